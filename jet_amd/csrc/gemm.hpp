// gemm.hpp -- complex GEMM kernels of the contraction path (gfx950).
//
// Every contraction reduces to the batched "NT" product
//     C[b][m][n] = sum_k A[b][m][k] * B[b][n][k]
// with A and B stored k-fastest (the permutation stage produces them in that
// order).  This is the row-major NoTrans/NoTrans product of the reference
// (TensorHelpers.hpp:47-61) with the right operand kept as [right][common]
// so both MFMA operands are read along k.
#pragma once

#include "errors.hpp"

#include <cstdint>

namespace jet_hip {

struct GemmArgs {
    const void *A;
    const void *B;
    void *C;
    int64_t M, N, K, batch;
    int64_t lda, ldb, ldc; // row strides in elements
    int64_t sA, sB, sC;    // batch strides in elements (0 = broadcast)
    int variant = 0;       // tile / thread-mapping variant (GemmChoice)
    // FP32 and FP64 matrix-core products: slices of slice_k k each write a
    // result of their own, slice_stride elements apart (tile_slices).
    int slices = 1;
    int64_t slice_k = 0, slice_stride = 0;
};

// Kernel families (also reported by jet_hip_plan_info).
enum GemmKernel {
    kGemmSmall = 0,     // VALU, one thread per output element
    kGemmSmallRed = 1,  // VALU, one block per output element (long K)
    kGemmF32Mfma = 2,   // FP32 products on the matrix cores: three BF16 pieces of
                        // each value and six products (gemm_f32x6.hip), or 4M
                        // complex on v_mfma_f32_16x16x4_f32 where that does
                        // not apply (k < 16)
    kGemmF64Mfma = 3,   // 4M complex on v_mfma_f64_16x16x4_f64 (gemm_f64.hip)
    kGemmBf16x3 = 4,    // 3M complex, split-BF16, v_mfma_f32_16x16x32_bf16
    kGemmBf16x4m = 5,   // 4M complex, split-BF16, v_mfma_f32_16x16x32_bf16
    kGemmSplitK = 6,    // VALU, few outputs and long k: k split over blocks,
                        // partial sums combined in FP64
    kGemmF16x4m = 7,    // 4M complex, split-FP16 with per-row power-of-two
                        // scales, v_mfma_f32_16x16x32_f16
};

// A GEMM kernel family and its tile (or thread-mapping) variant.  Variant 0
// lets the launcher pick by shape; the others force one form:
//   kGemmF32Mfma              1: 128x128  2: 64x128  3: 128x64 block tiles of
//                             the FP32 MFMA kernel
//   kGemmF64Mfma              1: its tile forms by shape
//   kGemmBf16x4m, kGemmF16x4m 1: 128x128  2: 128x192 block tiles
//                             3: 128x128 persistent (one work-group per
//                             CU walking the tiles)
//   kGemmSmall                1: one thread per output  2: short-K column
//                             blocks (K <= 16)  3: short-K row threads (K <= 16)
//   kGemmSmallRed, kGemmSplitK, kGemmBf16x3   1: their one form
struct GemmChoice {
    int kernel = kGemmSmall;
    int variant = 0;
};

// Variants 1..gemm_variants(kernel) exist for each kernel family.
int gemm_variants(int kernel);
// Whether the choice computes this shape in precision mode `mode` (0 fp32,
// 1 split-bf16 3M, 2 fp64, 3 split-bf16 4M, 4 split-fp16 4M): the data type
// matches, the kernel's grid fits and its operand limits hold.
bool gemm_choice_valid(int mode, int64_t M, int64_t N, int64_t K, int64_t batch,
                       GemmChoice c);

// Split-K: k range per block, and the FP64 partial-sum buffer it needs.
constexpr int64_t kSplitKChunk = 8192;
inline int64_t splitk_chunk(int64_t K)
{
    const int64_t c = ceil_div(K, 65535);
    return c > kSplitKChunk ? c : kSplitKChunk;
}
inline int64_t splitk_partials(int64_t outputs, int64_t K)
{
    return outputs * ceil_div(K, splitk_chunk(K));
}

// Whether the FP32 products run on the BF16 matrix cores: the lane offsets are
// 32 bits (rows to 2^21 k), and less than one k step is left to the FP32 MFMA kernel.
// Narrow products waste most of a 32x32 block here, but more of the FP32 kernel's
// 128x64 tiles (12x3000x1000 14.0 us and 160, 256x10x87 7.7 and 18.9, batches of 300
// 5x5x64 6.0 and 22).
inline bool f32x6_shape(int64_t M, int64_t N, int64_t K)
{
    return M >= 1 && N >= 1 && K >= 16 && K <= (int64_t(1) << 21);
}

// 4M split products with few 128x128 tiles: slices of k (at least 256 each)
// that fill the 256 CUs, each slice a result of its own, summed afterwards in
// FP64 (launch_sum_chunks).  One slice where half the CUs have a tile
// already, or for the other tile forms (variant > 1).  Measured with the operand
// passes: 140x150x12000 583 -> 58 us, 1024^3 72.6 -> 48.2.
inline int64_t x4m_slices(int64_t M, int64_t N, int64_t K, int64_t batch, int variant)
{
    const int64_t tiles = ceil_div(M, 128) * ceil_div(N, 128) * batch;
    const int64_t kt = ceil_div(K, 32);
    if (variant > 1 || tiles > 128 || kt < 16) return 1;
    const int64_t want = 256 / tiles < kt / 8 ? 256 / tiles : kt / 8;
    return ceil_div(kt, ceil_div(kt, want)); // no slice empty
}

// A tile form of the FP32 (gemm_f32x6.hip) or FP64 (gemm_f64.hip) matrix-core
// products, and the time in us that a product takes with it.  A CU that gets
// `per_cu` tiles (the fullest) runs them `occ` at a time; a stage of `kt` k
// takes `alone` us while they wait on latency and `full` us of matrix-core
// time per tile, and a tile costs `out` us beside its stages (prologue and
// stores).  Measured on shapes with one tile per CU and with many; FP32,
// predicted / measured us: 1024^3 62, 53, 56 / 65, 54, 55 for the 64x64, 64x32
// and 32x32 tiles, 2048^3 301, 353 / 308, 369 for 128x128 and 64x64,
// 256x65536x256 160, 173 / 160, 177 for 256x128 and 128x128; FP64: 1024^3 137,
// 137 / 144, 148 for 32x32 with and without slices in the tile, 1536x1536x512
// 158, 252 / 160, 256 for 32x32 and 128x128.  The FP32 choices are within 6% of
// the best of eleven forms timed on 19 shapes from 64^3 to 4096x4096x1024.
struct TileForm {
    int bm, bn, kt, occ;
    float alone, full, out;
};
constexpr TileForm kF32x6Forms[] = {{256, 128, 16, 1, 3.33f, 4.27f, 11.5f},
                                    {128, 128, 16, 1, 1.89f, 2.3f, 6.5f},
                                    {64, 64, 16, 3, 0.92f, 0.69f, 1.f},
                                    {64, 32, 32, 2, 1.05f, 0.77f, 0.6f},
                                    {32, 32, 64, 2, 1.1f, 0.8f, 0.4f}};
// Rows that are not 16-byte aligned (odd k): four times the load instructions, and
// registers for one work-group of the 32x32 form on a CU.  Predicted / measured us:
// 1030x1030x1001 106 / 100, 2050x1030x255 44 / 48 (64x64), 300x513x405 12.5 / 14.5
// (32x32; chosen by the aligned forms' times before, 1030x1030x17 took 24.8, now 8.3).
constexpr TileForm kF32x6DwordForms[] = {{64, 64, 16, 2, 1.2f, 0.81f, 1.75f},
                                         {32, 32, 64, 1, 1.25f, 1.23f, 3.7f}};
constexpr TileForm kF64Forms[] = {{128, 128, 8, 1, 3.8f, 3.92f, 9.f},
                                  {32, 32, 16, 3, 0.70f, 0.523f, 0.83f},
                                  {32, 32, 8, 6, 0.445f, 0.264f, 0.39f}};
// Tiles of a launch: fewer than 2^32 threads at 512 each.  Products with more of
// every form's take the first form, whose tiles are the largest.
constexpr int64_t kMaxTiles = (int64_t(1) << 23) - 1;
template <int COUNT>
inline double tile_time(const TileForm (&forms)[COUNT], int64_t M, int64_t N, int64_t K,
                        int64_t batch, int *form)
{
    constexpr int64_t kCus = 256;
    double best = -1.0;
    if (form) *form = 0;
    for (int i = 0; i < COUNT; i++) {
        const TileForm &f = forms[i];
        if (i > 0 && ceil_div(M, f.bm) * ceil_div(N, f.bn) > kMaxTiles) continue;
        const int64_t per_cu = ceil_div(ceil_div(M, f.bm) * ceil_div(N, f.bn) * batch, kCus);
        const double wait = f.alone * double(ceil_div(per_cu, f.occ)), work = f.full * double(per_cu);
        const double us = double(ceil_div(K, f.kt)) * (wait > work ? wait : work) +
                          f.out * double(per_cu);
        if (best < 0.0 || us < best) {
            best = us;
            if (form) *form = i;
        }
    }
    return best;
}

// Slices of k (multiples of 64) where a few tiles would walk a long k alone;
// their results are summed in FP64 (launch_sum_chunks: a launch, and the
// results read back at 3 TB/s).  time: with the sum.
template <int COUNT>
inline int tile_slices(const TileForm (&forms)[COUNT], int elem_bytes, int64_t M, int64_t N,
                       int64_t K, int64_t batch, double *time)
{
    int best = 1;
    double best_us = tile_time(forms, M, N, K, batch, nullptr);
    for (int s = 2; s <= 64 && K / s >= 128; s *= 2) {
        const int64_t k = ceil_div(ceil_div(K, s), 64) * 64;
        if (ceil_div(K, k) != s) continue;
        const double us = tile_time(forms, M, N, k, batch * s, nullptr) + 4.0 +
                          double(s) * double(batch) * double(M) * double(N) * elem_bytes / 3e6;
        if (us < 0.9 * best_us) {
            best_us = us;
            best = s;
        }
    }
    if (time) *time = best_us;
    return best;
}

// The FP32 products' slices.  Up to 2^17 outputs with a side of at most 128 and a
// long k were sums over the 256 threads of a work-group (kGemmSmallRed), whose
// error grows more slowly with k than a chain's: slices of at most 256 k, from 8192
// k on 512, keep the error below theirs on all tiles but the widest, which have
// one sum per output (4096x32x16384 2.2e-7 as a reduction, 2.8e-7 in four slices,
// 1.3e-7 in 32, 120 -> 161 us; 32x4096x1024 9.4e-8, in two slices 1.0e-7, in four
// 7.9e-8).
inline int f32x6_slices(int64_t M, int64_t N, int64_t K, int64_t batch, double *time)
{
    const int s = tile_slices(kF32x6Forms, 8, M, N, K, batch, time);
    if (K < 1024 || (M > 128 && N > 128) || batch * M * N > (int64_t(1) << 17)) return s;
    const int64_t parts = ceil_div(K, int64_t(K < 8192 ? 256 : 512)), least = parts < 64 ? parts : 64;
    const int64_t k = ceil_div(ceil_div(K, least), 64) * 64;
    if (least <= s || ceil_div(K, k) != least) return s; // none empty
    int form = 0;
    (void)tile_time(kF32x6Forms, M, N, k, batch * least, &form);
    return form == 0 ? s : int(least);
}

// Rows and k of the split-BF16 operand planes are padded to these multiples.
constexpr int kSplitRowPad = 16;
constexpr int kSplitKPad = 32;
// Longest padded k of the 4M split kernels: their per-lane load offsets
// within a tile of up to 192 operand rows stay below 2^32 bytes.
constexpr int64_t kX4mMaxK = int64_t(1) << 21;

// A split-FP16 operand read straight from an unpermuted source: the
// permutation to [batch][rows][K] is a permutation of the linear index bits
// (every extent a power of two), and one pass gathers LDS tiles made of all
// K bits and `xr` row bits -- the row bits that hold the source's lowest
// address bits, so reads are contiguous runs -- takes each tile row's
// maximum and writes the four planes and the scale (no permuted copy).
//   u: tile index in source order (bit j -> source bit su[j], ascending);
//   v: tile index in target order (bits 0..log2k-1 = k, then the tile's row
//      bits; u-bit j is v-bit u2v[j]; tile row bit i is row bit vrow[i]);
//   w: tile number (bit j -> source bit wsrc[j] and row bit wrow[j]).
constexpr int kGatherTileBits = 11; // 2048-element tiles (4096: 40% slower)
struct SplitGather {
    int tb = 0, log2k = 0, xr = 0, nw = 0;
    int8_t su[16] = {}, u2v[16] = {}, vrow[16] = {};
    int8_t wsrc[64] = {}, wrow[64] = {};
};

// A small contraction of power-of-two extents in one VALU pass that reads A
// and B and writes C in their own mode orders (no permuted copies, one
// launch instead of up to four).  Each group of modes (batch, left, right,
// common) is linearised with its last mode fastest; bit i of a group index
// sits at bit pos[i] of the element offset in the operand (row-major, every
// extent a power of two, so the modes' digits occupy disjoint bit ranges).
constexpr int kFusedMaxBits = 24;  // bits per group
constexpr int kFusedMaxLog2K = 12; // two words of fields (GroupBlock)
struct FusedBits {
    int n = 0;
    int8_t pos[kFusedMaxBits] = {};
};
struct FusedSmall {
    int lb = 0, lm = 0, ln = 0, lk = 0; // log2 of batch, M, N, K
    FusedBits a_b, a_m, a_k, b_b, b_n, b_k, c_b, c_m, c_n;
};

// One work-group's share of a group of independent small contractions that
// run in one launch (grouped_small_kernel): 256 >> lanes outputs of one
// contraction, from output `first` on, 2^lanes lanes per output.  a, b and c
// are slots of the pointer table that the launch is given.  An output's index
// holds its n, m and batch bits, lowest first; bit i goes to the address bit
// packed as the i-th five-bit field (six to a word) of oc, and of oa (ob)
// where the operand has it (mask_a, mask_b); k bits likewise in ka and kb.
constexpr int kGroupMaxLog2K = 10;
constexpr int kGroupMaxLog2Outputs = 14; // results kept apart from the arena's reuse
constexpr int kGroupMaxLog2Work = 20;    // outputs * K
constexpr int kSmallMaxLog2Outputs = 24; // four words of fields
struct GroupBlock {
    int32_t a = 0, b = 0, c = 0;
    int32_t first = 0, lanes = 0;
    int16_t lo = 0, lk = 0; // log2 of outputs and K
    int32_t wide = 0;       // complex64: a (1), b (2), c (4) hold FP64 values
    uint32_t mask_a = 0, mask_b = 0;
    uint32_t oa[4] = {}, ob[4] = {}, oc[4] = {};
    uint32_t ka[2] = {}, kb[2] = {};
};
// The record of a fused small contraction (lb + lm + ln <=
// kSmallMaxLog2Outputs); lanes, first and the slots are the caller's.
GroupBlock group_record(const FusedSmall &f);
// Lanes per output, at most `most` (log2): while each keeps four k and the
// contraction stays within 2^log2_threads threads.
inline int group_lanes(const GroupBlock &g, int most, int log2_threads)
{
    int lanes = 0;
    while (lanes < most && g.lk - lanes > 2 && g.lo + lanes < log2_threads) lanes++;
    return lanes;
}

// Split-BF16 operand: planes re hi/lo, im hi/lo[, re+im hi/lo].
//  * planar (3M kernel, six planes): plane p is [batch][rows_p][k_p] bf16 at
//    offset p * plane_elems;
//  * interleaved (4M kernel, four planes): [batch][rows_p][k_p / 32][4][32]
//    bf16, i.e. the four planes of one row and one 32-wide k tile form 256
//    contiguous bytes (two full cache lines per row and k tile).
//  * split-FP16 (4M kernel, four interleaved fp16 planes): each row r of
//    batch b is scaled by 2^(14 - e) before the split, e the exponent of the
//    row's largest |re| or |im|; rowmax[b * rows_p + r] holds that largest
//    magnitude's FP32 bit pattern and scale[b * rows_p + r] = 2^(e - 14), the
//    factor the GEMM applies to its outputs.
struct SplitOperand {
    void *base;
    int64_t rows_p, k_p, batch, plane_elems;
    int planes;
    int interleaved;
    uint32_t *rowmax = nullptr; // split-FP16 only
    float *scale = nullptr;     // split-FP16 only
};

inline int64_t split_plane_elems(int64_t batch, int64_t rows, int64_t k)
{
    const int64_t rp = ceil_div(rows, kSplitRowPad) * kSplitRowPad;
    const int64_t kp = ceil_div(k, kSplitKPad) * kSplitKPad;
    return batch * rp * kp;
}

// The built-in kernel rule for a shape and precision mode (0 = fp32/
// complex64, 1 = split-bf16 3M/complex64, 2 = fp64/complex128, 3 = split-bf16
// 4M/complex64, 4 = split-fp16 4M/complex64), variant 0.  Plans use the
// autotuned table (tuning.hpp) and fall back to this rule only for shapes
// the table does not cover.
int choose_gemm_kernel(int mode, int64_t M, int64_t N, int64_t K,
                       int64_t batch);

#if defined(__HIPCC__)
// `partials` (splitk_partials(batch*M*N, K) pairs of doubles) is only used by
// kGemmSplitK.
void launch_gemm(int kernel, int elem_bytes, const GemmArgs &g,
                 hipStream_t stream, void *partials = nullptr);
// The FP32 products on the BF16 matrix cores (gemm_f32x6.hip).
void launch_f32x6(const GemmArgs &g, hipStream_t stream);
// complex128 products (gemm_f64.hip).
void launch_f64(const GemmArgs &g, hipStream_t stream);
// src: complex64 [batch][rows][k] with row stride ld and batch stride s.
void launch_split_bf16(const void *src, int64_t rows, int64_t k, int64_t ld,
                       int64_t s, int64_t batch, const SplitOperand &dst,
                       hipStream_t stream);
void launch_gemm_bf16x4m(const SplitOperand &a, const SplitOperand &b, int64_t K_true,
                         void *C, int64_t M, int64_t N, int64_t ldc,
                         int64_t sC, int64_t batch, bool a_bcast, bool b_bcast,
                         hipStream_t stream, int variant = 0, int64_t slices = 1);
// Row maxima then the scaled fp16 planes of a split-FP16 operand.
void launch_split_f16(const void *src, int64_t rows, int64_t k, int64_t ld,
                      int64_t s, int64_t batch, const SplitOperand &dst,
                      hipStream_t stream);
// The same planes and scales gathered from an unpermuted source (SplitGather).
void launch_split_f16_gather(const void *src, const SplitGather &g, const SplitOperand &dst,
                             hipStream_t stream);
void launch_gemm_f16x4m(const SplitOperand &a, const SplitOperand &b, int64_t K_true,
                        void *C, int64_t M, int64_t N, int64_t ldc,
                        int64_t sC, int64_t batch, bool a_bcast, bool b_bcast,
                        hipStream_t stream, int variant = 0, int64_t slices = 1);
// n_blocks consecutive blocks of one group; `pointers` is the device table
// that their slots index.
void launch_grouped_small(const GroupBlock *blocks, int n_blocks, const void *const *pointers,
                          int elem_bytes, double flops, hipStream_t stream);
// pointers[first + i] = values[i] on the device, in stream order (the values
// travel as kernel arguments).
void launch_set_pointers(const void **pointers, const void *const *values, int n,
                         hipStream_t stream);
void launch_gemm_bf16x3(const SplitOperand &a, const SplitOperand &b, int64_t K_true,
                        void *C, int64_t M, int64_t N, int64_t ldc,
                        int64_t sC, int64_t batch, bool a_bcast, bool b_bcast,
                        hipStream_t stream);
// C = contract(A, B) through FusedSmall offsets.
void launch_fused_small(const FusedSmall &f, int elem_bytes, const void *a, const void *b,
                        void *c, hipStream_t stream);
#endif

} // namespace jet_hip
