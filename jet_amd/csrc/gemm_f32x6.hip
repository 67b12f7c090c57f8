// gemm_f32x6.hip -- complex64 GEMM at FP32 accuracy on the BF16 matrix cores
// (gfx950): the FP32 products of every precision mode.
//
// Each FP32 value is the sum of three BF16 pieces, 2^16 x = h + m + l (rounded
// to nearest: 3 x 8 significant bits, so the sum is exact; unscaled, the pieces
// of values under 2^-110 would fall below BF16's smallest subnormal), and a
// real product keeps the six terms hh, hm, mh, hl, lh, mm; the dropped ones are
// below 2^-24 of it.  Values from 2^111 on and sums from 2^95 on leave the scaled
// range, and with infinities and NaN their 32x32 blocks are computed again with
// the FP32 instruction (all of 4096^3 10.8 ms).  The scaling is one VALU
// instruction per value (4096^3 2380 -> 2405 us, 64x32 tiles 3% more).
//
// Four real products make 24 v_mfma_f32_32x32x16_bf16 per 32x32
// block and 16 k: at BF16's rate (16 times FP32's on the same matrix cores)
// that is 2.7 times the FP32 MFMA rate.  Measured (TFLOP/s of 8 M N K, FP32
// MFMA kernel before -> this one): 4096^3 121 -> 248, 4096x4096x1024 119 ->
// 238, 256x65536x256 113 -> 216, 1024^3 52 -> 166; 512^3 (which the VALU
// kernel ran) 368 -> 12 us.  Errors against 64 bits (normwise, random
// operands): 4096^3 1.6e-6 -> 1.4e-6, 1024^3 8.1e-7 -> 1.9e-7, 512^3 5.7e-7
// -> 9.8e-8, K = 64 7.4e-8 -> 5.6e-8: the accumulator takes fewer roundings
// per k than the K = 4 steps of the FP32 instruction, and (all tiles but the
// widest) the terms with a middle or low piece, 2^-8 of the product and
// less, sum in accumulators of their own, so that the main ones are rounded
// twice per 16 k.
//
// The operands stay FP32 in memory and in LDS (8 bytes per complex value:
// three pieces of each part would be 12) and are split in registers after
// the LDS read, 6.5 VALU instructions per value; there is no operand pass and
// no workspace.  A wave issues a VALU instruction every 8 cycles and an MFMA holds
// the matrix cores for 32, so a split hides behind the products where it is
// little work and stands beside them: the wide tiles give a wave 128x64 (64x64)
// outputs and one SIMD, 3.5 VALU instructions per MFMA, and read and split the
// next operands during the products (4096^3, eight waves of 64x64 that split
// first: 2520 us, matrix cores busy 60% of the cycles; four pipelined waves of 128x64:
// 2230, 75%, at a clock lowered for power).  Small tiles keep two or three
// waves per SIMD instead; pipelined they measured the same or less.
#include "common.hpp"
#include "gemm.hpp"
#include "gemm_device.hpp"
#include "profiler.hpp"

#include <algorithm>

namespace jet_hip {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// Three BF16 pieces of eight consecutive k of one operand row.
struct Pieces {
    u32x4 h, m, l;
};

__device__ __forceinline__ uint32_t pack_bf16(float a, float b)
{
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
}
__device__ __forceinline__ float low_bf16(uint32_t p) { return __uint_as_float(p << 16); }
__device__ __forceinline__ float high_bf16(uint32_t p)
{
    return __uint_as_float(p & 0xffff0000u);
}

// 2^16 x = h + m + l, each rounded to nearest: 24 significant bits, so the sum is
// exact, and the last bit of any FP32 number is at least BF16's smallest
// subnormal, which the conversions and the products keep.  Sums of products
// carry 2^32 until they are stored.
constexpr float kScale = 0x1p16f, kUnscale = 0x1p-32f;
__device__ __forceinline__ void split_pair(float a, float b, uint32_t &h, uint32_t &m, uint32_t &l)
{
    h = pack_bf16(a * kScale, b * kScale);
    const float ra = fmaf(a, kScale, -low_bf16(h)), rb = fmaf(b, kScale, -high_bf16(h));
    m = pack_bf16(ra, rb);
    l = pack_bf16(ra - low_bf16(m), rb - high_bf16(m));
}

__device__ __forceinline__ f32x16 mma(const u32x4 &a, const u32x4 &b, f32x16 c)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// BM x BN output tile, WM x WN waves of 32x32 blocks; with WK > 1 the waves
// also split every stage's k (WK slices of 16, summed through LDS at the
// end): small products have few tiles, and a tile's time is its k steps'
// latency.  Stages of 16 WK k come straight from global memory into NS LDS
// buffers with global_load_lds_dwordx4, two stages ahead with three buffers.
// Rows past M or N repeat the last row (their outputs are not stored); k past
// K is zeroed after the LDS read.  DW: dwords per lane of a load, 4, or 1 for
// rows that are not 16-byte aligned (odd k or strides).
template <int BM, int BN, int WM, int WN, int WK, int NS, bool DUAL, int DW>
__global__ __launch_bounds__(64 * WM * WN * WK,
                             WM * WN * WK / 4) void cgemm_f32x6_kernel(GemmArgs g)
{
    typedef __attribute__((address_space(3))) void lds_void;
    constexpr int NW = WM * WN * WK;
    constexpr int KT = 16 * WK; // complex k per stage
    constexpr int WTM = BM / WM, WTN = BN / WN;
    constexpr int FM = WTM / 32, FN = WTN / 32;
    constexpr int PER = 4 / DW; // loads per 16-byte chunk
    constexpr int A_IN = BM * 8 * WK * PER / (64 * NW);
    constexpr int B_IN = BN * 8 * WK * PER / (64 * NW);
    constexpr int L = A_IN + B_IN;
    constexpr int STAGE = (BM + BN) * 8 * WK; // 16-byte chunks
    static_assert(A_IN * 64 * NW == BM * 8 * WK * PER && B_IN * 64 * NW == BN * 8 * WK * PER,
                  "tile");
    static_assert(L < 64, "one stage of loads fits the wait counter");
    static_assert(NS == 2 || NS == 3, "two or three LDS stages");
    static_assert((WK - 1) * BM * BN * 8 <= STAGE * 16 * (NS == 2 ? 2 : 1), "wave sums fit");
    __shared__ f32x4 S0[NS == 2 ? 2 * STAGE : STAGE];
    __shared__ f32x4 S1x[NS == 2 ? 1 : STAGE], S2x[NS == 2 ? 1 : STAGE];
    f32x4 *const S1 = NS == 2 ? S0 + STAGE : S1x, *const S2 = NS == 2 ? S0 : S2x;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wk = wave % WK, wmn = wave / WK;
    const int wm = wmn / WN, wn = wmn % WN;
    const int64_t bz = blockIdx.z;
    int64_t tm, tn;
    tile_coords(blockIdx.x, (g.M + BM - 1) / BM, (g.N + BN - 1) / BN, tm, tn);
    const int64_t m0 = tm * BM, n0 = tn * BN;
    const int64_t k_first = int64_t(blockIdx.y) * g.slice_k; // of this slice
    const int K = int(g.slices > 1 ? min(g.K - k_first, g.slice_k) : g.K);
    const char *At = static_cast<const char *>(g.A) + (bz * g.sA + m0 * g.lda + k_first) * 8;
    const char *Bt = static_cast<const char *>(g.B) + (bz * g.sB + n0 * g.ldb + k_first) * 8;

    // One load instruction fills 64 consecutive chunks (or dwords) of a
    // stage; a stage is [k sixteenth][row of A, then of B][8 chunks], the
    // chunk of a row in slot chunk ^ (row & 7).
    uint32_t off[L]; // byte offset of the lane's row, and dword of its value
    int ck[L];       // the lane's first k
#pragma unroll
    for (int i = 0; i < L; i++) {
        const bool isa = i < A_IN;
        const int load = wave * (isa ? A_IN : B_IN) + (isa ? i : i - A_IN);
        const int64_t rows = isa ? g.M - m0 : g.N - n0;
        const int R = isa ? BM : BN;
        int r, kk;
        if (DW == 4) { // eight rows a load: the lane's k is the same in every load
            r = load * 8 % R + (lane >> 3), kk = load * 8 / R;
            ck[i] = 16 * kk + 2 * ((lane & 7) ^ (lane >> 3));
        }
        else {
            const int p = (load * 64 + lane) / PER;
            r = (p >> 3) % R, kk = (p >> 3) / R;
            ck[i] = 16 * kk + 2 * ((p & 7) ^ (r & 7)) + (lane % PER) * DW / 2;
        }
        const int64_t rr = r < rows ? r : rows - 1;
        off[i] = uint32_t(rr * (isa ? g.lda : g.ldb) * 8) + (DW == 4 ? 0 : ((lane % PER) & 1) * 4);
    }
    auto issue = [&](int kt, f32x4 *s) __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        const int k0 = kt * KT;
#pragma unroll
        for (int i = 0; i < L; i++) {
            const int k = k0 + ck[i];
            const uint32_t o = off[i] + (k < K ? uint32_t(k) * 8u : 0u);
            const void *src = (i < A_IN ? At : Bt) + uint64_t(o);
            float *dst = i < A_IN ? reinterpret_cast<float *>(s) + (wave * A_IN + i) * 64 * DW
                                  : reinterpret_cast<float *>(s + BM * 8 * WK) +
                                        (wave * B_IN + i - A_IN) * 64 * DW;
            if constexpr (DW == 4)
                __builtin_amdgcn_global_load_lds(src, (lds_void *)dst, 16, 0, 0);
            else
                __builtin_amdgcn_global_load_lds(src, (lds_void *)dst, 4, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };

    // DUAL: the products with a middle or low piece in sums of their own.
    constexpr int DM = DUAL ? FM : 1, DN = DUAL ? FN : 1;
    f32x16 cr[FM][FN], ci[FM][FN], dr[DM][DN], di[DM][DN];
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++) {
            cr[i][j] = f32x16{};
            ci[i][j] = f32x16{};
            if (DUAL) {
                dr[i % DM][j % DN] = f32x16{};
                di[i % DM][j % DN] = f32x16{};
            }
        }

    const int q = lane >> 5, j = lane & 31;
    // Eight complex values of one row from LDS, as the pieces of their real
    // and imaginary parts; kv: valid k of this lane's eight.
    auto fetch = [&](const f32x4 *row, int sw, bool tail, int kv, Pieces &re,
                     Pieces &im) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < 4; c++) {
            f32x4 v = row[(q * 4 + c) ^ sw];
            if (tail && 2 * c >= kv) v.x = v.y = 0.f;
            if (tail && 2 * c + 1 >= kv) v.z = v.w = 0.f;
            uint32_t h, m, l;
            split_pair(v.x, v.z, h, m, l);
            re.h[c] = h, re.m[c] = m, re.l[c] = l;
            split_pair(v.y, v.w, h, m, l);
            im.h[c] = h, im.m[c] = m, im.l[c] = l;
        }
    };
    // The products of one block: smallest terms first, the two accumulators by
    // turns.
    auto products = [&](int fm, int fn, const Pieces &ar, const Pieces &ai, const Pieces &br,
                        const Pieces &bi) __attribute__((always_inline)) {
        Pieces ni;
        ni.h = ai.h ^ 0x80008000u;
        ni.m = ai.m ^ 0x80008000u;
        ni.l = ai.l ^ 0x80008000u;
        f32x16 x = DUAL ? dr[fm % DM][fn % DN] : cr[fm][fn];
        f32x16 y = DUAL ? di[fm % DM][fn % DN] : ci[fm][fn];
        auto term = [&](u32x4 Pieces::*a, u32x4 Pieces::*b) __attribute__((always_inline)) {
            x = mma(ar.*a, br.*b, x);
            y = mma(ar.*a, bi.*b, y);
            x = mma(ni.*a, bi.*b, x);
            y = mma(ai.*a, br.*b, y);
        };
        term(&Pieces::l, &Pieces::h);
        term(&Pieces::h, &Pieces::l);
        term(&Pieces::m, &Pieces::m);
        term(&Pieces::m, &Pieces::h);
        term(&Pieces::h, &Pieces::m);
        if (DUAL) {
            dr[fm % DM][fn % DN] = x;
            di[fm % DM][fn % DN] = y;
            x = cr[fm][fn];
            y = ci[fm][fn];
        }
        term(&Pieces::h, &Pieces::h);
        cr[fm][fn] = x;
        ci[fm][fn] = y;
    };
    auto fetch_a = [&](const f32x4 *s, int fm, bool tail, int kt, Pieces &re,
                       Pieces &im) __attribute__((always_inline)) {
        const int r = wm * WTM + fm * 32 + j;
        fetch(s + (BM * wk + r) * 8, r & 7, tail, K - kt * KT - 16 * wk - 8 * q, re, im);
    };
    auto fetch_b = [&](const f32x4 *s, int fn, bool tail, int kt, Pieces &re,
                       Pieces &im) __attribute__((always_inline)) {
        const int r = wn * WTN + fn * 32 + j;
        fetch(s + (BM * WK + BN * wk + r) * 8, r & 7, tail, K - kt * KT - 16 * wk - 8 * q, re,
              im);
    };

    const int nk = (K + KT - 1) / KT, nfull = K / KT;
    // vmcnt(L), vmcnt(2 L): the loads of later stages may stay in flight.
    constexpr int kWaitAll = 0x0f70;
    constexpr int kWaitPrev = kWaitAll | (L & 15) | ((L >> 4) << 14);
    constexpr int kWaitTwo = kWaitAll | ((2 * L) & 15) | (((2 * L) >> 4) << 14);
    if constexpr (FM > 1) {
        // One wave per SIMD: the next operand of its own is read and split
        // beside each block's products, in the order in which registers get
        // free: B's second half beside (0, 0), A's row fm + 1 beside (fm, 1), and
        // beside the last row the next stage's A row 0 and first half of B.
        // That stage is in LDS for every wave once each has waited for its own
        // loads; every wave is then past its reads of this stage, whose buffer
        // takes the stage after the next two.
        static_assert(NS == 3 && WK == 1 && FN == 2 && DW == 4 && 2 * L < 64, "pipelined form");
        Pieces ar, ai, br[2], bi[2];
        // 24 products: six before the values just read are used, then by turns
        // with the VALU.
        auto interleave = [&]() __attribute__((always_inline)) {
            __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 6, 0);
#pragma unroll
            for (int i = 6; i < 24; i++) {
                __builtin_amdgcn_sched_group_barrier(0x002, 7, 0);
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        // Stage kt (in s) into LDS for every wave: own loads, zeros for k past K
        // (K is even here), own reads of the stage before; then the barrier.
        auto arrive = [&](int kt, f32x4 *s) __attribute__((always_inline)) {
            __builtin_amdgcn_sched_barrier(0);
            if (kt + 1 < nk) {
                if (kt == 0 && nk > 2)
                    __builtin_amdgcn_s_waitcnt(kWaitTwo);
                else
                    __builtin_amdgcn_s_waitcnt(kWaitPrev);
            }
            else {
                __builtin_amdgcn_s_waitcnt(kWaitAll);
                if (kt < nk && nk > nfull) {
                    asm volatile("" ::: "memory");
#pragma unroll
                    for (int i = 0; i < L; i++)
                        if (kt * KT + ck[i] >= K)
                            s[(i < A_IN ? wave * A_IN + i : BM / 8 + wave * B_IN + i - A_IN) * 64 +
                              lane] = f32x4{};
                }
            }
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt(0xc07f); // lgkmcnt(0)
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
        };
        // After the last stage what is read and split is not used.
        auto stage = [&](int kt, f32x4 *s, f32x4 *next) __attribute__((always_inline)) {
            Pieces nr, ni;
            fetch_b(s, 1, false, kt, br[1], bi[1]);
            products(0, 0, ar, ai, br[0], bi[0]);
            interleave();
#pragma unroll
            for (int fm = 0; fm + 1 < FM; fm++) {
                fetch_a(s, fm + 1, false, kt, nr, ni);
                products(fm, 1, ar, ai, br[1], bi[1]);
                interleave();
                ar = nr, ai = ni;
                if (fm + 2 < FM) {
                    products(fm + 1, 0, ar, ai, br[0], bi[0]);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            // split before the branches, beside the products above
            asm volatile(""
                         : "+v"(ar.h), "+v"(ar.m), "+v"(ar.l), "+v"(ai.h), "+v"(ai.m), "+v"(ai.l));
            arrive(kt + 1, next);
            if (kt + 3 < nk) issue(kt + 3, s);
            fetch_a(next, 0, false, kt + 1, nr, ni);
            products(FM - 1, 0, ar, ai, br[0], bi[0]);
            interleave();
            fetch_b(next, 0, false, kt + 1, br[0], bi[0]);
            products(FM - 1, 1, ar, ai, br[1], bi[1]);
            interleave();
            ar = nr, ai = ni;
        };
        issue(0, S0);
        if (nk > 1) issue(1, S1);
        if (nk > 2) issue(2, S2);
        arrive(0, S0);
        fetch_b(S0, 0, false, 0, br[0], bi[0]);
        fetch_a(S0, 0, false, 0, ar, ai);
        int kt = 0;
        for (; kt + 3 <= nk; kt += 3) {
            stage(kt, S0, S1);
            stage(kt + 1, S1, S2);
            stage(kt + 2, S2, S0);
        }
        for (int b = 0; kt < nk; kt++, b++) stage(kt, b == 0 ? S0 : S1, b == 0 ? S1 : S2);
    }
    else {
        auto compute = [&](const f32x4 *s, bool tail, int kt) __attribute__((always_inline)) {
            static_assert(FN == 1, "one block per wave");
            Pieces ar, ai, br, bi;
            fetch_b(s, 0, tail, kt, br, bi);
            fetch_a(s, 0, tail, kt, ar, ai);
            products(0, 0, ar, ai, br, bi);
        };
        issue(0, S0);
        if (NS == 3 && nk > 1) issue(1, S1);
        // Stage kt is in LDS for every wave once each has waited for its own
        // loads; every wave is then also past its reads of stage kt - 1, whose
        // buffer takes stage kt + NS - 1.
        auto arrive = [&](int kt, f32x4 *next) __attribute__((always_inline)) {
            __builtin_amdgcn_sched_barrier(0);
            if (NS == 3 && kt + 1 < nk)
                __builtin_amdgcn_s_waitcnt(kWaitPrev);
            else
                __builtin_amdgcn_s_waitcnt(kWaitAll);
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
            if (kt + NS - 1 < nk) issue(kt + NS - 1, next);
        };
        int kt = 0;
        if (NS == 3) {
            for (; kt + 3 <= nfull; kt += 3) {
                arrive(kt, S2);
                compute(S0, false, kt);
                arrive(kt + 1, S0);
                compute(S1, false, kt + 1);
                arrive(kt + 2, S1);
                compute(S2, false, kt + 2);
            }
            // At most three stages are left; only the third is still to be issued.
            for (int b = 0; kt < nk; kt++, b++) {
                arrive(kt, S2);
                compute(b == 0 ? S0 : b == 1 ? S1 : S2, true, kt);
            }
        }
        else {
            for (; kt + 2 <= nfull; kt += 2) {
                arrive(kt, S1);
                compute(S0, false, kt);
                arrive(kt + 1, S0);
                compute(S1, false, kt + 1);
            }
            for (int b = 0; kt < nk; kt++, b++) {
                arrive(kt, b == 0 ? S1 : S0);
                compute(b == 0 ? S0 : S1, true, kt);
            }
        }
    }

    if (DUAL) {
#pragma unroll
        for (int i = 0; i < FM; i++)
#pragma unroll
            for (int j2 = 0; j2 < FN; j2++) {
                cr[i][j2] += dr[i % DM][j2 % DN];
                ci[i][j2] += di[i % DM][j2 % DN];
            }
    }
    if (WK > 1) {
        // The sums of the K slices, added in slice order by the first.
        __syncthreads();
        float2 *sums = reinterpret_cast<float2 *>(S0);
        constexpr int SUM = FM * FN * 16 * 64;
        if (wk > 0) {
#pragma unroll
            for (int fm = 0; fm < FM; fm++)
#pragma unroll
                for (int fn = 0; fn < FN; fn++)
#pragma unroll
                    for (int i = 0; i < 16; i++)
                        sums[((wk - 1) * WM * WN + wmn) * SUM + ((fm * FN + fn) * 16 + i) * 64 +
                             lane] = float2{cr[fm][fn][i], ci[fm][fn][i]};
        }
        __syncthreads();
        if (wk > 0) return;
        for (int w = 0; w < WK - 1; w++)
#pragma unroll
            for (int fm = 0; fm < FM; fm++)
#pragma unroll
                for (int fn = 0; fn < FN; fn++)
#pragma unroll
                    for (int i = 0; i < 16; i++) {
                        const float2 v = sums[(w * WM * WN + wmn) * SUM +
                                              ((fm * FN + fn) * 16 + i) * 64 + lane];
                        cr[fm][fn][i] += v.x;
                        ci[fm][fn][i] += v.y;
                    }
    }

    float2 *C = static_cast<float2 *>(g.C) + bz * g.sC + int64_t(blockIdx.y) * g.slice_stride;
    bool bad = false;
    const int64_t row0 = m0 + wm * WTM + 4 * q, col0 = n0 + wn * WTN + j;
    const bool whole = m0 + BM <= g.M && n0 + BN <= g.N;
#pragma unroll
    for (int fm = 0; fm < FM; fm++)
#pragma unroll
        for (int fn = 0; fn < FN; fn++) {
            if constexpr (FM > 1) {
                // Block by block: all sums at once do not fit beside the matrix
                // cores' registers, and a spilled value read back between stores
                // waits for them.
                asm volatile("" : "+a"(cr[fm][fn]), "+a"(ci[fm][fn]));
                __builtin_amdgcn_sched_barrier(0);
            }
            float2 *const p = C + (row0 + fm * 32) * g.ldc + col0 + fn * 32;
            auto store = [&](bool masked) __attribute__((always_inline)) {
                float2 *o = p;
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const float2 v{cr[fm][fn][i] * kUnscale, ci[fm][fn][i] * kUnscale};
                    bad |= !(__builtin_isfinite(v.x) && __builtin_isfinite(v.y));
                    if (!masked || (col0 + fn * 32 < g.N &&
                                    row0 + fm * 32 + 8 * (i / 4) + (i & 3) < g.M))
                        *o = v;
                    // to the next row: 1 further, or past the other half's 4
                    o += ((i & 3) == 3 ? 5 : 1) * g.ldc;
                }
            };
            if (whole)
                store(false);
            else
                store(true);
        }
    if (!__any(bad)) return;
    // An infinite or NaN input, or values too large for the scaled sums: 32x32
    // blocks with such an output run again with the FP32 instruction, straight
    // from the operands, and give those outputs.  Lane l holds row (column) l % 32
    // at k = l / 32; results lie as above.
#pragma unroll 1
    for (int e = 0; e < FM * FN; e++) {
        const int64_t r0 = m0 + wm * WTM + (e / FN) * 32, col = n0 + wn * WTN + (e % FN) * 32 + j;
        const int rows = int(min(g.M - r0 - 4 * q, int64_t(32))); // of this lane
        float2 *const c = C + (r0 + 4 * q) * g.ldc + col;
        uint32_t again = 0; // bit 8 (i / 4) + i % 4 for the lane's result i
#pragma unroll 1
        for (int r = 0; r < 32; r++)
            if (!(r & 4) && r < rows && col < g.N) {
                const float2 v = c[r * g.ldc];
                if (!(__builtin_isfinite(v.x) && __builtin_isfinite(v.y))) again |= 1u << r;
            }
        if (!__any(again != 0)) continue;
        const float2 *a = static_cast<const float2 *>(g.A) + bz * g.sA +
                          min(r0 + j, g.M - 1) * g.lda + k_first;
        const float2 *b = static_cast<const float2 *>(g.B) + bz * g.sB +
                          min(col, g.N - 1) * g.ldb + k_first;
        f32x16 re{}, im{};
#pragma unroll 4
        for (int k = 0; k < K; k += 2) {
            const int kk = min(k + q, K - 1);
            float2 x = a[kk], y = b[kk];
            if (k + q >= K) x = y = float2{0.f, 0.f};
            re = __builtin_amdgcn_mfma_f32_32x32x2f32(x.x, y.x, re, 0, 0, 0);
            im = __builtin_amdgcn_mfma_f32_32x32x2f32(x.x, y.y, im, 0, 0, 0);
            re = __builtin_amdgcn_mfma_f32_32x32x2f32(-x.y, y.y, re, 0, 0, 0);
            im = __builtin_amdgcn_mfma_f32_32x32x2f32(x.y, y.x, im, 0, 0, 0);
        }
        float2 *o = c;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            if (again >> (8 * (i / 4) + (i & 3)) & 1) *o = float2{re[i], im[i]};
            o += ((i & 3) == 3 ? 5 : 1) * g.ldc;
        }
    }
}

template <int BM, int BN, int WM, int WN, int WK, int NS, bool DUAL, int DW = 4>
void launch_tile(const GemmArgs &g, hipStream_t stream)
{
    JH_REQUIRE(ceil_div(g.M, BM) * ceil_div(g.N, BN) <= 0x7fffffff, "Too many tiles.");
    dim3 grid((unsigned)(ceil_div(g.M, BM) * ceil_div(g.N, BN)), (unsigned)g.slices,
              (unsigned)g.batch);
    hipLaunchKernelGGL((cgemm_f32x6_kernel<BM, BN, WM, WN, WK, NS, DUAL, DW>), grid,
                       dim3(64 * WM * WN * WK), 0, stream, g);
    JH_HIP(hipGetLastError());
}

} // namespace

void launch_f32x6(const GemmArgs &g, hipStream_t stream)
{
    const bool aligned = reinterpret_cast<uintptr_t>(g.A) % 16 == 0 &&
                         reinterpret_cast<uintptr_t>(g.B) % 16 == 0 && g.K % 2 == 0 &&
                         g.lda % 2 == 0 && g.ldb % 2 == 0 &&
                         (g.batch == 1 || (g.sA % 2 == 0 && g.sB % 2 == 0));
    const int64_t k = g.slices > 1 ? g.slice_k : g.K, count = g.batch * g.slices;
    int form = 0;
    if (!aligned) {
        (void)tile_time(kF32x6DwordForms, g.M, g.N, k, count, &form);
        if (form == 0)
            launch_tile<64, 64, 2, 2, 1, 3, true, 1>(g, stream);
        else
            launch_tile<32, 32, 1, 1, 4, 2, true, 1>(g, stream);
        return;
    }
    (void)tile_time(kF32x6Forms, g.M, g.N, k, count, &form);
    switch (form) {
    case 0:
        launch_tile<256, 128, 2, 2, 1, 3, false>(g, stream);
        break;
    case 1:
        launch_tile<128, 128, 2, 2, 1, 3, true>(g, stream);
        break;
    case 2:
        launch_tile<64, 64, 2, 2, 1, 3, true>(g, stream);
        break;
    case 3:
        launch_tile<64, 32, 2, 1, 2, 3, true>(g, stream);
        break;
    default:
        launch_tile<32, 32, 1, 1, 4, 2, true>(g, stream);
        break;
    }
}

} // namespace jet_hip
