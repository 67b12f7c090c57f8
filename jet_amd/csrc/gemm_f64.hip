// gemm_f64.hip -- complex128 GEMM on the FP64 matrix cores (gfx950).
//
// Re C = Ar.Br - Ai.Bi and Im C = Ar.Bi + Ai.Br: four v_mfma_f64_16x16x4 per
// 16x16 block and 4 k, whose lane l holds row (column) l % 16 of A (B) at k = l /
// 16 and gets rows l / 16 + 4 r of column l % 16.  Bound by the matrix cores (64
// cycles an instruction); stages come from global memory straight into three
// LDS buffers, two stages ahead, and every operand value is one 16-byte LDS read.
// Tile forms from 128x128 to 32x32 tiles whose waves split k (kF64Forms).
// Measured (us; register-staged 128x64 tiles, or the VALU, before):
// 4096x2048x1024 1332 -> 1003 (68.5 TFLOP/s), 1024^3 468 -> 144, 512^3 406 ->
// 25, 256^3 44.5 -> 13.6; with slices of k 128x1024x65536 17900 -> 1320, and a
// contraction of 2^11 x 2^12 over 2^11 with its reorderings 2920 -> 2090.
// Error against extended precision as before with 128x128 tiles (K = 1024
// 1.5e-15 both), smaller with 32x32 (1.1e-15).
#include "common.hpp"
#include "gemm.hpp"
#include "gemm_device.hpp"
#include "profiler.hpp"

namespace jet_hip {

namespace {

typedef double f64x2 __attribute__((ext_vector_type(2)));
typedef double f64x4 __attribute__((ext_vector_type(4)));

// BM x BN output tile, WM x WN waves; with WK > 1 the waves also split every
// stage's k (WK slices of 8, summed through LDS at the end).  Rows past M or N
// repeat the last row (their outputs are not stored); k past K is zeroed after
// the LDS read.  DW: dwords per lane of a load, 4, or 1 for operands that are
// not 16-byte aligned.
template <int BM, int BN, int WM, int WN, int WK, int DW>
__global__ __launch_bounds__(64 * WM * WN * WK, WM * WN * WK / 4) void cgemm_f64_kernel(GemmArgs g)
{
    typedef __attribute__((address_space(3))) void lds_void;
    constexpr int NW = WM * WN * WK;
    constexpr int KT = 8 * WK; // complex k per stage: 128 bytes of a row per slice
    constexpr int WTM = BM / WM, WTN = BN / WN;
    constexpr int FM = WTM / 16, FN = WTN / 16;
    constexpr int PER = 4 / DW;
    constexpr int A_IN = BM * 8 * WK * PER / (64 * NW);
    constexpr int B_IN = BN * 8 * WK * PER / (64 * NW);
    constexpr int L = A_IN + B_IN;
    constexpr int STAGE = (BM + BN) * 8 * WK; // complex values
    static_assert(A_IN * 64 * NW == BM * 8 * WK * PER && B_IN * 64 * NW == BN * 8 * WK * PER,
                  "tile");
    static_assert(L < 64, "one stage of loads fits the wait counter");
    static_assert(WK == 1 || (WK - 1) * BM * BN / FM <= STAGE, "wave sums fit");
    __shared__ f64x2 S0[STAGE], S1[STAGE], S2[STAGE];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wk = wave % WK, wmn = wave / WK;
    const int wm = wmn / WN, wn = wmn % WN;
    const int64_t bz = blockIdx.z;
    int64_t tm, tn;
    tile_coords(blockIdx.x, (g.M + BM - 1) / BM, (g.N + BN - 1) / BN, tm, tn);
    const int64_t m0 = tm * BM, n0 = tn * BN;
    const int64_t k_first = int64_t(blockIdx.y) * g.slice_k; // of this slice
    const int64_t K = g.slices > 1 ? min(g.K - k_first, g.slice_k) : g.K;
    const char *At = static_cast<const char *>(g.A) + (bz * g.sA + m0 * g.lda + k_first) * 16;
    const char *Bt = static_cast<const char *>(g.B) + (bz * g.sB + n0 * g.ldb + k_first) * 16;

    // A stage is [k eighth][row of A, then of B][8 values], value k of a row
    // in slot k ^ (row & 7).
    int64_t off[L]; // byte offset of the lane's row, and dword of its value
    int ck[L];      // the lane's k
#pragma unroll
    for (int i = 0; i < L; i++) {
        const bool isa = i < A_IN;
        const int pd = (wave * (isa ? A_IN : B_IN) + (isa ? i : i - A_IN)) * 64 + lane;
        const int p = pd / PER, sub = (pd % PER) * DW;
        const int r = (p >> 3) % (isa ? BM : BN), slot = p & 7, kk = (p >> 3) / (isa ? BM : BN);
        const int64_t rows = isa ? g.M - m0 : g.N - n0;
        const int64_t rr = r < rows ? r : rows - 1;
        ck[i] = 8 * kk + (slot ^ (r & 7));
        off[i] = rr * (isa ? g.lda : g.ldb) * 16 + sub * 4;
    }
    auto issue = [&](int64_t kt, f64x2 *s) __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        const int64_t k0 = kt * KT;
#pragma unroll
        for (int i = 0; i < L; i++) {
            const int64_t k = k0 + ck[i];
            const void *src = (i < A_IN ? At : Bt) + off[i] + (k < K ? k * 16 : 0);
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

    f64x4 cr[FM][FN], ci[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++) cr[i][j] = ci[i][j] = f64x4{0, 0, 0, 0};

    const int q = lane >> 4, j = lane & 15;
    auto mma = [](double a, double b, f64x4 c) __attribute__((always_inline)) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    };
    auto compute = [&](const f64x2 *s, bool tail, int64_t kt) __attribute__((always_inline)) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int kk = 4 * h + q;
            const bool none = tail && kt * KT + 8 * wk + kk >= K;
            f64x2 b[FN];
#pragma unroll
            for (int fn = 0; fn < FN; fn++) {
                const int r = wn * WTN + fn * 16 + j;
                b[fn] = s[(BM * WK + BN * wk + r) * 8 + (kk ^ (r & 7))];
                if (none) b[fn] = f64x2{0, 0};
            }
#pragma unroll
            for (int fm = 0; fm < FM; fm++) {
                const int r = wm * WTM + fm * 16 + j;
                f64x2 a = s[(BM * wk + r) * 8 + (kk ^ (r & 7))];
                if (none) a = f64x2{0, 0};
#pragma unroll
                for (int fn = 0; fn < FN; fn++) {
                    cr[fm][fn] = mma(a.x, b[fn].x, cr[fm][fn]);
                    ci[fm][fn] = mma(a.x, b[fn].y, ci[fm][fn]);
                    cr[fm][fn] = mma(-a.y, b[fn].y, cr[fm][fn]);
                    ci[fm][fn] = mma(a.y, b[fn].x, ci[fm][fn]);
                }
            }
        }
    };

    const int64_t nk = (K + KT - 1) / KT;
    // vmcnt(L): the loads of the next stage may stay in flight.
    constexpr int kWaitPrev = 0x0f70 | (L & 15) | ((L >> 4) << 14);
    constexpr int kWaitAll = 0x0f70;
    issue(0, S0);
    if (nk > 1) issue(1, S1);
    // Stage kt is in LDS for every wave once each has waited for its own
    // loads; every wave is then also past its reads of stage kt - 1, whose
    // buffer takes stage kt + 2.
    auto arrive = [&](int64_t kt, f64x2 *next) __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        if (kt + 1 < nk)
            __builtin_amdgcn_s_waitcnt(kWaitPrev);
        else
            __builtin_amdgcn_s_waitcnt(kWaitAll);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        if (kt + 2 < nk) issue(kt + 2, next);
    };
    const int64_t nfull = K / KT;
    int64_t kt = 0;
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

    if (WK > 1) {
        // The sums of the k slices, added in slice order by the first, 16 rows at
        // a time.
        constexpr int SUM = FN * 4 * 64;
#pragma unroll
        for (int fm = 0; fm < FM; fm++) {
            __syncthreads();
            if (wk > 0) {
#pragma unroll
                for (int fn = 0; fn < FN; fn++)
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        S0[((wk - 1) * WM * WN + wmn) * SUM + (fn * 4 + r) * 64 + lane] =
                            f64x2{cr[fm][fn][r], ci[fm][fn][r]};
            }
            __syncthreads();
            if (wk > 0) continue;
            for (int w = 0; w < WK - 1; w++)
#pragma unroll
                for (int fn = 0; fn < FN; fn++)
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const f64x2 v = S0[(w * WM * WN + wmn) * SUM + (fn * 4 + r) * 64 + lane];
                        cr[fm][fn][r] += v.x;
                        ci[fm][fn][r] += v.y;
                    }
        }
        if (wk > 0) return;
    }

    double2 *C = static_cast<double2 *>(g.C) + bz * g.sC + int64_t(blockIdx.y) * g.slice_stride;
#pragma unroll
    for (int fm = 0; fm < FM; fm++)
#pragma unroll
        for (int fn = 0; fn < FN; fn++) {
            const int64_t col = n0 + wn * WTN + fn * 16 + j;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int64_t row = m0 + wm * WTM + fm * 16 + q + 4 * r;
                if (row < g.M && col < g.N)
                    C[row * g.ldc + col] = double2{cr[fm][fn][r], ci[fm][fn][r]};
            }
        }
}

template <int BM, int BN, int WM, int WN, int WK, int DW = 4>
void launch_tile(const GemmArgs &g, hipStream_t stream)
{
    JH_REQUIRE(ceil_div(g.M, BM) * ceil_div(g.N, BN) <= 0x7fffffff, "Too many tiles.");
    dim3 grid((unsigned)(ceil_div(g.M, BM) * ceil_div(g.N, BN)), (unsigned)g.slices,
              (unsigned)g.batch);
    hipLaunchKernelGGL((cgemm_f64_kernel<BM, BN, WM, WN, WK, DW>), grid, dim3(64 * WM * WN * WK), 0,
                       stream, g);
    JH_HIP(hipGetLastError());
}

} // namespace

void launch_f64(const GemmArgs &g, hipStream_t stream)
{
    const bool aligned = reinterpret_cast<uintptr_t>(g.A) % 16 == 0 &&
                         reinterpret_cast<uintptr_t>(g.B) % 16 == 0;
    if (!aligned) {
        launch_tile<64, 64, 2, 2, 1, 1>(g, stream);
        return;
    }
    int form = 0;
    (void)tile_time(kF64Forms, g.M, g.N, g.slices > 1 ? g.slice_k : g.K, g.batch * g.slices,
                    &form);
    switch (form) {
    case 0:
        launch_tile<128, 128, 4, 2, 1>(g, stream);
        break;
    case 1:
        launch_tile<32, 32, 2, 2, 2>(g, stream);
        break;
    default:
        launch_tile<32, 32, 2, 2, 1>(g, stream);
        break;
    }
}

} // namespace jet_hip
