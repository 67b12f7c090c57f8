// stream.hip -- contractions that read their operands once, in place (gfx950).
#include "common.hpp"
#include "profiler.hpp"
#include "stream.hpp"

#include <algorithm>

namespace jet_hip {

namespace {

template <class R> struct Pair;
template <> struct Pair<float> {
    using c = float2;
};
template <> struct Pair<double> {
    using c = double2;
};
typedef float f32x4 __attribute__((ext_vector_type(4)));

// How a thread's values lie in memory.
enum { kOneRow = 0, kTwoRows = 1, kPairsOfK = 2 };

template <class R> __device__ __forceinline__ void mac(R &re, R &im, R xr, R xi, R yr, R yi)
{
    re = fma(xr, yr, re);
    re = fma(-xi, yi, re);
    im = fma(xr, yi, im);
    im = fma(xi, yr, im);
}

// NPAIR: columns n and n + 1 are neighbours in C.  STAGE: a step's rows and all
// N columns are one contiguous piece of C: it is gathered in LDS (16-byte
// chunks, swizzled within a row) and written in order.
template <class R, int LK, int FORM, bool NPAIR, bool STAGE>
__global__ __launch_bounds__(256) void stream_shortk_kernel(
    const typename Pair<R>::c *__restrict__ X, const typename Pair<R>::c *__restrict__ Y,
    typename Pair<R>::c *__restrict__ C, StreamShortK p)
{
    using C2 = typename Pair<R>::c;
    constexpr int K = 1 << LK;
    constexpr int ROWS = FORM == kTwoRows ? 2 : 1;
    __shared__ C2 ys[1 << kStreamMaxLog2N][K];
    __shared__ uint32_t cns[1 << kStreamMaxLog2N];
    extern __shared__ f32x4 stage[];
    const int tid = threadIdx.x;
    const int N = 1 << p.ln;
    const uint32_t batch = blockIdx.y;
    const uint32_t yb = stream_bits(p.yb, p.lb, batch);
    for (int i = tid; i < N * K; i += 256)
        ys[i >> LK][i & (K - 1)] = Y[yb | stream_bits(p.yn, p.ln, i >> LK) |
                                     stream_bits(p.yk, LK, i & (K - 1))];
    if (tid < N) cns[tid] = stream_bits(p.cn, p.ln, tid);
    __syncthreads();
    const C2 *Xb = X + stream_bits(p.xb, p.lb, batch);
    C2 *Cb = C + stream_bits(p.cb, p.lb, batch);
    uint32_t xk[K];
#pragma unroll
    for (int k = 0; k < K; k++) xk[k] = stream_bits(p.xk, LK, k);
    const uint32_t rows = 1u << p.lr, stride = gridDim.x * 256u * ROWS;
    for (uint32_t row = (blockIdx.x * 256u + tid) * ROWS; row < rows; row += stride) {
        uint32_t xo, co;
        stream_row(p, row, &xo, &co);
        C2 x[ROWS][K];
        if constexpr (FORM == kTwoRows) {
#pragma unroll
            for (int k = 0; k < K; k++) {
                const f32x4 v = __builtin_nontemporal_load(
                    reinterpret_cast<const f32x4 *>(Xb + (xo | xk[k])));
                x[0][k] = C2{v.x, v.y};
                x[1][k] = C2{v.z, v.w};
            }
        }
        else if constexpr (FORM == kPairsOfK) {
#pragma unroll
            for (int k = 0; k < K; k += 2) {
                const f32x4 v = *reinterpret_cast<const f32x4 *>(Xb + (xo | xk[k]));
                x[0][k] = C2{v.x, v.y};
                x[0][k + 1] = C2{v.z, v.w};
            }
        }
        else {
#pragma unroll
            for (int k = 0; k < K; k++) x[0][k] = Xb[xo | xk[k]];
        }
#pragma unroll 1
        for (int n = 0; n < N; n += NPAIR ? 2 : 1) {
            C2 o[ROWS][NPAIR ? 2 : 1];
#pragma unroll
            for (int e = 0; e < (NPAIR ? 2 : 1); e++) {
                C2 y[K];
#pragma unroll
                for (int k = 0; k < K; k++) y[k] = ys[n + e][k];
#pragma unroll
                for (int r = 0; r < ROWS; r++) {
                    R re = 0, im = 0;
#pragma unroll
                    for (int k = 0; k < K; k++) mac(re, im, x[r][k].x, x[r][k].y, y[k].x, y[k].y);
                    o[r][e] = C2{re, im};
                }
            }
            C2 *dst = Cb + (co | cns[n]);
            if constexpr (STAGE) {
                const int cpr = N * int(sizeof(C2)) / 16;
#pragma unroll
                for (int r = 0; r < ROWS; r++) {
                    const int rl = tid * ROWS + r;
                    const int q = NPAIR ? n >> 1 : n;
                    f32x4 v;
                    if constexpr (NPAIR)
                        v = f32x4{o[r][0].x, o[r][0].y, o[r][1].x, o[r][1].y};
                    else
                        v = __builtin_bit_cast(f32x4, o[r][0]);
                    stage[rl * cpr + (q ^ (rl & (cpr - 1)))] = v;
                }
            }
            else if constexpr (NPAIR) {
#pragma unroll
                for (int r = 0; r < ROWS; r++)
                    *reinterpret_cast<f32x4 *>(r ? dst + (size_t(1) << p.segment[0].c) : dst) =
                        f32x4{o[r][0].x, o[r][0].y, o[r][1].x, o[r][1].y};
            }
            else if constexpr (FORM == kTwoRows) {
                if (p.segment[0].c == 0)
                    __builtin_nontemporal_store(
                        f32x4{o[0][0].x, o[0][0].y, o[1][0].x, o[1][0].y},
                        reinterpret_cast<f32x4 *>(dst));
                else {
                    dst[0] = o[0][0];
                    dst[size_t(1) << p.segment[0].c] = o[1][0];
                }
            }
            else
                dst[0] = o[0][0];
        }
        if constexpr (STAGE) {
            __syncthreads();
            const int cpr = N * int(sizeof(C2)) / 16, mask = cpr - 1;
            const int shift = p.ln - (sizeof(C2) == 8 ? 1 : 0);
            uint32_t x0, c0;
            stream_row(p, row - uint32_t(tid) * ROWS, &x0, &c0);
            f32x4 *dst = reinterpret_cast<f32x4 *>(Cb + c0);
            for (int i = tid; i < 256 * ROWS * cpr; i += 256) {
                const int rl = i >> shift;
                __builtin_nontemporal_store(stage[(rl << shift) + ((i & mask) ^ (rl & mask))],
                                            dst + i);
            }
            __syncthreads();
        }
    }
}

template <class R, int LK>
void launch_form(const StreamShortK &p, const void *x, const void *y, void *c, hipStream_t stream)
{
    using C2 = typename Pair<R>::c;
    const C2 *X = static_cast<const C2 *>(x), *Y = static_cast<const C2 *>(y);
    C2 *C = static_cast<C2 *>(c);
    const bool vec = sizeof(R) == 4 && reinterpret_cast<uintptr_t>(x) % 16 == 0 &&
                     reinterpret_cast<uintptr_t>(c) % 16 == 0;
    const bool two = vec && p.segment[0].x == 0;
    const bool kp = vec && LK >= 1 && p.xk[0] == 0;
    const bool np = vec && p.ln >= 1 && p.cn[0] == 0;
    // The columns fastest in C, then the rows of a whole step; with fewer
    // than 32 bytes of columns the stores of neighbouring threads meet in L2.
    bool staged = p.ln >= (sizeof(R) == 4 ? 2 : 1) && (vec || sizeof(R) == 8) && p.lr >= 9;
    for (int i = 0; i < p.n_segments; i++)
        staged = staged && (p.segment[i].row >= 9 || p.segment[i].c == p.segment[i].row + p.ln);
    for (int i = 0; i < p.ln; i++) staged = staged && p.cn[i] == i;
    const bool two_rows = two && !(staged && p.ln == 4); // 64 KiB of LDS otherwise
    const int64_t threads = (int64_t(1) << p.lr) >> (two_rows ? 1 : 0);
    const dim3 grid((unsigned)std::min<int64_t>(ceil_div(threads, int64_t(256)), 8192),
                    1u << p.lb);
    const size_t lds = staged ? (size_t(256) * sizeof(C2) << p.ln) * (two_rows ? 2 : 1) : 0;
#define JH_STREAM(FORM, NPAIR, STAGE)                                                         \
    hipLaunchKernelGGL((stream_shortk_kernel<R, LK, FORM, NPAIR, STAGE>), grid, dim3(256), lds, \
                       stream, X, Y, C, p)
    if constexpr (sizeof(R) == 4) {
        if (staged) {
            if (two_rows)
                JH_STREAM(kTwoRows, true, true);
            else if (kp)
                JH_STREAM(kPairsOfK, true, true);
            else
                JH_STREAM(kOneRow, true, true);
        }
        else if (two && np)
            JH_STREAM(kTwoRows, true, false);
        else if (two)
            JH_STREAM(kTwoRows, false, false);
        else if (kp && np)
            JH_STREAM(kPairsOfK, true, false);
        else if (kp)
            JH_STREAM(kPairsOfK, false, false);
        else
            JH_STREAM(kOneRow, false, false);
    }
    else if (staged)
        JH_STREAM(kOneRow, false, true);
    else
        JH_STREAM(kOneRow, false, false);
#undef JH_STREAM
}

template <class R>
void launch_typed(const StreamShortK &p, const void *x, const void *y, void *c, hipStream_t stream)
{
    switch (p.lk) {
    case 0:
        return launch_form<R, 0>(p, x, y, c, stream);
    case 1:
        return launch_form<R, 1>(p, x, y, c, stream);
    case 2:
        return launch_form<R, 2>(p, x, y, c, stream);
    case 3:
        return launch_form<R, 3>(p, x, y, c, stream);
    default:
        return launch_form<R, 4>(p, x, y, c, stream);
    }
}

} // namespace

void launch_stream_shortk(const StreamShortK &p, int elem_bytes, const void *a, const void *b,
                          void *c, hipStream_t stream)
{
    const double rows = double(int64_t(1) << (p.lr + p.lb));
    prof::Scope ps(prof::kGemmSmall, stream, 8.0 * rows * double(1 << (p.lk + p.ln)),
                   elem_bytes * rows * double((1 << p.lk) + (1 << p.ln)));
    const void *x = p.swap ? b : a, *y = p.swap ? a : b;
    if (elem_bytes == 8)
        launch_typed<float>(p, x, y, c, stream);
    else
        launch_typed<double>(p, x, y, c, stream);
    JH_HIP(hipGetLastError());
}

} // namespace jet_hip
