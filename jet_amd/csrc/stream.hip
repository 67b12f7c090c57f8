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

// A small tensor on a few modes of a large one (StreamShortK).  Bound by reading
// the large operand and writing the result once: 16-byte loads along its lowest
// mode, the small operand in LDS, products on the VALU.  Partial lines stored
// past the caches cost a read of the line each, so rows that are one piece of
// the result are gathered in LDS.  Measured: a two-qubit gate on 26 qubits (read
// and written twice with permuted copies before) 596 -> 188 us, 5.7 TB/s; gates
// of one to four qubits on 25 qubits 126-619 -> 77-124 us.
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
    const uint32_t yb = stream_all_bits(p.yb, batch);
    for (int i = tid; i < N * K; i += 256)
        ys[i >> LK][i & (K - 1)] = Y[yb | stream_all_bits(p.yn, i >> LK) |
                                     stream_all_bits(p.yk, i & (K - 1))];
    if (tid < N) cns[tid] = stream_all_bits(p.cn, tid);
    __syncthreads();
    const C2 *Xb = X + stream_all_bits(p.xb, batch);
    C2 *Cb = C + stream_all_bits(p.cb, batch);
    uint32_t xk[K];
#pragma unroll
    for (int k = 0; k < K; k++) xk[k] = stream_all_bits(p.xk, k);
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

// Few outputs, many k (StreamDot).  Bound by reading both operands once: a
// work-group walks tiles, the next tile's loads in registers while the current one
// is in LDS.  Thread bits, lowest first: the tile's batch bits, m bits beyond
// what a thread can sum, k.  Sums in FP64, as the split-K kernel's, first per
// thread, then over the threads, then over the work-groups (final kernel).
// Measured (permuted copies and the split-K kernel before): 4 x 2 outputs over
// 2^22 k 263 -> 48 us, 2 x 2 over 2^20 k in 128 batches 3089 -> 759 us (5.7 TB/s).
template <class R, int LM, int LN>
__global__ __launch_bounds__(256) void stream_dot_kernel(
    const typename Pair<R>::c *__restrict__ A, const typename Pair<R>::c *__restrict__ B,
    double2 *__restrict__ partials, StreamDot p, int log2_chunks, int vec)
{
    using C2 = typename Pair<R>::c;
    constexpr int EB = int(sizeof(C2)), CAP = EB == 8 ? kDotMaxLog2Tile : kDotMaxLog2Tile - 1;
    constexpr int VEC = 16 / EB; // elements per load
    constexpr int LOADS = (1 << CAP) / VEC / 256;
    constexpr int M = 1 << LM, N = 1 << LN;
    __shared__ f32x4 lds[(2 << CAP) / VEC];
    C2 *const as = reinterpret_cast<C2 *>(lds), *const bs = as + (1 << CAP);
    double2 *const red = reinterpret_cast<double2 *>(lds); // after the tiles
    static_assert(sizeof(lds) >= (4 << kDotMaxLog2Lanes) * sizeof(double2), "sums fit");
    const int tid = threadIdx.x;
    const int na = 1 << (p.lt + p.lm + p.tb), nb = 1 << (p.lt + p.ln + p.tb);
    const uint32_t chunk = blockIdx.x, batch = blockIdx.y;
    const C2 *Ab = A + stream_all_bits(p.oab, batch);
    const C2 *Bb = B + stream_all_bits(p.obb, batch);

    uint32_t offa[LOADS], offb[LOADS];
#pragma unroll
    for (int e = 0; e < LOADS; e++) {
        const uint32_t u = uint32_t(tid + e * 256) * VEC;
        offa[e] = stream_all_bits(p.a_pos, u);
        offb[e] = stream_all_bits(p.b_pos, u);
    }
    f32x4 na4[LOADS], nb4[LOADS];
    auto load = [&](const C2 *q) __attribute__((always_inline)) {
        if (EB == 16 || vec) return __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(q));
        return f32x4{float(q[0].x), float(q[0].y), float(q[1].x), float(q[1].y)};
    };
    auto fetch = [&](uint32_t t) __attribute__((always_inline)) {
        const C2 *at = Ab + stream_all_bits(p.oak, t);
        const C2 *bt = Bb + stream_all_bits(p.obk, t);
#pragma unroll
        for (int e = 0; e < LOADS; e++) {
            if ((tid + e * 256) * VEC < na) na4[e] = load(at + offa[e]);
            if ((tid + e * 256) * VEC < nb) nb4[e] = load(bt + offb[e]);
        }
    };
    auto put = [&](C2 *s, uint32_t u, f32x4 v) __attribute__((always_inline)) {
        if constexpr (EB == 8) {
            s[dot_slot(u, EB)] = C2{v.x, v.y};
            s[dot_slot(u + 1, EB)] = C2{v.z, v.w};
        }
        else
            s[dot_slot(u, EB)] = __builtin_bit_cast(C2, v);
    };

    // This thread's share of a tile.
    const int low = p.tb + p.xm;                // thread bits that are not k
    const int kl = 8 - low;                     // thread bits that are k
    const uint32_t tbv = tid & ((1 << p.tb) - 1), mx = (tid >> p.tb) & ((1 << p.xm) - 1);
    const uint32_t kv = tid >> low;
    const uint32_t ua = dot_slot(stream_all_bits(p.ab, tbv) |
                                     stream_all_bits(p.am, mx << LM) |
                                     stream_all_bits(p.ak, kv), EB);
    const uint32_t ub = dot_slot(stream_all_bits(p.bb, tbv) | stream_all_bits(p.bk, kv), EB);
    uint32_t sm[M], sn[N];
#pragma unroll
    for (int m = 0; m < M; m++) sm[m] = dot_slot(stream_all_bits(p.am, m), EB);
#pragma unroll
    for (int n = 0; n < N; n++) sn[n] = dot_slot(stream_all_bits(p.bn, n), EB);
    double re[M][N], im[M][N];
#pragma unroll
    for (int m = 0; m < M; m++)
#pragma unroll
        for (int n = 0; n < N; n++) re[m][n] = im[m][n] = 0.0;

    const uint32_t tiles = 1u << (p.lk - p.lt - log2_chunks); // of this work-group
    const uint32_t step = 1u << log2_chunks;
    const uint32_t iters = 1u << (p.lt - kl);
    fetch(chunk);
    for (uint32_t i = 0; i < tiles; i++) {
        __syncthreads();
#pragma unroll
        for (int e = 0; e < LOADS; e++) {
            const uint32_t u = uint32_t(tid + e * 256) * VEC;
            if (int(u) < na) put(as, u, na4[e]);
            if (int(u) < nb) put(bs, u, nb4[e]);
        }
        __syncthreads();
        if (i + 1 < tiles) fetch(chunk + (i + 1) * step);
        for (uint32_t it = 0; it < iters; it++) {
            const uint32_t xa = ua ^ dot_slot(stream_all_bits(p.ak, it << kl), EB);
            const uint32_t xb = ub ^ dot_slot(stream_all_bits(p.bk, it << kl), EB);
            C2 y[N];
#pragma unroll
            for (int n = 0; n < N; n++) y[n] = bs[xb ^ sn[n]];
#pragma unroll
            for (int m = 0; m < M; m++) {
                const C2 x = as[xa ^ sm[m]];
#pragma unroll
                for (int n = 0; n < N; n++)
                    mac(re[m][n], im[m][n], double(x.x), double(x.y), double(y[n].x),
                        double(y[n].y));
            }
        }
    }
    __syncthreads();
    // Over the k lanes of the wave, then over the waves.
    const int lane = tid & 63, wave = tid >> 6;
#pragma unroll
    for (int m = 0; m < M; m++)
#pragma unroll
        for (int n = 0; n < N; n++) {
            for (int off = 32; off >= 1 << low; off >>= 1) {
                re[m][n] += __shfl_xor(re[m][n], off);
                im[m][n] += __shfl_xor(im[m][n], off);
            }
            if (lane < 1 << low)
                red[(wave << kDotMaxLog2Lanes) + lane * (M * N) + m * N + n] =
                    double2{re[m][n], im[m][n]};
        }
    __syncthreads();
    const int sums = (1 << low) * M * N;
    for (int i = tid; i < sums; i += 256) {
        constexpr int W = 1 << kDotMaxLog2Lanes;
        const double2 a = red[i], b = red[W + i], c = red[2 * W + i], d = red[3 * W + i];
        const uint32_t l = i / (M * N), mn = i % (M * N);
        // output: outer batch, tile batch, m (thread bits highest), n
        const uint32_t m = ((l >> p.tb) << LM) | (mn >> LN);
        const int64_t o = (((int64_t(batch) << p.tb | (l & ((1u << p.tb) - 1))) << p.lm | m) << LN) |
                          (mn & (N - 1));
        partials[(o << log2_chunks) + chunk] =
            double2{(a.x + b.x) + (c.x + d.x), (a.y + b.y) + (c.y + d.y)};
    }
}

template <class R>
__global__ __launch_bounds__(256) void stream_dot_final_kernel(
    const double2 *__restrict__ partials, typename Pair<R>::c *__restrict__ C, StreamDot p,
    int log2_chunks)
{
    using C2 = typename Pair<R>::c;
    // one wave per output
    const int64_t o = int64_t(blockIdx.x) * 4 + (threadIdx.x >> 6);
    if (o >= int64_t(1) << (p.lb + p.lm + p.ln)) return;
    const int lane = threadIdx.x & 63;
    double re = 0, im = 0;
    for (int c = lane; c < 1 << log2_chunks; c += 64) {
        const double2 v = partials[(o << log2_chunks) + c];
        re += v.x;
        im += v.y;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        re += __shfl_xor(re, off);
        im += __shfl_xor(im, off);
    }
    if (lane == 0) {
        const uint32_t n = uint32_t(o) & ((1u << p.ln) - 1);
        const uint32_t m = uint32_t(o >> p.ln) & ((1u << p.lm) - 1);
        const uint32_t t = uint32_t(o >> (p.ln + p.lm)) & ((1u << p.tb) - 1);
        const uint32_t b = uint32_t(o >> (p.ln + p.lm + p.tb));
        C[stream_all_bits(p.cn, n) | stream_all_bits(p.cm, m) | stream_all_bits(p.ctb, t) |
          stream_all_bits(p.cob, b)] = C2{R(re), R(im)};
    }
}

template <class R, int LM>
void launch_dot_n(const StreamDot &p, const void *a, const void *b, double2 *partials,
                  int log2_chunks, hipStream_t stream)
{
    using C2 = typename Pair<R>::c;
    const dim3 grid(1u << log2_chunks, 1u << (p.lb - p.tb));
    const int vec = reinterpret_cast<uintptr_t>(a) % 16 == 0 &&
                    reinterpret_cast<uintptr_t>(b) % 16 == 0;
#define JH_DOT(LN)                                                                        \
    case LN:                                                                              \
        if constexpr (LM + LN <= kDotMaxLog2Sums)                                         \
            hipLaunchKernelGGL((stream_dot_kernel<R, LM, LN>), grid, dim3(256), 0, stream, \
                               static_cast<const C2 *>(a), static_cast<const C2 *>(b),    \
                               partials, p, log2_chunks, vec);                            \
        break
    switch (p.ln) {
        JH_DOT(0);
        JH_DOT(1);
        JH_DOT(2);
        JH_DOT(3);
        JH_DOT(4);
    }
#undef JH_DOT
}

template <class R>
void launch_dot(const StreamDot &p, const void *a, const void *b, void *c, double2 *partials,
                hipStream_t stream)
{
    int lc = 0;
    while ((int64_t(1) << lc) < p.chunks()) lc++;
    switch (p.lm - p.xm) {
    case 0:
        launch_dot_n<R, 0>(p, a, b, partials, lc, stream);
        break;
    case 1:
        launch_dot_n<R, 1>(p, a, b, partials, lc, stream);
        break;
    case 2:
        launch_dot_n<R, 2>(p, a, b, partials, lc, stream);
        break;
    case 3:
        launch_dot_n<R, 3>(p, a, b, partials, lc, stream);
        break;
    default:
        launch_dot_n<R, 4>(p, a, b, partials, lc, stream);
        break;
    }
    JH_HIP(hipGetLastError());
    hipLaunchKernelGGL(stream_dot_final_kernel<R>, dim3((unsigned)ceil_div(p.outputs(), int64_t(4))),
                       dim3(256), 0, stream, partials, static_cast<typename Pair<R>::c *>(c), p, lc);
}

} // namespace

void launch_stream_dot(const StreamDot &p, int elem_bytes, const void *a, const void *b, void *c,
                       void *partials, hipStream_t stream)
{
    const double batch = double(int64_t(1) << p.lb), k = double(int64_t(1) << p.lk);
    const double m = double(1 << p.lm), n = double(1 << p.ln);
    prof::Scope ps(prof::kGemmSplitK, stream, 8.0 * batch * m * n * k,
                   elem_bytes * batch * (m * k + n * k + m * n));
    if (p.swap) std::swap(a, b);
    if (elem_bytes == 8)
        launch_dot<float>(p, a, b, c, static_cast<double2 *>(partials), stream);
    else
        launch_dot<double>(p, a, b, c, static_cast<double2 *>(partials), stream);
    JH_HIP(hipGetLastError());
}

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
