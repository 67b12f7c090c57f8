// permute.hip -- LDS-tiled bit-permutation and gather kernels (gfx950).
#include "common.hpp"
#include "permute_plan.hpp"
#include "profiler.hpp"

#include <algorithm>
#include <numeric>

namespace jet_hip {

namespace {

// The plan's bit positions without a loop, as scalar registers: a loop over
// them (bits_tile_base) waits for a load of kernel arguments per bit, about 1 us of
// every tile and 5 us of a launch.  Positions past the last bit are zero
// and meet zero bits of v.
template <int N> __device__ __forceinline__ int64_t place_bits(const int8_t *pos, int64_t v)
{
    int64_t o = 0;
#pragma unroll
    for (int j = 0; j < N; j++) o |= ((v >> j) & 1) << pos[j];
    return o;
}

__device__ __forceinline__ void tile_base(const BitPermParams &p, int64_t w, int64_t *bin,
                                          int64_t *bout)
{
    constexpr int FAST = 24;
    int64_t i = place_bits<FAST>(p.outer_in, w), o = place_bits<FAST>(p.outer_out, w);
    for (int j = FAST; j < p.nr; j++) {
        i |= ((w >> j) & 1) << p.outer_in[j];
        o |= ((w >> j) & 1) << p.outer_out[j];
    }
    *bin = i;
    *bout = o;
}

__device__ __forceinline__ int64_t tile_in_offset(const BitPermParams &p, int u)
{
    return place_bits<kTileMaxBits>(p.tile_in, u);
}
__device__ __forceinline__ int64_t tile_out_offset(const BitPermParams &p, int v, int *u)
{
    *u = int(place_bits<kTileMaxBits>(p.v2u, v));
    return place_bits<kTileMaxBits>(p.tile_out, v);
}

template <class T>
__global__ __launch_bounds__(kPermThreads) void permute_bits_kernel(
    const T *__restrict__ in, T *__restrict__ out, BitPermParams p,
    int64_t ntiles)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    T *lds = reinterpret_cast<T *>(smem_raw);
    constexpr int EMAX = (1 << kTileMaxBits) / kPermThreads;
    const int tsize = 1 << p.tb;
    const int tid = threadIdx.x;

    // Per-thread in-tile offsets: identical for every tile this block visits.
    int64_t ioff[EMAX], ooff[EMAX];
    int lsrc[EMAX], ldst[EMAX];
#pragma unroll
    for (int e = 0; e < EMAX; e++) {
        const int u = tid + e * kPermThreads;
        int uu = 0;
        ioff[e] = tile_in_offset(p, u);
        ooff[e] = tile_out_offset(p, u, &uu);
        lsrc[e] = bits_lds_index(u, (int)sizeof(T));
        ldst[e] = bits_lds_index(uu, (int)sizeof(T));
    }

    for (int64_t w = blockIdx.x; w < ntiles; w += gridDim.x) {
        int64_t bin, bout;
        tile_base(p, w, &bin, &bout);
        __syncthreads();
#pragma unroll
        for (int e = 0; e < EMAX; e++)
            if (tid + e * kPermThreads < tsize) lds[lsrc[e]] = in[bin + ioff[e]];
        __syncthreads();
#pragma unroll
        for (int e = 0; e < EMAX; e++)
            if (tid + e * kPermThreads < tsize) out[bout + ooff[e]] = lds[ldst[e]];
    }
}

// complex64 tiles that hold both input bit 0 and output bit 0: each thread
// moves pairs of neighbouring elements, which are neighbours in the input
// (tile element u, u + 1 with u even) and in the output (tile element v,
// v + 1 in output order), with 16-byte loads and stores.
__global__ __launch_bounds__(kPermThreads) void permute_bits_pairs_kernel(
    const float2 *__restrict__ in, float2 *__restrict__ out, BitPermParams p, int64_t ntiles)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    float2 *lds = reinterpret_cast<float2 *>(smem_raw);
    constexpr int PMAX = (1 << kTileMaxBits) / kPermThreads / 2;
    const int tsize = 1 << p.tb;
    const int tid = threadIdx.x;
    int64_t ioff[PMAX], ooff[PMAX];
    int ls0[PMAX], ls1[PMAX], ld0[PMAX], ld1[PMAX];
#pragma unroll
    for (int e = 0; e < PMAX; e++) {
        const int u = 2 * (tid + e * kPermThreads);
        int uu0 = 0, uu1 = 0;
        ioff[e] = tile_in_offset(p, u);
        ooff[e] = tile_out_offset(p, u, &uu0);
        (void)tile_out_offset(p, u + 1, &uu1);
        ls0[e] = bits_lds_index(u, 8);
        ls1[e] = bits_lds_index(u + 1, 8);
        ld0[e] = bits_lds_index(uu0, 8);
        ld1[e] = bits_lds_index(uu1, 8);
    }
    // Non-temporal loads and stores: every element is read and written once
    // (5% over cached accesses on six rank-28 permutations, 1% over only the
    // stores non-temporal).
    typedef float f32x4v __attribute__((ext_vector_type(4)));
    for (int64_t w = blockIdx.x; w < ntiles; w += gridDim.x) {
        int64_t bin, bout;
        tile_base(p, w, &bin, &bout);
        __syncthreads();
#pragma unroll
        for (int e = 0; e < PMAX; e++) {
            if (2 * (tid + e * kPermThreads) < tsize) {
                const f32x4v x = __builtin_nontemporal_load(
                    reinterpret_cast<const f32x4v *>(in + bin + ioff[e]));
                lds[ls0[e]] = float2{x.x, x.y};
                lds[ls1[e]] = float2{x.z, x.w};
            }
        }
        __syncthreads();
#pragma unroll
        for (int e = 0; e < PMAX; e++) {
            if (2 * (tid + e * kPermThreads) < tsize) {
                const float2 a = lds[ld0[e]], b = lds[ld1[e]];
                __builtin_nontemporal_store(f32x4v{a.x, a.y, b.x, b.y},
                                            reinterpret_cast<f32x4v *>(out + bout + ooff[e]));
            }
        }
    }
}

template <class T>
__global__ __launch_bounds__(256) void permute_generic_kernel(
    const T *__restrict__ in, T *__restrict__ out, GenericPermParams p,
    int64_t numel)
{
    const int64_t stride = int64_t(gridDim.x) * blockDim.x;
    for (int64_t o = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; o < numel;
         o += stride) {
        const int64_t off = generic_in_offset(p, o);
        out[o] = in[off];
    }
}

// The same by tiles (TilePermParams): a work-group reads a tile in input order
// into LDS and writes it in output order; each thread's offsets, the same in
// every tile, are found once.  The gather above reads one element per line wherever
// the two orders' fastest axes differ.  Neighbouring tiles go to one XCD (one of 8
// in turn gets a work-group), whose L2 joins the lines that their runs share
// (complex64 2^26 350 -> 310 us).  Bound by partial lines at the ends of runs.
// Measured, complex64, gather before: 1260 x 1014 14.9 -> 8.9 us, 3000 x 7 x 500
// 116 -> 36, 100 x 100 x 100 x 10 183 -> 42, five random shapes of 2^23 elements 64 ->
// 27 and of 2^26 770 -> 318; complex128 2^26 1020 -> 431.
template <class T, int MAX>
__global__ __launch_bounds__(256) void permute_tiles_kernel(const T *__restrict__ in,
                                                            T *__restrict__ out, TilePermParams p)
{
    constexpr int PER = MAX / 256;
    __shared__ T lds[MAX + MAX / 32];
    const int tid = threadIdx.x;
    uint32_t ioff[PER], ooff[PER], src[PER];
#pragma unroll
    for (int e = 0; e < PER; e++) {
        const uint32_t u = tid + e * 256;
        if (int(u) >= p.elems) break;
        uint32_t unused;
        ioff[e] = tile_axes_offset(p.in_ext, p.in_rec, p.in_step, p.in_step, u, &unused);
        ooff[e] = tile_axes_offset(p.out_ext, p.out_rec, p.out_step, p.out_u, u, &src[e]);
        src[e] = tile_axes_slot(src[e]);
    }
    for (uint32_t w = blockIdx.x; w < p.tiles; w += gridDim.x) {
        uint32_t bin, bout;
        const uint32_t per = p.tiles >> 3; // of an XCD
        tile_axes_base(p, w < per * 8 ? (w & 7) * per + (w >> 3) : w, &bin, &bout);
        __syncthreads();
#pragma unroll
        for (int e = 0; e < PER; e++)
            if (tid + e * 256 < p.elems) lds[tile_axes_slot(tid + e * 256)] = in[bin + ioff[e]];
        __syncthreads();
#pragma unroll
        for (int e = 0; e < PER; e++)
            if (tid + e * 256 < p.elems) out[bout + ooff[e]] = lds[src[e]];
    }
}

// Device-to-device copy (the identity permutation): 16-byte vectors, four
// per thread and iteration with all four loads issued before the stores,
// non-temporal loads and stores (the data is streamed once).  Measured on
// a 2 GiB copy: 5.87 TB/s of read + write traffic, against 4.87 TB/s for
// hipMemcpyAsync and 5.1-5.7 TB/s with cached accesses.  `tail` (8 bytes,
// the last element of an odd number of complex64 values) is copied by the
// first thread.
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
constexpr int kCopyUnroll = 4;

__global__ __launch_bounds__(256) void copy16_kernel(const u32x4 *__restrict__ in,
                                                     u32x4 *__restrict__ out, int64_t n,
                                                     const uint2 *tail_in, uint2 *tail_out)
{
    const int64_t step = int64_t(gridDim.x) * 256 * kCopyUnroll;
    for (int64_t base = int64_t(blockIdx.x) * 256 * kCopyUnroll + threadIdx.x; base < n;
         base += step) {
        u32x4 v[kCopyUnroll];
#pragma unroll
        for (int u = 0; u < kCopyUnroll; u++) {
            const int64_t i = base + int64_t(u) * 256;
            if (i < n) v[u] = __builtin_nontemporal_load(in + i);
        }
#pragma unroll
        for (int u = 0; u < kCopyUnroll; u++) {
            const int64_t i = base + int64_t(u) * 256;
            if (i < n) __builtin_nontemporal_store(v[u], out + i);
        }
    }
    if (tail_in != nullptr && blockIdx.x == 0 && threadIdx.x == 0) *tail_out = *tail_in;
}

// 8-byte elements, for pointers that are not 16-byte aligned.
__global__ __launch_bounds__(256) void copy8_kernel(const uint2 *__restrict__ in,
                                                    uint2 *__restrict__ out, int64_t n)
{
    const int64_t stride = int64_t(gridDim.x) * 256;
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < n; i += stride)
        out[i] = in[i];
}

void launch_copy(const void *in, void *out, size_t bytes, hipStream_t stream)
{
    JH_REQUIRE(bytes % 8 == 0, "Copies move whole 8-byte units.");
    if (bytes == 0) return;
    const bool aligned = reinterpret_cast<uintptr_t>(in) % 16 == 0 &&
                         reinterpret_cast<uintptr_t>(out) % 16 == 0;
    if (aligned) {
        const int64_t n = int64_t(bytes / 16);
        const bool odd = bytes % 16 != 0;
        const uint2 *ti = odd ? reinterpret_cast<const uint2 *>(in) + 2 * n : nullptr;
        uint2 *to = odd ? reinterpret_cast<uint2 *>(out) + 2 * n : nullptr;
        const int grid = (int)std::max<int64_t>(
            1, std::min<int64_t>(ceil_div(n, 256 * kCopyUnroll), 16384));
        hipLaunchKernelGGL(copy16_kernel, dim3(grid), dim3(256), 0, stream,
                           static_cast<const u32x4 *>(in), static_cast<u32x4 *>(out), n, ti, to);
    }
    else {
        const int64_t n = int64_t(bytes / 8);
        const int grid = (int)std::max<int64_t>(1, std::min<int64_t>(ceil_div(n, 256), 16384));
        hipLaunchKernelGGL(copy8_kernel, dim3(grid), dim3(256), 0, stream,
                           static_cast<const uint2 *>(in), static_cast<uint2 *>(out), n);
    }
    JH_HIP(hipGetLastError());
}

} // namespace

template <class T>
static void launch_typed(const PermutePlan &plan, const void *in, void *out,
                         hipStream_t stream)
{
    const double bytes = 2.0 * sizeof(T) * double(plan.numel);
    if (plan.kind == PermutePlan::kCopy) {
        prof::Scope ps(prof::kCopy, stream, 0.0, bytes);
        launch_copy(in, out, sizeof(T) * size_t(plan.numel), stream);
        return;
    }
    if (plan.kind == PermutePlan::kBits) {
        prof::Scope ps(prof::kPermuteBits, stream, 0.0, bytes);
        const int64_t ntiles = int64_t(1) << plan.bits.nr;
        const int grid = (int)std::min<int64_t>(ntiles, 8192);
        const size_t lds = sizeof(T) << plan.bits.tb;
        const bool pairs = sizeof(T) == 8 && plan.bits.tb >= 9 && plan.bits.ti >= 1 &&
                           plan.bits.tile_out[0] == 0 &&
                           reinterpret_cast<uintptr_t>(in) % 16 == 0 &&
                           reinterpret_cast<uintptr_t>(out) % 16 == 0;
        if (pairs)
            hipLaunchKernelGGL(permute_bits_pairs_kernel, dim3(grid), dim3(kPermThreads), lds,
                               stream, static_cast<const float2 *>(in),
                               static_cast<float2 *>(out), plan.bits, ntiles);
        else
            hipLaunchKernelGGL(permute_bits_kernel<T>, dim3(grid), dim3(kPermThreads), lds,
                               stream, static_cast<const T *>(in), static_cast<T *>(out),
                               plan.bits, ntiles);
        JH_HIP(hipGetLastError());
        return;
    }
    prof::Scope ps(prof::kPermuteGeneric, stream, 0.0, bytes);
    const TilePermParams &tiles = sizeof(T) == 8 ? plan.tiles8 : plan.tiles16;
    if (tiles.elems > 0) {
        // Fewer work-groups find their offsets once for more tiles (2^23 31 -> 27
        // us); out of HBM more of them are faster (2^26 complex128 493 against 601).
        const dim3 grid(std::min(tiles.tiles, double(sizeof(T)) * double(plan.numel) >
                                                      double(kPermCacheBytes) ? 8192u : 4096u));
        const T *x = static_cast<const T *>(in);
        T *y = static_cast<T *>(out);
        if (tiles.cap <= 1024)
            hipLaunchKernelGGL((permute_tiles_kernel<T, 1024>), grid, dim3(256), 0, stream, x, y,
                               tiles);
        else if (tiles.cap == 2048)
            hipLaunchKernelGGL((permute_tiles_kernel<T, 2048>), grid, dim3(256), 0, stream, x, y,
                               tiles);
        else
            hipLaunchKernelGGL((permute_tiles_kernel<T, kTileBytes / int(sizeof(T))>), grid, dim3(256),
                               0, stream, x, y, tiles);
        JH_HIP(hipGetLastError());
        return;
    }
    const int grid = (int)std::min<int64_t>((plan.numel + 255) / 256, 16384);
    hipLaunchKernelGGL(permute_generic_kernel<T>, dim3(grid), dim3(256), 0, stream,
                       static_cast<const T *>(in), static_cast<T *>(out), plan.gen,
                       plan.numel);
    JH_HIP(hipGetLastError());
}

void launch_permute(const PermutePlan &plan, int elem_bytes, const void *in,
                    void *out, hipStream_t stream)
{
    if (plan.numel == 0) return;
    if (elem_bytes == 8)
        launch_typed<float2>(plan, in, out, stream);
    else if (elem_bytes == 16)
        launch_typed<double2>(plan, in, out, stream);
    else
        JH_FAIL(JET_HIP_ERROR_INVALID_VALUE, "Unsupported element size.");
}

} // namespace jet_hip
