// stream.hpp -- contractions bound by reading their operands once, in the
// operands' own mode orders (every extent a power of two): a small tensor on
// a few modes of a large one (a gate on a state), and two large tensors that
// share almost every mode (closing a network).
#pragma once

#include "errors.hpp"

#include <cstdint>
#include <vector>

namespace jet_hip {

// C[batch, row, n] = sum over k of X[batch, row, k] Y[batch, n, k] with few k
// and n and many rows.  Row bits are X's address bits that are neither k nor
// batch bits, in X's order; runs of them that stay adjacent in C move as one
// segment.  k bits are in X's order, n bits in C's, so that neighbouring
// elements are neighbours in registers where they are in memory.
constexpr int kStreamMaxLog2K = 4;
constexpr int kStreamMaxLog2N = 4;
constexpr int kStreamMaxSegments = 12;
constexpr int kStreamMaxBatch = 15; // grid rows
struct StreamSegment {
    int8_t row, len, x, c; // row bits row..row+len-1 -> bits x.. of X, c.. of C
};
struct StreamShortK {
    int lr = 0, lk = 0, ln = 0, lb = 0; // log2 of rows, K, N, batch
    int n_segments = 0;
    StreamSegment segment[kStreamMaxSegments] = {};
    int8_t xk[kStreamMaxLog2K] = {}, yk[kStreamMaxLog2K] = {};
    int8_t yn[kStreamMaxLog2N] = {}, cn[kStreamMaxLog2N] = {};
    int8_t xb[kStreamMaxBatch] = {}, yb[kStreamMaxBatch] = {}, cb[kStreamMaxBatch] = {};
    int swap = 0; // X is the second operand
};

// False where the form does not apply: an extent that is not a power of two,
// more than 16 k or n, more than 2^15 batches, an operand beyond 2^31 elements,
// a batch bit among the lowest address bits of X or C, or a result whose
// lowest bits (a 128-byte line) are not n bits or rows that neighbouring
// threads own.
bool plan_stream_shortk(const std::vector<int32_t> &a, const std::vector<int64_t> &ea,
                        const std::vector<int32_t> &b, const std::vector<int64_t> &eb,
                        const std::vector<int32_t> &c, StreamShortK &p);

// C[batch, m, n] = sum over k of A[batch, m, k] B[batch, n, k] with few m and n
// and many k, the operands' k in different orders.  A tile is all m and n, the
// k bits on the lowest address bits of A and of B and any batch bits there:
// both operands' parts of it are contiguous runs, and LDS makes up the
// difference of the orders.
constexpr int kDotMaxLog2Tile = 11; // elements of one operand's tile, complex64
constexpr int kDotMaxLog2MN = 4;    // each of M and N
constexpr int kDotMaxLog2Sums = 4;  // outputs of one thread
constexpr int kDotMaxTileBatch = 5;
constexpr int kDotMaxLog2Lanes = 9; // outputs of one tile
struct StreamDot {
    int lm = 0, ln = 0, lk = 0, lb = 0; // log2 of M, N, K, batch
    int lt = 0, tb = 0; // k and batch bits of a tile
    int xm = 0;         // m bits across threads, so that a thread has <= 16 sums
    int8_t a_pos[12] = {}, b_pos[12] = {}; // address bit of tile bit j (ascending)
    int8_t ak[12] = {}, bk[12] = {};       // tile bits of the tile's k bits
    int8_t am[4] = {}, bn[4] = {};         // of m and n
    int8_t ab[5] = {}, bb[5] = {};         // of the tile's batch bits
    int8_t oak[24] = {}, obk[24] = {};     // address bits of the other k bits
    int8_t oab[16] = {}, obb[16] = {};     // of the other batch bits
    int8_t cm[4] = {}, cn[4] = {}, ctb[5] = {}, cob[16] = {}; // bits in C
    int swap = 0; // A is the second operand: the one with more m than the other has n
    int64_t outputs() const { return int64_t(1) << (lb + lm + ln); }
    // Partial sums per output: about four work-groups per CU, at most 4 MiB.
    int64_t chunks() const
    {
        int64_t c = 1;
        const int64_t batches = int64_t(1) << (lb - tb), tiles = int64_t(1) << (lk - lt);
        while (c < tiles && c * batches < 1024 && c * 2 * outputs() <= (1 << 18)) c *= 2;
        return c;
    }
};

// False where the form does not apply: an extent that is not a power of two,
// more than 16 m or n or 64 of both, more than 2^16 outputs (2^15 batches),
// fewer than 2^12 k, or lowest address bits (128 bytes' worth) that do not fit in a tile.
bool plan_stream_dot(int elem_bytes, const std::vector<int32_t> &a, const std::vector<int64_t> &ea,
                     const std::vector<int32_t> &b, const std::vector<int64_t> &eb,
                     const std::vector<int32_t> &c, StreamDot &p);

// LDS slot of tile element u (a linear map over bits, so that slots of
// disjoint bits combine by xor): low bits, the banks of one 256-byte row,
// xored with the next ones.
JH_HD uint32_t dot_slot(uint32_t u, int elem_bytes)
{
    return elem_bytes == 8 ? u ^ (((u >> 5) ^ (u >> 10)) & 31u)
                           : u ^ (((u >> 4) ^ (u >> 8)) & 15u);
}

JH_HD uint32_t stream_bits(const int8_t *pos, int n, uint32_t v)
{
    uint32_t o = 0;
    for (int i = 0; i < n; i++) o |= ((v >> i) & 1u) << pos[i];
    return o;
}

// The same for v below 2^n, over the whole array without a loop: on the device
// the positions are then kernel arguments in scalar registers (a loop loads
// each as it comes to it).
template <int N> JH_HD uint32_t stream_all_bits(const int8_t (&pos)[N], uint32_t v)
{
    uint32_t o = 0;
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
#endif
    for (int i = 0; i < N; i++) o |= ((v >> i) & 1u) << pos[i];
    return o;
}

JH_HD void stream_row(const StreamShortK &p, uint32_t row, uint32_t *x, uint32_t *c)
{
    uint32_t xo = 0, co = 0;
    for (int i = 0; i < p.n_segments; i++) {
        const StreamSegment s = p.segment[i];
        const uint32_t v = (row >> s.row) & ((1u << s.len) - 1u);
        xo |= v << s.x;
        co |= v << s.c;
    }
    *x = xo;
    *c = co;
}

#if defined(__HIPCC__)
void launch_stream_shortk(const StreamShortK &p, int elem_bytes, const void *a, const void *b,
                          void *c, hipStream_t stream);
// partials: 16 bytes per output and chunk.
void launch_stream_dot(const StreamDot &p, int elem_bytes, const void *a, const void *b, void *c,
                       void *partials, hipStream_t stream);
#endif

} // namespace jet_hip
