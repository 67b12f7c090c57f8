// stream.hpp -- contractions bound by reading their operands once, in the
// operands' own mode orders (every extent a power of two): a small tensor on
// a few modes of a large one (a gate on a state).
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

JH_HD uint32_t stream_bits(const int8_t *pos, int n, uint32_t v)
{
    uint32_t o = 0;
    for (int i = 0; i < n; i++) o |= ((v >> i) & 1u) << pos[i];
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
#endif

} // namespace jet_hip
