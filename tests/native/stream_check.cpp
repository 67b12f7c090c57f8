// stream_check.cpp -- the offset arithmetic of the in-place contractions
// (jet_amd/csrc/stream.hpp) replayed on the CPU in complex128.
#include "../../jet_amd/csrc/contract_plan.hpp"

#include <vector>

using namespace jet_hip;

// C of a contraction through plan_stream_shortk.  Returns 1 where the form
// does not apply, 2 for an offset out of range, 3 for an element of C written
// twice or never.
extern "C" int stream_shortk_emulate(int ra, const int32_t *ma, const int64_t *ea, int rb,
                                     const int32_t *mb, const int64_t *eb, int rc,
                                     const int32_t *mc, const double *a, const double *b,
                                     int64_t nc, double *c)
{
    StreamShortK p;
    if (!plan_stream_shortk({ma, ma + ra}, {ea, ea + ra}, {mb, mb + rb}, {eb, eb + rb},
                            {mc, mc + rc}, p))
        return 1;
    int64_t na = 1, nb = 1;
    for (int i = 0; i < ra; i++) na *= ea[i];
    for (int i = 0; i < rb; i++) nb *= eb[i];
    const double *x = p.swap ? b : a, *y = p.swap ? a : b;
    const int64_t nx = p.swap ? nb : na, ny = p.swap ? na : nb;
    std::vector<char> seen(nc, 0);
    for (uint32_t bt = 0; bt < 1u << p.lb; bt++)
        for (uint32_t row = 0; row < 1u << p.lr; row++) {
            uint32_t xo, co;
            stream_row(p, row, &xo, &co);
            xo |= stream_bits(p.xb, p.lb, bt);
            co |= stream_bits(p.cb, p.lb, bt);
            for (uint32_t n = 0; n < 1u << p.ln; n++) {
                double re = 0, im = 0;
                for (uint32_t k = 0; k < 1u << p.lk; k++) {
                    const int64_t i = xo | stream_bits(p.xk, p.lk, k);
                    const int64_t j = stream_bits(p.yb, p.lb, bt) |
                                      stream_bits(p.yn, p.ln, n) | stream_bits(p.yk, p.lk, k);
                    if (i >= nx || j >= ny) return 2;
                    re += x[2 * i] * y[2 * j] - x[2 * i + 1] * y[2 * j + 1];
                    im += x[2 * i] * y[2 * j + 1] + x[2 * i + 1] * y[2 * j];
                }
                const int64_t o = co | stream_bits(p.cn, p.ln, n);
                if (o >= nc) return 2;
                if (seen[o]++) return 3;
                c[2 * o] = re;
                c[2 * o + 1] = im;
            }
        }
    for (char s : seen)
        if (!s) return 3;
    return 0;
}

// Whether plan_contraction routes complex64 operands (mode 0) to the form, and the
// workspace it then needs.
extern "C" int stream_route(int ra, const int32_t *ma, const int64_t *ea, int rb,
                            const int32_t *mb, const int64_t *eb, int rc, const int32_t *mc,
                            size_t *workspace)
{
    const ContractionDesc d = plan_contraction(8, 0, 0, ra, ma, ea, rb, mb, eb, rc, mc);
    *workspace = d.workspace;
    return d.stream_shortk ? 1 : d.stream_dot ? 2 : 0;
}

// C of a contraction through plan_stream_dot: every work-group's tiles, threads
// and slots as stream_dot_kernel computes them (complex64 tiles).  Returns 1
// where the form does not apply, 2 for an offset out of range, 3 for an operand
// value read into a tile twice or never, 4 for an output missed.
extern "C" int stream_dot_emulate(int elem_bytes, int ra, const int32_t *ma, const int64_t *ea,
                                  int rb, const int32_t *mb, const int64_t *eb, int rc,
                                  const int32_t *mc, const double *a, const double *b, int64_t nc,
                                  double *c)
{
    StreamDot p;
    if (!plan_stream_dot(elem_bytes, {ma, ma + ra}, {ea, ea + ra}, {mb, mb + rb}, {eb, eb + rb},
                         {mc, mc + rc}, p))
        return 1;
    int64_t na = 1, nb = 1;
    for (int i = 0; i < ra; i++) na *= ea[i];
    for (int i = 0; i < rb; i++) nb *= eb[i];
    if (p.swap) {
        std::swap(a, b);
        std::swap(na, nb);
    }
    const int64_t cap = elem_bytes == 8 ? 1 << kDotMaxLog2Tile : 1 << (kDotMaxLog2Tile - 1);
    const int la = p.lt + p.lm + p.tb, lb = p.lt + p.ln + p.tb;
    if ((1 << la) > cap || (1 << lb) > cap || p.chunks() > (int64_t(1) << (p.lk - p.lt))) return 2;
    std::vector<char> seen_a(na, 0), seen_b(nb, 0), seen_c(nc, 0);
    const int low = p.tb + p.xm, kl = 8 - low, LM = p.lm - p.xm;
    if (low > 6 || kl > p.lt || LM + p.ln > kDotMaxLog2Sums || low + LM + p.ln > kDotMaxLog2Lanes)
        return 2;
    std::vector<double> sa(2 * cap), sb(2 * cap);
    for (uint32_t bt = 0; bt < 1u << (p.lb - p.tb); bt++)
        for (uint32_t t = 0; t < 1u << (p.lk - p.lt); t++) {
            const uint32_t ba = stream_bits(p.oab, p.lb - p.tb, bt) | stream_bits(p.oak, p.lk - p.lt, t);
            const uint32_t bb = stream_bits(p.obb, p.lb - p.tb, bt) | stream_bits(p.obk, p.lk - p.lt, t);
            for (uint32_t u = 0; u < 1u << la; u++) {
                const int64_t i = ba + stream_bits(p.a_pos, la, u), s = dot_slot(u, elem_bytes);
                if (i >= na || s >= cap) return 2;
                if (seen_a[i]++) return 3;
                sa[2 * s] = a[2 * i], sa[2 * s + 1] = a[2 * i + 1];
            }
            for (uint32_t u = 0; u < 1u << lb; u++) {
                const int64_t i = bb + stream_bits(p.b_pos, lb, u), s = dot_slot(u, elem_bytes);
                if (i >= nb || s >= cap) return 2;
                if (seen_b[i]++) return 3;
                sb[2 * s] = b[2 * i], sb[2 * s + 1] = b[2 * i + 1];
            }
            for (uint32_t tid = 0; tid < 256; tid++) {
                const uint32_t tbv = tid & ((1u << p.tb) - 1), mx = (tid >> p.tb) & ((1u << p.xm) - 1);
                const uint32_t ua = dot_slot(stream_bits(p.ab, p.tb, tbv) |
                                                 stream_bits(p.am + LM, p.xm, mx) |
                                                 stream_bits(p.ak, kl, tid >> low), elem_bytes);
                const uint32_t ub = dot_slot(stream_bits(p.bb, p.tb, tbv) |
                                                 stream_bits(p.bk, kl, tid >> low), elem_bytes);
                for (uint32_t it = 0; it < 1u << (p.lt - kl); it++)
                    for (uint32_t m = 0; m < 1u << LM; m++)
                        for (uint32_t n = 0; n < 1u << p.ln; n++) {
                            const uint32_t x = ua ^ dot_slot(stream_bits(p.ak + kl, p.lt - kl, it), elem_bytes) ^
                                               dot_slot(stream_bits(p.am, LM, m), elem_bytes);
                            const uint32_t y = ub ^ dot_slot(stream_bits(p.bk + kl, p.lt - kl, it), elem_bytes) ^
                                               dot_slot(stream_bits(p.bn, p.ln, n), elem_bytes);
                            if (x >= cap || y >= cap) return 2;
                            const int64_t o = stream_bits(p.cn, p.ln, n) |
                                              stream_bits(p.cm, p.lm, (mx << LM) | m) |
                                              stream_bits(p.ctb, p.tb, tbv) |
                                              stream_bits(p.cob, p.lb - p.tb, bt);
                            if (o >= nc) return 2;
                            seen_c[o] = 1;
                            c[2 * o] += sa[2 * x] * sb[2 * y] - sa[2 * x + 1] * sb[2 * y + 1];
                            c[2 * o + 1] += sa[2 * x] * sb[2 * y + 1] + sa[2 * x + 1] * sb[2 * y];
                        }
            }
        }
    for (char s : seen_a)
        if (!s) return 3;
    for (char s : seen_b)
        if (!s) return 3;
    for (char s : seen_c)
        if (!s) return 4;
    return 0;
}
