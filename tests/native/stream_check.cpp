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
    return d.stream_shortk ? 1 : 0;
}
