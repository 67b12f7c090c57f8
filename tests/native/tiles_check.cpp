// tiles_check.cpp -- tiled generic permutations (jet_amd/csrc/permute_plan.hpp)
// replayed on the CPU.
#include "../../jet_amd/csrc/permute_plan.hpp"

#include <vector>

using namespace jet_hip;

// out[o] = input offset that the tiled kernel writes to output element o.
// Returns the elements of a tile (0: not tiled), or -1 for an offset or slot out
// of range, -2 for an element written twice or never.
extern "C" int tiled_permutation(int elem_bytes, int rank, const int64_t *ext, const int32_t *perm,
                                 int64_t *out)
{
    const PermutePlan plan = make_permute_plan(rank, ext, perm);
    if (plan.kind != PermutePlan::kGeneric) return 0;
    const TilePermParams &p = elem_bytes == 8 ? plan.tiles8 : plan.tiles16;
    if (!p.elems) return 0;
    const int64_t cap = p.cap;
    if (p.elems > cap || cap * elem_bytes > kTileBytes || int64_t(p.elems) * p.tiles != plan.numel) return -1;
    for (int64_t i = 0; i < plan.numel; i++) out[i] = -1;
    std::vector<int64_t> lds(cap + cap / 32);
    for (uint32_t w = 0; w < p.tiles; w++) {
        uint32_t bi, bo, src;
        tile_axes_base(p, w, &bi, &bo);
        for (int u = 0; u < p.elems; u++) {
            const int64_t i = int64_t(bi) + tile_axes_offset(p.in_ext, p.in_rec, p.in_step, p.in_step, u, &src);
            if (i >= plan.numel || tile_axes_slot(u) >= lds.size()) return -1;
            lds[tile_axes_slot(u)] = i;
        }
        for (int u = 0; u < p.elems; u++) {
            const int64_t o = int64_t(bo) + tile_axes_offset(p.out_ext, p.out_rec, p.out_step, p.out_u, u, &src);
            if (o >= plan.numel || src >= uint32_t(p.elems)) return -1;
            if (out[o] >= 0) return -2;
            out[o] = lds[tile_axes_slot(src)];
        }
    }
    for (int64_t i = 0; i < plan.numel; i++)
        if (out[i] < 0) return -2;
    return p.elems;
}
