// permute_plan.cpp -- host-side planning of tensor permutations (pure C++,
// also compiled into the CPU emulation used by the test suite).
#include "permute_plan.hpp"

#include <algorithm>
#include <cstdlib>
#include <numeric>
#include <vector>

namespace jet_hip {

namespace {

bool is_pow2(int64_t v) { return v > 0 && (v & (v - 1)) == 0; }

int ilog2(int64_t v)
{
    int r = 0;
    while (v > 1) {
        v >>= 1;
        r++;
    }
    return r;
}

// Tiles for a permutation of axes with extents `ext` (input order), output
// axis i being input axis perm[i]; elems 0 where no tile has runs of 64 bytes
// on both sides.
TilePermParams plan_tiles(std::vector<int64_t> ext, std::vector<int> perm, int elem_bytes,
                          int64_t cap)
{
    TilePermParams t;
    int64_t numel = 1;
    for (int64_t e : ext) numel *= e;
    // The gather kernel takes as long as a launch below 2^17 elements.
    if (numel < (int64_t(1) << 17) || numel >= (int64_t(1) << 31)) return t;
    // Split long axes at the divisor nearest 32 between 8 and 64.
    for (int a = 0; a < (int)ext.size(); a++) {
        if (ext[a] <= 64) continue;
        int64_t best = 0;
        for (int64_t d = 8; d <= 64; d++)
            if (ext[a] % d == 0 && (!best || std::abs(d - 32) < std::abs(best - 32))) best = d;
        if (!best || best == ext[a]) continue;
        ext.insert(ext.begin() + a + 1, best);
        ext[a] /= best;
        for (int &x : perm)
            if (x > a) x++;
        perm.insert(std::find(perm.begin(), perm.end(), a) + 1, a + 1);
        a++;
    }
    const int r = (int)ext.size();
    std::vector<int64_t> in_stride(r), out_stride(r);
    for (int64_t a = r - 1, s = 1; a >= 0; s *= ext[a], a--) in_stride[a] = s;
    for (int64_t i = r - 1, s = 1; i >= 0; s *= ext[perm[i]], i--) out_stride[perm[i]] = s;
    // Trailing axes of the input and the output in turn, the shorter run first,
    // until both runs reach 256 bytes and a tile 1024 elements.
    const int64_t want = 256 / elem_bytes;
    std::vector<char> in_tile(r, 0);
    int n_tile = 0;
    int64_t elems = 1;
    int ia = r - 1, io = r - 1; // next axis of each side
    int64_t run_in = 1, run_out = 1;
    bool open_in = true, open_out = true;
    while (open_in || open_out) {
        while (ia >= 0 && in_tile[ia]) run_in *= ext[ia--];
        while (io >= 0 && in_tile[perm[io]]) run_out *= ext[perm[io--]];
        open_in = open_in && ia >= 0;
        open_out = open_out && io >= 0;
        if (run_in >= want && run_out >= want && elems >= 1024) break;
        if (!open_in && !open_out) break;
        const bool side_in = open_in && (!open_out || run_in <= run_out);
        const int a = side_in ? ia : perm[io];
        if (n_tile == kTileAxes || ext[a] > 128 || elems * ext[a] > cap) {
            (side_in ? open_in : open_out) = false;
            continue;
        }
        in_tile[a] = 1;
        n_tile++;
        elems *= ext[a];
    }
    if (run_in * elem_bytes < 64 || run_out * elem_bytes < 64 || elems < 256 ||
        r - n_tile > kOuterAxes)
        return t;
    int n = 0;
    std::vector<uint32_t> step_u(r, 0);
    uint32_t u = 1;
    for (int a = r - 1; a >= 0; a--)
        if (in_tile[a]) {
            t.in_ext[n] = uint32_t(ext[a]);
            t.in_step[n++] = uint32_t(in_stride[a]);
            step_u[a] = u;
            u *= uint32_t(ext[a]);
        }
    int m = 0;
    for (int i = r - 1; i >= 0; i--) {
        const int a = perm[i];
        if (in_tile[a]) {
            t.out_ext[m] = uint32_t(ext[a]);
            t.out_step[m] = uint32_t(out_stride[a]);
            t.out_u[m++] = step_u[a];
        }
        else {
            t.outer_ext[t.n_outer] = uint32_t(ext[a]);
            t.outer_in[t.n_outer] = uint32_t(in_stride[a]);
            t.outer_out[t.n_outer++] = uint32_t(out_stride[a]);
        }
    }
    for (int i = 0; i < kTileAxes; i++) {
        if (i >= n) t.in_ext[i] = t.out_ext[i] = 1, t.in_step[i] = t.out_step[i] = t.out_u[i] = 0;
        t.in_rec[i] = (uint32_t(1 << 20) + t.in_ext[i] - 1) / t.in_ext[i];
        t.out_rec[i] = (uint32_t(1 << 20) + t.out_ext[i] - 1) / t.out_ext[i];
    }
    t.elems = int(elems);
    t.cap = int(cap);
    t.tiles = uint32_t(numel / elems);
    return t;
}

} // namespace

PermutePlan make_permute_plan(int rank, const int64_t *extents,
                              const int32_t *perm)
{
    PermutePlan plan;
    JH_REQUIRE(rank >= 0 && rank <= kMaxRank, "Permutation rank exceeds 64.");
    int64_t numel = 1;
    for (int i = 0; i < rank; i++) {
        JH_REQUIRE(extents[i] >= 1, "Tensor extents must be positive.");
        numel *= extents[i];
    }
    plan.numel = numel;
    {
        std::vector<int> seen(rank, 0);
        for (int i = 0; i < rank; i++) {
            JH_REQUIRE(perm[i] >= 0 && perm[i] < rank && !seen[perm[i]],
                       "New indices are an invalid permutation of the existing indices");
            seen[perm[i]] = 1;
        }
    }
    // Drop extent-1 axes.
    std::vector<int> keep_map(rank, -1);
    std::vector<int64_t> e;
    for (int a = 0; a < rank; a++) {
        if (extents[a] > 1) {
            keep_map[a] = (int)e.size();
            e.push_back(extents[a]);
        }
    }
    std::vector<int> p;
    for (int i = 0; i < rank; i++)
        if (keep_map[perm[i]] >= 0) p.push_back(keep_map[perm[i]]);
    // Merge runs of input axes that stay adjacent in the output.
    std::vector<std::vector<int>> groups;
    for (size_t i = 0; i < p.size(); i++) {
        if (!groups.empty() && groups.back().back() + 1 == p[i])
            groups.back().push_back(p[i]);
        else
            groups.push_back({p[i]});
    }
    const int r = (int)groups.size();
    if (r <= 1 || numel <= 1) {
        plan.kind = PermutePlan::kCopy;
        return plan;
    }
    std::vector<int> by_input(r);
    std::iota(by_input.begin(), by_input.end(), 0);
    std::sort(by_input.begin(), by_input.end(),
              [&](int x, int y) { return groups[x][0] < groups[y][0]; });
    std::vector<int> group_to_in(r);
    std::vector<int64_t> me(r);
    for (int a = 0; a < r; a++) {
        group_to_in[by_input[a]] = a;
        int64_t ext = 1;
        for (int ax : groups[by_input[a]]) ext *= e[ax];
        me[a] = ext;
    }
    std::vector<int> mp(r);
    for (int i = 0; i < r; i++) mp[i] = group_to_in[i];

    bool pow2 = true;
    for (int a = 0; a < r; a++) pow2 = pow2 && is_pow2(me[a]);

    if (!pow2) {
        plan.kind = PermutePlan::kGeneric;
        GenericPermParams &g = plan.gen;
        g.rank = r;
        std::vector<int64_t> in_stride(r);
        in_stride[r - 1] = 1;
        for (int a = r - 1; a > 0; a--) in_stride[a - 1] = in_stride[a] * me[a];
        for (int i = 0; i < r; i++) {
            g.out_ext[i] = me[mp[i]];
            g.in_stride[i] = in_stride[mp[i]];
        }
        // Small tiles first: a thread finds fewer offsets.  Past the last-level
        // cache longer runs count for more (2^26 complex128 493 us at 2048, 608 at
        // 1024; 2^23 complex64 31 us at 2048, 27 at 1024, 42 at 4096 alone).
        for (int64_t e : {8, 16}) {
            TilePermParams &t = e == 8 ? plan.tiles8 : plan.tiles16;
            for (int64_t cap = plan.numel * e > kPermCacheBytes ? 2048 : 1024;
                 cap * e <= kTileBytes && !t.elems; cap *= 2)
                t = plan_tiles(me, mp, int(e), cap);
        }
        return plan;
    }

    // Bit permutation: dst[b] = output bit of input bit b.
    std::vector<int> L(r), lo_in(r), lo_out(r);
    for (int a = 0; a < r; a++) L[a] = ilog2(me[a]);
    int acc = 0;
    for (int a = r - 1; a >= 0; a--) {
        lo_in[a] = acc;
        acc += L[a];
    }
    const int nbits = acc;
    JH_REQUIRE(nbits <= 62, "Tensor too large for the bit permutation kernel.");
    acc = 0;
    for (int i = r - 1; i >= 0; i--) {
        lo_out[i] = acc;
        acc += L[mp[i]];
    }
    std::vector<int> dst(nbits), src(nbits);
    for (int i = 0; i < r; i++)
        for (int j = 0; j < L[mp[i]]; j++) dst[lo_in[mp[i]] + j] = lo_out[i] + j;
    for (int b = 0; b < nbits; b++) src[dst[b]] = b;

    // Tile: alternately add the next lowest input bit and the input bit of
    // the next lowest output bit until the tile holds `target` bits.
    const int target = std::min(nbits, kTileMaxBits);
    std::vector<char> in_tile(nbits, 0);
    int count = 0, ti = 0, to = 0;
    while (count < target) {
        if (ti <= to && ti < nbits) {
            const int b = ti++;
            if (!in_tile[b]) {
                in_tile[b] = 1;
                count++;
            }
        }
        else if (to < nbits) {
            const int b = src[to++];
            if (!in_tile[b]) {
                in_tile[b] = 1;
                count++;
            }
        }
        else
            break;
    }
    BitPermParams &bp = plan.bits;
    bp.nbits = nbits;
    bp.tb = count;
    int contiguous = 0;
    while (contiguous < nbits && in_tile[contiguous]) contiguous++;
    bp.ti = contiguous;
    std::vector<int> tile_in, tile_by_out;
    for (int b = 0; b < nbits; b++)
        if (in_tile[b]) tile_in.push_back(b);
    for (int o = 0; o < nbits; o++)
        if (in_tile[src[o]]) tile_by_out.push_back(src[o]);
    for (int j = 0; j < count; j++) {
        bp.tile_in[j] = (int8_t)tile_in[j];
        bp.tile_out[j] = (int8_t)dst[tile_by_out[j]];
        const int upos = (int)(std::find(tile_in.begin(), tile_in.end(), tile_by_out[j]) -
                               tile_in.begin());
        bp.v2u[j] = (int8_t)upos;
    }
    // Past the last-level cache, tiles next to each other in the input and in
    // the output by turns (complex64 2^26 4.70 -> 5.17 TB/s, 2^28 4.60 -> 4.97); below,
    // in the input's order (2^23 5.0 TB/s, by turns 4.65).
    int nr = 0;
    std::vector<char> done(in_tile);
    for (int i = 0, o = 0, turn = 0;; turn ^= 1) {
        while (i < nbits && done[i]) i++;
        while (o < nbits && done[src[o]]) o++;
        if (i == nbits) break;
        const int b = turn && nbits >= kPermCacheBits ? src[o] : i;
        done[b] = 1;
        bp.outer_in[nr] = (int8_t)b;
        bp.outer_out[nr++] = (int8_t)dst[b];
    }
    bp.nr = nr;
    plan.kind = PermutePlan::kBits;
    return plan;
}

} // namespace jet_hip
