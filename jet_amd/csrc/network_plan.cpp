// network_plan.cpp -- host-side plan of a contraction sequence.
#include "network_plan.hpp"

#include <algorithm>
#include <iterator>
#include <limits>
#include <map>
#include <set>
#include <unordered_map>

namespace jet_hip {

namespace {

size_t align256(size_t x) { return (x + 255) & ~size_t(255); }

int find(const std::vector<int32_t> &v, int32_t x)
{
    for (size_t i = 0; i < v.size(); i++)
        if (v[i] == x) return (int)i;
    return -1;
}

// Best-fit allocator over a virtual address range; tracks the high-water mark.
class ArenaSim {
  public:
    size_t alloc(size_t bytes)
    {
        bytes = align256(std::max<size_t>(bytes, 256));
        auto best = free_.end();
        for (auto it = free_.begin(); it != free_.end(); ++it)
            if (it->second >= bytes && (best == free_.end() || it->second < best->second)) best = it;
        size_t off;
        if (best != free_.end()) {
            off = best->first;
            const size_t rest = best->second - bytes;
            free_.erase(best);
            if (rest) free_[off + bytes] = rest;
        }
        else {
            // Grow at the end (merging a free block that ends at the top).
            off = top_;
            if (!free_.empty()) {
                auto last = std::prev(free_.end());
                if (last->first + last->second == top_) {
                    off = last->first;
                    free_.erase(last);
                }
            }
            top_ = off + bytes;
        }
        used_[off] = bytes;
        return off;
    }
    void release(size_t off)
    {
        auto it = used_.find(off);
        if (it == used_.end()) return;
        size_t start = off, len = it->second;
        used_.erase(it);
        auto nx = free_.lower_bound(start);
        if (nx != free_.end() && start + len == nx->first) {
            len += nx->second;
            nx = free_.erase(nx);
        }
        if (nx != free_.begin()) {
            auto pv = std::prev(nx);
            if (pv->first + pv->second == start) {
                start = pv->first;
                len += pv->second;
                free_.erase(pv);
            }
        }
        free_[start] = len;
    }
    size_t high_water() const { return top_; }

  private:
    std::map<size_t, size_t> free_; // offset -> length
    std::map<size_t, size_t> used_;
    size_t top_ = 0;
};

// Fewer small steps than this run as launches of their own: a group saves 3-4 us a
// step and costs a table of pointers, set on each execution (2.6 us).
constexpr int kMinGrouped = 16;
constexpr int kDagWindow = 64, kDagOverlap = 4;

// Whether a step can run in a group, and its offsets there: the mode groups
// of plan_contraction (batch, left and right in the result's order, common
// in A's).
bool plan_small_step(const std::vector<int32_t> &A, const std::vector<int64_t> &ea,
                     const std::vector<int32_t> &B, const std::vector<int64_t> &eb,
                     const NetworkStep &st, FusedSmall &f)
{
    const ContractionDesc &d = st.desc;
    const double outputs = double(d.size_c), k = d.flops / (8.0 * outputs);
    if (outputs > double(1 << kGroupMaxLog2Outputs) || k > double(1 << kGroupMaxLog2K) ||
        outputs * k > double(1 << kGroupMaxLog2Work))
        return false;
    std::vector<int32_t> batch, left, right, common;
    for (int32_t m : st.modes) {
        const bool in_a = find(A, m) >= 0, in_b = find(B, m) >= 0;
        (in_a && in_b ? batch : in_a ? left : right).push_back(m);
    }
    for (int32_t m : A)
        if (find(B, m) >= 0 && find(st.modes, m) < 0) common.push_back(m);
    return plan_fused_small(A, ea, B, eb, st.modes, batch, left, right, common, f);
}

// Marks the steps that run in groups (none where they are few).
void choose_grouped(NetworkPlan &np, const std::vector<std::vector<int32_t>> &modes,
                    const std::vector<std::vector<int64_t>> &exts)
{
    int n = 0;
    for (NetworkStep &st : np.steps) {
        st.grouped = plan_small_step(modes[st.a], exts[st.a], modes[st.b], exts[st.b], st,
                                     st.small);
        n += st.grouped;
    }
    if (n < kMinGrouped)
        for (NetworkStep &st : np.steps) st.grouped = false;
    // complex64 results that only groups read stay in FP64, as they are summed:
    // rounded at the few steps that other kernels read, at no cost (the loads wait on
    // latency).  Products with a leaf (in DAGs, whose reverse steps have a leaf's
    // value in most products, of two leaves) are rounded like the leaves, which
    // is never less exact than FP32 results everywhere, but neither as exact for
    // the leaves' own values as FP64 everywhere: rings of 18 to 32 random leaves
    // 1.4-1.8e-7 with FP32 results, 0.8-1.1e-7 so, 0.2-0.3e-7 with FP64 ones.  It
    // stands for circuits, whose leaves are rounded roots of 1/2: their products
    // round back to what the gates' products are, which FP64 results keep from
    // happening.  Against the gates in 64 bits, in the same order: eight sets of
    // amplitudes of 42 qubits 1.2-1.6e-6, 0.9-1.8e-6, 1.6-2.3e-6, twelve losses of 36
    // qubits 1.2e-6, 0.9e-6, 2.0e-6, their gradients 1.5e-6, 1.0e-6, 2.1e-6.
    std::vector<int> depth(np.n_leaves, 0);
    for (size_t s = 0; s < np.steps.size(); s++) {
        NetworkStep &st = np.steps[s];
        depth.push_back(std::max(depth[st.a], depth[st.b]) + 1);
        st.wide = np.elem_bytes == 8 && st.grouped && !st.is_root && !(np.dag && np.kept[s]) &&
                  (np.dag ? depth.back() > 1 : st.a >= np.n_leaves && st.b >= np.n_leaves);
    }
    for (const NetworkStep &st : np.steps)
        if (!st.grouped)
            for (int x : {st.a, st.b})
                if (x >= np.n_leaves) np.steps[x - np.n_leaves].wide = false;
}

// The launches: the steps that run alone in their order, and before each (and
// after the last) the small steps that follow from what has run so far, by
// level.  With `delay` (contraction DAGs, whose recomputed values would
// otherwise all be computed first and live long) a small step goes at most
// kDagOverlap levels below the steps of earlier windows of kDagWindow steps, then
// moves to the last group before its first use (no launch more).  A step
// that reads the arena stays within the steps it stood between, which its
// operand outlives.  On the 4x4 depth-8 gradient with every fourth value
// kept: 31 levels instead of 24, 86 KB of results instead of 114.
// Returns the launch of every step.
std::vector<int> plan_launches(NetworkPlan &np, bool delay)
{
    const int n_steps = (int)np.steps.size();
    // (epoch, level): steps that run alone before the node, and its group's
    // level among the groups that follow the same ones
    typedef std::pair<int, int> Place;
    std::vector<Place> place(np.n_leaves + n_steps, Place(0, -1));
    Place top(0, -1), base(0, 0); // latest place so far; earliest of this window
    std::vector<int> single, before(n_steps);
    std::map<Place, std::vector<int>> groups;
    for (int s = 0; s < n_steps; s++) {
        const NetworkStep &st = np.steps[s];
        Place &p = place[np.n_leaves + s];
        before[s] = (int)single.size();
        if (!st.grouped) {
            single.push_back(s);
            p = Place((int)single.size(), -1);
            top = std::max(top, p);
            continue;
        }
        p = std::max(place[st.a], place[st.b]);
        p.second++;
        if (delay) {
            if (s % kDagWindow == 0) base = Place(top.first, std::max(0, top.second - kDagOverlap));
            p = std::max(p, base);
            top = std::max(top, p);
        }
        groups[p];
    }
    if (delay) {
        // last group at or before a place
        auto last_at = [&](Place p) { return std::prev(groups.upper_bound(p))->first; };
        std::vector<Place> latest(np.n_leaves + n_steps, Place(-1, -1));
        auto use = [&](int node, Place p) {
            if (latest[node].first < 0 || p < latest[node]) latest[node] = p;
        };
        for (int s = n_steps - 1; s >= 0; s--) {
            const NetworkStep &st = np.steps[s];
            Place &p = place[np.n_leaves + s];
            Place last(before[s], std::numeric_limits<int>::max());
            if (st.grouped) {
                Place l = latest[np.n_leaves + s];
                for (int x : {st.a, st.b})
                    if (x >= np.n_leaves && !np.steps[x - np.n_leaves].grouped && last < l)
                        l = last;
                if (l.first >= 0) p = std::max(p, last_at(l));
                last = Place(p.first, p.second - 1);
            }
            use(st.a, last);
            use(st.b, last);
        }
    }
    for (int s = 0; s < n_steps; s++)
        if (np.steps[s].grouped) groups[place[np.n_leaves + s]].push_back(s);

    std::vector<int> launch_of(n_steps);
    auto it = groups.begin();
    for (int e = 0; e <= (int)single.size(); e++) {
        for (; it != groups.end() && it->first.first == e; ++it) {
            if (it->second.empty()) continue;
            NetworkLaunch l;
            l.first_block = (int)np.blocks.size();
            for (int s : it->second) {
                const NetworkStep &st = np.steps[s];
                launch_of[s] = (int)np.launches.size();
                GroupBlock g = group_record(st.small);
                g.a = np.slot(st.a);
                g.b = np.slot(st.b);
                g.c = st.is_root ? np.n_leaves : np.slot(np.n_leaves + s);
                g.wide = np.wide(st.a) | np.wide(st.b) << 1 | st.wide << 2;
                g.lanes = group_lanes(g, 6, 16); // shuffles within a wave; 256 work-groups
                for (g.first = 0; g.first < 1 << g.lo; g.first += 256 >> g.lanes)
                    np.blocks.push_back(g);
                l.flops += st.desc.flops;
            }
            l.n_blocks = (int)np.blocks.size() - l.first_block;
            np.launches.push_back(l);
        }
        if (e < (int)single.size()) {
            NetworkLaunch l;
            l.step = single[e];
            l.flops = np.steps[l.step].desc.flops;
            launch_of[l.step] = (int)np.launches.size();
            np.launches.push_back(l);
        }
    }
    return launch_of;
}

} // namespace

NetworkPlan plan_network(int elem_bytes, int mode, int n_leaves,
                         const int32_t *leaf_ranks, const int32_t *leaf_modes,
                         const int64_t *leaf_extents, int n_steps,
                         const int32_t *path, int n_out,
                         const int32_t *out_modes)
{
    JH_REQUIRE(n_leaves >= 1, "An empty tensor network cannot be contracted.");
    JH_REQUIRE(n_steps >= 0 && n_out >= 0, "Invalid network description.");
    NetworkPlan np;
    np.elem_bytes = elem_bytes;
    np.n_leaves = n_leaves;
    np.out_modes.assign(out_modes, out_modes + n_out);
    const int n_nodes = n_leaves + n_steps;

    std::vector<std::vector<int32_t>> modes(n_nodes);
    std::vector<std::vector<int64_t>> exts(n_nodes);
    std::unordered_map<int32_t, int64_t> extent_of;
    size_t pos = 0;
    for (int i = 0; i < n_leaves; i++) {
        JH_REQUIRE(leaf_ranks[i] >= 0 && leaf_ranks[i] <= kMaxRank, "Leaf rank must be 0..64.");
        modes[i].assign(leaf_modes + pos, leaf_modes + pos + leaf_ranks[i]);
        exts[i].assign(leaf_extents + pos, leaf_extents + pos + leaf_ranks[i]);
        pos += leaf_ranks[i];
        for (size_t j = 0; j < modes[i].size(); j++) {
            auto it = extent_of.find(modes[i][j]);
            JH_REQUIRE(it == extent_of.end() || it->second == exts[i][j],
                       "An index has different extents in different tensors.");
            extent_of[modes[i][j]] = exts[i][j];
        }
    }
    np.leaf_modes.assign(modes.begin(), modes.begin() + n_leaves);
    np.leaf_extents.assign(exts.begin(), exts.begin() + n_leaves);
    for (int32_t m : np.out_modes) {
        JH_REQUIRE(extent_of.count(m), "Output index is not an index of the network.");
        np.out_extents.push_back(extent_of[m]);
    }
    const std::set<int32_t> open(np.out_modes.begin(), np.out_modes.end());

    // How many not-yet-consumed nodes hold each mode (hyperedges count > 2).
    std::unordered_map<int32_t, int> holders;
    for (int i = 0; i < n_leaves; i++)
        for (int32_t m : modes[i]) holders[m]++;

    std::vector<char> consumed(n_nodes, 0);
    std::vector<int> last_use(n_nodes, -1);
    for (int s = 0; s < n_steps; s++) {
        const int a = path[2 * s], b = path[2 * s + 1];
        JH_REQUIRE(a >= 0 && b >= 0 && a < n_leaves + s && b < n_leaves + s && a != b,
                   "Node ID in contraction path pair is invalid.");
        JH_REQUIRE(!consumed[a] && !consumed[b], "A node is contracted twice in the path.");
        consumed[a] = consumed[b] = 1;
        last_use[a] = last_use[b] = s;
    }
    if (n_steps > 0) {
        int unconsumed = 0;
        for (int i = 0; i < n_nodes; i++) unconsumed += !consumed[i];
        JH_REQUIRE(unconsumed == 1, "The path does not contract the network to one tensor.");
    }
    else {
        JH_REQUIRE(n_leaves == 1, "The path does not contract the network to one tensor.");
    }

    np.steps.resize(n_steps);
    for (int s = 0; s < n_steps; s++) {
        NetworkStep &st = np.steps[s];
        st.a = path[2 * s];
        st.b = path[2 * s + 1];
        const auto &A = modes[st.a], &B = modes[st.b];
        for (int32_t m : A) holders[m]--;
        for (int32_t m : B) holders[m]--;
        // Result: batch (shared and kept) in A's order, then A's free modes,
        // then B's free modes -- the GEMM's natural [batch][left][right].
        std::vector<int32_t> batch, left, right;
        for (int32_t m : A) {
            const bool in_b = find(B, m) >= 0;
            const bool keep = open.count(m) || holders[m] > 0;
            if (in_b && keep)
                batch.push_back(m);
            else if (!in_b)
                left.push_back(m);
        }
        for (int32_t m : B)
            if (find(A, m) < 0) right.push_back(m);
        std::vector<int32_t> out = batch;
        out.insert(out.end(), left.begin(), left.end());
        out.insert(out.end(), right.begin(), right.end());
        st.is_root = (s == n_steps - 1);
        if (st.is_root) {
            std::vector<int32_t> sorted_out = out, sorted_req = np.out_modes;
            std::sort(sorted_out.begin(), sorted_out.end());
            std::sort(sorted_req.begin(), sorted_req.end());
            JH_REQUIRE(sorted_out == sorted_req,
                       "Output indices do not match the indices left after the last step.");
            out = np.out_modes;
        }
        for (int32_t m : out) {
            st.modes.push_back(m);
            st.extents.push_back(extent_of[m]);
            holders[m]++;
        }
        modes[n_leaves + s] = st.modes;
        exts[n_leaves + s] = st.extents;
        st.desc = plan_contraction(elem_bytes, mode, 0, (int)A.size(), A.data(),
                                   exts[st.a].data(), (int)B.size(), B.data(),
                                   exts[st.b].data(), (int)st.modes.size(), st.modes.data());
        np.flops += st.desc.flops;
        np.workspace_bytes = std::max(np.workspace_bytes, st.desc.workspace);
    }
    choose_grouped(np, modes, exts);
    ArenaSim arena;
    std::vector<size_t> offset(n_nodes, 0);
    for (int s = 0; s < n_steps; s++) {
        NetworkStep &st = np.steps[s];
        if (!st.is_root && !st.grouped) {
            offset[n_leaves + s] = arena.alloc(np.result_bytes(s));
            st.offset = offset[n_leaves + s];
        }
        for (int id : {st.a, st.b})
            if (id >= n_leaves && last_use[id] == s && !np.steps[id - n_leaves].grouped)
                arena.release(offset[id]);
    }
    np.arena_bytes = arena.high_water();
    for (int s = 0; s < n_steps; s++) {
        NetworkStep &st = np.steps[s];
        if (!st.grouped || st.is_root) continue;
        st.offset = align256(np.arena_bytes);
        np.arena_bytes = st.offset + np.result_bytes(s);
    }
    plan_launches(np, false);
    if (n_steps == 0) {
        std::vector<int32_t> perm(np.out_modes.size());
        JH_REQUIRE(np.out_modes.size() == modes[0].size(),
                   "Output indices do not match the indices of the single tensor.");
        for (size_t i = 0; i < perm.size(); i++) {
            perm[i] = find(modes[0], np.out_modes[i]);
            JH_REQUIRE(perm[i] >= 0, "Output indices do not match the indices of the single tensor.");
        }
        np.root_copy = make_permute_plan((int)perm.size(), exts[0].data(), perm.data());
    }
    return np;
}


NetworkPlan plan_dag(int elem_bytes, int mode, int n_leaves, const int32_t *leaf_ranks,
                     const int32_t *leaf_modes, const int64_t *leaf_extents, int n_steps,
                     const int32_t *steps, int n_keep, const int32_t *keep)
{
    JH_REQUIRE(n_leaves >= 1 && n_steps >= 1 && n_keep >= 0, "Invalid contraction DAG.");
    NetworkPlan np;
    np.dag = true;
    np.elem_bytes = elem_bytes;
    np.n_leaves = n_leaves;
    const int n_nodes = n_leaves + n_steps;
    std::vector<std::vector<int32_t>> modes(n_nodes);
    std::vector<std::vector<int64_t>> exts(n_nodes);
    std::unordered_map<int32_t, int64_t> extent_of;
    size_t pos = 0;
    for (int i = 0; i < n_leaves; i++) {
        JH_REQUIRE(leaf_ranks[i] >= 0 && leaf_ranks[i] <= kMaxRank, "Leaf rank must be 0..64.");
        modes[i].assign(leaf_modes + pos, leaf_modes + pos + leaf_ranks[i]);
        exts[i].assign(leaf_extents + pos, leaf_extents + pos + leaf_ranks[i]);
        pos += leaf_ranks[i];
        for (size_t j = 0; j < modes[i].size(); j++) {
            auto it = extent_of.find(modes[i][j]);
            JH_REQUIRE(it == extent_of.end() || it->second == exts[i][j],
                       "An index has different extents in different tensors.");
            extent_of[modes[i][j]] = exts[i][j];
        }
    }
    np.leaf_modes.assign(modes.begin(), modes.begin() + n_leaves);
    np.leaf_extents.assign(exts.begin(), exts.begin() + n_leaves);

    std::vector<int> last_use(n_nodes, -1);
    for (int s = 0; s < n_steps; s++) {
        const int a = steps[2 * s], b = steps[2 * s + 1];
        JH_REQUIRE(a >= 0 && b >= 0 && a < n_leaves + s && b < n_leaves + s && a != b,
                   "Node ID in contraction path pair is invalid.");
        last_use[a] = last_use[b] = s;
    }
    np.kept.assign(n_steps, 0);
    std::vector<int> keep_order;
    for (int i = 0; i < n_keep; i++) {
        const int id = keep[i];
        JH_REQUIRE(id >= n_leaves && id < n_nodes, "Only step results can be kept.");
        JH_REQUIRE(!np.kept[id - n_leaves], "A step result is kept twice.");
        np.kept[id - n_leaves] = 1;
        keep_order.push_back(id - n_leaves);
    }

    np.steps.resize(n_steps);
    for (int s = 0; s < n_steps; s++) {
        NetworkStep &st = np.steps[s];
        st.a = steps[2 * s];
        st.b = steps[2 * s + 1];
        const auto &A = modes[st.a], &B = modes[st.b];
        for (int32_t m : A)
            if (find(B, m) < 0) st.modes.push_back(m);
        for (int32_t m : B)
            if (find(A, m) < 0) st.modes.push_back(m);
        for (int32_t m : st.modes) st.extents.push_back(extent_of[m]);
        modes[n_leaves + s] = st.modes;
        exts[n_leaves + s] = st.extents;
        st.desc = plan_contraction(elem_bytes, mode, 0, (int)A.size(), A.data(),
                                   exts[st.a].data(), (int)B.size(), B.data(),
                                   exts[st.b].data(), (int)st.modes.size(), st.modes.data());
        np.flops += st.desc.flops;
        np.workspace_bytes = std::max(np.workspace_bytes, st.desc.workspace);
    }
    choose_grouped(np, modes, exts);
    ArenaSim arena;
    std::vector<size_t> offset(n_nodes, 0);
    auto in_arena = [&](int s) { return !np.kept[s] && !np.steps[s].grouped; };
    for (int s = 0; s < n_steps; s++) {
        NetworkStep &st = np.steps[s];
        if (in_arena(s)) {
            offset[n_leaves + s] = arena.alloc(np.result_bytes(s));
            st.offset = offset[n_leaves + s];
        }
        for (int id : {st.a, st.b})
            if (id >= n_leaves && last_use[id] == s && in_arena(id - n_leaves))
                arena.release(offset[id]);
        // A result nothing uses is released at once (unless kept).
        if (last_use[n_leaves + s] < 0 && in_arena(s)) arena.release(st.offset);
    }
    // Kept results: one region after the working arena, in `keep` order.
    size_t top = align256(arena.high_water());
    // Results of the groups: a region of their own, reused in launch order.
    const std::vector<int> launch_of = plan_launches(np, true);
    std::vector<std::vector<int>> starts(np.launches.size()), ends(np.launches.size());
    auto in_groups = [&](int s) { return np.steps[s].grouped && !np.kept[s]; };
    std::vector<int> last_launch(launch_of);
    for (int s = 0; s < n_steps; s++)
        for (int id : {np.steps[s].a, np.steps[s].b})
            if (id >= n_leaves)
                last_launch[id - n_leaves] = std::max(last_launch[id - n_leaves], launch_of[s]);
    for (int s = 0; s < n_steps; s++)
        if (in_groups(s)) {
            starts[launch_of[s]].push_back(s);
            ends[last_launch[s]].push_back(s);
        }
    ArenaSim small;
    for (size_t l = 0; l < np.launches.size(); l++) {
        for (int s : starts[l])
            offset[n_leaves + s] = small.alloc(np.result_bytes(s));
        for (int s : ends[l]) small.release(offset[n_leaves + s]);
    }
    for (int s = 0; s < n_steps; s++)
        if (in_groups(s)) np.steps[s].offset = top + offset[n_leaves + s];
    top += align256(small.high_water());
    for (int s : keep_order) {
        np.steps[s].offset = top;
        top += align256(std::max<size_t>(256, (size_t)elem_bytes * (size_t)np.steps[s].desc.size_c));
    }
    np.arena_bytes = top;
    return np;
}

} // namespace jet_hip
