// group_check.cpp -- CPU checks of the launches of network and DAG plans: every
// step runs once, after the launches of its operands, and no two results that
// are alive at the same time share memory in launch order.
#include "../../jet_amd/csrc/network_plan.hpp"

#include <algorithm>
#include <cstring>
#include <vector>

using namespace jet_hip;

static int check(const NetworkPlan &np, int elem_bytes, int *n_launches, int *n_grouped)
{
    const int ns = (int)np.steps.size();
    std::vector<int> at(ns, -1);
    *n_grouped = 0;
    for (int l = 0; l < (int)np.launches.size(); l++) {
        const NetworkLaunch &x = np.launches[l];
        if (x.step >= 0) {
            if (at[x.step] >= 0 || np.steps[x.step].grouped) return 1;
            at[x.step] = l;
            continue;
        }
        for (int b = x.first_block; b < x.first_block + x.n_blocks; b++) {
            const GroupBlock &g = np.blocks[b];
            int s = -1;
            for (int i = 0; i < ns; i++)
                if (np.slot(np.n_leaves + i) == g.c || (np.steps[i].is_root && g.c == np.n_leaves))
                    s = i;
            if (s < 0 || !np.steps[s].grouped) return 2;
            const NetworkStep &st = np.steps[s];
            if (g.a != np.slot(st.a) || g.b != np.slot(st.b)) return 3;
            if (g.wide != (np.wide(st.a) | np.wide(st.b) << 1 | st.wide << 2)) return 10;
            if (at[s] >= 0 && at[s] != l) return 4;
            const int64_t lo = st.small.lb + st.small.lm + st.small.ln;
            if (int64_t(1) << lo != st.desc.size_c || g.first >= 1 << lo || g.lanes > 6) return 5;
            *n_grouped += at[s] < 0;
            at[s] = l;
        }
    }
    for (int s = 0; s < ns; s++) {
        if (at[s] < 0) return 6;
        for (int x : {np.steps[s].a, np.steps[s].b})
            if (x >= np.n_leaves && at[x - np.n_leaves] >= at[s]) return 7;
    }
    // FP64 results: read by groups alone, neither kept nor the root
    for (int s = 0; s < ns; s++) {
        const NetworkStep &st = np.steps[s];
        if (st.wide && (elem_bytes != 8 || !st.grouped || st.is_root || (np.dag && np.kept[s])))
            return 11;
        if (!st.grouped && (np.wide(st.a) || np.wide(st.b))) return 12;
    }
    // life in launches; kept results to the end
    std::vector<int> end(at);
    for (int s = 0; s < ns; s++)
        for (int x : {np.steps[s].a, np.steps[s].b})
            if (x >= np.n_leaves) end[x - np.n_leaves] = std::max(end[x - np.n_leaves], at[s]);
    for (int s = 0; s < ns; s++) {
        if (np.dag && np.kept[s]) end[s] = (int)np.launches.size();
        if (np.steps[s].is_root) continue;
        const size_t len = np.result_bytes(s);
        if (np.steps[s].offset + len > np.arena_bytes) return 8;
        for (int t = 0; t < s; t++) {
            if (np.steps[t].is_root || end[t] < at[s] || end[s] < at[t]) continue;
            const size_t lt = np.result_bytes(t);
            if (np.steps[s].offset < np.steps[t].offset + lt &&
                np.steps[t].offset < np.steps[s].offset + len)
                return 9;
        }
    }
    *n_launches = (int)np.launches.size();
    return 0;
}

extern "C" int check_launches(int dag, int n_leaves, const int32_t *ranks, const int32_t *modes,
                              const int64_t *exts, int n_steps, const int32_t *path, int n_out,
                              const int32_t *out, int *n_launches, int *n_grouped)
{
    return check(dag ? plan_dag(8, 0, n_leaves, ranks, modes, exts, n_steps, path, n_out, out)
                     : plan_network(8, 0, n_leaves, ranks, modes, exts, n_steps, path, n_out, out),
                 8, n_launches, n_grouped);
}
