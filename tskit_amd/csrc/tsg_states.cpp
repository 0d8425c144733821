// Host planner of the state plan (tsg_states.h): one pass along the genome.
//
// At each transition the edges out and in are applied in index order, and
// the nodes they touch (children, and the nodes on root paths) are compared
// before and after: a node whose samples below are the same keeps its state,
// whatever moved between the two, so above the point where a moved subtree's
// old and new root paths meet nothing is recorded.  (On coalescent trees
// about 14 states a transition against 43 path entries of the edge events.)
// "The same samples" is decided by a 128-bit sum of pseudo-random sample
// keys: two different sets agree with probability 2^-128.
#include <algorithm>
#include <cstring>
#include <unordered_map>

#include "tsg_states.h"
#include "tsg_treeseq.h"

namespace {

using Key = unsigned __int128;

uint64_t mix64(uint64_t x) {  // splitmix64 (Steele, Lea, Flood 2014)
    x += 0x9e3779b97f4a7c15ull;
    x = (x ^ (x >> 30)) * 0xbf58476d1ce4e5b9ull;
    x = (x ^ (x >> 27)) * 0x94d049bb133111ebull;
    return x ^ (x >> 31);
}

// The children of a node with more than TSG_STATE_IN of them, in slots that
// keep their places: groups of TSG_STATE_IN slots are summed by helper
// states, groups of those again, and a group none of whose members changed
// keeps its helper state.
struct Wide {
    std::vector<int32_t> slots;                         // child node or -1
    std::vector<std::vector<int32_t>> members, helper;  // per level
};

struct Planner {
    const tsg_treeseq *ts;
    // states in creation order: their direct inputs, and the inputs after
    // merging levels, with their level
    std::vector<int64_t> dir0;
    std::vector<int32_t> dir, level, in;
    std::unordered_map<int32_t, Wide> wide;
    std::vector<int32_t> slot_of;
    int64_t limit = 0;

    int32_t n() const { return ts->num_samples; }
    int32_t first() const { return 1 + ts->num_samples; }
    int32_t count() const { return (int32_t) level.size(); }

    const int32_t *inputs(int32_t s, int &m) const {
        m = (int) (dir0[s + 1] - dir0[s]);
        return dir.data() + dir0[s];
    }

    // A new state summing list[0..m), m <= TSG_STATE_IN.  The deepest inputs
    // are replaced by their own inputs while the list has room: fewer levels
    // (one launch each) for more gathers a state.  Measured on 2.8 M states
    // of 20000 samples: 44 levels of 2 inputs, 16 of up to 4, 8 of up to 8.
    int32_t add(const int32_t *list, int m) {
        const int32_t id = count();
        for (int i = 0; i < m; i++) dir.push_back(list[i]);
        dir0.push_back((int64_t) dir.size());
        int32_t l[TSG_STATE_IN];
        std::copy(list, list + m, l);
        for (;;) {
            int deep = -1;
            for (int i = 0; i < m; i++) {
                if (level[l[i]] > 0 && (deep < 0 || level[l[i]] > level[l[deep]])) deep = i;
            }
            if (deep < 0) break;
            int k;
            const int32_t *src = inputs(l[deep], k);
            if (m - 1 + k > TSG_STATE_IN) break;
            l[deep] = src[0];
            for (int i = 1; i < k; i++) l[m++] = src[i];
        }
        int32_t lev = 0;
        for (int i = 0; i < m; i++) lev = std::max(lev, level[l[i]]);
        level.push_back(lev + 1);
        for (int i = 0; i < TSG_STATE_IN; i++) in.push_back(i < m ? l[i] : 0);
        return id;
    }

    // the state summing the inputs given: an existing one where there is at
    // most one, helper states over groups where there are many
    int32_t sum(const int32_t *list, int m) {
        if (m == 0) return 0;
        if (m == 1) return list[0];
        return add(list, m);
    }

    int32_t sum_wide(int32_t u, const std::vector<int32_t> &par, const std::vector<int32_t> &lc,
                     const std::vector<int32_t> &rs, const std::vector<int32_t> &state) {
        Wide &w = wide[u];
        for (int32_t &c : w.slots) {
            if (c >= 0 && par[c] != u) c = -1;
        }
        size_t hole = 0;
        for (int32_t c = lc[u]; c >= 0; c = rs[c]) {
            if (slot_of[c] >= 0 && (size_t) slot_of[c] < w.slots.size() &&
                w.slots[slot_of[c]] == c) {
                continue;
            }
            while (hole < w.slots.size() && w.slots[hole] >= 0) hole++;
            if (hole == w.slots.size()) w.slots.push_back(-1);
            w.slots[hole] = c;
            slot_of[c] = (int32_t) hole;
        }
        std::vector<int32_t> cur(w.slots.size());
        for (size_t i = 0; i < cur.size(); i++) cur[i] = w.slots[i] >= 0 ? state[w.slots[i]] : 0;
        const int32_t own = ts->sample_index_map[u];
        if (own != TSG_NULL) cur.insert(cur.begin(), 1 + own);
        for (size_t lev = 0; cur.size() > 1; lev++) {
            if (w.members.size() <= lev) {
                w.members.emplace_back();
                w.helper.emplace_back();
            }
            std::vector<int32_t> &was = w.members[lev], &helper = w.helper[lev];
            const size_t g = (cur.size() + TSG_STATE_IN - 1) / TSG_STATE_IN;
            was.resize(g * TSG_STATE_IN, -1);
            helper.resize(g, -1);
            cur.resize(g * TSG_STATE_IN, 0);
            std::vector<int32_t> next(g);
            for (size_t i = 0; i < g; i++) {
                const int32_t *p = cur.data() + i * TSG_STATE_IN;
                int32_t *q = was.data() + i * TSG_STATE_IN;
                if (helper[i] < 0 || !std::equal(p, p + TSG_STATE_IN, q)) {
                    std::copy(p, p + TSG_STATE_IN, q);
                    int32_t l[TSG_STATE_IN];
                    int m = 0;
                    for (int t = 0; t < TSG_STATE_IN; t++) {
                        if (p[t] != 0) l[m++] = p[t];
                    }
                    helper[i] = sum(l, m);
                }
                next[i] = helper[i];
            }
            cur.swap(next);
        }
        return cur.empty() ? 0 : cur[0];
    }
};

}  // namespace

// Not usable (the statistics then run on the chunk plans) where the states
// outnumber what the tree sequence's size explains -- trees whose nodes
// change their samples far above every moved subtree -- or where there are
// so many merged levels that their launches would cost more than the chunk
// sweep (trees like caterpillars: 8 levels on 20000 coalescent samples).
int tsg_build_states(tsg_treeseq *ts) {
    tsg_stateplan &sp = ts->states;
    sp = tsg_stateplan();
    const int32_t N = ts->num_nodes, E = ts->num_edges, T = ts->num_trees, n = ts->num_samples;
    const int32_t *I = ts->I.data(), *O = ts->O.data();
    constexpr int32_t MOST_LEVELS = 64;
    Planner P;
    P.ts = ts;
    P.limit = 16 * ((int64_t) E + n) + 1024;
    P.level.assign(1 + (size_t) n, 0);
    P.dir0.assign(2 + (size_t) n, 0);
    P.slot_of.assign(N, -1);
    std::vector<int32_t> par(N, TSG_NULL), lc(N, -1), ls(N, -1), rs(N, -1), nch(N, 0);
    std::vector<int32_t> state(N, 0), stamp(N, -1), old_par(N, TSG_NULL), touched;
    std::vector<Key> key(N, 0), old_key(N, 0);
    for (int32_t u = 0; u < N; u++) {
        const int32_t s = ts->sample_index_map[u];
        if (s == TSG_NULL) continue;
        state[u] = 1 + s;
        key[u] = ((Key) mix64(2 * (uint64_t) s + 1) << 64) | mix64(2 * (uint64_t) s + 2);
    }
    std::vector<int32_t> ev_state, row_ref, list_ent;
    auto branch = [&](int32_t u, int32_t p) { return ts->time[p] - ts->time[u]; };
    sp.list_off.assign(1, 0);
    int32_t j = 0, k = 0;
    std::vector<int32_t> kids;
    for (int32_t t = 0; t < T; t++) {
        const double x = ts->breakpoints[t];
        touched.clear();
        auto touch = [&](int32_t u) {
            if (stamp[u] == t) return;
            stamp[u] = t;
            old_key[u] = key[u];
            old_par[u] = par[u];
            touched.push_back(u);
        };
        while (k < E && ts->right[O[k]] == x) {
            const int32_t p = ts->parent[O[k]], c = ts->child[O[k]];
            k++;
            touch(c);
            for (int32_t u = p; u != TSG_NULL; u = par[u]) {
                touch(u);
                key[u] -= key[c];
            }
            if (ls[c] >= 0) rs[ls[c]] = rs[c];
            else lc[p] = rs[c];
            if (rs[c] >= 0) ls[rs[c]] = ls[c];
            ls[c] = rs[c] = -1;
            par[c] = TSG_NULL;
            nch[p]--;
        }
        while (j < E && ts->left[I[j]] == x) {
            const int32_t p = ts->parent[I[j]], c = ts->child[I[j]];
            j++;
            touch(c);
            for (int32_t u = p; u != TSG_NULL; u = par[u]) {
                touch(u);
                key[u] += key[c];
            }
            rs[c] = lc[p];
            if (lc[p] >= 0) ls[lc[p]] = c;
            lc[p] = c;
            par[c] = p;
            nch[p]++;
        }
        // children before parents: a child is younger than its parent
        std::sort(touched.begin(), touched.end(), [&](int32_t a, int32_t b) {
            return ts->time[a] != ts->time[b] ? ts->time[a] < ts->time[b] : a < b;
        });
        for (int32_t u : touched) {
            const bool moved = key[u] != old_key[u];
            const double was = old_par[u] != TSG_NULL ? branch(u, old_par[u]) : 0.0;
            const double now = par[u] != TSG_NULL ? branch(u, par[u]) : 0.0;
            if (!moved) {
                if (now != was) {
                    ev_state.push_back(state[u]);
                    sp.ev_b.push_back(now - was);
                    sp.ev_pos.push_back(x);
                }
                continue;
            }
            if (was != 0.0) {
                ev_state.push_back(state[u]);
                sp.ev_b.push_back(-was);
                sp.ev_pos.push_back(x);
            }
            if (nch[u] + 1 > TSG_STATE_IN) {
                state[u] = P.sum_wide(u, par, lc, rs, state);
            } else {
                int32_t l[TSG_STATE_IN];
                int m = 0;
                if (ts->sample_index_map[u] != TSG_NULL) l[m++] = 1 + ts->sample_index_map[u];
                for (int32_t c = lc[u]; c >= 0; c = rs[c]) {
                    if (state[c] != 0) l[m++] = state[c];
                }
                state[u] = P.sum(l, m);
            }
            if (now != 0.0) {
                ev_state.push_back(state[u]);
                sp.ev_b.push_back(now);
                sp.ev_pos.push_back(x);
            }
        }
        if ((int64_t) P.level.size() > P.limit) return 0;
        // the rows of this tree's sites, from the states of their mutations'
        // nodes
        for (int32_t s = ts->tree_site0[t]; s < ts->tree_site0[t + 1]; s++) {
            const int32_t m0 = ts->site_mut0[s], m1 = ts->site_mut0[s + 1];
            if (m1 == m0 + 1 && ts->mut_allele[m0] == 1 && ts->mut_pallele[m0] == 0) {
                row_ref.push_back(state[ts->mut_node[m0]]);
                sp.row_pos.push_back(ts->site_pos[s]);
                continue;
            }
            for (int32_t al = 0; al < ts->site_nalleles[s]; al++) {
                row_ref.push_back(-1 - sp.num_lists++);
                sp.row_pos.push_back(ts->site_pos[s]);
                sp.list_kind.push_back(al == 0 ? TSG_ROW_ANCESTRAL : TSG_ROW_DERIVED);
                for (int32_t m = m0; m < m1; m++) {
                    const int32_t st = state[ts->mut_node[m]];
                    if (ts->mut_allele[m] == al) list_ent.push_back(2 * st);
                    if (ts->mut_pallele[m] == al) list_ent.push_back(2 * st + 1);
                }
                sp.list_off.push_back((int32_t) list_ent.size());
            }
        }
    }
    // number the states by level, within a level as created
    const int32_t S = P.count();
    if (S > INT32_MAX / 2 - 1 || ev_state.size() > (size_t) INT32_MAX ||
        row_ref.size() > (size_t) INT32_MAX || list_ent.size() > (size_t) INT32_MAX) {
        return 0;
    }
    int32_t levels = 0;
    for (int32_t l : P.level) levels = std::max(levels, l + 1);
    if (levels > MOST_LEVELS) return 0;
    sp.level0.assign(levels + 1, 0);
    for (int32_t l : P.level) sp.level0[l + 1]++;
    for (int32_t l = 0; l < levels; l++) sp.level0[l + 1] += sp.level0[l];
    std::vector<int32_t> id(S), next(sp.level0.begin(), sp.level0.end() - 1);
    for (int32_t s = 0; s < S; s++) id[s] = next[P.level[s]]++;
    const int32_t f = P.first();
    sp.in.resize((size_t) (S - f) * TSG_STATE_IN);
    for (int32_t s = f; s < S; s++) {
        const int32_t *src = P.in.data() + (size_t) (s - f) * TSG_STATE_IN;
        int32_t *dst = sp.in.data() + (size_t) (id[s] - f) * TSG_STATE_IN;
        for (int i = 0; i < TSG_STATE_IN; i++) dst[i] = id[src[i]];
    }
    for (int32_t &s : ev_state) s = id[s];
    for (int32_t &r : row_ref) r = r >= 0 ? id[r] : r;
    for (int32_t &e : list_ent) e = 2 * id[e >> 1] + (e & 1);
    sp.ev_state.swap(ev_state);
    sp.row_ref.swap(row_ref);
    sp.list_ent.swap(list_ent);
    sp.num_states = S;
    auto tiles = [](const std::vector<double> &pos, int tile, int32_t &count,
                    std::vector<double> &first) {
        count = (int32_t) std::max<size_t>(1, (pos.size() + tile - 1) / tile);
        first.assign(count, 0.0);
        for (int32_t t = 0; t < count; t++) {
            if ((size_t) t * tile < pos.size()) first[t] = pos[(size_t) t * tile];
        }
    };
    tiles(sp.ev_pos, TSG_BRANCH_TILE, sp.btiles, sp.btile_pos);
    tiles(sp.row_pos, TSG_SITE_TILE, sp.stiles, sp.stile_pos);
    sp.usable = true;
    return 0;
}
