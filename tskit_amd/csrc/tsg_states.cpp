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
#include <thread>

#include "tsg_states.h"
#include "tsg_threads.h"
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
// states, groups of those again, up to one.  A child that comes, leaves or
// changes its state marks its slot, and the next sum visits the groups above
// the marked slots alone, log8(children) a slot (visiting all children made a
// plan cost trees x children: 41 s for 50000 trees of 20 nodes with 5000
// children each, 0.7 s so).
struct Wide {
    static constexpr int32_t SELF = -2;        // the node's own sample
    std::vector<int32_t> slots;                // child node, SELF or -1
    std::vector<int32_t> free, marked;
    std::vector<std::vector<int32_t>> value;   // states of the slots, of their groups, ...

    int32_t take(int32_t c) {
        int32_t at = (int32_t) slots.size();
        if (free.empty()) {
            slots.push_back(c);
        } else {
            at = free.back();
            free.pop_back();
            slots[at] = c;
        }
        marked.push_back(at);
        return at;
    }
    void leave(int32_t at) {
        slots[at] = -1;
        free.push_back(at);
        marked.push_back(at);
    }
};

// What the pass keeps of a node: what a walk up a root path reads and writes
// on one cache line, the rest on the next.
struct alignas(128) Node {
    Key key = 0;              // of the samples below
    double time = 0;
    double last = 0;          // last update (branch pieces)
    int32_t par = TSG_NULL, stamp = -1, below = 0, state = 0;
    int32_t in_state = 0;     // samples below it in the state it is in
    int32_t last_piece = -1, lc = -1, rs = -1;

    Key old_key = 0;
    double ins = 0;           // its parent edge's insertion
    double from = 0;          // where its state began
    int32_t old_par = TSG_NULL, ls = -1, kids = 0, sample = TSG_NULL;
    int32_t wide = -1;        // its Wide, while it has one
    int32_t slot = -1;        // its slot there, while its parent has one
};

// Calls work(begin, end) over 0 .. count - 1, on a few threads where there is
// enough of it.
template <typename F>
void over(int64_t count, F work) {
    const int64_t P = std::max<int64_t>(
        1, std::min<int64_t>({(int64_t) std::thread::hardware_concurrency(), 8, count / 65536}));
    tsg_parallel((int) P, [&](int p) { work(count * p / P, count * (p + 1) / P); });
}

struct Planner {
    std::vector<Node> node;
    // states in creation order: their level after merging, their direct inputs
    // (two in place, more at `more`), and the inputs after merging levels
    struct State {
        int32_t level = 0, count = 0, d0 = 0, d1 = 0;
    };
    std::vector<State> state;
    std::vector<int32_t> more;
    std::vector<int32_t> *in = nullptr;
    std::vector<Wide> wide;
    std::vector<int32_t> unused;  // of them

    // A new state summing list[0..m), m <= TSG_STATE_IN.  The deepest inputs
    // are replaced by their own inputs while the list has room: fewer levels
    // (one launch each) for more gathers a state.  On 2.8 M states of 20000
    // samples: 44 levels of 2 inputs, 16 of up to 4, 8 of up to 8.
    int32_t add(const int32_t *list, int m) {
        const int32_t id = (int32_t) state.size();
        State made;
        made.count = m;
        if (m == 2) {
            made.d0 = list[0];
            made.d1 = list[1];
        } else {
            made.d0 = (int32_t) more.size();
            more.insert(more.end(), list, list + m);
        }
        const State *const st = state.data();
        int32_t l[TSG_STATE_IN] = {}, lev[TSG_STATE_IN] = {};
        for (int i = 0; i < m; i++) {
            l[i] = list[i];
            lev[i] = st[list[i]].level;
        }
        int32_t most;
        for (;;) {
            int32_t top = 0;  // level and place of the deepest input
            for (int i = 0; i < TSG_STATE_IN; i++) top = std::max(top, lev[i] * TSG_STATE_IN + i);
            most = top / TSG_STATE_IN;
            if (most == 0) break;
            const int deep = top % TSG_STATE_IN;
            const State d = st[l[deep]];
            if (m - 1 + d.count > TSG_STATE_IN) break;
            if (d.count == 2) {
                l[deep] = d.d0;
                lev[deep] = st[d.d0].level;
                l[m] = d.d1;
                lev[m++] = st[d.d1].level;
                continue;
            }
            const int32_t *src = more.data() + d.d0;
            l[deep] = src[0];
            lev[deep] = st[src[0]].level;
            for (int i = 1; i < d.count; i++, m++) {
                l[m] = src[i];
                lev[m] = st[src[i]].level;
            }
        }
        made.level = most + 1;
        state.push_back(made);
        in->insert(in->end(), l, l + TSG_STATE_IN);
        return id;
    }

    int32_t sum(const int32_t *list, int m) {
        return m == 0 ? 0 : m == 1 ? list[0] : add(list, m);
    }

    // u's children into slots
    void widen(int32_t u) {
        if (unused.empty()) {
            unused.push_back((int32_t) wide.size());
            wide.emplace_back();
        }
        node[u].wide = unused.back();
        unused.pop_back();
        Wide &w = wide[node[u].wide];
        if (node[u].sample != TSG_NULL) (void) w.take(Wide::SELF);
        for (int32_t c = node[u].lc; c >= 0; c = node[c].rs) node[c].slot = w.take(c);
    }
    void narrow(int32_t u) {
        wide[node[u].wide] = Wide();
        unused.push_back(node[u].wide);
        node[u].wide = -1;
    }

    int32_t sum_wide(int32_t u) {
        Wide &w = wide[node[u].wide];
        auto padded = [](size_t m) { return (m + TSG_STATE_IN - 1) / TSG_STATE_IN * TSG_STATE_IN; };
        if (w.value.empty()) w.value.emplace_back();
        w.value[0].resize(padded(w.slots.size()), 0);
        std::vector<int32_t> groups, next;
        for (const int32_t i : w.marked) {
            const int32_t c = w.slots[i];
            const int32_t st = c >= 0 ? node[c].state : c == Wide::SELF ? 1 + node[u].sample : 0;
            if (w.value[0][i] == st) continue;
            w.value[0][i] = st;
            groups.push_back(i / TSG_STATE_IN);
        }
        w.marked.clear();
        for (size_t lev = 0;; lev++) {
            const size_t g = w.value[lev].size() / TSG_STATE_IN;
            if (lev + 1 == w.value.size()) {  // a new top: of all groups
                w.value.emplace_back();
                groups.resize(g);
                for (size_t i = 0; i < g; i++) groups[i] = (int32_t) i;
            }
            const std::vector<int32_t> &from = w.value[lev];
            std::vector<int32_t> &to = w.value[lev + 1];
            to.resize(g == 1 ? 1 : padded(g), 0);
            std::sort(groups.begin(), groups.end());
            groups.erase(std::unique(groups.begin(), groups.end()), groups.end());
            next.clear();
            for (const int32_t i : groups) {
                int32_t l[TSG_STATE_IN];
                int m = 0;
                for (int t = 0; t < TSG_STATE_IN; t++) {
                    const int32_t st = from[(size_t) i * TSG_STATE_IN + t];
                    if (st != 0) l[m++] = st;
                }
                const int32_t st = sum(l, m);
                if (to[i] == st) continue;
                to[i] = st;
                next.push_back(i / TSG_STATE_IN);
            }
            if (g == 1) return to[0];
            groups.swap(next);
        }
    }

    // the state of u's samples from its children's states
    int32_t sum_of(int32_t u) {
        if (node[u].kids + 1 > TSG_STATE_IN) {
            if (node[u].wide < 0) widen(u);
            return sum_wide(u);
        }
        if (node[u].wide >= 0) narrow(u);
        int32_t l[TSG_STATE_IN];
        int m = 0;
        if (node[u].sample != TSG_NULL) l[m++] = 1 + node[u].sample;
        for (int32_t c = node[u].lc; c >= 0; c = node[c].rs) {
            if (node[c].state != 0) l[m++] = node[c].state;
        }
        return sum(l, m);
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
    // States from which they are numbered by level, so that a level's inputs
    // and rows are contiguous; below, the plan is a few MB and stays as made,
    // with a list of each level's states (half the memory written here).
    constexpr int64_t RENUMBER = 1 << 18;
    const int64_t most = 16 * ((int64_t) E + n) + 1024;
    Planner P;
    P.state.assign(1 + (size_t) n, Planner::State());
    P.node.assign(N, Node());
    Node *const node = P.node.data();
    for (int32_t u = 0; u < N; u++) {
        node[u].time = ts->time[u];
        const int32_t s = node[u].sample = ts->sample_index_map[u];
        if (s == TSG_NULL) continue;
        node[u].state = 1 + s;
        node[u].below = node[u].in_state = 1;
        node[u].key = ((Key) mix64(2 * (uint64_t) s + 1) << 64) | mix64(2 * (uint64_t) s + 2);
    }
    // (about 3 states and 6 events an edge on coalescent trees)
    P.in = &sp.in;
    P.state.reserve((size_t) n + 3 * (size_t) E);
    sp.in.reserve((size_t) E * 3 * TSG_STATE_IN);
    sp.ev_state.reserve((size_t) E * 6);
    sp.ev_b.reserve((size_t) E * 6);
    sp.ev_pos.reserve((size_t) E * 6);
    sp.node_pieces.reserve((size_t) E * 4);
    sp.pieces.reserve((size_t) E * 4);
    auto event = [&](double b, double x, int32_t state) {
        sp.ev_state.push_back(state);
        sp.ev_b.push_back(b);
        sp.ev_pos.push_back(x);
    };
    std::vector<int32_t> touched;
    // the branch piece of u that ends here (see tsg_states.h)
    auto update = [&](Node &v, double x) {
        const double from = v.last;
        if (!(from < x)) return;
        v.last = x;
        if (v.par == TSG_NULL || v.in_state <= 0 || v.in_state >= n) return;
        const double tp = node[v.par].time;
        if (v.last_piece >= 0) {
            TsgBranchPiece &l = sp.pieces[v.last_piece];
            if (l.to == from && l.state == v.state && l.tp == tp && l.ins == v.ins) {
                l.to = x;
                return;
            }
        }
        v.last_piece = (int32_t) sp.pieces.size();
        sp.pieces.push_back({v.time, tp, v.ins, from, x, v.state, 0});
    };
    sp.list_off.assign(1, 0);
    sp.mut_state.resize(ts->mut_node.size());
    int32_t j = 0, k = 0;
    for (int32_t t = 0; t < T; t++) {
        const double x = ts->breakpoints[t];
        touched.clear();
        auto touch = [&](Node &v, int32_t u) {
            if (v.stamp == t) return;
            v.stamp = t;
            v.old_key = v.key;
            v.old_par = v.par;
            touched.push_back(u);
        };
        auto walk = [&](int32_t p, Key d, int32_t b) {  // up the root path
            for (int32_t u = p; u != TSG_NULL; u = node[u].par) {
                Node &v = node[u];
                touch(v, u);
                update(v, x);
                v.key += d;
                v.below += b;
            }
        };
        while (k < E && ts->right[O[k]] == x) {
            const int32_t p = ts->parent[O[k]], c = ts->child[O[k]];
            k++;
            Node &v = node[c];
            touch(v, c);
            update(v, x);
            walk(p, -v.key, -v.below);
            if (v.ls >= 0) node[v.ls].rs = v.rs;
            else node[p].lc = v.rs;
            if (v.rs >= 0) node[v.rs].ls = v.ls;
            v.ls = v.rs = -1;
            v.par = TSG_NULL;
            node[p].kids--;
            if (node[p].wide >= 0) P.wide[node[p].wide].leave(v.slot);
        }
        while (j < E && ts->left[I[j]] == x) {
            const int32_t p = ts->parent[I[j]], c = ts->child[I[j]];
            j++;
            Node &v = node[c];
            touch(v, c);
            walk(p, v.key, v.below);
            v.rs = node[p].lc;
            if (v.rs >= 0) node[v.rs].ls = c;
            node[p].lc = c;
            v.par = p;
            v.ins = x;
            node[p].kids++;
            if (node[p].wide >= 0) v.slot = P.wide[node[p].wide].take(c);
        }
        // children before parents: a child is younger than its parent (a few
        // nodes, mostly in runs: by insertion; the first tree's by sorting)
        auto younger = [&](int32_t a, int32_t b) {
            return node[a].time != node[b].time ? node[a].time < node[b].time : a < b;
        };
        if (touched.size() > 64) {
            std::sort(touched.begin(), touched.end(), younger);
        } else {
            for (size_t i = 1; i < touched.size(); i++) {
                const int32_t u = touched[i];
                size_t h = i;
                for (; h > 0 && younger(u, touched[h - 1]); h--) touched[h] = touched[h - 1];
                touched[h] = u;
            }
        }
        for (int32_t u : touched) {
            Node &v = node[u];
            const double was = v.old_par != TSG_NULL ? node[v.old_par].time - v.time : 0.0;
            const double now = v.par != TSG_NULL ? node[v.par].time - v.time : 0.0;
            if (v.key == v.old_key) {
                if (now != was) event(now - was, x, v.state);
                continue;
            }
            if (was != 0.0) event(-was, x, v.state);
            const int32_t before = v.state;
            v.state = P.sum_of(u);
            v.in_state = v.below;
            if (v.state != before) {
                if (v.from < x) sp.node_pieces.push_back({u, before, v.from});
                v.from = x;
                if (v.par != TSG_NULL && node[v.par].wide >= 0) {
                    P.wide[node[v.par].wide].marked.push_back(v.slot);
                }
            }
            if (now != 0.0) event(now, x, v.state);
        }
        if ((int64_t) P.state.size() > most) {
            sp = tsg_stateplan();
            return 0;
        }
        // the rows of this tree's sites, from the states of their mutations'
        // nodes
        for (int32_t s = ts->tree_site0[t]; s < ts->tree_site0[t + 1]; s++) {
            const int32_t m0 = ts->site_mut0[s], m1 = ts->site_mut0[s + 1];
            for (int32_t m = m0; m < m1; m++) sp.mut_state[m] = node[ts->mut_node[m]].state;
            if (m1 == m0 + 1 && ts->mut_allele[m0] == 1 && ts->mut_pallele[m0] == 0) {
                const Node &v = node[ts->mut_node[m0]];
                sp.row_ref.push_back(v.state);
                sp.row_pos.push_back(ts->site_pos[s]);
                sp.row_all.push_back(v.in_state);
                continue;
            }
            for (int32_t al = 0; al < ts->site_nalleles[s]; al++) {
                sp.row_ref.push_back(-1 - sp.num_lists++);
                sp.row_pos.push_back(ts->site_pos[s]);
                sp.list_kind.push_back(al == 0 ? TSG_ROW_ANCESTRAL : TSG_ROW_DERIVED);
                int32_t all = al == 0 ? n : 0;
                for (int32_t m = m0; m < m1; m++) {
                    const Node &v = node[ts->mut_node[m]];
                    if (ts->mut_allele[m] == al) {
                        sp.list_ent.push_back(2 * v.state);
                        all += v.in_state;
                    }
                    if (ts->mut_pallele[m] == al) {
                        sp.list_ent.push_back(2 * v.state + 1);
                        all -= v.in_state;
                    }
                }
                sp.row_all.push_back(all);
                sp.list_off.push_back((int32_t) sp.list_ent.size());
            }
        }
    }
    for (int32_t u = 0; u < N; u++) {
        update(node[u], ts->L);
        sp.node_pieces.push_back({u, node[u].state, node[u].from});
    }
    const int64_t S = (int64_t) P.state.size();
    int32_t levels = 0;
    for (const Planner::State &st : P.state) levels = std::max(levels, st.level + 1);
    const size_t limit = (size_t) INT32_MAX / 2 - 1;
    if ((size_t) S > limit || sp.ev_state.size() > limit || sp.row_ref.size() > limit ||
        sp.list_ent.size() > limit || sp.node_pieces.size() > limit ||
        sp.pieces.size() > limit || levels > MOST_LEVELS) {
        sp = tsg_stateplan();
        return 0;
    }
    // the states by level, within a level as created
    sp.level0.assign(levels + 1, 0);
    for (const Planner::State &st : P.state) sp.level0[st.level + 1]++;
    for (int32_t l = 0; l < levels; l++) sp.level0[l + 1] += sp.level0[l];
    std::vector<int32_t> next(sp.level0.begin(), sp.level0.end() - 1);
    std::vector<int32_t> at(S);
    for (int64_t s = 0; s < S; s++) at[s] = next[P.state[s].level]++;
    if (S < RENUMBER) {
        sp.order.resize(S);
        for (int64_t s = 0; s < S; s++) sp.order[at[s]] = (int32_t) s;
    } else {
        const int32_t f = 1 + n;
        std::vector<int32_t> in(sp.in.size());
        over(S - f, [&](int64_t b, int64_t e) {
            for (int64_t s = b; s < e; s++) {
                const int32_t *src = sp.in.data() + s * TSG_STATE_IN;
                int32_t *dst = in.data() + (int64_t) (at[s + f] - f) * TSG_STATE_IN;
                for (int i = 0; i < TSG_STATE_IN; i++) dst[i] = at[src[i]];
            }
        });
        sp.in.swap(in);
        auto renumber = [&](auto &v, auto state) {
            over((int64_t) v.size(), [&](int64_t b, int64_t e) {
                for (int64_t i = b; i < e; i++) state(v[i]) = at[state(v[i])];
            });
        };
        auto whole = [](int32_t &s) -> int32_t & { return s; };
        auto member = [](auto &p) -> int32_t & { return p.state; };
        renumber(sp.ev_state, whole);
        renumber(sp.mut_state, whole);
        renumber(sp.pieces, member);
        renumber(sp.node_pieces, member);
        for (int32_t &r : sp.row_ref) r = r >= 0 ? at[r] : r;
        for (int32_t &e : sp.list_ent) e = 2 * at[e >> 1] + (e & 1);
    }
    sp.num_states = (int32_t) S;
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

void tsg_node_runs(const tsg_treeseq *ts, TsgNodeRuns &r) {
    const std::vector<TsgNodePiece> &pieces = ts->states.node_pieces;
    const int32_t N = ts->num_nodes;
    std::vector<int32_t> at(N + 1, 0);
    for (const TsgNodePiece &q : pieces) at[q.node + 1]++;
    for (int32_t u = 0; u < N; u++) at[u + 1] += at[u];
    r.state.resize(pieces.size());
    r.from.resize(pieces.size());
    for (int32_t u = 0; u < N; u++) {
        for (int32_t p = at[u]; p < at[u + 1]; p += TSG_NODE_RUN) {
            r.node.push_back(u);
            r.piece0.push_back(p);
        }
    }
    r.piece0.push_back((int32_t) pieces.size());
    for (const TsgNodePiece &q : pieces) {
        const int32_t to = at[q.node]++;
        r.state[to] = q.state;
        r.from[to] = q.from;
    }
}
