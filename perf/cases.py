"""The work that programs using this framework have it do, as timed cases.

A case is one pass through a public entry point on resident tree sequences:
windowed statistics in branch and site mode (single calls, a fused step, wide
requests, many replicates at once), the joint allele frequency spectrum, node
statistics, trait regression, and the sample x sample and genotype matrices.
Tree sequences come from the package's own coalescent generator (Ne = 1e4,
r = 1e-8), sample sets and trait weights from a seeded generator.

``exact`` recomputes the floating outputs in 64 bits with plain torch.
"""
import functools
import math

import numpy as np
import torch

import tskit_amd as ta

NE, RHO = 1e4, 1e-8


def listed():
    """The cases, smallest first."""
    return [
        # the smallest call: one statistic of a whole small sample, where
        # only latency counts (a notebook, a test, a simulation's inner loop)
        dict(name="tiny_diversity_site", op="stat", stat="diversity", mode="site", n=100, L=1e5,
             mu=1e-8, K=1, size=100, W=1),
        # two populations, ten windows: the first thing a user asks for
        dict(name="small_fst_branch", op="stat", stat="Fst", mode="branch", n=1000, L=1e6, mu=1e-8,
             K=2, size=500, W=10),
        # an f4 test over ragged sets and windows, from the genotypes
        dict(name="ragged_f4_site", op="stat", stat="f4", mode="site", n=4999, L=3.7e6, mu=1e-8,
             K=5, size=331, W=97),
        # centred relatedness between populations (polarised by default)
        dict(name="relatedness_branch", op="stat", stat="genetic_relatedness", mode="branch",
             n=2000, L=4e6, mu=1e-8, K=10, size=150, W=40),
        # a served request with many sets and windows
        dict(name="wide_divergence_branch", op="stat", stat="divergence", mode="branch", n=15000,
             L=2e6, mu=1e-8, K=64, size=200, W=2000),
        # genome scan by regression on two traits with two covariates
        dict(name="trait_regression_branch", op="weighted", mode="branch", n=2000, L=3e6, mu=1e-8,
             K=2, covariates=2, W=60),
        # joint spectrum of two populations, both modes
        dict(name="joint_spectrum", op="spectrum", n=5000, L=3e6, mu=2.75e-8, K=2, size=150, W=20),
        # one value per node and set of a resident tree sequence
        dict(name="node_diversity", op="stat", stat="diversity", mode="node", n=8000, L=4e6,
             mu=1e-8, K=8, size=500, W=1, resident=True),
        # relatedness of every two samples from the genotypes
        dict(name="relatedness_matrix_site", op="relatedness_matrix", n=2500, L=6e6, mu=2.75e-8,
             W=1),
        # genotypes of every sample at every site kept
        dict(name="genotype_matrix", op="genotypes", n=1500, L=5e6, mu=2e-8, sites=24000),
        # simulation replicates, every sweep in one launch
        dict(name="replicates", op="replicates", n=2000, L=1.5e6, mu=1e-8, K=16, size=400, W=500,
             count=40),
        # the large step: Fst over all pairs, Tajima's D and f4, both modes,
        # fused, on a resident tree sequence of many samples
        dict(name="large_step", op="step", n=20000, L=5e7, mu=1e-8, K=8, size=1000, W=1000,
             resident=True),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    """One more case of the same ranges."""
    op = rng.choice(["stat"] * 5 + ["step"] * 2 + ["weighted", "spectrum", "relatedness_matrix",
                                                   "genotypes", "replicates"])
    n = int(_log(rng, 100, 20000))
    L = float(int(_log(rng, 1e5, 6e6 if n <= 5000 else 2e6)))
    W = int(_log(rng, 1, 2000))
    K = int(_log(rng, 1, 64))
    c = dict(op=op, n=n, L=L, mu=1e-8)
    if op == "stat":
        stat = rng.choice(["diversity", "segregating_sites", "Tajimas_D", "divergence", "Fst", "f2",
                           "f3", "f4", "Y2", "genetic_relatedness"])
        mode = rng.choice(["branch", "branch", "site", "site", "node"])
        if stat == "Tajimas_D" and mode == "node":
            mode = "site"
        if mode == "node":
            K, W, c["resident"] = min(K, 8), 1, True
        K = max(K, {"f4": 4, "f3": 3, "divergence": 2, "Fst": 2, "f2": 2, "Y2": 2,
                    "genetic_relatedness": 2}.get(stat, 1))
        K = min(K, 12) if stat == "genetic_relatedness" else K
        return dict(c, stat=stat, mode=mode, K=K, size=_size(rng, n, K), W=W)
    if op == "step":
        K = min(max(K, 4), 12)
        return dict(c, K=K, size=_size(rng, n, K), W=W)
    if op == "weighted":
        n = min(n, 5000)
        return dict(c, n=n, mode=rng.choice(["branch", "site"]), K=min(K, 4),
                    covariates=rng.randint(1, 3), W=min(W, 300))
    if op == "spectrum":
        return dict(c, n=min(n, 8000), mu=2e-8, K=2, size=rng.randint(5, 45), W=min(W, 100))
    if op == "relatedness_matrix":
        return dict(c, n=min(n, 2500), mu=2e-8, W=min(W, 4))
    if op == "genotypes":
        n = min(n, 1500)
        return dict(c, n=n, mu=2e-8, sites=max(20, int(0.5 * _tables_size(n, L, 2e-8)[2])))
    return dict(c, n=int(_log(rng, 200, 2000)), L=1.5e6, K=min(K, 16), size=rng.randint(10, 400),
                W=min(W, 500), count=rng.randint(3, 30))


def _size(rng, n, K):
    return max(2, min(int(_log(rng, 10, 2000)), n // K))


# --- inputs ---------------------------------------------------------------

@functools.lru_cache(maxsize=2)
def _resident(n, L, mu):
    """The data set that a program loads once and queries for its whole life."""
    tables = ta.simulate_tables(n, L, NE, RHO, mu, 2)
    return tables, tables.tree_sequence()


def _tree_sequence(case, seed):
    n, L, mu = case["n"], case["L"], case["mu"]
    if case.get("resident"):
        return _resident(n, L, mu)
    tables = ta.simulate_tables(n, L, NE, RHO, mu, 1 + seed % (1 << 30))
    if "sites" in case:
        _keep_sites(tables, case["sites"])
    return tables, tables.tree_sequence()


def _keep_sites(tables, count):
    """The tables with their first ``count`` sites (one mutation each)."""
    for name in ("site_position", "ancestral_state", "mutation_site", "mutation_node",
                 "mutation_parent", "derived_state"):
        setattr(tables, name, getattr(tables, name)[:count])
    for name in ("ancestral_state_offset", "derived_state_offset"):
        setattr(tables, name, getattr(tables, name)[:count + 1])


def _sets(rng, n, K, size):
    """K disjoint sets of at most ``size`` samples, of slightly differing sizes."""
    size = max(2, min(size, n // K))
    perm = rng.permutation(n)
    return [np.sort(perm[k * size:(k + 1) * size - (k % 3 if size > 8 else 0)]).astype(np.int32)
            for k in range(K)]


def _indexes(stat, K):
    if stat in ("Fst", "f2", "Y2", "divergence", "genetic_relatedness"):
        if K <= 12:
            return [(i, j) for i in range(K) for j in range(i + 1, K)]
        return [(i, (i + 1) % K) for i in range(K)]
    if stat == "f3":
        return [(i, (i + 1) % K, (i + 2) % K) for i in range(K)]
    if stat == "f4":
        return [(i, (i + 1) % K, (i + 2) % K, (i + 3) % K) for i in range(K)]
    return None


def _inputs(case, seed):
    """Everything of a pass but the resident tree sequence."""
    op = case["op"]
    rng = np.random.default_rng([seed, 77])
    W = case.get("W", 1)
    s = dict(windows=np.linspace(0, case["L"], W + 1))
    if W > 2:  # window edges that fall anywhere, as genes and centimorgans do
        step = case["L"] / W
        s["windows"][1:-1] += rng.uniform(-0.3, 0.3, W - 1) * step
    if op == "weighted":
        n = case["n"]
        s["traits"] = rng.standard_normal((n, case["K"]))
        s["covariates"] = np.column_stack([np.ones(n), rng.standard_normal((n, case["covariates"]))])
    elif "K" in case and op != "replicates":
        s["sets"] = _sets(rng, case["n"], case["K"], case["size"])
    return s


def _replicate_cases(case):
    rng = np.random.default_rng([case["count"], case["n"], case["K"], case["W"]])
    out = []
    for i in range(case["count"]):
        n = int(round(math.exp(rng.uniform(math.log(100), math.log(case["n"])))))
        L = float(round(math.exp(rng.uniform(math.log(1e5), math.log(case["L"])))))
        K = int(rng.integers(1, case["K"] + 1))
        out.append(dict(op="replicate", n=n, L=L, mu=case["mu"], K=K,
                        size=int(rng.integers(min(10, case["size"]), case["size"] + 1)),
                        W=int(rng.integers(1, case["W"] + 1))))
    return out


def prepare(case, seed):
    op = case["op"]
    if op == "replicates":
        reps = []
        for i, c in enumerate(_replicate_cases(case)):
            tables, ts = _tree_sequence(c, seed + 7919 * i)
            ts.ll_tree_sequence.upload()
            reps.append(dict(_inputs(c, seed + 7919 * i), ts=ts, case=c))
        return dict(case=case, reps=reps)
    _, ts = _tree_sequence(case, seed)
    ts.ll_tree_sequence.upload()
    return dict(_inputs(case, seed), case=case, ts=ts)


# --- one pass -------------------------------------------------------------

def run(state):
    c = state["case"]
    op = c["op"]
    if op == "replicates":
        return _run_replicates(state["reps"])
    ts, w = state["ts"], state["windows"]
    if op == "stat":
        kw = dict(windows=w, mode=c["mode"])
        idx = _indexes(c["stat"], c["K"])
        if idx is not None:
            kw["indexes"] = idx
        if c["stat"] == "genetic_relatedness":
            kw["proportion"] = False
        return getattr(ts, c["stat"])(state["sets"], **kw)
    if op == "step":
        return _run_step(ts, state["sets"], w)
    if op == "weighted":
        return ts.trait_linear_model(state["traits"], state["covariates"], windows=w,
                                     mode=c["mode"])
    if op == "spectrum":
        return [ts.allele_frequency_spectrum(state["sets"], windows=w, mode=m, polarised=True)
                for m in ("site", "branch")]
    if op == "relatedness_matrix":
        return ts.genetic_relatedness_matrix(windows=w)
    return ts.genotype_matrix()


def _run_step(ts, sets, w):
    K = len(sets)
    pairs = [(i, j) for i in range(K) for j in range(i + 1, K)]
    b = ts.batch()
    pending = {}
    for mode in ("branch", "site"):
        pending[mode] = [b.Fst(sets, indexes=pairs, windows=w, mode=mode),
                         b.Tajimas_D(sets, windows=w, mode=mode),
                         b.f4(sets, indexes=[(0, 1, 2, 3)], windows=w, mode=mode)]
    b.run()
    return {mode: [p.result() for p in ps] for mode, ps in pending.items()}


def _run_replicates(reps):
    batches, pending = [], []
    for r in reps:
        b = r["ts"].batch()
        K = len(r["sets"])
        pairs = [(j, j + 1) for j in range(K - 1)]
        for mode in ("branch", "site"):
            pending.append(b.diversity(r["sets"], windows=r["windows"], mode=mode))
            if pairs:
                pending.append(b.divergence(r["sets"], indexes=pairs, windows=r["windows"],
                                            mode=mode))
        batches.append(b)
    ta.run_batches(batches)
    return np.concatenate([p.result().reshape(-1) for p in pending])


# --- what a pass cannot do without ----------------------------------------

def _tables_size(n, L, mu):
    """Expected edges, nodes and sites of the generator."""
    h = sum(1.0 / i for i in range(1, min(n, 10000))) + max(0.0, math.log(n / 10000))
    trees = 1 + 0.9 * 4 * NE * RHO * L * h
    return 2 * n + 3.7 * trees, 2 * n + 0.65 * trees, 4 * NE * mu * L * h


def work(case):
    """The tables read once (24 + 8 bytes an edge, 8 a node, 12 a site), the
    sample sets, the windows and the results; per edge the update of every
    column and the evaluation of every output."""
    op = case["op"]
    if op == "replicates":
        w = dict(bytes=0.0, flops=0.0)
        for c in _replicate_cases(case):
            K = c["K"]
            for mode in ("branch", "site"):
                one = work(dict(c, op="stat", stat="divergence", mode=mode))
                w = {k: w[k] + one[k] for k in w}
        return w
    n, L, W = case["n"], case["L"], case.get("W", 1)
    edges, nodes, sites = _tables_size(n, L, case["mu"])
    tables = 32 * edges + 8 * nodes + 12 * sites
    K = case.get("K", 1)
    if op == "spectrum":
        out = 2 * W * (case["size"] + 1) ** 2
        return dict(bytes=float(2 * tables + 2 * n + 8 * out), flops=float(2 * 2 * edges * 3))
    if op == "relatedness_matrix":
        return dict(bytes=float(tables + 8 * W * n * n), flops=float(2 * n * n * sites))
    if op == "genotypes":
        return dict(bytes=float(tables + 4 * n * case["sites"]), flops=float(n * case["sites"]))
    if op == "weighted":
        cols, out = K + case["covariates"] + 1, W * K
        return dict(bytes=float(tables + 8 * n * cols + 8 * out),
                    flops=float(2 * edges * cols + 2 * edges * (4 * cols + 6) * K))
    if op == "step":
        M = K * (K - 1) // 2 + K + 2 * K + 1
        out, modes = W * (K * (K - 1) // 2 + K + 1), 2
    else:
        idx = _indexes(case["stat"], K)
        M = len(idx) if idx is not None else K
        out, modes = (int(nodes) if case["mode"] == "node" else W) * M, 1
    return dict(bytes=float(modes * (tables + n * ((K + 7) // 8) + 8 * (W + 1) + 8 * out)),
                flops=float(modes * (2 * edges * K + 2 * edges * 4 * M)))


# --- 64-bit values --------------------------------------------------------

MOST_VALUES = 2e9  # (node, tree, column) values beyond which exact() gives none
REGION_VALUES = 1e8  # and how many are held at once


class _Trees:
    """Per node and tree of the region bp[t0] .. bp[t1] in which the node is
    alive, the sums of the columns over the samples below it: every edge,
    parents youngest first, adds its child's values over the trees it spans."""

    def __init__(self, tables, bp, columns, t0, t1, device):
        t = tables
        left, right = np.searchsorted(bp, t.edge_left), np.searchsorted(bp, t.edge_right)
        here = np.flatnonzero((left < t1) & (right > t0))
        here = here[np.argsort(t.node_time[t.edge_parent[here]], kind="stable")]
        self.t0, self.t1 = t0, t1
        self.el, self.er = np.maximum(left[here], t0) - t0, np.minimum(right[here], t1) - t0
        self.ep, self.ec = t.edge_parent[here], t.edge_child[here]
        N, T = len(t.node_time), t1 - t0
        a, b = np.full(N, T, np.int64), np.zeros(N, np.int64)
        for ids in (self.ep, self.ec):
            np.minimum.at(a, ids, self.el)
            np.maximum.at(b, ids, self.er)
        n, K = columns.shape
        a[:n], b[:n] = 0, T
        b = np.maximum(a, b)
        off = np.concatenate([[0], np.cumsum(b - a)])
        self.a, self.off = a, off
        x = np.zeros((int(off[-1]), K), columns.dtype)
        for s in range(n):
            x[off[s]:off[s + 1]] = columns[s]
        for p, c, l, r in zip(self.ep, self.ec, self.el, self.er):
            po, co = off[p] - a[p], off[c] - a[c]
            x[po + l:po + r] += x[co + l:co + r]
        self.x = torch.from_numpy(x).to(device)
        self.length = t.node_time[self.ep] - t.node_time[self.ec]
        self.device = device

    def blocks(self, lo, hi, ids, most=1 << 21):
        """(row in x, tree, item) of the items' trees lo[i] .. hi[i] - 1."""
        size = hi - lo
        i = 0
        while i < len(size):
            stop = max(i + 1, int(np.searchsorted(np.cumsum(size[i:]), most, side="right")) + i)
            item = np.repeat(np.arange(i, stop), size[i:stop])
            first = np.concatenate([[0], np.cumsum(size[i:stop])[:-1]])
            tree = lo[item] + np.arange(len(item)) - np.repeat(first, size[i:stop])
            node = ids[item]
            yield (torch.from_numpy(self.off[node] - self.a[node] + tree).to(self.device),
                   torch.from_numpy(tree).to(self.device), item)
            i = stop


def _summary(stat, x, n, idx):
    """One column per output at the counts x [rows, K] of sets of n samples."""
    if stat == "diversity":
        return x * (n - x) / (n * (n - 1))
    if stat == "segregating_sites":
        return (x > 0) * (1 - x / n)
    if stat == "genetic_relatedness":
        p = x / n
        mean = p.mean(dim=1, keepdim=True)
        i, j = idx[:, 0], idx[:, 1]
        return (p[:, i] - mean) * (p[:, j] - mean)
    i, j = idx[:, 0], idx[:, 1]
    xi, xj, ni, nj = x[:, i], x[:, j], n[i], n[j]
    if stat == "divergence":
        return xi * (nj - xj) / (ni * (nj - (i == j).to(nj.dtype)))
    if stat == "Y2":
        return xi * (nj - xj) * (nj - xj - 1) / (ni * nj * (nj - 1))
    if stat == "f2":
        return (xi * (xi - 1) * (nj - xj) * (nj - xj - 1)
                - xi * (ni - xi) * (nj - xj) * xj) / (ni * (ni - 1) * nj * (nj - 1))
    k = idx[:, 2]
    xk, nk = x[:, k], n[k]
    if stat == "f3":
        return (xi * (xi - 1) * (nj - xj) * (nk - xk)
                - xi * (ni - xi) * (nj - xj) * xk) / (ni * (ni - 1) * nj * nk)
    m = idx[:, 3]
    xm, nm = x[:, m], n[m]
    return (xi * (nj - xj) * xk * (nm - xm)
            - xi * (nj - xj) * (nk - xk) * xm) / (ni * nj * nk * nm)


class _Values:
    """Every region's trees in turn, for summaries evaluated together."""

    def __init__(self, tables, columns, device):
        t = self.tables = tables
        self.columns, self.device = columns, device
        self.bp = np.unique(np.concatenate([t.edge_left, t.edge_right, [0.0, t.sequence_length]]))
        live = 2 * len(columns) * columns.shape[1]
        self.fits = live * (len(self.bp) - 1) <= MOST_VALUES
        step = max(16, int(REGION_VALUES / live))
        T = len(self.bp) - 1
        self.regions = [(t0, min(T, t0 + step)) for t0 in range(0, T, step)]

    def all(self, fs, total, mode, polarised):
        """For each summary in ``fs``: per site, per tree or per node its
        value (the unpolarised form adds f at the complement)."""
        t, dev = self.tables, self.device

        def both(f, x):
            v = f(x)
            return v if polarised else v + f(total - x)

        out = [[] for _ in fs]
        zero = torch.zeros((1, self.columns.shape[1]), dtype=torch.float64, device=dev)
        zero = [both(f, zero) for f in fs]
        if mode == "node":
            out = [z.repeat(len(t.node_time), 1) * t.sequence_length for z in zero]
        pos = t.site_position[t.mutation_site]
        at = np.searchsorted(self.bp, pos, side="right") - 1
        for t0, t1 in self.regions:
            r = _Trees(t, self.bp, self.columns, t0, t1, dev)
            if mode == "site":
                m = np.flatnonzero((at >= t0) & (at < t1))
                node = t.mutation_node[m]
                rows = torch.from_numpy(r.off[node] + at[m] - t0 - r.a[node]).to(dev)
                for o, f in zip(out, fs):
                    o.append(both(f, r.x[rows].double()))
                continue
            if mode == "branch":
                spans, weight = (r.el, r.er, r.ec), torch.from_numpy(r.length).to(dev)
                sums = [torch.zeros((t1 - t0, z.shape[1]), dtype=torch.float64, device=dev)
                        for z in zero]
            else:
                spans = (r.a, r.a + np.diff(r.off), np.arange(len(r.a)))
                weight = torch.from_numpy(np.diff(self.bp[t0:t1 + 1])).to(dev)
                sums = out
            for rows, tree, item in r.blocks(*spans):
                item = torch.from_numpy(item).to(dev)
                for i in range(0, len(rows), 1 << 19):
                    s = slice(i, i + (1 << 19))
                    x = r.x[rows[s]].double()
                    for o, f, z in zip(sums, fs, zero):
                        if mode == "branch":
                            o.index_add_(0, tree[s], both(f, x) * weight[item[s], None])
                        else:
                            o.index_add_(0, item[s], (both(f, x) - z) * weight[tree[s], None])
            if mode == "branch":
                for o, v in zip(out, sums):
                    o.append(v)
        return out if mode == "node" else [torch.cat(o) for o in out]

    def windowed(self, fs, total, windows, mode, polarised, normalise):
        vals = self.all(fs, total, mode, polarised)
        if mode == "node":
            return [v / self.tables.sequence_length if normalise else v for v in vals]
        win = np.asarray(windows)
        bp = torch.from_numpy(self.bp).to(self.device)
        pos = self.tables.site_position[self.tables.mutation_site]
        at = np.searchsorted(pos, win)
        out = []
        for v in vals:
            rows = []
            for w in range(len(win) - 1):
                if mode == "site":
                    rows.append(v[at[w]:at[w + 1]].sum(dim=0))
                    continue
                t0 = int(np.searchsorted(self.bp, win[w], side="right")) - 1
                t1 = int(np.searchsorted(self.bp, win[w + 1], side="left"))
                span = (torch.clamp(bp[t0 + 1:t1 + 1], max=win[w + 1])
                        - torch.clamp(bp[t0:t1], min=win[w]))
                rows.append((v[t0:t1] * span[:, None]).sum(dim=0))
            o = torch.stack(rows)
            span = torch.from_numpy(np.diff(win)).to(self.device)[:, None]
            out.append(o / span if normalise else o)
        return out


def _stat_values(values, stat, sets, windows, mode, idx=None):
    dev = values.device
    K = len(sets)
    n = torch.tensor([float(len(s)) for s in sets], dtype=torch.float64, device=dev)
    idx = _indexes(stat, K) if idx is None else idx
    idx = torch.tensor(idx, device=dev) if idx is not None else None

    def several(names, normalise=True):
        fs = [functools.partial(lambda x, name: _summary(name, x, n, idx), name=name)
              for name in names]
        return values.windowed(fs, n, windows, mode, stat == "genetic_relatedness", normalise)

    if stat == "Tajimas_D":
        T, S = several(["diversity", "segregating_sites"], False)
        h, g = (torch.stack([torch.sum(1.0 / torch.arange(1, len(s), dtype=torch.float64,
                                                          device=dev) ** e) for s in sets])
                for e in (1, 2))
        a = (n + 1) / (3 * (n - 1) * h) - 1 / h**2
        b = 2 * (n**2 + n + 3) / (9 * n * (n - 1)) - (n + 2) / (h * n) + g / h**2
        return (T - S / h) / torch.sqrt(a * S + (b / (h**2 + g)) * S * (S - 1))
    if stat == "Fst":
        d, dxy = several(["diversity", "divergence"])
        du, dv = d[:, idx[:, 0]], d[:, idx[:, 1]]
        return 1 - 2 * (du + dv) / (du + dv + 2 * dxy)
    return several([stat])[0]


def _set_columns(n, sets):
    columns = np.zeros((n, len(sets)), np.int32)
    for k, s in enumerate(sets):
        columns[s, k] = 1
    return columns


def exact(case, seed):
    op = case["op"]
    if op not in ("stat", "step", "weighted") or case["n"] > 9000 or case["L"] > 7e6:
        return None
    device = "cuda" if torch.cuda.is_available() else "cpu"
    tables, _ = _tree_sequence(case, seed)
    s = _inputs(case, seed)
    w = s["windows"]
    if op == "weighted":
        return _exact_regression(case, tables, s, device)
    values = _Values(tables, _set_columns(case["n"], s["sets"]), device)
    if not values.fits:
        return None
    sets = s["sets"]
    if op == "stat":
        return _stat_values(values, case["stat"], sets, w, case["mode"]).cpu().numpy()
    return {mode: [_stat_values(values, "Fst", sets, w, mode).cpu().numpy(),
                   _stat_values(values, "Tajimas_D", sets, w, mode).cpu().numpy(),
                   _stat_values(values, "f4", sets, w, mode, [(0, 1, 2, 3)]).cpu().numpy()]
            for mode in ("branch", "site")}


def _exact_regression(case, tables, s, device):
    """trait_linear_model's value: the covariates made orthonormal (any basis
    of their span gives the same value)."""
    W = s["traits"]
    n, K = W.shape
    Z = np.linalg.qr(s["covariates"])[0]
    C = Z.shape[1]
    V = torch.from_numpy(W.T @ Z).to(device)
    columns = np.column_stack([W, Z, np.ones(n)])
    values = _Values(tables, columns, device)
    if not values.fits:
        return None

    def f(x):
        p, z, m = x[:, :K], x[:, K:K + C], x[:, K + C:]
        denom = m - (z * z).sum(dim=1, keepdim=True)
        a = p - z @ V.T
        good = (m > 0) & (m < n) & (denom > 1e-8)
        return torch.where(good, a * a / (2 * torch.where(good, denom, 1.0) ** 2), 0.0)

    total = torch.from_numpy(columns.sum(axis=0)).to(device)
    return values.windowed([f], total, s["windows"], case["mode"], False, True)[0].cpu().numpy()
