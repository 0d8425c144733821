"""The library's host code on a HIP runtime of host memory (host/
host_runtime.cpp): which kernels a call launches, with what grids, and what it
does where memory or threads are refused.  No kernel runs, so results are not
looked at."""
import json
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")

PRELUDE = """
import ctypes, json, sys
sys.path[:0] = [%r, %r]
import numpy as np
import cases
import tskit_amd as ta
H = ctypes.CDLL(None)
H.host_launches.restype = ctypes.c_char_p
H.host_held.restype = H.host_most.restype = ctypes.c_size_t
H.host_capacity.argtypes = H.host_most_new.argtypes = [ctypes.c_size_t]

def refuse(*sizes):
    H.host_refuse((ctypes.c_size_t * len(sizes))(*sizes), len(sizes))

def sizes():
    out = (ctypes.c_size_t * 4096)()
    return list(out[:H.host_sizes(out, 4096)])

def launches():
    rows = [r.split() for r in H.host_launches().decode().splitlines()]
    return [(r[0], [int(v) for v in r[1:]]) for r in rows]

def kernels():
    return [k for k, _ in launches()]

def on_states():
    return any("k_state" in k or "k_genotypes" in k or "k_site_bits" in k for k in kernels())
""" % (os.path.dirname(HERE), HERE)


@pytest.fixture(scope="session")
def host(tmp_path_factory):
    """Runs a snippet in a process of its own on the host runtime; what it
    assigns to ``out`` comes back."""
    lib = str(tmp_path_factory.mktemp("host") / "host_runtime.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I",
                    os.path.join(ROCM, "include"), "-o", lib,
                    os.path.join(HERE, "host", "host_runtime.cpp"), "-ldl"], check=True)

    def run(code):
        env = dict(os.environ, LD_PRELOAD=lib, OPENBLAS_NUM_THREADS="1")
        p = subprocess.run([sys.executable, "-c",
                            PRELUDE + code + "\nprint('\\n' + json.dumps(out))"],
                           env=env, capture_output=True, text=True, timeout=300)
        assert p.returncode == 0, (p.returncode, p.stderr[-3000:])
        return json.loads(p.stdout.splitlines()[-1])

    return run


CALLS = """
sets = [np.arange(0, 100), np.arange(100, 300)]
calls = {
    "branch": lambda ts: ts.diversity(sets, mode="branch"),
    "site": lambda ts: ts.diversity(sets, mode="site"),
    "node": lambda ts: ts.diversity(sets, mode="node"),
    "spectrum": lambda ts: ts.allele_frequency_spectrum([s[:5] for s in sets]),
    "genotypes": lambda ts: ts.genotype_matrix(),
    "matrix": lambda ts: ts.genetic_relatedness_matrix(),
}
tc = cases.generated(300, 3e5, 11)
"""


def test_plan_that_does_not_fit(host):
    """Where the state plan, or the part of it that a call adds on its first
    need, does not fit in device memory, the call runs on the chunk plans and
    the resident bytes are those that are there."""
    out = host(CALLS + """
ts = tc.tree_sequence()
ts.ll_tree_sequence.upload()
plan = sizes()[-1]                       # uploaded last
out = {"usual": {}, "refused": {}, "added": {}}
for name, call in calls.items():
    before = ts.ll_tree_sequence.get_device_bytes()
    H.host_reset()
    call(ts)
    out["usual"][name] = on_states()
    out["added"][name] = ts.ll_tree_sequence.get_device_bytes() - before
ts = tc.tree_sequence()
refuse(plan)
ts.ll_tree_sequence.upload()
out["held"] = [ts.ll_tree_sequence.get_device_bytes(), sum(sizes()[-2:])]
for name, call in calls.items():
    H.host_reset()
    call(ts)
    out["refused"][name] = on_states()
for name in ("node", "spectrum", "genotypes", "matrix"):
    refuse()
    ts = tc.tree_sequence()
    ts.ll_tree_sequence.upload()
    refuse(out["added"][name] or out["added"]["genotypes"])
    H.host_reset()
    calls[name](ts)
    out["refused"][name + " part"] = on_states()
""")
    assert all(out["usual"].values()), out
    assert all(out["added"][k] > 0 for k in ("node", "spectrum", "genotypes")), out
    assert not any(out["refused"].values()), out
    assert out["held"][0] < out["held"][1] + 1024


def test_rows_that_do_not_fit(host):
    """Where the device holds the plans and what a call on the chunk plans
    allocates, the call runs, whatever its rows on the state plan take."""
    out = host(CALLS + """
tc = cases.generated(3000, 1e6, 13)
sets = [np.arange(100 * i, 100 * i + 100) for i in range(24)]
calls["spectrum"] = lambda ts: ts.allele_frequency_spectrum([s[:2] for s in sets[:12]])
out = {}
for name, call in calls.items():
    ts = tc.tree_sequence()
    H.host_reset()
    ts.ll_tree_sequence.upload()
    plan = sizes()[-1]
    call(ts)                             # (the parts a call adds are resident)
    parts = ts.ll_tree_sequence.get_device_bytes()
    del ts
    ts = tc.tree_sequence()
    refuse(plan)
    H.host_reset()
    ts.ll_tree_sequence.upload()
    parts -= ts.ll_tree_sequence.get_device_bytes()
    call(ts)
    need = H.host_most()
    del ts
    refuse()
    ts = tc.tree_sequence()
    H.host_capacity(parts + need + 65536)
    H.host_reset()
    call(ts)
    out[name] = kernels()
    H.host_capacity(2 ** 64 - 1)
    del ts
""")
    assert set(out) == {"branch", "site", "node", "spectrum", "genotypes", "matrix"}
    for name, kernel in [("branch", "k_sweep"), ("site", "k_sweep"), ("matrix", "k_geno_hot")]:
        assert any(kernel in k for k in out[name]), (name, out[name])


STARS = """
def stars(n, trees):
    rng = np.random.default_rng(2)
    cur, since, rows = rng.integers(n, n + 2, n), np.zeros(n), []
    for t in range(1, trees):
        s = rng.integers(n)
        rows.append((since[s], t, cur[s], s))
        cur[s], since[s] = 2 * n + 1 - cur[s], t
    rows += [(since[s], trees, cur[s], s) for s in range(n)]
    rows += [(0, trees, n + 2, n), (0, trees, n + 2, n + 1)]
    tc = ta.TableCollection(float(trees))
    flags = np.zeros(n + 3, np.uint32)
    flags[:n] = 1
    tc.set_nodes(flags, np.concatenate([np.zeros(n), [1.0, 1.0, 2.0]]))
    a = np.array([r for r in rows if r[0] < r[1]])
    tc.set_edges(a[:, 0], a[:, 1], a[:, 2].astype(np.int32), a[:, 3].astype(np.int32))
    tc.sort_edges()
    return tc
"""


def test_no_more_threads(host):
    """Where no thread can be started, the calling thread does their work: the
    same plans, and the same launches."""
    out = host("""
tc = ta.simulate_tables(5000, 3e6, 1e4, 1e-8, 1e-8, 3)   # every pool is used
plans, calls, count = [], [], []
for none in (0, 1):
    H.host_no_threads(none)
    before = H.host_started()
    H.host_reset()
    ts = tc.tree_sequence()
    ll = ts.ll_tree_sequence
    plans.append([ll.get_state_plan(), ll.get_hot_plan()])
    ts.diversity([np.arange(100)], mode="branch")
    ts.genotype_matrix()
    bs = []
    for k in range(4):
        bs.append(ts.batch())
        bs[-1].diversity([np.arange(100 * k, 100 * k + 100)], mode="branch")
        bs[-1].diversity([np.arange(70)] + [np.arange(k, 70 + j) for j in range(70)], mode="site")
    ta.run_batches(bs)
    calls.append(launches())
    count.append(H.host_started() - before)
same = all(np.array_equal(a[k], b[k]) for a, b in zip(*plans) for k in a)
out = dict(same=bool(same), calls=calls[0] == calls[1], count=count)
""")
    assert out["same"] and out["calls"]
    assert out["count"][0] > 8 and out["count"][1] == 0


def test_no_more_memory(host):
    """Where the host has no memory for the state plan the tree sequence does
    without it; where it has none for the rest, that is an error."""
    out = host(STARS + """
tc = stars(200, 40000)
E = tc.num_edges
out = {}
for name, most in [("plan", E * 90), ("rest", E * 8)]:
    H.host_most_new(most)
    try:
        ts = tc.tree_sequence()
        out[name] = ts.ll_tree_sequence.get_state_plan_sizes()["usable"]
    except Exception as e:
        out[name] = str(e)
    H.host_most_new(2 ** 64 - 1)
out["usual"] = tc.tree_sequence().ll_tree_sequence.get_state_plan_sizes()["usable"]
""")
    assert out["plan"] == 0 and out["usual"] == 1
    assert "emory" in out["rest"]


def test_launches_stay_below_their_limit(host):
    """Grids of 2^32 threads or more are refused by the runtime: bit rows of
    many sites go in several launches, a request of 17 million windows to the
    chunk plans (which take no workgroup a window), and batches that are too
    large together in several launches of some of them."""
    out = host("""
n, S, T = 60000, 2300000, 1
tc = ta.TableCollection(1.0)
flags = np.ones(n + 1, np.uint32)
flags[n] = 0
tc.set_nodes(flags, np.concatenate([np.zeros(n), [1.0]]))
tc.set_edges(np.zeros(n), np.ones(n), np.full(n, n, np.int32), np.arange(n, dtype=np.int32))
tc.site_position = np.arange(S) / S
tc.ancestral_state = np.full(S, ord("0"), np.int8)
tc.ancestral_state_offset = np.arange(S + 1, dtype=np.uint64)
tc.mutation_site = np.arange(S, dtype=np.int32)
tc.mutation_node = (np.arange(S) % n).astype(np.int32)
tc.mutation_parent = np.full(S, -1, np.int32)
tc.derived_state = np.full(S, ord("1"), np.int8)
tc.derived_state_offset = np.arange(S + 1, dtype=np.uint64)
ts = tc.tree_sequence()
ts.genetic_relatedness_matrix(sample_sets=[[0], [1]])
grids = [g for k, g in launches() if "k_site_bits" in k]
out = dict(bits=[len(grids), sum(g[0] for g in grids) * 256 >= S * 1875])
del ts, tc
tc = cases.generated(300, 3e5, 11)
ts = tc.tree_sequence()
H.host_reset()
W = 17000000
ts.diversity([np.arange(100)], windows=np.linspace(0, 3e5, W + 1), mode="branch")
out["windows"] = on_states()
ts = [tc.tree_sequence() for _ in range(3)]
bs = [t.batch() for t in ts]
for b in bs:
    b.diversity([np.arange(100)], windows=np.linspace(0, 3e5, 8000001), mode="branch")
H.host_reset()
ta.run_batches(bs)
grids = [g for k, g in launches() if "k_states_windows" in k]
out["batches"] = [len(grids), sum(g[0] for g in grids)]
""")
    assert out["bits"] == [3, True]
    assert out["windows"] is False
    assert out["batches"][0] > 1 and out["batches"][1] == 24000000


def test_batches_of_more_columns_than_a_run(host):
    """A batch that does not fit one run on the state plan goes there in
    parts; the chunk sweeps take the queries that do not fit alone."""
    out = host("""
tc = cases.generated(300, 3e5, 11)
def fill(widths):
    b = tc.tree_sequence().batch()
    for i, K in enumerate(widths):
        sets = [np.arange(j, j + 5 + i) for j in range(K)]
        for mode in ("branch", "site"):
            b.diversity(sets, mode=mode)
    return b
out = {}
for name, widths in [("fit", (40, 20, 30, 30)), ("one", (40, 70, 30))]:
    H.host_reset()
    fill(widths).run()
    out[name] = kernels()
    bs = [fill(widths) for _ in range(2)]
    H.host_reset()
    ta.run_batches(bs)
    out[name + " together"] = kernels()
""")
    for name, ks in out.items():
        many = "together" in name
        evals = [k for k in ks if ("k_states_eval" if many else "k_state_eval") in k]
        sweeps = [k for k in ks if "k_sweep" in k]
        assert len(sweeps) == (2 if "one" in name else 0), (name, sweeps)
        # two runs; together one launch a mode over all of them
        assert len(evals) == (2 if many else 4), (name, evals)


def test_large_results(host):
    """A result that does not arrive leaves the caller's buffer as it was, and
    calls at one time share the threads that copy their results."""
    out = host("""
import threading
from tskit_amd import _lib
tc = ta.simulate_tables(2000, 1e6, 1e4, 1e-8, 2e-8, 3)
ts = tc.tree_sequence()
ll, lib = ts.ll_tree_sequence, _lib.lib()
shape = (ts.num_sites, 2000)
got = np.full(shape, 7, np.int32)
H.host_events(100000, 1)
rc = lib.tsg_treeseq_genotype_matrix(ll._h, 1, got.ctypes.data)
out = dict(bytes=got.nbytes, rc=rc, kept=bool((got == 7).all()))
H.host_events(20000, 0)
def call():
    ts.genotype_matrix()
python = [threading.Thread(target=call) for _ in range(6)]
for t in python: t.start()
for t in python: t.join()
out["threads"] = H.host_most_live()
""")
    assert out["bytes"] > 2 ** 25 and out["rc"] != 0 and out["kept"]
    assert out["threads"] <= 6 + 7


def test_tuning_the_chunks(host):
    """The tuner times the chunk sweeps, and a change of the chunk count
    leaves the state plan where it is."""
    out = host(CALLS + """
from tskit_amd import autotune
ts = tc.tree_sequence()
ll = ts.ll_tree_sequence
ll.upload()
plan = sizes()[-1]
H.host_reset()
got = autotune.tune(ts, candidates=(64, 256), reps=1, table={})
out = dict(states=on_states(), sweeps=sum("k_sweep" in k for k in kernels()))
b = [t.batch() for t in (ts, ts)]
def run():
    b = [ts.batch() for _ in range(2)]
    for x in b:
        x.diversity(sets, mode="branch")
    ta.run_batches(b)
import types
sys.modules["torch"] = types.SimpleNamespace(cuda=types.SimpleNamespace(synchronize=lambda: None))
H.host_reset()
autotune.tune_batch([ts], run, candidates=(64, 256), reps=1)
ks = kernels()
out["joint"] = [sum("k_sweep" in k for k in ks), sum("k_states_eval" in k for k in ks)]
out["sent"] = plan in sizes()
H.host_reset()
ts.diversity(sets, mode="branch")
out["after"] = on_states()
""")
    assert out["sweeps"] == 4 and not out["states"]
    assert out["joint"] == [4, 1]  # (the last run warms the usual plan)
    assert out["after"] and not out["sent"]


def test_serving_estimates_cover_what_a_launch_allocates(host):
    """The admission's estimate of a launch, on the state plan and on the
    chunk plans, is at least what the launch allocates and within a few times
    of it where that is large."""
    out = host("""
from tskit_amd import serve
tc = cases.generated(3000, 1e6, 13)
rng = np.random.default_rng(1)
def sets(k, size=60):
    return [rng.choice(3000, size, replace=False) for _ in range(k)]
pairs = [(i, i + 1) for i in range(9)]
w = np.linspace(0, 1e6, 41)
launches_ = {
    "one": [("diversity", dict(sample_sets=sets(1), mode="site"))],
    "wide": [("diversity", dict(sample_sets=sets(64), mode="branch", windows=np.linspace(0, 1e6, 2001)))],
    "mixed": [("Fst", dict(sample_sets=sets(10), indexes=pairs, windows=w, mode="branch")),
              ("Tajimas_D", dict(sample_sets=sets(12), windows=w, mode="branch")),
              ("f4", dict(sample_sets=sets(4), indexes=[(0, 1, 2, 3)], windows=w, mode="branch")),
              ("genetic_relatedness", dict(sample_sets=sets(7), indexes=[(0, 1)], windows=w,
                                           mode="branch"))],
    "site": [("divergence", dict(sample_sets=sets(10), indexes=pairs, windows=w, mode="site"))
             for _ in range(5)],
    "columns": [("diversity", dict(sample_sets=sets(70), windows=w, mode="site")),
                ("diversity", dict(sample_sets=sets(30), windows=w, mode="site")),
                ("diversity", dict(sample_sets=sets(50), windows=w, mode="site"))],
    "node": [("diversity", dict(sample_sets=sets(3), mode="node"))],
    "spectrum": [("allele_frequency_spectrum", dict(sample_sets=sets(2, 40), windows=w))],
}
out = {}
for name, asks in launches_.items():
    ts = tc.tree_sequence()
    srv = serve.StatServer([ts], max_inflight=1, memory_budget=1 << 40)
    reqs = [serve.Request(i, 0, stat, kw) for i, (stat, kw) in enumerate(asks)]
    for r in reqs:
        r.normalise(ts)
    resident, before = ts.ll_tree_sequence.get_device_bytes(), H.host_held()
    H.host_reset()
    srv._run([reqs])
    assert all(r.error is None for r in reqs), reqs[0].error
    parts = ts.ll_tree_sequence.get_device_bytes() - resident
    out[name] = [H.host_most() - before - parts, srv.job_bytes([reqs])]
""")
    for name, (held, estimate) in out.items():
        assert held <= estimate, (name, held, estimate)
        assert estimate <= 3 * held + (1 << 20), (name, held, estimate)
