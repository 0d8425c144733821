"""Genotypes as bits: the site divergence matrix at the edges of its tiles
(128 samples), words (32) and column chunks (128, 256).  Counts of differing
sites are whole numbers below 2^53: equal, not close."""
import numpy as np
import pytest

import cases
import tskit_amd as ta
from oracle.oracle import Oracle


def differing(G, pos, win):
    D = np.zeros((len(win) - 1, G.shape[1], G.shape[1]))
    for w in range(len(win) - 1):
        for row in G[(pos >= win[w]) & (pos < win[w + 1])]:
            D[w] += row[:, None] != row[None, :]
    return D


@pytest.mark.gpu
@pytest.mark.parametrize("n", [2, 31, 33, 64, 127, 129, 300])
@pytest.mark.parametrize("multi", [False, True])
def test_cross_products(require_gpu, n, multi):
    tc = (cases.multiallelic if multi else cases.generated)(n, 4e5, 40 + n)
    ts = tc.tree_sequence()
    G = Oracle(tc).genotype_matrix(False)
    pos, L = tc.site_position, tc.sequence_length
    S = len(pos)
    # windows of 0, 1, 127, 128, 129 sites and the rest (as far as there are)
    cuts = [i for i in np.cumsum([1, 127, 128, 129, 256, 257]) if i < S]
    win = np.unique(np.concatenate([[0, pos[0] / 2], pos[cuts], [L]]))
    for w in (np.array([0, L]), win, np.linspace(0, L, 40)):
        print("[case]", n, multi, S, len(w) - 1, flush=True)
        got = ts.divergence_matrix(windows=w, mode="site", span_normalise=False)
        assert np.array_equal(got, differing(G, pos, w))


@pytest.mark.gpu
def test_split_columns(require_gpu):
    """One tile and enough sites that their columns go to several workgroups."""
    tc = cases.generated(40, 6e6, 77, mu=1e-7)
    ts = tc.tree_sequence()
    assert ts.num_sites >= 3 * 8192
    G = Oracle(tc).genotype_matrix(False).astype(np.float64)
    C = G.T @ G
    d = np.diag(C)
    got = ts.divergence_matrix(mode="site", span_normalise=False)
    assert np.array_equal(got, d[:, None] + d[None, :] - 2 * C)


@pytest.mark.gpu
@pytest.mark.parametrize("make", ["generated", "multiallelic", "gapped"])
@pytest.mark.parametrize("n", [3, 15, 16, 17, 32, 33, 65, 129, 1000])
def test_genotypes(require_gpu, make, n):
    """Rows that start at every place of a 16-byte store, sites within one
    store, and results large enough to come as bytes (1000 samples)."""
    L = 1e6 if n == 1000 else 2e5
    tc = getattr(cases, make)(n, L, 60 + n)
    ts, orc = tc.tree_sequence(), Oracle(tc)
    for missing in (True, False):
        print("[case]", make, n, missing, ts.num_sites, flush=True)
        assert np.array_equal(ts.genotype_matrix(isolated_as_missing=missing),
                              orc.genotype_matrix(missing))


@pytest.mark.gpu
@pytest.mark.parametrize("alleles", [128, 129])
def test_many_alleles(require_gpu, alleles):
    """The last number of alleles whose indexes are bytes, and the next."""
    n, S = 200, 100
    tc = ta.TableCollection(100.0)
    flags = np.zeros(n + 1, np.uint32)
    flags[:n] = 1
    tc.set_nodes(flags, np.array([0.0] * n + [1.0]))
    tc.set_edges(np.zeros(n), np.full(n, 100.0), np.full(n, n, np.int32),
                 np.arange(n, dtype=np.int32))
    m = alleles - 1
    tc.site_position = np.arange(S, dtype=np.float64)
    tc.ancestral_state = np.zeros(S, np.int8)
    tc.ancestral_state_offset = np.arange(S + 1, dtype=np.uint64)
    tc.mutation_site = np.repeat(np.arange(S, dtype=np.int32), m)
    tc.mutation_node = np.tile(np.arange(m, dtype=np.int32), S)
    tc.mutation_parent = np.full(S * m, -1, np.int32)
    tc.derived_state = np.tile(np.arange(1, m + 1).astype(np.uint8).view(np.int8), S)
    tc.derived_state_offset = np.arange(S * m + 1, dtype=np.uint64)
    ts = tc.tree_sequence()
    exp = np.zeros((S, n), np.int32)
    exp[:, :m] = np.arange(1, m + 1)
    assert np.array_equal(ts.genotype_matrix(), exp)
