"""Genotypes as bits: the site divergence matrix at the edges of its tiles
(128 samples), words (32) and column chunks (128, 256).  Counts of differing
sites are whole numbers below 2^53: equal, not close."""
import numpy as np
import pytest

import cases
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
