"""The forward three-centre pass splits the pair slots over blocks whose size depends on the list
and the aux (256 to 8192 slots). gamma is checked against the oracle at list lengths on both sides
of the block edges, on ordered lists cut to that length, with aux counts that leave ragged record
blocks and with one that bounds the block from below (slots per block >= N / 8).

Tolerance: each term of gamma agrees with the oracle's to 1e-12 of its size (the bar of the parity
tests for gamma), so a sum differs by at most 1e-12 of the sum of the terms' magnitudes.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,n_aux", [(1, 1), (255, 11), (256, 12), (257, 13), (1023, 37),
                                     (2049, 36), (2600, 4099)])
def test_gamma_at_block_edges_matches_oracle(g, wl, orc, cuda, n, n_aux):
    s = wl.make_small(60, 7, n_atoms=5, seed=2, spread=4.0)
    i, j = (a.ravel().astype(np.int32) for a in np.divmod(np.arange(n) % (s.M * s.M), s.M))
    w = np.ones(n)
    rng = np.random.default_rng(n_aux)
    la = rng.uniform(np.log(0.1), np.log(20.0), n_aux)
    ac = s.centers[rng.integers(0, s.M, n_aux)] + rng.normal(0.0, 0.3, (n_aux, 3))
    basis = g.Splat(quat=s.quat, log_scale=s.log_scale, centers=s.centers)
    gam = g.df_coulomb_gamma_screened(basis, s.C, s.occ,
                                      g.IsotropicSplat(log_alpha=la, centers=ac),
                                      torch.tensor(i), torch.tensor(j),
                                      valid=torch.tensor(w)).cpu().numpy()
    ref = orc.gamma(s.quat, s.log_scale, s.centers, s.C, s.occ, la, ac, i, j, w)
    q = np.abs((s.C[i] * s.occ * s.C[j]).sum(1)).max()
    unit = orc.gamma(s.quat, s.log_scale, s.centers, np.ones((s.M, 1)), np.array([q]), la, ac, i,
                     j, w)
    print(f"[blocks] n={n} N={n_aux}: max error / bound "
          f"{np.max(np.abs(gam - ref) / (1e-12 * unit)):.2e}")
    assert np.all(np.abs(gam - ref) <= 1e-12 * unit)
