"""The nuclear pair pass at its edges: nuclei around the slab (16) and the force chunk (64), pair
counts around a workgroup (256) and a wave, nuclei that share a position, a single nucleus far off.

Node values are rounded to ~1e-15 of the sum, and a gradient sums terms that cancel to a few per
cent at most here: 1e-12 relative to the largest entry is a hundred times that.
"""
import numpy as np
import pytest
import torch

from conftest import rel_max

pytestmark = pytest.mark.gpu

BAR = 1e-12


def _cu(a, grad=False):
    return torch.tensor(np.asarray(a), device="cuda", dtype=torch.float64).requires_grad_(grad)


def _t(x, grad=False):
    t = torch.as_tensor(np.asarray(x), dtype=torch.float64).clone()
    return t.requires_grad_(grad) if grad else t


@pytest.mark.parametrize("forces", [True, False])
@pytest.mark.parametrize("atoms,pairs", [(1, 1), (1, 257), (15, 64), (16, 65), (17, 255), (63, 256),
                                         (64, 100), (65, 300), (129, 257)])
def test_nuclear_pass_edges(g, wl, orc, tr, cuda, atoms, pairs, forces):
    s = wl.make_small(40, 5, n_atoms=4, seed=atoms + pairs)
    pi, pj, w, _ = orc.neighbor_pairs(s.quat, s.log_scale, s.centers, s.eps, None, True)
    pi, pj, w = pi[:pairs], pj[:pairs], w[:pairs]
    assert len(pi) == pairs
    rng = np.random.Generator(np.random.PCG64(atoms))
    R = rng.normal(0.0, 4.0, (atoms, 3))
    Z = rng.uniform(1.0, 9.0, atoms)
    if atoms > 2:
        R[1] = R[0]                       # two nuclei at one point
        R[2] = R[2] + 60.0                # past the reach of most nodes
    print(f"[nuc edges] atoms={atoms} pairs={pairs} forces={forces}", flush=True)
    basis = g.Splat(quat=_cu(s.quat, True), log_scale=_cu(s.log_scale, True),
                    centers=_cu(s.centers, True))
    C, Rg = _cu(s.C, True), _cu(R, forces)
    E = g.screened_external_energy(basis, C, s.occ, pi, pj, Rg, Z, valid=w)
    E.backward()
    ref = [_t(s.quat, True), _t(s.log_scale, True), _t(s.centers, True), _t(s.C, True), _t(R, True)]
    idx = [torch.as_tensor(np.asarray(a, dtype=np.int64)) for a in (pi, pj)]
    Er = tr.screened_external_energy(*ref[:4], _t(s.occ), *idx, _t(w), ref[4], _t(Z))
    Er.backward()
    assert abs(E.item() - Er.item()) < BAR * abs(Er.item())
    got = [basis.quat, basis.log_scale, basis.centers, C] + ([Rg] if forces else [])
    for a, b in zip(got, ref):
        assert rel_max(a.grad.cpu().numpy(), b.grad.numpy()) < BAR
