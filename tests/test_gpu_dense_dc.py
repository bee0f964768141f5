"""dE/dC of the nuclear attraction by the dense product, against the sum over the list's pairs in
float64 torch: odd and even sizes, ordered and unique lists, repeated pairs in no order, and an
orbital coefficient that is not finite, which may reach its partners' rows only.

A row adds up to 2 M terms: 2 M 2^-53 times the sum of their magnitudes bounds either order.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _run(g, wl, M, k, unique, repeat, bad):
    s = wl.make_small(M, k, n_atoms=30, seed=M + k, spread=2.0)
    cu = lambda a: torch.tensor(np.asarray(a), device="cuda", dtype=torch.float64)
    b = g.Splat(quat=cu(s.quat).requires_grad_(True), log_scale=cu(s.log_scale),
                centers=cu(s.centers))
    C0 = cu(s.C)
    pi, pj, w = g.neighbor_pairs(b, eps=1e-7, unique=unique)
    w = w.to(torch.float64)
    if repeat:
        order = torch.randperm(len(pi), device="cuda", generator=torch.Generator("cuda").manual_seed(1))
        pick = torch.cat([order, order[:2000], order[:2000], order[500:1500]])
        pi, pj, w = pi[pick].contiguous(), pj[pick].contiguous(), w[pick].contiguous()
    assert M < 2048 or len(pi) * k > M * M * (0.04 * k + 8.0)         # the dense product's sizes
    if bad is not None:
        C0[7, 2] = bad
    C = C0.clone().requires_grad_(True)
    E = g.screened_external_energy(b, C, s.occ, pi, pj, s.atoms, s.charges, valid=w)
    E.backward()
    V = g.screened_nuclear_pairs(b, pi, pj, s.atoms, s.charges)
    i, j = pi.long(), pj.long()
    ref = torch.zeros_like(C0)
    mag = torch.zeros_like(C0)
    for a0 in range(0, len(i), 100000):
        c = slice(a0, a0 + 100000)
        x = (V[c] * w[c])[:, None]
        for p, q in ((i, j), (j, i)):
            ref.index_add_(0, p[c], x * C0[q[c]])
            mag.index_add_(0, p[c], (x * C0[q[c]]).abs())
    occ = cu(s.occ)
    return C.grad, ref * occ, mag * occ


@pytest.mark.parametrize("M,k,unique,repeat", [(2048, 96, True, False), (2049, 97, True, False),
                                               (2177, 128, False, False), (2300, 129, True, True),
                                               (2047, 96, True, False)])
def test_dense_dc(g, wl, cuda, M, k, unique, repeat):
    print(f"[dense dC] M={M} k={k} unique={unique} repeat={repeat}", flush=True)
    got, ref, mag = _run(g, wl, M, k, unique, repeat, None)
    again = _run(g, wl, M, k, unique, repeat, None)[0]
    assert torch.equal(got, again)
    assert bool(((got - ref).abs() <= 2 * M * 2.0 ** -53 * mag).all())


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_dense_dc_keeps_a_bad_coefficient_to_its_partners(g, wl, cuda, bad):
    got, ref, mag = _run(g, wl, 2100, 96, True, False, bad)
    fine = torch.isfinite(ref)
    assert bool((torch.isfinite(got) == fine).all()) and bool((~fine).any()) and bool(fine.any())
    assert bool(((got - ref).abs()[fine] <= 4200 * 2.0 ** -53 * mag[fine]).all())


def test_dense_dc_padding_inside_the_list(g, wl, cuda):
    """Weightless (0, 0) entries between the real ones change nothing but the order of sums: 2 M
    terms a row on each side, and V's nodes a few dozen roundings apart."""
    M, k = 2048, 96
    s = wl.make_small(M, k, n_atoms=30, seed=5, spread=2.0)
    cu = lambda a: torch.tensor(np.asarray(a), device="cuda", dtype=torch.float64)
    b = g.Splat(quat=cu(s.quat), log_scale=cu(s.log_scale), centers=cu(s.centers))
    pi, pj, w = g.neighbor_pairs(b, eps=1e-7, unique=True)
    w = w.to(torch.float64)
    h = len(pi) // 2
    got = []
    for pad in (0, 100001):
        z = lambda t: torch.cat([t[:h], torch.zeros(pad, dtype=t.dtype, device=t.device), t[h:]])
        C = cu(s.C).requires_grad_(True)
        g.screened_external_energy(b, C, s.occ, z(pi), z(pj), s.atoms, s.charges,
                                   valid=z(w)).backward()
        got.append(C.grad)
    x = (g.screened_nuclear_pairs(b, pi, pj, s.atoms, s.charges) * w).abs()
    mag = torch.zeros_like(got[0])
    for p, q in ((pi.long(), pj.long()), (pj.long(), pi.long())):
        mag.index_add_(0, p, x[:, None] * cu(s.C)[q].abs())
    mag *= cu(s.occ)
    assert bool(((got[0] - got[1]).abs() <= (4 * M + 64) * 2.0 ** -53 * mag).all())
