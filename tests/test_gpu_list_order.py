"""Slot order of the pairs. Lists of up to 65,536 entries keep their own order where it runs over i in
ascending order and are brought into ascending i otherwise; longer lists are sorted by the slot keys.
A wave leaves a node loop when all of its 64 pairs are out of reach, so on a long molecule the nodes
evaluated show whether neighbours share waves: the same pairs shuffled may not cost more than a tenth
more nodes than ascending (in shuffled order they cost 1.3 to 2 times as many).

The order decides which pairs share a wave and in which order lanes and slots are added: values agree to
the parity bars, 1e-12 of the largest for gamma, V and E, 1e-9 for gradients.
"""
import numpy as np
import pytest
import torch

from conftest import rel_max

pytestmark = pytest.mark.gpu


def _chain(g, wl, M, k):
    """Splats along a 50-Bohr alkane chain."""
    atoms = wl.alkane_atoms(20)
    rng = np.random.default_rng(17)
    cu = lambda a: torch.tensor(a, device="cuda", dtype=torch.float64).requires_grad_()
    own = np.arange(M) * len(atoms) // M
    basis = g.Splat(quat=cu(rng.normal(size=(M, 4))),
                    log_scale=cu(-np.log(2.0) - 2.0 * rng.uniform(np.log(0.3), np.log(3.0), (M, 3))),
                    centers=cu(atoms[own] + 0.4 * rng.normal(size=(M, 3))))
    return basis, cu(rng.normal(size=(M, k)) / np.sqrt(k)), np.ones(k), atoms


def _calls(g, basis, C, occ, atoms, pi, pj, w, what):
    leaves = [basis.quat, basis.log_scale, basis.centers, C]
    if what == "dfj":
        aux = g.init_product_aux(basis, scales=(0.5, 1.0, 2.0, 4.0))
        gam = g.df_coulomb_gamma_screened(basis, C, occ, aux, pi, pj, valid=w)
        v = torch.linspace(-1.0, 1.0, aux.n_basis, device="cuda", dtype=torch.float64)
        return gam, torch.autograd.grad(gam, leaves, v)
    if what == "nuclear":
        E = g.screened_external_energy(basis, C, occ, pi, pj, atoms, np.ones(len(atoms)), valid=w)
    else:
        E = g.screened_coulomb_energy(basis, C, occ, pi, pj, valid=w)
    return E, torch.autograd.grad(E, leaves)


@pytest.mark.parametrize("what,M", [("dfj", 330), ("dfj", 600), ("dfj", 700), ("nuclear", 600),
                                    ("exact", 330)])
def test_shuffled_list(g, wl, cuda, what, M):
    from gs_dft_amd import _lib
    ids = {"dfj": [_lib.PROF_GAMMA_FWD, _lib.PROF_GAMMA_BWD], "nuclear": [_lib.PROF_NUC_PAIRS],
           "exact": [_lib.PROF_ERI_BWD]}[what]
    basis, C, occ, atoms = _chain(g, wl, M, 12)
    pi, pj, w = g.neighbor_pairs(basis, eps=1e-7, unique=True)
    n = int((w != 0).sum())
    assert (n > 65536) == (M == 700)
    mix = torch.randperm(n, generator=torch.Generator().manual_seed(2)).cuda()
    by_j = torch.argsort(pj[:n], stable=True)        # one descent of i a column: still its own order
    out, nodes = [], []
    _lib.profile_enable(True)
    try:
        for order in (torch.arange(n, device="cuda"), mix, by_j):
            for kid in ids:
                _lib.profile_read_work(kid, reset=True)
            val, grads = _calls(g, basis, C, occ, atoms, pi[:n][order].contiguous(),
                                pj[:n][order].contiguous(), w[:n][order].contiguous(), what)
            nodes.append([_lib.profile_read_work(kid, reset=True) for kid in ids])
            out.append([x.detach().cpu().numpy() for x in (val, *grads)])
    finally:
        _lib.profile_enable(False)
    for name, got, cost in zip(("shuffled", "by j"), out[1:], nodes[1:]):
        ratio = [a / b for a, b in zip(cost, nodes[0])]
        errs = [rel_max(a, b) for a, b in zip(got, out[0])]
        print(f"[order] {what} n={n} {name}: nodes " + " ".join(f"{r:.3f}" for r in ratio) + " errors "
              + " ".join(f"{e:.1e}" for e in errs), flush=True)
        assert errs[0] < 1e-12 and max(errs[1:]) < 1e-9
        assert max(ratio) < 1.1


@pytest.mark.parametrize("M,n", [(2, 65), (1024, 1023), (1025, 4097), (1048577, 7001), (1100001, 65536)])
def test_shuffled_list_of_few_and_many_splats(g, cuda, M, n):
    """One, two and three digits of i; lists that divide no wave's part."""
    rng = np.random.default_rng(n)
    cu = lambda a: torch.tensor(a, device="cuda", dtype=torch.float64)
    basis = g.Splat(quat=cu(rng.normal(size=(M, 4))), log_scale=cu(rng.normal(-1.0, 0.3, (M, 3))),
                    centers=cu(rng.normal(0.0, 2.0, (M, 3))))
    C, occ = cu(rng.uniform(0.5, 1.0, (M, 2))), np.ones(2)
    aux = g.IsotropicSplat(log_alpha=rng.normal(size=5), centers=rng.normal(size=(5, 3)))
    i, j = np.sort(rng.integers(0, M, n)), rng.integers(0, M, n)
    w = rng.uniform(0.5, 1.0, n)
    mix = rng.permutation(n)
    out = [g.df_coulomb_gamma_screened(basis, C, occ, aux, torch.tensor(i[o].astype(np.int32)),
                                       torch.tensor(j[o].astype(np.int32)),
                                       valid=torch.tensor(w[o])).cpu().numpy()
           for o in (np.arange(n), mix)]
    print(f"[order] M={M} n={n}: {rel_max(out[1], out[0]):.1e}", flush=True)
    assert rel_max(out[1], out[0]) < 1e-12


def _repeated(M, n, rng):
    """Every ordered pair of M splats, over and over, shuffled; some entries dead."""
    a = rng.permutation(np.arange(n) % (M * M))
    w = rng.uniform(0.5, 2.0, n)
    w[::7] = 0.0
    w[-1] = 1.0
    return (a // M).astype(np.int32), (a % M).astype(np.int32), w


@pytest.mark.parametrize("n", [65536, 65537, 70001])
def test_long_list_against_oracle(g, wl, orc, cuda, n):
    """Both sides of the length from which lists are sorted, shared node lists in both passes."""
    s = wl.make_small(30, 6, n_atoms=4, seed=11, spread=4.0)
    rng = np.random.default_rng(n)
    i, j, w = _repeated(s.M, n, rng)
    la = (np.log(rng.uniform(0.1, 12.0, s.M))[None] + np.log(np.geomspace(0.5, 4.0, 4))[:, None])
    ac = np.tile(s.centers + rng.normal(0.0, 0.2, (s.M, 3)), (4, 1))
    t = lambda a: torch.tensor(a, device="cuda").requires_grad_()
    basis = g.Splat(quat=t(s.quat), log_scale=t(s.log_scale), centers=t(s.centers))
    C = t(s.C)
    gam = g.df_coulomb_gamma_screened(basis, C, s.occ,
                                      g.IsotropicSplat(log_alpha=la.ravel(), centers=ac),
                                      torch.tensor(i), torch.tensor(j), valid=torch.tensor(w))
    v = rng.normal(size=la.size)
    got = torch.autograd.grad(gam, [basis.quat, basis.log_scale, basis.centers, C],
                              torch.tensor(v, device="cuda"))
    ref = orc.gamma(s.quat, s.log_scale, s.centers, s.C, s.occ, la.ravel(), ac, i, j, w)
    back = orc.gamma_vjp(s.quat, s.log_scale, s.centers, s.C, s.occ, la.ravel(), ac, i, j, w, v)
    errs = [rel_max(gam.detach().cpu().numpy(), ref)] + [rel_max(a.cpu().numpy(), b)
                                                         for a, b in zip(got, back[-4:])]
    print(f"[order] oracle n={n}: " + " ".join(f"{e:.1e}" for e in errs), flush=True)
    assert errs[0] < 1e-12 and max(errs[1:]) < 1e-9


@pytest.mark.parametrize("n", [65536, 70001])
def test_nuclear_gradients_on_a_long_list(g, wl, tr, cuda, n):
    s = wl.make_small(24, 5, n_atoms=4, seed=6)
    rng = np.random.default_rng(n)
    i, j, w = _repeated(s.M, n, rng)
    t = lambda a: torch.tensor(a, device="cuda").requires_grad_()
    basis = g.Splat(quat=t(s.quat), log_scale=t(s.log_scale), centers=t(s.centers))
    C, R = t(s.C), t(np.asarray(s.atoms))
    E = g.screened_external_energy(basis, C, s.occ, torch.tensor(i), torch.tensor(j), R, s.charges,
                                   valid=torch.tensor(w))
    got = torch.autograd.grad(E, [basis.quat, basis.log_scale, basis.centers, C, R])
    # the oracle on the distinct pairs, their weights added
    W = np.zeros(s.M * s.M)
    np.add.at(W, i.astype(np.int64) * s.M + j, w)
    p, q = (torch.as_tensor(a) for a in np.divmod(np.arange(s.M * s.M), s.M))
    c = lambda a: torch.tensor(np.asarray(a), dtype=torch.float64)
    ref = [c(a).requires_grad_() for a in (s.quat, s.log_scale, s.centers, s.C, s.atoms)]
    Er = tr.screened_external_energy(*ref[:4], c(s.occ), p, q, c(W), ref[4], c(s.charges))
    want = torch.autograd.grad(Er, ref)
    errs = [abs(E.item() / Er.item() - 1)] + [rel_max(a.cpu().numpy(), b.numpy())
                                              for a, b in zip(got, want)]
    print(f"[order] nuclear n={n}: " + " ".join(f"{e:.1e}" for e in errs), flush=True)
    assert errs[0] < 1e-12 and max(errs[1:]) < 1e-9


def test_exchange_on_shared_lists_of_a_sorted_list(g, wl, cuda):
    """RI-K over 72,200 entries (every pair twice, shuffled), its groups in the sort's order: shared
    node lists against plain records (an aux chunk of 66 cuts their groups), and against the same entries
    in ascending order. lam = 1e-2 keeps the metric's condition near 1e4, as in test_gpu_node_sets.py."""
    s = wl.make_small(190, 5, n_atoms=6, seed=4, spread=3.0)
    t = lambda a: torch.tensor(a, device="cuda").requires_grad_()
    basis = g.Splat(quat=t(s.quat), log_scale=t(s.log_scale), centers=t(s.centers))
    C = t(s.C)
    aux = g.init_product_aux(basis, scales=(0.5, 1.0, 2.0, 4.0))
    L = g.aux_cholesky(aux, 1e-2)
    a = np.arange(2 * s.M * s.M) % (s.M * s.M)
    out = []
    for order, chunk in ((np.random.default_rng(1).permutation(len(a)), 66),
                         (np.random.default_rng(1).permutation(len(a)), 0), (np.argsort(a), 0)):
        i, j = (torch.tensor(x.astype(np.int32)) for x in np.divmod(a[order], s.M))
        E = g.df_exchange_energy_screened(basis, C, aux, i, j, cholV=L, aux_chunk=chunk)
        out.append([E.detach().cpu().numpy()] + [x.cpu().numpy() for x in torch.autograd.grad(
            E, [basis.quat, basis.log_scale, basis.centers, C])])
    for got in out[1:]:
        errs = [rel_max(x, y) for x, y in zip(got, out[0])]
        print("[order] exchange: " + " ".join(f"{e:.1e}" for e in errs), flush=True)
        assert errs[0] < 1e-10 and max(errs[1:]) < 1e-9
