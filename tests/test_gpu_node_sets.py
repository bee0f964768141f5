"""Shared node lists of the DF-J passes (lists of 32,768 pairs and more, aux with two and more scales
per centre): gamma and its reverse pass against the oracle's twenty nodes per function.

The cases are the forms the lists can take: 2 to 6 scales per centre (groups of four, the last one
ragged; gamma shares nodes from three scales on, the reverse with two and with multiples of four:
test_route), exponents over six decades, aux far from every pair, and aux whose functions do not share
a centre although their count is a multiple of the splats' (every function then keeps its own nodes).
One list is a single pair short, so it takes the plain records.

Tolerance: each (P|a) agrees with the oracle's to 1e-12 of itself (the parity bar for gamma, which
the lists' own error of a few 1e-15 does not move), so gamma differs by at most 1e-12 of the sum of
its terms' magnitudes, and each gradient row by 1e-9 of the largest (the parity bar).
"""
import numpy as np
import pytest
import torch

from conftest import rel_max

pytestmark = pytest.mark.gpu

N_MIN = 32768


def _case(wl, name):
    s = wl.make_small(30, 6, n_atoms=4, seed=11, spread=4.0)
    rng = np.random.default_rng(5)
    G = {"two": 2, "three": 3, "four": 4, "five": 5, "six": 6}.get(name, 4)
    la = np.log(rng.uniform(0.1, 12.0, s.M))[None] + np.log(np.geomspace(0.5, 4.0, G))[:, None]
    ac = np.repeat((s.centers + rng.normal(0.0, 0.2, (s.M, 3)))[None], G, 0)
    if name == "decades":
        la = rng.uniform(np.log(1e-3), np.log(1e3), (G, s.M))
    if name == "far":
        ac = ac + np.array([45.0, 30.0, -20.0])
    if name == "moved":            # one function of each second group stands elsewhere
        ac[2, ::2] += 0.25
    n = N_MIN - 1 if name == "short" else N_MIN + 77
    a = rng.integers(0, s.M * s.M, n)
    i, j = (a // s.M).astype(np.int32), (a % s.M).astype(np.int32)
    w = rng.uniform(0.5, 2.0, n)
    w[::7] = 0.0
    return s, la.ravel(), ac.reshape(-1, 3), i, j, w


@pytest.mark.parametrize("name", ["two", "three", "four", "five", "six", "decades", "far", "moved",
                                  "short"])
def test_gamma_and_reverse_match_oracle(g, wl, orc, cuda, name):
    s, la, ac, i, j, w = _case(wl, name)
    t = lambda a: torch.tensor(a, device="cuda").requires_grad_()
    basis = g.Splat(quat=t(s.quat), log_scale=t(s.log_scale), centers=t(s.centers))
    C = t(s.C)
    gam = g.df_coulomb_gamma_screened(basis, C, s.occ, g.IsotropicSplat(log_alpha=la, centers=ac),
                                      torch.tensor(i), torch.tensor(j), valid=torch.tensor(w))
    got = gam.detach().cpu().numpy()
    ref = orc.gamma(s.quat, s.log_scale, s.centers, s.C, s.occ, la, ac, i, j, w)
    # the terms' magnitudes, bounded: every orbital product by the largest one's
    big = np.full((s.M, 1), np.sqrt(np.abs((s.C * s.occ) @ s.C.T).max()))
    unit = orc.gamma(s.quat, s.log_scale, s.centers, big, np.ones(1), la, ac, i, j, w)
    print(f"[sets] {name}: N={len(la)} n={len(i)} gamma error / bound "
          f"{np.max(np.abs(got - ref) / (1e-12 * unit)):.2e}", flush=True)
    assert np.all(np.abs(got - ref) <= 1e-12 * unit)
    v = np.random.default_rng(3).normal(size=len(la)) / unit
    grads = torch.autograd.grad(gam, [basis.quat, basis.log_scale, basis.centers, C],
                                torch.tensor(v, device="cuda"))
    back = orc.gamma_vjp(s.quat, s.log_scale, s.centers, s.C, s.occ, la, ac, i, j, w, v)
    for what, a, b in zip(("quat", "log_scale", "centers", "C"), grads, back[-4:]):
        err = rel_max(a.cpu().numpy(), b)
        print(f"[sets] {name}: d{what} {err:.2e}", flush=True)
        assert err < 1e-9


@pytest.mark.parametrize("scales", [(0.5, 1.0, 2.0, 4.0), (0.5, 0.7, 1.0, 1.4, 2.0, 2.8, 4.0, 5.6)])
def test_exchange_on_shared_lists_matches_plain_records(g, wl, cuda, scales):
    """RI-K takes the shared lists when the scales come in fours and no aux chunk cuts a group; an
    aux chunk of 66 functions does, so the same call then runs on the plain records (checked against
    the oracle elsewhere). lam = 1e-2 keeps the metric's condition near 1e4, where two correct
    evaluations agree to the parity bars, 1e-10 for E_K and 1e-9 for gradients. Chunks of 64 and of
    100 functions leave ragged last blocks and slabs."""
    s = wl.make_small(190, 5, n_atoms=6, seed=4, spread=3.0)
    t = lambda a: torch.tensor(a, device="cuda").requires_grad_()
    basis = g.Splat(quat=t(s.quat), log_scale=t(s.log_scale), centers=t(s.centers))
    C = t(s.C)
    aux = g.init_product_aux(basis, scales=scales)
    pi, pj, v = g.neighbor_pairs(basis, eps=1e-9, unique=False)
    assert pi.shape[0] >= N_MIN
    L = g.aux_cholesky(aux, 1e-2)

    def run(chunk):
        E = g.df_exchange_energy_screened(basis, C, aux, pi, pj, valid=v, cholV=L, aux_chunk=chunk)
        return [E.detach()] + list(torch.autograd.grad(E, [basis.quat, basis.log_scale,
                                                           basis.centers, C]))

    plain = [x.cpu().numpy() for x in run(66)]
    for chunk in (0, 64, 100):
        got = [x.cpu().numpy() for x in run(chunk)]
        errs = [rel_max(a, b) for a, b in zip(got, plain)]
        print(f"[sets] exchange {len(scales)} scales, chunk {chunk}: n={pi.shape[0]} "
              + " ".join(f"{e:.1e}" for e in errs), flush=True)
        assert errs[0] < 1e-10 and max(errs[1:]) < 1e-9


def _aligned_gamma(mu, ls, ac, la, W):
    """gamma of splats whose precisions are all diagonal, (scales, centres), in the arithmetic of the
    arguments: with eigenvalues l = e^ls the pair's are L = l_i + l_j, and a node of exponent s takes
    prod_k (L_k + s)^(-1/2) exp(-s L_k d_k^2 / (L_k + s)). W holds the weights of the pairs (i, j)."""
    from oracle import oracle as orc
    t, wt = (a.astype(np.longdouble) for a in orc.quad_table())
    l = np.exp(ls)
    pi = 4 * np.arctan(np.longdouble(1))
    N = np.prod((2 * l / pi) ** np.longdouble(0.25), axis=1)
    L = l[:, None] + l[None]
    P = ((l * mu)[:, None] + (l * mu)[None]) / L
    D = mu[:, None] - mu[None]
    q = N[:, None] * N[None] * np.exp(-(l[:, None] * l[None] / L * D * D).sum(2)) * W
    out = np.zeros(la.shape, L.dtype)
    for c in range(la.shape[1]):
        d2 = (ac[c] - P) ** 2
        for g in range(la.shape[0]):
            b = np.exp(np.longdouble(la[g, c]))
            s = (t * t * b / (b + t * t))[:, None, None, None]
            f = np.prod(1 / np.sqrt(L + s), axis=3) * np.exp(-(s * L * d2 / (L + s)).sum(3))
            w = wt / ((b + t * t) * np.sqrt(b + t * t))
            out[g, c] = ((w[:, None, None] * f).sum(0) * q).sum() * (2 * b / pi) ** np.longdouble(0.75)
    return out * 2 * pi ** 3 / np.sqrt(pi)


@pytest.mark.parametrize("scales", [4, 2])
def test_compact_cluster_of_wide_splats(g, cuda, scales):
    """Splats ten times as long as they are thick, side by side within 0.2 Bohr, so that the widest
    pair's Gaussian reaches far past the box of the pairs' centres, and diffuse aux on them. The
    reference is 80-bit arithmetic, its derivatives by complex steps; all terms of gamma are positive.

    A node's value errs by at most 8e-15 of its prefactor (the hardware root's estimate, squared, and
    the exponential), so gamma errs by 1e-14, and a derivative, whose terms cancel to a few parts in
    ten here, by 1e-13 of the largest."""
    M, n = 8, N_MIN + 8
    rng = np.random.default_rng(3)
    mu = rng.normal(0.0, 0.1, (M, 3))
    ls = -np.log(2.0 * np.array([4.0, 0.3, 0.3]) ** 2) + rng.uniform(-0.05, 0.05, (M, 3))
    la = np.log(0.1 * np.geomspace(0.5, 4.0, scales))[:, None] + rng.uniform(-0.1, 0.1, M)[None]
    ac = mu.copy()
    a = np.arange(n) % (M * M)
    i, j = (a // M).astype(np.int32), (a % M).astype(np.int32)
    w = rng.uniform(0.5, 2.0, n)
    W = np.zeros((M, M), np.longdouble)
    np.add.at(W, (i, j), w.astype(np.longdouble))
    ref = _aligned_gamma(mu.astype(np.longdouble), ls.astype(np.longdouble), ac, la, W)
    h = np.longdouble(1e-30)
    dref = np.zeros((2, M, 3), np.longdouble)
    for v, m, k in np.ndindex(2, M, 3):
        x = [mu.astype(np.clongdouble), ls.astype(np.clongdouble)]
        x[v][m, k] += 1j * h
        dref[v, m, k] = _aligned_gamma(*x, ac, la, W).imag.sum() / h
    t = lambda a: torch.tensor(a, device="cuda").requires_grad_()
    quat = np.zeros((M, 4))
    quat[:, 0] = 1.0
    basis = g.Splat(quat=t(quat), log_scale=t(ls), centers=t(mu))
    aux = g.IsotropicSplat(log_alpha=la.ravel(), centers=np.tile(ac, (scales, 1)))
    gam = g.df_coulomb_gamma_screened(basis, np.ones((M, 1)), np.ones(1), aux, torch.tensor(i),
                                      torch.tensor(j), valid=torch.tensor(w))
    got = gam.detach().cpu().numpy().reshape(la.shape)
    dl, dc = torch.autograd.grad(gam.sum(), [basis.log_scale, basis.centers])
    errs = [float(np.abs(got / ref - 1).max())] + [
        float(np.abs(x.cpu().numpy() - y).max() / np.abs(y).max()) for x, y in zip((dc, dl), dref)]
    print(f"[sets] compact, {scales} scales: gamma {errs[0]:.1e} dcenters {errs[1]:.1e} "
          f"dlog_scale {errs[2]:.1e}", flush=True)
    assert errs[0] < 1e-14 and max(errs[1:]) < 1e-13


@pytest.mark.parametrize("scales", [3, 4])
@pytest.mark.parametrize("bad", ["centre", "exponent", "overflow"])
def test_bad_function_keeps_to_itself(g, wl, orc, cuda, scales, bad):
    """One aux function with a NaN centre, a NaN exponent or one past the largest double: gamma of every
    other function, those grouped with it included, agrees with the oracle (bar as above)."""
    s, la, ac, i, j, w = _case(wl, "three" if scales == 3 else "four")
    la, ac = la.copy(), ac.copy()
    at = s.M + 4                                   # second scale of the fifth centre
    if bad == "centre":
        ac[at, 1] = np.nan
    else:
        la[at] = np.nan if bad == "exponent" else 800.0
    basis = g.Splat(quat=s.quat, log_scale=s.log_scale, centers=s.centers)
    got = g.df_coulomb_gamma_screened(basis, s.C, s.occ, g.IsotropicSplat(log_alpha=la, centers=ac),
                                      torch.tensor(i), torch.tensor(j),
                                      valid=torch.tensor(w)).cpu().numpy()
    la[at], ac[at] = 0.0, 0.0
    ref = orc.gamma(s.quat, s.log_scale, s.centers, s.C, s.occ, la, ac, i, j, w)
    big = np.full((s.M, 1), np.sqrt(np.abs((s.C * s.occ) @ s.C.T).max()))
    unit = orc.gamma(s.quat, s.log_scale, s.centers, big, np.ones(1), la, ac, i, j, w)
    rest = np.arange(len(la)) != at
    assert not np.isfinite(got[at])
    assert np.all(np.abs(got - ref)[rest] <= 1e-12 * unit[rest])


@pytest.mark.parametrize("which", ["all", "some"])
def test_exchange_groups_without_a_common_centre(g, wl, cuda, which):
    """RI-K where no group of four functions, or only every second one, shares a centre, against the
    plain records (an aux chunk of 66); lam and the bars as above."""
    s = wl.make_small(190, 5, n_atoms=6, seed=4, spread=3.0)
    t = lambda a: torch.tensor(a, device="cuda").requires_grad_()
    basis = g.Splat(quat=t(s.quat), log_scale=t(s.log_scale), centers=t(s.centers))
    C = t(s.C)
    aux = g.init_product_aux(basis, scales=(0.5, 1.0, 2.0, 4.0))
    rng = np.random.default_rng(8)
    ac = aux.centers.detach().cpu().numpy().reshape(4, s.M, 3).copy()
    ac[:, ::1 if which == "all" else 2] += rng.normal(0.0, 0.3, ac[:, ::1 if which == "all" else 2].shape)
    aux = g.IsotropicSplat(log_alpha=aux.log_alpha.detach(), centers=ac.reshape(-1, 3))
    pi, pj, v = g.neighbor_pairs(basis, eps=1e-9, unique=False)
    assert pi.shape[0] >= N_MIN
    L = g.aux_cholesky(aux, 1e-2)
    out = []
    for chunk in (66, 0, 64):
        E = g.df_exchange_energy_screened(basis, C, aux, pi, pj, valid=v, cholV=L, aux_chunk=chunk)
        out.append([E.detach().cpu().numpy()] + [x.cpu().numpy() for x in torch.autograd.grad(
            E, [basis.quat, basis.log_scale, basis.centers, C])])
    for got in out[1:]:
        errs = [rel_max(a, b) for a, b in zip(got, out[0])]
        print(f"[sets] exchange, {which} apart: " + " ".join(f"{e:.1e}" for e in errs), flush=True)
        assert errs[0] < 1e-10 and max(errs[1:]) < 1e-9


@pytest.mark.parametrize("name,forward,reverse", [("two", False, True), ("three", True, False),
                                                  ("four", True, True), ("five", True, False),
                                                  ("six", True, False), ("short", False, False)])
def test_route(g, wl, cuda, name, forward, reverse):
    """Which scale counts share nodes, by the nodes each pass evaluates: plain records take all twenty of
    a function here (the system is compact: the screen leaves out 2%), shared lists of two scales nine
    tenths of them (18 a function), of more scales fewer."""
    from gs_dft_amd import _lib
    s, la, ac, i, j, w = _case(wl, name)
    ids = (_lib.PROF_GAMMA_FWD, _lib.PROF_GAMMA_BWD)
    t = lambda a: torch.tensor(a, device="cuda").requires_grad_()
    basis = g.Splat(quat=t(s.quat), log_scale=t(s.log_scale), centers=t(s.centers))
    _lib.profile_enable(True)
    try:
        for kid in ids:
            _lib.profile_read_work(kid, reset=True)
        gam = g.df_coulomb_gamma_screened(basis, t(s.C), s.occ,
                                          g.IsotropicSplat(log_alpha=la, centers=ac),
                                          torch.tensor(i), torch.tensor(j), valid=torch.tensor(w))
        gam.sum().backward()
        torch.cuda.synchronize()
        part = [_lib.profile_read_work(kid, reset=True) / (20.0 * len(la) * len(i)) for kid in ids]
    finally:
        _lib.profile_enable(False)
    print(f"[sets] {name}: of all nodes, forward {part[0]:.3f}, reverse {part[1]:.3f}", flush=True)
    for x, shared in zip(part, (forward, reverse)):
        assert x < 0.93 if shared else x > 0.96


def test_more_groups_than_one_grid_dimension_holds(g, cuda):
    """13.43 million centres of two functions: their lists' workgroups pass 2^32 work-items, which
    wraps a one-dimensional launch. J = sum_P v_P (P|a), all terms positive, against the plain records
    (a list of 64 pairs)."""
    from gs_dft_amd import ri
    M, n = 13_430_000, N_MIN
    assert M * 320 > 2 ** 32
    gen = torch.Generator("cuda").manual_seed(5)
    f8 = dict(device="cuda", dtype=torch.float64)
    centers = torch.randn(M, 3, generator=gen, **f8) * 2.0
    basis = g.Splat(quat=torch.randn(M, 4, generator=gen, **f8),
                    log_scale=torch.randn(M, 3, generator=gen, **f8) * 0.3 - 1.0, centers=centers)
    la = torch.rand(M, generator=gen, **f8)
    aux = g.IsotropicSplat(log_alpha=torch.cat([la, la + 1.0]), centers=torch.cat([centers, centers]))
    i = torch.arange(n, dtype=torch.int32, device="cuda") * 400
    w = torch.ones(n, **f8)
    v = torch.rand(2 * M, generator=gen, **f8) + 0.5
    out = []
    for m in (64, n):
        x = ri._Inputs(basis, torch.ones(M, 1, **f8), torch.ones(1, **f8), aux, i[:m], i[:m] + 1,
                       w[:m], None)
        print(f"[sets] {2 * M} functions, {m} pairs", flush=True)
        out.append(ri._gamma_vjp(x, v, None)[0].cpu().numpy())
        del x
        torch.cuda.empty_cache()
    assert np.all(np.abs(out[1][:64] - out[0]) <= 1e-12 * np.abs(out[0]))
