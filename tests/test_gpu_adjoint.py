"""Transposed operator and gradients on the GPU.

Pins, all on seeded synthetic Hamiltonians:
  * J^T from dpd_problem_sigma_t equals the transpose of the dense operator the
    oracle's sigma builds column by column (tiny system), and y.J x = x.J^T y on
    random blocks of vectors (C2v 24 orbitals, a small D2h system, every method);
  * d(L.J R)/d(theta) from dpd_problem_grad equals the central difference of the
    oracle's L.J(theta) R along random directions, one input at a time;
  * d w/d theta of an eigenvalue through the autograd Function equals the central
    difference of the GPU eigenvalue along random directions;
  * the FP32 and BF16x3 gradients stay within 1e-3 (relative 2-norm) of FP64.
"""
import numpy as np
import pytest

import oracle_sigma as OS

pytestmark = pytest.mark.gpu

TINY = dict(nso=(4, 1, 2, 3), nalpha=3, nbeta=1, seed=3)
C2V24 = dict(nso=(11, 2, 4, 7), nalpha=6, nbeta=4, seed=1)
SMALL_D2H = dict(nso=(5, 2, 3, 3, 4, 1, 2, 2), nalpha=5, nbeta=3, seed=5)
SMALL = dict(nso=(6, 2, 3, 5), nalpha=4, nbeta=2, seed=7)
INPUTS = {"sf-cis": ("eorb", "iabj"), "cisdoo": ("eorb", "iabj", "ijka", "abij", "abci"),
          "sf-cpsd": ("eorb", "iabj", "ijka", "ijkl", "abij", "abci", "abcd")}


@pytest.fixture(scope="module")
def torch():
    import torch as t
    assert t.cuda.is_available()
    return t


def make(cfg, method, symR):
    import dpdhip
    from test_gpu_sigma import ctx, oracle_problem
    sp, op = oracle_problem(cfg, method, symR)
    gp = dpdhip.Problem(ctx(len(cfg["nso"])), sp, method, symR)
    return sp, op, gp


@pytest.mark.parametrize("method", ["sf-cis", "cisdoo", "sf-cpsd"])
def test_sigma_t_is_dense_transpose(torch, method):
    sp, op, gp = make(TINY, method, 1)
    n = gp.dim
    print(f"[adjoint] dense transpose {method} dim={n}", flush=True)
    J = np.zeros((n, n))
    for k in range(n):
        e = np.zeros(n)
        e[k] = 1.0
        J[:, k] = op.sigma(e)
    rng = np.random.default_rng(1)
    Y = rng.standard_normal((3, n))
    T = gp.sigma_t(torch.tensor(Y.ravel(), device="cuda:0")).cpu().numpy().reshape(3, n)
    ref = Y @ J
    np.testing.assert_allclose(T, ref, rtol=0, atol=1e-12 * np.abs(ref).max())


@pytest.mark.parametrize("cfg,symR", [(C2V24, 1), (C2V24, 2), (SMALL_D2H, 1), (SMALL_D2H, 5)],
                         ids=["c2v-A1", "c2v-A2", "d2h-Ag", "d2h-B1u"])
@pytest.mark.parametrize("method", ["sf-cis", "cisdoo", "sf-cpsd"])
def test_adjoint_identity(torch, cfg, symR, method):
    import dpdhip
    from test_gpu_sigma import ctx
    sp = dpdhip.Spec(cfg["nso"], cfg["nalpha"], cfg["nbeta"], cfg["seed"])
    gp = dpdhip.Problem(ctx(len(cfg["nso"])), sp, method, symR)
    n = gp.dim
    print(f"[adjoint] identity {method} {cfg['nso']} symR={symR} dim={n}", flush=True)
    g = torch.Generator(device="cuda:0").manual_seed(5)
    X = torch.randn(4 * n, dtype=torch.float64, device="cuda:0", generator=g)
    Y = torch.randn(4 * n, dtype=torch.float64, device="cuda:0", generator=g)
    JX = gp.sigma(X).view(4, n)
    JtY = gp.sigma_t(Y).view(4, n)
    a = (Y.view(4, n) * JX).sum(1)
    b = (X.view(4, n) * JtY).sum(1)
    scale = Y.view(4, n).norm(dim=1) * JX.norm(dim=1)
    assert torch.all((a - b).abs() <= 1e-13 * scale), (a, b)


def _oracle_f(op, eorb, ints, L, R):
    """L . J(theta) R with the oracle's sigma at inputs theta"""
    o2 = OS.OracleProblem(op.sym, op.popo, op.popv, op.popa, op.popb, op.vrta, op.vrtb, eorb, ints, op.method,
                          op.symR)
    return float(L @ o2.sigma(R))


@pytest.mark.parametrize("method", ["sf-cis", "cisdoo", "sf-cpsd"])
def test_grad_matches_oracle_difference(torch, method):
    cfg, symR = SMALL, 2
    sp, op, gp = make(cfg, method, symR)
    n = gp.dim
    print(f"[adjoint] grad vs oracle difference {method} dim={n}", flush=True)
    rng = np.random.default_rng(11)
    L = rng.standard_normal(n)
    R = rng.standard_normal(n)
    g = gp.grad(torch.tensor(L, device="cuda:0"), torch.tensor(R, device="cuda:0"))
    base = {k: gp.get(k).cpu().numpy() for k in INPUTS[method]}
    h = 1e-5
    for name in INPUTS[method]:
        d = rng.standard_normal(base[name].size)
        d /= np.linalg.norm(d)
        vals = []
        for s in (1.0, -1.0):
            x = dict(base)
            x[name] = base[name] + s * h * d
            ints = {k: v for k, v in x.items() if k != "eorb"}
            vals.append(_oracle_f(op, x["eorb"], _full_ints(op, ints), L, R))
        fd = (vals[0] - vals[1]) / (2 * h)
        an = float(g[name].cpu().numpy() @ d)
        assert abs(fd - an) <= 1e-6 * max(1.0, abs(an)), (name, fd, an)


def _full_ints(op, ints):
    out = dict(op.ints)
    out.update(ints)
    return out


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_eigenvalue_gradient_matches_difference(torch, prec):
    import dpdhip
    from dpdhip.gradient import excitation_energy
    from test_gpu_sigma import ctx
    cfg = SMALL
    sp = dpdhip.Spec(cfg["nso"], cfg["nalpha"], cfg["nbeta"], cfg["seed"])
    gp = dpdhip.Problem(ctx(len(cfg["nso"])), sp, "sf-cpsd", 1)
    print(f"[adjoint] eigenvalue gradient {prec} dim={gp.dim}", flush=True)
    names = INPUTS["sf-cpsd"]
    base = {k: gp.get(k) for k in names}
    x = {k: v.clone().requires_grad_(True) for k, v in base.items()}
    solve = dict(nroot=2, conv=1e-10, max_dim=24, max_cyc=200)
    info = {}
    w = excitation_energy(gp, x, info=info, **solve)
    w.backward()
    grad = {k: x[k].grad.clone() for k in names}
    assert info["right"]["converged"] and info["left"]["converged"]
    assert abs(info["w_left"] - float(w.detach())) < 1e-9
    assert abs(info["w_right"] - float(w.detach())) < 1e-9
    # central differences of the FP64 eigenvalue along random directions
    gen = torch.Generator(device="cuda:0").manual_seed(3)
    h = 1e-4
    # spin-allowed elements only: a spin-forbidden one couples other sectors
    dirs = {k: torch.randn(v.numel(), dtype=torch.float64, device="cuda:0", generator=gen) * (v != 0)
            for k, v in base.items()}
    nrm = sum(float(d.norm() ** 2) for d in dirs.values()) ** 0.5
    dirs = {k: d / nrm for k, d in dirs.items()}
    if prec == "fp64":
        vals = []
        for s in (1.0, -1.0):
            xs = {k: base[k] + s * h * dirs[k] for k in names}
            vals.append(float(excitation_energy(gp, xs, **solve)))
        fd = (vals[0] - vals[1]) / (2 * h)
        an = sum(float(grad[k] @ dirs[k]) for k in names)
        assert abs(fd - an) <= 1e-6 * max(1.0, abs(an)), (fd, an)
        test_eigenvalue_gradient_matches_difference.ref = grad
    else:
        ref = getattr(test_eigenvalue_gradient_matches_difference, "ref", None)
        if ref is None:
            pytest.skip("needs the fp64 case first")
        gp.set_precision("fp32")
        try:
            x = {k: v.clone().requires_grad_(True) for k, v in base.items()}
            w32 = excitation_energy(gp, x, **dict(solve, conv=1e-5))
            w32.backward()
        finally:
            gp.set_precision("fp64")
        num = sum(float((x[k].grad - ref[k]).norm() ** 2) for k in names) ** 0.5
        den = sum(float(ref[k].norm() ** 2) for k in names) ** 0.5
        assert num <= 1e-3 * den, (num, den)


def test_set_requires_refresh(torch):
    import dpdhip
    from test_gpu_sigma import ctx
    sp = dpdhip.Spec(TINY["nso"], TINY["nalpha"], TINY["nbeta"], TINY["seed"])
    gp = dpdhip.Problem(ctx(4), sp, "sf-cpsd", 1)
    x = gp.get("abij")
    y0 = gp.sigma(torch.ones(gp.dim, dtype=torch.float64, device="cuda:0"))
    gp.set("abij", x)
    with pytest.raises(dpdhip.DpdError):
        gp.sigma(torch.ones(gp.dim, dtype=torch.float64, device="cuda:0"))
    with pytest.raises(dpdhip.DpdError):
        gp.set("mp2t", gp.get("mp2t"))
    gp.refresh()
    y1 = gp.sigma(torch.ones(gp.dim, dtype=torch.float64, device="cuda:0"))
    # the intermediates are recomputed (possibly with another autotuned tile, so
    # another summation order): equal to rounding
    assert float((y0 - y1).abs().max()) <= 1e-13 * float(y0.abs().max())


def test_interleaved_forwards_one_backward(torch):
    """Two forwards on the same problem with different inputs, then backward
    of the first: the gradient is evaluated at the first forward's inputs (the
    problem is re-set and refreshed), equal to a lone forward + backward."""
    import dpdhip
    from dpdhip.gradient import excitation_energy
    from test_gpu_sigma import ctx
    cfg = SMALL
    gp = dpdhip.Problem(ctx(len(cfg["nso"])), dpdhip.Spec(cfg["nso"], cfg["nalpha"], cfg["nbeta"], cfg["seed"]),
                        "sf-cpsd", 1)
    print(f"[adjoint] interleaved forwards dim={gp.dim}", flush=True)
    names = INPUTS["sf-cpsd"]
    base = {k: gp.get(k) for k in names}
    solve = dict(nroot=2, conv=1e-10, max_dim=24, max_cyc=200)
    x = {k: v.clone().requires_grad_(True) for k, v in base.items()}
    excitation_energy(gp, x, **solve).backward()
    ref = {k: x[k].grad.clone() for k in names}
    x1 = {k: v.clone().requires_grad_(True) for k, v in base.items()}
    w1 = excitation_energy(gp, x1, **solve)
    other = {k: (v * 1.05).requires_grad_(True) for k, v in base.items()}
    excitation_energy(gp, other, **solve)
    w1.backward()
    for k in names:
        err = float((x1[k].grad - ref[k]).abs().max())
        assert err <= 1e-8 * max(1.0, float(ref[k].abs().max())), (k, err)


@pytest.mark.timeout(300)
def test_gradient_c2v_100_orbitals_50_directions(torch):
    """The gradient workload at full size (C2v, 100 spatial orbitals [40,10,20,30],
    n_alpha=10, n_beta=8, dim 637 003): the FP64 eigenvalue gradient against
    central differences (h = 1e-4) of the eigenvalue along 50 seeded random unit
    directions over the spin-allowed integral elements and 5 in the orbital
    energies; FP32 and BF16x3 gradients within 1e-3 of FP64."""
    import dpdhip
    from dpdhip.gradient import excitation_energy
    ctx = dpdhip.Context(4, 0)
    gp = dpdhip.Problem(ctx, dpdhip.Spec((40, 10, 20, 30), 10, 8, 5), "sf-cpsd", 1)
    names = gp.INPUTS
    base = {k: gp.get(k) for k in names}
    solve = dict(nroot=1, conv=1e-9, max_dim=40, max_cyc=300)

    def run(x0, prec="fp64", conv=1e-9, warm=None):
        gp.set_precision(prec)
        x = {k: x0[k].clone().requires_grad_(True) for k in names}
        info = {}
        extra = {"R0": warm["R"], "L0": warm["L"]} if warm else {}
        w = excitation_energy(gp, x, info=info, **dict(solve, conv=conv), **extra)
        w.backward()
        return float(w.detach()), {k: x[k].grad for k in names}, info

    print(f"[adjoint] c2v-100 gradient dim={gp.dim}", flush=True)
    w0, g0, info = run(base)
    gn_eri = sum(float(g0[k].norm() ** 2) for k in names if k != "eorb") ** 0.5
    gen = torch.Generator(device="cuda:0").manual_seed(2024)
    h = 1e-4
    worst = 0.0
    for i in range(55):
        keys = ["eorb"] if i >= 50 else [k for k in names if k != "eorb"]
        d = {k: torch.randn(base[k].numel(), dtype=torch.float64, device="cuda:0", generator=gen) * (base[k] != 0)
             for k in keys}
        nrm = sum(float(v.norm() ** 2) for v in d.values()) ** 0.5
        vals = []
        for s in (1.0, -1.0):
            xs = {k: (base[k] + s * h * d[k] / nrm) if k in d else base[k] for k in names}
            vals.append(run(xs, warm=info)[0])
        fd = (vals[0] - vals[1]) / (2 * h)
        an = sum(float(g0[k] @ d[k]) for k in keys) / nrm
        worst = max(worst, abs(fd - an) / gn_eri)
        assert abs(fd - an) <= 1e-8 * gn_eri, (i, fd, an)
    print(f"[adjoint] worst |fd - analytic| / |grad| = {worst:.2e}", flush=True)
    den = sum(float(g0[k].norm() ** 2) for k in names) ** 0.5
    for prec in ("fp32", "bf16x3"):
        try:
            _, g, _ = run(base, prec, 1e-5)
        finally:
            gp.set_precision("fp64")
        err = sum(float((g[k] - g0[k]).norm() ** 2) for k in names) ** 0.5
        assert err <= 1e-3 * den, (prec, err, den)


@pytest.mark.parametrize("cfg,symR", [(TINY, 1), (C2V24, 1), (C2V24, 3), (SMALL_D2H, 1), (SMALL_D2H, 6),
                                      (dict(nso=(25, 4, 1, 9), nalpha=5, nbeta=3, seed=4), 2)],
                         ids=["tiny", "c2v-A1", "c2v-B1", "d2h-Ag", "d2h-B2u", "c2v-39"])
@pytest.mark.parametrize("method", ["sf-cis", "cisdoo"])
def test_orbital_energy_gradient_sums(torch, method, cfg, symR):
    """The orbital-energy part of the gradient is a sum over stored elements: with
    vectors of one excitation rank only (singles for SF-CIS, doubles for CIS(Doo),
    whose MP2 chain then vanishes), eorb_bar[p] = sum over the elements that hold p
    of +-scale*L*R.  Column lengths here lie below, at no multiple of and above the
    64 left pairs that a block of the reduction takes."""
    import oracle as O
    sp, op, gp = make(cfg, method, symR)
    print(f"[adjoint] orbital-energy sums {method} {cfg['nso']} symR={symR} dim={gp.dim}", flush=True)
    lay = sp.layout()
    n = len(cfg["nso"])
    O.Sym(n).activate()
    s = O.Sym(n)
    v, o = lay["popv"], lay["popo"]
    l1 = op.l1
    rng = np.random.default_rng(3)
    L, R = rng.standard_normal(gp.dim), rng.standard_normal(gp.dim)
    no = int(o.sum())
    ref, bound, count = np.zeros(no + int(v.sum())), np.zeros(no + int(v.sum())), np.zeros(no + int(v.sum()))
    if method == "sf-cis":
        a, i, _, _ = O.dpd_index(s, op.dR1)
        dims, w = ((no + a, 1.0), (i, -1.0)), 0.7 * L * R
    else:
        L[:l1] = R[:l1] = 0.0
        a, b, i, j = O.dpd_index(s, op.dR2)
        dims, w = ((no + a, 1.0), (no + b, 1.0), (i, -1.0), (j, -1.0)), 0.7 * L[l1:] * R[l1:]
    for at, sign in dims:
        np.add.at(ref, at, sign * w)
        np.add.at(bound, at, np.abs(w))
        np.add.at(count, at, 1.0)
    got = gp.grad(torch.tensor(L, device="cuda:0"), torch.tensor(R, device="cuda:0"), scale=0.7)["eorb"].cpu().numpy()
    # each sum of m terms is within (m + 2) 2^-53 of sum |w| of the exact one, on both sides
    assert np.all(np.abs(got - ref) <= 2 * (count + 2) * 2.0 ** -53 * bound + 1e-300), np.abs(got - ref).max()
