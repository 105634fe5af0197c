"""GPU parity of the HIP engine against the CPU oracle (same seeded inputs).

Covers the MFMA lane layout, the engine level (vv2v_dpd_444/424/442 fast paths,
fallback and scrambles, accumulation), the mod_contract surface with its
expand/antisymmetrise/compress semantics, every sort kernel and the Davidson
vector primitives.  FP64 tolerance: relative 1e-11 (only the summation order
differs from the oracle's BLAS)."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

RTOL, ATOL = 1e-11, 1e-12

PV = np.array([3, 1, 2, 2, 0, 0, 0, 0])
PO = np.array([2, 1, 0, 1, 0, 0, 0, 0])
PV8 = np.array([2, 1, 1, 2, 1, 0, 1, 1])
PO8 = np.array([1, 1, 0, 1, 1, 0, 0, 1])
# larger spaces so that tiles, split-K and several K segments are exercised
PVL = np.array([21, 9, 14, 17, 0, 0, 0, 0])
POL = np.array([4, 2, 3, 3, 0, 0, 0, 0])


@pytest.fixture(scope="module")
def torch():
    import torch as t
    assert t.cuda.is_available(), "GPU tests need a HIP device"
    return t


_ctxs = {}


def ctx_for(n):
    import dpdhip
    if n not in _ctxs:
        _ctxs[n] = dpdhip.Context(n, 0)
    return _ctxs[n]


# GEMM kernels (tile configuration, packing): automatic (timed) and automatic
# (cost model); first-generation
# kernel; gathering kernel with 64x64 / 128x64 / 64x128 / 128x128 tiles; the
# packed-panel kernel with automatic and with each fixed tile shape (7 names the tile of 2)
GEMM_CFGS = [(-1, 1), (-2, 1), (0, 0), (1, 0), (2, 0), (3, 0), (4, 0), (5, 0), (-1, 2), (1, 2), (2, 2), (3, 2),
             (4, 2), (5, 2), (6, 2), (7, 2)]
GEMM_IDS = ["auto", "model", "v1", "g64x64", "g128x64", "g64x128", "g128x128", "g32x32", "pk_auto", "pk64x64",
            "pk128x64", "pk64x128", "pk128x128", "pk32x32", "pk64x192", "pk128x64-7"]


@pytest.fixture(params=GEMM_CFGS, ids=GEMM_IDS)
def gemm_cfg(request, torch):
    cfg, packing = request.param
    for n in (4, 8):
        ctx_for(n).set_gemm_config(cfg, packing)
    yield request.param
    for n in (4, 8):
        ctx_for(n).set_gemm_config(-1, 1)


@pytest.fixture(params=[4, 8], ids=["c2v", "d2h"])
def sym(request, torch):
    s = O.Sym(request.param)
    s.activate()
    return s


def spaces(sym, large=False):
    if sym.nirrep == 4:
        return (PVL, POL) if large else (PV, PO)
    return PV8, PO8


def dev(torch, x):
    return torch.from_numpy(np.ascontiguousarray(x)).to("cuda:0")


def gopt(torch, sym, desc, x):
    import dpdhip
    arr = dev(torch, np.concatenate([x, [0.0]]))
    return dpdhip.Opt(ctx_for(sym.nirrep), *desc.pops, ioppq=desc.iop[0], ioprs=desc.iop[1], sym=desc.sym, arr=arr)


def test_mfma_lane_layout_single_tile(torch, sym):
    """A 16x16x4 block: the smallest GEMM, checks the MFMA operand/result layout."""
    s = sym
    p = np.zeros(8, np.int64)
    p[0] = 16
    k = np.zeros(8, np.int64)
    k[0] = 4
    d1 = O.Desc([p, k, O.ZORB, O.ZORB], (1, 1), 1)
    d2 = O.Desc([k, p, O.ZORB, O.ZORB], (1, 1), 1)
    d3 = O.Desc([p, p, O.ZORB, O.ZORB], (1, 1), 1)
    rng = np.random.default_rng(0)
    a = rng.standard_normal(64)
    b = rng.standard_normal(64)
    g1, g2, g3 = gopt(torch, s, d1, a), gopt(torch, s, d2, b), gopt(torch, s, d3, np.zeros(256))
    import dpdhip
    dpdhip.vv2v_222(g1, g2, g3, 1.0, "ik", "kj", "ij")
    got = g3.numpy().reshape(16, 16, order="F")
    exp = a.reshape(16, 4, order="F") @ b.reshape(4, 16, order="F")
    np.testing.assert_allclose(got, exp, rtol=1e-13, atol=1e-13)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("shape", [(16, 16, 4, "N", "N"), (70, 45, 37, "N", "N"), (65, 130, 100, "T", "N"),
                                   (33, 64, 17, "N", "T"), (128, 20, 300, "T", "T"),
                                   (257, 190, 129, "T", "N")])
def test_xgemm_layout_and_transposes(torch, prec, shape, gemm_cfg):
    """dense GEMM through the same MFMA kernel: pins the FP64 and FP32 MFMA operand
    and result layouts directly (one 16x16x4 tile first, then ragged tiles)."""
    import dpdhip
    m, n, k, ta, tb = shape
    rng = np.random.default_rng(m * 7 + n)
    A = rng.standard_normal((m, k) if ta == "N" else (k, m))
    B = rng.standard_normal((k, n) if tb == "N" else (n, k))
    C = rng.standard_normal((m, n))
    opA = A if ta == "N" else A.T
    opB = B if tb == "N" else B.T
    if prec == "fp32":
        exp = 1.5 * (opA.astype(np.float32).astype(np.float64) @ opB.astype(np.float32).astype(np.float64)) - 0.5 * C
        tol = dict(rtol=2e-5, atol=2e-5 * np.sqrt(k))
    else:
        exp = 1.5 * (opA @ opB) - 0.5 * C
        tol = dict(rtol=1e-13, atol=1e-13 * k)
    gA = dev(torch, A.flatten(order="F"))
    gB = dev(torch, B.flatten(order="F"))
    gC = dev(torch, C.flatten(order="F"))
    dpdhip.xgemm(ctx_for(4), ta, tb, m, n, k, 1.5, gA, A.shape[0], gB, B.shape[0], -0.5, gC, m, prec)
    got = gC.cpu().numpy().reshape(m, n, order="F")
    np.testing.assert_allclose(got, exp, **tol)


@pytest.mark.parametrize("shape", [(16, 16, 32, "N", "N"), (70, 45, 37, "N", "N"), (65, 130, 100, "T", "N"),
                                   (257, 190, 129, "T", "N"), (128, 20, 300, "T", "T")])
def test_xgemm_bf16x3(torch, shape, gemm_cfg):
    """BF16x3 MFMA path: matches hi*hi + hi*lo + lo*hi of the emulated split to
    FP32-accumulation accuracy, and the exact product to the split's accuracy."""
    import dpdhip
    if gemm_cfg[1] != 2 and gemm_cfg != (-1, 1):
        pytest.skip("BF16x3 always runs the packed kernel")
    m, n, k, ta, tb = shape
    rng = np.random.default_rng(m * 11 + k)
    A = rng.standard_normal((m, k) if ta == "N" else (k, m))
    B = rng.standard_normal((k, n) if tb == "N" else (n, k))
    C = rng.standard_normal((m, n))
    opA = A if ta == "N" else A.T
    opB = B if tb == "N" else B.T
    from bf16_emulation import bf16x3_split
    ah, al = bf16x3_split(opA)
    bh, bl = bf16x3_split(opB)
    emu = 1.5 * (ah @ bh + ah @ bl + al @ bh) - 0.5 * C
    gA = dev(torch, A.flatten(order="F"))
    gB = dev(torch, B.flatten(order="F"))
    gC = dev(torch, C.flatten(order="F"))
    dpdhip.xgemm(ctx_for(4), ta, tb, m, n, k, 1.5, gA, A.shape[0], gB, B.shape[0], -0.5, gC, m, "bf16x3")
    got = gC.cpu().numpy().reshape(m, n, order="F")
    mag = 1.5 * (np.abs(opA) @ np.abs(opB))
    # FP32 accumulation of the three products: at most k roundings of 2^-24
    assert np.all(np.abs(got - emu) <= max(k, 32) * 2.0 ** -24 * mag + 1e-12), np.abs(got - emu).max()
    exact = 1.5 * (opA @ opB) - 0.5 * C
    assert np.all(np.abs(got - exact) <= 3 * 2.0 ** -16 * mag + 1e-12)


def _engine_case(torch, sym, kind, pops, iops, syms, t1, t2, t3, f1=1.0, f2=0.0, seed=0):
    import dpdhip
    rng = np.random.default_rng(seed)
    d1 = O.Desc(pops[0], iops[0], syms[0])
    d2 = O.Desc(pops[1], iops[1], syms[1])
    d3 = O.Desc(pops[2], iops[2], syms[2])
    x1, x2, x3 = O.random_dpd(sym, d1, rng), O.random_dpd(sym, d2, rng), O.random_dpd(sym, d3, rng)
    ref = x3.copy()
    {444: O.vv2v_dpd_444, 424: O.vv2v_dpd_424, 442: O.vv2v_dpd_442}[kind](x1, d1, t1, x2, d2, t2, ref, d3, t3, f1, f2)
    g1, g2, g3 = gopt(torch, sym, d1, x1), gopt(torch, sym, d2, x2), gopt(torch, sym, d3, x3)
    {444: dpdhip.vv2v_dpd_444, 424: dpdhip.vv2v_dpd_424, 442: dpdhip.vv2v_dpd_442}[kind](g1, t1, g2, t2, g3, t3, f1,
                                                                                        f2)
    np.testing.assert_allclose(g3.numpy(), ref, rtol=RTOL, atol=ATOL)


def test_engine_fast_paths(torch, sym, gemm_cfg):
    for large in (False, True):
        if large and sym.nirrep == 8:
            continue
        V, Oc = spaces(sym, large)
        _engine_case(torch, sym, 444, [[V, V, V, V], [V, V, Oc, Oc], [V, V, Oc, Oc]], [(0, 0)] * 3, (1, 2, 2),
                     "abef", "efij", "abij")
        _engine_case(torch, sym, 444, [[V, V, Oc, Oc], [V, V, Oc, Oc], [Oc, Oc, Oc, Oc]], [(0, 0)] * 3, (1, 1, 1),
                     "efij", "efkl", "ijkl", f2=0.5)
        _engine_case(torch, sym, 444, [[V, V, Oc, Oc], [V, V, Oc, Oc], [V, V, V, V]], [(0, 0)] * 3, (3, 3, 1),
                     "abmn", "cdmn", "abcd")
        _engine_case(torch, sym, 444, [[Oc, Oc, V, V], [V, V, Oc, Oc], [V, V, V, V]], [(1, 1)] * 3, (2, 2, 1),
                     "mnab", "cdmn", "abcd", f2=0.5)


def test_engine_fallback_and_scrambles(torch, sym, gemm_cfg):
    V, Oc = spaces(sym)
    full = [(1, 1)] * 3
    _engine_case(torch, sym, 444, [[V, V, Oc, Oc]] * 3, full, (1, 2, 2), "aeim", "ebmj", "abij")
    _engine_case(torch, sym, 444, [[V, V, Oc, Oc]] * 3, full, (2, 1, 2), "eaim", "ebmj", "abij", f2=0.5)
    _engine_case(torch, sym, 444, [[Oc, V, V, Oc], [V, V, Oc, Oc], [Oc, V, Oc, V]], full, (1, 3, 3), "faeb", "iejf",
                 "baji", f2=0.5)
    _engine_case(torch, sym, 444, [[V, Oc, V, Oc], [V, Oc, V, Oc], [V, V, V, V]], full, (2, 3, 4), "pmqn", "rmsn",
                 "prqs")


def test_engine_errors(torch, sym):
    import dpdhip
    V, Oc = spaces(sym)
    d1 = O.Desc([V, V, Oc, Oc], (1, 1), 1)
    d2 = O.Desc([V, V, Oc, Oc], (0, 0), 1)
    g1 = gopt(torch, sym, d1, np.zeros(d1.length()))
    g2 = gopt(torch, sym, d2, np.zeros(d2.length()))
    with pytest.raises(dpdhip.DpdError) as e:
        dpdhip.vv2v_dpd_444(g1, "aeim", g2, "ebmj", g2, "abij", 1.0, 0.0)
    assert e.value.code == -4  # IOP barrier of the fallback
    d3 = O.Desc([V, Oc, V, Oc], (1, 1), 1)
    g3 = gopt(torch, sym, d3, np.zeros(d3.length()))
    with pytest.raises(dpdhip.DpdError) as e:
        dpdhip.vv2v_dpd_444(g3, "aeim", g1, "ebmj", g1, "abij", 1.0, 0.0)
    assert e.value.code == -3  # contracted populations differ
    with pytest.raises(dpdhip.DpdError):
        dpdhip.vv2v_444(g2, g2, g2, 1.0, "abef", "efij", "abij", 4)


def _surface_case(torch, sym, kind, ops, t, fact, anti, seed=1):
    import dpdhip
    rng = np.random.default_rng(seed)
    d1, d2, d3 = ops
    x1, x2, x3 = O.random_dpd(sym, d1, rng), O.random_dpd(sym, d2, rng), O.random_dpd(sym, d3, rng)
    v3 = O.Opt(d3, x3.copy())
    t1, t2, t3 = t
    fo = {"444": O.vv2v_444, "424": O.vv2v_424, "442": O.vv2v_442, "222": O.vv2v_222, "422": O.vv2v_422,
          "224": O.vv2v_224}[kind]
    fg = {"444": dpdhip.vv2v_444, "424": dpdhip.vv2v_424, "442": dpdhip.vv2v_442, "222": dpdhip.vv2v_222,
          "422": dpdhip.vv2v_422, "224": dpdhip.vv2v_224}[kind]
    extra = (anti,) if kind in ("444", "424", "224") else ()
    fo(O.Opt(d1, x1), O.Opt(d2, x2), v3, fact, t1, t2, t3, *extra)
    g3 = gopt(torch, sym, d3, x3)
    fg(gopt(torch, sym, d1, x1), gopt(torch, sym, d2, x2), g3, fact, t1, t2, t3, *extra)
    np.testing.assert_allclose(g3.numpy(), v3.arr, rtol=RTOL, atol=ATOL, err_msg=f"{kind} {t}")


@pytest.mark.parametrize("large", [False, True], ids=["small", "large"])
def test_contract_surface_sigma_calls(torch, sym, large, gemm_cfg):
    if large and sym.nirrep == 8:
        pytest.skip("large spaces are C2v only")
    V, Oc = spaces(sym, large)
    Z = O.ZORB
    for S in (1, 2):
        r1 = O.Desc([V, Oc, Z, Z], (1, 1), S)
        r2 = O.Desc([V, V, Oc, Oc], (0, 0), S)
        fab = O.Desc([V, V, Z, Z], (1, 1), 1)
        fij = O.Desc([Oc, Oc, Z, Z], (1, 1), 1)
        iabj = O.Desc([V, Oc, V, Oc], (1, 1), 1)
        abci = O.Desc([V, V, V, Oc], (0, 1), 1)
        ijka = O.Desc([Oc, Oc, Oc, V], (0, 1), 1)
        ijkl = O.Desc([Oc, Oc, Oc, Oc], (0, 0), 1)
        abcd = O.Desc([V, V, V, V], (0, 0), 1)
        _surface_case(torch, sym, "222", (fab, r1, r1), ("ae", "ei", "ai"), 1.0, 0)
        _surface_case(torch, sym, "222", (r1, fij, r1), ("am", "mi", "ai"), -1.0, 0)
        _surface_case(torch, sym, "422", (iabj, r1, r1), ("fnai", "fn", "ai"), 1.0, 0)
        _surface_case(torch, sym, "442", (abci, r2, r1), ("feam", "feim", "ai"), 1.0, 0)
        _surface_case(torch, sym, "442", (r2, ijka, r1), ("aemn", "mnie", "ai"), -1.0, 0)
        _surface_case(torch, sym, "424", (abci, r1, r2), ("abej", "ei", "abij"), 1.0, 2)
        _surface_case(torch, sym, "424", (ijka, r1, r2), ("ijmb", "am", "abij"), -1.0, 1)
        _surface_case(torch, sym, "444", (abcd, r2, r2), ("abef", "efij", "abij"), 1.0, 0)
        _surface_case(torch, sym, "444", (r2, ijkl, r2), ("abmn", "mnij", "abij"), 1.0, 0)
        _surface_case(torch, sym, "444", (r2, iabj, r2), ("aeim", "embj", "abij"), 1.0, 3)
    t2 = O.Desc([V, V, Oc, Oc], (0, 0), 1)
    fab = O.Desc([V, V, Z, Z], (1, 1), 1)
    fij = O.Desc([Oc, Oc, Z, Z], (1, 1), 1)
    iabj = O.Desc([V, Oc, V, Oc], (1, 1), 1)
    _surface_case(torch, sym, "442", (t2, t2, fab), ("afmn", "efmn", "ae"), -1.0, 0)
    _surface_case(torch, sym, "442", (t2, t2, fij), ("efmn", "efin", "mi"), 1.0, 0)
    _surface_case(torch, sym, "444", (t2, t2, iabj), ("fenm", "bfjn", "embj"), 1.0, 0)


def test_contract_surface_224(torch, sym):
    """mod_contract.f90:203-219 (vv2v_224): two 2-index tensors into a 4-index
    one, r1(a,i) r1(b,j) -> c2(ab,ij) with every antisymmetriser, and
    f(a,b) t(i,j) -> x(ab,ij) into a packed and an unpacked output"""
    V, Oc = spaces(sym, False)
    Z = O.ZORB
    for S1, S2 in ((1, 1), (2, 3)):
        S3 = O.xor_dirprd(sym.nirrep)[S1 - 1][S2 - 1]
        r1a = O.Desc([V, Oc, Z, Z], (1, 1), S1)
        r1b = O.Desc([V, Oc, Z, Z], (1, 1), S2)
        for anti, iop in ((0, 1), (1, 1), (2, 1), (3, 0), (3, 1)):
            c2 = O.Desc([V, V, Oc, Oc], (iop, iop), S3)
            _surface_case(torch, sym, "224", (r1a, r1b, c2), ("ai", "bj", "abij"), 0.5, anti)
        fab = O.Desc([V, V, Z, Z], (1, 1), S1)
        tij = O.Desc([Oc, Oc, Z, Z], (1, 1), S2)
        x = O.Desc([V, V, Oc, Oc], (1, 1), S3)
        _surface_case(torch, sym, "224", (fab, tij, x), ("ab", "ij", "abij"), -1.25, 0)


def test_engine_323(torch, sym):
    """vv2v_dpd_323 (libsrint/vv2v_dpd_323.f90) on the seven cases of its harness
    (vv2v_dpd_323_check.f90:98-280) against the oracle, and its error codes"""
    import dpdhip
    from test_oracle_engine import _cases323, _desc3
    V, Oc = spaces(sym, False)
    for case, (t1, p1, t2, p2, t3, p3, iop, f2) in enumerate(_cases323(V, Oc)):
        for s1, s2 in ((1, 1), (2, 3)):
            s3 = O.xor_dirprd(sym.nirrep)[s1 - 1][s2 - 1]
            rng = np.random.default_rng(case * 10 + s1)
            d1 = _desc3(p1, iop if t1 == "pqm" else 1, s1)
            d2 = O.desc2(p2[0], p2[1], 1, s2)
            d3 = _desc3(p3, iop if t3 == "pqr" else 1, s3)
            x1, x2, x3 = (O.random_dpd(sym, d, rng) for d in (d1, d2, d3))
            ref = x3.copy()
            O.vv2v_dpd_323(x1, d1, t1, x2, d2, t2, ref, d3, t3, 1.5, f2)
            g1, g2, g3 = gopt(torch, sym, d1, x1), gopt(torch, sym, d2, x2), gopt(torch, sym, d3, x3)
            dpdhip.vv2v_dpd_323(g1, t1, g2, t2, g3, t3, 1.5, f2)
            np.testing.assert_allclose(g3.numpy(), ref, rtol=RTOL, atol=ATOL, err_msg=f"case {case}")
    d1 = _desc3((V, Oc, Oc), 1, 1)
    d2 = O.desc2(Oc, V, 1, 1)
    d3 = _desc3((V, Oc, V), 1, 1)
    g1, g2, g3 = (gopt(torch, sym, d, np.zeros(d.length())) for d in (d1, d2, d3))
    with pytest.raises(dpdhip.DpdError):  # the contracted index kept in v3
        dpdhip.vv2v_dpd_323(g1, "pqm", g2, "mr", g3, "pqm", 1.0, 0.0)
    gp = gopt(torch, sym, O.desc2(Oc, V, 0, 1), np.zeros(O.desc2(Oc, V, 0, 1).length()))
    with pytest.raises(dpdhip.DpdError):  # v2 packed
        dpdhip.vv2v_dpd_323(g1, "pqm", gp, "mr", g3, "pqr", 1.0, 0.0)


def test_sort_kernels(torch, sym):
    import dpdhip
    c = ctx_for(sym.nirrep)
    V, Oc = spaces(sym)
    rng = np.random.default_rng(3)
    for irrepx in range(1, sym.nirrep + 1):
        d0 = O.Desc([V, V, Oc, Oc], (0, 0), irrepx)
        x = O.random_dpd(sym, d0, rng)
        for iexp in [(1, 0), (0, 1), (1, 1)]:
            ref = O.iexpso(x, V, V, 0, iexp[0], Oc, Oc, 0, iexp[1], irrepx)
            out = torch.zeros(len(ref) + 1, dtype=torch.float64, device="cuda:0")
            dpdhip.iexpso(c, dev(torch, x), out, V, V, 0, iexp[0], Oc, Oc, 0, iexp[1], irrepx)
            assert np.array_equal(out[: len(ref)].cpu().numpy(), ref)
        full = O.iexpso(x, V, V, 0, 1, Oc, Oc, 0, 0, irrepx)
        ref = O.icompso(full, V, V, 1, 0, Oc, Oc, 0, 1, irrepx)
        out = torch.zeros(len(ref) + 1, dtype=torch.float64, device="cuda:0")
        dpdhip.icompso(c, dev(torch, full), out, V, V, 1, 0, Oc, Oc, 0, 1, irrepx)
        assert np.array_equal(out[: len(ref)].cpu().numpy(), ref)
        d1 = O.Desc([V, Oc, V, Oc], (1, 1), irrepx)
        y = rng.standard_normal(d1.length())
        for icpq, icrs in [(1, 0), (0, 1), (1, 1)]:
            ref = O.isymtrso(y, V, Oc, 1, icpq, V, Oc, 1, icrs, irrepx)
            out = torch.zeros(len(y) + 1, dtype=torch.float64, device="cuda:0")
            dpdhip.isymtrso(c, dev(torch, y), out, V, Oc, 1, icpq, V, Oc, 1, icrs, irrepx)
            assert np.array_equal(out[: len(y)].cpu().numpy(), ref)
        ref = O.itranspso(y, V, Oc, 1, V, Oc, 1, irrepx)
        out = torch.zeros(len(y) + 1, dtype=torch.float64, device="cuda:0")
        dpdhip.itranspso(c, dev(torch, y), out, V, Oc, 1, V, Oc, 1, irrepx)
        assert np.array_equal(out[: len(y)].cpu().numpy(), ref)
        io = {0: (0, 1), 1: (1, 1), 2: (1, 1), 3: (1, 1), 4: (1, 0), 5: (1, 1)}
        for iop in range(6):
            di = O.Desc([V, V, Oc, Oc], io[iop], irrepx)
            z = O.random_dpd(sym, di, rng)
            ref = O.iassymso(z, irrepx, V, V, Oc, Oc, iop)
            out = torch.zeros(len(ref) + 1, dtype=torch.float64, device="cuda:0")
            dpdhip.iassymso(c, dev(torch, z), out, irrepx, V, V, Oc, Oc, iop)
            assert np.array_equal(out[: len(ref)].cpu().numpy(), ref), iop
        for t in ("3142", "2413", "4321", "1243"):
            ref = O.sstgenso(y, V, Oc, V, Oc, irrepx, t)
            out = torch.zeros(len(y) + 1, dtype=torch.float64, device="cuda:0")
            dpdhip.sstgenso(c, dev(torch, y), out, V, Oc, V, Oc, irrepx, t)
            assert np.array_equal(out[: len(y)].cpu().numpy(), ref)


def test_vector_primitives(torch):
    import dpdhip
    c = ctx_for(4)
    rng = np.random.default_rng(9)
    for n in (1, 7, 1000, 300001):
        x = rng.standard_normal(n)
        y = rng.standard_normal(n)
        gx, gy = dev(torch, x), dev(torch, y)
        assert dpdhip.dot(c, gx, gy) == pytest.approx(float(x @ y), rel=1e-12, abs=1e-12)
        assert dpdhip.nrm2(c, gx) == pytest.approx(float(np.linalg.norm(x)), rel=1e-12)
        # idamax: first index of the max |x|, 1-based
        x2 = x.copy()
        k = n // 2
        x2[k] = 10.0
        if n > 3:
            x2[n - 1] = -10.0
        i, v = dpdhip.amax(c, dev(torch, x2))
        assert i == k + 1 and v == 10.0
        dpdhip.axpy(c, -0.5, gx, gy)
        np.testing.assert_allclose(gy.cpu().numpy(), y - 0.5 * x, rtol=1e-15)
        dpdhip.scal(c, 3.0, gx)
        np.testing.assert_allclose(gx.cpu().numpy(), 3.0 * x, rtol=1e-15)
    # preconditioner with the 1e-4 clamp (mod_davidson.f90:417-428)
    d = np.array([1.0, 2.0, 0.50005, 0.49999, 3.0])
    e = np.array([1.0, 1.0, 1.0, 1.0, 2.0])
    p = torch.zeros(5, dtype=torch.float64, device="cuda:0")
    dpdhip.precondition(c, 0.5, dev(torch, d), dev(torch, e), p)
    exp = e / np.array([0.5 - 1.0, 0.5 - 2.0, -1e-4, 1e-4, 0.5 - 3.0])
    np.testing.assert_allclose(p.cpu().numpy(), exp, rtol=1e-15)


# sizes over which the estimate's choice of the packed-panel configuration goes through most of
# them: tile edges, remainders of 16 and of a K step, one K step only, fewer and more steps than
# the waves that share them (every configuration: test_every_panel_shape)
FR_SIZES = [(1, 1, 1), (5, 1, 3), (5, 1, 65), (16, 31, 2999), (17, 17, 65), (63, 97, 17), (65, 190, 600), (250, 250, 130),
            (5, 161, 3000), (250, 321, 97), (1000, 81, 97), (1000, 129, 130), (1000, 190, 130), (1000, 190, 33),
            (2999, 81, 33), (2999, 161, 33), (2999, 321, 33), (2999, 600, 33), (6001, 33, 33), (6001, 65, 33),
            (6001, 97, 33), (6001, 161, 33), (6001, 250, 33), (9001, 81, 33), (9001, 97, 33), (9001, 145, 33),
            (9001, 250, 3), (17001, 1, 3), (17001, 17, 33), (17001, 33, 33), (17001, 65, 33), (17001, 81, 33),
            (17001, 97, 33), (17001, 129, 33)]


@pytest.mark.parametrize("prec", ["fp64", "fp32", "bf16x3"])
@pytest.mark.parametrize("shape", FR_SIZES)
def test_xgemm_packed_shapes(torch, prec, shape):
    import dpdhip
    from bf16_emulation import bf16x3_split
    m, n, k = shape
    ctx = ctx_for(4)
    rng = np.random.default_rng(m + 3 * n + 5 * k)
    A, B, C = rng.standard_normal((m, k)), rng.standard_normal((k, n)), rng.standard_normal((m, n))
    g = [dev(torch, x.flatten(order="F")) for x in (A, B, C)]
    print(f"[engine] packed shapes {prec} {shape}", flush=True)
    ctx.set_gemm_config(-2, 2)
    try:
        dpdhip.xgemm(ctx, "N", "N", m, n, k, 1.5, g[0], m, g[1], k, -0.5, g[2], m, prec)
    finally:
        ctx.set_gemm_config(-1, 1)
    got = g[2].cpu().numpy().reshape(m, n, order="F")
    mag = 1.5 * (np.abs(A) @ np.abs(B)) + 0.5 * np.abs(C)
    exp = 1.5 * (A @ B) - 0.5 * C
    if prec == "fp64":  # k products and sums, two more roundings, on both sides
        bound = 2 * (k + 4) * 2.0 ** -53 * mag
    elif prec == "fp32":  # both operands rounded, then k roundings of the sum
        bound = (k + 4) * 2.0 ** -24 * mag
    else:  # the split loses 3 x 2^-16 of a product; k roundings of the FP32 sum
        (ah, al), (bh, bl) = bf16x3_split(A), bf16x3_split(B)
        exp = 1.5 * (ah @ bh + ah @ bl + al @ bh) - 0.5 * C
        bound = max(k, 32) * 2.0 ** -24 * mag
    assert np.all(np.abs(got - exp) <= bound + 1e-15), np.abs(got - exp).max()


# kFrShapes: rows and columns of every tile of the packed-panel kernel (0 is not one)
FR_TILES = [None, (64, 64), (128, 64), (64, 128), (128, 128), (32, 32), (64, 192), (128, 64), (64, 16), (128, 16), (64, 32),
            (128, 32), (64, 48), (128, 48), (64, 80), (128, 80), (64, 96), (128, 96), (64, 160), (128, 160), (16, 16),
            (32, 16), (16, 32)]


def test_panel_shapes_all_named(torch):
    from dpdhip import _lib
    L, h = _lib.lib(), ctx_for(4).h
    assert L.dpd_ctx_request_shape(h, len(FR_TILES) - 1, 0) == 0
    assert L.dpd_ctx_request_shape(h, len(FR_TILES), 0) != 0 and L.dpd_ctx_request_shape(h, 0, 0) != 0
    ctx_for(4).set_gemm_config(-1, 1)


@pytest.mark.parametrize("prec", ["fp64", "fp32", "bf16x3"])
@pytest.mark.parametrize("shape", range(1, len(FR_TILES)), ids=lambda i: "%dx%d" % FR_TILES[i] if i != 7 else "128x64d")
def test_every_panel_shape(torch, prec, shape):
    """every tile of the packed-panel kernel, with and without split-K, accumulating and not: one
    element, one less and one more than a tile, several tiles and the K steps of the unrolled loop's
    start, end and steady part"""
    import dpdhip
    from bf16_emulation import bf16x3_split
    from dpdhip import _lib
    bm, bn = FR_TILES[shape]
    ctx = ctx_for(4)
    print(f"[engine] panel shape {bm}x{bn} {prec}", flush=True)
    try:
        _lib.check(_lib.lib().dpd_ctx_request_shape(ctx.h, shape, 0))
        for m, n, k in ((1, 1, 1), (bm - 1, bn + 1, 17), (bm + 1, bn - 1, 33), (2 * bm + 5, 2 * bn + 3, 130),
                        (bm, bn, 1199), (bm + 15, 16, 3001)):
            rng = np.random.default_rng(m + 3 * n + 5 * k)
            A, B, C = rng.standard_normal((m, k)), rng.standard_normal((k, n)), rng.standard_normal((m, n))
            (ah, al), (bh, bl) = bf16x3_split(A), bf16x3_split(B)
            prod = ah @ bh + ah @ bl + al @ bh if prec == "bf16x3" else A @ B
            mag = 1.5 * (np.abs(A) @ np.abs(B)) + 0.5 * np.abs(C)
            # as in test_xgemm_packed_shapes
            bound = {"fp64": 2 * (k + 4) * 2.0 ** -53, "fp32": (k + 4) * 2.0 ** -24,
                     "bf16x3": max(k, 32) * 2.0 ** -24}[prec] * mag + 1e-15
            for split in (0, 1):
                ctx.set_split_k(split)
                for beta in (0.0, -0.5):
                    g = [dev(torch, x.flatten(order="F")) for x in (A, B, C)]
                    dpdhip.xgemm(ctx, "N", "N", m, n, k, 1.5, g[0], m, g[1], k, beta, g[2], m, prec)
                    got = g[2].cpu().numpy().reshape(m, n, order="F")
                    assert np.all(np.abs(got - 1.5 * prod - beta * C) <= bound), (m, n, k, split, beta)
    finally:
        ctx.set_split_k(-1)
        ctx.set_gemm_config(-1, 1)


@pytest.mark.parametrize("split", [0, 1])
def test_every_shape_beside_an_operand_in_place(torch, split):
    """every tile of the product that reads its row operand where it lies: one K segment and one K
    digit (pp-ladder), several segments and two K digits (c1_r2abci), ragged rows, columns and K's"""
    import dpdhip
    from dpdhip import _lib
    L = _lib.lib()
    pad = lambda p: np.array(list(p) + [0] * (8 - len(p)))
    cases = []
    for n, V, Oc, S, kind in ((1, [67], [5], 1, "444"), (2, [70, 61], [4, 3], 2, "442"), (4, [31, 20, 17, 25], [3, 1, 0, 2], 3, "444")):
        s = O.Sym(n)
        s.activate()
        V, Oc, Z = pad(V), pad(Oc), O.ZORB
        r1, r2 = O.Desc([V, Oc, Z, Z], (1, 1), S), O.Desc([V, V, Oc, Oc], (0, 0), S)
        if kind == "444":
            d, t = (O.Desc([V, V, V, V], (0, 0), 1), r2, r2), ("abef", "efij", "abij")
        else:
            d, t = (O.Desc([V, V, V, Oc], (0, 1), 1), r2, r1), ("feam", "feim", "ai")
        rng = np.random.default_rng(n)
        x = [O.random_dpd(s, q, rng) for q in d]
        o3 = O.Opt(d[2], x[2].copy())
        args = (O.Opt(d[0], x[0]), O.Opt(d[1], x[1]), o3, 1.0, *t)
        O.vv2v_444(*args, 0) if kind == "444" else O.vv2v_442(*args)
        cases.append((s, d, t, x, o3.arr, kind, [gopt(torch, s, q, y) for q, y in zip(d, x)]))
    shapes = [i for i in range(1, len(FR_TILES)) if L.dpd_ctx_request_shape(ctx_for(4).h, i, 1) == 0]
    assert len(shapes) == 16
    try:
        for shape in shapes:
            print(f"[engine] in place {FR_TILES[shape]} split={split}", flush=True)
            for s, d, t, x, ref, kind, g in cases:
                c = ctx_for(s.nirrep)
                s.activate()
                _lib.check(L.dpd_ctx_request_shape(c.h, shape, 1))
                c.set_split_k(split)
                g[2].arr[: len(x[2])] = dev(torch, x[2])
                dpdhip.vv2v_444(*g, 1.0, *t, 0) if kind == "444" else dpdhip.vv2v_442(*g, 1.0, *t)
                assert L.dpd_ctx_pack_code_bytes(c.h) > 0  # one side is packed
                # normal inputs: K products, partial sums of sqrt(K), so K roundings of 2^-53 sqrt(K)
                # add up to K 2^-53 in quadrature, on both sides; 16 of that
                K = 2300 if kind == "444" else 32_000
                assert abs(g[2].numpy() - ref).max() <= 16 * K * 2.0 ** -53, (FR_TILES[shape], kind)
    finally:
        for n in (1, 2, 4):
            ctx_for(n).set_split_k(-1)
            ctx_for(n).set_gemm_config(-1, 1)


@pytest.mark.parametrize("cfg", [1, 2, 4, 5, 6])
def test_fp32_sums_in_two_levels(torch, cfg):
    """k equal products: a single FP32 sum drifts with k (2^-24 per addition, all of one sign);
    two-level sums stay within the additions of one level plus those of the next: 256 k's and what
    is left at the end (96), or, in the 32x32 tile (5) whose four waves share the k's, 768 and 160,
    and one addition for each of those"""
    import dpdhip
    m, n, k = 37, 33, 200_003
    steps = cfg == 5
    bound = ((768 + 160 + k / 3072 if steps else 256 + 96 + k / 256) + 16) * 2.0 ** -24
    # one level, by element or by the four k's of an MFMA, is outside of that
    for per in (1, 4):
        one = np.cumsum(np.full(k // (4 * per if steps else per), per * np.float32(0.1), np.float32), dtype=np.float32)
        assert abs(one[-1] / (len(one) * float(per * np.float32(0.1))) - 1) > 1.5 * bound
    ctx = ctx_for(4)
    A, B, C = (torch.full((s,), x, dtype=torch.float64, device="cuda:0")
               for s, x in ((m * k, 0.1), (k * n, 1.0), (m * n, 0.0)))
    print(f"[engine] two-level sums cfg {cfg}", flush=True)
    ctx.set_gemm_config(cfg, 2)
    ctx.set_split_k(0)
    try:
        dpdhip.xgemm(ctx, "N", "N", m, n, k, 1.0, A, m, B, k, 0.0, C, m, "fp32")
    finally:
        ctx.set_gemm_config(-1, 1)
        ctx.set_split_k(-1)
    exp = k * float(np.float32(0.1))
    err = abs(C.cpu().numpy() / exp - 1).max()
    print(f"[engine] two-level sums cfg {cfg}: {err:.2e} of {bound:.2e}", flush=True)
    assert err <= bound


@pytest.mark.parametrize("nirrep,V,Oc,terms", [
    (1, [67], [5], "pp"), (1, [91], [6], "abci c1abci"), (4, [31, 20, 17, 25], [3, 1, 0, 2], "pp"),
    (4, [57, 41, 37, 44], [3, 1, 0, 2], "abci c1abci"), (8, [17, 9, 21, 16, 1, 19, 18, 20], [2, 1, 0, 1, 1, 0, 1, 1], "pp"),
    (2, [70, 61], [4, 3], "pp abci c1abci")], ids=["c1-pp", "c1-abci", "c2v-pp", "c2v-abci", "d2h-pp", "cs"])
def test_large_operand_read_where_it_lies(torch, nirrep, V, Oc, terms):
    """contractions whose row operand has 2^21 elements or more and is used a few times: read
    from the tensor by the GEMM (rows along its unit stride, K along it, one and two K digits,
    ragged rows and K's, several K segments) against the oracle; engine level with fact2 too"""
    import dpdhip
    from dpdhip import _lib
    ctx = ctx_for(nirrep)
    ctx.set_gemm_config(-1, 1)  # no plan is left
    codes = lambda: _lib.lib().dpd_ctx_pack_code_bytes(ctx.h)
    s = O.Sym(nirrep)
    s.activate()
    pad = lambda p: np.array(list(p) + [0] * (8 - len(p)))
    V, Oc, Z = pad(V), pad(Oc), O.ZORB
    for S in sorted({1, min(2, nirrep), nirrep}):
        r1, r2 = O.Desc([V, Oc, Z, Z], (1, 1), S), O.Desc([V, V, Oc, Oc], (0, 0), S)
        abci, abcd = O.Desc([V, V, V, Oc], (0, 1), 1), O.Desc([V, V, V, V], (0, 0), 1)
        print(f"[engine] large operand {nirrep} {terms} S={S}", flush=True)
        for term in terms.split():
            before = codes()
            if term == "pp":
                _surface_case(torch, s, "444", (abcd, r2, r2), ("abef", "efij", "abij"), 1.0, 0)
            elif term == "c1abci":
                _surface_case(torch, s, "442", (abci, r2, r1), ("feam", "feim", "ai"), 1.0, 0)
            else:
                _surface_case(torch, s, "424", (abci, r1, r2), ("abej", "ei", "abij"), 1.0, 2)
            assert codes() > before  # the other operand was packed: not the gathering kernel
        if "pp" in terms:
            before = codes()
            rng = np.random.default_rng(S)
            x1, x2, x3 = (O.random_dpd(s, d, rng) for d in (abcd, r2, r2))
            ref = x3.copy()
            O.vv2v_dpd_444(x1, abcd, "abef", x2, r2, "efij", ref, r2, "abij", 1.5, 0.5)
            g = [gopt(torch, s, d, x) for d, x in ((abcd, x1), (r2, x2), (r2, x3))]
            dpdhip.vv2v_dpd_444(g[0], "abef", g[1], "efij", g[2], "abij", 1.5, 0.5)
            assert codes() > before
            np.testing.assert_allclose(g[2].numpy(), ref, rtol=RTOL, atol=ATOL)


def _packed_product(torch, term):
    """a per-call FP64 product that is packed: a regrouped ring, an expanded operand beside a large
    one in place, an engine call; its inputs, result and a call that returns the result"""
    import dpdhip
    s = O.Sym(4)
    s.activate()
    V, Oc = (np.array([53, 37, 33, 40] + [0] * 4), np.array([3, 1, 0, 2] + [0] * 4)) if term == "c1abci" else \
        (PVL, np.array([5, 3, 4, 4] + [0] * 4))
    r2 = O.Desc([V, V, Oc, Oc], (0, 0), 2)
    W, f2 = O.Desc([V, Oc, V, Oc], (1, 1), 1), O.Desc([V, Oc, V, Oc], (1, 1), 2)
    abci, r1 = O.Desc([V, V, V, Oc], (0, 1), 1), O.Desc([V, Oc, O.ZORB, O.ZORB], (1, 1), 2)
    d = {"ring": (r2, W, r2), "c1abci": (abci, r2, r1), "engine": (W, f2, f2)}[term]
    t = {"ring": ("aeim", "embj", "abij"), "c1abci": ("feam", "feim", "ai"), "engine": ("aiem", "embj", "aibj")}[term]
    rng = np.random.default_rng(5)
    x = [O.random_dpd(s, q, rng) for q in d]
    ref = x[2].copy()
    if term == "engine":
        O.vv2v_dpd_444(x[0], d[0], t[0], x[1], d[1], t[1], ref, d[2], t[2], 1.5, 0.5)
    else:
        o3 = O.Opt(d[2], ref)
        (O.vv2v_444(O.Opt(d[0], x[0]), O.Opt(d[1], x[1]), o3, 1.0, *t, 3) if term == "ring" else
         O.vv2v_442(O.Opt(d[0], x[0]), O.Opt(d[1], x[1]), o3, 1.0, *t))
        ref = o3.arr

    def call(c):
        g = [dpdhip.Opt(c, *q.pops, ioppq=q.iop[0], ioprs=q.iop[1], sym=q.sym, arr=dev(torch, np.concatenate([v, [0.0]])))
             for q, v in zip(d, x)]
        if term == "engine":
            dpdhip.vv2v_dpd_444(g[0], t[0], g[1], t[1], g[2], t[2], 1.5, 0.5)
        elif term == "ring":
            dpdhip.vv2v_444(*g, 1.0, *t, 3)
        else:
            dpdhip.vv2v_442(*g, 1.0, *t)
        return g[2].numpy()
    return ref, call


@pytest.mark.parametrize("term", ["ring", "c1abci", "engine"])
def test_products_without_room_for_pack_codes(torch, term):
    """per-call FP64 products that are packed: where the codes of their panels do not fit, the call
    runs without them, to the same bits, and takes them up again once there is room"""
    import dpdhip
    from dpdhip import _lib
    L = _lib.lib()
    ref, call = _packed_product(torch, term)
    c = dpdhip.Context(4, 0)
    got = []
    for limit in (0, 0, 1 << 40, 0):
        print(f"[engine] pack codes {term} limit={limit}", flush=True)
        _lib.check(L.dpd_ctx_set_pack_code_limit(c.h, limit))
        got.append(call(c))
        assert (L.dpd_ctx_pack_code_bytes(c.h) > 0) == (len(got) > 2)  # kept once they are there
    c.set_gemm_config(-1, 1)
    assert L.dpd_ctx_pack_code_bytes(c.h) == 0
    np.testing.assert_allclose(got[0], ref, rtol=RTOL, atol=ATOL)
    for q in got[1:]:
        assert np.array_equal(q, got[0])
    c.close()


@pytest.mark.parametrize("term", ["c1abci", "engine"])
def test_products_without_room_for_panels(torch, term):
    """two of them (the ring's split-K sums take more than its panels) where the workspace has room
    for what the gathering kernel needs and not for panels: they run on that kernel, and on panels
    once there is room"""
    import dpdhip
    from dpdhip import _lib
    L = _lib.lib()
    ref, call = _packed_product(torch, term)
    c = dpdhip.Context(4, 0)
    limit, done = 1 << 16, 0
    while not done:
        _lib.check(L.dpd_ctx_set_workspace_limit(c.h, limit))
        try:
            got = call(c)
            done = 1
        except dpdhip.DpdError as e:
            assert e.code == -5, e  # out of memory, nothing else
            limit = limit * 9 // 8
            assert limit < 1 << 30
    print(f"[engine] no room for panels {term}: {limit} bytes do", flush=True)
    assert L.dpd_ctx_pack_code_bytes(c.h) == 0  # nothing was packed
    np.testing.assert_allclose(got, ref, rtol=RTOL, atol=ATOL)
    _lib.check(L.dpd_ctx_set_workspace_limit(c.h, -1))
    np.testing.assert_allclose(call(c), ref, rtol=RTOL, atol=ATOL)
    assert L.dpd_ctx_pack_code_bytes(c.h) > 0
    c.close()


def test_pack_codes_stay_within_their_limit(torch):
    """the panel codes that a context keeps for per-call products of ever new shapes stay within the
    limit, and go with the plans"""
    import dpdhip
    from dpdhip import _lib
    L = _lib.lib()
    O.Sym(4).activate()
    c = dpdhip.Context(4, 0)
    rng = np.random.default_rng(6)
    seen = []
    for limit in (-1, 3 << 20):
        _lib.check(L.dpd_ctx_set_pack_code_limit(c.h, limit))
        assert L.dpd_ctx_pack_code_bytes(c.h) == 0
        for n in range(5):
            V, Oc = np.array([21 + n, 9, 14, 17, 0, 0, 0, 0]), np.array([5, 3, 4, 4, 0, 0, 0, 0])
            d = O.Desc([V, Oc, V, Oc], (1, 1), 1)
            x = [O.random_dpd(O.Sym(4), d, rng) for _ in range(2)]
            g = [dpdhip.Opt(c, *d.pops, ioppq=1, ioprs=1, sym=1, arr=dev(torch, y)) for y in (*x, 0 * x[0])]
            print(f"[engine] pack code limit {limit} shape {n}", flush=True)
            dpdhip.vv2v_dpd_444(g[0], "aiem", g[1], "embj", g[2], "aibj", 1.0, 0.0)
            ref = np.zeros(d.length())
            O.vv2v_dpd_444(x[0], d, "aiem", x[1], d, "embj", ref, d, "aibj", 1.0, 0.0)
            np.testing.assert_allclose(g[2].numpy(), ref, rtol=RTOL, atol=ATOL)
            seen.append(L.dpd_ctx_pack_code_bytes(c.h))
        c.set_gemm_config(-1, 1)
    assert all(np.diff(seen[:5]) > 0) and seen[4] > 3 << 20  # every shape keeps its own
    assert 0 < seen[5] <= max(seen[5:]) <= 3 << 20 and seen[9] == seen[8]
    c.close()


def test_calls_on_alternating_streams(torch):
    """a context whose stream changes between calls: they share its workspace (here the panels of
    per-call products of several sizes), so each starts after the one before it"""
    import dpdhip
    s = O.Sym(4)
    s.activate()
    c = dpdhip.Context(4, 0)
    rng = np.random.default_rng(8)
    jobs = []
    for n in range(3):
        V, Oc = np.array([21 + 7 * n, 9, 14, 17 + n, 0, 0, 0, 0]), np.array([5, 3, 4, 4, 0, 0, 0, 0])
        d = O.Desc([V, Oc, V, Oc], (1, 1), 1)
        g = [dpdhip.Opt(c, *d.pops, ioppq=1, ioprs=1, sym=1, arr=dev(torch, O.random_dpd(s, d, rng))) for _ in range(3)]
        dpdhip.vv2v_dpd_444(g[0], "aiem", g[1], "embj", g[2], "aibj", 1.0, 0.0)
        torch.cuda.synchronize()
        jobs.append((g, g[2].arr.clone()))
    streams = [torch.cuda.Stream() for _ in range(2)]
    print("[engine] alternating streams", flush=True)
    for g, _ in jobs:
        g[2].arr.zero_()
    torch.cuda.synchronize()
    for rep in range(30):
        for i, (g, _) in enumerate(jobs):
            with torch.cuda.stream(streams[(rep + i) % 2]):
                c.use_current_stream()
                dpdhip.vv2v_dpd_444(g[0], "aiem", g[1], "embj", g[2], "aibj", 1.0, 0.0)
        if rep % 10 == 9:
            torch.cuda.synchronize()
            for g, ref in jobs:
                assert torch.equal(g[2].arr, ref)
                g[2].arr.zero_()
            torch.cuda.synchronize()
    c.use_current_stream()
    c.close()
