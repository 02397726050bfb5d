"""Edges of tiles and dispatch of the GPU kernels against the oracle: the
smallest and largest sizes of a kernel's range and sizes that leave
remainders in its tiles.  Tolerances are derived at each test."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
from test_oracle import _si_case  # noqa: E402

pytestmark = pytest.mark.gpu


def rel(a, b):
    a, b = np.ravel(a), np.ravel(b)
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


@pytest.mark.parametrize("ntru,nlev", [(1, 1), (5, 16), (21, 17), (42, 33), (10, 64)])
@pytest.mark.parametrize("dtype", ["float64", "float32"])
def test_si_apply_edges(oracle, gpu, ntru, nlev, dtype):
    """one level, whole and ragged groups of 16 levels and of 16 spectral
    reals, the largest level count.  FP64 arithmetic on both sides from the
    same bm1: sums of nlev <= 64 terms in the same order differ only by FMA
    contraction, a few 1e-16 per term of terms that cancel by less than 1e2,
    below 1e-12; FP32 arrays add the rounding of the results, 6e-8."""
    import torch

    from exoplasim_amd.semi_implicit import SemiImplicit

    print(f"si_apply T{ntru} L{nlev} {dtype}", flush=True)
    c = _si_case(ntru, nlev, seed=ntru + nlev)
    si = SemiImplicit(nlev, ntru, c["t0"], c["dsigma"], c["g"], c["tau"])
    si.makebm(c["delt"])
    dt = getattr(torch, dtype)
    names = ("sop", "spm", "atm", "adm", "stt", "sdt", "spt")
    t = {k: torch.from_numpy(np.ascontiguousarray(c[k])).to("cuda", dt) for k in names}
    host = {k: t[k].double().cpu().numpy() for k in names}
    si.apply(c["delt"], *[t[k] for k in names])
    torch.cuda.synchronize()
    want = oracle.si_apply(ntru, nlev, c["delt"], c["t0"], c["dsigma"], c["g"], c["tau"],
                           si.bm1(), *[host[k] for k in names])
    for k, w in zip(("stt", "sdt", "spt"), want):
        assert rel(t[k].double().cpu().numpy(), w) < (1e-12 if dtype == "float64" else 1e-6), k
    si.close()


@pytest.mark.parametrize("ntru,nlev", [(21, 1), (42, 8), (63, 9), (63, 17), (127, 3)])
@pytest.mark.parametrize("mode", ["f64", "f32"])
def test_direct_sums_edges(oracle, gpu, ntru, nlev, mode):
    """mktend, uv2dv and qtend where the 8 levels of a block are one, whole
    and one over, on three members, and the last wavenumber range of T42
    and T63 is ragged or full.  Random inputs: sums of <= 3 * 96 terms of
    equal size, rounding below sqrt(288) eps / 2 of the result: 1e-12 and 1e-6
    leave two orders and a half."""
    import torch

    from exoplasim_amd import sht

    print(f"direct sums T{ntru} L{nlev} {mode}", flush=True)
    p = sht.Plan(ntru)
    tab, one, nm = oracle.legini(ntru, p.nlat), np.ones(ntru + 1), 3
    rng = np.random.default_rng(ntru + nlev)
    f = [rng.standard_normal((nm, nlev, p.nlat, p.nlon)) for _ in range(6)]
    dt = p.dtype_of(mode)
    fd = [torch.from_numpy(x).to("cuda", dt) for x in f]
    out = [torch.full((nm, nlev, p.nrsp), float("nan"), dtype=dt, device="cuda")
           for _ in range(6)]
    p.mktend(mode, *out[:3], *fd, nlev)
    p.uv2dv(mode, fd[0], fd[1], out[3], out[4], nlev)
    p.qtend(mode, out[5], *fd[:3], nlev)
    got = [x.double().cpu().numpy() for x in out]
    a = (ntru, p.nlat, p.nlon, nlev)
    for k in range(nm):
        x = [y[k] for y in f]
        want = [*oracle.mktend(*a, tab["qc"], tab["qe"], tab["qm"], tab["qq"], one, *x),
                *oracle.uv2dv(*a, tab["qe"], tab["qm"], one, x[0], x[1]),
                oracle.qtend(*a, tab["qc"], tab["qe"], tab["qm"], one, *x[:3])]
        for i, w in enumerate(want):
            assert rel(got[i][k], w) < (1e-12 if mode == "f64" else 1e-6), (i, k)
    p.close()


sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden"))
from make_golden import (PLASIM_SCAL, gridpointa_humidity, gridpointa_state,  # noqa: E402
                         plasim_inputs)

CT = (6371220.0 * 7.292e-5) ** 2 / 287.0


def _vertical(oracle, nlev):
    return oracle.vertical(nlev, t0=np.linspace(220.0, 288.0, nlev) / CT)


def _gphi(f, v, nq):
    """the geopotential term in the form without the cancellation of (gt + t0)
    (1 + a) - t0 - gt, a = (1/rdbrv - 1) q of 1e-4 to 1e-3, which costs the
    oracle's form a factor 1 / a in rounding (up to 1e-12, and 1.35e-12 in the
    divergence tendency of T127 through the Laplacian)"""
    q = f["gq"] / f["gp"] if nq else f["dq"]
    corr = (f["gt"] + v["t0"][:, None]) * (1.0 / PLASIM_SCAL[0] - 1.0) * np.maximum(q, 0.0)
    return 2.0 / f["rcsq"] * (v["g"].T @ corr)


@pytest.mark.parametrize("nlev,nhor", [(2, 1), (3, 64), (7, 65), (9, 127), (64, 200)])
@pytest.mark.parametrize("mode", ["f64", "f32"])
def test_calcgp_edges(oracle, gpu, nlev, nhor, mode):
    """fewer levels than a block's waves, one more, the largest count; fewer
    points than a block, whole and one over.  Tolerances as for the other
    level counts: 1e-12 in FP64, 2e-5 in FP32 (the geopotential and sigma-dot
    sums cancel to about 1/20 of their terms)."""
    import torch

    from exoplasim_amd.dynamics import CALCGP_OUT, PRODUCTS, Dynamics

    print(f"calcgp L{nlev} x{nhor} {mode}", flush=True)
    v = _vertical(oracle, nlev)
    dyn = Dynamics.from_vertical(v, *PLASIM_SCAL)
    dt = torch.float64 if mode == "f64" else torch.float32
    f = {k: x[..., :nhor].copy() for k, x in plasim_inputs(nlev, 256, 5)[1].items()}
    if mode == "f32":
        f = {k: x.astype(np.float32).astype(np.float64) for k, x in f.items()}
    dev = {k: torch.from_numpy(np.ascontiguousarray(x)).to("cuda", dt) for k, x in f.items()}
    for k in CALCGP_OUT + PRODUCTS:
        dev[k] = torch.full((nlev, nhor), float("nan"), dtype=dt, device="cuda")
    dev["gvp"] = torch.full((nhor,), float("nan"), dtype=dt, device="cuda")
    dyn.calcgp(mode, dev, nqspec=1)
    got = {k: x.double().cpu().numpy() for k, x in dev.items()}
    want = oracle.calcgp(f, v, PLASIM_SCAL, 1)
    want["gphi"] = _gphi(f, v, 1)
    want.update(gut=f["gu"] * f["gt"], gvt=f["gv"] * f["gt"], guq=f["gu"] * f["gq"],
                gvq=f["gv"] * f["gq"], gke=f["gu"] ** 2 + f["gv"] ** 2 + want["gphi"])
    for k, w in want.items():
        assert rel(got[k], w) < (1e-12 if mode == "f64" else 2e-5), k
    dyn.close()


@pytest.mark.parametrize("ntru,nlev,mode", [(21, 2, "f64"), (21, 9, "f32"), (42, 7, "f64"),
                                            (42, 41, "f64"), (42, 33, "bf16x3"), (63, 5, "f32"),
                                            (127, 3, "f64")])
@pytest.mark.parametrize("nq", [1, 0])
def test_gridpointa_edges(oracle, gpu, ntru, nlev, mode, nq):
    """level counts around a block's 8 waves; rows transformed inside calcgp
    and outside it (FP64 above L40 at T42, T63, T127), three members.  The
    tendencies at 1e-12 in FP64 and 2e-5 in the FP32 modes, as for the other
    sizes; the Fourier fields of the work array too, from the oracle's grid
    fields through its gp2fc."""
    import torch

    from exoplasim_amd import sht
    from exoplasim_amd.dynamics import Dynamics, work_slots

    print(f"gridpointa T{ntru} L{nlev} {mode} nqspec={nq}", flush=True)
    tol = 1e-12 if mode == "f64" else 2e-5
    v = _vertical(oracle, nlev)
    plan, dyn = sht.Plan(ntru), Dynamics.from_vertical(v, *PLASIM_SCAL)
    st, work, tend = dyn.alloc_gridpointa(plan, 3, mode)
    nlat, nlon, sl = plan.nlat, plan.nlon, work_slots(nlev)
    states = [gridpointa_state(ntru, nlev, 0.9 + 0.1 * k) for k in range(3)]
    st.copy_(torch.from_numpy(np.stack(states)).to(st.dtype))
    hum = gridpointa_humidity(nlev, nlat * nlon)
    if nq == 0:
        for k, x in zip(("gq", "dq"), hum):
            work[:, sl[k]:sl[k] + nlev] = torch.from_numpy(
                x.reshape(nlev, nlat, nlon)).to("cuda", work.dtype)
    dyn.gridpointa(plan, mode, st, work, tend, nqspec=nq)
    got, wk = tend.double().cpu().numpy(), work.double().cpu().numpy()
    cast = (lambda x: x) if mode == "f64" else (lambda x: x.astype(np.float32).astype(np.float64))
    for k in (0, 2):
        want, f = oracle.gridpointa(ntru, nlev, cast(states[k]), v, PLASIM_SCAL, nq,
                                    gq=cast(hum[0]), dq=cast(hum[1]))
        f["gphi"] = _gphi(f, v, nq)
        f["gke"] = f["gu"] ** 2 + f["gv"] ** 2 + f["gphi"]
        tab, one = oracle.legini(ntru, nlat), np.ones(ntru + 1)
        four = {x: oracle.gp2fc(f[x].reshape(-1, nlat, nlon), nlon == 192)
                for x in ("gtn", "gvz", "guz", "gke", "gut", "gvt")}
        want[nlev:2 * nlev] = oracle.mktend(
            ntru, nlat, nlon, nlev, tab["qc"], tab["qe"], tab["qm"], tab["qq"], one,
            *[four[x] for x in ("gtn", "gvz", "guz", "gke", "gut", "gvt")])[0]
        for i in range(4 if nq else 3):
            s = slice(i * nlev, (i + 1) * nlev)
            assert rel(got[k, s], want[s]) < tol, (k, i)
        assert rel(got[k, 4 * nlev], want[4 * nlev]) < tol, k
        for name in ("gtn", "gqn", "guz", "gvz", "gut", "gvt", "gke", "gvp") + (
                ("guq", "gvq") if nq else ()):
            rows = f[name].reshape(-1, nlat, nlon)
            w = oracle.gp2fc(rows, nlon == 192)
            assert rel(wk[k, sl[name]:sl[name] + len(rows)], w) < tol, (k, name)
        for name in ("gphi", "dw", "gp", "rcsq"):
            w = f[name].reshape(-1, nlat, nlon)
            assert rel(wk[k, sl[name]:sl[name] + len(w)], w) < tol, (k, name)
    dyn.close()
    plan.close()


@pytest.mark.parametrize("nlev,ncol", [(2, 1), (5, 9), (7, 300), (31, 17), (32, 5), (63, 33)])
@pytest.mark.parametrize("fp64", [True, False])
def test_lwr_edges(oracle, gpu, nlev, ncol, fp64):
    """level counts whose pairs of levels leave lanes with short, empty or
    several-row runs, the last of 32 lanes and the first and last of 64, and
    ragged blocks of columns.  FP64 at the bar of the other lwr tests (1e-10:
    the layer emission cancels to 2e-11 of the flux where a transmissivity is
    clamped).  FP32: flux sums of up to 63 terms of about 400 W/m2 round at
    2.4e-5 each, layer differences of 0.1 W/m2 and more: 1e-3 of the heating,
    1e-4 of the OLR."""
    import torch

    import oracle as O
    from exoplasim_amd.radiation import LwrColumn, sigma_levels

    print(f"lwr L{nlev} x{ncol} fp64={fp64}", flush=True)
    rng = np.random.default_rng(nlev)
    s = sigma_levels(nlev)[0]
    t = 190.0 + 110.0 * np.sqrt(s) + rng.uniform(-2, 2, (ncol, nlev))
    cols = {"dt": np.concatenate([t, t[:, -1:] + rng.uniform(1, 5, (ncol, 1))], axis=1),
            "dq": np.exp(rng.uniform(np.log(1e-5), np.log(2e-2), (ncol, nlev))),
            "dp": rng.uniform(5e4, 1.5e5, ncol),
            "dqco2": np.repeat(np.exp(rng.uniform(3, 9, (ncol, 1))), nlev, axis=1),
            "dqo3": 1e-6 * rng.random((ncol, nlev)), "dcc": 0.5 * rng.random((ncol, nlev)),
            "dql": 1e-5 * rng.random((ncol, nlev)), "dls": (rng.random(ncol) < 0.5) * 1.0}
    dt = torch.float64 if fp64 else torch.float32
    dev = {k: torch.from_numpy(np.ascontiguousarray(x.T)).to("cuda", dt) for k, x in cols.items()}
    heat, olr, fu, fd = LwrColumn(nlev, fp64=fp64)(dev, fluxes=True)
    host = {k: np.ascontiguousarray(x.double().cpu().numpy().T) for k, x in dev.items()}
    wu, wd, wh, wo = O.lwr(oracle, host, nlev)
    tol = (1e-10, 1e-10) if fp64 else (1e-3, 1e-4)
    assert rel(heat.double().cpu().numpy(), wh.T * 86400.0) < tol[0]
    assert rel(olr.double().cpu().numpy(), wo) < tol[1]
    assert rel(fu.double().cpu().numpy(), wu.T) < tol[1]
    assert rel(fd.double().cpu().numpy(), wd.T) < tol[1]


@pytest.mark.parametrize("ntru,nlev,nmem", [(21, 5, 1), (21, 20, 40), (42, 10, 2), (42, 10, 5),
                                            (63, 7, 1), (63, 5, 4), (127, 6, 1), (127, 5, 3)])
@pytest.mark.parametrize("mode", ["f64", "f32", "bf16x3"])
def test_untuned_tiles(oracle, gpu, ntru, nlev, nmem, mode):
    """a plan that was not tuned chooses its tiles by the size of the call:
    below and above the sizes where the choice changes, against the oracle.
    The tolerances of the round trips at the default tiles: sums of <= 192
    terms and three FFT passes leave about 1e-15 and 2e-7 relative in the
    norm; 1e-12 and 1e-6."""
    import torch

    from exoplasim_amd import sht
    from exoplasim_amd.synth import ensemble

    print(f"untuned T{ntru} L{nlev} x{nmem} {mode}", flush=True)
    sp = ensemble(ntru, nlev, nmem, cfg=1)
    p = sht.Plan(ntru)
    x, gp, y = p.alloc_roundtrip(nmem, nlev, mode)
    x.copy_(torch.from_numpy(sp).to(x.dtype))
    p.roundtrip(mode, x, gp, y, nlev)
    torch.cuda.synchronize()
    tol = 1e-12 if mode == "f64" else 1e-6
    for k in (0, nmem - 1):
        want_g, want_s = oracle.roundtrip(ntru, nlev, x[k].double().cpu().numpy())
        assert rel(gp[k].double().cpu().numpy(), want_g) < tol
        assert rel(y[k].double().cpu().numpy(), want_s) < tol
    p.close()


@pytest.mark.parametrize("nbatch", [1, 15, 17, 256, 321, 1000, 4096, 4097, 4129])
def test_mlp_training_edges(gpu, nbatch):
    """the emulator's output and all gradients at ragged rows of a block, one
    and several batch splits, and both sides of the change from 16 to 32 rows
    per block, against the FP64 oracle with the kernels' bf16 roundings.
    What is left is FP32 accumulation and the bf16 values it flips to their
    neighbour: at most 2^-8 of a value, below 2^-9 = 2e-3 in the norm."""
    import sys as _sys

    _sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(__file__)), "oracle"))
    import mlp_oracle as MO
    import torch

    from exoplasim_amd.radiation import LwEmulator

    print(f"mlp training {nbatch}", flush=True)
    em = LwEmulator(seed=3)
    g = torch.Generator(device="cpu").manual_seed(nbatch)
    with torch.no_grad():
        for b in em.params[1::2]:
            b.copy_(0.1 * torch.randn(b.shape, generator=g))
    x = torch.randn(nbatch, 43, generator=g)
    gy = torch.randn(nbatch, 21, generator=g)
    y = em.raw(x.cuda())
    y.backward(gy.cuda())
    torch.cuda.synchronize()
    ps = [p.detach().double().cpu().numpy() for p in em.params]
    want, saved = MO.forward(x.double().numpy(), ps)
    grads = MO.backward(gy.double().numpy(), ps, saved)
    assert rel(y.detach().double().cpu().numpy(), want) < 2e-3
    for i, (p, w) in enumerate(zip(em.params, grads)):
        assert p.grad.shape == p.shape
        assert rel(p.grad.double().cpu().numpy(), w) < 2e-3, i


def test_mlp_saved_outputs_have_no_gradient(gpu):
    """a loss on a saved output alone reaches the backward pass without an
    output gradient: every parameter's gradient is zero"""
    import torch

    from exoplasim_amd.radiation import LwEmulator

    em = LwEmulator(seed=3)
    em.raw(torch.randn(20, 43, device="cuda"))
    out = torch.ops.exoplasim_amd.lw_mlp_forward(torch.randn(20, 43, device="cuda"), *em.params)
    out[2].sum().backward()
    assert all(p.grad is not None and not bool(p.grad.any()) for p in em.params)


@pytest.mark.parametrize("ncol", [1, 17, 4096, 4097])
def test_emulate_row_major_weights(gpu, ncol):
    """inference from row-major weights (exo_lw_emulate, guarded or not)
    against the fragment order that the class keeps, on both sides of the
    change from 16 to 32 columns per block: the same products in the same
    order, so equal to the last bit; and both guards flag the same columns"""
    import ctypes

    import torch

    from exoplasim_amd import radiation as R
    from exoplasim_amd._lib import lib
    from exoplasim_amd.columns import make_columns

    print(f"row-major emulate {ncol}", flush=True)
    em = R.LwEmulator(seed=5)
    cols = R.columns_to_device(make_columns(ncol, 20, 3), torch.float32)
    heat, olr = em.predict(cols)
    L, vp, ci = lib(), ctypes.c_void_p, ctypes.c_int
    ws = []
    for (nin, nout), (K, N), w in zip(R.LAYERS, R.PADDED, em.params[0::2]):
        W = torch.empty((N, K), dtype=torch.bfloat16, device="cuda")
        Wt = torch.empty((K, N), dtype=torch.bfloat16, device="cuda")
        assert L.exo_mlp_cast_weights(vp(w.data_ptr()), ci(nout), ci(nin), ci(N), ci(K),
                                      vp(W.data_ptr()), vp(Wt.data_ptr()), None) == 0
        ws.append((W, Wt))
    net = R._Net(20, (vp * 4)(*[W.data_ptr() for W, _ in ws]),
                 (vp * 4)(*[b.data_ptr() for b in em.params[1::2]]), em.ymean.data_ptr(),
                 em.ystd.data_ptr())
    x = [vp(cols[k].data_ptr()) for k in ("dt", "dq", "dp", "dqco2")]
    h, o = torch.empty_like(heat), torch.empty_like(olr)
    assert L.exo_lw_emulate(ctypes.byref(net), ci(ncol), *x, vp(h.data_ptr()), vp(o.data_ptr()),
                            None) == 0
    torch.cuda.synchronize()
    assert torch.equal(h, heat) and torch.equal(o, olr)
    f = R.features(cols)
    lo, hi = f.quantile(0.02, dim=0), f.quantile(0.98, dim=0)
    flags = [torch.empty(ncol, dtype=torch.int32, device="cuda") for _ in range(2)]
    assert L.exo_lw_emulate_guarded(ctypes.byref(net), vp(lo.data_ptr()), vp(hi.data_ptr()),
                                    ci(ncol), *x, vp(h.data_ptr()), vp(o.data_ptr()),
                                    vp(flags[0].data_ptr()), None) == 0
    assert L.exo_lw_emulate_packed(em._net_ref, vp(lo.data_ptr()), vp(hi.data_ptr()), ci(ncol),
                                   *x, vp(h.data_ptr()), vp(o.data_ptr()),
                                   vp(flags[1].data_ptr()), None) == 0
    torch.cuda.synchronize()
    assert torch.equal(h, heat) and torch.equal(o, olr) and torch.equal(*flags)


@pytest.mark.parametrize("ntru,nlev,nmem", [(21, 3, 9), (21, 11, 10), (42, 4, 5), (42, 21, 6)])
@pytest.mark.parametrize("mode", ["f64", "f32"])
def test_gridpointa_many_members(oracle, gpu, ntru, nlev, nmem, mode):
    """grids of more than one block per CU, whose levels a block shares among
    fewer waves, against each member alone (more waves, against the oracle
    above): the same sums in the same order, so that only the contraction of
    products and sums can differ, an ulp per term of sums that cancel by less
    than 1e2: 1e-12 and 2e-5."""
    import torch

    from exoplasim_amd import sht
    from exoplasim_amd.dynamics import Dynamics

    print(f"gridpointa T{ntru} L{nlev} x{nmem} {mode}", flush=True)
    plan = sht.Plan(ntru)
    dyn = Dynamics.from_vertical(_vertical(oracle, nlev), *PLASIM_SCAL)
    st, work, tend = dyn.alloc_gridpointa(plan, nmem, mode)
    st.copy_(torch.from_numpy(np.stack([gridpointa_state(ntru, nlev, 0.9 + 0.02 * k)
                                        for k in range(nmem)])).to(st.dtype))
    dyn.gridpointa(plan, mode, st, work, tend)
    st1, work1, tend1 = dyn.alloc_gridpointa(plan, 1, mode)
    tol = 1e-12 if mode == "f64" else 2e-5
    for k in (0, nmem - 1):
        st1.copy_(st[k:k + 1])
        dyn.gridpointa(plan, mode, st1, work1, tend1)
        torch.cuda.synchronize()
        for a, b in ((tend[k], tend1[0]), (work[k], work1[0])):
            assert rel(a.double().cpu().numpy(), b.double().cpu().numpy()) < tol
    dyn.close()
    plan.close()


@pytest.mark.parametrize("ntru,nlev,nmem,mode", [(63, 10, 33, "f64"), (42, 7, 300, "bf16x3")])
def test_noalloc_last_chunk(gpu, ntru, nlev, nmem, mode):
    """the no-allocation round trip of an untuned plan where the last chunk of
    members is small enough for other tiles than the whole call's: it uses
    the call's, so its outputs are the round trip's to the last bit"""
    import torch

    from exoplasim_amd import sht

    print(f"noalloc T{ntru} L{nlev} x{nmem} {mode}", flush=True)
    plan = sht.Plan(ntru)
    x, gp, y = plan.alloc_roundtrip(nmem, nlev, mode)
    x.normal_()
    plan.roundtrip(mode, x, gp, y, nlev)
    gp2, y2 = torch.full_like(gp, float("nan")), torch.full_like(y, float("nan"))
    plan.roundtrip_noalloc(mode, x, gp2, y2, nlev)
    torch.cuda.synchronize()
    assert torch.equal(gp, gp2) and torch.equal(y, y2)
    plan.close()


@pytest.mark.parametrize("ntru,nlev,nmem", [(21, 10, 1), (21, 9, 9), (42, 20, 1), (42, 7, 5)])
@pytest.mark.parametrize("mode", ["f64", "f32", "bf16x3"])
def test_gridpointa_dry_levels(oracle, gpu, ntru, nlev, nmem, mode):
    """humidity falling by 1e4 from the surface to the top: the rounding of a
    level's moisture tendency is that of its own terms, however much larger
    the other fields are.  Per level, the tolerances of the whole fields: a
    level's terms reach one level up and down, whose humidity is at most 4.6
    times its own (1e4^(1/6), L7), and cancel no more than the whole fields'
    do: 1e-12 and 2e-5.  A field that shared its row FFT with one 1e4 to 1e5
    times as large would keep 1e-16 * 1e5 and 1e-7 * 1e5."""
    import torch

    from exoplasim_amd import sht
    from exoplasim_amd.dynamics import Dynamics

    print(f"dry levels T{ntru} L{nlev} x{nmem} {mode}", flush=True)
    v = _vertical(oracle, nlev)
    plan, dyn = sht.Plan(ntru), Dynamics.from_vertical(v, *PLASIM_SCAL)
    st, work, tend = dyn.alloc_gridpointa(plan, nmem, mode)
    states = np.stack([gridpointa_state(ntru, nlev, 0.9 + 0.02 * k) for k in range(nmem)])
    states[:, 3 * nlev:4 * nlev] *= np.logspace(-4, 0, nlev)[:, None]
    st.copy_(torch.from_numpy(states).to(st.dtype))
    dyn.gridpointa(plan, mode, st, work, tend)
    got, host = tend.double().cpu().numpy(), st.double().cpu().numpy()
    for k in (0, nmem - 1):
        want, _ = oracle.gridpointa(ntru, nlev, host[k], v, PLASIM_SCAL, 1)
        for j in range(3 * nlev, 4 * nlev):
            assert rel(got[k, j], want[j]) < (1e-12 if mode == "f64" else 2e-5), (k, j)
    dyn.close()
    plan.close()


@pytest.mark.parametrize("ntru,nlev,nmem", [(21, 10, 1), (21, 9, 9), (42, 20, 1), (42, 7, 5),
                                            (63, 5, 1)])
@pytest.mark.parametrize("mode", ["f64", "f32", "bf16x3"])
def test_gridpointa_fields_apart(gpu, ntru, nlev, nmem, mode):
    """no field's values reach another through the transforms: a state
    without humidity has a moisture tendency of zeros, a humidity that is not
    a number at one level (which the virtual temperature takes as none)
    leaves the other tendencies as those of that level dry, to the last bit,
    and so does whatever lies in the grid humidity gq without spectral
    humidity, where only dq enters the temperature"""
    import torch

    from exoplasim_amd import sht
    from exoplasim_amd.dynamics import Dynamics, work_slots

    print(f"fields apart T{ntru} L{nlev} x{nmem} {mode}", flush=True)
    x = np.arange(1, nlev + 1) / nlev
    sh = 0.75 * x + 1.75 * x ** 3 - 1.5 * x ** 4
    ds = np.diff(np.concatenate([[0.0], sh]))
    g = np.tril(np.full((nlev, nlev), 0.2))
    v = dict(sigmah=sh, dsigma=ds, rdsig=0.5 / ds, t0=np.linspace(220.0, 288.0, nlev) / CT,
             t01s2=np.full(nlev, 0.01), tkp=np.full(nlev, 0.08), c=g.T, g=g, akap=0.286)
    plan, dyn = sht.Plan(ntru), Dynamics.from_vertical(v, *PLASIM_SCAL)
    st, work, tend = dyn.alloc_gridpointa(plan, nmem, mode)
    st.copy_(torch.from_numpy(np.stack([gridpointa_state(ntru, nlev, 0.9 + 0.02 * k)
                                        for k in range(nmem)])).to(st.dtype))
    sl, sq = work_slots(nlev), slice(3 * nlev, 4 * nlev)
    other = [i for i in range(4 * nlev + 1) if not 3 * nlev <= i < 4 * nlev]

    def run(nq=1):
        tend.fill_(float("nan"))
        dyn.gridpointa(plan, mode, st, work, tend, nqspec=nq)
        torch.cuda.synchronize()
        return tend[:, other].clone()

    wet = st[:, sq].clone()
    st[:, sq] = 0
    run()
    assert not bool(tend[:, sq].any())
    st[:, sq] = wet
    st[:, 3 * nlev + 2] = 0
    dry = run()
    assert bool(torch.isfinite(dry).all())
    st[:, 3 * nlev + 2] = float("nan")
    assert torch.equal(run(), dry)
    assert bool(torch.isfinite(tend[:, 4 * nlev - 1]).all())
    work[:, sl["dq"]:sl["dq"] + nlev] = 1e-3
    work[:, sl["gq"]:sl["gq"] + nlev] = 0
    dry = run(0)
    assert bool(torch.isfinite(dry).all())
    for bad in (1e30, float("inf"), float("nan")):
        work[:, sl["gq"]:sl["gq"] + nlev] = bad
        assert torch.equal(run(0), dry), bad
    dyn.close()
    plan.close()


@pytest.mark.parametrize("ntru", [21, 42, 63, 127])
@pytest.mark.parametrize("mode", ["f64", "f32", "f32mfma", "bf16x3"])
def test_tile_variants_same_bits(gpu, ntru, mode):
    """the tile variants sum in the same order and round in the same places,
    so that the choice among them, by tuning or by the size of a call, does
    not show in the results: equal to the last bit, in the inverse, the wind
    and the direct transforms"""
    import torch

    from exoplasim_amd import sht

    print(f"variants T{ntru} {mode}", flush=True)
    plan, nlev = sht.Plan(ntru), 5
    x, gp, y = plan.alloc_roundtrip(3, nlev, mode)
    x.normal_()
    first = None
    for v in range(4):
        plan.set_tiles(mode, v, v, v)
        gp.fill_(float("nan"))
        plan.inverse_all(mode, x, gp, nlev)
        out = [gp.clone()]
        plan.inverse_uv(mode, x, gp, nlev, 0, nlev, 3 * nlev + 2, 4 * nlev + 2)
        out.append(gp.clone())
        y.fill_(float("nan"))
        plan.direct(mode, out[0] if first is None else first[0], y, 3 * nlev + 1)
        out.append(y.clone())
        torch.cuda.synchronize()
        first = first or out
        assert all(torch.equal(a, b) for a, b in zip(out, first)), v
    plan.close()


@pytest.mark.parametrize("ntru,nlev,nmem", [(21, 20, 40), (42, 10, 9), (42, 20, 16), (63, 10, 16),
                                            (127, 5, 9)])
@pytest.mark.parametrize("mode", ["f64", "f32", "f32mfma", "bf16x3"])
def test_member_alone_same_bits(gpu, ntru, nlev, nmem, mode):
    """a member's round trip and dynamics step on an untuned plan are the same
    to the last bit alone, in a call whose tiles and waves per block are the
    small ones, and among as many members as take the large ones"""
    import torch

    from exoplasim_amd import sht
    from exoplasim_amd.dynamics import Dynamics

    print(f"member alone T{ntru} L{nlev} x{nmem} {mode}", flush=True)
    plan = sht.Plan(ntru)
    x, gp, y = plan.alloc_roundtrip(nmem, nlev, mode)
    x.normal_()
    plan.roundtrip(mode, x, gp, y, nlev)
    x1, gp1, y1 = plan.alloc_roundtrip(1, nlev, mode)
    x1.copy_(x[nmem - 1:])
    plan.roundtrip(mode, x1, gp1, y1, nlev)
    torch.cuda.synchronize()
    assert torch.equal(gp1[0], gp[nmem - 1]) and torch.equal(y1[0], y[nmem - 1])
    del x, gp, y
    s = np.arange(1, nlev + 1) / nlev
    g = np.tril(np.full((nlev, nlev), 0.2))
    v = dict(sigmah=s, dsigma=np.full(nlev, 1 / nlev), rdsig=np.full(nlev, nlev / 2),
             t0=np.linspace(220.0, 288.0, nlev) / CT, t01s2=np.full(nlev, 0.01),
             tkp=np.full(nlev, 0.08), c=g.T, g=g, akap=0.286)
    dyn = Dynamics.from_vertical(v, *PLASIM_SCAL)
    st, work, tend = dyn.alloc_gridpointa(plan, nmem, mode)
    st.copy_(torch.from_numpy(np.stack([gridpointa_state(ntru, nlev, 0.9 + 0.01 * k)
                                        for k in range(nmem)])).to(st.dtype))
    dyn.gridpointa(plan, mode, st, work, tend)
    st1, work1, tend1 = dyn.alloc_gridpointa(plan, 1, mode)
    st1.copy_(st[nmem - 1:])
    dyn.gridpointa(plan, mode, st1, work1, tend1)
    torch.cuda.synchronize()
    assert torch.equal(work1[0], work[nmem - 1]) and torch.equal(tend1[0], tend[nmem - 1])
    dyn.close()
    plan.close()


def test_emulator_columns_same_bits(gpu):
    """a column's heating and a row's network output are the same to the last
    bit in calls of 16 and of 32 columns per block"""
    import torch

    from exoplasim_amd import radiation as R
    from exoplasim_amd.columns import make_columns

    em = R.LwEmulator(seed=5)
    cols = R.columns_to_device(make_columns(8192, 20, 3), torch.float32)
    part = {k: v[..., 100:2000].contiguous() for k, v in cols.items()}
    (heat, olr), (h, o) = em.predict(cols), em.predict(part)
    assert torch.equal(heat[:, 100:2000], h) and torch.equal(olr[100:2000], o)
    x = R.features(cols)
    with torch.no_grad():
        assert torch.equal(em.raw(x)[100:2000], em.raw(x[100:2000]))


def test_tiles_saved_and_restored(gpu):
    """the choice by the size of each call is reported and can be set back"""
    from exoplasim_amd import sht
    from exoplasim_amd._lib import ExoError

    plan = sht.Plan(21)
    fresh = plan.tiles("f64")
    assert fresh == (-1, -1, -1)
    plan.set_tiles("f64", 2, 1, 3)
    assert plan.tiles("f64") == (2, 1, 3) and plan.tiles("f32") == fresh
    plan.set_tiles("f64", *fresh)
    assert plan.tiles("f64") == fresh
    for bad in ((-2, 0, 0), (0, 4, 0), (0, 0, -3)):
        with pytest.raises(ExoError):
            plan.set_tiles("f64", *bad)
    assert plan.tiles("f64") == fresh
    plan.close()


@pytest.mark.parametrize("nbatch", [1, 17, 64, 321, 1000])
def test_mlp_layer_entry_points(gpu, nbatch):
    """the layer-by-layer C entry points (casts, forward, input and weight
    gradients), chained as a caller of include/exo_rad.h would, against the
    FP64 oracle with the kernels' bf16 roundings, at ragged tiles of 64 rows
    and one and several batch splits.  What is left is FP32 accumulation and
    the bf16 values it flips to their neighbour: at most 2^-8 of a value,
    below 2^-9 = 2e-3 in the norm."""
    import ctypes
    import sys as _sys

    _sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(__file__)), "oracle"))
    import mlp_oracle as MO
    import torch

    from exoplasim_amd import radiation as R
    from exoplasim_amd._lib import lib

    print(f"mlp layers {nbatch}", flush=True)
    L, M, ci = lib(), nbatch, ctypes.c_int
    p = lambda t: None if t is None else ctypes.c_void_p(t.data_ptr())  # noqa: E731
    bf, f32 = torch.bfloat16, torch.float32
    new = lambda *s, dt=f32: torch.full(s, float("nan"), dtype=dt, device="cuda")  # noqa: E731
    g = torch.Generator(device="cpu").manual_seed(nbatch)
    ws = [torch.randn(o, i, generator=g) * (2.0 / i) ** 0.5 for i, o in R.LAYERS]
    bs = [0.1 * torch.randn(o, generator=g) for _, o in R.LAYERS]
    x, gy = torch.randn(M, R.NIN, generator=g), torch.randn(M, R.NOUT, generator=g)
    wd, bd = [w.cuda() for w in ws], [b.cuda() for b in bs]
    wb, wt = [], []
    for (nin, nout), (K, N), w in zip(R.LAYERS, R.PADDED, wd):
        wb.append(new(N, K, dt=bf))
        wt.append(new(K, N, dt=bf))
        assert L.exo_mlp_cast_weights(p(w), ci(nout), ci(nin), ci(N), ci(K), p(wb[-1]),
                                      p(wt[-1]), None) == 0
    xd, h = x.cuda(), [new(M, R.KIN, dt=bf)]
    assert L.exo_mlp_cast_rows(p(xd), ci(M), ci(R.NIN), ci(R.KIN), p(h[0]), None) == 0
    z = []
    for li in range(4):
        K, N = R.PADDED[li]
        out = new(M, N) if li < 3 else None
        hn, y = (new(M, N, dt=bf), None) if li < 3 else (None, new(M, N))
        assert L.exo_mlp_forward(p(h[li]), p(wb[li]), p(bd[li]), ci(M), ci(K), ci(N),
                                 ci(R.LAYERS[li][1]), ci(int(li < 3)), p(out), p(hn), p(y),
                                 None) == 0
        z.append(out)
        h.append(hn)
    dz32 = torch.zeros(M, R.NOUTP, device="cuda")
    dz32[:, :R.NOUT] = gy.cuda()
    dz = new(M, R.NOUTP, dt=bf)
    assert L.exo_mlp_cast_rows(p(dz32), ci(M), ci(R.NOUTP), ci(R.NOUTP), p(dz), None) == 0
    nsplit = max(1, min(64, M // 256))
    part, keep, grads = new(nsplit * R.NHID * R.NHID), [], [None] * 8
    for li in (3, 2, 1, 0):
        K, N = R.PADDED[li]
        nin, nout = R.LAYERS[li]
        dw, db = new(N, K), new(N)
        assert L.exo_mlp_backward_dw(p(dz), p(h[li]), p(dz32), ci(M), ci(N), ci(K), ci(nsplit),
                                     p(part), p(dw), p(db), None) == 0
        grads[2 * li], grads[2 * li + 1] = dw[:nout, :nin], db[:nout]
        if li:
            keep += [dz, dz32]
            ndz, ndz32 = new(M, K, dt=bf), new(M, K)
            assert L.exo_mlp_backward_dx(p(dz), p(wt[li]), p(z[li - 1]), ci(M), ci(N), ci(K),
                                         ci(R.LAYERS[li - 1][1]), p(ndz), p(ndz32), None) == 0
            dz, dz32 = ndz, ndz32
    torch.cuda.synchronize()
    ps = [t.double().numpy() for w, b in zip(ws, bs) for t in (w, b)]
    want, saved = MO.forward(x.double().numpy(), ps)
    assert rel(y[:, :R.NOUT].double().cpu().numpy(), want) < 2e-3
    for i, w in enumerate(MO.backward(gy.double().numpy(), ps, saved)):
        assert rel(grads[i].double().cpu().numpy(), w) < 2e-3, i


@pytest.mark.parametrize("nlev,nhor,nmem", [(2, 1, 1), (7, 130, 2), (20, 512, 1), (64, 65, 2)])
@pytest.mark.parametrize("mode", ["f64", "f32"])
@pytest.mark.parametrize("nq", [1, 0])
def test_calcgp_in_place(oracle, gpu, nlev, nhor, nmem, mode, nq):
    """outputs in the place of the inputs that a level reads from the next and
    the one before (temperature, humidity, winds) and of the vorticity: the
    same as in arrays of their own, to the last bit"""
    import torch

    from exoplasim_amd.dynamics import CALCGP_OUT, PRODUCTS, Dynamics

    print(f"calcgp in place L{nlev} x{nhor} x{nmem} {mode} nqspec={nq}", flush=True)
    dyn = Dynamics.from_vertical(_vertical(oracle, nlev), *PLASIM_SCAL)
    dt = torch.float64 if mode == "f64" else torch.float32
    host = {k: x[..., :nhor] for k, x in plasim_inputs(nlev, 512, 5)[1].items()}

    def fields():
        f = {}
        for k, x in host.items():
            x = np.stack([x * (1 + 0.1 * m) for m in range(nmem)])
            full = np.zeros((nmem, nlev, nhor))
            full[:, :x.shape[1] if x.ndim == 3 else 1] = x if x.ndim == 3 else x[:, None]
            f[k] = torch.from_numpy(full).to("cuda", dt)
        for k in CALCGP_OUT + PRODUCTS + ("gvp",):
            f[k] = torch.zeros((nmem, nlev, nhor), dtype=dt, device="cuda")
        return f

    def run(f):
        flat = {k: (x[0] if x.dim() == 3 else x).contiguous() if nmem == 1 else x
                for k, x in f.items()}
        if nmem == 1:
            for k in ("gp", "gpj", "gpm", "rcsq", "gvp"):
                flat[k] = f[k][0, 0]
        dyn.calcgp(mode, flat, nqspec=nq, nmem=nmem, member_stride=nlev * nhor if nmem > 1 else 0)
        torch.cuda.synchronize()

    a, b = fields(), fields()
    places = dict(gtn="gt", gqn="gq", guz="gv", gvz="gu", gke="gz", gphi="gd")
    for o, i in places.items():
        b[o] = b[i]
    run(a)
    run(b)
    for k in CALCGP_OUT + PRODUCTS + ("gvp",):
        assert torch.equal(a[k], b[k]), k
    dyn.close()


@pytest.mark.parametrize("nlev", [2, 10, 16, 17])
@pytest.mark.parametrize("mode", ["f64", "f32"])
def test_calcgp_many_points(oracle, gpu, nlev, mode):
    """more than 1024 blocks of 64 points, whose few levels 4 waves share
    instead of 8: points at both ends as in a call of their own (8 waves,
    against the oracle above), to the last bit"""
    import torch

    from exoplasim_amd.dynamics import CALCGP_OUT, PRODUCTS, Dynamics

    print(f"calcgp many points L{nlev} {mode}", flush=True)
    dyn = Dynamics.from_vertical(_vertical(oracle, nlev), *PLASIM_SCAL)
    dt, nhor = torch.float64 if mode == "f64" else torch.float32, 64 * 1025 + 1
    f = {k: torch.from_numpy(np.ascontiguousarray(x)).to("cuda", dt)
         for k, x in plasim_inputs(nlev, nhor, 5)[1].items()}

    def run(f):
        out = {k: torch.zeros((nlev, f["gt"].shape[1]), dtype=dt, device="cuda")
               for k in CALCGP_OUT + PRODUCTS}
        out["gvp"] = torch.zeros(f["gt"].shape[1], dtype=dt, device="cuda")
        dyn.calcgp(mode, {**f, **out}, nqspec=1)
        torch.cuda.synchronize()
        return out

    whole = run(f)
    for s in (slice(0, 130), slice(nhor - 70, nhor)):
        for k, x in run({k: x[..., s].contiguous() for k, x in f.items()}).items():
            assert torch.equal(x, whole[k][..., s]), k
    dyn.close()


@pytest.mark.parametrize("ntru,nlev,nmem", [(21, 3, 1), (42, 9, 2)])
@pytest.mark.parametrize("mode", ["f64", "f32"])
def test_mktend_in_place(gpu, ntru, nlev, nmem, mode):
    """the temperature tendency in the memory of ke and the vorticity's in that
    of tn, vt or ke, which the transforms before them have read: as in arrays
    of their own, to the last bit"""
    import torch

    from exoplasim_amd import sht

    print(f"mktend in place T{ntru} L{nlev} x{nmem} {mode}", flush=True)
    p = sht.Plan(ntru)
    dt = p.dtype_of(mode)
    tn, fu, fv, ke, ut, vt = (torch.randn(nmem, nlev, p.nlat, p.nlon, dtype=dt, device="cuda")
                              for _ in range(6))
    want = [torch.zeros((nmem, nlev, p.nrsp), dtype=dt, device="cuda") for _ in range(3)]
    p.mktend(mode, *want, tn, fu, fv, ke, ut, vt, nlev)
    for tat, zat in ((3, 0), (None, 5), (None, 3), (3, None)):
        f = [x.clone() for x in (tn, fu, fv, ke, ut, vt)]
        out = [torch.zeros_like(want[0])] + [
            torch.zeros_like(want[0]) if k is None
            else f[k].view(-1)[:want[0].numel()].view_as(want[0]) for k in (tat, zat)]
        p.mktend(mode, *out, *f, nlev)
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(out, want)), (tat, zat)
    p.close()


@pytest.mark.parametrize("ntru,nlev,mode", [(42, 42, "f64"), (42, 64, "f64"), (21, 64, "f64"),
                                            (42, 64, "f32")])
@pytest.mark.parametrize("nq", [1, 0])
def test_gridpointa_most_levels(oracle, gpu, ntru, nlev, mode, nq):
    """the level arrays of FP64 rows of 128 points fit a block's LDS up to L41
    (3072 L + 35840 bytes of 163840; above): from L42 on calcgp runs on the
    grid and the rows are transformed in a launch of their own.  The largest
    level count of the other row kernels, whose 10 waves then ask for 152128
    bytes.  Tolerances as above."""
    test_gridpointa_edges(oracle, gpu, ntru, nlev, mode, nq)


@pytest.mark.parametrize("ntru", [42, 63])
@pytest.mark.parametrize("mode", ["f64", "f32", "bf16x3"])
def test_untuned_tiles_many_blocks(oracle, gpu, ntru, mode):
    """calls far above the sizes where untuned plans take other tiles: 16
    members of L20.  Blocks at half the fields per block (V = 3), against the
    limits 256 and 512: inverse T42 4 pair blocks x (16 + 1 + 10) groups x 16
    members = 1728, T63 6 x (21 + 1 + 20) x 16 = 4032 (FP64, two fields per block,
    4 and 6 x (31 + 1 + 20) x 16 = 3328 and 4992); direct 61 fields x 16 = 976
    (T63 FP64, two latitude blocks: 1952).  So the whole tiles: V = 2, in the
    FP64 direct of T42 V = 0."""
    test_untuned_tiles(oracle, gpu, ntru, 20, 16, mode)


def test_plan_memory(gpu):
    """device memory of a T127 plan.  Tables of 96 x 8256 values: 8 in FP64 as
    built, 8 with the filters in FP64 and FP32 (50.7, 50.7 and 25.4 MB), the
    direct transform's one in both (9.5); the four inverse tables as matrix
    operands (2 x 50.3 MB, and split BF16) and the four direct ones: about 300
    MB.  All eight tables in the direct transform's order would add 67."""
    import torch

    from exoplasim_amd import sht

    sht.Plan(127).close()  # the library's own memory
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    plan = sht.Plan(127)
    used = free - torch.cuda.mem_get_info()[0]
    plan.close()
    print(f"T127 plan {used / 1e6:.0f} MB", flush=True)
    assert used < 320e6


@pytest.mark.parametrize("ntru,nlev", [(21, 10), (42, 7)])
@pytest.mark.parametrize("mode", ["f64", "f32"])
def test_gridpointa_unaligned_work(oracle, gpu, ntru, nlev, mode):
    """a work array that starts one value past an allocation, its members an
    odd number of values apart: a lane's two points are then not on their own
    size, and every value is that of the aligned call"""
    import torch

    from exoplasim_amd import sht
    from exoplasim_amd._lib import lib
    from exoplasim_amd.dynamics import Dynamics

    print(f"unaligned work T{ntru} L{nlev} {mode}", flush=True)
    plan, dyn = sht.Plan(ntru), Dynamics.from_vertical(_vertical(oracle, nlev), *PLASIM_SCAL)
    st, work, tend = dyn.alloc_gridpointa(plan, 3, mode)
    st.copy_(torch.from_numpy(np.stack([gridpointa_state(ntru, nlev, 0.9 + 0.1 * k)
                                        for k in range(3)])).to(st.dtype))
    dyn.gridpointa(plan, mode, st, work, tend)
    n, per = work[0].numel(), work[0].numel() + 3
    buf = torch.zeros(3 * per + 1, dtype=st.dtype, device="cuda")
    out = torch.zeros_like(tend)
    assert lib().exo_gridpointa(plan._h, dyn._h, 0 if mode == "f64" else 1, 3, 1, st.data_ptr(),
                                st[0].numel(), buf.data_ptr() + buf.element_size(), per,
                                out.data_ptr(), out[0].numel(),
                                torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    assert torch.equal(out, tend)
    for k in range(3):
        assert torch.equal(buf[1 + k * per:1 + k * per + n], work[k].view(-1))
    dyn.close()
    plan.close()
