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
