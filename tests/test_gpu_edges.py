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
