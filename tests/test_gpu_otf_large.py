"""P per call against stored tables on calls of many waves, where the forward
takes another kernel for all orders at once than for a tile of them: the two
kernels round alike, so the outputs are those of stored tables bit for bit.
Calls on both sides of the line, on FP64 plans and on a split-precision plan
below its own line, which runs the same products."""
import numpy as np
import pytest

from kemorin_mhd_amd import SHT_PREC_FP64, SHT_PREC_SPLIT_INT8, ShellConfig, SphTransPlan

pytestmark = pytest.mark.gpu

# (L, Nr, Ntheta, vectors, scalars, precision): 30400, 27456, 21760, 15616 and 10240 waves
CALLS = [(127, 190, 192, 8, 0, SHT_PREC_FP64), (127, 180, 192, 4, 12, SHT_PREC_SPLIT_INT8),
         (95, 170, 145, 0, 32, SHT_PREC_FP64), (127, 64, 192, 11, 4, SHT_PREC_FP64),
         (127, 64, 192, 8, 0, SHT_PREC_FP64)]


@pytest.mark.parametrize("L,nr,nth,nv,ns,prec", CALLS)
def test_large_calls_bitexact_vs_stored(torch_cuda, L, nr, nth, nv, ns, prec):
    t = torch_cuda
    print(f"[gpu] P per call vs stored L={L} Nr={nr} {nv}+{ns} precision={prec}", flush=True)
    cfg, nc = ShellConfig(L, nr, nth, 2 * nth), 3 * nv + ns
    g = t.Generator(device="cuda")
    g.manual_seed(L)
    rand = lambda n: t.randn(n, dtype=t.float64, device="cuda", generator=g)
    new = lambda n: t.full((n,), np.nan, dtype=t.float64, device="cuda")
    sp, grid = rand(cfg.n_rj(nc)), rand(cfg.n_rtp(nc))
    out = []
    for otf in (False, True):
        plan = SphTransPlan(cfg, max_ncomp=nc, precision=prec, p_on_the_fly=otf)
        try:
            v, w = new(cfg.n_rtp(nc)), new(cfg.n_rj(nc))
            plan.sph_backward_transforms(nv, ns, sp, v)
            plan.sph_forward_transforms(nv, ns, grid, w)
            t.cuda.synchronize()
            out.append((v, w))
        finally:
            plan.close()
    assert not t.isnan(out[0][1]).any()
    assert t.equal(out[0][0], out[1][0])
    assert t.equal(out[0][1], out[1][1])
