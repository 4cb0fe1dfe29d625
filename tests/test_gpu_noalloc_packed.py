"""sht_backward_noalloc on calls whose FP64 products pack their spectra: behind
the Fourier workspace in the fixed array, several shares of orders where little
of it is left, unpacked where one order's rows do not fit.  Bit for bit
sht_backward's results each time, also while sht_backward of the same plan runs
on another stream: the two share no buffer."""
import numpy as np
import pytest

from kemorin_mhd_amd import SHT_PREC_FP64, SHT_PREC_SPLIT_INT8, ShellConfig, SphTransPlan

pytestmark = pytest.mark.gpu

# Fourier workspace and what is left of 128 MiB, an order's packed rows (MB): 57 / 77, 0.6;
# 132.7 / 1.5, 1.0 (several shares); 134.0 / 0.3, 0.8 (unpacked); 52 / 82, 1.1 (scalars)
CALLS = [(63, 65, 96, 3, 0), (95, 67, 144, 3, 0), (127, 38, 192, 3, 0), (31, 360, 48, 0, 6)]


@pytest.mark.parametrize("prec", [SHT_PREC_FP64, SHT_PREC_SPLIT_INT8], ids=["fp64", "split"])
@pytest.mark.parametrize("otf", [False, True], ids=["tables", "per_call"])
@pytest.mark.parametrize("L,nr,nth,nv,ns", CALLS)
def test_bitexact(torch_cuda, L, nr, nth, nv, ns, otf, prec):
    t = torch_cuda
    if prec == SHT_PREC_SPLIT_INT8:
        nr //= 3  # its limit counts the sliced operand
    print(f"[gpu] noalloc L={L} Nr={nr} {nv}+{ns} per call={otf} precision={prec}", flush=True)
    cfg, nc = ShellConfig(L, nr, nth, 2 * nth), 3 * nv + ns
    sp = t.from_numpy(np.random.default_rng(L).standard_normal(cfg.n_rj(nc))).cuda()
    ref, got = (t.full((cfg.n_rtp(nc),), np.nan, dtype=t.float64, device="cuda") for _ in range(2))
    plan = SphTransPlan(cfg, max_ncomp=nc, precision=prec, p_on_the_fly=otf)
    try:
        plan.sph_backward_transforms(nv, ns, sp, ref)
        plan.sph_backward_transforms_noalloc(nv, ns, sp, got)
        t.cuda.synchronize()
    finally:
        plan.close()
    assert not t.isnan(ref).any()
    assert t.equal(got, ref)


@pytest.mark.parametrize("L,nr,nth,nv,ns", CALLS[:3])
def test_beside_sht_backward_of_the_same_plan(torch_cuda, L, nr, nth, nv, ns):
    t = torch_cuda
    print(f"[gpu] noalloc beside sht_backward L={L} Nr={nr}", flush=True)
    cfg, nc, rng = ShellConfig(L, nr, nth, 2 * nth), 3 * nv + ns, np.random.default_rng(L + 1)
    sp = [t.from_numpy(rng.standard_normal(cfg.n_rj(nc))).cuda() for _ in range(2)]
    ref, got = ([t.empty(cfg.n_rtp(nc), dtype=t.float64, device="cuda") for _ in range(2)] for _ in range(2))
    plan = SphTransPlan(cfg, max_ncomp=nc)
    streams = [t.cuda.Stream() for _ in range(2)]
    try:
        for x, y in zip(sp, ref):
            plan.sph_backward_transforms(nv, ns, x, y)
        t.cuda.synchronize()
        for _ in range(4):
            for y in got:
                y.fill_(np.nan)
            t.cuda.synchronize()
            with t.cuda.stream(streams[0]):
                plan.sph_backward_transforms(nv, ns, sp[0], got[0])
            with t.cuda.stream(streams[1]):
                plan.sph_backward_transforms_noalloc(nv, ns, sp[1], got[1])
            t.cuda.synchronize()
            assert t.equal(got[0], ref[0]) and t.equal(got[1], ref[1])
    finally:
        plan.close()
