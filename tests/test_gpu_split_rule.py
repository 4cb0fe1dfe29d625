"""Split-precision plans that run FP64 products (truncations below the rule's
line): the results of an FP64 plan, bit for bit, in every call form; the sliced
products where they are asked for, held to the oracle at sizes around their
chunks, with every form of them bit for bit the same; and the noalloc limit of
the sliced operand either way."""
import numpy as np
import pytest

import oracle as O
from kemorin_mhd_amd import (SHT_PREC_FP64, SHT_PREC_SPLIT_INT8, ShellConfig, ShtError,
                             SphTransPlan, synthetic_spectra)

pytestmark = pytest.mark.gpu

# 6 slices: backward 4.4e-12 and forward 1e-11 of a component as elsewhere
TOL = {4: 1e-6, 5: 1e-8, 6: 1e-11, 7: 1e-13}


def _calls(t, plan, cfg, nv, ns, sp, grid):
    nc = 3 * nv + ns
    new = lambda n: t.full((n,), np.nan, dtype=t.float64, device="cuda")
    v, w, rtm, w2 = new(cfg.n_rtp(nc)), new(cfg.n_rj(nc)), new(cfg.n_rtm(nc)), new(cfg.n_rj(nc))
    plan.sph_backward_transforms(nv, ns, sp, v)
    plan.sph_forward_transforms(nv, ns, grid, w)
    plan.legendre_backward(nv, ns, sp, rtm)
    plan.legendre_forward(nv, ns, rtm, w2)
    t.cuda.synchronize()
    return [x.cpu().numpy() for x in (v, w, rtm, w2)]


@pytest.mark.parametrize("L,nr,nth,nv,ns,S,otf", [(1, 1, 2, 1, 1, 0, False), (31, 33, 47, 2, 2, 6, True),
                                                  (63, 17, 96, 1, 3, 4, False), (127, 9, 191, 3, 0, 7, False),
                                                  (223, 5, 336, 1, 1, 4, False), (230, 5, 347, 1, 1, 5, True)])
def test_fp64_products(torch_cuda, L, nr, nth, nv, ns, S, otf):
    t = torch_cuda
    print(f"[gpu] split plan on FP64 products L={L} Nr={nr} S={S} per call={otf}", flush=True)
    cfg, nc = ShellConfig(L, nr, nth, max(2 * nth, 2 * L + 2)), 3 * nv + ns
    rng = np.random.default_rng(L)
    sp = t.from_numpy(rng.standard_normal(cfg.n_rj(nc))).cuda()
    grid = t.from_numpy(rng.standard_normal(cfg.n_rtp(nc))).cuda()
    out = []
    for prec in (SHT_PREC_FP64, SHT_PREC_SPLIT_INT8):
        plan = SphTransPlan(cfg, max_ncomp=nc, precision=prec, n_slices=S, p_on_the_fly=otf)
        try:
            out.append(_calls(t, plan, cfg, nv, ns, sp, grid))
        finally:
            plan.close()
    assert all(np.array_equal(a, b) for a, b in zip(*out))


@pytest.mark.parametrize("L,nr,nth,nv,ns,S", [
    (2, 3, 5, 1, 1, 6), (31, 17, 48, 2, 2, 6), (64, 16, 97, 3, 0, 5), (127, 5, 192, 0, 3, 4),
    (130, 9, 195, 1, 4, 7), (63, 33, 96, 1, 2, 6)])
@pytest.mark.parametrize("otf", [False, True])
def test_sliced_products(torch_cuda, L, nr, nth, nv, ns, S, otf):
    t = torch_cuda
    print(f"[gpu] sliced products selected L={L} Nr={nr} S={S} per call={otf}", flush=True)
    cfg, nc = ShellConfig(L, nr, nth, max(2 * nth, 2 * L + 2)), 3 * nv + ns
    orc = O.OraclePlan(cfg.L, cfg.nr, cfg.nth, cfg.nphi, cfg.radius(), full_tables=False)
    sp = synthetic_spectra(cfg, nv, ns, seed=L)
    grid = orc.backward(nv, ns, sp)
    plan = SphTransPlan(cfg, max_ncomp=nc, precision=SHT_PREC_SPLIT_INT8, n_slices=S, p_on_the_fly=otf)
    try:
        before = plan.device_bytes()
        plan.set_variant("split_all", 1)
        after = plan.device_bytes()
        assert after > before
        v, w, rtm, w2 = _calls(t, plan, cfg, nv, ns, t.from_numpy(sp).cuda(), t.from_numpy(grid).cuda())
        for name, value in (("split_fwd_mfma", 32), ("split_bwd_fused", 0)):
            plan.set_variant(name, value)
            form = _calls(t, plan, cfg, nv, ns, t.from_numpy(sp).cuda(), t.from_numpy(grid).cuda())
            assert all(np.array_equal(a, b) for a, b in zip(form, (v, w, rtm, w2)))
    finally:
        plan.close()

    def err(a, b, axis):
        a, b = (x.reshape(-1, nc) if axis == 0 else x.reshape(nc, -1).T for x in (a, b))
        return (np.linalg.norm(a - b, axis=0) / np.linalg.norm(b, axis=0)).max()

    assert err(v, grid, 1) <= TOL[S]
    assert err(w, orc.forward(nv, ns, grid), 0) <= TOL[S]
    assert err(rtm, orc.leg_bwd(nv, ns, sp), 0) <= TOL[S]


def test_noalloc_limit(torch_cuda):
    """L = 63, Nr = 65, 9 components: within the fixed workspace in FP64, above
    it with the slices of a split-precision plan, whichever products it runs."""
    t = torch_cuda
    cfg = ShellConfig(63, 65, 96, 192)
    sp = t.zeros(cfg.n_rj(9), dtype=t.float64, device="cuda")
    v = t.zeros(cfg.n_rtp(9), dtype=t.float64, device="cuda")
    for prec in (SHT_PREC_FP64, SHT_PREC_SPLIT_INT8):
        plan = SphTransPlan(cfg, max_ncomp=9, precision=prec)
        try:
            if prec == SHT_PREC_FP64:
                plan.sph_backward_transforms_noalloc(3, 0, sp, v)
            else:
                with pytest.raises(ShtError):
                    plan.sph_backward_transforms_noalloc(3, 0, sp, v)
                plan.set_variant("split_all", 1)
                with pytest.raises(ShtError):
                    plan.sph_backward_transforms_noalloc(3, 0, sp, v)
            t.cuda.synchronize()
        finally:
            plan.close()
