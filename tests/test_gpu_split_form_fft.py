"""The split-form FFT by name (fft_form 4) on lengths below 384, whose default
is the folded DFT: both against the oracle, on its smallest powers of two and
on both buffer layouts, and refused where the length has no such form."""
import numpy as np
import pytest

import oracle as O
from kemorin_mhd_amd import ShellConfig, ShtError, SphTransPlan, synthetic_spectra

pytestmark = pytest.mark.gpu

SHELLS = [ShellConfig(31, 3, 48, 96), ShellConfig(20, 5, 33, 64), ShellConfig(63, 7, 95, 192),
          ShellConfig(63, 2, 97, 320), ShellConfig(127, 3, 192, 384)]


def _rel(a, b, ncomp, comp_fastest):
    shape, axis = ((-1, ncomp), 0) if comp_fastest else ((ncomp, -1), 1)
    a, b = np.asarray(a).reshape(shape), np.asarray(b).reshape(shape)
    return (np.linalg.norm(a - b, axis=axis) / np.linalg.norm(b, axis=axis)).max()


@pytest.mark.parametrize("cfg", SHELLS, ids=lambda c: f"L{c.L}_N{c.nphi}")
def test_split_form(torch_cuda, cfg):
    t = torch_cuda
    print(f"[gpu] split-form FFT L={cfg.L} Nphi={cfg.nphi}", flush=True)
    nc = 4
    orc = O.OraclePlan(cfg.L, cfg.nr, cfg.nth, cfg.nphi, cfg.radius(), full_tables=False)
    sp = synthetic_spectra(cfg, 1, 1, seed=5)
    grid, rtm = orc.backward(1, 1, sp), orc.leg_bwd(1, 1, sp)
    new = lambda n: t.full((n,), np.nan, dtype=t.float64, device="cuda")
    d_grid, rtp = t.from_numpy(grid).cuda(), new(cfg.n_rtp(nc))
    plan = SphTransPlan(cfg, max_ncomp=nc)
    try:
        plan.set_variant("fft_form", 4)
        assert plan.get_variant("fft_form") == 4
        v, w, sv, srtp = new(cfg.n_rtp(nc)), new(cfg.n_rj(nc)), new(cfg.n_rtp(nc)), new(cfg.n_rtp(nc))
        plan.sph_backward_transforms(1, 1, t.from_numpy(sp).cuda(), v)
        plan.sph_forward_transforms(1, 1, d_grid, w)
        plan.exchange_rtm_to_rtp(nc, t.from_numpy(rtm).cuda(), rtp)
        plan.fft_backward(nc, rtp, sv)
        plan.fft_forward(nc, d_grid, srtp)
        t.cuda.synchronize()
    finally:
        plan.close()
    v, w, sv, srtp = (x.cpu().numpy() for x in (v, w, sv, srtp))
    assert _rel(v, grid, nc, False) <= 1e-12
    assert _rel(w, orc.forward(1, 1, grid), nc, True) <= 1e-12
    # log2 N butterfly levels of a few roundings each
    assert _rel(sv, grid, nc, False) <= 1e-13
    ref = orc.rtp_to_rtm(nc, orc.fft_fwd_to_rtp(nc, grid))
    assert _rel(orc.rtp_to_rtm(nc, srtp), ref, nc, True) <= 1e-13


@pytest.mark.parametrize("cfg", [ShellConfig(44, 3, 68, 138), ShellConfig(40, 3, 62, 126)],
                         ids=lambda c: f"L{c.L}_N{c.nphi}")
def test_refused_without_such_a_form(torch_cuda, cfg):
    plan = SphTransPlan(cfg, max_ncomp=4)
    try:
        with pytest.raises(ShtError) as e:
            plan.set_variant("fft_form", 4)
        assert e.value.status == 2  # SHT_ERR_UNSUPPORTED
        assert plan.get_variant("fft_form") == 1
    finally:
        plan.close()
