"""The folded real DFT of the zonal transform (the default for lengths below
384 and those without a fast FFT) against the oracle and the mixed-radix form.
Shells at the edges of its tiles: N/4 + 1 points at 32, 33 and one block, an
order count at the end of a K step and one past it, N divisible by 4 and not,
odd line counts, fewer lines than a block, and more waves than the small-grid
rule takes.  A sum of K products rounds within K 2^-53 of its terms' size:
K <= 300 and norms over many lines stay below 1e-13."""
import numpy as np
import pytest

import oracle as O
from kemorin_mhd_amd import ShellConfig, SphTransPlan, synthetic_spectra

pytestmark = pytest.mark.gpu

SHELLS = [ShellConfig(1, 1, 2, 4), ShellConfig(2, 3, 3, 6), ShellConfig(5, 1, 7, 14),
          ShellConfig(40, 3, 41, 124), ShellConfig(41, 5, 43, 128), ShellConfig(62, 7, 95, 190),
          ShellConfig(63, 4, 96, 192), ShellConfig(64, 3, 65, 130), ShellConfig(66, 2, 101, 202),
          ShellConfig(88, 65, 134, 268), ShellConfig(126, 3, 191, 382), ShellConfig(361, 2, 543, 1086)]


def _rel(a, b, ncomp, comp_fastest):
    shape, axis = ((-1, ncomp), 0) if comp_fastest else ((ncomp, -1), 1)
    a, b = np.asarray(a).reshape(shape), np.asarray(b).reshape(shape)
    return (np.linalg.norm(a - b, axis=axis) / np.linalg.norm(b, axis=axis)).max()


@pytest.mark.parametrize("cfg", SHELLS, ids=lambda c: f"L{c.L}_N{c.nphi}_lines{c.nr * c.nth}")
def test_folded_dft(torch_cuda, cfg):
    t = torch_cuda
    print(f"[gpu] folded DFT L={cfg.L} Nr={cfg.nr} Nphi={cfg.nphi}", flush=True)
    orc = O.OraclePlan(cfg.L, cfg.nr, cfg.nth, cfg.nphi, cfg.radius(), full_tables=False)
    plan = SphTransPlan(cfg, max_ncomp=4)
    gen = t.Generator(device="cuda")
    gen.manual_seed(17)
    nc = 4

    def rand(n):
        return t.randn(n, generator=gen, dtype=t.float64, device="cuda")

    def nan(n):
        return t.full((n,), np.nan, dtype=t.float64, device="cuda")

    sp, rtm, g = rand(cfg.n_rj(nc)), rand(cfg.n_rtm(nc)), rand(cfg.n_rtp(nc))
    rtp = t.empty(cfg.n_rtp(nc), dtype=t.float64, device="cuda")
    got = {}
    try:
        plan.exchange_rtm_to_rtp(nc, rtm, rtp)
        for form in (1, 0):
            plan.set_variant("fft_form", form)
            v, w, sv, srtp = nan(cfg.n_rtp(nc)), nan(cfg.n_rj(nc)), nan(cfg.n_rtp(nc)), t.zeros_like(rtp)
            plan.sph_backward_transforms(1, 1, sp, v)
            plan.sph_forward_transforms(1, 1, g, w)
            plan.fft_backward(nc, rtp, sv)
            plan.fft_forward(nc, g, srtp)
            t.cuda.synchronize()
            got[form] = [x.cpu().numpy() for x in (v, w, sv, srtp)]
    finally:
        plan.close()
    fastest = (False, True, False, True)
    for a, b, f in zip(got[1], got[0], fastest):
        assert _rel(a, b, nc, f) <= 1e-13
    v, w, sv, srtp = got[1]
    assert _rel(v, orc.backward(1, 1, sp.cpu().numpy()), nc, False) <= 1e-12
    assert _rel(w, orc.forward(1, 1, g.cpu().numpy()), nc, True) <= 1e-12
    assert _rel(sv, orc.fft_bwd_from_rtp(nc, orc.rtm_to_rtp(nc, rtm.cpu().numpy())), nc, False) <= 1e-13
    ref = orc.rtp_to_rtm(nc, orc.fft_fwd_to_rtp(nc, g.cpu().numpy()))
    assert _rel(orc.rtp_to_rtm(nc, srtp), ref, nc, True) <= 1e-13
