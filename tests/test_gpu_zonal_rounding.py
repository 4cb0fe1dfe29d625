"""Rounding of the default zonal transform, coefficients to grid, against
extended precision.  Coefficients fall with the order (m + 1)^-1.5, as a
transform's do: summed from the smallest up, the partial sums stay as small as
their terms, and what is left is the rounding of the table entries and of the
last few additions, each at most 2^-53 of the result: 2^-52 in the norm."""
import numpy as np
import pytest

from kemorin_mhd_amd import ShellConfig, SphTransPlan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,nr,nth,nphi", [(31, 3, 48, 96), (63, 4, 96, 192), (88, 3, 134, 268),
                                           (179, 3, 270, 540), (361, 2, 543, 1086)])
def test_backward_sums_from_the_smallest(torch_cuda, L, nr, nth, nphi):
    t = torch_cuda
    print(f"[gpu] zonal rounding L={L} Nphi={nphi}", flush=True)
    cfg, rng, lines = ShellConfig(L, nr, nth, nphi), np.random.default_rng(L), nr * nth
    m = np.arange(1, L + 1)
    a, b = (rng.standard_normal((L, lines)) * ((m + 1.0) ** -1.5)[:, None] for _ in range(2))
    rtp = np.zeros((nphi, lines))  # FFTPACK slots: a0, Nyquist, then cos and sin by turns
    rtp[0] = rng.standard_normal(lines)
    rtp[2 * m], rtp[2 * m + 1] = a, b
    w = 2 * np.longdouble("3.14159265358979323846264338327950288") / nphi
    ph = np.outer(np.arange(nphi), m) % nphi * w
    want = rtp[0] + np.cos(ph) @ a.astype(np.longdouble) + np.sin(ph) @ b.astype(np.longdouble)
    v = t.empty(cfg.n_rtp(1), dtype=t.float64, device="cuda")
    plan = SphTransPlan(cfg, max_ncomp=1)
    try:
        plan.fft_backward(1, t.from_numpy(rtp.reshape(-1)).cuda(), v)
        t.cuda.synchronize()
    finally:
        plan.close()
    d = (v.cpu().numpy().reshape(nphi, lines) - want).astype(np.float64)
    err = np.linalg.norm(d) / np.linalg.norm(want.astype(np.float64))
    print(f"    rel L2 {err:.2e}", flush=True)
    assert err <= 2.0 ** -52
