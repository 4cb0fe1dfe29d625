"""The staged FP64 forward Legendre kernel: radius-slowest input (the separate
stages) at the edges of its tiles, against the whole transform, whose direct
kernel the oracle tests cover; and calls large enough for it in the whole
transform, against the same fields one call each.  Both kernels add the same
products of one rounding each in the same order of K steps, over at most
Ntheta / 2 rows: 1e-14 of a component's norm per hundred rows and less."""
import numpy as np
import pytest

from kemorin_mhd_amd import ShellConfig, SphTransPlan

pytestmark = pytest.mark.gpu

# (L, Nr, Ntheta, vectors, scalars, P per call)
STAGES = [(1, 1, 2, 1, 1, False), (2, 2, 5, 0, 1, False), (5, 3, 7, 1, 2, False),
          (15, 17, 24, 2, 3, True), (31, 33, 47, 3, 0, False), (33, 16, 67, 1, 1, False),
          (64, 5, 97, 2, 1, False), (95, 40, 144, 1, 9, False), (127, 18, 191, 2, 3, True),
          (190, 9, 288, 2, 2, False)]
LARGE = [(65, 322, 99, 8, 3), (127, 180, 192, 4, 5)]


def _close(t, a, b):
    a, b = a.double(), b.double()
    assert not t.isnan(a).any()
    assert (t.linalg.norm(a - b, dim=0) <= 1e-13 * t.linalg.norm(b, dim=0)).all()


@pytest.mark.parametrize("L,nr,nth,nv,ns,otf", STAGES)
def test_radius_slowest(torch_cuda, L, nr, nth, nv, ns, otf):
    t = torch_cuda
    print(f"[gpu] staged forward L={L} Nr={nr} Ntheta={nth} {nv}+{ns} per call={otf}", flush=True)
    cfg, nc = ShellConfig(L, nr, nth, max(2 * nth, 2 * L + 2)), 3 * nv + ns
    grid = t.from_numpy(np.random.default_rng(L).standard_normal(cfg.n_rtp(nc))).cuda()
    new = lambda n: t.full((n,), np.nan, dtype=t.float64, device="cuda")
    rtp, rtm, w, ref = new(cfg.n_rtp(nc)), new(cfg.n_rtm(nc)), new(cfg.n_rj(nc)), new(cfg.n_rj(nc))
    plan = SphTransPlan(cfg, max_ncomp=nc, p_on_the_fly=otf)
    try:
        plan.fft_forward(nc, grid, rtp)
        plan.exchange_rtp_to_rtm(nc, rtp, rtm)
        plan.legendre_forward(nv, ns, rtm, w)
        plan.sph_forward_transforms(nv, ns, grid, ref)
        t.cuda.synchronize()
    finally:
        plan.close()
    _close(t, w.view(-1, nc), ref.view(-1, nc))


@pytest.mark.parametrize("L,nr,nth,nv,ns", LARGE)
def test_large_calls(torch_cuda, L, nr, nth, nv, ns):
    t = torch_cuda
    print(f"[gpu] staged forward L={L} Nr={nr} Ntheta={nth} {nv}+{ns}", flush=True)
    cfg, nc = ShellConfig(L, nr, nth, 2 * nth), 3 * nv + ns
    g = t.Generator(device="cuda")
    g.manual_seed(L)
    grid = t.randn(cfg.n_rtp(nc), dtype=t.float64, device="cuda", generator=g)
    w = t.full((cfg.n_rj(nc),), np.nan, dtype=t.float64, device="cuda")
    plan = SphTransPlan(cfg, max_ncomp=nc)
    try:
        plan.sph_forward_transforms(nv, ns, grid, w)
        w, v = w.view(-1, nc), grid.view(nc, -1)
        for c0, c1 in [(3 * i, 3 * i + 3) for i in range(nv)] + [(i, i + 1) for i in range(3 * nv, nc)]:
            one = t.full((cfg.n_rj(c1 - c0),), np.nan, dtype=t.float64, device="cuda")
            field = (1, 0) if c1 - c0 == 3 else (0, 1)
            plan.sph_forward_transforms(*field, v[c0:c1].contiguous().view(-1), one)
            t.cuda.synchronize()
            _close(t, w[:, c0:c1], one.view(-1, c1 - c0))
    finally:
        plan.close()


@pytest.mark.parametrize("L,nr,nth", [(127, 190, 194), (100, 300, 166)])
def test_repeats(torch_cuda, L, nr, nth):
    """A last chunk of fewer than four K steps (25 and 21 of them: 97 and 83 rows):
    the waves of a work-group leave the product loop without a barrier and turn
    their results in the LDS that held the rows; repeated calls agree bit for
    bit."""
    t = torch_cuda
    print(f"[gpu] staged forward repeated L={L} Nr={nr} Ntheta={nth}", flush=True)
    cfg, nv = ShellConfig(L, nr, nth, 2 * nth), 8
    g = t.Generator(device="cuda")
    g.manual_seed(L)
    grid = t.randn(cfg.n_rtp(3 * nv), dtype=t.float64, device="cuda", generator=g)
    plan = SphTransPlan(cfg, max_ncomp=3 * nv)
    out = []
    try:
        for _ in range(4):
            w = t.full((cfg.n_rj(3 * nv),), np.nan, dtype=t.float64, device="cuda")
            plan.sph_forward_transforms(nv, 0, grid, w)
            out.append(w)
        t.cuda.synchronize()
    finally:
        plan.close()
    assert all(t.equal(out[0], w) for w in out[1:])
