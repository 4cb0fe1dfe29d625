"""The FP64 Legendre kernels at the edges of their tiles and dispatch, against
the oracle: one degree per parity and less, order counts at the ends of a K
step, radii at, below and past a column tile (flattened over the fields), odd
Ntheta (an equator row), single kinds of field, calls on both sides of the
packing rule, and P tables per call.  Bound 1e-12 per call as elsewhere."""
import numpy as np
import pytest

import oracle as O
from kemorin_mhd_amd import ShellConfig, SphTransPlan

pytestmark = pytest.mark.gpu

# (L, Nr, Ntheta, vectors, scalars, P per call)
CASES = [(1, 1, 2, 1, 1, False), (2, 2, 5, 0, 1, False), (5, 3, 7, 1, 2, False),
         (7, 16, 9, 3, 0, True), (15, 17, 24, 2, 3, False), (31, 5, 48, 2, 2, False),
         (31, 33, 47, 0, 5, False), (40, 17, 43, 1, 3, True), (63, 33, 96, 3, 5, True),
         (64, 16, 97, 2, 1, False), (100, 20, 151, 2, 0, False), (127, 18, 192, 2, 1, True)]


@pytest.mark.parametrize("L,nr,nth,nv,ns,otf", CASES)
def test_fp64_legendre(torch_cuda, L, nr, nth, nv, ns, otf):
    t = torch_cuda
    print(f"[gpu] FP64 Legendre L={L} Nr={nr} Ntheta={nth} {nv}+{ns} per call={otf}", flush=True)
    cfg, nc = ShellConfig(L, nr, nth, max(2 * nth, 2 * L + 2)), 3 * nv + ns
    orc = O.OraclePlan(cfg.L, cfg.nr, cfg.nth, cfg.nphi, cfg.radius(), full_tables=False)
    rng = np.random.default_rng(L)
    sp, grid = rng.standard_normal(cfg.n_rj(nc)), rng.standard_normal(cfg.n_rtp(nc))
    v = t.full((cfg.n_rtp(nc),), np.nan, dtype=t.float64, device="cuda")
    w = t.full((cfg.n_rj(nc),), np.nan, dtype=t.float64, device="cuda")
    plan = SphTransPlan(cfg, max_ncomp=nc, p_on_the_fly=otf)
    try:
        plan.sph_backward_transforms(nv, ns, t.from_numpy(sp).cuda(), v)
        plan.sph_forward_transforms(nv, ns, t.from_numpy(grid).cuda(), w)
        t.cuda.synchronize()
    finally:
        plan.close()
    v, w = v.cpu().numpy().reshape(nc, -1), w.cpu().numpy().reshape(-1, nc)
    # the oracle field by field: in one call its FFTs pair neighbouring lines
    # of different components, and a radial component, l (l + 1) times the
    # others here, rounds into its neighbour (1.1e-12 of a scalar)
    rv, rw = np.empty_like(v), np.empty_like(w)
    sp, grid = sp.reshape(-1, nc), grid.reshape(nc, -1)
    for c0, c1 in [(3 * i, 3 * i + 3) for i in range(nv)] + [(i, i + 1) for i in range(3 * nv, nc)]:
        field = (1, 0) if c1 - c0 == 3 else (0, 1)
        rv[c0:c1] = orc.backward(*field, np.ascontiguousarray(sp[:, c0:c1]).ravel()).reshape(c1 - c0, -1)
        rw[:, c0:c1] = orc.forward(*field, np.ascontiguousarray(grid[c0:c1]).ravel()).reshape(-1, c1 - c0)
    assert (np.linalg.norm(v - rv, axis=1) <= 1e-12 * np.linalg.norm(rv, axis=1)).all()
    assert (np.linalg.norm(w - rw, axis=0) <= 1e-12 * np.linalg.norm(rw, axis=0)).all()
