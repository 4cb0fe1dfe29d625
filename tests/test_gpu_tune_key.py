"""What keeps autotuner cache entries apart: an entry of another kernel set
(files written before the set was part of the key) and one of the other kind
of products are not taken."""
import json

import pytest

from kemorin_mhd_amd import SHT_PREC_FP64, SHT_PREC_SPLIT_INT8, ShellConfig, SphTransPlan

pytestmark = pytest.mark.gpu


def test_entry_of_earlier_kernels_is_not_taken(torch_cuda, tmp_path):
    cfg = ShellConfig(44, 3, 68, 138)  # Nphi = 2 3 23
    cache = tmp_path / "tune.json"
    key = "L=44 nr=3 nth=68 nphi=138 prec=0 slices=0 p_otf=0 bwd=1,1 fwd=1,1"
    cache.write_text('{"kemorin_sht_autotune": 1, "entries": [\n{"key": "%s", "split_fwd_mfma": 16, '
                     '"fft_form": 0, "ms": 12345.0, "default_ms": 12345.0}\n]}\n' % key)
    print("[gpu] autotune with a cache entry of earlier kernels", flush=True)
    plan = SphTransPlan(cfg, max_ncomp=4, precision=SHT_PREC_FP64)
    try:
        r = plan.autotune(1, 1, 1, 1, cache=str(cache))
        assert r["ms"] < 12345.0
        assert len(json.loads(cache.read_text())["entries"]) == 2
        again = plan.autotune(1, 1, 1, 1, cache=str(cache))
        assert again["ms"] == pytest.approx(r["ms"], abs=1e-3)
    finally:
        plan.close()


def test_products_are_part_of_the_key(torch_cuda, tmp_path):
    cfg = ShellConfig(31, 5, 48, 96)
    cache = tmp_path / "tune.json"
    for n, split_all in ((1, 0), (2, 1), (2, 0), (2, 1)):
        print(f"[gpu] autotune split_all={split_all}", flush=True)
        plan = SphTransPlan(cfg, max_ncomp=4, precision=SHT_PREC_SPLIT_INT8)
        try:
            plan.set_variant("split_all", split_all)
            plan.autotune(1, 1, 1, 1, cache=str(cache))
        finally:
            plan.close()
        assert len(json.loads(cache.read_text())["entries"]) == n
