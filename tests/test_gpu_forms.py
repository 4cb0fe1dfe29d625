"""Sliced products and the mixed-radix FFT at the sizes of the other test
modules, where plans choose FP64 products and a folded DFT by default: the
tests of those modules once more, unchanged, on plans that are given the other
form when they are created.  Sliced: every slice count and spectrum, both MFMA
forms, fused scalars, 64 components, P per call, graph capture, the fixed
workspace, the autotuner, the finite check.  Mixed radix: its radices, direct
sums and Bluestein passes."""
import pytest

import test_gpu_batch
import test_gpu_finite
import test_gpu_many_fields
import test_gpu_otf
import test_gpu_shells64
import test_gpu_split
import test_gpu_sweep
import test_gpu_tune
import test_zz_no_alloc
from kemorin_mhd_amd import SHT_PREC_SPLIT_INT8, ShellConfig, SphTransPlan, batched_shell_draw
from test_gpu_split import case  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu

MODULES = (test_gpu_batch, test_gpu_finite, test_gpu_many_fields, test_gpu_otf, test_gpu_shells64,
           test_gpu_split, test_gpu_sweep, test_gpu_tune, test_zz_no_alloc)
SPLIT = SHT_PREC_SPLIT_INT8


class SlicedPlan(SphTransPlan):
    def __init__(self, *a, **kw):
        super().__init__(*a, **kw)
        if self.precision == SPLIT:
            self.set_variant("split_all", 1)


class MixedRadixPlan(SphTransPlan):
    def __init__(self, *a, **kw):
        super().__init__(*a, **kw)
        self.set_variant("fft_form", 0)


def _plans(monkeypatch, cls):
    for m in MODULES:
        monkeypatch.setattr(m, "SphTransPlan", cls)
    # the 64 shells of the batch test take long: the first dozen
    monkeypatch.setattr(test_gpu_shells64, "batched_shell_draw", lambda n: batched_shell_draw(n)[:12])


@pytest.fixture
def sliced(monkeypatch):
    _plans(monkeypatch, SlicedPlan)


@pytest.fixture
def mixed(monkeypatch):
    _plans(monkeypatch, MixedRadixPlan)


@pytest.mark.parametrize("S", [4, 5, 6, 7])
@pytest.mark.parametrize("slope", [1.5, 3.0])
def test_round_trip(case, torch_cuda, sliced, S, slope):  # noqa: F811
    test_gpu_split.test_split_roundtrip_vs_oracle(case, torch_cuda, S, slope)


def test_stage_scalars(case, torch_cuda, sliced):  # noqa: F811
    test_gpu_split.test_split_stage_scalars(case, torch_cuda)


@pytest.mark.parametrize("nv,ns", [(1, 1), (3, 4), (0, 3)])
def test_component_groups(case, torch_cuda, sliced, nv, ns):  # noqa: F811
    test_gpu_split.test_split_component_groups(case, torch_cuda, nv, ns)


@pytest.mark.parametrize("S", [4, 6, 7])
@pytest.mark.parametrize("nv,ns", [(3, 0), (1, 2), (0, 4)])
def test_mfma32(case, torch_cuda, sliced, S, nv, ns):  # noqa: F811
    test_gpu_split.test_forward_mfma32_bitexact_vs_mfma16(case, torch_cuda, S, nv, ns)


@pytest.mark.parametrize("S", [4, 5, 6, 7])
@pytest.mark.parametrize("nv,ns", [(2, 2), (1, 1), (2, 1), (1, 4), (3, 0)])
def test_fused_scalars(case, torch_cuda, sliced, S, nv, ns):  # noqa: F811
    test_gpu_split.test_backward_fused_scalars_bitexact(case, torch_cuda, S, nv, ns)


@pytest.mark.parametrize("otf", [False, True])
@pytest.mark.parametrize("name", list(test_gpu_many_fields.SHELLS))
def test_64_components(torch_cuda, sliced, name, otf):
    test_gpu_many_fields.test_64_components_vs_oracle(torch_cuda, name, otf, SPLIT, 1e-11)


@pytest.mark.parametrize("cfg", [ShellConfig(127, 9, 192, 384), ShellConfig(63, 5, 97, 196)],
                         ids=["L127", "L63_odd"])
def test_p_per_call(torch_cuda, sliced, cfg):
    test_gpu_otf.test_tables_per_call_bitexact_vs_stored(torch_cuda, SPLIT, cfg)


def test_p_per_call_graph(torch_cuda, sliced):
    test_gpu_otf.test_tables_per_call_under_graph_replay(torch_cuda)


def test_batch_graph(torch_cuda, sliced):
    test_gpu_batch.test_batch_graph_matches_eager(torch_cuda, SPLIT)


def test_shells_graph(torch_cuda, sliced):
    test_gpu_shells64.test_shells64_graph_vs_oracle(torch_cuda, SPLIT, 1e-11)


def test_autotune(torch_cuda, sliced, tmp_path):
    test_gpu_tune.test_autotune_cache_and_parity(torch_cuda, tmp_path, SPLIT, 1e-11)


def test_check_finite(torch_cuda, sliced):
    test_gpu_finite.test_check_finite_matches_output(torch_cuda, SPLIT)


def test_fixed_workspace(torch_cuda, sliced):
    test_zz_no_alloc.test_noalloc_matches_backward(torch_cuda, SPLIT)


@pytest.mark.parametrize("cfg", test_gpu_sweep.SHELLS + test_gpu_sweep.TINY,
                         ids=lambda c: f"L{c.L}_nth{c.nth}_nphi{c.nphi}")
@pytest.mark.parametrize("form", ["sliced", "mixed"])
def test_sweep(torch_cuda, request, form, cfg):
    request.getfixturevalue(form)
    if cfg in test_gpu_sweep.TINY:
        test_gpu_sweep.test_tiny_shells(torch_cuda, cfg)
    else:
        test_gpu_sweep.test_whole_transform_sweep(torch_cuda, cfg)


def test_mixed_radix_shells(torch_cuda, mixed):
    test_gpu_shells64.test_shells64_graph_vs_oracle(torch_cuda, 0, 1e-12)
