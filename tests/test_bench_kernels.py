"""The kernels that the bench names, and the work that it counts, for what a
plan runs: sliced products only where the plan says so, the zonal form that it
reports, the FP64 Legendre kernels by the waves of a launch.  The first tests
run on the host with made-up times; the last asks plans for what they run."""
import glob
import os
import re

import pytest

import bench
from kemorin_mhd_amd import SHT_PREC_FP64, SHT_PREC_SPLIT_INT8, ShellConfig, ShtError, SphTransPlan

CSRC = os.path.join(os.path.dirname(bench.__file__), "kemorin_mhd_amd", "csrc", "*.hip")
STAGES = ("legendre_backward", "fft_backward", "fft_forward", "legendre_forward", "exchange",
          "legendre_backward_vector_kernel", "legendre_forward_vector_kernel")


def _res(sliced, fft, fused=False, otf=False, slow="legendre_forward_vector_kernel"):
    return dict(timers={s: (8.0 if s == slow else 2.0, 2) for s in STAGES}, steps=2, sliced=sliced,
                fft=fft, bwd_fused=fused, otf=otf)


@pytest.mark.parametrize("cfg,res,names", [
    ("cfg2", _res(False, 4), ("k_leg_bwd<true>", "k_leg_fwd_lds<true>", "k_fft3_bwd<512, 4>", "k_fft3_fwd<512, 8>")),
    ("cfg2", _res(True, 4, True), ("k_leg_bwd_split<6, 4, true>", "k_leg_fwd_split<6, 3, true>",
                                   "k_fft3_bwd<512, 4>", "k_fft3_fwd<512, 8>")),
    ("cfg2", _res(True, 0), ("k_leg_bwd_split<6, 3, true>", "k_leg_fwd_split<6, 3, true>",
                             "k_fft_bwd (mixed radix)", "k_fft_fwd (mixed radix)")),
    ("cfg1", _res(False, 4), ("k_leg_bwd<true>", "k_leg_fwd_lds<true>", "k_fft3_bwd<256, 4>", "k_fft3_fwd<256, 8>")),
    ("cfg1", _res(False, 3, otf=True), ("k_leg_bwd<true>", "k_leg_fwd", "k_fftz_bwd", "k_fftz_fwd")),
    ("cfg0", _res(False, 5), ("k_leg_bwd<false>", "k_leg_fwd", "k_zfold_bwd<true>", "k_zfold_fwd<true>")),
    ("cfg4", _res(False, 4, otf=True), ("k_leg_bwd<true>", "k_leg_fwd_lds<true>", "k_fft3_bwd<1024, 2>",
                                        "k_fft3_fwd<1024, 4>"))])
def test_names(cfg, res, names):
    got = bench.kernel_names(bench.CONFIGS[cfg], res, 6)
    assert tuple(got[s] for s in ("legendre_backward_vector_kernel", "legendre_forward_vector_kernel",
                                  "fft_backward", "fft_forward")) == tuple("ksht::" + n for n in names)
    src = "".join(open(f).read() for f in glob.glob(CSRC))
    for n in names:
        assert re.search(r"__global__[^;{]*\b%s\(" % re.split(r"[<( ]", n)[0], src), n


@pytest.mark.parametrize("sliced,factor,peak", [(False, 1, bench.FP64_PEAK_TFLOPS), (True, 21, bench.INT8_PEAK_TOPS)])
def test_slice_products_are_counted_where_they_run(sliced, factor, peak):
    cfg = bench.CONFIGS["cfg1"]
    roof, _ = bench.kernel_roofline(cfg, _res(sliced, 4, sliced), "split", 6)
    assert roof["work_per_launch"] == 15 * bench.flops_per_contraction(cfg) * factor
    assert roof["peak"] == peak


@pytest.mark.gpu
def test_plans_say_what_they_run(torch_cuda):
    for cfg, prec, variants, sliced, fft in [
            (ShellConfig(31, 3, 48, 96), SHT_PREC_SPLIT_INT8, {}, 0, 5),
            (ShellConfig(31, 3, 48, 96), SHT_PREC_SPLIT_INT8, {"split_all": 1, "fft_form": 4}, 1, 4),
            (ShellConfig(127, 3, 192, 384), SHT_PREC_FP64, {"split_all": 1}, 0, 4),
            (ShellConfig(44, 3, 68, 138), SHT_PREC_FP64, {"fft_form": 0}, 0, 0),
            (ShellConfig(44, 3, 68, 138), SHT_PREC_FP64, {"fft_form": 3}, 0, 3)]:
        plan = SphTransPlan(cfg, max_ncomp=4, precision=prec)
        try:
            for k, v in variants.items():
                plan.set_variant(k, v)
            assert (plan.get_variant("sliced"), plan.get_variant("fft_kernels")) == (sliced, fft)
            for name in ("sliced", "fft_kernels"):
                with pytest.raises(ShtError):
                    plan.set_variant(name, 0)
        finally:
            plan.close()
