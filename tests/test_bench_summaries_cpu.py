"""The counter summaries that the bench line reads for the current kernels are
committed, and their figures lie between the bytes the kernels cannot do
without and half as much again (a tenth for the FFT)."""
import os
import re
import sys

from conftest import ROOT

sys.path.insert(0, ROOT)
import bench  # noqa: E402  (module level holds only helpers; main() runs under __main__)


def test_folded_mode_product_traffic_per_field_pass():
    v = bench.measured_traffic("k_modeprod_fold_192cube_hbm_counters.md", "traffic_bytes_per_field_pass")
    assert v is not None and 8 * 2 * 196 ** 3 <= v < 1.5 * 8 * 2 * 196 ** 3


def test_fft_pass_traffic_of_six_strains():
    """Six passes over three packed pairs (8 bytes a point, read and written); the first reads twelve FP32 fields
    in the pairs' place."""
    v = bench.measured_traffic("k_fft2_f32_192cube_hbm_counters.md")
    alg = (11 * 3 * 8 + 12 * 4) / 6 * 192 ** 3
    assert v is not None and alg <= v < 1.1 * alg


def test_every_summary_the_bench_names_is_there():
    names = set(re.findall(r'"(\w+_counters\.md)"', open(os.path.join(ROOT, "bench.py")).read()))
    assert len(names) >= 4
    for name in names:
        assert os.path.exists(os.path.join(ROOT, "profiles", name)), name
