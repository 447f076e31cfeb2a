"""The benchmark's recorded HBM traffic: every profile that a bench line quotes has its figure, of the kernel that the
line times and of about the kernel's own bytes."""
import os
import sys

import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))

import bench  # noqa: E402

N, NA = 1024 * 1024, {"color_sr_c1": 258 * 258, "color_sr_c3": 2052 * 2052}


@pytest.mark.parametrize("path,kernel,nbytes", [
    (bench.PROFILE, "k_cgcg_st2", 144 * N),
    (*bench.COLOR_TRAFFIC["color_sr_c1"], 4 * 8 * NA["color_sr_c1"] + 80 * 256 * 256),
    (*bench.COLOR_TRAFFIC["color_sr_c3"], 4 * 13 * NA["color_sr_c3"] + 80 * 2048 * 2048)])
def test_profiles_record_the_traffic_that_bench_quotes(path, kernel, nbytes):
    traffic = bench.measured_traffic(path)
    assert traffic is not None and 0.95 * nbytes < traffic < 1.5 * nbytes
    assert kernel in open(path).readline()
