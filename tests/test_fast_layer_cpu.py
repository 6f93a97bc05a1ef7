"""The fast instance's regrouped layer (p2r_fast_layer.inc) on the CPU.

tests/fast_layer_harness.cpp builds it on the host beside the same layer in FP64 by the reference's formulas
(tbb.cpp:656-812, :433-642).  A track that has no finite result there (a hit on the z axis, an infinite or missing
coordinate, a zero charge or curvature) has none in the fast arithmetic either, and ordinary tracks agree.
"""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_fast_layer_against_the_formulas_in_fp64(tmp_path):
    exe = str(tmp_path / "flh")
    subprocess.run(["g++", "-std=c++17", "-O1", "-o", exe, os.path.join(HERE, "fast_layer_harness.cpp")], check=True)
    *cases, last = subprocess.run([exe, "200000"], capture_output=True, text=True, check=True).stdout.splitlines()
    assert not cases, "an output is finite in one arithmetic only"
    par, cov = (float(v) for v in last.split()[1:])
    print(f"max difference over the propagated sigma: parameters {par:.1e}, covariance {cov:.1e}", flush=True)
    # x has the smallest propagated sigma, 4e-3 and more, and an ulp of 2e-6 at up to 20: four ulps over five steps
    assert par < 2e-3
    # a term of J P J^T is up to 10 times its sum (j00 = 1 + U g0 all but cancels) at 2^-24 each, over 20 products
    assert cov < 2e-3
