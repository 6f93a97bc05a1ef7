"""The exact instance's short forms (p2r_lane_math.inc) on the CPU: its own sine and cosine against long double, and which
forms a propagation takes.

tests/exact_forms_harness.cpp builds that code on the host.  A wavefront with an operand that the short forms do not
cover goes straight to the general ones, and an angle whose sine or cosine is in doubt costs the library's call and
nothing else: none of it works an iteration out twice.
"""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def lines(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("forms") / "forms")
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-o", exe,
                    os.path.join(HERE, "exact_forms_harness.cpp")], check=True)
    out = subprocess.run([exe, "331"], capture_output=True, text=True, check=True).stdout
    return {name: [float(v) for v in rest] for name, *rest in (line.split() for line in out.splitlines())}


def test_short_sincos_against_long_double(lines):
    e_sin, e_cos = lines["ulps"]
    print(f"sin {e_sin} cos {e_cos} ulps of FP64, |r| - pi/4 up to {lines['remainder'][0]}", flush=True)
    # 256 ulps from a midpoint decide: half of that is the margin asked for
    assert e_sin < 128 and e_cos < 128
    assert lines["remainder"][0] < 1.7e-4
    assert lines["words"] == [0]


def test_forms_taken(lines):
    """[short square roots, general square roots, library sine/cosine calls]; a propagation has 7 roots."""
    short, general = [7, 0, 0], [0, 7, 0]
    assert lines["ordinary"] == short
    assert lines["phi=0"] == lines["phi=-0"] == short
    for name in ("x=0", "y=-0", "ipt=0", "ipt=NaN"):
        assert lines[name] == general, name
    for name in ("phi=unsure", "theta=unsure", "phi=8192"):
        assert lines[name] == [7, 0, 2], name
    # seen only by the iterations themselves: a radius beyond 2^12, sin theta = 0, a NaN angle
    for name, library in (("x=2^13", 0), ("theta=0", 0), ("phi=NaN", 2)):
        assert lines[name] == [7, 7, library], name
