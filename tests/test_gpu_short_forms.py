"""The exact arithmetic's short square root, reciprocal, division and sine/cosine (p2r_lane_math.inc) against the general
ones, word for word: the roots, reciprocals and angles by exhaustion over their range and beyond, the quotients over every
divisor significand with half the dividends aimed at rounding midpoints, FP64 reciprocals at random."""
import ctypes
import os

import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "p2r-tests_amd", "lib",
                   "libp2r_short_forms.so")


def _bits(exponent):
    return (127 + exponent) << 23


@pytest.fixture(scope="module")
def count():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    lib = ctypes.CDLL(LIB)

    def run(name, *args):
        counts = torch.zeros(2, dtype=torch.int64, device="cuda")
        stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        assert getattr(lib, name)(*args, ctypes.c_void_p(counts.data_ptr()), stream) == 0
        bad, compared = counts.tolist()
        print(f"{name}: {bad} of {compared} differ", flush=True)
        return bad, compared
    return run


@pytest.mark.parametrize("which", [0, 1])
def test_every_root_and_reciprocal(count, which):
    lo, hi = _bits(-60), _bits(60)
    assert count("short_forms_floats", ctypes.c_uint32(lo), ctypes.c_uint32(hi), which) == (0, hi - lo + 1)


def test_every_sine_and_cosine(count):
    """Every angle of -2^12 .. 2^12 whose sine and cosine the short form is sure of: all but a few in a million."""
    hi = _bits(12)
    bad, compared = count("short_forms_floats", ctypes.c_uint32(0), ctypes.c_uint32(hi), 2)
    assert bad == 0
    assert (1 - 1e-5) * 2 * (hi + 1) < compared <= 2 * (hi + 1)


def test_quotients(count):
    assert count("short_forms_quotients", 64) == (0, 64 << 23)


def test_fp64_reciprocals(count):
    assert count("short_forms_reciprocals64", ctypes.c_uint64(1 << 30)) == (0, 1 << 30)
