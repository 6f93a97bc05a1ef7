"""The exact arithmetic's short square root, reciprocal and division, and the general ones a wavefront falls back
to, on both sides of the line between them (operands of 2^-24 .. 2^24): every word equals the oracle's.

Each edge sits in one lane of an otherwise ordinary wavefront, and a batch of one track has it alone."""
import numpy as np
import pytest

from p2r_amd import Shape

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def ctx():
    import p2r_amd
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return p2r_amd.Context(0)


def _two(e):
    return np.float32(2.0 ** e)


ALL_ONES = np.float32(np.ldexp(2 ** 24 - 1, -20))  # a significand of ones, the reciprocal's hardest operand

# (field of the track or of layer 0's hit, value) per lane
EDGES = [
    [("par", 0, np.float32(0.0))], [("par", 1, np.float32(-0.0))], [("par", 0, np.float32(0.0)), ("par", 1, np.float32(0.0))],
    [("par", 0, _two(-24))], [("par", 0, np.nextafter(_two(-24), np.float32(0)))], [("par", 1, -_two(-30))],
    [("par", 0, _two(11))], [("par", 0, _two(12))], [("par", 1, _two(13))], [("par", 0, _two(40))],
    [("par", 3, _two(24))], [("par", 3, _two(25))], [("par", 3, _two(-24))], [("par", 3, -_two(-25))],
    [("par", 3, ALL_ONES)], [("par", 0, ALL_ONES), ("par", 1, _two(-24))],
    [("par", 5, np.float32(0.0))], [("par", 5, _two(-25))], [("par", 5, np.float32(np.pi))], [("par", 4, np.float32(1e6))],
    [("hit", 0, np.float32(0.0)), ("hit", 1, np.float32(0.0))], [("hit", 0, _two(12))], [("hit", 1, _two(20))],
    [("hit", 0, np.float32(0.0))], [("hit", 0, np.float32(3.0)), ("hit", 1, ALL_ONES)], [("par", 2, np.float32(np.inf))],
    [("par", 3, np.float32(np.nan))], [("hit", 1, np.float32(np.inf))],
]


@pytest.mark.parametrize("semantics", ["reference", "chained"])
@pytest.mark.parametrize("nlayer", [1, 3])
def test_exact_words_on_both_sides_of_the_short_forms_range(orc, ctx, semantics, nlayer):
    from test_gpu_parity import check_exact
    import p2r_amd
    for bsize in (32, 1):
        n = 64 * len(EDGES) if bsize == 32 else len(EDGES)
        shape = Shape(1, n, nlayer, bsize)
        trk, hits = p2r_amd.gen_uniform(shape)
        t = trk.reshape(shape.nblk, 28, bsize)
        h = hits.reshape(shape.nblk, nlayer, 9, bsize)
        for i, edge in enumerate(EDGES):
            g = 64 * i + (i * 7) % 64 if bsize == 32 else i
            for kind, f, v in edge:
                (t[g // bsize, f] if kind == "par" else h[g // bsize, 0, f])[g % bsize] = v
        check_exact(orc, ctx, trk, hits, shape, semantics, f"range edges bsize {bsize} nlayer {nlayer}")


@pytest.mark.parametrize("kfact", [2.0 ** -24, 2.0 ** -25, -2.0 ** 24, 2.0 ** 25, 0.0])
def test_exact_propagation_at_the_ends_of_kfact(orc, ctx, kfact):
    """The curvature constant at the range's ends and outside, through the block entry point."""
    import p2r_amd
    bs, nblk = 32, 4
    shape = Shape(1, bs * nblk, 1, bs)
    trk, hits = p2r_amd.gen_uniform(shape)
    dt, dh = torch.from_numpy(trk).cuda(), torch.from_numpy(hits).cuda()
    do = torch.zeros_like(dt)
    ctx.propagateToR(dt[6 * bs:], dt[0:], dt[27 * bs:], dh, do[6 * bs:], do[0:], bs, nblk, 28 * bs, 9 * bs, kfact=kfact)
    gpu = do.cpu().numpy().reshape(nblk, 28, bs)
    orc.lib.orc_set_trig_mode(1)
    try:
        for b in range(nblk):
            tb = trk.reshape(nblk, 28 * bs)[b]
            e, p = orc.propagate_block(bs, kfact, tb[6 * bs:27 * bs].copy(), tb[:6 * bs].copy(),
                                       tb[27 * bs:].view(np.int32).copy(), hits.reshape(nblk, 9 * bs)[b, :3 * bs].copy())
            want, got = np.concatenate([p, e]), gpu[b, :27].ravel()
            same = (want.view(np.uint32) == got.view(np.uint32)) | (np.isnan(want) & np.isnan(got))
            assert same.all()
    finally:
        orc.lib.orc_set_trig_mode(0)


# angles (FP32 bits) whose sine or cosine lies within 250 ulps of FP64 of the midpoint between two floats
UNSURE = [0xc0259f7c, 0x40096e02, 0xbfe3343a, 0xc04549a0, 0xbfe9c645, 0x3e659fc6, 0x3cb0bc91, 0x4010a4bf, 0x3ffedd26,
          0x3fadffc7, 0xbe5c11ed]
# the ends of the range of the kernels' own sine and cosine, and around it; multiples of pi/2
ANGLES = [2.0 ** -24, np.nextafter(np.float32(2.0 ** -24), np.float32(0)), -(2.0 ** -30), 0.0, -0.0, 1e-40, 4096.0,
          np.nextafter(np.float32(4096), np.float32(5000)), -4095.9, 1e5, 3e38, np.inf, np.nan,
          *(k * np.pi / 2 for k in (-2607, -5, -2, -1, 1, 2, 3, 4, 101, 2607)), np.pi / 4, -3 * np.pi / 4, 2.356]


@pytest.mark.parametrize("field", [4, 5])
@pytest.mark.parametrize("semantics", ["reference", "chained"])
def test_exact_sine_and_cosine_words(orc, ctx, semantics, field):
    """phi (4) and theta (5) at the ends of their range, at multiples of pi/2 and where the FP32 rounding of a sine or
    cosine is in doubt, one per wavefront and all in a few wavefronts."""
    from test_gpu_parity import check_exact
    import p2r_amd
    angles = np.concatenate([np.array(UNSURE, np.uint32).view(np.float32), np.array(ANGLES, np.float32)])
    for spread in (64, 1):
        n = 32 * (-(-len(angles) * spread // 32))
        shape = Shape(1, n, 2, 32)
        trk, hits = p2r_amd.gen_uniform(shape)
        t = trk.reshape(shape.nblk, 28, 32)
        for i, a in enumerate(angles):
            t[i * spread // 32, field, i * spread % 32] = a
        check_exact(orc, ctx, trk, hits, shape, semantics, f"angles field {field} spread {spread}")
