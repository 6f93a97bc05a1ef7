"""Small batches in reference semantics, whose layers are dealt to several wavefronts: in exact arithmetic every word of
the tracks and of chi2 (summed and per layer) equals the oracle's, at tile ends, with layer counts that leave wavefronts without a layer,
on both sides of the line to the one-wavefront kernel, and with the output over the input."""
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


def _same(a, b):
    a, b = np.asarray(a, np.float32).ravel(), np.asarray(b, np.float32).ravel()
    return bool(((a.view(np.uint32) == b.view(np.uint32)) | (np.isnan(a) & np.isnan(b))).all())


@pytest.mark.parametrize("n,nlayer,bsize", [(1, 2, 1), (63, 3, 1), (65, 17, 1), (64, 64, 32), (132, 20, 33), (4096, 5, 64),
                                            (131072, 3, 32), (131104, 3, 32)])
@pytest.mark.parametrize("options", [0, 7])
def test_split_layers_match_oracle(orc, ctx, n, nlayer, bsize, options):
    import p2r_amd
    shape = Shape(1, n, nlayer, bsize)
    trk, hits = p2r_amd.gen_uniform(shape)
    if options:
        trk.reshape(shape.nblk, 28, bsize)[:, 3] *= -1  # the charge option flips these
    want, want_chi2 = orc.run_f32(trk, hits, shape.nblk, nlayer, bsize, semantics=0, cr_trig=True, chi2=True,
                                  options=options)
    dt, dh = torch.from_numpy(trk).cuda(), torch.from_numpy(hits).cuda()
    params = p2r_amd.default_params("exact", options=options)
    for chi2 in (False, True):
        for in_place in (False, True):
            src = dt.clone()
            out = src if in_place else torch.full_like(src, 5.0)
            c = torch.full((n * (nlayer if options & 4 else 1),), -1.0, device="cuda") if chi2 else None
            ctx.forward(src, dh, out, shape, "reference", params=params, chi2=c)
            what = f"n {n} nlayer {nlayer} bsize {bsize} options {options} chi2 {chi2} in place {in_place}"
            assert _same(out.cpu().numpy(), want), what
            if chi2:
                assert _same(c.cpu().numpy(), want_chi2), what


@pytest.mark.parametrize("n,nlayer", [(96000, 20), (65536, 7), (131072, 3)])
def test_split_layers_in_fast_arithmetic(orc, ctx, n, nlayer):
    """Tracks and chi2 are as close to the oracle as the reference's own fast-math build is (with no chi2, summed and per
    layer: a kernel each), and the sum over the layers, taken in their order from what the wavefronts left, is the sum
    of the chi2 per layer to the word."""
    import oracle
    import p2r_amd
    import parity
    shape = Shape(1, n, nlayer, 32)
    trk, hits = p2r_amd.gen_uniform(shape)
    cpu, c2_cpu = orc.run_f32(trk, hits, shape.nblk, nlayer, 32, semantics=0, chi2=True)
    alt, c2_alt = oracle.Oracle("liboracle_bench.so").run_f32(trk, hits, shape.nblk, nlayer, 32, semantics=0, chi2=True)
    par64, cov64, _ = orc.run_f64(trk, hits, shape.nblk, nlayer, 32, semantics=0)
    dt, dh = torch.from_numpy(trk).cuda(), torch.from_numpy(hits).cuda()

    def run(options, chi2):
        out = torch.empty_like(dt)
        c = torch.full((n * (nlayer if options & 4 else 1),), -1.0, device="cuda") if chi2 else None
        ctx.forward(dt, dh, out, shape, "reference", params=p2r_amd.default_params("fast", options=options), chi2=c)
        res = parity.compare_statistical(out.cpu().numpy(), cpu, alt, 32, par64, cov64)
        assert res["ok"], res
        return c.cpu().numpy() if chi2 else None

    run(0, False)
    total, layers = run(0, True), run(4, True).reshape(nlayer, n)
    want = np.zeros(n, np.float32)
    for row in layers:
        want += row
    assert _same(total, want)

    def distance(c):
        return np.quantile(np.abs(c - c2_cpu) / np.abs(c2_cpu), [0.5, 0.9, 0.99])

    got, allowed = distance(total), distance(c2_alt)
    print(f"chi2 against the oracle, quantiles 0.5 0.9 0.99: {got}, the reference's fast-math build {allowed}", flush=True)
    assert (got <= 2 * allowed).all()  # the same sums grouped differently: no closer agreement is asked for
