"""Checkpoint strides of the adjoint on both sides of the workspace line below which every layer's state is kept: a
batch above it (every stride's own kernels, the last workgroup partly filled) against its own leading tracks run as a
batch below it, and the strides against each other."""
import numpy as np
import pytest

from p2r_amd import Shape

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

# 48 MiB hold 24 500 tracks x 20 layers of FP32 states and 12 000 of FP64 ones
LARGE, SMALL, BS, NL = 33000, 1056, 33, 20


@pytest.fixture(scope="module")
def ctx():
    import p2r_amd
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return p2r_amd.Context(0)


def _run(ctx, dt, dh, n, gp, stride):
    shape = Shape(1, n, NL, BS)
    out = torch.empty_like(dt)
    g = {"chi2": torch.empty(n, device="cuda"), "grad_par": torch.empty(6 * n, device="cuda"),
         "grad_hits": torch.empty(3 * NL * n, device="cuda"), "grad_kfact": torch.empty(n, device="cuda")}
    ctx.forward_adjoint(dt, dh, out, shape, grad_precision=gp, checkpoint_stride=stride, **g)
    return [t.cpu().numpy() for t in (out, *g.values())]


# F32 recomputes the forward pass's words; the FP64 states of the others may differ in their last bits, which shows
# in the FP32 outputs as a last-bit difference here and there (MIXED: as its FP32 reverse amplifies it)
@pytest.mark.parametrize("gp,tol", [("f32", 0.0), ("mixed", 1e-5), ("f64", 2.0 ** -23)])
def test_strides_agree_across_the_workspace_line(ctx, gp, tol):
    import p2r_amd
    trk, hits = p2r_amd.gen_uniform(Shape(1, LARGE, NL, BS))
    dt, dh = torch.from_numpy(trk).cuda(), torch.from_numpy(hits).cuda()
    small = _run(ctx, dt[:28 * SMALL].clone(), dh[:9 * NL * SMALL].clone(), SMALL, gp, 4)
    ref = None
    for stride in (1, 2, 4, 8):
        large = _run(ctx, dt, dh, LARGE, gp, stride)
        ref = large if ref is None else ref
        for a, b, s in zip(large, ref, small):
            if tol == 0.0:
                assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), stride
                assert np.array_equal(a[:s.size].view(np.uint32), s.view(np.uint32)), stride
            else:
                for x, y in ((a, b), (a[:s.size], s)):
                    ok = np.isfinite(y)
                    assert np.array_equal(ok, np.isfinite(x))
                    assert np.linalg.norm((x - y)[ok]) <= tol * np.linalg.norm(y[ok]), stride


@pytest.mark.parametrize("gp", ["f32", "mixed", "f64"])
def test_a_context_warmed_with_its_largest_batch_allocates_no_more(gp):
    """A batch below the line keeps every layer's state and so can need more workspace than a larger one above it: the
    larger one's call reserves that too, so that no smaller batch makes the context allocate, which a stream capture
    would not allow."""
    import p2r_amd
    ctx = p2r_amd.Context(0)
    n = LARGE
    trk, hits = p2r_amd.gen_uniform(Shape(1, n, NL, BS))
    dt, dh = torch.from_numpy(trk).cuda(), torch.from_numpy(hits).cuda()
    out, chi2 = torch.empty_like(dt), torch.empty(n, device="cuda")
    gg = torch.empty(4 * NL + 1, device="cuda", dtype=torch.float64)

    def call(m):
        ctx.forward_adjoint(dt, dh, out, Shape(1, m // BS * BS, NL, BS), grad_precision=gp, checkpoint_stride=4, chi2=chi2,
                            grad_global=gg)

    call(n)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    sizes = (24000, 22000, 12100, 11900, 5000, 64)
    for m in sizes:
        call(m)
        torch.cuda.synchronize()
        assert torch.cuda.mem_get_info()[0] == free, m
    # and under capture, which refuses an allocation
    for m in sizes[1:4]:
        call(m)
        want = [t.clone() for t in (out, chi2, gg)]
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            call(m)
        for _ in range(3):
            for t in (out, chi2, gg):
                t.fill_(float("nan"))
            g.replay()
            torch.cuda.synchronize()
            k = m // BS * BS
            for a, b, c in ((out, want[0], 28 * k), (chi2, want[1], k), (gg, want[2], gg.numel())):
                assert torch.equal(a[:c].view(torch.uint8), b[:c].view(torch.uint8)), m
    ctx.close()
