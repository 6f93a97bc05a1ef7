"""Checkpoint strides of the adjoint on both sides of the workspace line below which every layer's state is kept (all
strides run alike there, so a stride's own kernels are reached only above it): batches above the line, the last
workgroup partly filled, against their own leading tracks run as a batch below it, the strides against each other in
every precision and arithmetic, and fits shorter than the stride or ending in a short segment."""
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


def _above_the_line(gp, nlayer):
    """Tracks just above the line: 48 MiB of workspace at stride 1 (p2r.h, p2r_forward_adjoint)."""
    size = 4 if gp == "f32" else 8
    per_track = (max(nlayer - 1, 1) * 27 + 1) * size + (112 if gp == "mixed" else 0)
    n = ((48 << 20) // per_track // BS + 1) * BS
    return n + BS if n % 256 == 0 else n


def _run_all(ctx, dt, dh, n, nlayer, gp, precision, stride):
    """All outputs of the first n tracks, on the GPU: {name: tensor}; per-track rows of the gradients as "grads"."""
    out = torch.empty(28 * n, device="cuda")
    g = {"chi2": torch.empty(n, device="cuda"), "grad_par": torch.empty(6 * n, device="cuda"),
         "grad_hits": torch.empty(3 * nlayer * n, device="cuda"), "grad_kfact": torch.empty(n, device="cuda"),
         "grad_global": torch.empty(4 * nlayer + 1, device="cuda", dtype=torch.float64)}
    ctx.forward_adjoint(dt, dh, out, Shape(1, n, nlayer, BS), grad_precision=gp, precision=precision,
                        checkpoint_stride=stride, **g)
    rows = [g["grad_par"].view(-1, 6, BS).transpose(1, 2).reshape(n, 6),
            g["grad_hits"].view(-1, 3 * nlayer, BS).transpose(1, 2).reshape(n, 3 * nlayer), g["grad_kfact"].view(n, 1)]
    return {"out": out, **g, "grads": torch.cat(rows, 1).double()}


def _bytes_equal(a, b):
    return torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8))


# bounds per track on the gradients' difference between strides, normwise: exact F32 recomputes the forward pass's words;
# elsewhere the compiler fuses the forward pass and a segment's recompute differently, and the last bits of a state
# show as tests/test_gpu_adjoint.py::test_checkpoint_stride_with_fused_arithmetic says
STRIDE_CASES = [("f32", "exact", 0.0), ("f32", "fast", 1.5e-2), ("mixed", "exact", 1e-5), ("mixed", "fast", 1e-5),
                ("f64", "exact", 1e-8)]


@pytest.mark.parametrize("nlayer", [1, 3, 5, 9, 20])
@pytest.mark.parametrize("gp,precision,tol", STRIDE_CASES)
def test_strides_above_the_line(ctx, gp, precision, tol, nlayer):
    """Every stride's own kernels (fits shorter than the stride, last segments of one layer, segment states in LDS and
    in the workspace) give the same gradients and global sums, and a track's words do not depend on how far the last
    workgroup is filled."""
    import p2r_amd
    n = _above_the_line(gp, nlayer)
    trk, hits = p2r_amd.gen_uniform(Shape(1, n + BS, nlayer, BS))
    dt, dh = torch.from_numpy(trk).cuda(), torch.from_numpy(hits).cuda()
    ref = _run_all(ctx, dt, dh, n, nlayer, gp, precision, 4)
    size = ref["grads"].norm(dim=1)
    total = ref["grads"][:, 6:6 + 3 * nlayer].abs().sum(0).view(nlayer, 3)  # per translation
    for stride in (1, 2, 4, 8):
        r = _run_all(ctx, dt, dh, n, nlayer, gp, precision, stride)
        longer = _run_all(ctx, dt, dh, n + BS, nlayer, gp, precision, stride)
        for k in ("out", "chi2", "grad_par", "grad_hits", "grad_kfact"):
            assert _bytes_equal(longer[k][:r[k].numel()], r[k]), (stride, k)
        if tol == 0.0:
            for k in r:
                assert _bytes_equal(r[k], ref[k]), (stride, k)
            continue
        assert torch.equal(torch.isfinite(r["grads"]), torch.isfinite(ref["grads"]))
        e = ((r["grads"] - ref["grads"]).norm(dim=1) / size)
        lead = e[:2048].max().item()
        within = (e < tol).double().mean().item()
        sums = ((r["grad_global"] - ref["grad_global"])[:-1].view(nlayer, 4)[:, :3].abs() / total).max().item()
        print(f"{gp} ({precision}) {nlayer} layers stride {stride} vs 4: 2048 tracks max {lead:.1e}, within {tol:g} "
              f"{within:.6f} of {n}, sums over the sum of magnitudes {sums:.1e}", flush=True)
        assert lead < tol and within > 0.999 and sums < tol


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
