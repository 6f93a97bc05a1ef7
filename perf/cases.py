"""Timed workloads of the p2r library: what its users have it do, from one Matriplex block pair to the largest
batches, through the public entry points of p2r_amd.

Forward fits (uniform batches, both layer semantics, both arithmetics), uneven batches with masked layers, and the
chained fit with its adjoint (per-track gradients, the alignment sums, and the torch.autograd.Function).  Inputs are
the library's own benchmark distribution (p2r_gen.h, P2R_GEN_CONSISTENT) drawn on the GPU: each track's true state is
the base state smeared by 10 %, its hits lie on its own helix plus 100 um of noise, and the fit starts from the true
state plus noise of the input covariance.
"""
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "p2r-tests_amd"))
import p2r_amd  # noqa: E402
from p2r_amd import Shape  # noqa: E402

FLOPS_FORWARD = 1212  # useful FP32 operations of one track-layer update
FLOPS_ADJOINT = 3319  # the same with its reverse


def _forward(name, nevts, ntrks, nlayer, bsize, semantics, precision, chi2=False, options=0):
    return {"name": name, "kind": "forward", "nevts": nevts, "ntrks": ntrks, "nlayer": nlayer, "bsize": bsize,
            "semantics": semantics, "precision": precision, "chi2": chi2, "options": options}


def _ragged(name, nevts, median, nlayer, bsize, semantics, precision, chi2):
    return {"name": name, "kind": "ragged", "nevts": nevts, "median": median, "nlayer": nlayer, "bsize": bsize,
            "semantics": semantics, "precision": precision, "chi2": chi2}


def _adjoint(name, nevts, ntrks, nlayer, bsize, precision, grad, stride, outputs):
    return {"name": name, "kind": "adjoint", "nevts": nevts, "ntrks": ntrks, "nlayer": nlayer, "bsize": bsize,
            "precision": precision, "grad": grad, "stride": stride, "outputs": outputs}


def listed():
    return [
        # The smallest call: a wavefront's worth of tracks through all layers, as an online fit of one region does.
        _forward("blocks_chained", 1, 64, 20, 32, "chained", "exact", chi2=True),
        # One event of the reference's own size, its layer semantics: the unit an event loop hands over.
        _forward("event_reference", 1, 9600, 20, 32, "reference", "exact"),
        # One event fitted in the fast arithmetic.
        _forward("event_chained_fast", 1, 9600, 20, 32, "chained", "fast", chi2=True),
        # Ten events, the chained Kalman fit: the configuration that also runs on a CPU.
        _forward("ten_events_chained", 10, 9600, 20, 32, "chained", "exact"),
        # Odd sizes with every physics option: a detector of 13 layers, a Matriplex width of 17, chi2 per layer.
        _forward("odd_options", 7, 5627, 13, 17, "chained", "exact", chi2=True, options=7),
        # The headline batch: 100 events in the reference's semantics, bit-exact.
        _forward("batch_reference", 100, 9600, 20, 32, "reference", "exact"),
        # The same batch as a chained fit in the fast arithmetic, with its chi2.
        _forward("batch_chained_fast", 100, 9600, 20, 32, "chained", "fast", chi2=True),
        # 500 events of lognormal sizes, each track missing layers: a day's uneven batch in one launch.
        _ragged("uneven_500", 500, 9600, 20, 32, "chained", "exact", True),
        # A gradient of the fit for the whole batch, the default precision and checkpoints: calibration.
        _adjoint("batch_gradient", 100, 9600, 20, 32, "exact", "mixed", 4, "tracks"),
        # The FP64 gradient of one event: the gradient that others are checked against.
        _adjoint("event_gradient_f64", 1, 9600, 20, 32, "exact", "f64", 0, "tracks"),
        # Alignment: the sums over a million tracks of 40 layers, FP32 fit and reverse, FP64 reduction.
        _adjoint("alignment", 1, 1000000, 40, 32, "exact", "f32", 4, "global"),
        # The torch.autograd.Function on a small sample, inside somebody's training loop.
        {"name": "autograd_sample", "kind": "autograd", "ntrks": 2048, "nlayer": 20, "bsize": 32, "grad": "mixed"},
    ]


def draw(rng):
    def log(lo, hi):
        return math.exp(rng.uniform(math.log(lo), math.log(hi)))

    kind = rng.choice(["forward", "forward", "forward", "ragged", "adjoint", "adjoint", "autograd"])
    bsize = rng.choice([8, 16, 17, 24, 32, 32, 33, 64])
    nlayer = rng.randint(3, 40 if kind in ("forward", "adjoint") else 26)
    # The reference's layer semantics is a matter of its exact words.  It restarts every layer from the broad input
    # covariance, whose FP32 update cancels: two correct builds in the fast arithmetic differ by percents of the norm.
    semantics = rng.choice(["reference", "chained"])
    precision = "exact" if semantics == "reference" else rng.choice(["exact", "fast"])
    tracks = log(64, min(960000, 18e6 / nlayer))
    if kind == "forward":
        nevts = rng.choice([1, 1, 3, 10, 50])
        ntrks = max(1, round(tracks / nevts / bsize)) * bsize
        c = _forward("", nevts, ntrks, nlayer, bsize, semantics, precision, rng.random() < 0.5, rng.choice([0, 0, 0, 7]))
    elif kind == "ragged":
        # tracks with few layers are near-singular: a few of them would make up the fast arithmetic's whole difference
        fast = precision == "fast"
        c = _ragged("", max(1, round(log(1, 20 if fast else 300))), max(64, round(log(64, 9600))),
                    max(12, nlayer) if fast else nlayer, bsize, semantics, precision, not fast and rng.random() < 0.5)
    elif kind == "adjoint":
        nevts = rng.choice([1, 1, 4])
        ntrks = max(1, round(tracks / 2 / nevts / bsize)) * bsize
        grad = rng.choice(["f32", "mixed", "mixed", "f64"])
        # FP32 gradients of single ill-conditioned tracks carry percents; their sums over the batch do not
        c = _adjoint("", nevts, ntrks, nlayer, bsize, precision, grad, rng.choice([0, 1, 2, 4, 8]),
                     "global" if grad == "f32" else rng.choice(["tracks", "tracks", "global"]))
    else:
        c = {"kind": "autograd", "ntrks": max(1, round(log(64, 30000) / bsize)) * bsize, "nlayer": nlayer,
             "bsize": bsize, "grad": rng.choice(["mixed", "f64"])}
    c.pop("name", None)
    return c


# ---- inputs -------------------------------------------------------------------------------------------------
BASE_PAR = (-12.806846618652344, -7.723824977874756, 38.13014221191406, 0.23732035065189902, -2.613372802734375,
            0.35594117641448975)
BASE_VAR = (6.290299552347278e-07, 7.526661534029699e-07, 9.626245400795597e-08, 0.00253512163402557,
            0.00040678296006807003, 0.0002306247719158348)
# lower triangle of the input state's correlation (the base correlations shrunk to a positive-definite matrix)
BASE_CORR = (1.0, 0.0450986548, 1.0, 0.639253060, 0.429973660, 1.0, -0.0526633327, 0.106779774, 0.0127184711, 1.0,
             -0.0113448587, 0.0184841575, 0.000372372297, 0.682356945, 1.0, -0.0482922236, 0.0959419324, 0.0106280377,
             0.825944011, 0.180137097, 1.0)
HIT_VAR = 1e-4
KFACT = float(np.float32(100 / (-0.299792458 * 3.8112)))


@functools.lru_cache(maxsize=None)
def _context():
    return p2r_amd.Context(0)


def _blocks(rows, bsize):
    """[fields][tracks] -> [blocks][fields][bsize], the Matriplex order."""
    return torch.stack(rows).view(len(rows), -1, bsize).transpose(0, 1)


def _inputs(ntrk, nlayer, bsize, seed):
    """Track and hit buffers (float32, Matriplex layout) of `ntrk` tracks."""
    g = torch.Generator("cuda").manual_seed(seed)

    def normal(*size):
        return torch.randn(*size, generator=g, device="cuda", dtype=torch.float64)

    truth = [b * (1 + 0.1 * normal(ntrk).clamp(-3, 3)) for b in BASE_PAR]
    q = torch.where(torch.rand(ntrk, generator=g, device="cuda") < 0.5, -1, 1).to(torch.int32)
    corr = torch.zeros(6, 6, dtype=torch.float64)
    corr[tuple(np.tril_indices(6))] = torch.tensor(BASE_CORR, dtype=torch.float64)
    corr = corr + corr.tril(-1).T
    low = torch.linalg.cholesky(corr).tolist()
    sig = [math.sqrt(v) * (1 + 0.1 * normal(ntrk)).abs() for v in BASE_VAR]
    z = [normal(ntrk) for _ in range(6)]
    trk = torch.empty(ntrk // bsize, 28, bsize, device="cuda")
    trk[:, :6] = _blocks([truth[i] + sig[i] * sum(low[i][j] * z[j] for j in range(i + 1)) for i in range(6)], bsize)
    trk[:, 6:27] = _blocks([corr[i, j].item() * sig[i] * sig[j] for i in range(6) for j in range(i + 1)], bsize)
    trk[:, 27] = q.view(torch.float32).view(-1, bsize)
    hits = torch.empty(ntrk // bsize, nlayer, 9, bsize, device="cuda")
    hits[:, :, 3:] = torch.tensor([HIT_VAR, 0, HIT_VAR, 0, 0, HIT_VAR], device="cuda")[:, None]
    # the track's circle: centre (cx, cy), signed radius k pt; the crossing with radius r first met along the momentum
    x, y, zt, ipt, phi, theta = truth
    kpt = q * KFACT / ipt
    cx, cy = x - kpt * torch.sin(phi), y + kpt * torch.cos(phi)
    d2 = cx * cx + cy * cy
    d, sign, cot = d2.sqrt(), torch.sign(kpt), torch.cos(theta) / torch.sin(theta)
    for layer in range(nlayer):
        r = 20.0 + (5.0 if nlayer <= 26 else 2.5) * layer
        aa = (r * r - kpt * kpt + d2) / (2 * d)
        h = (r * r - aa * aa).clamp(min=0).sqrt()
        turn = None
        for s in (-1.0, 1.0):
            px, py = (aa * cx - s * h * cy) / d, (aa * cy + s * h * cx) / d
            a = torch.remainder(sign * (torch.atan2((px - cx) / kpt, (cy - py) / kpt) - phi), 2 * math.pi)
            turn = a if turn is None else torch.minimum(turn, a)
        a = sign * turn
        p = [cx + kpt * torch.sin(a + phi), cy - kpt * torch.cos(a + phi), zt + kpt * a * cot]
        meets = r * r > aa * aa  # else the hit lies radially outward of the start
        out = r / torch.hypot(x, y)
        p = [torch.where(meets, v, w) + math.sqrt(HIT_VAR) * normal(ntrk) for v, w in zip(p, (x * out, y * out, zt))]
        hits[:, layer, :3] = _blocks(p, bsize)
    return trk.view(-1), hits.view(-1)


def _counts(case):
    """Track counts of an uneven batch's events: a property of the case, so that its work is known."""
    hi = min(40000, 5 * case["median"])
    return p2r_amd.lognormal_counts(case["nevts"], median=case["median"], sigma=0.5, lo=min(500, case["median"]), hi=hi)


def _present(nlayer):
    """Range of present layers of a track: a quarter of them up to all."""
    return max(1, nlayer // 4), nlayer


def _layout(case):
    blocks = -(-_counts(case).astype(np.int64) // case["bsize"])
    return np.concatenate([[0], np.cumsum(blocks)])


def prepare(case, seed):
    kind, nlayer, bsize = case["kind"], case["nlayer"], case["bsize"]
    state = {"case": case}
    if kind == "ragged":
        offsets = _layout(case)
        nslot = int(offsets[-1]) * bsize
        trk, hits = _inputs(nslot, nlayer, bsize, seed)
        g = torch.Generator("cuda").manual_seed(seed + 1)
        lo, hi = _present(nlayer)
        keys = torch.rand(nslot, nlayer, generator=g, device="cuda")
        count = torch.randint(lo, hi + 1, (nslot,), generator=g, device="cuda")
        present = keys.argsort(1).argsort(1) < count[:, None]
        first = torch.from_numpy(offsets[:-1] * bsize).cuda()
        event = torch.bucketize(torch.arange(nslot, device="cuda"), first, right=True) - 1
        real = torch.arange(nslot, device="cuda") - first[event] < torch.from_numpy(_counts(case)).cuda()[event]
        bits = (present & real[:, None]).long() << torch.arange(nlayer, device="cuda")
        state.update(offsets=offsets, mask=bits.sum(1).to(torch.int32))
        n = nslot
    else:
        n = case.get("nevts", 1) * case["ntrks"]
        trk, hits = _inputs(n, nlayer, bsize, seed)
    state.update(ctx=_context(), trk=trk, hits=hits)
    if kind == "autograd":
        from p2r_amd import autograd
        par, cov, q = autograd.split_tracks(trk, bsize)
        pos, hit_cov = autograd.split_hits(hits, nlayer, bsize)
        g = torch.Generator("cuda").manual_seed(seed + 2)
        state.update(fit=autograd.fit, par=par.clone().requires_grad_(), cov=cov.clone(), q=q.clone(),
                     pos=pos.clone().requires_grad_(), hit_cov=hit_cov.clone(),
                     weight=0.5 + torch.rand(n, generator=g, device="cuda"))
        return state
    out = torch.empty_like(trk)
    o = out.view(-1, 28, bsize)
    result = {"par": o[:, :6], "cov": o[:, 6:27], "q": o[:, 27].view(torch.int32)}
    state.update(out=out, result=result, chi2=None)
    if kind != "ragged":
        state["shape"] = Shape(case["nevts"], case["ntrks"], nlayer, bsize)
    if kind == "adjoint":
        state["chi2"] = result["chi2"] = torch.empty(n, device="cuda")
        state["grads"] = {}
        if case["outputs"] == "tracks":
            state["grads"] = {"grad_par": torch.empty(n * 6, device="cuda"),
                              "grad_hits": torch.empty(n * 3 * nlayer, device="cuda"),
                              "grad_kfact": torch.empty(n, device="cuda")}
        else:
            state["grads"] = {"grad_global": torch.empty(4 * nlayer + 1, device="cuda", dtype=torch.float64)}
        result.update(state["grads"])
    elif case["chi2"]:
        per_layer = case.get("options", 0) & p2r_amd.P2R_OPT_CHI2_PER_LAYER
        state["chi2"] = result["chi2"] = torch.empty(n * (nlayer if per_layer else 1), device="cuda")
    state["params"] = p2r_amd.default_params(case["precision"], options=case.get("options", 0))
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "forward":
        state["ctx"].forward(state["trk"], state["hits"], state["out"], state["shape"], case["semantics"],
                             params=state["params"], chi2=state["chi2"])
    elif kind == "ragged":
        state["ctx"].forward_ragged(state["trk"], state["hits"], state["out"], state["offsets"], state["mask"],
                                    case["nlayer"], case["bsize"], case["semantics"], params=state["params"],
                                    chi2=state["chi2"])
    elif kind == "adjoint":
        state["ctx"].forward_adjoint(state["trk"], state["hits"], state["out"], state["shape"],
                                     params=state["params"], grad_precision=case["grad"],
                                     checkpoint_stride=case["stride"], chi2=state["chi2"], **state["grads"])
    else:
        chi2, par_out, cov_out = state["fit"](state["par"], state["cov"], state["q"], state["pos"], state["hit_cov"],
                                              grad_precision=case["grad"])
        grad_par, grad_pos = torch.autograd.grad((state["weight"] * chi2).sum(), (state["par"], state["pos"]))
        return {"chi2": chi2.detach(), "par": par_out, "cov": cov_out, "grad_par": grad_par, "grad_pos": grad_pos}
    return state["result"]


def work(case):
    nlayer = case["nlayer"]
    if case["kind"] == "ragged":
        n = int(_counts(case).sum())
        updates = n * sum(_present(nlayer)) / 2
    else:
        n = case.get("nevts", 1) * case["ntrks"]
        updates = n * nlayer
    size = n * 224 + updates * 36  # tracks in and out, the hits of the present layers
    if case["kind"] in ("adjoint", "autograd"):
        size += n * 4
        size += n * 28 + updates * 12 if case.get("outputs", "tracks") == "tracks" else 8 * (4 * nlayer + 1)
        return {"bytes": size, "flops": updates * FLOPS_ADJOINT}
    if case["kind"] == "ragged":
        size += n * 4
    if case["chi2"]:
        size += 4 * (updates if case.get("options", 0) & p2r_amd.P2R_OPT_CHI2_PER_LAYER else n)
    return {"bytes": size, "flops": updates * FLOPS_FORWARD}


def tolerance(case):
    """The exact arithmetic is a promise of words.  Otherwise about four times the distance from 64 bits that was
    measured over the listed cases and forty drawn ones: in FP32 the covariance update cancels and chi2 is up to 5e-3
    off (a few tracks make up most of it); MIXED gradients are 3e-4 off, single ones 2e-2; with FP64 states only the
    rounding of the outputs is left."""
    if case["kind"] in ("forward", "ragged"):
        return "exact" if case["precision"] == "exact" else {"rel": 0.02, "max": 0.9}
    return {"f32": {"rel": 0.02, "max": 0.9}, "mixed": {"rel": 2e-3, "max": 0.1}, "f64": {"rel": 1e-7, "max": 1e-6}}[case["grad"]]


# ---- the same in 64 bits --------------------------------------------------------------------------------------
C6, C24 = float(np.float32(0.16666667)), float(np.float32(0.04166667))  # the turning angle's Taylor polynomials
INV_2PI = float(np.float32(1 / (2 * math.pi)))


def _sincos4(x):
    x2 = x * x
    return x - C6 * x * x2, 1 - 0.5 * x2 + C24 * x2 * x2


def _sym(i, j):
    i, j = max(i, j), min(i, j)
    return i * (i + 1) // 2 + j


def _layer(par, cov, k, hit, hit_var):
    """One propagation to the hit's radius and update; lists of FP64 tensors per field.  -> par, cov, chi2"""
    x, y, z, ipt, phi, theta = par
    r, r0 = torch.hypot(hit[0], hit[1]), torch.hypot(x, y)
    pt = 1 / ipt
    sin_p, cos_p, sin_t, cos_t = torch.sin(phi), torch.cos(phi), torch.sin(theta), torch.cos(theta)
    px, py = cos_p * pt, sin_p * pt
    zero = torch.zeros_like(x)
    D, Ddx, Ddy, Ddi, Ddp = zero, -x / r0, -y / r0, zero, zero
    xo, yo = x, y
    for i in range(5):
        r0 = torch.hypot(xo, yo)
        step = r - r0
        D = D + step
        sa, ca = _sincos4(step * ipt / k)
        if i < 4:
            o = torch.where(step.abs() < 1e-4, 1 / r0, zero)
            dx, dy, di = -xo * ipt / k * o, -yo * ipt / k * o, step / k * ipt
            c, s = px * ca - py * sa, py * ca + px * sa
            Ddx = Ddx - (xo * (1 + k * dx * c) + yo * k * dx * s) * o
            Ddy = Ddy - (xo * k * dy * c + yo * (1 + k * dy * s)) * o
            Ddi = Ddi - k * (xo * (c * di - s + py) + yo * (s * di + c - px)) * pt * o
            Ddp = Ddp + k * (xo * (py * sa - px + px * ca) - yo * (px * sa - py + py * ca)) * o
        xo, yo = xo + k * (px * sa - py * (1 - ca)), yo + k * (py * sa + px * (1 - ca))
        px, py = px * ca - py * sa, py * ca + px * sa
    alpha, dx, dy, di, dp = D * ipt / k, Ddx * ipt / k, Ddy * ipt / k, (ipt * Ddi + D) / k, Ddp * ipt / k
    sa, ca = _sincos4(alpha)
    cs, sc, v, w = cos_p * ca - sin_p * sa, sin_p * ca + cos_p * sa, ipt * di, k * cos_t * pt / sin_t
    one = torch.ones_like(x)
    jac = [[1 + k * dx * cs * pt, k * dy * cs * pt, None, k * (cos_p * (v * ca - sa) + sin_p * ((1 - ca) - v * sa)) * pt * pt,
            k * (dp * cs + cs - cos_p) * pt, None],
           [k * dx * sc * pt, 1 + k * dy * sc * pt, None, k * (sin_p * (v * ca - sa) + cos_p * (v * sa - (1 - ca))) * pt * pt,
            k * (dp * sc + sc - sin_p) * pt, None],
           [w * dx, w * dy, one, w * (v - alpha) * pt, w * dp, -k * alpha * pt / (sin_t * sin_t)],
           [None, None, None, one, None, None],
           [dx, dy, None, di, 1 + dp, None],
           [None, None, None, None, None, one]]

    def row(m, terms):
        return functools.reduce(torch.add, [m[t] * a for t, a in terms])

    a = [[row([cov[_sym(t, j)] for t in range(6)], [(t, jac[i][t]) for t in range(6) if jac[i][t] is not None])
          for j in range(6)] for i in range(6)]
    cov = [row(a[i], [(t, jac[j][t]) for t in range(6) if jac[j][t] is not None]) for i in range(6) for j in range(i + 1)]
    par = [xo, yo, z + w * alpha, ipt, phi + alpha, theta]
    ra, rb = -(hit[1] + par[1]) / (2 * r), (hit[0] + par[0]) / (2 * r)
    u = [cov[e] + hit_var[e] for e in range(6)]
    s00, s01, s11 = (ra * u[0] + rb * u[1]) * ra + (ra * u[1] + rb * u[2]) * rb, u[3] * ra + u[4] * rb, u[5]
    det = s00 * s11 - s01 * s01
    s00, s01, s11 = s11 / det, -s01 / det, s00 / det
    h0 = [cov[_sym(i, 0)] * ra + cov[_sym(i, 1)] * rb for i in range(6)]
    h1 = [cov[_sym(i, 2)] for i in range(6)]
    k0 = [h0[i] * s00 + h1[i] * s01 for i in range(6)]
    k1 = [h0[i] * s01 + h1[i] * s11 for i in range(6)]
    e0, e1 = ra * (hit[0] - par[0]) + rb * (hit[1] - par[1]), hit[2] - par[2]
    chi2 = e0 * (s00 * e0 + s01 * e1) + e1 * (s01 * e0 + s11 * e1)
    cov = [cov[_sym(i, j)] - (k0[i] * h0[j] + k1[i] * h1[j]) for i in range(6) for j in range(i + 1)]
    return [par[i] + k0[i] * e0 + k1[i] * e1 for i in range(6)], cov, chi2


def _fit(par, cov, q, hits, chained, mask, options):
    """The whole fit in 64 bits.  par, cov: fields; q: charge; hits: [layer][field].  -> par, cov, [chi2 of each layer]"""
    start, now, chi2s = (par, cov, q), (par, cov, q), []
    for layer, h in enumerate(hits):
        p, c, ch = now if chained else start
        p, c, chi2 = _layer(p, c, ch * KFACT, h[:3], h[3:])
        if options & 1:
            p[4] = p[4] - torch.floor((p[4] + math.pi) * INV_2PI) * (2 * math.pi)
        if options & 2:
            ch = torch.where(p[3] < 0, -ch, ch)
            p[3] = p[3].abs()
        if mask is not None:
            there = (mask >> layer) & 1 == 1
            p = [torch.where(there, a, b) for a, b in zip(p, now[0])]
            c = [torch.where(there, a, b) for a, b in zip(c, now[1])]
            chi2 = torch.where(there, chi2, torch.zeros_like(chi2))
        now = (p, c, ch)
        chi2s.append(chi2)
    return now[0], now[1], chi2s


def exact(case, seed):
    kind, nlayer, bs = case["kind"], case["nlayer"], case["bsize"]
    grads = kind in ("adjoint", "autograd")
    state = prepare(case, seed)
    nblk = state["trk"].numel() // (28 * bs)
    if grads and nblk * bs * nlayer > 20e6:
        return None  # minutes
    t, hit = state["trk"].view(nblk, 28, bs), state["hits"].view(nblk, nlayer, 9, bs)
    mask = state["mask"].view(nblk, bs) if kind == "ragged" else None
    parts, per_layer = [], case.get("options", 0) & 4
    chunk = max(1, int((1.5e6 if grads else 40e6) / nlayer / bs))
    for b in range(0, nblk, chunk):
        tc = t[b:b + chunk]
        par = tc[:, :6].double().detach().requires_grad_(grads)
        pos = hit[b:b + chunk, :, :3].double().detach().requires_grad_(grads)
        hv, cov, q = hit[b:b + chunk, :, 3:].double(), tc[:, 6:27].double(), tc[:, 27].view(torch.int32).double()
        scale = torch.ones_like(q, requires_grad=grads)  # of the charge times kfact
        with torch.set_grad_enabled(grads):
            p, c, chi2 = _fit([par[:, f] for f in range(6)], [cov[:, f] for f in range(21)], q * scale,
                              [[pos[:, i, f] for f in range(3)] + [hv[:, i, f] for f in range(6)] for i in range(nlayer)],
                              grads or case["semantics"] == "chained", mask[b:b + chunk] if mask is not None else None,
                              case.get("options", 0))
            total = functools.reduce(torch.add, chi2)
        got = {"par": torch.stack(p, 1).detach(), "cov": torch.stack(c, 1).detach(),
               "chi2": (torch.stack(chi2) if per_layer else total).detach()}
        if grads:
            weight = state["weight"].view(nblk, bs)[b:b + chunk].double() if kind == "autograd" else 1.0
            got["grad_par"], got["grad_pos"], gk = torch.autograd.grad((weight * total).sum(), (par, pos, scale))
            got["grad_kfact"] = gk / KFACT
            gx, gy, gz = (got["grad_pos"][:, :, f] for f in range(3))
            turn = pos[:, :, 0].detach() * gy - pos[:, :, 1].detach() * gx
            fine = torch.isfinite(total.detach())
            got["sums"] = torch.cat([
                torch.stack([torch.where(fine[:, None], v, 0.0).sum((0, 2)) for v in (gx, gy, gz, turn)], 1).view(-1),
                -torch.where(fine, gk, 0.0).sum().view(1)])
        parts.append(got)
        del p, c, chi2, total
    join = {f: torch.cat([x[f] for x in parts], 1 if f == "chi2" and per_layer else 0) for f in parts[0] if f != "sums"}
    if kind == "autograd":
        return {"chi2": join["chi2"].view(-1), "par": join["par"], "cov": join["cov"], "grad_par": join["grad_par"],
                "grad_pos": join["grad_pos"]}
    result = {"par": join["par"], "cov": join["cov"], "q": None}
    if state["chi2"] is not None:
        result["chi2"] = join["chi2"].reshape(-1)
    if grads and case["outputs"] == "tracks":
        result.update(grad_par=join["grad_par"].reshape(-1), grad_hits=join["grad_pos"].reshape(-1),
                      grad_kfact=join["grad_kfact"].view(-1))
    elif grads:
        result["grad_global"] = sum(x["sums"] for x in parts)
    return result
