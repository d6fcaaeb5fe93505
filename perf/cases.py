"""The work a program has this framework do, as cases that can be timed and checked.

``listed()`` names the cases, ``draw(rng)`` gives another one of the same ranges,
``prepare(case, seed)`` makes what a program holds before the call, ``run(state)`` is one pass
through the public entry points, ``work(case)`` the bytes and operations a pass cannot do
without, and ``exact(case, seed)`` the pass's outputs in 64 bits, in plain torch.
"""
import math
import os

import numpy as np
import torch

from hindemith_amd import batched, kernels
from hindemith_amd.autograd import horn_schunck

DEV = "cuda"

# Horn & Schunck's stencils (weights, column offsets, row offsets).
_Q, _E, _C = 0.25, 1.0 / 6.0, 1.0 / 12.0
TAPS = {
    "Dx": (np.float32([-_Q, _Q, -_Q, _Q]), np.int32([0, 1, 0, 1]), np.int32([0, 0, 1, 1])),
    "Dy": (np.float32([-_Q, _Q, -_Q, _Q]), np.int32([0, 0, 1, 1]), np.int32([0, 1, 0, 1])),
    "Dt": (np.float32([_Q, _Q, _Q, _Q]), np.int32([0, 1, 0, 1]), np.int32([0, 0, 1, 1])),
    "Avg": (np.float32([_E, _E, _E, _E, _C, _C, _C, _C]),
            np.int32([-1, 1, 0, 0, -1, 1, -1, 1]), np.int32([0, 0, -1, 1, -1, -1, 1, 1])),
}
LAP5 = (np.float32([4, -1, -1, -1, -1]), np.int32([0, -1, 1, 0, 0]), np.int32([0, 0, 0, -1, 1]))
POWERS = 8  # operator powers of a communication-avoiding CG step
LAM = 0.125


def listed():
    return [
        # a coarse pyramid level (1080p / 8): the smallest solve of a coarse-to-fine flow, where
        # each launch's latency counts
        dict(name="solve_135x240", kind="solve", H=135, W=240, iters=100, alpha=1.0),
        # a camera-sized pair
        dict(name="solve_480x640", kind="solve", H=480, W=640, iters=200, alpha=1.0),
        # an odd crop: no row starts on a cache line, and partial tiles on two sides
        dict(name="solve_613x977", kind="solve", H=613, W=977, iters=200, alpha=0.5),
        # the headline workload
        dict(name="solve_1080x1920", kind="solve", H=1080, W=1920, iters=500, alpha=1.0),
        # a 4K frame
        dict(name="solve_2160x3840", kind="solve", H=2160, W=3840, iters=500, alpha=1.0),
        # many pairs of uneven sizes in one call (a video server's queue)
        dict(name="batched_32", kind="batched", pairs=32, lo=64, hi=1024, iters=200),
        # a training step through the solver: forward and backward of a batch
        dict(name="train_8x512x512", kind="train", B=8, H=512, W=512, iters=200, every=20,
             start=False),
        # the same on odd crops, with gradients to a predicted starting flow too
        dict(name="train_3x243x331", kind="train", B=3, H=243, W=331, iters=100, every=16,
             start=True),
        # the front end: the canonical program, called with host arrays as the reference is
        dict(name="program_1080x1920", kind="program", H=1080, W=1920, iters=500, alpha=1.0),
        # the building blocks of a program that composes them: the 5-point operator as a
        # stencil, as diagonal planes and as CSR, and a residual's sum
        dict(name="operators_2048x2048", kind="operators", H=2048, W=2048),
        # an irregular sparse operator (row lengths from a truncated Zipf law)
        dict(name="powerlaw_2048x2048", kind="powerlaw", rows=2048 * 2048),
        # one outer step of the preconditioned-CG solver on a warped pair
        dict(name="cg_2160x3840", kind="cg", H=2160, W=3840),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["solve", "solve", "solve", "batched", "train", "program", "operators",
                       "powerlaw", "cg"])
    if kind == "solve":
        return dict(kind=kind, H=_log(rng, 48, 2160), W=_log(rng, 64, 3840),
                    iters=rng.randint(50, 500), alpha=rng.choice([0.5, 1.0, 1.5, 2.0]))
    if kind == "batched":
        lo = _log(rng, 32, 256)
        return dict(kind=kind, pairs=rng.randint(2, 32), lo=lo,
                    hi=max(lo + 16, _log(rng, 128, 1024)), iters=rng.randint(50, 250))
    if kind == "train":
        return dict(kind=kind, B=rng.randint(1, 8), H=_log(rng, 64, 512), W=_log(rng, 64, 512),
                    iters=rng.randint(40, 200), every=rng.randint(8, 25),
                    start=rng.random() < 0.5)
    if kind == "program":
        return dict(kind=kind, H=_log(rng, 64, 1080), W=_log(rng, 64, 1920),
                    iters=rng.choice([100, 500]), alpha=rng.choice([0.5, 1.0, 2.0]))
    if kind == "operators":
        return dict(kind=kind, H=_log(rng, 256, 2048), W=_log(rng, 256, 2048))
    if kind == "powerlaw":
        return dict(kind=kind, rows=_log(rng, 1 << 17, 1 << 22))
    return dict(kind=kind, H=_log(rng, 128, 2160), W=_log(rng, 128, 3840))


# ---------------------------------------------------------------------------
# inputs


def _gen(seed, salt=0):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 1009 + salt)


def _pair(H, W, g, blobs=32):
    """Two float32 frames: Gaussian blobs and noise, the second moved by a constant flow."""
    def uni(n, lo, hi):
        return torch.rand(n, generator=g, device=DEV, dtype=torch.float64) * (hi - lo) + lo
    P = 4  # the moved frame is cut from a larger one
    ys = torch.arange(-P, H + P, device=DEV, dtype=torch.float64)
    xs = torch.arange(-P, W + P, device=DEV, dtype=torch.float64)
    cy, cx = uni(blobs, 0, H), uni(blobs, 0, W)
    sg, am = uni(blobs, 8.0, 24.0), uni(blobs, 0.0, 1.0)
    gy = am[:, None] * torch.exp(-((ys - cy[:, None]) ** 2) / (2 * sg[:, None] ** 2))
    gx = torch.exp(-((xs - cx[:, None]) ** 2) / (2 * sg[:, None] ** 2))
    big = (gy.float().T.contiguous() @ gx.float())
    big += 0.01 * torch.randn(big.shape, generator=g, device=DEV)
    fx, fy = (float(t) for t in uni(2, -3.0, 3.0).cpu())
    ix, iy = math.floor(-fx), math.floor(-fy)
    ax, ay = -fx - ix, -fy - iy

    def cut(dy, dx):
        return big[P + dy:P + dy + H, P + dx:P + dx + W]
    f2 = ((1 - ay) * ((1 - ax) * cut(iy, ix) + ax * cut(iy, ix + 1)) +
          ay * ((1 - ax) * cut(iy + 1, ix) + ax * cut(iy + 1, ix + 1)))
    return cut(0, 0).contiguous(), f2.contiguous()


def _batch_sizes(case, seed):
    # sizes are the case's own, not the seed's: a queue of the same streams
    r = np.random.default_rng(case["pairs"] * 7919 + case["lo"] * 31 + case["hi"])
    n = case["pairs"]
    hs, ws = (r.integers(case["lo"], case["hi"] + 1, n) for _ in range(2))
    al = np.round(r.uniform(0.5, 2.0, n) * 8) / 8
    return [(int(h), int(w), float(a)) for h, w, a in zip(hs, ws, al)]


def _train_inputs(case, seed):
    B, H, W = case["B"], case["H"], case["W"]
    ps = [_pair(H, W, _gen(seed, b)) for b in range(B)]
    g = _gen(seed, 500)
    d = dict(I1=torch.stack([p[0] for p in ps]), I2=torch.stack([p[1] for p in ps]),
             alpha=0.5 + torch.rand(B, generator=g, device=DEV),
             gu=torch.randn(B, H, W, generator=g, device=DEV) / (H * W),
             gv=torch.randn(B, H, W, generator=g, device=DEV) / (H * W))
    if case["start"]:
        d["u0"] = torch.randn(B, H, W, generator=g, device=DEV)
        d["v0"] = torch.randn(B, H, W, generator=g, device=DEV)
    return d


def _operator_inputs(case, seed):
    H, W = case["H"], case["W"]
    g = _gen(seed)
    base = torch.tensor(LAP5[0], device=DEV)[:, None, None]
    A = base * (0.5 + torch.rand(5, H, W, generator=g, device=DEV))
    x = torch.randn(H, W, generator=g, device=DEV)
    n = H * W
    p = torch.arange(n, device=DEV)
    r, c = p // W, p % W
    cols, ok = [], []
    for ox, oy in zip(LAP5[1].tolist(), LAP5[2].tolist()):
        ok.append((r + oy >= 0) & (r + oy < H) & (c + ox >= 0) & (c + ox < W))
        cols.append(p + oy * W + ox)
    ok, cols = torch.stack(ok, 1), torch.stack(cols, 1)
    d = torch.arange(5, device=DEV)[None, :].expand(n, 5)
    indices = cols[ok]
    data = A.reshape(5, n)[d[ok], indices]
    indptr = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    indptr[1:] = torch.cumsum(ok.sum(1), 0)
    return dict(A=A, x=x, indptr=indptr.int(), indices=indices.int(), data=data)


def _powerlaw_inputs(case, seed):
    n, g = case["rows"], _gen(seed)
    k = torch.arange(1, 513, device=DEV, dtype=torch.float64)
    cdf = torch.cumsum(k ** -1.5, 0)
    cdf = cdf / cdf[-1]
    lens = 1 + torch.searchsorted(cdf, torch.rand(n, generator=g, device=DEV,
                                                  dtype=torch.float64)).clamp(max=511)
    indptr = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    indptr[1:] = torch.cumsum(lens, 0)
    nnz = int(indptr[-1])
    indices = torch.randint(0, n, (nnz,), generator=g, device=DEV, dtype=torch.int32)
    data = torch.randn(nnz, generator=g, device=DEV)
    x = torch.randn(n, generator=g, device=DEV)
    return dict(indptr=indptr.int(), indices=indices, data=data, x=x)


def _cg_inputs(case, seed):
    H, W = case["H"], case["W"]
    g = _gen(seed)
    I1, I2 = _pair(H, W, g)

    def smooth(scale):
        t = torch.randn(1, 1, H // 16 + 2, W // 16 + 2, generator=g, device=DEV) * scale
        return torch.nn.functional.interpolate(t, size=(H, W), mode="bilinear")[0, 0].contiguous()
    d0, d1 = (torch.rand(H, W, generator=g, device=DEV) for _ in range(2))
    off = 0.5 * (torch.rand(H, W, generator=g, device=DEV) - 0.5) * torch.minimum(d0, d1)
    return dict(I1=I1, I2=I2, fx=smooth(2.0), fy=smooth(2.0), diag0=d0, diag1=d1, offdiag=off,
                r0=torch.randn(H, W, generator=g, device=DEV),
                r1=torch.randn(H, W, generator=g, device=DEV))


# the stencil whose weight 2 enters the preconditioner's diagonal blocks
PRECOND_STENCIL = (np.float32([-LAM, -LAM, LAM, -LAM, -LAM]), np.int32([0, -1, 0, 1, 0]),
                   np.int32([-1, 0, 0, 0, 1]))

_programs = {}


def _program(iters):
    """The canonical @hm program of that many iterations."""
    if not _programs:
        os.environ["HM_GPU0"] = "1"
        from hindemith_amd import hindemith as front
        front.defines.update(nd20=1, nd21=1, nt20=8, nt21=8, ne20=2, ne21=2)
        hm = front.hm

        @hm
        def hs_100(I1, I2, Dx, Dy, Dt, Avg, alpha2, u, v):
            Ix = Dx * I1 + Dx * I2
            Iy = Dy * I1 + Dy * I2
            It = Dt * I2 - Dt * I1
            den = alpha2 + Ix * Ix + Iy * Iy
            for i in range(100):
                ubar = Avg * u
                vbar = Avg * v
                t = (Ix * ubar + Iy * vbar + It) / den
                u = ubar - Ix * t
                v = vbar - Iy * t
            return u, v

        @hm
        def hs_500(I1, I2, Dx, Dy, Dt, Avg, alpha2, u, v):
            Ix = Dx * I1 + Dx * I2
            Iy = Dy * I1 + Dy * I2
            It = Dt * I2 - Dt * I1
            den = alpha2 + Ix * Ix + Iy * Iy
            for i in range(500):
                ubar = Avg * u
                vbar = Avg * v
                t = (Ix * ubar + Iy * vbar + It) / den
                u = ubar - Ix * t
                v = vbar - Iy * t
            return u, v

        _programs.update({100: hs_100, 500: hs_500, "Stencil": front.Stencil})
    return _programs[iters], _programs["Stencil"]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "solve":
        I1, I2 = _pair(case["H"], case["W"], _gen(seed))
        return dict(case=case, I1=I1, I2=I2,
                    work=torch.empty(5, case["H"], case["W"], device=DEV))
    if kind == "batched":
        sizes = _batch_sizes(case, seed)
        ps = [_pair(h, w, _gen(seed, i)) for i, (h, w, _) in enumerate(sizes)]
        return dict(case=case, solver=batched.BatchedHS([p[0] for p in ps], [p[1] for p in ps],
                                                        [s[2] for s in sizes],
                                                        iters=case["iters"], taps=TAPS))
    if kind == "train":
        d = _train_inputs(case, seed)
        for n in ("I1", "I2", "alpha", "u0", "v0"):
            if n in d:
                d[n].requires_grad_(True)
        return dict(case=case, **d)
    if kind == "program":
        fn, Stencil = _program(case["iters"])
        I1, I2 = (t.cpu().numpy() for t in _pair(case["H"], case["W"], _gen(seed)))
        return dict(case=case, fn=fn, kwargs=dict(
            I1=I1, I2=I2, alpha2=np.float32(case["alpha"] ** 2), u=np.zeros_like(I1),
            v=np.zeros_like(I1), **{k: Stencil(*t) for k, t in TAPS.items()}))
    if kind == "operators":
        return dict(case=case, partials=torch.empty(1024, device=DEV, dtype=torch.float64),
                    **_operator_inputs(case, seed))
    if kind == "powerlaw":
        d = _powerlaw_inputs(case, seed)
        sl = kernels.CSRSlices(d["indptr"].cpu().numpy(), d["indices"].cpu().numpy(),
                               case["rows"], DEV)
        return dict(case=case, slices=sl, values=sl.values(d["data"]), x=d["x"])
    return dict(case=case, partials=torch.empty(1024, device=DEV, dtype=torch.float64),
                **_cg_inputs(case, seed))


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "solve":
        return kernels.hs_solve(s["I1"], s["I2"], case["alpha"] ** 2, TAPS, case["iters"],
                                workspace=s["work"])
    if kind == "batched":
        return s["solver"].run()
    if kind == "train":
        u, v = horn_schunck(s["I1"], s["I2"], s["alpha"], iters=case["iters"],
                            ckpt_every=case["every"], taps=TAPS, u0=s.get("u0"), v0=s.get("v0"))
        wrt = [s[n] for n in ("I1", "I2", "alpha", "u0", "v0") if n in s]
        return (u.detach(), v.detach()) + torch.autograd.grad([u, v], wrt, [s["gu"], s["gv"]])
    if kind == "program":
        # the program updates u, v in place: every call starts from a zero flow
        s["kwargs"]["u"].fill(0.0)
        s["kwargs"]["v"].fill(0.0)
        return s["fn"](**s["kwargs"])
    if kind == "operators":
        y1 = kernels.stencil2d(s["x"], LAP5)
        y2 = kernels.dia2d_spmv(s["A"], LAP5[1], LAP5[2], s["x"])
        y3 = kernels.csr_spmv(s["indptr"], s["indices"], s["data"], s["x"].reshape(-1))
        return y1, y2, y3, kernels.sum2d(y2, partials=s["partials"])
    if kind == "powerlaw":
        return kernels.csr_spmv_sliced(s["slices"], s["values"], s["x"])
    w = kernels.warp_img2d(s["I2"], s["fx"], s["fy"])
    Ix, Iy, It = kernels.hs_setup(s["I1"], w, TAPS["Dx"], TAPS["Dy"], TAPS["Dt"])
    z0, z1 = kernels.hs_precondition(PRECOND_STENCIL, s["diag0"], s["diag1"], s["offdiag"],
                                     s["r0"], s["r1"])
    V0, V1 = kernels.hs_matrix_powers(LAM, Ix, Iy, z0, z1, POWERS)
    return w, Ix, Iy, It, z0, z1, V0, V1, kernels.sum2d(It, partials=s["partials"])


# ---------------------------------------------------------------------------
# what a pass cannot do without: every input read once, every output written once


def work(case):
    kind = case["kind"]
    # a pixel's iteration: two 8-tap sums (32), three products and sums of the data term and its
    # denominator's quotient (5), the update (4)
    it, setup = 41, 6 * 8 + 8
    if kind in ("solve", "program"):
        px = case["H"] * case["W"]
        more = 8 if kind == "program" else 0  # the starting flow is an argument there
        return dict(bytes=px * (16 + more), flops=px * (it * case["iters"] + setup))
    if kind == "batched":
        px = sum(h * w for h, w, _ in _batch_sizes(case, 0))
        return dict(bytes=px * 16, flops=px * (it * case["iters"] + setup))
    if kind == "train":
        px = case["B"] * case["H"] * case["W"]
        # frames, flow, its gradient, the frames' gradients (and the start and its gradients);
        # a reverse iteration takes two transposed sums and about 30 operations, once the
        # forward iteration it reverses is known
        return dict(bytes=px * (8 + 8 + 8 + 8 + (16 if case["start"] else 0)),
                    flops=px * (case["iters"] * (it + 62) + 3 * setup))
    if kind == "operators":
        n = case["H"] * case["W"]
        # one x for all, each operator's own arrays, three results; the sum reads one of them
        return dict(bytes=n * (4 + 20 + 8 * 5 + 4 + 12), flops=n * (10 + 10 + 10 + 1))
    if kind == "powerlaw":
        k = np.arange(1, 513, dtype=np.float64)
        p = k ** -1.5
        nnz = float(case["rows"] * (k * p).sum() / p.sum())
        return dict(bytes=8 * nnz + 12 * case["rows"], flops=2 * nnz)
    px = case["H"] * case["W"]
    return dict(bytes=px * 4 * (9 + 6 + 2 * POWERS), flops=px * (20 + setup + 20 + 22 * POWERS))


# ---------------------------------------------------------------------------
# the same in 64 bits


def _shift(p, ox, oy, H, W):
    """The H x W window of a once-padded array at a tap's offset."""
    return p[..., 1 + oy:1 + oy + H, 1 + ox:1 + ox + W]


def _pad(x, mode="replicate"):
    lead = x.shape[:-2]
    x = x.reshape((-1, 1) + tuple(x.shape[-2:]))
    x = torch.nn.functional.pad(x, (1, 1, 1, 1), mode=mode)
    return x.reshape(tuple(lead) + tuple(x.shape[-2:]))


def _stencil(x, st):
    H, W = x.shape[-2:]
    p = _pad(x)
    out = 0.0
    for w, ox, oy in zip(st[0].tolist(), st[1].tolist(), st[2].tolist()):
        out = out + w * _shift(p, ox, oy, H, W)
    return out


def _derivatives(I1, I2):
    return (_stencil(I1, TAPS["Dx"]) + _stencil(I2, TAPS["Dx"]),
            _stencil(I1, TAPS["Dy"]) + _stencil(I2, TAPS["Dy"]),
            _stencil(I2, TAPS["Dt"]) - _stencil(I1, TAPS["Dt"]))


def _iterate(u, v, Ix, Iy, It, den, iters):
    for _ in range(iters):
        ub, vb = _stencil(u, TAPS["Avg"]), _stencil(v, TAPS["Avg"])
        t = (Ix * ub + Iy * vb + It) / den
        u, v = ub - Ix * t, vb - Iy * t
    return u, v


def _solve(I1, I2, alpha2, iters):
    Ix, Iy, It = _derivatives(I1.double(), I2.double())
    z = torch.zeros_like(Ix)
    return _iterate(z, z, Ix, Iy, It, alpha2 + Ix * Ix + Iy * Iy, iters)


def _train(case, seed):
    from torch.utils.checkpoint import checkpoint
    d = {k: t.double() for k, t in _train_inputs(case, seed).items()}
    wrt = [d[n].requires_grad_(True) for n in ("I1", "I2", "alpha", "u0", "v0") if n in d]
    Ix, Iy, It = _derivatives(d["I1"], d["I2"])
    den = (d["alpha"] ** 2)[:, None, None] + Ix * Ix + Iy * Iy
    u = d.get("u0", torch.zeros_like(Ix))
    v = d.get("v0", torch.zeros_like(Ix))
    left = case["iters"]
    while left > 0:
        n = min(10, left)
        u, v = checkpoint(_iterate, u, v, Ix, Iy, It, den, n, use_reentrant=False)
        left -= n
    return (u.detach(), v.detach()) + torch.autograd.grad([u, v], wrt, [d["gu"], d["gv"]])


def _csr(indptr, indices, data, x):
    n = indptr.numel() - 1
    y = torch.zeros(n, device=x.device, dtype=torch.float64)
    rows = torch.repeat_interleave(torch.arange(n, device=x.device),
                                   (indptr[1:] - indptr[:-1]).long())
    return y.index_add_(0, rows, data.double() * x.double()[indices.long()])


def _operators(case, seed):
    d = _operator_inputs(case, seed)
    H, W = case["H"], case["W"]
    x = d["x"].double()
    y1 = _stencil(x, LAP5)
    y2 = 0.0
    for A, ox, oy in zip(d["A"].double(), LAP5[1].tolist(), LAP5[2].tolist()):
        y2 = y2 + _shift(_pad(A * x, mode="constant"), ox, oy, H, W)
    y3 = _csr(d["indptr"], d["indices"], d["data"], d["x"].reshape(-1))
    return y1, y2, y3, None  # (the sum is of y2 as it was rounded)


def _warp(src, ox, oy):
    H, W = src.shape
    mx, my = torch.floor(ox), torch.floor(oy)
    # a whole negative offset splits one step lower, with a fraction of 1: the same sample, but
    # another pixel beyond the border; random fields hold none
    r = torch.arange(H, device=src.device)[:, None]
    c = torch.arange(W, device=src.device)[None, :]
    sx, sy = c + mx.long(), r + my.long()
    inside = (sx >= 0) & (sx + 1 < W) & (sy >= 0) & (sy + 1 < H)
    x0, y0 = sx.clamp(0, W - 2), sy.clamp(0, H - 2)
    ax, ay = ox.double() - mx.double(), oy.double() - my.double()
    s = src.double()
    out = ((1 - ay) * ((1 - ax) * s[y0, x0] + ax * s[y0, x0 + 1]) +
           ay * ((1 - ax) * s[y0 + 1, x0] + ax * s[y0 + 1, x0 + 1]))
    return torch.where(inside, out, s)


def _cg(case, seed):
    d = _cg_inputs(case, seed)
    H, W = case["H"], case["W"]
    w = _warp(d["I2"], d["fx"], d["fy"])
    Ix, Iy, It = _derivatives(d["I1"].double(), w)
    nb = torch.full((H, W), 4.0, device=DEV, dtype=torch.float64)
    nb[0] -= 1
    nb[-1] -= 1
    nb[:, 0] -= 1
    nb[:, -1] -= 1
    a, b = d["diag0"].double() + nb * LAM, d["offdiag"].double()
    dd = d["diag1"].double() + nb * LAM
    r0, r1 = d["r0"].double(), d["r1"].double()
    det = a * dd - b * b
    z0, z1 = (r0 * dd - b * r1) / det, (a * r1 - b * r0) / det

    def lap(x):  # replicated borders: a neighbour outside the image adds nothing
        return LAM * _stencil(x, LAP5)
    V0, V1 = [z0], [z1]
    for _ in range(POWERS - 1):
        dot = Ix * V0[-1] + Iy * V1[-1]
        n0, n1 = Ix * dot + lap(V0[-1]), Iy * dot + lap(V1[-1])
        V0.append(n0)
        V1.append(n1)
    return w, Ix, Iy, It, z0, z1, torch.stack(V0), torch.stack(V1), None


def exact(case, seed):
    kind = case["kind"]
    if kind in ("solve", "program"):
        I1, I2 = _pair(case["H"], case["W"], _gen(seed))
        return _solve(I1, I2, case["alpha"] ** 2, case["iters"])
    if kind == "batched":
        out = []
        for i, (h, w, a) in enumerate(_batch_sizes(case, seed)):
            I1, I2 = _pair(h, w, _gen(seed, i))
            out.append(_solve(I1, I2, a * a, case["iters"]))
        return out
    if kind == "train":
        return _train(case, seed)
    if kind == "operators":
        return _operators(case, seed)
    if kind == "powerlaw":
        d = _powerlaw_inputs(case, seed)
        return _csr(d["indptr"], d["indices"], d["data"], d["x"])
    return _cg(case, seed)
