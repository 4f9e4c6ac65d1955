"""The work this package is used for, as cases to time: whole objectives, pair sums, images of warped events, the
per-event operators, voxel grids and the look-up table, each through its public entry point, forward and backward
where it has a gradient.

listed() are the cases of the benchmark's and the tests' sizes, draw() more of the same ranges, prepare() a user's
inputs on the GPU, run() one pass, work() its unavoidable bytes and operations, tolerance() how far another correct
fp32 implementation may be off, and exact() the same numbers in 64 bits from plain torch."""
from __future__ import annotations

import math

import torch
import torch.nn.functional as nnf

from x_amd.core import EventPacket
from x_amd.motion import DenseLinearFlow, PixelTrajectories, Translation
from x_amd.objectives import AnchoredExact, AnchoredTrajectories, IWEConfig, MotionPriorCMaxLoss, iwe_at_events, iwe_variance
from x_amd.ops import ats_pair_sums, gather, layout_scope, splat, voxel_grid
from x_amd.ops.functional import ats_pair_sums_reference_layout

DEV = "cuda"
SLICES, CUT, STEPS = 16, 3.0, 6


# ----------------------------------------------------------------------------------------------- the cases
def listed():
    return [
        # the anchored score, forward + backward to a dense flow: a step of an alignment or training loop.
        # A small window, where launches and host work count (the smoke test's size).
        dict(name="score_small", kind="score", n=3000, B=1, H=40, W=48, Hg=40, Wg=48, h=1.0, tau=0.2, vmax=6.0),
        # the benchmark's headline: 1M events on 640x480, a flow vector per pixel
        dict(name="score_1m", kind="score", n=1_000_000, B=1, H=480, W=640, Hg=480, Wg=640, h=1.0, tau=0.2, vmax=20.0),
        # three ragged windows on an odd sensor, a coarse flow grid, the wide kernel of an annealing schedule's start
        dict(name="score_ragged_h2", kind="score", n=251_117, B=3, H=259, W=345, Hg=65, Wg=87, h=2.0, tau=0.3,
             vmax=14.0),
        # the bare pair sums of a subset of anchors over all sources, whole window as time range (the reference's
        # operator benchmark: 20k anchors, 100k sources, 240x320)
        dict(name="pairs_20k_of_100k", kind="pairs", scene="uniform", n=100_000, m=20_000, B=1, H=240, W=320, h=1.0,
             tau=1.0, vmax=20.0),
        # the contention workload: 4M events, 90% of them in five small blobs, thousands of pairs per event
        dict(name="pairs_4m_blobs", kind="pairs", scene="blobs", n=4_000_000, m=4_000_000, B=1, H=480, W=640, h=1.0,
             tau=0.2, vmax=40.0),
        # the reference's own call pattern: its plan layout built on the device, then the plan's two operators
        dict(name="reflayout_400k", kind="reflayout", scene="segments", n=400_003, m=400_003, B=1, H=480, W=640, h=1.0,
             tau=0.2, vmax=20.0),
        # contrast maximisation's inner loop: warp, image of warped events, its values at the events, and back
        dict(name="iwe_1m", kind="iwe", motion="dense", n=1_000_000, B=1, H=480, W=640, Hg=480, Wg=640, vmax=20.0),
        dict(name="iwe_translation_100k", kind="iwe", motion="translation", n=100_000, B=1, H=180, W=240, Hg=1, Wg=1,
             vmax=2.4),
        # the operators by themselves, Gaussian votes (the reference's operator benchmark, 100k events at 240x320)
        dict(name="splat_gauss_100k", kind="ops", kernel="gauss", sigma=1.0, n=100_000, B=1, H=240, W=320),
        # a network's input: 15 time bins, normalised
        dict(name="voxel_1m", kind="voxel", n=1_000_000, B=1, C=15, H=480, W=640),
        # continuous-time trajectories: 4 windows of 500k events, per-pixel cubic B-splines of 10 control points,
        # the anchored score less the image contrast, back to the control points
        dict(name="traj_4x500k", kind="traj", n=2_000_000, B=4, H=480, W=640, K=10, tile=1, tau=0.8),
        # the nearest-trajectory table of a trained network's loss: 15 bins x 19200 cells, 32 neighbours
        dict(name="lut_640x480", kind="lut", B=1, H=480, W=640, K=10, tile=4, bins=15, knn=32),
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["score", "score", "pairs", "pairs", "reflayout", "iwe", "iwe", "ops", "voxel", "traj", "lut"])
    H, W = rng.randint(90, 480), rng.randint(120, 640)
    c = dict(kind=kind, H=H, W=W)
    if kind == "lut":
        c.update(B=rng.randint(1, 2), K=rng.randint(3, 10), tile=4, bins=rng.randint(5, 15), knn=rng.randint(8, 32))
        return c
    c["B"] = rng.randint(1, 4)
    n = min(size(2000, 2_000_000), 4 * H * W * c["B"])
    if kind == "score":
        full = rng.random() < 0.5
        c.update(n=min(n, 1_000_000), Hg=H if full else rng.randint(2, 60), Wg=W if full else rng.randint(2, 80),
                 h=rng.choice([0.5, 1.0, 2.0, round(rng.uniform(0.5, 2.0), 3)]), tau=round(rng.uniform(0.05, 0.5), 3),
                 vmax=round(rng.uniform(1.0, 25.0), 2))
    elif kind in ("pairs", "reflayout"):
        n = min(n, 1_000_000)
        c.update(scene=rng.choice(["uniform", "segments", "blobs"]), n=n,
                 m=n if rng.random() < 0.5 else size(max(n // 50, 100), n), h=round(rng.uniform(0.5, 2.0), 3),
                 tau=round(rng.uniform(0.1, 1.0), 3), vmax=round(rng.uniform(1.0, 25.0), 2))
        if c["scene"] == "blobs":           # crowded: thousands of pairs per event already at 200k events
            c["n"], c["m"] = min(n, 200_000), min(c["m"], n, 200_000)
    elif kind == "iwe":
        if rng.random() < 0.7:
            full = rng.random() < 0.5
            c.update(motion="dense", Hg=H if full else rng.randint(2, 60), Wg=W if full else rng.randint(2, 80))
        else:
            c.update(motion="translation", Hg=1, Wg=1)
        c.update(n=n, vmax=round(rng.uniform(1.0, 25.0), 2))
    elif kind == "ops":
        c.update(kernel=rng.choice(["bilinear", "gauss"]), sigma=round(rng.uniform(0.6, 1.6), 2), n=n)
        if c["kernel"] == "gauss":
            c["n"] = min(n, 1_000_000)
    elif kind == "voxel":
        c.update(n=n, C=rng.choice([5, 9, 15]))
    else:
        c.update(n=min(n, 1_000_000), K=rng.randint(4, 10), tile=rng.choice([1, 4]), tau=round(rng.uniform(0.2, 0.8), 3))
    return c


# ----------------------------------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device=DEV)


def _smooth(g, B, C, H, W, H0, W0, vmax):
    """A smooth random field (B, C, H, W) of an H0 x W0 sensor (nodes about every 40 px), whose longest vector (pairs
    of channels k and k + C/2) is vmax."""
    lo = torch.randn(B, C, max(H0 // 40, 1) + 3, max(W0 // 40, 1) + 3, generator=g, device=DEV)
    f = nnf.interpolate(lo, size=(H, W), mode="bicubic", align_corners=True)
    half = C // 2
    return (f * (vmax / (f[:, :half] ** 2 + f[:, half:] ** 2).sqrt().max())).contiguous()


def _points(g, n, H, W, scene):
    """Scene points (n, 2): 70% near 50 line segments, or 90% in five blobs of sigma 8 px; the rest uniform."""
    ext = torch.tensor([W - 1.0, H - 1.0], device=DEV)
    p = _rand(g, n, 2) * ext
    if scene == "segments":
        a, d = _rand(g, 50, 2) * ext, _rand(g, 50, 2) * ext
        d = d - a
        k = torch.randint(0, 50, (n,), generator=g, device=DEV)
        nrm = torch.stack([-d[:, 1], d[:, 0]], 1) / d.norm(dim=1, keepdim=True).clamp(min=1e-6)
        q = a[k] + _rand(g, n, 1) * d[k] + nrm[k] * (2 * _rand(g, n, 1) - 1)
        return torch.where(_rand(g, n, 1) < 0.7, q, p)
    if scene == "blobs":
        c = _rand(g, 5, 2) * ext
        q = c[torch.randint(0, 5, (n,), generator=g, device=DEV)] + 8.0 * torch.randn(n, 2, generator=g, device=DEV)
        return torch.where(_rand(g, n, 1) < 0.9, q, p)
    return p


def _events(g, n, B, H, W, scene, move=None):
    """Events sorted by (window, time), windows of different sizes: pixel positions (a sensor reports whole pixels),
    times, polarities and window numbers; ``move(p, b, t)`` carries the scene points along the motion."""
    share = 1.0 + 0.5 * _rand(g, B)
    b = torch.searchsorted(torch.cumsum(share / share.sum(), 0), (torch.arange(n, device=DEV) + 0.5) / n)
    b = b.clamp(max=B - 1)
    t = _rand(g, n).clamp(max=1 - 2.0 ** -24)
    t = t[torch.argsort(b.double() * 4 + t.double())]
    p = _points(g, n, H, W, scene)
    if move is not None:
        p = move(p, b, t)
    ext = torch.tensor([W - 1.0, H - 1.0], device=DEV)
    out = ((p < 0) | (p > ext)).any(1, keepdim=True)
    xy = torch.where(out, _rand(g, n, 2) * ext, p).round()
    pol = torch.where(_rand(g, n) < 0.5, 1.0, -1.0)
    return xy.contiguous(), t.contiguous(), pol, b


def _packet(ev, B, H, W):
    xy, t, p, b = ev
    return EventPacket(xy, t, p, b, B, H, W, torch.ones(B, device=DEV), {"sorted": True})


def _flow_at(grid, p, b, H, W):
    Hg, Wg = grid.shape[-2:]
    return _bilinear(grid, torch.stack([p[:, 0] * ((Wg - 1) / max(W - 1, 1)), p[:, 1] * ((Hg - 1) / max(H - 1, 1))], 1), b)


def _inputs(c, seed):
    """The raw inputs of a case: what prepare() wraps and exact() starts from."""
    g, k = _gen(seed), c["kind"]
    B, H, W = c["B"], c["H"], c["W"]
    if k == "score" or k == "iwe":
        grid = (_smooth(g, B, 2, c["Hg"], c["Wg"], H, W, c["vmax"]) if k == "score" or c["motion"] == "dense" else
                (torch.rand(B, 2, 1, 1, generator=g, device=DEV) - 0.5) * (2 * c["vmax"]))
        # the scene moves along the flow; the estimate differs from it, as during a fit
        move = lambda p, b, t: p + _flow_at(grid, p, b, H, W) * t[:, None]  # noqa: E731
        ev = _events(g, c["n"], B, H, W, "segments", move)
        est = grid + 0.05 * c["vmax"] * torch.randn(B, 2, 1, 1, generator=g, device=DEV)
        d = dict(ev=ev, grid=est.contiguous())
        if k == "iwe":
            d["gv"] = torch.randn(c["n"], generator=g, device=DEV)
        return d
    if k in ("pairs", "reflayout"):
        n, m = c["n"], min(c["m"], c["n"])
        xy, t, _, b = _events(g, n, B, H, W, c["scene"])
        x = xy + _rand(g, n, 2) - 0.5
        v = _flow_at(_smooth(g, B, 2, H, W, H, W, c["vmax"]), x, b, H, W).contiguous()
        anchors = None if m == n else torch.sort(torch.randperm(n, generator=g, device=DEV)[:m]).values
        xa = (x if anchors is None else x[anchors]) + c["h"] * torch.randn(m, 2, generator=g, device=DEV)
        return dict(x=x, t=t, b=b, v=v, anchors=anchors, xa=xa, gS=(0.5 + _rand(g, m)) / m)
    if k == "ops":
        n = c["n"]
        ext = torch.tensor([W + 1.0, H + 1.0], device=DEV)
        b = torch.randint(0, B, (n,), generator=g, device=DEV)
        return dict(pos=_rand(g, n, 2) * ext - 1.0, w=torch.randn(n, generator=g, device=DEV), b=b,
                    gi=torch.randn(B, H, W, generator=g, device=DEV), gv=torch.randn(n, generator=g, device=DEV))
    if k == "voxel":
        return dict(ev=_events(g, c["n"], B, H, W, "segments"))
    K = c["K"]
    coef = _smooth(g, B, 2 * K, H, W, H, W, 5.0 if k == "traj" else 25.0)
    if k == "lut":
        shape = B, c["bins"], -(-H // 4), -(-W // 4), 2
        return dict(coef=coef, t_ref=_rand(g, 1)[0], gt=torch.randn(shape, generator=g, device=DEV))
    return dict(coef=coef, ev=_events(g, c["n"], B, H, W, "segments"))


def prepare(case, seed):
    c, d = case, _inputs(case, seed)
    s = dict(case=c, d=d)
    k, B, H, W = c["kind"], c["B"], c["H"], c["W"]
    if k == "score":
        s["ev"] = _packet(d["ev"], B, H, W)
        s["motion"] = DenseLinearFlow(B, H, W, grid=(c["Hg"], c["Wg"]), init=d["grid"]).to(DEV)
        s["obj"] = AnchoredExact(h=c["h"], tau=c["tau"], cut=CUT, n_slices=SLICES, n_anchors=None, seed=int(seed),
                                 rng="device")
    elif k == "iwe":
        s["ev"] = _packet(d["ev"], B, H, W)
        s["motion"] = (DenseLinearFlow(B, H, W, grid=(c["Hg"], c["Wg"]), init=d["grid"]) if c["motion"] == "dense" else
                       Translation(B, H, W, init=d["grid"].view(B, 2))).to(DEV)
        s["cfg"] = IWEConfig(kernel="bilinear", sigma=0.0, mask_border=True)
    elif k in ("pairs", "reflayout"):
        d["v"].requires_grad_(True)
    elif k == "ops":
        d["pos"].requires_grad_(True)
        d["w"].requires_grad_(True)
    elif k == "traj":
        s["ev"] = _packet(d["ev"], B, H, W)
        d["coef"].requires_grad_(True)
        s["obj"] = AnchoredTrajectories(h=1.0, tau=c["tau"], cut=CUT, n_slices=SLICES, n_anchors=None, seed=int(seed),
                                        rng="device")
    elif k == "lut":
        d["coef"].requires_grad_(True)
        s["obj"] = MotionPriorCMaxLoss(num_bins=c["bins"], num_knn=c["knn"], lut=4)
    return s


# ----------------------------------------------------------------------------------------------- one pass
def run(state):
    c, d = state["case"], state["d"]
    k, B, H, W = c["kind"], c["B"], c["H"], c["W"]
    if k == "score":
        m = state["motion"]
        m.grid.grad = None
        loss = state["obj"](state["ev"], m)["loss"]
        loss.backward()
        return {"loss": loss, "grad": m.grid.grad}
    if k == "iwe":
        m = state["motion"]
        m.theta.grad = None
        img, vals = iwe_at_events(state["ev"], m, 0.5, state["cfg"])
        vals.backward(d["gv"])
        return {"img": img, "vals": vals, "grad": m.theta.grad}
    if k in ("pairs", "reflayout"):
        d["v"].grad = None
        op = ats_pair_sums if k == "pairs" else ats_pair_sums_reference_layout
        S = op(d["x"], d["t"], d["v"], d["b"], B, H, W, d["anchors"], c["h"], c["tau"], CUT, SLICES, anchor_xy=d["xa"])
        S.backward(d["gS"])
        return {"S": S, "grad": d["v"].grad}
    if k == "ops":
        d["pos"].grad = d["w"].grad = None
        img = splat(d["pos"], d["w"], d["b"], B, H, W, kernel=c["kernel"], sigma=c["sigma"])
        vals = gather(img, d["pos"], d["b"])
        torch.autograd.backward([img, vals], [d["gi"], d["gv"]])
        return {"img": img, "vals": vals, "gpos": d["pos"].grad, "gw": d["w"].grad}
    if k == "voxel":
        xy, t, p, b = d["ev"]
        return {"vox": voxel_grid(xy, t, p, b, B, c["C"], H, W, normalize="mean_std")}
    if k == "traj":
        d["coef"].grad = None
        with layout_scope():
            m = PixelTrajectories(d["coef"], c["K"], "bspline", tile=c["tile"])
            loss = state["obj"](state["ev"], m)["loss"] - iwe_variance(state["ev"], m, 0.5)
        loss.backward()
        return {"loss": loss, "grad": d["coef"].grad}
    d["coef"].grad = None
    m = PixelTrajectories(d["coef"], c["K"], "bspline", tile=c["tile"])
    table, _ = state["obj"].lut_flow(m, H, W, d["t_ref"])
    table.backward(d["gt"])
    return {"table": table, "grad": d["coef"].grad}


# ----------------------------------------------------------------------------------------------- work
def _pairs_per_anchor(c):
    """Expected contributing pairs of an anchor: the density times the disc times the time range, and how much the
    scene concentrates it (for the segments as counted on the 1M-event window at h = 0.5, 1 and 2)."""
    n, area = c["n"] / c["B"], c["H"] * c["W"]
    tau = c["tau"]
    near = (2 * tau - tau * tau) * n
    h = c.get("h", 1.0)
    flat = near * math.pi * (CUT * h) ** 2 / area
    if c.get("scene") == "blobs":
        return 0.81 / 5 * near * (1 - math.exp(-((CUT * h) ** 2) / (4 * 64.0))) + 0.1 * flat
    return flat if c.get("scene") == "uniform" else flat * (1 + 3 * h ** -0.75)


def work(case):
    c, k = case, case["kind"]
    B, H, W = c["B"], c["H"], c["W"]
    px = B * H * W
    if k == "score":
        # positions, noise (three draws read back as positions), times, windows; the grid and its gradient; 13 flops
        # a pair forward and 19 backward
        pairs = c["n"] * _pairs_per_anchor(c)
        return {"bytes": 36 * c["n"] + 16 * B * c["Hg"] * c["Wg"], "flops": 32 * pairs}
    if k in ("pairs", "reflayout"):
        m = min(c["m"], c["n"])
        return {"bytes": 36 * c["n"] + 24 * m, "flops": 32 * m * _pairs_per_anchor(c)}
    if k == "iwe":
        return {"bytes": 48 * c["n"] + 4 * px + 16 * B * c["Hg"] * c["Wg"], "flops": 150 * c["n"]}
    if k == "ops":
        # positions, weights, windows, value gradients in, values and both gradients out; the images
        taps = 4 if c["kernel"] == "bilinear" else (2 * math.ceil(3 * c["sigma"]) + 1) ** 2
        return {"bytes": 40 * c["n"] + 8 * px, "flops": (30 * taps + 80) * c["n"]}
    if k == "voxel":
        return {"bytes": 24 * c["n"] + 4 * c["C"] * px, "flops": 30 * c["n"] + 8 * c["C"] * px}
    K = c["K"]
    if k == "traj":
        # 13 + 19 + 10 flops a pair; per event 6 fixed-point steps of two transports and one exposure start, each 8
        # flops a corner and channel, and twice that back; the grid and its gradient
        pairs = c["n"] * _pairs_per_anchor(dict(c, h=1.0))
        return {"bytes": 36 * c["n"] + 16 * K * px, "flops": 42 * pairs + c["n"] * 16 * K * (3 * 14 + 7)}
    q = -(-H // 4) * -(-W // 4)
    nt = B * c["bins"] * q
    # coefficients at the tile centres and the gradient of the whole grid, the table and its gradient; a neighbour
    # search cannot do with less than a distance per chosen neighbour
    return {"bytes": 8 * K * (px + B * q) + 16 * nt, "flops": nt * (4 * K + 10 * c["knn"])}


# About four times the largest error of the fp32 path against exact() over the listed and some drawn cases.  Sums in
# another order change results by 1e-7 (1.7e-6 over the blobs' thousands of pairs); the rest comes from what a rounding
# decides: a pair at the cut or the end of the time range, an event at a pixel's border (whose bilinear gradient jumps),
# a neighbour at the same distance.  The per-event operators have none of these inside a pixel.
_REL = {"score": 1.4e-3, "pairs": 8e-4, "reflayout": 8e-4, "iwe": 8e-3, "ops": 1e-5, "voxel": 1e-5, "traj": 4e-3,
        "lut": 2.5e-3}


def tolerance(case):
    return {"rel": _REL[case["kind"]]}


# ----------------------------------------------------------------------------------------------- 64 bits
F64 = torch.float64


def _bilinear(field, gp, b):
    """(N, C) bilinear sample of (B, C, Hg, Wg) at grid coordinates gp, clamped to the border."""
    B, C, Hg, Wg = field.shape
    x, y = gp[:, 0].clamp(0, Wg - 1), gp[:, 1].clamp(0, Hg - 1)
    x0 = torch.floor(x.detach()).clamp(max=max(Wg - 2, 0))
    y0 = torch.floor(y.detach()).clamp(max=max(Hg - 2, 0))
    ax, ay = (x - x0)[:, None], (y - y0)[:, None]
    i, j = x0.long(), y0.long()
    i1, j1 = (i + 1).clamp(max=Wg - 1), (j + 1).clamp(max=Hg - 1)
    rows = field.permute(0, 2, 3, 1).reshape(B * Hg * Wg, C)
    at = lambda jj, ii: rows.index_select(0, (b * Hg + jj) * Wg + ii)  # noqa: E731
    return ((at(j, i) * (1 - ax) + at(j, i1) * ax) * (1 - ay) + (at(j1, i) * (1 - ax) + at(j1, i1) * ax) * ay)


def _noise(xy, seed, h):
    """The first draw of the objectives' device noise (Philox4x32-10, Salmon et al. 2011; key: the seed, counter: the
    event's number and the draw's, 0): positions + U(-1/2, 1/2), and those + h N(0, 1) by Box and Muller."""
    n, mask = xy.shape[0], 0xFFFFFFFF
    i = torch.arange(n, device=xy.device)
    zero = torch.zeros_like(i)
    x = [i & mask, i >> 32, zero, zero]
    k0, k1 = seed & mask, (seed >> 32) & mask
    for _ in range(10):
        p0, p1 = x[0] * 0xD2511F53, x[2] * 0xCD9E8D57          # wraps modulo 2^64, as wanted
        x = [((p1 >> 32) & mask) ^ x[1] ^ k0, p1 & mask, ((p0 >> 32) & mask) ^ x[3] ^ k1, p0 & mask]
        k0, k1 = (k0 + 0x9E3779B9) & mask, (k1 + 0xBB67AE85) & mask
    u = [(w >> 8).to(F64) / 2.0 ** 24 for w in x]
    xs = xy.to(F64) + torch.stack([u[0] - 0.5, u[1] - 0.5], 1)
    rad = torch.sqrt(-2 * torch.log(u[2] + 2.0 ** -24))
    return xs, xs + h * torch.stack([rad * torch.cos(2 * math.pi * u[3]), rad * torch.sin(2 * math.pi * u[3])], 1)


def _pairs64(source, t, b, xa, ta, ba, aid, h, tau, gS=None, give=None):
    """S of every anchor over the sources seen from its time slice, sum of exp(-r^2 / 2 h^2) over |r| <= CUT h,
    |dt| <= tau, another event of the same window, r = xa - y - v (t_a - c); ``source(ids, c)`` gives the positions y
    and velocities v of sources at the slice centre c.  With gS, ``give(ids, c, gy, gv)`` gets their gradients."""
    S = torch.zeros(ta.shape[0], dtype=F64, device=DEV)
    slc = torch.floor(ta * SLICES).clamp(0, SLICES - 1)
    for s in range(SLICES):
        c = (s + 0.5) / SLICES
        ids = torch.nonzero((t - c).abs() <= tau + 0.5 / SLICES + 1e-6)[:, 0]
        anc = torch.nonzero(slc == s)[:, 0]
        if not len(ids) or not len(anc):
            continue
        y, v = source(ids, c)
        at = ta[anc] - c
        R = CUT * h + float(v.norm(dim=1).max() * at.abs().max()) + 1e-3
        lo = torch.minimum(xa[anc].amin(0), y.amin(0)) - 2 * R
        hi = torch.maximum(xa[anc].amax(0), y.amax(0)) + 2 * R
        GW, GH = (int(q) + 2 for q in torch.ceil((hi - lo) / R).tolist())
        cell = lambda p, bb: (bb * GH + ((p[:, 1] - lo[1]) / R).long()) * GW + ((p[:, 0] - lo[0]) / R).long()  # noqa: E731
        key, perm = torch.sort(cell(y, b[ids]))
        y, v, src = y[perm], v[perm], ids[perm]
        tj = t[src]
        ak, order = torch.sort(cell(xa[anc], ba[anc]))
        anc, at = anc[order], at[order]
        near = ak[:, None] + torch.tensor([-GW, 0, GW], device=DEV)
        first = torch.searchsorted(key, near - 1)
        cnt = torch.searchsorted(key, near + 1, right=True) - first
        ends = torch.cumsum(cnt.sum(1), 0)
        gy, gv = torch.zeros_like(y), torch.zeros_like(y)
        a0 = 0
        while a0 < len(anc):
            done = int(ends[a0 - 1]) if a0 else 0
            a1 = max(a0 + 1, int(torch.searchsorted(ends, done + 50_000_000, right=True)))
            k3 = cnt[a0:a1].reshape(-1)
            tot = int(k3.sum())
            seg = torch.repeat_interleave(torch.arange(len(k3), device=DEV), k3, output_size=tot)
            j = first[a0:a1].reshape(-1)[seg] + torch.arange(tot, device=DEV) - (torch.cumsum(k3, 0) - k3)[seg]
            i = seg // 3 + a0
            r = xa[anc][i] - y[j] - v[j] * at[i][:, None]
            keep = torch.nonzero(((r * r).sum(1) <= (CUT * h) ** 2) & ((ta[anc][i] - tj[j]).abs() <= tau)
                                 & (aid[anc][i] != src[j]))[:, 0]
            i, j, r = i[keep], j[keep], r[keep]
            k = torch.exp(-(r * r).sum(1) / (2 * h * h))
            S.index_add_(0, anc[i], k)
            if gS is not None:
                gr = (gS[anc[i]] * k / (h * h))[:, None] * r
                gy.index_add_(0, j, gr)
                gv.index_add_(0, j, gr * at[i][:, None])
            a0 = a1
        if gS is not None:
            give(src, c, gy, gv)
    return S


def _linear64(x, v, t):
    """source() and give() of motion linear at the event, and the velocities' gradient that give() adds up."""
    g = torch.zeros_like(v)

    def give(ids, c, gy, gv):
        g.index_add_(0, ids, gy * (c - t[ids])[:, None] + gv)

    return (lambda ids, c: (x[ids] + v[ids] * (c - t[ids])[:, None], v[ids])), give, g


def _weights64(t, b, ta, ba, at_time, B, H, W, tau):
    """Window counts times the exposure's visible share; ``at_time(c)`` gives the anchors' positions at time c."""
    key = b.to(F64) * 4 + t
    ki = ba.to(F64) * 4 + ta
    wc = (torch.searchsorted(key, ki + tau, right=True) - torch.searchsorted(key, ki - tau) - 1).clamp(min=0).to(F64)
    counts = torch.bincount(b * 16 + (t * 16).long().clamp(0, 15), minlength=B * 16).to(F64).view(B, 16)
    vis, tot = torch.zeros_like(ta), torch.zeros_like(ta)
    for q in range(16):
        c = (q + 0.5) / 16
        y = at_time(c)
        w = counts[ba, q] * ((ta - c).abs() <= tau)
        vis += w * ((y[:, 0] >= 0) & (y[:, 0] <= W - 1) & (y[:, 1] >= 0) & (y[:, 1] <= H - 1))
        tot += w
    return wc.clamp(min=1) * (vis / tot.clamp(min=1)).clamp(min=1e-3)


def _score64(S, Wn, h, H, W):
    D = Wn * 2 * math.pi * h * h
    rho = 1e-2 / (H * W) + S / D
    return -torch.log(rho).mean(), -1.0 / (rho * D * len(S))


def _splat64(pos, w, b, B, H, W, kernel="bilinear", sigma=1.0):
    if kernel == "bilinear":
        base, taps = torch.floor(pos.detach()), [(x, y) for y in (0, 1) for x in (0, 1)]
    else:
        base, r = torch.round(pos.detach()), math.ceil(3 * sigma)
        taps = [(x, y) for y in range(-r, r + 1) for x in range(-r, r + 1)]
    img = pos.new_zeros(B * H * W)
    d = pos - base
    i0 = base.long()
    for x, y in taps:
        i, j = i0[:, 0] + x, i0[:, 1] + y
        wt = ((1 - (d[:, 0] - x).abs()) * (1 - (d[:, 1] - y).abs()) if kernel == "bilinear" else
              torch.exp(-((d[:, 0] - x) ** 2 + (d[:, 1] - y) ** 2) / (2 * sigma ** 2)) / (2 * math.pi * sigma ** 2))
        ok = torch.nonzero((i >= 0) & (i < W) & (j >= 0) & (j < H))[:, 0]
        img = img.index_add(0, ((b * H + j) * W + i)[ok], (w * wt)[ok])
    return img.view(B, H, W)


def _gather64(img, pos, b):
    return _bilinear(nnf.pad(img, (1, 1, 1, 1))[:, None], (pos + 1).clamp(min=0), b)[:, 0]


def _inside64(y, H, W):
    y = y.detach()
    return ((y[:, 0] >= 0) & (y[:, 0] <= W - 1) & (y[:, 1] >= 0) & (y[:, 1] <= H - 1)).to(F64)


def _bspline64(t, K):
    """(..., K): the clamped uniform cubic (K >= 3) B-splines N_1..N_K of K + 1 at t, by Cox and de Boor's recursion."""
    P = min(3, K)
    L = K + 1 - P
    u = [min(max(i - P, 0), L) / L for i in range(K + P + 2)]
    j = torch.floor(t * L).clamp(0, L - 1)
    N = [(j == i - P).to(F64) for i in range(K + P + 1)]
    for q in range(1, P + 1):
        N = [((t - u[i]) / (u[i + q] - u[i]) * N[i] if u[i + q] > u[i] else 0 * t)
             + ((u[i + q + 1] - t) / (u[i + q + 1] - u[i + 1]) * N[i + 1] if u[i + q + 1] > u[i + 1] else 0 * t)
             for i in range(K + P + 1 - q)]
    return torch.stack(N[1:K + 1], -1)


def _traj64(c, coef, ev, seed):
    xy, t, _, b = ev
    B, H, W, K, tile = c["B"], c["H"], c["W"], c["K"], c["tile"]
    t = t.to(F64)
    full = coef.detach().to(F64).requires_grad_(True)
    off = tile // 2
    fld = full if tile == 1 else full[:, :, off::tile, off::tile]
    rows = lambda p: _bilinear(fld, (p - off) / tile if tile > 1 else p, b)  # noqa: E731

    def disp(cf, g):                            # rows [y_1.. y_K, x_1.. x_K] and the basis -> (x, y)
        return torch.stack([(cf[:, K:] * g).sum(1), (cf[:, :K] * g).sum(1)], 1)

    def origin(q, steps=STEPS):
        p, g = q, _bspline64(t, K)
        for _ in range(steps):
            p = q - disp(rows(p), g)
        return p

    def table(cc):                              # basis and derivative at one time
        tt = torch.tensor([cc], dtype=F64, device=DEV, requires_grad=True)
        val = _bspline64(tt, K)[0]
        der = torch.stack([torch.autograd.grad(val[k], tt, retain_graph=True)[0][0] for k in range(K)])
        return val.detach(), der

    xs, xa = _noise(xy, int(seed), 1.0)
    start = origin(xs)
    cf = rows(start)
    p0, c0 = start.detach(), cf.detach()
    gp, gc = torch.zeros_like(p0), torch.zeros_like(c0)

    def source(ids, cc):
        val, der = table(cc)
        return p0[ids] + disp(c0[ids], val), disp(c0[ids], der)

    def give(ids, cc, gy, gv):
        val, der = table(cc)
        gp.index_add_(0, ids, gy)
        gc.index_add_(0, ids, torch.cat([gy[:, 1:] * val + gv[:, 1:] * der, gy[:, :1] * val + gv[:, :1] * der], 1))

    aid = torch.arange(len(t), device=DEV)
    S = _pairs64(source, t, b, xa, t, b, aid, 1.0, c["tau"])
    with torch.no_grad():
        pa = origin(xa)
        ca = rows(pa)
        Wn = _weights64(t, b, t, b, lambda cc: pa + disp(ca, _basis_at64(cc, K)), B, H, W, c["tau"])
    loss, gS = _score64(S, Wn, 1.0, H, W)
    _pairs64(source, t, b, xa, t, b, aid, 1.0, c["tau"], gS, give)
    torch.autograd.backward([start, cf], [gp, gc])
    del start, cf
    pos = origin(xy.to(F64))
    y = pos + disp(rows(pos), _basis_at64(0.5, K))
    var = _splat64(y, _inside64(y, H, W), b, B, H, W).var(dim=(-2, -1)).mean()
    (-var).backward()
    return {"loss": loss - var.detach(), "grad": full.grad}


def _basis_at64(cc, K):
    return _bspline64(torch.tensor(cc, dtype=F64, device=DEV), K)


def exact(case, seed):
    c, d = case, _inputs(case, seed)
    k, B, H, W = c["kind"], c["B"], c["H"], c["W"]
    if k == "score":
        xy, t, _, b = d["ev"]
        t = t.to(F64)
        grid = d["grid"].to(F64).requires_grad_(True)
        xs, xa = _noise(xy, int(seed), c["h"])
        v = _flow_at(grid, xs, b, H, W)
        source, give, g = _linear64(xs, v.detach(), t)
        aid = torch.arange(len(t), device=DEV)
        S = _pairs64(source, t, b, xa, t, b, aid, c["h"], c["tau"])
        va = _flow_at(grid.detach(), xa, b, H, W)
        Wn = _weights64(t, b, t, b, lambda cc: xa + va * (cc - t)[:, None], B, H, W, c["tau"])
        loss, gS = _score64(S, Wn, c["h"], H, W)
        _pairs64(source, t, b, xa, t, b, aid, c["h"], c["tau"], gS, give)
        v.backward(g)
        return {"loss": loss, "grad": grid.grad}
    if k in ("pairs", "reflayout"):
        if min(c["m"], c["n"]) * _pairs_per_anchor(c) > 5e9:      # minutes of 64-bit pairs
            return None
        x, t, v, xa = (d[q].to(F64) for q in ("x", "t", "v", "xa"))
        a = torch.arange(c["n"], device=DEV) if d["anchors"] is None else d["anchors"]
        source, give, g = _linear64(x, v, t)
        S = _pairs64(source, t, d["b"], xa, t[a], d["b"][a], a, c["h"], c["tau"], d["gS"].to(F64), give)
        return {"S": S, "grad": g}
    if k == "iwe":
        xy, t, _, b = d["ev"]
        grid = d["grid"].to(F64).requires_grad_(True)
        y = xy.to(F64) + _flow_at(grid, xy.to(F64), b, H, W) * (0.5 - t.to(F64))[:, None]
        img = _splat64(y, _inside64(y, H, W), b, B, H, W)
        vals = _gather64(img, y, b)
        vals.backward(d["gv"].to(F64))
        return {"img": img, "vals": vals, "grad": grid.grad if c["motion"] == "dense" else grid.grad.view(B, 2)}
    if k == "ops":
        pos, w = d["pos"].to(F64).requires_grad_(True), d["w"].to(F64).requires_grad_(True)
        img = _splat64(pos, w, d["b"], B, H, W, c["kernel"], c["sigma"])
        vals = _gather64(img, pos, d["b"])
        torch.autograd.backward([img, vals], [d["gi"].to(F64), d["gv"].to(F64)])
        return {"img": img, "vals": vals, "gpos": pos.grad, "gw": w.grad}
    if k == "voxel":
        xy, t, p, b = d["ev"]
        tn = t.to(F64) * (c["C"] - 1)
        t0 = torch.floor(tn)
        vox = torch.zeros(B * c["C"], H, W, dtype=F64, device=DEV)
        for tb in (t0, t0 + 1):
            ok = torch.nonzero(tb < c["C"])[:, 0]
            vox += _splat64(xy.to(F64)[ok], (p * (1 - (tb - tn).abs()))[ok], b[ok] * c["C"] + tb.long()[ok],
                            B * c["C"], H, W)
        vox = vox.view(B, -1)
        for q in range(B):
            nz = vox[q] != 0
            x = vox[q][nz]
            vox[q][nz] = (x - x.mean()) / x.std()
        return {"vox": vox.view(B, c["C"], H, W)}
    if k == "traj":
        return _traj64(c, d["coef"], d["ev"], seed)
    full = d["coef"].to(F64).requires_grad_(True)
    fld = full[:, :, 2::4, 2::4]
    Hq, Wq = fld.shape[-2:]
    K = c["K"]
    tt = torch.cat([d["t_ref"].to(F64).view(1), (torch.arange(c["bins"], device=DEV) + 0.5).to(F64) / c["bins"]])
    cf = fld.reshape(B, 2, K, Hq * Wq).flip(1)
    disp = torch.einsum("tk,bckn->btnc", _bspline64(tt, K), cf)
    cent = torch.cartesian_prod(torch.arange(Hq, device=DEV), torch.arange(Wq, device=DEV)).flip(-1).to(F64) * 4 + 2
    Hl, Wl = -(-H // 4), -(-W // 4)
    q = torch.cartesian_prod(torch.arange(Hl, device=DEV), torch.arange(Wl, device=DEV)).flip(-1).to(F64) * 4 + 1.5
    kk = min(c["knn"], Hq * Wq)
    planes = []
    for bb in range(B):
        for s in range(c["bins"]):
            pts = (cent + disp[bb, 1 + s]).detach()
            idx = []
            for r in range(0, len(q), 4096):
                dx = q[r:r + 4096, None, 0] - pts[None, :, 0]
                dy = q[r:r + 4096, None, 1] - pts[None, :, 1]
                idx.append(torch.topk(dx * dx + dy * dy, kk, dim=1, largest=False).indices)
            idx = torch.cat(idx)
            mv = disp[bb, 0] - disp[bb, 1 + s]
            planes.append(mv.index_select(0, idx.reshape(-1)).view(-1, kk, 2).mean(1))
    table = torch.stack(planes).view(B, c["bins"], Hl, Wl, 2)
    table.backward(d["gt"].to(F64))
    return {"table": table, "grad": full.grad}
