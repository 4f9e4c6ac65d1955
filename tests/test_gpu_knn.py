"""The HIP k-nearest-neighbour pass of MotionPriorCMax's look-up table against the oracle (bit-exact indices, in
order), and the look-up table and loss on the device against the package's CPU path."""
import numpy as np
import pytest
import torch

import oracle as O
from x_amd.ops import functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda"
F32 = np.float32


def _knn(q, pts, k):
    """pts (P, n, 2) numpy -> (P, Q, k) from the HIP pass."""
    qt = torch.as_tensor(q, device=DEV)
    pt = torch.as_tensor(pts, device=DEV)[None]
    out = F.knn_indices(qt, pt, k)
    torch.cuda.synchronize()
    return out[0].cpu().numpy()


@pytest.mark.parametrize("k", [1, 5, 8, 9, 16, 17, 32])
def test_knn_random_planes_match_oracle(k):
    print(f"knn random planes k={k}", flush=True)
    rng = np.random.default_rng(k)
    q = (rng.random((1500, 2)) * [160, 120]).astype(F32)
    pts = (rng.random((3, 700, 2)) * [170, 130] - 5).astype(F32)
    assert np.array_equal(_knn(q, pts, k), O.knn_indices(q, pts, k))


def test_knn_ties_on_a_lattice_in_index_order():
    print("knn lattice ties", flush=True)
    gy, gx = np.meshgrid(np.arange(12) * 4.0 + 2, np.arange(16) * 4.0 + 2, indexing="ij")
    pts = np.stack([gx.ravel(), gy.ravel()], 1).astype(F32)[None].repeat(2, 0)
    pts[1] = pts[1][::-1]                                       # same points, reversed indices
    hy, hx = np.meshgrid(np.arange(0, 48, 4) + 1.5, np.arange(0, 64, 4) + 1.5, indexing="ij")
    q = np.stack([hx.ravel(), hy.ravel()], 1).astype(F32)
    for k in (4, 8, 32):
        assert np.array_equal(_knn(q, pts, k), O.knn_indices(q, pts, k))


def test_knn_edge_cases():
    rng = np.random.default_rng(7)
    print("knn: points far outside the query box, coincident points, k = n", flush=True)
    q = (rng.random((300, 2)) * 30).astype(F32)
    pts = np.concatenate([(rng.random((1, 40, 2)) * 30).astype(F32),
                          np.array([[[1e4, 1e4], [-5e3, 7.0], [3.0, -2e4]]], F32),
                          np.full((1, 5, 2), 12.25, F32)], 1)
    for k in (1, 7, 32):
        assert np.array_equal(_knn(q, pts, k), O.knn_indices(q, pts, k))
    small = pts[:, :6]
    assert np.array_equal(_knn(q, small, 6), O.knn_indices(q, small, 6))
    print("knn: a single query, a single point", flush=True)
    assert np.array_equal(_knn(q[:1], pts[:, :1], 1), np.zeros((1, 1, 1), np.int64))
    with pytest.raises(ValueError):
        F.knn_indices(torch.as_tensor(q, device=DEV), torch.as_tensor(pts, device=DEV)[None], 33)


def _smooth_coeffs(B, C, H, W, seed, scale):
    g = torch.Generator().manual_seed(seed)
    c = torch.randn(B, C, H, W, generator=g)
    c = torch.nn.functional.avg_pool2d(c, 31, 1, 15, count_include_pad=False)
    return (c / c.abs().amax() * scale).float()


def test_knn_look_up_table_shape_against_oracle():
    # MotionPriorCMax's DSEC configuration: 480x640, 4 px cells (19200 queries), tile-4 trajectories (19200 points
    # per plane), 15 time bins, 32 neighbours; the oracle checks 2 planes on 1500 queries
    from x_amd.motion import PixelTrajectories
    from x_amd.objectives import MotionPriorCMaxLoss
    print("knn look-up table shape: 15 planes x 19200 points, 19200 queries, k = 32", flush=True)
    coef = _smooth_coeffs(1, 20, 480, 640, 0, 25.0).to(DEV)
    m = PixelTrajectories(coef, 10, "bspline", tile=4)
    loss = MotionPriorCMaxLoss()
    edges = torch.linspace(0, 1, 16, device=DEV)
    mids = (edges[:-1] + edges[1:]) * 0.5
    pts = m.tile_trajectories(mids)[0].contiguous()             # (15, 19200, 2)
    q = loss.cell_centres(480, 640, DEV)
    got = F.knn_indices(q, pts[None], 32)[0]
    torch.cuda.synchronize()
    rng = np.random.default_rng(0)
    sel = rng.choice(q.shape[0], 1500, replace=False)
    for plane in (0, 14):
        want = O.knn_indices(q.cpu().numpy()[sel], pts[plane:plane + 1].cpu().numpy(), 32)[0]
        assert np.array_equal(got[plane].cpu().numpy()[sel], want)


def test_mpcm_loss_device_matches_cpu():
    from x_amd import synth
    from x_amd.core import EventPacket
    from x_amd.motion import PixelTrajectories
    from x_amd.objectives import MotionPriorCMaxLoss
    print("mpcm loss device vs cpu", flush=True)
    win = synth.small_window(seed=4, n=6000, B=2)
    coef = _smooth_coeffs(2, 6, win.height, win.width, 1, 3.0)
    res = {}
    for dev in ("cpu", DEV):
        ev = EventPacket.from_window(win, dev)
        g = coef.clone().to(dev).requires_grad_(True)
        out = MotionPriorCMaxLoss(num_knn=16, t_ref=0.35)(ev, PixelTrajectories(g, 3, "bspline", tile=4))
        out["loss"].backward()
        res[dev] = (float(out["loss"].detach()), g.grad.detach().cpu().numpy())
    (l0, g0), (l1, g1) = res["cpu"], res[DEV]
    assert abs(l1 - l0) <= 1e-5 * abs(l0)
    assert np.abs(g1 - g0).max() <= 1e-4 * np.abs(g0).max()


def _lattice_case(kind, rng, n_side=(30, 44)):
    """tr (B, 1 + T, n, 2): tile trajectories on a 4 px lattice, displaced by ``kind``."""
    hy, hx = n_side
    gy, gx = np.meshgrid(np.arange(hy) * 4.0 + 2, np.arange(hx) * 4.0 + 2, indexing="ij")
    start = np.stack([gx.ravel(), gy.ravel()], 1)
    n = start.shape[0]
    tr = np.tile(start, (2, 4, 1, 1)).astype(F32)
    if kind == "smooth":
        tr += np.cumsum(rng.normal(size=(2, 4, 1, 2)) * 6, 1).astype(F32) + rng.normal(size=tr.shape).astype(F32)
    elif kind == "crowded":                        # most points in two corners, the rest uniform; planes differ
        tr[:, 1:] = (rng.random((2, 3, n, 2)) ** 4 * [4.0 * hx, 4.0 * hy]).astype(F32)
    elif kind == "far":                            # all but a few points hundreds of pixels outside the lattice
        tr[:, 1:, 5:] += F32(3000.0) + rng.random((2, 3, n - 5, 2)).astype(F32) * 500
    return tr                                      # "still": every displacement zero but ties everywhere


@pytest.mark.parametrize("k", [1, 7, 32])
@pytest.mark.parametrize("kind,lattice", [("smooth", (44, 30, 4.0)), ("still", (43, 29, 4.0)), ("crowded", (44, 30, 4.0)),
                                          ("far", (9, 5, 4.0)), ("smooth", (1, 1, 3.0)), ("smooth", (17, 65, 2.0))])
def test_lut_table_equals_the_indices_path(kind, lattice, k):
    print(f"lut table {kind} {lattice} k={k}", flush=True)
    nx, ny, step = lattice
    rng = np.random.default_rng(nx * 100 + k)
    tr = torch.as_tensor(_lattice_case(kind, rng), device=DEV)
    if kind == "still":
        tr[:, 0] += torch.rand_like(tr[:, 0])      # the ties' choice shows in the mean
    half = step / 2 - 0.5
    cy, cx = torch.arange(ny, device=DEV) * step + half, torch.arange(nx, device=DEV) * step + half
    centres = torch.cartesian_prod(cy, cx).flip(-1).contiguous()
    g = torch.as_tensor(rng.normal(size=(2, 3, nx * ny, 2)), dtype=torch.float32, device=DEV)
    a, b = tr.clone().requires_grad_(True), tr.double().requires_grad_(True)
    got = F.lut_table(a, half, half, step, nx, ny, k)
    want = F.lut_table_torch(b, centres, k)        # the same fp32 choice, averaged in fp64
    got.backward(g)
    want.backward(g.double())
    # k fp32 differences and additions of magnitude m: (k + 2) ulp
    m = float((b[:, :1] - b[:, 1:]).detach().abs().max())
    assert (got - want).abs().max().item() <= (k + 2) * 2.0 ** -24 * max(m, 1e-30) * 2 + 2.0 ** -24 * float(tr.abs().max())
    # a point's gradient adds at most Q terms of |g| / k; the reference row adds the bins'
    mass = torch.zeros_like(b)
    idx = F.knn_indices(centres, tr[:, 1:], k).view(2, 3, -1, 1).expand(-1, -1, -1, 2)
    mass[:, 1:].scatter_add_(2, idx, (g.double().abs() / k)[:, :, :, None].expand(-1, -1, -1, k, -1).reshape(2, 3, -1, 2))
    mass[:, 0] = mass[:, 1:].sum(1)
    hits = torch.zeros_like(mass[:, 1:]).scatter_add_(2, idx, torch.ones_like(idx, dtype=torch.float64)).max().item()
    assert ((a.grad - b.grad).abs() <= (hits + 4) * 2.0 ** -23 * mass).all()


def test_lut_table_differentiates_twice_and_leaves_transforms_to_torch():
    from x_amd.motion import PixelTrajectories
    from x_amd.objectives import MotionPriorCMaxLoss
    coef = _smooth_coeffs(1, 8, 41, 54, 3, 9.0).to(DEV).requires_grad_(True)
    obj = MotionPriorCMaxLoss(num_bins=3, num_knn=5)
    t_ref = torch.tensor(0.3, device=DEV)
    fn = lambda c: obj.lut_flow(PixelTrajectories(c, 4, "bspline", tile=4), 41, 54, t_ref)[0]  # noqa: E731
    table = fn(coef)
    g, = torch.autograd.grad((table ** 2).sum(), coef, create_graph=True)
    gg, = torch.autograd.grad((g ** 2).sum(), coef)
    # the table is J c: g = 2 J'J c and its squared norm's gradient 4 J'J g
    with torch.autograd.forward_ad.dual_level():
        d = torch.autograd.forward_ad.make_dual(coef.detach(), g.detach())
        jg = torch.autograd.forward_ad.unpack_dual(fn(d)).tangent
    want, = torch.autograd.grad((fn(coef) * jg).sum() * 4, coef)
    assert (gg - want).abs().max() <= 1e-4 * want.abs().max()      # fp32 sums of some hundred terms
    times = torch.rand(5, device=DEV)
    sq = lambda c: (PixelTrajectories(c, 4, "bspline", tile=4).tile_trajectories(times) ** 2).sum()  # noqa: E731
    want, = torch.autograd.grad(sq(coef), coef)
    assert (torch.func.grad(sq)(coef.detach()) - want).abs().max() <= 1e-5 * want.abs().max()


@pytest.mark.parametrize("K,tile,kind,nt", [(1, 4, "bspline", 1), (3, 1, "bezier", 5), (10, 4, "bspline", 16),
                                            (16, 3, "polynomial", 6), (4, 4, "bspline", 1000)])
def test_tile_trajectories_match_torch(K, tile, kind, nt):
    from x_amd.motion import PixelTrajectories
    from x_amd.motion.trajectories import basis
    g = torch.Generator().manual_seed(K)
    coef = torch.randn(2, 2 * K, 23, 37, generator=g)
    times = torch.rand(nt, generator=g)
    gout = None
    res = []
    for dev, dt in ((DEV, torch.float32), ("cpu", torch.float64)):
        c = coef.to(dev, dt).requires_grad_(True)
        m = PixelTrajectories(c, K, kind, tile=tile)
        if dt is torch.float32:
            pos = m.tile_trajectories(times.to(dev))
            gout = torch.randn(pos.shape, generator=g)
        else:
            gt = basis(times.double(), K, kind)
            disp = torch.einsum("tk,bckn->btnc", gt, m.tile_c.reshape(2, 2, K, -1).flip(1))
            start = torch.cartesian_prod(torch.arange(m.Hq) * tile + m.offset, torch.arange(m.Wq) * tile + m.offset).flip(-1)
            pos = start + disp
        pos.backward(gout.to(dev, dt))
        res.append((pos.detach().cpu().double(), c.grad.cpu().double()))
    (p0, g0), (p1, g1) = res
    # the basis to a few ulp of its recursions, K (nt) additions, positions up to 40 px
    assert (p0 - p1).abs().max() <= (K + 8) * 2.0 ** -23 * (coef.abs().max() * 4 + 40)
    assert (g0 - g1).abs().max() <= (nt + 8) * 2.0 ** -23 * (gout.abs().max() * nt ** 0.5 * 4)


def test_tile_trajectories_and_table_take_batched_gradients():
    """Several gradients at once through the backward (is_grads_batched: vmap over it), as the torch operations allow."""
    from x_amd.motion import PixelTrajectories
    from x_amd.objectives import MotionPriorCMaxLoss
    coef = _smooth_coeffs(1, 8, 41, 54, 3, 9.0).to(DEV).requires_grad_(True)
    obj = MotionPriorCMaxLoss(num_bins=3, num_knn=5)
    m = PixelTrajectories(coef, 4, "bspline", tile=4)
    for out in (m.tile_trajectories(torch.rand(5, device=DEV)), obj.lut_flow(m, 41, 54, torch.tensor(0.3, device=DEV))[0]):
        g = torch.randn(3, *out.shape, device=DEV)
        got, = torch.autograd.grad(out, coef, g, retain_graph=True, is_grads_batched=True)
        want = torch.stack([torch.autograd.grad(out, coef, gi, retain_graph=True)[0] for gi in g])
        assert (got - want).abs().max() <= 1e-5 * want.abs().max()     # fp32 sums of some hundred terms


@pytest.mark.parametrize("where", ["subclass", "class", "instance"])
def test_table_of_other_cell_centres(where, monkeypatch):
    """Centres that a user puts in the place of the lattice are the ones looked up."""
    from x_amd.motion import PixelTrajectories
    from x_amd.objectives import MotionPriorCMaxLoss

    def centres(self, H, W, device):
        return torch.rand(-(-H // self.lut) * -(-W // self.lut), 2, device=device, generator=torch.Generator(device).manual_seed(2)) * 40

    cls = type("Other", (MotionPriorCMaxLoss,), {"cell_centres": centres} if where == "subclass" else {})
    if where == "class":
        monkeypatch.setattr(MotionPriorCMaxLoss, "cell_centres", centres)
    obj = cls(num_bins=3, num_knn=5)
    if where == "instance":
        obj.cell_centres = lambda H, W, device: centres(obj, H, W, device)
    m = PixelTrajectories(_smooth_coeffs(1, 8, 41, 54, 3, 9.0).to(DEV), 4, "bspline", tile=4)
    t_ref = torch.tensor(0.3, device=DEV)
    mids = (torch.arange(3, device=DEV) + 0.5) / 3
    tr = m.tile_trajectories(torch.cat([t_ref.reshape(1), mids]))
    want = F.lut_table_torch(tr, centres(obj, 41, 54, DEV), 5)
    got = obj.lut_flow(m, 41, 54, t_ref)[0]
    assert (got.view_as(want) - want).abs().max() <= 1e-5 * want.abs().max()
