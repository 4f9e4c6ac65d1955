"""Fused pair-sum path (atl_fast_*) against the oracle: per-anchor neighbour counts bit-exact, sums within
1e-5 relative, velocity gradients within 1e-4 (relative to the largest magnitude, as gradient sums cancel).

The fused path bins positions on its own fine grid; these tests check that it finds exactly the reference's
contributing pairs (counts) and sums them to the reference's values, on the reference test shapes, on the
edge cases of the plan (empty inputs, clamped positions far outside the sensor, coincident events, anchor
subsets in any order) and at the full 1M-event size against the reference-layout kernels."""
import numpy as np
import pytest
import torch

import oracle as O
from tests.conftest import assert_sums_close, rand_events
from x_amd import synth
from x_amd.ops import functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda"
F32 = np.float32


def T(a):
    return torch.as_tensor(np.ascontiguousarray(a), device=DEV)


def N(t):
    return t.detach().cpu().numpy()


def close_rel(got, want, rel):
    scale = max(float(np.abs(want).max()), 1e-30) if want.size else 1.0
    err = float(np.abs(got.astype(np.float64) - want.astype(np.float64)).max()) if want.size else 0.0
    assert err <= rel * scale, f"max err {err:.3e} vs scale {scale:.3e} (rel {err / scale:.2e})"


def _case(seed=0, n=6000, B=2, H=40, W=48, h=1.0):
    win = synth.small_window(seed=seed, n=n // B, H=H, W=W, B=B)
    v, _, _ = O.dense_velocity(win.motion["grid"], win.xy, win.b, H, W)
    rng = np.random.default_rng(seed + 100)
    xs = (win.xy + rng.uniform(-0.5, 0.5, win.xy.shape)).astype(F32)
    xa = (xs + h * rng.standard_normal(xs.shape)).astype(F32)
    return win, xs, v, xa


class _PlannedSums(F.FastPairPlan):
    """The fused path with its plan, also where few events would be summed directly."""

    def _geometry(self, *sizes):
        super()._geometry(*sizes)
        self.geo.direct = 0.0


def check_against_oracle(xs, t, v, b, B, H, W, anchors, xa, h, tau, S, seed=0, index_free=False):
    """Counts, sums and gradients of the fused path vs the oracle on the reference plan, with its plan and, where few
    events are summed directly, that way too.  ``index_free``: the anchors are every event in order and the fused plan
    gets no index array (the benchmarked form)."""
    print(f"fast pair case N={len(t)} M={len(anchors)} B={B} HxW={H}x{W} h={h} tau={tau} S={S}", flush=True)
    p = O.build_pair_plan(xs, t, v, b, B, H, W, anchors, h, tau, 3.0, S, anchor_xy=xa)
    want, wcnt = O.ats_pair_fwd(p, h, tau, 3.0, with_counts=True)
    if index_free:
        assert np.array_equal(anchors, np.arange(len(t)))
    gS = np.random.default_rng(seed + 3).standard_normal(len(anchors)).astype(F32)
    want_g = O.ats_pair_bwd(gS, p, h, tau, 3.0, len(t))
    direct = False
    for cls in (F.FastPairPlan, _PlannedSums):
        plan = cls(T(xs), T(t), T(v), T(b), B, H, W, None if index_free else T(anchors), h, tau, 3.0, S,
                   None if xa is None else T(xa))
        if cls is _PlannedSums and not direct:
            break                                  # the plan was taken already
        direct = plan.geo.direct != 0
        assert np.array_equal(N(plan.counts()), wcnt)
        assert_sums_close(N(plan.forward()), want)
        close_rel(N(plan.backward(T(gS))), want_g, 1e-4)
    return wcnt


# at most 8, 9, 12 and 16 slices per source (the entry passes keep up to 12 in registers, more take two passes)
@pytest.mark.parametrize("tau,S,h", [(0.2, 16, 1.0), (1.0, 8, 1.5), (0.05, 4, 0.5), (0.2, 16, 2.0), (0.3, 16, 1.0),
                                     (0.6, 16, 1.0)])
def test_fast_matches_oracle(tau, S, h):
    win, xs, v, xa = _case(seed=11, h=h)
    cnt = check_against_oracle(xs, win.t, v, win.b, 2, 40, 48, np.arange(win.n), xa, h, tau, S)
    assert cnt.sum() > win.n                 # the case has real neighbourhoods


def test_fast_anchor_subsets_and_raw_positions():
    win, xs, v, xa = _case(seed=12)
    rng = np.random.default_rng(0)
    perm = rng.permutation(win.n)[: win.n // 3]              # unsorted subset, smoothed positions
    check_against_oracle(xs, win.t, v, win.b, 2, 40, 48, perm, xa[perm], 1.0, 0.2, 16)
    every3 = np.arange(0, win.n, 3)                          # x[anchors] (anchor_xy None)
    check_against_oracle(xs, win.t, v, win.b, 2, 40, 48, every3, None, 1.0, 0.2, 16)


def test_fast_duplicate_anchors():
    """An event listed twice among the anchors: both records skip exactly their own event (leave-one-out by id,
    the backward's fallback from the own-record position test)."""
    win, xs, v, xa = _case(seed=15)
    anchors = np.concatenate([np.arange(0, win.n, 2), np.arange(0, win.n, 6)])
    check_against_oracle(xs, win.t, v, win.b, 2, 40, 48, anchors, None, 1.0, 0.2, 16)
    check_against_oracle(xs, win.t, v, win.b, 2, 40, 48, anchors, xa[anchors], 1.0, 0.2, 16)


def test_fast_reference_test_shape():
    """tests/test_ops.py:62-77 shape: n=600, B=2, 20x24, positions in [-2, W+2), v = 6 N(0,1), h=1.5."""
    pos, _, b, t = rand_events(n=600, seed=3)
    v = (np.random.default_rng(1).standard_normal((600, 2)) * 6).astype(F32)
    anchors = np.arange(0, 600, 3)
    for tau, S in [(1.0, 8), (0.2, 16), (0.05, 4)]:
        check_against_oracle(pos, t, v, b, 2, 20, 24, anchors, None, 1.5, tau, S)


def test_fast_edge_cases():
    rng = np.random.default_rng(5)
    # coincident events: many at the same position and time (ties in t, d2 = 0, leave-one-out by id)
    n = 400
    xs = np.repeat(np.array([[10.0, 7.0], [30.0, 20.0]], F32), n // 2, axis=0)
    t = np.sort(np.repeat(rng.random(n // 8).astype(F32), 8))
    v = np.zeros((n, 2), F32)
    b = np.zeros(n, np.int64)
    check_against_oracle(xs, t, v, b, 1, 40, 48, np.arange(n), None, 1.0, 0.2, 16)
    # positions and slice-centre positions far outside the sensor (clamped bins), large velocities
    win, xs, v, xa = _case(seed=13)
    xs2 = xs.copy()
    xs2[::7] += F32(300.0)
    xs2[1::7] -= F32(250.0)
    v2 = (v * F32(8.0)).astype(F32)
    check_against_oracle(xs2, win.t, v2, win.b, 2, 40, 48, np.arange(win.n), xa, 1.0, 0.2, 16)
    # times exactly on slice boundaries and at 0 / 1
    t3 = np.sort(np.concatenate([np.arange(17, dtype=F32) / F32(16), rng.random(583).astype(F32)]))
    xs3 = (rng.random((600, 2)) * [48, 40]).astype(F32)
    v3 = (rng.standard_normal((600, 2)) * 3).astype(F32)
    check_against_oracle(xs3, t3, v3, np.zeros(600, np.int64), 1, 40, 48, np.arange(600), None, 1.0, 0.2, 16)


def test_fast_empty_inputs():
    x = torch.zeros(0, 2, device=DEV)
    t = torch.zeros(0, device=DEV)
    b = torch.zeros(0, dtype=torch.int64, device=DEV)
    plan = F.FastPairPlan(x, t, x, b, 1, 40, 48, b, 1.0, 0.2)
    assert plan.forward().shape == (0,) and plan.backward(t).shape == (0, 2)
    # events but no anchors
    win, xs, v, xa = _case(seed=14)
    plan = F.FastPairPlan(T(xs), T(win.t), T(v), T(win.b), 2, 40, 48, torch.zeros(0, dtype=torch.int64, device=DEV),
                          1.0, 0.2)
    assert plan.forward().shape == (0,)
    assert float(plan.backward(torch.zeros(0, device=DEV)).abs().sum()) == 0.0


def test_fast_api_autograd_matches_bruteforce():
    """ats_pair_sums on device (the fused path) vs the O(MN) fp64 brute force, values and gradients."""
    pos, _, b, t = rand_events(n=600, seed=3)
    rng = np.random.default_rng(1)
    v = (rng.standard_normal((600, 2)) * 6).astype(F32)
    anchors = np.arange(0, 600, 3)
    for tau, S in [(1.0, 8), (0.2, 16), (0.05, 4)]:
        tv = T(v).requires_grad_(True)
        s_ext = F.ats_pair_sums(T(pos), T(t), tv, T(b), 2, 20, 24, T(anchors), 1.5, tau, cut=3.0, n_slices=S)
        Sb, _, grad = O.pair_sums_fp64(pos, t, v, b, anchors, 1.5, tau, 3.0)
        assert np.allclose(N(s_ext), Sb, atol=1e-4, rtol=1e-4)
        gS = rng.standard_normal(len(anchors)).astype(F32)
        s_ext.backward(T(gS))
        assert np.allclose(N(tv.grad), grad(gS), atol=1e-4, rtol=1e-3)


def test_fast_plumbing_size_matches_oracle():
    """100k events on 240x180 (translation 2.0, -1.25 px per window): every event an anchor, vs the oracle."""
    win = synth.plumbing_translation(seed=0)
    rng = np.random.default_rng(21)
    xs = (win.xy + rng.uniform(-0.5, 0.5, win.xy.shape)).astype(F32)
    xa = (xs + rng.standard_normal(xs.shape)).astype(F32)
    v = np.broadcast_to(np.asarray(win.motion["theta"][:2], F32), xs.shape).copy()
    check_against_oracle(xs, win.t, v, win.b, 1, win.height, win.width, np.arange(win.n), xa, 1.0, 0.2, 16)


@pytest.mark.parametrize("h", [1.0, 0.5, 2.0])
def test_fast_full_size_matches_oracle(h):
    """The headline window at full size, directly against the oracle: 1M events at 640x480 (dense flow,
    dequantised sources, smoothed anchors, every event an anchor without an index array, as benchmarked), tau =
    0.2, 16 slices: every per-anchor count bit-exact, sums within 1e-5, velocity gradients within 1e-4."""
    win = synth.dense_flow_window(seed=0)
    rng = np.random.default_rng(0)
    xs = (win.xy + rng.uniform(-0.5, 0.5, win.xy.shape)).astype(F32)
    xa = (xs + h * rng.standard_normal(xs.shape)).astype(F32)
    v, _, _ = O.dense_velocity(win.motion["grid"], xs, win.b, 480, 640)
    cnt = check_against_oracle(xs, win.t, v, win.b, 1, 480, 640, np.arange(win.n), xa, h, 0.2, 16, index_free=True)
    assert cnt.sum() > 10 * win.n


def test_fast_blob_contention_matches_oracle():
    """Contention shape against the oracle: 4M events, 90% in 5 Gaussian blobs (sigma 8 px), Sim2 flow
    (0, 0, 0.1, 0.1), h = 1, a random 40k-anchor subset (thousands of neighbours each): counts bit-exact, sums
    within 1e-5, gradients within 1e-4."""
    win = synth.blob_window(seed=0)
    rng = np.random.default_rng(1)
    xs = (win.xy + rng.uniform(-0.5, 0.5, win.xy.shape)).astype(F32)
    th = win.motion["theta"].astype(F32)
    c = np.array([(640 - 1) / 2.0, (480 - 1) / 2.0], F32)
    d = (xs - c).astype(F32)
    v = np.stack([th[0] + (th[2] * d[:, 0] - th[3] * d[:, 1]), th[1] + (th[3] * d[:, 0] + th[2] * d[:, 1])],
                 1).astype(F32)
    anchors = np.sort(rng.choice(win.n, 40_000, replace=False))
    xa = (xs[anchors] + rng.standard_normal((len(anchors), 2))).astype(F32)
    cnt = check_against_oracle(xs, win.t, v, win.b, 1, 480, 640, anchors, xa, 1.0, 0.2, 16)
    assert cnt.mean() > 1000


@pytest.mark.parametrize("h", [1.0, 0.5, 2.0])
def test_fast_full_size_matches_reference_layout(h):
    """1M events at 640x480 (dense flow, dequantised sources, smoothed anchors, all anchors): the fused path
    against the reference-layout device plan + kernels (themselves pinned to the oracle above): counts
    bit-exact, sums within 1e-5, gradients within 1e-4."""
    print(f"full size h={h}", flush=True)
    win = synth.dense_flow_window(seed=0)
    rng = np.random.default_rng(0)
    xs = (win.xy + rng.uniform(-0.5, 0.5, win.xy.shape)).astype(F32)
    xa = (xs + h * rng.standard_normal(xs.shape)).astype(F32)
    v, _, _ = O.dense_velocity(win.motion["grid"], xs, win.b, 480, 640)
    anchors = T(np.arange(win.n))
    tx, tt, tv, tb, txa = T(xs), T(win.t), T(v), T(win.b), T(xa)
    ref_plan = F.build_pair_plan(tx, tt, tv, tb, 1, 480, 640, anchors, h, 0.2, 3.0, 16, anchor_xy=txa)
    want_cnt = N(F.pair_counts(ref_plan, h, 0.2, 3.0))
    e = F.get_ext()
    p = ref_plan
    want = N(e.ats_pair_fwd(p.src_y, p.src_v, p.src_t, p.src_id, p.cell_start, p.anc_x, p.anc_t, p.anc_cell,
                            p.anc_id, p.slice_c, p.S, p.GH, p.GW, h, 0.2, 3.0))
    plan = F.FastPairPlan(tx, tt, tv, tb, 1, 480, 640, anchors, h, 0.2, 3.0, 16, txa)
    assert np.array_equal(N(plan.counts()), want_cnt)
    assert_sums_close(N(plan.forward()), want)
    gS = torch.randn(win.n, device=DEV, generator=torch.Generator(device=DEV).manual_seed(4))
    gv_ref = N(e.ats_pair_bwd(gS, p.src_y, p.src_v, p.src_t, p.src_id, p.cell_start, p.anc_x, p.anc_t, p.anc_cell,
                              p.anc_id, p.slice_c, p.S, p.GH, p.GW, h, 0.2, 3.0, win.n))
    close_rel(N(plan.backward(gS)), gv_ref, 1e-4)


def test_fast_blob_contention_matches_reference_layout():
    """Contention stress shape: 4M events, 90% in 5 Gaussian blobs (sigma 8 px), Sim2 flow (0, 0, 0.1, 0.1),
    h = 1, a random 40k-anchor subset: fused path against the reference-layout device plan and kernels
    (counts bit-exact, sums within 1e-5, gradients within 1e-4)."""
    print("blob contention, 4M events", flush=True)
    win = synth.blob_window(seed=0)
    rng = np.random.default_rng(0)
    xs = (win.xy + rng.uniform(-0.5, 0.5, win.xy.shape)).astype(F32)
    th = win.motion["theta"].astype(F32)
    c = np.array([(640 - 1) / 2.0, (480 - 1) / 2.0], F32)
    d = (xs - c).astype(F32)
    v = np.stack([th[0] + (th[2] * d[:, 0] - th[3] * d[:, 1]), th[1] + (th[3] * d[:, 0] + th[2] * d[:, 1])],
                 1).astype(F32)
    anchors = np.sort(rng.choice(win.n, 40_000, replace=False))
    xa = (xs[anchors] + rng.standard_normal((len(anchors), 2))).astype(F32)
    tx, tt, tv, tb, ta, txa = T(xs), T(win.t), T(v), T(win.b), T(anchors), T(xa)
    ref_plan = F.build_pair_plan(tx, tt, tv, tb, 1, 480, 640, ta, 1.0, 0.2, 3.0, 16, anchor_xy=txa)
    want_cnt = N(F.pair_counts(ref_plan, 1.0, 0.2, 3.0))
    assert want_cnt.mean() > 1000                       # dense neighbourhoods
    e = F.get_ext()
    p = ref_plan
    args = (p.src_y, p.src_v, p.src_t, p.src_id, p.cell_start, p.anc_x, p.anc_t, p.anc_cell, p.anc_id, p.slice_c,
            p.S, p.GH, p.GW, 1.0, 0.2, 3.0)
    want = N(e.ats_pair_fwd(*args))
    plan = F.FastPairPlan(tx, tt, tv, tb, 1, 480, 640, ta, 1.0, 0.2, 3.0, 16, txa)
    assert np.array_equal(N(plan.counts()), want_cnt)
    assert_sums_close(N(plan.forward()), want)
    gS = torch.randn(len(anchors), device=DEV, generator=torch.Generator(device=DEV).manual_seed(5))
    close_rel(N(plan.backward(gS)), N(e.ats_pair_bwd(gS, *args, win.n)), 1e-4)


@pytest.mark.parametrize("planned", [False, True])
@pytest.mark.parametrize("B,H,W,Hg,Wg,h", [(2, 40, 48, 40, 48, 1.0), (2, 37, 53, 9, 14, 0.5), (1, 30, 36, 30, 1, 2.0),
                                            (3, 24, 20, 2, 2, 1.0)])
def test_pair_sums_flow_matches_oracle(B, H, W, Hg, Wg, h, planned, monkeypatch):
    """ats_pair_sums_flow (the flow sampled inside, its gradient accumulated over the plan's source records) against
    the oracle: sums within 1e-5, and the flow-grid gradient (pair backward, then sample_grid's adjoint) within
    1e-4, on full-resolution, coarse and degenerate grids, with sources far outside the sensor (clamped into the
    border nodes and the plan's box, so that their records fall outside the tile's window).  ``planned``: with the plan,
    also where the events are few enough for the direct sums."""
    if planned:
        monkeypatch.setattr(F, "FastPairPlan", _PlannedSums)
    print(f"pair sums flow B={B} {H}x{W} grid {Hg}x{Wg} h={h}", flush=True)
    rng = np.random.default_rng(B * 100 + Hg)
    n = 2500 * B
    win = synth.small_window(seed=Hg + Wg, n=n // B, H=H, W=W, B=B)
    grid = (rng.standard_normal((B, 2, Hg, Wg)) * 4.0).astype(F32)
    xs = (win.xy + rng.uniform(-0.5, 0.5, win.xy.shape)).astype(F32)
    xs[::97] = np.array([-40.0, 7.5], F32)                       # far outside: clamped in the grid and the box
    xs[1::101] = np.array([W + 30.0, H + 25.0], F32)
    xa = (xs + h * rng.standard_normal(xs.shape)).astype(F32)
    v, idx, wts = O.dense_velocity(grid, xs, win.b, H, W)
    anchors = np.arange(win.n)
    p = O.build_pair_plan(xs, win.t, v, win.b, B, H, W, anchors, h, 0.2, 3.0, 16, anchor_xy=xa)
    want = O.ats_pair_fwd(p, h, 0.2, 3.0)
    gS = rng.standard_normal(win.n).astype(F32)
    want_g = O.sample_grid_bwd(O.ats_pair_bwd(gS, p, h, 0.2, 3.0, win.n), idx, wts, grid.shape)
    tg = T(grid).requires_grad_(True)
    S = F.ats_pair_sums_flow(tg, T(xs), T(win.t), T(win.b), B, H, W, None, h, 0.2, 3.0, 16, anchor_xy=T(xa))
    assert_sums_close(N(S), want)
    (S * T(gS)).sum().backward()
    close_rel(N(tg.grad), want_g, 1e-4)


def test_pair_sums_flow_full_size_matches_composed():
    """1M events, 640x480, dense flow: the flow path's sums and grid gradient against sampling the flow and calling
    ats_pair_sums (whose own backward goes through sample_grid's binned adjoint)."""
    print("pair sums flow vs composed, 1M events", flush=True)
    win = synth.dense_flow_window(seed=0)
    H, W = win.height, win.width
    rng = np.random.default_rng(5)
    xs = T((win.xy + rng.uniform(-0.5, 0.5, win.xy.shape)).astype(F32))
    xa = T((N(xs) + rng.standard_normal(win.xy.shape)).astype(F32))
    t, b = T(win.t), T(win.b)
    gS = torch.randn(win.n, device=DEV)
    res = []
    for fused in (True, False):
        tg = T(win.motion["grid"]).requires_grad_(True)
        if fused:
            S = F.ats_pair_sums_flow(tg, xs, t, b, 1, H, W, None, 1.0, 0.2, 3.0, 16, anchor_xy=xa)
        else:
            v = F.sample_grid_hip(tg, xs, b, img_hw=(H, W))
            S = F.ats_pair_sums(xs, t, v, b, 1, H, W, None, 1.0, 0.2, 3.0, 16, anchor_xy=xa)
        (S * gS).sum().backward()
        res.append((N(S), N(tg.grad)))
    # the same pairs; the within-cell record order follows the plan's LDS atomics, so sums differ in the last bits
    assert_sums_close(res[0][0], res[1][0])
    close_rel(res[0][1], res[1][1], 1e-4)


@pytest.mark.parametrize("n,m,B,S,h,tau", [(1, None, 1, 16, 1.0, 0.2), (15, 7, 2, 1, 2.0, 0.4), (64, None, 1, 3, 1.0, 1.0),
                                           (65, 130, 3, 16, 0.7, 0.05), (2049, None, 2, 16, 1.0, 0.2),
                                           (16384, 2048, 4, 8, 1.5, 0.3)])
def test_direct_sums_equal_the_planned_ones(n, m, B, S, h, tau):
    print(f"direct sums n={n} m={m} B={B} S={S}", flush=True)
    rng = np.random.default_rng(n)
    H, W = 40, 48
    x = (rng.random((n, 2)) * [W + 3, H + 3] + 12).astype(F32)   # none near the corner where the plan keeps a NaN
    t = (rng.random(n) * 1.2 - 0.1).astype(F32)
    v = (rng.normal(size=(n, 2)) * 15).astype(F32)
    b = rng.integers(0, B, n)
    if n > 60:
        if S >= 8:                                 # outside every planned walk while these are short
            x[3] = np.nan
        x[5:9] = x[4]
        t[5:9] = t[4]
        b[10], b[11] = -1, B                       # left out
        v[12] = 60.0
    anchors = None if m is None else rng.integers(0, n, m)     # repeated events among them
    xa = x if m is None else x[anchors]
    xa = (xa + h * rng.normal(size=xa.shape)).astype(F32)
    gS = rng.normal(size=xa.shape[0]).astype(F32)
    res = []
    for cls in (F.FastPairPlan, _PlannedSums):
        p = cls(T(x), T(t), T(v), T(b), B, H, W, None if m is None else T(anchors), h, tau, 3.0, S, T(xa))
        assert (p.geo.direct != 0) == (cls is F.FastPairPlan)
        res.append((N(p.counts()), N(p.forward()), N(p.backward(T(gS))), N(p.backward_flow(T(gS), B, 7, 9, H, W))))
    (c0, s0, g0, f0), (c1, s1, g1, f1) = res
    assert np.array_equal(c0, c1)                  # the same pairs
    # the same fp32 terms (all below 1) in another order
    assert np.abs(s0 - s1).max() <= 2.0 ** -22 * max(c1.max(), 1)
    # a source's term is at most |gS| tau r / h^2 with r <= 3 h; fp32 sums of up to m of them
    bound = float(np.abs(gS).max()) * tau * 3.0 / h
    assert np.abs(g0 - g1).max() <= 2.0 ** -21 * bound * max(c1.max(), 1) * 4
    assert np.abs(f0 - f1).max() <= 2.0 ** -20 * max(np.abs(f1).max(), bound)


def test_direct_sums_end_at_their_limits():
    for n, m, direct in ((16384, 2048, True), (16385, 16, False), (5793, 5793, False), (5792, 5792, True)):
        x = torch.zeros(n, 2, device=DEV)
        a = torch.zeros(m, dtype=torch.int64, device=DEV)
        p = F.FastPairPlan(x, x[:, 0], x, a.new_zeros(n), 1, 40, 48, a, 1.0, 0.2)
        assert (p.geo.direct != 0) == direct


def test_entries_past_32_bit_offsets():
    """A second window whose entries stand behind 2^28 others of 16 bytes (byte offsets past 32 bits): its sums, counts
    and gradients are those of the window alone."""
    n0, n1, H, W, h, tau, S = 1 << 24, 3000, 512, 512, 1.0, 1.0, 16
    print(f"entries past 32-bit offsets: {n0 * S} in front", flush=True)
    rng = np.random.default_rng(8)
    xs = (rng.random((n1, 2)) * 40 + 200).astype(F32)
    t = np.sort(rng.random(n1)).astype(F32)
    v = (rng.normal(size=(n1, 2)) * 4).astype(F32)
    p = O.build_pair_plan(xs, t, v, np.zeros(n1, np.int64), 1, H, W, np.arange(n1), h, tau, 3.0, S)
    want, wcnt = O.ats_pair_fwd(p, h, tau, 3.0, with_counts=True)
    gS = rng.normal(size=n1).astype(F32)
    gen = torch.Generator(device=DEV).manual_seed(1)
    x_all = torch.cat([torch.rand(n0, 2, device=DEV, generator=gen) * H, T(xs)])
    t_all = torch.cat([torch.rand(n0, device=DEV, generator=gen), T(t)])
    v_all = torch.cat([torch.zeros(n0, 2, device=DEV), T(v)])
    b_all = torch.cat([torch.zeros(n0, dtype=torch.int64, device=DEV), torch.ones(n1, dtype=torch.int64, device=DEV)])
    anchors = torch.arange(n0, n0 + n1, device=DEV)
    plan = F.FastPairPlan(x_all, t_all, v_all, b_all, 2, H, W, anchors, h, tau, 3.0, S)
    assert np.array_equal(N(plan.counts()), wcnt)
    assert_sums_close(N(plan.forward()), want)
    gv = plan.backward(T(gS))
    close_rel(N(gv[n0:]), O.ats_pair_bwd(gS, p, h, tau, 3.0, n1), 1e-4)
    assert not gv[:n0].any()


def _crowd(B=3, per=47_001, H=60, W=72, seed=4):
    """Windows of events in two dense spots and a little noise, enough of them that the forward takes 16 anchors a wave."""
    rng = np.random.default_rng(seed)
    n = B * per
    x = np.where(rng.random((n, 1)) < 0.5, [20.0, 25.0], [50.0, 30.0]) + 5 * rng.normal(size=(n, 2))
    x = np.where(rng.random((n, 1)) < 0.1, rng.random((n, 2)) * [W, H], x).astype(F32)
    t = np.sort(rng.random((B, per)).astype(F32), 1).ravel()
    v = (rng.normal(size=(n, 2)) * 6).astype(F32)
    return x, t, v, np.repeat(np.arange(B), per), B, H, W


def test_crowd_of_many_anchors_matches_oracle():
    x, t, v, b, B, H, W = _crowd()
    xa = (x + np.random.default_rng(5).normal(size=x.shape)).astype(F32)
    cnt = check_against_oracle(x, t, v, b, B, H, W, np.arange(len(t)), xa, 1.0, 0.05, 16)
    assert cnt.mean() > 50


def test_crowd_with_velocities_that_are_not_finite():
    """Anchors taken 16 at a time from a common neighbourhood meet the same sources as in the passes of smaller anchor
    sets, those of NaN, infinite and huge velocities among them (a NaN distance counts as a visit)."""
    x, t, v, b, B, H, W = _crowd()
    n, per = len(t), len(t) // B
    v[per + 11], v[per + 30_000], v[2 * per + 7], v[2 * per + 8] = [np.nan, 0], [0, np.nan], [np.inf, 0], [1e31, -1e31]
    print(f"crowd with wild velocities n={n}", flush=True)
    run = lambda a: F.FastPairPlan(T(x), T(t), T(v), T(b), B, H, W, T(a), 1.0, 0.05, 3.0, 16)  # noqa: E731
    parts = [run(a) for a in np.array_split(np.arange(n), 2)]      # below the count that takes 16 anchors a wave
    cnt, want = (np.concatenate([N(f(p)) for p in parts]) for f in (lambda p: p.counts(), lambda p: p.forward()))
    plan = run(np.arange(n))
    assert np.isnan(want).any() and np.isfinite(want).mean() > 0.3
    assert np.array_equal(N(plan.counts()), cnt)
    got, fin = N(plan.forward()), np.isfinite(want)
    assert np.array_equal(np.isfinite(got), fin)
    assert_sums_close(got[fin], want[fin])


def test_backward_with_products_past_the_float_range():
    """A pair that no test admits adds nothing, also where its velocity times its time offset is past the float range."""
    rng = np.random.default_rng(6)
    n, H, W = 400, 40, 48
    x = (rng.random((n, 2)) * [W, H]).astype(F32)
    t = np.sort(rng.random(n)).astype(F32)
    v = (rng.normal(size=(n, 2)) * 4).astype(F32)
    t[-1], t[-2] = 1e10, 0.97                      # an anchor far past the window, in the last slice with the others
    v[-2], v[-5] = [9e29, 0], [1e25, -1e29]
    print("products past the float range", flush=True)
    gS = rng.normal(size=n).astype(F32)
    run = lambda cls: N(cls(T(x), T(t), T(v), T(np.zeros(n, np.int64)), 1, H, W, None, 1.0, 0.2, 3.0, 16).backward(T(gS)))  # noqa: E731
    got, want = run(_PlannedSums), run(F.FastPairPlan)   # the direct sums select every term
    assert np.isfinite(want).all() and np.isfinite(got).all()
    close_rel(got, want, 1e-4)
    coef = np.zeros((n, 2), F32)                   # K = 1: the displacement grows linearly in time
    coef[:, 0], coef[:, 1] = v[:, 1], v[:, 0]
    from x_amd.motion import PixelTrajectories
    tab = PixelTrajectories(torch.zeros(1, 2, 4, 5), 1, "polynomial", tile=1).slice_tables(16, DEV)
    p = F.FastPairPlan(T(x), T(t), None, T(np.zeros(n, np.int64)), 1, H, W, None, 1.0, 0.2, 3.0, 16, T(x), traj=(T(coef), 1, tab))
    assert all(bool(torch.isfinite(g).all()) for g in p.backward_traj(T(gS)))


@pytest.mark.parametrize("B,Hg,Wg", [(1, 1, 1), (1, 2, 2), (2, 1, 30), (2, 30, 1), (1, 32, 64), (1, 32, 65), (3, 40, 48)])
@pytest.mark.parametrize("crowd", [False, True])
def test_direct_flow_gradient_on_every_grid(B, Hg, Wg, crowd):
    """The adjoint of the direct sums, in LDS up to 4096 floats of gradient and with global atomics above, sources on
    the same cell merged by their wave: against the sources' own gradients put through the grid's adjoint."""
    print(f"direct flow gradient B={B} {Hg}x{Wg} crowd={crowd}", flush=True)
    rng = np.random.default_rng(Hg)
    n, H, W = 2500, 40, 48
    x = (rng.random((n, 2)) * [W + 30, H + 30] - 15).astype(F32)
    if crowd:
        x[rng.random(n) < 0.6] = [20.3, 17.6]
    t, v = np.sort(rng.random(n)).astype(F32), (rng.normal(size=(n, 2)) * 4).astype(F32)
    b = rng.integers(-1, B + 1, n)
    gS = rng.normal(size=n).astype(F32)
    p = F.FastPairPlan(T(x), T(t), T(v), T(b), B, H, W, None, 1.0, 0.2, 3.0, 16)
    assert p.geo.direct
    gv, got = N(p.backward(T(gS))), N(p.backward_flow(T(gS), B, Hg, Wg, H, W))
    keep = (b >= 0) & (b < B)
    _, idx, wts = O.dense_velocity(np.zeros((B, 2, Hg, Wg), F32), x[keep], b[keep], H, W)
    want = O.sample_grid_bwd(gv[keep], idx, wts, got.shape)
    mass = O.sample_grid_bwd(np.abs(gv[keep]), idx, wts, got.shape)
    assert (np.abs(got - want) <= 2.0 ** -19 * mass + 1e-12).all()     # fp32 sums in another order


@pytest.mark.parametrize("B,S", [(5, 13), (63, 1), (65, 1), (33, 4), (300, 16), (4500, 1)])
def test_backward_over_many_planes(B, S):
    """Windows times slices around and past 64 and 64^2 planes, most of them empty, in the planned backward: the
    gradients of the direct sums."""
    print(f"many planes B={B} S={S}", flush=True)
    rng = np.random.default_rng(B)
    n, H, W = 3000, 20, 24
    full = rng.choice(B, max(B // 3, 1), replace=False)
    b = np.sort(np.concatenate([full[rng.integers(0, len(full), n - 2)], [0, B - 1]]))
    x, t = (rng.random((n, 2)) * [W, H]).astype(F32), rng.random(n).astype(F32)
    v = (rng.normal(size=(n, 2)) * 3).astype(F32)
    gS = rng.normal(size=n).astype(F32)
    plans = [cls(T(x), T(t), T(v), T(b), B, H, W, None, 1.5, 0.2, 3.0, S) for cls in (_PlannedSums, F.FastPairPlan)]
    assert np.array_equal(*(N(p.counts()) for p in plans))
    close_rel(*(N(p.backward(T(gS))) for p in plans), 1e-4)


@pytest.mark.parametrize("m,S,wild", [(2000, 1, False), (900, 16, False), (700, 16, True), (None, 5, False)])
def test_backward_source_by_source(m, S, wild):
    """Sparse anchors of many sources take the backward source by source: unsorted and repeated anchors, one and several
    slices, a velocity past the bounds of the plain sums; against the oracle."""
    rng = np.random.default_rng(S + 2)
    n, B, H, W = 140_001, 3, 200, 260
    x = (rng.random((n, 2)) * [W + 20, H + 20] - 10).astype(F32)
    if m is None:                                  # all of them anchors, on a sensor that leaves few pairs
        H, W = 900, 1200
        x = (rng.random((n, 2)) * [W, H]).astype(F32)
    t = rng.random(n).astype(F32)
    v = (rng.normal(size=(n, 2)) * 3).astype(F32)
    if wild:
        v[7] = [5e18, 0]
    b = np.sort(rng.integers(0, B, n))
    anchors = np.arange(n) if m is None else np.concatenate([rng.integers(0, n, m), [7, 7, n - 1, 0]])
    check_against_oracle(x, t, v, b, B, H, W, anchors, None, 1.0, 0.1, S)


@pytest.mark.parametrize("n", [131_073, 500_001, 790_000])
def test_plans_of_every_block_size(n):
    """Event counts of each block size of the plan's passes, none a multiple of a block, half of them anchors: the linear
    sums and the flow gradient against the oracle."""
    rng = np.random.default_rng(n)
    B, H, W, Hg, Wg = 2, 300, 400, 9, 14
    x = (rng.random((n, 2)) * [W, H]).astype(F32)
    t = rng.random(n).astype(F32)
    b = np.sort(rng.integers(0, B, n))
    grid = (rng.normal(size=(B, 2, Hg, Wg)) * 4).astype(F32)
    v, idx, wts = O.dense_velocity(grid, x, b, H, W)
    anchors = np.sort(rng.choice(n, n // 2, replace=False))
    check_against_oracle(x, t, v, b, B, H, W, anchors, None, 1.0, 0.05, 16)
    p = F.FastPairPlan(T(x), T(t), T(v), T(b), B, H, W, T(anchors), 1.0, 0.05, 3.0, 16)
    gS = rng.normal(size=len(anchors)).astype(F32)
    want = O.sample_grid_bwd(N(p.backward(T(gS))), idx, wts, grid.shape)
    close_rel(N(p.backward_flow(T(gS), B, Hg, Wg, H, W)), want, 1e-4)


@pytest.mark.parametrize("n", [196_609, 530_001])
def test_reference_layout_of_every_block_size(n):
    """The reference-layout entries where pass A of its plan and of its anchors takes two and four items per thread:
    counts, sums and gradients of the fused path."""
    print(f"reference layout n={n}", flush=True)
    rng = np.random.default_rng(n)
    B, H, W = 2, 240, 320
    x, t = T((rng.random((n, 2)) * [W, H]).astype(F32)), T(rng.random(n).astype(F32))
    v, b = T((rng.normal(size=(n, 2)) * 4).astype(F32)), T(np.sort(rng.integers(0, B, n)))
    a = torch.arange(n, device=DEV)
    q = F.build_pair_plan(x, t, v, b, B, H, W, a, 1.0, 0.05, 3.0, 16)
    p = F.FastPairPlan(x, t, v, b, B, H, W, None, 1.0, 0.05, 3.0, 16)
    assert np.array_equal(N(F.pair_counts(q, 1.0, 0.05, 3.0)), N(p.counts()))
    tv = v.clone().requires_grad_(True)
    S = F._ATSPair.apply(tv, q, 1.0, 0.05, 3.0)
    assert_sums_close(N(S), N(p.forward()))
    gS = torch.randn(n, device=DEV, generator=torch.Generator(device=DEV).manual_seed(2))
    S.backward(gS)
    close_rel(N(tv.grad), N(p.backward(gS)), 1e-4)
