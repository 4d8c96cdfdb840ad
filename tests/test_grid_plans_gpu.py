"""Which calls the Chebyshev grids take (pypo_hip_last_grids), against the CPU
oracle on both sides of the decision, at sizes well inside the range where a
plan is tried.

Tolerances.  Mixed: FP32 phases (2e-7 rad), sines and products of terms whose
sizes add up to a few times the peak: 2e-6 of it; unit Poynting vectors (EHP)
the repository's 1e-5.  FP64: phases of 3e3 rad rounded to 2^-53: 1e-12;
gradients, which are differences of such sums, 2e-6 and 1e-11 of the largest."""

import ctypes

import numpy as np
import pytest

from helpers import current_rows, grid_rows
from oracle import adjoint as OA
from oracle import bind as OB
from pypo_amd import adjoint as PA
from pypo_amd import geometry as G
from pypo_amd import types as T

pytestmark = pytest.mark.gpu

TOL = {"mixed": 2e-6, "fp64": 1e-12}
K = 2 * np.pi
OFF, ON = 1, 2


@pytest.fixture
def grids(hip):
    """A call's eight numbers about its grids."""
    old = hip.pypo_hip_set_timing(1)

    def last():
        info = (ctypes.c_int * 8)()
        assert hip.pypo_hip_last_grids(info) == 0
        return list(info)

    yield last
    hip.pypo_hip_set_timing(old)


def _plane(h, n, z=0.0, flip=False, deg=0.0):
    p = G.plane({"gmode": "xy", "lims_x": [-h, h], "lims_y": [-h, h], "gridsize": [n, n], "flip": flip})
    a = np.radians(deg)
    r = np.eye(4)
    r[0, 0] = r[2, 2] = np.cos(a)
    r[0, 2], r[2, 0] = np.sin(a), -np.sin(a)
    p["transf"] = G.mat_translate([0, 0, z], r)
    return p


def _dish(n_u, n_v, d, f):
    return G.paraboloid({"pmode": "focus", "vertex": [0, 0, 0], "focus_1": [0, 0, f], "gmode": "uv",
                         "lims_u": [0, d / 2], "lims_v": [0, 360], "gridsize": [n_u, n_v]})


def _aoe(az, el, n_az, n_el):
    return G.plane({"gmode": "AoE", "lims_Az": az, "lims_El": el, "gridsize": [n_az, n_el]})


def _aperture(n, sign):
    """A tapered Huygens aperture with a smooth phase, travelling along sign z."""
    x = np.linspace(-1, 1, n)
    e = np.exp(-(x[:, None] ** 2 + x[None, :] ** 2) / 0.3) * np.exp(1j * (0.4 * x[:, None] - 0.3 * x[None, :] ** 2))
    z = 0 * e
    return T.currents(-e, -0.02 * e, z, sign * 0.02 * e, -sign * e, z)


FEED = _plane(1.8, 41, 240.0, True)
DISH = _dish(497, 503, 600.0, 240.0)
NEAR = {
    "feed_dish": (FEED, DISH, -1.0),
    "feed_small_dish": (_plane(1.0, 41, 240.0, True), _dish(497, 503, 300.0, 240.0), -1.0),   # no null on the dish
    "planes": (_plane(12.0, 101), _plane(40.0, 257, 220.0), 1.0),
    "too_near": (_plane(9.0, 101), _plane(30.0, 259, 20.0), 1.0),
    "part_in_shadow": (_plane(2.0, 61, 0.0, False, 60.0), _plane(200.0, 401, 120.0), 1.0),
}


def _oracle(port, mode, g_s, cells, vals, pts):
    if mode != "scalar":
        return OB.propagate_on_grids(port, mode, g_s, cells, pts, vals, K)
    _, nu, nv = cells                       # Propagation.h:1279-1331
    w = np.ones((nu, nv))
    w[[0, -1]] *= 0.5
    w[:, [0, -1]] *= 0.5
    u = (vals[0] + 1j * vals[1]) * w.ravel() * g_s[6]
    r = np.sqrt(((pts[:3, :, None] - g_s[:3, None, :]) ** 2).sum(0))
    f = (u * np.exp(1j * K * r) / r).sum(1) * (-K ** 2 / (4 * float(np.float32(3.14159265359))))
    return np.stack([f.real, f.imag])


@pytest.mark.parametrize("name,mode,prec,state", [
    ("feed_dish", "JM", "mixed", ON), ("feed_dish", "JM", "fp64", ON), ("feed_dish", "JMEH", "mixed", ON),
    ("feed_small_dish", "EHP", "mixed", ON), ("planes", "scalar", "mixed", ON), ("planes", "scalar", "fp64", ON),
    ("planes", "EH", "mixed", ON), ("planes", "EH", "fp64", ON), ("too_near", "EH", "mixed", OFF),
    ("too_near", "scalar", "mixed", OFF), ("part_in_shadow", "JM", "mixed", OFF),
    ("part_in_shadow", "EH", "fp64", OFF)])
def test_near_plans(grids, port, name, mode, prec, state):
    import torch
    from pypo_amd import device as D
    src, tgt, sign = NEAR[name]
    n = int(src["gridsize"][0])
    g_s, g_t = D.generate_grid(src), D.generate_grid(tgt)
    cur = _aperture(n, sign)
    vals = D.scalar_tensor(T.scalarfield(cur.components()[0])) if mode == "scalar" else D.currents_tensor(cur)
    out = D.propagate(mode, g_s, g_t, vals, src, K, precision=prec).cpu().numpy()
    info = grids()
    n_t = g_t.shape[1]
    idx = np.unique(np.concatenate([np.random.default_rng(1).integers(0, n_t, 150), [0, n_t - 1]]))
    pts = g_t[:, torch.as_tensor(idx, device="cuda")].cpu().numpy()
    ref = _oracle(port, mode, g_s.cpu().numpy(), (int(src["gmode"]), n, n), vals.cpu().numpy(), pts)
    step = 2 if mode == "scalar" else (3 if mode == "EHP" else 6)
    worst = 0.0
    for g in range(0, ref.shape[0], step):
        pk = np.max(np.abs(out[g:g + step]))
        worst = max(worst, np.max(np.abs(out[g:g + step, idx] - ref[g:g + step])) / pk if pk > 0 else 0.0)
        assert pk > 0 or np.all(ref[g:g + step] == 0)
    print(f"{name} {mode} {prec}: {info} {worst:.2e} of peak")
    assert info[0] == 0 and info[4] == state
    assert worst <= (1e-5 if mode == "EHP" else TOL[prec])


def test_not_finite_near(grids):
    """A target that is not a number, and an infinite scalar source: off."""
    import torch
    from pypo_amd import device as D
    src, tgt, _ = NEAR["planes"]
    g_s, g_t = D.generate_grid(src), D.generate_grid(tgt)
    u = D.scalar_tensor(T.scalarfield(_aperture(101, 1.0).components()[0]))
    ref = D.propagate("scalar", g_s, g_t, u, src, K)
    assert grids()[4] == ON
    bad = g_t.clone()
    bad[1, 4321] = float("nan")
    out = D.propagate("scalar", g_s, bad, u, src, K)
    assert grids()[4] == OFF
    assert torch.isnan(out[:, 4321]).all()
    keep = torch.arange(g_t.shape[1], device="cuda") != 4321
    assert ((out - ref)[:, keep].abs().max() / ref.abs().max()).item() <= 2 * TOL["mixed"]
    u[0, 77] = float("inf")
    out = D.propagate("scalar", g_s, g_t, u, src, K)
    assert grids()[4] == OFF
    assert not torch.isfinite(out[0]).any()


@pytest.mark.parametrize("az,el,magnetic,prec,state", [
    ([-1.5, 1.5], [-1.5, 1.5], True, "mixed", ON), ([-1.5, 1.5], [-1.5, 1.5], False, "fp64", ON),
    ([-70.0, 20.0], [-60.0, 60.0], True, "mixed", OFF)])
def test_far_plans(grids, port, az, el, magnetic, prec, state):
    """Rows of equal azimuth in grid order, none once shuffled; off where part
    of the box is in shadow."""
    import torch
    from pypo_amd import device as D
    src, ff = _dish(301, 302, 300.0, 120.0), _aoe(az, el, 121, 119)
    g_s, g_t = D.generate_grid(src), D.generate_grid(ff)
    e = torch.polar(torch.exp(-2 * (g_s[0] ** 2 + g_s[1] ** 2) / 150.0 ** 2), -K * torch.sqrt(
        g_s[0] ** 2 + g_s[1] ** 2 + (g_s[2] - 120.0) ** 2)).cpu().numpy().reshape(301, 302)
    z = 0 * e
    cur = T.currents(e, 0.1 * e, 0.3 * e, 0.2 * e if magnetic else z, e if magnetic else z, z)
    c = D.currents_tensor(cur)
    idx = np.unique(np.random.default_rng(2).integers(0, g_t.shape[1], 120))
    ref, _ = OB.farfield_subset(port, src, ff, cur, K, idx)
    out = D.propagate("FF", g_s, g_t, c, src, K, precision=prec)
    info = grids()
    full = D.tensor_to_complex6(out)
    worst = max(np.max(np.abs(full[g:g + 3, idx] - ref[g:g + 3])) / np.max(np.abs(full[g:g + 3])) for g in (0, 3))
    print(f"{az} {prec}: {info} {worst:.2e} of peak")
    assert info[0] == state and info[4] == 0 and info[3] == (119 if state == ON else 0)
    assert worst <= TOL[prec]
    D.propagate("FF", g_s, g_t[:, torch.randperm(g_t.shape[1], device="cuda")].contiguous(), c, src, K, precision=prec)
    assert grids()[0] in (OFF, state) and grids()[3] == 0


def test_two_streams_with_different_plans(grids, hip):
    """On and off on two streams at once: each as by itself."""
    import torch
    from pypo_amd import device as D
    calls = []
    for name in ("feed_dish", "part_in_shadow"):
        src, tgt, sign = NEAR[name]
        g_s, g_t = D.generate_grid(src), D.generate_grid(tgt)
        calls.append((g_s, g_t, D.currents_tensor(_aperture(int(src["gridsize"][0]), sign)), src))
    want = []
    for c, state in zip(calls, (ON, OFF)):
        want.append(D.propagate("JM", *c, K))
        assert grids()[4] == state
    hip.pypo_hip_set_timing(0)      # timing waits for every call
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    got = [[], []]
    for _ in range(4):
        for s, c, g in zip(streams, calls, got):
            with torch.cuda.stream(s):
                g.append(D.propagate("JM", *c, K))
    torch.cuda.synchronize()
    for w, g in zip(want, got):
        assert all(torch.equal(w, o) for o in g)
    for s in streams:
        D.release_scratch(s)


@pytest.mark.parametrize("n_dish,n_ff,n_feed,focal,ff_deg,far,near", [
    (401, 121, 45, 300.0, 1.0, ON, (ON, ON)), (401, 121, 45, 120.0, 65.0, OFF, (ON, OFF)),
    (151, 41, 15, 120.0, 1.0, 0, (0, 0))])
def test_gradient_plans(grids, port, n_dish, n_ff, n_feed, focal, ff_deg, far, near):
    """near: mixed and FP64, whose node counts do not pay over the half sky that
    a dish of f / D = 0.4 spans."""
    import torch
    feed, cur, dish, ff, k, radius = PA.surface_error_workload(
        n_dish=n_dish, n_ff=n_ff, n_feed=n_feed, diameter=300.0, focal=focal, lam=3.0, ff_deg=ff_deg)
    fr, dr, ffr = grid_rows(port, feed), grid_rows(port, dish), grid_rows(port, ff)
    d = PA.zernike_displacement(dr[0], dr[1], radius, sigma=0.05, seed=4)
    rng = np.random.default_rng(n_ff)
    E, g = rng.standard_normal((12, n_ff * n_ff)), rng.standard_normal(n_ff * n_ff)
    idx = np.arange(0, n_dish * n_dish, 1201)
    sub = OA.displace(dr, d)[:, idx].copy()
    sub[6] *= 2 * OA.trapezoid_weights(dish["gmode"], n_dish, n_dish)[idx]   # a grid of one row has weights of a half
    ref = OA.power_grad(fr, (feed["gmode"], n_feed, n_feed), current_rows(cur), sub, (1, 1, idx.size), ffr, E, g, k)
    prob = PA.ShapeProblem(feed, cur, dish, ff, k)
    for prec, bar, state in (("mixed", 2e-6, near[0]), ("fp64", 1e-11, near[1])):
        got = prob.power_grad(*(torch.tensor(v, device="cuda") for v in (d, E, g)), precision=prec).cpu().numpy()[idx]
        info = grids()
        worst = np.abs(got - ref).max() / np.abs(ref).max()
        print(f"{n_dish}^2 x {n_ff}^2, feed {n_feed}^2, +-{ff_deg} deg {prec}: {info} {worst:.2e}")
        assert info[0] == far and info[4] == state
        assert worst <= bar


@pytest.mark.parametrize("n_dish,n_ff,ff_deg,far", [(90, 300, 9.0, OFF), (64, 400, 6.0, OFF), (401, 121, 1.0, ON)])
def test_gradient_plan_counts_the_moments(grids, n_dish, n_ff, ff_deg, far):
    """A small dish under many targets: the targets' moments, one for every node
    and target, cost more than the reverse sums they would save."""
    import torch
    feed, cur, dish, ff, k, _ = PA.surface_error_workload(n_dish=n_dish, n_ff=n_ff, n_feed=9, ff_deg=ff_deg,
                                                          diameter=300.0, focal=120.0, lam=3.0)
    prob = PA.ShapeProblem(feed, cur, dish, ff, k)
    gen = torch.Generator(device="cuda").manual_seed(1)
    E = torch.randn((12, n_ff * n_ff), dtype=torch.float64, device="cuda", generator=gen)
    prob.power_grad(torch.zeros(n_dish * n_dish, dtype=torch.float64, device="cuda"), E, E[0])
    assert grids()[0] == far


def test_far_plan_of_a_scan_back_and_forth(grids):
    """Few sources, many targets: the series pays along rows of equal azimuth
    only.  Rows alternately reversed are none, though the first targets look like
    one: the sums at the targets then, and the same field."""
    import torch
    from pypo_amd import device as D
    src, ff = _plane(16.0, 36), _aoe([-12.0, 12.0], [-12.0, 12.0], 701, 703)
    g_s, g_t = D.generate_grid(src), D.generate_grid(ff)
    c = D.currents_tensor(_aperture(36, 1.0))
    ref = D.propagate("FF", g_s, g_t, c, src, K)
    info = grids()
    assert info[0] == ON and info[3] == 703
    order = torch.arange(701 * 703, device="cuda").view(701, 703).clone()
    order[1::2] = order[1::2].flip(1)
    order = order.reshape(-1)
    out = D.propagate("FF", g_s, g_t[:, order].contiguous(), c, src, K)
    print(info, grids())
    assert grids()[0] == OFF
    assert ((out - ref[:, order]).abs().max() / ref.abs().max()).item() <= TOL["mixed"]
