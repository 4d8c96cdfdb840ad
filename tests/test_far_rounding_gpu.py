"""Rounding of FP64 far fields: what the Chebyshev grid adds to it."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,z,half,n_az,n_el", [(1000.0, 0.0, 8e-3, 201, 201), (1000.0, -700.0, 8e-3, 203, 199),
                                                (300.0, 2500.0, 25e-3, 181, 171)])
def test_fp64_far_field_rounds_like_its_sums(hip, d, z, half, n_az, n_el):
    """A focused dish of d wavelengths, z from the origin.  The reference takes
    the same directions (cosines in FP64, a common rounding of up to 2 pi z / 2^54
    otherwise), phases in extended precision and sums them in FP64.  A sum's own
    error is its phases' rounding, 2 pi |r| / 2^54 a source and mostly averaged out
    over tens of thousands; the bar leaves a quarter of that for what sources
    share, and 1e-14 for the polynomials (3e-15) and the sums."""
    import torch
    from pypo_amd import device as D
    from pypo_amd import geometry as G
    k = 2 * np.pi
    src = G.paraboloid({"pmode": "focus", "vertex": [0, 0, 0], "focus_1": [0, 0, 0.4 * d], "gmode": "uv",
                        "lims_u": [0, d / 2], "lims_v": [0, 360], "gridsize": [301, 300]})
    src["transf"] = G.mat_translate([0, 0, z])
    deg = np.degrees(half)
    ff = G.plane({"gmode": "AoE", "lims_Az": [-deg, deg], "lims_El": [-deg, deg], "gridsize": [n_az, n_el]})
    g, t = D.generate_grid(src), D.generate_grid(ff)
    p = g[0:3].clone()
    p[2] -= z + 0.4 * d
    r = torch.linalg.norm(p, dim=0)
    wave = torch.polar(torch.exp(-1.15 * (g[0] ** 2 + g[1] ** 2) / (d / 2) ** 2), -k * r)
    zero = torch.zeros_like(r)
    cur = torch.stack([wave.real, zero, zero, wave.imag] + [zero] * 8).contiguous()
    out = D.propagate("FF", g, t, cur, src, k, precision="fp64").cpu().numpy()
    rng = np.random.default_rng(3)
    idx = rng.integers(0, t.shape[1], 120)
    th, ph = t[0].cpu()[idx], t[1].cpu()[idx]
    th, ph = th.cuda(), ph.cuda()
    u = torch.stack([torch.cos(ph) * torch.sin(th), torch.sin(ph) * torch.sin(th), torch.cos(th)]).cpu().numpy()
    pos = g[0:3].cpu().numpy().astype(np.longdouble)
    w = np.ones((301, 300))
    w[[0, -1]] *= 0.5                        # the trapezoid weights of a uv grid
    c = wave.cpu().numpy() * w.ravel() * g[6].cpu().numpy()
    sums = []
    for i in range(idx.size):
        rev = pos[0] * u[0, i] + pos[1] * u[1, i] + pos[2] * u[2, i]
        sums.append((c * np.exp(2j * np.pi * (rev - np.rint(rev)).astype(np.float64))).sum())
    # E_x of J along x: -j pref (S - r_x^2 S)
    ref = -1j * np.array(sums) * (1 - u[0] ** 2)
    got = (out[0] + 1j * out[3])[idx]
    got = got * (np.vdot(got, ref) / np.vdot(got, got)).real     # the prefactor
    err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    bar = 1e-14 + 0.25 * k * (abs(z) + d / 4) * 2.0 ** -54
    print(f"{d} at {z}: {err:.2e}, bar {bar:.2e}")
    assert err <= bar
