"""A gradient with more feed points than 65 536 tiles, the largest grid.y of a launch."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_feed_of_more_tiles_than_a_launch_has_rows(hip):
    """Mixed against FP64 (the mixed gradient's bar, 1e-5 of the largest)."""
    import torch
    from pypo_amd import adjoint as PA
    from pypo_amd import geometry as G
    n = 4100
    assert (n * n + 255) // 256 > 65536
    feed = G.plane({"gmode": "xy", "lims_x": [-1.5, 1.5], "lims_y": [-1.5, 1.5], "gridsize": [n, n], "flip": True})
    feed["transf"] = G.mat_translate([0, 0, 60.0])
    dish = G.paraboloid({"pmode": "focus", "vertex": [0, 0, 0], "focus_1": [0, 0, 60.0], "gmode": "uv",
                         "lims_u": [0, 50.0], "lims_v": [0, 360], "gridsize": [33, 34]})
    ff = G.plane({"gmode": "AoE", "lims_Az": [-1, 1], "lims_El": [-1, 1], "gridsize": [9, 9]})
    x = torch.linspace(-1, 1, n, dtype=torch.float64, device="cuda")
    e = torch.exp(-(x[:, None] ** 2 + x[None, :] ** 2) / 0.4).reshape(-1)
    cur = torch.zeros((12, n * n), dtype=torch.float64, device="cuda")
    cur[0], cur[7] = -e, e
    prob = PA.ShapeProblem(feed, cur, dish, ff, 2 * np.pi)
    d = torch.zeros(prob.n_dish, dtype=torch.float64, device="cuda")
    field = torch.randn((12, 81), dtype=torch.float64, device="cuda", generator=torch.Generator("cuda").manual_seed(2))
    got = [prob.power_grad(d, field, field[0], precision=p) for p in ("fp64", "mixed")]
    assert torch.isfinite(got[0]).all() and got[0].abs().max() > 0
    assert ((got[1] - got[0]).abs().max() / got[0].abs().max()).item() <= 1e-5
