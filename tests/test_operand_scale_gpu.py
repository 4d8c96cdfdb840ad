"""The matrix kernels' FP16 operands (hi and lo halves, scaled per tile of 256):
small amplitudes beside large ones keep their 22 bits."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_src,ratio", [(256, 1e-3), (256, 1e-4), (1021, 1e-4), (300, 1e-5)])
def test_small_sources_beside_one_in_shadow(hip, n_src, ratio):
    """One source `ratio`^-1 larger than the rest of its tile faces away from
    all targets and adds nothing; the others' sum is held to 1e-6 of its peak:
    256 terms' FP32 phases and products, 1e-7 each of their own size, with room
    for a field that partly cancels."""
    import torch
    from pypo_amd import device as D
    from pypo_amd import geometry as G
    rng = np.random.default_rng(n_src)
    src = G.plane({"gmode": "xy", "lims_x": [-2, 2], "lims_y": [-2, 2], "gridsize": [n_src, 1]})
    ff = G.plane({"gmode": "AoE", "lims_Az": [-20, 20], "lims_El": [-20, 20], "gridsize": [31, 29]})
    g = torch.zeros((7, n_src), dtype=torch.float64)
    g[0:2] = torch.as_tensor(rng.uniform(-2, 2, (2, n_src)))
    g[5] = 1.0
    g[6] = 0.01
    cur = ratio * torch.as_tensor(rng.standard_normal((12, n_src)))
    cur[:, 0:6] += ratio * 2     # some of the sum adds up
    g[5, 100] = -1.0
    cur[:, 100] = 1.0
    g, cur, g_t = g.cuda(), cur.cuda(), D.generate_grid(ff)
    out = [D.propagate("FF", g, g_t, cur, src, 2 * np.pi, precision=p) for p in ("mixed", "fp64")]
    err = ((out[0] - out[1]).abs().max() / out[1].abs().max()).item()
    print(f"{n_src} sources, {ratio}: {err:.2e} of peak")
    assert err <= 1e-6


@pytest.mark.parametrize("kernel,bar", [("matrix", 1.9e-7), ("vector", 2.1e-7)])
def test_gradient_of_a_beam_is_as_good_as_its_sums(hip, kernel, bar):
    """Gradient of a far-field fit, mixed against FP64 for the same far field.
    Summed over every far-field target it is off by 1.7e-7 to 2.4e-7 of its norm
    (FP32 currents and phases; rms of these four 1.9e-7, 2.1e-7 on the vector
    ALUs); the sums at Chebyshev nodes have to be no worse."""
    import torch
    from pypo_amd import adjoint as PA
    from pypo_amd import bind as B
    feed, cur, dish, ff, k, radius = PA.surface_error_workload(n_dish=401, n_ff=151, n_feed=33)
    prob = PA.ShapeProblem(feed, cur, dish, ff, k)
    x, y = prob.g_dish0[0].cpu().numpy(), prob.g_dish0[1].cpu().numpy()
    ideal = (prob.far_field(torch.zeros_like(prob.g_dish0[0]), "fp64")[0:6] ** 2).sum(0)
    errs = []
    for seed in (5, 6, 7, 8):
        d = torch.tensor(PA.zernike_displacement(x, y, radius, sigma=0.02, seed=seed), device="cuda")
        e = prob.far_field(d, "fp64")
        g = 2 * ((e[0:6] ** 2).sum(0) - ideal) / ideal.max() ** 2
        B.set_ff_kernel(kernel)
        try:
            ref, got = (prob.power_grad(d, e, g, p) for p in ("fp64", "mixed"))
        finally:
            B.set_ff_kernel("matrix")
        errs.append((torch.linalg.norm(got - ref) / torch.linalg.norm(ref)).item())
    print(kernel, "gradient errors", ["%.2e" % v for v in errs])
    assert np.sqrt(np.mean(np.square(errs))) <= bar
