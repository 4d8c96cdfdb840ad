"""The gradient of a fit of far-field powers, forward and backward in mixed
precision: errors of the forward sums that neighbouring targets share do not
average out of the difference of two powers."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kernel,direct", [("matrix", 3.4e-7), ("vector", 3.9e-7)])
def test_gradient_of_a_power_difference(hip, kernel, direct):
    """|P(d) - P(0)|^2 of a 401^2 dish, 151^2 targets, against the same in FP64.
    direct: what sums at every target, which share no error, were off by, rms
    over these surfaces; the bar leaves a quarter."""
    import torch
    from pypo_amd import adjoint as PA
    from pypo_amd import bind as B
    feed, cur, dish, ff, k, radius = PA.surface_error_workload(n_dish=401, n_ff=151, n_feed=33)
    prob = PA.ShapeProblem(feed, cur, dish, ff, k)
    x, y = prob.g_dish0[0].cpu().numpy(), prob.g_dish0[1].cpu().numpy()

    def grad(d, prec):
        e0, e = (prob.far_field(v, prec) for v in (torch.zeros_like(d), d))
        p0, p = ((v[0:6] ** 2).sum(0) for v in (e0, e))
        return prob.power_grad(d, e, 2 * (p - p0) / p0.max() ** 2, prec)

    errs = []
    B.set_ff_kernel(kernel)
    try:
        for seed in range(20, 32):
            d = torch.tensor(PA.zernike_displacement(x, y, radius, sigma=0.02, seed=seed), device="cuda")
            ref, got = grad(d, "fp64"), grad(d, "mixed")
            errs.append((torch.linalg.norm(got - ref) / torch.linalg.norm(ref)).item())
    finally:
        B.set_ff_kernel("matrix")
    print("gradient errors", ["%.2e" % v for v in errs], "rms %.2e" % np.sqrt(np.mean(np.square(errs))))
    assert np.sqrt(np.mean(np.square(errs))) <= 1.25 * direct
