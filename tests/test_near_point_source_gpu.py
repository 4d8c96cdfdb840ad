"""Near fields of sources much smaller than a wavelength, on targets within and
around the near zone, against the CPU oracle: there the 1 / (k R) and
1 / (k R)^2 terms set how fast the field changes with the distance, not the
sources' extent.  Sizes at which the Chebyshev patches are tried.

Tolerances: the repository's bars, 1e-5 of each field's peak mixed and 1e-10
FP64."""

import numpy as np
import pytest

from oracle import bind as OB
from pypo_amd import geometry as G
from pypo_amd import types as T

pytestmark = pytest.mark.gpu

TOL = {"fp64": 1e-10, "mixed": 1e-5}
K = 2 * np.pi
N_S, N_T = 33, 491


def _plane(h, n, z):
    p = G.plane({"gmode": "xy", "lims_x": [-h, h], "lims_y": [-h, h], "gridsize": [n, n]})
    p["transf"] = G.mat_translate([0, 0, z])
    return p


# half width of the source and distance of the targets in wavelengths, and how
# far (a share of their distance) the targets scatter off their plane
@pytest.mark.parametrize("hw,dist,spread", [(2e-6, 0.2, 1.0), (2e-6, 1.3, 0.0), (2e-6, 20.0, 0.0), (1e-4, 0.03, 1.0),
                                            (1e-3, 0.1, 0.1), (1e-2, 0.4, 0.5), (0.1, 1.3, 0.3)])
@pytest.mark.parametrize("mode,prec,exp", [("JM", "mixed", "fwd"), ("EH", "mixed", "bwd"), ("JM", "fp64", "bwd"),
                                           ("JMEH", "fp64", "fwd")])
def test_point_like_source_matches_oracle(hip, port, hw, dist, spread, mode, prec, exp):
    import torch
    from pypo_amd import device as D
    src = _plane(hw, N_S, 0.0)
    g_s, g_t = D.generate_grid(src), D.generate_grid(_plane(0.8 * dist, N_T, dist))
    n_t = g_t.shape[1]
    rng = np.random.default_rng(7)
    if spread:
        g_t[0:3] *= 1.0 + spread * torch.as_tensor(rng.random(n_t), device="cuda")
    c = [rng.standard_normal((N_S, N_S)) + 1j * rng.standard_normal((N_S, N_S)) for _ in range(6)]
    vals = D.currents_tensor(T.currents(*c))
    out = D.propagate(mode, g_s, g_t, vals, src, K, exp=exp, precision=prec).cpu().numpy()
    idx = np.unique(np.concatenate([rng.integers(0, n_t, 250), [0, N_T - 1, n_t // 2, n_t - 1]]))
    pts = g_t[:, torch.as_tensor(idx, device="cuda")].cpu().numpy()
    ref = OB.propagate_on_grids(port, mode, g_s.cpu().numpy(), (int(src["gmode"]), N_S, N_S), pts, vals.cpu().numpy(),
                                K, exp=exp)
    for g in range(0, ref.shape[0], 6):
        pk = np.max(np.abs(out[g:g + 6]))
        if pk == 0:
            assert np.all(ref[g:g + 6] == 0)
            continue
        err = np.max(np.abs(out[g:g + 6, idx] - ref[g:g + 6])) / pk
        print(f"{hw} at {dist}, spread {spread}, {mode} {prec} {exp} rows {g}: {err:.2e} of peak")
        assert err <= TOL[prec]
