"""The point tool's nearest-sample search against the oracle (GPU).

The search shares a wave's lanes out to the nodes that ask for a sample, so
the cases vary how many do: samples filling the whole block (every node of
the grid, up to 64 per wave), one sample (single nodes), sample counts around
multiples of the wave and past the stride-2 decimation (n >= 8000), and a
partly filled last wave (grids that are no multiple of 64 nodes).  Two equally
near samples: the first one counts.  Tolerances as in the parity tests:
normwise 1e-9 in FP64 and 1e-5 in FP32 (the step's own rounding; the search
is FP64 in both).
"""
import numpy as np
import pytest

import parity
import workloads

pytestmark = pytest.mark.gpu
H = workloads.H


def case(cells, n, seed, twins=False):
    cx, cy, cz = cells
    rng = np.random.default_rng(seed)
    pts = rng.uniform(0.0, 1.0, (n, 3)) * np.array([cx, cy, cz]) * H
    if n == 1:
        pts = np.array([[0.5 * cx * H, 0.5 * cy * H, (cz - 0.3) * H]])
    if twins:   # mirrored pairs about the planes of nodes: equal distances
        pts = np.concatenate([pts, pts])
    cfg = workloads.scaled(workloads.slab_config0(), cells, steps=2, name=f"points_{n}")
    return dict(cfg, tool=("points", pts, 1.5 * H), vel=(-1.0, 0.3, -0.5))


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-9), ("fp32", 1e-5)])
@pytest.mark.parametrize("cells,n,twins", [((4, 4, 2), 1, False), ((5, 3, 2), 63, False), ((4, 4, 2), 65, True),
                                           ((7, 5, 3), 1000, False), ((6, 6, 4), 8191, False)])
def test_nearest_sample_matches_oracle(cells, n, twins, prec, tol):
    res = parity.run_case(case(cells, n, n, twins), prec, nsteps=2)
    e = res["errors"]
    m = res["metrics"]
    print(f"\n[points {n} {prec}] force {m[0].contact_force:.6g}/{m[1].contact_force:.6g} "
          + " ".join(f"{k}={v:.2e}" for k, v in sorted(e.items())), flush=True)
    assert res["status_mismatch"] == 0 and res["grid_same"]
    assert m[1].contact_force > 0 and abs(m[0].contact_force - m[1].contact_force) <= 10 * tol * m[1].contact_force
    for k in ("pos", "vel", "temperature", "plastic_strain", "grid_mass", "grid_momentum"):
        assert e[k] <= tol, (k, e[k])
