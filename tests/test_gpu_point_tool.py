"""The point tool's nearest-sample search against the oracle (GPU).

The search shares a wave's lanes out to the nodes that ask for a sample, so
the cases vary how many do: samples filling the whole block (every node of
the grid, up to 64 per wave), one sample (single nodes), sample counts around
multiples of the wave and past the stride-2 decimation (n >= 8000), and a
partly filled last wave (grids that are no multiple of 64 nodes).  Every sample
given twice changes nothing.  Of two equally near samples on opposite sides of a
node the first one counts, wherever the lanes find them (a lattice of binary
fractions, on which the distances are exact).  Tolerances as in the parity tests:
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
    if twins:   # every sample a second time
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


# a cell size that makes node positions, sample positions and squared
# distances exact
HB = 2.0 ** -12


def mirrored(cells, seed, fill):
    """Pairs of samples mirrored about nodes of the block, in a random order
    among `fill` samples further away from every node."""
    rng = np.random.default_rng(seed)
    nodes = np.stack(np.meshgrid(*(np.arange(c + 1) for c in cells), indexing="ij"), -1).reshape(-1, 3)
    nodes = nodes[rng.permutation(len(nodes))[:max(1, len(nodes) // 3)]]
    off = rng.integers(2, 5, nodes.shape) * rng.choice([-1, 1], nodes.shape)   # sixteenths of a cell
    pairs = np.concatenate([nodes + off / 16.0, nodes - off / 16.0])
    far = rng.integers(0, np.array(cells), (fill, 3)) + 0.5
    pts = np.concatenate([pairs, far])
    return pts[rng.permutation(len(pts))] * HB


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-9), ("fp32", 1e-5)])
@pytest.mark.parametrize("cells,fill", [((2, 1, 1), 0), ((60, 2, 1), 200), ((5, 4, 3), 500), ((13, 9, 4), 64)])
def test_first_of_equally_near_samples(cells, fill, prec, tol):
    cfg = workloads.scaled(workloads.slab_config0(), cells, steps=1, name=f"mirrored_{cells}")
    pts = mirrored(cells, 5, fill)
    cfg = dict(cfg, tool=("points", pts, 1.5 * HB), vel=(-1.0, 0.7, -0.5), tip=(0.0, 0.0, 0.0),
               params=dict(cfg["params"], cell_size=HB, tool_contact_radius=1.5 * HB))

    def mutate(d):   # the grid's origin on the lattice: a particle at the block's own
        d["pos"][:] = np.round(d["pos"] / HB * 64.0) / 64.0 * HB
        d["pos"][0] = 0.0

    def force(p):
        res = parity.run_case(dict(cfg, tool=("points", p, 1.5 * HB)), prec, nsteps=1, mutate=mutate)
        return res, [m.contact_force for m in res["metrics"]]

    res, f = force(pts)
    _, back = force(pts[::-1])
    e = res["errors"]
    print(f"\n[mirrored {cells} {prec}] force {f[0]:.6g}/{f[1]:.6g}, other order {back[1]:.6g} "
          + " ".join(f"{k}={v:.2e}" for k, v in sorted(e.items())), flush=True)
    assert res["status_mismatch"] == 0 and res["grid_same"]
    assert abs(back[1] - f[1]) > 1e-3 * f[1], "the order of the samples shows nothing here"
    for a, b in (f, back):
        assert abs(a - b) <= 10 * tol * b
    for k in ("pos", "vel", "temperature", "grid_mass", "grid_momentum"):
        assert e[k] <= tol, (k, e[k])
