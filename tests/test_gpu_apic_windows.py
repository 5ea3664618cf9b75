"""The APIC pass's per-wave windows where they can go wrong (GPU, against the
oracle).

* ``spread``: particles uniform in the slab, so that the particles of a wave
  share base nodes and take turns, and every tile is uneven.
* ``heap``: a cell of more particles than the slot table has columns, over a
  slab of one particle a cell.
* ``up``/``down``/``aside``: a translation by 1.6 cells between two binnings:
  particles leave their wave's window (queued), fill the queue and leave
  their tile's window (node accumulators).

Tolerances are the parity tests' (1e-9 normwise in FP64, 1e-5 in FP32).  The
forces of an FP32 translation have one of their own: a node's velocity of
2e3 m/s is a ratio of two sums of some 27 rounded terms, wrong by about
7 * 6e-8 of itself; the weights' gradients, 1.5 / h in all, turn that into a
strain rate of 5 / s, and 20 steps of 1e-8 s with a modulus of 1.1e11 Pa into
1.1e5 Pa, 1e-3 of the 1e8 Pa that the particles start with.
"""
import numpy as np
import pytest

import parity
import workloads

pytestmark = pytest.mark.gpu
H = workloads.H
STEPS, DT, STRESS = 20, 1e-8, 1e8


def case(kind, cells):
    cfg = workloads.scaled(workloads.drill_config1(), cells, steps=STEPS)
    cfg = dict(cfg, dt=DT, transfer="apic", params=dict(cfg["params"], fixture_thickness=0.0))
    o, _ = parity.build_oracle(cfg)
    d = o.get_particles()
    rng = np.random.default_rng(7)
    d["stress"][:] = rng.uniform(-STRESS, STRESS, d["stress"].shape)
    if kind == "spread":
        d["pos"][:] = rng.uniform(0.0, 1.0, d["pos"].shape) * (np.array(cells) * H)
    elif kind == "heap":
        d = {k: np.ascontiguousarray(v[::8]) for k, v in d.items()}
        d["pos"][5:55] = (np.array([2.0, 2.0, 1.0]) + rng.uniform(0.0, 1.0, (50, 3))) * H
    else:
        v = {"up": (0.0, 0.0, 1.6), "down": (0.0, 0.0, -1.6), "aside": (1.6, -1.6, 0.4)}[kind]
        d["vel"][:] = np.array(v) * H / (STEPS * DT)
        name, desc, pose = cfg["tool"]   # out of the way: contact would add heat at nearly empty surface nodes
        x, y, z = pose["center"]
        cfg["tool"] = (name, desc, dict(pose, center=(x, y, z + 1.0)))
    return cfg, d


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-9), ("fp32", 1e-5)])
@pytest.mark.parametrize("kind,cells", [("spread", (9, 8, 5)), ("spread", (24, 17, 8)), ("heap", (9, 9, 5)),
                                        ("up", (17, 9, 9)), ("down", (17, 9, 9)), ("aside", (17, 9, 9))])
def test_windows_match_oracle(kind, cells, prec, tol):
    cfg, d = case(kind, cells)
    n = 1 if kind in ("spread", "heap") else STEPS
    res = parity.run_from_state(cfg, prec, d, n)
    errs = res["errors"]
    print(f"\n[{kind} {cells} {prec}] " + " ".join(f"{k}={v:.1e}" for k, v in sorted(errs.items())), flush=True)
    assert res["status_mismatch"] == 0
    for k in ("pos", "vel", "temperature", "grid_mass", "grid_momentum", "grid_force"):
        bound = 1e-3 if k == "grid_force" and prec == "fp32" and n > 1 else tol
        assert errs[k] <= bound, (k, errs[k])


def test_out_of_window_counts_device_memory_visits():
    """A particle that left its wave's window but not its tile's is added in
    LDS: the diagnostics count it in neither precision.  A translation by
    0.55 cells takes 5 % of the particles out of their wave's window (too few to
    fill a queue), a quarter of those out of the tile's; particles that the
    rounding of a position puts on the other side may differ."""
    cfg, d = case("up", (17, 9, 9))
    d["vel"][:] = np.array([0.0, 0.0, 0.55]) * H / (STEPS * DT)
    out = {}
    for prec in ("fp64", "fp32"):
        s = parity.build_gpu(cfg, prec, particles=d)
        s.run(STEPS, DT)
        out[prec] = s.diagnostics()["out_of_window"]
        s.close()
    print(f"\n[out of window] {out}", flush=True)
    assert out["fp64"] > 100 and abs(out["fp32"] - out["fp64"]) <= 0.02 * out["fp64"]


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-9), ("fp32", 1e-5)])
@pytest.mark.parametrize("kind,cells", [("spread", (9, 8, 5)), ("heap", (9, 9, 5)), ("pile", (9, 9, 5)),
                                        ("spread", (56, 48, 20)), ("pile", (56, 48, 20))])
def test_fused_pass_on_uneven_tiles(kind, cells, prec, tol):
    """Two steps, so that the fused pass walks the uneven tiles too, shared and
    (210 tiles) not; a pile is one cell of 400 (the small slab's) or 700
    particles, more than the slot table has columns."""
    cfg, d = case("heap" if kind == "pile" else kind, cells)
    rng = np.random.default_rng(11)
    if kind == "pile":
        d["pos"][5:min(705, len(d["pos"]))] = (np.array([3.0, 2.0, 1.0]) +
                                               rng.uniform(0.0, 1.0, (min(705, len(d["pos"])) - 5, 3))) * H
    d["stress"][:] = 0.0
    d["vel"][:] = rng.uniform(-1.0, 1.0, 3) + 200.0 * d["pos"][:, ::-1]
    res = parity.run_from_state(cfg, prec, d, 2)
    errs = res["errors"]
    print(f"\n[uneven {kind} {cells} {prec}] " + " ".join(f"{k}={v:.1e}" for k, v in sorted(errs.items())), flush=True)
    assert res["status_mismatch"] == 0
    for k in ("pos", "vel", "temperature", "grid_mass", "grid_momentum"):
        assert errs[k] <= tol, (k, errs[k])
