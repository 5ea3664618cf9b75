"""Tiles shared by several workgroups (GPU).

A workpiece of few tiles shares each tile among 2, 4 or 8 workgroups, alone and
in a batch.  A member's particles must stay those of the workpiece stepped
alone: up to the order of the sums that are formed with atomics, i.e. to
rounding carried through the steps (1e-9 normwise in FP64, 1e-5 in FP32, the
parity tests' tolerances), across a grid rebuild and across joining and
leaving.
"""
import numpy as np
import pytest

import mpmw
import parity
import workloads

pytestmark = pytest.mark.gpu
GATED = ("pos", "vel", "temperature", "plastic_strain", "stress")


def solver(cells, prec, transfer="pic"):
    cfg = dict(workloads.scaled(workloads.drill_config1(), cells, steps=30), transfer=transfer)
    return parity.build_gpu(cfg, prec)


@pytest.mark.parametrize("transfer", ["pic", "apic"])
@pytest.mark.parametrize("prec,tol", [("fp64", 1e-9), ("fp32", 1e-5)])
@pytest.mark.parametrize("cells", [(3, 2, 2), (17, 9, 6), (40, 33, 9)])
def test_member_sharing_changes_with_the_launch(cells, prec, tol, transfer):
    ref, mem, big = solver(cells, prec, transfer), solver(cells, prec, transfer), solver((64, 48, 24), prec, transfer)
    dt = 1e-8
    for _ in range(28):
        ref.step(dt)
    b = mpmw.Batch()
    b.add(big)
    for k in range(28):
        if k in (2, 24):     # into the large launch, the second time at the step before a rebuild
            b.add(mem)
        if k in (7, 26):     # and out of it
            b.remove(mem)
        if mem in b.members:
            b.step(dt)
        else:
            mem.step(dt)
    errs, mism = parity.compare_particles(mem.get_particles(), ref.get_particles())
    print(f"\n[{cells} {prec} {transfer}] " + " ".join(f"{k}={v:.1e}" for k, v in sorted(errs.items())), flush=True)
    assert mism == 0
    for k in GATED:
        assert errs[k] <= tol, (k, errs[k])
    b.close()
    for s in (ref, mem, big):
        s.close()


@pytest.mark.parametrize("cells", [(1, 1, 1), (9, 8, 4), (24, 24, 12), (41, 30, 20)])
def test_shared_tiles_match_oracle(cells):
    """One workgroup's share empty (1 particle per slot), tile edges, and a
    workpiece on each side of the sharing steps, against the oracle."""
    cfg = workloads.scaled(workloads.slab_config0(), cells, steps=3)
    res = parity.run_case(cfg, "fp64")
    assert res["status_mismatch"] == 0 and res["grid_same"]
    for k in GATED + ("grid_mass", "grid_momentum", "grid_force"):
        assert res["errors"][k] <= 1e-9, (k, res["errors"][k])


def wedge_case(cells):
    top = cells[2] * workloads.H
    edge = (workloads.H, 0.0, top - 0.5e-3)
    pose = dict(center=edge, angle=0.0, vel=(2.0, 0.0, 0.0), omega=0.0)
    return dict(workloads.scaled(workloads.slab_config0(), cells), vel=(0.0, 0.0, 0.0), tip=edge,
                tool=("wedge", workloads.wedge_desc_values(), pose))


@pytest.mark.parametrize("transfer", ["pic", "apic"])
@pytest.mark.parametrize("prec,tol", [("fp64", 1e-9), ("fp32", 1e-5)])
def test_tool_and_mode_change_under_shared_tiles(prec, tol, transfer):
    """The grid update after a change of the tool still reads the windows that
    the last P2G left, shared or not: a wedge, a point tool, the wedge again, and
    (the trilinear transfer) the deterministic mode on and off, against the
    oracle, with a grid rebuild on the way."""
    cells = (17, 13, 9)
    cfg = dict(wedge_case(cells), transfer=transfer)
    pts = workloads.rake_face_samples(0.0, cells[1] * workloads.H, cells[2] * workloads.H - 0.5e-3)
    o, _ = parity.build_oracle(cfg)
    s = parity.build_gpu(cfg, prec)

    def go(n):
        for _ in range(n):
            o.step(1e-8)
            s.step(1e-8)

    def wedge():
        for q, m in ((s, mpmw), (o, parity.oracle)):
            d = m.ToolDesc()
            for k, v in cfg["tool"][1].items():
                setattr(d, k, v)
            q.set_tool_analytic(d)

    go(4)
    for q in (o, s):
        q.set_tool_samples(pts, 1.5 * workloads.H)
    go(24)
    wedge()
    go(2)
    if transfer == "pic":
        s.set_deterministic(True)
        go(3)
        s.set_deterministic(False)
        go(3)
    errs, mism = parity.compare_particles(s.get_particles(), o.get_particles())
    print(f"\n[tools {prec} {transfer}] " + " ".join(f"{k}={v:.1e}" for k, v in sorted(errs.items())), flush=True)
    assert mism == 0
    for k in ("pos", "vel", "temperature"):
        assert errs[k] <= tol, (k, errs[k])


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-9), ("fp32", 1e-5)])
@pytest.mark.parametrize("move", [(0.0, 0.0, 1.6), (1.6, -1.6, 0.4)])
def test_more_leave_their_cell_than_the_queue_holds(move, prec, tol):
    """A translation by 1.6 cells between two binnings: every particle leaves its
    cell, 1024 of a workgroup's at least (tiles unshared in FP32, shared two ways
    in FP64) where the queue holds 512.  The forces of the FP32 translation as in
    the APIC windows' test."""
    cells, steps, dt = (41, 33, 9), 20, 1e-8
    cfg = dict(workloads.scaled(workloads.drill_config1(), cells), dt=dt)
    cfg["params"] = dict(cfg["params"], fixture_thickness=0.0)
    name, desc, pose = cfg["tool"]   # out of the way
    x, y, z = pose["center"]
    cfg["tool"] = (name, desc, dict(pose, center=(x, y, z + 1.0)))
    _, d = parity.build_oracle(cfg)
    d["stress"][:] = np.random.default_rng(7).uniform(-1e8, 1e8, d["stress"].shape)
    d["vel"][:] = np.array(move) * workloads.H / (steps * dt)
    errs = parity.run_from_state(cfg, prec, d, steps)["errors"]
    print(f"\n[queue {move} {prec}] " + " ".join(f"{k}={v:.1e}" for k, v in sorted(errs.items())), flush=True)
    for k in ("pos", "vel", "temperature", "grid_mass", "grid_momentum", "grid_force"):
        bound = 1e-3 if k == "grid_force" and prec == "fp32" else tol
        assert errs[k] <= bound, (k, errs[k])
