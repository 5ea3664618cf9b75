"""An FP32 workpiece that moves keeps the order of its P2G sums (GPU).

Along the surface of a workpiece that moves through the grid, nearly empty
nodes turn the last bits of their sums into velocity and contact heat, so the
tiles of such a workpiece are not shared among workgroups, whatever its tool
and however the velocity was given.  Its sums are then those of the
deterministic mode, bit for bit, as long as no particle leaves its cell (a
displacement of 4e-11 m, away from the planes of the particles nearest to the
grid's origin; the tool stays clear, and the deterministic mode counts its
re-binnings).  A workpiece at rest is the control: its tiles are shared, and its bits differ.
"""
import numpy as np
import pytest

import parity
import workloads

pytestmark = pytest.mark.gpu
H = workloads.H
STEPS, DT, CELLS = 4, 1e-8, (17, 17, 9)


def config(tool, vel):
    cfg = workloads.scaled(workloads.drill_config1(), CELLS)
    cfg = dict(cfg, vel=vel, params=workloads.params_dict(fixture=0.0))
    if tool != "drill":
        edge = (H, 0.0, CELLS[2] * H - 0.5e-3)
        pose = dict(center=edge, angle=0.0, vel=(1.0, 0.0, 0.0), omega=0.0)
        cfg = dict(cfg, tool=("wedge", workloads.wedge_desc_values(), pose), tip=edge, name="batch")
        if tool == "voxel":
            cfg = workloads.voxel_tool_case(cfg)
    name, desc, pose, *mesh = cfg["tool"]
    x, y, z = pose["center"]
    cfg["tool"] = (name, desc, dict(pose, center=(x, y, z + 1.0)), *mesh)
    return cfg


def run(cfg, det, upload):
    s = parity.build_gpu(cfg, "fp32", det)
    d = s.get_particles()
    if upload:
        s.set_particles(d)
    s.run(STEPS, DT)
    g = s.get_particles()
    rebins = s.diagnostics()["det_rebins"]
    s.close()
    return d, g, rebins


@pytest.mark.parametrize("upload", [False, True])
@pytest.mark.parametrize("tool", ["wedge", "drill", "voxel"])
def test_sums_keep_their_order(tool, upload):
    for vel, moving in (((0.001, 0.0005, 0.001), True), ((0.0, 0.0, 0.0), False)):
        d, ref, rebins = run(config(tool, vel), True, upload)
        assert rebins == 0, "a particle left its cell: the case shows nothing"
        _, got, _ = run(config(tool, vel), False, upload)
        o, q = np.argsort(ref["id"]), np.argsort(got["id"])
        same = all(np.array_equal(got[k][q].view(np.uint8), ref[k][o].view(np.uint8))
                   for k in ("pos", "vel", "temperature", "stress"))
        assert same == moving, (tool, vel)
