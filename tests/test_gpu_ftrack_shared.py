"""F-tracking passes whose tiles are shared by several workgroups (GPU).

A block of few tiles shares each among 2, 4 or 8 workgroups (by the particle
count and the precision), and the step skips the external force and backstress
arrays while they hold zeros.  Sizes on both sides of the sharing steps, a
workgroup's share empty (a handful of particles), forces applied between
steps, backstress loaded or not; against the FP64 oracle, with the parity
tests' tolerances (normwise 1e-9 in FP64; 1e-5 in FP32 on the gated fields).
"""
import numpy as np
import pytest

import ftrack
import mpms
import parity
from test_gpu_ftrack import FIELDS, GATED, compare, grid_errors, oracle_view

pytestmark = pytest.mark.gpu


def block(dims, jitter, seed, **kw):
    kw = dict(dict(jc_A=250e6, jc_B=300e6, jc_n=0.4, jc_C=0.015, jc_m=1.0, lod_active_radius=0.002,
                   lod_near_radius=0.006, fixture_thickness=0.0, domain_min=(-0.02, -0.02, -0.02),
                   domain_max=(0.04, 0.04, 0.04)), **kw)
    sp = 2.5e-4
    rng = np.random.default_rng(seed)
    z, y, x = np.meshgrid(*(np.arange(d) for d in dims[::-1]), indexing="ij")
    pos = np.stack([x, y, z], -1).reshape(-1, 3) * sp + rng.uniform(-jitter, jitter, (x.size, 3)) * sp + 0.07 * sp
    a = mpms.new_particles(len(pos))
    a["x"], a["y"], a["z"] = pos.T
    a["mass"], a["volume"], a["temperature"] = 4430.0 * sp ** 3, sp ** 3, 300.0
    a["vx"], a["vy"], a["vz"] = rng.uniform(-3, 3, (3, len(pos)))
    a["id"] = np.arange(len(pos))
    a["status"] = np.where(pos[:, 2] < 0.1 * dims[2] * sp, mpms.FIXED, mpms.ACTIVE)
    return kw, a, pos


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("dims", [(2, 1, 1), (7, 5, 3), (63, 64, 32), (64, 64, 32), (97, 96, 30)])
def test_shared_tiles_match_oracle(dims, prec):
    kw, a, pos = block(dims, 0.2, dims[0])
    o = mpms.Oracle(mpms.default_params(**kw))
    o.set_particles(a)
    s = ftrack.Solver(ftrack.default_params(**kw, precision=ftrack.FP64 if prec == "fp64" else ftrack.FP32))
    s.set_particles(oracle_view(a))
    c = pos.mean(0) + [0, 0, 0.3 * dims[2] * 2.5e-4]
    for q in (o, s):
        q.set_tool_position(*c)
        q.set_tool_nodes(c[None] + [[0, 0, 0], [5e-4, 0, 0]], np.tile([0.0, 0.0, -20.0], (2, 1)))
    for _ in range(3):
        o.step(1e-8)
        s.step(1e-8)
    errs, mism = compare(s.get_particles(), oracle_view(o.get_particles()))
    errs.update(grid_errors(s, o))
    print(f"\n[{dims} {prec}] " + " ".join(f"{k}={v:.1e}" for k, v in sorted(errs.items())), flush=True)
    assert mism == 0
    for k in (errs if prec == "fp64" else GATED):
        assert errs[k] <= (1e-9 if prec == "fp64" else 1e-5), (k, errs[k])
    s.close()


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("back", [False, True])
def test_forces_come_and_go(back, graph):
    """Steps without any external force, with one pending from the start, and
    with forces applied between steps."""
    kw, a, pos = block((12, 10, 8), 0.2, 5)
    if back:
        a["a"] = np.random.default_rng(1).uniform(-2e7, 2e7, a["a"].shape)
    for pending in (False, True):
        if pending:
            a["efx"] = 0.01
        o = mpms.Oracle(mpms.default_params(**kw))
        o.set_particles(a)
        s = ftrack.Solver(ftrack.default_params(**kw, precision=ftrack.FP64))
        s.set_graph(graph)
        s.set_particles(oracle_view(a))
        for q in (o, s):
            q.set_tool_position(*pos.mean(0))
        for k in range(7):
            if k in (2, 3, 5):
                for q in (o, s):
                    q.apply_external_force(pos.mean(0), 1e-3, np.array([0.0, 0.02, -0.05]))
            o.step(1e-8)
            s.step(1e-8)
        g = s.get_particles()
        errs, mism = compare(g, oracle_view(o.get_particles()))
        assert mism == 0 and not g["fext"].any()
        for k in FIELDS:
            assert errs[k] <= 1e-9, (pending, k, errs[k])
        s.close()
