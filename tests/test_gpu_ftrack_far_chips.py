"""F-tracking step of a small block whose box two far chips stretch (GPU).

Nearly all tiles of such a box are empty, and every tile takes its windows and
workgroups whether it holds particles or not: its tiles are not shared, and
past some 80 thousand of them one workgroup does both jobs of the P2G.  The
device memory stays that of one window set a tile, and the results are the
oracle's, with the parity tests' tolerances (normwise 1e-9 in FP64; 1e-5 in
FP32 on the gated fields).
"""
import ctypes as C

import numpy as np
import pytest

import ftrack
import mpms
import mpmw
from test_gpu_ftrack import GATED, compare, grid_errors, oracle_view
from test_gpu_ftrack_shared import block

pytestmark = pytest.mark.gpu
NODES = 10 * 10 * 6   # nodes of a tile's window


def free_bytes():
    free, total = C.c_size_t(), C.c_size_t()
    assert mpmw.lib().hipMemGetInfo(C.byref(free), C.byref(total)) == 0   # the library's own runtime
    return free.value


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("far", [0.04, 0.12])
def test_far_chips(far, prec):
    kw, a, pos = block((12, 10, 8), 0.2, 3, domain_max=(far, far, far))
    for k, at in ((0, -0.0185), (1, far - 0.0015)):
        a["x"][k] = a["y"][k] = a["z"][k] = at
        a["vx"][k] = a["vy"][k] = a["vz"][k] = 1.0
        a["status"][k] = mpms.ACTIVE
    o = mpms.Oracle(mpms.default_params(**kw))
    o.set_particles(a)
    P = ftrack.default_params(**kw, precision=ftrack.FP64 if prec == "fp64" else ftrack.FP32)
    s = ftrack.Solver(P)   # loads what a first solver of the process loads
    s.init_box((0, 0, 0), (1e-3, 1e-3, 1e-3), 2.5e-4)
    s.step(1e-8)
    s.close()
    free = free_bytes()
    s = ftrack.Solver(P)
    s.set_particles(oracle_view(a))
    for q in (o, s):
        q.set_tool_position(*pos.mean(0))
        for _ in range(2):
            q.step(1e-8)
    errs, mism = compare(s.get_particles(), oracle_view(o.get_particles()))
    errs.update(grid_errors(s, o))
    used = free - free_bytes()
    n = np.array(s.diagnostics()["box_n"])
    nt, r = int(np.prod(-(-n // [8, 8, 4]))), 8 if prec == "fp64" else 4
    # one window set a tile and the node block, a quarter over; the rest is small
    bound = 1.25 * (nt * NODES * 8 * r + int(np.prod(n)) * (10 * r + 4)) + (256 << 20)
    print(f"\n[{far} {prec}] {nt} tiles, {used / 1e6:.0f} MB of {bound / 1e6:.0f} "
          + " ".join(f"{k}={v:.1e}" for k, v in sorted(errs.items())), flush=True)
    assert (nt > 80100) == (far > 0.1) and used <= bound
    assert mism == 0
    for k in (errs if prec == "fp64" else GATED):
        assert errs[k] <= (1e-9 if prec == "fp64" else 1e-5), (k, errs[k])
    s.close()
