"""Tiles shared by several workgroups (GPU).

A workpiece of few tiles shares each tile among 2, 4 or 8 workgroups, alone and
in a batch.  A member's particles must stay those of the workpiece stepped
alone: up to the order of the sums that are formed with atomics, i.e. to
rounding carried through the steps (1e-9 normwise in FP64, 1e-5 in FP32, the
parity tests' tolerances), across a grid rebuild and across joining and
leaving.
"""
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
