"""A member of a batch has the sums it has alone (GPU, the atomic mode).

How many workgroups share a tile groups the sums of the P2G, so it may depend
on the workpiece but not on what else is in the launch.  While every particle
stays in its cell nothing is added with atomics either, and the state of a
member must then be that of the same workpiece stepped alone, bit for bit:
workpieces on each side of the sharing steps (27 to 280 tiles) beside one
whose tiles alone fill the chip, with a grid rebuild on the way.
"""
import numpy as np
import pytest

import mpmw
import parity
import workloads

pytestmark = pytest.mark.gpu
STEPS, DT = 30, 1e-8


def solver(cells, prec, transfer, graph):
    s = parity.build_gpu(dict(workloads.scaled(workloads.drill_config1(), cells), transfer=transfer), prec)
    s.set_graph(graph)
    return s


@pytest.mark.parametrize("transfer,prec", [("pic", "fp32"), ("pic", "fp64"), ("apic", "fp32")])
@pytest.mark.parametrize("graph", [0, 1])
def test_member_equals_alone(transfer, prec, graph):
    sizes = [(17, 17, 9), (32, 32, 16), (48, 40, 20), (64, 56, 20), (96, 80, 32)]
    alone = []
    for c in sizes[:-1]:
        s = solver(c, prec, transfer, graph)
        s.run(STEPS, DT)
        alone.append(s.get_particles())
        s.close()
    members = [solver(c, prec, transfer, 0) for c in sizes]
    b = mpmw.Batch()
    for s in members:
        b.add(s)
    b.set_graph(graph)
    for _ in range(STEPS):
        b.step(DT)
    for c, s, a in zip(sizes, members, alone):
        g = s.get_particles()
        for k, v in a.items():
            if v is not None:
                assert np.array_equal(np.asarray(g[k]).view(np.uint8), np.asarray(v).view(np.uint8)), (c, k)
    b.close()
    for s in members:
        s.close()
