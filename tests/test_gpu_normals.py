"""Normals of the next-to-wall nodes at triangle counts around the kernel's chunk of 64 (8 a thread) and node
counts around its blocks of 16 and 64 nodes, against the oracle's sum over every triangle in file order."""
import numpy as np
import pytest

from pv_dec_original_amd import Simulation, SubDomain
from pv_dec_original_amd.workloads import fluid_box_case, xfaces
from tests import oracle_ctypes as O

pytestmark = pytest.mark.gpu


# a box of fluid of this size in a grid two wider: few nodes (blocks of 16, full and not) and past
# 65536 next-to-wall nodes (blocks of 64)
@pytest.mark.parametrize("box,ntri", [((3, 3, 3), 1), ((5, 4, 3), 7), ((9, 6, 5), 63), ((9, 6, 5), 64),
                                      ((17, 16, 15), 65), ((17, 16, 15), 200), ((112, 109, 107), 9),
                                      ((112, 109, 107), 129)])
def test_normals_against_file_order_sums(box, ntri):
    nx, ny, nz = box
    case = fluid_box_case(q=19, box=(nx + 2, ny + 2, nz + 2), tau=0.8)
    fluid = np.zeros((nz + 2, ny + 2, nx + 2), dtype=np.uint8)
    fluid[1:-1, 1:-1, 1:-1] = 1
    case.geometry.fluid = fluid
    rng = np.random.default_rng(ntri)
    tri = rng.uniform(-3.0, max(box) + 3.0, (ntri, 12))
    tri[ntri // 2, 3:9] = np.tile(tri[ntri // 2, :3], 2)  # two vertices on the first: no area
    case.geometry.globalTriangles = tri
    sd = SubDomain(case.geometry, xfaces(case.geometry), storage="fp64", tau=case.tau)
    nrm = sd.normals()
    xyz = Simulation(sd, case.tau).wss()[:, :3]
    assert len(xyz) == nrm.shape[1] > 0 and (len(xyz) >= 65536) == (min(box) > 100)
    # bit for bit: the same sums in the same order, division and square root correctly rounded
    assert np.array_equal(nrm, O.normal_at(tri, xyz), equal_nan=True)
