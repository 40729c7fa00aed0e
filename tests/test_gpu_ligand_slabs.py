"""GPU: the ligand voxelizer of grids above one workgroup's LDS works on slabs of planes, bit-exact with
the oracle: slabs that end inside the grid and at its end, more atoms than one list of 4096 takes,
atoms outside the grid, and the core rule that reaches two planes over a slab's edge."""
import numpy as np
import pytest

import megadock_amd as M
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("na,ng,extent,delta", [(5000, 80, 50.0, 2.0), (4097, 110, 70.0, 2.0), (4096, 98, 20.0, 1.0),
                                                (300, 162, 100.0, -3.5)])
def test_slabs(na, ng, extent, delta):
    rng = np.random.default_rng(na + ng)
    xyz = rng.uniform(-extent, extent, (na, 3)).astype(np.float32)
    xyz[: na // 8] = xyz[na // 8: 2 * (na // 8)]  # voxels with several atoms
    radius = rng.choice([0.0, 1.2, 1.63, 1.87, 2.1, 6.0], na).astype(np.float32)
    charge = rng.choice([0.0, 0.1, -0.15, 0.33, -0.57, 1e-3], na).astype(np.float32)
    center = np.array([0.3, -0.2, 0.1], np.float32)
    ctx = M.Context(2 * ng, ng, na, t=1, max_batch=2)
    ctx.set_ligand(xyz, center, radius, charge, O.grid_coord(ng, 1.2), 1.2, delta)
    ang = O.load_rotations(360)[[3, 201]]
    for _ in range(2):  # the charge grid and the counts are handed back empty
        gr, gi = ctx.voxelize(M.rotation_coefs(ang))
        for q in range(2):
            rot = O.rotate_ligand(xyz, center, O.rotation_coef(ang[q]))
            er, ei = O.ligand_voxel(ng, 1.2, rot, radius, charge, delta)
            print("na=%d ng=%d rotation %d" % (na, ng, q), flush=True)
            assert np.array_equal(gr[q], er)
            assert np.array_equal(gi[q], ei)
    ctx.close()
