"""GPU: the ligand voxelizer at the edges of its forms, bit-exact with the oracle: one atom, an atom's
planes in five threads and in one (512 and 513 atoms), more atoms than the charges' table takes,
boxes that end at a word or at the grid, atoms outside the grid, voxels with one, two and many atoms,
and grids in one workgroup's LDS and above."""
import numpy as np
import pytest

import megadock_amd as M
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("na,ng,extent,delta", [(1, 9, 1.0, 1.0), (512, 33, 12.0, 1.0), (513, 33, 12.0, 2.0),
                                                (640, 24, 3.0, 1.0), (1300, 63, 40.0, 1.0), (5120, 72, 30.0, 1.0),
                                                (5121, 72, 30.0, 2.0), (2561, 63, 4.0, 1.0), (9000, 32, 25.0, 1.0),
                                                (3000, 75, 45.0, 1.0), (700, 3, 5.0, 1.0)])
def test_ligand_grids(na, ng, extent, delta):
    rng = np.random.default_rng(na + ng)
    xyz = rng.uniform(-extent, extent, (na, 3)).astype(np.float32)
    xyz[na // 3: na // 2] = xyz[: na // 2 - na // 3]  # voxels with several atoms
    radius = rng.choice([0.0, 1.2, 1.63, 1.87, 2.1], na).astype(np.float32)
    charge = rng.choice([0.0, 0.1, -0.15, 0.33, -0.57, 1e-3], na).astype(np.float32)
    center = np.array([0.3, -0.2, 0.1], np.float32)
    ctx = M.Context(2 * ng, ng, na, t=1, max_batch=3)
    ctx.set_ligand(xyz, center, radius, charge, O.grid_coord(ng, 1.2), 1.2, delta)
    ang = O.load_rotations(360)[[0, 101, 355]]
    for _ in range(2):  # the charge grid is handed back empty
        gr, gi = ctx.voxelize(M.rotation_coefs(ang))
        for q in range(3):
            rot = O.rotate_ligand(xyz, center, O.rotation_coef(ang[q]))
            er, ei = O.ligand_voxel(ng, 1.2, rot, radius, charge, delta)
            print("na=%d ng=%d rotation %d" % (na, ng, q), flush=True)
            assert np.array_equal(gr[q], er)
            assert np.array_equal(gi[q], ei)
    ctx.close()
