"""GPU: the ligand voxelizer of grids above one workgroup's LDS sets the bits of up to four rotations in
memory and those of more in slabs of planes; both sides of that line, bit-exact with the oracle, and one
rotation of a large ligand takes little more time than one of a small ligand."""
import time

import numpy as np
import pytest

import megadock_amd as M
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("na,ng,extent,delta", [(1, 77, 1.0, 1.0), (25, 90, 60.0, 2.0), (4097, 110, 70.0, 2.0),
                                                (5000, 80, 50.0, 1.0), (300, 162, 100.0, -3.5)])
def test_four_rotations_and_five(na, ng, extent, delta):
    rng = np.random.default_rng(na + ng)
    xyz = rng.uniform(-extent, extent, (na, 3)).astype(np.float32)
    xyz[: na // 8] = xyz[na // 8: 2 * (na // 8)]  # voxels with several atoms
    radius = rng.choice([0.0, 1.2, 1.63, 1.87, 2.1, 6.0], na).astype(np.float32)
    charge = rng.choice([0.0, 0.1, -0.15, 0.33, -0.57, 1e-3], na).astype(np.float32)
    center = np.array([0.3, -0.2, 0.1], np.float32)
    ctx = M.Context(2 * ng, ng, na, t=1, max_batch=5)
    ctx.set_ligand(xyz, center, radius, charge, O.grid_coord(ng, 1.2), 1.2, delta)
    ang = O.load_rotations(360)[[3, 50, 120, 201, 333]]
    want = []
    for a in ang:
        rot = O.rotate_ligand(xyz, center, O.rotation_coef(a))
        want.append(O.ligand_voxel(ng, 1.2, rot, radius, charge, delta))
    for n in (4, 5, 1, 5, 4):  # each form behind the other
        print("na=%d ng=%d rotations=%d" % (na, ng, n), flush=True)
        gr, gi = ctx.voxelize(M.rotation_coefs(ang[:n]))
        for q in range(n):
            assert np.array_equal(gr[q], want[q][0])
            assert np.array_equal(gi[q], want[q][1])
    ctx.close()


def test_time_of_one_rotation():
    """One rotation at 160^3, 30000 atoms a voxel or more apart against 300: three times the time in slabs,
    of which one rotation has ten."""
    ng = 80
    at = (np.stack(np.meshgrid(*[np.arange(32)] * 3, indexing="ij"), -1).reshape(-1, 3) - 15.5) * 2.0
    took = []
    for na in (300, 30000):
        ctx = M.Context(2 * ng, ng, na, t=1, max_batch=1)
        z = np.zeros(ng ** 3, np.float32)
        ctx.set_receptor(z, z)
        ctx.set_ligand(at[:na].astype(np.float32), np.zeros(3, np.float32), np.full(na, 1.6, np.float32),
                       np.full(na, 0.1, np.float32), M.grid_coord(ng), 1.2)
        rot, ids = np.eye(3, dtype=np.float32).reshape(1, 9), np.zeros(1, np.int32)
        best = np.inf
        for _ in range(30):
            t0 = time.perf_counter()
            ctx.dock(rot, ids)
            best = min(best, time.perf_counter() - t0)
        ctx.close()
        took.append(best)
    print("300 atoms %.0f us, 30000 atoms %.0f us" % (took[0] * 1e6, took[1] * 1e6), flush=True)
    assert took[1] < 2.2 * took[0]
