"""GPU: Context.dock takes few results straight to host memory and copies more; both sides of that line,
one and several results per rotation, and grids whose voxelizer reads the rotations once or often,
give what the resident rotation loop gives, in the caller's rotation numbers."""
import os

import numpy as np
import pytest

import megadock_amd as M
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ng,t,counts", [(32, 1, (1, 255, 256, 257)), (32, 3, (85, 86)), (32, 16, (16, 17)),
                                         (80, 2, (1, 130)), (32, 40, (2, 7))])
def test_both_ways(golden_dir, ng, t, counts):
    rec = O.Protein(os.path.join(golden_dir, "1gcq_r.pdb"))
    lig = O.Protein(os.path.join(golden_dir, "1gcq_l.pdb"))
    n = max(counts)
    ctx = M.Context(2 * ng, ng, lig.na, t=t, max_batch=n)
    ctx.set_receptor(*O.receptor_voxel(ng, 1.2, rec))
    ctx.set_ligand(lig.xyz, lig.center, lig.radius, lig.charge, O.grid_coord(ng, 1.2), 1.2)
    rot = M.rotation_coefs(O.load_rotations(360)[:n])
    ctx.set_rotations(rot)
    ctx.dock_range(0, n)
    want = ctx.results(0, n).reshape(n, t)
    for B in counts:
        print("ng=%d t=%d B=%d" % (ng, t, B), flush=True)
        ids = 1000 + np.arange(B, dtype=np.int32)
        got = ctx.dock(rot[:B], ids).reshape(B, t)
        ref = want[:B].copy()
        ref["index"][:, :, 0] += 1000
        assert got.tobytes() == ref.tobytes()
    ctx.close()
