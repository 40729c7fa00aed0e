"""GPU: receptor atoms far outside the grid, up to infinite coordinates, have empty boxes: the grids are
those of the other atoms."""
import os

import numpy as np
import pytest

import megadock_amd as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("far", [1e5, -1e5, 2.6e9, -2.6e9, 1e30, -1e30, np.inf, -np.inf])
@pytest.mark.parametrize("axis", [0, 2])
def test_far_atoms(golden_dir, far, axis):
    prot = M.Protein(os.path.join(golden_dir, "synth_l40.pdb"))
    ng = 40
    xyz = np.ascontiguousarray(prot.xyz - prot.center[None, :], np.float32)
    gone = np.zeros(prot.na, bool)
    gone[::7] = True
    moved = xyz.copy()
    moved[gone, axis] = far
    ctx = M.Context(2 * ng, ng, 8, t=1, max_batch=1)
    print("far=%g axis %d" % (far, axis), flush=True)
    ctx.set_receptor_atoms(moved, prot.radius, prot.charge, prot.ace, M.grid_coord(ng))
    got = ctx.receptor_grids()
    ctx.set_receptor_atoms(xyz[~gone], prot.radius[~gone], prot.charge[~gone], prot.ace[~gone], M.grid_coord(ng))
    want = ctx.receptor_grids()
    ctx.close()
    assert want[0].any() and want[1].any()
    for g, w in zip(got, want):
        assert np.array_equal(g.view(np.uint32), w.view(np.uint32))
