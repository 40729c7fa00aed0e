"""GPU: the device receptor producer works on rows of 32-voxel words; rows that end inside a
word, at its edge, and every count of words that a sweep kernel is built for, are bit-exact with
the host producer, as are a core value of 0 and a receptor without atoms."""
import os

import numpy as np
import pytest

import megadock_amd as M

pytestmark = pytest.mark.gpu


def _device(xyz, radius, charge, ace, ng, rec_core=-45.0):
    ctx = M.Context(2 * ng, ng, 8, t=1, max_batch=1)
    ctx.set_receptor_atoms(xyz, radius, charge, ace, M.grid_coord(ng), rec_core=rec_core)
    out = ctx.receptor_grids()
    ctx.close()
    return out


@pytest.mark.parametrize("ng,core", [(9, -45.0), (32, -45.0), (33, -45.0), (36, 0.0), (65, -45.0), (98, -45.0),
                                     (130, -45.0), (162, -45.0), (200, -45.0)])
def test_rows_of_words(golden_dir, ng, core):
    prot = M.Protein(os.path.join(golden_dir, "synth_r120.pdb"))
    gr, gi = M.receptor_grids(prot, ng, rec_core=core)
    xyz = (prot.xyz - prot.center[None, :]).astype(np.float32)
    dr, di = _device(xyz, prot.radius, prot.charge, prot.ace, ng, core)
    print("ng=%d core=%g" % (ng, core), flush=True)
    assert np.array_equal(gr.view(np.uint32), dr.view(np.uint32))
    assert np.array_equal(gi.view(np.uint32), di.view(np.uint32))


def test_no_atoms():
    z = np.zeros(0, np.float32)
    dr, di = _device(z, z, z, z, 24)
    assert not dr.any() and not di.any()
