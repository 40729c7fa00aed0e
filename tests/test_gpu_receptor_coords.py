"""GPU: receptor grids whose coordinates are the voxel centres only nearly or not at all (shifted,
stretched, moved one by one), where the surface's boxes may not be cut to an atom's reach, bit-exact
with the oracle's restatement of the reference; also atoms that reach over the box and beyond the grid."""
import ctypes as C
import os

import numpy as np
import pytest

import megadock_amd as M
from oracle import oracle as O

pytestmark = pytest.mark.gpu

NG = 44


def _coords(kind):
    rng = np.random.default_rng(1)
    gc = M.grid_coord(NG).astype(np.float64)
    if kind == "nearly":
        gc += rng.uniform(-0.29, 0.29, NG)  # within a quarter of the pitch of 1.2
    elif kind == "one":
        gc[NG // 2] += 0.31
    elif kind == "shifted":
        gc += 0.7
    elif kind == "far":
        gc += 5.0
    elif kind == "stretched":
        gc *= 1.1
    elif kind == "jittered":
        gc += rng.uniform(-0.6, 0.6, NG)
    return gc.astype(np.float32)


@pytest.mark.parametrize("radius", [0.0, 4.0])
@pytest.mark.parametrize("kind", ["centres", "nearly", "one", "shifted", "far", "stretched", "jittered"])
def test_coordinates(golden_dir, kind, radius):
    prot = M.Protein(os.path.join(golden_dir, "1gcq_l.pdb"))
    xyz = np.ascontiguousarray(prot.xyz - prot.center[None, :], np.float32)
    rad = (prot.radius + np.float32(radius)).astype(np.float32)
    gc = _coords(kind)
    ctx = M.Context(2 * NG, NG, 8, t=1, max_batch=1)
    ctx.set_receptor_atoms(xyz, rad, prot.charge, prot.ace, gc)
    dr, di = ctx.receptor_grids()
    ctx.close()
    gr, gi = np.zeros(NG ** 3, np.float32), np.zeros(NG ** 3, np.float32)
    O.lib().or_receptor_voxel(C.c_int(NG), C.c_float(1.2), C.c_int(prot.na), O._fp(xyz), O._fp(rad), O._fp(prot.charge),
                              O._fp(prot.ace), O._fp(gc), C.c_float(1.0), C.c_float(-45.0), C.c_float(1.0), O._fp(gr), O._fp(gi))
    print("%s, radius + %g: core %d, surface %d" % (kind, radius, (gr == -45).sum(), (gr > 0).sum()), flush=True)
    assert (gr > 0).any() and gi.any()
    assert np.array_equal(gr.view(np.uint32), dr.view(np.uint32))
    assert np.array_equal(gi.view(np.uint32), di.view(np.uint32))
