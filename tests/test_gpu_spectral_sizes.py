"""GPU: the spectral score is a kernel of its own for every FFT size with specialised kernels; sizes on
either side of its layout's lines (columns that end inside a chunk of 16, forward passes fused and
apart, the largest), against float64 and, above that, against the docked scores at grid points."""
import os

import numpy as np
import pytest

import megadock_amd as M
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def pair(golden_dir):
    return O.Protein(os.path.join(golden_dir, "1gcq_r.pdb")), O.Protein(os.path.join(golden_dir, "1gcq_l.pdb"))


def _ctx(pair, nf, t):
    rec, lig = pair
    gr, gi = O.receptor_voxel(nf // 2, 1.2, rec)
    c = M.Context(nf, nf // 2, lig.na, t=t, max_batch=2)
    c.set_receptor(gr, gi)
    c.set_ligand(lig.xyz, lig.center, lig.radius, lig.charge, O.grid_coord(nf // 2, 1.2), 1.2)
    return c, gr, gi


@pytest.mark.parametrize("nf", [64, 66, 90, 128, 162, 176, 180, 198])
def test_float64(pair, nf):
    """Beside the docked translations, where the gradient is of the score's order (far away it is a
    millionth of it, and its float error no small part of it); bounds as in the tests at 96, 100, 126."""
    lig = pair[1]
    c, gr, gi = _ctx(pair, nf, 1)
    ang = O.load_rotations(3600)[[44, 2100]]
    rot = M.rotation_coefs(ang)
    t = c.dock(rot, np.arange(2, dtype=np.int32))["index"][:, 1:] + np.float32([0.3, -0.2, 0.4])
    t = t.astype(np.float32)
    got = c.score_spectral(rot, t)
    c.close()
    remb = O.embed(nf // 2, nf, gr, gi)
    for q in range(2):
        xyz = O.rotate_ligand(lig.xyz, lig.center, O.rotation_coef(ang[q]))
        lr, li = O.ligand_voxel(nf // 2, 1.2, xyz, lig.radius, lig.charge)
        Q = O.folded_spectrum_fp64(nf, remb, O.embed(nf // 2, nf, lr, li))
        s, g = O.spectral_score_fp64(nf, Q, t[q].astype(np.float64))
        print("nf=%d pose %d" % (nf, q), flush=True)
        assert abs(got[q, 0] - s) <= 2e-6 * np.abs(np.fft.ifftn(Q)).max()
        assert np.linalg.norm(got[q, 1:] - g) <= 1e-3 * np.linalg.norm(g)


@pytest.mark.parametrize("nf", [210, 216, 242, 264, 288, 308, 320])
def test_docked_scores(pair, nf):
    c, _, _ = _ctx(pair, nf, 3)
    rot = M.rotation_coefs(O.load_rotations(3600)[[5, 3000]])
    res = c.dock(rot, np.arange(2, dtype=np.int32))
    got = c.score_spectral(np.repeat(rot, 3, axis=0), res["index"][:, 1:].astype(np.float32))
    c.close()
    print("nf=%d" % nf, flush=True)
    assert (np.abs(got[:, 0] - res["score"]) <= 1e-5 * np.maximum(np.abs(res["score"]), 1e-3)).all()
