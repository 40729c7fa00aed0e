"""GPU: a companion score whose atoms have positions that are not numbers is not a number itself, in
value and gradients (a 0 would pass for the score of a ligand outside the grid, and refinement
would take it); far and infinite positions count as outside, and other poses of the call stay
as they are."""
import os

import numpy as np
import pytest

import megadock_amd as M

pytestmark = pytest.mark.gpu

EYE = np.eye(3, dtype=np.float32).ravel()


@pytest.fixture(scope="module")
def pair(golden_dir):
    return M.Protein(os.path.join(golden_dir, "synth_r120.pdb")), M.Protein(os.path.join(golden_dir, "synth_l40.pdb"))


def _ctx(pair, xyz=None):
    rec, lig = pair
    ng = 40
    c = M.Context(2 * ng, ng, lig.na, t=1, max_batch=4)
    c.set_receptor(*M.receptor_grids(rec, ng))
    c.set_ligand(lig.xyz if xyz is None else xyz, lig.center, lig.radius, lig.charge, M.grid_coord(ng), 1.2)
    return c


@pytest.mark.parametrize("where", ["translation", "one axis", "rotation", "coordinate"])
def test_not_a_number(pair, where):
    xyz = pair[1].xyz.copy()
    rot, t = np.tile(EYE, (3, 1)), np.zeros((3, 3), np.float32)
    if where == "translation":
        t[1] = np.nan
    elif where == "one axis":
        t[1, 2] = np.nan
    elif where == "rotation":
        rot[1, 4] = np.nan
    else:
        xyz[len(xyz) // 2, 0] = np.nan
    c, plain = _ctx(pair, xyz), _ctx(pair)
    out, ref = c.score_companion(rot, t), plain.score_companion(np.tile(EYE, (3, 1)), np.zeros((3, 3), np.float32))
    c.close()
    plain.close()
    assert np.isfinite(ref).all()
    assert np.isnan(out[1]).all()
    for b in (0, 2):
        assert np.isnan(out[b]).all() if where == "coordinate" else np.array_equal(out[b], ref[b])


@pytest.mark.parametrize("t", [1000.0, -1000.0, 3.0e38, np.inf, -np.inf])
def test_outside(pair, t):
    c = _ctx(pair)
    out = c.score_companion(EYE[None], np.full((1, 3), t, np.float32))
    c.close()
    assert np.array_equal(out, np.zeros((1, 7), np.float32))
