"""GPU: the companion score where atoms leave the receptor grid or have no position, and for pose
counts around its launch sizes.  A pose far outside scores 0 with zero gradients; poses scored
together equal poses scored one by one."""
import os

import numpy as np
import pytest

import megadock_amd as M

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx(golden_dir):
    rec = M.Protein(os.path.join(golden_dir, "synth_r120.pdb"))
    lig = M.Protein(os.path.join(golden_dir, "synth_l40.pdb"))
    ng = 40
    c = M.Context(2 * ng, ng, lig.na, t=1, max_batch=4)
    c.set_receptor(*M.receptor_grids(rec, ng))
    c.set_ligand(lig.xyz, lig.center, lig.radius, lig.charge, M.grid_coord(ng), 1.2)
    yield c
    c.close()


@pytest.mark.parametrize("t", [1000.0, -3.0e8, np.inf, np.nan])
def test_far_poses_score_zero(ctx, t):
    out = ctx.score_companion(np.eye(3, dtype=np.float32).ravel()[None], np.full((1, 3), t, np.float32))
    assert np.array_equal(out, np.zeros((1, 7), np.float32))


@pytest.mark.parametrize("n", [1, 3, 5, 257])
def test_pose_counts(ctx, n):
    rng = np.random.default_rng(n)
    q = rng.normal(size=(n, 3, 3))
    rot = np.linalg.qr(q)[0].reshape(n, 9).astype(np.float32)
    t = rng.uniform(-30, 30, (n, 3)).astype(np.float32)
    out = ctx.score_companion(rot, t)
    one = np.concatenate([ctx.score_companion(rot[b:b + 1], t[b:b + 1]) for b in range(n)])
    assert np.array_equal(out, one) and np.isfinite(out).all()
    assert ctx.score_companion(rot[:0], t[:0]).shape == (0, 7)
