"""GPU: t around the line between the two per-rotation selects (one wide histogram up to t = 512,
byte levels above): every t's list is a prefix of the longest one, bit for bit, for scores of
both signs, with some equal and with all negative."""
import os

import numpy as np
import pytest

import megadock_amd as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nf", [22, 64, 100])
@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_lists_are_prefixes_of_each_other(golden_dir, nf, sign):
    rec = M.Protein(os.path.join(golden_dir, "synth_r120.pdb"))
    lig = M.Protein(os.path.join(golden_dir, "synth_l40.pdb"))
    ng = nf // 2
    gr, gi = M.receptor_grids(rec, ng)
    ang = M.rotation_set(3600)[::1200]
    rc = M.rotation_coefs(ang)
    ids = np.arange(len(rc), dtype=np.int32)

    def run(t):
        c = M.Context(nf, ng, lig.na, t=t, max_batch=len(rc))
        c.set_receptor(sign * np.abs(gr), np.zeros_like(gi))  # the score keeps one sign, zeros are tied
        c.set_ligand(lig.xyz, lig.center, lig.radius, np.zeros_like(lig.charge), M.grid_coord(ng), 1.2)
        out = c.dock(rc, ids).reshape(len(rc), t)
        c.close()
        return out

    full = run(700)
    for t in (17, 18, 63, 511, 512, 513):
        got = run(t)
        print("nf=%d sign=%g t=%d" % (nf, sign, t), flush=True)
        assert np.array_equal(got.view(np.uint8), np.ascontiguousarray(full[:, :t]).view(np.uint8)), t
