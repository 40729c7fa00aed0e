"""GPU: the generic passes choose their workgroup by the size; in each choice (256 threads up to about 146,
512 up to about 290, 1024 above) score maps follow the float64 correlation, and the best results,
one or several per rotation, are the map's."""
import os

import numpy as np
import pytest

import megadock_amd as M
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nf", [22, 130, 156, 208, 260, 324])
def test_sizes(golden_dir, nf):
    rec = O.Protein(os.path.join(golden_dir, "1gcq_r.pdb"))
    lig = O.Protein(os.path.join(golden_dir, "1gcq_l.pdb"))
    ng = nf // 2
    gr, gi = O.receptor_voxel(ng, 1.2, rec)
    angle = O.load_rotations(360)[77]
    rot = M.rotation_coefs(angle[None])
    lr, li = O.ligand_voxel(ng, 1.2, O.rotate_ligand(lig.xyz, lig.center, O.rotation_coef(angle)), lig.radius, lig.charge)
    ref = O.correlation_fp64(nf, O.embed(ng, nf, gr, gi), O.embed(ng, nf, lr, li)).ravel()
    for t in (1, 3):
        print("nf=%d t=%d" % (nf, t), flush=True)
        ctx = M.Context(nf, ng, lig.na, t=t, max_batch=1)
        ctx.set_receptor(gr, gi)
        ctx.set_ligand(lig.xyz, lig.center, lig.radius, lig.charge, O.grid_coord(ng, 1.2), 1.2)
        smap = ctx.score_map(rot[0])
        assert np.abs(smap.astype(np.float64) - ref).max() < 2e-6 * np.abs(ref).max()
        got = ctx.dock(rot, np.zeros(1, np.int32))
        # equal scores: the lowest index first; t > 1 orders by the score over nf^3
        key = smap if t == 1 else smap / np.float32(nf ** 3)
        best = np.lexsort((np.arange(key.size), -key.astype(np.float64)))[:t]
        idx = got["index"].astype(np.int64)
        assert ((idx[:, 1] * nf + idx[:, 2]) * nf + idx[:, 3]).tolist() == best.tolist()
        ctx.close()
