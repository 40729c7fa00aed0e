"""GPU: the off-grid scores' buffers are there from a context's creation on for as many poses as its
batch, larger calls grow them and go through blocks of 65536 poses; results do not depend on what
was called before or on the block that a pose falls in."""
import os

import numpy as np
import pytest

import megadock_amd as M

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _poses(n, span):
    rng = np.random.default_rng(n)
    rot = M.rotation_coefs(rng.uniform(0, 3, (n, 3)).astype(np.float32))
    return rot, rng.uniform(0, span, (n, 3)).astype(np.float32)


def _ctx(golden_dir, nf, batch):
    lig = M.Protein(os.path.join(golden_dir, "synth_l40.pdb"))
    rng = np.random.default_rng(nf)
    c = M.Context(nf, nf // 2, lig.na, t=1, max_batch=batch)
    c.set_receptor(rng.normal(size=(nf // 2) ** 3), rng.normal(size=(nf // 2) ** 3))
    c.set_ligand(lig.xyz, lig.center, lig.radius, lig.charge, M.grid_coord(nf // 2), 1.2)
    return c


def test_first_call_allocates_nothing(golden_dir):
    """60000 poses of 19 words are 4.6 MB, more than any pool of small allocations gives.  (The runtime
    takes memory of its own when a process first calls the kernels: another context does.)"""
    n = 60000
    rot, t = _poses(n, 8)
    c = _ctx(golden_dir, 8, n)
    c.score_companion(rot, t)
    c.close()
    c = _ctx(golden_dir, 8, n)
    c.sync()
    before = torch.cuda.mem_get_info()[0]
    first = c.score_companion(rot, t)
    assert torch.cuda.mem_get_info()[0] == before
    assert np.array_equal(c.score_companion(rot, t), first)
    c.close()


@pytest.mark.parametrize("score", ["companion", "spectral"])
def test_rising_counts_and_blocks(golden_dir, score):
    """One pose more than a block, and a short call in a layout of its own."""
    nf, n = 64, 65536 + 3
    c = _ctx(golden_dir, nf, 200)
    f = getattr(c, "score_" + score)
    rot, t = _poses(n, nf)
    rot[1000:], t[1000:] = rot[np.arange(1000, n) % 1000], t[np.arange(1000, n) % 1000]  # the first 1000 again
    counts = (1, 2, 3, 199, 200, 201, 333, 1000, 7)
    want = f(rot[:1000], t[:1000])
    for k in counts:
        print("%s: %d poses" % (score, k), flush=True)
        assert np.array_equal(f(rot[:k], t[:k]), want[:k])
    print("%s: %d poses" % (score, n), flush=True)
    assert np.array_equal(f(rot, t), want[np.arange(n) % 1000])
    assert np.array_equal(f(rot[:5], t[:5]), want[:5])
    c.close()
