"""GPU: 16 < t <= 512 results per rotation where more scores reach the t-th best than one list of the
select takes (maps of one value, of two values, and beside them maps without ties in the same
batch): the results are the score map's own best ones, equal scores by the lower index, and
such maps take the whole GPU as others do."""
import os
import time

import numpy as np
import pytest

import megadock_amd as M

pytestmark = pytest.mark.gpu


def _best(smap, nf, t):
    key = smap / np.float32(nf ** 3) + np.float32(0)
    return key, np.lexsort((np.arange(key.size), -key.astype(np.float64)))[:t]


def _check(got, smap, nf, t):
    key, best = _best(smap, nf, t)
    idx = got["index"].astype(np.int64)
    assert ((idx[:, 1] * nf + idx[:, 2]) * nf + idx[:, 3]).tolist() == best.tolist()
    assert np.array_equal(got["score"], key[best])


def _ctx(lig, nf, t, batch, xyz=None, center=None):
    c = M.Context(nf, nf // 2, lig.na, t=t, max_batch=batch)
    c.set_ligand(lig.xyz if xyz is None else xyz, lig.center if center is None else center, lig.radius, lig.charge,
                 M.grid_coord(nf // 2), 1.2)
    return c


@pytest.fixture(scope="module")
def lig(golden_dir):
    return M.Protein(os.path.join(golden_dir, "synth_l40.pdb"))


@pytest.mark.parametrize("nf,t", [(22, 17), (22, 512), (64, 17), (64, 512), (100, 64), (144, 300), (200, 64)])
@pytest.mark.parametrize("values", [0, 1, 2])
def test_few_values(lig, nf, t, values):
    re, im = np.zeros((nf, nf, nf), np.float32), np.zeros((nf, nf, nf), np.float32)
    if values:
        re[0, 0, 0] = 3.0
    if values > 1:
        re[0, nf // 2, 0] = re[nf // 2, nf // 2, nf // 2] = 1.0  # two or more values along y
    c = _ctx(lig, nf, t, 3)
    c.set_receptor_spectrum(re, im)
    rot = M.rotation_coefs(M.rotation_set(24)[[0, 7, 20]])
    got = c.dock(rot, np.arange(3, dtype=np.int32)).reshape(3, t)
    for b in range(3):
        print("nf=%d t=%d values=%d rotation %d" % (nf, t, values, b), flush=True)
        _check(got[b], c.score_map(rot[b]), nf, t)
    c.close()


@pytest.mark.parametrize("nf,t", [(22, 17), (64, 33), (64, 512), (112, 64), (144, 512)])
@pytest.mark.parametrize("kind", ["close", "along_z", "along_x"])
def test_one_wide_bucket(lig, nf, t, kind):
    """Scores that differ but lie within 6% of each other, and equal ones that lie apart in the map."""
    rng = np.random.default_rng(nf + t)
    re, im = np.zeros((nf, nf, nf), np.float32), np.zeros((nf, nf, nf), np.float32)
    if kind == "close":
        re[0, 0, 0] = 1e5
        re[:3, :3, 1:4], im[:3, :3, 1:4] = rng.normal(size=(2, 3, 3, 3)).astype(np.float32)
    else:
        re[(0, 0, nf // 2) if kind == "along_z" else (nf // 2, 0, 0)] = 1.0
    c = _ctx(lig, nf, t, 2)
    c.set_receptor_spectrum(re, im)
    rot = M.rotation_coefs(M.rotation_set(24)[[3, 11]])
    got = c.dock(rot, np.arange(2, dtype=np.int32)).reshape(2, t)
    for b in range(2):
        print("nf=%d t=%d %s rotation %d" % (nf, t, kind, b), flush=True)
        _check(got[b], c.score_map(rot[b]), nf, t)
    c.close()


def test_beside_other_maps(golden_dir, lig):
    """A ligand off its centre: rotations that carry it out of the grid give maps of zeros."""
    nf, t = 64, 40
    rec = M.Protein(os.path.join(golden_dir, "synth_r120.pdb"))
    gr, _ = M.receptor_grids(rec, nf // 2)
    xyz = lig.xyz - lig.center + np.float32([36.0, 0.0, 0.0])
    c = M.Context(nf, nf // 2, lig.na, t=t, max_batch=16)
    c.set_receptor(gr, np.zeros_like(gr))
    c.set_ligand(xyz, np.zeros(3, np.float32), lig.radius, np.zeros_like(lig.charge), M.grid_coord(nf // 2), 1.2)
    rot = M.rotation_coefs(M.rotation_set(360)[::24][:15])
    rot[::4] = np.eye(3, dtype=np.float32).ravel()
    got = c.dock(rot, np.arange(15, dtype=np.int32)).reshape(15, t)
    tied = 0
    for b in range(15):
        smap = c.score_map(rot[b])
        tied += not smap.any()
        _check(got[b], smap, nf, t)
    c.close()
    assert 0 < tied < 15


def test_batches_one_after_another(golden_dir, lig):
    """A context docks tied maps, others and tied ones again, as many rotations or fewer each time."""
    nf, t = 64, 40
    rec = M.Protein(os.path.join(golden_dir, "synth_r120.pdb"))
    grids, zero = M.receptor_grids(rec, nf // 2), (np.zeros((nf // 2) ** 3, np.float32),) * 2
    rot = M.rotation_coefs(M.rotation_set(24)[:6])
    c, want = _ctx(lig, nf, t, 6), {}
    for tied in (False, True):
        fresh = _ctx(lig, nf, t, 6)
        fresh.set_receptor(*(zero if tied else grids))
        want[tied] = fresh.dock(rot, np.arange(6, dtype=np.int32)).reshape(6, t)
        fresh.close()
    for tied, n in ((True, 6), (False, 6), (True, 2), (False, 4), (False, 6), (True, 6), (False, 1), (False, 6)):
        print("tied=%d rotations=%d" % (tied, n), flush=True)
        c.set_receptor(*(zero if tied else grids))
        got = c.dock(rot[:n], np.arange(n, dtype=np.int32)).reshape(n, t)
        assert np.array_equal(got, want[tied][:n])
    c.close()


def test_more_tied_maps_than_workgroups(lig):
    nf, t, n = 22, 20, 700
    c = _ctx(lig, nf, t, n)
    z = np.zeros(nf ** 3, np.float32)
    c.set_receptor_spectrum(z, z)
    rot = M.rotation_coefs(M.rotation_set(3600)[:n])
    got = c.dock(rot, np.arange(n, dtype=np.int32)).reshape(n, t)
    c.close()
    assert not got["score"].any()
    assert (got["index"][:, :, 0] == np.arange(n)[:, None]).all()
    assert (got["index"][:, :, 1:] == np.array([[0, k // nf, k % nf] for k in range(t)])[None]).all()


def test_time_of_a_tied_map(golden_dir, lig):
    """One tied map takes no more than ten times another (it is read twice more; one workgroup
    took seventy times as long)."""
    nf, t = 112, 64
    rec = M.Protein(os.path.join(golden_dir, "synth_r120.pdb"))
    c = _ctx(lig, nf, t, 1)
    rot, ids = M.rotation_coefs(M.rotation_set(24)[:1]), np.zeros(1, np.int32)
    took = []
    for grids in (M.receptor_grids(rec, nf // 2), (np.zeros((nf // 2) ** 3, np.float32),) * 2):
        c.set_receptor(*grids)
        best = np.inf
        for _ in range(10):
            t0 = time.perf_counter()
            c.dock(rot, ids)
            best = min(best, time.perf_counter() - t0)
        took.append(best)
    c.close()
    print("plain %.0f us, tied %.0f us" % (took[0] * 1e6, took[1] * 1e6), flush=True)
    assert took[1] < 10 * took[0]
