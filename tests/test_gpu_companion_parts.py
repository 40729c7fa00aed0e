"""GPU: the companion score sums a large ligand in parts, a workgroup each: a pose's bits do not depend
on how many poses there are, its values are the float64 companion's, and one pose of a large
ligand takes little more time than one of a small ligand."""
import time

import numpy as np
import pytest

import megadock_amd as M
from oracle import oracle as O

pytestmark = pytest.mark.gpu

NG = 48


def _ligand(na):
    rng = np.random.default_rng(na)
    xyz = rng.uniform(-25, 25, (na, 3)).astype(np.float32)
    return xyz, np.zeros(3, np.float32), rng.choice([1.4, 1.63, 1.87], na).astype(np.float32), \
        rng.choice([0.1, -0.15, 0.33, -0.57, 0.0], na).astype(np.float32)


def _receptor():
    rng = np.random.default_rng(3)
    return rng.normal(size=NG ** 3).astype(np.float32), rng.normal(size=NG ** 3).astype(np.float32)


def _ctx(na, batch=8):
    c = M.Context(2 * NG, NG, na, t=1, max_batch=batch)
    c.set_receptor(*_receptor())
    c.set_ligand(*_ligand(na), M.grid_coord(NG), 1.2)
    return c


def _poses(n):
    rng = np.random.default_rng(n)
    return (np.linalg.qr(rng.normal(size=(n, 3, 3)))[0].reshape(n, 9).astype(np.float32),
            rng.uniform(-15, 15, (n, 3)).astype(np.float32))


@pytest.mark.parametrize("na", [1023, 2559, 2560, 2561, 4096, 4097, 16384, 17000, 65535])
def test_few_poses_and_many(na):
    c = _ctx(na)
    rot, t = _poses(1200)
    many = c.score_companion(rot, t)
    for n in (1, 2, 63, 300):
        print("na=%d poses=%d" % (na, n), flush=True)
        assert np.array_equal(c.score_companion(rot[:n], t[:n]).view(np.uint32), many[:n].view(np.uint32))
    c.close()
    assert np.isfinite(many).all()


def test_more_poses_than_a_launch_takes():
    c = _ctx(17000)  # 16 parts, 4096 poses
    rot, t = _poses(8200)
    many = c.score_companion(rot, t)
    for a, b in ((4090, 4100), (8190, 8200), (4096, 8200)):
        assert np.array_equal(c.score_companion(rot[a:b], t[a:b]).view(np.uint32), many[a:b].view(np.uint32))
    c.close()


@pytest.mark.parametrize("na", [2560, 5000])
def test_against_float64(na):
    """A float position is off by at most 2^-22 * 2 * 25 / 1.2 * sqrt(3) ~ 2e-5 voxels (25 A, a few
    roundings); values and gradients of a grid of order 1 (up to 5) change by up to 10 times that an atom, in
    sums whose terms have a random sign: within 1e-3 of the root of the sum of squares."""
    c = _ctx(na)
    rot, t = _poses(2)
    got = c.score_companion(rot, t)
    c.close()
    xyz, cen, rad, chg = _ligand(na)
    gr, gi = _receptor()
    ws = 4.0 / 3.0 * np.pi * rad.astype(np.float64) ** 3 / 1.2 ** 3
    scale = np.sqrt((ws ** 2 + chg.astype(np.float64) ** 2).sum())
    for q in range(2):
        s, dt, dw = O.companion_fp64(gr, gi, NG, np.float64(np.float32(1.2)), xyz, cen, rad, chg, rot[q].reshape(3, 3),
                                     t[q], 2 * NG)
        # an atom whose cell differs between float and double takes another slope: a few of 5000
        assert abs(got[q, 0] - s) <= 1e-3 * scale
        assert np.linalg.norm(got[q, 1:4] - dt) <= 0.2 * scale
        assert np.linalg.norm(got[q, 4:7] - dw) <= 0.2 * 25 * scale


def test_time_of_one_pose():
    """30000 atoms against 300, one pose: 7.2 times the time in one workgroup, under 2 in parts."""
    took = []
    for na in (300, 30000):
        c = _ctx(na)
        rot, t = _poses(1)
        best = np.inf
        for _ in range(40):
            t0 = time.perf_counter()
            c.score_companion(rot, t)
            best = min(best, time.perf_counter() - t0)
        c.close()
        took.append(best)
    print("300 atoms %.0f us, 30000 atoms %.0f us" % (took[0] * 1e6, took[1] * 1e6), flush=True)
    assert took[1] < 4 * took[0]
