"""Grids in which few columns hold boundary voxels."""
import numpy as np
import pytest

from conftest import compare_results, say

pytestmark = pytest.mark.gpu


def _cluster(n, size, at, seed):
    rng = np.random.default_rng(seed)
    return np.ascontiguousarray(at + size * rng.uniform(0, 1, (n, 9)), np.float32)


# one, two and four columns a wave, words with one and several occupied columns, both ends of a row
@pytest.mark.parametrize("l1,n2", [(64, 16), (132, 9), (256, 8), (256, 5), (256, 4), (260, 1), (20, 4)])
def test_few_occupied_columns(gv, orc, l1, n2):
    soup = np.concatenate([_cluster(15, 0.03, a, 40 + k) for k, a in enumerate((0.0, 0.31, 0.5, 0.97))])
    bmin, bmax, mms = np.zeros(3, np.float32), np.array([1, 0.9, 0.8], np.float32), np.float32(1)
    want = orc.voxelize(soup, orc.grid_setup(bmin, bmax, mms, l1, n2), orc.ORC_FAST)
    mesh = {"soup": soup, "bmin": bmin, "bmax": bmax, "mms": mms, "voxel_count": l1, "voxel_count2": n2}
    other = {"soup": soup[:20], "bmin": bmin, "bmax": bmax, "mms": mms, "voxel_count": 24, "voxel_count2": 3}
    wother = orc.voxelize(soup[:20], orc.grid_setup(bmin, bmax, mms, 24, 3), orc.ORC_FAST)
    with gv.Context() as c:
        say(f"few occupied columns {l1}/{n2}")
        for _ in range(2):
            g = c.voxelize(soup, bmin, bmax, mms, l1, n2)
            compare_results(f"{l1}/{n2}", g.download(), want, n2)
            g.release()
        grids = c.voxelize_batch([other, mesh, other])
        for g, w, n in zip(grids, (wother, want, wother), (3, n2, 3)):
            compare_results(f"batch {l1}/{n2}", g.download(), w, n)
            g.release()
        g = c.create(soup, bmin, bmax, mms, l1, n2)     # the staged form, its bins made twice
        g.classify_tessellation()
        g.classify_inout()
        g.compact_boundary()
        g.compact_boundary()
        g.classify_tessellation_level2()
        g.classify_inout_level2()
        g.finish()
        compare_results(f"staged {l1}/{n2}", g.download(), want, n2)
        g.release()


# columns taken by several waves (up to 1,024 of them) and not; more boundary voxels than one
# window of a column holds, more entries than the waves stage at once, and few of either
@pytest.mark.parametrize("thin,l1,n2", [(0.02, 400, 16), (0.02, 400, 8), (0.03, 300, 11), (0.05, 600, 1), (0.05, 600, 4),
                                        (0.124, 256, 8), (0.14, 256, 8), (0.124, 256, 16), (1, 12, 16), (1, 4, 5)])
def test_few_tall_columns(gv, orc, thin, l1, n2):
    v, f = gv.mixed(1, 9000, 51)
    v = np.asarray(v, np.float64).copy()
    v[:, :2] *= thin
    v = v.astype(np.float32)
    soup = gv.flatten(v, f)
    bmin, bmax, mms = gv.mesh_bbox(v)
    want = orc.voxelize(soup, orc.grid_setup(bmin, bmax, mms, l1, n2), orc.ORC_FAST)
    mesh = {"soup": soup, "bmin": bmin, "bmax": bmax, "mms": mms, "voxel_count": l1, "voxel_count2": n2}
    with gv.Context() as c:
        say(f"few tall columns x{thin} {l1}/{n2}")
        g = c.voxelize(soup, bmin, bmax, mms, l1, n2)
        say(f"grid {g.info()['n']}, {g.info()['nb']} boundary voxels")
        compare_results(f"alone {l1}/{n2}", g.download(), want, n2)
        g.release()
        for g in c.voxelize_batch([mesh, mesh]):
            compare_results(f"batch {l1}/{n2}", g.download(), want, n2)
            g.release()


# columns of many entries among many columns: one, two and four columns a wave, batches of
# meshes with different ones, more of them than blocks of a round
@pytest.mark.parametrize("l1,n2,n,size", [(256, 8, 400, 0.1), (256, 4, 400, 0.1), (256, 3, 300, 0.3), (128, 16, 300, 0.1), (100, 5, 500, 0.2),
                                          (128, 9, 300, 0.1), (40, 1, 900, 0.3), (64, 12, 129, 0.05)])
def test_columns_of_many_entries(gv, orc, l1, n2, n, size):
    soup = np.concatenate([_cluster(n, size, 0.5, 60 + n2), _cluster(40, 0.6, 0.2, 61)])
    bmin, bmax, mms = np.zeros(3, np.float32), np.ones(3, np.float32), np.float32(1)
    want = orc.voxelize(soup, orc.grid_setup(bmin, bmax, mms, l1, n2), orc.ORC_FAST)
    mesh = {"soup": soup, "bmin": bmin, "bmax": bmax, "mms": mms, "voxel_count": l1, "voxel_count2": n2}
    other = {"soup": soup[:200], "bmin": bmin, "bmax": bmax, "mms": mms, "voxel_count": 40, "voxel_count2": 7}
    wother = orc.voxelize(soup[:200], orc.grid_setup(bmin, bmax, mms, 40, 7), orc.ORC_FAST)
    with gv.Context() as c:
        for overlap in (1, 0):
            c.set_tune(l2_overlap=overlap, l2_parity_waves=1 if overlap else 4)
            say(f"columns of many entries {l1}/{n2}, overlap {overlap}")
            g = c.voxelize(soup, bmin, bmax, mms, l1, n2)
            compare_results(f"{l1}/{n2}", g.download(), want, n2)
            g.release()
            for g, w, k in zip(c.voxelize_batch([other, mesh]), (wother, want), (7, n2)):
                compare_results(f"batch {l1}/{n2}", g.download(), w, k)
                g.release()
        g = c.create(soup, bmin, bmax, mms, l1, n2)     # the staged form, its parity made three times
        while g.classify_tessellation():    # its bins grow
            pass
        g.classify_inout()
        g.compact_boundary()
        for _ in range(3):
            g.classify_inout_level2()
        g.classify_tessellation_level2()
        g.finish()
        compare_results(f"staged {l1}/{n2}", g.download(), want, n2)
        g.release()


def test_empty_columns_cost_little(gv):
    """The Level2 parity of 27 boundary voxels in 262,144 columns of 512 layers: 0.89 ms
    with a scan of every column, 0.05 ms with the occupied ones only."""
    soup = _cluster(20, 0.005, 0.5, 7)
    bmin, bmax = np.zeros(3, np.float32), np.ones(3, np.float32)
    with gv.Context() as c:
        say("empty columns")
        ms = []
        for _ in range(5):
            g = c.voxelize(soup, bmin, bmax, 1.0, 512, 16)
            ms.append(g.info()["ms_stage"][4])
            g.release()
        say(f"Level2 parity {min(ms):.3f} ms")
        assert min(ms) < 0.3


def test_few_columns_share_the_chip(gv):
    """The Level2 parity of a rod of 12 x 12 columns and 512 layers at n2 = 16: 0.63 ms with
    a wave to a column, 0.18 ms with four."""
    v, f = gv.mixed(1, 60000, 31)
    v = np.asarray(v, np.float32).copy()
    v[:, :2] *= np.float32(0.02)
    soup, box = gv.flatten(v, f), gv.mesh_bbox(v)
    with gv.Context() as c:
        say("few columns")
        ms = []
        for _ in range(5):
            g = c.voxelize(soup, *box, 512, 16)
            ms.append(g.info()["ms_stage"][4])
            g.release()
        say(f"Level2 parity {min(ms):.3f} ms")
        assert min(ms) < 0.4


def test_few_heavy_columns_are_shared(gv):
    """2,000 overlapping triangles in a tenth of a 256/8 grid: the Level2 parity took 1.6 ms
    with a wave to two columns whatever they hold, 0.54 with four waves to those of many."""
    soup = _cluster(2000, 0.1, 0.5, 2)
    bmin, bmax = np.zeros(3, np.float32), np.ones(3, np.float32)
    with gv.Context() as c:
        say("few heavy columns")
        ms = []
        for _ in range(5):
            g = c.voxelize(soup, bmin, bmax, 1.0, 256, 8)
            ms.append(g.info()["ms_stage"][4])
            g.release()
        say(f"Level2 parity {min(ms):.3f} ms")
        assert min(ms) < 0.9


@pytest.mark.parametrize("layers,n2", [(700, 8), (1500, 3), (500, 16)])
def test_columns_of_many_windows(gv, orc, layers, n2):
    """A rod of few columns and many layers, so that a column's voxels take many windows."""
    v, f = gv.mixed(1, 3000, 33)
    v = np.asarray(v, np.float32).copy()
    v[:, :2] *= np.float32(0.06)
    soup, (bmin, bmax, mms) = gv.flatten(v, f), gv.mesh_bbox(v)
    say(f"many windows {layers}/{n2}")
    want = orc.voxelize(soup, orc.grid_setup(bmin, bmax, mms, layers, n2), orc.ORC_FAST)
    with gv.Context() as c:
        g = c.voxelize(soup, bmin, bmax, float(mms), layers, n2)
        compare_results(f"many windows {layers}/{n2}", g.download(), want, n2)
        g.release()


def test_tall_columns_are_scanned_once(gv):
    """The Level2 parity of a rod of 7,488 columns and 8,192 layers at n2 = 8: 13 ms with every
    layer scanned for each window, 2.4 with those that hold the window's voxels."""
    v, f = gv.mixed(1, 60000, 31)
    v = np.asarray(v, np.float32).copy()
    v[:, :2] *= np.float32(0.01)
    soup, box = gv.flatten(v, f), gv.mesh_bbox(v)
    with gv.Context() as c:
        say("tall columns")
        ms = []
        for _ in range(4):
            g = c.voxelize(soup, *box, 8192, 8)
            ms.append(g.info()["ms_stage"][4])
            g.release()
        say(f"Level2 parity {min(ms):.3f} ms")
        assert min(ms) < 6


def test_columns_of_many_windows_share_the_chip(gv):
    """The Level2 parity of a rod of some 1,200 columns and 4,096 layers at n2 = 16: 3.5 ms with a
    wave to a column, 1.5 with four."""
    v, f = gv.mixed(1, 60000, 31)
    v = np.asarray(v, np.float32).copy()
    v[:, :2] *= np.float32(0.01)
    soup, box = gv.flatten(v, f), gv.mesh_bbox(v)
    with gv.Context() as c:
        say("columns of many windows")
        ms = []
        for _ in range(4):
            g = c.voxelize(soup, *box, 4096, 16)
            ms.append(g.info()["ms_stage"][4])
            g.release()
        say(f"Level2 parity {min(ms):.3f} ms")
        assert min(ms) < 2.6
