"""Whole grids on both sides of the sizes where a launch changes its form: the
blocks of the set-up (256 triangles), of the flag packing (1024 words) and of
the scans (4096), the tile offsets by the count's last block, the Level2
SAT's rows in pieces (n2 > 8), waves without columns in the ray expansion, and downloads
in one launch or in chunks.  Against the oracle, every product, bit for bit."""
import numpy as np
import pytest

from conftest import compare_results, say

pytestmark = pytest.mark.gpu


def _soup(gv, n, seed):
    """n triangles: a closed mesh, repeated and cut to the count."""
    v, f = gv.icosphere(5, 0.4, (0.5, 0.5, 0.5), 0.02, seed=seed)
    s = gv.flatten(v, f).reshape(-1, 9)
    s = np.concatenate([s] * (n // len(s) + 1))[:n]
    return np.ascontiguousarray(s, np.float32), np.asarray(v, np.float32)


@pytest.mark.parametrize("n,l1,n2", [(1, 8, 4), (255, 8, 4), (257, 8, 4), (4096, 20, 3), (4097, 20, 3),
                                     (65536, 40, 4), (65537, 40, 4), (70001, 36, 0)])
def test_triangle_counts(gv, orc, n, l1, n2):
    soup, v = _soup(gv, n, 21)
    bmin, bmax, mms = gv.mesh_bbox(v)
    want = orc.voxelize(soup, orc.grid_setup(bmin, bmax, mms, l1, n2), orc.ORC_FAST)
    with gv.Context() as c:
        say(f"triangles {n}, {l1}/{n2}")
        for _ in range(2):
            g = c.voxelize(soup, bmin, bmax, mms, l1, max(n2, 1), n2 > 0)
            compare_results(f"{n} triangles", g.download(), want, n2)
            g.release()


# words of a Level1 plane around 1024 and 4096, columns around a tile of the sorts, rows in pieces
@pytest.mark.parametrize("l1,n2", [(28, 9), (32, 8), (36, 16), (60, 4), (64, 5), (68, 11), (128, 2), (132, 1)])
def test_grid_sizes(gv, orc, l1, n2):
    v, f = gv.icosphere(3, 0.4, (0.5, 0.5, 0.5), 0.02, seed=22)
    soup = gv.flatten(v, f)
    bmin, bmax, mms = gv.mesh_bbox(v)
    want = orc.voxelize(soup, orc.grid_setup(bmin, bmax, mms, l1, n2), orc.ORC_FAST)
    with gv.Context() as c:
        say(f"grid {l1}/{n2}")
        g = c.voxelize(soup, bmin, bmax, mms, l1, n2)
        compare_results(f"grid {l1}/{n2}", g.download(), want, n2)
        g.release()


def test_walls_without_columns(gv, orc):
    """Long runs of triangles that no ray column meets (vertical ones) between flat
    faces whose crossings share words."""
    rng = np.random.default_rng(23)
    a = rng.uniform(0.1, 0.9, (40000, 2)).astype(np.float32)
    z = rng.uniform(0.2, 0.8, (40000, 2)).astype(np.float32)
    walls = np.zeros((40000, 3, 3), np.float32)
    walls[:, 0, :2] = walls[:, 1, :2] = a
    walls[:, 2, :2] = a + np.float32(0.01)
    walls[:, :, 2] = np.stack([z[:, 0], z[:, 1], z[:, 0]], 1)
    flat = np.array([[[0.05, 0.05, h], [0.95, 0.05, h], [0.95, 0.95, h]] for h in (0.11, 0.34, 0.52, 0.77)] +
                    [[[0.05, 0.05, h], [0.95, 0.95, h], [0.05, 0.95, h]] for h in (0.11, 0.34, 0.52, 0.77)], np.float32)
    soup = np.ascontiguousarray(np.concatenate([flat[:4], walls, flat[4:]]).reshape(-1, 9))
    bmin, bmax, mms = gv.mesh_bbox(soup.reshape(-1, 3))
    want = orc.voxelize(soup, orc.grid_setup(bmin, bmax, mms, 70, 3), orc.ORC_FAST)
    with gv.Context() as c:
        say("walls")
        g = c.voxelize(soup, bmin, bmax, mms, 70, 3)
        compare_results("walls", g.download(), want, 3)
        g.release()


def test_download_with_little_memory(gv):
    """The arrays of a download one after the other where the device memory for
    their exports does not hold two of them."""
    v, f = gv.icosphere(4, 0.4, (0.5, 0.5, 0.5), 0.02, seed=24)
    soup = gv.flatten(v, f)
    bmin, bmax, mms = gv.mesh_bbox(v)
    with gv.Context() as c:
        say("download with little memory")
        g = c.voxelize(soup, bmin, bmax, mms, 96, 2)
        want = g.download()
        n1 = want["l1"].size
        need = 1 << (4 * n1 - 1).bit_length()
        assert want["l2"].size <= need
        c.set_mem_limit(c.pool_stats()["live_bytes"] + need)
        got = g.download()
        for k in ("l1", "prefix", "bidx", "l2"):
            assert np.array_equal(got[k], want[k]), k
        c.set_mem_limit(0)
        g.release()
