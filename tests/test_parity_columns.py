"""The Level2 parity by columns: the crossing bounds (gpview_amd/csrc/
gpv_parcol.hpp) against the float ray test over whole columns, and grids with
many boundary voxels per column against the oracle.  No tolerance: the claims
are exact."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from conftest import ROOT, compare_results, say
from test_sat_rows import _triangles

NATIVE = os.path.join(ROOT, "tests", "native")
EPS_ABOVE = 0x358637BE      # the smallest float above 1e-6


@pytest.fixture(scope="module")
def columns():
    so = os.path.join(NATIVE, "libparcol.so")
    if not os.path.exists(so):
        subprocess.run(["make", "-s", "-C", NATIVE, so], check=True)
    L = ctypes.CDLL(so)
    f32 = np.ctypeslib.ndpointer(dtype=np.float32, flags="C_CONTIGUOUS")
    L.parcol_batch.argtypes = [ctypes.c_int64, ctypes.c_int, ctypes.c_int] + [f32] * 4 + \
        [np.ctypeslib.ndpointer(dtype=np.int32, flags="C_CONTIGUOUS")] + [f32] * 5 + \
        [ctypes.c_int, ctypes.c_uint32, np.ctypeslib.ndpointer(dtype=np.int64, flags="C_CONTIGUOUS")]
    return L.parcol_batch


@pytest.mark.parametrize("fam", ["random", "small", "lattice", "near", "axis", "sliver"])
def test_crossings_never_contradict_the_ray_test(columns, gv, fam):
    rng = np.random.default_rng(100 + ["random", "small", "lattice", "near", "axis", "sliver"].index(fam))
    accepted = 0
    for k, (vc, n2) in enumerate([(256, 8), (64, 4), (64, 16), (8, 4), (33, 5), (128, 1), (4, 16), (100, 7), (33, 11)]):
        size = [1.0, 1e3, 10.0, 1.0, 0.1][k % 5]
        ext = rng.uniform(0.2, 1, 3) * size
        off = [0.0, 0.5, -1.0, 30.0, 3000.0][(k * 2) % 5] * rng.uniform(-1, 1, 3) * size
        bmin, bmax = off.astype(np.float32), (off + ext).astype(np.float32)
        info = gv.grid_derive(bmin, bmax, float((bmax - bmin).max()), vc, n2)
        cuda = k % 4 == 3
        nn, g1, g2 = np.array(list(info.n)), np.array(list(info.g), float), np.array(list(info.g2), np.float32)
        tabs = [gv.grid_centers(info, 3, a, cuda) for a in range(3)]
        n = int(max(60, min(2000, 3e7 / (len(tabs[2]) * n2 * n2))))
        idx = np.stack([rng.integers(0, nn[a], n) for a in range(3)], 1)
        ox, oy = (np.ascontiguousarray(tabs[a].reshape(nn[a], n2)[idx[:, a]]) for a in (0, 1))
        tv = _triangles(rng, fam, bmin + (idx + 0.5) * g1, g1, g2.astype(float), n2)
        l0 = np.ascontiguousarray(np.clip(idx[:, 2] + rng.integers(-1, 2, n), 0, nn[2] - 1) * n2, dtype=np.int32)
        h = (g2 / np.float32(2)).astype(np.float32)
        each = [np.ascontiguousarray(np.broadcast_to(x, (n, 3)), np.float32).ravel() for x in (bmin, bmax, g2, h)]
        out = np.zeros((n, 6), np.int64)
        columns(n, n2, len(tabs[2]), tv.ravel(), ox.ravel(), oy.ravel(), tabs[2], l0, *each,
                np.full(n, info.g[2], np.float32), int(cuda), EPS_ABOVE, out.ravel())
        got, outside, cand, wrong, _, _ = out.sum(0)
        assert outside == 0, f"{vc}/{n2}: {outside} accepted sub-columns outside the candidate range"
        assert wrong == 0, f"{vc}/{n2}: {wrong} layers contradict the crossing bounds"
        assert cand <= max(4 * got, got + 200 * n) or fam == "sliver"
        accepted += int(got)
    assert accepted > (100 if fam == "sliver" else 1000)   # most slivers fail the det test


@pytest.mark.parametrize("fam", ["random", "small", "lattice", "near", "axis", "sliver"])
def test_level1_crossings_never_contradict_the_ray_test(columns, gv, fam):
    """Level1: the certain layers of a column against the float test at every layer."""
    L = ctypes.CDLL(os.path.join(NATIVE, "libparcol.so"))
    f32 = np.ctypeslib.ndpointer(dtype=np.float32, flags="C_CONTIGUOUS")
    L.parl1_batch.argtypes = [ctypes.c_int64, ctypes.c_int] + [f32] * 4 + [ctypes.c_float] * 2 + \
        [ctypes.c_uint32, np.ctypeslib.ndpointer(dtype=np.int64, flags="C_CONTIGUOUS")]
    rng = np.random.default_rng(200 + ["random", "small", "lattice", "near", "axis", "sliver"].index(fam))
    accepted = left = 0
    for k, vc in enumerate([256, 64, 8, 33, 128, 4, 100, 512, 700]):
        size = [1.0, 1e3, 10.0, 1.0, 0.1][k % 5]
        ext = rng.uniform(0.2, 1, 3) * size
        off = [0.0, 0.5, -1.0, 30.0, 3000.0][(k * 2) % 5] * rng.uniform(-1, 1, 3) * size
        bmin, bmax = off.astype(np.float32), (off + ext).astype(np.float32)
        info = gv.grid_derive(bmin, bmax, float((bmax - bmin).max()), vc, 4)
        nn, g1 = np.array(list(info.n)), np.array(list(info.g), float)
        tabs = [gv.grid_centers(info, 1, a, False) for a in range(3)]
        n = int(max(2000, min(20000, 2e7 / nn[2])))
        idx = np.stack([rng.integers(0, nn[a], n) for a in range(3)], 1)
        ox, oy = (np.ascontiguousarray(tabs[a][idx[:, a]]) for a in (0, 1))
        assert np.all(np.diff(tabs[2]) >= 0)
        tv = _triangles(rng, fam, bmin + (idx + 0.5) * g1, g1, (g1 / 4), 4)
        out = np.zeros((n, 4), np.int64)
        L.parl1_batch(n, int(nn[2]), tv.ravel(), ox, oy, tabs[2], float(bmin[2]), float(bmax[2]), EPS_ABOVE, out.ravel())
        got, wrong, und, _ = out.sum(0)
        assert wrong == 0, f"{vc}: {wrong} layers contradict the crossing bounds"
        accepted += int(got)
        left += int(und)
    assert accepted > (20 if fam == "sliver" else 500)   # most slivers fail the det test
    assert left < 20 * accepted


def _tall(gv, seed):
    """A steep closed surface: dozens of boundary voxels in its columns."""
    v, f = gv.icosphere(4, 0.4, (0.5, 0.5, 0.5), 0.02, seed=seed)
    v = np.ascontiguousarray(v * np.float32([1, 1, 6]))
    return v, f


@pytest.mark.gpu
@pytest.mark.parametrize("n2", [1, 3, 4, 5, 8, 9, 16])
def test_tall_columns(gv, orc, n2):
    """More boundary voxels in a column than one pass of a wave holds, more
    than 64 layers, and a second mesh of another resolution in the batch; the
    whole-column candidates of the CUDA kernels' arithmetic as well."""
    from gpview_amd import workloads
    v, f = _tall(gv, 5)
    v2, f2 = gv.mixed(1, 2500, 12)
    ms = [workloads.mesh_entry(gv, v, f, 200, n2), workloads.mesh_entry(gv, v2, f2, 30, 8 if n2 != 8 else 4)]
    want = [orc.voxelize(m["soup"], orc.grid_setup(m["bmin"], m["bmax"], m["mms"], m["voxel_count"], m["voxel_count2"]),
                         orc.ORC_FAST) for m in ms]
    per_column = np.bincount(want[0]["bidx"] % (want[0]["l1"].size // 200))
    assert per_column.max() > 32
    with gv.Context() as c:
        say(f"tall columns: n2={n2}")
        m = ms[0]
        g = c.voxelize(m["soup"], m["bmin"], m["bmax"], m["mms"], 200, n2)
        compare_results(f"tall {n2}", g.download(), want[0], n2)
        g.release()
        for i, g in enumerate(c.voxelize_batch(ms)):
            compare_results(f"tall batch {n2}, mesh {i}", g.download(), want[i], ms[i]["voxel_count2"])
            g.release()
        gc = orc.grid_setup(m["bmin"], m["bmax"], m["mms"], 200, n2, cuda_l2=True)
        g = c.voxelize(m["soup"], m["bmin"], m["bmax"], m["mms"], 200, n2, cuda_level2=True)
        compare_results(f"tall cuda {n2}", g.download(), orc.voxelize(m["soup"], gc, orc.ORC_FAST), n2)
        g.release()


@pytest.mark.gpu
@pytest.mark.parametrize("n2", [4, 5, 8])
def test_many_columns(gv, orc, n2):
    """Enough columns for waves of two and four, columns of more boundary voxels
    than such a wave's window holds among them."""
    from gpview_amd import workloads
    v, f = gv.icosphere(4, 0.4, (0.5, 0.5, 0.5), 0.02, seed=9)
    m = workloads.mesh_entry(gv, v, f, 260, n2)
    want = orc.voxelize(m["soup"], orc.grid_setup(m["bmin"], m["bmax"], m["mms"], 260, n2), orc.ORC_FAST)
    per_column = np.bincount(want["bidx"] % (want["l1"].size // 260))
    assert per_column.size >= 1 << 16 and per_column.max() > 16
    with gv.Context() as c:
        say(f"many columns: n2={n2}")
        g = c.voxelize(m["soup"], m["bmin"], m["bmax"], m["mms"], 260, n2)
        compare_results(f"many columns {n2}", g.download(), want, n2)
        g.release()
