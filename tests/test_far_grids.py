"""Grids so far from the origin that a float hardly tells one sub-voxel from the
next: the Level2 SAT's rows and the ray parities' crossings with the positions
taken from the tables (gpview_amd/csrc/gpv_satrow.hpp, gpv_parcol.hpp) against
the float predicates, and whole calls against the oracle.  No tolerance: the claims
are exact."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from conftest import ROOT, compare_results, say
from test_sat_rows import _triangles

NATIVE = os.path.join(ROOT, "tests", "native")
FAMILIES = ["random", "small", "lattice", "near", "axis", "sliver"]
EPS_ABOVE = 0x358637BE      # the smallest float above 1e-6


def _lib(name):
    so = os.path.join(NATIVE, name)
    if not os.path.exists(so):
        subprocess.run(["make", "-s", "-C", NATIVE, so], check=True)
    return ctypes.CDLL(so)


def _nd(t):
    return np.ctypeslib.ndpointer(dtype=t, flags="C_CONTIGUOUS")


# voxel counts, Level2 sizes, extents and distances from the origin in sub-voxels
GRIDS = [(8, 8, 1.0, 1e6), (8, 16, 1.0, 4e6), (33, 5, 1e3, 2e7), (64, 11, 1e-3, 1e5), (16, 4, 10.0, 1e7), (4, 9, 1.0, 3e7),
         (64, 1, 1.0, 1e8), (8, 16, 1.0, 3e7), (33, 7, 1.0, 3e3)]


def _grid(gv, rng, vc, n2, size, dist):
    ext = rng.uniform(0.4, 1, 3) * size
    off = rng.choice([-1, 1], 3) * rng.uniform(0.3, 1, 3) * dist * size / (vc * n2)
    bmin = off.astype(np.float32)
    bmax = (off + ext).astype(np.float32)
    bmax = np.where(bmax > bmin, bmax, np.nextafter(bmin, np.float32(np.inf)))
    info = gv.grid_derive(bmin, bmax, float((bmax - bmin).max()), vc, n2)
    return bmin, bmax, info, np.array(list(info.n)), np.array(list(info.g), float), np.array(list(info.g2), np.float32)


@pytest.mark.parametrize("piece", [1, 4, 16])
@pytest.mark.parametrize("fam", FAMILIES)
def test_far_rows_never_contradict_the_sat(gv, orc, fam, piece):
    f = _lib("libsatrow.so").satrow_far
    f.argtypes = [ctypes.c_int64, ctypes.c_int, ctypes.c_int] + [_nd(np.float32)] * 8 + \
        [ctypes.c_int, _nd(np.uint32), _nd(np.uint32), _nd(np.uint8)]
    rng = np.random.default_rng(700 + 10 * FAMILIES.index(fam) + piece)
    hits = left = 0
    for k, (vc, n2, size, dist) in enumerate(GRIDS):
        bmin, bmax, info, nn, g1, g2 = _grid(gv, rng, vc, n2, size, dist)
        cuda = k % 3 == 1
        n = max(150, min(1500, 150000 // n2 ** 3))
        idx = np.stack([rng.integers(0, nn[a], n) for a in range(3)], 1)
        tv = _triangles(rng, fam, bmin + (idx + 0.5) * g1, g1, g2.astype(float), n2)
        c = [np.ascontiguousarray(gv.grid_centers(info, 2, a, cuda).reshape(nn[a], n2)[idx[:, a]]) for a in range(3)]
        h = (g2 / np.float32(2)).astype(np.float32)
        each = [np.ascontiguousarray(np.broadcast_to(x, (n, 3)), np.float32).ravel() for x in (bmin, bmax, g2, h)]
        inn, may = np.zeros((n, n2, n2), np.uint32), np.zeros((n, n2, n2), np.uint32)
        f(n, n2, piece, tv.ravel(), c[0].ravel(), c[1].ravel(), c[2].ravel(), *each, int(cuda), inn.ravel(), may.ravel(),
          np.zeros(n, np.uint8))
        r = np.arange(n2, dtype=np.uint32)
        inn, may = (((m[..., None] >> r) & 1).astype(bool) for m in (inn, may))      # [case, q, p, r]
        cc = np.empty((n, n2, n2, n2, 3), np.float32)
        cc[..., 0], cc[..., 1], cc[..., 2] = c[0][:, None, :, None], c[1][:, :, None, None], c[2][:, None, None, :]
        big = np.broadcast_to(tv[:, None, None, None], (n, n2, n2, n2, 9)).reshape(-1, 9)
        hit = orc.tri_box(cc.reshape(-1, 3), np.broadcast_to(h, (len(big), 3)), big).reshape(inn.shape).astype(bool)
        assert not np.any(inn & ~hit), f"{vc}/{n2}: {np.count_nonzero(inn & ~hit)} boxes accepted that the SAT rejects"
        assert not np.any(hit & ~may), f"{vc}/{n2}: {np.count_nonzero(hit & ~may)} SAT hits dropped"
        hits += int(hit.sum())
        left += int((may & ~inn).sum())
    assert hits > 2000
    if fam == "random":
        assert left < 0.1 * hits    # the float SAT is the exception, not the rule


@pytest.mark.parametrize("fam", FAMILIES)
def test_far_crossings_never_contradict_the_ray_test(gv, fam):
    f = _lib("libparcol.so").parcol_far
    f.argtypes = [ctypes.c_int64, ctypes.c_int, ctypes.c_int] + [_nd(np.float32)] * 4 + [_nd(np.int32)] + \
        [_nd(np.float32)] * 5 + [ctypes.c_int, ctypes.c_uint32, _nd(np.int64)]
    rng = np.random.default_rng(800 + FAMILIES.index(fam))
    accepted = 0
    for k, (vc, n2, size, dist) in enumerate(GRIDS):
        bmin, bmax, info, nn, g1, g2 = _grid(gv, rng, vc, n2, size * 30, dist)
        cuda = k % 3 == 1
        tabs = [gv.grid_centers(info, 3, a, cuda) for a in range(3)]
        n = int(max(60, min(2000, 3e7 / (len(tabs[2]) * n2 * n2))))
        idx = np.stack([rng.integers(0, nn[a], n) for a in range(3)], 1)
        ox, oy = (np.ascontiguousarray(tabs[a].reshape(nn[a], n2)[idx[:, a]]) for a in (0, 1))
        tv = _triangles(rng, fam, bmin + (idx + 0.5) * g1, g1, g2.astype(float), n2)
        l0 = np.ascontiguousarray(np.clip(idx[:, 2] + rng.integers(-1, 2, n), 0, nn[2] - 1) * n2, dtype=np.int32)
        h = (g2 / np.float32(2)).astype(np.float32)
        each = [np.ascontiguousarray(np.broadcast_to(x, (n, 3)), np.float32).ravel() for x in (bmin, bmax, g2, h)]
        out = np.zeros((n, 6), np.int64)
        f(n, n2, len(tabs[2]), tv.ravel(), ox.ravel(), oy.ravel(), tabs[2], l0, *each,
          np.full(n, info.g[2], np.float32), int(cuda), EPS_ABOVE, out.ravel())
        got, outside, _, wrong, _, _ = out.sum(0)
        assert outside == 0, f"{vc}/{n2}: {outside} accepted sub-columns outside the candidate range"
        assert wrong == 0, f"{vc}/{n2}: {wrong} layers contradict the crossing bounds"
        accepted += int(got)
    assert accepted > (100 if fam == "sliver" else 1000)   # most slivers fail the det test


def _mesh(gv, tris, seed, scale, off):
    v, f = gv.mixed(1, tris, seed)
    return (np.asarray(v, np.float64) * scale + np.asarray(off)).astype(np.float32), f


@pytest.mark.gpu
@pytest.mark.parametrize("n2", [1, 3, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("cuda", [False, True])
def test_far_grids_on_the_device(gv, orc, n2, cuda):
    """Offsets on both sides of the line between the two forms, alone and in a batch
    with a mesh at the origin; few columns, and enough for waves of their own."""
    from gpview_amd import workloads
    with gv.Context() as c:
        for vc, tris in ((16, 800), (72, 6000)):
            ms, want = [], []
            for k, o in enumerate((0.0, 300.0, 5e3, 2e4, 1e5)):
                v, f = _mesh(gv, tris, 60 + k, 1.0, (o, -o, 0.7 * o))
                m = workloads.mesh_entry(gv, v, f, vc, n2)
                m["cuda_level2"] = cuda
                ms.append(m)
                want.append(orc.voxelize(m["soup"], orc.grid_setup(m["bmin"], m["bmax"], m["mms"], vc, n2, cuda_l2=cuda),
                                         orc.ORC_FAST))
                say(f"far {vc}/{n2} offset {o:g} cuda={cuda}")
                g = c.voxelize(m["soup"], m["bmin"], m["bmax"], m["mms"], vc, n2, cuda_level2=cuda)
                compare_results(f"far {vc}/{n2} at {o:g}", g.download(), want[-1], n2)
                g.release()
            for i, g in enumerate(c.voxelize_batch(ms)):
                compare_results(f"far batch {vc}/{n2}, mesh {i}", g.download(), want[i], n2)
                g.release()
