"""The rows of the Level2 SAT (gpview_amd/csrc/gpv_satrow.hpp) walked as the
kernel walks them, in pieces begun at any column, entries that are loose
included: no box that the reference's SAT accepts is dropped and none that it
rejects is accepted.  No tolerance: the claims are exact."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from conftest import ROOT
from test_sat_rows import _triangles

NATIVE = os.path.join(ROOT, "tests", "native")
FAMILIES = ["tiny", "random", "near", "axis", "sliver"]


@pytest.fixture(scope="module")
def pieces():
    so = os.path.join(NATIVE, "libsatrow.so")
    if not os.path.exists(so):
        subprocess.run(["make", "-s", "-C", NATIVE, so], check=True)
    f = ctypes.CDLL(so).satrow_pieces
    f32 = np.ctypeslib.ndpointer(dtype=np.float32, flags="C_CONTIGUOUS")
    u32 = np.ctypeslib.ndpointer(dtype=np.uint32, flags="C_CONTIGUOUS")
    u8 = np.ctypeslib.ndpointer(dtype=np.uint8, flags="C_CONTIGUOUS")
    f.argtypes = [ctypes.c_int64, ctypes.c_int, ctypes.c_int] + [f32] * 8 + [ctypes.c_int, u32, u32, u8]
    f.restype = None
    return f


def _tiny(rng, n, g1):
    """Triangles around the origin with one or two edges whose x and y differences
    are not zero but too small for a finite reciprocal."""
    t = rng.uniform(-1, 1, (n, 3, 3)) * g1 * rng.choice([1, 3], (n, 1, 1))
    small = rng.choice([-1, 1], (n, 3, 2)) * 10.0 ** rng.uniform(-44.8, -36, (n, 3, 2))
    a = rng.integers(0, 3, n)
    k = np.arange(n)
    for b in (a, (a + 1) % 3):
        t[k, b, :2] = small[k, b]
    m = rng.random(n) < 0.2
    t[m, (a[m] + 2) % 3, :2] = small[m, (a[m] + 2) % 3]
    return np.ascontiguousarray(t.reshape(n, 9).astype(np.float32))


@pytest.mark.parametrize("piece", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("fam", FAMILIES)
def test_pieces_never_contradict_the_sat(pieces, gv, orc, fam, piece):
    rng = np.random.default_rng(300 + 10 * FAMILIES.index(fam) + piece)
    hits = loose_hits = 0
    for vc, n2, size in [(8, 8, 1.0), (8, 16, 1.0), (33, 5, 1e3), (64, 11, 1e-3), (16, 4, 1e6), (4, 9, 1.0)]:
        ext = rng.uniform(0.4, 1, 3) * size
        bmin = (-ext * rng.uniform(0.3, 0.7, 3)).astype(np.float32)
        bmax = (bmin + ext).astype(np.float32)
        info = gv.grid_derive(bmin, bmax, float((bmax - bmin).max()), vc, n2)
        nn, g1, g2 = np.array(list(info.n)), np.array(list(info.g), float), np.array(list(info.g2), np.float32)
        n = max(150, min(1500, 150000 // n2 ** 3))
        if fam == "tiny":      # the voxel that holds the origin and its neighbours
            idx = np.floor(-bmin / g1).astype(int) + rng.integers(-1, 2, (n, 3))
            idx = np.clip(idx, 0, nn - 1)
            tv = _tiny(rng, n, g1)
        else:
            idx = np.stack([rng.integers(0, nn[a], n) for a in range(3)], 1)
            tv = _triangles(rng, fam, bmin + (idx + 0.5) * g1, g1, g2.astype(float), n2)
        c = [np.ascontiguousarray(gv.grid_centers(info, 2, a, False).reshape(nn[a], n2)[idx[:, a]]) for a in range(3)]
        h = (g2 / np.float32(2)).astype(np.float32)
        each = [np.ascontiguousarray(np.broadcast_to(x, (n, 3)), np.float32).ravel() for x in (bmin, bmax, g2, h)]
        inn, may = np.zeros((n, n2, n2), np.uint32), np.zeros((n, n2, n2), np.uint32)
        loose = np.zeros(n, np.uint8)
        pieces(n, n2, piece, tv.ravel(), c[0].ravel(), c[1].ravel(), c[2].ravel(), *each, 0, inn.ravel(), may.ravel(), loose)
        r = np.arange(n2, dtype=np.uint32)
        inn, may = (((m[..., None] >> r) & 1).astype(bool) for m in (inn, may))      # [case, q, p, r]
        cc = np.empty((n, n2, n2, n2, 3), np.float32)
        cc[..., 0], cc[..., 1], cc[..., 2] = c[0][:, None, :, None], c[1][:, :, None, None], c[2][:, None, None, :]
        big = np.broadcast_to(tv[:, None, None, None], (n, n2, n2, n2, 9)).reshape(-1, 9)
        hit = orc.tri_box(cc.reshape(-1, 3), np.broadcast_to(h, (len(big), 3)), big).reshape(inn.shape).astype(bool)
        assert not np.any(inn & ~hit), f"{vc}/{n2}: {np.count_nonzero(inn & ~hit)} boxes accepted that the SAT rejects"
        assert not np.any(hit & ~may), f"{vc}/{n2}: {np.count_nonzero(hit & ~may)} SAT hits dropped"
        hits += int(hit.sum())
        loose_hits += int(hit[loose != 0].sum())
    assert hits > 2000
    if fam == "tiny":
        assert loose_hits > 500     # the family reaches the loose form


@pytest.mark.gpu
@pytest.mark.parametrize("n2", [8, 16])
def test_near_zero_edges_on_the_device(gv, orc, n2):
    """Whole calls on a soup of such triangles."""
    from conftest import compare_results, say
    rng = np.random.default_rng(350 + n2)
    bmin, bmax = np.full(3, -0.5, np.float32), np.full(3, 0.5, np.float32)
    soup = _tiny(rng, 400, np.full(3, 0.12))
    say(f"near-zero edges, 8/{n2}")
    want = orc.voxelize(soup, orc.grid_setup(bmin, bmax, np.float32(1), 8, n2), orc.ORC_FAST)
    with gv.Context() as c:
        g = c.voxelize(soup, bmin, bmax, 1.0, 8, n2)
        compare_results(f"near-zero edges 8/{n2}", g.download(), want, n2)
        g.release()
