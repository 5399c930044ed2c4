"""The row form of the Level2 SAT (gpview_amd/csrc/gpv_satrow.hpp) against the
reference's SAT: every box it accepts for certain is a SAT hit and every hit
is a box it accepts or leaves to the float SAT.  No tolerance: the claims are
exact.  The tables are the library's own (gpv_grid_centers)."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from conftest import ROOT, compare_results, say

NATIVE = os.path.join(ROOT, "tests", "native")


@pytest.fixture(scope="module")
def rows():
    so = os.path.join(NATIVE, "libsatrow.so")
    if not os.path.exists(so):
        subprocess.run(["make", "-s", "-C", NATIVE, so], check=True)
    L = ctypes.CDLL(so)
    f32 = np.ctypeslib.ndpointer(dtype=np.float32, flags="C_CONTIGUOUS")
    u32 = np.ctypeslib.ndpointer(dtype=np.uint32, flags="C_CONTIGUOUS")
    L.satrow_batch.argtypes = [ctypes.c_int64, ctypes.c_int] + [f32] * 8 + [ctypes.c_int, u32, u32]
    i32, i64 = (np.ctypeslib.ndpointer(dtype=d, flags="C_CONTIGUOUS") for d in (np.int32, np.int64))
    L.satcol_batch.argtypes = [ctypes.c_int64, f32, i32, i32] + [f32] * 6 + [i64, i32]
    L.satrow_batch.columns = L.satcol_batch
    L.sataxis_batch.argtypes = [ctypes.c_int64, ctypes.c_int] + [f32] * 6 + [ctypes.c_int, i32]
    L.satrow_batch.axis = L.sataxis_batch
    return L.satrow_batch


def _triangles(rng, fam, C, g1, g2, n2):
    """Triangles around voxels with centers C, sizes g1 and sub-voxels g2."""
    n = len(C)
    near = C[:, None] + rng.uniform(-0.6, 0.6, (n, 1, 3)) * g1
    if fam == "random":
        t = near + rng.normal(0, 1, (n, 3, 3)) * 10.0 ** rng.uniform(-2, 1.3, (n, 1, 1)) * g1 * 0.5
    elif fam == "small":
        t = near + rng.normal(0, 1, (n, 3, 3)) * g2 * rng.uniform(0.1, 4, (n, 1, 1))
    elif fam == "lattice":      # vertices on sub-voxel faces and centers
        t = (C - 0.5 * g1)[:, None] + rng.integers(-1, n2 + 2, (n, 3, 3)) * rng.choice([1, 0.5], (n, 1, 1)) * g2
    elif fam == "near":         # a hair off them
        k = rng.integers(-2, 2 * n2 + 4, (n, 3, 3)) * 0.5
        t = (C - 0.5 * g1)[:, None] + k * g2 * (1 + rng.choice([0, 1, -1], (n, 3, 3)) * 10.0 ** rng.uniform(-9, -3, (n, 3, 3)))
    elif fam == "axis":         # edges and planes along the axes, repeated vertices
        t = near + rng.normal(0, 1, (n, 3, 3)) * g1 * 0.6
        for i in range(3):
            j, a = (i + 1) % 3, rng.integers(0, 3, n)
            for b in (a, (a + 1) % 3):
                m = rng.random(n) < 0.4
                t[m, j, b[m]] = t[m, i, b[m]]
        m = rng.random(n) < 0.2
        t[m, 0] = t[m, 1] + rng.choice([0, 1e-6, 1e-4], (m.sum(), 1)) * g1
    else:                       # slivers
        d = rng.normal(0, 1, (n, 3)) * g1 * 10.0 ** rng.uniform(-1, 1, (n, 1))
        w = rng.normal(0, 1, (n, 3)) * g1 * 10.0 ** rng.uniform(-8, -2, (n, 1))
        t = np.stack([near[:, 0] - d, near[:, 0] + d, near[:, 0] + w + d * rng.uniform(-1, 1, (n, 1))], 1)
    return np.ascontiguousarray(t.reshape(n, 9).astype(np.float32))


@pytest.mark.parametrize("fam", ["random", "small", "lattice", "near", "axis", "sliver"])
def test_rows_never_contradict_the_sat(rows, gv, orc, fam):
    rng = np.random.default_rng(["random", "small", "lattice", "near", "axis", "sliver"].index(fam))
    hits = left = 0
    # voxel counts, Level2 sizes, extents and offsets from the origin (in extents)
    for k, (vc, n2) in enumerate([(256, 8), (512, 16), (64, 4), (8, 4), (33, 5), (512, 1), (4, 16), (100, 7), (256, 11)]):
        size = [1.0, 1e3, 1e-3, 1e8, 1e-8][k % 5]
        ext = rng.uniform(0.2, 1, 3) * size
        off = [0.0, 0.5, -1.0, 30.0, 3000.0][(k * 2) % 5] * rng.uniform(-1, 1, 3) * size
        bmin, bmax = off.astype(np.float32), (off + ext).astype(np.float32)
        info = gv.grid_derive(bmin, bmax, float((bmax - bmin).max()), vc, n2)
        cuda = k % 4 == 3
        nn, g1, g2 = np.array(list(info.n)), np.array(list(info.g), float), np.array(list(info.g2), np.float32)
        tabs = [gv.grid_centers(info, 2, a, cuda).reshape(nn[a], n2) for a in range(3)]
        n = max(200, min(4000, 400000 // n2 ** 3))
        idx = np.stack([rng.integers(0, nn[a], n) for a in range(3)], 1)
        c = [np.ascontiguousarray(tabs[a][idx[:, a]]) for a in range(3)]
        tv = _triangles(rng, fam, bmin + (idx + 0.5) * g1, g1, g2.astype(float), n2)
        h = (g2 / np.float32(2)).astype(np.float32)
        each = [np.ascontiguousarray(np.broadcast_to(x, (n, 3)), np.float32).ravel() for x in (bmin, bmax, g2, h)]
        inn, may = np.zeros((n, n2, n2), np.uint32), np.zeros((n, n2, n2), np.uint32)
        rows(n, n2, tv.ravel(), c[0].ravel(), c[1].ravel(), c[2].ravel(), *each, int(cuda), inn.ravel(), may.ravel())
        r = np.arange(n2, dtype=np.uint32)
        inn, may = (((m[..., None] >> r) & 1).astype(bool) for m in (inn, may))      # [case, q, p, r]
        cc = np.empty((n, n2, n2, n2, 3), np.float32)
        cc[..., 0], cc[..., 1], cc[..., 2] = c[0][:, None, :, None], c[1][:, :, None, None], c[2][:, None, None, :]
        big = np.broadcast_to(tv[:, None, None, None], (n, n2, n2, n2, 9)).reshape(-1, 9)
        hit = orc.tri_box(cc.reshape(-1, 3), np.broadcast_to(h, (len(big), 3)), big).reshape(inn.shape).astype(bool)
        assert not np.any(inn & ~hit), f"{vc}/{n2}: {np.count_nonzero(inn & ~hit)} boxes accepted that the SAT rejects"
        assert not np.any(hit & ~may), f"{vc}/{n2}: {np.count_nonzero(hit & ~may)} SAT hits dropped"
        hits += int(hit.sum())
        left += int((may & ~inn).sum()) if size == 1.0 and abs(off).max() <= 1 else 0
    assert hits > 5000
    if fam in ("random", "small"):
        assert left < 0.1 * hits    # the float SAT is the exception, not the rule


@pytest.mark.gpu
@pytest.mark.parametrize("n2", [1, 6, 7, 8, 10, 13, 15, 16])
@pytest.mark.parametrize("below", [0, 1 << 20])
def test_level2_sat_groups(gv, orc, n2, below):
    """Level2 sizes on either side of the accumulator's byte and 16-bit forms,
    one voxel per wave and as many as fit, meshes that end inside a group."""
    from gpview_amd import workloads
    v, f = gv.mixed(2, 6000, 40 + n2)
    v2, f2 = gv.mixed(0, 1500, 90 + n2)
    ms = [workloads.mesh_entry(gv, v, f, 24, n2), workloads.mesh_entry(gv, v2, f2, 17, n2)]
    want = [orc.voxelize(m["soup"], orc.grid_setup(m["bmin"], m["bmax"], m["mms"], m["voxel_count"], n2), orc.ORC_FAST)
            for m in ms]
    with gv.Context() as c:
        c.set_tune(l2_group_below=below)
        say(f"Level2 SAT groups: n2={n2} below={below}")
        for w, m in zip(want, ms):
            g = c.voxelize(m["soup"], m["bmin"], m["bmax"], m["mms"], m["voxel_count"], n2)
            compare_results(f"alone {n2}", g.download(), w, n2)
            g.release()
        grids = c.voxelize_batch(ms)
        for w, g in zip(want, grids):
            compare_results(f"batch {n2}", g.download(), w, n2)
        for g in grids:
            g.release()


@pytest.mark.gpu
def test_level2_sat_huge_bin(gv, orc):
    """One voxel that holds every triangle of a fine mesh: more bin entries
    than a queued box's 16-bit entry number counts."""
    v, f = gv.icosphere(7, 0.05, (0.43, 0.43, 0.43), 0.02, seed=3)
    soup = gv.flatten(v, f)
    bmin, bmax = np.zeros(3, np.float32), np.ones(3, np.float32)
    assert len(soup) > 4 * 65536
    say(f"Level2 SAT, one bin of {len(soup)} entries")
    want = orc.voxelize(soup, orc.grid_setup(bmin, bmax, np.float32(1), 4, 4), orc.ORC_FAST)
    with gv.Context() as c:
        g = c.voxelize(soup, bmin, bmax, 1.0, 4, 4)
        compare_results("huge bin", g.download(), want, 4)
        assert g.info()["max_tris_per_voxel"] > 65536
        g.release()


@pytest.mark.parametrize("cuda", [False, True])
def test_box_axis_ends(rows, gv, cuda):
    """Where the box-axis runs are called clear, they are the float test's."""
    rng = np.random.default_rng(9 + cuda)
    clear = total = 0
    for k, (vc, n2) in enumerate([(256, 8), (512, 16), (64, 4), (8, 4), (33, 5), (512, 1), (100, 7)] * 2):
        size = [1.0, 1e3, 1e-3, 1e8, 1e-8][k % 5]
        ext = rng.uniform(0.2, 1, 3) * size
        off = [0.0, 0.5, -1.0, 30.0, 3000.0][(k * 2) % 5] * rng.uniform(-1, 1, 3) * size
        bmin, bmax = off.astype(np.float32), (off + ext).astype(np.float32)
        info = gv.grid_derive(bmin, bmax, float((bmax - bmin).max()), vc, n2)
        nn, g2 = np.array(list(info.n)), np.array(list(info.g2), np.float32)
        for a in range(3):
            n = 4000
            c = np.ascontiguousarray(gv.grid_centers(info, 2, a, cuda).reshape(nn[a], n2)[rng.integers(0, nn[a], n)])
            d = float(g2[a])
            u = rng.integers(-3, 2 * n2 + 3, (n, 2)) * 0.5 + rng.choice([0.0, 1e-7, -1e-7, 1e-5, 0.1], (n, 2))
            u[::2] = rng.uniform(-3, n2 + 3, (n // 2 + n % 2, 2)) * rng.choice([1, 1000], (n // 2 + n % 2, 1))
            e = np.sort((c[:, :1] + u * d).astype(np.float32), 1)
            lo, hi = np.ascontiguousarray(e[:, 0]), np.ascontiguousarray(e[:, 1])
            h = np.float32(g2[a] / np.float32(2))
            end = np.zeros((n, 3), np.int32)
            rows.axis(n, n2, lo, hi, c.ravel(), np.full(n, bmin[a]), np.full(n, bmax[a]), np.full(n, g2[a]), int(cuda), end.ravel())
            first = (lo[:, None] - c > h).sum(1)              # monotone: the centers that fail come first
            last = n2 - 1 - (hi[:, None] - c < -h).sum(1)
            ok = end[:, 2] != 0
            np.testing.assert_array_equal(np.clip(end[ok, 0], 0, n2), first[ok])
            np.testing.assert_array_equal(np.clip(end[ok, 1], -1, n2 - 1), last[ok])
            clear += int(ok.sum()) if size == 1.0 and abs(off).max() <= 1 else 0
            total += n if size == 1.0 and abs(off).max() <= 1 else 0
    assert clear > 0.4 * total


@pytest.mark.parametrize("fam", ["random", "small", "lattice", "near", "axis", "sliver"])
def test_columns_never_contradict_the_sat(rows, gv, orc, fam):
    """The same claims for the Level1 columns of a triangle's index AABB."""
    from test_slab_filter import _index_box
    rng = np.random.default_rng(70 + ["random", "small", "lattice", "near", "axis", "sliver"].index(fam))
    hits = left = 0
    for k, vc in enumerate([256, 64, 8, 512, 33, 100]):
        size = [1.0, 1e3, 1e-3, 1e8, 1e-8][k % 5]
        ext = rng.uniform(0.2, 1, 3) * size
        off = [0.0, 0.5, -1.0, 30.0, 3000.0][(k * 2) % 5] * rng.uniform(-1, 1, 3) * size
        bmin, bmax = off.astype(np.float32), (off + ext).astype(np.float32)
        info = gv.grid_derive(bmin, bmax, float((bmax - bmin).max()), vc, 1)
        nn, g1 = np.array(list(info.n)), np.array(list(info.g), np.float32)
        tabs = [gv.grid_centers(info, 0, a) for a in range(3)]
        idx = np.stack([rng.integers(0, nn[a], 500) for a in range(3)], 1)
        big = g1.astype(float) * [1, 8, 3][k % 3]
        tv = _triangles(rng, fam, bmin + (idx + 0.5) * g1.astype(float), big, g1.astype(float), 3)
        lo, hi = _index_box(tv, bmin, bmax, nn)
        dd = np.maximum(hi - lo + 1, 0)
        keep = (dd > 0).all(1) & (dd.prod(1) < 40000)
        tv, lo, dd = (np.ascontiguousarray(x[keep], t) for x, t in ((tv, np.float32), (lo, np.int32), (dd, np.int32)))
        at = np.concatenate([[0], np.cumsum(dd[:, 0].astype(np.int64) * dd[:, 1])]).astype(np.int64)
        out = np.zeros((at[-1], 4), np.int32)
        rows.columns(len(tv), tv.ravel(), lo.ravel(), dd.ravel(), *tabs, np.array(list(info.bmin), np.float32),
                     np.array(list(info.bmax), np.float32), g1, at, out.ravel())
        own = np.repeat(np.arange(len(tv)), np.diff(at))
        loc = np.arange(at[-1]) - at[own]
        col = np.repeat(np.arange(len(own)), dd[own, 2])
        z = np.arange(len(col)) - np.repeat(np.cumsum(dd[own, 2]) - dd[own, 2], dd[own, 2])
        c = np.stack([tabs[0][lo[own, 0] + loc % dd[own, 0]][col], tabs[1][lo[own, 1] + loc // dd[own, 0]][col],
                      tabs[2][lo[own[col], 2] + z]], 1)
        h = np.broadcast_to((g1 / np.float32(2)).astype(np.float32), c.shape)
        hit = orc.tri_box(c, h, tv[own[col]]).astype(bool)
        am, ai, bi, bm = out[col].T
        inn, may = (z >= ai) & (z < bi), (z >= am) & (z < bm)
        assert not np.any(inn & ~hit), f"{vc}: {np.count_nonzero(inn & ~hit)} boxes accepted that the SAT rejects"
        assert not np.any(hit & ~may), f"{vc}: {np.count_nonzero(hit & ~may)} SAT hits dropped"
        hits += int(hit.sum())
        left += int((may & ~inn).sum()) if size == 1.0 and abs(off).max() <= 1 else 0
    assert hits > 2000
    if fam in ("random", "small"):
        assert left < 0.1 * hits    # the float SAT is the exception, not the rule


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["one", "tall", "walls", "empty"])
def test_level1_sat_columns(gv, orc, kind):
    """Columns of more than 64 layers (steep slivers; upright walls that
    overflow a block's append buffer in one round) and long runs of triangles
    without a column between others, alone and in a batch."""
    from gpview_amd import workloads
    rng = np.random.default_rng(5)
    bmin, bmax = np.zeros(3, np.float32), np.array([0.5, 0.4, 1.0], np.float32)
    if kind == "one":
        soup = rng.uniform(0.1, 0.4, (1, 9))
    elif kind == "tall":        # slivers along z, a few columns each
        a = np.concatenate([rng.uniform(0.05, 0.35, (300, 2)), rng.uniform(0, 0.2, (300, 1))], 1)
        b = a + np.concatenate([rng.normal(0, 0.01, (300, 2)), rng.uniform(0.3, 0.8, (300, 1))], 1)
        soup = np.concatenate([a, b, a + rng.normal(0, 0.02, (300, 3))], 1)
    elif kind == "walls":       # x = const and slightly tilted, the whole box high and wide
        x = rng.uniform(0.05, 0.45, (40, 1))
        e = rng.normal(0, 1e-3, (40, 3)) * (np.arange(40) % 2)[:, None]
        o, w = np.zeros((40, 1)), np.ones((40, 1))
        soup = np.concatenate([x + e[:, :1], o, o, x + e[:, 1:2], w * 0.8, o, x + e[:, 2:], o, w * 2], 1)
    else:                       # only every 500th triangle meets the grid
        soup = rng.uniform(2, 3, (4000, 9))
        soup[::500] = rng.uniform(0.05, 0.35, (8, 9))
    soup = np.ascontiguousarray(soup, np.float32)
    v, f = gv.mixed(1, 2000, 3)
    say(f"Level1 SAT columns: {kind}")
    mms = np.float32(1)
    mesh = {"soup": soup, "bmin": bmin, "bmax": bmax, "mms": mms, "voxel_count": 150, "voxel_count2": 2, "level2": True,
            "initial_capacity": 0}
    other = workloads.mesh_entry(gv, v, f, 20, 2)
    want = [orc.voxelize(m["soup"], orc.grid_setup(m["bmin"], m["bmax"], m["mms"], m["voxel_count"], 2), orc.ORC_FAST)
            for m in (mesh, other)]
    with gv.Context() as c:
        g = c.voxelize(soup, bmin, bmax, float(mms), 150, 2)
        compare_results(f"{kind} alone", g.download(), want[0], 2)
        g.release()
        grids = c.voxelize_batch([mesh, other, mesh])
        for w, g in zip([want[0], want[1], want[0]], grids):
            compare_results(f"{kind} batch", g.download(), w, 2)
        for g in grids:
            g.release()
