"""Triangles two of whose vertices are the same (segments): the Level2 SAT's rows and the
Level1 SAT's columns bound them like any other, so that few boxes are left to the float
SAT, and never contradict it."""
import numpy as np
import pytest

from test_sat_row_pieces import pieces  # noqa: F401
from test_sat_rows import rows          # noqa: F401
from test_slab_filter import _index_box


def _segments(rng, C, size, which):
    n = len(C)
    t = C[:, None] + rng.uniform(-0.6, 0.6, (n, 1, 3)) * size + rng.normal(0, 1, (n, 3, 3)) * size * 10.0 ** rng.uniform(-1.5, 1, (n, 1, 1))
    t = t.astype(np.float32)
    t[:, (which + 1) % 3] = t[:, which]
    flat = rng.random(n) < 0.2                   # along an axis or in a coordinate plane
    for a in range(3):
        m = flat & (rng.random(n) < 0.5)
        t[m, :, a] = t[m, :1, a]
    return np.ascontiguousarray(t.reshape(n, 9))


@pytest.mark.parametrize("which", [0, 1, 2])
@pytest.mark.parametrize("vc,n2", [(64, 8), (16, 16), (100, 5)])
def test_rows_of_segments(pieces, gv, orc, vc, n2, which):  # noqa: F811
    rng = np.random.default_rng(500 + 10 * n2 + which)
    bmin, bmax = np.float32([-0.3, 0.1, -0.6]), np.float32([0.6, 0.9, 0.3])
    info = gv.grid_derive(bmin, bmax, 0.9, vc, n2)
    nn, g1, g2 = np.array(list(info.n)), np.array(list(info.g), float), np.array(list(info.g2), np.float32)
    n = 600
    idx = np.stack([rng.integers(0, nn[a], n) for a in range(3)], 1)
    tv = _segments(rng, bmin + (idx + 0.5) * g1, g1, which)
    c = [np.ascontiguousarray(gv.grid_centers(info, 2, a, False).reshape(nn[a], n2)[idx[:, a]]) for a in range(3)]
    h = (g2 / np.float32(2)).astype(np.float32)
    each = [np.ascontiguousarray(np.broadcast_to(x, (n, 3)), np.float32).ravel() for x in (bmin, bmax, g2, h)]
    inn, may = np.zeros((n, n2, n2), np.uint32), np.zeros((n, n2, n2), np.uint32)
    loose = np.zeros(n, np.uint8)
    pieces(n, n2, 4, tv.ravel(), c[0].ravel(), c[1].ravel(), c[2].ravel(), *each, 0, inn.ravel(), may.ravel(), loose)
    r = np.arange(n2, dtype=np.uint32)
    inn, may = (((m[..., None] >> r) & 1).astype(bool) for m in (inn, may))
    cc = np.empty((n, n2, n2, n2, 3), np.float32)
    cc[..., 0], cc[..., 1], cc[..., 2] = c[0][:, None, :, None], c[1][:, :, None, None], c[2][:, None, None, :]
    big = np.broadcast_to(tv[:, None, None, None], (n, n2, n2, n2, 9)).reshape(-1, 9)
    hit = orc.tri_box(cc.reshape(-1, 3), np.broadcast_to(h, (len(big), 3)), big).reshape(inn.shape).astype(bool)
    assert not np.any(inn & ~hit) and not np.any(hit & ~may)
    assert hit.sum() > 500
    points = (tv.reshape(n, 3, 3) == tv.reshape(n, 3, 3)[:, :1]).all((1, 2))
    assert not np.any(loose[~points])
    assert (may & ~inn)[~points].sum() < 0.1 * hit.sum()


@pytest.mark.parametrize("which", [0, 1, 2])
def test_columns_of_segments(rows, gv, orc, which):  # noqa: F811
    rng = np.random.default_rng(530 + which)
    bmin, bmax = np.float32([-0.3, 0.1, -0.6]), np.float32([0.6, 0.9, 0.3])
    info = gv.grid_derive(bmin, bmax, 0.9, 64, 1)
    nn, g1 = np.array(list(info.n)), np.array(list(info.g), np.float32)
    tabs = [gv.grid_centers(info, 0, a) for a in range(3)]
    idx = np.stack([rng.integers(0, nn[a], 300) for a in range(3)], 1)
    tv = _segments(rng, bmin + (idx + 0.5) * g1.astype(float), 3 * g1.astype(float), which)
    lo, hi = _index_box(tv, bmin, bmax, nn)
    dd = np.maximum(hi - lo + 1, 0)
    keep = (dd > 0).all(1) & (dd.prod(1) < 40000)
    tv, lo, dd = (np.ascontiguousarray(x[keep], t) for x, t in ((tv, np.float32), (lo, np.int32), (dd, np.int32)))
    at = np.concatenate([[0], np.cumsum(dd[:, 0].astype(np.int64) * dd[:, 1])]).astype(np.int64)
    out = np.zeros((at[-1], 4), np.int32)
    rows.columns(len(tv), tv.ravel(), lo.ravel(), dd.ravel(), *tabs, bmin, bmax, g1, at, out.ravel())
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
    assert not np.any(inn & ~hit) and not np.any(hit & ~may)
    assert hit.sum() > 1000
    assert (may & ~inn).sum() < 0.1 * hit.sum()
