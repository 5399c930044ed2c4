"""Where the bytes of a download go (gpview_amd/csrc/gpv_download.hpp), on the host with
stand-ins for the HIP calls; and whole downloads into page-locked memory on the device."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from conftest import ROOT, say

NATIVE = os.path.join(ROOT, "tests", "native")
PAGEABLE, LOCKED, DEVICE = None, 0, 1
SMALL = 256 << 10      # up to this total a download is one launch


class Harness:
    def __init__(self, L):
        self.L, self.d = L, L.dl_new()

    def close(self):
        self.L.dl_delete(self.d)

    def run(self, pieces, no_locked=False, no_events=False):
        """pieces: (bytes, kind of destination, offset of the source); checks the bytes and
        returns the stand-ins' log."""
        L = self.L
        L.dl_reset(int(no_locked), int(no_events))
        rng = np.random.default_rng(len(pieces) + sum(n for n, *_ in pieces))
        src = [rng.integers(0, 256, n + at, np.uint8) for n, _, at in pieces]
        dst = [np.zeros(n + 1, np.uint8) for n, *_ in pieces]
        for d, (n, kind, _) in zip(dst, pieces):
            if kind is not PAGEABLE:
                L.dl_known(d.ctypes.data, n + 1, kind)
        arr = lambda v: (ctypes.c_void_p * len(v))(*v)
        log = np.zeros(6, np.int64)
        n = np.array([p[0] for p in pieces], np.int64)
        r = L.dl_run(self.d, len(pieces), arr([d.ctypes.data for d in dst]),
                     arr([s.ctypes.data + at for s, (_, _, at) in zip(src, pieces)]), n.ctypes.data, log.ctypes.data)
        assert r == 0
        for d, s, (k, _, at) in zip(dst, src, pieces):
            assert np.array_equal(d[:k], s[at:]) and d[k] == 0
        out = dict(zip(("kernels", "kernel_bytes", "copies", "copy_bytes", "waits", "error"), log.tolist()))
        assert out["waits"] > 0 and out["error"] == 0
        assert out["kernel_bytes"] + out["copy_bytes"] == n.sum()
        return out


@pytest.fixture
def down():
    so = os.path.join(NATIVE, "libdownload.so")
    if not os.path.exists(so):
        subprocess.run(["make", "-s", "-C", NATIVE, so], check=True)
    L = ctypes.CDLL(so)
    vp, i = ctypes.c_void_p, ctypes.c_int
    L.dl_new.restype = vp
    L.dl_delete.argtypes = [vp]
    L.dl_known.argtypes = [vp, ctypes.c_int64, i]
    L.dl_reset.argtypes = [i, i]
    L.dl_run.argtypes = [vp, i, vp, vp, vp, vp]
    h = Harness(L)
    yield h
    h.close()


@pytest.mark.parametrize("n", [SMALL + 1, 3 << 20, (40 << 20) + 13])
def test_page_locked_destinations_are_written_once(down, n):
    """Larger results go straight into page-locked memory; the rest of the same call
    by the staging."""
    log = down.run([(n, LOCKED, 0)])
    assert log["copy_bytes"] == n and log["kernels"] == 0
    log = down.run([(n, LOCKED, 4), (n + 5, PAGEABLE, 0), (0, LOCKED, 0), (777, LOCKED, 8)])
    assert log["copy_bytes"] == n + 777 and log["kernel_bytes"] == n + 5
    log = down.run([(n, PAGEABLE, 0)])
    assert log["kernel_bytes"] == n


@pytest.mark.parametrize("n", [1, 4096, SMALL, SMALL + 1, 5 << 20])
def test_device_destinations_are_never_written_by_the_host(down, n):
    assert down.run([(n, DEVICE, 0)])["copy_bytes"] == n
    log = down.run([(100, PAGEABLE, 0), (n, DEVICE, 0), (50, LOCKED, 0)])
    assert log["copy_bytes"] >= n


@pytest.mark.parametrize("what", ["no_locked", "no_events"])
@pytest.mark.parametrize("n", [100, SMALL, SMALL + 1, 5 << 20])
def test_downloads_without_staging(down, n, what):
    """No page-locked memory or no events left: the download still arrives, leaves no error
    behind, and the next one has its staging again."""
    pieces = [(n, PAGEABLE, 0), (n // 2, PAGEABLE, 4)]
    log = down.run(pieces, **{what: True})
    assert log["copy_bytes"] in (0, n + n // 2)
    assert down.run(pieces)["kernel_bytes"] == n + n // 2


@pytest.mark.gpu
@pytest.mark.parametrize("l1,n2", [(8, 4), (40, 5), (100, 3)])
def test_page_locked_download(gv, l1, n2):
    """Every product into page-locked arrays equals the one into ordinary arrays, alone and
    for batch members, whose arrays begin at any element."""
    from gpview_amd import workloads
    say(f"page-locked download {l1}/{n2}")
    ms = [dict(workloads.mesh_entry(gv, *gv.mixed(k, 1500 + 700 * k, 80 + k), l1 + 3 * k, n2), normals=True) for k in range(3)]
    with gv.Context() as c:
        m = ms[0]
        grids = [c.voxelize(m["soup"], m["bmin"], m["bmax"], m["mms"], l1, n2, normals=True)] + c.voxelize_batch(ms)
        for g in grids:
            d, (l1n, l2n) = g.download(), g.download_normals()
            want = [d["l1"], d["prefix"], d["bidx"], d["l2"], l1n, l2n, *g.download_bits()]
            locked = [gv.PinnedArray((max(w.size, 1),), w.dtype) for w in want]
            p = [a.array.ctypes.data for a in locked]
            L = gv.lib()
            assert L.gpv_grid_download(c.h, g.h, *p[:4]) == 0
            assert L.gpv_grid_download_normals(c.h, g.h, *p[4:6]) == 0
            assert L.gpv_grid_download_bits(c.h, g.h, *p[6:]) == 0
            for k, (w, a) in enumerate(zip(want, locked)):
                assert np.array_equal(a.array[:w.size], w.ravel()), f"array {k}"
            for a in locked:
                a.close()
            g.release()
