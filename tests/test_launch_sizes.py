"""Launch sizes against what the kernels index, on the host
(gpview_amd/csrc/gpv_internal.hpp)."""
import ctypes
import os
import subprocess

import pytest

from conftest import ROOT

NATIVE = os.path.join(ROOT, "tests", "native")


@pytest.fixture(scope="module")
def launch():
    so = os.path.join(NATIVE, "liblaunch.so")
    if not os.path.exists(so):
        subprocess.run(["make", "-s", "-C", NATIVE, so], check=True)
    L = ctypes.CDLL(so)
    L.tiles_of.argtypes, L.tiles_of.restype = [ctypes.c_uint64], ctypes.c_int64
    L.scan_lds_bytes.argtypes, L.scan_lds_bytes.restype = [ctypes.c_int] * 2, ctypes.c_int64
    L.scan_touched_bytes.argtypes, L.scan_touched_bytes.restype = [ctypes.c_int], ctypes.c_int64
    return L


# keys of a sort: none, a tile or so, the largest with one shift and the first with the
# next, just above 2^26 (more than 8192 tiles), the most that a run takes
KEYS = [0, 1, 256, 257, 65536, 2097152, 2097153, 16700000, 16777216, 2 ** 26 - 8192, 2 ** 26, 2 ** 26 + 1, 8200 * 8200,
        100000000, 2 ** 27]


def test_tile_scan_fits_its_lds(launch):
    """Both sorts of a launch share its LDS: neither scan reaches past it."""
    tiles = sorted({launch.tiles_of(k) for k in KEYS} | set(range(8160, 8225)))
    assert tiles[0] == 0 and tiles[-1] == 16384 and 8209 in tiles
    need = {t: launch.scan_touched_bytes(t) for t in tiles}
    bad = [(a, b) for a in tiles for b in tiles if max(need[a], need[b]) > launch.scan_lds_bytes(a, b)]
    assert not bad, f"{len(bad)} pairs of tile counts, the first {bad[0]}"
    assert max(launch.scan_lds_bytes(a, b) for a in tiles for b in tiles) <= 65536


def test_batch_offsets_are_fixed(launch):
    """The Level1 parity reads the offsets on its own stream while the boundary scan and
    the group plan of the main one write theirs: not into the same table."""
    assert launch.offsets_are_fixed() == 1


def test_autotuner_tries_the_defaults(launch):
    """From any shapes set by hand the autotuner can come back to the default ones."""
    assert launch.sweeps_without_default() == 0
