// Host harness for launch sizes (gpview_amd/csrc/gpv_internal.hpp):
// tests/test_launch_sizes.py checks them against what the kernels index.  Test
// tooling only.
#include "gpv_internal.hpp"

// the tiles of a counting sort with nkeys keys
extern "C" int64_t tiles_of(uint64_t nkeys) { return (int64_t)gpv::ts_tiles(nkeys); }

// bytes of LDS of the scan launch for sorts of na and nb tiles
extern "C" int64_t scan_lds_bytes(int na, int nb) { return 4 * (int64_t)gpv::ts_scan_lds(na, nb); }

// bytes of LDS that the scan of n tiles touches: tile t lies at word t + (t >> pad)
extern "C" int64_t scan_touched_bytes(int n)
{
    int64_t top = 0;
    for (int t = 0; t < n; ++t) {
        const int64_t at = t + (t >> gpv::ts_pad(n)) + 1;
        top = at > top ? at : top;
    }
    return 4 * top;
}
