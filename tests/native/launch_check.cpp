// Host harness for launch sizes (gpview_amd/csrc/gpv_internal.hpp):
// tests/test_launch_sizes.py checks them against what the kernels index.  Test
// tooling only.
#include "gpv_internal.hpp"

#include <type_traits>

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

// Whether kernels get a batch's table of offsets read-only, with nothing in it that
// is known only after the boundary scan: kernels of both streams read it.
template <typename T, typename = void>
struct has_ranks : std::false_type {};
template <typename T>
struct has_ranks<T, std::void_t<decltype(T::b0)>> : std::true_type {};
extern "C" int offsets_are_fixed()
{
    using Entry = std::remove_pointer_t<decltype(gpv::Meshes::off)>;
    return std::is_const<Entry>::value && !has_ranks<Entry>::value;
}

// how many of the fields that the autotuner sweeps do not try the default
extern "C" int sweeps_without_default()
{
    int bad = 0;
    for (const gpv::TuneField& f : gpv::kTuneSweep) {
        bool found = false;
        for (int k = 0; k < f.n; ++k) found = found || f.values[k] == gpv::kTuneDefault.*f.field;
        bad += found ? 0 : 1;
    }
    return bad;
}
