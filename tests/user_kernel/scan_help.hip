// The pair scan with blocks that never wait: a tile that is not published yet
// is summed at once by the block that needs it, as in the library after
// kHelpSpins turns.  Built with the package for tests/test_gpu_scan_help.py.
#define NLH_HELP_SPINS 0
#define nlh nlh_scan_help   // symbols of its own beside libnlhip.so's
#include "../../neighbourlists.jl_amd/csrc/kernels.hip"

// Device pointers: counts (n), pair_off (n + 1), first (n + 1, TI), tile_atom
// (2 tile_cap), status, lookback (lookback_entries(1, n)).  Sets *words to the
// number of lookback words when it is given, and launches nothing.
extern "C" int scan_help(const int32_t *counts, int64_t n, int32_t ti_bytes, int64_t *pair_off, void *first,
                         int32_t *tile_atom, int64_t tile_cap, void *status, uint64_t *lookback, int64_t *words)
{
    if (words) {
        *words = nlh::lookback_entries(1, n);
        return 0;
    }
    if (n <= 0 || nlh::scan_tiles(n) > nlh::kLookbackTiles || tile_cap < 2) return 1;
    nlh::PipelineBufs b{};
    b.nsys = 1;
    b.nat = n;
    b.sort.n_sort = 1;
    b.pair_count = const_cast<int32_t *>(counts);
    b.pair_off = pair_off;
    b.first_out = first;
    b.tile_atom = tile_atom;
    b.tile_cap = tile_cap;
    b.fill_pairs = 256;
    b.pair_capacity = INT64_MAX;
    b.status = static_cast<nlh::Status *>(status);
    b.lookback = lookback;
    b.ti_bytes = ti_bytes;
    nlh::launch_clear_pair_lookback(b, nullptr);
    nlh::launch_scan_pairs(b, nullptr);
    if (hipGetLastError() != hipSuccess) return 2;
    return hipDeviceSynchronize() == hipSuccess ? 0 : 3;
}
