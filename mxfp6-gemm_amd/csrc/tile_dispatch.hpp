// Which kernel a descriptor's tile plan (MXFP6_KERNEL_TILE) runs on, and as how many computing waves.
// Plain C++: the HIP launch code acts on it and the host plan answers mxfp6_plan_kernel from it, so
// that the query and the launch cannot differ. Every kernel gives the plan's bits; the rules below are
// about time. The sweeps they cite are on MI355X (256 CUs), operands of several sets in turn so that
// none is still cached from the call before.
#pragma once
#include "hip_layer.h"
#include "mxfp6_gemm.h"

namespace mxfp6_dispatch {

struct TileRun {
    int kernel;   // mxfp6_tile_kernel
    int waves;    // computing waves of a workgroup (STREAM, BAND), else 0
    bool nt_b;    // STREAM, BAND: B loaded nontemporally
};

inline long ceil_div(long a, long b) { return (a + b - 1) / b; }

inline double b_bytes(const mxfp6_launch_desc& d) { return (double)d.N * (d.Kp / 4 * 3); }

constexpr double LLC_HALF = 128.0 * (1 << 20);  // half of MI355X's 256 MiB last-level cache

// The skinny tile's workgroups against the rounds of the CUs that 128 x 256 wide tiles would take: the
// workgroups a CU of the skinny tile in the time of a round of wide ones.
inline double skinny_rounds(const mxfp6_launch_desc& d, long cus) {
    const long tile = ceil_div(d.M, d.MT) * ceil_div(d.N, d.NT) * d.splits;
    const long wide = ceil_div(d.M, 128) * ceil_div(d.N, 256) * d.splits;
    return (double)tile / (double)(cus * ceil_div(wide, cus));
}

// Whether a skinny tile's plan (32 or 64 rows) on row-major A runs on 128 x 256 wide tiles with the
// skinny tile's scale groups: by the work of the busiest CU. A round of wide workgroups takes as long
// as 1.1 (64 x 256), 1.4 (32 x 256) or 2 (the 128-column tiles) of the skinny tile's workgroups a CU,
// and a wide workgroup counts as much when few of its 128 rows exist; so the wide tiles have to
// replace that many times their own number of workgroups. In profiles/skinny_tiles_on_row_major_a.txt
// (539 routed plans) the rule's pick is 1.0% slower than the better of the two on average and 1.37x at
// worst (448 x 5760 x 16320 in 3 segments, stream 102.8 us, wide 74.9). One tile row never goes wide
// (32 x 32768 x 1024: stream 9.3 us, wide 15.2; 64 x 32768 x 8192: 41.3 and 64.8), many rows do (2784
// x 2304 x 11392: stream 142.8, wide 79.9). `one` K-tile a segment, on 32 x 128: from 4.2 (slab 13.2 us,
// wide 14.1 at 3.97, 608 x 13696; 16.0 and 14.4 at 4.8, 3168 x 3200).
// Rows whose 128 offsets pass 32 bits stay on the tile's own kernel.
inline bool skinny_runs_wide(const mxfp6_launch_desc& d, long cus, bool one) {
    const double least = d.NT == 256 ? (d.MT == 64 ? 1.1 : 1.4) : one && d.MT == 32 ? 4.2 : 2.0;
    return skinny_rounds(d, cus) > least && 127.0 * d.A_row_bytes < 2147483648.0;
}

// Whether a skinny tile's plan of one K-tile a segment that does not go wide runs on the slab kernel: the
// stream kernel loads two ahead. 64 x 128 (slab 4.1-4.9 us, stream 4.6-5.6 on 10 plans) and 64 x 256 on no more
// workgroups than CUs (four waves; 5.2-6.6 against 5.5-7.1), on more where no block is masked (10.5 and 11.7 at
// 832 x 9472; masked 10.4 and 9.3 at 832 x 5248); 32 x 128 on more than two workgroups a CU (7.3 and 8.1 at
// 1120 x 3712; to two within 5% either way). From two K-tiles on the stream kernel is as fast or
// faster (profiles/skinny_tiles_short_k.txt).
inline bool one_k_tile_on_slab(const mxfp6_launch_desc& d, long cus, int waves) {
    if (d.MT == 64) return d.NT == 128 || waves == 4 || (d.M % 64 == 0 && d.N % 256 == 0);
    return d.NT == 128 && skinny_rounds(d, cus) > 2.0;
}

// Computing waves of a stream workgroup (four as the router counts the tile): fewer where four would
// leave CUs idle or load them unevenly.
//   one 32-column block a wave (NT 128): two waves below 3/5 of the CUs, and on 32 rows one where two
//   stay below that as well (32 x 384 x 12928 in 16 segments, 48 workgroups of four: four 1.13x, two
//   1.04x, one 1; 16 x 1024 x 10880, 128: four 1.11x, two 1);
//   two blocks a wave: two waves on more workgroups than CUs, which four waves' registers run one round
//   at a time (96 x 23552 x 2112, 276 workgroups: four 1.25x two; 2240 x 2176 x 576, 315: 1.21x; on
//   144-256 workgroups four are 0-12% faster).
inline int stream_waves(const mxfp6_launch_desc& d, long cus, bool nt_b) {
    auto wgs = [&](int waves) {
        return ceil_div(d.M, d.MT) * ceil_div(d.N, d.NT / 4 * waves) * d.splits;
    };
    if (d.NT != 128) return wgs(4) > cus && !nt_b ? 2 : 4;
    if (d.MT == 32 && 5 * wgs(2) < 3 * cus) return 1;
    return 5 * wgs(4) < 3 * cus ? 2 : 4;
}

// Computing waves of the 128-row bands that run a wide tile's plan on row-major A, or 0 where the wide
// kernel is the better one: the fewest with which the plan's workgroups run in one round of the CUs. On 110
// routed plans drawn at random the bands were 1.09-1.60x as fast as the wide kernel
// (profiles/bands_against_wide_tiles.txt: three waves 1.44x on average, four 1.32x, five 1.19x). Five only
// where B is no small part of the 256 MiB last-level cache (57 MB 1.03-1.08x unsplit, 0.90 split; 75 MB 1.29x,
// 126 MB in two segments 1.18x, 170 MB 1.32x; 28 MB 0.91, 42 MB 1.00), for there the wide kernel's loads, one
// K-tile ahead, wait on HBM; six lost but for one shape (682 x 1280 x 27520 in 6 segments 0.76, 256 x 7040 x
// 9920 in 3 0.89; 128 x 6016 x 18944 in 8 1.15x). Segments of fewer than eight K-tiles keep the wide
// kernel, which has short paths for them.
inline int band_waves(const mxfp6_launch_desc& d, long cus) {
    if (d.a_layout != MXFP6_A_ROWS || d.out_stream || d.Kp / 192 < 8 * d.splits) return 0;
    const long rows = ceil_div(d.M, 128) * d.splits, blks = ceil_div(d.N, 32);
    const int most = b_bytes(d) > LLC_HALF / 2 ? 5 : 4;
    for (int waves = 2; waves <= most; waves++)
        if (rows * ceil_div(blks, waves) <= cus) return waves;
    return 0;
}

// Wide tiles: four waves side by side, A's scale groups of four row blocks.
inline bool is_wide(const mxfp6_launch_desc& d) {
    return d.mpw == 4 && (d.NT == 512 || d.NT == 384 || (d.NT == 256 && d.npw == 2));
}

// cus: the device's compute units, or 0 where the runtime reports none (an MI355X's 256 then).
inline TileRun tile_run(const mxfp6_launch_desc& d, long cus) {
    if (cus <= 0) cus = 256;
    if (d.MT == 32 && d.NT == 32) return {MXFP6_TILE_TINY, 0, false};
    if (is_wide(d)) {
        const int waves = band_waves(d, cus);
        if (waves == 0) return {MXFP6_TILE_WIDE, 0, false};
        // B read by one workgroup row, and more than half the last-level cache
        return {MXFP6_TILE_BAND, waves, d.M <= 128 && b_bytes(d) > LLC_HALF};
    }
    if (d.MT > 64 || d.a_layout != MXFP6_A_ROWS) return {MXFP6_TILE_SLAB, 0, false};
    const bool one = d.Kp / 192 <= d.splits;  // K-tile a segment
    if (skinny_runs_wide(d, cus, one)) return {MXFP6_TILE_WIDE, 0, false};
    const bool nt_b = d.M <= d.MT && b_bytes(d) > LLC_HALF;
    const int waves = stream_waves(d, cus, nt_b);
    if (one && one_k_tile_on_slab(d, cus, waves)) return {MXFP6_TILE_SLAB, 0, false};
    return {MXFP6_TILE_STREAM, waves, nt_b && waves == 4};
}

}  // namespace mxfp6_dispatch
