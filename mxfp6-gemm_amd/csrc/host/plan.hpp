// Internal declarations of the host plan (router, split-K planner, checks).
#pragma once
#include <cstddef>
#include <cstdint>

#include "mxfp6/gemm.hpp"

namespace mxfp6 {
namespace plan {

// Compute units the router plans for when the HIP runtime reports no device (a host without a
// GPU): MI355X's 256 (8 XCDs x 32 CUs). On a device the count is read from it (plan.cpp).
constexpr int DEFAULT_CUS = 256;
// Plan-time model of the router (plan.cpp): fitted on MI355X measurements, microseconds.
constexpr int SPLIT_CHOICES[] = {1, 2, 3, 4, 6, 8, 12, 16};  // K segments considered
constexpr double T_LAUNCH = 2.40452;       // one kernel launch (and its ramp), back to back
constexpr double T_WG = 0.806055;           // fixed cost of one workgroup
constexpr double T_SLAB_MIN = 0.183313;      // latency floor of one 64-wide K slab
constexpr double T_MFMA = 0.00394993;        // per MFMA per wave per slab, per workgroup on the busiest CU
constexpr double T_COPY_KB = 0.0165642;      // per KiB copied global->LDS per slab, per workgroup
constexpr double T_BREG_KB = 0.00831597;     // per KiB of B loaded into registers per slab (wide tiles)
constexpr double T_L2_KB = 7.1085e-05;     // per KiB per slab of every workgroup in flight (L2 -> CUs)
constexpr double T_OUT_KB = 0.0216756;      // per KiB of output (FP16 tile or FP32 partial) per workgroup
constexpr double REPACK_BYTES_PER_US = 5.5e6;        // A repack traffic (measured kernel rate)
constexpr double SPLIT_BYTES_PER_US = 4059650.0;   // split-K partials written and read back
constexpr double A_ROWS_COST = 0.572519;    // extra copy cost per byte of a row-major A slab
constexpr double A_ROWS_COST_WIDE = 0.0675946;  // the same for the wide tiles' K-tile chunks
constexpr double A_ROWS_LONG = 0.158036;    // more per doubling of Kp past 8192 (row-major A)
constexpr double PLAN_MIN_GAIN = 0.01;     // lead a more complex plan needs over a simpler one
// An unsplit plan on a wide tile writes D with nontemporal stores by what it reads (operands, scales, the
// repacked A: "in", at most MI355X's 256 MiB last-level cache) and writes ("out"):
//   in + out > STREAM_FOOTPRINT_BYTES: D no longer evicts the operands the tiles re-read (6-22% faster,
//   8192x16384x2048, 4096x51200x1024, 16384x16384x4096, 1024x102272x2048, 2048x102272x1024; no
//   difference once the operands alone exceed the cache, 2048x102272x4096), and a kernel that reads D next
//   would not find it cached either (the pair 5-10% faster on 8192x16384x2048 and 4096x28672x4096);
//   16-bit D, in + out from half the cache to STREAM_MID_BYTES, D no less than STREAM_MID_RATIO of in: two
//   such calls in a row no longer fit the cache together, and the plain stores of one wait for the other's
//   D to be written back. profiles/gemm_d_stores_with_a_reader.txt, 17 to 25 shapes, streamed against plain:
//   the GEMM alone takes 0.88 times as long where operands and D rotate (8192x8192x1024 86.6 -> 70.2 us,
//   8192x8192x4096 202.9 -> 175.4), 0.94 where D is one buffer (0.83-1.04), and with a kernel after it that
//   reads D and writes as much 0.965 and 0.98 (0.92-1.04). A kernel that only reads D gives the gain back:
//   0.985 where D rotates, 1.065 where it is one buffer (8192x8192x1024 97.2 -> 113.2). The ratio
//   keeps out the plans that run as 128-row bands (tile_dispatch.hpp), whose D is small. STREAM_MID_BYTES is
//   not where the gain ends: from there to STREAM_FOOTPRINT_BYTES streaming measured 0.87 alone and 0.95 with
//   a kernel that reads and writes (8192^3 346.2 -> 329.6 and 388.3 -> 380.2; only reading, 370.7 -> 378.3);
//   plain stores have stayed there but for D of at least STREAM_D_RATIO times in (short K: 8192x14336x512
//   96.5 -> 84.9).
// D whose rows are no whole number of cache lines, or that does not begin on one, is never streamed: a store past
// the caches writes a part of a line, and the memory has to merge it. Streamed against plain
// (profiles/gemm_d_stores_by_row_alignment.txt, 280 shapes), odd N: 1.05-2.96 times as long below 280 MB
// (2091 x 23035 x 2218 159.7 us against 119.6) and 1.00-2.86 above; even N 0.80-2.46 and 0.77-2.49, 1.2 and
// 1.3 on average; whole lines 0.91. Tiles of an odd number of blocks a wave (128x384) store the last one's
// rows as half lines: below 280 MB 0.90-1.02 alone on average and 1.04-1.09 with a reader that writes, so not
// there.
// FP32 D up to STREAM_FOOTPRINT_BYTES is stored the ordinary way: what reads it next is prepare_a, and the pair
// is 3-8% slower with D streamed (4096x8192x2048 96.7 -> 105.5 us, one D 85.6 -> 100.1), as the GEMM alone
// is where D is one buffer (60.2 -> 71.1).
constexpr double LLC_BYTES = 268435456.0;
constexpr long STREAM_LINE_BYTES = 128;
constexpr double STREAM_FOOTPRINT_BYTES = 280e6;
constexpr double STREAM_MID_BYTES = 236e6;
constexpr double STREAM_MID_RATIO = 0.4;
constexpr double STREAM_D_RATIO = 8.0;

TileChoice route(int M, int N, int Kp);
int splitk_segments(int M, int N, int Kp);
size_t workspace_bytes(int M, int N, int Kp);
size_t preferred_workspace_bytes(int M, int N, int Kp);
bool route_repacks(int M, int N, int Kp);
bool streams_output(int out_type, int M, int N, int Kp, const TileChoice& tc, int S, bool repack,
                    int A_row_bytes);
int tune(int out_type, int M, int N, int Kp, const void* dA, const void* dBsh, const uint8_t* dsA,
         const uint8_t* dsB, void* dD, int A_row_bytes, void* ws, size_t ws_bytes,
         int candidates, void* stream, int tile_out[4], int* splits_out, int* repack_out);
int tuned(int out_type, int M, int N, int Kp, int tile_out[4], int* splits_out, int* repack_out);
void tune_reset();
int tune_save(const char* path, int* count);
int tune_load(const char* path, int* loaded, int* skipped);
int plan_info(int out_type, int M, int N, int Kp, size_t ws_bytes, int tile_out[4],
              int* splits_out, int* repack_out);
size_t plan_bytes(int M, int N, int Kp, int S, bool repack);
int check_common(int out_type, int M, int N, int Kp, const void* dA, const void* dBsh,
                 const void* dsA, const void* dsB, const void* dD, int A_row_bytes);
const char* status_text(int st);

}  // namespace plan
}  // namespace mxfp6
