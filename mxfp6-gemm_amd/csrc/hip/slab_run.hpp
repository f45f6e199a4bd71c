// Declarations of the tile kernel's launch entry (definitions in slab_kernel.hpp). The launch
// code of each kernel output type is compiled in a translation unit of its own (slab_split.hip,
// slab_f32.hip, slab_f16.hip, slab_bf16.hip), so the instantiations build in parallel and
// launch.hip compiles none of them.
#pragma once
#include "../hip_layer.h"
#include "device_common.hpp"

namespace mxfp6_dev {

// (MT, NT, MPW, NPW) -> wave grid: the scale grouping fixes how many 32-blocks one wave holds,
// so it also selects between the 4-wave and 8-wave instantiation of a tile.
inline bool tile_supported(int MT, int NT, int mpw, int npw) {
    return (MT == 32 && NT == 32 && mpw == 1 && npw == 1) ||  // tiny_kernel.hpp (launch.hip)
           (MT == 32 && NT == 128 && mpw == 1 && npw == 1) ||
           (MT == 32 && NT == 256 && mpw == 1 && npw == 2) ||
           (MT == 64 && NT == 128 && mpw == 2 && npw == 1) ||
           (MT == 64 && NT == 256 && mpw == 2 && npw == 2) ||
           (MT == 128 && NT == 128 && mpw == 2 && npw == 2) ||
           (MT == 128 && NT == 256 && mpw == 2 && npw == 4) ||
           (MT == 128 && NT == 384 && mpw == 4 && npw == 3) ||
           (MT == 128 && NT == 512 && mpw == 4 && npw == 4) ||
           (MT == 128 && NT == 256 && mpw == 4 && npw == 2) ||
           (MT == 256 && NT == 256 && mpw == 4 && npw == 2) ||
           (MT == 256 && NT == 256 && mpw == 4 && npw == 4) ||
           (MT == 256 && NT == 192 && mpw == 4 && npw == 3) ||
           (MT == 256 && NT == 256 && mpw == 2 && npw == 4);
}

// Whether a skinny tile's plan (32 or 64 rows) runs faster on 128 x 256 wide tiles reading row-major A
// with the skinny tile's scale groups. Three operand sets in turn:
//   plans that would repack A first: every one of 31 measured, from 108 wide workgroups on,
//   1.22-2.55x (3616 x 17024 x 4096, M an odd number of 32-row blocks: 512.7 -> 266.4 us; 5216 x 2688 x
//   14464 507.2 -> 198.5; 576 x 8192 x 6016 59.7 -> 34.1);
//   plans on row-major A (stream kernel): from half as many workgroups as CUs, unless the last of
//   several rounds leaves the CUs more than two fifths idle in all: 15 of 15 faster, 1.09-2.84x
//   (4128 x 1024 x 6653, 132 workgroups: 55.6 -> 38.3; 3264 x 1408 x 6590, 156: 50.4 -> 38.3; 288 x
//   2560 x 30656 in 8 segments, 240: 87.6 -> 30.9); below that 78 of 81 slower (192 x 12288 x 3072,
//   96: 0.76, 320 x 25600 x 292, 300: 0.84).
inline bool skinny_runs_wide(int M, int N, int splits, bool repack) {
    const int reported = mxfp6_hip_device_cus();
    const long cus = reported > 0 ? reported : 256;
    const long wgs = (long)((M + 127) / 128) * ((N + 255) / 256) * splits;
    if (repack) return 5 * wgs >= 2 * cus;
    return 2 * wgs >= cus && (wgs <= cus || 5 * wgs >= 3 * ((wgs + cus - 1) / cus * cus));
}

// Runs the descriptor's plan on the tile kernel (after the A repack when a_layout asks for it):
// KT = the kernel's output type, SPLIT = FP32 partials of d->splits K segments into d->ws (KT =
// float). Returns 0, 1 when no instantiation matches the tile, 2 when a launch fails.
template <typename KT, bool SPLIT>
int slab_run(const mxfp6_launch_desc* d, hipStream_t st);

extern template int slab_run<float, true>(const mxfp6_launch_desc*, hipStream_t);
extern template int slab_run<float, false>(const mxfp6_launch_desc*, hipStream_t);
extern template int slab_run<__half, false>(const mxfp6_launch_desc*, hipStream_t);
extern template int slab_run<__hip_bfloat16, false>(const mxfp6_launch_desc*, hipStream_t);

}  // namespace mxfp6_dev
