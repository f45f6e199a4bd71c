// Stream kernels of libmxfp6gemm for gfx950: the skinny tiles (32 and 64 rows) and, on small grids, the
// wide tiles (as 128-row bands) on row-major A, B read straight into registers.
//
// A workgroup computes an MT x NT tile of D with MT = 32 MB and NT = 32 NPW WN: WN computing waves
// side by side, each owning all MT rows and 32 NPW columns, and one copying wave. (MB, NPW) is the
// tile's scale grouping: 32 x 128 (1, 1), 32 x 256 (1, 2), 64 x 128 (2, 1), 64 x 256 (2, 2); WN does
// not change the arithmetic of a wave, so the output bits are the tile's for every WN.
//   B       each computing wave loads its own blocks from the preshuffled layout into MFMA operand
//           registers, L = 2 K-tiles ahead (per 64-wide slab and block a 16- and an 8-byte load a
//           lane, contiguous), and its scales with them; a slab's loads for K-tile c + L are issued
//           right after the MFMAs that read K-tile c's.
//   A       chunks of CK = 2 K-tiles, copied by the copying wave along the rows (a row's 288 bytes
//           are 3.1 cache lines on average, where two K-tile pieces of 144 bytes take 4) into a
//           ring of NB = 3 LDS buffers, rows 304 bytes apart (16-byte pieces, one of padding), with
//           the A scales of the chunk (one 12-byte copy a K-tile). A computing wave reads K-tile
//           c + 1 from LDS into the other of two register sets while it multiplies K-tile c.
//   sync    one workgroup barrier per chunk: the copying wave has waited for chunk g + 1 (its own
//           vmcnt count: it issues nothing else), every computing wave for its reads of chunk g,
//           whose buffer then takes chunk g + NB.
// What bounds it: the read requests a CU keeps in flight, about a hundred of at most 128 bytes, whether
// they go to registers or to LDS (104 a CU on 64 x 28672 x 8192 and 93 on the bands of 256 x 18432 x 12288
// by the counters, profiles/stream_kernel_*_pmc.txt; MFMAs busy 8 and 18% of the cycles): 64 x 8192 x 8192
// on 64 CUs moved 29 KB/us a CU from HBM and 48 from the Infinity Cache, the same with 2, 4 or 6 K-tiles
// of loads ahead. So lead past two K-tiles is worth nothing; the lines of A, the padded scale dwords and
// the number of CUs in use are what counts. That is why A comes in two K-tiles per row piece, only one wave
// loads A's scales, and WN shrinks when the grid is small (tile_dispatch.hpp). 64 x 28672 x 8192 (three
// operand sets in turn, B from HBM): 52.1 us on the slab kernel (B and A through LDS a slab at a time,
// every wave copying), 38.2 here: 5.0 TB/s of operands; without A's copies and scales 30.5.
// NT: B's loads are nontemporal where B exceeds half the last-level cache and is read by one tile row. A
// layer's weights are read again only after the other layers': with three or more sets in turn 24 plans
// of 140-271 MB of B are 7-15% faster so (64 x 28672 x 8192 43.4 -> 38.0 us, 32 x 28672 x 6400 34.4 ->
// 30.9), and prepare_b followed by the GEMM 4-7%. The same B again at once loses what the cache would
// have kept (140-212 MB: 3-26%, 64 x 28672 x 8192 32.4 -> 36.9; 64 x 8192 x 8192, B 50 MB: 20.9 -> 31.4;
// from 240 MB on 0-8%).
// BAND (WN = 0 in the template; 128 rows, scale groups of four row blocks): a wave owns 128 rows and
// one 32-column block, byte blk % npw of its scale group of npw blocks, so that the launch can
// choose how many columns a workgroup takes (2 to 5 computing waves, all in one round of the CUs)
// whatever the tile: same bits as the wide kernel's tiles of that grouping. Two copying waves share
// a chunk's copies, and the A operands are read a slab ahead (a K-tile's would not fit the
// registers). Against the wide kernel on a grid that leaves CUs idle each CU in use has fewer cache
// lines to fetch: per K-tile 26 KB of A and 5.4 KB a wave, where a 128 x 256 tile takes 76 KB
// (256 x 18432 x 12288, 144 workgroups of 128 x 256 or 232 of five waves: 88.1 -> 66.6 us).
// MASK (ragged M or N): rows past M repeat the last one, blocks and scale groups past the end the last
// that exists; stores are masked.
#pragma once

#include "../tile_dispatch.hpp"
#include "device_common.hpp"
#include "epilogue.hpp"
#include "lds_dma.hpp"
#include "wide_kernel.hpp"

namespace mxfp6_dev {

template <int MB_, int NPW_, int WN_>
struct StreamGeom {
    static constexpr int MB = MB_, NPW = NPW_, WN = WN_;
    static constexpr bool BAND = WN == 0;                       // WN given by the launch
    static constexpr int NCW = BAND ? 2 : 1;                    // copying waves
    static constexpr int MAXWN = BAND ? 5 : WN;
    static constexpr int L = 2;                                 // K-tiles of B in flight
    static constexpr int CK = 2;                                // K-tiles of A a chunk
    static constexpr int NB = 3;                                // chunk buffers
    static constexpr int MT = 32 * MB, NT = 32 * NPW * WN;
    static constexpr int THREADS = 64 * (MAXWN + NCW);
    static constexpr int ROW = 9 * CK + 1;                      // 16-byte LDS pieces a row, one of padding
    static constexpr int PIECES = MT * ROW;
    static constexpr int COPIES = (PIECES + 63) / 64;           // wave copies of a chunk's rows
    // operations of a copying wave for a chunk: its rows' copies and one of a K-tile's scales
    static constexpr int OPS = (COPIES + CK) / NCW;
    static constexpr int CST = (COPIES + CK) * 1024;            // LDS buffer stride
    static constexpr int LDS = NB * CST;
    static constexpr int PASS = 2;                              // K-tiles of a pass of the K loop
    static_assert(PASS % CK == 0 && PASS % L == 0 && PASS % 2 == 0, "ring positions are constants");
    static_assert(COPIES % NCW == 0 && CK % NCW == 0, "copies shared evenly");
    static_assert((NB - 1) * OPS <= 63, "vmcnt range");
    static_assert(LDS <= 160 * 1024, "LDS budget");
};

// f(T), f(T + 1), ... for the first `left` of the PASS positions (left < PASS).
template <int T, int PASS, typename F>
__device__ __forceinline__ void stream_tail(int left, F&& f) {
    if constexpr (T + 1 < PASS) {
        if (left > 0) {
            f(std::integral_constant<int, T>{});
            stream_tail<T + 1, PASS>(left - 1, f);
        }
    }
}

template <int MB_, int NPW_, int WN_, int XG, typename OutT, bool SPLIT, bool MASK, bool NTB>
__global__ void __launch_bounds__(64 * (WN_ == 0 ? 7 : WN_ + 1), 1)
    stream_kernel(const uint8_t* __restrict__ A, const uint8_t* __restrict__ Bsh,
                  const uint8_t* __restrict__ sA, const uint8_t* __restrict__ sB,
                  OutT* __restrict__ D, float* __restrict__ ws, int M, int N, int Kp,
                  int A_row_bytes, int S, int npw) {
    using G = StreamGeom<MB_, NPW_, WN_>;
    constexpr int MT = G::MT, MB = G::MB, NPW = G::NPW, NCW = G::NCW, L = G::L;
    constexpr int CK = G::CK, NB = G::NB;
    constexpr int AUX = NTB ? 2 : 0;  // cache policy of the B loads (2: nontemporal)
    __shared__ __attribute__((aligned(1024))) char lds[G::LDS];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int wg_m = blockIdx.x, wg_n = blockIdx.y, wg_z = SPLIT ? (int)blockIdx.z : 0;
    if constexpr (XG > 0) {
        const int gm = (int)gridDim.x, gn = (int)gridDim.y;
        if (!SPLIT || (gm * gn) % NXCD == 0)
            xcd_tile(gm, gn, XG, (int)(blockIdx.y * gridDim.x + blockIdx.x), wg_m, wg_n);
    }
    const int k64n = Kp / 64, k_tiles = Kp / 192;
    int kt0 = 0, nkt = k_tiles;
    if (SPLIT) split_segment(k_tiles, S, wg_z, kt0, nkt);
    const int kt_last = kt0 + nkt - 1;

    const int WN = G::BAND ? (int)(blockDim.x >> 6) - NCW : G::WN;

    if (wave >= WN) {
        // the copying wave: copy i moves LDS piece p = 64 i + l of a chunk (16 bytes, lane l) from
        // piece p % ROW of row p / ROW; the padding piece is not copied, nor are the pieces past the
        // segment's end. Every copy has at least one lane to copy, so a chunk is OPS operations.
        const int rows = MASK ? min(MT, M - wg_m * MT) : MT;
        const uint8_t* a_tile = A + (size_t)wg_m * MT * A_row_bytes + (size_t)kt0 * (SUBS * SLAB_BYTES);
        const int cw = wave - WN;  // copies cw, cw + NCW, ...
        uint32_t voff[G::COPIES / NCW];
#pragma unroll
        for (int i = 0; i < G::COPIES / NCW; i++) {
            const int p = (i * NCW + cw) * 64 + lane, row = p / G::ROW, col = p - row * G::ROW;
            voff[i] = p < G::PIECES && col < 9 * CK
                          ? (uint32_t)((MASK ? min(row, rows - 1) : row) * A_row_bytes + 16 * col)
                          : ~0u;
        }
        int ga = wg_m;
        if (MASK) ga = min(ga, ((M + 31) / 32 + MB - 1) / MB - 1);
        const uint8_t* sa_grp = sA + ((size_t)ga * k_tiles + kt0) * 64 * 12;
        const uint32_t lds0 = lds_u32(lds), sc_voff = 12 * lane;
        const int nch = (nkt + CK - 1) / CK;
        auto copy = [&](int ch) {
            const uint8_t* src = a_tile + (size_t)ch * (CK * SUBS * SLAB_BYTES);
            const uint32_t dst = __builtin_amdgcn_readfirstlane(lds0 + ch % NB * G::CST + cw * 1024);
            const int kts = min(CK, nkt - ch * CK);
            if (kts == CK) {
#pragma unroll
                for (int i = 0; i < G::COPIES / NCW; i++)
                    if (voff[i] != ~0u) dma16(dst + i * NCW * 1024, src, voff[i]);
            } else {
#pragma unroll
                for (int i = 0; i < G::COPIES / NCW; i++) {
                    const int col = ((i * NCW + cw) * 64 + lane) % G::ROW;
                    if (voff[i] != ~0u && col < 9 * kts) dma16(dst + i * NCW * 1024, src, voff[i]);
                }
            }
            const uint32_t sdst =
                __builtin_amdgcn_readfirstlane(lds0 + ch % NB * G::CST + G::COPIES * 1024);
            for (int t = cw; t < CK; t += NCW)
                dma12_at<0>(sdst + t * 1024, sa_grp + (size_t)(ch * CK + min(t, kts - 1)) * 768, sc_voff);
        };
        for (int ch = 0; ch < NB && ch < nch; ch++) copy(ch);
        // chunk ch landed, up to NB - 1 newer ones (OPS copies each) in flight
        auto landed = [&](int ch, auto newer) {
            if (ch + decltype(newer)::value < nch)
                wait_vmcnt<decltype(newer)::value * G::OPS>();
            else
                wait_vmcnt0();
        };
        landed(0, std::integral_constant<int, NB - 1>{});
        ring_barrier();
        for (int ch = 0; ch < nkt / CK; ch++) {
            landed(ch + 1, std::integral_constant<int, NB - 2>{});
            ring_barrier();  // chunk ch + 1 landed, chunk ch read by every wave
            if (ch + NB < nch) copy(ch + NB);
        }
        return;
    }

    const int b_blk_last = (N + 31) / 32 - 1;
    rsrc_t b_rs[NPW];
#pragma unroll
    for (int ni = 0; ni < NPW; ni++) {
        int blk = (wg_n * WN + wave) * NPW + ni;
        if (MASK) blk = min(blk, b_blk_last);
        b_rs[ni] = raw_rsrc(opaque_gptr(Bsh + (size_t)blk * k64n * OPBLK_BYTES));
    }
    // the wave's B scale group; BAND: its one block is byte b_shift / 8 of a group of npw blocks
    int gb = wg_n * WN + wave, b_shift = 0;
    if constexpr (G::BAND) {
        const int blk = min(gb, b_blk_last);
        gb = blk / npw;
        b_shift = 8 * (blk - gb * npw);
    } else if (MASK) {
        gb = min(gb, ((N + 31) / 32 + NPW - 1) / NPW - 1);
    }
    const rsrc_t sb_rs = raw_rsrc(opaque_gptr(sB + (size_t)gb * k_tiles * 64 * 12));
    const int v_b0 = (int)opaque_v(16 * lane), v_b1 = (int)opaque_v(1024 + 8 * lane);
    const int v_sc = (int)opaque_v(12 * lane);

    v8i RB[L][SUBS][NPW];  // B operands and scales of K-tile c in slot c % L
    v3i sc_b[L];
    auto load_b = [&](v8i& v, int ni, int kt, int s) {
        const int so = kt * (SUBS * OPBLK_BYTES);
        const v4i y0 = __builtin_bit_cast(
            v4i, __builtin_amdgcn_raw_buffer_load_b128(b_rs[ni], v_b0 + s * OPBLK_BYTES, so, AUX));
        const v2i y1 = __builtin_bit_cast(
            v2i, __builtin_amdgcn_raw_buffer_load_b64(b_rs[ni], v_b1 + s * OPBLK_BYTES, so, AUX));
        const v4i y1w = __builtin_shufflevector(y1, y1, 0, 1, -1, -1);
        v = __builtin_shufflevector(y0, y1w, 0, 1, 2, 3, 4, 5, -1, -1);
    };
    auto load_scales = [&](v3i& b, int kt) {
        b = __builtin_bit_cast(v3i, __builtin_amdgcn_raw_buffer_load_b96(sb_rs, v_sc, kt * 768, AUX));
    };
    const lds_cptr lds3 = (lds_cptr)lds;
    const uint32_t a_rd = (uint32_t)((lane & 31) * G::ROW * 16 + (lane >> 5) * 24);

    v16f acc[MB][NPW];
#pragma unroll
    for (int i = 0; i < MB; i++)
#pragma unroll
        for (int j = 0; j < NPW; j++) acc[i][j] = v16f{};

#pragma unroll
    for (int c = 0; c < L; c++) {
        const int kt = min(kt0 + c, kt_last);
#pragma unroll
        for (int s = 0; s < SUBS; s++)
#pragma unroll
            for (int ni = 0; ni < NPW; ni++) {
                load_b(RB[c][s][ni], ni, kt, s);
                asm volatile("" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
            }
        load_scales(sc_b[c], kt);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    }
    // A operands, two sets: of a K-tile, or (BAND, whose sets are larger) of a slab; A scales of a
    // K-tile, two sets
    constexpr int US = G::BAND ? 1 : SUBS;
    v8i RA[2][US][MB];
    v3i sc_a[2];
    // the A scales of K-tile KT of the chunk in buffer buf to set Q
    auto read_sc = [&](auto qq, auto tt, int buf) {
        constexpr int Q = decltype(qq)::value, KT = decltype(tt)::value;
        sc_a[Q] = *reinterpret_cast<const __attribute__((address_space(3))) v3i*>(
            lds3 + opaque_v(16 * lane + buf * G::CST) + (G::COPIES + KT) * 1024);
    };
    // and the A operands of its slabs s0 .. s0 + US - 1
    auto read_a = [&](auto qq, auto tt, int s0, int buf) {
        constexpr int Q = decltype(qq)::value, KT = decltype(tt)::value;
        const uint32_t base = opaque_v(a_rd + buf * G::CST);
#pragma unroll
        for (int s = 0; s < US; s++)
#pragma unroll
            for (int mi = 0; mi < MB; mi++) {
                const v6i_a8 x = *reinterpret_cast<const __attribute__((address_space(3))) v6i_a8*>(
                    lds3 + base + mi * 32 * G::ROW * 16 + KT * SUBS * SLAB_BYTES + (s0 + s) * SLAB_BYTES);
                RA[Q][s][mi] = __builtin_shufflevector(x, x, 0, 1, 2, 3, 4, 5, -1, -1);
            }
    };
    using I0 = std::integral_constant<int, 0>;
    ring_barrier();
    read_sc(I0{}, I0{}, 0);
    read_a(I0{}, I0{}, 0, 0);
    int buf = 0;
    auto ktile = [&](int c, auto tt) {
        constexpr int T = decltype(tt)::value % L, P = decltype(tt)::value % 2;
        constexpr int KT = decltype(tt)::value % CK, NEXT = (KT + 1) % CK;
        using NextC = std::integral_constant<int, NEXT>;
        using ScC = std::integral_constant<int, 1 - P>;
        // K-tile c + 1 is read from here on: at a chunk's end once it has landed
        auto next_ktile = [&] {
            if constexpr (NEXT == 0) {
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                ring_barrier();
                buf = buf == NB - 1 ? 0 : buf + 1;
            }
            read_sc(ScC{}, NextC{}, buf);
        };
        if constexpr (US == SUBS) {
            next_ktile();
            read_a(ScC{}, NextC{}, 0, buf);
            __builtin_amdgcn_sched_barrier(0);
        }
        const int kt_next = min(kt0 + c + L, kt_last);
        const v3i ca = sc_a[P], cb = sc_b[T];
        static_for<SUBS>([&](auto ss) {
            constexpr int s = decltype(ss)::value;
            constexpr int Q = US == SUBS ? P : (P + s) % 2;  // 3 c + s, modulo 2
            if constexpr (US == 1) {
                if constexpr (s + 1 < SUBS) {
                    read_a(std::integral_constant<int, 1 - Q>{}, std::integral_constant<int, KT>{}, s + 1, buf);
                } else {
                    next_ktile();
                    read_a(std::integral_constant<int, 1 - Q>{}, NextC{}, 0, buf);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            const int sa = s == 0 ? ca.x : s == 1 ? ca.y : ca.z;
            int sb = s == 0 ? cb.x : s == 1 ? cb.y : cb.z;
            if constexpr (G::BAND) sb = (int)((uint32_t)sb >> b_shift);
#pragma unroll
            for (int ni = 0; ni < NPW; ni++) {
#pragma unroll
                for (int mi = 0; mi < MB; mi++)
                    wide_mfma<MB, NPW>(acc, mi, ni, RA[Q][US == SUBS ? s : 0][mi], RB[T][s][ni], sa, sb);
                __builtin_amdgcn_sched_barrier(0);
                load_b(RB[T][s][ni], ni, kt_next, s);
                asm volatile("" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
                if (s == SUBS - 1 && ni == NPW - 1) {
                    load_scales(sc_b[T], kt_next);
                    asm volatile("" ::: "memory");
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        });
    };
    // Whole passes, then the K-tiles left. No exit inside a pass: where it met the loop's back edge
    // the compiler would wait for loads just issued. For the same reason a K-tile's scale load comes
    // after the last MFMA that uses the slot's old ones (a copy of them would be waited for).
    constexpr int PASS = G::PASS;
    int c = 0;
    for (; c + PASS <= nkt; c += PASS) static_for<PASS>([&](auto tt) { ktile(c + decltype(tt)::value, tt); });
    stream_tail<0, PASS>(nkt - c, [&](auto tt) { ktile(c + decltype(tt)::value, tt); });
    const int le = lane_id();
    store_tile<MB, NPW, OutT, SPLIT, MASK>(acc, D, ws, M, N, wg_m * MT + 4 * (le >> 5),
                                           (wg_n * WN + wave) * NPW * 32 + (le & 31), le, wg_z);
}

// One launch for a tile of grouping (MB, NPW) with WN computing waves a workgroup. The K-segment
// partials go to d->ws when SPLIT.
template <int MB, int NPW, int WN, typename KT, bool SPLIT>
hipError_t stream_launch_w(const mxfp6_launch_desc* d, bool ntb, hipStream_t st) {
    using G = StreamGeom<MB, NPW, WN>;
    const bool mask = d->M % G::MT != 0 || d->N % G::NT != 0;
    const dim3 grid((unsigned)((d->M + G::MT - 1) / G::MT), (unsigned)((d->N + G::NT - 1) / G::NT),
                    (unsigned)d->splits);
    auto k = mask ? stream_kernel<MB, NPW, WN, 4, KT, SPLIT, true, false>
                  : stream_kernel<MB, NPW, WN, 4, KT, SPLIT, false, false>;
    if constexpr (WN == 4) {
        if (ntb)
            k = mask ? stream_kernel<MB, NPW, WN, 4, KT, SPLIT, true, true>
                     : stream_kernel<MB, NPW, WN, 4, KT, SPLIT, false, true>;
    }
    return launch_kernel(k, grid, dim3(G::THREADS), st, static_cast<const uint8_t*>(d->A),
                         static_cast<const uint8_t*>(d->Bsh), d->sA, d->sB,
                         SPLIT ? nullptr : static_cast<KT*>(d->D), SPLIT ? d->ws : nullptr, d->M,
                         d->N, d->Kp, d->A_row_bytes, SPLIT ? d->splits : 1, NPW);
}

// run.waves computing waves (tile_dispatch.hpp). Returns 0, or 2 when the launch fails.
template <int MB, int NPW, typename KT, bool SPLIT>
int stream_launch(const mxfp6_launch_desc* d, const mxfp6_dispatch::TileRun& run, hipStream_t st) {
    hipError_t e;
    if (run.waves == 4)
        e = stream_launch_w<MB, NPW, 4, KT, SPLIT>(d, run.nt_b, st);
    else if (MB == 1 && NPW == 1 && run.waves == 1)
        e = stream_launch_w<MB, NPW, MB == 1 && NPW == 1 ? 1 : 2, KT, SPLIT>(d, run.nt_b, st);
    else
        e = stream_launch_w<MB, NPW, 2, KT, SPLIT>(d, run.nt_b, st);
    return e == hipSuccess ? 0 : 2;
}

// BAND with run.waves computing waves. Returns 0, or 2 when the launch fails.
template <typename KT, bool SPLIT>
int band_launch(const mxfp6_launch_desc* d, const mxfp6_dispatch::TileRun& run, hipStream_t st) {
    using G = StreamGeom<4, 1, 0>;
    const int wn = run.waves;
    const dim3 grid((unsigned)((d->M + 127) / 128), (unsigned)((d->N + 32 * wn - 1) / (32 * wn)),
                    (unsigned)d->splits);
    const hipError_t e = launch_kernel(
        run.nt_b ? stream_kernel<4, 1, 0, 4, KT, SPLIT, true, true>
                 : stream_kernel<4, 1, 0, 4, KT, SPLIT, true, false>,
        grid, dim3(64 * (wn + G::NCW)), st, static_cast<const uint8_t*>(d->A),
        static_cast<const uint8_t*>(d->Bsh), d->sA, d->sB, SPLIT ? nullptr : static_cast<KT*>(d->D),
        SPLIT ? d->ws : nullptr, d->M, d->N, d->Kp, d->A_row_bytes, SPLIT ? d->splits : 1, d->npw);
    return e == hipSuccess ? 0 : 2;
}

}  // namespace mxfp6_dev
