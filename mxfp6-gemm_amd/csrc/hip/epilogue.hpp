// Epilogue shared by the tile kernels: a wave's MPW x NPW block of FP32 accumulators to D (FP32,
// FP16 or BF16, row-major, ld = N) or, for a split-K segment, to its FP32 partials ws[z][M][N].
// Lane l of block (mi, ni) holds column n_w + 32 ni and rows m_w + 32 mi + 8 g + r in
// acc[mi][ni][4 g + r], with m_w = (first row of the wave) + 4 (l / 32) and n_w = (first column of
// the wave) + l % 32. PAIR stores two side-by-side blocks of 16-bit D together. MASK stores only rows < M and columns < N. NT writes D with nontemporal
// stores (streamed past the caches, for plans whose D would evict the operands the tiles re-read).
#pragma once
#include "device_common.hpp"

namespace mxfp6_dev {

// *p = v, nontemporal when NT
template <bool NT, typename T>
__device__ __forceinline__ void store_out(T* p, T v) {
    if constexpr (!NT)
        *p = v;
    else if constexpr (sizeof(T) == 2)
        __builtin_nontemporal_store((uint16_t)half_bits(v), reinterpret_cast<uint16_t*>(p));
    else
        __builtin_nontemporal_store(v, p);
}

template <int MPW, int NPW, typename OutT, bool SPLIT, bool MASK, bool NT = false, bool PAIR = NT>
__device__ __forceinline__ void store_tile(const v16f (&acc)[MPW][NPW], OutT* __restrict__ D,
                                           float* __restrict__ ws, int M, int N, int m_w, int n_w,
                                           int lane, int wg_z) {
    if constexpr (!SPLIT && sizeof(OutT) == 2) {
        if (!MASK || (N & 1) == 0) {
            // 16-bit output in 4-byte stores: lanes 2k and 2k+1 (columns c, c+1) trade halves so
            // that the even lane holds rows +0 and +2 of both columns and the odd lane rows +1
            // and +3 (one quad_perm DPP move and three byte permutes per 4 values), halving the
            // store instructions. The conversions are the per-element ones of cvt_out.
            // PAIR: a row of one block is 64 bytes, half a cache line. Where a wave owns two blocks side by
            // side they are stored together, 128 contiguous bytes of a row (two of them) an instruction
            // in place of four half lines. Past the caches (NT) half lines are slow: 8192 x 8192 x 1024
            // 76.7 -> 71.0 us with pairs, 8192 x 28672 x 1024 254 -> 220. Stores through the caches merge there,
            // and the second trade costs up to 3% (profiles/epilogue16_plain_stores.txt: 8192 x 6144 x 512
            // 39.3 -> 40.3, 3000 x 5000 x 4096 45.8 -> 46.1), but for whole 256 x 256 tiles of long K
            // (wide_launch_st).
            constexpr int PAIRED = PAIR ? NPW / 2 * 2 : 0;
            const bool odd = (lane & 1) != 0;
            const uint32_t sel_send = odd ? 0x05040100u : 0x07060302u;
            const uint32_t sel_a = odd ? 0x03020504u : 0x05040100u;
            const uint32_t sel_b = odd ? 0x03020706u : 0x07060100u;
            const int m_p = m_w + (lane & 1), n_p = n_w & ~1;
            auto swap_pair = [](uint32_t v) {
                // quad_perm [1, 0, 3, 2]
                return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xF, 0xF, false);
            };
            // values 4 g .. 4 g + 3 of a block: rows +0 / +1 (even / odd lane) in oa, +2 / +3 in ob
            auto rows4 = [&](const v16f& a, int g, uint32_t& oa, uint32_t& ob) {
                const uint32_t p01 = half_bits(cvt_out<OutT>(a[4 * g])) |
                                     (half_bits(cvt_out<OutT>(a[4 * g + 1])) << 16);
                const uint32_t p23 = half_bits(cvt_out<OutT>(a[4 * g + 2])) |
                                     (half_bits(cvt_out<OutT>(a[4 * g + 3])) << 16);
                const uint32_t recv = swap_pair(__builtin_amdgcn_perm(p23, p01, sel_send));
                oa = __builtin_amdgcn_perm(recv, p01, sel_a);
                ob = __builtin_amdgcn_perm(recv, p23, sel_b);
            };
            auto put = [&](int m, int n, uint32_t v) {
                if (!MASK || m < M) store_out<NT>(reinterpret_cast<uint32_t*>(D + (size_t)m * N + n), v);
            };
#pragma unroll
            for (int mi = 0; mi < MPW; mi++) {
#pragma unroll
                for (int ni = 0; ni + 1 < PAIRED; ni += 2)
#pragma unroll
                    for (int g = 0; g < 4; g++) {
                        // the pair trades again: the even lane holds all four rows of block ni, the
                        // odd lane those of block ni + 1
                        uint32_t a0, b0, a1, b1;
                        rows4(acc[mi][ni], g, a0, b0);
                        rows4(acc[mi][ni + 1], g, a1, b1);
                        const uint32_t ra = swap_pair(odd ? a0 : a1), rb = swap_pair(odd ? b0 : b1);
                        const int m = m_w + mi * 32 + 8 * g, n = n_p + (ni + (lane & 1)) * 32;
                        if (MASK && n >= N) continue;  // n even and N even: n + 1 < N as well
                        put(m, n, odd ? ra : a0);
                        put(m + 1, n, odd ? a1 : ra);
                        put(m + 2, n, odd ? rb : b0);
                        put(m + 3, n, odd ? b1 : rb);
                    }
#pragma unroll
                for (int ni = PAIRED; ni < NPW; ni++)
#pragma unroll
                    for (int g = 0; g < 4; g++) {
                        uint32_t oa, ob;
                        rows4(acc[mi][ni], g, oa, ob);
                        const int m = m_p + mi * 32 + 8 * g, n = n_p + ni * 32;
                        if (MASK && n >= N) continue;
                        put(m, n, oa);
                        put(m + 2, n, ob);
                    }
            }
            return;
        }
    }
#pragma unroll
    for (int mi = 0; mi < MPW; mi++)
#pragma unroll
        for (int ni = 0; ni < NPW; ni++)
#pragma unroll
            for (int g = 0; g < 4; g++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int m = m_w + mi * 32 + 8 * g + r, n = n_w + ni * 32;
                    if (MASK && (m >= M || n >= N)) continue;
                    const size_t idx = (size_t)m * N + n;
                    if (SPLIT)
                        ws[(size_t)wg_z * M * N + idx] = acc[mi][ni][4 * g + r];
                    else
                        store_out<NT>(D + idx, cvt_out<OutT>(acc[mi][ni][4 * g + r]));
                }
}

}  // namespace mxfp6_dev
