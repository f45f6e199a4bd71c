"""The stream kernel (stream_kernel.hpp): the skinny tiles on row-major A. Bit for bit the output of
the direct kernel, and on ragged shapes of the slab kernel on the repacked A, where its chunks (two
K-tiles), its passes, its number of computing waves, its masks, its output type and its loads of B change. Every
case says how many computing waves it is for, and the plan's kernel is asked. One K-tile a segment runs on the slab
kernel where that is faster: row-major A there, against the same references."""
import numpy as np
import pytest
import torch

import checks
import mxfp6_amd as mx
import gpu_util as g

pytestmark = pytest.mark.gpu

T32_128, T32_256, T64_128, T64_256 = (32, 128, 1, 1), (32, 256, 1, 2), (64, 128, 2, 1), (64, 256, 2, 2)
T3 = {"dist_a": mx.DIST_STUDENT_T3, "dist_b": mx.DIST_STUDENT_T3}


def same(a, b):
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


def problem(M, N, K, seed, **kw):
    return checks.spread_scales(mx.make_problem(M, N, K, **T3, seed=seed, **kw), seed=seed)


def streams(dp, out_type, S, waves):
    p = dp.p
    slab = p.Kp // 192 <= S and dp.tile[0] == 64
    assert mx.plan_kernel(out_type, p.M, p.N, p.Kp, dp.tile, S, A_row_bytes=p.a_row_bytes) == (
        ("slab", 0, False) if slab else ("stream", waves, False))


@pytest.mark.parametrize("K", [192, 384, 576, 768, 960])
@pytest.mark.parametrize("tile,M,N,waves", [(T32_128, 64, 256, 1), (T32_128, 256, 2048, 2),
                                            (T32_128, 512, 2048, 4), (T32_256, 64, 256, 4),
                                            (T32_256, 320, 7168, 2), (T64_128, 64, 256, 2),
                                            (T64_128, 512, 4096, 4), (T64_256, 64, 256, 4),
                                            (T64_256, 320, 13824, 2)])
def test_stream_bitwise_equals_direct(tile, M, N, waves, K):
    """One to five K-tiles (odd and even: partial chunks and passes) on grids of one workgroup up to more
    workgroups than CUs."""
    dp = g.DevProblem(problem(M, N, K, M + N + K), tile)
    for ot in (mx.OUT_F32, mx.OUT_F16 if K % 384 else mx.OUT_BF16):
        streams(dp, ot, 1, waves)
        same(g.run_explicit(dp, ot), g.run_direct(dp, ot))


@pytest.mark.parametrize("K,S", [(576, 3), (1344, 3), (2304, 3)])
@pytest.mark.parametrize("tile,M,N,waves", [(T32_128, 64, 256, 1), (T32_128, 128, 1024, 2),
                                            (T32_128, 256, 2048, 4), (T32_256, 64, 256, 4),
                                            (T32_256, 256, 3584, 2), (T64_128, 64, 256, 2),
                                            (T64_128, 512, 2048, 4), (T64_256, 64, 256, 4),
                                            (T64_256, 512, 2816, 2)])
def test_stream_split_bitwise_equals_direct(tile, M, N, waves, K, S):
    """One to four K-tiles a segment, segments of two lengths."""
    dp = g.DevProblem(problem(M, N, K, M + N + K + S), tile)
    streams(dp, mx.OUT_F32, S, waves)
    same(g.run_explicit(dp, mx.OUT_F32, splits=S), g.run_direct(dp, mx.OUT_F32, splits=S))


@pytest.mark.parametrize("tile", [T32_128, T32_256, T64_128, T64_256])
@pytest.mark.parametrize("M,N,K,S", [(1, 1, 192, 1), (13, 1000, 1100, 1), (31, 33, 600, 2),
                                     (65, 127, 2000, 1), (95, 4097, 400, 1), (33, 300, 5000, 7)])
@pytest.mark.parametrize("compact", [True, False])
def test_stream_ragged_equals_slab(tile, M, N, K, S, compact):
    dp = g.DevProblem(problem(M, N, K // 32 * 32, M + K, compact=compact), tile)
    p = dp.p
    assert mx.plan_kernel(mx.OUT_F32, M, N, p.Kp, tile, S, A_row_bytes=p.a_row_bytes)[0] == (
        "slab" if K == 192 and tile[0] == 64 else "stream")
    same(g.run_explicit(dp, mx.OUT_F32, splits=S), g.run_explicit(dp, mx.OUT_F32, splits=S, a_layout=1))


@pytest.mark.parametrize("tile,M,N,K,S", [(T64_128, 37, 545, 96, 1), (T64_128, 130, 260, 350, 2),
                                          (T64_256, 61, 1001, 192, 1), (T64_256, 832, 9472, 160, 1),
                                          (T32_128, 1119, 3714, 192, 1), (T32_128, 1120, 3712, 64, 1)])
@pytest.mark.parametrize("out_type", [mx.OUT_F32, mx.OUT_F16, mx.OUT_BF16])
def test_one_k_tile_on_rows_equals_repacked(tile, M, N, K, S, out_type):
    dp = g.DevProblem(problem(M, N, K // 32 * 32, M + K), tile)
    p = dp.p
    assert mx.plan_kernel(out_type, M, N, p.Kp, tile, S, A_row_bytes=p.a_row_bytes)[0] == "slab"
    same(g.run_explicit(dp, out_type, splits=S), g.run_explicit(dp, out_type, splits=S, a_layout=1))


@pytest.mark.parametrize("tile,M,N,waves", [(T32_128, 33, 130, 1), (T32_128, 250, 2040, 2),
                                            (T32_128, 500, 2031, 4), (T32_256, 300, 7100, 2),
                                            (T32_256, 37, 1001, 4), (T64_128, 61, 1034, 2),
                                            (T64_128, 500, 4090, 4), (T64_256, 319, 13790, 2),
                                            (T64_256, 130, 2050, 4)])
@pytest.mark.parametrize("out_type", [mx.OUT_F32, mx.OUT_F16, mx.OUT_BF16])
def test_stream_masked_waves_equal_slab(tile, M, N, waves, out_type):
    """Partial tile rows and columns at every number of computing waves."""
    dp = g.DevProblem(problem(M, N, 544, M + N), tile)
    streams(dp, out_type, 1, waves)
    same(g.run_explicit(dp, out_type), g.run_explicit(dp, out_type, a_layout=1))


@pytest.mark.parametrize("tile,M,N,Kp,S", [(T32_128, 32, 20480, 8832, 1), (T32_128, 13, 20450, 8832, 1),
                                           (T32_128, 32, 20480, 8832, 2), (T32_256, 32, 16384, 11136, 1),
                                           (T32_256, 13, 16382, 11136, 1), (T32_256, 32, 16384, 11136, 3),
                                           (T64_128, 64, 20480, 8832, 1), (T64_128, 61, 20480, 8832, 1),
                                           (T64_128, 61, 20450, 8832, 2), (T64_256, 64, 16384, 11136, 1),
                                           (T64_256, 61, 16384, 11136, 1), (T64_256, 64, 16384, 11136, 3)])
@pytest.mark.parametrize("out_type,dtype", [(mx.OUT_F32, torch.float32), (mx.OUT_BF16, torch.bfloat16)])
def test_stream_large_b_equals_slab(tile, M, N, Kp, S, out_type, dtype):
    """B over half the last-level cache under one tile row: its loads are nontemporal."""
    assert mx.plan_kernel(out_type, M, N, Kp, tile, S) == ("stream", 4, True)
    gen = torch.Generator(device="cuda").manual_seed(5)
    b = lambda n, lo, hi: torch.randint(lo, hi, (n,), generator=gen, device="cuda", dtype=torch.uint8)  # noqa: E731
    row = mx.packed_bytes(Kp)
    a, bsh = b(M * row, 0, 256), b(mx.preshuffled_bytes(N, Kp), 0, 256)
    sa, sb = b(mx.tiled_scale_bytes(M, Kp, tile[2]), 110, 128), b(mx.tiled_scale_bytes(N, Kp, tile[3]), 110, 128)
    D = []
    for layout in (0, 1):
        n = max(4, mx.plan_workspace_size(M, N, Kp, S, layout == 1))
        ws = torch.empty(n, dtype=torch.uint8, device="cuda")
        d = torch.empty(M, N, dtype=dtype, device="cuda")
        rc = mx.gemm_explicit(out_type, M, N, Kp, tile, S, a.data_ptr(), bsh.data_ptr(), sa.data_ptr(),
                              sb.data_ptr(), d.data_ptr(), row, ws.data_ptr(), n, a_layout=layout)
        assert rc == 0, mx.STATUS.get(rc, rc)
        torch.cuda.synchronize()
        D.append(d.float().cpu().numpy())
    same(D[0], D[1])
