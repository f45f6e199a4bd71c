"""The stream kernel (stream_kernel.hpp): the skinny tiles on row-major A. Bit for bit the output of
the direct kernel, and on ragged shapes of the slab kernel on the repacked A, where its chunks (two
K-tiles), its passes, its number of computing waves and its masks change."""
import numpy as np
import pytest

import checks
import mxfp6_amd as mx
import gpu_util as g

pytestmark = pytest.mark.gpu

SKINNY = [(32, 128, 1, 1), (32, 256, 1, 2), (64, 128, 2, 1), (64, 256, 2, 2)]
T3 = {"dist_a": mx.DIST_STUDENT_T3, "dist_b": mx.DIST_STUDENT_T3}


def same(a, b):
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


@pytest.mark.parametrize("tile", SKINNY)
@pytest.mark.parametrize("K,S", [(192, 1), (384, 1), (576, 1), (768, 1), (960, 1), (576, 3),
                                 (1344, 3), (2304, 5)])
@pytest.mark.parametrize("M,N", [(64, 256), (512, 2048), (1024, 5120)])
def test_stream_bitwise_equals_direct(tile, K, S, M, N):
    """K-tile counts 1 to 5 a segment (odd and even: partial chunks and passes) on grids of one
    workgroup up to more workgroups than CUs (one, two and four computing waves)."""
    seed = M + N + K + S
    p = checks.spread_scales(mx.make_problem(M, N, K, **T3, seed=seed), seed=seed)
    dp = g.DevProblem(p, tile)
    same(g.run_explicit(dp, mx.OUT_F32, splits=S), g.run_direct(dp, mx.OUT_F32, splits=S))


@pytest.mark.parametrize("tile", SKINNY)
@pytest.mark.parametrize("M,N,K,S", [(1, 1, 192, 1), (13, 1000, 1100, 1), (31, 33, 600, 2),
                                     (65, 127, 2000, 1), (95, 4097, 400, 1), (33, 300, 5000, 7)])
@pytest.mark.parametrize("compact", [True, False])
def test_stream_ragged_equals_slab(tile, M, N, K, S, compact):
    K = K // 32 * 32
    p = checks.spread_scales(mx.make_problem(M, N, K, **T3, seed=M + K, compact=compact), seed=M + K)
    dp = g.DevProblem(p, tile)
    same(g.run_explicit(dp, mx.OUT_F32, splits=S), g.run_explicit(dp, mx.OUT_F32, splits=S, a_layout=1))


@pytest.mark.parametrize("tile,M,S", [((64, 128, 2, 1), 61, 1), ((32, 256, 1, 2), 32, 3)])
def test_stream_large_b_equals_slab(tile, M, S):
    """B over half the last-level cache under one tile row: its loads are nontemporal."""
    import torch
    N, Kp = 16384, 11136
    gen = torch.Generator(device="cuda").manual_seed(5)
    b = lambda n, lo, hi: torch.randint(lo, hi, (n,), generator=gen, device="cuda", dtype=torch.uint8)  # noqa: E731
    row = mx.packed_bytes(Kp)
    a, bsh = b(M * row, 0, 256), b(mx.preshuffled_bytes(N, Kp), 0, 256)
    sa, sb = b(mx.tiled_scale_bytes(M, Kp, tile[2]), 110, 128), b(mx.tiled_scale_bytes(N, Kp, tile[3]), 110, 128)
    D = []
    for layout in (0, 1):
        n = max(4, mx.plan_workspace_size(M, N, Kp, S, layout == 1))
        ws = torch.empty(n, dtype=torch.uint8, device="cuda")
        d = torch.empty(M, N, device="cuda")
        rc = mx.gemm_explicit(mx.OUT_F32, M, N, Kp, tile, S, a.data_ptr(), bsh.data_ptr(), sa.data_ptr(),
                              sb.data_ptr(), d.data_ptr(), row, ws.data_ptr(), n, a_layout=layout)
        assert rc == 0, mx.STATUS.get(rc, rc)
        torch.cuda.synchronize()
        D.append(d.cpu().numpy())
    same(D[0], D[1])
