"""Skinny-tile plans (32 and 64 rows) on many workgroups run on 128 x 256 wide tiles that read the
skinny tile's scale groups: bit for bit the direct kernel's output, the slab kernel's on the repacked A on
ragged shapes, and the routed gemm on its plan's workspace."""
import numpy as np
import pytest

import checks
import mxfp6_amd as mx
import gpu_util as g

pytestmark = pytest.mark.gpu

SKINNY = [(32, 128, 1, 1), (32, 256, 1, 2), (64, 128, 2, 1), (64, 256, 2, 2)]
T3 = {"dist_a": mx.DIST_STUDENT_T3, "dist_b": mx.DIST_STUDENT_T3}


def runs_wide(dp, out_type, S):
    p = dp.p
    return mx.plan_kernel(out_type, p.M, p.N, p.Kp, dp.tile, S, A_row_bytes=p.a_row_bytes)[0] == "wide"


def same(a, b):
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


@pytest.mark.parametrize("tile", SKINNY)
@pytest.mark.parametrize("K,S", [(192, 1), (384, 1), (576, 1), (768, 1), (1500, 1), (1344, 2)])
def test_bitwise_equals_direct(tile, K, S):
    """One to eight K-tiles (its short paths, which two B groups a wave end at two K-tiles, and its
    main loop), split and not, the last tile row partly past M."""
    M, N = 2112 if S == 1 else 1088, 2304  # 153 or 162 workgroups of 128 x 256
    p = checks.spread_scales(mx.make_problem(M, N, K // 32 * 32, **T3, seed=K), seed=K)
    dp = g.DevProblem(p, tile)
    assert runs_wide(dp, mx.OUT_F32, S)
    same(g.run_explicit(dp, mx.OUT_F32, splits=S), g.run_direct(dp, mx.OUT_F32, splits=S))


@pytest.mark.parametrize("tile", SKINNY)
@pytest.mark.parametrize("M,N,K,S", [(2017, 2049, 800, 1), (2000, 4700, 192, 1), (97, 19000, 700, 2)])
@pytest.mark.parametrize("out_type", [mx.OUT_F32, mx.OUT_F16])
def test_ragged_equals_slab(tile, M, N, K, S, out_type):
    K = K // 32 * 32
    p = checks.spread_scales(mx.make_problem(M, N, K, **T3, seed=M + K), seed=M + K)
    dp = g.DevProblem(p, tile)
    assert runs_wide(dp, out_type, S)
    same(g.run_explicit(dp, out_type, splits=S), g.run_explicit(dp, out_type, splits=S, a_layout=1))


@pytest.mark.parametrize("M,N,K,kernel", [(3616, 5120, 4096, "wide"), (1184, 25856, 1536, "wide"),
                                          (576, 8192, 6016, "wide"), (1056, 1920, 17408, "stream")])
def test_routed_plans(M, N, K, kernel):
    p = checks.spread_scales(mx.make_problem(M, N, K, **T3, seed=M), seed=M)
    tile, S, rp = mx.gemm_plan(mx.OUT_F32, M, N, p.Kp, mx.preferred_workspace_size(M, N, p.Kp))
    assert not rp and tile[0] <= 64
    dp = g.DevProblem(p, tile)
    assert mx.plan_kernel(mx.OUT_F32, M, N, p.Kp, tile, S, A_row_bytes=p.a_row_bytes)[0] == kernel
    same(g.run_routed(dp, mx.OUT_F32), g.run_explicit(dp, mx.OUT_F32, splits=S, a_layout=1))
