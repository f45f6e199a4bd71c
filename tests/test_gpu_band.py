"""Wide-tile plans on row-major A whose grid leaves CUs idle run as 128-row bands of the stream kernel
(stream_kernel.hpp, BAND), as many computing waves a workgroup as one round of the CUs needs. Bit for
bit the direct kernel's output, and on ragged shapes the wide kernel's on the repacked A."""
import numpy as np
import pytest
import torch

import checks
import mxfp6_amd as mx
import gpu_util as g

pytestmark = pytest.mark.gpu

WIDE = [(128, 256, 4, 2), (128, 384, 4, 3), (128, 512, 4, 4), (256, 256, 4, 2)]
T3 = {"dist_a": mx.DIST_STUDENT_T3, "dist_b": mx.DIST_STUDENT_T3}


def same(a, b):
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


@pytest.mark.parametrize("tile", WIDE)
@pytest.mark.parametrize("M,N,K,S,waves", [(128, 384, 1536, 1, 2),    # a whole number of chunks
                                           (256, 768, 1728, 1, 2),    # nine K-tiles: a partial chunk
                                           (512, 6144, 1536, 1, 3),
                                           (512, 7680, 1600, 1, 4),   # the last K-tile half values
                                           (256, 1536, 4992, 3, 2)])  # segments of nine and eight K-tiles
def test_band_bitwise_equals_direct(tile, M, N, K, S, waves):
    assert mx.plan_kernel(mx.OUT_F32, M, N, mx.kpad(K), tile, S) == ("band", waves, False)
    seed = M + N + K
    p = checks.spread_scales(mx.make_problem(M, N, K, **T3, seed=seed), seed=seed)
    dp = g.DevProblem(p, tile)
    same(g.run_explicit(dp, mx.OUT_F32, splits=S), g.run_direct(dp, mx.OUT_F32, splits=S))


@pytest.mark.parametrize("tile", WIDE)
@pytest.mark.parametrize("M,N,K,S", [(1, 1, 1600, 1), (100, 1000, 1760, 1), (131, 6143, 1536, 1),
                                     (300, 517, 3300, 2)])
@pytest.mark.parametrize("out_type", [mx.OUT_F32, mx.OUT_BF16])
def test_band_ragged_equals_wide(tile, M, N, K, S, out_type):
    K = K // 32 * 32
    p = checks.spread_scales(mx.make_problem(M, N, K, **T3, seed=M + K), seed=M + K)
    dp = g.DevProblem(p, tile)
    assert mx.plan_kernel(out_type, M, N, p.Kp, tile, S, A_row_bytes=p.a_row_bytes)[0] == "band"
    same(g.run_explicit(dp, out_type, splits=S), g.run_explicit(dp, out_type, splits=S, a_layout=1))


@pytest.mark.parametrize("M,N,Kp,waves,nt", [
    (250, 18432, 4992, 5, False),   # B of a quarter of the last-level cache: five waves
    (128, 24576, 7488, 3, True),    # half of it, one tile row: nontemporal loads
    (123, 40950, 4416, 5, True)])   # both, masked
@pytest.mark.parametrize("out_type,dtype", [(mx.OUT_F32, torch.float32), (mx.OUT_F16, torch.float16)])
def test_band_large_b_equals_wide(M, N, Kp, waves, nt, out_type, dtype):
    tile = (128, 256, 4, 2)
    assert mx.plan_kernel(out_type, M, N, Kp, tile) == ("band", waves, nt)
    gen = torch.Generator(device="cuda").manual_seed(5)
    b = lambda n, lo, hi: torch.randint(lo, hi, (n,), generator=gen, device="cuda", dtype=torch.uint8)  # noqa: E731
    row = mx.packed_bytes(Kp)
    a, bsh = b(M * row, 0, 256), b(mx.preshuffled_bytes(N, Kp), 0, 256)
    sa, sb = b(mx.tiled_scale_bytes(M, Kp, 4), 110, 128), b(mx.tiled_scale_bytes(N, Kp, 2), 110, 128)
    D = []
    for layout in (0, 1):
        n = max(4, mx.plan_workspace_size(M, N, Kp, 1, layout == 1))
        ws = torch.empty(n, dtype=torch.uint8, device="cuda")
        d = torch.empty(M, N, dtype=dtype, device="cuda")
        rc = mx.gemm_explicit(out_type, M, N, Kp, tile, 1, a.data_ptr(), bsh.data_ptr(), sa.data_ptr(),
                              sb.data_ptr(), d.data_ptr(), row, ws.data_ptr(), n, a_layout=layout)
        assert rc == 0, mx.STATUS.get(rc, rc)
        torch.cuda.synchronize()
        D.append(d.float().cpu().numpy())
    same(D[0], D[1])
