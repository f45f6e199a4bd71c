"""The 16-bit epilogue (epilogue.hpp): each value is the tile's FP32 result rounded once, at every column
remainder of a pair of blocks, with nothing written outside D. (Streamed D, which is stored two blocks of a wave
together, is in test_stream_out_short_k.py.)"""
import numpy as np
import pytest
import torch

import checks
import mxfp6_amd as mx
import gpu_util as g

pytestmark = pytest.mark.gpu

GUARD = 4096  # bytes before and after D
TILES = [(32, 256, 1, 2), (64, 128, 2, 1), (128, 256, 4, 2), (128, 384, 4, 3), (128, 512, 4, 4),
         (256, 256, 4, 2), (256, 256, 2, 4)]


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("M,N", [(256, 1536), (37, 2), (133, 30), (37, 34), (133, 62), (37, 66), (133, 94),
                                 (130, 126), (37, 130), (261, 610), (261, 1000), (131, 545)])
@pytest.mark.parametrize("out_type,dtype", [(mx.OUT_F16, torch.float16), (mx.OUT_BF16, torch.bfloat16)])
def test_rounded_once_and_in_bounds(tile, M, N, out_type, dtype):
    rounded_once(tile, M, N, 320, out_type, dtype)


@pytest.mark.parametrize("M,N,K", [(256, 256, 4096), (4096, 4352, 4096), (4096, 4352, 4032)])
@pytest.mark.parametrize("out_type,dtype", [(mx.OUT_F16, torch.float16), (mx.OUT_BF16, torch.bfloat16)])
def test_long_k_whole_tiles(M, N, K, out_type, dtype):
    """K on both sides of the line from which whole 256 x 256 tiles store pairs of blocks (more tiles than CUs:
    they do not run as bands)."""
    rounded_once((256, 256, 4, 2), M, N, K, out_type, dtype)


def rounded_once(tile, M, N, K, out_type, dtype):
    p = checks.spread_scales(mx.make_problem(M, N, K, seed=M + N), span=3, seed=N)
    dp = g.DevProblem(p, tile)
    want = torch.from_numpy(g.run_explicit(dp, mx.OUT_F32)).reshape(M, N).to(dtype)
    buf = torch.full((2 * M * N + 2 * GUARD,), 0x5A, dtype=torch.uint8, device="cuda")
    a, b, sa, sb = dp.ptrs()
    rc = mx.gemm_explicit(out_type, M, N, p.Kp, tile, 1, a, b, sa, sb, buf.data_ptr() + GUARD,
                          p.a_row_bytes, 0, 0, a_layout=0)
    assert rc == 0, mx.STATUS.get(rc, rc)
    torch.cuda.synchronize()
    out = buf.cpu()
    assert torch.equal(out[GUARD:-GUARD].view(torch.int16).reshape(M, N), want.view(torch.int16))
    assert np.all(out[:GUARD].numpy() == 0x5A) and np.all(out[-GUARD:].numpy() == 0x5A)
