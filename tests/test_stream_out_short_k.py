"""Unsplit plans on wide tiles whose operands and 16-bit D fill half the 256 MiB last-level cache or more
write D with nontemporal stores where D is at least 0.4 times the operands (up to 236 MB in all) or 8 times
(above), FP32 D only past 280 MB, and either only in rows of whole 128-byte lines: the rule's edges, and the values against the direct kernel bit for bit."""
import pytest

import checks
import mxfp6_amd as mx


@pytest.mark.parametrize("M,N,K,out_type,want", [
    (8192, 8192, 1024, mx.OUT_BF16, True),    # D 134 MB, 10x the operands
    (8192, 7936, 960, mx.OUT_BF16, True),     # 130 + 12 MB: over half the cache
    (8192, 7168, 1024, mx.OUT_BF16, False),   # 131 MB in all: under it
    (8192, 8192, 4096, mx.OUT_BF16, True),    # D 2.5x, 187 MB in all
    (8192, 4096, 8192, mx.OUT_BF16, True),    # D 0.85x, 146 MB
    (256, 18432, 12288, mx.OUT_F32, False),   # D a tenth of the operands
    (8192, 12288, 3072, mx.OUT_BF16, False),  # 251 MB in all, D 4x
    (8192, 15360, 512, mx.OUT_BF16, True),    # 262 MB, D over 8x
    (4096, 10240, 1024, mx.OUT_F32, False),   # FP32 D of 168 MB: prepare_a finds it cached
    (4096, 8192, 2048, mx.OUT_F32, False),
    (4096, 16384, 512, mx.OUT_F32, False),    # 268 + 8 MB
    (4096, 17408, 512, mx.OUT_F32, True),     # 285 + 8 MB
    (4096, 10240, 1024, mx.OUT_F16, False),
    (2048, 28672, 1024, mx.OUT_F16, True),
    # rows that are no whole number of 128-byte lines, below and above 280 MB
    (2091, 23035, 2218, mx.OUT_BF16, False), (8192, 8194, 1024, mx.OUT_BF16, False),
    (8191, 8224, 1024, mx.OUT_F16, False), (8191, 8256, 1024, mx.OUT_F16, True),
    (2048, 102271, 1024, mx.OUT_F16, False), (2048, 102272, 1024, mx.OUT_F16, True),
    (4096, 17424, 512, mx.OUT_F32, False), (4096, 17472, 512, mx.OUT_F32, True),
    (10368, 9600, 142, mx.OUT_F16, False)])   # 128x384: three blocks a wave
def test_rule(M, N, K, out_type, want):
    Kp = mx.kpad(K)
    assert mx.splitk_segments(M, N, Kp) == 1
    assert mx.plan_kernel(out_type, M, N, Kp, mx.choose_tile(M, N, Kp))[0] in ("wide", "band")
    assert mx.streams_output(out_type, M, N, Kp, mx.packed_bytes(Kp)) == want


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,out_type", [(8192, 8192, 1024, mx.OUT_BF16), (2048, 28672, 1344, mx.OUT_F16),
                                            (8192, 10240, 960, mx.OUT_F16),
                                            (4096, 17408, 512, mx.OUT_F32)])
def test_equals_direct_kernel(M, N, K, out_type):
    from gpu_util import DevProblem, run_direct, run_routed
    p = checks.spread_scales(mx.make_problem(M, N, K, seed=M + N + K), seed=K)
    assert mx.streams_output(out_type, M, N, p.Kp, p.a_row_bytes)
    dp = DevProblem(p, mx.choose_tile(M, N, p.Kp))
    assert (run_routed(dp, out_type).view("u4") == run_direct(dp, out_type).view("u4")).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(2040, 28736, 1344),    # 256 x 256 or 128 x 512 tiles, masked on both sides
                                   (8191, 8256, 1024), (8100, 8384, 320), (16000, 4672, 384)])
@pytest.mark.parametrize("out_type,name", [(mx.OUT_F16, "float16"), (mx.OUT_BF16, "bfloat16")])
def test_masked_in_bounds(M, N, K, out_type, name):
    """Streamed D of tiles that divide neither M nor N: the FP32 result rounded once, nothing outside."""
    import torch
    from gpu_util import DevProblem, run_explicit
    guard, dtype = 4096, getattr(torch, name)
    p = checks.spread_scales(mx.make_problem(M, N, K, seed=M + N + K), span=3, seed=K)
    tile = mx.choose_tile(M, N, p.Kp)
    assert M % tile[0] != 0 and N % tile[1] != 0
    assert mx.streams_output(out_type, M, N, p.Kp, p.a_row_bytes)
    dp = DevProblem(p, tile)
    want = torch.from_numpy(run_explicit(dp, mx.OUT_F32)).reshape(M, N).to(dtype)
    buf = torch.full((2 * M * N + 2 * guard,), 0x5A, dtype=torch.uint8, device="cuda")
    rc = mx.gemm_explicit(out_type, M, N, p.Kp, tile, 1, *dp.ptrs(), buf.data_ptr() + guard, p.a_row_bytes)
    assert rc == 0, mx.STATUS.get(rc, rc)
    torch.cuda.synchronize()
    out = buf.cpu()
    assert torch.equal(out[guard:-guard].view(torch.int16).reshape(M, N), want.view(torch.int16))
    assert bool((out[:guard] == 0x5A).all()) and bool((out[-guard:] == 0x5A).all())
