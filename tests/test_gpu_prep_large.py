"""The preparation kernels past the sizes where they bound the waves in flight and load B
nontemporally: the bytes of the whole operand against those of its pieces, each under those sizes
(rows of A are independent, and so are the 32-column blocks of B's layout)."""
import pytest
import torch

import mxfp6_amd as mx

pytestmark = pytest.mark.gpu


def values(rows, cols, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(rows, cols, generator=gen, device="cuda")
    return x * torch.exp(2 * torch.randn(rows, 1, generator=gen, device="cuda"))


def out(n):
    return torch.full((n,), 0x5A, dtype=torch.uint8, device="cuda")


@pytest.mark.parametrize("rows,cols,shift,few", [(8256, 2048, 0, 1), (8224, 2049, 0, 1), (4160, 4100, 1, 1),
                                                 (8256, 1025, 2, 1), (8256, 1024, 2, 0), (8256, 31, 3, 0),
                                                 (2080, 16127, 0, 1)])
def test_rows(rows, cols, shift, few):
    """More than 32 waves a CU, in fewer at a time (FEW) where a wave has more than 1024 values, rows of any
    length and inputs of any 4-byte alignment."""
    assert mx.lib().mxfp6_hip_prep_few_waves(rows, cols) == few
    x = torch.empty(rows * cols + 4, device="cuda")[shift:shift + rows * cols].view(rows, cols)
    x.copy_(values(rows, cols, cols))
    Kp = mx.kpad(cols)
    row = mx.packed_bytes(Kp)

    def quantise(v):
        n = v.shape[0]
        p, s = out(n * row), out(n * (Kp // 32))
        assert mx.quantize_dev(v.data_ptr(), n, cols, p.data_ptr(), row, s.data_ptr(), Kp // 32) == 0
        return p.view(n, row), s.view(n, Kp // 32)

    p, s = quantise(x)
    for r0 in range(0, rows, 1031):
        part = x[r0:r0 + 1031].clone()  # 16-byte aligned whatever x's alignment
        pp, ps = quantise(part)
        assert torch.equal(p[r0:r0 + 1031], pp) and torch.equal(s[r0:r0 + 1031], ps)


@pytest.mark.parametrize("K,N", [(8192, 4096), (4099, 8256), (16384, 12288), (110000, 330)])
@pytest.mark.parametrize("group", [2, 3])
def test_b(K, N, group):
    """B of half the last-level cache and more."""
    assert mx.lib().mxfp6_hip_prep_b_few(K, N)
    B = values(K, N, N)

    def prepare(b):
        n = b.shape[1]
        p, t = out(mx.preshuffled_bytes(n, K)), out(mx.tiled_scale_bytes(n, K, group))
        assert mx.prepare_b_dev(b.data_ptr(), K, n, group, p.data_ptr(), t.data_ptr()) == 0
        return p, t

    p, t = prepare(B)
    w = 32 * group * 10
    for n0 in range(0, N, w):
        pp, pt = prepare(B[:, n0:n0 + w].contiguous())
        blk = mx.preshuffled_bytes(32, K)
        assert torch.equal(p[n0 // 32 * blk:][:pp.numel()], pp)
        g = mx.tiled_scale_bytes(32 * group, K, group)
        assert torch.equal(t[n0 // (32 * group) * g:][:pt.numel()], pt)
