"""Performance cases of the MXFP6 GEMM library: the calls a program makes through its public entry
points (mxfp6-gemm_amd/mxfp6_amd.py), over the range of sizes they are made with.

Four kinds of call:
  gemm    D = A.B with both operands already in the device layouts (choose_tile, the preferred
          workspace and gemm, as INTEGRATION.md's calling sequence does);
  linear  a layer's call: float activations A are quantised on the device (prepare_a) and
          multiplied with weights B that were laid out once;
  prep_a  prepare_a alone: float A to packed rows and tiled scales;
  prep_b  prepare_b alone: float B[K][N] to the preshuffled operand and tiled scales (loading
          weights, or the moving operand of a training step).
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "mxfp6-gemm_amd"))
import mxfp6_amd as mx  # noqa: E402

DTYPE = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
OUT = {"f32": mx.OUT_F32, "f16": mx.OUT_F16, "bf16": mx.OUT_BF16}

MAX_FLOPS = 2.0 * 2048 * 5120 * 105728  # the largest listed case
MAX_B = 5120 * 105728                   # values of its weights
MAX_PREP = 8192 * 28672                 # values of the largest listed preparation


def listed():
    return [
        # one small product, where launch and latency are all of the time
        {"name": "gemm_small", "kind": "gemm", "M": 256, "N": 256, "K": 1024, "out": "f32"},
        # decoding a small batch: few rows against a large weight, activations ready
        {"name": "gemm_decode", "kind": "gemm", "M": 64, "N": 28672, "K": 8192, "out": "bf16"},
        # one decode step of a layer from float activations; 13 rows fill no tile
        {"name": "linear_decode", "kind": "linear", "M": 13, "N": 8192, "K": 8192, "out": "bf16"},
        # a middle-sized batch against a wide weight
        {"name": "gemm_batch", "kind": "gemm", "M": 256, "N": 18432, "K": 12288, "out": "f16"},
        # short K: a projection whose output is larger than its operands
        {"name": "gemm_short_k", "kind": "gemm", "M": 8192, "N": 8192, "K": 1024, "out": "bf16"},
        # sizes that no tile divides
        {"name": "gemm_ragged", "kind": "gemm", "M": 3000, "N": 5000, "K": 4096, "out": "f16"},
        # the benchmark's large square product
        {"name": "gemm_square", "kind": "gemm", "M": 8192, "N": 8192, "K": 8192, "out": "f16"},
        # very long K with few output tiles: K is split
        {"name": "gemm_long_k", "kind": "gemm", "M": 2048, "N": 1024, "K": 105728, "out": "f16"},
        # the same with more columns: the largest product of the benchmark
        {"name": "gemm_long_k_wide", "kind": "gemm", "M": 2048, "N": 5120, "K": 105728,
         "out": "bf16"},
        # prefill of a layer from float activations, with the sizes of a benchmark product
        {"name": "linear_prefill", "kind": "linear", "M": 2048, "N": 6144, "K": 16128,
         "out": "f16"},
        # activations of a large batch to the GEMM's format
        {"name": "prep_a", "kind": "prep_a", "dim": 8192, "K": 8192, "group": 4},
        # weights to the GEMM's format
        {"name": "prep_b", "kind": "prep_b", "dim": 28672, "K": 8192, "group": 2},
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _dim(rng, low, high, whole, odd):
    """A size from low to high over its logarithm: a multiple of `whole`, or, with probability
    `odd`, any number."""
    n = _log(rng, low, high)
    return n if rng.random() < odd else min(high, max(whole, (n + whole // 2) // whole * whole))


def draw(rng):
    kind = rng.choice(["gemm", "gemm", "gemm", "linear", "linear", "prep_a", "prep_b"])
    while True:
        if kind in ("prep_a", "prep_b"):
            dim = _dim(rng, 16 if kind == "prep_a" else 256, 28672, 32, 0.3)
            K = _dim(rng, 256, 32768, 64, 0.3)
            if 1 << 16 <= dim * K <= MAX_PREP:
                return {"kind": kind, "dim": dim, "K": K, "group": rng.choice([1, 2, 2, 3, 4, 4])}
            continue
        if rng.random() < 0.15:  # long K
            M, N = _dim(rng, 128, 4096, 128, 0.2), _dim(rng, 256, 8192, 128, 0.2)
            K = _dim(rng, 16384, 105728, 64, 0.3)
        else:
            M, N = _dim(rng, 1, 8192, 32, 0.4), _dim(rng, 256, 28672, 128, 0.25)
            K = _dim(rng, 256, 16384, 64, 0.3)
        if 2.0 * M * N * K <= MAX_FLOPS and N * K <= MAX_B:
            return {"kind": kind, "M": M, "N": N, "K": K,
                    "out": rng.choice(["f16", "bf16", "bf16", "f32"])}


def _values(rows, cols, sigma, gen, by_row):
    """Normal values whose channels (rows or columns) differ in size, as weights' and
    activations' do."""
    x = torch.randn(rows, cols, generator=gen, device="cuda")
    size = torch.exp(0.5 * torch.randn(rows if by_row else cols, generator=gen, device="cuda"))
    return x.mul_((sigma * size)[:, None] if by_row else sigma * size)


def _operands(case, seed):
    """Float A [M][K] and B [K][N]: activations of unit size, weights of 1 / sqrt(K)."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    A = _values(case["M"], case["K"], 1.0, gen, False)
    B = _values(case["K"], case["N"], 1.0 / math.sqrt(case["K"]), gen, True)
    return A, B


def _prep_input(case, seed):
    """Float A [dim][K], or B [K][dim]."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dim, K = case["dim"], case["K"]
    if case["kind"] == "prep_a":
        return _values(dim, K, 1.0, gen, False)
    return _values(K, dim, 1.0 / math.sqrt(K), gen, True)


def _ok(rc):
    if rc != 0:
        raise RuntimeError("mxfp6: " + mx.STATUS.get(rc, str(rc)))


def _bytes(n):
    return torch.empty(n, dtype=torch.uint8, device="cuda")


def prepare(case, seed):
    s = {"kind": case["kind"], "stream": torch.cuda.current_stream().cuda_stream}
    K = case["K"]
    Kp = mx.kpad(K)
    row = mx.packed_bytes(Kp)
    if case["kind"] in ("prep_a", "prep_b"):
        dim, group = case["dim"], case["group"]
        s.update(x=_prep_input(case, seed), dim=dim, K=K, group=group, row=row,
                 packed=_bytes(dim * row if case["kind"] == "prep_a" else
                               mx.preshuffled_bytes(dim, K)),
                 tiled=_bytes(mx.tiled_scale_bytes(dim, K, group)))
        return s
    M, N = case["M"], case["N"]
    tile = mx.choose_tile(M, N, Kp)
    ws_bytes = mx.preferred_workspace_size(M, N, Kp)
    A, B = _operands(case, seed)
    s.update(out=OUT[case["out"]], M=M, N=N, K=K, Kp=Kp, row=row, group=tile[2], x=A,
             a=_bytes(M * row), sa=_bytes(mx.tiled_scale_bytes(M, K, tile[2])),
             b=_bytes(mx.preshuffled_bytes(N, K)), sb=_bytes(mx.tiled_scale_bytes(N, K, tile[3])),
             ws=_bytes(max(ws_bytes, 4)), ws_bytes=ws_bytes,
             D=torch.empty(M, N, dtype=DTYPE[case["out"]], device="cuda"))
    _ok(mx.prepare_b_dev(B.data_ptr(), K, N, tile[3], s["b"].data_ptr(), s["sb"].data_ptr(),
                         stream=s["stream"]))
    if case["kind"] == "gemm":
        _quantise_a(s)
        s["x"] = None
    torch.cuda.current_stream().synchronize()  # the float inputs are released here
    return s


def _quantise_a(s):
    _ok(mx.prepare_a_dev(s["x"].data_ptr(), s["M"], s["K"], s["group"], s["a"].data_ptr(),
                         s["row"], s["sa"].data_ptr(), stream=s["stream"]))


def run(s):
    if s["kind"] == "prep_a":
        _ok(mx.prepare_a_dev(s["x"].data_ptr(), s["dim"], s["K"], s["group"],
                             s["packed"].data_ptr(), s["row"], s["tiled"].data_ptr(),
                             stream=s["stream"]))
        return [s["packed"], s["tiled"]]
    if s["kind"] == "prep_b":
        _ok(mx.prepare_b_dev(s["x"].data_ptr(), s["K"], s["dim"], s["group"],
                             s["packed"].data_ptr(), s["tiled"].data_ptr(), stream=s["stream"]))
        return [s["packed"], s["tiled"]]
    if s["kind"] == "linear":
        _quantise_a(s)
    _ok(mx.gemm(s["out"], s["M"], s["N"], s["Kp"], s["a"].data_ptr(), s["b"].data_ptr(),
                s["sa"].data_ptr(), s["sb"].data_ptr(), s["D"].data_ptr(), s["row"],
                s["ws"].data_ptr() if s["ws_bytes"] else 0, s["ws_bytes"], stream=s["stream"]))
    return s["D"]


def work(case):
    """Bytes: float operands once where the call takes them, 3/4 byte a packed value, one scale
    byte per 32 values, D once."""
    K = case["K"]
    mx_bytes = 0.75 + 1.0 / 32
    if case["kind"] in ("prep_a", "prep_b"):
        return {"bytes": case["dim"] * K * (4.0 + mx_bytes), "flops": 0}
    M, N = case["M"], case["N"]
    a = M * K * (4.0 if case["kind"] == "linear" else mx_bytes)
    return {"bytes": a + N * K * mx_bytes + M * N * DTYPE[case["out"]].itemsize,
            "flops": 2.0 * M * N * K}


def tolerance(case):
    """Packed bytes are defined bit for bit. D: the products of codes and scales are exact and
    summed in 32 bits (another order or split moves a sum by a few 1e-7), then rounded once."""
    if case["kind"] in ("prep_a", "prep_b"):
        return "exact"
    return {"rel": {"f32": 2e-6, "f16": 8e-4, "bf16": 6.5e-3}[case["out"]]}


# ---- the same results in 64 bits, from the formats' definitions (plain torch) ------------------

def _blocks(x):
    """x [rows][K] as 32-blocks [rows][ceil(K / 32)][32], the last one filled with zeros."""
    rows, K = x.shape
    return torch.nn.functional.pad(x, (0, -K % 32)).view(rows, -1, 32)


def _quantised(x):
    """(magnitudes of the E2M3 values in steps of 1/8, signs, exponents): the scale of a block is
    the smallest power of two >= amax / 7.5, a value the nearest E2M3 number (ties to even), at
    most 7.5."""
    b = _blocks(x)
    amax = b.abs().amax(-1)
    m, e = torch.frexp(amax / 7.5)
    e = (e - (m == 0.5).to(e.dtype)).clamp(-127, 127)
    e = torch.where(amax == 0, torch.zeros_like(e), e)
    q = torch.ldexp(b.double(), -e[..., None].double())
    mag = q.abs()
    step = torch.where(mag < 2, 0.125, torch.where(mag < 4, 0.25, 0.5)).to(mag.dtype)
    eighths = torch.round(mag / step).mul_(step).clamp_(max=7.5).mul_(8)
    return eighths, q < 0, e


def _dequantised(x):
    out = []
    for rows in x.split(max(1, (1 << 26) // x.shape[1])):
        eighths, neg, e = _quantised(rows)
        v = torch.ldexp(torch.where(neg, -eighths, eighths) / 8, e[..., None].double())
        out.append(v.view(rows.shape[0], -1)[:, :x.shape[1]])
    return torch.cat(out)


def _formatted(x):
    """(24 packed bytes of each 32-block [rows][nb][24], scale codes [rows][nb])."""
    eighths, neg, e = _quantised(x)
    v = eighths.to(torch.int32)
    # 0..15: the value is its own code; 16..30 by 2: exponent 2; 32..60 by 4: exponent 3
    code = torch.where(v < 16, v, torch.where(v < 32, 16 + (v - 16) // 2, 24 + (v - 32) // 4))
    code = (code | (neg.to(torch.int32) << 5)).view(*v.shape[:2], 8, 4)
    word = code[..., 0] | code[..., 1] << 6 | code[..., 2] << 12 | code[..., 3] << 18
    packed = torch.stack([word & 255, word >> 8 & 255, word >> 16], -1).to(torch.uint8)
    return packed.view(*v.shape[:2], 24), (e + 127).to(torch.uint8)


def _tiled(scales, dim, Kp, group):
    """Scale codes [dim][Kp/32] as (group of 32-row blocks, K-tile of 192, half, row, slab, row
    block of the group in whole dwords); 127 past the last row."""
    groups = -(-dim // (32 * group))
    s = torch.nn.functional.pad(scales, (0, 0, 0, groups * 32 * group - dim), value=127)
    s = s.view(groups, group, 32, Kp // 192, 3, 2).permute(0, 3, 5, 2, 4, 1)
    return torch.nn.functional.pad(s, (0, -group % 4)).reshape(-1)


def exact(case, seed):
    K = case["K"]
    if case["kind"] in ("prep_a", "prep_b"):
        a, dim, Kp = case["kind"] == "prep_a", case["dim"], -(-K // 192) * 192
        x = _prep_input(case, seed)
        x = x if a else x.t()
        parts = [_formatted(rows) for rows in x.split(max(1, (1 << 26) // K))]
        packed, scales = torch.cat([p[0] for p in parts]), torch.cat([p[1] for p in parts])
        more = Kp // 32 - scales.shape[1]
        packed = torch.nn.functional.pad(packed, (0, 0, 0, more))
        tiled = _tiled(torch.nn.functional.pad(scales, (0, more), value=127), dim, Kp,
                       case["group"])
        if a:
            return [packed.view(-1), tiled]
        p = torch.nn.functional.pad(packed, (0, 0, 0, 0, 0, -dim % 32))
        p = p.view(-1, 32, Kp // 64, 2, 24).permute(0, 2, 3, 1, 4)  # [n/32][k/64][half][column][24]
        p = torch.cat([p[..., :16].flatten(2), p[..., 16:].flatten(2)], -1)
        return [p.reshape(-1), tiled]
    A, B = _operands(case, seed)
    a = _dequantised(A)
    del A
    b = _dequantised(B.t().contiguous())
    del B
    return a @ b.t()
