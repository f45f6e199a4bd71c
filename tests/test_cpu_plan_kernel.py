"""mxfp6_plan_kernel, from the rules that the launches act on (csrc/tile_dispatch.hpp): which kernel a plan's
tile runs on, against the recorded times of the candidates."""
import math
import os

import pytest

PROFILE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "profiles",
                       "skinny_tiles_on_row_major_a.txt")
SHORT = PROFILE.replace("on_row_major_a", "short_k")


def _skinny_times():
    with open(PROFILE) as f:
        for line in f:
            if not line.startswith("#"):
                v = line.split()
                yield [int(x) for x in v[:7]], dict(zip(("slab", "stream", "wide"), map(float, v[7:])))


def _kernel(mx, M, N, K, MT, NT, S, **kw):
    return mx.plan_kernel(mx.OUT_BF16, M, N, mx.kpad(K), (MT, NT, MT // 32, NT // 128), S, **kw)


def test_skinny_tiles_run_on_the_faster_kernel(mx):
    """Of the recorded plans none runs slower on the kernel it is given than on the slab kernel (which
    the tiles ran on before, A repacked or not), nor more than 1.4 times the faster one of stream and
    wide, 1% on average."""
    over = []
    for (M, N, K, MT, NT, S, rp), t in _skinny_times():
        us = t[_kernel(mx, M, N, K, MT, NT, S)[0]]
        assert us <= 1.03 * t["slab"], (M, N, K, MT, NT, S, t)
        over.append(us / min(t["stream"], t["wide"]))
        assert over[-1] < 1.4, (M, N, K, MT, NT, S, t)
    assert len(over) > 400 and math.exp(sum(map(math.log, over)) / len(over)) < 1.01


def test_short_skinny_plans_run_on_the_faster_kernel(mx):
    """One to seven K-tiles a segment: none slower than on the slab kernel by more than 8%, 4% for one
    K-tile (and 0.2 us, the spread of the launches that set the times of about 4 us)."""
    n = 0
    with open(SHORT) as f:
        lines = [line.split() for line in f if not line.startswith("#")]
    for v in lines:
        nk, M, N, K, MT, NT, S = map(int, v[:7])
        us = float(v[{"slab": 7, "stream": 8, "wide": 9}[_kernel(mx, M, N, K, MT, NT, S)[0]]])
        assert us <= float(v[7]) * (1.04 if nk == 1 else 1.08) + 0.2, v
        n += 1
    assert n > 300


@pytest.mark.parametrize("MT,NT,want", [(64, 128, "slab"), (64, 256, "slab"), (32, 128, "stream"),
                                        (32, 256, "stream")])
def test_one_k_tile(mx, MT, NT, want):
    assert _kernel(mx, 320, 3584, 130, MT, NT, 1)[0] == want
    assert _kernel(mx, 96, 3584, 576, MT, NT, 3)[0] == want
    assert _kernel(mx, 320, 3584, 384, MT, NT, 1)[0] == "stream"
    assert _kernel(mx, 1120, 3712, 192, 32, 128, 1)[0] == "slab"
    assert _kernel(mx, 832, 9472, 192, 64, 256, 1)[0] == "slab"
    assert _kernel(mx, 832, 5248, 192, 64, 256, 1)[0] == "stream"
    assert _kernel(mx, 4096, 8192, 192, MT, NT, 1)[0] == "wide"


@pytest.mark.parametrize("MT,NT", [(32, 128), (32, 256), (64, 128), (64, 256)])
def test_one_row_of_tiles_is_streamed(mx, MT, NT):
    """A wide tile on one row of skinny tiles would be half to 31/32 repeated rows, however many
    columns and segments there are."""
    for N in (256, 4096, 28672, 32768, 65536, 102272):
        for M in (1, MT // 2 + 1, MT):
            for S in (1, 3, 8, 16):
                assert _kernel(mx, M, N, 28672, MT, NT, S)[0] == "stream", (M, N, S)


def test_long_rows_keep_the_tile(mx):
    """128 row offsets of the wide tile stay within 31 bits: longer rows run on the 32- and 64-row tiles."""
    args = (4096, 8192, 4096, 64, 256, 1)
    assert _kernel(mx, *args)[0] == "wide"
    assert _kernel(mx, *args, A_row_bytes=2**31 // 127 // 4 * 4)[0] == "wide"
    assert _kernel(mx, *args, A_row_bytes=2**31 // 127 // 4 * 4 + 4)[0] == "stream"


def test_other_layouts_and_tiles(mx):
    k = lambda tile, layout, S=1: mx.plan_kernel(mx.OUT_F16, 256, 6144, 4224, tile, S, layout)[0]  # noqa: E731
    assert k((64, 256, 2, 2), mx.A_REPACK) == k((32, 128, 1, 1), mx.A_PRESHUFFLED) == "slab"
    assert k((128, 128, 2, 2), mx.A_ROWS) == k((256, 256, 4, 4), mx.A_ROWS) == "slab"
    assert k((256, 192, 4, 3), mx.A_ROWS) == "slab"
    assert k((128, 256, 4, 2), mx.A_ROWS) == k((128, 384, 4, 3), mx.A_ROWS) == "band"
    assert k((128, 256, 4, 2), mx.A_REPACK) == "wide"
    assert k((32, 32, 1, 1), mx.A_ROWS, 8) == "tiny"
    for bad in ((256, 128, 4, 2), (64, 64, 2, 2)):
        with pytest.raises(ValueError):
            k(bad, mx.A_ROWS)
    with pytest.raises(ValueError):
        k((64, 256, 2, 2), mx.A_ROWS, 23)


def test_plans_say_what_runs(mx):
    """The recorded plans that repacked A for the slab kernel read its rows now: every query says so, the
    workspace holds the K segments only, and with those bytes the plan is the same one."""
    n = 0
    for (M, N, K, MT, NT, S, rp), _ in _skinny_times():
        if not rp:
            continue
        Kp, tile = mx.kpad(K), (MT, NT, MT // 32, NT // 128)
        assert not mx.repacks_a(M, N, Kp), (M, N, K)
        split = 4 * S * M * N if S > 1 else 0
        assert mx.workspace_size(M, N, Kp) == split
        assert mx.preferred_workspace_size(M, N, Kp) == -(-split // 256) * 256
        for ws in (split, 1 << 40):
            assert mx.gemm_plan(mx.OUT_F16, M, N, Kp, ws) == (tile, S, False), (M, N, K, ws)
        n += 1
    assert n > 200


def test_loaded_skinny_plan_reads_rows(mx, tmp_path):
    M, N, Kp = 3616, 5120, mx.kpad(4096)
    tile = mx.choose_tile(M, N, Kp)
    assert tile[0] <= 64
    f = tmp_path / "plans.txt"
    f.write_text(" ".join(map(str, (1, M, N, Kp, *tile, 1, 1))) + "\n")
    mx.tune_reset()
    try:
        assert mx.tune_load(str(f)) == (1, 0)
        assert mx.tuned_plan(1, M, N, Kp) == (tuple(tile), 1, False)
        assert mx.gemm_plan(1, M, N, Kp, 0) == (tuple(tile), 1, False)
    finally:
        mx.tune_reset()


@pytest.mark.parametrize("M,N,K,want", [(256, 256, 1024, "tiny_kernel"), (8192, 8192, 8192, "wide_kernel"),
                                        (2048, 5120, 105728, "wide_kernel"),
                                        (64, 28672, 8192, "stream_kernel"),
                                        (256, 18432, 12288, "stream_kernel")])
def test_bench_names_the_kernel(mx, M, N, K, want):
    import types
    import bench
    Kp = mx.kpad(K)
    w = types.SimpleNamespace(ot=mx.OUT_F16, M=M, N=N, tile=mx.choose_tile(M, N, Kp),
                              S=mx.splitk_segments(M, N, Kp), repack=mx.repacks_a(M, N, Kp),
                              p=types.SimpleNamespace(Kp=Kp, a_row_bytes=mx.packed_bytes(K)))
    assert bench.tile_kernel_name(w) == want
