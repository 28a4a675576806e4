"""The plan of the wide-workgroup GEMMs (hip_compiler tile_plan / tile_group) and their tile order, on the CPU."""

import ctypes
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def order(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    so = str(tmp_path_factory.mktemp("order") / "liborder.so")
    subprocess.run(["g++", "-O2", "-shared", "-fPIC", "-I", os.path.join(HERE, "..", "pytorch-apple_amd", "csrc", "kernels"),
                    os.path.join(HERE, "tile_host.cpp"), "-o", so], check=True)
    lib = ctypes.CDLL(so)

    def f(gx, gy, gz, gn):
        out = (ctypes.c_uint * (3 * gx * gy * gz))()
        lib.order(gx, gy, gz, gn, out)
        return [tuple(out[i:i + 3]) for i in range(0, len(out), 3)]

    return f


def test_tile_order_covers_every_tile_once(order):
    """The grouped tile order (tile.hip's own, built for the host) over grids that do and do not divide by 8 or by the
    group: every (row tile, column tile, split) exactly once, and each XCD's share one stretch of the order."""
    for gx, gy, gz, gn in ((11, 16, 1, 5), (63, 8, 1, 1), (16, 16, 1, 7), (1, 1, 1, 1), (13, 3, 5, 4), (7, 9, 2, 7)):
        tiles = order(gx, gy, gz, gn)
        assert sorted(tiles) == [(m, n, z) for m in range(gy) for n in range(gx) for z in range(gz)]
        in_order = [(m, n, z) for z in range(gz) for g in range(0, gx, gn) for m in range(gy)
                    for n in range(g, min(g + gn, gx))]
        assert [t for xcd in range(8) for t in tiles[xcd::8]] == in_order


@pytest.mark.parametrize("kind,bounds", [("one", ()), ("silu", ()), ("grp", (1536, 1792)), ("grp", (512, 576))])
def test_plan_covers_the_product(kind, bounds):
    """Any size: the tile is one of the kernels, splits tile K exactly and stay within the scratch limit,
    groups lie within the grid."""
    from hip_compiler.subgraph_analyzer import GEMM_MIN_KCHUNK, TILE_COST, TILE_MAX_PART, tile_group, tile_plan

    for M in (1, 16, 33, 63, 64, 65, 129, 300, 1000, 4096, 70000):
        for N in (1, 8, 96, 513, 1536, 2048, 8960, 151936):
            for K in (64, 128, 320, 1536, 8960):
                bm, bn, waves, ks = tile_plan(M, N, K, kind, bounds)
                assert (bm, bn, waves) in TILE_COST[kind] and not any(b % bn for b in bounds)
                chunk = -(-(K // 64) // ks) * 64
                assert ks == 1 or (kind == "one" and (ks - 1) * chunk < K <= ks * chunk and chunk >= GEMM_MIN_KCHUNK
                                   and ks * M * N * 4 <= TILE_MAX_PART)
                assert 1 <= tile_group(M, N, bm, bn, 2 if kind == "silu" else 1, ks) <= -(-N // bn)


@pytest.mark.parametrize("kind,N,K,rows,tile", [
    ("silu", 8960, 1536, (129, 160, 192, 256), (128, 80)),       # on 64 x 64, one per CU, 420 tiles were two rounds
    ("silu", 8960, 1536, (513, 640, 768), (192, 144)),
    ("silu", 8960, 1536, (1025, 1088, 1152, 1280), (192, 144)),  # on 128 x 144 three rounds
    ("one", 1536, 1536, (1025, 1152, 1281), (64, 64)),           # two per CU: one round of half-size workgroups
])
def test_rows_just_past_a_full_round(kind, N, K, rows, tile):
    """Row counts just past a full round of the larger tiles take tiles that fill the CUs again, not a
    nearly empty last round of the larger ones."""
    from hip_compiler.subgraph_analyzer import tile_plan

    for M in rows:
        assert tile_plan(M, N, K, kind)[:2] == tile, M


def test_two_workgroups_per_cu_are_one_round():
    """The second pair of a TILE_COST entry: 257 to 512 workgroups are one round of shared CUs, and what is
    left of a round goes at the rate of a CU to each."""
    from hip_compiler.subgraph_analyzer import TILE_COST, tile_us

    tile = (64, 64, 8)
    step, fixed, step2, fixed2 = TILE_COST["one"][tile]
    alone, both = 10 * step + fixed, 10 * step2 + fixed2
    for wgs, us in ((1, alone), (256, alone), (257, both), (512, both), (600, both + alone), (1024, 2 * both)):
        assert tile_us("one", tile, wgs, 10) == pytest.approx(us)
    assert tile_us("one", (128, 128, 8), 257, 10) == pytest.approx(2 * tile_us("one", (128, 128, 8), 256, 10))


@pytest.mark.parametrize("N,HW,C,Cout,k,kernel,ksplit", [
    (4, 56, 128, 64, 3, "k_gemm_f16_convg_m64n64_w8_k64d", 1),        # 196 tiles of 64 x 64: within a round
    (11, 56, 128, 64, 3, "k_gemm_f16_convg_m128n64_k64d2", 1),        # 539: no half-empty 128-column tiles
    (64, 28, 256, 32, 3, "k_gemm_f16_convg_m128n64_k64d2", 1),
    (16, 56, 128, 72, 3, "k_gemm_f16_convg_m128n128_w8_k64d", 1),
    (16, 56, 1088, 64, 1, "k_gemm_f16_conv_m128n64_k64d2", 1),
    (1, 16, 2048, 2048, 1, "k_gemm_f16_conv_m64n64_w8_k64d", 1),      # the gathers' rates split K four ways here
])
def test_long_k_convolutions_take_the_tiles_that_fit_their_channels(N, HW, C, Cout, k, kernel, ksplit):
    from hip_compiler import compile_subgraph
    from test_gpu_parity import _conv_chain_ir

    prog = compile_subgraph(_conv_chain_ir(N, 64, HW, HW, C, Cout, k, 1, k // 2, False))
    (step,) = [s for s in prog.steps if s.kind == "conv" and s.args.get("N") == Cout and s.module in ("gemm", "tile")]
    assert (step.kernel, step.args["ksplit"]) == (kernel, ksplit)
