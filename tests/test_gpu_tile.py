"""The wide-workgroup MFMA GEMMs (csrc/kernels/tile.hip) against float64 products of the same values:
every tile shape with each epilogue, at sizes one past and one short of a tile, rows that are no
multiple of 16 bytes, the shortest K, a K of more stages than the LDS ring holds, and split K.

The bounds are the kernels' own rounding points. With u the unit roundoff of the type (2^-8 for
bfloat16, 2^-11 for float16) and s the fp32 sum's error, at most K 2^-24 sum |x w|:
  bias   |out - y| <= u |y| + s
  resid  |out - (r + y)| <= u |y| + u |r + y| + 2 s
  silu   |out - silu(g) h| <= u (1.1 |g| |h| + 4 |out|) + 2 s (1 + |g| + |h|): silu' is at most 1.1 in
         size, and g, h, silu(g) and the product are each rounded once
"""

import numpy as np
import pytest
import torch

from conftest import gpu_available

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a ROCm GPU")]


def _tiles():
    from hip_compiler.subgraph_analyzer import TILE_COST

    return [(kind, t) for kind in ("one", "silu") for t in TILE_COST[kind]]


def _run(ir, inputs, backend):
    from hip_compiler import compile_subgraph, is_hip_op_supported
    from npu_compiler import partition
    from npu_runtime import DAGExecutor

    ex = DAGExecutor(partition(ir, is_hip_op_supported), backend, compile_fn=compile_subgraph)
    ex.load_weights({})
    out = ex.execute({k: backend.allocate_buffer(v) for k, v in inputs.items()})
    torch.cuda.synchronize()
    (prog,) = ex.npu_programs.values()
    return {k: v.to_torch().clone() for k, v in out.items()}, prog


def _graph(epi, M, N, K, dtype, bias):
    from irgen.builder import IRBuilder
    from irgen.qwen import linear

    b = IRBuilder("tile")
    x, w = b.input("x", [M, K], dtype), b.input("w", [N, K], dtype)
    bv = b.input("b", [N], dtype) if bias else None
    y = linear(b, x, w, bv)
    if epi == "resid":
        y = b.op("aten.add.Tensor", [b.input("r", [M, N], dtype), y])
    if epi == "silu":
        w2 = b.input("w2", [N, K], dtype)
        b2 = b.input("b2", [N], dtype) if bias else None
        y = b.op("aten.mul.Tensor", [b.op("aten.silu.default", [y]), linear(b, x, w2, b2)])
    b.output(y)
    return b.to_dict()


def _check(epi, M, N, K, dtype, bias, backend, tile=None, ksplit=None):
    ir = _graph(epi, M, N, K, dtype, bias)
    td = {"bfloat16": torch.bfloat16, "float16": torch.float16}[dtype]
    g = torch.Generator(device="cuda").manual_seed(M * 7 + N * 3 + K)
    mk = lambda *s, std=1.0: (std * torch.randn(s, generator=g, device="cuda")).to(td)
    ins = {"x": mk(M, K), "w": mk(N, K, std=K ** -0.5)}
    if bias:
        ins["b"] = mk(N)
    if epi == "resid":
        ins["r"] = mk(M, N)
    if epi == "silu":
        ins["w2"] = mk(N, K, std=K ** -0.5)
        if bias:
            ins["b2"] = mk(N)
    print(f"[case] tile {epi} {M}x{N}x{K} {dtype} bias={bias} tile={tile} ksplit={ksplit}", flush=True)
    got, prog = _run(ir, ins, backend)
    main = [s for s in prog.steps if s.module == "tile"]
    assert len(main) == 1 and main[0].kernel.endswith("_k64d"), [s.kernel for s in prog.steps]
    if tile:
        assert main[0].params["tile"] == tile[:2] and main[0].block[0] == 64 * tile[2]
    if ksplit:
        assert main[0].args["ksplit"] == ksplit
    (out,) = got.values()
    d = {k: v.double() for k, v in ins.items()}
    u = 2.0 ** -8 if dtype == "bfloat16" else 2.0 ** -11
    y = d["x"] @ d["w"].T + (d["b"] if bias else 0.0)
    s = K * 2.0 ** -24 * (d["x"].abs() @ d["w"].abs().T + 1.0)
    if epi == "bias":
        ref, tol = y, u * y.abs() + s
    elif epi == "resid":
        ref = d["r"] + y
        tol = u * (y.abs() + ref.abs()) + 2 * s
    else:
        h = d["x"] @ d["w2"].T + (d["b2"] if bias else 0.0)
        s = torch.maximum(s, K * 2.0 ** -24 * (d["x"].abs() @ d["w2"].abs().T + 1.0))
        ref = y * torch.sigmoid(y) * h
        tol = u * (1.1 * y.abs() * h.abs() + 4 * ref.abs()) + 2 * s * (1 + y.abs() + h.abs())
    tol = 1.02 * tol + 1e-6   # second-order terms of the roundings; the smallest float16 spacing
    bad = (out.double() - ref).abs() > tol
    assert not bad.any(), (int(bad.sum()), bad.nonzero()[0].tolist())


@pytest.mark.parametrize("kind,tile", _tiles() if gpu_available() else [])
def test_every_tile_shape_at_its_edges(backend, kind, tile, monkeypatch):
    """One tile shape forced: a row and 8 columns past a tile with a K of many stages, one row and one
    column short (rows of odd length: the element-wise stores), and the shortest K."""
    import hip_compiler.subgraph_analyzer as SA

    monkeypatch.setitem(SA.TILE_COST, kind, {tile: SA.TILE_COST[kind][tile]})
    monkeypatch.setattr(SA, "TILE_MAX_SPLIT", 1)
    bm, bn, _ = tile
    m0 = max(1, -(-129 // bm))   # past the rows of the skinny and wide kernels
    for M, N, K in ((m0 * bm + 1, 2 * bn + 8, 64 * 11), (m0 * bm + bm - 1, 3 * bn - 1, 192), (m0 * bm, bn, 64)):
        for epi in (("bias", "resid") if kind == "one" else ("silu",)):
            _check(epi, M, N, K, "bfloat16", True, backend, tile)
        if kind == "one":
            _check("bias", M, N, K, "float16", N % 2 == 0, backend, tile)


@pytest.mark.parametrize("ks,M,N,K", [(3, 130, 200, 64 * 13), (5, 257, 1004, 64 * 20), (16, 129, 99, 64 * 64)])
def test_split_k_partials(backend, ks, M, N, K, monkeypatch):
    """fp32 partials of each split (an uneven last one; N % 4 != 0: element-wise partials) and their reduce."""
    import hip_compiler.subgraph_analyzer as SA

    real = SA.tile_plan
    monkeypatch.setattr(SA, "tile_plan", lambda *a, **k: real(*a, **k)[:3] + (ks,))
    for epi in ("bias", "resid"):
        _check(epi, M, N, K, "bfloat16", True, backend, ksplit=ks)


def test_grouped_projections_do_not_depend_on_the_tile(backend, monkeypatch):
    """q | k | v of a prefill layer with each grouped tile: K is summed in the same order whatever the
    tile, so logits and caches are bit-identical."""
    import hip_compiler.subgraph_analyzer as SA
    from irgen.qwen import QwenConfig, build_decode_ir
    from irgen.workloads import make_weights, prefill_inputs

    cfg = QwenConfig(layers=1, vocab=4096)
    T = 129
    ir = build_decode_ir(132, cfg, tokens=T)
    w, x = make_weights(ir, cfg, norm_std=0.02, device="cuda"), prefill_inputs(T, 132, cfg, device="cuda")
    from hip_compiler import compile_subgraph, is_hip_op_supported
    from npu_compiler import partition
    from npu_runtime import DAGExecutor

    outs, real = [], dict(SA.TILE_COST["grp"])
    for tile in real:
        monkeypatch.setitem(SA.TILE_COST, "grp", {tile: real[tile]})
        print(f"[case] grouped projections, tile {tile}", flush=True)
        ex = DAGExecutor(partition(ir, is_hip_op_supported), backend, compile_fn=compile_subgraph)
        ex.load_weights(w)
        out = ex.execute({k: backend.allocate_buffer(v.clone()) for k, v in x.items()})
        (prog,) = ex.npu_programs.values()
        assert f"k_gemm_bf16_grp_m{tile[0]}n{tile[1]}_k64d" in [s.kernel for s in prog.steps]
        outs.append({k: v.to_numpy() for k, v in out.items()})
    for o in outs[1:]:
        assert all(np.array_equal(o[k], outs[0][k]) for k in o)


def test_silu_of_every_16_bit_value(backend):
    """gm_silu over every finite bfloat16 value, through a one-column-of-ones product: at most one unit
    in the last place from the correctly rounded float64 value (the library form's own distance)."""
    K, N = 64, 8
    vals = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    vals = vals[torch.isfinite(vals) & (vals.abs() < 3e38)]
    M = vals.numel()
    x = torch.zeros(M, K, dtype=torch.bfloat16)
    x[:, 0], x[:, 1] = vals, 1.0
    w, w2 = torch.zeros(N, K, dtype=torch.bfloat16), torch.zeros(N, K, dtype=torch.bfloat16)
    w[:, 0], w2[:, 1] = 1.0, 1.0
    print(f"[case] silu of {M} values", flush=True)
    got, prog = _run(_graph("silu", M, N, K, "bfloat16", False), {"x": x.cuda(), "w": w.cuda(), "w2": w2.cuda()}, backend)
    (out,) = got.values()
    v = vals.double()
    ref = v * torch.sigmoid(v)
    out = out.cpu().double()
    assert all(torch.equal(out[:, 0], out[:, j]) for j in range(1, N))
    # one unit in the last place of bfloat16. From v = -128 ln 2 = -88.7 on the fraction's denominator
    # (2^(-v log2 e - 2) + 1/4) passes 2^126 and its reciprocal is flushed to zero, and so the result,
    # 88.7 e^-88.7 = 2^-121.5 at most (expf overflows at the same place); everything smaller may be too
    tol = torch.maximum(ref.abs() * 2.0 ** -7, torch.full_like(ref, 2.0 ** -121))
    assert ((out[:, 0] - ref).abs() <= tol).all()
    exact = ref.bfloat16().double()
    assert ((out[:, 0] != exact) & (ref.abs() > 2.0 ** -121)).sum() <= 24   # 17 measured, as with expf and /


@pytest.mark.parametrize("tile", [(64, 64, 8), (64, 128, 8), (128, 128, 8)])
@pytest.mark.parametrize("N,H,W,C,Cout,k,stride,pad,add,dtype,ks", [
    (1, 7, 7, 192, 96, 3, 1, 1, True, "float16", 1),      # 49 pixels, padded taps on every side, residual
    (3, 9, 11, 128, 200, 3, 2, 1, False, "float16", 3),   # stride 2, odd sizes, ragged columns, split K
    (2, 8, 9, 1088, 72, 1, 1, 0, True, "bfloat16", 1),    # the image rows as they are, 17 steps
    (2, 13, 6, 1152, 68, 1, 2, 0, False, "float16", 2),   # strided 1 x 1; 68 columns: element-wise stores
    (1, 6, 5, 128, 64, 5, 1, 2, False, "bfloat16", 1),    # 5 x 5: more padding than the image's half
])
def test_long_k_convolutions(backend, N, H, W, C, Cout, k, stride, pad, add, dtype, ks, tile, monkeypatch):
    """Channels-last convs with K > 1024 (tile.hip's conv kernels) + batch norm (+ residual) + ReLU against
    float64. Bound: with y the conv, v = r(r(y) a + b) (+ r): u |y| |a| + u |v| + u |out|, fp32 sums as above."""
    import hip_compiler.subgraph_analyzer as SA
    from irgen.builder import IRBuilder

    monkeypatch.setattr(SA, "tile_plan", lambda M, n, K, kind, *a, **kw: tile + (ks,))
    monkeypatch.setattr(SA, "CONV_TILE_MIN_WGS", 1)
    td, u = (torch.float16, 2.0 ** -11) if dtype == "float16" else (torch.bfloat16, 2.0 ** -8)
    g = torch.Generator(device="cuda").manual_seed(C + Cout)
    rn = lambda *s, std=1.0, mean=0.0: (mean + std * torch.randn(s, generator=g, device="cuda")).to(td)
    b = IRBuilder("conv")
    x = b.input("x", [N, 64, H, W], dtype)
    ident = b.weight("w0", [C, 64, 1, 1], dtype)   # a 1 x 1 that copies channels first: its output is channels-last
    norm = lambda y, n, sfx: b.op("aten.batch_norm.default", [y] + [b.weight(q + sfx, [n], dtype) for q in (
        "g", "beta", "mu", "var")], {"training": False, "momentum": 0.1, "eps": 1e-5, "cudnn_enabled": True})
    h = b.op("aten.conv2d.default", [x, ident], {"stride": [1, 1], "padding": [0, 0], "dilation": [1, 1], "groups": 1})
    h = b.op("aten.relu.default", [norm(h, C, "0")])   # (a factor of 1 / sqrt(1 + 1e-5): rounded away)
    w = b.weight("w", [Cout, C, k, k], dtype)
    y = b.op("aten.conv2d.default", [h, w], {"stride": [stride, stride], "padding": [pad, pad], "dilation": [1, 1],
                                             "groups": 1})
    y = norm(y, Cout, "")
    if add:
        y = b.op("aten.add.Tensor", [y, b.input("r", list(y.shape), dtype)])
    b.output(b.op("aten.relu.default", [y]))
    ir = b.to_dict()
    K = C * k * k
    pick = torch.arange(C) % 64
    ws = {"w0": torch.eye(64, device="cuda")[pick.cuda()].reshape(C, 64, 1, 1).to(td), "w": rn(Cout, C, k, k, std=K ** -0.5),
          "g": rn(Cout, std=0.1, mean=1.0), "beta": rn(Cout, std=0.1), "mu": rn(Cout, std=0.1),
          "var": (torch.rand(Cout, generator=g, device="cuda") + 0.5).to(td)}
    one, zero = torch.ones(C, dtype=td, device="cuda"), torch.zeros(C, dtype=td, device="cuda")
    ws.update(g0=one, beta0=zero, mu0=zero, var0=one)
    ins = {"x": rn(N, 64, H, W).abs()}
    if add:
        ins["r"] = rn(*[N, Cout, (H + 2 * pad - k) // stride + 1, (W + 2 * pad - k) // stride + 1])
    print(f"[case] conv {N}x{C}x{H}x{W} -> {Cout} k{k} s{stride} p{pad} {dtype} tile {tile} ks {ks}", flush=True)
    from hip_compiler import compile_subgraph, is_hip_op_supported
    from npu_compiler import partition
    from npu_runtime import DAGExecutor

    ex = DAGExecutor(partition(ir, is_hip_op_supported), backend, compile_fn=compile_subgraph)
    ex.load_weights(ws)
    (out,) = ex.execute({n: backend.allocate_buffer(v) for n, v in ins.items()}).values()
    (prog,) = ex.npu_programs.values()
    main = [s for s in prog.steps if s.module == "tile" and s.params["kernel"] == [k, k] and s.args["N"] == Cout]
    assert main and main[-1].kernel.endswith("_w8_k64d") and main[-1].args["ksplit"] == ks
    d = {n: v.double().cpu() for n, v in {**ws, **ins}.items()}
    d["x"] = d["x"][:, pick]
    conv = lambda t, f: torch.nn.functional.conv2d(t, f, stride=stride, padding=pad)
    yy, mag = conv(d["x"], d["w"]), conv(d["x"], d["w"].abs())
    col = lambda t: t.reshape(1, -1, 1, 1)
    a = d["g"] / torch.sqrt(d["var"] + 1e-5)
    v = yy * col(a) + col(d["beta"] - d["mu"] * a)
    ref = v + (d["r"] if add else 0.0)
    s32 = K * 2.0 ** -24 * (mag + 1.0)
    tol = 1.02 * (u * (yy.abs() * col(a).abs() + v.abs() + ref.abs()) + s32 * (1 + col(a).abs())) + 1e-6
    bad = (out.to_torch().cpu().double() - ref.clamp(min=0)).abs() > tol
    assert not bad.any(), (int(bad.sum()), bad.nonzero()[0].tolist())
