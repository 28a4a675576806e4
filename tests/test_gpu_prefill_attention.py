"""k_attn_prefill over head groupings, types and masks at the edges of its 32 x 32 blocks, against float64.

With the scores rounded as the kernel rounds them (r(r(q.k) scale) + mask), what is left is the rounding
of P (at most u = 2^-8 of each term for bfloat16, 2^-11 for float16) and of the output, and the fp32
sums: |out - ref| <= 1.1 u (sum p |v| + |ref|), where a score that falls on the other side of a
rounding boundary moves by u |s|, so its probability by that factor: the bound takes u (1 + 2 max |s|)."""

import numpy as np
import pytest
import torch

from conftest import gpu_available

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a ROCm GPU")]


def _graph(T, S, H, KVH, dtype, mask_dtype):
    from irgen.builder import IRBuilder
    from irgen.qwen import repeat_kv

    b = IRBuilder("PrefillAttention")
    q, k, v = (b.input(n, s, dtype) for n, s in (("q", [1, H, T, 128]), ("k", [1, KVH, S, 128]), ("v", [1, KVH, S, 128])))
    kt = b.op("aten.transpose.int", [repeat_kv(b, k, H // KVH)], {"dim0": 2, "dim1": 3})
    sc = b.op("aten.mul.Tensor", [b.op("aten.matmul.default", [q, kt])], {"other": 128 ** -0.5})
    if mask_dtype:
        sc = b.op("aten.add.Tensor", [sc, b.input("mask", [1, 1, T, S], mask_dtype)])
    p = b.op("aten.softmax.int", [sc], {"dim": -1, "dtype": "float32"})
    p = b.op("aten.to.dtype", [p], {"dtype": dtype}, base="to")
    b.output(b.op("aten.matmul.default", [p, repeat_kv(b, v, H // KVH)]))
    return b.to_dict()


# causal over a prefix, a window that closes blocks in the middle and at the start, a fully open row next
# to a row open at one position, and the type's lowest value instead of -inf (rows where it is all there is)
def _mask(kind, T, S):
    t, s = torch.arange(T)[:, None], torch.arange(S)[None, :]
    m = torch.zeros(T, S)
    if kind == "causal":
        m[s > t + (S - T)] = -torch.inf
    elif kind == "window":
        m[(s > t + (S - T)) | (s < t + (S - T) - 40)] = -torch.inf
    elif kind == "one":
        m[1::2][:, :] = -torch.inf
        m[1::2, S // 2] = 0.0
    elif kind == "lowest":
        m[s > t] = torch.finfo(torch.bfloat16).min
        m[T // 2] = torch.finfo(torch.bfloat16).min
    elif kind == "bias":    # values in every open block
        m = -(t + (S - T) - s).clamp(min=0) / 64
        m[s > t + (S - T)] = -torch.inf
    elif kind == "mixed":   # open blocks, then values, then closed blocks, then values to the end
        m = torch.cos(0.37 * s + t) * (s >= 170)
        m[:, 400:520] = -torch.inf
    return m


@pytest.mark.parametrize("T,S,H,KVH,dtype,mask_dtype,kind", [
    (33, 36, 12, 2, "bfloat16", "bfloat16", "causal"),     # one query and one position past a block
    (31, 160, 12, 2, "bfloat16", "bfloat16", "causal"),    # fewer queries than a block, five position blocks
    (97, 300, 6, 1, "bfloat16", "bfloat16", "window"),
    (64, 292, 8, 4, "bfloat16", "bfloat16", "causal"),     # two heads per KV head
    (40, 129, 5, 5, "bfloat16", None, "open"),             # a KV head each, no mask, S % 32 = 1
    (65, 131, 4, 4, "bfloat16", "float32", "causal"),
    (45, 100, 12, 2, "bfloat16", "bfloat16", "one"),
    (45, 100, 12, 4, "bfloat16", "float32", "one"),
    (50, 132, 12, 2, "bfloat16", "bfloat16", "lowest"),
    (66, 260, 12, 2, "float16", "float16", "causal"),
    (34, 96, 4, 2, "float16", None, "open"),
    (45, 700, 12, 2, "bfloat16", "bfloat16", "bias"),      # mask values over several rounds of blocks
    (33, 644, 6, 1, "bfloat16", "bfloat16", "mixed"),
    (33, 644, 4, 2, "bfloat16", "float32", "mixed"),
    (40, 388, 12, 2, "float16", "float16", "mixed"),
])
@pytest.mark.parametrize("heads", [1, 2, 3])
def test_prefill_attention_vs_float64(backend, T, S, H, KVH, dtype, mask_dtype, kind, heads, monkeypatch):
    import hip_compiler.patterns as P
    from hip_compiler import compile_subgraph, is_hip_op_supported
    from npu_compiler import partition
    from npu_runtime import DAGExecutor

    if H // KVH % heads:
        pytest.skip("not a divisor of the head group")
    # the limit at which `heads` heads per workgroup are the fewest that fit it
    monkeypatch.setattr(P, "PREFILL_ATTN_WGS", -(-T // 32) * (H // heads))
    ir = _graph(T, S, H, KVH, dtype, mask_dtype)
    ex = DAGExecutor(partition(ir, is_hip_op_supported), backend, compile_fn=compile_subgraph)
    ex.load_weights({})
    td = getattr(torch, dtype)
    g = torch.Generator().manual_seed(T + S)
    x = {"q": torch.randn(1, H, T, 128, generator=g).to(td), "k": torch.randn(1, KVH, S, 128, generator=g).to(td),
         "v": torch.randn(1, KVH, S, 128, generator=g).to(td)}
    m = torch.zeros(T, S, dtype=torch.float64)
    if mask_dtype:
        x["mask"] = _mask(kind, T, S).to(getattr(torch, mask_dtype)).reshape(1, 1, T, S)
        m = x["mask"][0, 0].double()
    print(f"[case] prefill attention T={T} S={S} H={H}/{KVH} {dtype} mask {mask_dtype} {kind}", flush=True)
    (o,) = ex.execute({k: backend.allocate_buffer(v) for k, v in x.items()}).values()
    (prog,) = ex.npu_programs.values()
    (step,) = [s for s in prog.steps if s.kernel.startswith("k_attn_prefill")]
    assert step.block[0] == 256 * heads and step.grid[1] == H // heads
    assert step.kernel.endswith(f"_h{heads}") == (heads > 1)
    rd = lambda t: t.to(td).double()
    q, k, v = x["q"][0].double(), *(x[n][0].double().repeat_interleave(H // KVH, 0) for n in "kv")
    s = rd(rd(q @ k.transpose(1, 2)) * 128 ** -0.5)
    if mask_dtype:
        s = rd(s + m) if mask_dtype == dtype else (s + m).float().double()
    p = torch.softmax(s, -1)
    ref = p @ v
    u = 2.0 ** -8 if dtype == "bfloat16" else 2.0 ** -11
    big = torch.where(torch.isfinite(s) & (s > -1e30), s.abs(), 0.0).amax(-1, keepdim=True)
    tol = 1.1 * u * ((1 + 2 * big) * (p @ v.abs()) + ref.abs())
    err = (o.to_torch().cpu().double()[0] - ref).abs()
    assert (err <= tol).all(), float((err / tol).max())
    # on the whole the error is the roundings', far below that bound
    assert float((err ** 2).sum().sqrt() / ref.norm()) <= 1.5 * u
