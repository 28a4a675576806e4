"""1 x 1 convolutions with a CU to each workgroup on the four-stage kernels, and the K-split rule of short K."""

import numpy as np
import pytest
import torch

from hip_compiler import subgraph_analyzer as SA

from test_gpu_parity import _conv_chain_ir, host, run_hip


@pytest.mark.gpu
@pytest.mark.parametrize("N,HW,C,Cout,add", [
    (1, 9, 128, 64, False),     # two K steps: fewer than the ring holds
    (1, 8, 192, 192, True),     # three steps: the ring exactly ahead; residual
    (2, 7, 256, 200, False),    # four steps: the first buffer is used twice
    (4, 32, 320, 256, False),   # five steps, 256 workgroups: the largest grid of the rule
    (3, 5, 960, 64, False),     # 15 steps, the longest K that is not split
])
def test_four_stage_1x1_conv_matches_two_stages(backend, monkeypatch, N, HW, C, Cout, add):
    """The same MFMAs in the same order: bit-identical to the two-stage kernels."""
    ir = _conv_chain_ir(N, 64, HW, HW, C, Cout, 1, 1, 0, add)
    g = torch.Generator().manual_seed(C + Cout)
    w = {}
    for i, (co, ci) in enumerate(((C, 64), (Cout, C))):
        w[f"w{i}"] = (ci ** -0.5 * torch.randn(co, ci, 1, 1, generator=g)).half()
        for n, m in (("g", 1.0), ("beta", 0.0), ("mu", 0.0)):
            w[f"{n}{i}"] = (m + 0.1 * torch.randn(co, generator=g)).half()
        w[f"var{i}"] = (0.5 + torch.rand(co, generator=g)).half()
    x = {"x": torch.randn(N, 64, HW, HW, generator=g).half()}
    print(f"[case] 1 x 1 conv {N}x{C}x{HW}x{HW} -> {Cout}, residual {add}", flush=True)
    outs, kernels = [], []
    for wgs in (0, SA.CONV_D_WGS):
        monkeypatch.setattr(SA, "CONV_D_WGS", wgs)
        got, ex = run_hip(ir, host(x), host(w), backend)
        (prog,) = ex.npu_programs.values()
        kernels.append([s for s in prog.steps if s.kind == "conv"][-1].kernel)
        outs.append(next(iter(got.values())))
    assert kernels[0].endswith("_m64n64_k64d2") and kernels[1].endswith("_m64n64_k64d"), kernels
    assert np.isfinite(np.asarray(outs[0], dtype=np.float32)).all() and np.array_equal(outs[0], outs[1])


def test_short_k_splits_only_over_few_tiles():
    for K, M, splits in ((960, 64, False), (1024, 63 * 64, True), (1024, 64 * 64, False), (1984, 64 * 64, False),
                         (2048, 64 * 64, True), (2048, 255 * 64, True)):
        assert (SA.conv_gemm_tiling(M, 64, K)[2] > 1) == splits, (K, M)
