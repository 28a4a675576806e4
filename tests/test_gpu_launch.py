"""Launch lists run directly and as HIP graphs give the same results, whichever buffers change."""

import pytest
import torch

from conftest import gpu_available

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a ROCm GPU")]


def test_direct_and_graph_launches_agree_when_buffers_change(backend):
    """An MLP block (two launches: direct by default) fed from two input buffers in turn, then with new
    weights and the old ones again: every result equals the graph executor's and the single-buffer one."""
    from hip_compiler import compile_subgraph, is_hip_op_supported
    from hip_runtime.hip_executor import GRAPH_MIN_STEPS
    from irgen.qwen import QwenConfig, build_mlp_ir
    from irgen.workloads import make_weights, mlp_inputs
    from npu_compiler import partition
    from npu_runtime import DAGExecutor

    cfg = QwenConfig(hidden=512, intermediate=1024)
    ir = build_mlp_ir(1, cfg)
    ws = [make_weights(ir, cfg, seed=s, norm_std=0.02, device="cuda") for s in (0, 7)]
    xs = [backend.allocate_buffer(mlp_inputs(1, cfg, seed=s)["x"].cuda()) for s in (1, 2)]
    runs = {}
    for graph in (False, True):
        ex = DAGExecutor(partition(ir, is_hip_op_supported), backend, compile_fn=compile_subgraph)
        (hexec,) = ex.npu_executors.values()
        assert len(hexec.program.steps) < GRAPH_MIN_STEPS and hexec.use_graph is False
        hexec.use_graph = graph
        out = []
        for w, x in ((0, 0), (0, 1), (0, 0), (1, 0), (1, 1), (0, 1)):
            print(f"[case] graph={graph} weights {w} input {x}", flush=True)
            ex.load_weights(ws[w])
            (y,) = ex.execute({"x": xs[x]}).values()
            out.append(y.to_torch().clone())
        assert bool(hexec._graphs) == graph
        assert torch.equal(out[0], out[2]) and torch.equal(out[1], out[5])
        assert not torch.equal(out[0], out[1]) and not torch.equal(out[0], out[3])
        runs[graph] = out
    assert all(torch.equal(a, b) for a, b in zip(runs[False], runs[True]))


def test_short_launches_become_a_graph_on_their_second_call(backend):
    """A list of 13 short launches (a two-layer decode without the one-launch step): a pointer set's first call
    is launched directly, its second captured and its third the same graph, with equal results; another set
    starts directly again."""
    from hip_compiler import compile_subgraph, is_hip_op_supported
    from irgen.qwen import QwenConfig, build_decode_ir
    from irgen.workloads import decode_inputs, make_weights
    from npu_compiler import partition
    from npu_runtime import DAGExecutor

    cfg = QwenConfig(hidden=512, intermediate=1024, layers=2, heads=4, kv_heads=2, head_dim=128, vocab=4096)
    ir = build_decode_ir(256, cfg, argmax=True)
    ex = DAGExecutor(partition(ir, is_hip_op_supported), backend,
                     compile_fn=lambda sub: compile_subgraph(sub, persistent=False))
    ex.load_weights(make_weights(ir, cfg, device="cuda"))
    (hexec,) = ex.npu_executors.values()
    assert hexec.use_graph
    sets = [{k: backend.allocate_buffer(v.cuda()) for k, v in decode_inputs(256, 100, cfg, seed=s).items()} for s in (1, 2)]
    names, out, graphs = [o["name"] for o in ir["graph_outputs"]], [], []
    for i in (0, 0, 0, 1, 0, 1):
        print(f"[case] input set {i}", flush=True)
        y = ex.execute(sets[i])
        out.append([y[n].to_torch().clone() for n in names])
        graphs.append(len(hexec._graphs))
    assert graphs == [0, 1, 1, 1, 1, 2]
    for i, j in ((0, 1), (0, 2), (0, 4), (3, 5)):
        assert all(torch.equal(a, b) for a, b in zip(out[i], out[j]))
    assert not torch.equal(out[0][0], out[3][0])


@pytest.mark.parametrize("layers", [2, 7])
def test_calls_inside_a_callers_capture(backend, layers):
    """A list that runs as a graph by default (13 short launches, and more than 32), captured by its caller after
    calls that made the executor's own graph: every replay, with eager work and a synchronisation between, equals
    the eager result for the inputs the buffers hold then."""
    from hip_compiler import compile_subgraph, is_hip_op_supported
    from irgen.qwen import QwenConfig, build_decode_ir
    from irgen.workloads import decode_inputs, make_weights
    from npu_compiler import partition
    from npu_runtime import DAGExecutor

    cfg = QwenConfig(hidden=512, intermediate=1024, layers=layers, heads=4, kv_heads=2, head_dim=128, vocab=4096)
    ir = build_decode_ir(256, cfg, argmax=True)
    ex = DAGExecutor(partition(ir, is_hip_op_supported), backend,
                     compile_fn=lambda sub: compile_subgraph(sub, persistent=False))
    ex.load_weights(make_weights(ir, cfg, device="cuda"))
    (hexec,) = ex.npu_executors.values()
    assert hexec.use_graph and (len(hexec.program.steps) > 32) == (layers == 7)
    x = {k: backend.allocate_buffer(v.cuda()) for k, v in decode_inputs(256, 100, cfg, seed=1).items()}
    names = [o["name"] for o in ir["graph_outputs"]]
    read = lambda y: [y[n].to_torch().clone() for n in names]
    ids = x["input_ids"].native_handle
    want = []
    for tok in (3, 77, 1234):
        ids.fill_(tok)
        for _ in range(3):
            y = read(ex.execute(x))
        want.append(y)
    assert len(hexec._graphs) == 1
    print(f"[case] capture of {len(hexec.program.steps)} launches", flush=True)
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g):
        out = ex.execute(x)
    for rep in range(2):
        for tok, w in zip((3, 77, 1234), want):
            ids.fill_(tok)
            g.replay()
            torch.cuda.synchronize()
            assert all(torch.equal(a, b) for a, b in zip(read(out), w)), (rep, tok)
            assert all(torch.equal(a, b) for a, b in zip(read(ex.execute(x)), w)), (rep, tok)
