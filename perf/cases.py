"""What is timed when this backend is measured: the calls a user's program makes, as cases.

A case is one graph of the ``irgen`` builders at one size, compiled through ``partition`` and
``DAGExecutor`` and run with ``DAGExecutor.execute`` on device buffers the program keeps (the
zero-copy calling convention of a serving loop). ``listed()`` holds the sizes the repository's own
benchmark and tests name plus ragged ones; ``draw`` spreads over the same ranges.

kinds:

* ``mlp``      RMSNorm -> gate/up -> SiLU * up -> down -> + residual on ``tokens`` rows: the larger half
               of a decoder layer, from one decode token to a long prompt.
* ``attention``one decode token's attention block over a cache of ``kv_len`` rows, all open (q/k/v, RoPE,
               cache update in place, GQA attention, o_proj).
* ``decode``   one step of the whole model over a static cache of ``kv_len`` rows at position ``pos``:
               logits, updated caches and the greedy token.
* ``prefill``  ``tokens`` prompt tokens through ``layers`` decoder layers and the head over a static cache
               of ``kv_len`` rows (a padded prompt of a generation, or a prompt scored at every position).
* ``resnet``   a ResNet-50 forward of ``batch`` images of ``image`` x ``image`` pixels, float16.
"""

from __future__ import annotations

import math
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "pytorch-apple_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

HIDDEN, INTER, HEADS, KV_HEADS, HEAD_DIM, VOCAB, LAYERS = 1536, 8960, 12, 2, 128, 151936, 28
EPS, THETA = 1e-6, 1e6
SMALL_VOCAB = 4096      # heads of the few-layer prefill cases: the layers are what they time
RESNET_BLOCKS, RESNET_WIDTHS, CLASSES = (3, 4, 6, 3), (64, 128, 256, 512), 1000


def listed():
    return [
        # one decode token through the MLP: the smallest call, two launches
        {"name": "mlp_t1", "kind": "mlp", "tokens": 1},
        # a small batch of sequences, or the verification of a few speculated tokens
        {"name": "mlp_t16", "kind": "mlp", "tokens": 16},
        # a short padded prompt
        {"name": "mlp_t128", "kind": "mlp", "tokens": 128},
        # a ragged prompt, no multiple of any tile
        {"name": "mlp_t1000", "kind": "mlp", "tokens": 1000},
        # one decode token's attention over an odd cache
        {"name": "attention_kv1025", "kind": "attention", "kv_len": 1025},
        # the headline: one decode step of the whole model near the end of a 2048-position cache
        {"name": "decode_kv2048", "kind": "decode", "layers": LAYERS, "kv_len": 2048, "pos": 2015},
        # decoder layers over a long cache that is nearly full (the layers the long context weighs on)
        {"name": "decode_kv32768", "kind": "decode", "layers": 4, "kv_len": 32768, "pos": 32639},
        # time to first token: a prompt padded to 128 tokens over the generation's cache
        {"name": "prefill_t128", "kind": "prefill", "layers": 4, "vocab": VOCAB, "tokens": 128, "kv_len": 2048},
        # a 512-token prompt scored at every position, the real head with a quarter of the layers (over
        # all 28, two correct bf16 evaluations drift apart by nearly 3%)
        {"name": "prefill_t512", "kind": "prefill", "layers": 7, "vocab": VOCAB, "tokens": 512, "kv_len": 512},
        # decoder layers over a long ragged prompt
        {"name": "prefill_t2000", "kind": "prefill", "layers": 2, "vocab": SMALL_VOCAB, "tokens": 2000, "kv_len": 2048},
        # one image: latency of a network of small launches
        {"name": "resnet_b1", "kind": "resnet", "batch": 1, "image": 224},
        # the benchmark's batch
        {"name": "resnet_b32", "kind": "resnet", "batch": 32, "image": 224},
    ]


def _log(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["mlp", "mlp", "attention", "decode", "prefill", "prefill", "resnet"])
    if kind == "mlp":
        return {"kind": kind, "tokens": _log(rng, 1, 4096)}
    if kind == "attention":
        return {"kind": kind, "kv_len": _log(rng, 16, 16384)}
    if kind == "decode":
        kv = _log(rng, 64, 32768)
        return {"kind": kind, "layers": rng.randint(1, 4), "kv_len": kv, "pos": rng.randint(kv // 2, kv - 1)}
    if kind == "prefill":
        t = _log(rng, 16, 2048)
        kv = t if rng.random() < 0.5 else min(4096, t + rng.randint(1, 2048))
        kv += -kv % 4           # prefill attention reads its 16-bit mask in rows of a multiple of 4
        return {"kind": kind, "layers": rng.randint(1, 2), "vocab": SMALL_VOCAB, "tokens": t, "kv_len": kv}
    return {"kind": kind, "batch": _log(rng, 1, 32), "image": rng.randint(64, 224)}


# ---------------------------------------------------------------- inputs, from the seed alone

def _gen(seed, salt):
    return torch.Generator(device="cuda").manual_seed(1_000_003 * int(seed) + salt)


def _normal(shape, std, dtype, gen, mean=0.0):
    return torch.randn(shape, generator=gen, device="cuda").mul_(std).add_(mean).to(dtype)


def _inv_freq():
    i = torch.arange(0, HEAD_DIM, 2, dtype=torch.float64, device="cuda")
    return (THETA ** (-i / HEAD_DIM)).float()


def _attention_weights(pre, gen):
    bf, nq, nk = torch.bfloat16, HEADS * HEAD_DIM, KV_HEADS * HEAD_DIM
    w = {}
    for name, n in (("q_proj", nq), ("k_proj", nk), ("v_proj", nk)):
        w[f"{pre}{name}.weight"] = _normal((n, HIDDEN), 0.02, bf, gen)
        w[f"{pre}{name}.bias"] = _normal((n,), 0.02, bf, gen)
    w[f"{pre}o_proj.weight"] = _normal((HIDDEN, nq), 0.02, bf, gen)
    return w


def _mlp_weights(pre, gen):
    bf = torch.bfloat16
    return {f"{pre}gate_proj.weight": _normal((INTER, HIDDEN), 0.02, bf, gen),
            f"{pre}up_proj.weight": _normal((INTER, HIDDEN), 0.02, bf, gen),
            f"{pre}down_proj.weight": _normal((HIDDEN, INTER), 0.02, bf, gen)}


def _norm_weight(gen):
    return _normal((HIDDEN,), 0.02, torch.bfloat16, gen, mean=1.0)


def _model_weights(case, gen):
    w = {"model.embed_tokens.weight": _normal((case.get("vocab", VOCAB), HIDDEN), 0.02, torch.bfloat16, gen),
         "model.rotary_emb.inv_freq": _inv_freq(), "model.norm.weight": _norm_weight(gen)}
    for li in range(case["layers"]):
        pre = f"model.layers.{li}."
        w[pre + "input_layernorm.weight"] = _norm_weight(gen)
        w[pre + "post_attention_layernorm.weight"] = _norm_weight(gen)
        w.update(_attention_weights(pre + "self_attn.", gen))
        w.update(_mlp_weights(pre + "mlp.", gen))
    return w


def _convs(case):
    """(key, cin, cout, kernel, stride, padding, input size) of every convolution, in graph order."""
    size = (case["image"] + 6 - 7) // 2 + 1
    out = [("conv1", 3, 64, 7, 2, 3, case["image"])]
    size = (size + 2 - 3) // 2 + 1
    cin = 64
    for si, (n, width) in enumerate(zip(RESNET_BLOCKS, RESNET_WIDTHS)):
        for bi in range(n):
            key, stride = f"layer{si + 1}.{bi}", 2 if bi == 0 and si > 0 else 1
            after = (size + 2 - 3) // stride + 1
            out += [(key + ".conv1", cin, width, 1, 1, 0, size), (key + ".conv2", width, width, 3, stride, 1, size),
                    (key + ".conv3", width, 4 * width, 1, 1, 0, after)]
            if bi == 0:
                out.append((key + ".downsample.0", cin, 4 * width, 1, stride, 0, size))
            cin, size = 4 * width, after
    return out


def _bn_key(conv):
    return conv.replace("downsample.0", "downsample.1") if "downsample" in conv else conv.replace("conv", "bn")


def _resnet_weights(case, gen):
    h = torch.float16
    w = {}
    for key, cin, cout, k, _, _, _ in _convs(case):
        w[key + ".weight"] = _normal((cout, cin, k, k), (2.0 / (cin * k * k)) ** 0.5, h, gen)
        bn = _bn_key(key)
        # the last batch norm of a block starts small, so that activations keep their size with depth
        w[bn + ".weight"] = torch.full((cout,), 0.25 if ".conv3" in key else 1.0, dtype=h, device="cuda")
        w[bn + ".bias"] = torch.zeros((cout,), dtype=h, device="cuda")
        w[bn + ".running_mean"] = _normal((cout,), 0.1, h, gen)
        w[bn + ".running_var"] = (torch.rand((cout,), generator=gen, device="cuda") + 0.5).to(h)
    w["fc.weight"] = _normal((CLASSES, 2048), 0.01, h, gen)
    w["fc.bias"] = torch.zeros((CLASSES,), dtype=h, device="cuda")
    return w


def _weights(case, seed):
    gen = _gen(seed, 1)
    if case["kind"] == "mlp":
        return {"post_attention_layernorm.weight": _norm_weight(gen), **_mlp_weights("mlp.", gen)}
    if case["kind"] == "attention":
        return {"model.rotary_emb.inv_freq": _inv_freq(), **_attention_weights("model.layers.0.self_attn.", gen)}
    return _resnet_weights(case, gen) if case["kind"] == "resnet" else _model_weights(case, gen)


def _inputs(case, seed):
    gen, bf = _gen(seed, 2), torch.bfloat16
    if case["kind"] == "mlp":
        return {"x": _normal((case["tokens"], HIDDEN), 1.0, bf, gen)}
    if case["kind"] == "resnet":
        return {"x": _normal((case["batch"], 3, case["image"], case["image"]), 1.0, torch.float16, gen)}
    S, T = case["kv_len"], case.get("tokens", 1)
    first = {"prefill": 0, "decode": case.get("pos"), "attention": S - 1}[case["kind"]]
    at = torch.arange(first, first + T, dtype=torch.int64, device="cuda")
    mask = torch.zeros((T, S), device="cuda").masked_fill_(torch.arange(S, device="cuda")[None, :] > at[:, None], -math.inf)
    d = {"attention_mask": mask.to(bf).reshape(1, 1, T, S), "position_ids": at.reshape(1, T), "cache_position": at.clone()}
    if case["kind"] == "attention":
        d["hidden_states"] = _normal((1, 1, HIDDEN), 1.0, bf, gen)
    else:
        d["input_ids"] = torch.randint(0, case.get("vocab", VOCAB), (1, T), generator=gen, device="cuda")
    for li in range(case.get("layers", 1)):
        for kind in ("key", "value"):   # the rows before the call's own tokens are filled
            t = torch.zeros((1, KV_HEADS, S, HEAD_DIM), dtype=bf, device="cuda")
            t[:, :, :first] = _normal((1, KV_HEADS, first, HEAD_DIM), 1.0, bf, gen)
            d[f"past_{kind}_{li}"] = t
    return d


# ---------------------------------------------------------------- the calls

def _graph(case):
    from irgen.qwen import QwenConfig, build_attention_ir, build_decode_ir, build_mlp_ir
    from irgen.resnet import build_resnet50_ir

    if case["kind"] == "mlp":
        return build_mlp_ir(case["tokens"])
    if case["kind"] == "attention":
        return build_attention_ir(case["kv_len"])
    if case["kind"] == "resnet":
        return build_resnet50_ir(case["batch"], case["image"])
    cfg = QwenConfig(layers=case["layers"], vocab=case.get("vocab", VOCAB))
    return build_decode_ir(case["kv_len"], cfg, argmax=True, tokens=case.get("tokens", 1))


def prepare(case, seed):
    from hip_compiler import compile_subgraph, is_hip_op_supported
    from hip_runtime import HIPBackend
    from npu_compiler import partition
    from npu_runtime import DAGExecutor

    ir, backend = _graph(case), HIPBackend(0)
    ex = DAGExecutor(partition(ir, is_hip_op_supported), backend, compile_fn=compile_subgraph)
    ex.load_weights(_weights(case, seed))
    inputs = {k: backend.allocate_buffer(v) for k, v in _inputs(case, seed).items()}
    names = [o["name"] for o in ir["graph_outputs"]]
    if case["kind"] == "prefill":
        # the last output is the greedy token of every position: over hundreds of them several are
        # near ties that fall either way, and the logits they are taken from are returned whole
        names = names[:-1]
    return {"executor": ex, "inputs": inputs, "outputs": names}


def run(state):
    out = state["executor"].execute(state["inputs"])
    return [out[name].to_torch() for name in state["outputs"]]


# ---------------------------------------------------------------- what a pass cannot do without

def _layer_weights():
    nq, nk = HEADS * HEAD_DIM, KV_HEADS * HEAD_DIM
    return HIDDEN * nq + 2 * HIDDEN * nk + nq + 2 * nk + nq * HIDDEN + 3 * HIDDEN * INTER + 2 * HIDDEN


def work(case):
    kind = case["kind"]
    if kind == "mlp":
        T = case["tokens"]
        return {"bytes": 2 * (3 * HIDDEN * INTER + HIDDEN + 2 * T * HIDDEN), "flops": 6 * T * HIDDEN * INTER}
    if kind == "resnet":
        convs, n = _convs(case), case["batch"]
        flops = sum(2 * n * cin * cout * k * k * ((s + 2 * p - k) // st + 1) ** 2 for _, cin, cout, k, st, p, s in convs)
        weights = sum(cin * cout * k * k + 4 * cout for _, cin, cout, k, _, _, _ in convs) + 2048 * CLASSES + CLASSES
        return {"bytes": 2 * (weights + 3 * n * case["image"] ** 2 + n * CLASSES), "flops": flops + 2 * n * 2048 * CLASSES}
    S, nq, nk = case["kv_len"], HEADS * HEAD_DIM, KV_HEADS * HEAD_DIM
    if kind == "attention":
        w = HIDDEN * nq + 2 * HIDDEN * nk + nq + 2 * nk + nq * HIDDEN
        return {"bytes": 2 * (w + 2 * nk * S + 2 * nk + S + 2 * HIDDEN), "flops": 2 * w + 4 * nq * S}
    T, L, V = case.get("tokens", 1), case["layers"], case.get("vocab", VOCAB)
    first = case.get("pos", 0)
    pairs = T * first + T * (T + 1) // 2          # (query, open position) pairs
    rows = first + T                              # cache rows read, the call's own among them
    tables = V * HIDDEN + T * HIDDEN + HIDDEN     # the head, the tokens' embedding rows, the last norm
    size = L * _layer_weights() + tables + L * 2 * nk * (rows + T) + T * S + T * V
    return {"bytes": 2 * size, "flops": 2 * T * (L * _layer_weights() + V * HIDDEN) + L * 4 * nq * pairs}


def tolerance(case):
    """About four times what the same graph with its sums in another order (other tiles and splits,
    the launch list instead of the one-launch step) was measured to differ by: relative 2-norm / largest
    difference 4e-5 / 8e-3 for the MLP, 4e-4 / 1.6e-3 for ResNet-50, 4.5e-3 / 3e-2 for two decoder
    layers, 1.3e-2 / 0.12 for four to eight, 2.3e-2 / 0.1 for the 28-layer decode step. The MLP's and
    the attention block's are stated as what one more or one less 16-bit rounding inside gives
    (their distance to 64 bits is 3.4e-3 and 5.1e-3)."""
    kind = case["kind"]
    if kind == "mlp":
        return {"rel": 1e-3, "max": 0.04}
    if kind == "attention":
        return {"rel": 0.01, "max": 0.06}
    if kind == "resnet":
        return {"rel": 2e-3, "max": 0.01}
    return {"rel": 0.02 if case["layers"] <= 2 and kind == "prefill" else 0.03, "max": 0.5, "differ": 0.0}


# ---------------------------------------------------------------- the same in 64 bits

def _rms64(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _mlp64(w, pre, x, norm):
    h = _rms64(x, norm)
    act = torch.nn.functional.silu(h @ w[pre + "gate_proj.weight"].double().T) * (h @ w[pre + "up_proj.weight"].double().T)
    return x + act @ w[pre + "down_proj.weight"].double().T


def _attention64(w, pre, x, inp, li):
    """x [T, hidden] -> the block's output [T, hidden] and the updated caches."""
    T, S = x.shape[0], inp["attention_mask"].shape[-1]

    def heads(name, n):
        return (x @ w[f"{pre}{name}.weight"].double().T + w[f"{pre}{name}.bias"].double()).reshape(T, n, HEAD_DIM).transpose(0, 1)

    at = inp["position_ids"].reshape(-1)
    ang = at.double()[:, None] * w["model.rotary_emb.inv_freq"].double()[None, :]
    cos, sin = torch.cat([ang, ang], -1).cos(), torch.cat([ang, ang], -1).sin()

    def rotate(t):
        half = HEAD_DIM // 2
        return t * cos + torch.cat([-t[..., half:], t[..., :half]], -1) * sin

    q, k, v = rotate(heads("q_proj", HEADS)), rotate(heads("k_proj", KV_HEADS)), heads("v_proj", KV_HEADS)
    kc, vc = inp[f"past_key_{li}"][0].double(), inp[f"past_value_{li}"][0].double()
    kc[:, inp["cache_position"]], vc[:, inp["cache_position"]] = k, v
    mask = inp["attention_mask"].reshape(T, S).double()
    per, out = HEADS // KV_HEADS, []
    for h in range(HEADS):
        s = q[h] @ kc[h // per].T.contiguous() * HEAD_DIM ** -0.5 + mask
        out.append(torch.softmax(s, -1) @ vc[h // per])
    o = torch.stack(out, 1).reshape(T, HEADS * HEAD_DIM)
    return o @ w[pre + "o_proj.weight"].double().T, kc[None], vc[None]


def _model64(case, w, inp):
    T = case.get("tokens", 1)
    x = w["model.embed_tokens.weight"][inp["input_ids"].reshape(-1)].double()
    caches = []
    for li in range(case["layers"]):
        pre = f"model.layers.{li}."
        a, kc, vc = _attention64(w, pre + "self_attn.", _rms64(x, w[pre + "input_layernorm.weight"]), inp, li)
        x = _mlp64(w, pre + "mlp.", x + a, w[pre + "post_attention_layernorm.weight"])
        caches += [kc, vc]
    logits = _rms64(x, w["model.norm.weight"]) @ w["model.embed_tokens.weight"].double().T
    token = [None] if case["kind"] == "decode" else []      # the greedy token: a tie may fall either way
    return [logits.reshape(1, T, -1)] + caches + token


def _conv64(x, w, k, stride, pad):
    """conv2d as one product per image over its unfolded taps."""
    n, _, h, wd = x.shape
    ho, wo = (h + 2 * pad - k) // stride + 1, (wd + 2 * pad - k) // stride + 1
    m = w.double().reshape(w.shape[0], -1)
    cols = [torch.nn.functional.unfold(x[i:i + 1], k, padding=pad, stride=stride)[0] for i in range(n)]
    return torch.stack([(m @ c).reshape(w.shape[0], ho, wo) for c in cols])


def _resnet64(case, w, x):
    shape = {key: (k, st, p) for key, _, _, k, st, p, _ in _convs(case)}

    def conv_bn(x, key):
        bn = _bn_key(key)
        g, b, m, v = (w[f"{bn}.{n}"].double().reshape(1, -1, 1, 1) for n in ("weight", "bias", "running_mean", "running_var"))
        return (_conv64(x, w[key + ".weight"], *shape[key]) - m) / torch.sqrt(v + 1e-5) * g + b

    h = torch.relu(conv_bn(x.double(), "conv1"))
    h = torch.nn.functional.max_pool2d(h, 3, 2, 1)
    for si, n in enumerate(RESNET_BLOCKS):
        for bi in range(n):
            key = f"layer{si + 1}.{bi}"
            y = torch.relu(conv_bn(h, key + ".conv1"))
            y = conv_bn(torch.relu(conv_bn(y, key + ".conv2")), key + ".conv3")
            h = torch.relu(y + (conv_bn(h, key + ".downsample.0") if bi == 0 else h))
    return [h.mean((2, 3)) @ w["fc.weight"].double().T + w["fc.bias"].double()]


def exact(case, seed):
    w, inp = _weights(case, seed), _inputs(case, seed)
    if case["kind"] == "mlp":
        return [_mlp64(w, "mlp.", inp["x"].double(), w["post_attention_layernorm.weight"])]
    if case["kind"] == "attention":
        o, kc, vc = _attention64(w, "model.layers.0.self_attn.", inp["hidden_states"].reshape(1, HIDDEN).double(), inp, 0)
        return [o.reshape(1, 1, HIDDEN), kc, vc]
    if case["kind"] == "resnet":
        return _resnet64(case, w, inp["x"])
    return _model64(case, w, inp)
