"""The framework's work as a user's program has it: one dict per case, over the whole range of calls.

``listed()`` names the measured cases, ``draw()`` gives more of the same ranges; ``prepare()`` makes
what a program holds before the call (patched modules, inputs, a captured decode step), ``run()`` is
one pass through the public entry points, ``exact()`` the same values in 64 bits from plain torch.

Four kinds of pass:

* ``decode``: one token step through a stack of expert layers (1-8 tokens), eager as a generate loop
  calls it or replayed from the HIP graph that a serving program captured once.
* ``forward``: one expert layer on a batch of tokens: a serving batch (tens to hundreds of tokens)
  or a prompt (hundreds to thousands), bare or through an ``ExpertsLoRA`` with a trained adapter.
* ``train``: forward and backward of one ``ExpertsLoRA`` layer: gradients of the tokens, of the
  router weights (they depend on the tokens even where the router is frozen) and of the adapters.
* ``quantize``: ``from_float`` of one layer's expert stacks, what loading a model does per layer.
"""
import math

import torch

import experts4bit_qlora_amd as e4b

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}

# (experts, hidden, intermediate, top-k, weights renormalised): OLMoE-1B-7B, Qwen3-30B-A3B and
# gpt-oss-20b layers, and a small generic one whose widths are multiples of 64 but not of 128
GEOMETRY = {
    "olmoe": (64, 2048, 1024, 8, False),
    "qwen3": (128, 2048, 768, 8, True),
    "gptoss": (32, 2880, 2880, 4, True),
    "small": (16, 1216, 704, 4, True),
}
ALPHA, LIMIT = 1.702, 7.0  # gpt-oss clamped GLU


def _case(kind, name=None, **kw):
    c = {"kind": kind, "geometry": "olmoe", "fmt": "nf4", "dtype": "bf16", "tokens": 1, "layers": 1, "graph": False,
         "rank": 0, "adapter": "fp32", "zipf": 0.0}
    c.update(kw)
    return c if name is None else {"name": name, **c}


def listed():
    return [
        # one token through the 16 layers of OLMoE, replayed from the serving program's graph
        _case("decode", "decode_1_olmoe", layers=16, graph=True),
        # the same step with a trained rank-16 adapter served unmerged
        _case("decode", "decode_1_olmoe_lora", layers=16, graph=True, rank=16),
        # a few sequences at once, eager (a generate loop), double-quantized absmax
        _case("decode", "decode_5_qwen3_dq", geometry="qwen3", fmt="nf4_dq", tokens=5, layers=8),
        # MXFP4 experts with biases and the clamped GLU, eager
        _case("decode", "decode_3_gptoss", geometry="gptoss", fmt="mxfp4", tokens=3, layers=4),
        # a serving batch: every expert has a few rows
        _case("forward", "batch_37_qwen3_dq", geometry="qwen3", fmt="nf4_dq", tokens=37),
        # a larger batch from an fp16 model
        _case("forward", "batch_150_olmoe_fp16", tokens=150, dtype="fp16"),
        # a long prompt with skewed expert popularity
        _case("forward", "prefill_4096_qwen3_dq", geometry="qwen3", fmt="nf4_dq", tokens=4096, zipf=1.1),
        # a prompt through MXFP4 experts
        _case("forward", "prefill_2048_gptoss", geometry="gptoss", fmt="mxfp4", tokens=2048),
        # a prompt of odd length through a trained adapter
        _case("forward", "prefill_1531_olmoe_lora", tokens=1531, rank=16),
        # one micro-batch of fine-tuning: the step this project is named for
        _case("train", "train_2048_olmoe", tokens=2048, rank=16),
        # a short odd sequence, double-quantized base, bf16 adapters of a larger rank
        _case("train", "train_509_qwen3_dq", geometry="qwen3", fmt="nf4_dq", tokens=509, rank=32, adapter="bf16",
              zipf=0.7),
        # loading: one layer's dense bf16 expert stacks to NF4
        _case("quantize", "quantize_olmoe"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("decode", "decode", "forward", "forward", "forward", "train", "train", "quantize"))
    geometry = rng.choice(("olmoe", "qwen3", "gptoss", "small"))
    fmt = "mxfp4" if geometry == "gptoss" else rng.choice(("nf4", "nf4_dq"))
    dtype = rng.choice(("bf16", "bf16", "bf16", "fp16"))
    rank = rng.choice((0, 0, 8, 16, 32, 64)) if fmt != "mxfp4" else 0
    adapter = rng.choice(("fp32", "bf16"))
    zipf = rng.choice((0.0, round(rng.uniform(0.3, 1.2), 2)))
    if kind == "quantize":
        if geometry == "gptoss":
            geometry, fmt = "small", "nf4"
        return _case(kind, geometry=geometry, fmt=fmt, dtype=rng.choice(("bf16", "fp16", "fp32")))
    if kind == "train":
        if geometry == "gptoss":
            geometry, fmt = "olmoe", "nf4"
        return _case(kind, geometry=geometry, fmt=fmt, dtype=dtype, tokens=_log_int(rng, 48, 2048),
                     rank=rng.choice((8, 12, 16, 32, 64)), adapter=adapter, zipf=zipf)
    if kind == "decode":
        return _case(kind, geometry=geometry, fmt=fmt, dtype=dtype, tokens=rng.randint(1, 8), layers=rng.randint(4, 8),
                     graph=rng.random() < 0.5, rank=rank, adapter=adapter, zipf=zipf)
    return _case(kind, geometry=geometry, fmt=fmt, dtype=dtype, tokens=_log_int(rng, 9, 4096 if fmt != "mxfp4" else 2048),
                 rank=rank, adapter=adapter, zipf=zipf)


# ------------------------------------------------------------------------------ inputs

_NF4 = (-1.0, -0.6961928009986877, -0.5250730514526367, -0.39491748809814453, -0.28444138169288635,
        -0.18477343022823334, -0.09105003625154495, 0.0, 0.07958029955625534, 0.16093020141124725,
        0.24611230194568634, 0.33791524171829224, 0.44070982933044434, 0.5626170039176941, 0.7229568362236023, 1.0)
_E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0)


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _dynamic_map():
    """The signed dynamic 8-bit map that double-quantized absmax codes index."""
    vals = [0.0, 1.0]
    for i in range(7):
        b = torch.linspace(0.1, 1, 2 ** i + 1)
        m = ((b[:-1] + b[1:]) / 2 * 10 ** (i - 6)).tolist()
        vals += m + [-v for v in m]
    return torch.tensor(sorted(vals + [0.0] * (256 - len(vals))), dtype=torch.float32)


def _nf4_stack(E, n, k, g, dq):
    """Packed NF4 bytes and scales of an N(0, 0.02) stack, as a checkpoint holds them."""
    code = torch.tensor(_NF4, device=DEV)
    mids = (code[:-1] + code[1:]) / 2
    packed = torch.empty(E, n * k // 2, dtype=torch.uint8, device=DEV)
    absmax = torch.empty(E, n * k // 64, device=DEV)
    for e0 in range(0, E, 16):
        w = torch.randn(min(16, E - e0), n * k // 64, 64, generator=g, device=DEV) * 0.02
        am = w.abs().amax(-1)
        q = torch.bucketize(w / am.unsqueeze(-1), mids, out_int32=True).to(torch.uint8).reshape(w.shape[0], -1)
        packed[e0:e0 + 16] = (q[:, 0::2] << 4) | q[:, 1::2]
        absmax[e0:e0 + 16] = am
    if not dq:
        return {"packed": packed, "absmax": absmax}
    offset = absmax.mean(-1)
    c2 = _dynamic_map().to(DEV)
    nb = absmax.shape[1]
    c = torch.nn.functional.pad(absmax - offset[:, None], (0, -nb % 256)).reshape(E, -1, 256)
    a2 = c.abs().amax(-1)
    q = torch.bucketize(c / a2.unsqueeze(-1), (c2[:-1] + c2[1:]) / 2, out_int32=True).to(torch.uint8)
    return {"packed": packed, "absmax": q.reshape(E, -1)[:, :nb].contiguous(), "absmax2": a2, "offset": offset}


def _mxfp4_stack(E, n, k, g):
    """e2m1 blocks ``[E, n, k / 32, 16]`` and e8m0 scales ``[E, n, k / 32]`` of an N(0, 0.02) stack."""
    mids = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], device=DEV)
    blocks = torch.empty(E, n, k // 32, 16, dtype=torch.uint8, device=DEV)
    scales = torch.empty(E, n, k // 32, dtype=torch.uint8, device=DEV)
    for e0 in range(0, E, 8):
        w = torch.randn(min(8, E - e0), n, k // 32, 32, generator=g, device=DEV) * 0.02
        x = torch.floor(torch.log2(w.abs().amax(-1))) - 2
        w = torch.ldexp(w, -x.unsqueeze(-1))
        q = torch.bucketize(w.abs(), mids, out_int32=True).to(torch.uint8) | ((w < 0).to(torch.uint8) << 3)
        blocks[e0:e0 + 8] = (q[..., 1::2] << 4) | q[..., 0::2]
        scales[e0:e0 + 8] = (x + 127).to(torch.uint8)
    return {"blocks": blocks, "scales": scales}


def _weights(case, seed):
    """Stored weights of each layer, and its adapter."""
    E, H, I, _, _ = GEOMETRY[case["geometry"]]
    out = []
    for l in range(case["layers"]):
        g = _gen(1000 * seed + l)
        if case["fmt"] == "mxfp4":
            d = {"up": _mxfp4_stack(E, 2 * I, H, g), "down": _mxfp4_stack(E, H, I, g)}
            d["up_bias"] = (torch.randn(E, 2 * I, generator=g, device=DEV) * 0.02).to(DTYPES[case["dtype"]])
            d["down_bias"] = (torch.randn(E, H, generator=g, device=DEV) * 0.02).to(DTYPES[case["dtype"]])
        else:
            dq = case["fmt"] == "nf4_dq"
            d = {"up": _nf4_stack(E, 2 * I, H, g, dq), "down": _nf4_stack(E, H, I, g, dq)}
        r = case["rank"]
        if r:
            adt = DTYPES[case["adapter"]]

            def normal(*shape, std):
                return (torch.randn(*shape, generator=g, device=DEV) * std).to(adt)

            d["lora"] = {"gate_up_lora_A": normal(E, r, H, std=1 / r), "gate_up_lora_B": normal(E, 2 * I, r, std=0.02),
                         "down_lora_A": normal(E, r, I, std=1 / r), "down_lora_B": normal(E, H, r, std=0.02)}
        out.append(d)
    return out


def _tokens(case, seed):
    """Per layer: activations after a norm, the router's ids and weights, and (training) the output's gradient."""
    E, H, _, k, renorm = GEOMETRY[case["geometry"]]
    dt, T = DTYPES[case["dtype"]], case["tokens"]
    out = []
    for l in range(case["layers"]):
        g = _gen(1000 * seed + 500 + l)
        x = torch.randn(T, H, generator=g, device=DEV).to(dt)
        logits = torch.randn(T, E, generator=g, device=DEV)
        if case["zipf"]:
            rank = torch.randperm(E, generator=g, device=DEV) + 1
            logits = logits - case["zipf"] * torch.log(rank.float())
        w, idx = torch.topk(torch.softmax(logits, -1), k, dim=-1)
        if renorm:
            w = w / w.sum(-1, keepdim=True)
        grad = torch.randn(T, H, generator=g, device=DEV).to(dt) if case["kind"] == "train" else None
        out.append((x, idx, w.to(dt), grad))
    return out


def _dense(case, seed):
    E, H, I, _, _ = GEOMETRY[case["geometry"]]
    g = _gen(seed)
    return [torch.randn(E, n, k, generator=g, device=DEV, dtype=torch.float32).mul_(0.02).to(DTYPES[case["dtype"]])
            for n, k in ((2 * I, H), (H, I))]


def _module(case, d):
    """One expert layer over the stored weights, through the loaders a program uses."""
    E, H, I, _, _ = GEOMETRY[case["geometry"]]
    cd = DTYPES[case["dtype"]]
    if case["fmt"] == "mxfp4":
        return e4b.GptOssExpertsMxfp4.from_gptoss_mxfp4(
            d["up"]["blocks"], d["up"]["scales"], d["up_bias"], d["down"]["blocks"], d["down"]["scales"], d["down_bias"],
            alpha=ALPHA, limit=LIMIT, compute_dtype=cd)
    mod = e4b.Experts4bit(E, H, I, compute_dtype=cd, quant_type="nf4", device=DEV,
                          compress_statistics=case["fmt"] == "nf4_dq")
    state = {}
    for name, s in (("gate_up", d["up"]), ("down", d["down"])):
        state[f"{name}_proj"], state[f"{name}_absmax"] = s["packed"], s["absmax"]
        if "offset" in s:
            state[f"{name}_absmax2"], state[f"{name}_absmax_offset"] = s["absmax2"], s["offset"]
    mod.load_state_dict({**mod.state_dict(), **state})
    if case["rank"]:
        mod = e4b.ExpertsLoRA(mod, r=case["rank"], alpha=2 * case["rank"], dtype=DTYPES[case["adapter"]]).to(DEV)
        mod.load_state_dict({**mod.state_dict(), **d["lora"]})
    return mod


def prepare(case, seed):
    if case["kind"] == "quantize":
        return {"case": case, "dense": _dense(case, seed)}
    mods = [_module(case, d) for d in _weights(case, seed)]
    inputs = _tokens(case, seed)
    state = {"case": case, "mods": mods, "inputs": inputs}
    if case["kind"] == "train":
        mods[0].train()
        assert e4b.enable_fast_train(mods[0]) == 1
        x, idx, w, grad = inputs[0]
        state["inputs"] = [(x.requires_grad_(), idx, w.requires_grad_(), grad)]
        return state
    for m in mods:
        m.eval()
        assert e4b.enable_fast(m) == 1
    if case["graph"]:  # the serving program's decode step, captured once
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for _ in range(2):
                _forward(state)
        torch.cuda.current_stream().wait_stream(side)
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]):
            state["out"] = _forward(state)
    return state


# ------------------------------------------------------------------------------- passes


def _forward(state):
    with torch.no_grad():
        return [m(x, idx, w) for m, (x, idx, w, _) in zip(state["mods"], state["inputs"])]


def run(state):
    kind = state["case"]["kind"]
    if kind == "quantize":
        mod = e4b.Experts4bit.from_float(*state["dense"], compute_dtype=torch.bfloat16,
                                         compress_statistics=state["case"]["fmt"] == "nf4_dq")
        return {k: v for k, v in mod.state_dict().items() if torch.is_tensor(v)}
    if kind == "train":
        mod = state["mods"][0]
        x, idx, w, grad = state["inputs"][0]
        x.grad = w.grad = None
        mod.zero_grad(set_to_none=True)
        out = mod(x, idx, w)
        out.backward(grad)
        return {"out": out.detach(), "x": x.grad, "router": w.grad,
                **{n: p.grad for n, p in mod.named_parameters() if p.grad is not None}}
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    return _forward(state)


def work(case):
    """Bytes: the routed experts' stored weights, adapters, activations and outputs, once each
    (training: both directions read the weights; gradients are outputs). Flops: the projections
    of every routed row and the adapters' products."""
    E, H, I, k, _ = GEOMETRY[case["geometry"]]
    T, r, L = case["tokens"], case["rank"], case["layers"]
    scale = {"nf4": 4 / 64, "nf4_dq": 1 / 64 + 4 / (64 * 256), "mxfp4": 1 / 32}[case["fmt"]]
    per_value = 0.5 + scale
    if case["kind"] == "quantize":
        n = E * 3 * I * H
        return {"bytes": n * (per_value + DTYPES[case["dtype"]].itemsize), "flops": 3.0 * n}
    p = [1.0 / (e + 1) ** case["zipf"] for e in range(E)]  # the chance that a token's k ids hold an expert
    hit = sum(1 - (1 - min(1.0, k * v / sum(p))) ** T for v in p)
    M, it = T * k, DTYPES[case["dtype"]].itemsize
    weights = hit * 3 * I * H * per_value
    ab = hit * r * (H + 2 * I + I + H) * DTYPES[case["adapter"]].itemsize
    tokens = 2 * T * H * it + M * 8 + M * it
    flops = M * (6.0 * I * H + 2 * r * (H + 2 * I + I + H))
    if case["kind"] == "train":
        ab_grad = E * r * (2 * H + 3 * I) * DTYPES[case["adapter"]].itemsize
        return {"bytes": 2 * weights + ab + ab_grad + 2 * tokens, "flops": M * (12.0 * I * H + 6 * r * (2 * H + 3 * I))}
    return {"bytes": L * (weights + ab + tokens), "flops": L * flops}


def tolerance(case):
    if case["kind"] == "quantize":
        return "exact"
    # measured against exact(): forward 2.3e-3 to 3.6e-3 in bf16 and 5e-4 in fp16 (h and the output are
    # rounded), training 4.4e-3 to 5.2e-3 in bf16; four times that
    rel = 0.02 if case["kind"] == "train" else 0.012
    if case["dtype"] == "fp16":
        rel /= 6
    return {"rel": rel, "max": 20 * rel}


# ------------------------------------------------------------------- 64-bit plain torch


def _dense64(case, d, which, e):
    """Expert e's dense weight in 64 bits from its stored bytes."""
    E, H, I, _, _ = GEOMETRY[case["geometry"]]
    n, k = (2 * I, H) if which == "up" else (H, I)
    s = d[which]
    if case["fmt"] == "mxfp4":
        b = s["blocks"][e].long()
        v = torch.tensor(_E2M1, dtype=torch.float64, device=DEV)[torch.stack([b & 15, b >> 4], -1)].reshape(n, k // 32, 32)
        return (v * torch.pow(2.0, s["scales"][e].double() - 127).unsqueeze(-1)).reshape(n, k)
    b = s["packed"][e].long()
    v = torch.tensor(_NF4, dtype=torch.float32).double().to(DEV)[torch.stack([b >> 4, b & 15], -1)].reshape(-1, 64)
    am = s["absmax"][e]
    if "offset" in s:
        a2 = s["absmax2"][e].double().repeat_interleave(256)[:am.numel()]
        am = _dynamic_map().double().to(DEV)[am.long()] * a2 + s["offset"][e].double()
    return (v * am.double()[:, None]).reshape(n, k)


def _layer64(case, d, x, idx, w, adapter):
    out = torch.zeros_like(x)
    scaling = 2.0
    for e in torch.unique(idx).tolist():
        tok, slot = torch.where(idx == e)
        rows = x[tok]
        proj = rows @ _dense64(case, d, "up", e).T
        if adapter:
            proj = proj + scaling * (rows @ adapter["gate_up_lora_A"][e].T) @ adapter["gate_up_lora_B"][e].T
        if case["fmt"] == "mxfp4":
            proj = proj + d["up_bias"][e].double()
            gate, up = proj[:, 0::2].clamp(max=LIMIT), proj[:, 1::2].clamp(min=-LIMIT, max=LIMIT)
            h = (up + 1) * gate * torch.sigmoid(ALPHA * gate)
        else:
            gate, up = proj.chunk(2, dim=-1)
            h = gate * torch.sigmoid(gate) * up
        down = h @ _dense64(case, d, "down", e).T
        if adapter:
            down = down + scaling * (h @ adapter["down_lora_A"][e].T) @ adapter["down_lora_B"][e].T
        if case["fmt"] == "mxfp4":
            down = down + d["down_bias"][e].double()
        out = out.index_add(0, tok, down * w[tok, slot].unsqueeze(-1))
    return out


def exact(case, seed):
    if case["kind"] == "quantize":
        return None
    outs = []
    for d, (x, idx, w, grad) in zip(_weights(case, seed), _tokens(case, seed)):
        x, w = x.double(), w.double()
        adapter = {n: p.double() for n, p in d["lora"].items()} if case["rank"] else None
        if case["kind"] == "train":
            leaves = [x, w, *adapter.values()]
            for t in leaves:
                t.requires_grad_()
            out = _layer64(case, d, x, idx, w, adapter)
            out.backward(grad.double())
            return {"out": out.detach(), "x": x.grad, "router": w.grad, **{n: p.grad for n, p in adapter.items()}}
        with torch.no_grad():
            outs.append(_layer64(case, d, x, idx, w, adapter))
    return outs
