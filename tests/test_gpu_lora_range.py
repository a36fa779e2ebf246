"""Adapters over expert weights, token rows and adapter values at the ends of the number range. The fp16
matrix-core mode scales its operands by powers of two and a delta is formed in those scaled sums, so
all-zero scales, tiny rows and infinities reach it at its largest and smallest factors."""
import pytest
import torch

import experts4bit_qlora_amd as e4b
from experts4bit_qlora_amd import train
from oracle_weights import oracle_weights

pytestmark = pytest.mark.gpu
DEV = "cuda"
ADAPTERS = ("gate_up_lora_A", "gate_up_lora_B", "down_lora_A", "down_lora_B")


def _announce(msg):
    print(f"[case] {msg}", flush=True)


def _rel(got, want):
    return ((got.double() - want).norm() / want.norm().clamp_min(1e-30)).item()


def _module(E, hid, inter, r, dq, alpha=None, gate_up=None, down=None):
    torch.manual_seed(31)
    gu = (torch.randn(E, 2 * inter, hid) * 0.05 if gate_up is None else gate_up).to(DEV)
    dn = (torch.randn(E, hid, inter) * 0.05 if down is None else down).to(DEV)
    base = e4b.Experts4bit.from_float(gu, dn, compute_dtype=torch.bfloat16, compress_statistics=dq)
    mod = e4b.ExpertsLoRA(base, r=r, alpha=2 * r if alpha is None else alpha, dtype=torch.float32).to(DEV)
    with torch.no_grad():
        for p in (mod.gate_up_lora_B, mod.down_lora_B):
            p.normal_(0, 0.02)
    return mod


def _layer_fp64(mod, x, idx, w, grad=None):
    """The layer over the oracle-decoded weights in fp64, and its gradients for ``grad``."""
    base = mod.base
    W1, W2 = ([torch.from_numpy(W[e]).double().to(DEV) for e in range(base.num_experts)] for W in oracle_weights(base))
    x, w = x.detach().double().requires_grad_(), w.detach().double().requires_grad_()
    p = {n: getattr(mod, n).detach().double().requires_grad_() for n in ADAPTERS}
    out = torch.zeros_like(x)
    for e in range(base.num_experts):
        tok, slot = torch.where(idx == e)
        xe = x[tok]
        proj = xe @ W1[e].T + mod.scaling * (xe @ p["gate_up_lora_A"][e].T) @ p["gate_up_lora_B"][e].T
        gate, up = proj.chunk(2, -1)
        h = torch.nn.functional.silu(gate) * up
        down = h @ W2[e].T + mod.scaling * (h @ p["down_lora_A"][e].T) @ p["down_lora_B"][e].T
        out = out.index_add(0, tok, down * w[tok, slot, None])
    if grad is None:
        return {"out": out.detach()}
    out.backward(grad.double())
    return {"out": out.detach(), "x": x.grad, "w": w.grad, **{n: p[n].grad for n in ADAPTERS}}


def _zeroed_stacks(E, hid, inter):
    """Expert 0 without a gate_up projection, expert 1 without a down projection, expert 2 without either."""
    torch.manual_seed(30)
    gu, dn = torch.randn(E, 2 * inter, hid) * 0.05, torch.randn(E, hid, inter) * 0.05
    gu[[0, 2]], dn[[1, 2]] = 0.0, 0.0
    return gu, dn


# 256-row tiles (and halved ones); 32-row tiles, K a multiple of 256; 32-row tiles, K off 256
SHAPES = [(1200, 4, 256, 256), (60, 6, 256, 256), (60, 6, 192, 320)]


@pytest.mark.parametrize("T,E,hid,inter", SHAPES)
@pytest.mark.parametrize("dq", (False, True))
@pytest.mark.parametrize("alpha", (32, 4096))
def test_training_with_all_zero_expert_weights(T, E, hid, inter, dq, alpha):
    """The deltas of experts whose block scales are all zero, all-zero token rows among the others, and a
    scaling of 256. bf16 roundings of x, h, the rows and their gradients: 1e-2 in norm."""
    _announce(f"train zero experts T={T} E={E} hid={hid} inter={inter} dq={dq} alpha={alpha}")
    gu, dn = _zeroed_stacks(E, hid, inter)
    mod = _module(E, hid, inter, 16, dq, alpha, gu, dn).train()
    assert e4b.enable_fast_train(mod) == 1
    x = torch.randn(T, hid, device=DEV).to(torch.bfloat16)
    x[3] = 0.0
    x[5] *= 2.0 ** -120
    x.requires_grad_()
    idx = torch.rand(T, E, device=DEV).argsort(1)[:, :2].contiguous()
    idx[3, 0], idx[5, 0] = 0, 2
    idx[3, 1], idx[5, 1] = 1, 3
    w = torch.rand(T, 2, device=DEV).to(torch.bfloat16).requires_grad_()
    grad = torch.randn(T, hid, device=DEV).to(torch.bfloat16)
    grad[7] = 0.0
    assert train._layer_inputs(mod, x.detach(), idx, w) is not None
    out = mod(x, idx, w)
    out.backward(grad)
    want = _layer_fp64(mod, x, idx, w, grad)
    got = {"out": out.detach(), "x": x.grad, "w": w.grad, **{n: getattr(mod, n).grad for n in ADAPTERS}}
    for n in want:
        assert got[n].isfinite().all(), n
        assert _rel(got[n], want[n]) < 1e-2, (n, _rel(got[n], want[n]))


@pytest.mark.parametrize("T,E,hid,inter", SHAPES)
@pytest.mark.parametrize("dq", (False, True))
def test_inference_with_all_zero_expert_weights(T, E, hid, inter, dq):
    _announce(f"infer zero experts T={T} E={E} hid={hid} inter={inter} dq={dq}")
    gu, dn = _zeroed_stacks(E, hid, inter)
    mod = _module(E, hid, inter, 16, dq, 4096, gu, dn).eval()
    assert e4b.enable_fast(mod) == 1
    x = torch.randn(T, hid, device=DEV).to(torch.bfloat16)
    x[3] = 0.0
    idx = torch.rand(T, E, device=DEV).argsort(1)[:, :2].contiguous()
    idx[3, 0], idx[3, 1] = 0, 1
    w = torch.rand(T, 2, device=DEV).to(torch.bfloat16)
    with torch.no_grad():
        out = mod(x, idx, w)
    want = _layer_fp64(mod, x, idx, w)["out"]
    assert out.isfinite().all()
    assert _rel(out, want) < 1e-2, _rel(out, want)
