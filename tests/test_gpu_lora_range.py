"""Adapters over expert weights, token rows and adapter values at the ends of the number range. The fp16
matrix-core mode scales its operands by powers of two and a delta is formed in those scaled sums, so
all-zero scales, tiny rows and infinities reach it at its largest and smallest factors."""
import pytest
import torch

import experts4bit_qlora_amd as e4b
from experts4bit_qlora_amd import ops, train
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


def _same_specials(got, want, tol):
    """Infinities of one sign and NaNs where ``want`` has them, the rest within ``tol`` in norm."""
    got = got.double()
    inf, fin = want.isinf(), want.isfinite()
    assert bool((got.isnan() == want.isnan()).all()) and bool((got.isinf() == inf).all())
    assert bool((got[inf] == want[inf]).all())
    assert _rel(got[fin], want[fin]) < tol


@pytest.mark.parametrize("T,E,hid,inter", SHAPES)
@pytest.mark.parametrize("adt", (torch.float32, torch.float16, torch.bfloat16))
@pytest.mark.parametrize("r", (3, 16))
def test_an_infinity_stays_one(T, E, hid, inter, adt, r):
    """Weights, adapters and tokens all positive, so one infinite activation or gradient makes sums of one sign
    infinite and leaves the others alone. The adapters fit one bf16 part: what is split off is zero.
    The largest finite gradient is dL/dA1 = scaling u1 x over 600 rows: u1 = 512 . 22 . 0.06 = 676 for
    gradients of 0.06, 4.9e5 in all, beyond fp16; with gradients of 0.06 . 2^-6 it is 7.6e3."""
    _announce(f"infinities T={T} E={E} hid={hid} inter={inter} {adt} r={r}")
    mod = _module(E, hid, inter, r, False, gate_up=torch.full((E, 2 * inter, hid), 0.01),
                  down=torch.full((E, hid, inter), 0.01)).train()
    for n in ADAPTERS:
        p = getattr(mod, n)
        setattr(mod, n, torch.nn.Parameter((torch.rand_like(p) * 0.1 + 0.01).to(torch.bfloat16).to(adt)))
    assert e4b.enable_fast_train(mod) == 1
    torch.manual_seed(33)
    x = (torch.rand(T, hid, device=DEV) + 0.1).to(torch.bfloat16)
    idx = torch.rand(T, E, device=DEV).argsort(1)[:, :2].contiguous()
    idx[3, 0], idx[3, 1], idx[9, 0], idx[9, 1] = 0, 1, 0, 1
    w = torch.rand(T, 2, device=DEV).to(torch.bfloat16) + 0.1
    grad = ((torch.rand(T, hid, device=DEV) * 0.1 + 0.01) * 2.0 ** -6).to(torch.bfloat16)
    x[3, 5] = float("inf")
    with torch.no_grad():
        out = mod(x, idx, w)
    want = _layer_fp64(mod, x, idx, w)["out"]
    assert want[3].isinf().all() and want[4].isfinite().all()
    _same_specials(out, want, 1e-2)
    x[3, 5] = 1.0
    grad[9, 7] = float("inf")
    x, w = x.requires_grad_(), w.requires_grad_()
    out = mod(x, idx, w)
    out.backward(grad)
    want = _layer_fp64(mod, x, idx, w, grad)
    assert want["x"][9].isinf().all() and want["gate_up_lora_A"][0].isinf().all()
    for n, got in (("x", x.grad), ("w", w.grad), *((n, getattr(mod, n).grad) for n in ADAPTERS)):
        _same_specials(got, want[n], 1e-2)


@pytest.mark.parametrize("adt", (torch.bfloat16, torch.float16))
def test_weight_gradients_keep_infinities(adt):
    """u and rows of exact leading parts, one infinity in each: sums of one sign."""
    rb = ops._routing_from_sizes([70, 5], [0, 1], 2, DEV)[0]
    u = torch.full((75, 8), 0.5, device=DEV)
    a = torch.full((75, 136), 0.25, device=DEV).to(adt)
    u[3, 2], a[71, 9] = float("inf"), float("inf")
    got = ops.lora_wgrad(u, a, rb, 75, 2, 1.0)
    want = torch.stack([u[:70].T @ a[:70].float(), u[70:].T @ a[70:].float()])
    assert want[0, 2].isinf().all() and want[1, :, 9].isinf().all()
    assert torch.equal(got, want)
