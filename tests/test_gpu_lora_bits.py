"""The adapters' products in the training layer keep 32 bits: t = x . A^T and u = g . B run on the bf16 matrix
cores over the adapter's exact bf16 parts, so only the fp32 sums round. Adapter values of 1 + 2^-9 + 2^-18,
all products of one sign: two parts of 8 bits lose 2^-18 of every one of them."""
import pytest
import torch

import experts4bit_qlora_amd as e4b
from experts4bit_qlora_amd import _native as N
from experts4bit_qlora_amd import fast as F
from experts4bit_qlora_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
BITS = 1 + 2.0 ** -9 + 2.0 ** -18  # rounded to the adapter's dtype where that is narrower


def _announce(msg):
    print(f"[case] {msg}", flush=True)


def _signs(*shape):
    return torch.randint(0, 2, shape, device=DEV).float() * 2 - 1


def _base(E, hid, inter):
    torch.manual_seed(41)
    base = e4b.Experts4bit.from_float((torch.randn(E, 2 * inter, hid) * 0.05).to(DEV),
                                      (torch.randn(E, hid, inter) * 0.05).to(DEV), compute_dtype=torch.bfloat16)
    return base, F._for_tokens(F._qweights(base), 64)


def _saved_rows(saved, M, H, inter, r):
    """(sorted flat order, h, t1, t2) out of the forward's buffer: each part begins 256-byte aligned, the
    order first, h, the down rows, t1 and t2 last."""
    size = lambda n: (n + 255) // 256 * 256  # noqa: E731
    at = saved.numel() - 2 * size(4 * M * r)
    rows = lambda o, n, dt: saved[o:o + n].view(dt)  # noqa: E731
    h_at = at - size(2 * M * H) - size(2 * M * inter)
    return (rows(0, 4 * M, torch.int32).long(), rows(h_at, 2 * M * inter, torch.bfloat16).view(M, inter),
            rows(at, 4 * M * r, torch.float32).view(M, r), rows(at + size(4 * M * r), 4 * M * r, torch.float32).view(M, r))


@pytest.mark.parametrize("T,E,hid,inter", [(150, 2, 512, 192), (20, 4, 256, 320), (1, 2, 64, 64)])
@pytest.mark.parametrize("adt", (torch.float32, torch.float16, torch.bfloat16))
@pytest.mark.parametrize("r", (1, 16, 20, 33, 64))
def test_t_keeps_32_bits(T, E, hid, inter, adt, r):
    """64- and 32-row parts, every rank block. Sums of at most 512 products of one sign: below 2^-20."""
    _announce(f"t T={T} E={E} hid={hid} {adt} r={r}")
    base, (w1, w2) = _base(E, hid, inter)
    sign = _signs(hid)
    x = sign.expand(T, hid).to(torch.bfloat16).contiguous()
    a1 = (BITS * sign * torch.arange(1, r + 1, device=DEV)[:, None]).expand(E, r, hid).to(adt).contiguous()
    b1, b2 = (torch.randn(E, n, r, device=DEV).mul_(0.02).to(adt) for n in (2 * inter, hid))
    a2 = (BITS * torch.randn(E, r, inter, device=DEV)).to(adt)
    idx = torch.randint(0, E, (T, 1), device=DEV)
    _, saved = ops.train_forward(x, idx, torch.ones(T, 1, device=DEV), w1, w2, (a1, b1, a2, b2), 1.0, N.EPI_SWIGLU, 0.0,
                                 torch.float32)
    order, h, t1, t2 = _saved_rows(saved, T, hid, inter, r)
    e = idx.flatten()[order]
    for got, rows, a in ((t1, x[order], a1), (t2, h, a2)):
        want = (rows.double().unsqueeze(1) @ a[e].double().transpose(1, 2)).squeeze(1)
        mag = (rows.double().abs().unsqueeze(1) @ a[e].double().abs().transpose(1, 2)).squeeze(1)
        assert torch.all((got - want).abs() <= mag * 2.0 ** -20), ((got - want).abs() / mag).max()


@pytest.mark.parametrize("T,E", [(64, 1), (24, 24)])
@pytest.mark.parametrize("adt", (torch.float32, torch.float16))
@pytest.mark.parametrize("r", (1, 16, 20, 33, 64))
def test_u_keeps_32_bits(T, E, adt, r):
    """dL/dA2 = u^T h of one row per expert, or of 64 equal rows of one expert (64-row parts): u to the fp32
    rounding of 320 products of one sign, the product with h and a sum of 64: below 2^-20. The gradient
    itself leaves in the adapter's dtype, so an fp16 one also rounds to it (2^-11)."""
    _announce(f"u T={T} E={E} {adt} r={r}")
    hid, inter = 320, 128
    base, (w1, w2) = _base(E, hid, inter)
    x = torch.randn(1, hid, device=DEV).expand(T, hid).to(torch.bfloat16).contiguous()
    sign = _signs(hid)
    grad = sign.expand(T, hid).to(torch.bfloat16).contiguous()
    a1, a2 = (torch.randn(E, r, n, device=DEV).div_(r).to(adt) for n in (hid, inter))
    b1 = torch.zeros(E, 2 * inter, r, device=DEV, dtype=adt)
    b2 = (BITS * sign[:, None] * torch.arange(1, r + 1, device=DEV)).expand(E, hid, r).to(adt).contiguous()
    idx = (torch.arange(T, device=DEV) % E).unsqueeze(1)
    w = torch.ones(T, 1, device=DEV)
    lora = (a1, b1, a2, b2)
    _, saved = ops.train_forward(x, idx, w, w1, w2, lora, 2.0 ** -8, N.EPI_SWIGLU, 0.0, torch.bfloat16)
    grads = ops.train_backward(grad, x, w, w1, w2, lora, 2.0 ** -8, N.EPI_SWIGLU, 0.0, saved, (False,) * 4 + (True, False))
    _, h, _, _ = _saved_rows(saved, T, hid, inter, r)
    u = sign.double() @ b2[0].double()  # the same for every row
    rows = h.double() * 2.0 ** -8
    want = (torch.einsum("q,mc->mqc", u, rows) if E > 1 else torch.einsum("q,mc->qc", u, rows).unsqueeze(0))
    mag = (u.abs()[:, None] * (rows.abs() if E > 1 else rows.abs().sum(0, keepdim=True)).unsqueeze(1))
    err = (grads[4].double() - want).abs()
    assert torch.all(err <= mag * 2.0 ** -20 + (want.abs() * 2.0 ** -11 + 2.0 ** -24 if adt == torch.float16 else 0.0)), (err / mag).max()


def test_t_is_no_further_from_64_bits_than_the_vector_units():
    """Against the fp32 multiply-adds of e4b_lora_t on N(0, 1) rows and A ~ N(0, 1 / r)."""
    T, E, hid, inter, r = 512, 4, 2048, 256, 16
    base, (w1, w2) = _base(E, hid, inter)
    x = torch.randn(T, hid, device=DEV).to(torch.bfloat16)
    a1 = torch.randn(E, r, hid, device=DEV) / r
    a2, b1, b2 = (torch.zeros(E, *s, device=DEV) for s in ((r, inter), (2 * inter, r), (hid, r)))
    idx = torch.randint(0, E, (T, 1), device=DEV)
    _, saved = ops.train_forward(x, idx, torch.ones(T, 1, device=DEV), w1, w2, (a1, b1, a2, b2), 1.0, N.EPI_SWIGLU, 0.0,
                                 torch.float32)
    order, _, t1, _ = _saved_rows(saved, T, hid, inter, r)
    e = idx.flatten()[order]
    want = (x[order].double().unsqueeze(1) @ a1[e].double().transpose(1, 2)).squeeze(1)
    rb = ops.route(idx, E)
    old = ops.lora_t(x, rb, T, E, a1, gather_k=1)
    got, ref = ((v.double() - want).norm() / want.norm() for v in (t1, old))
    print(f"t rel error {got:.3e}, vector units {ref:.3e}", flush=True)
    assert got <= ref
