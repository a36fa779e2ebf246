"""The adapters' products in the training layer keep 32 bits: t = x . A^T and u = g . B run on the bf16 matrix
cores over the adapter's exact bf16 parts, so only the fp32 sums round. Adapter values of 1 + 2^-9 + 2^-18,
all products of one sign: two parts of 8 bits lose 2^-18 of every one of them."""
import pytest
import torch

import experts4bit_qlora_amd as e4b
from experts4bit_qlora_amd import _native as N
from experts4bit_qlora_amd import fast as F
from experts4bit_qlora_amd import ops
from experts4bit_qlora_amd import quant as Q

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


def _zero_layer(hid, inter):
    """Descriptors of one ungated expert whose block scales are all zero."""
    code = Q.code_4bit("nf4", DEV)
    return [ops.with_weight_shift(ops.nf4_qweight(torch.zeros(1, n * k // 2, dtype=torch.uint8, device=DEV),
                                                  torch.zeros(1, n * k // 64, device=DEV), code, n, k, num_experts=1))
            for n, k in ((inter, hid), (hid, inter))]


# (1 + 2^-9 + 2^-18) - (1 + 2^-9), and the last bits of (1 + 2^-9)^2 less its first two terms
CANCEL = [((1 + 2.0 ** -9 + 2.0 ** -18, 1 + 2.0 ** -9), (1.0, -1.0)),
          ((1.0, 1.0), (1 + 2.0 ** -9 + 2.0 ** -18, -1 - 2.0 ** -9)),
          ((1 + 2.0 ** -9, 1.0), (1 + 2.0 ** -9, -1 - 2.0 ** -8))]


@pytest.mark.parametrize("T,hid,inter", [(150, 192, 256), (300, 256, 192), (20, 256, 256), (20, 192, 320)])
@pytest.mark.parametrize("adt,case", [(torch.float32, 0), (torch.float32, 1), (torch.float32, 2), (torch.float16, 0),
                                      (torch.float16, 2), (torch.bfloat16, 0)])  # the adapters that dtype holds exactly
def test_deltas_keep_32_bits(T, hid, inter, adt, case):
    """Deltas t . B (forward) and u . A (backward) of two ranks that cancel to 2^-18, over zero weights:
    halved and whole 256-row tiles, 32-row tiles with K a multiple of 256 and not. Every product and sum is exact,
    so the rows are equal."""
    _announce(f"delta bits T={T} hid={hid} inter={inter} {adt} case={case}")
    (t0, t1), (b0, b1) = CANCEL[case]
    pair = torch.tensor([b0, b1], device=DEV)
    w1, w2 = _zero_layer(hid, inter)
    bits = torch.zeros(hid, device=DEV)
    bits[:3] = torch.tensor([1.0, 2.0 ** -9, 2.0 ** -18])
    x = bits.expand(T, hid).to(torch.bfloat16).contiguous()
    pick = lambda v: torch.tensor([1.0, float(v >= 1 + 2.0 ** -9), float(v > 1 + 2.0 ** -9)], device=DEV)  # noqa: E731
    side = lambda n: torch.nn.functional.pad(torch.stack([pick(t0), pick(t1)]), (0, n - 3))  # [2, n]  # noqa: E731
    idx, w = torch.zeros(T, 1, dtype=torch.int64, device=DEV), torch.ones(T, 1, device=DEV)
    one = lambda v: v.to(adt).unsqueeze(0).contiguous()  # noqa: E731
    # forward: t = (t0, t1), B1 rows (b0, b1)
    lora = (one(side(hid)), one(pair.expand(inter, 2)), one(torch.zeros(2, inter, device=DEV)),
            one(torch.zeros(hid, 2, device=DEV)))
    _, saved = ops.train_forward(x, idx, w, w1, w2, lora, 1.0, N.EPI_ACT, 0.0, torch.float32)
    size = lambda n: (n + 255) // 256 * 256  # noqa: E731
    at = saved.numel() - 2 * size(8 * T) - size(2 * T * hid) - 2 * size(2 * T * inter)
    proj = saved[at:at + 2 * T * inter].view(torch.bfloat16)
    assert torch.all(proj == 2.0 ** -18), proj
    # backward: u = (t0, t1) from the gradient x and B2, A2 columns (b0, b1); proj = 0, so dL/dproj = dh / 2, and with
    # t1 = 1 in both ranks dL/dB1 = T dh / 2
    lora = (one(torch.nn.functional.pad(torch.ones(2, 1, device=DEV), (0, hid - 1))), one(torch.zeros(inter, 2, device=DEV)),
            one(pair[:, None].expand(2, inter)), one(side(hid).t()))
    _, saved = ops.train_forward(x, idx, w, w1, w2, lora, 1.0, N.EPI_ACT, 0.0, torch.float32)
    grads = ops.train_backward(x, x, w, w1, w2, lora, 1.0, N.EPI_ACT, 0.0, saved, (False,) * 3 + (True, False, False))
    assert torch.all(grads[3].float() == torch.tensor(T * 2.0 ** -19).to(adt).float().item()), grads[3]
