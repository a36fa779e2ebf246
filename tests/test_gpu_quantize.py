"""``e4b_quantize_4bit`` against the torch formulation in ``quant.py``, bit for bit: packed codes and
block scales are the stored bytes, so nothing may differ."""
import pytest
import torch

from experts4bit_qlora_amd import quant as Q

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _special_blocks(quant_type, dtype):
    """Blocks where a nearest-code search can go wrong: zeros, exact midpoints and codes (and their
    neighbours), a NaN, infinities, subnormal and huge scales."""
    mids = torch.tensor(Q._host_table_4bit(quant_type)[0])
    code = Q.code_4bit(quant_type)
    up, down = torch.full_like(mids, 2.0), torch.full_like(mids, -2.0)
    edge = torch.cat([mids, torch.nextafter(mids, up), torch.nextafter(mids, down), code, torch.ones(3)])
    rows = [torch.zeros(64), edge, -edge]
    g = torch.Generator().manual_seed(5)
    for scale in (1e-44, 3e-39, 1.1754944e-38, 1e-30, 3.0e38, 1.8e38):
        rows.append((torch.rand(64, generator=g) * 2 - 1) * scale)
    for special in (float("nan"), float("inf"), -float("inf")):
        row = torch.randn(64, generator=g)
        row[17] = special
        rows += [row, torch.where(torch.arange(64) == 3, torch.full((64,), special), torch.zeros(64))]
    return torch.stack(rows).to(dtype)


@pytest.mark.parametrize("dtype", (torch.float32, torch.bfloat16, torch.float16))
@pytest.mark.parametrize("quant_type", ("nf4", "fp4"))
def test_codes_and_scales_are_the_torch_formulations(quant_type, dtype):
    g = torch.Generator().manual_seed(1)
    # one block; the edges of a 1,024-piece workgroup (128 blocks); an odd stack
    stacks = [torch.randn(s, generator=g) * 0.02 for s in ((1, 64), (1, 127 * 64), (128, 64), (129, 64), (3, 5 * 64 * 37))]
    for w in [s.to(dtype) for s in stacks] + [_special_blocks(quant_type, dtype)]:
        w = w.to(DEV)
        assert Q._on_kernel(w, 64)
        packed, absmax = Q.quantize_4bit(w, quant_type)
        want_packed, want_absmax = Q._quantize_4bit_torch(w, quant_type, 64)
        assert torch.equal(packed, want_packed)
        assert torch.equal(absmax.isnan(), want_absmax.isnan())
        assert torch.equal(absmax.nan_to_num(-1.0), want_absmax.nan_to_num(-1.0))


def test_views_other_dtypes_and_the_torch_route():
    w = torch.randn(64 * 64 + 2, device=DEV) * 0.1
    views = (w[2:].view(64, 64), w[:4096].view(64, 64).t(), w[:4096].view(64, 64).double(), w[1:4097])
    for v in views:
        packed, absmax = Q.quantize_4bit(v)
        want_packed, want_absmax = Q._quantize_4bit_torch(v.float(), "nf4", 64)
        assert torch.equal(packed, want_packed) and torch.equal(absmax, want_absmax)
        assert packed.shape == want_packed.shape and absmax.shape == want_absmax.shape
    assert not Q._on_kernel(w[:4096].view(64, 64), 32)
    recorded = w[:4096].view(64, 64).clone().requires_grad_()
    assert not Q._on_kernel(recorded, 64) and Q.quantize_4bit(recorded)[1].requires_grad


@pytest.mark.parametrize("shape", ((1, 1), (3, 255), (2, 256), (5, 257), (7, 1000), (4096,)))
def test_double_quant_is_the_torch_formulation(shape):
    """Block edges, a padded last block, blocks of equal values (all zeros once the offset is off), a NaN."""
    g = torch.Generator().manual_seed(3)
    a = (torch.rand(shape, generator=g) * 0.1).to(DEV)
    cases = [a, torch.full_like(a, 0.25), torch.zeros_like(a)]
    if len(shape) == 2 and shape[0] > 2:
        bad = a.clone()
        bad[1, -1] = float("nan")
        cases.append(bad)
    for c in cases:
        got, want = Q.double_quant(c), Q.double_quant(c, code2=Q.dynamic_map().to(DEV))
        assert all(torch.equal(p.nan_to_num(-1.0), q.nan_to_num(-1.0)) and p.dtype == q.dtype for p, q in zip(got, want))


def test_tangents_and_traces_follow_the_torch_formulation():
    """Forward-mode tangents of the scales, and a traced function on another input."""
    g = torch.Generator().manual_seed(4)
    w, t, other = (torch.randn(8, 256, generator=g).to(DEV) for _ in range(3))
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(w, t)
        unpack = torch.autograd.forward_ad.unpack_dual
        got, want = Q.quantize_4bit(dual)[1], Q._quantize_4bit_torch(dual, "nf4", 64)[1]
        assert torch.equal(unpack(got).tangent, unpack(want).tangent)
        got, want = Q.double_quant(dual), Q.double_quant(dual, code2=Q.dynamic_map().to(DEV))
        assert torch.equal(unpack(got[1]).tangent, unpack(want[1]).tangent)
    traced = torch.jit.trace(lambda v: Q.quantize_4bit(v), (w,), check_trace=False)
    assert all(torch.equal(a, b) for a, b in zip(traced(other), Q.quantize_4bit(other)))
    traced = torch.jit.trace(lambda v: Q.double_quant(v), (w.abs(),), check_trace=False)
    assert all(torch.equal(a, b) for a, b in zip(traced(other.abs()), Q.double_quant(other.abs())))
