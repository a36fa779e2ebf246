"""The grouped GEMM's tile heights against each other and against fp64, where the tiles' edges lie: output
widths off the vector stores' runs, row counts around a half, a whole and two tiles."""
import pytest
import torch

from experts4bit_qlora_amd import _native as N
from experts4bit_qlora_amd import ops
from experts4bit_qlora_amd import quant as Q

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _routing(sizes, tile_m):
    """Groups of `sizes` rows, expert by expert, as 256- / 128- / 32-row tiles."""
    idx = torch.repeat_interleave(torch.arange(len(sizes)), torch.tensor(sizes)).unsqueeze(1).to(DEV)
    return ops.route(idx, len(sizes), tile_m=tile_m)


@pytest.mark.parametrize("n", (64, 100, 136, 528))
@pytest.mark.parametrize("epi,bias,f32", [(N.EPI_NONE, False, True), (N.EPI_NONE, True, True), (N.EPI_NONE, False, False),
                                          (N.EPI_NONE, True, False), (N.EPI_SWIGLU, False, False),
                                          (N.EPI_GPTOSS, True, False), (N.EPI_GPTOSS, True, True), (N.EPI_ACT, False, False)])
def test_mxfp4_256_row_tiles_equal_the_128_row_ones(n, epi, bias, f32):
    """Both kernels multiply the same exact operands in the same order along k: equal bit for bit."""
    g = torch.Generator().manual_seed(n + epi)
    sizes, K = [1, 128, 0, 129, 256, 300, 31], 192
    E, M = len(sizes), sum(sizes)
    blocks, scales = Q.quantize_mxfp4(torch.randn(E, n, K, generator=g) * 0.05)
    b = (torch.randn(E, n, generator=g) * 0.1).to(torch.bfloat16).to(DEV) if bias else None
    qw = ops.mxfp4_qweight(blocks.to(DEV), scales.to(DEV), n, K, num_experts=E, bias=b)
    a = torch.randn(M, K, generator=g).to(torch.bfloat16).to(DEV)
    out = [ops.grouped_gemm(a, qw, _routing(sizes, tm), M, M, epilogue=epi, gather_k=1, path=N.PATH_MFMA,
                            out_dtype=torch.float32 if f32 else None) for tm in (256, 128)]
    assert torch.equal(*out)


@pytest.mark.parametrize("n", (64, 100, 272))
@pytest.mark.parametrize("dq", (False, True))
@pytest.mark.parametrize("epi", (N.EPI_NONE, N.EPI_SWIGLU))
def test_fp16_32_row_tiles_use_the_exact_weights(n, dq, epi):
    """fp16 activations over 32-row tiles against fp64 products of the weights as e4b_dequant gives them in
    fp16: fp32 sums of 512 products (2^-16 of the sum of magnitudes), one rounding to fp16 (2^-11)."""
    g = torch.Generator().manual_seed(n)
    sizes, K = [1, 16, 17, 0, 32, 33, 70], 512
    E, M = len(sizes), sum(sizes)
    packed, absmax = Q.quantize_4bit((torch.randn(E, n * K, generator=g) * 0.05).to(DEV))
    code = Q.code_4bit("nf4", DEV)
    if dq:
        q, a2, off = Q.double_quant(absmax)
        qw = ops.nf4_dq_qweight(packed, q, a2, off, code, Q.dynamic_map().to(DEV), n, K, num_experts=E)
    else:
        qw = ops.nf4_qweight(packed, absmax, code, n, K, num_experts=E)
    a = torch.randn(M, K, generator=g).to(torch.float16).to(DEV)
    got = ops.grouped_gemm(a, qw, _routing(sizes, 32), M, M, epilogue=epi, gather_k=1, path=N.PATH_MFMA).double()
    W = ops.dequant(qw, dtype=torch.float16).double()
    e = torch.repeat_interleave(torch.arange(E), torch.tensor(sizes)).tolist()
    want = torch.stack([a[m].double() @ W[e[m]].T for m in range(M)])
    bound = torch.stack([a[m].double().abs() @ W[e[m]].abs().T for m in range(M)]) * 2.0 ** -16
    if epi == N.EPI_SWIGLU:
        gate, up = want.chunk(2, -1)
        bg, bu = bound.chunk(2, -1)
        want = torch.nn.functional.silu(gate) * up
        bound = 1.1 * bg * up.abs() + bu * gate.abs() + bg * bu + 2.0 ** -20 * want.abs()  # |silu'| <= 1.1
    assert torch.all((got - want).abs() <= bound + 2.0 ** -11 * want.abs() + 2.0 ** -24)


@pytest.mark.parametrize("dq", (False, True))
def test_fp16_32_row_tiles_hold_the_dequantized_weights_bit_for_bit(dq):
    """One activation of 1 per row: every output is one weight, rounded to fp32 and then to fp16 as e4b_dequant rounds
    it (of the 417,792 products, about 25 lie where a single rounding gives another fp16 value)."""
    g = torch.Generator().manual_seed(9)
    E, n, K = 3, 272, 512
    packed, absmax = Q.quantize_4bit((torch.randn(E, n * K, generator=g) * 0.05).to(DEV))
    code = Q.code_4bit("nf4", DEV)
    if dq:
        q, a2, off = Q.double_quant(absmax)
        qw = ops.nf4_dq_qweight(packed, q, a2, off, code, Q.dynamic_map().to(DEV), n, K, num_experts=E)
    else:
        qw = ops.nf4_qweight(packed, absmax, code, n, K, num_experts=E)
    a = torch.eye(K, dtype=torch.float16, device=DEV).repeat(E, 1)
    got = ops.grouped_gemm(a, qw, _routing([K] * E, 32), E * K, E * K, gather_k=1, path=N.PATH_MFMA)
    want = ops.dequant(qw, dtype=torch.float16).view(E, n, K).transpose(1, 2).reshape(E * K, n)
    assert torch.equal(got, want), int((got != want).sum())
