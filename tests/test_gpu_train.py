"""The training lane (``enable_fast_train``) under the reference's parity contract
(``tests/test_fused_train_parity.py:50-224``): forward values, dL/dx and dL/d(every LoRA
parameter) within the measured bf16 noise (forward < 1.5e-2, gradients < 1e-2 relative norm)
against the reference ``ExpertsLoRA.forward`` with a load-bearing adapter; the same assertions
REJECT a 1% LoRA-scaling mutant (the control), and forward parity alone would not.

Below the contract, each kernel of the backward against an independent computation: the grouped
dgrad against fp64 products over the oracle-decoded weights, the per-expert weight gradient
against numpy, the split LoRA passes against the fused one bit for bit.
"""
import numpy as np
import pytest
import torch

import experts4bit_qlora_amd as e4b
from experts4bit_qlora_amd import _native as N
from experts4bit_qlora_amd import fast as F
from experts4bit_qlora_amd import ops, train
from oracle_weights import oracle_weights

pytestmark = pytest.mark.gpu
DEV = "cuda"
E, HID, INTER, TOP_K = 8, 128, 192, 2
FWD_TOL = 1.5e-2
GRAD_TOL = 1.0e-2


def _announce(msg):
    print(f"[case] {msg}", flush=True)


def _rel(got, want):
    want = want.float()
    return ((got.float() - want).norm() / want.norm().clamp_min(1e-12)).item()


def _build(seed=0, scaling_bug=1.0, E_=E, hid=HID, inter=INTER, r=8, dq=False):
    """An ExpertsLoRA over a real NF4 base, B nonzero (test_fused_train_parity.py:76-95)."""
    torch.manual_seed(seed)
    gate_up = (torch.randn(E_, 2 * inter, hid) * 0.1).to(DEV)
    down = (torch.randn(E_, hid, inter) * 0.1).to(DEV)
    base = e4b.Experts4bit.from_float(gate_up, down, quant_type="nf4", compute_dtype=torch.bfloat16,
                                      compress_statistics=dq)
    mod = e4b.ExpertsLoRA(base, r=r, alpha=2 * r, dtype=torch.float32).to(DEV)
    with torch.no_grad():
        for p in (mod.gate_up_lora_B, mod.down_lora_B):
            p.normal_(0, 0.02)
    mod.scaling *= scaling_bug
    return mod.train()


def _inputs(n_tok=64, seed=1, E_=E, hid=HID, top_k=TOP_K):
    torch.manual_seed(seed)
    hs = torch.randn(n_tok, hid, dtype=torch.bfloat16, device=DEV)
    idx = torch.randint(0, E_, (n_tok, top_k), device=DEV)
    wts = torch.rand(n_tok, top_k, dtype=torch.bfloat16, device=DEV)
    torch.manual_seed(seed + 100)
    loss_w = torch.randn(n_tok, hid, device=DEV)
    return hs, idx, wts, loss_w


def _forward_backward(mod, hs, idx, wts, loss_w):
    hs = hs.clone().requires_grad_(True)
    for p in mod.parameters():
        p.grad = None
    out = mod(hs, idx, wts)
    assert out.requires_grad, "a training path that returns a detached tensor trains nothing"
    (out.float() * loss_w).sum().backward()
    grads = {n: p.grad.detach().clone() for n, p in mod.named_parameters() if p.grad is not None}
    assert grads, "no parameter received a gradient"
    return out.detach(), hs.grad.detach().clone(), grads


def assert_parity(candidate, reference, args=None, fwd_tol=FWD_TOL, grad_tol=GRAD_TOL):
    ref_p = dict(reference.named_parameters())
    for n, p in candidate.named_parameters():
        assert torch.equal(p.detach(), ref_p[n].detach()), f"fixtures differ at {n}"
    args = args or _inputs()
    ref_out, ref_dx, ref_grads = _forward_backward(reference, *args)
    got_out, got_dx, got_grads = _forward_backward(candidate, *args)
    measured = {"forward": _rel(got_out, ref_out), "dL/dx": _rel(got_dx, ref_dx)}
    assert measured["forward"] < fwd_tol, f"forward {measured['forward']:.3e}"
    assert measured["dL/dx"] < grad_tol, f"dL/dx {measured['dL/dx']:.3e}"
    assert set(got_grads) == set(ref_grads), sorted(set(got_grads) ^ set(ref_grads))
    for n in ref_grads:
        measured[f"dL/d{n}"] = _rel(got_grads[n], ref_grads[n])
        assert measured[f"dL/d{n}"] < grad_tol, f"dL/d{n} {measured[f'dL/d{n}']:.3e}"
    return measured


def test_training_path_matches_reference_forward_and_gradients():
    """test_fused_train_parity.py:180-189 for the enable_fast_train lane."""
    _announce("train parity contract")
    reference = _build(seed=0)
    candidate = _build(seed=0)
    assert e4b.enable_fast_train(candidate) == 1
    measured = assert_parity(candidate, reference)
    print("enable_fast_train: " + "  ".join(f"{k}={v:.2e}" for k, v in measured.items()), flush=True)


@pytest.mark.parametrize("n_tok,E_,hid,inter,r,dq", [(2048, 8, 256, 128, 16, False), (512, 16, 192, 256, 20, True),
                                                     (3, 8, 128, 192, 8, False)])
def test_training_path_contract_at_other_shapes(n_tok, E_, hid, inter, r, dq):
    """The contract with 128-row tiles (2048 tokens over 8 experts), double-quantized weights and
    an odd rank, and a 3-token batch."""
    _announce(f"train parity n_tok={n_tok} E={E_} hid={hid} inter={inter} r={r} dq={dq}")
    reference = _build(seed=5, E_=E_, hid=hid, inter=inter, r=r, dq=dq)
    candidate = _build(seed=5, E_=E_, hid=hid, inter=inter, r=r, dq=dq)
    assert e4b.enable_fast_train(candidate) == 1
    measured = assert_parity(candidate, reference, args=_inputs(n_tok, seed=6, E_=E_, hid=hid))
    print(f"n_tok={n_tok}: " + "  ".join(f"{k}={v:.2e}" for k, v in measured.items()), flush=True)


def test_contract_detects_a_wrong_gradient():
    """The control (test_fused_train_parity.py:192-205): a 1% LoRA-scaling error must fail."""
    _announce("train contract control")
    reference = _build(seed=0)
    mutant = _build(seed=0, scaling_bug=1.01)
    assert e4b.enable_fast_train(mutant) == 1
    with pytest.raises(AssertionError):
        assert_parity(mutant, reference)


def test_forward_parity_alone_would_miss_a_gradient_bug():
    """test_fused_train_parity.py:208-224, on the fused lane: the mutant's forward passes, its
    parameter gradients do not."""
    _announce("train forward-only control")
    reference = _build(seed=0)
    mutant = _build(seed=0, scaling_bug=1.01)
    assert e4b.enable_fast_train(mutant) == 1
    args = _inputs()
    ref_out, _, ref_grads = _forward_backward(reference, *args)
    got_out, _, got_grads = _forward_backward(mutant, *args)
    assert _rel(got_out, ref_out) < FWD_TOL
    worst = max(_rel(got_grads[n], ref_grads[n]) for n in ref_grads)
    assert worst > GRAD_TOL, worst


def test_enable_disable_markers_and_idempotence():
    _announce("train enable/disable")
    mod = _build(seed=0)
    ref_forward = mod.forward
    assert e4b.enable_fast_train(mod) == 1
    assert hasattr(mod, "_e4b_train_ref") and mod._e4b_dgrad is False
    assert e4b.enable_fast_train(mod) == 0  # already patched
    with pytest.warns(RuntimeWarning, match="dgrad"):
        assert e4b.enable_fast_train(mod, dgrad=True) == 0
    assert e4b.disable_fast_train(mod) == 1
    assert not hasattr(mod, "_e4b_train_ref") and not hasattr(mod, "_e4b_dgrad")
    assert mod.forward == ref_forward
    assert e4b.disable_fast_train(mod) == 0
    mod._e4b_batched_ref = mod.forward  # another lane's marker: skipped
    assert e4b.enable_fast_train(mod) == 0


# ------------------------------------------------------------------ the backward's kernels


def _nf4(E_, n, k, seed, dq=False):
    """A base whose gate_up weights are [E, n, k] (n output features, the dgrad's reduction)."""
    torch.manual_seed(seed)
    return e4b.Experts4bit.from_float((torch.randn(E_, n, k) * 0.05).to(DEV), (torch.randn(E_, k, n) * 0.05).to(DEV),
                                      compute_dtype=torch.bfloat16, has_gate=False, compress_statistics=dq)


@pytest.mark.parametrize("E_,n,k,T,top,tile,gdt,dq", [(8, 256, 320, 700, 2, 128, torch.bfloat16, False),
                                                       (8, 128, 192, 90, 2, 32, torch.bfloat16, True),
                                                       (4, 192, 512, 300, 3, 128, torch.float16, False),
                                                       (16, 64, 128, 33, 4, 32, torch.float16, True)])
def test_grouped_dgrad_matches_fp64(E_, n, k, T, top, tile, gdt, dq):
    """out[m] = g[m] . deq(W[e_m]) against fp64 products over the oracle-decoded weights, rounded
    to the gradient dtype as the kernel's operands are: tolerance 2^-16 of sum |g||w| per output
    (fp32 accumulation only: a wrong row, scale or nibble is off by O(1) of it); 128- and 32-row
    tiles, columns not a multiple of the tile."""
    _announce(f"grouped dgrad E={E_} n={n} k={k} T={T} top={top} tile={tile} g={gdt} dq={dq}")
    base = _nf4(E_, n, k, seed=7, dq=dq)
    w1, _ = F._qweights(base)
    g_ = torch.Generator(device=DEV).manual_seed(8)
    idx = torch.rand(T, E_, generator=g_, device=DEV).argsort(dim=1)[:, :top]  # distinct experts per token
    rb = ops.route(idx, E_, tile_m=tile)
    M = T * top
    g = torch.randn(M, n, generator=g_, device=DEV).to(gdt)
    got = ops.grouped_dgrad(g, w1, rb, M).double().cpu().numpy()
    W = oracle_weights(base)[0]
    Wr = {e: torch.from_numpy(W[e]).to(gdt).double().numpy() for e in range(E_)}  # the kernel's operand values
    offs = rb.offsets.cpu().numpy()
    gd = g.double().cpu().numpy()
    for e in range(E_):
        s, t = int(offs[e]), int(offs[e + 1])
        if s == t:
            continue
        want = gd[s:t] @ Wr[e]
        bound = np.abs(gd[s:t]) @ np.abs(Wr[e])
        assert np.all(np.abs(got[s:t] - want) <= bound * 2.0 ** -16 + 1e-30), e


@pytest.mark.parametrize("r,adt,gather", [(8, torch.float32, True), (20, torch.bfloat16, False), (64, torch.float32, True)])
def test_lora_wgrad_matches_numpy(r, adt, gather):
    """out[e] = scale * u_e^T a_e per expert over its sorted rows (gathered token rows or sorted
    rows), zeros for an expert without rows."""
    _announce(f"lora wgrad r={r} gather={gather}")
    E_, T, top, cols = 12, 150, 2, 320
    g_ = torch.Generator(device=DEV).manual_seed(9)
    idx = torch.randint(0, E_ - 2, (T, top), generator=g_, device=DEV)  # the last two experts get no rows
    rb = ops.route(idx, E_)
    M = T * top
    u = torch.randn(M, r, generator=g_, device=DEV)
    a = torch.randn(T if gather else M, cols, generator=g_, device=DEV).to(torch.bfloat16)
    got = ops.lora_wgrad(u, a, rb, M, E_, 1.5, gather_k=top if gather else 0).double().cpu().numpy()
    offs = rb.offsets.cpu().numpy()
    sf = rb.sorted_flat.cpu().numpy()[:M]
    ud, ad = u.double().cpu().numpy(), a.double().cpu().numpy()
    for e in range(E_):
        s, t = int(offs[e]), int(offs[e + 1])
        rows = ad[sf[s:t] // top] if gather else ad[s:t]
        want = 1.5 * ud[s:t].T @ rows if t > s else np.zeros((r, cols))
        bound = 1.5 * np.abs(ud[s:t]).T @ np.abs(rows) if t > s else np.zeros((r, cols))
        assert np.all(np.abs(got[e] - want) <= bound * 2.0 ** -16 + 1e-30), e


def test_split_lora_passes_equal_the_fused_delta():
    """e4b_lora_t then e4b_lora_t_add == e4b_lora_delta, bit for bit (the same kernels)."""
    _announce("lora split passes")
    E_, T, top, k_in, n_out, r = 8, 200, 2, 256, 384, 16
    g_ = torch.Generator(device=DEV).manual_seed(10)
    idx = torch.randint(0, E_, (T, top), generator=g_, device=DEV)
    rb = ops.route(idx, E_)
    M = T * top
    x = torch.randn(T, k_in, generator=g_, device=DEV).to(torch.bfloat16)
    A = torch.randn(E_, r, k_in, generator=g_, device=DEV) / r
    B = torch.randn(E_, n_out, r, generator=g_, device=DEV) * 0.02
    base = torch.randn(M, n_out, generator=g_, device=DEV)
    fused = ops.lora_delta(x, rb, M, E_, A, B, 2.0, base.clone(), gather_k=top, delta_dtype=torch.float32)
    t = ops.lora_t(x, rb, M, E_, A, gather_k=top)
    split = ops.lora_t_add(t, rb, M, E_, B, 2.0, base.clone())
    assert torch.equal(fused, split)


@pytest.mark.parametrize("n_tok,E_,top", [(64, 8, 2), (1024, 8, 4)])
def test_training_lane_is_bit_identical_across_runs(n_tok, E_, top):
    """ref tests/test_deterministic_scatter.py:62-80: the training forward and every gradient are
    bit-identical over repeated runs (no float atomics anywhere in the lane). 1,024 tokens x 4
    slots over 8 experts runs the 128-row tiles; 64 x 2 the 32-row ones."""
    _announce(f"train determinism n_tok={n_tok} E={E_} top={top}")
    mod = _build(seed=3, E_=E_)
    assert e4b.enable_fast_train(mod) == 1
    args = _inputs(n_tok=n_tok, seed=4, E_=E_, top_k=top)
    out0, dx0, g0 = _forward_backward(mod, *args)
    assert set(g0) == {"gate_up_lora_A", "gate_up_lora_B", "down_lora_A", "down_lora_B"}, sorted(g0)
    for run in range(1, 8):
        out, dx, grads = _forward_backward(mod, *args)
        assert torch.equal(out, out0), f"run {run}: forward differs"
        assert torch.equal(dx, dx0), f"run {run}: dL/dx differs"
        for n in g0:
            assert torch.equal(grads[n], g0[n]), f"run {run}: dL/d{n} differs"


@pytest.mark.parametrize("r,adt,top,cols", [(1, torch.bfloat16, 1, 8), (16, torch.float16, 2, 136), (17, torch.bfloat16, 3, 100),
                                            (33, torch.float16, 2, 392), (64, torch.bfloat16, 4, 129)])
def test_lora_wgrad_edges(r, adt, top, cols):
    """Ranks and columns off the 16-rank and 128-column tiles, row counts around the 64-row rounds, rows
    that are not whole 16-byte pieces, both 16-bit types. Products are exact and summed in fp32, so
    2^-16 of the sum of magnitudes holds up to 256 rows (2^-24 each)."""
    _announce(f"lora wgrad edges r={r} {adt} cols={cols}")
    sizes = [63, 0, 64, 65, 1, 128, 200]
    E_ = len(sizes)
    rb = ops._routing_from_sizes(sizes, list(range(E_)), E_, DEV)[0]
    M = sum(sizes)
    g_ = torch.Generator(device=DEV).manual_seed(12)
    u = torch.randn(M, r, generator=g_, device=DEV) * torch.logspace(-6, 6, M, device=DEV).unsqueeze(1)
    a = torch.randn(M, cols, generator=g_, device=DEV).to(adt)
    got = ops.lora_wgrad(u, a, rb, M, E_, 0.5).double()
    at = 0
    for e, s in enumerate(sizes):
        ue, ae = u[at:at + s].double(), a[at:at + s].double()
        want, bound = 0.5 * ue.T @ ae, 0.5 * ue.abs().T @ ae.abs()
        assert torch.all((got[e] - want).abs() <= bound * 2.0 ** -16 + 1e-30), e
        at += s
    u[70, 0] = float("inf")  # expert 2's alone
    got = ops.lora_wgrad(u, a, rb, M, E_, 0.5)
    assert not got[2, 0].isfinite().any() and got[[0, 1, 3, 4, 5, 6]].isfinite().all()


def _layer_fp64(base, mod, x, idx, w, grad, act):
    """The layer and its gradients in fp64 autograd over the oracle-decoded weights, nothing rounded."""
    W1, W2 = ([torch.from_numpy(W[e]).double().to(DEV) for e in range(base.num_experts)] for W in oracle_weights(base))
    x, w = x.double().requires_grad_(), w.double().requires_grad_()
    p = {n: t.detach().double().requires_grad_() for n, t in mod.named_parameters() if "lora" in n}
    out = torch.zeros_like(x)
    for e in range(base.num_experts):
        tok, slot = torch.where(idx == e)
        if not len(tok):
            continue
        proj = x[tok] @ W1[e].T + mod.scaling * (x[tok] @ p["gate_up_lora_A"][e].T) @ p["gate_up_lora_B"][e].T
        h = act(proj)
        down = h @ W2[e].T + mod.scaling * (h @ p["down_lora_A"][e].T) @ p["down_lora_B"][e].T
        out = out.index_add(0, tok, down * w[tok, slot, None])
    out.backward(grad.double())
    return {"out": out.detach(), "x": x.grad, "w": w.grad, **{n: t.grad for n, t in p.items()}}


def _swiglu64(limit=0.0):
    """With a limit the gradient jumps at it, and a value within the layer's rounding of the limit may lie on
    either side: a share of 2^-8 of the limit times the density there, its root in norm (0.7 under a
    density of 0.2: 2e-2). So the clamp sees proj as the layer stores it, rounded to bf16 (gradient
    passed straight through), and the limit of 4 lies beyond two standard deviations, where the
    weights' own rounding (2^-11) moves few values across (a density of 0.015: 4e-3)."""
    def act(proj):
        if limit:
            proj = proj + (proj.to(torch.bfloat16).double() - proj).detach()
        g, u = proj.chunk(2, -1)
        if limit:
            g, u = g.clamp(max=limit), u.clamp(-limit, limit)
        return torch.nn.functional.silu(g) * u

    return act


@pytest.mark.parametrize("T,E_,top,hid,inter,r,adt,dq,kind,xdt", [
    (2048, 8, 2, 256, 128, 16, torch.float32, False, "swiglu", torch.bfloat16),   # 256-row tiles, whole step pairs
    (700, 4, 2, 192, 320, 20, torch.bfloat16, True, "swiglu", torch.bfloat16),    # halved tiles; k off 256 and 128
    (300, 3, 1, 320, 192, 64, torch.float16, False, "clamp", torch.float32),      # tails of 1..32 rows, fp32 tokens
    (33, 16, 4, 128, 64, 1, torch.float32, True, "act", torch.bfloat16),          # 32-row tiles only, one gate half
    (1, 8, 2, 64, 64, 8, torch.float32, False, "swiglu", torch.bfloat16),
])
def test_fused_layer_matches_fp64(T, E_, top, hid, inter, r, adt, dq, kind, xdt):
    """The two-call layer against fp64 autograd: outputs and every gradient. bf16 rounds x, proj, h, the down
    rows and their gradients (2^-9 each, independent): 1e-2 in norm is the contract's bar. Dropped ids
    (-1 and E) contribute nothing and get zero router gradients."""
    _announce(f"fused layer T={T} E={E_} hid={hid} inter={inter} r={r} {kind}")
    torch.manual_seed(21)
    gated = kind != "act"
    gu = (torch.randn(E_, (2 if gated else 1) * inter, hid) * 0.1).to(DEV)
    dn = (torch.randn(E_, hid, inter) * 0.1).to(DEV)
    if kind == "clamp":
        base = e4b.DeepseekV4Experts4bit.from_deepseek_v4(gu, dn, limit=4.0, compute_dtype=torch.bfloat16,
                                                          compress_statistics=dq)
    else:
        base = e4b.Experts4bit.from_float(gu, dn, has_gate=gated, compute_dtype=torch.bfloat16, compress_statistics=dq)
    mod = e4b.ExpertsLoRA(base, r=r, alpha=2 * r, dtype=adt).to(DEV).train()
    with torch.no_grad():
        for p in (mod.gate_up_lora_B, mod.down_lora_B):
            p.normal_(0, 0.05)
    assert e4b.enable_fast_train(mod) == 1
    x = torch.randn(T, hid, device=DEV).to(torch.bfloat16).to(xdt).requires_grad_()
    idx = torch.rand(T, E_, device=DEV).argsort(1)[:, :top].contiguous()
    if T > 2:
        idx[1, 0], idx[2, top - 1] = -1, E_
    w = torch.rand(T, top, device=DEV).to(torch.bfloat16).requires_grad_()
    grad = torch.randn(T, hid, device=DEV).to(xdt)
    assert train._layer_inputs(mod, x.detach().to(torch.bfloat16), idx, w) is not None
    out = mod(x, idx, w)
    out.backward(grad)
    got = {"out": out.detach(), "x": x.grad, "w": w.grad, **{n: p.grad for n, p in mod.named_parameters() if "lora" in n}}
    act = {"swiglu": _swiglu64(), "clamp": _swiglu64(4.0), "act": torch.nn.functional.silu}[kind]
    want = _layer_fp64(base, mod, x.detach(), idx, w.detach(), grad, act)
    assert out.dtype == xdt and x.grad.dtype == xdt
    for n in want:
        assert _rel(got[n], want[n]) < GRAD_TOL, (n, _rel(got[n], want[n]))
    if T > 2:
        assert w.grad[1, 0] == 0 and w.grad[2, top - 1] == 0


def test_fused_layer_gives_only_the_gradients_asked_for():
    """Each subset of leaves alone gives the bits that all of them together give."""
    _announce("fused layer partial gradients")
    mod = _build(seed=9)
    assert e4b.enable_fast_train(mod) == 1
    hs, idx, wts, loss_w = _inputs(n_tok=90, seed=11)
    names = ("gate_up_lora_A", "gate_up_lora_B", "down_lora_A", "down_lora_B")

    def grads(leaves):
        x, w = hs.clone().requires_grad_("x" in leaves), wts.clone().requires_grad_("w" in leaves)
        for n in names:
            getattr(mod, n).requires_grad_(n in leaves).grad = None
        mod(x, idx, w).backward(loss_w.to(torch.bfloat16))
        return {"x": x.grad, "w": w.grad, **{n: getattr(mod, n).grad for n in names}}

    full = grads(("x", "w", *names))
    for n in full:
        only = grads((n,))
        assert torch.equal(only[n], full[n]) and all(only[m] is None for m in only if m != n), n


@pytest.mark.parametrize("adt", (torch.float32, torch.bfloat16))
def test_a_backward_without_tokens_writes_zero_adapter_gradients(adt):
    """The adapters' gradients have their size whatever the tokens: written, not left as they were allocated."""
    _announce(f"no tokens {adt}")
    E_, hid, inter, r = 3, 128, 64, 5
    w1, w2 = F._for_tokens(F._qweights(_build(E_=E_, hid=hid, inter=inter, r=r).base), 64)
    lora = [torch.ones(E_, *s, dtype=adt, device=DEV) for s in ((r, hid), (2 * inter, r), (r, inter), (hid, r))]
    x, idx = torch.zeros(0, hid, dtype=torch.bfloat16, device=DEV), torch.zeros(0, 2, dtype=torch.int64, device=DEV)
    w = torch.zeros(0, 2, device=DEV)
    out, saved = ops.train_forward(x, idx, w, w1, w2, lora, 1.0, N.EPI_SWIGLU, 0.0, torch.bfloat16)
    assert out.shape == (0, hid)
    stale = [torch.full_like(t, float("nan")) for t in lora]
    del stale  # the allocator hands these blocks out again
    grads = ops.train_backward(out, x, w, w1, w2, lora, 1.0, N.EPI_SWIGLU, 0.0, saved, (True,) * 6)
    assert grads[0].shape == x.shape and grads[1].shape == w.shape
    for g, t in zip(grads[2:], lora):
        assert g.shape == t.shape and g.dtype == adt and not g.any()
    only = ops.train_backward(out, x, w, w1, w2, lora, 1.0, N.EPI_SWIGLU, 0.0, saved, (False,) * 3 + (True,) + (False,) * 2)
    assert [t is None for t in only] == [True, True, True, False, True, True]


@pytest.mark.parametrize("T,E_,top,hid,inter,cdt,kind", [
    (60, 8, 2, 256, 512, torch.float16, "swiglu"),     # fp16 over 32-row tiles, K a multiple of 256: exact weights in registers
    (60, 8, 2, 192, 320, torch.float16, "swiglu"),     # ... and off it
    (900, 4, 2, 256, 128, torch.float16, "swiglu"),    # 128-row tiles
    (300, 4, 2, 192, 128, torch.bfloat16, "gelu"),     # an activation that only the base's Python code knows
    (300, 4, 2, 192, 128, torch.bfloat16, "ranks"),    # two ranks
    (40, 4, 2, 256, 128, torch.bfloat16, "dtypes"),    # adapters of two dtypes
])
def test_per_projection_functions_match_fp64(T, E_, top, hid, inter, cdt, kind):
    """Layers that the two-call form does not take, projection by projection: outputs and every gradient against
    fp64 autograd, dropped ids among them. 1e-2 in norm for bf16, as above; fp16 keeps three more bits (an
    eighth), twice that."""
    _announce(f"per projection T={T} E={E_} hid={hid} inter={inter} {cdt} {kind}")
    torch.manual_seed(23)
    act = torch.nn.functional.gelu if kind == "gelu" else None
    base = e4b.Experts4bit.from_float((torch.randn(E_, 2 * inter, hid) * 0.1).to(DEV), (torch.randn(E_, hid, inter) * 0.1).to(DEV),
                                      compute_dtype=cdt, **({"activation": act} if act else {}))
    mod = e4b.ExpertsLoRA(base, r=16, alpha=32, dtype=torch.float32).to(DEV).train()
    with torch.no_grad():
        for p in (mod.gate_up_lora_B, mod.down_lora_B):
            p.normal_(0, 0.05)
    if kind == "ranks":
        mod.down_lora_A = torch.nn.Parameter(torch.randn(E_, 5, inter, device=DEV) / 5)
        mod.down_lora_B = torch.nn.Parameter(torch.randn(E_, hid, 5, device=DEV) * 0.05)
    if kind == "dtypes":
        for n in ("down_lora_A", "down_lora_B"):
            setattr(mod, n, torch.nn.Parameter(getattr(mod, n).detach().to(torch.bfloat16)))
    assert e4b.enable_fast_train(mod) == 1
    x = torch.randn(T, hid, device=DEV).to(cdt).requires_grad_()
    idx = torch.rand(T, E_, device=DEV).argsort(1)[:, :top].contiguous()
    idx[1, 0], idx[2, top - 1] = -1, E_
    w = torch.rand(T, top, device=DEV).to(cdt).requires_grad_()
    grad = torch.randn(T, hid, device=DEV).to(cdt)
    assert train._layer_inputs(mod, x.detach(), idx, w) is None
    out = mod(x, idx, w)
    out.backward(grad)

    def gated(proj):
        g, u = proj.chunk(2, -1)
        return act(g) * u

    want = _layer_fp64(base, mod, x.detach(), idx, w.detach(), grad, gated if act else _swiglu64())
    got = {"out": out.detach(), "x": x.grad, "w": w.grad, **{n: p.grad for n, p in mod.named_parameters() if "lora" in n}}
    tol = GRAD_TOL if cdt == torch.bfloat16 else GRAD_TOL / 4
    for n in want:
        assert got[n].dtype == (out.dtype if n in ("out", "x", "w") else getattr(mod, n).dtype)
        assert _rel(got[n], want[n]) < tol, (n, _rel(got[n], want[n]))
    assert w.grad[1, 0] == 0 and w.grad[2, top - 1] == 0


@pytest.mark.parametrize("T,E_", [(600, 4), (60, 8)])
def test_wide_gradient_rows_are_no_further_from_fp64(T, E_, monkeypatch):
    """Gradient rows whose values span 2^-30 .. 1: the fp16 mode's scaled rows (values below 2^-31 of a row's
    largest lose bits) against the per-projection functions' bf16 rows and weights."""
    _announce(f"wide gradient rows T={T} E={E_}")
    args = _inputs(T, seed=13, E_=E_)
    g_ = torch.Generator(device=DEV).manual_seed(14)
    scale = torch.exp2(-30 * torch.rand(args[0].shape, generator=g_, device=DEV))
    err = {}
    for lane in ("layer", "projections"):
        mod = _build(seed=12, E_=E_)
        assert e4b.enable_fast_train(mod) == 1
        if lane == "projections":
            monkeypatch.setattr(train, "_layer_inputs", lambda *a: None)
        hs, grad = args[0].clone().requires_grad_(), (args[3] * scale).to(torch.bfloat16)
        mod(hs, *args[1:3]).backward(grad)
        want = _layer_fp64(mod.base, mod, args[0], args[1], args[2], grad, _swiglu64())
        err[lane] = {"x": _rel(hs.grad, want["x"]), **{n: _rel(p.grad, want[n]) for n, p in mod.named_parameters() if "lora" in n}}
    print(err, flush=True)
    for n in err["layer"]:
        assert err["layer"][n] <= err["projections"][n], n
