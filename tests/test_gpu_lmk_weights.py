"""The differentiable landmark weights (dsalt_lmk_weights and its backward) against float64
torch autograd of the hybrid score and its weight at the selected positions: packed and
table layouts, grouped value heads, 16-bit and fp32 operands, strided views, sequences
without a candidate. Bars: a norm's fp32 sum carries ~1e-6 of its value, which
standardising magnifies by norm / std (about 50 here): 1e-4 of the largest value; 16-bit
gradients add their own rounding, 2^-8 (bf16) or 2^-11 (fp16) of each element."""
import numpy as np
import pytest
import torch

from dsalt import _hip
from dsalt.kernels._lmk_weights import landmark_weights

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)
ULP = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}

CASES = {
    # lens, d, H, n_kv, D, x dtype, v dtype, k, table, strided
    "mha-bf16": ([300, 0, 45, 700], 512, 8, 8, 64, torch.bfloat16, torch.bfloat16, 16, False, False),
    "gqa-autocast": ([257, 90], 256, 8, 2, 128, torch.float32, torch.bfloat16, 33, False, False),
    "mqa-fp16-strided": ([130, 64, 1], 128, 6, 1, 64, torch.float16, torch.float16, 8, False, True),
    "fp32-no-candidate": ([20, 500], 192, 3, 3, 64, torch.float32, torch.float32, 5, False, False),
    "table-bf16": ([333], 256, 4, 2, 64, torch.bfloat16, torch.bfloat16, 16, True, False),
    "table-fp32-all-keys": ([9], 64, 2, 1, 64, torch.float32, torch.float32, 9, True, True),
    "many-value-heads": ([70], 64, 128, 128, 64, torch.float32, torch.float32, 3, False, False),
}


def reference(x, v, alpha, pos, cu, tau, table):
    T, H, n_kv = x.shape[0], alpha.shape[0], v.shape[1]

    def standardise(n):
        return (n - n.mean(0, keepdim=True)) / n.std(0, keepdim=True).clamp(min=1e-6)

    z_v = standardise(v.norm(dim=-1)).repeat_interleave(H // n_kv, dim=1)
    s = alpha * z_v + (1 - alpha) * standardise(x.norm(dim=-1)).unsqueeze(1)
    w = torch.log(torch.sigmoid(s / tau).clamp(min=1e-20)).t()
    tok = torch.tensor(cu[:-1], device=DEV).view(1, -1, 1) + pos.clamp(min=0)
    if table:
        on = torch.zeros(H, T, dtype=torch.bool, device=DEV).scatter(1, tok[:, 0], True)
        return torch.where(on, w, float("-inf"))
    return w.gather(1, tok.view(H, -1)).view(pos.shape).masked_fill(pos < 0, float("-inf"))


@pytest.mark.parametrize("case", list(CASES))
def test_landmark_weights_match_float64_autograd(case):
    lens, d, H, n_kv, D, xdt, vdt, k, table, strided = CASES[case]
    print(f"landmark weights {case}", flush=True)
    g = torch.Generator().manual_seed(len(case))
    cu = [0] + np.cumsum(lens).tolist()
    T = cu[-1]
    x = torch.randn(T, 2 * d if strided else d, generator=g).to(DEV, xdt)[:, :d]
    v = torch.randn(T, n_kv * (2 if strided else 1), D, generator=g).to(DEV, vdt)[:, :n_kv]
    x, v = x.detach().requires_grad_(), v.detach().requires_grad_()
    alpha = torch.rand(H, generator=g).to(DEV).requires_grad_()
    w = (1 + 40 * torch.rand(T, generator=g)).to(DEV)
    if table:
        w = torch.zeros(1, device=DEV).expand(T)  # every key is a candidate, as in the dense variant
    cu_t = torch.tensor(cu, dtype=torch.int32, device=DEV)
    # 16-bit norms unrounded, as under autocast: the reference's norms are exact
    with torch.autocast("cuda", dtype=torch.bfloat16):
        v_out, weight, pos, w_disc = landmark_weights(x, v, alpha, w, cu_t, k, max(lens), 2.0, table)
    assert torch.equal(v_out, v) and (table or torch.equal(w_disc, w.floor()))
    gw = torch.randn(weight.shape, generator=g).to(DEV)
    gv = torch.randn(v.shape, generator=g).to(DEV, vdt)
    torch.autograd.backward([weight, v_out], [gw, gv])

    x64, v64, a64 = (t.detach().double().requires_grad_() for t in (x, v, alpha))
    ref = reference(x64, v64, a64, pos, cu, 2.0, table)
    fin = torch.isfinite(ref)
    assert torch.equal(fin, torch.isfinite(weight)) and bool((weight[~fin] == float("-inf")).all())
    assert bool(fin.any())
    assert float((weight[fin] - ref[fin]).detach().abs().max()) < 1e-4
    torch.autograd.backward([torch.where(fin, ref, 0.0), v64], [torch.where(fin, gw, 0.0).double(), gv.double()])
    for name, got, want, dt in (("x", x.grad, x64.grad, xdt), ("v", v.grad, v64.grad, vdt),
                                ("alpha", alpha.grad, a64.grad, torch.float32)):
        assert got.dtype == dt if name != "alpha" else True
        bar = 1e-4 * float(want.abs().max()) + ULP[dt] * want.abs()
        assert bool(((got.double() - want).abs() <= bar).all()), f"{name}: {float((got.double() - want).abs().max())}"


def test_landmark_weights_without_weight_gradient():
    """Only v's gradient arrives (no landmark took part in the loss): it passes through."""
    print("landmark weights pass-through", flush=True)
    x = torch.randn(50, 64, device=DEV, requires_grad=True)
    v = torch.randn(50, 1, 64, device=DEV, requires_grad=True)
    cu = torch.tensor([0, 50], dtype=torch.int32, device=DEV)
    v_out, *_ = landmark_weights(x, v, torch.full((2,), 0.6, device=DEV), torch.full((50,), 9.0, device=DEV), cu, 4, 50,
                                 2.0)
    gv = torch.randn_like(v)
    v_out.backward(gv)
    assert x.grad is None and torch.equal(v.grad, gv)


@pytest.mark.parametrize("what,T", [("x nan", 70), ("x inf", 70), ("v nan", 70), ("v inf", 70), ("one token", 1)])
@pytest.mark.parametrize("table", [False, True])
def test_non_finite_norms_give_nan(what, T, table):
    """A norm that is not finite, or the std of one token, makes every score NaN: no landmark is
    selected, a selected one would weigh NaN, and the gradients are NaN where autograd's are
    (a zero gradient times NaN)."""
    print(f"landmark weights {what} table={table}", flush=True)
    g = torch.Generator().manual_seed(T)
    H, n_kv = 4, 2
    x, v = torch.randn(T, 64, generator=g).to(DEV), torch.randn(T, n_kv, 64, generator=g).to(DEV)
    if T > 1:
        t = x if what[0] == "x" else v.view(T, -1)
        t[T // 2, 3] = float(what[2:])
    x, v = x.requires_grad_(), v.requires_grad_()
    alpha = torch.full((H,), 0.6, device=DEV, requires_grad=True)
    w = torch.zeros(1, device=DEV).expand(T) if table else torch.ones(T, device=DEV)
    cu = torch.tensor([0, T], dtype=torch.int32, device=DEV)
    v_out, weight, pos, _ = landmark_weights(x, v, alpha, w, cu, 3, T, 2.0, table)
    x64, v64, a64 = (t.detach().double().requires_grad_() for t in (x, v, alpha))
    ref = reference(x64, v64, a64, pos, [0, T], 2.0, table)
    if table:  # the reference weighs what is selected; here nothing may be, in the NaN heads
        ref = torch.where(torch.isfinite(weight), ref, float("-inf"))
    assert torch.equal(torch.isfinite(ref), torch.isfinite(weight))
    fin = torch.isfinite(ref).detach()
    torch.autograd.backward([weight, v_out], [torch.where(fin, 1.0, 0.0), torch.zeros_like(v)])
    torch.where(fin, ref, 0.0).sum().backward()
    assert bool(a64.grad.isnan().any())
    for got, want in ((x, x64), (v, v64), (alpha, a64)):
        assert torch.equal(got.grad.isnan(), want.grad.isnan())
    # a slot that names a token whose score is NaN
    sel = _hip.SelectHybridLauncher(x.detach(), v.detach(), alpha.detach(), H, w, cu, 3, max_seqlen=T, quantize=not table)
    sel()
    named = _hip.lmk_weights(sel.norms, alpha.detach(), torch.zeros_like(pos), sel.cu, T, n_kv, 2.0, table)
    first = named[:, 0] if table else named[:, 0, 0]
    nan_heads = a64.grad.isnan()
    assert torch.equal(first.isnan(), nan_heads)
