"""The transformer block's differentiable passes (dsalt_norm_train, dsalt_swiglu_rows and the
functions over them) against float64 and against torch's composition of the same ops."""
import pytest
import torch
import torch.nn.functional as F

from dsalt import _hip
from dsalt.kernels import _block_train
from dsalt.kernels.RMSENorm import RMSENorm
from dsalt.modules import DSALTAttention
from dsalt.modules.dsalt_transformer import DSALTTransformerBlock, SwiGLUFFN

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF, HF, FP = torch.bfloat16, torch.float16, torch.float32
EPS = {BF: 2.0 ** -8, HF: 2.0 ** -11, FP: 2.0 ** -20}


def close(got, want, dtype, what):
    """One rounding to the dtype (half an ulp is EPS/2 relative) plus fp32 sums over a row, as
    a share of the largest value of the tensor's row sums: 2^-20 of its norm."""
    want = want.double()
    err = (got.double() - want).abs()
    tol = EPS[dtype] * want.abs() + 2.0 ** -18 * want.abs().max() + (2.0 ** -24 if dtype == HF else 0)
    assert bool((err <= tol).all()), (what, float((err - tol).max()))


@pytest.mark.parametrize("xd,hd,wd", [(FP, BF, FP), (FP, HF, FP), (FP, FP, FP), (BF, BF, BF), (BF, BF, FP), (HF, HF, HF),
                                      (HF, HF, FP)])
@pytest.mark.parametrize("rows,d", [(1, 8), (3, 512), (5, 520), (3101, 1024), (7, 1032), (2, 2056), (1601, 4096)])
def test_norm_train(xd, hd, wd, rows, d):
    """d: both edges of one wave per row (two chunks per lane) and of four; more rows than the
    backward's workgroups take at once."""
    print(f"norm_train {xd} {hd} {wd} {rows}x{d}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(rows + d)
    rnd = lambda dt, *s: torch.randn(*s, device=DEV, generator=g).to(dt)
    x, h, w, dy, ds = rnd(xd, rows, d), rnd(hd, rows, d), rnd(wd, d), rnd(hd, rows, d), rnd(xd, rows, d)
    cast = hd if xd == FP and hd != FP else None
    s, y, yc, rstd = _hip.norm_train(x, h, w, 1e-6, True, cast)
    assert torch.equal(s, x + h)
    s64, w64 = s.double().requires_grad_(), w.double().requires_grad_()
    y64 = s64 * torch.rsqrt(s64.square().mean(-1, keepdim=True) + 1e-6) * w64
    close(y, y64.detach(), xd, "y")
    if cast is not None:
        assert torch.equal(yc, y.to(cast))
        assert torch.equal(_hip.norm_train(x, h, w, 1e-6, False, cast)[2], yc)
    gx, gw = torch.autograd.grad(y64, (s64, w64), dy.double())
    for res in (ds, None):
        dx, dh, dw = _hip.norm_train_bwd(s, w, rstd, dy, res, hd if hd != xd else None, True, True)
        want = gx if res is None else gx + res.double()
        close(dx, want, xd, "dx")
        close(dw, gw, wd, "dw")
        if dh is not None:
            assert torch.equal(dh, dx.to(hd))
    assert _hip.norm_train_bwd(s, w, rstd, dy, ds, None, False, True)[0] is None
    s0, y0, _, _ = _hip.norm_train(s, None, w, 1e-6)
    assert s0 is None and torch.equal(y0, y)
    assert torch.equal(_hip.norm_train(x, h, None, 0.0)[0], s)


@pytest.mark.parametrize("dtype", [BF, HF, FP])
@pytest.mark.parametrize("rows,f", [(1, 8), (37, 24), (3, 2048), (300, 2816)])
def test_swiglu_rows(dtype, rows, f):
    print(f"swiglu_rows {dtype} {rows}x{f}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(f)
    gu = (3 * torch.randn(rows, 2 * f, device=DEV, generator=g)).to(dtype)
    gu[0, 0], gu[0, 1], gu[0, 2] = 60.0, -60.0, 0.0  # ends of the sigmoid
    da = torch.randn(rows, f, device=DEV, generator=g).to(dtype)
    gate, up = gu[:, :f].contiguous(), gu[:, f:].contiguous()
    assert torch.equal(_hip.swiglu_rows(gu), _hip.swiglu(gate, up))
    got = _hip.swiglu_rows(gu, da)
    g64 = gate.double().requires_grad_()
    dg, = torch.autograd.grad(F.silu(g64) * up.double(), g64, da.double())
    close(got[:, :f], dg, dtype, "dgate")
    close(got[:, f:], da.double() * F.silu(gate).double(), dtype, "dup")


@pytest.mark.parametrize("dtype,autocast", [(BF, False), (HF, False), (FP, False), (FP, True)])
def test_swiglu_function(dtype, autocast):
    """Against the module's projections called one by one: the gradients differ by the roundings
    between torch's passes (a few half ulps, here as a share of each tensor's norm)."""
    print(f"swiglu function {dtype} autocast={autocast}", flush=True)
    torch.manual_seed(3)
    ffn = SwiGLUFFN(128, 264).to(DEV, dtype)
    x = torch.randn(2, 75, 128, device=DEV).to(dtype)
    dy = torch.randn(2, 75, 128, device=DEV)
    out = []
    for one in (True, False):
        ffn.zero_grad()
        xx = x.clone().requires_grad_()
        with torch.autocast("cuda", dtype=BF, enabled=autocast):
            assert _block_train.swiglu_supported(ffn, xx)
            y = ffn(xx) if one else ffn.down_proj(F.silu(ffn.gate_proj(xx)) * ffn.up_proj(xx))
        y.backward(dy.to(y.dtype))
        out.append([y.detach(), xx.grad] + [p.grad for p in ffn.parameters()])
    tol = 4 * EPS[BF if autocast else dtype]
    for a, b in zip(*out):
        assert a.dtype == b.dtype and a.shape == b.shape
        assert float((a.double() - b.double()).norm()) <= tol * float(b.double().norm())


def test_twice_differentiable_and_transformed():
    """What torch's composition allowed is kept: a graph of the backward, functorch transforms,
    forward mode, hooks on a projection, a frozen weight."""
    print("block functions: second order, transforms, hooks", flush=True)
    torch.manual_seed(4)
    ffn, norm = SwiGLUFFN(64, 72).to(DEV), RMSENorm(64).to(DEV)
    x = torch.randn(5, 64, device=DEV, requires_grad=True)
    h = torch.randn(5, 64, device=DEV, requires_grad=True)
    v = torch.randn(5, 64, device=DEV)

    def second(f):
        gx, = torch.autograd.grad((f() * v).sum(), x, create_graph=True)
        return torch.autograd.grad(gx.square().sum(), (x, h), allow_unused=True)

    def plain_ffn(t):
        return ffn.down_proj(F.silu(ffn.gate_proj(t)) * ffn.up_proj(t))

    def pair(s, y):
        return s.tanh() + y

    cases = [(lambda: ffn(x + h), lambda: plain_ffn(x + h)),
             (lambda: pair(*_block_train.add_norm(x, h, norm)), lambda: pair(x + h, norm(x + h))),
             (lambda: pair(*_block_train.add_norm(x, None, norm)), lambda: pair(x, norm(x)))]
    for one, ref in cases:
        for a, b in zip(second(one), second(ref)):
            assert (a is None) == (b is None)
            if a is not None:
                assert float((a - b).norm()) <= 1e-4 * float(b.norm())
    one = torch.func.jacrev(lambda t: ffn(t).sum())(x.detach())
    ref, = torch.autograd.grad(plain_ffn(x).sum(), x)
    assert float((one - ref).norm()) <= 1e-4 * float(ref.norm())
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(x.detach(), v)
        assert torch.autograd.forward_ad.unpack_dual(ffn(dual)).tangent is not None
    seen = []
    hook = ffn.up_proj.register_forward_hook(lambda m, a, o: seen.append(1))
    ffn(x)
    assert seen == [1]
    hook.remove()
    ffn.up_proj.weight.requires_grad_(False)
    ffn.zero_grad()
    ffn(x).sum().backward()
    assert ffn.up_proj.weight.grad is None and ffn.gate_proj.weight.grad is not None


@pytest.mark.parametrize("fwd", [None, HF, BF])
@pytest.mark.parametrize("bwd", [HF, BF])
@pytest.mark.parametrize("part", ["ffn", "attention"])
def test_backward_inside_autocast(part, fwd, bwd):
    """A backward called inside an autocast, of the forward's type or another, gives the gradients
    that it gives outside."""
    print(f"{part}: backward inside autocast fwd={fwd} bwd={bwd}", flush=True)
    torch.manual_seed(5)
    if part == "ffn":
        mod = SwiGLUFFN(128, 264).to(DEV)
        run = mod
    else:
        mod = DSALTAttention(128, 2, 4, 30, 4, max_seq_len=100).to(DEV).train()
        mod._apply_out_proj = lambda o: o  # torch's linear follows the autocast around its backward
        cu = torch.tensor([0, 75], dtype=torch.int32, device=DEV)
        run = lambda x: mod(x, cu_seqlens=cu)[0]  # noqa: E731
    x = torch.randn(75, 128, device=DEV, requires_grad=True)
    got = []
    for inside in (False, True):
        with torch.autocast("cuda", dtype=fwd or BF, enabled=fwd is not None):
            y = run(x)
        with torch.autocast("cuda", dtype=bwd, enabled=inside):
            got.append(torch.autograd.grad(y, [x, *(p for n, p in mod.named_parameters() if "out_proj" not in n)],
                                           torch.ones_like(y)))
    for a, b in zip(*got):
        assert a.dtype == b.dtype and torch.equal(a, b)


@pytest.mark.parametrize("name", ["gate_proj", "up_proj", "down_proj"])
@pytest.mark.parametrize("x_grad", [True, False])
def test_weights_changed_before_the_backward(name, x_grad):
    """As with linears: gate's and up's weights are refused where x takes a gradient, down's always
    (its input takes one), and the others are free to change."""
    print(f"swiglu changed {name} x_grad={x_grad}", flush=True)
    torch.manual_seed(5)
    ffn = SwiGLUFFN(64, 72).to(DEV)
    x = torch.randn(9, 64, device=DEV).requires_grad_(x_grad)
    want = torch.autograd.grad(ffn(x).sum(), list(ffn.parameters()))
    y = ffn(x)
    with torch.no_grad():
        getattr(ffn, name).weight.mul_(1.5)
    if x_grad or name == "down_proj":
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            y.sum().backward()
    else:
        for a, b in zip(torch.autograd.grad(y.sum(), list(ffn.parameters())), want):
            assert torch.equal(a, b)


@pytest.mark.parametrize("dtype,autocast", [(FP, True), (BF, False)])
@pytest.mark.parametrize("shape", [(40, 128), (1, 40, 128)])
def test_outputs_can_be_modified_in_place(dtype, autocast, shape):
    """Hooks that scale the feed-forward's or the attention's output in place, as on torch's ops."""
    print(f"block in place {dtype} {shape}", flush=True)
    torch.manual_seed(2)
    block = DSALTTransformerBlock(128, 2, 4, 30, 4, 100, 264).to(DEV, dtype).train()
    x = torch.randn(shape, device=DEV).to(dtype)
    packed = {} if len(shape) == 3 else {"cu_seqlens": torch.tensor([0, 40], dtype=torch.int32, device=DEV)}
    got = []
    for inplace in (True, False):
        hooks = [block.ffn.register_forward_hook(lambda m, a, o: o.mul_(2) if inplace else o * 2),
                 block.attn.register_forward_hook(lambda m, a, o: (o[0].mul_(2) if inplace else o[0] * 2, o[1]))]
        xx = x.clone().requires_grad_()
        with torch.autocast("cuda", dtype=BF, enabled=autocast):
            y, _ = block(xx, **packed)
        got.append([y.detach(), *torch.autograd.grad(y.float().sum(), [xx, *block.parameters()])])
        for hk in hooks:
            hk.remove()
    for a, b in zip(*got):
        assert torch.equal(a, b)


def test_second_order_of_dependent_inputs():
    """A graph of the backward where one input is computed from another (the norm's weight and the
    feed-forward's weights from x): each gradient counts its own share once."""
    print("block functions: dependent inputs", flush=True)
    torch.manual_seed(7)
    ffn, norm = SwiGLUFFN(64, 72).to(DEV), RMSENorm(64).to(DEV)
    x = torch.randn(5, 64, device=DEV, requires_grad=True)
    ws = {n: p.detach() for n, p in ffn.named_parameters()}

    def one():
        own = {n: p * x.mean() for n, p in ws.items()}
        w = 1 + x[0]
        t = RMSENorm(64).to(DEV)
        t.__dict__["_parameters"] = {"weight": w}
        s, y = _block_train.add_norm(x, None, t)
        return torch.func.functional_call(ffn, own, (s + y,))

    def ref():
        g, u, d = (ws[f"{n}_proj.weight"] * x.mean() for n in ("gate", "up", "down"))
        h = x + F.rms_norm(x, (64,), 1 + x[0], norm.eps)
        return F.linear(F.silu(F.linear(h, g)) * F.linear(h, u), d)

    for f in (one, ref):
        first, = torch.autograd.grad(f().square().sum(), x, create_graph=True)
        second, = torch.autograd.grad(first.square().sum(), x)
        if f is one:
            want = first.detach(), second
    for a, b in zip(want, (first, second)):
        assert float((a - b).norm()) <= 1e-4 * float(b.norm())


@pytest.mark.parametrize("dtype,autocast", [(FP, True), (BF, False), (BF, True)])
@pytest.mark.parametrize("checkpoint", [False, True])
def test_block_matches_separate_ops(dtype, autocast, checkpoint):
    """A training step of the block with its fused passes and with torch's ops in their place
    (fp32 parameters with a bf16 stream in the third case: no projection takes the one-function
    route there unless autocast rounds it)."""
    print(f"block {dtype} autocast={autocast} checkpoint={checkpoint}", flush=True)
    torch.manual_seed(6)
    block = DSALTTransformerBlock(256, 4, 8, 64, 8, 512, 704).to(DEV, FP if autocast else dtype).train()
    with torch.no_grad():  # weights of 1 leave all rows one norm, whose standardised scores are noise
        block.attn_norm.weight.uniform_(0.2, 1.8)
    cu = torch.tensor([0, 200, 333], dtype=torch.int32, device=DEV)
    x = torch.randn(333, 256, device=DEV).to(dtype)
    dy = torch.randn(333, 256, device=DEV)
    out = []
    for fused in (True, False):
        block.zero_grad()
        block._fuse_norms = fused
        hooks = [] if fused else [block.ffn.up_proj.register_forward_hook(lambda m, a, o: None)]
        xx = x.clone().requires_grad_()
        with torch.autocast("cuda", dtype=BF, enabled=autocast):
            y, _ = block(xx, cu_seqlens=cu, cu_list=[0, 200, 333], gradient_checkpointing=checkpoint)
        assert y.dtype == dtype
        y.backward(dy.to(y.dtype))
        out.append({"y": y.detach(), "x": xx.grad, **{n: p.grad for n, p in block.named_parameters()}})
        for hk in hooks:
            hk.remove()
    for n, a in out[0].items():
        b = out[1][n]
        assert a.dtype == b.dtype
        # each of the separate ops rounds once more on the way (2^-9 a time, five to eight of them);
        # the gate's bias and alpha sum cancelling terms over the tokens and the slots
        share = 2.0 ** -5 if n in ("attn.win_gate.bias", "attn.alpha_w") else 2.0 ** -7
        assert float((a.double() - b.double()).norm()) <= share * float(b.double().norm()), n
