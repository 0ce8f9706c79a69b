"""The attention module's core as one function (RoPE, selection, weights, attention): its
operands against dsalt_rope and a cast, the un-rotated gradients of the backward kernels
against rotating them afterwards, and the module's output and gradients against the
composed route (separate RoPE, selection and attention functions)."""
import math

import pytest
import torch

from dsalt import _hip
from dsalt.kernels.window_utils import build_rope_cache
from dsalt.modules import DSALTAttention

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def tables(rows, D, cat=True, seed=0):
    if cat:
        return tuple(t.to(DEV) for t in build_rope_cache(rows, D, torch.device("cpu")))
    g = torch.Generator().manual_seed(seed)
    return tuple(torch.randn(rows, D, generator=g).to(DEV) for _ in range(2))


@pytest.mark.parametrize("H,n_kv,D,dtype,strided,cat,rows", [
    (4, 4, 64, torch.bfloat16, True, True, 300), (6, 2, 128, torch.float16, False, False, 300),
    (8, 4, 64, torch.float32, False, True, 300), (3, 1, 128, torch.float32, True, False, 300),
    (2, 2, 64, torch.bfloat16, False, True, 100)], ids=["bf16-strided", "fp16-d128-gqa", "fp32", "fp32-mqa-strided", "past"])
def test_norms_pass_operands_equal_rope_then_cast(H, n_kv, D, dtype, strided, cat, rows):
    print(f"operands H={H} n_kv={n_kv} D={D} {dtype}", flush=True)
    g = torch.Generator().manual_seed(H + D)
    lens, d = [257, 0, 30], 192
    T = sum(lens)
    cu = torch.tensor([0, 257, 257, 287], dtype=torch.int32, device=DEV)
    wide = torch.randn(T, H + 2 * n_kv, D, generator=g).to(DEV, dtype)
    q, k, v = wide[:, :H], wide[:, H:H + n_kv], wide[:, H + n_kv:]
    if not strided:
        q, k, v = q.contiguous(), k.contiguous(), v.contiguous()
    x = torch.randn(T, d, generator=g).to(DEV, dtype)
    w = (1 + 60 * torch.rand(T, generator=g)).to(DEV)
    alpha = torch.rand(H, generator=g).to(DEV)
    cos, sin = tables(rows, D, cat)
    q_r, k_r = _hip.rope(q, k, cos, sin, cu)
    f = _hip.SelectHybridLauncher(x, v, alpha, H, w, cu, 16, max_seqlen=257, rope_k=(k, cos, sin, cu), rope_q=q)
    f()  # rotates q and k in place unless they are fp32
    w_ref, pos_ref, _ = _hip.select_hybrid(x, v, alpha, H, w, cu, 16, max_seqlen=257)
    cdt = _hip.compute_dtype(dtype)
    assert f.q_out.dtype == f.k_out.dtype == f.v_out.dtype == cdt
    for got, want in ((f.q_out, q_r.to(cdt)), (f.k_out, k_r.to(cdt)), (f.v_out, v.to(cdt))):
        assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(), want.nan_to_num())
    assert torch.equal(f.out, pos_ref) and torch.equal(f.w_out, w_ref)


@pytest.mark.parametrize("cat,rows", [(True, 400), (False, 400), (True, 200)], ids=["module-tables", "any-tables", "past"])
@pytest.mark.parametrize("mode,D,dtype", [(_hip.MODE_HARD, 64, torch.bfloat16), (_hip.MODE_SOFT, 64, torch.float16),
                                          (_hip.MODE_SOFT, 128, torch.bfloat16), (_hip.MODE_DENSE, 64, torch.bfloat16)])
def test_backward_unrotates_like_rope(mode, D, dtype, cat, rows):
    """dq and dk returned un-rotated against dsalt_rope's transposed rotation of the plain
    backward's, in fp32 (the two contract products differently: a few ulp of each pair)."""
    print(f"bwd rope mode={mode} D={D} {dtype} cat={cat} rows={rows}", flush=True)
    g = torch.Generator().manual_seed(D + mode)
    H, lens = 2, [331] if mode == _hip.MODE_DENSE else [331, 1, 96]
    T = sum(lens)
    cu_list = [0, 331] if mode == _hip.MODE_DENSE else [0, 331, 332, 428]
    cu = torch.tensor(cu_list, dtype=torch.int32, device=DEV)
    q, k, v, do = (torch.randn(T, H, D, generator=g).to(DEV, dtype) for _ in range(4))
    w = (2 + 80 * torch.rand(T, generator=g)).to(DEV)
    cos, sin = tables(rows, D, cat)
    scale = 1 / math.sqrt(D)
    # the tables rounded as the forward's rotation rounds them
    cos_r, sin_r = cos.to(dtype).float(), sin.to(dtype).float()
    if mode == _hip.MODE_DENSE:
        out, lse = _hip.dense_fwd(q, k, v, w, None, scale)
        run = lambda rope: _hip.dense_bwd(q, k, v, out, lse, do, w, None, scale, grad_dtype=torch.float32, rope=rope)  # noqa: E731
    else:
        if mode == _hip.MODE_HARD:
            w = w.floor()
        pos = _hip.select_landmarks(torch.randn(T, H, generator=g).to(DEV), w.floor(), cu, 12)
        out, lse = _hip.fwd(mode, q, k, v, w, pos, None, cu, scale)
        run = lambda rope: _hip.bwd(mode, q, k, v, out, lse, do, w, pos, None, cu, scale,  # noqa: E731
                                    need_dw=mode == _hip.MODE_SOFT, grad_dtype=torch.float32, rope=rope)
    plain, fused = run(None), run((cos, sin, dtype))
    dq, dk = _hip.rope(plain[0], plain[1], cos_r, sin_r, cu, transpose=True)
    for got, want in ((fused[0], dq), (fused[1], dk)):
        assert torch.equal(got.isnan(), want.isnan()) and bool(got.isnan().any()) == (rows < 331)
        got, want = got.nan_to_num(), want.nan_to_num()
        assert float((got - want).abs().max()) <= 1e-5 * float(want.abs().max())
    for got, want in zip(fused[2:], plain[2:]):
        assert (got is None and want is None) or torch.equal(got, want)


CASES = {
    # heads, n_kv, D, lens (None: unpacked), dtype, k, autocast
    "bf16": (4, 4, 64, [300, 77, 512], torch.bfloat16, 16, False),
    "bf16-gqa-d128": (4, 2, 128, [260, 65], torch.bfloat16, 8, False),
    "fp32": (3, 3, 64, [200, 130], torch.float32, 8, False),
    "autocast": (4, 4, 64, [300, 77], torch.float32, 16, True),
    "no-landmarks": (2, 2, 64, [150], torch.bfloat16, 0, False),
    "dense-bf16": (4, 4, 64, None, torch.bfloat16, 16, False),
    "dense-fp32-gqa": (4, 1, 64, None, torch.float32, 16, False),
    "dense-d128": (2, 2, 128, None, torch.bfloat16, 8, False),
}


@pytest.mark.parametrize("case", list(CASES))
def test_module_training_equals_composed_route(case):
    """Output and every gradient against the route of separate functions. Both round their
    operands and outputs alike; the composed route also rounds dq and dk before rotating
    them back, so the difference is bounded by a few roundings of the compute type."""
    H, n_kv, D, lens, dtype, k, autocast = CASES[case]
    print(f"module attention {case}", flush=True)
    torch.manual_seed(3)
    T = 333 if lens is None else sum(lens)
    mod = DSALTAttention(H * D, H, 8, 100, k, max_seq_len=600, n_kv_heads=n_kv).to(DEV, dtype).train()
    x = torch.randn(T, H * D, device=DEV).to(dtype)
    dy = torch.randn(T, H * D, device=DEV)
    packed = {}
    if lens is None:
        x, dy = x[None], dy[None]
    else:
        cu = torch.tensor([0, *torch.tensor(lens).cumsum(0).tolist()], dtype=torch.int32, device=DEV)
        packed = {"cu_seqlens": cu, "cu_list": cu.tolist()}
    got = {}
    for route in ("one", "composed"):
        if route == "composed":
            mod._one_function = lambda *a: False
        mod.zero_grad(set_to_none=True)
        xx = x.clone().requires_grad_()
        with torch.autocast("cuda", dtype=torch.bfloat16, enabled=autocast):
            y, _ = mod(xx, **packed)
        y.backward(dy.to(y.dtype))
        got[route] = {"y": y.detach(), "x": xx.grad, **{n: p.grad for n, p in mod.named_parameters()}}
        got[route]["sel"] = mod._last_selection[1]
    assert torch.equal(got["one"].pop("sel"), got["composed"].pop("sel"))
    tol = 1e-2 if dtype == torch.bfloat16 or autocast else 2e-3
    for name, a in got["one"].items():
        b = got["composed"][name]
        if a is None or b is None:  # no landmark: alpha takes no gradient
            assert a is None and b is None and k == 0 and name == "alpha_w"
            continue
        assert a.dtype == b.dtype
        if name == "win_gate.bias":  # a sum of cancelling terms: on the scale of its weight's gradient
            assert abs(float(a - b)) <= tol * float(got["composed"]["win_gate.weight"].double().norm())
            continue
        bar = tol
        if name == "alpha_w" and lens is None and dtype == torch.bfloat16:
            # the composed dense route takes torch's norms: where their fp32 sum rounds to the
            # other bf16 neighbour a z moves by ulp / std = 2^-5 / 0.4, one of H k terms here
            bar = 4 * 2 ** -5 / 0.4 / math.sqrt(H * k)
        a, b = a.double(), b.double()
        assert float((a - b).norm()) <= bar * float(b.norm()), name


def small_module(dtype=torch.bfloat16):
    torch.manual_seed(9)
    mod = DSALTAttention(256, 4, 8, 100, 16, max_seq_len=400, n_kv_heads=2).to(DEV, dtype).train()
    cu = torch.tensor([0, 250, 333], dtype=torch.int32, device=DEV)
    return mod, torch.randn(333, 256, device=DEV).to(dtype), {"cu_seqlens": cu, "cu_list": [0, 250, 333]}


def test_hooked_projections_are_called():
    """A hook on a projection takes the route of separate functions, where it runs."""
    print("module attention hooks", flush=True)
    mod, x, packed = small_module()
    assert mod._one_function(x)
    seen = []
    h = mod.k_proj.register_forward_hook(lambda m, a, o: seen.append(o.shape))
    assert not mod._one_function(x)
    mod(x, **packed)[0].float().sum().backward()
    assert seen == [(333, 128)]
    h.remove()
    assert mod._one_function(x)


class OwnSteps(DSALTAttention):
    """A subclass with its own balance, windows and landmark weights."""

    def _alpha(self):
        return torch.sigmoid(3 * self.alpha_w)

    def _window_continuous(self, x):
        return 0.5 * super()._window_continuous(x)

    def _train_selectors(self, *a, **k):
        w, pos, logw = super()._train_selectors(*a, **k)
        return w, pos, logw - 1.0


@pytest.mark.parametrize("where", ["subclass", "instance", "class"])
@pytest.mark.parametrize("dense", [False, True])
def test_replaced_steps_are_called(where, dense, monkeypatch):
    """The steps that the one function and the landmark weights' function stand for, replaced in a
    subclass, on an instance or on the class: each is called."""
    print(f"module attention own steps {where} dense={dense}", flush=True)
    mod, x, packed = small_module()
    seen = []

    def counted(name):
        step = getattr(OwnSteps, name)
        return lambda self, *a, **k: (seen.append(name), step(self, *a, **k))[1]

    if where == "subclass":
        mod.__class__ = type("Counted", (OwnSteps,), {n: counted(n) for n in ("_alpha", "_window_continuous", "_train_selectors")})
    else:
        base = {n: getattr(DSALTAttention, n) for n in ("_alpha", "_window_continuous", "_train_selectors")}
        for n, step in base.items():
            f = lambda self, *a, _n=n, _s=step, **k: (seen.append(_n), _s(self, *a, **k))[1]  # noqa: E731
            if where == "class":
                monkeypatch.setattr(DSALTAttention, n, f)
            else:
                mod.__dict__[n] = f.__get__(mod)
    y = mod(x[None])[0] if dense else mod(x, **packed)[0]
    y.float().sum().backward()
    assert {"_alpha", "_window_continuous"} <= set(seen) and ("_train_selectors" in seen) == (not dense)
    if where == "subclass" and not dense:
        assert not torch.equal(y, small_module()[0](x, **packed)[0])


@pytest.mark.parametrize("frozen", [("q_proj.weight",), ("k_proj.weight", "v_proj.weight", "alpha_w"),
                                    ("win_gate.weight", "win_gate.bias"), ("q_proj.weight", "k_proj.weight", "v_proj.weight")])
@pytest.mark.parametrize("x_grad", [True, False])
def test_frozen_parameters_take_no_gradient(frozen, x_grad):
    """The other gradients are what they are without the freezing (the weights' GEMMs are
    taken apart, so up to their rounding)."""
    print(f"module attention frozen {frozen} x_grad={x_grad}", flush=True)
    mod, x, packed = small_module()
    dy = torch.randn(333, 256, device=DEV).to(x.dtype)
    want = {}
    for pas in ("all", "frozen"):
        mod.zero_grad(set_to_none=True)
        for n, p in mod.named_parameters():
            p.requires_grad_(pas == "all" or n not in frozen)
        xx = x.clone().requires_grad_(pas == "all" or x_grad)
        mod(xx, **packed)[0].backward(dy)
        got = {"x": xx.grad, **{n: p.grad for n, p in mod.named_parameters()}}
        if pas == "all":
            want = got
    for n, g in got.items():
        if n in frozen or (n == "x" and not x_grad):
            assert g is None, n
        else:
            w = want[n].double()
            assert float((g.double() - w).norm()) <= 2 ** -8 * float(w.norm()), n


@pytest.mark.parametrize("name", ["q_proj", "k_proj", "v_proj", "win_gate", "alpha_w"])
@pytest.mark.parametrize("x_grad", [True, False])
def test_weights_changed_before_the_backward(name, x_grad):
    """As with linears: a projection's weight changed in place between the passes is refused where
    it is needed for x's gradient, and taken where x has none."""
    print(f"module attention changed {name} x_grad={x_grad}", flush=True)
    mod, x, packed = small_module()
    x.requires_grad_(x_grad)
    dy = torch.randn(333, 256, device=DEV).to(x.dtype)
    ps = [p for n, p in mod.named_parameters() if n != "out_proj.weight"]
    want = torch.autograd.grad(mod(x, **packed)[0], ps, dy)
    y = mod(x, **packed)[0]
    with torch.no_grad():
        (mod.alpha_w if name == "alpha_w" else getattr(mod, name).weight).mul_(1.5)
    if x_grad and name != "alpha_w":
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            y.backward(dy)
    else:
        for a, b in zip(torch.autograd.grad(y, ps, dy), want):
            assert torch.equal(a, b)


@pytest.mark.parametrize("dtype,autocast", [(torch.bfloat16, False), (torch.float16, False), (torch.float32, True)])
def test_training_windows_are_the_rounded_gate(dtype, autocast):
    """The windows of the norms pass are torch's formula on the correctly rounded logits."""
    print(f"module attention windows {dtype} autocast={autocast}", flush=True)
    mod, x, packed = small_module(dtype)
    with torch.no_grad():
        mod.win_gate.weight.mul_(8)
    cdt = torch.bfloat16 if autocast else dtype
    with torch.autocast("cuda", dtype=torch.bfloat16, enabled=autocast):
        mod(x, **packed)
    w, b = mod.win_gate.weight.to(cdt).double(), mod.win_gate.bias.to(cdt).double()
    logit = (x.to(cdt).double() @ w.t() + b).squeeze(-1).to(cdt)
    want = mod.n_min + torch.sigmoid(logit) * (mod.n_max - mod.n_min)
    assert torch.equal(mod._last_selection[0], want.float().floor().clamp(min=1))


def test_alpha_takes_no_gradient_without_landmarks():
    """With k_lmk = 0 no weight depends on alpha: its gradient is None (an optimizer leaves it
    alone), not zeros. The dense variant's table holds a weight for every key, so zeros there."""
    print("module attention alpha without landmarks", flush=True)
    mod, x, packed = small_module()
    mod.k_lmk = 0
    mod(x, **packed)[0].float().sum().backward()
    assert mod.alpha_w.grad is None and mod.v_proj.weight.grad is not None
    mod(x[None])[0].float().sum().backward()
    assert bool((mod.alpha_w.grad == 0).all())


@pytest.mark.parametrize("dtype,autocast", [(torch.bfloat16, False), (torch.float32, False), (torch.float32, True)])
def test_dense_last_selection_keeps_its_types(dtype, autocast):
    """The dense variant's _last_selection: windows in the gate's type on either route."""
    print(f"module attention dense selection {dtype} autocast={autocast}", flush=True)
    mod, x, _ = small_module(dtype)
    got = []
    for hip in (True, False):
        mod._hip_scores = hip
        with torch.autocast("cuda", dtype=torch.bfloat16, enabled=autocast):
            mod(x[None])
        got.append(mod._last_selection)
    (w1, p1), (w2, p2) = got
    assert w1.dtype == w2.dtype == (torch.bfloat16 if autocast else dtype) and p1.dtype == p2.dtype == torch.int64
    assert float((w1.double() - w2.double()).abs().max()) <= 2.0 ** (-20 if w1.dtype == torch.float32 else -7) * mod.n_max


@pytest.mark.parametrize("T,k", [(1, 0), (1, 4), (70, 0), (70, 4)])
def test_non_finite_scores_in_training(T, k):
    """The scores' gradients with one token or an infinite state are autograd's: NaN (0 times
    NaN) with landmark slots, and without any nothing comes in through them."""
    print(f"module attention non-finite T={T} k={k}", flush=True)
    got = {}
    for hip in (True, False):
        torch.manual_seed(5)
        mod = DSALTAttention(256, 4, 8, 100, k, max_seq_len=400, n_kv_heads=2).to(DEV, torch.bfloat16).train()
        mod._hip_scores = hip  # False: torch's ops
        x = torch.randn(T, 256, device=DEV).to(torch.bfloat16)
        if T > 1:
            x[T // 2, 3] = float("inf")
        x.requires_grad_()
        assert mod._one_function(x) == hip
        mod(x, cu_seqlens=torch.tensor([0, T], dtype=torch.int32, device=DEV))[0].float().sum().backward()
        got[hip] = {"x": x.grad, **{n: p.grad for n, p in mod.named_parameters()}}
    for n, want in got[False].items():
        a = got[True][n]
        if want is not None:
            assert torch.equal(a.isnan(), want.isnan()), n
    assert got[True]["alpha_w"] is None if k == 0 else bool(got[True]["alpha_w"].isnan().all())


def second_order(mod, x, packed, dy, autocast=False):
    """First gradients (with a graph) of x and the parameters, and the gradients of their squares'
    sum."""
    ps = [x, *mod.parameters()]
    with torch.autocast("cuda", dtype=torch.bfloat16, enabled=autocast):
        y = mod(x, **packed)[0]
        first = torch.autograd.grad(y, ps, dy.to(y.dtype), create_graph=True, allow_unused=True)
        penalty = sum(g.float().square().sum() for g in first if g is not None)
    return first, torch.autograd.grad(penalty, ps, allow_unused=True)


SECOND = {  # H, n_kv, D, dense, dtype, k, autocast
    "fp32": (4, 4, 64, False, torch.float32, 8, False), "fp32-gqa-d128": (4, 2, 128, False, torch.float32, 8, False),
    "bf16": (4, 2, 64, False, torch.bfloat16, 8, False), "autocast": (4, 2, 64, False, torch.float32, 8, True),
    "no-landmarks": (2, 2, 64, False, torch.float32, 0, False), "dense": (4, 2, 64, True, torch.float32, 8, False),
    "dense-d128": (2, 2, 128, True, torch.float32, 8, False), "dense-autocast": (2, 1, 64, True, torch.float32, 8, True),
}


@pytest.mark.parametrize("case", list(SECOND))
@pytest.mark.parametrize("route", ["one", "weights"])
def test_second_order_gradients(case, route):
    """A graph of the backward holds what torch's projections, gate and landmark weights hold: both
    the one function and the landmark weights' function ("weights") against torch's ops, whose
    attention core is a constant in the graph on every route."""
    H, n_kv, D, dense, dtype, k, autocast = SECOND[case]
    print(f"module attention second order {case} {route}", flush=True)
    lens = [130, 77]
    got = {}
    for r in (route, "torch"):
        torch.manual_seed(8)
        mod = DSALTAttention(H * D, H, 4, 32, k, max_seq_len=300, n_kv_heads=n_kv).to(DEV, dtype).train()
        mod._fuse_qkv, mod._hip_scores = r == "one", r != "torch"
        x = torch.randn(sum(lens), H * D, device=DEV).to(dtype)
        dy = torch.randn(sum(lens), H * D, device=DEV)
        assert mod._one_function(x) == (r == "one")
        packed = {} if dense else {"cu_seqlens": torch.tensor([0, 130, 207], dtype=torch.int32, device=DEV)}
        x, dy = (x[None], dy[None]) if dense else (x, dy)
        got[r] = second_order(mod, x.detach().requires_grad_(), packed, dy, autocast)
    # a few roundings of the compute type (the projections' in fp32 take part in fp16 attention)
    tol = 2e-2 if dtype == torch.bfloat16 or autocast else 2e-3
    names = ["x", *(n for n, _ in mod.named_parameters())]
    for order in (0, 1):
        for n, a, b in zip(names, got[route][order], got["torch"][order]):
            assert (a is None) == (b is None) and (a is None or a.requires_grad == b.requires_grad), (order, n)
            if a is None or n == "win_gate.bias":  # a sum of cancelling terms
                continue
            a, b = a.detach().double(), b.detach().double()
            assert float((a - b).norm()) <= tol * float(b.norm()), (order, n, float((a - b).norm() / b.norm()))


def test_fp32_windows():
    """fp32 modules form their windows in the norms pass too: expf within 2 ulp, a division, a
    product and a sum rounded once each, all relative to at most n_max: 2^-21 n_max."""
    print("module attention fp32 windows", flush=True)
    mod, x, _ = small_module(torch.float32)
    with torch.no_grad():
        mod.win_gate.weight.mul_(8)
        mod(x[None])
    logit = x.double() @ mod.win_gate.weight.double().squeeze(0) + mod.win_gate.bias.double()
    want = mod.n_min + torch.sigmoid(logit) * (mod.n_max - mod.n_min)
    assert float((mod._last_selection[0].double() - want).abs().max()) <= 2.0 ** -21 * mod.n_max


# tokens per workgroup of the states' pass (8, 16 from 4096 tokens, 32 from 16384; the last
# workgroup partly filled) and rows of one, exactly and just over 256 column chunks
@pytest.mark.parametrize("T,d,H,n_kv,dtype", [
    (33, 64, 2, 2, torch.bfloat16), (4095, 2048, 2, 1, torch.bfloat16), (4099, 2056, 2, 1, torch.float16),
    (16387, 72, 3, 3, torch.bfloat16), (4097, 1028, 2, 2, torch.float32), (16384, 1024, 2, 1, torch.float32)])
def test_module_grads_at_the_edges_of_its_shapes(T, d, H, n_kv, dtype):
    """dsalt_module_grads_v and _x against float64 autograd of the scores, the weights and the gate."""
    print(f"module grads T={T} d={d} H={H}/{n_kv} {dtype}", flush=True)
    g = torch.Generator().manual_seed(T + d)
    rnd = lambda *s: torch.randn(*s, generator=g).to(DEV)  # noqa: E731
    D, k, tau, n_min, n_max = 64, 12, 2.0, 4.0, 60.0
    lens = [T // 3, T - T // 3]
    cu = torch.tensor([0, lens[0], T], dtype=torch.int32, device=DEV)
    x, v = rnd(T, d).to(dtype), rnd(T, n_kv, D).to(dtype)
    aw = rnd(H)
    alpha = torch.sigmoid(aw)
    sel = _hip.SelectHybridLauncher(x, v, alpha, H, 1 + 30 * torch.rand(T, generator=g).to(DEV), cu, k,
                                    max_seqlen=max(lens), norms_f32=True)
    sel()
    _hip.lmk_weights(sel.norms, alpha, sel.out, sel.cu, T, n_kv, tau)
    dlw = rnd(H, 2, k) * 0.1
    dk_h, dv_h, dx_in, dw = rnd(T, H, D).to(dtype), rnd(T, H, D).to(dtype), rnd(T, d).to(dtype), rnd(T) * 0.1
    wg = (rnd(1, d) / d ** 0.5).to(dtype)
    logit = rnd(T).to(dtype).float()
    m = _hip.ModuleGrads(x, v, sel.norms, alpha, sel.out, sel.cu, dlw, tau, False)
    dk, dv = torch.empty(T, n_kv, D, device=DEV, dtype=dtype), torch.empty(T, n_kv, D, device=DEV, dtype=dtype)
    da = m.values(dk_h, dv_h, dk, dv, alpha_sigmoid=True)
    dx, dwg, dbg = m.states(dx_in, True, (wg, logit, dw, dtype, n_min, n_max))

    x64, v64, a64 = (t.detach().double().requires_grad_() for t in (x, v, aw))
    sig = torch.sigmoid(a64)
    z = [(n - n.mean(0)) / n.std(0) for n in (x64.norm(dim=-1), v64.norm(dim=-1))]
    s = sig * z[1].repeat_interleave(H // n_kv, 1) + (1 - sig) * z[0].unsqueeze(1)
    tok = cu[:-1].long().view(1, 2, 1) + sel.out.clamp(min=0)
    filled = sel.out >= 0
    logw = torch.log(torch.sigmoid(s.t().gather(1, tok.view(H, -1)).view(tok.shape) / tau))
    logw[filled].backward(dlw[filled].double())
    assert bool(filled.any()) and bool(filled.all()) == (T > 33)
    sg = torch.sigmoid(logit.double()).to(dtype).double()  # the gate as the forward rounded it
    dl = dw.double() * (n_max - n_min) * sg * (1 - sg)
    want = {"dx": x64.grad + dx_in.double() + dl[:, None] * wg.double(),
            "dv": v64.grad + dv_h.double().view(T, n_kv, -1, D).sum(2), "dwg": (dl @ x.double())[None], "dbg": dl.sum()[None],
            "da": a64.grad}
    if n_kv != H:
        want["dk"] = dk_h.double().view(T, n_kv, -1, D).sum(2)
    # fp32 sums: 1e-4 of the largest value where the standardised norms take part (see the weights'
    # own test), 1e-5 of the terms' sum for the gate's; each result rounded once
    ulp = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -23}[dtype]
    terms = {"dwg": dl.abs() @ x.double().abs(), "dbg": dl.abs().sum()}
    for n, w in want.items():
        got = {"dx": dx, "dv": dv, "dwg": dwg, "dbg": dbg, "da": da, "dk": dk}[n].double()
        bar = ulp * w.abs() + (1e-5 * terms[n] if n in terms else 1e-4 * w.abs().max())
        assert bool(((got - w).abs() <= bar).all()), (n, float(((got - w).abs() - bar).max()))
