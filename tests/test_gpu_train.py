"""GPU: the training side of the layer (not on the forward path).

- requant / fused_lion_requant on device buffers replay the reference's own
  outputs bit for bit (tests/golden/golden_requant.npz, kernel/fp8_tile.py:240-285;
  the CPU replay is tests/test_requant.py).
- A SwiFFN_MoE training step (model.py:557-585 under autograd): the input
  gradient, the router-weight gradient (through the selected probabilities,
  model.py:559-563) and every executed expert's bf16 weight gradients
  (kernel/fp8_tile.py:172-197) against a float64 autograd restatement of the
  same layer on the decoded weights with the same routing.  Bar: relative
  1e-1 of the largest magnitude -- the layer computes in bf16 activations
  (x, the SwiGLU product, expert outputs), so the gradients carry bf16
  rounding; unselected experts get no gradient.
- The same training step against the reference layer's own step
  (tests/golden/golden_train.npz, make_golden_train.py): x.grad, the router
  gradient and every _gw within rel-L2 2e-3.
- Eval mode with grad on keeps the input gradient.
"""
import pytest
import torch
import torch.nn.functional as F

from smaulnative_amd import MoEConfig, SwiFFN_MoE
from smaulnative_amd.fp8_tile import decode_block

pytestmark = pytest.mark.gpu
DEV = "cuda"


def test_requant_and_lion_match_reference_on_device():
    from test_requant import replay
    print("case requant/lion replay on the device", flush=True)
    replay(DEV)


def _dense(lin):
    return decode_block(lin.w8, lin.sc, 0, lin.out_f, lin.in_f, lin.tile).double().cpu()


def rel(a, b):
    a, b = a.double().cpu(), b.double().cpu()
    return float((a - b).abs().max() / b.abs().max().clamp_min(1e-300))


@pytest.mark.parametrize("E,k", [(4, 2), (8, 1)])
def test_moe_training_step_gradients(E, k):
    print(f"case moe training step E={E} k={k}", flush=True)
    torch.manual_seed(11 + E)
    cfg = MoEConfig(d_model=128, ffn_mult=2.5, tile=64, num_experts=E, num_experts_per_tok=k)
    moe = SwiFFN_MoE(cfg).to(DEV).train()
    x = torch.randn(2, 40, 128, device=DEV).to(torch.bfloat16).requires_grad_(True)
    c = torch.randn(2, 40, 128, device=DEV)
    out = moe(x)
    assert out.dtype == torch.bfloat16 and out.shape == x.shape
    (out.float() * c).sum().backward()
    topi = moe.last_topi.cpu().reshape(-1, k)

    # float64 restatement with the module's routing
    xs = x.detach().double().cpu().reshape(-1, 128).requires_grad_(True)
    gw = moe.gate.weight.detach().double().cpu().requires_grad_(True)
    ws = [{n: _dense(getattr(ex, n)).requires_grad_(True) for n in ("gate", "up", "down")} for ex in moe.experts]
    prob = torch.softmax(xs @ gw.t(), -1)
    topv = prob.gather(-1, topi)
    topv = topv / topv.sum(-1, keepdim=True)
    ref = torch.zeros_like(xs)
    for e in range(E):
        wsel = torch.where(topi == e, topv, torch.zeros_like(topv)).sum(-1)
        rows = torch.nonzero(wsel > 0).squeeze(-1)
        if rows.numel():
            xm = xs.index_select(0, rows)
            h = F.silu(xm @ ws[e]["gate"].t()) * (xm @ ws[e]["up"].t())
            ref = ref.index_add(0, rows, (h @ ws[e]["down"].t()) * wsel.index_select(0, rows).unsqueeze(-1))
    (ref * c.double().cpu().reshape(-1, 128)).sum().backward()

    assert rel(out.float().reshape(-1, 128), ref.detach()) < 3e-2
    assert rel(x.grad.float().reshape(-1, 128), xs.grad) < 1e-1
    assert torch.isfinite(moe.gate.weight.grad).all()
    if k == 1:
        # one expert per token: the renormalised weight is p / p = 1, so the
        # router's gradient is zero up to rounding (model.py:565-567)
        assert float(gw.grad.abs().max()) < 1e-9
        assert float(moe.gate.weight.grad.abs().max()) < 1e-4
    else:
        assert rel(moe.gate.weight.grad, gw.grad) < 1e-1
    counts = moe.expert_token_counts
    assert sum(counts) == 80 * k
    for e, ex in enumerate(moe.experts):
        for n in ("gate", "up", "down"):
            lin = getattr(ex, n)
            if counts[e] == 0:
                assert lin._gw is None
            else:
                assert lin._gw is not None and lin._gw.dtype == torch.bfloat16
                assert rel(lin._gw.float(), ws[e][n].grad) < 1e-1, (e, n)


def test_eval_mode_keeps_input_gradient():
    """In eval mode with grad on, SwiFFN_MoE and SwiFFN still record autograd
    (as the reference's FP8Linear function does, kernel/fp8_tile.py:162-170):
    the input gradient equals the train-mode one bit for bit, and no expert
    accumulates _gw (that is the training flag's only effect).  Under no_grad
    the fused entries run and return outputs without a graph."""
    from smaulnative_amd import SwiFFN
    print("case eval-mode input gradient", flush=True)
    torch.manual_seed(5)
    cfg = MoEConfig(d_model=128, ffn_mult=2.5, tile=64, num_experts=4, num_experts_per_tok=2)
    moe = SwiFFN_MoE(cfg).to(DEV)
    x = torch.randn(2, 24, 128, device=DEV).to(torch.bfloat16)
    c = torch.randn(2, 24, 128, device=DEV)
    grads = {}
    for mode in ("train", "eval"):
        moe.train(mode == "train")
        for ex in moe.experts:
            for n in ("gate", "up", "down"):
                getattr(ex, n)._gw = None
        xi = x.clone().requires_grad_(True)
        out = moe(xi)
        assert out.grad_fn is not None, mode
        (out.float() * c).sum().backward()
        grads[mode] = xi.grad.clone()
        gws = [getattr(ex, n)._gw for ex in moe.experts for n in ("gate", "up", "down")]
        if mode == "eval":
            assert all(g is None for g in gws)
        else:
            assert any(g is not None for g in gws)
    assert torch.equal(grads["train"], grads["eval"])
    with torch.no_grad():
        assert moe(x).grad_fn is None

    ffn = SwiFFN(cfg).to(DEV).eval()
    xi = x.clone().requires_grad_(True)
    y = ffn(xi)
    assert y.grad_fn is not None
    (y.float() * c).sum().backward()
    assert xi.grad is not None and torch.isfinite(xi.grad.float()).all() and float(xi.grad.abs().max()) > 0


def _bf(a):
    return torch.from_numpy(a).view(torch.bfloat16)


def test_moe_training_step_vs_reference():
    """One SwiFFN_MoE training step on rocm against the reference layer's own
    step (tests/golden/golden_train.npz, written by make_golden_train.py from
    model.py:506-585 with the reference's fp8_cpu.cpp forward and backward
    kernels).  Two steps accumulate _gw, as the reference's blockwise bf16 add
    does (kernel/fp8_tile.py:172-197).

    Routing and counts are exact.  The rest carries bf16 rounding points
    whose inputs differ from the reference's only by fp32 summation order, so
    an element can land one bf16 ulp away.  Bars: rel-L2 2e-3 for the output
    (the forward bar), x.grad, gate.weight.grad and every _gw; at most 1 % of
    the _gw elements differing at all, none by more than one bf16 ulp of the
    tensor's largest magnitude.  (Measured on MI355X: rel-L2 1e-4 to 2e-4,
    0.2 % of elements, 0.24 ulp.)"""
    import os
    import numpy as np
    print("case moe training step vs the reference's", flush=True)
    g = np.load(os.path.join(os.path.dirname(__file__), "golden", "golden_train.npz"))
    E, d = 4, 128
    cfg = MoEConfig(d_model=d, ffn_mult=2.5, tile=64, num_experts=E, num_experts_per_tok=2)
    moe = SwiFFN_MoE(cfg)
    with torch.no_grad():
        moe.gate.weight.copy_(torch.from_numpy(g["gate_w"]))
        for e, ex in enumerate(moe.experts):
            for n in ("gate", "up", "down"):
                getattr(ex, n).w8.copy_(torch.from_numpy(g[f"e{e}_{n}_w8"]))
                getattr(ex, n).sc.copy_(torch.from_numpy(g[f"e{e}_{n}_sc"]))
    moe = moe.to(DEV).train()
    x0 = _bf(g["x"]).to(DEV)
    c = torch.from_numpy(g["c"]).to(DEV)

    def rl2(a, b):
        a, b = a.double().cpu(), b.double().cpu()
        return float((a - b).norm() / b.norm().clamp_min(1e-300))
    for step in range(2):
        x = x0.clone().requires_grad_(True)
        y = moe(x)
        (y.float() * c).sum().backward()
        if step == 0:
            assert torch.equal(moe.last_topi.cpu(), torch.from_numpy(g["topi"]))
            assert moe.expert_token_counts == g["counts"].tolist()
            errs = {"out": rl2(y.float(), _bf(g["out"]).float()),
                    "x_grad": rl2(x.grad.float(), _bf(g["x_grad"]).float()),
                    "gate_grad": rl2(moe.gate.weight.grad, torch.from_numpy(g["gate_grad"]))}
    for e, ex in enumerate(moe.experts):
        for n in ("gate", "up", "down"):
            gw = getattr(ex, n)._gw
            assert (gw is not None) == bool(g[f"e{e}_{n}_gw_ran"]), (e, n)
            if gw is None:
                continue
            ref = _bf(g[f"e{e}_{n}_gw"]).float()
            got = gw.float().cpu()
            errs[f"e{e}_{n}_gw"] = rl2(got, ref)
            frac = float((got != ref).float().mean())
            # worst difference in bf16 ulps of the tensor's largest magnitude: an
            # element that cancels across the two steps can sit near zero, where
            # its own ulp says nothing about the rounding that moved it
            worst = float((got - ref).abs().max() / (ref.abs().max() * 2.0 ** -7))
            print(f"expert {e} {n}: _gw rel_l2 {errs[f'e{e}_{n}_gw']:.2e}, {frac:.2%} elements differ, "
                  f"worst {worst:.3f} ulp of max|_gw|", flush=True)
            assert frac <= 0.01 and worst <= 1.0, (e, n, frac, worst)
    print({k: f"{v:.2e}" for k, v in errs.items()}, flush=True)
    for k, v in errs.items():
        assert v <= 2e-3, (k, v)


@pytest.mark.parametrize("T,E,k,dtype", [(1, 4, 2, torch.float32), (70, 8, 3, torch.bfloat16),
                                         (257, 5, 1, torch.float32), (130, 2, 2, torch.float32)])
def test_training_dispatch_is_the_masked_loop(T, E, k, dtype):
    """The experts of a training step through the backend's dispatch against the
    loop over masks: outputs, counts and the gradients of x and of the routing
    weights, with slots of zero weight (no row) and an expert without a token.
    The same rows go through the same kernels, each token's k products added in
    the same order: fp32 rounding of k terms apart (k = 3, 2^-22)."""
    print(f"case training dispatch T={T} E={E} k={k} {dtype}", flush=True)
    torch.manual_seed(T + E)
    moe = SwiFFN_MoE(MoEConfig(d_model=128, ffn_mult=2.5, tile=64, num_experts=E, num_experts_per_tok=k)).to(DEV)
    moe.train()
    topi = torch.stack([torch.randperm(max(k, E - 1), device=DEV)[:k] for _ in range(T)])
    w0 = torch.rand(T, k, device=DEV)
    if T > 64:
        w0[::7, 0] = 0.0
    x0 = torch.randn(T, 128, device=DEV).to(dtype)
    c = torch.randn(T, 128, device=DEV)
    got = []
    for f in (moe._experts_by_mask, moe._experts_dispatched):
        for ex in moe.experts:
            for m in (ex.gate, ex.up, ex.down):
                m._gw = None
        x, w = x0.clone().requires_grad_(True), w0.clone().requires_grad_(True)
        out, counts = f(x, topi, w)
        (out * c).sum().backward()
        gws = [None if m._gw is None else m._gw.clone() for ex in moe.experts for m in (ex.gate, ex.up, ex.down)]
        got.append((out.detach(), x.grad, torch.where(w0 > 0, w.grad, torch.zeros_like(w0)), counts, gws))
    (o0, gx0, gw0, c0, g0), (o1, gx1, gw1, c1, g1) = got
    assert c0 == c1 and sum(c0) == int((w0 > 0).sum())
    bar = 2.0 ** -22 if dtype == torch.float32 else 2.0 ** -7   # x.grad is rounded to bf16 per term or once
    assert rel(o1, o0) <= 2.0 ** -22 and rel(gw1, gw0) < 1e-5 and rel(gx1, gx0) <= 4 * bar
    for a, b in zip(g0, g1):
        assert (a is None) == (b is None) and (a is None or torch.equal(a, b))


@pytest.mark.parametrize("shape,dtype", [((3, 5), torch.float32), ((257, 1280), torch.float32),
                                         ((64, 640), torch.bfloat16), ((0, 64), torch.float32)])
def test_swiglu_vs_float64(shape, dtype):
    """The training path's SwiGLU product and gradients against float64: a few
    fp32 roundings (2^-20 of the largest value), then the dtype's."""
    from smaulnative_amd.compute import get_backend
    print(f"case swiglu {shape} {dtype}", flush=True)
    torch.manual_seed(5)
    g, u, d = ((3 * torch.randn(shape, device=DEV)).to(dtype) for _ in range(3))
    be = get_backend("rocm")
    out = be.swiglu(g, u)
    dg, du = be.swiglu_backward(d, g, u)
    g64, u64 = g.double().requires_grad_(True), u.double().requires_grad_(True)
    ref = F.silu(g64) * u64
    ref.backward(d.double())
    step = 0.0 if dtype == torch.float32 else 2.0 ** -8
    for a, r in ((out, ref.detach()), (dg, g64.grad), (du, u64.grad)):
        assert a.dtype == dtype and a.shape == r.shape
        if a.numel():
            assert bool(((a.double() - r).abs() <= step * r.abs() + 2.0 ** -20 * r.abs().max()).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("spread", [1.0, 30.0])
def test_swiglu_is_as_near_float64_as_the_tensor_operations(dtype, spread):
    """Product and gradients no further from float64 than the operations they
    replace, F.silu(g.float()) * u.float() and autograd's (1 % for ties of the
    mean): large and small sigmoids, the underflow of both, infinities."""
    from smaulnative_amd.compute import get_backend
    print(f"case swiglu error {dtype} {spread}", flush=True)
    torch.manual_seed(6)
    g, u, d = ((s * torch.randn(1 << 18, device=DEV)).to(dtype) for s in (spread, 1.0, 1.0))
    g[:8] = torch.tensor([0.0, -0.0, 88.0, -88.0, -88.5, -104.0, float("inf"), -float("inf")], device=DEV).to(dtype)
    be = get_backend("rocm")
    got = (be.swiglu(g, u), *be.swiglu_backward(d, g, u))
    gf, uf = g.clone().requires_grad_(True), u.clone().requires_grad_(True)
    out = (F.silu(gf.float()) * uf.float()).to(dtype)
    out.backward(d)
    g64, u64 = g.double().requires_grad_(True), u.double().requires_grad_(True)
    exact = F.silu(g64) * u64
    exact.backward(d.double())
    # relative to each value, where it is a normal number of the arithmetic
    for a, b, x in zip(got, (out.detach(), gf.grad, uf.grad), (exact.detach(), g64.grad, u64.grad)):
        assert torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(torch.isinf(a), torch.isinf(b))
        ok = torch.isfinite(x) & (x.abs() > 1e-35)
        mine, theirs = (((t.double() - x) / x)[ok].square().mean().sqrt() for t in (a, b))
        print(f"  {float(mine):.4e} {float(theirs):.4e} bits differ {int((a != b).sum())}", flush=True)
        assert float(mine) <= 1.01 * float(theirs)
