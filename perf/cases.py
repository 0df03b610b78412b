"""The work a program has this framework do, as measurable cases.

Every case goes through a public entry point of ``smaulnative_amd`` (a module
or a backend method) on inputs of the distributions the path meets in use:
hidden states N(0, 1) (the layers read normalised activations), weights
N(0, 0.02) quantized to tiled E4M3, router weights N(0, 0.02), elu + 1
attention features.  ``kind`` selects the path:

- ``moe``: one inference pass of a mixture-of-experts layer;
- ``decode``: the MoE layers of one decode step, captured once as a HIP graph
  and replayed, as a serving loop does;
- ``swiffn``: one dense SwiGLU feed-forward layer;
- ``linear``: one tiled-FP8 projection;
- ``moe_train``: forward and backward of a MoE layer, with the experts' weight
  gradients;
- ``attn`` / ``attn_train`` / ``attn_step``: the linear-attention recurrence,
  as a prefill, as a training step and as one decode step;
- ``update``: one Lion step on a tiled-FP8 weight (decode, update, quantize).
"""
import torch
import torch.nn.functional as F

from smaulnative_amd import FP8Linear, MoEConfig, SwiFFN, SwiFFN_MoE
from smaulnative_amd.compute import get_backend
from smaulnative_amd.fp8_tile import quantize_tiles

DEV = "cuda"
EPS = 1e-6
LION = dict(lr=1e-4, wd=0.1, b1=0.9, b2=0.99)
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}


def listed():
    return [
        # one generated token of a single sequence through the layer of the small byte model
        # (d=512, 4 experts, top-2): launches and host latency are all there is
        dict(name="moe_token_f32", kind="moe", entry="module", T=1, d=512, h=1280, E=4, k=2, dtype="f32", tile=64,
             skew="none"),
        # a decode step of 64 sequences: eight MoE layers of a deep model, whose codes (535 MB) come from HBM
        dict(name="moe_decode_64_bf16", kind="decode", T=64, d=1024, h=2560, E=8, k=2, dtype="bf16", layers=8),
        # the small byte model's layer on its batch of 2 x 256 byte tokens
        dict(name="moe_batch_512_f32", kind="moe", entry="module", T=512, d=512, h=1280, E=4, k=2, dtype="f32",
             tile=64, skew="none"),
        # prefill of 16384 tokens, eight experts with a mild imbalance: the headline workload
        dict(name="moe_prefill_16k_bf16", kind="moe", entry="backend", T=16384, d=1024, h=2560, E=8, k=2,
             dtype="bf16", tile=64, skew="mild"),
        # the same layer on fp32 hidden states and a prompt of no round length
        dict(name="moe_prefill_odd_f32", kind="moe", entry="backend", T=10007, d=1024, h=2560, E=8, k=2,
             dtype="f32", tile=64, skew="mild"),
        # the largest: 16 experts, one of which takes about 40 % of the tokens and three of which take next to none
        dict(name="moe_skew_64k_bf16", kind="moe", entry="backend", T=65536, d=2048, h=5120, E=16, k=2,
             dtype="bf16", tile=64, skew="heavy"),
        # the dense feed-forward layer of a model without routing
        dict(name="swiffn_4096_f32", kind="swiffn", rows=4096, d=512, h=1280, dtype="f32", tile=64),
        # a projection whose widths divide by nothing, with the finer scale tiles
        dict(name="linear_odd_f32", kind="linear", rows=3001, i=1000, o=777, dtype="f32", tile=32),
        # a training step of the MoE layer: 8 x 256 tokens, forward, backward, weight gradients
        dict(name="moe_train_2048_f32", kind="moe_train", T=2048, d=512, h=1280, E=4, k=2, dtype="f32", tile=64),
        # the attention of a prefill that goes on to decode: outputs and final state
        dict(name="attn_prefill_256", kind="attn", B=2, T=256, H=8, D=64),
        # the attention of the training step's batch: forward and backward
        dict(name="attn_train_256", kind="attn_train", B=8, T=256, H=8, D=64),
        # the optimizer's step on one expert matrix
        dict(name="lion_update_2560x1024", kind="update", o=2560, i=1024, tile=64),
    ]


def _log(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm; every second one is odd."""
    n = int(round(lo * (hi / lo) ** rng.random()))
    return max(lo, min(hi, n | 1 if rng.random() < 0.5 else n))


def draw(rng):
    kind = rng.choice(["moe", "moe", "moe", "moe", "decode", "swiffn", "linear", "linear", "moe_train", "attn",
                       "attn_train", "attn_step", "update"])
    dtype = rng.choice(["f32", "bf16"])
    if kind == "moe":
        d, h = rng.choice([(256, 640), (512, 1280), (768, 1920), (1024, 2560), (2048, 5120)])
        E = rng.choice([2, 4, 8, 16])
        most = {256: 65536, 512: 65536, 768: 32768, 1024: 16384, 2048: 8192}[d]
        # other scale tiles than 64 are an option of smaller layers
        tile = rng.choice([64, 64, 64, 64, 32, 128]) if d <= 512 else 64
        if tile != 64:
            most //= 8
        return dict(kind="moe", entry="backend", T=_log(rng, 1, most), d=d, h=h, E=E,
                    k=rng.choice([1, 2, 2, 3]) if E > 2 else 2, dtype=dtype, tile=tile,
                    skew=rng.choice(["none", "mild", "heavy"] if E >= 8 else ["none", "mild"]))
    if kind == "decode":
        return dict(kind="decode", T=_log(rng, 1, 64), d=1024, h=2560, E=8, k=rng.choice([1, 2]), dtype=dtype,
                    layers=rng.randint(4, 8))
    if kind == "swiffn":
        d, h = rng.choice([(256, 640), (512, 1280), (1024, 2560)])
        return dict(kind="swiffn", rows=_log(rng, 1, 16384), d=d, h=h, dtype=dtype, tile=64)
    if kind == "linear":
        tile = rng.choice([32, 64, 64, 64, 128])
        if rng.random() < 0.5:
            i, o = 64 * rng.randint(2, 40), 64 * rng.randint(2, 40)
        else:
            i, o = _log(rng, 100, 2000), _log(rng, 100, 2000)
        return dict(kind="linear", rows=_log(rng, 1, 16384), i=i, o=o, dtype=dtype, tile=tile)
    if kind == "moe_train":
        d, h = rng.choice([(256, 640), (512, 1280)])
        return dict(kind="moe_train", T=_log(rng, 128, 4096), d=d, h=h, E=rng.choice([2, 4, 8]), k=2,
                    dtype=dtype, tile=64)
    if kind in ("attn", "attn_train"):
        return dict(kind=kind, B=rng.randint(1, 8), T=_log(rng, 16, 512), H=rng.choice([4, 8, 16]),
                    D=rng.choice([32, 48, 64, 64, 128]))
    if kind == "attn_step":
        return dict(kind="attn_step", B=_log(rng, 1, 64), T=1, H=rng.choice([4, 8, 16]),
                    D=rng.choice([32, 64, 64, 128]))
    return dict(kind="update", o=_log(rng, 200, 4000), i=_log(rng, 200, 4000), tile=rng.choice([32, 64, 64, 128]))


# ---- inputs -----------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _n(gen, *shape, std=1.0):
    return torch.randn(*shape, generator=gen, device=DEV) * std


def _matrix(gen, o, i, tile):
    return quantize_tiles(_n(gen, o, i, std=0.02), tile)


def _expert(gen, d, h, tile):
    return _matrix(gen, h, d, tile) + _matrix(gen, h, d, tile) + _matrix(gen, d, h, tile)


def _moe_inputs(case, seed):
    """(x, router weight, router bias or None, experts) of a layer, from the seed alone."""
    gen = _gen(seed)
    T, d, h, E = case["T"], case["d"], case["h"], case["E"]
    x = _n(gen, T, d).to(DTYPES[case["dtype"]])
    gw = _n(gen, E, d, std=0.02)
    gb = None
    skew = case.get("skew", "mild")
    if skew == "mild":
        gb = _n(gen, E, std=0.5)
    elif skew == "heavy":  # one popular expert, three that hardly a token takes (logits have a spread of 0.02 sqrt(d))
        gb = torch.zeros(E, device=DEV)
        spread = 0.02 * d ** 0.5
        gb[0] = 2.2 * spread
        gb[E - 3:] = -2.5 * spread
    return x, gw, gb, [_expert(gen, d, h, case.get("tile", 64)) for _ in range(E)]


def _fill(linear, pair):
    linear.w8.copy_(pair[0])
    linear.sc.copy_(pair[1])


def _module(cls, case, experts, gw=None):
    d, h = case["d"], case["h"]
    E = case.get("E", 1)
    cfg = MoEConfig(d_model=d, ffn_mult=h / d, tile=case["tile"], num_experts=E, num_experts_per_tok=case.get("k", 1))
    with torch.device(DEV), torch.no_grad():
        m = cls(cfg)
        for ex, bufs in zip(m.experts if gw is not None else [m], experts):
            for n, lin in enumerate((ex.gate, ex.up, ex.down)):
                _fill(lin, bufs[2 * n:2 * n + 2])
        if gw is not None:
            m.gate.weight.copy_(gw)
    return m


def _attn_inputs(case, seed):
    gen = _gen(seed)
    shape = (case["B"], case["T"], case["H"], case["D"])
    q = F.elu(_n(gen, *shape, std=0.45)) + 1.0
    k = F.elu(_n(gen, *shape, std=0.45)) + 1.0
    return q, k, _n(gen, *shape, std=0.45), _n(gen, *shape)


def _update_inputs(case, seed):
    gen = _gen(seed)
    o, i = case["o"], case["i"]
    w8, sc = _matrix(gen, o, i, case["tile"])
    return w8, sc, _n(gen, o, i, std=1e-3).to(torch.bfloat16), _n(gen, o, i, std=1e-3)


def prepare(case, seed):
    kind, dt = case["kind"], DTYPES[case.get("dtype", "f32")]
    st = {"case": case, "be": get_backend()}
    if kind == "moe":
        x, gw, gb, experts = _moe_inputs(case, seed)
        if case["entry"] == "module":
            st.update(x=x, layer=_module(SwiFFN_MoE, case, experts, gw).eval())
        else:
            st.update(x=x, gw=gw, gb=gb, experts=experts)
    elif kind == "decode":
        layers = [_moe_inputs(case, seed * 64 + n) for n in range(case["layers"])]
        be = st["be"]

        def step():
            return [be.moe_forward(x, gw, gb, ex, case["k"], 64)[:3] for x, gw, gb, ex in layers]

        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            step()
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            outs = step()
        st.update(layers=layers, graph=graph, outs=outs)
    elif kind == "swiffn":
        gen = _gen(seed)
        x = _n(gen, case["rows"], case["d"]).to(dt)
        st.update(x=x, layer=_module(SwiFFN, case, [_expert(gen, case["d"], case["h"], case["tile"])]).eval())
    elif kind == "linear":
        gen = _gen(seed)
        st["x"] = _n(gen, case["rows"], case["i"]).to(dt)
        with torch.device(DEV), torch.no_grad():
            st["layer"] = FP8Linear(case["i"], case["o"], case["tile"]).eval()
            _fill(st["layer"], _matrix(gen, case["o"], case["i"], case["tile"]))
    elif kind == "moe_train":
        x, gw, _, experts = _moe_inputs(case, seed)
        st.update(x=x.requires_grad_(True), layer=_module(SwiFFN_MoE, case, experts, gw).train(),
                  dout=_n(_gen(seed + 1), case["T"], case["d"]).to(dt))
    elif kind in ("attn", "attn_train"):
        st["qkv"] = _attn_inputs(case, seed)
    elif kind == "attn_step":
        q, k, v, _ = _attn_inputs(case, seed)
        # the state of a sequence of some hundred tokens; it is advanced in place by every pass
        S, z = _step_state(case, seed)
        st.update(q=q[:, 0].contiguous(), k=k[:, 0].contiguous(), v=v[:, 0].contiguous(), S=S, z=z)
    else:
        w8, sc, g, m = _update_inputs(case, seed)
        with torch.device(DEV), torch.no_grad():
            lin = FP8Linear(case["i"], case["o"], case["tile"])
            _fill(lin, (w8, sc))
        st.update(layer=lin, gw=g, momentum=m)
    return st


def _step_state(case, seed):
    B, H, D = case["B"], case["H"], case["D"]
    gen = _gen(seed + 2)
    z = 10.0 + 0.5 * _n(gen, B, H, D).abs()
    return _n(gen, B, H, D, D), z


# ---- one pass ---------------------------------------------------------------


def run(st):
    case, be = st["case"], st["be"]
    kind = case["kind"]
    if kind == "moe":
        if case["entry"] == "module":
            with torch.no_grad():
                out = st["layer"](st["x"])
            return out, st["layer"].last_prob, st["layer"].last_topi
        return be.moe_forward(st["x"], st["gw"], st["gb"], st["experts"], case["k"], case["tile"])[:3]
    if kind == "decode":
        st["graph"].replay()
        return st["outs"]
    if kind in ("swiffn", "linear"):
        with torch.no_grad():
            return st["layer"](st["x"])
    if kind == "moe_train":
        x, layer = st["x"], st["layer"]
        x.grad = layer.gate.weight.grad = None  # as after an optimizer step
        linears = [m for ex in layer.experts for m in (ex.gate, ex.up, ex.down)]
        for m in linears:
            m._gw = None
        out = layer(x)
        out.backward(st["dout"])
        # an expert that no token took has no gradient
        return [out.detach(), x.grad, layer.gate.weight.grad] + [m._gw for m in linears]
    if kind == "attn":
        q, k, v, _ = st["qkv"]
        y, _, S, z = be.attn_forward(q, k, v, EPS, False, need_state=True)
        return y, S, z
    if kind == "attn_train":
        q, k, v, dy = st["qkv"]
        y, den, _, _ = be.attn_forward(q, k, v, EPS, True)
        return (y, den) + tuple(be.attn_backward(dy, q, k, v, y, den, EPS))
    if kind == "attn_step":
        return be.attn_step(st["S"], st["z"], st["q"], st["k"], st["v"], EPS)
    st["layer"].fused_lion_requant(st["gw"], st["momentum"], **LION)
    return st["layer"].w8, st["layer"].sc, st["momentum"]


# ---- what a pass cannot do without ------------------------------------------


def _weights(n_out, n_in, tile):
    return n_out * n_in + 4 * n_out * -(-n_in // tile)


def work(case):
    kind = case["kind"]
    size = 2 if case.get("dtype") == "bf16" else 4
    if kind in ("moe", "decode", "moe_train"):
        T, d, h, E, k, tile = case["T"], case["d"], case["h"], case["E"], case["k"], case.get("tile", 64)
        # experts a batch of T tokens reaches (all of them but for the smallest batches)
        hit = min(E, T * k) if T > 8 else E * (1 - (1 - k / E) ** T)
        expert = 2 * _weights(h, d, tile) + _weights(d, h, tile)
        io = 2 * T * d * size + T * E * 4 + T * k * 8 + E * d * 4
        byts, flops = io + hit * expert, 6.0 * T * k * d * h + 2.0 * T * d * E
        if kind == "moe_train":  # the output gradient in, the input's, the router's and the weights' out
            byts += 2 * T * d * size + E * d * 4 + hit * (3 * d * h * 2)
            flops *= 3
        n = case.get("layers", 1)
        return {"bytes": float(n * byts), "flops": float(n * flops)}
    if kind == "swiffn":
        rows, d, h, tile = case["rows"], case["d"], case["h"], case["tile"]
        return {"bytes": float(2 * rows * d * size + 2 * _weights(h, d, tile) + _weights(d, h, tile)),
                "flops": 6.0 * rows * d * h}
    if kind == "linear":
        rows, i, o = case["rows"], case["i"], case["o"]
        return {"bytes": float(rows * (i + o) * size + _weights(o, i, case["tile"])), "flops": 2.0 * rows * i * o}
    if kind in ("attn", "attn_train", "attn_step"):
        B, T, H, D = case["B"], case["T"], case["H"], case["D"]
        n, state = B * T * H * D, B * H * D * (D + 1)
        if kind == "attn":  # per step: S += kn (x) v, q . S, z, q . z
            return {"bytes": 4.0 * (4 * n + state), "flops": 4.0 * n * (D + 1)}
        if kind == "attn_step":
            return {"bytes": 4.0 * (4 * n + 2 * state), "flops": 4.0 * n * (D + 1)}
        # q, k, v, dy in; y, den, dq, dk, dv out; the forward, S again with dq, and the adjoint with dk and dv
        return {"bytes": 4.0 * (8 * n + B * T * H), "flops": 4.0 * n * (D + 1) + 4.0 * n * D + 6.0 * n * D}
    o, i, tile = case["o"], case["i"], case["tile"]
    return {"bytes": float(2 * _weights(o, i, tile) + o * i * (2 + 8)), "flops": 10.0 * o * i}


def tolerance(case):
    kind = case["kind"]
    if kind == "update" or kind.startswith("attn"):
        # the codes, and the recurrence's order of sums, are what these entries promise bit for bit
        return "exact"
    if kind == "moe_train":
        # the weight gradients are stored in bf16
        return {"rel": 1e-2}
    if case["dtype"] == "bf16":
        # two equally good sums round to neighbouring bf16 values; prob is fp32, a near tie may go either way
        return {"rel": 1e-2, "max": 0.9, "differ": 1e-3} if kind in ("moe", "decode") else {"rel": 1e-2}
    # fp32 sums over two bf16 terms of x: measured 4e-6 against 64 bits
    return {"rel": 2e-5, "max": 0.9, "differ": 1e-3} if kind in ("moe", "decode") else {"rel": 2e-5}


# ---- the same in 64 bits ----------------------------------------------------


def _decode64(w8, sc, tile):
    """lut[code] * scale of E4M3 codes without infinities or NaN (0x7F / 0xFF are +-448), in float64."""
    c = torch.arange(256, device=w8.device)
    e, m = (c >> 3) & 15, (c & 7).double()
    lut = torch.where(e == 0, m / 512.0, (1.0 + m / 8.0) * torch.exp2(e.double() - 7.0))
    lut = torch.where((c & 127) == 127, torch.full_like(lut, 448.0), lut)
    lut = torch.where(c >= 128, -lut, lut)
    return lut[w8.long()] * sc.double().repeat_interleave(tile, 1)[:, :w8.shape[1]]


def _route64(x, gw, gb, k):
    logits = x @ gw.double().t()
    if gb is not None:
        logits = logits + gb.double()
    prob = torch.softmax(logits, -1)
    val, idx = torch.topk(prob, k, -1)
    return prob, idx, val / val.sum(-1, keepdim=True)


def _swiglu64(x, ws, rows=8192):
    parts = []
    for n in range(0, x.shape[0], rows):
        c = x[n:n + rows]
        parts.append((F.silu(c @ ws[0].t()) * (c @ ws[1].t())) @ ws[2].t())
    return torch.cat(parts) if parts else x.new_zeros(0, ws[2].shape[0])


def _moe64(x, gw, gb, experts, k, tile):
    x = x.double()
    prob, idx, wt = _route64(x, gw, gb, k)
    out = torch.zeros_like(x)
    for e, bufs in enumerate(experts):
        sel = torch.where(idx == e, wt, torch.zeros_like(wt)).sum(-1)
        rows = torch.nonzero(sel > 0).squeeze(-1)
        ws = [_decode64(bufs[2 * n], bufs[2 * n + 1], tile) for n in range(3)]
        out.index_add_(0, rows, _swiglu64(x[rows], ws) * sel[rows].unsqueeze(-1))
    return out, prob, None


def _moe_train64(case, seed):
    x, gw, _, experts = _moe_inputs(case, seed)
    x = x.double().requires_grad_(True)
    gw = gw.double().requires_grad_(True)
    ws = [[_decode64(b[2 * n], b[2 * n + 1], case["tile"]).requires_grad_(True) for n in range(3)] for b in experts]
    _, idx, wt = _route64(x, gw, None, case["k"])
    out = torch.zeros_like(x)
    for e in range(case["E"]):
        sel = torch.where(idx == e, wt, torch.zeros_like(wt)).sum(-1)
        rows = torch.nonzero((idx == e).any(-1)).squeeze(-1)
        if rows.numel():
            out = out.index_add(0, rows, _swiglu64(x[rows], ws[e]) * sel[rows].unsqueeze(-1))
    out.backward(_n(_gen(seed + 1), case["T"], case["d"]).to(DTYPES[case["dtype"]]).double())
    return [out.detach(), x.grad, gw.grad] + [w.grad for e in ws for w in e]


def _attn64(q, k, v):
    """(y, den, S, z) of the recurrence, from the causal products of all steps at once."""
    q, k, v = (t.double().transpose(1, 2) for t in (q, k, v))  # [B, H, T, D]
    kn = k / k.norm(dim=-1, keepdim=True).clamp_min(1e-6)
    a = torch.matmul(q, kn.transpose(-1, -2).contiguous()).tril()
    den = a.sum(-1).clamp_min(EPS)
    y = torch.matmul(a, v) / den.unsqueeze(-1)
    S = torch.matmul(kn.transpose(-1, -2).contiguous(), v)
    return y.transpose(1, 2), den.transpose(1, 2), S, kn.sum(2)


def exact(case, seed):
    kind = case["kind"]
    if kind == "moe":
        return _moe64(*_moe_inputs(case, seed), case["k"], case["tile"])
    if kind == "decode":
        return [_moe64(*_moe_inputs(case, seed * 64 + n), case["k"], 64) for n in range(case["layers"])]
    if kind == "swiffn":
        gen = _gen(seed)
        x = _n(gen, case["rows"], case["d"]).to(DTYPES[case["dtype"]])
        b = _expert(gen, case["d"], case["h"], case["tile"])
        return _swiglu64(x.double(), [_decode64(b[2 * n], b[2 * n + 1], case["tile"]) for n in range(3)])
    if kind == "linear":
        gen = _gen(seed)
        x = _n(gen, case["rows"], case["i"]).to(DTYPES[case["dtype"]])
        return x.double() @ _decode64(*_matrix(gen, case["o"], case["i"], case["tile"]), case["tile"]).t()
    if kind == "moe_train":
        return _moe_train64(case, seed)
    if kind == "attn":
        y, _, S, z = _attn64(*_attn_inputs(case, seed)[:3])
        return y, S, z
    if kind == "attn_train":
        q, k, v, dy = _attn_inputs(case, seed)
        q, k, v = (t.double().requires_grad_(True) for t in (q, k, v))
        y, den, _, _ = _attn64(q, k, v)
        y.backward(dy.double())
        return y.detach(), den.detach(), q.grad, k.grad, v.grad
    if kind == "attn_step":
        q, k, v, _ = (t[:, 0].double() for t in _attn_inputs(case, seed))
        S, z = (t.double() for t in _step_state(case, seed))
        kn = k / k.norm(dim=-1, keepdim=True).clamp_min(1e-6)
        S = S + kn.unsqueeze(-1) * v.unsqueeze(-2)
        z = z + kn
        den = (q * z).sum(-1, keepdim=True).clamp_min(EPS)
        return (q.unsqueeze(-1) * S).sum(-2) / den, S, z
    # the codes and their scales depend on which of two neighbours a value rounds to
    _, _, g, m = _update_inputs(case, seed)
    return None, None, m.double() * LION["b2"] + g.double() * (1.0 - LION["b2"])
