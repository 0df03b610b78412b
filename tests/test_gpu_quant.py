"""GPU parity of the tiled-E4M3 quantizer (the backend's fp8_quantize_tiles).

Bar: codes, scales and the non-finite count bit-identical to the reference
quantizer -- its golden vectors (the 12 special-value cases of
tests/test_linear_fp8.py:484-510 x tiles 32/64/128, written from the
reference by tests/golden/make_golden.py) and the oracle's torch path
(kernel/fp8_tile.py:100-113), which the CPU tests pin to those vectors.
"""
import os
import warnings

import numpy as np
import pytest
import torch

import oracle
from smaulnative_amd.compute import get_backend
from smaulnative_amd.fp8_tile import decode_tile, quantize_tiles

pytestmark = pytest.mark.gpu

DEV = "cuda"
GOLD = os.path.join(os.path.dirname(__file__), "golden", "golden_fp8_moe.npz")
QCASES = ["uniform", "tiny", "huge", "zeros", "half_zero", "codebook", "midpoints", "saturating",
          "subnormal", "odd_shape", "padded_tile", "nonfinite"]


@pytest.mark.parametrize("tile", [32, 64, 128])
def test_device_quantizer_golden(tile):
    g = np.load(GOLD)
    be = get_backend("rocm")
    for name in QCASES:
        w = torch.from_numpy(np.array(g[f"q_{name}_w"]))
        print(f"case quant {name} {tuple(w.shape)} tile={tile}", flush=True)
        codes, sc, bad = be.fp8_quantize_tiles(w.to(DEV), tile)
        in_f = w.shape[1]
        assert codes.shape[1] == -(-in_f // tile) * tile
        assert bool((codes[:, in_f:] == 0).all())                     # the padding of the last tile
        assert np.array_equal(codes[:, :in_f].cpu().numpy(), g[f"q_{name}_t{tile}_codes"])
        assert np.array_equal(sc.cpu().numpy().view(np.uint32), g[f"q_{name}_t{tile}_sc"].view(np.uint32))
        assert bad == int((~torch.isfinite(w)).sum())


@pytest.mark.parametrize("out_f,in_f,tile", [(2560, 1024, 64), (77, 333, 32), (64, 200, 48), (33, 1000, 100),
                                             (16, 640, 128), (9, 70, 1), (40, 96, 8), (5, 300, 256)])
def test_device_quantizer_vs_oracle(out_f, in_f, tile):
    print(f"case quant random {out_f}x{in_f} tile={tile}", flush=True)
    gen = torch.Generator().manual_seed(out_f * 31 + in_f + tile)
    w = torch.randn(out_f, in_f, generator=gen) * 0.02
    w[torch.rand(out_f, in_f, generator=gen) < 0.01] = 0.0
    ref_c, ref_s = oracle.quantize_tiles(w, tile)
    c, s = quantize_tiles(w.to(DEV), tile)          # the product entry, device path
    assert c.is_cuda and c.dtype == torch.uint8 and tuple(c.shape) == (out_f, in_f)
    assert torch.equal(c.cpu(), ref_c)
    assert torch.equal(s.cpu(), ref_s)
    # decoding on the device gives the oracle's values
    t = min(1, s.shape[1] - 1)
    assert torch.equal(decode_tile(c, s, 0, out_f, t, tile).cpu(), oracle.decode_tile(ref_c, ref_s, 0, out_f, t, tile))


def test_device_quantizer_warns_on_nonfinite():
    w = torch.randn(8, 64)
    w[0, 0], w[1, 1] = float("nan"), float("inf")
    with warnings.catch_warnings(record=True) as rec:
        warnings.simplefilter("always")
        c, s = quantize_tiles(w.to(DEV), 64)
    assert any("2 non-finite" in str(r.message) for r in rec)
    ref_c, ref_s = oracle.quantize_tiles(w, 64)
    assert torch.equal(c.cpu(), ref_c) and torch.equal(s.cpu(), ref_s)


@pytest.mark.parametrize("out_f,in_f,tile,gdtype", [
    # the four-weights-a-lane kernel (4 to 256 wide tiles, ragged last ones), the
    # scalar ones (widths and tiles it does not take)
    (70, 1024, 64, torch.bfloat16), (33, 100, 32, torch.float32), (5, 4, 4, torch.bfloat16),
    (9, 516, 256, torch.float32), (33, 333, 32, torch.bfloat16), (17, 200, 48, torch.bfloat16),
    (3, 1500, 512, torch.float32), (40, 90, 2, torch.float32)])
def test_device_requant_is_the_tensor_operations(out_f, in_f, tile, gdtype):
    """requant and the Lion step in one pass against the tensor operations they
    replace (decode_block, in-place arithmetic, quantize_tiles): codes, scales
    and momentum bit for bit, non-finite weights and every code included."""
    from smaulnative_amd.fp8_tile import FP8Linear, decode_block
    print(f"case requant {out_f}x{in_f} tile={tile} {gdtype}", flush=True)
    gen = torch.Generator().manual_seed(out_f * 13 + in_f + tile)
    w8 = torch.randint(0, 256, (out_f, in_f), generator=gen, dtype=torch.int64).to(torch.uint8).to(DEV)
    sc = (torch.rand(out_f, -(-in_f // tile), generator=gen) * 0.01 + 1e-4).to(DEV)
    upd = (torch.randn(out_f, in_f, generator=gen) * 0.1).to(DEV)
    upd[0, 0], upd[-1, -1] = float("nan"), float("inf")
    g = (torch.randn(out_f, in_f, generator=gen) * 1e-3).to(gdtype).to(DEV)
    m = (torch.randn(out_f, in_f, generator=gen) * 1e-3).to(DEV)
    m[0, :2] = 0.0
    g[0, :2] = 0.0   # a zero step
    lr, wd, b1, b2 = 1e-2, 0.1, 0.9, 0.99

    def module():
        lin = FP8Linear(in_f, out_f, tile).to(DEV)
        lin.w8.copy_(w8)
        lin.sc.copy_(sc)
        return lin

    for update, decay in ((upd, 0.0), (upd, 0.03), (None, 0.03), (None, 0.0)):
        w = decode_block(w8, sc, 0, out_f, in_f, tile)
        if decay:
            w.mul_(1 - decay)
        if update is not None:
            w.sub_(update)
        with warnings.catch_warnings(record=True) as rec:
            warnings.simplefilter("always")
            rc, rs = quantize_tiles(w, tile)
            lin = module()
            version = lin.w8._version
            lin.requant(update, decay)
        assert len(rec) == (0 if update is None else 2) and len({str(r.message) for r in rec}) <= 1
        assert lin.w8._version > version   # what caches made from the codes go by
        assert torch.equal(lin.w8, rc) and torch.equal(lin.sc, rs)
    st, ref = m.clone(), m.clone()
    lin = module()
    lin.fused_lion_requant(g, st, lr, wd, b1, b2)
    step = (ref * b1 + g.float() * (1.0 - b1)).sign() * lr
    ref.mul_(b2).add_(g.float(), alpha=1.0 - b2)
    rc, rs = quantize_tiles(decode_block(w8, sc, 0, out_f, in_f, tile).mul_(1 - lr * wd).sub_(step), tile)
    assert torch.equal(st, ref) and torch.equal(lin.w8, rc) and torch.equal(lin.sc, rs)
