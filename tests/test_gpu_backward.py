"""GPU parity of the tiled-FP8 linear's backward (training; not on the forward path).

fp8_backward_input (kernel/compute.py:145-153) against the oracle's
restatement of kernel/fp8_cpu.cpp:167-259, which the CPU tests pin bit-exact
to the reference's own kernel.  Bar: max relative difference 1e-5 -- the
GPU sums the output dimension in another fp32 order (the reference's own
test holds its kernel to 1e-5 against autograd, test_linear_fp8.py:186-199).
The module test runs FP8Linear forward + backward in training mode: the
input gradient, and the weight gradient accumulated in bf16 ``_gw``
(kernel/fp8_tile.py:172-197) by the backend's kernel or in 64-row blocks.
"""
import pytest
import torch

import oracle
from smaulnative_amd.compute import get_backend

pytestmark = pytest.mark.gpu
DEV = "cuda"


def rel_max(a, b):
    a, b = a.detach().double().cpu(), b.detach().double().cpu()
    return float((a - b).abs().max() / b.abs().max().clamp_min(1e-300))


@pytest.mark.parametrize("rows,in_f,out_f,tile", [(64, 128, 128, 64), (33, 70, 100, 64), (4096, 512, 1280, 64),
                                                  (50, 300, 130, 32), (17, 96, 200, 128), (1, 1024, 64, 64),
                                                  (0, 64, 64, 64)])
def test_backward_input_vs_oracle(rows, in_f, out_f, tile):
    print(f"case backward rows={rows} in_f={in_f} out_f={out_f} tile={tile}", flush=True)
    gen = torch.Generator().manual_seed(rows * 3 + in_f + out_f)
    g = torch.randn(rows, out_f, generator=gen)
    w, s = oracle.quantize_tiles(torch.randn(out_f, in_f, generator=gen) * 0.05, tile)
    dx = get_backend("rocm").fp8_backward_input(g.to(DEV), w.to(DEV), s.to(DEV), in_f, out_f, tile)
    assert dx.dtype == torch.float32 and tuple(dx.shape) == (rows, in_f)
    if rows == 0:
        return
    ref = oracle.fp8_backward_input(g, w, s, in_f, out_f, tile)
    assert rel_max(dx, ref) < 1e-5, rel_max(dx, ref)


@pytest.mark.parametrize("rows,in_f,out_f", [
    # 32-row tiles and chunks of 128 (few tiles): a row tile's edge, ragged both;
    # out_f a multiple of 64 but not of 128, and many tiles, are 64-row ones
    (1, 64, 128), (33, 128, 640), (95, 192, 320), (40, 100, 130), (2100, 2048, 128)])
def test_backward_input_row_tiles(rows, in_f, out_f):
    print(f"case backward tiles rows={rows} in_f={in_f} out_f={out_f}", flush=True)
    gen = torch.Generator().manual_seed(rows + in_f + out_f)
    g = torch.randn(rows, out_f, generator=gen)
    w, s = oracle.quantize_tiles(torch.randn(out_f, in_f, generator=gen) * 0.05, 64)
    dx = get_backend("rocm").fp8_backward_input(g.to(DEV), w.to(DEV), s.to(DEV), in_f, out_f, 64)
    assert rel_max(dx, oracle.fp8_backward_input(g, w, s, in_f, out_f, 64)) < 1e-5


@pytest.mark.parametrize("rows,in_f,out_f", [
    # either side of the lines between 32- and 64-row tiles on 256 CUs: guarded
    # loads at 128 / 132 tiles and at one chunk of 64 or more, vectors at 511 / 512
    (2000, 200, 300), (2050, 200, 300), (70, 512, 64 - 3), (70, 512, 64 + 3), (4640, 448, 128), (4090, 512, 256)])
def test_backward_input_tile_rule(rows, in_f, out_f):
    print(f"case backward rule rows={rows} in_f={in_f} out_f={out_f}", flush=True)
    gen = torch.Generator().manual_seed(rows + in_f + out_f)
    g = torch.randn(rows, out_f, generator=gen)
    w, s = oracle.quantize_tiles(torch.randn(out_f, in_f, generator=gen) * 0.05, 64)
    dx = get_backend("rocm").fp8_backward_input(g.to(DEV), w.to(DEV), s.to(DEV), in_f, out_f, 64)
    assert rel_max(dx, oracle.fp8_backward_input(g, w, s, in_f, out_f, 64)) < 1e-5


@pytest.mark.parametrize("rows,in_f,out_f,dtype", [
    # rows about the kernel's chunks of 16 (four waves take every fourth) and
    # outputs about its 64 x 64 tiles
    (1, 64, 64, torch.float32), (15, 65, 63, torch.float32), (64, 1, 129, torch.bfloat16),
    (129, 192, 100, torch.float32), (1000, 512, 320, torch.bfloat16), (0, 40, 24, torch.float32),
    (70, 700, 800, torch.float32)])  # over 128 of them: 64 x 64 tiles, else 32 x 32
def test_weight_grad_vs_float64(rows, in_f, out_f, dtype):
    """gw += g^T x in fp32, one rounding to bf16: against the float64 sum the
    fp32 sum is within rows * 2^-24 * sum |g||x| (any order), and the rounding
    within half a bf16 step: 8 significant bits, so 2^-8 of the result at most."""
    print(f"case weight grad rows={rows} in_f={in_f} out_f={out_f} {dtype}", flush=True)
    gen = torch.Generator().manual_seed(rows + in_f + out_f)
    g = torch.randn(rows, out_f, generator=gen)
    x = torch.randn(rows, in_f, generator=gen).to(dtype)
    gw = torch.randn(out_f, in_f, generator=gen).to(torch.bfloat16)
    be = get_backend("rocm")
    for fresh in (False, True):
        got = gw.to(DEV)
        be.fp8_weight_grad(g.to(DEV), x.to(DEV), got, fresh)
        start = torch.zeros_like(gw) if fresh else gw
        ref = start.double() + g.double().t() @ x.double()
        slack = (rows + 1) * 2.0 ** -24 * (g.double().abs().t() @ x.double().abs() + start.double().abs())
        bound = slack + (ref.abs() + slack) * 2.0 ** -8
        assert bool(((got.cpu().double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_fp8linear_training_step(dtype):
    from smaulnative_amd import FP8Linear
    torch.manual_seed(3)
    m = FP8Linear(192, 130, 64).to(DEV).train()
    x = torch.randn(2, 40, 192, device=DEV).to(dtype).requires_grad_(True)
    c = torch.randn(2, 40, 130, device=DEV)
    for step in range(2):  # the weight gradient accumulates across backward calls
        y = m(x)
        assert y.dtype == dtype
        (y.float() * c).sum().backward()
    # the module's output is in x's dtype, so the gradient reaching its backward
    # is c rounded to that dtype
    g = c.reshape(-1, 130).to(dtype).float().cpu()
    w, s = m.w8.cpu(), m.sc.cpu()
    gx = oracle.fp8_backward_input(g, w, s, 192, 130, 64).reshape(2, 40, 192)
    # two steps add the same gradient twice
    assert rel_max(x.grad.float(), (2 * gx).to(dtype).float()) < (1e-5 if dtype == torch.float32 else 8e-3)
    # _gw: per 64-row block, g^T x formed in fp32 and added to the bf16 buffer (rounded once per add)
    xr = x.detach().reshape(-1, 192).float().cpu()
    gw = torch.zeros(130, 192, dtype=torch.bfloat16)
    for _ in range(2):
        for o0 in range(0, 130, 64):
            gw[o0:o0 + 64].add_(g[:, o0:o0 + 64].t() @ xr)
    assert m._gw.dtype == torch.bfloat16 and tuple(m._gw.shape) == (130, 192)
    # the fp32 products are summed in another order on the device: a bf16
    # rounding may flip, and where the sum cancels the fp32 error bound (a few
    # units of 2^-24 of the sum of |terms|) can exceed one bf16 ulp of the result
    diff = (m._gw.cpu().float() - gw.float()).abs()
    ulp = gw.float().abs() * 2.0 ** -7
    terms = 2 * (g.abs().t() @ xr.abs())
    assert bool((diff <= 2 * ulp + terms * 2.0 ** -18).all())


@pytest.mark.parametrize("tile", [64, 128])
def test_backward_input_raw_codes(tile):
    """Every one of the 256 codes as stored (0x7F / 0xFF decode to +-448, NaN
    in OCP E4M3), scales spanning 2^-20..2^4, and a gradient with a wide
    dynamic range: the matrix-core form (tile a multiple of 64) splits g * s
    into three bf16 terms exactly and decodes the codes exactly."""
    rows, in_f, out_f = 200, 320, 512
    gen = torch.Generator().manual_seed(tile)
    w = torch.randint(0, 256, (out_f, in_f), generator=gen, dtype=torch.uint8)
    nt = (in_f + tile - 1) // tile
    s = torch.exp2(torch.randint(-20, 5, (out_f, nt), generator=gen).float()) * (1 + torch.rand(out_f, nt, generator=gen))
    g = torch.randn(rows, out_f, generator=gen) * torch.exp2(torch.randint(-30, 30, (rows, 1), generator=gen).float())
    dx = get_backend("rocm").fp8_backward_input(g.to(DEV), w.to(DEV), s.to(DEV), in_f, out_f, tile)
    ref = oracle.fp8_backward_input(g, w, s, in_f, out_f, tile)
    # per row: the rows differ by up to 2^60 in scale
    err = ((dx.cpu().double() - ref.double()).abs().amax(1) / ref.double().abs().amax(1).clamp_min(1e-300)).max()
    assert float(err) < 1e-5, float(err)


def test_backward_input_zero_sizes_abi():
    """in_f or out_f of 0 are accepted, as by the reference kernel
    (fp8_cpu.cpp:227-228): out_f == 0 is an empty sum (dx all zeros, g / w / s
    not read), in_f == 0 leaves nothing to write."""
    from smaulnative_amd import _lib
    lib = _lib.load()
    print("case backward_input zero sizes", flush=True)
    stream = torch.cuda.current_stream().cuda_stream
    dx = torch.full((3, 5), 7.0, device=DEV)
    _lib.check(lib.smaul_fp8_backward_input(None, None, None, dx.data_ptr(), 3, 5, 0, 64, stream), "out_f 0")
    _lib.check(lib.smaul_fp8_backward_input(None, None, None, None, 3, 0, 4, 64, stream), "in_f 0")
    torch.cuda.synchronize()
    assert torch.equal(dx.cpu(), torch.zeros(3, 5))
    assert lib.smaul_fp8_backward_input(None, None, None, dx.data_ptr(), 3, -1, 4, 64, stream) == _lib.SMAUL_ERR_INVALID


@pytest.mark.parametrize("rows,in_f,tile", [(3, 64, 64), (70, 192, 64), (33, 128, 128), (5, 256, 32)])
def test_backward_input_empty_sum_reads_nothing(rows, in_f, tile):
    """out_f == 0 with in_f a multiple of 64 and null g / w / s, whose alignment
    is that of the vector loads: dx all zeros, nothing read."""
    from smaulnative_amd import _lib
    lib = _lib.load()
    print(f"case backward empty sum rows={rows} in_f={in_f} tile={tile}", flush=True)
    dx = torch.full((rows, in_f), 7.0, device=DEV)
    stream = torch.cuda.current_stream().cuda_stream
    _lib.check(lib.smaul_fp8_backward_input(None, None, None, dx.data_ptr(), rows, in_f, 0, tile, stream), "out_f 0")
    assert torch.equal(dx.cpu(), torch.zeros(rows, in_f))


def test_weight_grad_of_more_rows_than_a_grid_dimension():
    """out_f past 64 * 65535, the tiles that fit a launch's second dimension, as
    the blocks of 64 rows took it: the last rows are computed like the first
    (the products of two rows are exact in fp32 here, one bf16 rounding)."""
    out_f, in_f, rows = 64 * 65535 + 65, 3, 2
    print(f"case weight grad out_f={out_f}", flush=True)
    gen = torch.Generator(device=DEV).manual_seed(7)
    g = torch.randint(-8, 9, (rows, out_f), generator=gen, device=DEV).float()
    x = torch.randint(-8, 9, (rows, in_f), generator=gen, device=DEV).float()
    gw = torch.randint(-8, 9, (out_f, in_f), generator=gen, device=DEV).to(torch.bfloat16)
    ref = (gw.float() + g[0, :, None] * x[0] + g[1, :, None] * x[1]).to(torch.bfloat16)
    get_backend("rocm").fp8_weight_grad(g, x, gw)
    assert torch.equal(gw, ref)


def test_kernels_that_write_in_place_bump_the_version():
    """What autograd saved and a kernel then overwrote is noticed, as with the
    in-place operations: the accumulated weight gradient and the Lion momentum."""
    from smaulnative_amd import FP8Linear
    print("case in-place versions", flush=True)
    lin = FP8Linear(64, 32).to(DEV).train()
    x = torch.randn(5, 64, device=DEV, requires_grad=True)
    lin(x).sum().backward()
    w = torch.ones(32, 64, device=DEV, dtype=torch.bfloat16, requires_grad=True)
    held = w * lin._gw
    lin(x).sum().backward()  # adds to _gw in place
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        held.sum().backward()
    momentum = torch.zeros(32, 64, device=DEV)
    held = w.float() * momentum
    lin.fused_lion_requant(lin._gw, momentum, 1e-3, 0.1, 0.9, 0.99)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        held.sum().backward()


@pytest.mark.parametrize("rows,in_f,out_f,dtype,kernel", [
    # about the lines of the rule: one block of 64 rows (by rows and by rows x
    # in_f), two, three; and bf16 x converted for the kernel, or not
    (16383, 8, 64, torch.float32, torch.float32), (16384, 8, 64, torch.float32, None),
    (4095, 4096, 16, torch.bfloat16, torch.bfloat16), (4096, 4096, 16, torch.bfloat16, None),
    (65535, 24, 65, torch.bfloat16, torch.float32), (65536, 24, 65, torch.float32, None),
    (65536, 24, 129, torch.float32, torch.float32), (1023, 70, 1100, torch.bfloat16, torch.bfloat16),
    (1024, 70, 1024, torch.bfloat16, torch.float32)])
def test_weight_grad_route(rows, in_f, out_f, dtype, kernel, monkeypatch):
    """Few outputs over many rows go to the 64-row blocks (None), which a library
    product fills the device with; both give g^T x within its fp32 sums' bound."""
    from smaulnative_amd import FP8Linear
    print(f"case weight grad route rows={rows} in_f={in_f} out_f={out_f} {dtype}", flush=True)
    bk = get_backend("rocm")
    run, took = bk.fp8_weight_grad, []
    monkeypatch.setattr(bk, "fp8_weight_grad", lambda g, x, gw, fresh: (took.append(x.dtype), run(g, x, gw, fresh)))
    torch.manual_seed(rows)
    lin = FP8Linear(in_f, out_f).to(DEV).train()
    x = torch.randn(rows, in_f, device=DEV).to(dtype).requires_grad_(True)
    g = torch.randn(rows, out_f, device=DEV).to(dtype)
    lin(x).backward(g)
    assert took == ([] if kernel is None else [kernel])
    ref = g.double().t() @ x.detach().double()
    slack = rows * 2.0 ** -24 * (g.double().abs().t() @ x.detach().double().abs())
    assert bool(((lin._gw.double() - ref).abs() <= slack + (ref.abs() + slack) * 2.0 ** -8).all())
