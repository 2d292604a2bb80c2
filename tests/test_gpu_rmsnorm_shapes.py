"""RMSNorm at the edges of its launch shapes: rows owned by part of a wavefront,
by one and by a workgroup, in 16-byte chunks and element by element, with as
many rows as leave owners idle, fill them once and make them walk on."""
import pytest
import torch

from oracle import rms_oracle as rorc

pytestmark = pytest.mark.gpu

EPS = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -23}


def _check(x, dy, w):
    import tritonops_amd as ta

    dt, (rows, dim) = x.dtype, x.shape
    xc, dc, wc = x.cpu(), dy.cpu(), w.cpu()
    y, rs = ta.rmsnorm_fwd(x, w, 1e-6)
    dx, dw = ta.rmsnorm_bwd(dy, x, w, rs, 1e-6)
    want = rorc.rms_norm(xc.double(), wc.double(), 1e-6)
    wdx, wdw = rorc.rms_norm_backward(dc, xc, wc, 1e-6)
    # results: one rounding to the storage type (half an ulp) and fp32 sums of dim terms (a few 2^-23 relative to the
    # largest partial sum, below 2^-23 * dim / 8 by the in-lane and butterfly order)
    tol = EPS[dt] + 2.0 ** -23 * (8 + dim / 8)
    assert ((y.cpu().double() - want).abs() <= tol * (want.abs() + 1e-3)).all()
    assert (dx.cpu().double() - wdx).abs().max() <= tol * max(1.0, wdx.abs().max().item())
    # dw: fp32 sums over the rows of terms of magnitude |dy x r|, then one rounding to the weight's type
    mag = (dc.double().abs() * xc.double().abs() * torch.rsqrt((xc.double() ** 2).mean(-1, keepdim=True))).sum(0)
    wtol = EPS[w.dtype] * wdw.abs() + 2.0 ** -23 * (8 + rows / 64) * mag
    assert ((dw.cpu().double() - wdw).abs() <= wtol).all()


def _inputs(rows, dim, dt, wdt, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn((rows, dim), generator=g, device="cuda").to(dt)
    dy = torch.randn((rows, dim), generator=g, device="cuda").to(dt)
    w = (1 + 0.1 * torch.randn((dim,), generator=g, device="cuda")).to(wdt)
    return x, dy, w


@pytest.mark.parametrize("rows,dim", [
    (5, 1), (4099, 7), (129, 255), (300, 257), (4097, 511), (33, 513), (5, 1023), (4100, 1025), (3, 2047), (1025, 2049),
    (1500, 4095), (7, 4097), (1100, 5001), (3, 8191), (3, 8193)])
@pytest.mark.parametrize("dt,wdt", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32),
                                    (torch.float32, torch.float32)])
def test_element_wise_rows(rows, dim, dt, wdt):
    _check(*_inputs(rows, dim, dt, wdt))


@pytest.mark.parametrize("rows", [1, 7, 31, 33, 2048 * 32 + 5])
@pytest.mark.parametrize("dim", [8, 56, 64, 72, 96, 128, 136, 256, 264, 512])
def test_rows_of_part_of_a_wavefront(rows, dim):
    _check(*_inputs(rows, dim, torch.bfloat16, torch.bfloat16))
    if rows < 100:
        _check(*_inputs(rows, dim // 2, torch.float32, torch.float32))


@pytest.mark.parametrize("dim", [64, 512, 1024, 4096])
def test_rows_that_are_not_aligned(dim):
    """Widths of the 16-byte path whose rows start between 16-byte boundaries."""
    x, dy, w = _inputs(77, dim, torch.bfloat16, torch.bfloat16)
    wide = torch.empty((77, dim + 3), device="cuda", dtype=torch.bfloat16)
    xs = wide[:, 1:dim + 1]
    xs.copy_(x)
    _check(xs, dy, w)
    flat = torch.empty(77 * dim + 1, device="cuda", dtype=torch.bfloat16)
    ds = flat[1:].view(77, dim)
    ds.copy_(dy)
    _check(x, ds, w)
