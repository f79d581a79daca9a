"""LayerNorm on the HIP kernels: values and gradients against float64, and the calls that stay with
torch."""
import importlib

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF, F32 = torch.bfloat16, torch.float32


@pytest.fixture(scope="module")
def modules():
    return importlib.import_module("rwkv-megatron_amd").modules


def _norm(modules, C, wdt, bdt):
    g = torch.Generator().manual_seed(C)
    ln = modules.LayerNorm(C, eps=1e-5, device=DEV)
    ln.weight = torch.nn.Parameter((torch.randn(C, generator=g) * 0.5 + 1).to(wdt).to(DEV))
    ln.bias = torch.nn.Parameter(torch.randn(C, generator=g).to(bdt).to(DEV))
    return ln


def _case(shape, C):
    g = torch.Generator().manual_seed(7 * C + shape[0])
    mk = lambda: torch.randn(*shape, C, generator=g).to(BF).to(DEV)
    return mk() * 3 + 0.5, mk()


def _exact(x, w, b, dy, eps):
    x, w, b, dy = (t.double() for t in (x, w, b, dy))
    m = x.mean(-1, keepdim=True)
    r = ((x - m).square().mean(-1, keepdim=True) + eps).rsqrt()
    xh, g = (x - m) * r, dy * w
    dx = r * (g - g.mean(-1, keepdim=True) - xh * (g * xh).mean(-1, keepdim=True))
    rows = tuple(range(x.dim() - 1))
    return xh * w + b, dx, (dy * xh).sum(rows), dy.sum(rows)


# Rows at the edges of a wave's pieces (C = 8 .. 4096: one to eight of 512 channels, full and with a
# remainder), of the four rows of a block, of the backward's ranges (8 rows; more than 8 above 4096),
# and every mix of parameter dtypes.  A bf16 result is rounded once, 2^-9 of itself; fp32 sums of n
# terms of size s differ by less than 2^-23 n s, and n s <= 5000 * 16 here: the absolute part.
@pytest.mark.parametrize("shape,C,wdt,bdt", [
    ((1,), 8, F32, F32), ((3,), 64, BF, BF), ((5, 1), 512, F32, BF), ((4,), 520, BF, F32),
    ((9,), 1024, F32, F32), ((2, 4), 1032, BF, BF), ((777, 1), 2048, F32, F32), ((33,), 2056, F32, F32),
    ((17,), 4096, BF, BF), ((4099,), 512, F32, F32), ((512, 2), 512, torch.float16, torch.float16)])
def test_layer_norm_matches_float64(modules, shape, C, wdt, bdt):
    ln = _norm(modules, C, wdt, bdt)
    x, dy = _case(shape, C)
    if len(shape) == 2:                                   # rows apart in memory
        x = x.transpose(0, 1).contiguous().transpose(0, 1)
    x.requires_grad_(True)
    y = ln(x)
    assert "LayerNormBackward" in type(y.grad_fn).__name__ or "LayerNorm" in y.grad_fn.name()
    assert "Native" not in y.grad_fn.name()
    got = [y.detach(), *torch.autograd.grad(y, (x, ln.weight, ln.bias), dy)]
    y2 = ln(x)
    again = [y2.detach(), *torch.autograd.grad(y2, (x, ln.weight, ln.bias), dy)]
    ref = _exact(x.detach(), ln.weight.detach(), ln.bias.detach(), dy, ln.eps)
    for a, b, c, dt in zip(got, again, ref, (BF, BF, wdt, bdt)):
        assert a.dtype == dt and a.shape == c.shape and torch.equal(a, b)
        half = {BF: 2.0 ** -8, torch.float16: 2.0 ** -10, F32: 2.0 ** -20}[dt]
        bound = half * c.abs() + 2.0 ** -23 * (16 * max(x.numel() // C, C))
        assert bool(((a.double() - c).abs() <= bound).all()), float(((a.double() - c).abs() - bound).max())


def test_layer_norm_calls_that_stay_with_torch(modules):
    ln = _norm(modules, 64, F32, F32)
    x, dy = _case((6,), 64)
    cast = lambda t: F.layer_norm(t, (64,), ln.weight.to(t.dtype), ln.bias.to(t.dtype), ln.eps)
    for t in (x.float(), x.half(), x[:0]):
        assert torch.equal(ln(t), cast(t))
    big, bx = _norm(modules, 4104, BF, BF), _case((3,), 4104)[0]
    assert torch.equal(big(bx), F.layer_norm(bx, (4104,), big.weight, big.bias, big.eps))
    with torch.autocast("cuda", dtype=BF):
        assert torch.equal(ln(x), cast(x)) and ln(x).dtype == cast(x).dtype
    assert torch.equal(torch.func.vmap(ln)(x), cast(x))
    out, tan = torch.func.jvp(ln, (x,), (dy,))
    assert torch.equal(out, cast(x)) and torch.equal(tan, torch.func.jvp(cast, (x,), (dy,))[1])
    with pytest.raises(RuntimeError):
        ln(x[:, :32])
    traced = torch.jit.trace(ln, (x,), check_trace=False)
    other = _case((6,), 64)[1]
    assert torch.equal(traced(other), cast(other))


# Second derivatives go through torch's differentiable form.  Forward values differ from torch's by
# the rounding of the cast parameters, 2^-9, and every bf16 intermediate by another: 2^-5 of the
# largest entry covers the eight of the chain.
def test_layer_norm_second_derivative_and_updates(modules):
    ln = _norm(modules, 64, F32, F32)
    x, dy = _case((6,), 64)
    x.requires_grad_(True)

    def second(f):
        gx, gw = torch.autograd.grad(f(x), (x, ln.weight), dy, create_graph=True)
        return torch.autograd.grad(gx.float().square().sum() + gw.float().square().sum(), (x, ln.weight))

    a, b = second(ln), second(lambda t: F.layer_norm(t, (64,), ln.weight.to(BF), ln.bias.to(BF), ln.eps))
    for p, q in zip(a, b):
        assert float((p.float() - q.float()).abs().max()) <= 2.0 ** -5 * float(q.float().abs().max())
    # the backward uses the weight that the forward saw
    want = torch.autograd.grad(ln(x), x, dy)[0]
    y = ln(x)
    with torch.no_grad():
        ln.weight.mul_(2)
    assert torch.equal(torch.autograd.grad(y, x, dy)[0], want)


# The same chain, so the same bound, for an input that the kernels read through a dense copy: strided, or
# off the 16-byte grid.  x enters the loss a second time, so that a lost d(dx)/dx would not be an error.
@pytest.mark.parametrize("form", ["transposed", "shifted"])
@pytest.mark.parametrize("wdt", [F32, BF])
def test_layer_norm_second_derivative_of_a_copied_input(modules, form, wdt):
    ln = _norm(modules, 64, wdt, wdt)
    x, dy = _case((6, 5), 64)
    x = x.transpose(0, 1) if form == "transposed" else torch.cat([x.reshape(-1)[:1], x.reshape(-1)])[1:].view(x.shape)
    dy = dy.transpose(0, 1) if form == "transposed" else dy
    x = x.detach().requires_grad_(True)
    assert not x.is_contiguous() or x.data_ptr() % 16

    def second(f):
        gx, gw = torch.autograd.grad(f(x), (x, ln.weight), dy, create_graph=True)
        return torch.autograd.grad(gx.float().square().sum() + gw.float().square().sum() + x.float().sum(), (x, ln.weight))

    a, b = second(ln), second(lambda t: F.layer_norm(t, (64,), ln.weight.to(BF), ln.bias.to(BF), ln.eps))
    for p, q in zip(a, b):
        assert float((p.float() - q.float()).abs().max()) <= 2.0 ** -5 * float(q.float().abs().max())
