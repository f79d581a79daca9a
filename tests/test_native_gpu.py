"""The C++ autograd functions (csrc/autograd.cpp) where a Python autograd function has rules that
they must keep: saved-tensor hooks, in-place changes of saved tensors, outputs no loss uses,
inputs that need a copy, function transforms and forward-mode differentiation (refused)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _ops(pkg):
    """name -> (function of its leaves, leaves)."""
    g = torch.Generator().manual_seed(5)
    bf = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16).to(DEV)
    T, B, C = 70, 2, 128
    w = -torch.rand(1, 2, T, 64, generator=g).to(torch.bfloat16).to(DEV)
    hd = lambda: bf(1, 2, T, 64)
    tm, cm = pkg.timemix, pkg.channelmix
    return {
        "wkv": (lambda r, k, v, w, u, h: pkg.chunk_rwkv6(r, k, v, w, u, 1.0, h, True),
                [hd(), hd(), hd(), w, bf(2, 64).float(), bf(1, 2, 64, 64).float()]),
        "seqfirst": (lambda r, k, v, d, u: pkg.wkv6_seqfirst(r, k, v, d, u, 2, output_final_state=True),
                     [bf(T, B, C), bf(T, B, C), bf(T, B, C), bf(T, B, C), bf(2, 64)]),
        "mix": (tm.token_shift_mix, [bf(T, B, C), bf(C), bf(C, 5, 32) * 0.05, bf(5, 32, C) * 0.1, bf(5, C)]),
        "decay": (tm.decay_lora, [bf(T, B, C), bf(C, 1, 64) * 0.05, bf(1, 64, C) * 0.1, bf(1, C)]),
        "gn": (lambda o, x, ga, be: tm.group_norm_gate(o, x, ga, be, 1e-5), [bf(B, 2, T, 64), bf(T, B, C), bf(C), bf(C)]),
        "lerp": (cm.cmix_lerp, [bf(T, B, C), bf(2, C)]),
        "relu": (cm.relu_sq, [bf(T, B, C)]),
        "gate": (cm.sigmoid_gate, [bf(T, B, C), bf(T, B, C)]),
        "linear": (pkg._lib.native().linear, [bf(T, B, C), bf(64, C).float()]),
    }


NAMES = ["wkv", "seqfirst", "mix", "decay", "gn", "lerp", "relu", "gate", "linear"]


def _outs(o):
    return [t for t in (o if isinstance(o, (tuple, list)) else (o,)) if t is not None]


@pytest.mark.parametrize("name", NAMES)
def test_saved_tensor_hooks_and_versions(pkg, name):
    fn, leaves = _ops(pkg)[name]
    leaves = [t.requires_grad_(True) for t in leaves]
    base = torch.autograd.grad(sum(t.float().square().sum() for t in _outs(fn(*leaves))), leaves)
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (packed.append(t), t.cpu())[1], lambda t: t.to(DEV)):
        out = _outs(fn(*leaves))
    assert packed
    again = torch.autograd.grad(sum(t.float().square().sum() for t in out), leaves)
    assert all(torch.equal(a, b) for a, b in zip(base, again))
    out = _outs(fn(*leaves))
    with torch.no_grad():
        leaves[0].add_(1)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(sum(t.float().square().sum() for t in out), leaves)


@pytest.mark.parametrize("name", NAMES)
@pytest.mark.parametrize("kind", [TypeError, ValueError])
def test_an_error_of_a_saved_tensor_hook_is_raised_itself(pkg, name, kind):
    fn, leaves = _ops(pkg)[name]

    def pack(t):
        raise kind("from the hook")

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t), pytest.raises(kind, match="from the hook"):
        fn(*[t.requires_grad_(True) for t in leaves])


@pytest.mark.parametrize("name", ["wkv", "seqfirst", "mix", "lerp"])
def test_unused_outputs_have_zero_gradients(pkg, name):
    """A loss on one output alone: the same gradients as with zero gradients for the others."""
    fn, leaves = _ops(pkg)[name]
    leaves = [t.requires_grad_(True) for t in leaves]
    n = len(_outs(fn(*leaves)))
    for i in range(n):
        out = _outs(fn(*leaves))
        dy = [torch.ones_like(t) if j == i else torch.zeros_like(t) for j, t in enumerate(out)]
        want = torch.autograd.grad(out, leaves, dy)
        got = torch.autograd.grad(_outs(fn(*leaves))[i], leaves, torch.ones_like(out[i]))
        assert all(torch.equal(a, b) for a, b in zip(want, got))


@pytest.mark.parametrize("name", NAMES)
def test_copied_inputs(pkg, name):
    """Strided inputs and inputs off the 16-byte grid give the results of their dense copies."""
    fn, leaves = _ops(pkg)[name]

    def strided(t):
        return torch.stack([t, t], -1)[..., 0]

    def shifted(t):
        return torch.cat([t.reshape(-1)[:1], t.reshape(-1)])[1:].view(t.shape)

    def run(ls):
        ls = [t.detach().requires_grad_(True) for t in ls]
        out = _outs(fn(*ls))
        return out + list(torch.autograd.grad(out, ls, [strided(torch.ones_like(t)) for t in out]))

    want = run(leaves)
    for make in (strided, shifted):
        assert all(torch.equal(a, b) for a, b in zip(want, run([make(t) for t in leaves])))


@pytest.mark.parametrize("name", NAMES)
def test_transforms_are_refused(pkg, name):
    fn, leaves = _ops(pkg)[name]
    with pytest.raises(RuntimeError):
        torch.func.vmap(fn)(*[torch.stack([t, t]) for t in leaves])
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda t: _outs(fn(t, *leaves[1:]))[0].float().sum())(leaves[0])
    import torch.autograd.forward_ad as fwd
    with fwd.dual_level(), pytest.raises((RuntimeError, NotImplementedError)):
        _outs(fn(fwd.make_dual(leaves[0].clone().requires_grad_(True), torch.ones_like(leaves[0])), *leaves[1:]))


# Token tiles of 32 (eight waves: few workgroups; four) and 64, their remainders, a tail of the 64 or 128
# inputs of a step, outputs that do not fill a tile.  Both operands are exact in bf16, so the result differs
# from float64's by its own rounding, 2^-9, and the fp32 sums' 2^-23 I sum |x w|; the bf16 weight that the
# backward multiplies with gives the library path's dx bit for bit.
@pytest.mark.parametrize("N,O,I", [(1, 4, 8), (31, 64, 64), (32, 68, 72), (33, 200, 712), (65, 60, 2048),
                                   (1030, 512, 136), (2050, 512, 64), (2112, 516, 200)])
def test_linear_of_an_fp32_weight(pkg, N, O, I):
    g = torch.Generator().manual_seed(N + O)
    x = torch.randn(N, 1, I, generator=g).to(torch.bfloat16).to(DEV).requires_grad_(True)
    w = (torch.randn(O, I, generator=g) * I ** -0.5).to(DEV).requires_grad_(True)
    dy = torch.randn(N, 1, O, generator=g).to(torch.bfloat16).to(DEV)
    linear = pkg._lib.native().linear
    y = linear(x, w)
    wb = w.detach().to(torch.bfloat16).requires_grad_(True)
    ref = x.detach().double() @ wb.detach().double().t()
    mag = x.detach().double().abs() @ wb.detach().double().abs().t()
    assert y.shape == (N, 1, O) and y.dtype == torch.bfloat16
    assert bool(((y.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 2.0 ** -23 * I * mag).all())
    dx, dw = torch.autograd.grad(y, (x, w), dy)
    dxb, _ = torch.autograd.grad(linear(x, wb), (x, wb), dy)
    assert torch.equal(dx, dxb) and dw.dtype == torch.float32 and dw.shape == w.shape
    with torch.no_grad():
        assert torch.equal(linear(x, w), y) and torch.equal(linear(x[:1, 0], w), linear(x[:1], w)[0])
    strided = x.detach().transpose(0, 2).contiguous().transpose(0, 2)
    assert torch.equal(linear(strided, w), y)


# dx = dy W and dW = dy^T x are linear, so d(sum dW * m)/dx = dy m and so on: exact in bf16 operands up to
# one rounding, 2^-9, of each bf16 result and the fp32 sums.  One chunk of tokens, odd (N = 33), and a
# count that the plain backward splits (10240).
@pytest.mark.parametrize("N", [33, 10240])
@pytest.mark.parametrize("wdt", [torch.float32, torch.bfloat16])
def test_linear_second_derivative(pkg, N, wdt):
    g = torch.Generator().manual_seed(N)
    bf = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16).to(DEV)
    x, dy, m = bf(N, 64).requires_grad_(True), bf(N, 32).requires_grad_(True), bf(32, 64)
    w = (bf(32, 64).float() * 0.125).to(wdt).requires_grad_(True)
    y = pkg._lib.native().linear(x, w)
    plain = torch.autograd.grad(y, w, dy.detach(), retain_graph=True)[0]
    dw = torch.autograd.grad(y, w, dy, create_graph=True)[0]
    ref = dy.detach().double().t() @ x.detach().double()
    for t in (plain, dw):
        assert t.dtype == wdt
        half = 2.0 ** -8 if wdt == torch.bfloat16 else 0.0
        assert bool(((t.double() - ref).abs() <= half * ref.abs() + 2.0 ** -23 * N * 16).all())
    gx, gdy = torch.autograd.grad((dw * m).sum(), (x, dy))
    for got, want in ((gx, dy.detach().double() @ m.double()), (gdy, x.detach().double() @ m.double().t())):
        assert bool(((got.double() - want).abs() <= 2.0 ** -7 * want.abs() + 2.0 ** -23 * 64 * 16).all())


# The weight gradient's chunks of tokens: one, two and four of them, on both sides of each line (a chunk of
# 2560 tokens for few output tiles, of 4096 for more than 32; counts that do not divide), for every parameter
# type.  Exact bf16 operands: off by the result's own rounding and that of the fp32 sums, N additions to sums
# of up to 4 sqrt(N), 2^-24 each like a random walk: 2^-22 N, and four times that as the bound.
@pytest.mark.parametrize("N,O,I,chunks", [
    (5119, 256, 256, 1), (5118, 256, 256, 1), (5120, 256, 256, 2), (5121, 256, 256, 1), (10238, 256, 256, 2),
    (10240, 256, 256, 4), (10242, 256, 256, 2), (20480, 200, 72, 4), (8190, 2048, 1280, 1),
    (8192, 2048, 1280, 2), (8193, 2048, 1280, 1), (16384, 1280, 2048, 4)])
@pytest.mark.parametrize("wdt", [torch.bfloat16, torch.float32, torch.float16])
def test_linear_weight_gradient(pkg, N, O, I, chunks, wdt):
    tiles = -(-O // 256) * -(-I // 256)
    least, s = 4096 if tiles > 32 else 2560, 1
    while s < 4 and tiles * s < 256 and N % (2 * s) == 0 and N // (2 * s) >= least:
        s *= 2
    assert s == chunks                                     # the rule of csrc/autograd.cpp, restated
    g = torch.Generator(device=DEV).manual_seed(N + O)
    x = torch.randn(N, I, generator=g, device=DEV).to(torch.bfloat16)
    dy = torch.randn(N, O, generator=g, device=DEV).to(torch.bfloat16)
    w = (torch.randn(O, I, generator=g, device=DEV) * I ** -0.5).to(wdt).requires_grad_(True)
    grads = [torch.autograd.grad(pkg._lib.native().linear(x, w), w, dy)[0] for _ in range(2)]
    ref = dy.double().t() @ x.double()
    assert grads[0].dtype == wdt and torch.equal(*grads)
    half = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -10, torch.float32: 0.0}[wdt]
    bound = half * ref.abs() + 2.0 ** -20 * N
    assert bool(((grads[0].double() - ref).abs() <= bound).all())
