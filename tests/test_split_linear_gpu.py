"""fp32 products on the 16-bit matrix cores: against float64, and no further from it than torch's fp32 products."""
import pytest
import torch

from quick_ssm_amd import split_linear

pytestmark = pytest.mark.gpu


def _error(got, ref):
    return ((got.double() - ref).norm() / ref.norm()).item()


# Bound of the relative error (2-norm): 2^-23 for the split (what it leaves out of a pair is below 2^-24 of it) plus the
# fp32 accumulation of up to K / 16 * 3 sums of a part, 2^-24 * sqrt(3 K / 16) and no more.
def _bound(k):
    return 2.0 ** -23 + 2.0 ** -24 * (3 * k / 16) ** 0.5


# tiles are 128 x 128 and stages 16 long: one below, on and above each edge, several launches' worth, and the
# layer's own ratios
SHAPES = [(256, 16, 128, 1), (255, 20, 132, 1), (257, 12, 124, 5), (1, 64, 64, 1), (1000, 72, 260, 2), (4096, 256, 1280, 1),
          (2048, 256, 512, 5), (515, 1024, 256, 1), (16384, 36, 64, 3)]


@pytest.mark.parametrize("rows,k,n,count", SHAPES)
def test_products_and_gradients_match_float64(gpu, rows, k, n, count):
    gen = torch.Generator().manual_seed(rows + k)
    u = torch.randn(rows, k, generator=gen).to(gpu)
    u *= torch.logspace(-6, 6, rows, device=gpu)[:, None] if rows > 1 else 1.0      # rows of very different size
    ws = [((torch.rand(n, k, generator=gen) * 2 - 1) * k ** -0.5).to(gpu) for _ in range(count)]
    bias = [torch.randn(n, generator=gen).to(gpu)] + [None] * (count - 1)
    wide = torch.randn(rows, count * n, generator=gen).to(gpu) * 1e-4
    gs = [wide[:, i * n:(i + 1) * n] for i in range(count)]
    outs, maxima = split_linear.forward(u, ws, bias, True, True)
    du, dws = split_linear.backward(gs, u, ws, maxima, True, True)
    u64, w64, g64 = u.double(), [w.double() for w in ws], [g.double() for g in gs]
    for i in range(count):
        ref = u64 @ w64[i].t()
        got = outs[i].double() - (bias[i].double() if bias[i] is not None else 0.0)
        # row by row, each with its own scale; the bias adds its own rounding
        slack = 2.0 ** -23 * (ref.abs().amax(1) + (bias[i].abs().max().item() if bias[i] is not None else 0.0)) * n ** 0.5
        assert bool(((got - ref).norm(dim=1) <= _bound(k) * u64.norm(dim=1) * w64[i].norm() + slack).all())
        ref = g64[i].t() @ u64
        assert _error(dws[i], ref) <= _bound(rows)
    ref = sum(g @ w for g, w in zip(g64, w64))
    assert bool(((du.double() - ref).norm(dim=1) <= _bound(n * count) * ref.norm(dim=1) * 4).all())


def test_no_further_from_float64_than_fp32_products(gpu):
    gen = torch.Generator().manual_seed(1)
    for rows, k, n in ((2048, 64, 256), (2048, 256, 1024), (4096, 1024, 1024), (8192, 128, 512)):
        u = torch.randn(rows, k, generator=gen).to(gpu)
        w = ((torch.rand(n, k, generator=gen) * 2 - 1) * k ** -0.5).to(gpu)
        g = torch.randn(rows, n, generator=gen).to(gpu)
        (y,), maxima = split_linear.forward(u, [w], [None], True, True)
        du, (dw,) = split_linear.backward([g], u, [w], maxima, True, True)
        for got, lib, ref in ((y, u @ w.t(), u.double() @ w.double().t()), (du, g @ w, g.double() @ w.double()),
                              (dw, g.t() @ u, g.double().t() @ u.double())):
            assert _error(got, ref) <= 1.1 * _error(lib, ref)


def test_infinities_nan_zeros_and_extremes_behave_as_in_fp32(gpu):
    gen = torch.Generator().manual_seed(2)
    u = torch.randn(600, 64, generator=gen).to(gpu)
    w = torch.randn(300, 64, generator=gen).to(gpu)
    u[3, 5], u[70, 9], u[400, 63], w[7, 11] = float("inf"), float("nan"), float("-inf"), float("-inf")
    u[301] = 0.0
    u[302], u[303] = 1e-30, 1e36
    u[304, 0] = 3.4e38
    (y,), _ = split_linear.forward(u, [w], [None], False, False)
    ref = u @ w.t()
    assert torch.equal(torch.isnan(y), torch.isnan(ref)) and torch.equal(torch.isposinf(y), torch.isposinf(ref))
    assert torch.equal(torch.isneginf(y), torch.isneginf(ref))
    assert not bool(y[301, 8:].any())
    fine = torch.isfinite(ref).all(1) & (torch.arange(600, device=gpu) != 301)
    cols = torch.arange(300, device=gpu) != 7
    exact = (u[fine].double() @ w[cols].double().t())
    assert bool(((y[fine][:, cols].double() - exact).norm(dim=1) <= 1e-6 * exact.norm(dim=1)).all())


def test_a_layer_takes_them_and_repeats_bit_for_bit(gpu, monkeypatch):
    from quick_ssm_amd import SSM

    calls = []
    for name in ("forward", "backward"):
        monkeypatch.setattr(split_linear, name, lambda *a, _f=getattr(split_linear, name): (calls.append(1), _f(*a))[1])
    torch.manual_seed(0)
    layer = SSM(1024, 4, device=gpu)
    x = torch.randn(3, 1400, 1024, device=gpu, requires_grad=True)
    dy = torch.randn_like(x)

    def step():
        layer.zero_grad()
        return torch.autograd.grad(layer(x), [x, *layer.parameters()], dy)

    first, second = step(), step()
    assert len(calls) == 8 and all(torch.equal(a, b) for a, b in zip(first, second))
    monkeypatch.setattr(split_linear, "usable", lambda *a: False)
    for got, want in zip(first, step()):
        # the gates round to fp16, so a product's last bit may move an operand by 2^-11
        assert _error(got, want.double()) < 2e-3


@pytest.mark.parametrize("k,n,count,gradients,taken", [
    (128, 32, 1, False, False), (144, 192, 5, False, False), (128, 256, 5, False, True), (144, 1024, 1, False, True),
    (124, 4096, 5, False, False), (256, 32, 1, False, True), (128, 32, 1, True, True), (124, 64, 5, True, True)])
def test_narrow_inputs_and_outputs_stay_with_the_library_in_inference(gpu, k, n, count, gradients, taken):
    rows = split_linear.MIN_WORK // (k * n * count) + 1
    u, ws = torch.empty(rows, k, device=gpu), [torch.empty(n, k, device=gpu) for _ in range(count)]
    assert split_linear.usable(u, ws, gradients) == taken
    assert not split_linear.usable(u[:rows // 2], ws, gradients)
