"""A 16-bit layer in training takes its five projections as one product; everything about it but the speed is as with five."""
import pytest
import torch

from quick_ssm_amd import SSM, layers

pytestmark = pytest.mark.gpu


def _step(layer, x, dy):
    layer.zero_grad()
    y = layer(x)
    return [y.detach(), *torch.autograd.grad(y, [x, *(p for p in layer.parameters() if p.requires_grad)], dy)]


@pytest.mark.parametrize("hidden,mult,shape", [(128, 2, (5, 333)), (96, 1.25, (2, 700)), (64, 1, (3, 129))], ids=str)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=str)
def test_matches_the_five_products(gpu, monkeypatch, hidden, mult, shape, dtype):
    monkeypatch.setattr(SSM, "_BATCHED_PROJECTION_LIMIT", 0)   # small shapes count as large ones
    torch.manual_seed(1)
    layer = SSM(hidden, mult, dtype=dtype, device=gpu, compute_dtype=dtype)
    x = torch.randn(*shape, hidden, device=gpu, dtype=dtype, requires_grad=True)
    dy = torch.randn_like(x)
    pointers = [p.data_ptr() for p in layer.parameters()]
    calls = []
    monkeypatch.setattr(layers._WideProjections, "apply", lambda *a, _f=layers._WideProjections.apply: (calls.append(1), _f(*a))[1])
    got = _step(layer, x, dy)
    assert calls and pointers == [p.data_ptr() for p in layer.parameters()]     # the parameters stay where they are
    layer.B_proj.weight.requires_grad_(False)
    assert len(_step(layer, x, dy)) == len(got) - 1
    layer.B_proj.weight.requires_grad_(True)
    n = len(calls)
    layer.D_proj.register_forward_hook(lambda *a: None)                         # a hook wants the module to be called
    want = _step(layer, x, dy)
    assert len(calls) == n
    with torch.no_grad():
        layer(x)
    assert len(calls) == n
    for g, w in zip(got, want):
        # the five products round once more each on the way to the input's gradient
        assert (g.double() - w.double()).norm() <= 4 * torch.finfo(dtype).eps * w.double().norm()


def test_a_weight_changed_before_the_backward_is_an_error_and_second_derivatives_reach_the_weights(gpu, monkeypatch):
    monkeypatch.setattr(SSM, "_BATCHED_PROJECTION_LIMIT", 0)
    torch.manual_seed(1)
    layer = SSM(64, 1, dtype=torch.bfloat16, device=gpu, compute_dtype=torch.bfloat16, use_norm=False)
    x = torch.randn(2, 200, 64, device=gpu, dtype=torch.bfloat16, requires_grad=True)
    y = layer(x)
    with torch.no_grad():
        layer.C_proj_a.weight.mul_(0.5)
    with pytest.raises(RuntimeError, match="inplace operation"):
        y.sum().backward()
    (dx,) = torch.autograd.grad(layer(x).float().sum(), x, create_graph=True)
    grads = torch.autograd.grad(dx.float().pow(2).sum(), [layer.A_proj.weight, layer.D_proj.weight])
    assert all(bool(g.any()) for g in grads)


def test_nothing_is_kept_for_the_backward_that_five_products_would_not_keep(gpu, monkeypatch):
    monkeypatch.setattr(SSM, "_BATCHED_PROJECTION_LIMIT", 0)
    layer = SSM(512, 4, dtype=torch.bfloat16, device=gpu, compute_dtype=torch.bfloat16)
    x = torch.randn(1, 128, 512, device=gpu, dtype=torch.bfloat16, requires_grad=True)
    kept = {}
    for name in ("five", "one"):
        monkeypatch.setattr(SSM, "_WIDE_PRODUCT_LIMIT", 0 if name == "five" else 1 << 26)
        layer(x).sum().backward()                       # buffers of the launches exist from here on
        layer.zero_grad()
        x.grad = None
        before = torch.cuda.memory_allocated(gpu)
        y = layer(x)
        kept[name] = torch.cuda.memory_allocated(gpu) - before
        del y
    # (the five weights are 10 MB, what the graph keeps of the activations 3; tensors are rounded up to 512 bytes)
    assert kept["one"] <= kept["five"] + (1 << 17)


@pytest.mark.parametrize("dtype,compute", [(torch.float32, torch.float16), (torch.bfloat16, torch.bfloat16)], ids=["f32", "bf16"])
def test_autocast_calls_the_projections_themselves(gpu, monkeypatch, dtype, compute):
    # Under autocast torch decides what type a product runs in: neither the split products nor the one wide product may
    # stand in for the modules' calls.
    monkeypatch.setattr(SSM, "_BATCHED_PROJECTION_LIMIT", 0)
    monkeypatch.setattr(layers.split_linear, "MIN_WORK", 1)
    torch.manual_seed(2)
    layer = SSM(256, 2, dtype=dtype, device=gpu, compute_dtype=compute)
    x = torch.randn(2, 150, 256, device=gpu, dtype=dtype, requires_grad=True)
    dy = torch.randn_like(x)

    def step():
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y = layer(x)
            return [y.detach(), *torch.autograd.grad(y, [x, *layer.parameters()], dy.to(y.dtype))]

    def refuse(*a, **k):
        raise AssertionError("not under autocast")

    calls = []
    handles = [m.register_forward_hook(lambda *a: calls.append(1)) for m in layer._projections(False)[0]]
    want = step()
    for h in handles:
        h.remove()
    assert len(calls) == 5
    monkeypatch.setattr(layers.split_linear, "forward", refuse)
    monkeypatch.setattr(layers._WideProjections, "apply", refuse)
    for got, ref in zip(step(), want):
        assert got.dtype == ref.dtype and torch.equal(got, ref)
