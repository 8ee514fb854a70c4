"""The layer's own weight gradients: the kernel at the edges of its tiles, stages and parts, and the rule that calls it."""
import ctypes

import pytest
import torch

from quick_ssm_amd import SSM, _lib, hip_scan, layers

pytestmark = pytest.mark.gpu


class _Counted:
    """The native module, with the weight gradients counted that it computes."""

    def __init__(self, native):
        self.native, self.taken = native, 0

    def __getattr__(self, name):
        return getattr(self.native, name)

    def weight_gradient(self, g, u):
        dw = self.native.weight_gradient(g, u)
        self.taken += dw is not None
        return dw


def _launch(a, b, pad=0):
    (K, M), N = a.shape, b.shape[1]
    lib = _lib.load()
    lib.qssm_weight_gradient_floats.restype = ctypes.c_uint64
    floats = lib.qssm_weight_gradient_floats(M, N, K)
    partial = torch.full((max(floats, 1),), float("nan"), device=a.device)
    c = torch.full((M, N + pad), 7.0, device=a.device, dtype=a.dtype)
    p = ctypes.c_void_p
    _lib.check(lib.qssm_weight_gradient(
        p(a.data_ptr()), ctypes.c_int64(a.stride(0)), p(b.data_ptr()), ctypes.c_int64(b.stride(0)), p(c.data_ptr()),
        ctypes.c_int64(N + pad), M, N, K, _lib.QSSM_BF16 if a.dtype == torch.bfloat16 else _lib.QSSM_F16, p(partial.data_ptr()),
        ctypes.c_uint64(floats), p(torch.cuda.current_stream().cuda_stream)))
    torch.cuda.synchronize()
    assert bool((c[:, N:] == 7.0).all())
    return c[:, :N]


# tiles are 256 x 256, stages 64 rows, at least four to a part: one piece of 8 columns below, on and above the edges
SHAPES = [(8, 8, 1), (256, 256, 64), (248, 264, 63), (264, 248, 65), (256, 512, 511), (520, 256, 1000), (1024, 1024, 4096),
          (264, 1032, 20000), (4200, 3000, 600)]


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=str)
def test_edges_match_float64(gpu, M, N, K, dtype):
    gen = torch.Generator(device=gpu).manual_seed(M + K)
    a, b = (torch.empty(K, n + 16, device=gpu).normal_(generator=gen).to(dtype)[:, 8:8 + n] for n in (M, N))
    got = _launch(a, b, pad=8)
    ref = a.double().t().contiguous() @ b.double()
    size = a.double().abs().t().contiguous() @ b.double().abs()
    # K sums and the parts' sums in fp32, one rounding to 8 or 11 significant bits, i.e. by at most 2^-8 or 2^-11 of the
    # value (fp16: of numbers down to its subnormals)
    unit = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    assert bool(((got.double() - ref).abs() <= unit * 1.01 * ref.abs() + 2.0 ** -24 * (K + 64) * size + 2.0 ** -25).all())
    assert torch.equal(got, _launch(a, b, pad=8))


def test_infinities_and_nan_stay_where_they_belong(gpu):
    gen = torch.Generator(device=gpu).manual_seed(3)
    a, b = (torch.empty(1090, n, device=gpu).normal_(generator=gen).bfloat16() for n in (264, 520))
    a[1089, 5], b[1088, 9], a[3, 263], b[3, 519] = float("inf"), float("nan"), float("-inf"), 0.0   # -inf x 0: NaN
    got, ref = _launch(a, b), a.float().t().contiguous() @ b.float()
    assert torch.equal(torch.isnan(got), torch.isnan(ref)) and torch.equal(torch.isposinf(got), torch.isposinf(ref))
    assert torch.equal(torch.isneginf(got), torch.isneginf(ref))


@pytest.mark.parametrize("params,compute,rows", [(torch.bfloat16, torch.bfloat16, 8192), (torch.float16, torch.float16, 8200),
                                                 (torch.float32, torch.bfloat16, 8192)], ids=str)
def test_a_layer_takes_them_and_nothing_else_changes(gpu, monkeypatch, params, compute, rows):
    native = hip_scan._native or hip_scan._load_native()
    counted = _Counted(native)
    monkeypatch.setattr(hip_scan, "_native", counted)
    torch.manual_seed(0)
    layer = SSM(128, 2, device=gpu, dtype=params, compute_dtype=compute)
    x = torch.randn(8, rows // 8, 128, device=gpu, dtype=params, requires_grad=True)
    dy = torch.randn_like(x)

    def step():
        counted.taken = 0
        return torch.autograd.grad(layer(x), [x, *layer.parameters()], dy)

    got = step()
    assert counted.taken == 2   # the five projections' and out_proj's
    monkeypatch.setattr(layers, "_GRADIENT_ROWS", 1 << 40)
    monkeypatch.setattr(layers, "_GRADIENT_WORK", 1 << 60)
    want = step()
    assert counted.taken == 0
    for (name, _), g, w in zip([("x", x), *layer.named_parameters()], got, want):
        if name.endswith("weight") and "norm" not in name:
            assert g.dtype == w.dtype and (g.double() - w.double()).norm() <= (2e-6 if params == torch.float32 else 4e-3) * w.double().norm()
        else:
            assert torch.equal(g, w), name
    u, g = x.detach().reshape(-1, 128), dy.reshape(-1, 128)
    assert native.weight_gradient(g, u) is not None
    # what the kernel does not take goes to the library
    assert native.weight_gradient(g[:, :100], u) is None or params == torch.float32
    assert native.weight_gradient(g.t().contiguous().t(), u) is None
    assert native.weight_gradient(g[:1].expand(rows, 128), u) is None
    assert native.weight_gradient(g, u.double()) is None
    if params != torch.float32:
        assert native.weight_gradient(g[:4096], u[:4096]) is None


@pytest.mark.parametrize("n,k,taken", [(16, 16, False), (400, 16, False), (16, 400, False), (20, 20, True), (100, 20, True), (64, 64, True)])
def test_narrow_fp32_gradients(gpu, monkeypatch, n, k, taken):
    counted = _Counted(hip_scan._native or hip_scan._load_native())
    monkeypatch.setattr(hip_scan, "_native", counted)
    gen = torch.Generator(device=gpu).manual_seed(n)
    rows = 40000
    g, u = (torch.empty(rows, c, device=gpu).normal_(generator=gen) for c in (n, k))
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    with torch.no_grad():
        got = layers._weight_gradient(g, u)
    assert counted.taken == taken
    if taken:   # the operand's copy (twice the operands at most) and sums of up to 64 parts
        assert torch.cuda.max_memory_allocated() - before <= 2 * 4 * rows * (n + k) + 65 * 4 * n * k + (1 << 20)
    ref, size = g.double().t().contiguous() @ u.double(), g.double().abs().t().contiguous() @ u.double().abs()
    assert bool(((got.double() - ref).abs() <= 2.0 ** -24 * (2 * rows + 8) * size).all())


@pytest.mark.parametrize("rows,n,k,taken", [(64, 8200, 8200, 0), (120, 6400, 6400, 0), (128, 6144, 6144, 1), (512, 4096, 2048, 0),
                                            (512, 4096, 2052, 1)])
def test_fp32_gradients_of_few_rows(gpu, monkeypatch, rows, n, k, taken):
    counted = _Counted(hip_scan._native or hip_scan._load_native())
    monkeypatch.setattr(hip_scan, "_native", counted)
    gen = torch.Generator(device=gpu).manual_seed(rows)
    g, u = (torch.empty(rows, c, device=gpu).normal_(generator=gen) for c in (n, k))
    with torch.no_grad():
        got = layers._weight_gradient(g, u)
    assert counted.taken == taken and got.shape == (n, k)
    ref, size = g[:, :64].double().t() @ u.double(), g[:, :64].double().abs().t() @ u.double().abs()
    assert bool(((got[:64].double() - ref).abs() <= 2.0 ** -24 * (2 * rows + 8) * size).all())
