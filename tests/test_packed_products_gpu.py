"""fp32 products with one operand packed: the edges of its tiles and stages, either operand packed, and the launch without
scratch, all through the C ABI."""
import ctypes

import pytest
import torch

from quick_ssm_amd import _lib
from tests.test_split_linear_host import _Call

pytestmark = pytest.mark.gpu


def _call(a, b, c, bias, M, N, K, a_ks, b_ks, segments=1):
    call = _Call(M=M, N=N, K=K, lda=a[0].stride(0), ldb=b[0].stride(0), ldc=c[0].stride(0), batch=len(c),
                 segments=segments, splits=1, a_kstrided=a_ks, b_kstrided=b_ks)
    for field, tensors in (("a", a), ("b", b), ("c", c), ("bias", bias)):
        for i, t in enumerate(tensors):
            getattr(call, field)[i] = t.data_ptr()
    return call


def _run(call, packed, splits, gpu):
    lib = _lib.load()
    for fn in (lib.qssm_gemm_f32, lib.qssm_gemm_f32_packed, lib.qssm_gemm_f32_packed_plan):
        fn.restype = ctypes.c_int
    nbytes = ctypes.c_uint64()
    _lib.check(lib.qssm_gemm_f32_packed_plan(ctypes.byref(call), ctypes.byref(nbytes)))
    if splits:
        call.splits = splits
    partial = torch.empty(call.splits * call.batch * call.M * call.N, device=gpu)
    call.partial, call.partial_floats = partial.data_ptr(), partial.numel()
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    if packed:
        # (the plan names no bytes for products this small; this is what either operand takes at most)
        most = -(-max(call.M, call.N) // 256) * max(call.batch, call.segments) * -(-call.K // 32) * 49152
        assert nbytes.value <= most
        scratch = torch.empty(most, dtype=torch.uint8, device=gpu)
        _lib.check(lib.qssm_gemm_f32_packed(ctypes.byref(call), ctypes.c_void_p(scratch.data_ptr()), ctypes.c_uint64(most), stream))
    else:
        _lib.check(lib.qssm_gemm_f32(ctypes.byref(call), stream))
    torch.cuda.synchronize()


# tiles of 128 x 256 and stages of 32: one below, on and above the edges; N > M packs A instead of B (each with whole and with
# ragged stages)
SHAPES = [(128, 256, 32), (129, 260, 36), (127, 252, 28), (384, 64, 64), (64, 384, 96), (1, 4, 4), (300, 1024, 260), (260, 512, 31),
          (384, 64, 44), (640, 260, 99)]


@pytest.mark.parametrize("packed", [True, False])
@pytest.mark.parametrize("kind", ["outputs", "input gradient", "weight gradients", "one input"])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_edges_match_float64(gpu, M, N, K, kind, packed):
    if kind != "weight gradients":
        K = -(-K // 4) * 4
    gen = torch.Generator(device=gpu).manual_seed(M + N)
    pad4 = lambda n: -(-n // 4) * 4  # noqa: E731

    def new(rows, cols):   # rows that are not next to each other
        return torch.empty(rows, pad4(cols) + 8, device=gpu).normal_(generator=gen)[:, :cols]

    many = 1 if kind == "outputs" else 3
    a_ks, b_ks = kind == "weight gradients", kind in ("input gradient", "weight gradients")
    a = [new(K, M) if a_ks else new(M, K) for _ in range(1 if kind == "one input" else many)] * (many if kind == "one input" else 1)
    b = [new(K, N) if b_ks else new(N, K) for _ in range(many)]
    segments = many if kind == "input gradient" else 1
    c = [torch.full((M, N + 4), 7.0, device=gpu) for _ in range(many if segments == 1 else 1)]
    bias = [torch.randn(N, device=gpu, generator=gen)] if kind == "outputs" else []
    pairs = [((x.t() if a_ks else x).double(), (y.t() if b_ks else y).double()) for x, y in zip(a, b)]
    refs, sizes = [[p @ q.t().contiguous() for p, q in pairs], [p.abs() @ q.abs().t().contiguous() for p, q in pairs]]
    if segments > 1:
        refs, sizes = [sum(refs)], [sum(sizes)]
    for splits in (0, 2, 5):
        _run(_call(a, b, c, bias, M, N, K, a_ks, b_ks, segments), packed, splits, gpu)
        for i, t in enumerate(c):
            got, ref, size = t[:, :N].double(), refs[i], sizes[i]
            if i < len(bias):
                ref, size = ref + bias[i].double(), size + bias[i].double().abs()
            # k products with 2^-24 each left out of them at most, k sums rounded at 2^-24 of the size so far, the parts'
            # sums and the bias
            assert bool(((got - ref).abs() <= 2.0 ** -24 * (2 * segments * K + 8) * size).all()), (splits, i)
            assert bool((t[:, N:] == 7.0).all())


@pytest.mark.parametrize("value", [float("inf"), float("nan"), 3e38])
def test_what_bf16_does_not_hold_ends_as_fp32_does_in_either_operand(gpu, value):
    gen = torch.Generator(device=gpu).manual_seed(1)
    for M, N in ((300, 520), (520, 300)):   # A packed, B packed
        for which in range(2):
            a, b = (torch.empty(n, 64, device=gpu).normal_(generator=gen) for n in (M, N))
            (a, b)[which][70, 9] = value
            c = torch.empty(M, N, device=gpu)
            _run(_call([a], [b], [c], [], M, N, 64, False, False), True, 0, gpu)
            ref = a @ b.t()
            assert torch.equal(torch.isnan(c), torch.isnan(ref)) and torch.equal(torch.isinf(c), torch.isinf(ref))
            fine = torch.isfinite(ref)
            size = (a.abs().double() @ b.abs().double().t().contiguous())[fine]
            assert bool(((c.double() - a.double() @ b.double().t().contiguous())[fine].abs() <= 2.0 ** -24 * 65 * size).all())
