"""The native autograd node of scan() and scan_chunk(): what autograd promises beyond the values of the gradients."""
import pytest
import torch

from helpers import TOL, assert_close, make_inputs, oracle_all
from quick_ssm_amd import hip_scan, scan, scan_chunk

pytestmark = pytest.mark.gpu


def test_a_graph_is_walked_once_unless_kept_and_frees_what_it_saved(gpu):
    x, a, b, c, dy = make_inputs((2, 300, 24), seed=5)
    ref = oracle_all(x, a, b, c, dy)
    leaves = [t.to(gpu).requires_grad_(True) for t in (x, a, b, c)]
    y = scan(*leaves, checkpoint=False)
    first = torch.autograd.grad(y, leaves, dy.to(gpu), retain_graph=True)
    second = torch.autograd.grad(y, leaves, dy.to(gpu))
    for name, g1, g2 in zip(("dx", "da", "db", "dc"), first, second):
        assert torch.equal(g1, g2), name
        assert_close(name, g1.cpu(), ref[name], TOL[torch.float32])
    assert y.grad_fn.h_saved is None
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(y, leaves, dy.to(gpu))
    y = scan(*leaves)
    with torch.no_grad():
        leaves[1].mul_(0.5)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.backward(dy.to(gpu))


@pytest.mark.parametrize("used", ["y", "state", "both"])
@pytest.mark.parametrize("dtypes", [(torch.float32,) * 4, (torch.float16, torch.float32, torch.bfloat16, torch.float64)],
                         ids=["f32", "mixed"])
def test_either_output_of_a_piece_may_go_unused(gpu, used, dtypes):
    x, a, b, c, dy = make_inputs((3, 90, 20), seed=8)
    st, dst = torch.randn(3, 20, generator=torch.Generator().manual_seed(1)), torch.ones(3, 20)
    ops = [t.to(d) for t, d in zip((x, a, b, c), dtypes)] + [st.half() if dtypes[0] != torch.float32 else st]

    def grads(backend, device):
        leaves = [t.to(device).requires_grad_(True) for t in ops]
        ins = leaves if backend == "hip" else [t.double() for t in leaves]
        y, h = scan_chunk(*ins, out_dtype=torch.float32 if backend == "hip" else torch.float64, backend=backend)
        loss = 0.0
        if used != "state":
            loss = loss + (y * dy.to(y)).sum()
        if used != "y":
            loss = loss + (h * dst.to(h)).sum()
        return torch.autograd.grad(loss, leaves, allow_unused=True)

    for name, got, want in zip(("dx", "da", "db", "dc", "dstate"), grads("hip", gpu), grads("torch", "cpu")):
        if want is None:          # c when only the state is used
            assert got is None or not bool(got.any()), name
            continue
        assert got.dtype == want.dtype, name
        # float32 arithmetic, one rounding to the operand's own type
        assert_close(name, got.cpu().float(), want.float().numpy(), max(1e-5, torch.finfo(got.dtype).eps))
    assert hip_scan.workspace_status() == 0


class _NoGradient(torch.autograd.Function):
    @staticmethod
    def forward(ctx, t):
        return t * 2

    @staticmethod
    def backward(ctx, g):
        return None


def test_no_gradient_from_a_function_behind_the_scan_is_a_gradient_of_zeros(gpu):
    x, a, b, c, _ = make_inputs((2, 70, 24), seed=6)
    leaves = [t.to(gpu).requires_grad_(True) for t in (x, a, b, c, torch.ones(2, 24))]
    y, h = scan_chunk(*leaves)
    (_NoGradient.apply(scan(*leaves[:4])).sum() + _NoGradient.apply(y).sum() + _NoGradient.apply(h).sum()).backward()
    for t in leaves:
        assert t.grad is not None and not bool(t.grad.any())


@pytest.mark.parametrize("out", [torch.int32, torch.bool], ids=str)
def test_an_output_of_a_type_without_gradients_is_returned_without_one(gpu, out):
    x, a, b, c, _ = make_inputs((2, 70, 24), seed=7)
    leaves = [(8 * t).to(gpu).requires_grad_(True) for t in (x, a / 8, b, c)]
    y = scan(*leaves, out_dtype=out)
    with torch.no_grad():
        want, final = scan_chunk(*leaves, out_dtype=out)
    assert y.dtype == out and not y.requires_grad and torch.equal(y, want)
    y, h = scan_chunk(*leaves, out_dtype=out)
    assert not y.requires_grad and torch.equal(y, want) and torch.equal(h, final)
    grads = torch.autograd.grad(h.sum(), leaves[:3])
    full, h = scan_chunk(*leaves)
    for got, ref in zip(grads, torch.autograd.grad(h.sum(), leaves[:3])):
        assert torch.equal(got, ref)


def test_a_trace_records_the_scan_instead_of_its_result(gpu):
    first, second = ([t.to(gpu) for t in make_inputs((2, 130, 24), seed=s)[:4]] for s in (1, 2))
    state = torch.randn(2, 24, generator=torch.Generator().manual_seed(3)).to(gpu)
    for fn, more in ((lambda x, a, b, c: scan(x, a, b, c), []),
                     (lambda x, a, b, c, h: scan_chunk(x, a, b, c, h)[0], [state])):
        traced = torch.jit.trace(fn, (*first, *more), check_trace=False)
        assert torch.equal(traced(*second, *more), fn(*second, *more))


def test_what_the_node_cannot_do_is_refused(gpu):
    import torch.autograd.forward_ad as fwd

    x, a, b, c = (t.to(gpu) for t in make_inputs((2, 30, 8), seed=1)[:4])
    calls = (lambda x: scan(x, a, b, c), lambda x: scan_chunk(x, a, b, c)[0])
    for fn in calls:
        with fwd.dual_level(), pytest.raises(RuntimeError):
            fn(fwd.make_dual(x, torch.ones_like(x)))
        with pytest.raises(RuntimeError):
            torch.func.grad(lambda x: fn(x).sum())(x)
        with pytest.raises(RuntimeError):
            torch.func.vmap(fn)(torch.stack([x, x]))
        assert torch.isfinite(fn(x)).all()


@pytest.mark.parametrize("dtype,compute", [(torch.bfloat16, torch.bfloat16), (torch.float32, torch.float16)], ids=str)
def test_a_wide_tensor_and_its_five_blocks_are_the_same_launch(gpu, dtype, compute):
    from quick_ssm_amd import gated_scan

    gen = torch.Generator(device=gpu).manual_seed(1)
    wide = torch.empty(2, 70, 5 * 136, device=gpu).normal_(generator=gen).to(dtype).requires_grad_(True)
    dy = torch.empty(2, 70, 136, device=gpu).normal_(generator=gen).to(dtype)
    blocks = [t.detach().contiguous().requires_grad_(True) for t in wide.split(136, 2)]
    assert gated_scan.supported_wide(wide, compute, dtype) and gated_scan.supported(blocks, compute, dtype)
    got = gated_scan.gated_scan_wide(wide, compute_dtype=compute)
    want = gated_scan.gated_scan(*blocks, compute_dtype=compute)
    assert torch.equal(got, want)
    (dwide,) = torch.autograd.grad(got, wide, dy)
    for a, b in zip(dwide.split(136, 2), torch.autograd.grad(want, blocks, dy)):
        assert torch.equal(a, b)
    # the two rules agree, block by block, on widths and rows that 16 bytes do not divide
    for width, at in ((128, 0), (132, 0), (136, 4), (136, 8), (124, 0)):
        odd = torch.empty(2, 5, 5 * width + 16, device=gpu, dtype=dtype)[..., at:at + 5 * width]
        five = [odd[..., k * width:(k + 1) * width] for k in range(5)]
        assert gated_scan.supported_wide(odd, compute, dtype) == gated_scan.supported(five, compute, dtype), (width, at)


def test_a_wide_tensor_that_is_more_than_five_blocks(gpu):
    # four columns behind the last block
    from quick_ssm_amd import gated_scan

    gen = torch.Generator(device=gpu).manual_seed(2)
    rows = torch.empty(2, 70, 684, device=gpu).normal_(generator=gen)
    wide, five = (rows[..., :n].detach().requires_grad_(True) for n in (684, 680))
    got, want = (gated_scan.gated_scan_wide(t, compute_dtype=torch.float16) for t in (wide, five))
    assert torch.equal(got, want)
    (dwide,), (dfive,) = torch.autograd.grad(got.sum(), wide), torch.autograd.grad(want.sum(), five)
    assert dwide.shape == wide.shape and torch.equal(dwide[..., :680], dfive) and not dwide[..., 680:].any()
    with pytest.raises(ValueError):
        gated_scan.gated_scan_wide(rows[0])
