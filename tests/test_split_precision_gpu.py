"""The split products keep fp32's precision element by element, whatever else is in a row, a column or a batch."""
import pytest
import torch

from quick_ssm_amd import split_linear

pytestmark = pytest.mark.gpu

ROWS, K, N = 700, 256, 260


def _few(n):
    def make(u, w, g, gen):
        keep = torch.rand(u.shape, generator=gen, device=u.device).argsort(1) < n
        return u * keep, w, g
    return make


def _loud_feature(p, weight):
    """One feature 2^p above the others, its weight 0 or as far below."""
    def make(u, w, g, gen):
        u, w = u.clone(), w.clone()
        u[:, 5] *= 2.0 ** p
        w[:, 5] *= 2.0 ** -p if weight else 0.0
        return u, w, g
    return make


def _loud_token(p):
    """One token's gradient 2^p above the others, its input 0."""
    def make(u, w, g, gen):
        u, g = u.clone(), g.clone()
        g[7] *= 2.0 ** p
        u[7] = 0.0
        return u, w, g
    return make


def _spread(u, w, g, gen):
    wide = lambda t: t * torch.exp(torch.empty_like(t).normal_(generator=gen) * 6)  # noqa: E731
    return wide(u), wide(w), wide(g)


CASES = {
    "dense": lambda u, w, g, gen: (u, w, g),
    **{f"{n} nonzeros": _few(n) for n in (1, 2, 4, 16)},
    **{f"loud feature 2^{p}": _loud_feature(p, False) for p in (20, 40, 100)},
    **{f"raw feature 2^{p}": _loud_feature(p, True) for p in (20, 40, 100)},
    **{f"loud token 2^{p}": _loud_token(p) for p in (26, 60)},
    "spread": _spread,
    "small": lambda u, w, g, gen: (u * 2.0 ** -120, w * 2.0 ** 20, g * 2.0 ** 20),
    "subnormal": lambda u, w, g, gen: (u * 2.0 ** -132, w * 2.0 ** 30, g * 2.0 ** 30),
}


def _inputs(gpu, seed=3):
    gen = torch.Generator(device=gpu).manual_seed(seed)
    new = lambda *s: torch.empty(*s, device=gpu).normal_(generator=gen)  # noqa: E731
    return new(ROWS, K), new(N, K), new(ROWS, N), gen


@pytest.mark.parametrize("case", CASES)
def test_every_element_is_as_close_as_fp32_sums_are(gpu, case):
    u, w, g, gen = _inputs(gpu)
    u, w, g = CASES[case](u, w, g, gen)
    (y,), saved = split_linear.forward(u, [w], [None], True, True)
    du, (dw,) = split_linear.backward([g], u, [w], saved, True, True)
    for name, got, a, b in (("y", y, u, w.t()), ("du", du, g, w), ("dw", dw, g.t(), u)):
        a64, b64 = a.double(), b.double().contiguous()
        ref, size = a64 @ b64, a64.abs() @ b64.abs()
        # k products of 2^-24 each at most for what is left out of them, and k sums rounded at 2^-24 of the size so far;
        # results below fp32's normal numbers at half of their spacing
        k = a.shape[1]
        error = (got.double() - ref).abs()
        assert bool((error <= 2.0 ** -24 * (k + 1) * size + 2.0 ** -150).all()), (case, name)
        # and in the mean no further off than the library's fp32 product.  Each element relative to its own sum of
        # magnitudes: the norm of the "spread" matrix is that of its one largest element, whose last bit is chance.  The
        # 5 %: a sum of one pair is rounded once by fp32, here after the sum of its parts (2 %), and 67600 elements' mean
        # square has a standard error of 1 %.
        some = size > 2.0 ** -110
        mean = lambda e: (e[some] / size[some]).pow(2).mean().sqrt().item()  # noqa: E731
        ours, lib = mean(error), mean(((a @ b.contiguous()).double() - ref).abs())
        print(f"{case} {name}: {ours:.2e}, library {lib:.2e}")
        assert ours <= 1.05 * lib, (case, name)


def test_a_row_with_a_single_one_picks_the_weights_exactly(gpu):
    u, w, g, gen = _inputs(gpu)
    pick = torch.randint(K, (ROWS,), generator=gen, device=gpu)
    one = torch.zeros_like(u)
    one[torch.arange(ROWS, device=gpu), pick] = 1.0
    (y,), saved = split_linear.forward(one, [w], [None], True, True)
    assert torch.equal(y, w.t()[pick])
    one = torch.zeros_like(g)
    one[torch.arange(ROWS, device=gpu), pick % N] = -2.0
    du, _ = split_linear.backward([one], u, [w], saved, True, False)
    assert torch.equal(du, -2.0 * w[pick % N])


def test_numbers_beyond_bf16_in_a_product_of_several_parts(gpu):
    # 20000 rows summed in parts (split over workgroups); one of them holds an infinity, one a number no bf16 value
    # holds, one numbers whose product overflows.
    gen = torch.Generator(device=gpu).manual_seed(5)
    u = torch.empty(20000, 64, device=gpu).normal_(generator=gen)
    g = torch.empty(20000, 132, device=gpu).normal_(generator=gen)
    w = torch.empty(132, 64, device=gpu).normal_(generator=gen)
    u[17, 3], u[9000, 40], u[15000, 9], g[15000, 100] = float("inf"), 3.4e38, 2.0 ** 100, -2.0 ** 60
    g[9000] = 0.0
    g[9000, 7] = 1e-3
    _, (dw,) = split_linear.backward([g], u, [w], None, False, True)
    ref = g.double().t() @ u.double()
    for column in (3, 40, 9):
        for row in (7, 8, 100, 131):
            want = ref[row, column].float()
            if torch.isfinite(want):
                assert (dw[row, column] - want).abs() <= 2.0 ** -24 * 20001 * (g[:, row].double().abs() @ u[:, column].double().abs())
            else:
                assert torch.equal(dw[row, column], want), (row, column)
    rest = [k for k in range(64) if k not in (3, 40, 9)]
    assert (dw[:, rest].double() - ref[:, rest]).norm() <= 2e-6 * ref[:, rest].norm()
