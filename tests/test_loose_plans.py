"""Plans for rows that are not aligned to, or not divided by, the lanes' width (qssm_plan_scan_loose)."""
import ctypes

import numpy as np
import pytest
import torch

from helpers import TOL, assert_close, make_inputs, oracle_all
from quick_ssm_amd import _lib, hip_scan, scan, scan_chunk


def _plan(B, L, D, dtype, out_dtype, direction, align, stride=0):
    code = {torch.float32: 0, torch.float16: 1, torch.bfloat16: 2}
    p = _lib.Plan()
    lib = _lib.load()
    _lib.check(lib.qssm_plan_scan_loose(B, L, D, code[dtype], code[out_dtype], direction, align, stride, 0, ctypes.byref(p)))
    return p


@pytest.mark.parametrize("D", [1, 3, 31, 32, 33, 34, 36, 63, 65, 127, 129, 255, 257, 258, 511, 513, 777, 1000, 1027, 4095])
def test_every_column_is_covered_and_nothing_beyond_the_rows(D):
    for dtype, out in ((torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32)):
        for align in (1, 2, 4, 8):
            if align > 1 and D % align:
                continue
            for B, L in ((1, 1), (2, 300), (1, 5000), (4, 2048)):
                back = _plan(B, L, D, dtype, out, _lib.QSSM_BACKWARD, align)
                ahead = _plan(B, L, D, dtype, out, _lib.QSSM_FORWARD, align, back.seg_len)
                assert ahead.n_ckpt == back.n_ckpt
                for p, direction in ((back, _lib.QSSM_BACKWARD), (ahead, _lib.QSSM_FORWARD)):
                    tight = hip_scan.make_plan(B, L, D, dtype, out, direction, align, p.ckpt_stride if p is ahead else 0)
                    if not p.element_aligned:   # the same plan as without the freedom
                        assert p.describe() == tight.describe()
                        assert D % p.vec == 0 and align % p.vec == 0
                        continue
                    assert D >= 32 and p.vec > tight.vec and p.vec <= 4
                    lanes = np.arange(p.n_strips * (1 << p.g_log2)) * p.vec
                    first = np.minimum(lanes[lanes < D], D - p.vec)
                    assert first.min() >= 0 and set((first[:, None] + np.arange(p.vec)).ravel()) == set(range(D))
                    # a tile's base and a lane's offset from it are both non-negative
                    strip = np.minimum(lanes[lanes < D] // p.strip_cols * p.strip_cols, D - p.vec)
                    assert (first >= strip).all()


def test_loose_plans_describe_launches_that_stay_in_bounds():
    # What the sweeps over strict plans check, for the plans that scan() launches: geometry, buffer sizes, and every
    # lane's elements, saved states and words.
    import random

    from test_host_logic import _tile_accesses

    rng = random.Random(77)
    pairs = [(torch.float32, torch.float32), (torch.float16, torch.float16), (torch.bfloat16, torch.bfloat16),
             (torch.float16, torch.float32), (torch.bfloat16, torch.float32)]
    loose = 0
    for _ in range(150):
        B, L = rng.choice([1, 2, 3]), rng.choice([1, 5, 31, 33, 64, 127, 200, 513, 1030])
        D = rng.choice([1, 3, 31, 32, 33, 34, 47, 63, 65, 77, 130, 255, 258, 333, 514, 777])
        dt, odt = rng.choice(pairs)
        align = rng.choice([a for a in (1, 2, 4, 8) if a == 1 or D % a == 0])
        tune = rng.choice([0, 0, 4, 6, 8]) | (rng.choice([0, 4, 8]) << 8) | (rng.choice([0, 1, 3]) << 28)
        try:
            bwd = hip_scan.make_plan(B, L, D, dt, odt, _lib.QSSM_BACKWARD, align, 0, tune, loose=True)
            fwd = hip_scan.make_plan(B, L, D, dt, odt, _lib.QSSM_FORWARD, align, bwd.seg_len, loose=True)
        except Exception as exc:   # a forced geometry the planner refuses is fine; anything else is not
            assert tune and ("LDS" in str(exc) or "ckpt_stride" in str(exc)), (B, L, D, dt, odt, align, tune, str(exc))
            continue
        for p in (bwd, fwd):
            what = (B, L, D, dt, odt, align, tune, p.describe())
            loose += p.element_aligned
            assert p.vec <= D and (p.element_aligned or (D % p.vec == 0 and align % p.vec == 0)), what
            assert p.seg_len == p.steps * (p.threads >> p.g_log2) and p.seg_len % p.ckpt_stride == 0, what
            assert p.n_strips == -(-D // p.strip_cols) and p.n_seg == -(-L // p.seg_len), what
            assert 0 < p.lds_bytes <= 64 * 1024, what
            assert p.ckpt_elems == B * p.n_ckpt * D and p.n_ckpt == -(-L // p.ckpt_stride), what
            lo, hi, hi_ckpt, hi_word = _tile_accesses(p, B, L, D)
            assert lo >= 0 and hi == B * L * D - 1, what
            assert hi_ckpt < p.ckpt_elems and hi_word <= p.workspace_bytes, what
        assert fwd.ckpt_stride == bwd.ckpt_stride == bwd.seg_len
    assert loose >= 80


def test_a_misaligned_backward_reads_the_states_of_a_gated_forward():
    # The gated scan's two-pass backward takes y's gradient as autograd hands it over, one element off alignment if it
    # must be: a loose plan that meets the spacing the gated forward saved its states with.
    from quick_ssm_amd import gated_scan

    for dtype, compute, out in ((torch.bfloat16, torch.bfloat16, torch.float32), (torch.float16, torch.float16, torch.float32),
                                (torch.float32, torch.float16, torch.float32), (torch.float32, torch.float32, torch.float32)):
        for B in (1, 3, 16):
            for L in (1, 2, 5, 6, 7, 9, 17, 33, 100, 1000, 4096, 65536):
                for S in (128, 132, 136, 264, 688, 1008, 1024, 4096):
                    stride = gated_scan._plan(B, L, S, dtype, compute, dtype, _lib.QSSM_BACKWARD, 0).seg_len
                    for align in (1, 2, 4, 8):
                        p = hip_scan.make_plan(B, L, S, compute, out, _lib.QSSM_BACKWARD, align, stride, loose=True)
                        assert p.ckpt_stride == stride and p.seg_len % stride == 0, (B, L, S, dtype, compute, align)


SHAPES = [(2, 300, 33), (3, 100, 35), (2, 1100, 257), (1, 700, 258), (2, 513, 777), (1, 5000, 61), (64, 1, 1027)]


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("dtypes", [(torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32)],
                         ids=["f32", "bf16", "f16-f32"])
@pytest.mark.parametrize("shift", [0, 1], ids=["dense", "shifted"])
def test_scan_and_gradients_match_the_oracle(gpu, shape, dtypes, shift):
    dtype, out = dtypes
    x, a, b, c, dy = make_inputs(shape, dtype=dtype, seed=sum(shape), out_dtype=out)
    ref = oracle_all(x, a, b, c, dy)

    def place(t):
        """On the GPU, its rows starting one element into wider ones when `shift`."""
        if not shift:
            return t.to(gpu)
        wide = torch.full((*t.shape[:2], t.shape[2] + 3), float("nan"), dtype=t.dtype, device=gpu)
        view = wide[..., 1:1 + t.shape[2]]
        view.copy_(t)
        return view

    for checkpoint in (True, False):
        leaves = [place(t).requires_grad_(True) for t in (x, a, b, c)]
        y = scan(*leaves, checkpoint=checkpoint, out_dtype=out)
        grads = torch.autograd.grad(y, leaves, place(dy))
        assert hip_scan.workspace_status() == 0
        assert_close("y", y.detach().cpu(), ref["y"], TOL[out])
        for name, g in zip(("dx", "da", "db", "dc"), grads):
            assert_close(name, g.cpu(), ref[name], TOL[dtype])


@pytest.mark.gpu
def test_states_cross_pieces_of_odd_rows(gpu):
    x, a, b, c, dy = (t.to(gpu) for t in make_inputs((2, 900, 333), seed=4))
    whole = [t.clone().requires_grad_(True) for t in (x, a, b, c)]
    parts = [t.clone().requires_grad_(True) for t in (x, a, b, c)]
    y = scan(*whole)
    ys, state = [], torch.zeros(2, 333, device=gpu)
    for lo, hi in ((0, 101), (101, 500), (500, 900)):
        piece, state = scan_chunk(*(t[:, lo:hi] for t in parts), state)
        ys.append(piece)
    for got, want in zip((torch.cat(ys, 1), *torch.autograd.grad(torch.cat(ys, 1), parts, dy)),
                         (y, *torch.autograd.grad(y, whole, dy))):
        assert_close("piecewise", got.detach().cpu(), want.detach().cpu().numpy(), 1e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(64, 1, 1027), (3, 40, 333), (2, 900, 515)], ids=lambda s: "x".join(map(str, s)))
def test_a_state_carried_in_place_is_read_before_it_is_written(gpu, shape):
    # Two lanes share columns of a row, and a chain's last tile writes the state that its first ones read.
    x, a, b, c, dy = (t.to(gpu) for t in make_inputs(shape, seed=9))
    state = torch.randn(shape[0], shape[2], generator=torch.Generator().manual_seed(1)).to(gpu)
    want = torch.empty_like(state)
    y, _, ckpt, stride = hip_scan.scan_forward(x, a, b, c, out_dtype=torch.float32, want_ckpt=True, h_init=state, h_final=want)
    for _ in range(20):
        moved = state.clone()
        again = hip_scan.scan_forward(x, a, b, c, out_dtype=torch.float32, h_init=moved, h_final=moved)[0]
        assert torch.equal(again, y) and torch.equal(moved, want)
    grad, out = torch.randn_like(state), torch.empty_like(state)
    args = dict(ckpt=ckpt, ckpt_stride=stride, h_init=state)
    want = hip_scan.scan_backward(x, a, b, c, dy, dh_final=grad, dh_init=out, **args)
    for _ in range(20):
        moved = grad.clone()
        got = hip_scan.scan_backward(x, a, b, c, dy, dh_final=moved, dh_init=moved, **args)
        assert torch.equal(moved, out) and all(torch.equal(g, w) for g, w in zip(got, want))
    assert hip_scan.workspace_status() == 0
