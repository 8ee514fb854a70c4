"""Host side of the HIP scan: workspace, launch numbering, and the two launches.

Everything here and in csrc/torch_scan.cpp (output tensors, plans, the call itself) is plumbing around
`qssm_scan_forward` / `qssm_scan_backward` (include/quick_ssm_hip.h).  It takes the place of the launch code in the reference's
`block_scan_forward_3d` (quick_ssm/triton_forwards.py:134-172) and `block_scan_backward_3d`
(quick_ssm/triton_backwards.py:168-209): no fp32 upcast copies, no N-sized scratch, one launch per
direction.
"""
from __future__ import annotations

import ctypes
import os
import threading
from typing import Dict, List, Optional, Sequence, Tuple

import torch

from . import _lib
from ._lib import Plan

Tensor = torch.Tensor

_DTYPE_CODE = {torch.float32: _lib.QSSM_F32, torch.float16: _lib.QSSM_F16, torch.bfloat16: _lib.QSSM_BF16}
# (storage of x,a,b,c) -> storages of y the kernels are built for
_BUILT_OUT = {
    torch.float32: (torch.float32,),
    torch.float16: (torch.float16, torch.float32),
    torch.bfloat16: (torch.bfloat16, torch.float32),
}

_ws_lock = threading.Lock()
_EPOCH_MAX = 0xFFFFFFFF


class ScanLaunchError(RuntimeError):
    """A scan launch reported failure through its control block's status word.

    status 1: a tile gave up waiting for a neighbour's word (about a second); outputs downstream of it are NaN.
    status 2: a ticket counter was not zero when the launch started; every output of the launch is NaN.
    By the time this is raised the control block and workspace have been zero-filled again, so the next launch
    on the stream starts clean; results of launches since the last check must be discarded.
    """

    def __init__(self, status: int, where: str):
        super().__init__(
            f"quick_ssm_amd: a scan launch on {where} failed with status {status} "
            f"({'a tile gave up waiting for a neighbour' if status == 1 else 'the control block was not zero on entry' if status == 2 else 'both kinds of failure'}); "
            "its outputs are NaN. Control block and workspace have been reset; repeat the step.")
        self.status = status


def _env_int(name: str, default: int) -> int:
    try:
        return int(os.environ.get(name, default))
    except ValueError:
        return default


# Every `_check_every`-th launch on a pair of buffers is followed by an asynchronous copy of the status word to
# pinned host memory, looked at (without waiting) before each later launch: a failed launch is reported within two
# such periods.  QSSM_CHECK_STATUS=1 checks behind every launch, 0 never; set_status_check_period() at run time.
_check_every = _env_int("QSSM_CHECK_STATUS", 64)


def set_status_check_period(launches: int) -> int:
    """Look at the status word every `launches`-th launch (0: never).  Returns the old period."""
    global _check_every
    old, _check_every = _check_every, max(0, int(launches))
    return old


class _Buffers:
    """Per (device, stream, who numbers the launches): control block, workspace, the host's launch count, and the
    pinned word the status is copied to."""

    __slots__ = ("control", "workspace", "epoch", "ctl_ptr", "ctl_size", "ws_ptr", "ws_size", "captured",
                 "pinned", "seen", "since_check", "device", "where")

    def __init__(self, device: torch.device, where: str):
        self.control: Optional[Tensor] = None
        self.workspace: Optional[Tensor] = None
        self.epoch = 0
        self.ctl_ptr = self.ctl_size = self.ws_ptr = self.ws_size = 0
        self.captured = False          # a graph holds these addresses: never free or move them
        # The status word is copied here by a raw asynchronous copy that torch's pinned-memory allocator knows
        # nothing about: the block must never go back to it, or a copy still queued when the entry is dropped
        # would land in somebody else's tensor.  Four bytes per (device, stream) ever used.
        self.pinned = torch.zeros(1, dtype=torch.int32, pin_memory=True)
        _pinned_words.append(self.pinned)
        self.seen = ctypes.c_int32.from_address(self.pinned.data_ptr())
        self.since_check = 0
        self.device = device
        self.where = where


# One entry per (device, raw stream handle, device-counted) ever launched on.  Entries stay until reset_workspaces():
# a stream handle says nothing about whether its stream still exists, and an entry costs its control block and
# workspace (tens of MiB for large shapes), so a program that keeps making streams should call reset_workspaces()
# now and then.
_buffers: Dict[Tuple[int, int, bool], _Buffers] = {}
_pinned_words: List[Tensor] = []
# Buffers a recorded graph still points to, after they have been replaced by larger ones or dropped by
# reset_workspaces(): kept alive until the process ends, because replaying that graph writes to them.
_retired: List[Tensor] = []


def kernel_dtypes(in_dtypes: Sequence[torch.dtype], out_dtype: torch.dtype) -> Tuple[torch.dtype, torch.dtype]:
    """Storage types the launch will use for (x,a,b,c / grads) and for (y / dy).

    Arithmetic is fp32 in every case.  Operands of mixed or unsupported storage are cast to a
    common supported one on the host; an unsupported y storage is produced as fp32 and cast.
    """
    common = in_dtypes[0]
    for dt in in_dtypes[1:]:
        if dt != common:
            common = torch.promote_types(common, dt)
    if common not in _DTYPE_CODE:
        common = torch.float32
    k_out = out_dtype if out_dtype in _BUILT_OUT[common] else torch.float32
    return common, k_out


def _align_elems(tensors: Sequence[Optional[Tensor]], D: int) -> int:
    """Largest v in (8, 4, 2, 1) such that D, every stride and every base address (in elements) divide by v."""
    bits = D
    for t in tensors:
        if t is None:
            continue
        es = t.element_size()
        ptr = t.data_ptr()
        if ptr % es:
            return 1
        bits |= (ptr // es) | t.stride(0) | t.stride(1)
    low = bits & -bits
    return 8 if low == 0 or low > 8 else low


# (device index, stream handle) -> how many `device_counted_launches` contexts are open on it
_device_counted: Dict[Tuple[int, int], int] = {}


def _raw_stream(dev_index: int) -> int:
    return torch._C._cuda_getCurrentRawStream(dev_index)


class device_counted_launches:
    """Context manager: scan launches made on the stream that is current when it is entered, while it is open and
    from any thread (autograd runs the backward on its own, on the forward's stream), number themselves in their
    control block (epoch argument 0), as launches recorded into a graph do, and use the buffers kept for such
    launches.  Launches on other streams or devices are not affected.

    Launches being recorded into a graph do this by themselves, but cannot allocate: run the work once inside this
    context, on the stream that will capture, and the control block and workspace exist (large enough) when the
    capture starts.  Buffers a capture has used are never freed: if a later launch needs larger ones, new buffers
    take their place for new launches and the old ones stay alive for the graph that points to them.  Two graphs
    recorded on one stream share their buffers: replay them on that stream, one at a time.
    """

    def __enter__(self):
        index = torch.cuda.current_device()
        self._key = (index, _raw_stream(index))
        with _ws_lock:
            _device_counted[self._key] = _device_counted.get(self._key, 0) + 1
        return self

    def __exit__(self, *exc):
        with _ws_lock:
            left = _device_counted.get(self._key, 0) - 1
            if left > 0:
                _device_counted[self._key] = left
            else:
                _device_counted.pop(self._key, None)
        return False


def _grow_buffers(key: Tuple[int, int, bool], device: torch.device, need_c: int, need_w: int, capturing: bool) -> _Buffers:
    """Slow path of `_launch_buffers`: first use of a (device, stream), a larger shape, or a used-up numbering."""
    with _ws_lock:
        return _grow_buffers_locked(key, device, need_c, need_w, capturing)


def _grow_buffers_locked(key: Tuple[int, int, bool], device: torch.device, need_c: int, need_w: int, capturing: bool) -> _Buffers:
    """`_grow_buffers` for a caller that holds `_ws_lock`."""
    buf = _buffers.get(key)
    grow_c = buf is None or buf.control is None or buf.ctl_size < need_c
    grow_w = grow_c or buf.workspace is None or buf.ws_size < need_w or buf.epoch >= _EPOCH_MAX
    if capturing and grow_w:   # before anything is allocated: an allocation would spoil the recording
        raise RuntimeError(
            "quick_ssm_amd: a scan launch being recorded into a graph cannot allocate its control block and "
            "workspace; run the same work once inside `hip_scan.device_counted_launches()` on this stream first")
    if buf is None:
        buf = _Buffers(device, f"device {key[0]}, stream {key[1]:#x}")
    if buf.captured and grow_w:
        # a recorded graph points at the old pair: keep it alive and untouched, new launches get a new pair
        _retired.extend(t for t in (buf.control, buf.workspace) if t is not None)
        buf.captured = False
        grow_c = True
    if grow_c:
        # a new control block restarts the device-side count: the workspace must not keep words of the old numbering
        buf.control = torch.zeros(max(1 << 16, 1 << (need_c - 1).bit_length()), dtype=torch.uint8, device=device)
        buf.ctl_ptr, buf.ctl_size = buf.control.data_ptr(), buf.control.numel()
    if grow_w:
        buf.workspace = torch.zeros(max(1 << 20, 1 << (need_w - 1).bit_length()), dtype=torch.uint8, device=device)
        buf.ws_ptr, buf.ws_size = buf.workspace.data_ptr(), buf.workspace.numel()
        buf.epoch = 0
    _buffers[key] = buf
    return buf


def _recover(buf: _Buffers, stream: int) -> int:
    """Zero-fill a failed pair of buffers on `stream`, forget the host's numbering, and return the status seen."""
    lib = _lib.load()
    with torch.cuda.device(buf.device):
        _lib.check(lib.qssm_zero_fill(buf.ctl_ptr, buf.ctl_size, stream))
        _lib.check(lib.qssm_zero_fill(buf.ws_ptr, buf.ws_size, stream))
        out = ctypes.c_int32(0)
        _lib.check(lib.qssm_control_status(buf.ctl_ptr, stream, ctypes.byref(out)))   # waits: copies in flight have landed
    with _ws_lock:
        status = int(buf.seen.value)
        buf.seen.value = 0
        buf.epoch = 0
        buf.since_check = 0
    return status


# (entry, control block, workspace, their addresses and sizes in turn): what one launch works with.  The launch holds
# the two tensors until it is on its stream; the entry may have been given others by then.
_Taken = Tuple[_Buffers, Tensor, Tensor, int, int, int, int]


def _launch_buffers(device: torch.device, dev_index: int, stream: int, need_c: int, need_w: int) -> Tuple[_Taken, int, bool]:
    """Buffers and epoch argument of the next launch on (device, stream), and whether the stream is capturing.

    Both buffers are zero-filled when they are allocated (torch.zeros runs a fill kernel on the
    current stream, ahead of the launch that uses them) and grown on demand.  Every launch leaves
    the control block's status word and ticket counters zero.  The workspace is never cleared:
    every launch gets the next epoch.  Eager launches are numbered here.  Launches recorded into a
    graph (and those inside `device_counted_launches`) use a pair of buffers of their own and are
    numbered in the control block itself (epoch argument 0), so that replays number themselves, at
    the price of a one-lane counting kernel behind each launch.  A workspace that has to grow, or
    whose 32-bit host numbering is used up, is replaced by a fresh zeroed one.  A status word that an
    earlier check found nonzero raises ScanLaunchError here, after the buffers have been reset.
    """
    capturing = torch._C._cuda_isCurrentStreamCapturing()
    on_device = capturing or ((dev_index, stream) in _device_counted)
    key = (dev_index, stream, on_device)
    # Looking the buffers up and taking the next number is one step under the lock: the forward of the next step on
    # the caller's thread and a backward on autograd's thread may launch on one stream at the same time, and two
    # launches with one number would read each other's words as their own.  The addresses are read in the same step:
    # a larger launch on the other thread replaces the tensors, and a number only means something to its own buffers.
    # Callers pass on these addresses, never the entry's.
    with _ws_lock:
        buf = _buffers.get(key)
        if buf is None or buf.ctl_size < need_c or buf.ws_size < need_w or buf.epoch >= _EPOCH_MAX:
            buf = _grow_buffers_locked(key, device, need_c, max(need_w, 256), capturing)
        failed = buf.seen.value != 0 and not capturing
        epoch = 0
        if not failed:
            if capturing:
                buf.captured = True
            if not on_device:
                buf.epoch += 1
                epoch = buf.epoch
        taken = (buf, buf.control, buf.workspace, buf.ctl_ptr, buf.ctl_size, buf.ws_ptr, buf.ws_size)
    if failed:
        raise ScanLaunchError(_recover(buf, stream), buf.where)
    return taken, epoch, capturing


def _status_check_due(buf: _Buffers, capturing: bool) -> bool:
    """Counts a launch; True behind every `_check_every`-th."""
    if _check_every <= 0 or capturing:
        return False
    with _ws_lock:
        buf.since_check += 1
        due = buf.since_check >= _check_every
        if due:
            buf.since_check = 0
    return due


def _after_launch(taken: _Taken, stream: int, capturing: bool) -> None:
    """Every `_check_every`-th launch: ask for the status word, to be looked at before a later launch."""
    buf = taken[0]
    if _status_check_due(buf, capturing):
        _lib.check(_lib.load().qssm_control_status_async(taken[3], buf.pinned.data_ptr(), stream))


_devices: Dict[int, torch.device] = {}


def _take_launch(dev_index: int, stream: int, need_c: int, need_w: int) -> tuple:
    """What the native launches (csrc/torch_scan.cpp) ask for, from whatever thread they run on: the addresses and
    sizes of control block and workspace, the epoch argument, the pinned word the status is to be copied to behind this
    launch (0: not this time), and the two tensors, which the caller holds until the launch is on its stream."""
    device = _devices.get(dev_index)
    if device is None:
        device = _devices[dev_index] = torch.device("cuda", dev_index)
    (buf, control, workspace, cp, cs, wp, ws), epoch, capturing = _launch_buffers(device, dev_index, stream, need_c, need_w)
    status_to = buf.pinned.data_ptr() if _status_check_due(buf, capturing) else 0
    return cp, cs, wp, ws, epoch, status_to, control, workspace


def workspace_status(device: Optional[torch.device] = None, all_streams: bool = False) -> int:
    """Status words of the current stream's control blocks (of every stream of the device with `all_streams`),
    or-ed; synchronises those streams.  0 = all launches completed."""
    device = torch.device("cuda", torch.cuda.current_device()) if device is None else device
    index = device.index if device.index is not None else torch.cuda.current_device()
    stream = _raw_stream(index)
    with _ws_lock:
        bufs = [(k, b) for k, b in _buffers.items()
                if k[0] == index and (all_streams or k[1] == stream) and b.control is not None]
    status = 0
    for key, buf in bufs:
        out = ctypes.c_int32(0)
        with torch.cuda.device(device):
            _lib.check(_lib.load().qssm_control_status(buf.ctl_ptr, key[1], ctypes.byref(out)))
        status |= int(out.value)
    return status


def reset_workspaces() -> None:
    """Drop every cached buffer (the next launch allocates fresh zeroed ones).  Buffers that a recorded graph
    points to are not freed, but no later launch uses them: such graphs still replay, on their own old buffers."""
    with _ws_lock:
        for buf in _buffers.values():
            if buf.captured:
                _retired.extend(t for t in (buf.control, buf.workspace) if t is not None)
        _buffers.clear()


_plans: Dict[tuple, Plan] = {}
_forward_keep = True


def set_forward_keep(flag):
    """Whether forwards that save states for a backward (plain and gated) follow the planner's cache policy from now
    on (`plan.keep_tiles`: the last tiles of every chain load their operands with ordinary loads, for a backward
    that starts there; True), stream every operand past the caches (False), or keep at most that many tiles per
    chain (an int).  Forwards that save nothing always stream.  Results are the same bit for bit; only what a launch
    leaves in the caches differs.  Returns the old setting."""
    global _forward_keep
    old = _forward_keep
    _forward_keep = flag if isinstance(flag, bool) else max(0, int(flag))
    return old


def make_plan(B: int, L: int, D: int, in_dtype: torch.dtype, out_dtype: torch.dtype, direction: int,
              align_elems: int, ckpt_stride: int = 0, tune: int = 0, loose: bool = False) -> Plan:
    """Launch geometry for a shape: with `loose` the plan that `scan_forward` and `scan_backward` launch
    (qssm_plan_scan_loose), without it that of callers whose rows are all aligned to the lanes' width (qssm_plan_scan;
    the two differ only where they are not).  `tune` overrides single choices, for a test or sweep.  Plans depend on
    nothing but the arguments, so they are kept.  Callers must not modify the result."""
    key = (B, L, D, in_dtype, out_dtype, direction, align_elems, ckpt_stride, tune, loose)
    plan = _plans.get(key)
    if plan is None:
        plan = Plan()
        lib = _lib.load()
        planner = lib.qssm_plan_scan_loose if loose else lib.qssm_plan_scan_tuned
        _lib.check(planner(B, L, D, _DTYPE_CODE[in_dtype], _DTYPE_CODE[out_dtype], direction, align_elems, ckpt_stride,
                           tune, ctypes.byref(plan)))
        if len(_plans) >= 4096:
            _plans.clear()
        _plans[key] = plan
    return plan


_native = None


def _load_native():
    """csrc/torch_scan.cpp's module, with the two callables it works with."""
    global _native
    _native = _lib.load_native(_take_launch)
    return _native


def scan_forward(
    x: Tensor, a: Tensor, b: Tensor, c: Optional[Tensor], *,
    out_dtype: torch.dtype,
    want_y: bool = True,
    want_h: bool = False,
    want_ckpt: bool = True,
    tune: int = 0,
    bwd_tune: int = 0,
    h_init: Optional[Tensor] = None,
    h_final: Optional[Tensor] = None,
) -> Tuple[Optional[Tensor], Optional[Tensor], Optional[Tensor], int]:
    """One forward launch.  Operands must already share one supported storage type.

    Returns (y, h, ckpt, ckpt_stride): y in `out_dtype` (a storage the kernels are built for), h
    the full fp32 state if `want_h`, ckpt the fp32 states h(t-1) at t = k*ckpt_stride if
    `want_ckpt` (what the backward rebuilds h from).  `h_init` (fp32 [B, D], contiguous) is the
    state before the first step instead of zero; `h_final` (same layout) receives h(L-1).
    """
    # Operands are left in the caches only for a backward: a forward that saves no states has none coming.
    keep = _forward_keep if (want_ckpt or want_h) else False
    native = _native or _load_native()
    return native.scan_forward(x, a, b, c, _DTYPE_CODE[out_dtype], want_y | want_h << 1 | want_ckpt << 2,
                               -1 if keep is True else int(keep), tune, bwd_tune, h_init, h_final)


def scan_backward(
    x: Tensor, a: Tensor, b: Tensor, c: Tensor, dy: Tensor, *,
    h: Optional[Tensor] = None,
    ckpt: Optional[Tensor] = None,
    ckpt_stride: int = 0,
    need: Sequence[bool] = (True, True, True, True),
    tune: int = 0,
    h_init: Optional[Tensor] = None,
    dh_final: Optional[Tensor] = None,
    dh_init: Optional[Tensor] = None,
) -> Tuple[Optional[Tensor], Optional[Tensor], Optional[Tensor], Optional[Tensor]]:
    """One backward launch.  x, a, b, c share one storage type; dy has the storage of y.

    Exactly one of `h` (full fp32 state) and `ckpt` (+ its `ckpt_stride`) must be given.  Returns
    (dx, da, db, dc) in the storage type of the operands; entries not in `need` are None.
    `h_init` is the state the forward started from, `dh_final` the gradient arriving at h(L-1),
    `dh_init` receives the gradient of h(-1); all fp32 [B, D], contiguous, optional.
    """
    native = _native or _load_native()
    mask = sum(1 << i for i, n in enumerate(need) if n)
    return native.scan_backward(x, a, b, c, dy, h, ckpt, ckpt_stride, mask, tune, h_init, dh_final, dh_init)


def attach(y: Tensor, h: Optional[Tensor], ckpt: Optional[Tensor], stride: int, x: Tensor, a: Tensor, b: Tensor,
           c: Tensor, k_in: torch.dtype, k_out: torch.dtype, h_final: Optional[Tensor] = None,
           state: Optional[Tensor] = None, h_init: Optional[Tensor] = None) -> None:
    """Make `y` (and `h_final`) the outputs of an autograd node over the operands (and the incoming `state`): what
    `scan_forward` computed and kept, with the operands as the caller gave them and the storage types of the launch.
    `h_init` is the state the launch started from."""
    native = _native or _load_native()
    native.attach_scan(y, h, ckpt, stride, x, a, b, c, _DTYPE_CODE[k_in], _DTYPE_CODE[k_out], h_final, state, h_init)


def block_scan_forward_3d(x: Tensor, a: Tensor, b: Tensor, BLOCK_L: int = 256) -> Tuple[Tensor, Tensor]:
    """Device forward of h(t) = a(t) h(t-1) + b(t) x(t).

    Same contract as the reference's function of this name (quick_ssm/triton_forwards.py:134-172):
    3-D GPU inputs, returns fp32 `(out_a, out_x)` with out_x = h and out_a the running product of
    a.  `BLOCK_L` is accepted for compatibility; the launch geometry no longer depends on it.
    """
    for t in (x, a, b):
        assert t.dim() == 3, "All inputs should be [B, L, D]."
        assert t.device.type == "cuda", "Inputs must be on a GPU device."
    B, L, D = x.shape
    if L == 0:
        return torch.empty_like(a), torch.empty_like(x)
    k_in, _ = kernel_dtypes([x.dtype, a.dtype, b.dtype], torch.float32)
    xs, as_, bs = (t if t.dtype == k_in else t.to(k_in) for t in (x, a, b))
    h, _, _, _ = scan_forward(xs, as_, bs, None, out_dtype=torch.float32, want_ckpt=False)
    # out_a is discarded by every caller of the reference; it is kept for the tuple's shape.
    out_a = torch.cumprod(a.to(torch.float32), dim=1)
    return out_a, h


def block_scan_backward_3d(a: Tensor, b: Tensor, c: Tensor, x: Tensor, h: Tensor, grad_y: Tensor,
                           BLOCK_L: int = 256) -> Tuple[Tensor, Tensor, Tensor, Tensor]:
    """Device backward given the forward states h; returns fp32 (dx, da, db, dc).

    Same contract and argument order as the reference's function of this name
    (quick_ssm/triton_backwards.py:168-209), which upcasts every operand to fp32 first.
    """
    for t in (a, b, c, x, h, grad_y):
        assert t.dim() == 3, "All inputs should be [B, L, D]."
        assert t.device.type == "cuda", "Inputs must be on a GPU device."
    B, L, D = x.shape
    if L == 0:
        return (torch.empty_like(x), torch.empty_like(a), torch.empty_like(b), torch.empty_like(c))
    f32 = torch.float32
    a, b, c, x, h, grad_y = (t if t.dtype == f32 else t.to(f32) for t in (a, b, c, x, h, grad_y))
    return scan_backward(x, a, b, c, grad_y, h=h)
