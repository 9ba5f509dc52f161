"""Mamba-2 SSD forward on MI355X -- the host side of ``SSDLayer._ssd_core``.

Reference: ``workloads/mamba/model_ref.py`` (MR) in ShouyangDong/WorkloadSuite,
``SSDLayer._ssd_core(X_b, B_b, C_b, dt_b, A_dt_b, batch)`` (MR:123-162).  This
module keeps its argument meaning in unchunked form:

    MR (after MR:97-110)                 here
    X_b    [b, c, l, h, p]  fp16         X  [b, L, h, P]   f32 / bf16 / f16
    A_dt_b [b, c, l, h]     fp32         A  [b, L, h]      f32 (the log-decay A*dt)
    B_b, C_b [b, c, l, h, n] (repeated)  B, C [b, L, g, N] (group i // (h/g), no repeat)
    dt_b   [b, c, l, h]                  dt [b, L, h] or None (None: X is already scaled)
    block_len                            chunk_size
    (zeros, MR:153)                      initial_states [b, h, P, N] or None
    (discarded, MR:156)                  final state [b, h, P, N] when requested
    returns Y_diag + Y_off [b,c,l,h,p]   returns Y [b, L, h, P] in X's dtype

and its error behaviour: a seqlen that is not a multiple of the chunk size
(MR:106-110 raises in einops) and heads not divisible by groups (MR:37-38,
``ValueError``) raise ``ValueError`` here too.  Like MR, the op is pure: it
allocates fresh outputs and never mutates its inputs.

All arithmetic runs in libssd.so's HIP kernels on the tensors' device
and on torch's current stream.  There is no CPU path: tensors on another
device, or a missing library, raise.  The op is forward-only (no autograd),
as the reference harness runs it under ``torch.inference_mode()``.
"""

from __future__ import annotations

import ctypes
from typing import NamedTuple

import torch

from . import _lib

__all__ = [
    "ssd_forward",
    "forward_chunk",
    "walk_plan",
    "ssd_forward_noalloc",
    "ssd_core",
    "chunk_cumsum",
    "chunk_prep",
    "chunk_state",
    "state_passing",
    "state_passing_",
    "chunk_scan",
    "decode_step",
    "layer_prep",
    "ssd_layer",
    "workspace_bytes",
    "SSDError",
    "F16SStates",
    "F16SLocalStates",
]

SSDError = _lib.SSDError

_DTYPES = {torch.float32: _lib.DTYPE_F32, torch.bfloat16: _lib.DTYPE_BF16, torch.float16: _lib.DTYPE_F16}
_STATE_DTYPES = {torch.float32: _lib.DTYPE_F32, torch.bfloat16: _lib.DTYPE_BF16}
# f32 states stored as 16-bit (hi, lo) pairs of the inputs' type, or ("f16s")
# as f16 rows with a power-of-two scale per row
_SPLIT_STATES = {torch.bfloat16: _lib.STATE_SPLIT_BF16, torch.float16: _lib.STATE_SPLIT_F16,
                 "f16s": _lib.STATE_F16S}


class F16SStates(NamedTuple):
    """States handed to chunk_scan as f16 rows with a power-of-two scale per
    row (SSD_STATE_F16S): ``states`` [b, c, h, P, N] float32 storage whose
    rows hold N f16 values in their first half, ``scales`` [b, c, h, P]
    float32; state[..., p, n] = f16 value * scales[..., p]."""
    states: torch.Tensor
    scales: torch.Tensor

    def decode(self) -> torch.Tensor:
        N = self.states.shape[-1]
        return self.states.view(torch.float16)[..., :N].float() * self.scales[..., None]


class F16SLocalStates(NamedTuple):
    """Local states as ``chunk_state(..., state_dtype="f16s")`` writes them
    (SSD_STATE_F16S_LOCAL): ``states`` [b, c, h, P, N] float32 storage whose
    rows hold N f16 values in their first half; the power-of-two scales of
    each [P, N] item, one per row p and 16-column tile t, sit in (p, t) order
    in the second halves of its first rows; state[..., p, n] = f16 value *
    scale[p, n // 16].  ``state_passing`` takes them in place of f32 local
    states."""
    states: torch.Tensor

    def scales(self) -> torch.Tensor:
        """[b, c, h, P, N / 16] float32: the scale of each row's 16-column tiles."""
        P, N = self.states.shape[-2:]
        rows = P * (N // 16) // (N // 2)
        return self.states[..., :rows, N // 2:].reshape(*self.states.shape[:-2], P, N // 16)

    def decode(self) -> torch.Tensor:
        N = self.states.shape[-1]
        return self.states.view(torch.float16)[..., :N].float() * self.scales().repeat_interleave(16, -1)


def _handover(state_format, dtype, state_dtype):
    """state_dtype code for ssd_forward: the storage of the per-chunk states
    and, for f32 states, the format K3 hands them to K4 in (None: the
    library's choice, f16 rows with per-row scales where the chunk-256 kernels
    run; "split": hi/lo pairs of the inputs' type; "f16s")."""
    sd = _STATE_DTYPES.get(state_dtype)
    if sd is None:
        raise ValueError(f"unsupported state dtype {state_dtype}")
    if state_format is None:
        return sd
    if state_dtype != torch.float32 or dtype == torch.float32:
        raise ValueError("state_format needs float32 states and 16-bit inputs")
    if state_format == "split":
        return _SPLIT_STATES[dtype]
    if state_format == "f16s":
        return _lib.STATE_F16S
    raise ValueError(f"unknown state_format {state_format!r}")


def _device_check(*ts):
    dev = None
    for t in ts:
        if t is None:
            continue
        if t.device.type != "cuda":
            raise ValueError(f"libssd runs on HIP devices only; got a tensor on {t.device}")
        if dev is None:
            dev = t.device
        elif t.device != dev:
            raise ValueError(f"tensors on different devices: {dev} and {t.device}")
    return dev


def _vec_operand(t: torch.Tensor) -> torch.Tensor:
    """Unit inner stride, 16-byte aligned base and row strides (vector loads)."""
    es = t.element_size()
    ok = (t.stride(-1) == 1 and t.data_ptr() % 16 == 0
          and all(s >= 0 and (s * es) % 16 == 0 for s in t.stride()[:-1]))
    return t if ok else t.clone(memory_format=torch.contiguous_format)


def _f32_operand(t):
    if t is None:
        return None
    t = t.detach()
    if t.dtype != torch.float32:
        t = t.float()
    if any(s < 0 for s in t.stride()):
        t = t.contiguous()
    return t


def _f32_contig(t):
    if t is None:
        return None
    t = t.detach().to(torch.float32)
    if not t.is_contiguous() or t.data_ptr() % 16:
        t = t.clone(memory_format=torch.contiguous_format)
    return t


def _ptr(t):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


def _stream(dev):
    return ctypes.c_void_p(torch.cuda.current_stream(dev).cuda_stream)


# torch's current stream of a device as a raw handle, without building a
# Stream object (the accessor torch's own generated code uses), where present
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def _stream_fast(dev):
    return _raw_stream(dev.index) if _raw_stream is not None else _stream(dev)


def _shape_check(X, A, B, C, chunk_size, dt, initial_states):
    if X.dim() != 4:
        raise ValueError(f"X must be [batch, seqlen, nheads, headdim], got {tuple(X.shape)}")
    b, L, h, P = X.shape
    if A.shape != (b, L, h):
        raise ValueError(f"A must be {(b, L, h)}, got {tuple(A.shape)}")
    if B.dim() != 4 or B.shape[:2] != (b, L) or C.shape != B.shape:
        raise ValueError(f"B and C must be [batch, seqlen, ngroups, dstate] with batch={b}, seqlen={L}; "
                         f"got {tuple(B.shape)} and {tuple(C.shape)}")
    g, N = B.shape[2], B.shape[3]
    if h % g != 0:
        raise ValueError("n_heads must be divisible by n_groups")
    if chunk_size < 1 or L % chunk_size != 0:
        raise ValueError(f"seqlen {L} is not a multiple of chunk size {chunk_size}")
    if dt is not None and dt.shape != (b, L, h):
        raise ValueError(f"dt must be {(b, L, h)}, got {tuple(dt.shape)}")
    if initial_states is not None and initial_states.shape != (b, h, P, N):
        raise ValueError(f"initial_states must be {(b, h, P, N)}, got {tuple(initial_states.shape)}")
    if X.dtype not in _DTYPES:
        raise ValueError(f"unsupported dtype {X.dtype}")
    if B.dtype != X.dtype or C.dtype != X.dtype:
        raise ValueError(f"B and C must have X's dtype {X.dtype}, got {B.dtype} and {C.dtype}")
    return b, L, h, P, g, N


def _dims(b, L, h, P, N, g, Q):
    d = _lib.dims(b, L, h, P, N, g, Q)
    rc = _lib.load().ssd_check_dims(ctypes.byref(d), _lib.DTYPE_F32)
    _lib.check(rc)
    return d


def _expect(name, t, shape, dtype=None):
    """Shape (and dtype) of a per-kernel operand the C ABI takes without sizes."""
    if t is None:
        return
    if tuple(t.shape) != tuple(shape):
        raise ValueError(f"{name} must be {tuple(shape)}, got {tuple(t.shape)}")
    if dtype is not None and t.dtype != dtype:
        raise ValueError(f"{name} must be {dtype}, got {t.dtype}")


def _check_prep(prep, d):
    """chunk_prep's buffer must be at least what the dims need (it is read without a size)."""
    if prep is None:
        return
    need = _lib.load().ssd_chunk_prep_bytes(ctypes.byref(d))
    if need == 0 or prep.dtype != torch.uint8 or prep.numel() < need:
        raise ValueError(f"prep must be chunk_prep(B, C, Q)'s buffer for these shapes ({need} bytes)")


def workspace_bytes(batch, seqlen, nheads, headdim, dstate, ngroups, chunk_size,
                    state_dtype=torch.float32) -> int:
    d = _lib.dims(batch, seqlen, nheads, headdim, dstate, ngroups, chunk_size)
    n = _lib.load().ssd_workspace_bytes(ctypes.byref(d), _STATE_DTYPES[state_dtype])
    if n == 0:
        _lib.check(_lib.load().ssd_check_dims(ctypes.byref(d), _lib.DTYPE_F32))
    return n


def forward_chunk(batch, seqlen, nheads, headdim, dstate, ngroups, chunk_size, dtype,
                  state_dtype=torch.float32, state_format=None) -> int:
    """The chunk length ``ssd_forward`` runs these dims at (the library's
    ``ssd_forward_chunk``): ``chunk_size``, or 256 for 16-bit inputs with
    float32 states, seqlen % 256 == 0 and d_state 64 / 128 where that
    workspace is not the larger one."""
    d = _lib.dims(batch, seqlen, nheads, headdim, dstate, ngroups, chunk_size)
    q = _lib.load().ssd_forward_chunk(ctypes.byref(d), _DTYPES[dtype], _handover(state_format, dtype, state_dtype))
    if q == 0:
        _lib.check(_lib.load().ssd_check_dims(ctypes.byref(d), _DTYPES[dtype]))
    return q


class WalkPlan(NamedTuple):
    """How a core runs as a walk along its (batch, head) chains (``walk_plan``)."""
    segments: int  # of each chain
    steps: int     # 64-token steps per segment
    heads: int     # per workgroup
    linked: bool   # the states entering the segments come from a launch of their own
    hilo: bool     # the state enters C.S as a hi + lo pair of the input type (else as f16 rows with a scale each)


def walk_plan(batch, seqlen, nheads, headdim, dstate, ngroups, chunk_size, dtype, state_dtype=torch.float32,
              state_format=None, gated=False, in_place=False):
    """How the library runs ``ssd_forward`` (``gated``: ``ssd_layer``) of these
    dims, for operands it takes as they are (``in_place``: with the final state
    written over the initial one, as the C ABI allows): a WalkPlan, or None for the stage
    kernels.  Without a device, as for 256 CUs."""
    d = _lib.dims(batch, seqlen, nheads, headdim, dstate, ngroups, chunk_size)
    p = _lib.SSDWalkPlan()
    _lib.check(_lib.load().ssd_forward_plan(ctypes.byref(d), _DTYPES[dtype], _handover(state_format, dtype, state_dtype),
                                            int(gated), int(in_place), ctypes.byref(p)))
    return WalkPlan(p.segments, p.steps, p.heads, bool(p.linked), bool(p.hilo)) if p.segments else None


# ssd_forward's per-call host work, kept per layout: the ctypes dims and
# stride arrays, the workspace size and the output shapes, for operands that
# the kernels take as they are (no copy).  Keyed by every shape, stride,
# dtype and device the checks depend on; data pointers (16-byte alignment)
# are checked on every call.
_PLANS = {}
_PLANS_MAX = 256
_NO_WORKSPACE = {}  # device -> a 256-byte buffer for the forwards that use no workspace


class _Plan(NamedTuple):
    dims: object
    dtype: int
    sd: int
    ws_n: int
    strides: tuple   # X, A, B, C, dt (or None), Y
    y_shape: tuple
    f_shape: tuple


def _layout_key(t):
    return None if t is None else (t.shape, t.stride(), t.dtype, t.device)


def _unchanged(t, t0):
    """t is t0's memory as it was (no copy or conversion on the way)."""
    if t is None or t0 is None:
        return t is None and t0 is None
    return t.data_ptr() == t0.data_ptr() and t.dtype == t0.dtype and t.stride() == t0.stride()


def _aligned(*ts):
    return all(t is None or t.data_ptr() % 16 == 0 for t in ts)


def _no_workspace(dev):
    buf = _NO_WORKSPACE.get(dev)
    if buf is None:
        buf = _NO_WORKSPACE[dev] = torch.empty(256, dtype=torch.uint8, device=dev)
    return buf


def ssd_forward(X, A, B, C, chunk_size, dt=None, initial_states=None,
                return_final_states=False, state_dtype=torch.float32, state_format=None):
    """Chunked SSD forward (MR:123-162) on the HIP device.

    Returns Y, or (Y, final_states) with ``return_final_states``.

    ``chunk_size`` is MR's block_len and only has to divide the seqlen: every
    chunking evaluates the same linear recurrence (MR:152-161).  For 16-bit
    inputs with float32 states, seqlen % 256 == 0 and d_state 64 / 128 the
    library runs chunk 64 / 128 at 256 (``forward_chunk``), which changes
    rounding only.

    ``state_dtype`` is the storage type of the per-chunk states (float32, or
    bfloat16 for 16-bit inputs); the recurrence itself always runs in
    float32.  ``state_format`` (float32 states, 16-bit inputs): how the states
    entering each chunk reach chunk_scan --

    * None (the default): the library's choice.  At d_state 128 with an even
      number of heads per group and enough work for the GPU the whole core
      runs as a walk along the (batch, head) chains with the state in float32
      registers, and no states are handed over at all (float32 inputs: at
      d_state 64 / 128 with more than two chains per CU; ``walk_plan`` tells).
      Otherwise f16 rows
      with a power-of-two scale per row ("f16s") wherever a 16-bit chunk_scan
      reads them: chunk 256 with d_state 64 / 128, and chunk 64 / 128 with
      chunk x d_state <= 8192.
      Where chunk_state and state_passing then run as two launches (chunk 256
      outside the one-launch state chain, and the chain's segments) the local
      states between them cross HBM as f16 rows with a scale per row and
      16-column tile (SSD_STATE_F16S_LOCAL); the state chain keeps them in
      float32 registers.  Which launches run, and how a walk cuts its chains,
      depends on batch x heads and the device's CU count, so the last bits of Y and of the final state are not
      invariant to the batch size (within the 16-bit tolerance, and the final
      state within ~1e-3 of its scale).
    * "split": hi/lo pairs of the inputs' type at chunk 256 (plain float32
      at chunk 64 / 128); every local state stays float32.
    * "f16s": f16 rows as above, never the walk.
    """
    key = (_layout_key(X), _layout_key(A), _layout_key(B), _layout_key(C), _layout_key(dt),
           _layout_key(initial_states), chunk_size, return_final_states, state_dtype, state_format)
    plan = _PLANS.get(key)
    if plan is not None and _aligned(X, B, C, initial_states):
        dev = X.device
        Y = torch.empty(plan.y_shape, dtype=X.dtype, device=dev)
        final = torch.empty(plan.f_shape, dtype=torch.float32, device=dev) if return_final_states else None
        ws = _no_workspace(dev) if plan.ws_n <= 256 else torch.empty(plan.ws_n, dtype=torch.uint8, device=dev)
        sx, sa, sb, sc, sdt, sy = plan.strides
        _lib.check(_lib.load().ssd_forward(
            ctypes.byref(plan.dims), plan.dtype, X.data_ptr(), sx, A.data_ptr(), sa, B.data_ptr(), sb,
            C.data_ptr(), sc, None if dt is None else dt.data_ptr(), sdt,
            None if initial_states is None else initial_states.data_ptr(), Y.data_ptr(), sy,
            None if final is None else final.data_ptr(), ws.data_ptr(), plan.ws_n, plan.sd, _stream_fast(dev)))
        return (Y, final) if return_final_states else Y
    out = _ssd_forward(X, A, B, C, chunk_size, dt, initial_states, return_final_states, state_dtype,
                       state_format, key)
    return out


def _ssd_forward(X, A, B, C, chunk_size, dt, initial_states, return_final_states, state_dtype, state_format, key):
    """The checks, operand conversions and call of ssd_forward (and its plan for the layout)."""
    b, L, h, P, g, N = _shape_check(X, A, B, C, chunk_size, dt, initial_states)
    dev = _device_check(X, A, B, C, dt, initial_states)
    lib = _lib.load()
    d = _dims(b, L, h, P, N, g, chunk_size)
    X0, B0, C0, A0, dt0, init0 = X, B, C, A, dt, initial_states
    X = _vec_operand(X.detach())
    Bm = _vec_operand(B.detach())
    Cm = _vec_operand(C.detach())
    A = _f32_operand(A)
    dt = _f32_operand(dt)
    init = _f32_contig(initial_states)
    Y = torch.empty((b, L, h, P), dtype=X.dtype, device=dev)
    final = torch.empty((b, h, P, N), dtype=torch.float32, device=dev) if return_final_states else None
    sd = _handover(state_format, X.dtype, state_dtype)
    # the workspace of the chunk the library runs at
    dw = _lib.dims(b, L, h, P, N, g, lib.ssd_forward_chunk(ctypes.byref(d), _DTYPES[X.dtype], sd))
    ws_n = lib.ssd_workspace_bytes(ctypes.byref(dw), sd)
    ws = _no_workspace(dev) if ws_n <= 256 else torch.empty(ws_n, dtype=torch.uint8, device=dev)
    strides = (_lib.strides(X), _lib.strides(A), _lib.strides(Bm), _lib.strides(Cm),
               _lib.strides(dt) if dt is not None else None, _lib.strides(Y))
    rc = lib.ssd_forward(ctypes.byref(d), _DTYPES[X.dtype],
                         _ptr(X), strides[0], _ptr(A), strides[1], _ptr(Bm), strides[2], _ptr(Cm), strides[3],
                         _ptr(dt), strides[4], _ptr(init), _ptr(Y), strides[5], _ptr(final),
                         _ptr(ws), ws_n, sd, _stream(dev))
    _lib.check(rc)
    # the same layout next time: no checks or conversions, where none were needed
    as_is = all(_unchanged(t, t0) for t, t0 in ((X, X0), (Bm, B0), (Cm, C0), (A, A0), (dt, dt0), (init, init0)))
    if as_is and len(_PLANS) < _PLANS_MAX:
        _PLANS[key] = _Plan(d, _DTYPES[X.dtype], sd, ws_n, strides, tuple(Y.shape),
                            None if final is None else tuple(final.shape))
    return (Y, final) if return_final_states else Y


def ssd_forward_noalloc(X, A, B, C, chunk_size, dt=None, initial_states=None,
                        return_final_states=False, state_dtype=torch.float32, state_format=None):
    """``ssd_forward`` through the C ABI's ``ssd_forward_noalloc``: the library
    takes its workspace from a device array it keeps per device instead of a
    buffer allocated here (for callers that cannot allocate: graph capture,
    serving loops).  Same results (a call too large for the array runs in batch
    slices: those of ``ssd_forward`` on each slice).  Only the outputs are allocated (by torch,
    before the call); inputs that are not already in the kernels' layout are
    copied first, as in ``ssd_forward``.  Calls that overlap on one device race
    on that array."""
    b, L, h, P, g, N = _shape_check(X, A, B, C, chunk_size, dt, initial_states)
    dev = _device_check(X, A, B, C, dt, initial_states)
    lib = _lib.load()
    d = _dims(b, L, h, P, N, g, chunk_size)
    sd = _handover(state_format, X.dtype, state_dtype)
    X = _vec_operand(X.detach())
    Bm = _vec_operand(B.detach())
    Cm = _vec_operand(C.detach())
    A = _f32_operand(A)
    dt = _f32_operand(dt)
    init = _f32_contig(initial_states)
    Y = torch.empty((b, L, h, P), dtype=X.dtype, device=dev)
    final = torch.empty((b, h, P, N), dtype=torch.float32, device=dev) if return_final_states else None
    rc = lib.ssd_forward_noalloc(ctypes.byref(d), _DTYPES[X.dtype],
                                 _ptr(X), _lib.strides(X), _ptr(A), _lib.strides(A),
                                 _ptr(Bm), _lib.strides(Bm), _ptr(Cm), _lib.strides(Cm),
                                 _ptr(dt), _lib.strides(dt) if dt is not None else None,
                                 _ptr(init), _ptr(Y), _lib.strides(Y), _ptr(final), sd, _stream(dev))
    _lib.check(rc)
    return (Y, final) if return_final_states else Y


def ssd_core(X_b, B_b, C_b, dt_b, A_dt_b, batch=None, state_dtype=torch.float32):
    """``SSDLayer._ssd_core`` (MR:123-162) with the reference's own arguments.

    X_b [b, c, l, h, p]; B_b, C_b [b, c, l, h, n] (already GQA-repeated,
    MR:97-99); dt_b, A_dt_b [b, c, l, h]; ``batch`` is accepted and ignored
    (MR passes it to size its zero initial state).  Returns Y [b, c, l, h, p]
    in X_b's dtype, like MR:162.  The block length is l (MR's block_len).
    """
    b, c, l, h, p = X_b.shape
    L = c * l
    Y = ssd_forward(X_b.reshape(b, L, h, p), A_dt_b.reshape(b, L, h),
                    B_b.reshape(b, L, h, B_b.shape[-1]), C_b.reshape(b, L, h, C_b.shape[-1]),
                    chunk_size=l, dt=dt_b.reshape(b, L, h), state_dtype=state_dtype)
    return Y.reshape(b, c, l, h, p)


# ---------------------------------------------------------------------------
# The four kernels one at a time (per-kernel parity tests and timing).
# ---------------------------------------------------------------------------

def chunk_cumsum(A, chunk_size):
    """K1: A [b, L, h] -> (Acs [b, h, c, Q], chunk_decay [b, h, c]) (MR:135-136, 150)."""
    if A.dim() != 3:
        raise ValueError("A must be [batch, seqlen, nheads]")
    b, L, h = A.shape
    dev = _device_check(A)
    if chunk_size < 1 or L % chunk_size != 0:
        raise ValueError(f"seqlen {L} is not a multiple of chunk size {chunk_size}")
    d = _dims(b, L, h, 64, 16, 1, chunk_size)
    A = _f32_operand(A)
    nc = L // chunk_size
    Acs = torch.empty((b, h, nc, chunk_size), dtype=torch.float32, device=dev)
    decay = torch.empty((b, h, nc), dtype=torch.float32, device=dev)
    _lib.check(_lib.load().ssd_chunk_cumsum(ctypes.byref(d), _ptr(A), _lib.strides(A), _ptr(Acs),
                                            _ptr(decay), _stream(dev)))
    return Acs, decay


def chunk_prep(B, C, chunk_size):
    """K0: the chunk-256 kernels' per-(batch, chunk, group) operands -- C.B^T
    (MR:143) and B in their register order -- as an opaque uint8 buffer for
    ``chunk_state`` / ``chunk_scan`` (``prep=``), or None for shapes and dtypes
    without that path (the kernels then rebuild them themselves)."""
    b, L, g, N = B.shape
    if C.shape != B.shape:
        raise ValueError("B and C must have the same shape [batch, seqlen, ngroups, dstate]")
    dev = _device_check(B, C)
    if chunk_size < 1 or L % chunk_size != 0:
        raise ValueError(f"seqlen {L} is not a multiple of chunk size {chunk_size}")
    lib = _lib.load()
    d = _dims(b, L, g, 64, N, g, chunk_size)
    n = lib.ssd_chunk_prep_bytes(ctypes.byref(d))
    if n == 0 or B.dtype == torch.float32:
        return None
    Bm, Cm = _vec_operand(B.detach()), _vec_operand(C.detach())
    prep = torch.empty(n, dtype=torch.uint8, device=dev)
    _lib.check(lib.ssd_chunk_prep(ctypes.byref(d), _DTYPES[Bm.dtype], _ptr(Bm), _lib.strides(Bm), _ptr(Cm),
                                  _lib.strides(Cm), _ptr(prep), n, _stream(dev)))
    return prep


def chunk_state(X, B, Acs, dt=None, state_dtype=torch.float32, prep=None):
    """K2: local states [b, c, h, P, N] (MR:144, 148-149).  ``prep``: chunk_prep(B, C, Q) or None.

    ``state_dtype="f16s"`` (16-bit inputs at chunk 256, d_state 64 / 128):
    the f32 local states rounded to f16 rows with a power-of-two scale per
    row, as an ``F16SLocalStates`` (what the forward hands from K2 to K3
    there when S_in goes to chunk_scan as "f16s")."""
    b, L, h, P = X.shape
    g, N = B.shape[2], B.shape[3]
    Q = Acs.shape[-1]
    dev = _device_check(X, B, Acs, dt, prep)
    d = _dims(b, L, h, P, N, g, Q)
    _expect("Acs", Acs, (b, h, L // Q, Q))
    _expect("dt", dt, (b, L, h))
    _check_prep(prep, d)
    f16l = isinstance(state_dtype, str) and state_dtype == "f16s"
    if not f16l and state_dtype not in _STATE_DTYPES:
        raise ValueError(f"unsupported state dtype {state_dtype}")
    X, Bm = _vec_operand(X.detach()), _vec_operand(B.detach())
    Acs = _f32_contig(Acs)
    dt = _f32_operand(dt)
    states = torch.empty((b, L // Q, h, P, N), dtype=torch.float32 if f16l else state_dtype, device=dev)
    _lib.check(_lib.load().ssd_chunk_state(
        ctypes.byref(d), _DTYPES[X.dtype], _ptr(X), _lib.strides(X), _ptr(Bm), _lib.strides(Bm),
        _ptr(dt), _lib.strides(dt) if dt is not None else None, _ptr(Acs), _ptr(states),
        _lib.STATE_F16S_LOCAL if f16l else _STATE_DTYPES[state_dtype], _ptr(prep), _stream(dev)))
    return F16SLocalStates(states) if f16l else states


def state_passing(states, chunk_decay, initial_states=None, return_final_states=True, split=None):
    """K3: (S_in [b, c, h, P, N], final [b, h, P, N]) from local states (MR:152-157).

    Works on a copy: the input ``states`` is left unchanged.  ``split``
    (f32 states only): torch.bfloat16 / torch.float16 store S_in as that
    type's (hi, lo) pairs for ``chunk_scan(..., split=True)``; "f16s" as f16
    rows with a power-of-two scale per row for ``chunk_scan(..., split="f16s")``.
    ``states`` may be ``chunk_state(..., state_dtype="f16s")``'s
    ``F16SLocalStates`` (S_in then goes out as "f16s").
    """
    local = isinstance(states, F16SLocalStates)
    if local:
        if split not in (None, "f16s"):
            raise ValueError('f16 local states give f16s S_in: split must be "f16s" or None')
        split, states = "f16s", states.states
    S = states.detach().clone(memory_format=torch.contiguous_format)
    final = (torch.empty((S.shape[0], S.shape[2], S.shape[3], S.shape[4]), dtype=torch.float32, device=S.device)
             if return_final_states else None)
    scales = torch.empty(S.shape[:4], dtype=torch.float32, device=S.device) if split == "f16s" else None
    state_passing_(S, chunk_decay, initial_states, final, split=split, scales=scales, f16_local=local)
    return (F16SStates(S, scales) if scales is not None else S), final


def state_passing_(states, chunk_decay, initial_states=None, final_states=None, split=None, scales=None,
                   f16_local=False):
    """K3 in place on a contiguous ``states`` buffer (local states in, S_in out);
    ``final_states`` (optional, [b, h, P, N] float32) receives the last state;
    ``scales`` ([b, c, h, P] float32) the row scales when split="f16s";
    ``f16_local``: the buffer holds SSD_STATE_F16S_LOCAL local states (split "f16s")."""
    b, nc, h, P, N = states.shape
    dev = _device_check(states, chunk_decay, initial_states, final_states)
    if not states.is_contiguous():
        raise ValueError("state_passing_ needs a contiguous states buffer")
    d = _dims(b, nc * 64, h, P, N, 1, 64)
    if states.dtype not in _STATE_DTYPES:
        raise ValueError(f"unsupported state dtype {states.dtype}")
    _expect("chunk_decay", chunk_decay, (b, h, nc))
    _expect("initial_states", initial_states, (b, h, P, N))
    decay = _f32_contig(chunk_decay)
    init = _f32_contig(initial_states)
    if final_states is not None and (final_states.dtype != torch.float32 or not final_states.is_contiguous()
                                     or final_states.shape != (b, h, P, N)):
        raise ValueError("final_states must be a contiguous float32 [b, h, P, N] tensor")
    if split is not None and (states.dtype != torch.float32 or split not in _SPLIT_STATES):
        raise ValueError('split storage needs float32 states and split=torch.bfloat16, torch.float16 or "f16s"')
    sd = _STATE_DTYPES[states.dtype] if split is None else _SPLIT_STATES[split]
    if f16_local:
        if split != "f16s":
            raise ValueError('f16 local states need split="f16s"')
        sd = _lib.STATE_F16S_LOCAL
    if split == "f16s":
        _expect("scales", scales, (b, nc, h, P), torch.float32)
        if scales is None or not scales.is_contiguous() or scales.device != dev:
            raise ValueError(f"f16s states need a contiguous float32 scales tensor {(b, nc, h, P)} on {dev}")
    _lib.check(_lib.load().ssd_state_passing(ctypes.byref(d), _ptr(states), sd, _ptr(scales if split == "f16s" else None),
                                             _ptr(decay), _ptr(init), _ptr(final_states), _stream(dev)))
    return states


def chunk_state_passing(X, B, Acs, chunk_decay, dt=None, prep=None, initial_states=None,
                        return_final_states=True, split=None, state_dtype=torch.float32):
    """K2 then K3 as ``ssd_forward`` runs them (MR:144-157): (S_in [b, c, h, P, N],
    final [b, h, P, N] or None).  Same values as ``chunk_state`` followed by
    ``state_passing``; with ``split`` (the inputs' 16-bit type) and ``prep`` at
    chunk 256 the two run as one launch where that is faster on the device."""
    b, L, h, P = X.shape
    g, N = B.shape[2], B.shape[3]
    Q = Acs.shape[-1]
    dev = _device_check(X, B, Acs, chunk_decay, dt, initial_states, prep)
    d = _dims(b, L, h, P, N, g, Q)
    _expect("Acs", Acs, (b, h, L // Q, Q))
    _expect("chunk_decay", chunk_decay, (b, h, L // Q))
    _expect("dt", dt, (b, L, h))
    _expect("initial_states", initial_states, (b, h, P, N))
    _check_prep(prep, d)
    X, Bm = _vec_operand(X.detach()), _vec_operand(B.detach())
    Acs = _f32_contig(Acs)
    decay = _f32_contig(chunk_decay)
    dt = _f32_operand(dt)
    init = _f32_contig(initial_states)
    if split is not None:
        if split not in _SPLIT_STATES:
            raise ValueError('split must be torch.bfloat16, torch.float16 or "f16s"')
        sd, store = _SPLIT_STATES[split], torch.float32
    else:
        sd, store = _STATE_DTYPES[state_dtype], state_dtype
    states = torch.empty((b, L // Q, h, P, N), dtype=store, device=dev)
    final = torch.empty((b, h, P, N), dtype=torch.float32, device=dev) if return_final_states else None
    scales = torch.empty((b, L // Q, h, P), dtype=torch.float32, device=dev) if split == "f16s" else None
    _lib.check(_lib.load().ssd_chunk_state_passing(
        ctypes.byref(d), _DTYPES[X.dtype], _ptr(X), _lib.strides(X), _ptr(Bm), _lib.strides(Bm),
        _ptr(dt), _lib.strides(dt) if dt is not None else None, _ptr(Acs), _ptr(decay), _ptr(prep), _ptr(init),
        _ptr(states), sd, _ptr(scales), _ptr(final), _stream(dev)))
    return (F16SStates(states, scales) if scales is not None else states), final


def _epilogue(X, D, z, dev):
    """The skip / gate epilogue struct (or None) and the tensors it points into."""
    if D is None and z is None:
        return None, ()
    epi = _lib.SSDEpilogue()
    keep = []
    if D is not None:
        D = _f32_contig(D.reshape(-1))
        if D.device != dev or D.numel() != X.shape[2]:
            raise ValueError(f"D must be [{X.shape[2]}] on {dev}")
        epi.D = D.data_ptr()
        keep.append(D)
    if z is not None:
        if z.shape != X.shape or z.dtype != X.dtype or z.device != dev:
            raise ValueError(f"z must match X: {tuple(X.shape)} {X.dtype} on {dev}")
        z = z.detach()
        if z.stride(-1) != 1 or any(st < 0 for st in z.stride()):
            z = z.contiguous()
        epi.z = z.data_ptr()
        for k in range(4):
            epi.z_strides[k] = z.stride(k)
        keep.append(z)
    return epi, keep


def chunk_scan(X, B, C, Acs, states, dt=None, prep=None, split=False, D=None, z=None):
    """K4: Y [b, L, h, P] from the states entering each chunk (MR:139-145, 160-162).
    ``prep``: chunk_prep(B, C, Q) or None.  ``split``: True when ``states``
    holds state_passing(..., split=X.dtype)'s (hi, lo) pairs, "f16s" for
    state_passing(..., split="f16s")'s scaled f16 rows.  ``D`` [h] and / or
    ``z`` (X's shape and dtype): the layer's skip and gate fused into the write,
    Y = (Y + D x) * silu(z) (MR:116-118)."""
    b, L, h, P = X.shape
    g, N = B.shape[2], B.shape[3]
    Q = Acs.shape[-1]
    scales = None
    if isinstance(states, F16SStates):
        if split not in (False, "f16s"):
            raise ValueError('F16SStates are read with split="f16s"')
        split, states, scales = "f16s", states.states, states.scales
    elif split == "f16s":
        raise ValueError('split="f16s" needs the F16SStates that state_passing(..., split="f16s") returns')
    dev = _device_check(X, B, C, Acs, states, dt, prep, scales)
    d = _dims(b, L, h, P, N, g, Q)
    if scales is not None:
        _expect("scales", scales, (b, L // Q, h, P), torch.float32)
        scales = scales.contiguous()
    if C.shape != B.shape or C.dtype != B.dtype:
        raise ValueError("B and C must have the same shape and dtype")
    _expect("Acs", Acs, (b, h, L // Q, Q))
    _expect("dt", dt, (b, L, h))
    # the kernels read [b, c, h, P, N] rows of the states' element size: a
    # wrongly shaped or typed buffer would be read past its end
    _expect("states", states, (b, L // Q, h, P, N), torch.float32 if split else None)
    if not split and states.dtype not in _STATE_DTYPES:
        raise ValueError(f"unsupported state dtype {states.dtype}")
    if split and X.dtype not in (torch.bfloat16, torch.float16):
        raise ValueError("split states need 16-bit inputs")
    if split not in (False, True, "f16s"):
        raise ValueError(f'split must be False, True or "f16s", got {split!r}')
    _check_prep(prep, d)
    X, Bm, Cm = _vec_operand(X.detach()), _vec_operand(B.detach()), _vec_operand(C.detach())
    Acs = _f32_contig(Acs)
    dt = _f32_operand(dt)
    S = states.detach()
    if not S.is_contiguous():
        S = S.contiguous()
    Y = torch.empty((b, L, h, P), dtype=X.dtype, device=dev)
    epi, _keep = _epilogue(X, D, z, dev)
    _lib.check(_lib.load().ssd_chunk_scan(
        ctypes.byref(d), _DTYPES[X.dtype], _ptr(X), _lib.strides(X), _ptr(Bm), _lib.strides(Bm),
        _ptr(Cm), _lib.strides(Cm), _ptr(dt), _lib.strides(dt) if dt is not None else None,
        _ptr(Acs), _ptr(S), (_SPLIT_STATES["f16s" if split == "f16s" else X.dtype] if split
                             else _STATE_DTYPES[S.dtype]), _ptr(scales), _ptr(Y),
        _lib.strides(Y), _ptr(prep), ctypes.byref(epi) if epi is not None else None, _stream(dev)))
    return Y


# decode_step's and ssd_layer's per-call host work, kept per layout as
# ssd_forward's is (_PLANS): for operands the kernels take as they are.  Nothing
# of a call's own is kept: pointers go into structs made for the call.
_DECODE_PLANS = {}
_LAYER_PLANS = {}


class _DecodePlan(NamedTuple):
    dims: object
    dtype: int
    strides: tuple     # x, B, C, a (and dt), y
    z_strides: object  # or None
    y_shape: tuple


class _LayerPlan(NamedTuple):
    dims: object
    dtype: int
    width: int         # conv kernel width
    strides: tuple     # x, z, B, C, dt, y
    nbytes: int


def decode_step(state, x, B, C, a, dt=None, D=None, z=None):
    """One token of the recurrence, in place on ``state`` [b, h, P, N] f32
    (e.g. ssd_forward's final state): state = exp(a) state + dt x B^T, then
    y = state C (+ D x, * silu(z)).  x, z [b, h, P]; B, C [b, g, N] of x's
    dtype; a, dt [b, h] f32 (dt None means 1).  Returns y [b, h, P]."""
    key = (_layout_key(state), _layout_key(x), _layout_key(B), _layout_key(C), _layout_key(a), _layout_key(dt),
           _layout_key(D), _layout_key(z))
    plan = _DECODE_PLANS.get(key)
    if plan is None or not _aligned(state, a, dt, D):
        return _decode_step(state, x, B, C, a, dt, D, z, key)
    dev = x.device
    y = torch.empty(plan.y_shape, dtype=x.dtype, device=dev)
    sx, sb, sc, sad, sy = plan.strides
    epi = None
    if plan.z_strides is not None:
        epi = ctypes.byref(_lib.SSDEpilogue(0 if D is None else D.data_ptr(), 0 if z is None else z.data_ptr(),
                                            plan.z_strides))
    _lib.check(_lib.load().ssd_decode_step(
        ctypes.byref(plan.dims), plan.dtype, state.data_ptr(), x.data_ptr(), sx, B.data_ptr(), sb, C.data_ptr(), sc,
        a.data_ptr(), None if dt is None else dt.data_ptr(), sad, y.data_ptr(), sy, epi, _stream_fast(dev)))
    return y


def _decode_step(state, x, B, C, a, dt, D, z, key):
    """The checks, operand conversions and call of decode_step (and its plan for the layout)."""
    if state.dim() != 4 or state.dtype != torch.float32:
        raise ValueError("state must be [b, h, P, N] float32")
    b, h, P, N = state.shape
    if x.shape != (b, h, P) or B.dim() != 3 or B.shape[0] != b or B.shape[2] != N or C.shape != B.shape:
        raise ValueError(f"x must be {(b, h, P)} and B, C [b, g, {N}]")
    g = B.shape[1]
    if h % g != 0:
        raise ValueError("n_heads must be divisible by n_groups")
    if a.shape != (b, h) or (dt is not None and dt.shape != (b, h)):
        raise ValueError(f"a and dt must be {(b, h)}")
    if x.dtype not in _DTYPES or B.dtype != x.dtype or C.dtype != x.dtype:
        raise ValueError("x, B and C must share a supported dtype")
    if not state.is_contiguous() or state.data_ptr() % 16:
        raise ValueError("state must be contiguous and 16-byte aligned (it is updated in place)")
    dev = _device_check(state, x, B, C, a, dt, D, z)
    if D is not None and D.numel() != h:
        raise ValueError(f"D must have {h} elements")
    d = _lib.dims(b, 1, h, P, N, g, 1)
    given = (x, B, C, a, dt, D, z)
    x, Bm, Cm = _rows3(x), _rows3(B), _rows3(C)
    a = _f32_contig(a)
    dt = _f32_contig(dt)
    y = torch.empty((b, h, P), dtype=x.dtype, device=dev)
    epi, _keep = None, ()
    if D is not None or z is not None:
        epi = _lib.SSDEpilogue()
        keep = []
        if D is not None:
            D = _f32_contig(D.reshape(h))
            epi.D = D.data_ptr()
            keep.append(D)
        if z is not None:
            if z.shape != (b, h, P) or z.dtype != x.dtype or z.device != dev:
                raise ValueError(f"z must match x: {(b, h, P)} {x.dtype}")
            z = _rows3(z)
            epi.z = z.data_ptr()
            epi.z_strides[0], epi.z_strides[1], epi.z_strides[2], epi.z_strides[3] = z.stride(0), 0, z.stride(1), 1
            keep.append(z)
        _keep = keep
    st2 = lambda t: (ctypes.c_int64 * 2)(t.stride(0), t.stride(1))  # noqa: E731
    strides = (st2(x), st2(Bm), st2(Cm), st2(a), st2(y))
    _lib.check(_lib.load().ssd_decode_step(
        ctypes.byref(d), _DTYPES[x.dtype], _ptr(state), _ptr(x), strides[0], _ptr(Bm), strides[1], _ptr(Cm), strides[2],
        _ptr(a), _ptr(dt), strides[3], _ptr(y), strides[4], ctypes.byref(epi) if epi is not None else None, _stream(dev)))
    del _keep
    # the same layout next time, where nothing was copied or converted (D, of
    # any shape with h elements in a row, is read as its h floats)
    x0, B0, C0, a0, dt0, D0, z0 = given
    if (all(_unchanged(t, t0) for t, t0 in ((x, x0), (Bm, B0), (Cm, C0), (a, a0), (dt, dt0), (z, z0)))
            and (D0 is None or (D.data_ptr() == D0.data_ptr() and D0.dtype == torch.float32))
            and len(_DECODE_PLANS) < _PLANS_MAX):
        _DECODE_PLANS[key] = _DecodePlan(d, _DTYPES[x.dtype], strides, None if epi is None else epi.z_strides, (b, h, P))
    return y


# ---------------------------------------------------------------------------
# the layer around the core (SSDLayer.forward, MR:76-118)
# ---------------------------------------------------------------------------

def _layer_params(conv_weight, conv_bias, dt_bias, A_log, D, d_inner, nheads, dtype, dev):
    k = conv_weight.shape[-1]
    if conv_weight.numel() != d_inner * k:
        raise ValueError(f"conv weight must be [{d_inner}, 1, k], got {tuple(conv_weight.shape)}")
    w = conv_weight.detach().reshape(d_inner, k).to(dtype).contiguous()
    bias = None if conv_bias is None else conv_bias.detach().reshape(d_inner).to(dtype).contiguous()
    dtb = dt_bias.detach().reshape(nheads).to(dtype).contiguous()
    alog = _f32_contig(A_log.reshape(nheads))
    Dv = None if D is None else _f32_contig(D.reshape(nheads))
    for t in (w, bias, dtb, alog, Dv):
        if t is not None and t.device != dev:
            raise ValueError(f"layer parameters must be on {dev}, got {t.device}")
    prm = _lib.SSDLayerParams(k, w.data_ptr(), 0 if bias is None else bias.data_ptr(), dtb.data_ptr(),
                              alog.data_ptr(), 0 if Dv is None else Dv.data_ptr())
    return prm, (w, bias, dtb, alog, Dv)


def _rows3(t):
    t = t.detach()
    if t.stride(-1) != 1 or any(st < 0 for st in t.stride()):
        t = t.contiguous()
    return t


def layer_prep(x, dt, conv_weight, conv_bias, dt_bias, A_log, chunk_size, nheads, ngroups=1, dstate=64):
    """Pre-SSD prep (MR:83-103) in two HIP launches.

    ``x`` [b, L, h*P] and ``dt`` [b, L, h] are in_proj's output slices (any
    strides, unit inner stride).  Returns ``(X, dt, Acs, chunk_decay)``: X =
    silu(causal depthwise conv1d(x) + bias) as [b, L, h, P] in x's dtype, dt =
    softplus(dt + dt_bias) in float32, and K1's cumsum of A dt with A =
    -exp(A_log).  ``ngroups`` / ``dstate`` only enter the shape validation."""
    b, L, d_inner = x.shape
    if dt.shape != (b, L, nheads) or d_inner % nheads != 0:
        raise ValueError(f"dt must be {(b, L, nheads)} and d_inner a multiple of nheads")
    P = d_inner // nheads
    if x.dtype not in _DTYPES or dt.dtype != x.dtype:
        raise ValueError(f"x and dt must share a supported dtype, got {x.dtype} and {dt.dtype}")
    if chunk_size < 1 or L % chunk_size != 0:
        raise ValueError(f"seqlen {L} is not a multiple of chunk size {chunk_size}")
    dev = _device_check(x, dt, conv_weight, dt_bias, A_log)
    d = _dims(b, L, nheads, P, dstate, ngroups, chunk_size)
    prm, _keep = _layer_params(conv_weight, conv_bias, dt_bias, A_log, None, d_inner, nheads, x.dtype, dev)
    x, dt = _rows3(x), _rows3(dt)
    X = torch.empty((b, L, nheads, P), dtype=x.dtype, device=dev)
    dto = torch.empty((b, L, nheads), dtype=torch.float32, device=dev)
    c = L // chunk_size
    Acs = torch.empty((b, nheads, c, chunk_size), dtype=torch.float32, device=dev)
    dec = torch.empty((b, nheads, c), dtype=torch.float32, device=dev)
    _lib.check(_lib.load().ssd_layer_prep(
        ctypes.byref(d), _DTYPES[x.dtype], ctypes.byref(prm), _ptr(x), _lib.strides(x), _ptr(dt),
        _lib.strides(dt), _ptr(X), _ptr(dto), _ptr(Acs), _ptr(dec), _stream(dev)))
    return X, dto, Acs, dec


def ssd_layer(x, z, B, C, dt, conv_weight, conv_bias, dt_bias, A_log, D, chunk_size, nheads):
    """SSDLayer.forward between its projections (MR:76-118), one C-ABI call:
    pre-SSD prep, the SSD core and the skip + gate fused into its output.

    ``x``, ``z`` [b, L, h*P]; ``B``, ``C`` [b, L, g, N]; ``dt`` [b, L, h] --
    in_proj's output slices, all of one dtype (MR: float16).  ``conv_weight``
    [h*P, 1, k], ``conv_bias`` [h*P] or None, ``dt_bias`` [h], ``A_log`` [h],
    ``D`` [h] or None: MR's parameters.  Returns y [b, L, h*P] in x's dtype,
    out_proj's input."""
    key = (_layout_key(x), _layout_key(z), _layout_key(B), _layout_key(C), _layout_key(dt), _layout_key(conv_weight),
           _layout_key(conv_bias), _layout_key(dt_bias), _layout_key(A_log), _layout_key(D), chunk_size, nheads)
    plan = _LAYER_PLANS.get(key)
    if plan is None or not _aligned(B, C, A_log):
        return _ssd_layer(x, z, B, C, dt, conv_weight, conv_bias, dt_bias, A_log, D, chunk_size, nheads, key)
    dev = x.device
    Dv = None if D is None else _f32_contig(D)
    prm = _lib.SSDLayerParams(plan.width, conv_weight.data_ptr(), 0 if conv_bias is None else conv_bias.data_ptr(),
                              dt_bias.data_ptr(), A_log.data_ptr(), 0 if Dv is None else Dv.data_ptr())
    sx, sz, sb, sc, sdt, sy = plan.strides
    ws = torch.empty(max(plan.nbytes, 1), dtype=torch.uint8, device=dev)
    y = torch.empty(x.shape, dtype=x.dtype, device=dev)
    _lib.check(_lib.load().ssd_layer_forward(
        ctypes.byref(plan.dims), plan.dtype, ctypes.byref(prm), x.data_ptr(), sx, z.data_ptr(), sz, B.data_ptr(), sb,
        C.data_ptr(), sc, dt.data_ptr(), sdt, y.data_ptr(), sy, ws.data_ptr(), plan.nbytes, _stream_fast(dev)))
    return y


def _ssd_layer(x, z, B, C, dt, conv_weight, conv_bias, dt_bias, A_log, D, chunk_size, nheads, key):
    """The checks, operand conversions and call of ssd_layer (and its plan for the layout)."""
    b, L, d_inner = x.shape
    if z.shape != x.shape or dt.shape != (b, L, nheads) or d_inner % nheads != 0:
        raise ValueError("x and z must be [b, L, h*P] and dt [b, L, h]")
    if B.dim() != 4 or B.shape[:2] != (b, L) or C.shape != B.shape:
        raise ValueError(f"B and C must be [b, L, g, N], got {tuple(B.shape)} and {tuple(C.shape)}")
    P = d_inner // nheads
    g, N = B.shape[2], B.shape[3]
    if nheads % g != 0:
        raise ValueError("n_heads must be divisible by n_groups")
    if chunk_size < 1 or L % chunk_size != 0:
        raise ValueError(f"seqlen {L} is not a multiple of chunk size {chunk_size}")
    dtype = x.dtype
    if dtype not in _DTYPES or any(t.dtype != dtype for t in (z, B, C, dt)):
        raise ValueError("x, z, B, C and dt must share a supported dtype")
    dev = _device_check(x, z, B, C, dt, conv_weight, dt_bias, A_log)
    d = _dims(b, L, nheads, P, N, g, chunk_size)
    prm, keep = _layer_params(conv_weight, conv_bias, dt_bias, A_log, D, d_inner, nheads, dtype, dev)
    given = (x, z, dt, B, C)
    x, z, dt = _rows3(x), _rows3(z), _rows3(dt)
    Bm, Cm = _vec_operand(B.detach()), _vec_operand(C.detach())
    lib = _lib.load()
    nbytes = lib.ssd_layer_workspace_bytes(ctypes.byref(d), _DTYPES[dtype])
    ws = torch.empty(max(nbytes, 1), dtype=torch.uint8, device=dev)
    y = torch.empty((b, L, d_inner), dtype=dtype, device=dev)
    strides = tuple(_lib.strides(t) for t in (x, z, Bm, Cm, dt, y))
    _lib.check(lib.ssd_layer_forward(
        ctypes.byref(d), _DTYPES[dtype], ctypes.byref(prm), _ptr(x), strides[0], _ptr(z), strides[1],
        _ptr(Bm), strides[2], _ptr(Cm), strides[3], _ptr(dt), strides[4], _ptr(y), strides[5], _ptr(ws), nbytes,
        _stream(dev)))
    # the same layout next time, where nothing but D was copied or converted
    w, bias, dtb, alog, _ = keep
    as_is = (all(_unchanged(t, t0) for t, t0 in zip((x, z, dt, Bm, Cm), given))
             and all((t is None and t0 is None) or (t.data_ptr() == t0.data_ptr() and t.dtype == t0.dtype)
                     for t, t0 in ((w, conv_weight), (bias, conv_bias), (dtb, dt_bias), (alog, A_log))))
    if as_is and len(_LAYER_PLANS) < _PLANS_MAX:
        _LAYER_PLANS[key] = _LayerPlan(d, _DTYPES[dtype], conv_weight.shape[-1], strides, nbytes)
    return y
