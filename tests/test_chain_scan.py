"""The chain walk (csrc/ssd_chain_scan.hip): ssd_forward and ssd_layer on 16-bit
inputs at d_state 128 with at least ten (chain, 64-token step) pairs per CU.

GPU: against the float64 oracle (chunked evaluation at 64), at shapes that
take one segment, segments whose entering state each workgroup forms itself
(up to 4) and segments that state_passing finishes (each shape's plan is
asserted), with ragged last segments, both types, dt, an initial state, strided operands and state rows
outside f16's range.  y within 2e-2 (the 16-bit tolerance); the final state,
whose products run on hi + lo pairs of the input type, to f32 accuracy: the
pair is within 2^-17 of each product, so 3e-5 of max|state| (as
tests/test_gpu_parity.py holds chunk_state).

CPU: the per-lane LDS address formulas, restated and pinned to the source."""

import ctypes
import os
import re
import subprocess

import numpy as np
import pytest
import torch

from oracle import ssd_oracle as O
from test_address_bounds import inside, pin
from workloadsuite_amd import _lib, build
from workloadsuite_amd import ssd as S

DEV = "cuda"
F = "ssd_chain_scan.hip"


def case(dtype, b, L, h, g, seed, scale=None):
    gen = torch.Generator().manual_seed(seed)
    X = torch.randn(b, L, h, 64, generator=gen)
    if scale is not None:
        X = X * scale
    A = -torch.rand(b, L, h, generator=gen) * 0.2
    B = torch.randn(b, L, g, 128, generator=gen) * 128 ** -0.5
    C = torch.randn(b, L, g, 128, generator=gen) * 128 ** -0.5
    dt = torch.rand(b, L, h, generator=gen) + 0.1
    init = torch.randn(b, h, 64, 128, generator=gen)
    return X.to(dtype), A, B.to(dtype), C.to(dtype), dt, init


def check(Y, final, ref, fref, tol=2e-2):
    torch.testing.assert_close(Y.double().cpu(), ref, rtol=tol, atol=tol)
    torch.testing.assert_close(final.double().cpu(), fref, rtol=0, atol=3e-5 * fref.abs().max().item())


SHAPES = [
    # b, L, h, g: one segment (512 chains of 6 steps); eight; 49 (16 chains of
    # 193 steps); a prime number of steps; six heads per group
    (8, 384, 64, 4),
    (2, 2496, 64, 8),
    (1, 12352, 16, 2),
    (1, 64 * 67, 48, 1),
    (3, 1088, 96, 16),
]


# b, L, h, g: segments, steps per segment, heads per workgroup, linked by a launch of their own, S as a hi + lo pair
PLANS = {
    (8, 384, 64, 4): (1, 6, 2, False, False),
    (2, 2496, 64, 8): (8, 5, 2, True, False),
    (1, 12352, 16, 2): (49, 4, 2, True, False),
    (1, 64 * 67, 48, 1): (17, 4, 2, True, False),
    (3, 1088, 96, 16): (1, 17, 2, False, False),
    # entering states formed by each workgroup: four segments (groups of 80 heads) and three (of six)
    (3, 1216, 80, 1): (4, 5, 2, False, False),
    (3, 1472, 48, 8): (3, 8, 2, False, False),
    # groups of six heads, linked by a launch
    (3, 2368, 24, 4): (7, 6, 2, True, False),
    # strided operands
    (2, 1344, 64, 4): (7, 3, 2, True, False),
}
GATED_PLANS = {
    (8, 384, 128, 8): (1, 6, 4, False, True),
    (2, 1216, 128, 8): (4, 5, 4, False, True),
    (1, 2752, 64, 1): (15, 3, 4, True, True),
    # two heads per workgroup
    (4, 512, 128, 8): (1, 8, 2, False, False),
    (3, 1216, 96, 8): (1, 19, 2, False, True),
    (1, 2752, 96, 16): (5, 9, 2, True, True),
    (3, 1472, 48, 8): (3, 8, 2, False, True),
    (3, 1344, 96, 8): (3, 7, 2, False, True),
    # lengths that 256 divides: four heads per workgroup, two (one segment above), and two segments of groups of six
    (8, 256, 128, 8): (1, 4, 4, False, False),
    (5, 1024, 48, 8): (2, 8, 2, False, False),
}


@pytest.mark.parametrize("gated", [False, True])
def test_plans(gated):
    """Every shape of the GPU tests below takes the walk it is there for (256 CUs)."""
    for (b, L, h, g), want in (GATED_PLANS if gated else PLANS).items():
        for dtype in (torch.bfloat16, torch.float16):
            assert S.walk_plan(b, L, h, 64, 128, g, 64, dtype, gated=gated) == want, (b, L, h, g)
    assert {k[:4] for k in SHAPES + MORE_SHAPES} <= set(PLANS)
    assert {k for k in SPANS + SPANS_TWO} == set(GATED_PLANS)
    # what the walk does not take: a named hand-over format, an odd number of heads per group, d_state 64, small calls
    assert S.walk_plan(8, 384, 64, 64, 128, 4, 64, torch.float16, state_format="f16s") is None
    assert S.walk_plan(8, 384, 64, 64, 128, 64, 64, torch.float16) is None
    assert S.walk_plan(8, 384, 64, 64, 64, 4, 64, torch.float16) is None
    assert S.walk_plan(1, 384, 64, 64, 128, 4, 64, torch.float16) is None


def on_the_walk(b, L, h, g, dtype, gated=False):
    """The call below runs the walk planned above also on this device."""
    got = S.walk_plan(b, L, h, 64, 128, g, 64, dtype, gated=gated)
    assert got == (GATED_PLANS if gated else PLANS)[b, L, h, g], got


MORE_SHAPES = [(3, 1216, 80, 1), (3, 1472, 48, 8), (3, 2368, 24, 4)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,L,h,g", SHAPES + MORE_SHAPES)
@pytest.mark.parametrize("opts", [True, False])
def test_forward(dtype, b, L, h, g, opts):
    on_the_walk(b, L, h, g, dtype)
    print("CASE chain walk", dtype, b, L, h, g, opts, flush=True)
    X, A, B, C, dt, init = case(dtype, b, L, h, g, seed=L + h)
    dt, init = (dt, init) if opts else (None, None)
    hs = [0, 1, h // 2, h - 1]   # heads of the first, a middle and the last workgroup
    grp = [k // (h // g) for k in hs]
    ref, fref = O.ssd_chunked(X[:, :, hs], A[:, :, hs], B[:, :, grp], C[:, :, grp], 64,
                              dt=None if dt is None else dt[:, :, hs], initial_states=None if init is None else init[:, hs])
    d = lambda t: None if t is None else t.to(DEV)  # noqa: E731
    Y, final = S.ssd_forward(d(X), d(A), d(B), d(C), 64, dt=d(dt), initial_states=d(init), return_final_states=True)
    torch.cuda.synchronize()
    assert torch.isfinite(Y).all() and torch.isfinite(final).all()
    check(Y[:, :, hs], final[:, hs], ref, fref)


@pytest.mark.gpu
def test_state_rows_outside_f16():
    """x scaled per column p over 16 decades (states from ~1e-9 to ~1e6): rows
    take their power-of-two scale.  Each column of y against its own scale."""
    print("CASE chain walk, wide rows", flush=True)
    col = torch.logspace(-9, 6, 64)
    X, A, B, C, dt, init = case(torch.bfloat16, 8, 384, 64, 4, seed=5, scale=col)
    init = init * col[:, None]
    hs = [0, 31, 63]
    grp = [k // 16 for k in hs]
    ref, fref = O.ssd_chunked(X[:, :, hs], A[:, :, hs], B[:, :, grp], C[:, :, grp], 64, dt=dt[:, :, hs],
                              initial_states=init[:, hs])
    Y, final = S.ssd_forward(*(t.to(DEV) for t in (X, A, B, C)), 64, dt=dt.to(DEV), initial_states=init.to(DEV),
                             return_final_states=True)
    torch.cuda.synchronize()
    check(Y[:, :, hs].double().cpu() / col, final[:, hs].double().cpu() / col[:, None].double(), ref / col,
          fref / col[:, None])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,L,h,g", [(8, 384, 64, 4), (3, 1216, 80, 1), (2, 2496, 64, 8)])
@pytest.mark.parametrize("small", [-12, -20, -24])
def test_small_entries_of_a_state_row(dtype, b, L, h, g, small):
    """C picks entries 2^small below their row's largest: with the row scaled to
    [2^14, 2^15) they keep f16's 11 bits down to 2^-29 of it, so y is within the
    rounding of S (half an ulp of 11 bits: 2^-11) and its own (2^-11 in f16, 2^-8
    in bf16)."""
    print("CASE chain walk, small entries", dtype, b, L, h, g, small, flush=True)
    on_the_walk(b, L, h, g, dtype)
    gen = torch.Generator().manual_seed(4)
    init = torch.zeros(b, h, 64, 128)
    init[..., 3] = 1 + torch.rand(b, h, 64, generator=gen)             # the row's largest
    init[..., 40] = (1 + torch.rand(b, h, 64, generator=gen)) * 2.0 ** small
    C = torch.zeros(b, L, g, 128)
    C[..., 40] = 2.0 ** min(-small, 15)
    X, A, B = torch.zeros(b, L, h, 64), torch.zeros(b, L, h), torch.zeros(b, L, g, 128)
    Y = S.ssd_forward(X.to(DEV, dtype), A.to(DEV), B.to(DEV, dtype), C.to(DEV, dtype), 64, initial_states=init.to(DEV))
    want = (init[..., 40].double() * 2.0 ** min(-small, 15)).to(DEV)[:, None]
    eps = 2.0 ** -11 + (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11)
    assert ((Y.double() - want).abs() <= 1.01 * eps * want).all()


@pytest.mark.gpu
def test_scales_of_c_and_s_cancel():
    """C near bf16's largest values times a tiny state: the two scales are
    multiplied first, so that neither alone overflows the sum."""
    print("CASE chain walk, scales cancel", flush=True)
    b, L, h, g = 8, 384, 64, 4
    on_the_walk(b, L, h, g, torch.bfloat16)
    init = torch.full((b, h, 64, 128), 2.0 ** -80, device=DEV)
    C = torch.full((b, L, g, 128), 2.0 ** 114, device=DEV, dtype=torch.bfloat16)
    X, A = torch.zeros(b, L, h, 64, device=DEV, dtype=torch.bfloat16), torch.zeros(b, L, h, device=DEV)
    Y = S.ssd_forward(X, A, torch.zeros_like(C), C, 64, initial_states=init)
    assert (Y == 2.0 ** 41).all()


@pytest.mark.gpu
def test_strided_operands_match_contiguous_ones():
    """x, B, C as column slices of a wider tensor, A and dt transposed: the bits of the contiguous call."""
    print("CASE chain walk, strides", flush=True)
    L = 1344
    on_the_walk(2, L, 64, 4, torch.float16)
    X, A, B, C, dt, init = (t.to(DEV) for t in case(torch.float16, 2, L, 64, 4, seed=9))
    wide = torch.zeros(2, L, 64 * 64 + 2 * 4 * 128 + 16, device=DEV, dtype=torch.float16)
    xs, bs, cs = wide[..., 8:8 + 4096], wide[..., 4104:4104 + 512], wide[..., 4616:4616 + 512]
    xs.copy_(X.flatten(2)), bs.copy_(B.flatten(2)), cs.copy_(C.flatten(2))
    At, dtt = A.transpose(1, 2).contiguous().transpose(1, 2), dt.transpose(1, 2).contiguous().transpose(1, 2)
    Y0, f0 = S.ssd_forward(X, A, B, C, 64, dt=dt, initial_states=init, return_final_states=True)
    Y1, f1 = S.ssd_forward(xs.unflatten(2, (64, 64)), At, bs.unflatten(2, (4, 128)), cs.unflatten(2, (4, 128)), 64, dt=dtt,
                           initial_states=init, return_final_states=True)
    torch.cuda.synchronize()
    assert torch.equal(Y0, Y1) and torch.equal(f0, f1)


@pytest.mark.gpu
@pytest.mark.parametrize("b,L,h,g", [(3, 1216, 80, 1), (3, 1472, 48, 8), (2, 2496, 64, 8)])
def test_growth_beyond_f32_over_a_segment(b, L, h, g):
    """Log-decays of +0.4 over the first 256 tokens (a factor e^102) with x zero
    there: no state exists yet, and the rest is as if the sequence began later.
    (bf16: in f16 the weights of one 64-token block, up to e^25, are infinite.)"""
    print("CASE chain walk, growth over a segment", b, L, h, g, flush=True)
    dtype = torch.bfloat16
    on_the_walk(b, L, h, g, dtype)
    assert PLANS[b, L, h, g][0] > 1 and PLANS[b, L, h, g][1] > 4
    X, A, B, C, dt, _ = case(dtype, b, L, h, g, seed=6)
    A[:, :256] = 0.4
    X[:, :256] = 0
    hs = [0, h // 2, h - 1]
    grp = [k // (h // g) for k in hs]
    ref, fref = O.ssd_chunked(*(t[:, 256:] for t in (X[:, :, hs], A[:, :, hs], B[:, :, grp], C[:, :, grp])), 64,
                              dt=dt[:, 256:, hs])
    Y, final = S.ssd_forward(*(t.to(DEV) for t in (X, A, B, C)), 64, dt=dt.to(DEV), return_final_states=True)
    check(Y[:, 256:, hs], final[:, hs], ref, fref)
    assert (Y[:, :256] == 0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("what", ["x", "B", "C"])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("b,L,h,g", [(8, 384, 64, 4), (3, 1216, 80, 1)])
def test_one_bad_value(b, L, h, g, what, bad):
    """An infinity or NaN reaches the outputs it belongs to (the products of a
    32-token block see the whole block, as in the stage kernels) and no others:
    those keep their bits."""
    print("CASE chain walk, one bad value", b, L, h, g, what, bad, flush=True)
    on_the_walk(b, L, h, g, torch.bfloat16)
    X, A, B, C, dt, _ = (t.to(DEV) for t in case(torch.bfloat16, b, L, h, g, seed=1))
    call = lambda: S.ssd_forward(X, A, B, C, 64, dt=dt, return_final_states=True)  # noqa: E731
    Y0, f0 = call()
    l, bb = 64 * (L // 128) + 37, b - 1  # noqa: E741
    hit = torch.zeros_like(Y0, dtype=torch.bool)       # what may change
    fhit = torch.zeros_like(f0, dtype=torch.bool)
    if what == "x":
        X[bb, l, 5, 9] = bad
        hit[bb, l - l % 32:, 5, 9] = True
        fhit[bb, 5, 9] = True
    elif what == "B":
        B[bb, l, 0, 77] = bad
        hit[bb, l:, :h // g] = True
        fhit[bb, :h // g, :, 77] = True
    else:
        C[bb, l, 0, 77] = bad
        hit[bb, l, :h // g] = True
    Y, final = call()
    torch.cuda.synchronize()
    assert torch.equal(Y[~hit], Y0[~hit]) and torch.equal(final[~fhit], f0[~fhit])
    own = Y[bb, l, 5, 9] if what == "x" else Y[bb, l, :h // g]
    assert not torch.isfinite(own).any()
    if what != "C":
        assert not torch.isfinite(final[fhit]).any()


def test_in_place_state_waits_for_every_segment():
    """With final_states = initial_states no workgroup of a cut chain may read the
    initial state: at 6 x 16384 tokens of 112 heads 1008 workgroups share 512 places,
    so the last segment of a chain can end before an earlier one starts."""
    segs, _, heads, linked, _ = S.walk_plan(6, 16384, 112, 64, 128, 1, 64, torch.bfloat16)
    assert (segs, linked) == (3, False) and 6 * segs * 112 // heads > 512
    for b, L, h, g in [(6, 16384, 112, 1), (3, 1216, 80, 1), (3, 1472, 48, 8), (2, 2496, 64, 8)]:
        assert S.walk_plan(b, L, h, 64, 128, g, 64, torch.bfloat16, in_place=True).linked
    assert not S.walk_plan(8, 384, 64, 64, 128, 4, 64, torch.bfloat16, in_place=True).linked  # whole chains


@pytest.mark.gpu
@pytest.mark.parametrize("b,L,h,g", [(8, 384, 64, 4), (3, 1216, 80, 1), (3, 1472, 48, 8), (2, 2496, 64, 8)])
def test_state_updated_in_place(b, L, h, g):
    """ssd_forward of the C ABI with final_states = initial_states: y and the state
    of a call with two buffers (to the order in which the segments are linked)."""
    print("CASE chain walk, in place", b, L, h, g, flush=True)
    X, A, B, C, dt, init = (t.to(DEV) for t in case(torch.float16, b, L, h, g, seed=2))
    Y0, f0 = S.ssd_forward(X, A, B, C, 64, dt=dt, initial_states=init, return_final_states=True)
    n = S.workspace_bytes(b, L, h, 64, 128, g, 64)
    ws, Y = torch.empty(n, dtype=torch.uint8, device=DEV), torch.empty_like(X)
    d, lib = _lib.dims(b, L, h, 64, 128, g, 64), _lib.load()
    st = _lib.strides
    _lib.check(lib.ssd_forward(ctypes.byref(d), _lib.DTYPE_F16, X.data_ptr(), st(X), A.data_ptr(), st(A), B.data_ptr(), st(B),
                               C.data_ptr(), st(C), dt.data_ptr(), st(dt), init.data_ptr(), Y.data_ptr(), st(Y),
                               init.data_ptr(), ws.data_ptr(), n, _lib.DTYPE_F32, torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    # one f32 rounding per linked segment apart; y one f16 rounding where that crosses a boundary
    torch.testing.assert_close(init, f0, rtol=0, atol=1e-6 * f0.abs().max().item())
    torch.testing.assert_close(Y.float(), Y0.float(), rtol=2e-3, atol=2e-3)


SPANS = [(8, 384, 128, 8), (2, 1216, 128, 8), (1, 2752, 64, 1), (8, 256, 128, 8)]


# chunk 128, odd multiples: one segment, four, fourteen linked ones, three of groups of six heads
CHUNK_128 = {(4, 640, 64, 8): (1, 10, 2, False, True), (3, 1152, 80, 1): (4, 5, 2, False, True),
             (1, 2688, 64, 8): (14, 3, 2, True, True), (3, 1152, 48, 8): (3, 6, 2, False, True)}


def test_state_operand_follows_the_stage_kernels():
    """S enters C.S as a hi + lo pair where the stage kernels take it so (chunk
    128, the gate at lengths that 256 does not divide), else as f16 rows."""
    for dtype in (torch.bfloat16, torch.float16):
        for (b, L, h, g), want in CHUNK_128.items():
            assert S.walk_plan(b, L, h, 64, 128, g, 128, dtype) == want
        for b, L, h, g, chunk, gated, hilo in [(4, 640, 64, 8, 64, False, False), (4, 1024, 80, 1, 128, False, False),
                                               (4, 1024, 80, 1, 256, False, False), (8, 384, 128, 8, 128, True, True),
                                               (8, 512, 128, 8, 128, True, False), (8, 512, 128, 8, 64, True, False)]:
            assert S.walk_plan(b, L, h, 64, 128, g, chunk, dtype, gated=gated).hilo == hilo, (L, chunk, gated)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,L,h,g", list(CHUNK_128))
@pytest.mark.parametrize("opts", [True, False])
def test_forward_chunk_128(dtype, b, L, h, g, opts):
    """As test_forward, at chunk 128; then a state whose entries nearly cancel:
    y = S[3] - S[40] with S[3] = (1 + 1.5 2^-11) S[40], which 11 bits of S do not
    resolve.  A bf16 pair of values below 2 is within 2^-17 of each (2^-16 of the
    larger binade), an f16 pair closer; y's own rounding is 2^-8 (bf16)."""
    print("CASE chain walk, chunk 128", dtype, b, L, h, g, opts, flush=True)
    assert S.walk_plan(b, L, h, 64, 128, g, 128, dtype) == CHUNK_128[b, L, h, g]
    X, A, B, C, dt, init = case(dtype, b, L, h, g, seed=L + h)
    dt, init = (dt, init) if opts else (None, None)
    hs = [0, 1, h // 2, h - 1]
    grp = [k // (h // g) for k in hs]
    ref, fref = O.ssd_chunked(X[:, :, hs], A[:, :, hs], B[:, :, grp], C[:, :, grp], 64,
                              dt=None if dt is None else dt[:, :, hs], initial_states=None if init is None else init[:, hs])
    d = lambda t: None if t is None else t.to(DEV)  # noqa: E731
    Y, final = S.ssd_forward(d(X), d(A), d(B), d(C), 128, dt=d(dt), initial_states=d(init), return_final_states=True)
    check(Y[:, :, hs], final[:, hs], ref, fref)
    state = torch.zeros(b, h, 64, 128, device=DEV)
    state[..., 40] = 1 + torch.rand(b, h, 64, device=DEV)
    state[..., 3] = state[..., 40] * (1 + 1.5 * 2.0 ** -11)
    C = torch.zeros(b, L, g, 128, device=DEV, dtype=dtype)
    C[..., 3], C[..., 40] = 1, -1
    zero = lambda t: torch.zeros_like(t, device=DEV)  # noqa: E731
    Y = S.ssd_forward(zero(X), zero(A), zero(B), C, 128, dt=d(dt), initial_states=state)
    want = (state[..., 3].double() - state[..., 40].double())[:, None]
    assert ((Y.double() - want).abs() <= 2 * 2.0 ** -16 + 2.0 ** -8 * want).all()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,L,h,g", [(8, 384, 128, 8), (2, 1216, 128, 8), (3, 1216, 96, 8), (3, 1472, 48, 8)])
def test_layer_span_resolves_the_state(dtype, b, L, h, g):
    """The same near-cancellation in the gated walk: S[3] - S[40] = 1.5 2^-11 S[40]
    from the first two tokens, read by all from the second 64 on."""
    print("CASE chain walk, gated, near-cancelling state", dtype, b, L, h, g, flush=True)
    on_the_walk(b, L, h, g, dtype, gated=True)
    assert GATED_PLANS[b, L, h, g][4]
    x = torch.zeros(b, L, h * 64, device=DEV)
    x[:, 0] = x[:, 1] = 1 + torch.rand(b, h * 64, device=DEV)
    B, C = torch.zeros(2, b, L, g, 128, device=DEV, dtype=dtype)
    B[:, 0, :, 3] = B[:, 0, :, 40] = 1
    B[:, 1, :, 3] = 1.5 * 2.0 ** -11
    C[..., 3], C[..., 40] = 1, -1
    z = torch.full((b, L, h * 64), 8.0, device=DEV, dtype=dtype)
    dt = torch.full((b, L, h), 0.5, device=DEV, dtype=dtype)
    w = torch.zeros(h * 64, 1, 4, device=DEV, dtype=dtype)
    w[..., 3] = 1
    zero = torch.zeros(h, device=DEV)
    x = x.to(dtype)
    y = S.ssd_layer(x, z, B, C, dt, w, None, zero.to(dtype), zero - 30, zero, 64, h)
    # x as the conv leaves it, dt = softplus(0.5), decays 1 - 1e-10
    xv = torch.nn.functional.silu(x[:, 0].double()).to(dtype).double() * torch.nn.functional.softplus(dt[0, 0, 0].double())
    gate = torch.nn.functional.silu(torch.tensor(8.0, dtype=torch.float64, device=DEV))
    want = (xv * 1.5 * 2.0 ** -11 * gate)[:, None]
    # S below 4: a pair is within 2^-15 of each entry; x's rounding after the conv may differ by an ulp (2^-8)
    assert ((y[:, 64:].double() - want).abs() <= gate * 2 * 2.0 ** -15 + 2 * 2.0 ** -8 * want).all()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,L,h,g", SPANS)
def test_layer_span(dtype, b, L, h, g):
    """The gated variant with four heads per workgroup (one segment, four, and
    fifteen; S as a hi + lo pair, and at 256 tokens as f16 rows) against the stage entry points on the same prepared operands, 2e-2."""
    on_the_walk(b, L, h, g, dtype, gated=True)
    from test_layer_kernels import layer_case, split
    print("CASE chain walk, layer span", dtype, b, L, h, g, flush=True)
    proj, prm = layer_case(dtype, b=b, L=L, h=h, P=64, g=g, N=128)
    x, z, B, C, dt = split(proj.to(DEV), h, 64, g, 128)
    p = {k: v.to(DEV) for k, v in prm.items()}
    y = S.ssd_layer(x, z, B, C, dt, p["conv_w"], p["conv_b"], p["dt_bias"], p["A_log"], p["D"], 64, h)
    X, dto, Acs, dec = S.layer_prep(x, dt, p["conv_w"], p["conv_b"], p["dt_bias"], p["A_log"], 64, h)
    S_in, _ = S.chunk_state_passing(X, B, Acs, dec, dt=dto)
    ref = S.chunk_scan(X, B, C, Acs, S_in, dt=dto, D=p["D"], z=z.reshape(b, L, h, 64))
    torch.cuda.synchronize()
    torch.testing.assert_close(y.float(), ref.reshape(b, L, -1).float(), rtol=2e-2, atol=2e-2)


SPANS_TWO = [(4, 512, 128, 8), (3, 1216, 96, 8), (1, 2752, 96, 16), (3, 1472, 48, 8), (3, 1344, 96, 8), (5, 1024, 48, 8)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,L,h,g", SPANS_TWO)
def test_layer_span_two_heads(dtype, b, L, h, g):
    """The gated variant with two heads per workgroup: whole chains, and in
    segments with groups of six and of twelve heads.  Against the stage entry
    points, 2e-2, and a second call gives the bits of the first."""
    on_the_walk(b, L, h, g, dtype, gated=True)
    from test_layer_kernels import layer_case, split
    print("CASE chain walk, layer span, two heads", dtype, b, L, h, g, flush=True)
    proj, prm = layer_case(dtype, b=b, L=L, h=h, P=64, g=g, N=128)
    x, z, B, C, dt = split(proj.to(DEV), h, 64, g, 128)
    p = {k: v.to(DEV) for k, v in prm.items()}
    y, y2 = (S.ssd_layer(x, z, B, C, dt, p["conv_w"], p["conv_b"], p["dt_bias"], p["A_log"], p["D"], 64, h) for _ in range(2))
    X, dto, Acs, dec = S.layer_prep(x, dt, p["conv_w"], p["conv_b"], p["dt_bias"], p["A_log"], 64, h)
    S_in, _ = S.chunk_state_passing(X, B, Acs, dec, dt=dto)
    ref = S.chunk_scan(X, B, C, Acs, S_in, dt=dto, D=p["D"], z=z.reshape(b, L, h, 64))
    torch.cuda.synchronize()
    torch.testing.assert_close(y.float(), ref.reshape(b, L, -1).float(), rtol=2e-2, atol=2e-2)
    assert torch.equal(y, y2)


@pytest.mark.gpu
@pytest.mark.parametrize("b,L,h,g", [(8, 384, 64, 4), (3, 1216, 80, 1), (2, 2496, 64, 8)])
def test_captured_in_a_graph(b, L, h, g):
    """A captured walk (one segment; four; eight linked ones) replayed on new
    inputs, with eager calls between: the bits of the eager call each time."""
    print("CASE chain walk, graph", b, L, h, g, flush=True)
    on_the_walk(b, L, h, g, torch.bfloat16)
    sets = [[t.to(DEV) for t in case(torch.bfloat16, b, L, h, g, seed)] for seed in (1, 2, 3)]
    call = lambda X, A, B, C, dt, init: S.ssd_forward(X, A, B, C, 64, dt=dt, initial_states=init,  # noqa: E731
                                                      return_final_states=True)
    args = [t.clone() for t in sets[0]]
    call(*args)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        Y, final = call(*args)
    for s in (sets[1], sets[2], sets[0], sets[1]):
        for t, v in zip(args, s):
            t.copy_(v)
        graph.replay()
        torch.cuda.synchronize()
        Y0, f0 = call(*s)
        torch.cuda.synchronize()
        assert torch.equal(Y, Y0) and torch.equal(final, f0)


# ---------------------------------------------------------------------------
# addresses (CPU)
# ---------------------------------------------------------------------------

def test_lds_addresses():
    """Copies and operand reads of a step meet: every byte of B, C, x and W
    that a lane reads lies inside its buffer and holds the element the
    product needs."""
    pin(F, "return (2 * row) & 14;",
        "const int row = 4 * (DPW * wave + m) + crow;",
        "(cslot ^ bsw(row & 15))", "(cslot ^ (row & 15))",
        "boff[nt] = trow * kN + 8 * ((4 * nt + 2 * (g & 1) + (q & 1)) ^ bsw(trow)) + 4 * (q >> 1);",
        "const int coff = r * kN + 8 * (hl ^ (r & 15));",
        "cl + (coff ^ (16 * kb)) + 32 * t * kN",
        "const int xoff = trow * kP + 8 * ((4 * w + 2 * (g & 1) + (q >> 1)) ^ (trow & 7)) + 4 * (q & 1);",
        "const int q = i & 3, trow = 4 * hl + (i >> 2);",
        "lds_read_tr(bs + boff[nt] + 16 * kb * kN), lds_read_tr(bs + boff[nt] + (16 * kb + 8) * kN)",
        "lds_read_tr(xb + xoff + 16 * kb * kP), lds_read_tr(xb + xoff + (16 * kb + 8) * kP)")
    lane = np.arange(64)
    hl, r, g, i = lane >> 5, lane & 31, lane >> 4, lane & 15
    q, trow = i & 3, 4 * hl + (i >> 2)
    bsw = lambda row: (2 * row) & 14  # noqa: E731
    # LDS images: [row, column] of each 16-bit slot, as the copies place them
    img_b, img_c = np.full((64 * 128, 2), -1), np.full((64 * 128, 2), -1)
    img_x = np.full((64 * 64, 2), -1)
    for d in range(16):
        row, slot = 4 * d + (lane >> 4), lane & 15
        for e in range(8):
            dst = d * 512 + lane * 8 + e
            img_b[dst] = np.stack([row, 8 * (slot ^ bsw(row & 15)) + e], 1)
            img_c[dst] = np.stack([row, 8 * (slot ^ (row & 15)) + e], 1)
    for blk in range(8):
        row = 8 * blk + (lane >> 3)
        for e in range(8):
            img_x[blk * 512 + lane * 8 + e] = np.stack([row, 8 * ((lane & 7) ^ (lane >> 3)) + e], 1)
    for img in (img_b, img_c, img_x):
        assert (img >= 0).all()

    def tr(addr):
        """element [lane] <- 4 consecutive elements through the transposing read: [64, 4] slots"""
        out = np.empty((64, 4), np.int64)
        for k in range(64):
            base, j = k & 48, k & 15
            for rr in range(4):
                out[k, rr] = addr[base + 4 * rr + j // 4] + j % 4
        return out

    for kb in range(4):
        tokens = np.stack([16 * kb + 8 * (j // 4) + 4 * hl + j % 4 for j in range(8)], 1)
        for nt in range(4):
            a0 = trow * 128 + 8 * ((4 * nt + 2 * (g & 1) + (q & 1)) ^ bsw(trow)) + 4 * (q >> 1)
            slots = np.concatenate([tr(a0 + 16 * kb * 128), tr(a0 + (16 * kb + 8) * 128)], 1)
            inside("B", slots, 0, 64 * 128)
            # row r of the tile is n = 32 nt + 16 (k >> 1) + 8 h + 4 (k & 1) + jj for r = 8 k + 4 h + jj
            k, h2, jj = r >> 3, (r >> 2) & 1, r & 3
            n = 32 * nt + 16 * (k >> 1) + 8 * h2 + 4 * (k & 1) + jj
            assert (img_b[slots][..., 0] == tokens).all() and (img_b[slots][..., 1] == n[:, None]).all()
        for w in range(2):
            a0 = trow * 64 + 8 * ((4 * w + 2 * (g & 1) + (q >> 1)) ^ (trow & 7)) + 4 * (q & 1)
            slots = np.concatenate([tr(a0 + 16 * kb * 64), tr(a0 + (16 * kb + 8) * 64)], 1)
            inside("x", slots, 0, 64 * 64)
            assert (img_x[slots][..., 0] == tokens).all() and (img_x[slots][..., 1] == (32 * w + r)[:, None]).all()
    for kb in range(8):
        for t in range(2):
            a0 = ((r * 128 + 8 * (hl ^ (r & 15))) ^ (16 * kb)) + 32 * t * 128
            slots = a0[:, None] + np.arange(8)
            inside("C", slots, 0, 64 * 128)
            assert (img_c[slots][..., 0] == (32 * t + r)[:, None]).all()
            # S's lane values of K step kb: n = 16 kb + 8 hl + j
            assert (img_c[slots][..., 1] == (16 * kb + 8 * hl)[:, None] + np.arange(8)).all()


@pytest.mark.parametrize("src", ["ssd_chain_scan.hip", "ssd_chain_scan_f32.hip"])
def test_counted_waits(src, tmp_path):
    """The compiled kernels: a barrier's counted wait leaves in flight only
    accesses issued after the copies that the barrier publishes, and there are no
    flat accesses, which may retire out of that order.  (The scan's first barrier
    leaves the next step's x copies, its second none; the segment-state kernel's
    leaves the copies of the step after next.)"""
    out = tmp_path / "walk.s"
    cmd = [build.hipcc(), *build.COMMON_FLAGS, *build.DEVICE_FLAGS, "-Wno-error", "--cuda-device-only", "-S",
           os.path.join(build.CSRC, src), "-o", str(out)]
    subprocess.run(cmd, check=True, capture_output=True)
    name, body, seen = None, [], 0
    for ln in out.read_text().splitlines():
        m = re.match(r"(_Z\w+):", ln)
        if m:
            name, body = m.group(1), []
        elif name and re.match(r"\t[a-z]", ln):
            body.append(ln.split(";")[0].strip())
            if body[-1] != "s_endpgm" or "prep" in name:
                continue
            seen += 1
            assert not [x for x in body if x.startswith("flat_")], name
            waits = {}
            for k, x in enumerate(body):
                if x == "s_barrier":
                    at, n = max((j, int(w.group(1))) for j in range(k) if (w := re.search(r"vmcnt\((\d+)\)", body[j])))
                    ops = [y for y in body[:at] if re.match(r"(global|buffer)_", y)]
                    waits[n] = len([y for y in ops[len(ops) - n:] if "_lds_" in y])
            if "state_kernel" in name:
                assert len(waits) == 1 and all(n == copies > 0 for n, copies in waits.items()), (name, waits)
            elif "f32" in src:
                assert waits == {0: 0, 40: 0}, (name, waits)
            else:
                gated = re.search(r"ELb[01]ELb([01])ELb[01]EEEvNS_13ChainScanArgsE$", name).group(1) == "1"
                assert waits == {0: 0, 9: 0, 8 if gated else 4: 4}, (name, waits)
    assert seen == {"ssd_chain_scan.hip": 24, "ssd_chain_scan_f32.hip": 4}[src]


def test_w_tiles():
    """The ten causal tiles, five per wave, fill their halves of W's blocks in
    the order the diagonal product reads them; the two tiles above the
    diagonal inside the blocks are the zeroed ones."""
    pin("ssd_chain_step.h", "constexpr int kT[5] = {0, 2, 1, 2, 2}, kDT[5] = {1, 1, 2, 1, 1};",
        "constexpr int kS[5] = {0, 2, 0, 0, 1}, kDS[5] = {1, 1, 2, 1, -1};")
    pin(F, "constexpr int dS[3] = {1, 2, -1}, dW[3] = {512 + 128, 2048, -512 + 128};",
        "asoff[k] = 16 * dS[k] * w + 4 * g;", "woff[k] = dW[k] * w + ((g & 1) * 32 + i) * 8 + 4 * (g >> 1);",
        "if (k < 2) aloff[k] = 16 * dS[k] * w + i;",
        "constexpr int kDI[5] = {0, 0, 1, 0, 2}, kTI[5] = {0, 0, 1, 0, 0};",
        "woff[kDI[kb]] + ((t0 >> 1) * 2 + s0) * 512 + (t0 & 1) * 128",
        "&wl[hh][(w == 0 ? 1 : 5) * 512 + ((g & 1) * 32 + i) * 8 + 4 * (g >> 1)]")
    kT, kDT, kS, kDS = [0, 2, 1, 2, 2], [1, 1, 2, 1, 1], [0, 2, 0, 0, 1], [1, 1, 2, 1, -1]
    dS, dW, kDI, kTI = [1, 2, -1], [640, 2048, -384], [0, 0, 1, 0, 2], [0, 0, 1, 0, 0]
    lane = np.arange(64)
    g, i = lane >> 4, lane & 15
    img = np.full((6 * 512, 2), -1)   # (s, l) of each slot of W
    for w in range(2):
        zero = (1 if w == 0 else 5) * 512 + ((g & 1) * 32 + i) * 8 + 4 * (g >> 1)
        for jj in range(4):
            img[zero + jj] = -2
    seen = set()
    for w in range(2):
        for m in range(5):
            t, s = kT[m] + kDT[m] * w, kS[m] + kDS[m] * w
            assert 0 <= s <= t <= 3 and (s == t) == (m < 2)
            seen.add((t, s))
            assert (16 * dS[kDI[m]] * w + 4 * g + 16 * kS[m] == 16 * s + 4 * g).all()
            assert (16 * dS[kTI[m]] * w + i + 16 * kT[m] == 16 * t + i).all()
            at = dW[kDI[m]] * w + ((g & 1) * 32 + i) * 8 + 4 * (g >> 1) + ((kT[m] >> 1) * 2 + kS[m]) * 512 + (kT[m] & 1) * 128
            inside("W", at, 0, 6 * 512 - 3)
            for jj in range(4):
                assert (img[at + jj] == -1).all()
                img[at + jj] = np.stack([16 * s + 4 * g + jj, 16 * t + i], 1)
    assert len(seen) == 10
    hl, r = lane >> 5, lane & 31
    for blk, (tile, kb) in enumerate([(0, 0), (0, 1), (1, 0), (1, 1), (1, 2), (1, 3)]):
        for j in range(8):
            got = img[blk * 512 + lane * 8 + j]
            s = 16 * kb + 8 * (j // 4) + 4 * hl + j % 4
            l = 32 * tile + r  # noqa: E741
            above = (s // 16) > (l // 16)
            assert (got[above] == -2).all()
            assert (got[~above, 0] == s[~above]).all() and (got[~above, 1] == l[~above]).all()
