"""The one-kernel Winograd conv (csrc/winograd_fused.hip) where split sums are not
finite, or too small for their operands' bits: the workgroups that met one do their
items again on the f32 instructions, so outputs and GroupNorm partials are what the
f32 products give, for odd values in the input and in the weights, with the residual,
the prologue and the upsample."""
from __future__ import annotations

import ctypes
import time

import numpy as np
import pytest

import oracle
from moebius_cpu_amd import engine as E
from tests.test_gpu_split import odd_values, same_kind
from tests.util import rel_l2

pytestmark = pytest.mark.gpu
HUGE = np.float32(3.4e38)  # finite, and infinite as a bf16


@pytest.fixture(scope="module")
def ctx():
    c = E.Context(0)
    yield c
    c.synchronize()
    c.close()


def conv(ctx, x, wt, b, up=False, aff=None, res=None):
    """The conv's output, its GroupNorm partials (blocks, c_out, 2) and the pixels per block."""
    n, h, w, ci = x.shape
    co, s = wt.shape[0], 2 if up else 1
    cv = E.Conv3x3(ctx, ci, co, E.Param(ctx, wt), b, upsample2x=up, winograd=True)
    dev = {k: E.DeviceArray.from_numpy(ctx, v) for k, v in
           dict(x=x, b=b, r=res, sc=aff and aff[0], sh=aff and aff[1]).items() if v is not None}
    ptr = {k: dev[k].ptr if k in dev else None for k in ("x", "b", "r", "sc", "sh")}
    tiles = n * -(-h * s // 2) * -(-w * s // 2)
    out = E.DeviceArray(ctx, (n, h * s, w * s, co))
    part = E.DeviceArray(ctx, (-(-tiles // 32), co, 2))
    rows = ctypes.c_uint32(99)
    ctx.set_tuning("wino_fused", "1")
    try:
        E.check(E.lib().mh_conv3x3_winograd_gn_partials(ctx.h, ptr["x"], n, h, w, ci, cv.u.ptr, co, ptr["b"], int(up),
                                                        ptr["sc"], ptr["sh"], 0, ptr["r"], out.ptr, part.ptr,
                                                        ctypes.byref(rows)))
        return out.numpy(), part.numpy(), rows.value
    finally:
        ctx.set_tuning("wino_fused", None)


def inputs(n, h, w, ci, co, up, pro, res):
    rng = np.random.default_rng(h + w + ci + co)
    x = rng.standard_normal((n, h, w, ci)).astype(np.float32)
    wt = (rng.standard_normal((co, 3, 3, ci)) / np.sqrt(9 * ci)).astype(np.float32)
    b = (rng.standard_normal(co) * 0.02).astype(np.float32)
    s = 2 if up else 1
    aff = ((1 + 0.1 * rng.random(n * ci)).astype(np.float32), rng.standard_normal(n * ci).astype(np.float32)) if pro else None
    r = rng.standard_normal((n, h * s, w * s, co)).astype(np.float32) if res else None
    return x, wt, b, aff, r


def want(x, wt, b, up, aff, res):
    y = oracle.conv3x3(x, wt, b, upsample2x=up, prologue=aff and (*aff, False))
    return y if res is None else y + res


CASES = [(1, 16, 16, 32, 64, False, False, False), (2, 16, 32, 64, 64, False, True, True),
         (1, 16, 16, 64, 128, True, False, True), (2, 13, 11, 64, 64, False, True, True),
         # blocks that straddle items (32 and 96 tiles each): partials of 32 tiles
         (3, 8, 16, 32, 64, False, False, True), (2, 16, 24, 64, 128, False, True, False),
         # several items per workgroup, of which one is flagged
         (1, 192, 192, 32, 64, False, False, True)]


@pytest.mark.parametrize("n,h,w,ci,co,up,pro,res", CASES)
def test_a_huge_finite_value(ctx, n, h, w, ci, co, up, pro, res):
    x, wt, b, aff, r = inputs(n, h, w, ci, co, up, pro, res)
    wt *= np.float32(1e-21)  # outputs to 1e17, their squares to 1e34
    x[n - 1, h // 2, w // 2, 7] = HUGE / 4 if up else HUGE  # upsampled, a patch's transform adds four of it
    if pro:  # the prologue leaves it as it is
        aff[0][(n - 1) * ci + 7], aff[1][(n - 1) * ci + 7] = 1, 0
    print(f"huge {n}x{h}x{w} {ci}->{co} up={up} pro={pro} res={res}", flush=True)
    got, part, rows = conv(ctx, x, wt, b, up, aff, r)
    assert np.isfinite(got).all() and rel_l2(got, want(x, wt, b, up, aff, r)) <= 1e-5
    if (h % 2, w % 2) == (0, 0):
        assert rows == (256 if got[0].shape[0] * got[0].shape[1] % 256 == 0 else 128)
        blocks = got[0].shape[0] * got[0].shape[1] // rows
        p = part.reshape(-1, co, 2)[:n * blocks].astype(np.float64).reshape(n, blocks, co, 2).sum(axis=1)
        g = got.astype(np.float64).reshape(n, -1, co)
        # 256 values a partial, summed in f32 by adds of at most 32 in a chain
        assert np.abs(p[..., 1] - (g * g).sum(axis=1)).max() <= 64 * 2.0 ** -24 * (g * g).sum(axis=1).max()
        assert np.abs(p[..., 0] - g.sum(axis=1)).max() <= 64 * 2.0 ** -24 * np.abs(g).sum(axis=1).max()
    else:
        assert rows == 0


@pytest.mark.parametrize("n,h,w,ci,co,up,pro,res", CASES)
def test_infinities_and_nan(ctx, n, h, w, ci, co, up, pro, res):
    x, wt, b, aff, r = inputs(n, h, w, ci, co, up, pro, res)
    x = odd_values(x)
    print(f"odd {n}x{h}x{w} {ci}->{co} up={up} pro={pro} res={res}", flush=True)
    got, ref = conv(ctx, x, wt, b, up, aff, r)[0], want(x, wt, b, up, aff, r)
    assert same_kind(got, ref)


def test_odd_values_in_the_weights(ctx):
    """Each spoils its own output channel as in f32, and no other; a huge finite one none."""
    x, wt, b, _, _ = inputs(1, 16, 16, 64, 64, False, False, False)
    x *= np.float32(1e-4)
    wt[3, 1, 1, 5], wt[9, 0, 0, 10], wt[40, 2, 1, 63] = np.inf, HUGE, np.nan
    got, ref = conv(ctx, x, wt, b)[0], oracle.conv3x3(x, wt, b)
    assert same_kind(got, ref)
    assert np.isfinite(got[..., 9]).all() and rel_l2(got[..., 9], ref[..., 9]) <= 1e-5
    rest = [c for c in range(64) if c not in (3, 9, 40)]
    assert rel_l2(got[..., rest], ref[..., rest]) <= 2e-6


@pytest.mark.parametrize("value", [np.nan, np.inf, HUGE])
def test_the_repair_is_bounded(ctx, value):
    """A map of nothing but odd values: the f32 products once more, no dearer per output."""
    h = w = 256
    x, wt, b, _, _ = inputs(1, h, w, 128, 128, False, False, False)
    cv = E.Conv3x3(ctx, 128, 128, E.Param(ctx, wt), b, winograd=True)

    def us(x):
        t, out = E.Tensor.from_numpy(ctx, x), E.Tensor(ctx)
        best = np.inf
        for _ in range(4):
            ctx.synchronize()
            t0 = time.perf_counter()
            cv.forward(t, out)
            ctx.synchronize()
            best = min(best, time.perf_counter() - t0)
        return best * 1e6

    base, odd = us(x), us(np.full_like(x, value))
    print(f"repair: {base:.0f} us finite, {odd:.0f} us all {value}", flush=True)
    assert odd <= 6 * base + 200  # the split conv and the f32 one, and the host's jitter


# bf16 holds 24 bits of an operand down to 2^-110; an f32 sum's last bit is at 2^-149 at the least
@pytest.mark.parametrize("exponent", [-105, -114, -119])
@pytest.mark.parametrize("where", ["input", "half", "weights"])
def test_small_operands(ctx, exponent, where):
    """The whole input, its right half beside values around 1, or the weights."""
    h, w, ci, co = 16, 48, 64, 64
    x, wt, _, _, _ = inputs(1, h, w, ci, co, False, False, False)
    scale = np.float32(2.0 ** exponent)
    if where == "weights":
        wt *= scale
    else:
        x[:, :, w // 2 if where == "half" else 0:] *= scale
    got = conv(ctx, x, wt, None)[0].astype(np.float64) * 2.0 ** -exponent
    xp = np.pad(x.astype(np.float64), ((0, 0), (1, 1), (1, 1), (0, 0)))
    ref = sum(xp[:, ky:ky + h, kx:kx + w] @ wt[:, ky, kx].T.astype(np.float64)
              for ky in range(3) for kx in range(3)) * 2.0 ** -exponent
    if where == "half":  # the tiles that touch no value around 1
        got, ref = got[:, :, w // 2 + 2:], ref[:, :, w // 2 + 2:]
    # as for ordinary values: a sum of 2^-119 and more rounds to 2^-30 of it or its 24 bits
    assert rel_l2(got, ref) <= 8 * 2.0 ** -24
