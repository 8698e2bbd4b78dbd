"""The split GEMM (csrc/gemm_split.hpp) where its sums are not finite, or too small for
their operands' bits: such tiles are redone on the f32 instructions in every tiling and
A-operand form, for little more than the f32 kernel's time."""
from __future__ import annotations

import ctypes
import time

import numpy as np
import pytest

from moebius_cpu_amd import engine as E
from tests.test_gpu_split import TILES, odd_values, rel, same_kind

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = E.Context(0)
    yield c
    c.synchronize()
    c.close()


def f32_bound(k):
    """A chain of k / 4 f32 sums of four products, each rounded once, and the epilogue."""
    return 2.0 ** -24 * (4 + np.sqrt(k / 4))


def conv1x1(ctx, x, wt, f16=False, b=None, res=None):
    out = E.Tensor(ctx)
    E.Conv1x1(ctx, wt.shape[1], wt.shape[0], E.Param(ctx, wt, f16=f16), b).forward(
        E.Tensor.from_numpy(ctx, x), out, None if res is None else E.Tensor.from_numpy(ctx, res))
    return out.numpy()


# bf16 holds 24 bits of an operand down to 2^-110; an f32 sum's last bit is at 2^-149 at the least
@pytest.mark.parametrize("tile", TILES[1:])
@pytest.mark.parametrize("where,exponent", [("input", -114), ("rows", -119), ("weights", -119), ("input", -105)])
def test_small_operands(ctx, tune, tile, where, exponent):
    """The whole input, its last rows beside values around 1, or the weights."""
    h, w, ci, co = 9, 15, 200, 72
    rng = np.random.default_rng(ci - exponent)
    x = rng.standard_normal((2, h, w, ci)).astype(np.float32)
    wt = (rng.standard_normal((co, ci)) / np.sqrt(ci)).astype(np.float32)
    scale = np.float32(2.0 ** exponent)
    if where == "weights":
        wt *= scale
    else:
        x[1 if where == "rows" else 0:] *= scale
    tune("gemm_split", tile)
    got = conv1x1(ctx, x, wt).astype(np.float64)
    want = x.astype(np.float64) @ wt.T.astype(np.float64)
    assert rel(got[1] * 2.0 ** -exponent, want[1] * 2.0 ** -exponent) <= f32_bound(ci)


# the gathers of test_conv_tilings: 64 channels to a K step and 4, stride 2, the upsample; a GroupNorm prologue
@pytest.mark.parametrize("tile", TILES[1:])
@pytest.mark.parametrize("h,w,ci,co,stride,up,pro", [(13, 9, 64, 80, 1, False, False), (15, 11, 36, 52, 2, False, False),
                                                     (7, 5, 64, 40, 1, True, True), (6, 9, 20, 33, 1, False, True)])
def test_conv_odd_values(ctx, tune, tile, h, w, ci, co, stride, up, pro):
    rng = np.random.default_rng(h + ci + co)
    x = odd_values(rng.standard_normal((2, h, w, ci)).astype(np.float32))
    wt = (rng.standard_normal((co, 3, 3, ci)) / np.sqrt(9 * ci)).astype(np.float32)
    aff = None
    if pro:
        sc = np.where(rng.random((2, ci)) < 0.5, 0.9, 1.0).astype(np.float32)
        sh = rng.standard_normal((2, ci)).astype(np.float32)
        aff = E.Affine(E.DeviceArray.from_numpy(ctx, sc), E.DeviceArray.from_numpy(ctx, sh), False)

    def run(tile, x):
        tune("gemm_split", tile)
        out = E.Tensor(ctx)
        E.Conv3x3(ctx, ci, co, E.Param(ctx, wt), stride=stride, upsample2x=up).forward_prologue(
            E.Tensor.from_numpy(ctx, x), aff, out)
        return out.numpy()

    got, want = run(tile, x), run("0", x)
    assert same_kind(got, want) and not np.isfinite(got).all()
    ok = np.isfinite(want) & (np.abs(want) < 1e30)  # but for the outputs of the huge value
    assert ok.any() and rel(got[ok].astype(np.float64), want[ok].astype(np.float64)) <= 2 * f32_bound(9 * ci)
    small = np.float32(2.0 ** -119) * rng.standard_normal(x.shape).astype(np.float32)
    if not pro:
        assert rel(run(tile, small).astype(np.float64), run("0", small).astype(np.float64)) <= 2 * f32_bound(9 * ci)


@pytest.mark.parametrize("value", [np.nan, np.inf, np.float32(3.4e38), np.float32(2.0 ** -120)])
def test_the_redo_is_bounded(ctx, tune, value):
    rng = np.random.default_rng(2)
    wt = (rng.standard_normal((1280, 1280)) / 36).astype(np.float32)
    x = rng.standard_normal((2, 32, 32, 1280)).astype(np.float32)
    conv = E.Conv1x1(ctx, 1280, 1280, E.Param(ctx, wt))

    def us(x):
        t, out, best = E.Tensor.from_numpy(ctx, x), E.Tensor(ctx), np.inf
        for _ in range(5):
            ctx.synchronize()
            t0 = time.perf_counter()
            conv.forward(t, out)
            ctx.synchronize()
            best = min(best, time.perf_counter() - t0)
        return best * 1e6

    base, odd = us(x), us(np.full_like(x, value))
    print(f"redo: {base:.0f} us finite, {odd:.0f} us all {value}", flush=True)
    assert odd <= 6 * base + 200  # the split tile and the f32 one, and the host's jitter
