"""EXACT products on the bf16 matrix instructions, every f32 operand split in three
bf16 parts (csrc/split_bf16.hpp): no further from 64 bits than an f32 sum, at the
tile edges, and infinities, NaN and values next to the largest f32 as the f32
products give them (a part product of an infinite value with a zero part is NaN)."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from moebius_cpu_amd import engine as E

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = E.Context(0)
    yield c
    c.synchronize()
    c.close()


def rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def same_kind(got, want):
    """Infinite, NaN and finite in the same places, infinities of the same sign."""
    return (np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isposinf(got), np.isposinf(want))
            and np.array_equal(np.isneginf(got), np.isneginf(want)))


def odd_values(x):
    """Infinities, a NaN and a value that rounds to infinity in bf16, far apart."""
    h, w, c = x.shape[1:]
    x[0, 1, 1, 3] = np.inf
    x[0, h - 2, w // 2, c - 1] = -np.inf
    x[0, 1, w - 2, 5] = np.nan
    x[0, h // 2, 2, 7] = np.float32(3.4e38)
    return x


# the one-kernel Winograd conv: whole and partial tile blocks, one and several
# channel blocks, more items than workgroups, the upsample
@pytest.mark.parametrize("n,h,w,ci,co,up", [(1, 16, 16, 32, 64, False), (2, 13, 11, 64, 64, False),
                                            (1, 70, 66, 96, 192, False), (1, 9, 14, 128, 64, True),
                                            (1, 190, 180, 32, 64, False)])
def test_winograd_error_and_odd_values(ctx, n, h, w, ci, co, up):
    rng = np.random.default_rng(n + h + ci)
    x = rng.standard_normal((n, h, w, ci)).astype(np.float32)
    wt = (rng.standard_normal((co, 3, 3, ci)) * np.sqrt(2.0 / (9 * ci))).astype(np.float32)
    b = (rng.standard_normal(co) * 0.02).astype(np.float32)

    def run(x, fused):
        ctx.set_tuning("wino_fused", fused)
        try:
            cv = E.Conv3x3(ctx, ci, co, E.Param(ctx, wt), b, upsample2x=up, winograd=True)
            out = E.Tensor(ctx)
            cv.forward(E.Tensor.from_numpy(ctx, x), out)
            return out.numpy()
        finally:
            ctx.set_tuning("wino_fused", None)

    print(f"split wino {n}x{h}x{w} {ci}->{co} up={up}", flush=True)
    xs = x.astype(np.float64)
    if up:
        xs = xs.repeat(2, axis=1).repeat(2, axis=2)
    xp = np.pad(xs, ((0, 0), (1, 1), (1, 1), (0, 0)))
    want = sum(xp[:, ky:ky + xs.shape[1], kx:kx + xs.shape[2]] @ wt[:, ky, kx].T.astype(np.float64)
               for ky in range(3) for kx in range(3)) + b
    # the f32 transforms (two sums of two either side) and the sums over ci: a few
    # roundings of 2^-24 each, amplified by F(2x2, 3x3) to under 8 of them in 2-norm
    assert rel(run(x, 1), want) <= 8 * 2.0 ** -24 * max(1.0, np.sqrt(ci / 64))
    x = odd_values(x)
    assert same_kind(run(x, 1), oracle.conv3x3(x, wt, b, upsample2x=up))
    assert same_kind(run(np.full_like(x, np.nan), 1), np.full(want.shape, np.nan))
