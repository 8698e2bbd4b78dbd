"""EXACT products on the bf16 matrix instructions, every f32 operand split in three
bf16 parts (csrc/split_bf16.hpp): no further from 64 bits than an f32 sum, at the
tile edges, and infinities, NaN and values next to the largest f32 as the f32
products give them (a part product of an infinite value with a zero part is NaN)."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from moebius_cpu_amd import engine as E
from moebius_cpu_amd import unet_params as U
from moebius_cpu_amd.unet import UNet

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


# every tiling of the split GEMM (csrc/gemm_split.hpp) and the planner's choice
TILES = ["1", "16,80,8,1", "16,64,8,1", "16,80,4,2", "16,64,4,2", "16,48,4,2", "16,80,2,4", "16,64,2,4", "16,48,2,4",
         "16,32,2,4"]


def gemm_bound(k):
    """A chain of k / 32 f32 sums, each rounded once (2^-24 in 2-norm at most), the
    sum of the small part products and the epilogue's two additions."""
    return 2.0 ** -24 * (4 + np.sqrt(k / 32))


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("f16", [False, True])
# one row, one K step; rows, columns and K past their last whole tile, stage and quad
@pytest.mark.parametrize("h,w,ci,co", [(1, 1, 4, 4), (9, 11, 200, 70), (33, 3, 36, 324), (16, 16, 1284, 96)])
def test_gemm_tilings(ctx, tune, tile, f16, h, w, ci, co):
    rng = np.random.default_rng(h + ci + co)
    x = rng.standard_normal((2, h, w, ci)).astype(np.float32)
    wt = (rng.standard_normal((co, ci)) / np.sqrt(ci)).astype(np.float16 if f16 else np.float32)
    b = rng.standard_normal(co).astype(np.float32)
    r = rng.standard_normal((2, h, w, co)).astype(np.float32)
    param = E.Param(ctx, wt, f16=f16)

    def run(x, tile):
        tune("gemm_split", tile)
        out = E.Tensor(ctx)
        E.Conv1x1(ctx, ci, co, param, b).forward(E.Tensor.from_numpy(ctx, x), out, E.Tensor.from_numpy(ctx, r))
        return out.numpy()

    print(f"split gemm {tile} 2x{h}x{w} {ci}->{co} f16={f16}", flush=True)
    want = x.astype(np.float64) @ wt.T.astype(np.float64) + b + r
    assert rel(run(x, tile), want) <= gemm_bound(ci)
    if h > 3 and w > 4:
        x = odd_values(x)
        assert same_kind(run(x, tile), run(x, "0"))


@pytest.mark.parametrize("tile", TILES)
# the gathers: 64 channels to a K step and 4, stride 2, the upsample; a GroupNorm prologue
@pytest.mark.parametrize("h,w,ci,co,stride,up,pro", [(13, 9, 64, 80, 1, False, False), (15, 11, 36, 52, 2, False, False),
                                                     (7, 5, 64, 40, 1, True, True), (6, 9, 20, 33, 1, False, True)])
def test_conv_tilings(ctx, tune, tile, h, w, ci, co, stride, up, pro):
    rng = np.random.default_rng(h + ci + co)
    x = rng.standard_normal((2, h, w, ci)).astype(np.float32)
    wt = (rng.standard_normal((co, 3, 3, ci)) / np.sqrt(9 * ci)).astype(np.float32)
    b = rng.standard_normal(co).astype(np.float32)
    aff, xs = None, x.astype(np.float64)
    if pro:
        sc = (1 + 0.2 * rng.standard_normal((2, ci))).astype(np.float32)
        sh = rng.standard_normal((2, ci)).astype(np.float32)
        aff = E.Affine(E.DeviceArray.from_numpy(ctx, sc), E.DeviceArray.from_numpy(ctx, sh), False)
        xs = xs * sc.reshape(2, 1, 1, ci) + sh.reshape(2, 1, 1, ci)
    if up:
        xs = xs.repeat(2, axis=1).repeat(2, axis=2)
    xp = np.pad(xs, ((0, 0), (1, 1), (1, 1), (0, 0)))
    oh, ow = -(-xs.shape[1] // stride), -(-xs.shape[2] // stride)
    want = b + sum(xp[:, ky:ky + stride * oh:stride, kx:kx + stride * ow:stride][:, :oh, :ow]
                   @ wt[:, ky, kx].T.astype(np.float64) for ky in range(3) for kx in range(3))
    print(f"split conv {tile} 2x{h}x{w} {ci}->{co} stride={stride} up={up} pro={pro}", flush=True)
    tune("gemm_split", tile)
    out = E.Tensor(ctx)
    E.Conv3x3(ctx, ci, co, E.Param(ctx, wt), b, stride=stride, upsample2x=up).forward_prologue(
        E.Tensor.from_numpy(ctx, x), aff, out)
    assert rel(out.numpy(), want) <= gemm_bound(9 * ci)


def test_unet_step_every_tiling(ctx, tune):
    """A whole step: the concatenated, segmented, grouped and batched forms, LayerNorm
    and GroupNorm partials and prologues, against the f32 products' step."""
    net = UNet(ctx, U.random_unet())
    inp = U.unet_input()
    tune("gemm_split", "0")
    want = net.forward_host(inp.x, inp.timestep)
    for tile in TILES:
        print(f"split unet {tile}", flush=True)
        tune("gemm_split", tile)
        # both are f32 results of one network, each within 2.5e-6 of its 64-bit value
        assert rel(net.forward_host(inp.x, inp.timestep), want) <= 5e-6


# the rule's line: one full round of workgroups, half a round, and one workgroup past a round
@pytest.mark.parametrize("n,h,w,ci,co,fused", [(2, 64, 64, 512, 512, 1), (1, 64, 64, 512, 512, 0),
                                               (1, 108, 148, 256, 256, 1), (1, 96, 98, 256, 512, 0)])
def test_winograd_rule(ctx, tune, n, h, w, ci, co, fused):
    rng = np.random.default_rng(n + ci)
    x = E.Tensor.from_numpy(ctx, rng.standard_normal((n, h, w, ci), dtype=np.float32))
    wt = rng.standard_normal((co, 3, 3, ci), dtype=np.float32) / np.float32(np.sqrt(9 * ci))
    conv = E.Conv3x3(ctx, ci, co, E.Param(ctx, wt), winograd=True)

    def run(v):
        tune("wino_fused", v)
        out = E.Tensor(ctx)
        conv.forward(x, out)
        return out.numpy()

    print(f"wino rule {n}x{h}x{w} {ci}->{co}", flush=True)
    got = run(-1)
    assert np.array_equal(got, run(fused)) and rel(run(1 - fused), got) <= 2e-6
