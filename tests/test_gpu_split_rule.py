"""Which kernel an EXACT GEMM takes (plan_split in csrc/gemm_split.hpp), at the lines of
its rule, read from the launch timing's configuration; and the results either way."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

from moebius_cpu_amd import engine as E
from tests.test_gpu_split import TILES

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = E.Context(0)
    yield c
    c.synchronize()
    c.close()


def run(ctx, tune, conv, x):
    """The output and the kernel that made it."""
    t, out = E.Tensor.from_numpy(ctx, x), E.Tensor(ctx)
    tune("gemm_time", 1)
    ctx.gemm_times()
    conv.forward(t, out)
    recs = ctx.gemm_times()
    tune("gemm_time", 0)
    assert len(recs) == 1
    return out.numpy(), recs[0]["config"].split(" mode")[0]


def close(a, b, k):
    a, b = a.astype(np.float64), b.astype(np.float64)
    return np.linalg.norm(a - b) <= 2 * 2.0 ** -24 * (4 + np.sqrt(k / 4)) * np.linalg.norm(b)


# up to 32 rows: the narrowest tile whose columns are one round of 256 CUs
@pytest.mark.parametrize("m,n,k,tile", [(2, 8192, 1024, "32x32"), (32, 8224, 1024, "32x48"), (1, 11200, 1280, "32x48"),
                                        (3, 12320, 768, "32x64"), (32, 20480, 768, "32x80"), (16, 1280, 11520, "32x32"),
                                        (32, 20500, 768, None), (32, 16384, 512, None), (2, 6560, 1280, "32x32"),
                                        (2, 6400, 1280, None)])
def test_few_rows(ctx, tune, m, n, k, tile):
    rng = np.random.default_rng(m + n)
    x = rng.standard_normal((1, 1, m, k), dtype=np.float32)
    conv = E.Conv1x1(ctx, k, n, E.Param(ctx, rng.standard_normal((n, k), dtype=np.float32) / np.float32(np.sqrt(k))))
    print(f"few rows {m}x{n}x{k}", flush=True)
    got, config = run(ctx, tune, conv, x)
    assert config.startswith(f"f32 split {tile} waves 2x1x4" if tile else "f32 ") and ("split" in config) == (tile is not None)
    tune("gemm_split", "0")
    assert close(got, run(ctx, tune, conv, x)[0], k)


# few output pixels of a deep conv: K split over workgroups on the f32 instructions
@pytest.mark.parametrize("h,w,ci,co,stride", [(8, 8, 1280, 1280, 2), (7, 7, 1280, 1280, 2), (5, 5, 1280, 640, 1),
                                              (8, 8, 640, 2560, 2)])
def test_few_pixels(ctx, tune, h, w, ci, co, stride):
    rng = np.random.default_rng(h + ci)
    x = rng.standard_normal((1, h, w, ci), dtype=np.float32)
    wt = rng.standard_normal((co, 3, 3, ci), dtype=np.float32) / np.float32(np.sqrt(9 * ci))
    conv = E.Conv3x3(ctx, ci, co, E.Param(ctx, wt), stride=stride)
    print(f"few pixels {h}x{w} {ci}->{co}", flush=True)
    got, config = run(ctx, tune, conv, x)
    assert config.startswith("f32 ") and "split" not in config
    tune("gemm_split", "16,32,2,4")
    assert close(got, run(ctx, tune, conv, x)[0], 9 * ci)


# rows per item that 128, or 64 and 128, do not divide: the taller tiles are faster but for the
# statistics launch that the next GroupNorm would need
@pytest.mark.parametrize("h,w", [(56, 56), (51, 64), (32, 49), (64, 64)])
def test_group_norm_partials_are_kept(ctx, h, w):
    c = 512
    rng = np.random.default_rng(h)
    x = rng.standard_normal((1, h, w, c), dtype=np.float32)
    wt = E.Param(ctx, rng.standard_normal((c, c), dtype=np.float32) / np.float32(np.sqrt(c)))
    out, part = E.DeviceArray(ctx, (1, h, w, c)), E.DeviceArray(ctx, (-(-h * w // 32), c, 2))
    xd, rows = E.DeviceArray.from_numpy(ctx, x), ctypes.c_uint32()
    E.check(E.lib().mh_conv1x1_gn_partials(ctx.h, xd.ptr, 1, h, w, c, wt.ptr, wt.dtype, c, None, None, out.ptr, part.ptr,
                                           ctypes.byref(rows)))
    assert rows.value > 0 and h * w % rows.value == 0
    y = out.numpy().reshape(-1, c).astype(np.float64)
    sums = part.numpy()[:h * w // rows.value].astype(np.float64).sum(axis=0)
    # 32 to 128 values a partial, summed in f32
    assert np.abs(sums[:, 1] - (y * y).sum(axis=0)).max() <= 128 * 2.0 ** -24 * (y * y).sum(axis=0).max()


# the forced tilings of the split kernel's tests are the ones that run, and the planner's choice at a
# shape above its line is one of them
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("f16", [False, True])
def test_the_tiling_that_runs(ctx, tune, tile, f16):
    rng = np.random.default_rng(5)
    tune("gemm_split", tile)
    px, ci, co = ((64, 64), 320, 320) if tile == "1" else ((9, 11), 64, 70)
    x = rng.standard_normal((1, *px, ci), dtype=np.float32)
    dense = E.Conv1x1(ctx, ci, co, E.Param(ctx, rng.standard_normal((co, ci)).astype(np.float16 if f16 else np.float32),
                                           f16=f16))
    conv = E.Conv3x3(ctx, ci, co, E.Param(ctx, rng.standard_normal((co, 3, 3, ci)).astype(np.float16 if f16 else np.float32),
                                          f16=f16))
    for op in (dense, conv):
        config = run(ctx, tune, op, x)[1]
        if tile == "1":
            assert config.startswith("f32 split ")
        else:
            tm, bn, wm, wk = (int(v) for v in tile.split(","))
            assert config.startswith(f"f32 split {tm * wm}x{bn} waves {wm}x1x{wk}")


@pytest.mark.parametrize("value", ["16,80,8", "16,80,8,1,1", "16,80,8,1 ", "16,96,8,1", "32,80,4,1", "2", "-1", "x"])
def test_an_unknown_tiling_is_refused(ctx, value):
    with pytest.raises(E.MoebiusError):
        ctx.set_tuning("gemm_split", value)
    ctx.set_tuning("gemm_split", None)
