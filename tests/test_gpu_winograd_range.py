"""The one-kernel Winograd conv's range (csrc/winograd_fused.hip): maps of a row or two,
where a patch's rows reach further than the whole input, against the oracle; and an
input above 1 GiB, against the same conv of its last rows."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from moebius_cpu_amd import engine as E
from tests.test_gpu_winograd_repair import conv as conv_partials
from tests.util import rel_l2

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = E.Context(0)
    yield c
    c.synchronize()
    c.close()


def conv(ctx, tune, x, wt, up=False, fused=1):
    tune("wino_fused", fused)
    out = E.Tensor(ctx)
    E.Conv3x3(ctx, wt.shape[3], wt.shape[0], E.Param(ctx, wt), None, upsample2x=up, winograd=True).forward(
        E.Tensor.from_numpy(ctx, x), out)
    return out.numpy()


@pytest.mark.parametrize("n,h,w,ci,co,up", [(1, 1, 1, 32, 64, False), (1, 1, 300, 64, 64, False),
                                            (1, 2, 71, 96, 64, False), (2, 1, 5, 512, 128, False),
                                            (1, 1, 9, 64, 64, True), (1, 2, 33, 32, 64, True),
                                            (1, 200, 1, 64, 64, False)])
def test_strips(ctx, tune, n, h, w, ci, co, up):
    rng = np.random.default_rng(h + w + ci)
    x = rng.standard_normal((n, h, w, ci)).astype(np.float32)
    wt = (rng.standard_normal((co, 3, 3, ci)) / np.sqrt(9 * ci)).astype(np.float32)
    print(f"strip {n}x{h}x{w} {ci}->{co} up={up}", flush=True)
    assert rel_l2(conv(ctx, tune, x, wt, up), oracle.conv3x3(x, wt, upsample2x=up)) <= 4e-6


def test_an_input_above_1_gib(ctx):
    h, w, ci, co = 1100, 1024, 256, 64  # 1.07 GiB
    rng = np.random.default_rng(3)
    x = np.resize(rng.standard_normal(999983).astype(np.float32), (1, h, w, ci))
    wt = (rng.standard_normal((co, 3, 3, ci)) / np.sqrt(9 * ci)).astype(np.float32)
    print("wino fused above 1 GiB", flush=True)
    got, _, rows = conv_partials(ctx, x, wt, None)
    assert rows > 0  # the one-kernel path
    # the same products in the same order, but for the row at the crop's edge
    last = conv_partials(ctx, np.ascontiguousarray(x[:, -64:]), wt, None)[0]
    assert np.array_equal(got[:, -62:], last[:, 2:])
    first = conv_partials(ctx, np.ascontiguousarray(x[:, :64]), wt, None)[0]
    assert np.array_equal(got[:, :62], first[:, :62])
