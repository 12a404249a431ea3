"""GPU parity: every tile shape and split of the int4 tile kernel, at the edges of its tiles, units and splits, against the
float64 value of the same stored operands; the plan itself on the host."""

import ctypes
import random

import pytest
import torch

from keras_amd import _lib, ops as kops
from keras_amd.layers import Dense
from tests.helpers import c_w4_matmul_f64
from tests.test_gpu_int4_matmul import make_layer
from tests.test_gpu_int4_strip_rows import magnitude


def plan_of(rows, parts, K, N):
    out = (ctypes.c_int * 4)()
    assert _lib.load().k3qt_w4_tile_plan(rows, parts, K, N, out) == 0
    return tuple(out)


def test_plan_covers_k():
    rng = random.Random(7)
    for _ in range(3000):
        rows, parts = rng.choice((1, 17, rng.randint(1, 1024))), rng.choice((1, 2, 3))
        units, N = rng.randint(1, 130), 32 * rng.randint(1, 900)
        mb, bn, ks, steps = plan_of(rows, parts, 128 * units, N)
        kq = 256 // bn
        assert mb in (1, 2, 4) and bn in (128, 256) and (bn == 128 or mb == 4) and (parts != 2 or mb > 1)
        assert 1 <= ks <= 8 and (ks - 1) * steps * kq < units <= ks * steps * kq


# rows, K, N, group, float32, the plan (blocks of rows, columns, splits) the shape stands for
CASES = [
    (17, 128, 32, 128, False, (1, 128, 1)),       # one unit: the second slice of K has none
    (33, 384, 96, 128, False, (1, 128, 1)),       # an odd number of units, a row past a tile
    (31, 2944, 1056, 128, False, (1, 128, 3)),    # splits that end inside a step
    (128, 5504, 2080, None, False, (1, 128, 3)),
    (300, 1664, 6400, 128, False, (2, 128, 1)),
    (200, 4096, 8192, None, False, (2, 128, 1)),
    (511, 896, 8160, 128, False, (4, 128, 1)),    # columns past the last whole tile
    (500, 640, 8224, 128, False, (4, 256, 1)),
    (512, 1152, 14368, None, False, (4, 256, 1)),
    (700, 1152, 4160, 128, False, (4, 128, 1)),
    (65, 384, 1024, 128, True, (2, 128, 1)),      # two parts of a row in one tile
    (40, 2944, 4096, 128, True, (2, 128, 3)),
    (300, 1152, 4128, None, True, (4, 128, 1)),
    (512, 640, 14368, 128, True, (4, 256, 1)),
    (50, 376, 1052, 128, True, (1, 128, 1)),      # three parts of a row
]


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,N,block_size,f32,plan", CASES)
def test_tile_plans(dev, M, K, N, block_size, f32, plan):
    dtype = torch.float32 if f32 else torch.bfloat16
    parts = 1 if not f32 else 3 if N % 8 or K % 16 else 2
    assert plan_of(M, parts, -(-K // 128) * 128, -(-N // 32) * 32)[:3] == plan
    qk, bias = make_layer(K, N, block_size, seed=M, with_bias=(M % 2 == 1))
    g = torch.Generator().manual_seed(K)
    x = torch.randn(M, K, generator=g).to(dtype)
    scale, kernel = qk["kernel_scale"].to(dtype), qk["kernel"].to(dev)
    zero = qk["kernel_zero"] if block_size else None
    b = None if bias is None else bias.to(dtype)
    exact = c_w4_matmul_f64(x, qk["kernel"], scale, zero, block_size, b, N)
    mag = magnitude(x, kernel, scale, zero, block_size, N)
    strip = kops.int4_strip_copy(kernel, N)
    b = None if b is None else b.to(dev)

    def rows_entry(x):
        return kops.int4_matmul_tiles_rows(
            x, strip, N, kops.int4_tile_columns(scale.to(dev), N) if block_size else scale.to(dev),
            kernel_zero=kops.int4_tile_columns(zero.to(dev), N) if block_size else None, block_size=block_size, bias=b)

    calls = [("rows", rows_entry)]
    if kops.int4_tiles_strip_supported(M, K, N, block_size) and not f32:
        calls.append(("strip", lambda x: kops.int4_matmul_tiles_strip(
            x, strip, N, scale.to(dev), kernel_zero=None if zero is None else zero.to(dev), block_size=block_size, bias=b)))
    for name, call in calls:
        # poisoned scratch, twice: a partial or a sum that is read before it is written shows, as does anything left over
        got = []
        for fill in (0xFF, 0x7F):
            kops._workspace(dev, 64 << 20).fill_(fill)
            got.append(call(x.to(dev)))
        torch.cuda.synchronize()
        assert torch.equal(got[0], got[1]), name
        assert got[0].dtype == dtype and tuple(got[0].shape) == (M, N)
        err = (got[0].double().cpu() - exact).abs()
        # (the bounds of test_tiles_rows; an offset of 136 sums terms up to 17 times the largest weight's)
        if f32:
            split = 2.0 ** -17 if parts == 2 else 0.0
            bound = mag * (split + 4 * 2.0 ** -24 * K ** 0.5) + exact.abs() * 2.0 ** -22
        else:
            size = exact.abs() + (0 if b is None else 2 * b.double().abs().cpu())
            bound = mag * (17 if name == "strip" else 4) * 2.0 ** -24 * K ** 0.5 + size * 3.05 * 2.0 ** -8
        assert bool((err <= bound).all()), (name, float((err / bound).max()))


@pytest.mark.gpu
@pytest.mark.parametrize("rows,K,units,tiles", [(640, 4096, 1024, True), (640, 1024, 128, False), (1025, 256, 4096, False)])
def test_bfloat16_layers_on_both_sides_of_the_line(dev, rows, K, units, tiles):
    layer = Dense(units, dtype="mixed_bfloat16", device="cuda:0", use_bias=False)
    layer.build((None, K))
    layer.quantize("int4")
    x = torch.randn(rows, K, generator=torch.Generator().manual_seed(rows)).to(torch.bfloat16)
    y = layer(x.to(dev))
    assert ("w4s" in layer._cache) == tiles
    q = layer._kernel.value.cpu()
    scale, zero = layer.kernel_scale.value.to(torch.bfloat16).cpu(), layer.kernel_zero.value.cpu()
    exact = c_w4_matmul_f64(x, q, scale, zero, 128, None, units)
    # each weight of the de-quantised kernel is rounded to bfloat16, the tiles' are not
    mag = magnitude(x, layer._kernel.value, scale, zero, 128, units)
    bound = mag * (17 * 2.0 ** -24 * K ** 0.5 + (0 if tiles else 2.0 ** -9)) + exact.abs() * 2.0 ** -8
    err = (y.double().cpu() - exact).abs()
    assert bool((err <= bound).all()), float((err / bound).max())
