"""The launches of an int4 tile call of more rows than one takes (k3q_gemm_w4_rows): on the host, that each covers K with its
own plan and has room for its partial sums; on the GPU, rows of the first and the last launch against float64."""

import ctypes
import random

import pytest
import torch

from keras_amd import _lib, ops as kops
from tests.helpers import c_w4_matmul_f64
from tests.test_gpu_int4_matmul import make_layer
from tests.test_gpu_int4_strip_rows import magnitude


def launches(f32, M, K, N, block_size):
    """[(rows, mb, bn, ks, steps, bytes of partials, room)] of a call."""
    lib, out, m0 = _lib.load(), [], 0
    while m0 < M:
        v = (ctypes.c_int64 * 7)()
        assert lib.k3qt_w4_rows_launch(_lib.K3Q_F32 if f32 else _lib.K3Q_BF16, M, K, N, block_size, m0, v) == 0
        out.append(tuple(v))
        m0 += v[0]
    assert m0 == M
    return out


def test_every_launch_covers_k_and_has_room():
    rng = random.Random(11)
    changes = 0
    for _ in range(6000):
        f32, M = rng.random() < 0.5, rng.randint(1, 4096)
        K = rng.choice((8 * rng.randint(2, 1800), 128 * rng.randint(1, 112)))
        N = rng.choice((rng.randint(1, 14336), 32 * rng.randint(1, 448)))
        bs = rng.choice((128, -1))
        ran = launches(f32, M, K, N, bs)
        units = -(-K // 128)
        for rows, mb, bn, ks, steps, partials, room in ran:
            kq = 256 // bn
            assert (ks - 1) * steps * kq < units <= ks * steps * kq, (f32, M, K, N, bs, ran)
            assert partials <= room, (f32, M, K, N, bs, ran)
        head = _lib.load().k3q_gemm_w4_rows_workspace_bytes(_lib.K3Q_F32 if f32 else _lib.K3Q_BF16, M, K, N, bs)
        assert head >= ran[0][6] + ran[0][0] * 2 * K
        # (another tile or other splits for the last launch: what one shared plan got wrong)
        changes += ran[0][1:5] != ran[-1][1:5]
    assert changes > 300


def test_kernels_beyond_the_tiles_offsets_are_not_promised():
    """K and N that 32-bit lane offsets do not reach are not taken (they go to the kernels on the stored weights) instead of
    failing at the launch."""
    assert kops.int4_tiles_rows_supported(1 << 20, 1 << 16, 128)
    for K, N in ((1 << 24, 64), (1 << 21, 1 << 16), (1 << 21, (1 << 16) - 8)):
        for bs in (128, None):
            assert not kops.int4_tiles_rows_supported(K, N, bs)
        for dtype in (_lib.K3Q_F32, _lib.K3Q_BF16):
            assert _lib.load().k3q_gemm_w4_rows_workspace_bytes(dtype, 100, K, N, 128) == 0


# the plans of the first and of the last launch: (blocks of rows, columns, splits)
CASES = [
    (612, 6400, 2560, True, (4, 256, 3), (2, 128, 3)),
    (800, 8192, 4096, True, (4, 128, 1), (4, 256, 3)),
    (648, 11008, 4096, True, (4, 128, 1), (4, 256, 5)),
    (860, 14336, 2048, True, (4, 128, 2), (4, 256, 5)),
    (409, 4096, 2337, True, (4, 256, 3), (2, 128, 3)),     # three parts a row
    (1505, 6400, 2049, False, (4, 256, 3), (4, 128, 3)),
    (1700, 11008, 3333, False, (4, 128, 1), (4, 256, 3)),
]


@pytest.mark.gpu
@pytest.mark.parametrize("block_size", [128, None])
@pytest.mark.parametrize("M,K,N,f32,first,last", CASES)
def test_last_launch(dev, M, K, N, f32, first, last, block_size):
    dtype = torch.float32 if f32 else torch.bfloat16
    ran = launches(f32, M, K, N, block_size or -1)
    assert len(ran) > 1 and ran[0][1:4] == first and ran[-1][1:4] == last
    qk, bias = make_layer(K, N, block_size, seed=M, with_bias=True)
    g = torch.Generator().manual_seed(K)
    x = torch.randn(M, K, generator=g).to(dtype)
    scale, kernel, b = qk["kernel_scale"].to(dtype), qk["kernel"].to(dev), bias.to(dtype)
    zero = qk["kernel_zero"] if block_size else None
    need = _lib.load().k3q_gemm_w4_rows_workspace_bytes(_lib.K3Q_F32 if f32 else _lib.K3Q_BF16, M, K, N, block_size or -1)
    kops._workspace(dev, need).fill_(0xFF)
    got = kops.int4_matmul_tiles_rows(
        x.to(dev), kops.int4_strip_copy(kernel, N), N,
        kops.int4_tile_columns(scale.to(dev), N) if block_size else scale.to(dev),
        kernel_zero=kops.int4_tile_columns(zero.to(dev), N) if block_size else None, block_size=block_size, bias=b.to(dev))
    start = M - ran[-1][0]
    rows = torch.tensor([0, 1, start - 1, start, start + 1, start + 33, M - 2, M - 1])
    got, x = got.cpu()[rows], x[rows]
    exact = c_w4_matmul_f64(x, qk["kernel"], scale, zero, block_size, b, N)
    mag = magnitude(x, kernel, scale, zero, block_size, N)
    err = (got.double() - exact).abs()
    if f32:  # (the bounds of test_tile_plans)
        split = 2.0 ** -17 if N % 8 == 0 and K % 16 == 0 else 0.0
        bound = mag * (split + 4 * 2.0 ** -24 * K ** 0.5) + exact.abs() * 2.0 ** -22
    else:
        bound = mag * 4 * 2.0 ** -24 * K ** 0.5 + (exact.abs() + 2 * b.double().abs()) * 3.05 * 2.0 ** -8
    assert bool((err <= bound).all()), float((err / bound).max())


@pytest.mark.parametrize("rows,parts,K,N,plan", [
    (65, 1, 5120, 11008, (4, 256, 5)), (64, 1, 5120, 11008, (2, 128, 2)), (329, 2, 8192, 2048, (4, 256, 5)),
    (338, 1, 5120, 2048, (4, 128, 5)), (920, 1, 8192, 2048, (4, 128, 2)),
    (96, 1, 4096, 14336, (2, 128, 1)), (102, 2, 3200, 4544, (2, 128, 1)),
])
def test_splits_where_they_pay(rows, parts, K, N, plan):
    """Measured: the best plan of each, 6 to 33 % ahead of fewer splits (the last two: of more)."""
    out = (ctypes.c_int * 4)()
    assert _lib.load().k3qt_w4_tile_plan(rows, parts, K, N, out) == 0 and tuple(out)[:3] == plan


@pytest.mark.gpu
@pytest.mark.parametrize("block_size", [128, None])
@pytest.mark.parametrize("M,K,N,plan", [
    (65, 5120, 11008, (4, 256, 5)), (338, 5120, 2048, (4, 128, 5)), (64, 5120, 11008, (2, 128, 2)), (96, 14336, 2048, (2, 128, 8)),
])
def test_large_tiles_with_splits(dev, M, K, N, plan, block_size):
    """Through the entry of the layers' own shapes: partial sums of every row, added by the second pass."""
    out = (ctypes.c_int * 4)()
    assert _lib.load().k3qt_w4_tile_plan(M, 1, K, N, out) == 0 and tuple(out)[:3] == plan
    qk, bias = make_layer(K, N, block_size, seed=M, with_bias=True)
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(K)).to(torch.bfloat16)
    scale, kernel, b = qk["kernel_scale"].to(torch.bfloat16), qk["kernel"].to(dev), bias.to(torch.bfloat16)
    zero = qk["kernel_zero"] if block_size else None
    got = []
    for fill in (0xFF, 0x7F):
        kops._workspace(dev, 64 << 20).fill_(fill)
        got.append(kops.int4_matmul_tiles_strip(
            x.to(dev), kops.int4_strip_copy(kernel, N), N, scale.to(dev), kernel_zero=None if zero is None else zero.to(dev),
            block_size=block_size, bias=b.to(dev)).cpu())
    assert torch.equal(got[0], got[1])
    rows = torch.tensor([0, 1, 31, 32, M // 2, M - 2, M - 1])
    exact = c_w4_matmul_f64(x[rows], qk["kernel"], scale, zero, block_size, b, N)
    mag = magnitude(x[rows], kernel, scale, zero, block_size, N)
    # (the bound of test_tile_plans with an offset of 136)
    bound = mag * 17 * 2.0 ** -24 * K ** 0.5 + (exact.abs() + 2 * b.double().abs()) * 3.05 * 2.0 ** -8
    err = (got[0][rows].double() - exact).abs()
    assert bool((err <= bound).all()), float((err / bound).max())
