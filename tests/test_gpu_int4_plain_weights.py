"""GPU parity: the general int4 kernels on shapes with N % 8 or K % 16, where they take the weights without an offset, against
the kernel on the stored weights, which multiplies float32 values for these shapes."""

import pytest
import torch

from keras_amd import ops as kops
from tests.helpers import c_w4_matmul_f64
from tests.test_gpu_int4_matmul import make_layer

pytestmark = pytest.mark.gpu

SHAPES = [(2048, 5247, 128), (1000, 777, 128), (2056, 904, None), (136, 5, None), (3000, 9001, 128), (24, 31, 128),
          (8192, 1005, 128)]


class Kernel:
    def __init__(self, dev, dtype, K, N, block_size):
        self.qk, _ = make_layer(K, N, block_size, seed=K + N, with_bias=False)
        self.N, self.block_size = N, block_size
        self.scale, self.zero = self.qk["kernel_scale"].to(dtype), self.qk["kernel_zero"] if block_size else None
        self.packed, scale = self.qk["kernel"].to(dev), self.scale.to(dev)
        zero = self.zero.to(dev) if block_size else None
        self.copy = kops.int4_strip_copy(self.packed, N)
        grouped = dict(block_size=block_size)
        self.stored = lambda x: kops.int4_matmul(x, self.packed, scale, N, kernel_zero=zero, **grouped)
        if block_size:
            params = kops.int4_strip_rows_params(scale, zero, K, N, block_size)
            self.decode = lambda x: kops.int4_matmul_strip_rows(x, self.copy, N, gparams=params, **grouped)
            columns = [kops.int4_tile_columns(t, N) for t in (scale, zero)]
            self.tiles = lambda x: kops.int4_matmul_tiles_rows(x, self.copy, N, columns[0], kernel_zero=columns[1], **grouped)
        else:
            self.decode = lambda x: kops.int4_matmul_strip_rows(x, self.copy, N, kernel_scale=scale)
            self.tiles = lambda x: kops.int4_matmul_tiles_rows(x, self.copy, N, scale)

    def __call__(self, x):
        return self.decode(x) if x.shape[0] <= 16 else self.tiles(x)


@pytest.mark.parametrize("K,N,block_size", SHAPES)
@pytest.mark.parametrize("M", [1, 5, 16, 40, 130])
def test_float32_rows_without_negative_values_lose_nothing(dev, M, K, N, block_size):
    """Rows behind a relu have large sums that an offset on the weights would have to cancel."""
    kernel = Kernel(dev, torch.float32, K, N, block_size)
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(M)).relu()
    exact = c_w4_matmul_f64(x, kernel.qk["kernel"], kernel.scale, kernel.zero, block_size, None, N)
    off = lambda y: float((y.double().cpu() - exact).norm() / exact.norm())
    # (both are float32 sums in some order: a result is rounded to half an ulp whatever the order)
    assert off(kernel(x.to(dev))) <= max(off(kernel.stored(x.to(dev))), 2.0 ** -24)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("K,N,block_size", SHAPES)
@pytest.mark.parametrize("M", [4, 40])
def test_rows_that_are_not_finite(dev, dtype, M, K, N, block_size):
    """An infinity gives what a float product gives, and nothing to the other rows."""
    kernel = Kernel(dev, dtype, K, N, block_size)
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(K)).to(dtype)
    rest = x.clone()
    for row, value in ((0, float("inf")), (1, float("-inf")), (2, float("nan"))):
        x[row, (7 * row + 3) % K] = value
        rest[row] = 0
    x[M - 1, 0], x[M - 1, K - 1], rest[M - 1] = float("inf"), float("inf"), 0
    got, want, others = (kernel(x.to(dev)).float(), kernel.stored(x.to(dev)).float(), kernel(rest.to(dev)).float())
    special = [0, 1, 2, M - 1]
    assert torch.equal(got[special].nan_to_num(nan=3.0), want[special].nan_to_num(nan=3.0))
    assert bool(got[[0, 1]].isinf().any()) and bool(got[2].isnan().all())
    if M > 4:
        assert torch.equal(got[3:M - 1], others[3:M - 1])


@pytest.mark.parametrize("dtype,bound", [(torch.float32, 2.0 ** -20), (torch.bfloat16, 2.0 ** -7)])
@pytest.mark.parametrize("K,N,block_size", [s for s in SHAPES if s[0] >= 128])
@pytest.mark.parametrize("M", [3, 33])
def test_rows_of_huge_values(dev, dtype, bound, M, K, N, block_size):
    """24 times the sum of such a row is beyond float32, its products with the kernel are not.  (A bfloat16 result is
    rounded twice, half an ulp or 2^-8 each; float32 sums of up to 3000 terms differ by far less than 2^-20.)"""
    kernel = Kernel(dev, dtype, K, N, block_size)
    x = ((torch.rand(M, K, generator=torch.Generator().manual_seed(N)) + 1) * 1.4e35).to(dtype).to(dev)
    got, want = kernel(x).double(), kernel.stored(x).double()
    assert bool(want.isfinite().all()) and bool(got.isfinite().all())
    assert float(((got - want) * 2.0 ** -100).norm()) <= bound * float((want * 2.0 ** -100).norm())
