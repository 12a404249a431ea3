"""GPU: what a prompt's attention makes of infinite values, NaN and positions that see no row: what the library's kernel and
float64 make of them."""

import math

import pytest
import torch

from keras_amd import ops as kops
from tests.test_gpu_prompt_attention import attention64

pytestmark = pytest.mark.gpu


def library(q, k, v, mask):
    return torch.nn.functional.scaled_dot_product_attention(q.transpose(1, 2), k, v, attn_mask=mask[None, None]).transpose(1, 2)


def same_kind(a, b):
    return torch.equal(a.isnan(), b.isnan()) and torch.equal(a == math.inf, b == math.inf) and torch.equal(a == -math.inf, b == -math.inf)


# (one block of rows with a short end, whole blocks, a short last block)
@pytest.mark.parametrize("max_len,T", [(20, 5), (64, 64), (132, 70), (256, 17)])
def test_values_that_are_no_numbers(dev, max_len, T):
    g = torch.Generator().manual_seed(max_len)
    mk = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16)
    q, k, v = mk(2, T, 3, 128), mk(2, 3, max_len, 128), mk(2, 3, max_len, 128)
    mask = mk(T, max_len)
    mask[:, 1:4] = 0
    mask[T // 2:, 2] = float("-inf")  # a row that half of the positions see
    v[:, :, 0, 3], v[:, :, 2, 7] = math.inf, -math.inf
    v[:, :, max_len - 1, 9], v[:, :, max_len // 2, 11] = -math.inf, math.nan
    v[1, 2, 0, 20], v[1, 2, max_len - 1, 20] = math.inf, -math.inf
    args = [t.to(dev) for t in (q, k, v, mask)]
    got, want = kops.prompt_attention(*args), attention64(*args)
    assert same_kind(got.double(), want) and same_kind(got, library(*args))
    # results of finite values are those of the same call without the others
    clean = torch.where(args[2].isfinite(), args[2], torch.zeros_like(args[2]))
    plain = kops.prompt_attention(args[0], args[1], clean, args[3])
    assert torch.equal(got[want.isfinite()], plain[want.isfinite()])


def test_position_that_sees_nothing(dev):
    mk = lambda *s: torch.randn(*s, generator=torch.Generator().manual_seed(4)).to(torch.bfloat16).to(dev)
    q, k, v = mk(1, 70, 2, 128), mk(1, 2, 96, 128), mk(1, 2, 96, 128)
    mask = torch.zeros(70, 96, dtype=torch.bfloat16, device=dev)
    mask[3], mask[65:] = float("-inf"), float("-inf")
    got, lib = kops.prompt_attention(q, k, v, mask), library(q, k, v, mask)
    assert not got[:, 3].any() and not got[:, 65:].any() and not lib[:, 3].any()
    assert bool(got.isfinite().all()) and bool(got[:, 4].any())


@pytest.mark.parametrize("value", [torch.finfo(torch.bfloat16).min, -2.4e38, -2.3e38, -1e9, -30.0])
def test_masks_of_low_finite_values(dev, value):
    """A row that is low all over, and rows that are low in part."""
    mk = lambda *s: torch.randn(*s, generator=torch.Generator().manual_seed(6)).to(torch.bfloat16).to(dev)
    q, k, v = mk(1, 20, 2, 128), mk(1, 2, 128, 128), mk(1, 2, 128, 128)
    mask = torch.zeros(20, 128, dtype=torch.bfloat16, device=dev)
    mask[3] = value
    mask[4, 64:], mask[5, :64], mask[6, ::2] = value, value, value
    mask[7], mask[7, 100] = value, 0
    got, lib = kops.prompt_attention(q, k, v, mask).double(), library(q, k, v, mask).double()
    assert bool(got.isfinite().all())
    assert torch.equal(got[:, 3] == 0, lib[:, 3] == 0)
    # (either is a rounding of the result to bfloat16 and a few of its probabilities away from float64's)
    assert float((got - lib).norm() / lib.norm()) < 2.0 ** -8
    for row in (3, 4, 5, 6, 7):
        assert float((got[:, row] - lib[:, row]).abs().max()) <= 2.0 ** -6 * max(1.0, float(lib[:, row].abs().max()))
