"""GPU parity: the tied int4 table as the LM head on the general form of the strip-linear decode kernel (float32 scales,
tables that the kernel proper does not fit), against the float64 value of the stored table and the kernel in place."""

import pytest
import torch

from keras_amd import ops as kops, quantizers
from keras_amd.layers import ReversibleEmbedding
from keras_amd.quantization_config import Int4QuantizationConfig

pytestmark = pytest.mark.gpu


def make(policy, vocab, dim, block_size, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    layer = ReversibleEmbedding(
        vocab, dim, dtype=policy, device="cuda:0",
        embeddings_initializer=lambda s, d: (torch.randn(s, generator=g, device="cuda") * 0.02).to(d))
    layer.build()
    layer.quantize("int4", config=Int4QuantizationConfig(block_size=block_size))
    return layer


def operands(layer, block_size):
    w = quantizers.unpack_int4(layer._embeddings.value, layer.output_dim, axis=-1).double()
    scale = layer.embeddings_scale.value.double()
    if block_size > 0:
        group = torch.arange(layer.output_dim, device=w.device) // block_size
        return (w - layer.embeddings_zero.value.double()[:, group]), scale[:, group]
    return w, 1 / scale.reshape(-1, 1)


def check(layer, x, block_size):
    w, scale = operands(layer, block_size)
    exact = x.double() @ (w * scale).t()
    got = layer(x, reverse=True)
    # (an offset of up to 24 + 8 on every weight is taken out of the sums again)
    mag = x.double().abs() @ ((w.abs() + 48) * scale.abs()).t()
    K = x.shape[1]
    if got.dtype == torch.float32:
        # two parts of a float32 value leave 2^-17 of it; float32 sums of K terms 2^-24 sqrt(K) of the magnitudes, four times
        # that; the result's own roundings
        split = 2.0 ** -17 if x.dtype == torch.float32 else 0.0
        bound = mag * (split + 4 * 2.0 ** -24 * K ** 0.5) + exact.abs() * 2.0 ** -22
    else:  # sum and quotient rounded to bfloat16, half an ulp or 2^-8 each
        bound = mag * 4 * 2.0 ** -24 * K ** 0.5 + exact.abs() * 2.05 * 2.0 ** -8
    err = (got.double() - exact).abs()
    assert bool((err <= bound).all()), float((err / bound).max())
    return got


@pytest.mark.parametrize("policy,block_size,vocab,dim", [
    ("mixed_bfloat16", 128, 1000, 4096), ("mixed_bfloat16", 128, 1003, 4224), ("float32", 128, 1000, 2048),
    ("float32", -1, 1000, 4096), ("float32", 128, 1003, 2048), ("float32", -1, 1001, 2056), ("bfloat16", 128, 1003, 2048),
    ("bfloat16", -1, 1000, 2064), ("float32", 128, 1000, 4544),
])
@pytest.mark.parametrize("M", [1, 4])
def test_tied_rows(dev, policy, block_size, vocab, dim, M):
    layer = make(policy, vocab, dim, block_size)
    x = torch.randn(M, dim, generator=torch.Generator().manual_seed(M)).to(dev)
    x = x if policy == "float32" else x.to(torch.bfloat16)
    check(layer, x, block_size)
    assert "w4s" in layer._cache and ("w4s_rows_params" in layer._cache) == (block_size > 0)
    params = layer._cache["w4s_rows_params"][2].data_ptr() if block_size > 0 else None
    # other parameters: the packed ones are rebuilt where they lie
    layer.embeddings_scale.assign(layer.embeddings_scale.value.flip(0))
    if block_size > 0:
        layer.embeddings_zero.assign(-layer.embeddings_zero.value)
    check(layer, x, block_size)
    assert params is None or layer._cache["w4s_rows_params"][2].data_ptr() == params


@pytest.mark.parametrize("block_size", [128, -1])
@pytest.mark.parametrize("policy", ["float32", "bfloat16", "mixed_bfloat16"])
def test_tied_rows_where_the_kernel_in_place_multiplies_float32(dev, policy, block_size):
    """K % 128: no further from 64 bits than that kernel, and an infinity gives what a float product gives."""
    dim = 4544
    layer = make(policy, 2000, dim, block_size)
    x = torch.randn(3, dim, generator=torch.Generator().manual_seed(1)).to(dev)
    x = x if policy == "float32" else x.to(torch.bfloat16)
    zero = layer.embeddings_zero.value if block_size > 0 else None
    in_place = lambda x: kops.int4_matmul_nk(x, layer._embeddings.value, layer.embeddings_scale.value, zero=zero,
                                             block_size=block_size if block_size > 0 else None)
    w, scale = operands(layer, block_size)
    for rows in (x, x.relu()):
        exact = rows.double() @ (w * scale).t()
        off = lambda y: float((y.double() - exact).norm() / exact.norm())
        got, want = layer(rows, reverse=True), in_place(rows)
        if got.dtype == torch.float32 and (policy == "float32" or block_size > 0):
            assert off(got) <= max(off(want), 2.0 ** -24)
        else:  # (roundings to bfloat16 hide the sums)
            assert off(got) <= 1.02 * off(want)
    x[1, 7] = float("inf")
    got, want = layer(x, reverse=True).float()[1], in_place(x).float()[1]
    assert torch.equal(got.nan_to_num(nan=3.0), want.nan_to_num(nan=3.0)) and bool(got.isinf().any())
