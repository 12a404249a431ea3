"""`quantize()` hands the new variables their values as they are made: what they hold, and what a value that cannot be
held as it is (another dtype, another shape) does, is what building them and assigning afterwards gives."""

import pytest
import torch

from keras_amd.layers import Dense, EinsumDense
from keras_amd.quantization_config import Int4QuantizationConfig, Int8QuantizationConfig
from keras_amd.quantizers import AbsMaxQuantizer


class OddQuantizer(AbsMaxQuantizer):
    """Values as float32 integers, scales as float64 or with one entry too many."""

    short = False

    def __call__(self, x, to_numpy=False):
        q, scale = super().__call__(x, to_numpy=to_numpy)
        scale = scale.to(torch.float64)
        return q.to(torch.float32), torch.cat([scale, scale[..., :1]], -1) if self.short else scale


def build(kind, device):
    gen = torch.Generator().manual_seed(5)
    value = torch.randn(48, 40, generator=gen)
    layer = (Dense(40, use_bias=False, device=device, kernel_initializer=lambda s, d: value.to(d)) if kind == "dense" else
             EinsumDense("ab,bc->ac", (40,), device=device, kernel_initializer=lambda s, d: value.to(d)))
    layer.build((None, 48))
    return layer


def held(layer, mode, config):
    layer.quantize(mode, config=config)
    return {v.name.split("/")[-1]: (v.value.dtype, tuple(v.shape), v.version, v.value.clone()) for v in layer._variables}


def by_assign(layer, mode, config, monkeypatch):
    monkeypatch.setattr(type(layer), "_quantized_build_with",
                        lambda self, shape, mode, config, **values: self.quantized_build(shape, mode, config))
    out = held(layer, mode, config)
    monkeypatch.undo()
    return out


CONFIGS = [("int8", lambda: None), ("int8", lambda: Int8QuantizationConfig(weight_quantizer=OddQuantizer(axis=0))),
           ("int4", lambda: Int4QuantizationConfig(block_size=-1)), ("int4", lambda: Int4QuantizationConfig(block_size=20)),
           ("int4", lambda: Int4QuantizationConfig(block_size=16))]


def same(a, b):
    assert a.keys() == b.keys()
    for name in a:
        assert a[name][:3] == b[name][:3], name
        assert torch.equal(a[name][3], b[name][3]), name


@pytest.mark.parametrize("kind", ["dense", "einsum"])
@pytest.mark.parametrize("case", range(2))  # (int4 kernels are packed on the device only)
def test_values(kind, case, monkeypatch):
    mode, config = CONFIGS[case]
    same(held(build(kind, "cpu"), mode, config()), by_assign(build(kind, "cpu"), mode, config(), monkeypatch))


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["dense", "einsum"])
@pytest.mark.parametrize("case", range(len(CONFIGS)))
def test_values_on_the_device(kind, case, monkeypatch):
    mode, config = CONFIGS[case]
    same(held(build(kind, "cuda:0"), mode, config()), by_assign(build(kind, "cuda:0"), mode, config(), monkeypatch))


def test_a_value_of_another_shape_is_refused():
    quantizer = OddQuantizer(axis=0)
    quantizer.short = True
    with pytest.raises(ValueError, match="must match"):
        build("dense", "cpu").quantize("int8", config=Int8QuantizationConfig(weight_quantizer=quantizer))
