"""Derived operands that a layer keeps: rebuilt when the variable is assigned, never in the caller's memory."""

import pytest
import torch

from keras_amd import ops as kops
from keras_amd.layers import Dense, EinsumDense, ReversibleEmbedding
from keras_amd.layers.dense import strip_rows_params, tile_rows_operands


def quantized(kind, policy, source="_from_float32"):
    """A layer built in its quantized form."""
    policy += source
    if kind == "einsum":
        layer = EinsumDense("btd,dnh->btnh", (None, 4, 8), bias_axes="nh", dtype=policy, device="cpu")
        layer.build((None, None, 256))
    elif kind == "tied":
        layer = ReversibleEmbedding(32, 256, dtype=policy, device="cpu")
        layer.build()
    else:
        layer = Dense(32, dtype=policy, device="cpu")
        layer.build((None, 256))
    return layer


OPERANDS = {
    # name: (layer, variable, operand of the variable's value)
    "dense_bias": (lambda: quantized("dense", "int8"), "bias", lambda l: l._read_cached("bias", l.bias)),
    "dense_scale": (lambda: quantized("dense", "int8"), "kernel_scale",
                    lambda l: l._read_cached("kernel_scale", l.kernel_scale)),
    "dense_tile_scale_per_channel": (lambda: quantized("dense", "int4/-1"), "kernel_scale",
                                     lambda l: tile_rows_operands(l, torch.float32, 32, False)["kernel_scale"]),
    "dense_tile_scale": (lambda: quantized("dense", "int4/128"), "kernel_scale",
                         lambda l: tile_rows_operands(l, torch.float32, 32, True)["kernel_scale"]),
    "einsum_scale": (lambda: quantized("einsum", "int4/-1"), "kernel_scale",
                     lambda l: l._cached("kernel_scale", l.kernel_scale, lambda t: t.reshape(-1).contiguous())),
    "tied_scale": (lambda: quantized("tied", "int8"), "embeddings_scale",
                   lambda l: l._cached("scale", l.embeddings_scale, lambda t: t.contiguous())),
}


@pytest.mark.parametrize("name", OPERANDS)
def test_rebuild_leaves_the_assigned_tensors_alone(name):
    make, variable, operand = OPERANDS[name]
    layer = make()
    var = getattr(layer, variable)
    a, b = torch.full(var.shape, 1.0), torch.full(var.shape, 2.0)
    var.assign(a)
    first = operand(layer)
    assert torch.equal(first.flatten(), a.flatten())
    var.assign(b)
    second = operand(layer)
    assert torch.equal(second.flatten(), b.flatten())
    assert second.data_ptr() == first.data_ptr()  # (a captured graph holds it)
    assert bool((a == 1.0).all()) and bool((b == 2.0).all())
    var.assign(a)
    assert torch.equal(operand(layer).flatten(), torch.full(var.shape, 1.0).flatten())


def test_operand_of_the_same_type_follows_writes_into_the_variable():
    layer = quantized("dense", "int8")
    read = lambda: layer._read_cached("bias", layer.bias)
    before = read()
    layer.bias.value.add_(3.0)
    assert torch.equal(read(), layer.bias.value) and read().data_ptr() == before.data_ptr()


def test_packed_parameters_of_two_types_live_side_by_side(monkeypatch):
    made = []

    def pack(scale, zero, input_dim, units, block_size):
        made.append(scale.dtype)
        return torch.full((scale.numel() * scale.element_size(),), float(scale.flatten()[0]))

    monkeypatch.setattr(kops, "int4_strip_rows_params", pack)
    layer = quantized("dense", "int4/128")
    read = lambda dtype: strip_rows_params(layer, dtype, 256, 32, 128)
    wide, narrow = read(torch.float32), read(torch.bfloat16)
    assert read(torch.float32) is wide and read(torch.bfloat16) is narrow and len(made) == 2
    layer.kernel_scale.assign(torch.full(layer.kernel_scale.shape, 3.0))
    # rebuilt where they lie
    assert read(torch.float32) is wide and read(torch.bfloat16) is narrow
    assert float(wide[0]) == float(narrow[0]) == 3.0


def test_shared_launch_packs_nothing_for_rows_of_another_type(monkeypatch):
    packed = []
    monkeypatch.setattr(kops, "int4_strip_rows_params", lambda *a: packed.append("params") or torch.zeros(1))
    monkeypatch.setattr(kops, "int4_strip_copy", lambda *a: packed.append("copy") or torch.zeros(1))
    layer = Dense(24, dtype="int4/128_from_mixed_bfloat16", device="cpu", use_bias=False)
    layer.build((None, 256))
    spec = layer._int4_together_spec(torch.zeros(4, 256))  # float32 rows: the layer's call casts them first
    assert spec is not None and spec["rows"] is None and packed == []
    assert layer._int4_together_spec(torch.zeros(4, 256, dtype=torch.bfloat16))["rows"] is not None


@pytest.mark.parametrize("kind", ["dense", "einsum"])
def test_packed_parameters_of_the_decode_kernel_keep_their_address(monkeypatch, kind):
    monkeypatch.setattr(kops, "int4_strip_supported", lambda *a: True)
    monkeypatch.setattr(kops, "int4_strip_copy", lambda *a: torch.zeros(1))
    monkeypatch.setattr(kops, "int4_strip_params", lambda scale, *a: scale.clone())
    layer = quantized(kind, "int4/128", "_from_mixed_bfloat16")
    read = lambda: layer._strip_operands(1, 256, 32, True, 128)["gparams"]
    before = read()
    layer.kernel_scale.assign(torch.full(layer.kernel_scale.shape, 3.0))
    after = read()
    assert after.data_ptr() == before.data_ptr() and bool((after == 3.0).all())
