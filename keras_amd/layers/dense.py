"""`Dense` with the int8 / int4 quantized forward on MI355X.

Mirrors the quantization-related surface of `keras.layers.Dense`
(keras/src/layers/core/dense.py): variable names, shapes and dtypes
(`_kernel`, `kernel_scale`, `kernel_zero`, `g_idx`, `bias`), `quantize(mode,
config)`, the dtype-policy names it leaves behind, the positional
`save_own_variables` / `load_own_variables` order, and `_int8_call` /
`_int4_call`.  The two call methods run the k3q HIP kernels; the float `call`
is a plain torch matmul and exists so that a float layer can be built,
compared against and converted.
"""

import math

import torch

from keras_amd import dtype_policies, ops as kops, quantizers
from keras_amd.layers.layer import (Layer, as_tensor, cached_operand, cached_params, require_default_g_idx,
                                    to_torch_dtype)
from keras_amd.layers.together import quantize_rows, quantizes_alone
from keras_amd.quantization_config import QuantizationConfig, get_block_size_for_layer

_ACTIVATIONS = {
    None: None,
    "linear": None,
    "relu": torch.relu,
    "gelu": torch.nn.functional.gelu,
    "silu": torch.nn.functional.silu,
    "swish": torch.nn.functional.silu,
    "sigmoid": torch.sigmoid,
    "tanh": torch.tanh,
}

# `exact_epilogue` of a layer: None / True reproduce the reference's rounding chain bit for
# bit (the default: it costs under 2 % of a prefill-sized matmul); False rounds once at the end.


def activation_name(fn):
    for name, f in _ACTIVATIONS.items():
        if f is fn:
            return name
    raise ValueError(f"activation {fn} has no serializable name")


def serialize_quantization_config(config):
    if config is None:
        return None
    return {"class_name": type(config).__name__, "config": config.get_config()}


def glorot_uniform(shape, dtype, generator=None):
    """U(-L, L), L = sqrt(6 / (fan_in + fan_out))
    (keras/src/initializers/random_initializers.py:292-318)."""
    fan_in, fan_out = shape[0], shape[-1]
    if len(shape) > 2:
        receptive = 1
        for d in shape[:-2]:
            receptive *= d
        fan_in, fan_out = shape[-2] * receptive, shape[-1] * receptive
    limit = math.sqrt(6.0 / (fan_in + fan_out))
    return ((torch.rand(shape, generator=generator) * 2.0 - 1.0) * limit).to(dtype)


def he_uniform(shape, dtype, generator=None):
    """U(-L, L), L = sqrt(6 / fan_in) (keras/src/initializers/random_initializers.py, `HeUniform`)."""
    fan_in = shape[0]
    if len(shape) > 2:
        receptive = 1
        for d in shape[:-2]:
            receptive *= d
        fan_in = shape[-2] * receptive
    limit = math.sqrt(6.0 / max(fan_in, 1))
    return ((torch.rand(shape, generator=generator) * 2.0 - 1.0) * limit).to(dtype)


LORA_INITIALIZERS = {"he_uniform": he_uniform, "zeros": "zeros", "ones": "ones"}


def lora_initializer(spec):
    if callable(spec):
        return spec
    if spec not in LORA_INITIALIZERS:
        raise ValueError(f"Unknown initializer: {spec}")
    return LORA_INITIALIZERS[spec]


# rows for which the int4 forward reads the kernel as int4 tiles, from the strip-linear copy or (groups of 64) a
# K-contiguous one, measured against the 32-row passes below it (17 rows 13.4 us at K=N=4096, where the tiles take 14.5)
# and the de-quantise + GEMM route above it (512 rows: K=4096, N=14336 98 against 69; K=N=4096 45 against 29; K=14336,
# N=4096 102 against 74).  What larger calls of the strip-linear copy keep on tiles: int4_tile_rows_route.
KMAJOR_MIN_ROWS, KMAJOR_MAX_ROWS = 33, 512
# from 17 rows on kernels at least this wide or this large (17 rows, groups of 128, us:
# K=5120, N=13824: 26 against 36; K=13824, N=5120: 29 against 37; K=11008, N=4096: 25 against
# 27; K=8192, N=28672: 59 against 129; K=N=5120: 18 against 18.5 and K=N=4096: 14.5 against
# 13.4, both left on the decode kernel)
KMAJOR_MIN_ROWS_WIDE, KMAJOR_WIDE_UNITS, KMAJOR_LARGE_WEIGHTS = 17, 8192, 40 << 20


def kmajor_rows(rows, units, input_dim=0):
    """Whether `rows` bfloat16 rows into `units` outputs take the K-contiguous int4 route."""
    wide = units >= KMAJOR_WIDE_UNITS or units * input_dim >= KMAJOR_LARGE_WEIGHTS
    low = KMAJOR_MIN_ROWS_WIDE if wide else KMAJOR_MIN_ROWS
    return low <= rows <= KMAJOR_MAX_ROWS


def int4_strip_rows_route(dtype, rows, input_dim, units, block_size):
    """Whether an int4 call of these rows goes to `ops.int4_matmul_strip_rows`: what the strip kernel proper
    (`ops.int4_strip_supported`) does not take of up to 16 rows -- float32 rows, narrow, short or ragged kernels.
    A launch costs what one of the kernel on the stored weights costs, which takes 8 float32 or 16 bfloat16 rows
    (us, 1 / 8 / 16 rows, stored against strip: K=4096, N=14336 float32 15.5 / 16.5 / 31.8 against 10.9 / 12.1 / 33.9
    in three launches; K=N=4096 8.2 / 9.5 / 18.6 against 4.7 / 6.6 / 12.3; bfloat16 K=1600, N=6400 7.1 / 8.4 / 10.2
    against 5.4 / 5.9 / 6.1; K=11008, N=4096 at 8 rows 16.1 against 16.5 in two launches).  Where N % 8 or K % 16
    leave only the kernel of one output per thread (N = 5247: 220 ... 490 us) every shape goes here."""
    if not (dtype in (torch.float32, torch.bfloat16) and 0 < rows <= kops.STRIP_MAX_ROWS):
        return False
    launches = kops.int4_strip_rows_launches(dtype, rows, input_dim, units, block_size)
    if units % 8 or input_dim % 16:
        return launches > 0
    # All of K stays inside a workgroup here, however few columns there are; the kernel on the stored weights splits K.  At
    # the widths it fills the chip with, a long enough K is faster split (us, stored against strip, 1 row: 24576 x 768
    # float32 12.1 / 13.3, 28672 x 1024 13.9 / 14.9, 32768 x 576 13.2 / 16.0; bfloat16 43008 x 512 15.4 / 17.6).  Wider or
    # narrower it is not (24576 x 512 float32 16.5 / 13.1, 28672 x 512 25.5 / 14.6, 32768 x 256 25.7 / 15.6, 1152 16.8 / 16.4).
    if 384 < units <= 1024 and input_dim >= (24576 if units > 640 else 32768):
        return False
    return 0 < launches <= (-(-rows // 8) if dtype == torch.float32 else 1)


ROWS_PARAMS = {torch.float32: "w4s_rows_params", torch.bfloat16: "w4s_rows_params_bfloat16"}


def strip_rows_params(layer, dtype, input_dim, units, block_size):
    """The grouped parameters of `ops.int4_matmul_strip_rows` in `dtype`: made on first use, rebuilt in place
    when a variable they come from is assigned (a captured graph holds their address).  Each dtype has its own."""
    scale, zero, key = layer.kernel_scale, layer.kernel_zero, ROWS_PARAMS[dtype]
    hit = layer._cache.get(key)
    if hit is not None and hit[0] == (id(scale), scale.version, id(zero), zero.version):
        return hit[2]
    return cached_params(layer._cache, key, scale, zero, lambda: kops.int4_strip_rows_params(
        as_tensor(scale).to(dtype), as_tensor(zero), input_dim, units, block_size))


# Rows up to which the int4 tile kernel beats the GEMM on the de-quantised kernel (us, GEMM route / tiles).  Float32: grouped
# K=N=4096 1024 rows 138 / 93, 2048 225 / 186; K=8192, N=4096 800 rows 249 / 146; K=4096, N=11008 2048 rows 688 / 462; 1024 rows of
# K=N=2048 53 / 43, K=4096, N=1024 56.5 / 55.0; K=N=2048 4000 rows 132 / 180: small kernels up to 1024.  Per channel (two parts a
# weight fewer for the GEMM) K=N=4096 700 rows 97 / 74, 1024 98 / 101.  Bfloat16: while the tiles are one turn of the chip,
# and enough for it (weights without an offset, as the GEMM's): 1024 rows K=N=4096 55 / 41, K=14336, N=4096 153 / 128, K=N=2048
# 36 / 19, 640 rows K=N=4096 51 / 38, K=4096, N=1024 28 / 24; with an offset K=4096, N=14336 138 / 143.
TILE_ROWS_MAX_F32, TILE_ROWS_MAX_F32_LARGE, TILE_ROWS_MAX_F32_CHANNEL, TILE_LARGE_WEIGHTS = 1024, 2048, 768, 16 << 20
TILE_ROWS_MAX_BF16, TILE_COUNTS_BF16 = 1024, (32, 256)


def int4_tile_rows_route(dtype, rows, input_dim, units, block_size):
    """Whether an int4 call of more rows than the decode kernels take goes to `ops.int4_matmul_tiles_rows`: shapes
    that neither the tile kernel's aligned entry (`ops.int4_kmajor_supported`) nor the GEMM on the de-quantised kernel takes
    (K % 128, N % 64), which went in passes of 32 bfloat16 or 8 float32 rows over the kernel (us, passes / tiles: K=1600,
    N=6400 bfloat16 48 rows 25.6 / 13, 300 137 / 17; float32 17 rows 25 / 14, 300 307 / 24; one pass, up to 32 bfloat16 rows of a
    kernel this small, is as good), and rows of aligned shapes up to the limits above.  Where N % 8 or K % 16 leave only the
    kernel of one output per thread (K=2048, N=5247: 480 us at 32 rows, 6.1 ms at 1200, against 15 and 55) every shape
    goes here."""
    if not (dtype in (torch.float32, torch.bfloat16) and rows > kops.STRIP_MAX_ROWS
            and kops.int4_tiles_rows_supported(input_dim, units, block_size)):
        return False
    if units % 8 or input_dim % 16:
        return True
    gemm = input_dim % 128 == 0 and units % 64 == 0
    if not gemm:
        return dtype == torch.float32 or rows >= KMAJOR_MIN_ROWS or kmajor_rows(rows, units, input_dim)
    if dtype == torch.float32:
        if not block_size:
            return rows <= TILE_ROWS_MAX_F32_CHANNEL
        return rows <= (TILE_ROWS_MAX_F32_LARGE if input_dim * units >= TILE_LARGE_WEIGHTS else TILE_ROWS_MAX_F32)
    low, high = TILE_COUNTS_BF16
    return KMAJOR_MAX_ROWS < rows <= TILE_ROWS_MAX_BF16 and low <= -(-rows // 128) * -(-units // 128) <= high


def tile_rows_operands(layer, dtype, units, grouped):
    """Scales and zero points of `ops.int4_matmul_tiles_rows` in `dtype`, kept while the variables do not change."""
    if not grouped:
        return dict(kernel_scale=layer._cached("kernel_scale", layer.kernel_scale, lambda t: t.to(dtype).contiguous()))
    return dict(kernel_scale=layer._cached("tile_scale", layer.kernel_scale,
                                           lambda t: kops.int4_tile_columns(t.to(dtype), units)),
                kernel_zero=(layer._cached("tile_zero", layer.kernel_zero, lambda t: kops.int4_tile_columns(t, units))
                             if units % 32 else as_tensor(layer.kernel_zero)))


def int8_strip_route(quantizer, x2, units, strict=False):
    """Whether an int8 call of these rows goes to `ops.int8_dense_strip`: rows on the device, few
    enough, a plain abs-max quantizer (whatever its range and epsilon), a shape the kernel takes.
    Every shape it takes is faster there than behind the two-launch routes (rows 1, 4, 8 and 16,
    quantizer included, us, strip against stored kernel or tiles: K=N=4096 float32 8.8 / 9.6 / 9.8 / 10.3
    against 12.2 / 13.3 / 14.0 / 29.4; K=1600, N=6400 8.5 ... 10.6 against 10.6 ... 12.2; K=8192, N=1024
    8.6 ... 11.9 against 13.9 ... 48.7; K=N=768 6.7 ... 7.5 against 9.2 ... 13.3).  So it is for a long K on few columns,
    all of which stays in a workgroup (cold weights: K=28672, 1 row, N=16 / 512 / 1024 / 8192 float32 19.0 / 20.8 / 23.1 /
    51.4 against 27.9 / 35.1 / 40.6 / 58.1; K=14336, N=128, 8 rows 16.2 against 21.5).
    strict: only bfloat16 rows and the widths of `ops.int8_strip_supported`: what a launch that several
    layers share takes, and what a tied table keeps a copy for."""
    if not (type(quantizer) is quantizers.AbsMaxQuantizer and quantizer.output_dtype == "int8"
            and x2.is_cuda and 0 < x2.shape[0] <= kops.INT8_STRIP_MAX_ROWS):
        return False
    if x2.dtype == torch.bfloat16 and kops.int8_strip_supported(x2.shape[0], x2.shape[1], units):
        return True
    return (not strict and x2.dtype in (torch.float32, torch.bfloat16)
            and kops.int8_strip_rows_supported(x2.shape[0], x2.shape[1], units))


def int8_rows_route(x2, dtype, units, bias):
    """Whether an int8 call of more rows than the decode kernels take goes to `ops.int8_dense_rows`: everything the tile
    GEMM reads from the strip-linear copy, with a bias for all rows.  (The same launches as quantizer and product called one by
    one; eager, us, one by one / in one call: 64 rows of 4096 x 4096 float32 32.0 / 20.2, 100 of 1600 x 6400 bfloat16 27.5 / 18.7.)"""
    return (x2.is_cuda and x2.dtype == dtype and dtype in (torch.float32, torch.bfloat16) and x2.shape[1] % 64 == 0
            and x2.shape[0] > kops.INT8_STRIP_MAX_ROWS and (bias is None or bias.numel() == units))


class Dense(Layer):
    def __init__(self, units, activation=None, use_bias=True, kernel_initializer=None,
                 bias_initializer="zeros", dtype=None, name=None, device=None,
                 quantization_config=None, lora_rank=None, lora_alpha=None):
        super().__init__(dtype=dtype, name=name, device=device)
        self.quantization_config = quantization_config  # dense.py:98-130
        self.lora_rank = lora_rank
        self.lora_alpha = lora_alpha if lora_alpha is not None else lora_rank
        if not isinstance(units, int) or units <= 0:
            raise ValueError(
                f"Received an invalid value for `units`, expected a positive integer. Received: units={units}"
            )
        self.units = units
        self.activation = activation if callable(activation) else _ACTIVATIONS[activation]
        self.use_bias = use_bias
        self.kernel_initializer = kernel_initializer or glorot_uniform
        self.bias_initializer = bias_initializer
        self.lora_enabled = False
        self.exact_epilogue = None
        self._cache = {}

    # ---- build --------------------------------------------------------------
    def build(self, input_shape):
        self._build_input_shape = tuple(input_shape)
        kernel_shape = (input_shape[-1], self.units)
        if self.quantization_mode:
            self.quantized_build(kernel_shape, mode=self.quantization_mode,
                                 config=self.quantization_config)
        if self.quantization_mode not in ("int8", "int4"):
            self._kernel = self.add_weight(
                name="kernel", shape=kernel_shape, initializer=self.kernel_initializer, trainable=True
            )
        if self.use_bias:
            self.bias = self.add_weight(
                name="bias", shape=(self.units,), initializer=self.bias_initializer, trainable=True
            )
        else:
            self.bias = None
        self.built = True
        if self.lora_rank:
            self.enable_lora(self.lora_rank)  # (dense.py:160-161: the alpha is not passed on)

    @property
    def kernel(self):
        """The kernel as a consumer sees it: the int4 kernel comes back unpacked to
        `[input_dim, units]` int8; with LoRA enabled the low-rank update is added and the sum
        cast to the compute dtype (keras/src/layers/core/dense.py:163-236)."""
        if not self.built:
            raise AttributeError("You must build the layer before accessing `kernel`.")
        kernel = as_tensor(self._kernel)
        if self.quantization_mode == "int4":
            kernel = quantizers.unpack_int4(kernel, self._orig_output_dim, axis=-1)
        if self.lora_enabled:
            delta = (self.lora_alpha / self.lora_rank) * torch.matmul(
                as_tensor(self.lora_kernel_a), as_tensor(self.lora_kernel_b))
            kernel = torch.add(kernel, delta).to(to_torch_dtype(self.compute_dtype))
        return kernel

    def enable_lora(self, rank, lora_alpha=None, a_initializer="he_uniform", b_initializer="zeros"):
        """keras/src/layers/core/dense.py:251-312: float32 `lora_kernel_a` [input_dim, rank] and
        `lora_kernel_b` [rank, units]; the forward adds (alpha / rank) * (x . a) . b."""
        if not self.built:
            raise ValueError("Cannot enable lora on a layer that isn't yet built.")
        if self.lora_enabled:
            raise ValueError("lora is already enabled. This can only be done once per layer.")
        if self.quantization_mode == "int4" and hasattr(self, "_orig_input_dim"):
            input_dim = self._orig_input_dim
        else:
            input_dim = self._kernel.shape[0]
        self.lora_kernel_a = self.add_weight(name="lora_kernel_a", shape=(input_dim, rank), dtype="float32",
                                             initializer=lora_initializer(a_initializer), trainable=True)
        self.lora_kernel_b = self.add_weight(name="lora_kernel_b", shape=(rank, self.units), dtype="float32",
                                             initializer=lora_initializer(b_initializer), trainable=True)
        self.lora_enabled = True
        self.lora_rank = rank
        self.lora_alpha = lora_alpha if lora_alpha is not None else rank

    def _quantized_call_with_lora(self, quantized_call, inputs):
        """The reference's order with LoRA enabled (dense.py:972-986, :1085-1095): the de-scaled
        quantized product first, then the low-rank term, the cast, the bias, the activation --
        so the kernels run without their fused bias here."""
        bias, activation = self.bias, self.activation
        self.bias, self.activation, self.lora_enabled = None, None, False
        try:
            x = quantized_call(inputs)
        finally:
            self.bias, self.activation, self.lora_enabled = bias, activation, True
        x = torch.add(x, self._lora_term(inputs)).to(to_torch_dtype(self.compute_dtype))
        if bias is not None:
            x = torch.add(x, self.read(bias))
        if activation is not None:
            x = activation(x)
        return x

    def _lora_term(self, inputs):
        """(alpha / rank) * (inputs . a) . b as the quantized calls add it (dense.py:977-980,
        :1086-1089): two small float matmuls in the compute dtype."""
        lora_x = torch.matmul(inputs, self.read(self.lora_kernel_a))
        lora_x = torch.matmul(lora_x, self.read(self.lora_kernel_b))
        return (self.lora_alpha / self.lora_rank) * lora_x

    def call(self, inputs, training=None):
        if self.lora_enabled:
            x = torch.matmul(inputs, self.kernel)
            if self.bias is not None:
                x = torch.add(x, self.read(self.bias))
            return self.activation(x) if self.activation is not None else x
        x = torch.matmul(inputs, self.read(self._kernel))
        if self.bias is not None:
            x = torch.add(x, self.read(self.bias))
        if self.activation is not None:
            x = self.activation(x)
        return x

    # ---- quantized variables --------------------------------------------------
    def quantized_build(self, kernel_shape, mode, config=None):
        if mode == "int8":
            self._int8_build(kernel_shape, config)
        elif mode == "int4":
            self._int4_build(kernel_shape, config)
        else:
            raise self._quantization_mode_error(mode)
        self._is_quantized = True

    def _int8_build(self, kernel_shape, config=None):
        self.inputs_quantizer = QuantizationConfig.activation_quantizer_or_default(
            config, quantizers.AbsMaxQuantizer()
        )
        self._kernel = self.add_weight(name="kernel", shape=kernel_shape, dtype="int8")
        self.kernel_scale = self.add_weight(name="kernel_scale", shape=(self.units,), initializer="ones")

    def _int4_build(self, kernel_shape, config=None):
        self.inputs_quantizer = QuantizationConfig.activation_quantizer_or_default(config, None)
        input_dim, output_dim = kernel_shape
        packed_cols = (output_dim + 1) // 2
        self._kernel = self.add_weight(name="kernel", shape=(input_dim, packed_cols), dtype="int8")
        block_size = get_block_size_for_layer(self, config)
        self._int4_block_size = block_size
        if block_size is None or block_size == -1:
            scale_shape = (self.units,)
        else:
            scale_shape = (math.ceil(input_dim / block_size), self.units)
        self.kernel_scale = self.add_weight(name="kernel_scale", shape=scale_shape, initializer="ones")
        if block_size is not None and block_size > 0:
            self.kernel_zero = self.add_weight(name="kernel_zero", shape=scale_shape, dtype="int8")
            # float32 on purpose, as in the reference (dense.py:868-889); made where it stays: a copy from the host would
            # wait for the quantizer that is running
            self.g_idx = self.add_weight(
                name="g_idx", shape=(input_dim,), dtype="float32",
                initializer=lambda shape, dtype: torch.floor_divide(
                    torch.arange(input_dim, dtype=dtype, device=self.device), block_size),
            )
        self._orig_input_dim = input_dim
        self._orig_output_dim = output_dim

    # ---- quantize (one-time, host side) --------------------------------------
    def _quantize(self, mode, config, type_check=True):
        if type_check and type(self) is not Dense:
            raise self._not_implemented_error(self.quantize)
        self.quantization_config = config
        kernel_shape = self._kernel.shape
        if mode == "int8":
            weight_quantizer = QuantizationConfig.weight_quantizer_or_default(
                config, quantizers.AbsMaxQuantizer(axis=0)
            )
            kernel_value, kernel_scale = weight_quantizer(as_tensor(self._kernel), to_numpy=True)
            kernel_scale = torch.squeeze(kernel_scale, dim=0)
            self._drop_float_kernel()
            self._quantized_build_with(kernel_shape, mode, config, kernel=kernel_value, kernel_scale=kernel_scale)
            self._kernel.assign(kernel_value)
            self.kernel_scale.assign(kernel_scale)
        elif mode == "int4":
            block_size = get_block_size_for_layer(self, config)
            kernel_zero = None
            if block_size is None or block_size == -1:
                weight_quantizer = QuantizationConfig.weight_quantizer_or_default(
                    config,
                    quantizers.AbsMaxQuantizer(axis=0, value_range=(-8, 7), output_dtype="int8"),
                )
                kernel_value_int4, kernel_scale = weight_quantizer(as_tensor(self._kernel), to_numpy=True)
                kernel_scale = torch.squeeze(kernel_scale, dim=0)
                packed, _, _ = quantizers.pack_int4(kernel_value_int4.to(self.device), axis=-1)
            else:
                packed, kernel_scale, kernel_zero = quantizers.quantize_and_pack_grouped(
                    as_tensor(self._kernel), block_size, self.device)
            self._drop_float_kernel()
            self._quantized_build_with(kernel_shape, mode, config, kernel=packed, kernel_scale=kernel_scale,
                                       kernel_zero=kernel_zero)
            self._kernel.assign(packed)
            self.kernel_scale.assign(kernel_scale)
            if kernel_zero is not None:
                self.kernel_zero.assign(kernel_zero)
        else:
            raise self._quantization_mode_error(mode)

        if self.dtype_policy.quantization_mode is None:
            policy_name = mode
            if mode == "int4":
                block_size = get_block_size_for_layer(self, config)
                policy_name = f"int4/{-1 if block_size is None else block_size}"
            self._dtype_policy = dtype_policies.get(f"{policy_name}_from_{self.dtype_policy.name}")
        self._cache.clear()

    def _drop_float_kernel(self):
        self._variables = [v for v in self._variables if v is not self._kernel]
        del self._kernel

    # ---- cached derived operands ------------------------------------------------
    def _cached(self, key, var, make):
        """Value derived from a variable, rebuilt when the variable is assigned."""
        hit = self._cache.get(key)
        # (the test of `cached_operand`, without a call: a decode-sized call looks up three or four operands)
        if hit is not None and hit[1] is var and hit[0] == var.version and (
                hit[3] is None or hit[3] == var._value._version):
            return hit[2]
        return cached_operand(self._cache, key, var, make)

    def _read_cached(self, key, var):
        hit = self._cache.get(key)
        if hit is not None and hit[1] is var and hit[0] == var.version and (
                hit[3] is None or hit[3] == var._value._version):
            return hit[2]
        cd = to_torch_dtype(self.compute_dtype)
        return self._cached(key, var, lambda t: t.to(cd).contiguous())

    def _strip_operands(self, rows, input_dim, units, grouped, block_size):
        """The operands of the strip-linear decode route (`ops.int4_matmul_strip`) when it takes
        `rows` bfloat16 rows of this layer, else None: the copy of the kernel it streams and, for
        grouped kernels, the re-ordered scales / zero points -- made on first use, kept while the
        variables they come from do not change."""
        if not (0 < rows <= kops.STRIP_MAX_ROWS and to_torch_dtype(self.compute_dtype) == torch.bfloat16
                and kops.int4_strip_supported(rows, input_dim, units, block_size if grouped else None)):
            return None
        spec = dict(units=units,
                    shadow=self._cached("w4s", self._kernel, lambda t: kops.int4_strip_copy(t, units)))
        if grouped:
            scale, zero = self.kernel_scale, self.kernel_zero
            spec["gparams"] = cached_params(self._cache, "w4s_params", scale, zero, lambda: kops.int4_strip_params(
                as_tensor(scale), as_tensor(zero), input_dim, units, block_size))
        else:
            spec["kernel_scale"] = self._read_cached("kernel_scale", self.kernel_scale)
        return spec

    def _strip_rows_operands(self, inputs, grouped, block_size):
        """The operands of `ops.int4_matmul_strip_rows` for these inputs."""
        units = self._orig_output_dim
        spec = dict(units=units, shadow=self._cached("w4s", self._kernel, lambda t: kops.int4_strip_copy(t, units)))
        if grouped:
            spec["gparams"] = strip_rows_params(self, inputs.dtype, inputs.shape[-1], units, block_size)
        else:
            spec["kernel_scale"] = self._read_cached("kernel_scale", self.kernel_scale)
        return spec

    def _tile_operand(self, input_dim):
        """The derived copy of the int8 kernel that the tile GEMM reads, as a keyword of
        `ops.int8_matmul`: the decode kernel's strip-linear copy where the tile kernel can take it
        (one derived copy per layer; same bits and speed as from a [N, K] copy), else the [N, K] copy."""
        if input_dim % 64 == 0:
            return dict(strip=self._cached("w8s", self._kernel, kops.int8_strip_copy))
        return dict(prepacked=self._cached("prepacked", self._kernel, kops.prepack_int8_kernel))

    # ---- quantized forward --------------------------------------------------------
    def _int8_call(self, inputs, training=None):
        """keras/src/layers/core/dense.py:938-986: quantise rows, int8 GEMM, de-scale, bias."""
        if self.lora_enabled:
            return self._quantized_call_with_lora(self._int8_call, inputs)
        if not self.inputs_quantizer:
            # weight-only: float activations against the int8 kernel, then the de-scale
            y = kops.int8_weight_only_matmul(
                inputs, as_tensor(self._kernel),
                self._read_cached("kernel_scale", self.kernel_scale),
                bias=self._call_bias(),
                prepacked=self._cached("prepacked", self._kernel, kops.prepack_int8_kernel),
            )
            if self.activation is not None:
                y = self.activation(y)
            return y
        lead = inputs.shape[:-1]
        x2 = inputs if inputs.dim() == 2 else inputs.reshape(-1, inputs.shape[-1])
        M, N = x2.shape[0], self.units
        exact = self.exact_epilogue
        if exact is None:
            exact = True
        alone = exact and quantizes_alone(self.inputs_quantizer)
        if exact and int8_strip_route(self.inputs_quantizer, x2, N):
            # decode sizes: quantizer, matmul and de-scale in one launch, from the strip-linear copy
            y = kops.int8_dense_strip(
                x2, self._cached("w8s", self._kernel, kops.int8_strip_copy), N,
                self._read_cached("kernel_scale", self.kernel_scale), bias=self._call_bias(),
                epsilon=self.inputs_quantizer.epsilon, value_range=self.inputs_quantizer.value_range,
                quantize=None if alone else lambda rows: quantize_rows(self.inputs_quantizer, rows))
            y = y if len(lead) == 1 else y.reshape(*lead, N)
            if self.activation is not None:
                y = self.activation(y)
            return y
        bias = self._call_bias()
        if alone and int8_rows_route(x2, to_torch_dtype(self.compute_dtype), N, bias):
            # more rows: quantizer and tile GEMM in one call
            y = kops.int8_dense_rows(
                x2, self._cached("w8s", self._kernel, kops.int8_strip_copy), N,
                self._read_cached("kernel_scale", self.kernel_scale), bias=bias, epsilon=self.inputs_quantizer.epsilon,
                value_range=self.inputs_quantizer.value_range)
        else:
            q, scale = quantize_rows(self.inputs_quantizer, x2)
            y = kops.int8_matmul(
                q, as_tensor(self._kernel), a_scale=scale,
                kernel_scale=self._read_cached("kernel_scale", self.kernel_scale),
                bias=bias,
                out_dtype=to_torch_dtype(self.compute_dtype),
                exact_epilogue=exact, **self._tile_operand(x2.shape[1]),
            )
        y = y if len(lead) == 1 else y.reshape(*lead, N)
        if self.activation is not None:
            y = self.activation(y)
        return y

    def _int4_call(self, inputs, training=None):
        """keras/src/layers/core/dense.py:988-1095, weight-only: the packed kernel is
        consumed in place (no unpack, no de-quantised copy)."""
        if self.lora_enabled:
            return self._quantized_call_with_lora(self._int4_call, inputs)
        block_size = getattr(self, "_int4_block_size", None)
        grouped = block_size is not None and block_size > 0
        # (a grouped kernel ignores an activation quantizer, as the reference's sub-channel branch
        # does: dense.py:1040-1084 never reads it)
        if self.inputs_quantizer and not grouped:
            # activation-quantized, per-channel (dense.py:1023-1031): int8 rows against the
            # nibbles unpacked to int8 in scratch, exact int32 accumulation, one de-scale
            lead = inputs.shape[:-1]
            x2 = inputs.reshape(-1, inputs.shape[-1])
            q, scale = quantize_rows(self.inputs_quantizer, x2)
            units = self._orig_output_dim
            operand = {}
            if x2.shape[1] % 128 == 0 and x2.shape[0] > kops.SKINNY_MAX_ROWS:
                # the tile GEMM reads a strip-linear int8 copy of the unpacked kernel, made once and kept
                # while the kernel does not change (one byte per weight beside the stored half byte: this
                # configuration, which the reference does not default to, holds 3x the stored bytes)
                # instead of unpacking the whole kernel into scratch on every call
                unpacked = None
                operand = dict(strip=self._cached(
                    "w8s_unpacked", self._kernel,
                    lambda t: kops.int8_strip_copy(quantizers.unpack_int4(t, units, axis=-1))))
            else:
                unpacked = quantizers.unpack_int4(as_tensor(self._kernel), units, axis=-1)
            y = kops.int8_matmul(
                q, unpacked, a_scale=scale,
                kernel_scale=self._read_cached("kernel_scale", self.kernel_scale),
                bias=self._call_bias(),
                out_dtype=to_torch_dtype(self.compute_dtype), exact_epilogue=True, kernel_shape=(x2.shape[1], units),
                **operand,
            )
            y = y.reshape(*lead, self._orig_output_dim)
            if self.activation is not None:
                y = self.activation(y)
            return y
        if grouped:
            require_default_g_idx(self, block_size)
        rows = inputs.numel() // inputs.shape[-1] if inputs.shape[-1] else 0
        strip = (self._strip_operands(rows, inputs.shape[-1], self._orig_output_dim, grouped, block_size)
                 if inputs.dtype == torch.bfloat16 else None)
        if strip is not None:
            # decode sizes: the strip-linear copy of the kernel, streamed once, all of K inside a
            # workgroup (one launch, no scratch)
            bias = self._call_bias()
            per_row = bias is not None and rows > 1 and bias.numel() == rows * self._orig_output_dim
            y = kops.int4_matmul_strip(
                inputs, strip["shadow"], self._orig_output_dim, kernel_scale=strip.get("kernel_scale"),
                gparams=strip.get("gparams"), block_size=block_size if grouped else None,
                bias=None if per_row else bias, addend=bias if per_row else None)
        elif int4_strip_rows_route(inputs.dtype, rows, inputs.shape[-1], self._orig_output_dim,
                                   block_size if grouped else None):
            y = kops.int4_matmul_strip_rows(inputs, block_size=block_size if grouped else None, bias=self._call_bias(),
                                            **self._strip_rows_operands(inputs, grouped, block_size))
        elif (inputs.dtype == torch.bfloat16 and kmajor_rows(rows, self._orig_output_dim, inputs.shape[-1])
                and kops.int4_kmajor_supported(rows, inputs.shape[-1], self._orig_output_dim,
                                               block_size if grouped else None)):
            # a few dozen to a hundred-odd rows: from the K-contiguous copy of the kernel (made
            # on first use, kept while the kernel does not change), read once as int4
            units = self._orig_output_dim
            if kops.int4_tiles_strip_supported(rows, inputs.shape[-1], units, block_size if grouped else None):
                # ... from the SAME strip-linear copy the decode kernel streams: one derived copy per layer
                y = kops.int4_matmul_tiles_strip(
                    inputs, self._cached("w4s", self._kernel, lambda t: kops.int4_strip_copy(t, units)), units,
                    self._read_cached("kernel_scale", self.kernel_scale),
                    kernel_zero=as_tensor(self.kernel_zero) if grouped else None,
                    block_size=block_size if grouped else None, bias=self._call_bias())
            else:
                y = kops.int4_matmul_kmajor(
                    inputs, self._cached("kmajor", self._kernel, lambda t: kops.int4_kmajor_copy(t, units)),
                    self._read_cached("kernel_scale", self.kernel_scale),
                    kernel_zero=as_tensor(self.kernel_zero) if grouped else None,
                    block_size=block_size if grouped else None,
                    bias=self._call_bias(),
                )
        elif int4_tile_rows_route(inputs.dtype, rows, inputs.shape[-1], self._orig_output_dim,
                                  block_size if grouped else None):
            units = self._orig_output_dim
            y = kops.int4_matmul_tiles_rows(
                inputs, self._cached("w4s", self._kernel, lambda t: kops.int4_strip_copy(t, units)), units,
                block_size=block_size if grouped else None, bias=self._call_bias(),
                **tile_rows_operands(self, inputs.dtype, units, grouped))
        else:
            y = kops.int4_matmul(
                inputs, as_tensor(self._kernel),
                self._read_cached("kernel_scale", self.kernel_scale), self._orig_output_dim,
                kernel_zero=as_tensor(self.kernel_zero) if grouped else None,
                block_size=block_size if grouped else None,
                bias=self._call_bias(),
            )
        if self.activation is not None:
            y = self.activation(y)
        return y

    def _call_bias(self):
        """The bias of this call: the layer's own, or -- for a layer without one -- the rows
        that `call_add` lends for the duration of a call (one row: a bias; a row per row of the
        input: the int4 decode kernel's addend)."""
        if self.bias is None:
            return getattr(self, "_row_bias", None)
        return self._read_cached("bias", self.bias)

    def _row_bias_ok(self):
        return self.bias is None and self.activation is None

    def _rows_of(self, inputs):
        return inputs.numel() // inputs.shape[-1]

    def _int8_together_spec(self, inputs):
        """What `call_together` needs to run this layer's int8 forward in a launch shared with other
        layers (decode sizes, the strip-linear copy): rows, quantizer settings, operands, and the
        step from the [M, N] result to the layer's output.  None when the layer's forward is
        anything else."""
        if (not self.built or self.quantization_mode != "int8" or self.lora_enabled
                or self.exact_epilogue is False):
            return None
        x2 = inputs.reshape(-1, inputs.shape[-1])
        if not int8_strip_route(self.inputs_quantizer, x2, self.units, strict=True):
            return None
        bias = self._call_bias()
        if bias is not None and bias.numel() != self.units:
            return None
        lead = inputs.shape[:-1]

        def finish(y2):
            y = y2.reshape(*lead, self.units)
            return self.activation(y) if self.activation is not None else y

        q = self.inputs_quantizer
        return dict(x2=x2, settings=(float(q.epsilon), tuple(float(v) for v in q.value_range)), quantizer=q,
                    kernel=dict(shadow=self._cached("w8s", self._kernel, kops.int8_strip_copy), units=self.units,
                                kernel_scale=self._read_cached("kernel_scale", self.kernel_scale), bias=bias),
                    finish=finish)

    def _int4_together_spec(self, inputs):
        """What `call_together` needs to run this layer's weight-only int4 forward in a launch
        shared with other layers: the [M, K] rows, the kernel's operands and the step that
        turns the [M, N] result into the layer's output.  None when the layer's forward is
        anything else."""
        if (not self.built or self.quantization_mode != "int4" or self.inputs_quantizer
                or self.lora_enabled):
            return None
        block_size = getattr(self, "_int4_block_size", None)
        grouped = block_size is not None and block_size > 0
        if grouped:
            require_default_g_idx(self, block_size)
        lead = inputs.shape[:-1]

        def finish(y2):
            y = y2.reshape(*lead, self._orig_output_dim)
            return self.activation(y) if self.activation is not None else y

        x2 = inputs.reshape(-1, inputs.shape[-1])
        strip = (self._strip_operands(x2.shape[0], x2.shape[1], self._orig_output_dim, grouped, block_size)
                 if x2.dtype == torch.bfloat16 else None)
        rows = None
        if strip is not None:
            strip["bias"] = self._call_bias()
        elif x2.dtype == to_torch_dtype(self.compute_dtype) and int4_strip_rows_route(
                x2.dtype, x2.shape[0], x2.shape[1], self._orig_output_dim, block_size if grouped else None):
            # (`call_add` asks before the cast of its inputs: what it runs has the compute dtype)
            rows = dict(self._strip_rows_operands(x2, grouped, block_size), bias=self._call_bias())
        return dict(
            x2=x2, block_size=block_size if grouped else None, strip=strip, rows=rows,
            kernel=dict(kernel_packed=as_tensor(self._kernel),
                        kernel_scale=self._read_cached("kernel_scale", self.kernel_scale),
                        units=self._orig_output_dim,
                        kernel_zero=as_tensor(self.kernel_zero) if grouped else None,
                        bias=self._call_bias()),
            finish=finish)

    # ---- serialization ---------------------------------------------------------------
    @property
    def variable_serialization_spec(self):
        """Order of variables in a store, per mode (dense.py:486-541)."""
        return {
            None: ["kernel", "bias"],
            "int8": ["kernel", "bias", "kernel_scale"],
            "int4": ["kernel", "bias", "kernel_scale", "kernel_zero", "g_idx"],
        }

    def _get_kernel_with_merged_lora(self):
        """`(kernel, kernel_scale, kernel_zero)` as they are saved
        (keras/src/layers/core/dense.py:1301-1427): without LoRA the variables themselves; with
        it the kernel is de-quantised (int8: `cast(q, compute) / scale`; int4: unpack, then
        divide or `dequantize_with_sz_map`), `(alpha / rank) * a . b` is added in float, and the sum
        is quantised again the way `quantize()` does it (host numpy path), giving new scales
        (and zero points)."""
        mode = self.quantization_mode
        if mode is None:
            return self.kernel, None, None
        kernel_value = as_tensor(self._kernel)
        kernel_scale = as_tensor(self.kernel_scale)
        kernel_zero = as_tensor(self.kernel_zero) if hasattr(self, "kernel_zero") else None
        if not self.lora_enabled:
            return kernel_value, kernel_scale, kernel_zero
        cd = to_torch_dtype(self.compute_dtype)
        block_size = getattr(self, "_int4_block_size", None)
        grouped = block_size is not None and block_size != -1
        if mode == "int4":
            unpacked = quantizers.unpack_int4(kernel_value, self._orig_output_dim, axis=-1)
            if grouped:
                float_kernel = quantizers.dequantize_with_sz_map(
                    unpacked, kernel_scale, kernel_zero, as_tensor(self.g_idx), group_axis=0).to(cd)
            else:
                float_kernel = torch.divide(unpacked.to(cd), kernel_scale)
            quant_range = (-8, 7)
        elif mode == "int8":
            float_kernel = torch.divide(kernel_value.to(cd), kernel_scale)
            quant_range = (-127, 127)
        else:
            raise self._quantization_mode_error(mode)
        delta = (self.lora_alpha / self.lora_rank) * torch.matmul(
            as_tensor(self.lora_kernel_a), as_tensor(self.lora_kernel_b))
        merged = torch.add(float_kernel, delta)
        if mode == "int4" and grouped:
            requantized, kernel_scale, kernel_zero = quantizers.abs_max_quantize_grouped_with_zero_point(
                merged, block_size=block_size, to_numpy=True)
        else:
            requantized, kernel_scale = quantizers.abs_max_quantize(
                merged, axis=0, value_range=quant_range, dtype="int8", to_numpy=True)
            kernel_scale = torch.squeeze(kernel_scale, dim=0)
            kernel_zero = None
        if mode == "int4":
            kernel_value, _, _ = quantizers.pack_int4(requantized.to(self.device), axis=-1)
        else:
            kernel_value = requantized
        return kernel_value, kernel_scale, kernel_zero

    def save_own_variables(self, store):
        """Write variables under "0", "1", ... in spec order, skipping absent ones; a LoRA update
        is merged into what is written (dense.py:314-378)."""
        if not self.built:
            return
        mode = self.quantization_mode
        if mode not in self.variable_serialization_spec:
            raise self._quantization_mode_error(mode)
        kernel_value, merged_scale, merged_zero = self._get_kernel_with_merged_lora()
        idx = 0
        for name in self.variable_serialization_spec[mode]:
            if name == "kernel":
                value = kernel_value
            elif name == "bias" and self.bias is None:
                continue
            elif name == "kernel_zero" and mode == "int4":
                if merged_zero is None:
                    continue
                value = merged_zero
            elif name == "g_idx" and not hasattr(self, name):
                continue
            elif name == "kernel_scale" and mode in ("int4", "int8"):
                value = merged_scale
            else:
                value = getattr(self, name)
            store[str(idx)] = as_tensor(value)
            idx += 1

    def load_own_variables(self, store):
        if not self.built:
            return
        mode = self.quantization_mode
        if mode not in self.variable_serialization_spec:
            raise self._quantization_mode_error(mode)
        idx = 0
        for name in self.variable_serialization_spec[mode]:
            if name == "kernel":
                target = self._kernel
            elif name == "bias" and self.bias is None:
                continue
            elif name in ("kernel_zero", "g_idx") and not hasattr(self, name):
                continue
            else:
                target = getattr(self, name)
            target.assign(store[str(idx)])
            idx += 1
        if self.lora_enabled:
            # what was saved has the update merged in (dense.py:428-430)
            self.lora_kernel_a.assign(torch.zeros_like(as_tensor(self.lora_kernel_a)))
            self.lora_kernel_b.assign(torch.zeros_like(as_tensor(self.lora_kernel_b)))
        self._cache.clear()

    def get_config(self):
        config = {
            "name": self.name,
            "units": self.units,
            "activation": activation_name(self.activation),
            "use_bias": self.use_bias,
            "dtype": self.dtype_policy.name,
            "quantization_config": serialize_quantization_config(self.quantization_config),
        }
        if self.lora_rank:
            config["lora_rank"] = self.lora_rank
            config["lora_alpha"] = self.lora_alpha
        return config
