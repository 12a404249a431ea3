"""Layer plumbing shared by `Dense` and `EinsumDense`.

Only what the quantized forward needs of `keras.layers.Layer` is restated:
the dtype policy, the cast of inputs to the compute dtype, reading float
variables in the compute dtype (autocast), the `quantize()` argument checks and
the dispatch to `_int8_call` / `_int4_call`
(keras/src/layers/layer.py:243-261, :797-849, :874-1003, :1366-1458).
"""

import re

import numpy as np
import torch

from keras_amd import dtype_policies
from keras_amd.quantization_config import validate_and_resolve_config

_TORCH_DTYPES = {
    "float32": torch.float32,
    "bfloat16": torch.bfloat16,
    "float16": torch.float16,
    "int8": torch.int8,
    "uint8": torch.uint8,
    "int32": torch.int32,
}


def _snake_case(name):
    name = re.sub(r"\W+", "", name)
    name = re.sub("(.)([A-Z][a-z]+)", r"\1_\2", name)
    return re.sub("([a-z])([A-Z])", r"\1_\2", name).lower()


def to_torch_dtype(name):
    if isinstance(name, torch.dtype):
        return name
    return _TORCH_DTYPES[name]


def default_device():
    return torch.device("cuda", torch.cuda.current_device()) if torch.cuda.is_available() else torch.device("cpu")


class Variable:
    """A named tensor with `assign`, as far as the quantized layers use it."""

    def __init__(self, value, name, trainable=False):
        self.name = name
        self.trainable = trainable
        self._value = value
        self.version = 0  # bumped by assign(); caches derived from the value key on it

    @property
    def value(self):
        return self._value

    @property
    def shape(self):
        return tuple(self._value.shape)

    @property
    def dtype(self):
        return str(self._value.dtype).replace("torch.", "")

    @property
    def device(self):
        return self._value.device

    def assign(self, value):
        if isinstance(value, Variable):
            value = value.value
        if not isinstance(value, torch.Tensor):
            value = torch.as_tensor(np.asarray(value))
        if tuple(value.shape) != self.shape:
            raise ValueError(
                "The shape of the target variable and the shape of the target value in "
                f"`variable.assign(value)` must match. variable.shape={self.shape}, "
                f"Received: value.shape={tuple(value.shape)}. Target variable: {self.name}"
            )
        self._value = value.to(device=self._value.device, dtype=self._value.dtype).contiguous()
        self.version += 1

    def numpy(self):
        v = self._value.detach().cpu()
        return (v.float() if v.dtype == torch.bfloat16 else v).numpy()

    def __repr__(self):
        return f"<Variable {self.name} shape={self.shape} dtype={self.dtype}>"


def as_tensor(x):
    return x.value if isinstance(x, Variable) else x


def cached_operand(cache, key, var, make):
    """`make(value of var)`, kept in `cache` and rebuilt when the variable is assigned.  A rebuilt tensor keeps its
    address: a captured HIP graph that holds the old one's goes on reading live memory (the new values) instead of
    memory that was freed.  The rebuild writes into the tensor that is kept, so that one never shares storage with the
    variable's (a cast to the dtype it has already, a `contiguous()` of what lies so, return the variable's own
    tensor, and that may be the caller's): it is cloned, and follows writes into the variable's tensor, too."""
    if var is None:
        return None
    hit = cache.get(key)
    if (hit is not None and hit[1] is var and hit[0] == var.version
            and (hit[3] is None or hit[3] == var._value._version)):
        return hit[2]
    t = as_tensor(var)
    value = make(t)
    writes, shared = None, False
    if isinstance(value, torch.Tensor):
        if value.untyped_storage().data_ptr() == t.untyped_storage().data_ptr():
            writes = None if t.is_inference() else t._version  # (inference tensors do not count)
            shared = True
        if (hit is not None and isinstance(hit[2], torch.Tensor) and hit[2].shape == value.shape
                and hit[2].dtype == value.dtype and hit[2].device == value.device):
            hit[2].copy_(value.detach())
            value = hit[2]
        elif shared:
            value = value.detach().clone()
    cache[key] = (var.version, var, value, writes)
    return value


def cached_params(cache, key, first, second, make):
    """`make()`, a tensor packed from two variables, kept in `cache` and rebuilt in place (as `cached_operand`)
    when one of them is assigned."""
    stamp = (id(first), first.version, id(second), second.version)
    hit = cache.get(key)
    if hit is None or hit[0] != stamp:
        value = make()
        if (hit is not None and hit[2].shape == value.shape and hit[2].dtype == value.dtype
                and hit[2].device == value.device):
            hit[2].copy_(value)
            value = hit[2]
        hit = cache[key] = (stamp, None, value)
    return hit[2]


def require_default_g_idx(layer, block_size):
    """The grouped int4 kernels take the group of row k to be `k // block_size`; the reference
    looks it up in the `g_idx` variable (keras/src/quantizers/quantizers.py:1659-1668), which
    `quantize()` fills with exactly that (keras/src/layers/core/dense.py:868-889).  A stored
    `g_idx` holding any other map would silently compute something else here, so it is
    rejected: checked once per value of the variable (one small device-to-host read)."""
    var = getattr(layer, "g_idx", None)
    if var is None:
        return
    stamp = (id(var), var.version)
    if getattr(layer, "_g_idx_checked", None) == stamp:
        return
    g = as_tensor(var)
    want = torch.floor_divide(torch.arange(g.numel(), dtype=torch.float32, device=g.device),
                              float(block_size))
    if g.shape != want.shape or not bool(torch.equal(g.to(torch.float32), want)):
        raise ValueError(
            f"{type(layer).__name__} '{layer.name}': g_idx is not floor(arange(n) / {block_size}); "
            "group maps other than the one quantize() writes are not supported by the fused "
            "int4 kernels")
    layer._g_idx_checked = stamp


class Layer:
    def __init__(self, dtype=None, name=None, device=None):
        # default name: the snake-cased class name (keras/src/utils/naming.py; the reference
        # also appends a per-process counter to later instances)
        self.name = name or _snake_case(type(self).__name__)
        self._dtype_policy = dtype_policies.get(dtype)
        self.device = torch.device(device) if device is not None else default_device()
        self.built = False
        self._is_quantized = False
        self.quantization_config = None
        self._variables = []

    # ---- dtype policy ------------------------------------------------------
    @property
    def dtype_policy(self):
        return self._dtype_policy

    @dtype_policy.setter
    def dtype_policy(self, value):
        policy = dtype_policies.get(value)
        # keras/src/layers/layer.py:797-817: a quantized policy set on a built float layer
        # converts the layer
        if policy.quantization_mode is not None and self.built and not self._is_quantized:
            self.quantize(policy.quantization_mode, type_check=False)
        self._dtype_policy = policy

    @property
    def compute_dtype(self):
        return self._dtype_policy.compute_dtype

    @property
    def variable_dtype(self):
        return self._dtype_policy.variable_dtype

    @property
    def quantization_mode(self):
        return self._dtype_policy.quantization_mode

    # ---- variables ----------------------------------------------------------
    def add_weight(self, name, shape, dtype=None, initializer="zeros", trainable=False):
        tdtype = to_torch_dtype(dtype or self.variable_dtype)
        value = self.__dict__.get("_build_values", {}).get(name)
        if (isinstance(value, torch.Tensor) and tuple(value.shape) == tuple(shape) and value.dtype == tdtype
                and value.device == self.device and value.is_contiguous()):
            pass  # (what `assign` would make of it: the value itself)
        elif callable(initializer):
            value = initializer(tuple(shape), tdtype)
            if not isinstance(value, torch.Tensor):
                value = torch.as_tensor(np.asarray(value))
            value = value.to(device=self.device, dtype=tdtype)
        elif initializer == "ones":
            value = torch.ones(tuple(shape), dtype=tdtype, device=self.device)
        elif initializer == "zeros":
            value = torch.zeros(tuple(shape), dtype=tdtype, device=self.device)
        else:
            raise ValueError(f"Unknown initializer: {initializer}")
        var = Variable(value, name=f"{self.name}/{name}", trainable=trainable)
        self._variables.append(var)
        return var

    def _quantized_build_with(self, shape, mode, config, **values):
        """`quantized_build`, for a caller that assigns `values` (by the names of the weights) to the variables right
        after it.  A weight that can hold its value as it is takes it at once, and its initial zeros or ones are never
        written: of a 4096 x 14336 kernel that is 34 MB and three launches.  One that cannot (another shape, dtype or
        device) is made as ever and left to `assign`."""
        self._build_values = values
        try:
            self.quantized_build(shape, mode, config)
        finally:
            del self._build_values

    def read(self, var):
        """Value of a variable as `call` sees it: float variables are read in the compute
        dtype under a mixed policy (AutocastScope,
        keras/src/backend/common/variables.py:245-249, :677-708)."""
        if var is None:
            return None
        t = as_tensor(var)
        cd = to_torch_dtype(self.compute_dtype)
        if t.dtype.is_floating_point and t.dtype != cd:
            # the cast copy is kept while the variable holds the same value (assign() bumps the
            # variable's version, an in-place write the tensor's): a decode step reads the same
            # gains and scales thousands of times
            cache = self.__dict__.setdefault("_read_cache", {})
            stamp = (var.version, t.data_ptr(), t._version, cd)
            hit = cache.get(id(var))
            if hit is not None and hit[0] == stamp and hit[1] is var:
                return hit[2]
            value = t.to(cd)
            cache[id(var)] = (stamp, var, value)
            return value
        return t

    def resident_bytes(self):
        """Device memory this layer holds, split into what the reference's layer stores and what
        this build derives from it: `{"stored": bytes of the variables, "derived": bytes of the
        copies kept for the kernels (strip-linear / K-contiguous / prepacked kernels, cast
        scales)}`.  Storage shared by several tensors is counted once.  No counterpart in the
        reference."""
        seen, stored = set(), 0
        for var in getattr(self, "_variables", []):
            t = as_tensor(var)
            key = t.untyped_storage().data_ptr()
            if key not in seen:
                seen.add(key)
                stored += t.untyped_storage().nbytes()
        derived = 0

        def visit(value):
            nonlocal derived
            if isinstance(value, torch.Tensor):
                key = value.untyped_storage().data_ptr()
                if value.is_cuda and key not in seen:
                    seen.add(key)
                    derived += value.untyped_storage().nbytes()
            elif isinstance(value, (list, tuple)):
                for v in value:
                    visit(v)
            elif isinstance(value, dict):
                for v in value.values():
                    visit(v)

        visit(self.__dict__.get("_cache", {}))
        visit(self.__dict__.get("_read_cache", {}))
        return {"stored": stored, "derived": derived}

    # ---- config ---------------------------------------------------------------
    @classmethod
    def from_config(cls, config):
        """Layer from `get_config()` output (keras/src/layers/layer.py `from_config`; the
        quantization config travels as {"class_name", "config"})."""
        from keras_amd import quantization_config as qc

        config = dict(config)
        config.pop("trainable", None)
        spec = config.pop("quantization_config", None)
        if isinstance(config.get("dtype"), dict):  # a serialized policy object
            config["dtype"] = dtype_policies.get(config["dtype"]["config"].get("name")
                                                 or config["dtype"]["config"])
        if spec is not None:
            classes = {c.__name__: c for c in (qc.Int8QuantizationConfig, qc.Int4QuantizationConfig)}
            if spec["class_name"] not in classes:
                raise ValueError(f"Unknown quantization config class: {spec['class_name']}")
            config["quantization_config"] = classes[spec["class_name"]].from_config(spec["config"])
        return cls(**config)

    # ---- stores ---------------------------------------------------------------
    def save_own_variables(self, store):
        """Every variable under "0", "1", ... in creation order
        (keras/src/layers/layer.py:1478-1489); quantized layers override the order."""
        for i, v in enumerate(self._variables):
            store[str(i)] = v.value

    def load_own_variables(self, store):
        if len(store.keys()) != len(self._variables):
            raise ValueError(
                f"Layer '{self.name}' expected {len(self._variables)} variables, but received "
                f"{len(store.keys())} variables during loading. "
                f"Expected: {[v.name for v in self._variables]}"
            )
        for i, v in enumerate(self._variables):
            v.assign(store[str(i)])

    # ---- call ---------------------------------------------------------------
    def __call__(self, inputs, training=None):
        if not isinstance(inputs, torch.Tensor):
            inputs = torch.as_tensor(np.asarray(inputs))
        if not self.built:
            self.build(tuple(inputs.shape))
        if inputs.device != self.device:
            inputs = inputs.to(self.device)
        cd = to_torch_dtype(self.compute_dtype)
        if inputs.dtype.is_floating_point and inputs.dtype != cd:
            inputs = inputs.to(cd)
        if self.quantization_mode is not None:
            return self.quantized_call(inputs, training=training)
        return self.call(inputs, training=training)

    def quantized_call(self, *args, **kwargs):
        mode = self.quantization_mode
        if mode == "int8":
            return self._int8_call(*args, **kwargs)
        if mode == "int4":
            return self._int4_call(*args, **kwargs)
        raise self._quantization_mode_error(mode)

    def _int8_call(self, *args, **kwargs):
        raise self._not_implemented_error(self._int8_call)

    def _int4_call(self, *args, **kwargs):
        raise self._not_implemented_error(self._int4_call)

    # ---- quantize -----------------------------------------------------------
    def quantize(self, mode=None, config=None, **kwargs):
        """Argument checks of `quantize_wrapper`, then the layer's own conversion."""
        config = validate_and_resolve_config(mode, config)
        mode = config.mode
        self._check_quantize_args(mode, self.compute_dtype)
        return self._quantize(mode=mode, config=config, **kwargs)

    def _quantize(self, mode, config, type_check=True):
        raise self._not_implemented_error(self.quantize)

    def _check_quantize_args(self, mode, compute_dtype):
        if not self.built:
            raise ValueError(
                "Cannot quantize a layer that isn't yet built. "
                f"Layer '{self.name}' (of type '{self.__class__.__name__}') "
                "is not built yet."
            )
        if getattr(self, "_is_quantized", False):
            raise ValueError(
                f"Layer '{self.name}' is already quantized with "
                f"dtype_policy='{self.dtype_policy.name}'. "
                f"Received: mode={mode}"
            )
        if mode not in dtype_policies.QUANTIZATION_MODES:
            raise ValueError(
                "Invalid quantization mode. "
                f"Expected one of {dtype_policies.QUANTIZATION_MODES}. "
                f"Received: mode={mode}"
            )
        if mode == "int8" and compute_dtype == "float16":
            raise ValueError(
                f"Quantization mode='{mode}' doesn't work well with "
                "compute_dtype='float16'. Consider loading model/layer with "
                "another dtype policy such as 'mixed_bfloat16' or "
                "'mixed_float16' before calling `quantize()`."
            )

    def _not_implemented_error(self, attr, msg=None):
        if callable(attr):
            attr_name, attr_type = attr.__name__, "method"
        else:
            attr_name, attr_type = str(attr), "attribute"
        msg = f" {msg}" if msg is not None else ""
        return NotImplementedError(
            f"Layer {self.__class__.__name__} does not have a `{attr_name}` "
            f"{attr_type} implemented.{msg}"
        )

    def _quantization_mode_error(self, mode):
        return NotImplementedError(
            "Invalid quantization mode. Expected one of "
            f"{dtype_policies.QUANTIZATION_MODES}. "
            f"Received: quantization_mode={mode}"
        )
