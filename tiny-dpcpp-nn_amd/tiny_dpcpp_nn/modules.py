"""torch.nn.Module front end of the MI355X implementation: Network, Encoding, NetworkWithInputEncoding.

The public surface is the reference's (dpcpp_bindings/tiny_dpcpp_nn/modules.py: autograd function :65-136, Module base
:139-261, Network :264-307, Encoding :309-354, NetworkWithInputEncoding :357-421): the same class names, constructor
arguments and attributes (`params`, `tnn_module`, `n_input_dims`, `n_output_dims`, `width`, `n_hidden_layers`,
`loss_scale`, ...), the same padding rules (network input columns to the network width, filled with ones when `use_bias` and
zeros otherwise; any number of rows), the same loss scaling (128 for fp16, 1 for bf16) and the same
layout conventions (`params` of a network is the packed layout, `set_params(tensor)` takes unpacked matrices). The device
is PyTorch-ROCm's "cuda" where the reference has "xpu".

As in the reference (modules.py:253), every forward pushes `params` to the native module first, so that any way of
writing them is seen, `params.data[...] = ...` included. The push is part of the forward kernel, or one small kernel in front of it. A caller that only
ever updates `params` through operations PyTorch's version counter sees (optimizers, copy_(), load_state_dict) can switch
the push off for unchanged parameters with `module.push_params_every_forward = False`.

One difference in behaviour, a saving: a grid encoding and its network run as one kernel, in evaluation and in training.

All compute goes through the extension module `tiny_dpcpp_nn_pybind_module` (HIP kernels); importing this file fails if it
is not built. There is no PyTorch fallback.
"""
import torch

from .tiny_dpcpp_nn_pybind_module import Activation, create_encoding, create_network, set_initial_weight_seed

MIN_BATCH_SIZE = 8  # the kernels take batches that are multiples of 8 rows
DEFAULT_DEVICE = "cuda"

_ACTIVATIONS = {"relu": Activation.ReLU, "tanh": Activation.Tanh, "sigmoid": Activation.Sigmoid, "linear": Activation.Linear,
                "none": Activation.Linear}
_NETWORK_DTYPES = (torch.float16, torch.bfloat16)


def manual_seed(seed):
    """Networks created from now on get reproducible initial weights: seeds counted up from `seed`. Without this call every
    network is seeded from std::random_device, as in the reference (include/network/Network.h:262-263 there), and two runs of a
    program train different networks. No counterpart in the reference."""
    set_initial_weight_seed(int(seed) & (2 ** 64 - 1))


def free_temporary_memory():
    """Nothing to free: every workspace belongs to a module and goes with it. Kept because callers of the reference call it."""


def get_dpcpp_activation(name):
    try:
        return _ACTIVATIONS[name.lower()]
    except KeyError:
        raise NotImplementedError(f"Activation: {name} not defined") from None


def unpad_tensor_to_input_dim(padded_tensor, output_dim):
    if output_dim > padded_tensor.shape[1]:
        raise ValueError("input_dim must be less than or equal to the current width of the tensor")
    return padded_tensor[:, :output_dim]


def to_packed_layout_coord(idx, rows, cols):
    """Flat index of row-major element `idx` of a rows x cols matrix in the packed parameter layout, where the two rows of
    a pair are interleaved element by element."""
    row, col = divmod(idx, cols)
    return (row & ~1) * cols + 2 * col + (row & 1)


def from_packed_layout_coord(idx, rows, cols):
    """Inverse of to_packed_layout_coord."""
    pair, within = divmod(idx, 2 * cols)
    return (2 * pair + (within & 1)) * cols + within // 2


class _RecordedCall(torch.autograd.Function):
    """A module's call as torch.jit.trace can record it: one operator, which calls the module again when the trace is replayed."""

    @staticmethod
    def forward(ctx, owner, x, *params):
        recorder = torch._C._get_tracing_state()  # None when a trace is replayed
        torch._C._set_tracing_state(None)  # what the call consists of is not recorded
        try:
            with torch.set_grad_enabled(any(ctx.needs_input_grad)):
                x = x.detach().requires_grad_(ctx.needs_input_grad[1])
                y = owner.forward(x)
            ctx.inner = (x, *params), y
            shape, values = tuple(y.shape), y.data
        finally:
            torch._C._set_tracing_state(recorder)
        if recorder is None:
            return values
        result = torch.empty(shape, dtype=values.dtype, device=values.device)  # (a tensor the recorder knows)
        torch._C._set_tracing_state(None)
        result.copy_(values)
        torch._C._set_tracing_state(recorder)
        return result

    @staticmethod
    def backward(ctx, dy):
        inputs, y = ctx.inner
        wanted = [t for t, needed in zip(inputs, ctx.needs_input_grad[1:]) if needed]
        grads = iter(torch.autograd.grad(y, wanted, dy, retain_graph=True, allow_unused=True))
        return (None, *(next(grads) if needed else None for needed in ctx.needs_input_grad[1:]))


class Module(torch.nn.Module):
    """Base of the three front-end classes: owns the native module (`tnn_module`) and the PyTorch-side parameter tensor
    `params` (fp32 when `store_params_as_full_precision`, else the module's dtype; a network's is in the packed layout)."""

    _is_network = False

    def __init__(self, dtype, device=DEFAULT_DEVICE, store_params_as_full_precision=True, use_bias=True, init_module=True):
        super().__init__()
        self.dtype = dtype
        self.device = device
        self.use_bias = use_bias
        self.store_params_as_full_precision = store_params_as_full_precision
        self.loss_scale = 128.0 if dtype == torch.float16 else 1.0
        # True (the reference's behaviour): every forward pushes `params` first. False: only when the tensor's identity, storage
        # address or version counter changed since the last push -- a write through `.data` changes none of them and then
        # needs an explicit set_params().
        self.push_params_every_forward = True
        self._pushed = None  # (tensor identity, storage address, version) of `params` when the native module last took it
        if not init_module:
            return
        self.tnn_module = self.create_module()
        if self.tnn_module.n_params() == 0:
            print("No params initialised, as n_params = 0. This is correct for Encodings (apart from grid encodings).")
            self.params = torch.nn.Parameter(torch.zeros(1, device=self.device), requires_grad=False)
            return
        held = torch.float32 if store_params_as_full_precision else dtype
        # PyTorch's own memory, not a view of the native module's arrays
        self.params = torch.nn.Parameter(self.tnn_module.initial_params().detach().clone().to(held), requires_grad=True)

    # ---- parameters ----------------------------------------------------------------------------------------------
    def _params_state(self):
        p = self.params
        return (id(p), p.data_ptr(), p._version)

    def _push(self, tensor, packed):
        t = tensor.detach()
        # a network on the GPU converts fp32 / fp16 / bf16 to its own type in the kernel that copies; everything else is cast here
        if not (self._is_network and t.is_cuda and t.dtype in (torch.float32,) + _NETWORK_DTYPES):
            t = t.to(self.dtype)
        self.tnn_module.set_params(t.contiguous(), packed)

    def set_params(self, params=None):
        """`params` given: a flat tensor of unpacked [in][out] matrices (network) or the table (encoding); it is pushed to the
        native module and `self.params` takes what the module then holds. `None`: push `self.params` as it is (a network's is
        already packed)."""
        if self.tnn_module.n_params() == 0:
            if params is not None:
                raise RuntimeError("Network has no parameters. Cannot set params")
            return
        if params is None:
            self._push(self.params, packed=self._is_network)
        else:
            assert isinstance(params, torch.Tensor), "Params is not a torch.Tensor"
            self._push(params, packed=False)
            with torch.no_grad():
                self.params.copy_(self.get_params().reshape(self.params.shape))
        self._pushed = self._params_state()

    def _must_push(self):
        """What the reference does in front of every forward (modules.py:253): set_params(). With push_params_every_forward
        switched off, only when `params` is known to have changed: in-place updates (optimizer steps, copy_, load_state_dict)
        raise the tensor's version and a replaced tensor has another identity or address; writes through `.data` do neither."""
        return self.push_params_every_forward or self._pushed != self._params_state()

    def _has_pushed(self):
        """Called once the pass has taken the parameters over: after one that raised, the next pushes again."""
        if not self.push_params_every_forward:
            self._pushed = self._params_state()

    def get_params(self):
        """The parameters as the native module holds them (a network's: packed layout)."""
        return self.tnn_module.get_params()

    # ---- evaluation ----------------------------------------------------------------------------------------------
    def forward(self, x):
        # one entry into the native module: push, padding and conversion, the pass, and its node in the autograd graph
        y = self.tnn_module.call(x, self.params, self._must_push(), self.training, self.loss_scale)
        if y is None:  # torch.jit.trace is recording
            return _RecordedCall.apply(self, x, self.params)
        self._has_pushed()
        return y


class Network(Module):
    _is_network = True
    name = "network"

    def __init__(self, n_input_dims, n_output_dims, network_config, store_params_as_full_precision=True, device=DEFAULT_DEVICE,
                 dtype=torch.float16, use_bias=True):
        assert dtype in _NETWORK_DTYPES, f"Only torch.float16 or torch.bfloat16 supported, got: {dtype}"
        self.n_input_dims = n_input_dims
        self.n_output_dims = n_output_dims
        self.network_config = network_config
        self.width = network_config["n_neurons"]
        self.n_hidden_layers = network_config["n_hidden_layers"]
        self.activation = get_dpcpp_activation(network_config["activation"])
        self.output_activation = get_dpcpp_activation(network_config["output_activation"])
        super().__init__(dtype=dtype, device=device, store_params_as_full_precision=store_params_as_full_precision, use_bias=use_bias)

    def create_module(self):
        return create_network(self.n_input_dims, self.n_output_dims, self.n_hidden_layers, self.activation, self.output_activation,
                              self.width, str(self.dtype), self.use_bias)


class Encoding(Module):
    name = "encoding"

    def __init__(self, n_input_dims, encoding_config, n_output_dims=None, device=DEFAULT_DEVICE, dtype=torch.float,
                 store_params_as_full_precision=True):
        assert dtype == torch.float, "Only torch.float is currently supported for encoding (the grid gradients are float atomics)"
        self.n_input_dims = n_input_dims
        self.encoding_config = encoding_config
        self.encoding_config.setdefault("n_dims_to_encode", n_input_dims)
        self.encoding_name = encoding_config["otype"]
        self.padded_output_dims = n_output_dims  # None: the encoding's own width
        super().__init__(dtype=dtype, device=device, store_params_as_full_precision=store_params_as_full_precision)
        self.n_output_dims = self.tnn_module.n_output_dims()  # known once the native module exists

    def create_module(self):
        return create_encoding(self.encoding_name, self.encoding_config, self.padded_output_dims)


class NetworkWithInputEncoding(Module):
    name = "network_with_encoding"

    def __init__(self, n_input_dims, n_output_dims, network_config, encoding_config, device=DEFAULT_DEVICE,
                 store_params_as_full_precision=True, dtype=torch.float16, use_bias=True):
        assert dtype in _NETWORK_DTYPES, (f"Only torch.float16 or torch.bfloat16 supported, got: {dtype}."
                                          " Note, that dtype here only refers to dtype of Network, the Encoding is always float.")
        super().__init__(dtype=dtype, init_module=False)
        self.n_input_dims = n_input_dims
        self.n_output_dims = n_output_dims
        self.network_config = network_config
        self.encoding_config = encoding_config
        self.width = network_config["n_neurons"]
        self.n_hidden_layers = network_config["n_hidden_layers"]
        self.activation = get_dpcpp_activation(network_config["activation"])
        self.output_activation = get_dpcpp_activation(network_config["output_activation"])
        # the encoding pads its rows to the network width itself, so the network never pads its input
        self.encoding = Encoding(n_input_dims, encoding_config, n_output_dims=self.width, device=device, dtype=torch.float,
                                 store_params_as_full_precision=store_params_as_full_precision)
        assert self.encoding.n_output_dims == self.width
        self.network = Network(self.width, n_output_dims, network_config, store_params_as_full_precision=store_params_as_full_precision,
                               device=device, dtype=dtype, use_bias=use_bias)
        self.network_with_encoding = torch.nn.Sequential(self.encoding, self.network)
        self._fused = None  # whether the pair runs as one call: (without autograd, with it)

    @property
    def params(self):
        return self.network.params  # the table is `self.encoding.params`

    def get_params(self):
        raise RuntimeError("Not implemented.")

    def set_params(self, params=None):
        self.network.set_params(params)

    def forward(self, x):
        network, encoding = self.network, self.encoding
        if self._fused is None:  # (fixed once the two native modules exist)
            self._fused = (network.tnn_module.can_fuse_encoding(encoding.tnn_module), network.tnn_module.can_train_with_encoding(encoding.tnn_module))
        if not self._fused[torch.is_grad_enabled()]:
            return self.network_with_encoding(x)
        # a grid encoding and its network as one call into the native module each way, with the values of the two
        # modules in turn, the reference's only route
        y = network.tnn_module.call_with_encoding(encoding.tnn_module, x, network.params, encoding.params, network._must_push(), encoding._must_push(),
                                                  network.loss_scale)
        if y is None:
            return _RecordedCall.apply(self, x, network.params, encoding.params) if torch.jit.is_tracing() else self.network_with_encoding(x)
        network._has_pushed()
        encoding._has_pushed()
        return y
