"""The work that programs built on this framework have it do, as cases that can be timed and whose outputs can be compared.

A case is a dict of plain values. Its "kind" names the entry point a user's program calls:

  network     tiny_dpcpp_nn.Network: `with torch.no_grad(): net(x)` (op "infer") or `net(x)` and `.backward(dy)` (op "train")
  field       tiny_dpcpp_nn.NetworkWithInputEncoding, a hash grid in front of a network: the same two ops on positions
  encoding    tiny_dpcpp_nn.Encoding, a hash grid on its own: the same two ops
  step        one optimisation step of a network through the C ABI (tnn_mlp_train_step_l2_adam)
  field_step  one optimisation step of a hash grid and its network through the C ABI (tnn_grid_order_points,
              tnn_grid_mlp_train_step_l2_adam, tnn_adam_step on the table)

Outputs, gradients and updated optimiser state come back whole.
"""
import ctypes
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "tiny-dpcpp-nn_amd"))
import tiny_dpcpp_nn as tnn  # noqa: E402
from tiny_dpcpp_nn import _lib  # noqa: E402

DEVICE = "cuda"
TORCH_DTYPE = {"bf16": torch.bfloat16, "fp16": torch.float16}
ABI_DTYPE = {"bf16": _lib.TNN_BF16, "fp16": _lib.TNN_FP16}
ADAM = dict(lr=1e-3, beta1=0.9, beta2=0.99, eps=1e-15)


# ---- the cases -----------------------------------------------------------------------------------------------------------

def _network(op, width, hidden, dtype, n_in, n_out, batch, given="same", dx=False, output_activation="None"):
    return {"kind": "network", "op": op, "width": width, "hidden": hidden, "dtype": dtype, "n_in": n_in, "n_out": n_out, "batch": batch,
            "given": given, "dx": dx, "output_activation": output_activation}


def _grid(dims, log2, scale, levels=16, features=2, base=16, interpolation="Linear"):
    return {"dims": dims, "log2": log2, "scale": scale, "levels": levels, "features": features, "base": base, "interpolation": interpolation}


def _field(op, grid, width, hidden, dtype, n_out, batch, points="uniform"):
    return {"kind": "field", "op": op, "width": width, "hidden": hidden, "dtype": dtype, "n_out": n_out, "batch": batch, "points": points, **grid}


def _encoding(op, grid, batch):
    return {"kind": "encoding", "op": op, "batch": batch, **grid}


def _step(width, hidden, dtype, batch, dx=False):
    return {"kind": "step", "width": width, "hidden": hidden, "dtype": dtype, "batch": batch, "dx": dx}


def _field_step(grid, hidden, dtype, batch):
    return {"kind": "field_step", "width": 64, "hidden": hidden, "dtype": dtype, "batch": batch, **grid}


def listed():
    return [
        # a control loop or an interactive viewer asks for a few rows at a time, in float32, and waits for the answer
        dict(_network("infer", 64, 4, "bf16", 32, 16, 100, given="float32"), name="network_infer_100"),
        # bulk evaluation of the same kind of network, full width in and out
        dict(_network("infer", 64, 4, "bf16", 64, 64, 2 ** 20), name="network_infer_w64_1m"),
        # bulk evaluation of the deepest network of the configurations, a batch that is no round number
        dict(_network("infer", 128, 8, "fp16", 128, 128, 200_003), name="network_infer_w128_200k"),
        # a small network on raw coordinates trained on small ragged batches, in the package's default type
        dict(_network("train", 32, 4, "fp16", 3, 3, 5001, given="float32"), name="network_train_w32_5k"),
        # the reference's headline network in a PyTorch training loop
        dict(_network("train", 64, 4, "bf16", 64, 64, 2 ** 18), name="network_train_w64_256k"),
        # a deep network behind another differentiable module, which wants dL/dx
        dict(_network("train", 128, 8, "fp16", 128, 128, 2 ** 17, dx=True), name="network_train_w128_128k"),
        # the sample: a 2-D hash grid and a network learn an image
        dict(_field("train", _grid(2, 15, 1.5), 64, 2, "bf16", 3, 2 ** 16), name="field_train_image_64k"),
        # the same with a large table and a large batch, in the package's default type
        dict(_field("train", _grid(2, 19, 1.5), 64, 2, "fp16", 3, 2 ** 18), name="field_train_image_256k"),
        # a 3-D neural field evaluated at scattered points
        dict(_field("infer", _grid(3, 22, 1.447), 64, 3, "fp16", 16, 2 ** 21), name="field_infer_3d_2m"),
        # the encoding benchmark: a 3-D grid on its own, forward and backward, in front of a user's own model
        dict(_encoding("train", _grid(3, 19, 1.447, interpolation="Smoothstep"), 2 ** 20), name="encoding_train_3d_1m"),
        # the headline optimisation step, for native programs
        dict(_step(64, 4, "bf16", 2 ** 18), name="step_w64_256k"),
        # image regression as one optimisation step with a half-precision table, for native programs
        dict(_field_step(_grid(2, 19, 1.5), 2, "fp16", 2 ** 18), name="field_step_image_256k"),
    ]


def _between(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _rows_of_8(rng, lo, hi):
    return 8 * _between(rng, lo // 8, hi // 8)


def draw(rng):
    kind = rng.choice(["network infer", "network train", "network train", "field infer", "field train", "encoding", "step", "field step"])
    dtype = rng.choice(["bf16", "fp16"])
    width, hidden = rng.choice([(16, 2), (32, 4), (64, 2), (64, 3), (64, 4), (128, 4), (128, 8)])
    if kind.startswith("network"):
        op = kind.split()[1]
        n_in = rng.choice([width, rng.randint(2, width)])
        n_out = rng.choice([width, rng.randint(1, width)])
        most = 2 ** 20 if width < 128 else 2 ** 18
        return _network(op, width, hidden, dtype, n_in, n_out, _between(rng, 1, most if op == "infer" else most // 2), given=rng.choice(["same", "float32"]),
                        dx=op == "train" and rng.random() < 0.5, output_activation=rng.choice(["None", "None", "Sigmoid"]))
    if kind == "step":
        return _step(width, hidden, dtype, _rows_of_8(rng, 256, 2 ** 20 if width < 128 else 2 ** 18), dx=rng.random() < 0.25)
    dims = rng.choice([2, 3])
    grid = _grid(dims, rng.randint(14, 22 if kind == "field infer" else 19), rng.choice([1.3, 1.447, 1.5, 2.0]), levels=rng.choice([8, 12, 16]),
                 interpolation=rng.choice(["Linear", "Linear", "Smoothstep"]))
    if kind == "field step":
        return _field_step(grid, rng.randint(1, 4), dtype, _rows_of_8(rng, 2 ** 10, 2 ** 18))
    if kind == "encoding":
        grid["features"] = rng.choice([2, 2, 4])
        return _encoding(rng.choice(["infer", "train"]), grid, _between(rng, 100, 2 ** 20))
    op = kind.split()[1]
    return _field(op, grid, 64, rng.randint(1, 4), dtype, rng.randint(1, 16), _between(rng, 100, 2 ** 21 if op == "infer" else 2 ** 18),
                  points=rng.choice(["uniform", "raster"]) if op == "infer" else "uniform")


# ---- what a program has in hand before the call ---------------------------------------------------------------------------

def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _uniform(gen, shape, lo, hi):
    return torch.rand(shape, generator=gen, device=DEVICE).mul_(hi - lo).add_(lo)


def _normal(gen, shape, sigma):
    return torch.randn(shape, generator=gen, device=DEVICE).mul_(sigma)


def _network_config(case):
    return {"otype": "FullyFusedMLP", "activation": "ReLU", "output_activation": case.get("output_activation", "None"), "n_neurons": case["width"],
            "n_hidden_layers": case["hidden"]}


def _encoding_config(case):
    return {"otype": "HashGrid", "type": "Hash", "n_levels": case["levels"], "n_features_per_level": case["features"], "log2_hashmap_size": case["log2"],
            "base_resolution": case["base"], "per_level_scale": case["scale"], "interpolation": case["interpolation"]}


def _positions(case, gen):
    """Positions in the unit square or cube: scattered, as a training batch or a volume renderer's samples are, or the rows of
    a picture (a slice of the volume in 3-D), as a viewer asks for them."""
    n, dims = case["batch"], case["dims"]
    if case.get("points", "uniform") == "uniform":
        return _uniform(gen, (n, dims), 0.0, 1.0)
    across = max(1, math.isqrt(n))
    i = torch.arange(n, device=DEVICE)
    corner = torch.rand(dims, generator=gen, device=DEVICE)
    xy = torch.stack([(i % across) / across, (i // across) / (n // across + 1)], dim=1)
    return torch.cat([(xy + corner[:2]) % 1.0, corner[2:].expand(n, dims - 2)], dim=1).contiguous()


def _gradient(case, gen, shape):
    """dL/dy as a scaled loss gives it: clear of fp16's smallest values."""
    return _normal(gen, shape, 1e-3)


def _weights(case, gen):
    """Unpacked Xavier-uniform matrices of a width x width network, flat."""
    bound = math.sqrt(6.0 / (2 * case["width"]))
    return _uniform(gen, ((case["hidden"] + 1) * case["width"] ** 2,), -bound, bound)


def _prepare_network(case, gen, seed):
    tnn.manual_seed(seed)
    dtype = TORCH_DTYPE[case["dtype"]]
    net = tnn.Network(case["n_in"], case["n_out"], _network_config(case), dtype=dtype)
    x = _uniform(gen, (case["batch"], case["n_in"]), -1.0, 1.0)
    x = x if case["given"] == "float32" else x.to(dtype)
    if case["op"] == "infer":
        net.eval()
        return {"model": net, "x": x}
    dy = _gradient(case, gen, (case["batch"], case["n_out"])).to(dtype)
    return {"model": net, "x": x.requires_grad_(case["dx"]), "dy": dy}


def _prepare_field(case, gen, seed):
    tnn.manual_seed(seed)
    dtype = TORCH_DTYPE[case["dtype"]]
    model = tnn.NetworkWithInputEncoding(case["dims"], case["n_out"], _network_config(case), _encoding_config(case), dtype=dtype, use_bias=False)
    with torch.no_grad():  # a table that has been trained for a while; a fresh one holds values within 1e-4
        model.encoding.params.copy_(_normal(gen, model.encoding.params.shape, 0.1))
    state = {"model": model, "x": _positions(case, gen)}
    if case["op"] == "infer":
        model.eval()
    else:
        state["dy"] = _gradient(case, gen, (case["batch"], case["n_out"])).to(dtype)
    return state


def _prepare_encoding(case, gen, seed):
    enc = tnn.Encoding(case["dims"], _encoding_config(case))
    with torch.no_grad():
        enc.params.copy_(_normal(gen, enc.params.shape, 0.1))
    state = {"model": enc, "x": _positions(case, gen)}
    if case["op"] == "train":
        state["dy"] = _normal(gen, (case["batch"], enc.n_output_dims), 1e-3)
    return state


def _p(t):
    return ctypes.c_void_p(t.data_ptr()) if t is not None else None


def _prepare_optimiser(case, gen, seed):
    """Weights, their operand copies and Adam's state after some hundred steps, as a native program holds them on the device."""
    lib, dtype = _lib.load(), TORCH_DTYPE[case["dtype"]]
    desc = _lib.MlpDesc(ABI_DTYPE[case["dtype"]], case["width"], case["hidden"], _lib.ACT_RELU, _lib.ACT_NONE)
    master = _weights(case, gen)
    size = lib.tnn_mlp_prepared_bytes(ctypes.byref(desc)) // 2
    s = {"lib": lib, "desc": desc, "step": 200, "loss_scale": 1.0 if case["dtype"] == "bf16" else 1024.0, "master": master,
         "m": _normal(gen, master.shape, 1e-4), "v": _uniform(gen, master.shape, 1e-9, 1e-8), "packed": torch.empty_like(master, dtype=dtype),
         "fwd": torch.empty(size, dtype=dtype, device=DEVICE), "bwd": torch.empty(size, dtype=dtype, device=DEVICE),
         "loss": torch.zeros(1, device=DEVICE)}
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    _lib.check(lib.tnn_mlp_prepare_weights(ctypes.byref(desc), _p(master), 1, _p(s["fwd"]), _p(s["bwd"]), stream))
    s["stream"] = stream
    s["targets"] = _uniform(gen, (case["batch"], case["width"]), 0.0, 1.0)
    return s


def _prepare_step(case, gen, seed):
    s = _prepare_optimiser(case, gen, seed)
    n = case["batch"]
    s["x"] = _uniform(gen, (n, case["width"]), -1.0, 1.0).to(TORCH_DTYPE[case["dtype"]])
    s["dx"] = torch.empty_like(s["x"]) if case["dx"] else None
    size = s["lib"].tnn_mlp_train_step_workspace_bytes(ctypes.byref(s["desc"]), n)
    s["workspace"] = torch.empty(size, dtype=torch.uint8, device=DEVICE)
    s["before"] = (ctypes.byref(s["desc"]), _p(s["fwd"]), _p(s["bwd"]), _p(s["x"]), _p(s["targets"]), s["loss_scale"], None, _p(s["loss"]), _p(s["master"]),
                   _p(s["m"]), _p(s["v"]))
    s["after"] = (ADAM["lr"], ADAM["beta1"], ADAM["beta2"], ADAM["eps"], _p(s["packed"]), _p(s["dx"]), n, _p(s["workspace"]), size, None, s["stream"])
    return s


def _prepare_field_step(case, gen, seed):
    s = _prepare_optimiser(case, gen, seed)
    lib, n = s["lib"], case["batch"]
    grid = _lib.GridDesc()
    interpolation = {"Linear": 1, "Smoothstep": 2}[case["interpolation"]]
    _lib.check(lib.tnn_grid_desc_init(ctypes.byref(grid), case["dims"], case["levels"], case["features"], case["log2"], case["base"], case["scale"],
                                      0, 1, interpolation, _lib.TNN_FP16))
    n_params = lib.tnn_grid_n_params(ctypes.byref(grid))
    s["grid"], s["n_params"] = grid, n_params
    s["x"] = _positions(case, gen)
    s["table_master"] = _normal(gen, (n_params,), 0.1)
    s["table"] = s["table_master"].to(torch.float16)
    s["table_m"], s["table_v"] = _normal(gen, (n_params,), 1e-6), _uniform(gen, (n_params,), 1e-13, 1e-12)
    s["table_grad"] = torch.empty(n_params, device=DEVICE)
    order_bytes = lib.tnn_grid_order_bytes(ctypes.byref(grid), n)
    s["order"] = torch.empty(order_bytes, dtype=torch.uint8, device=DEVICE)
    size = lib.tnn_grid_mlp_train_step_workspace_bytes(ctypes.byref(grid), ctypes.byref(s["desc"]), n)
    assert size > 0
    s["workspace"] = torch.empty(size, dtype=torch.uint8, device=DEVICE)
    s["ordering"] = (ctypes.byref(grid), _p(s["x"]), n, _p(s["order"]), order_bytes, s["stream"])
    s["before"] = (ctypes.byref(grid), ctypes.byref(s["desc"]), None, _p(s["order"]), _p(s["table"]), _p(s["fwd"]), _p(s["bwd"]), _p(s["targets"]),
                   s["loss_scale"], None, _p(s["loss"]), _p(s["master"]), _p(s["m"]), _p(s["v"]))
    s["after"] = (ADAM["lr"], ADAM["beta1"], ADAM["beta2"], ADAM["eps"], _p(s["packed"]), _p(s["table_grad"]), 1, n, _p(s["workspace"]), size, s["stream"])
    s["table_before"] = (_p(s["table_master"]), _p(s["table_m"]), _p(s["table_v"]), _p(s["table_grad"]), _lib.TNN_FP32, 1.0 / s["loss_scale"], n_params)
    s["table_after"] = (ADAM["lr"], ADAM["beta1"], ADAM["beta2"], ADAM["eps"], _p(s["table"]), _lib.TNN_FP16, s["stream"])
    return s


_PREPARE = {"network": _prepare_network, "field": _prepare_field, "encoding": _prepare_encoding, "step": _prepare_step, "field_step": _prepare_field_step}


def prepare(case, seed):
    state = _PREPARE[case["kind"]](case, _generator(seed), seed)
    state["kind"], state["op"] = case["kind"], case.get("op", "train")
    return state


# ---- one pass ---------------------------------------------------------------------------------------------------------------

def _infer(s):
    with torch.no_grad():
        return s["model"](s["x"])


def _train(s):
    model, x = s["model"], s["x"]
    x.grad = None
    for p in model.parameters():
        p.grad = None
    y = model(x)
    y.backward(s["dy"])
    out = {"y": y.detach(), "dx": x.grad}
    out.update(("d" + name, p.grad) for name, p in model.named_parameters())
    return out


def _optimise_network(s):
    s["step"] += 1
    _lib.check(s["lib"].tnn_mlp_train_step_l2_adam(*s["before"], s["step"], *s["after"]))
    return {k: s[k] for k in ("loss", "master", "m", "v", "packed", "dx")}


def _optimise_field(s):
    lib = s["lib"]
    s["step"] += 1
    _lib.check(lib.tnn_grid_order_points(*s["ordering"]))
    _lib.check(lib.tnn_grid_mlp_train_step_l2_adam(*s["before"], s["step"], *s["after"]))
    _lib.check(lib.tnn_adam_step(*s["table_before"], s["step"], *s["table_after"]))
    return {k: s[k] for k in ("loss", "master", "m", "v", "packed", "table_grad", "table_master", "table_m", "table_v", "table")}


def run(state):
    kind = state["kind"]
    if kind == "step":
        return _optimise_network(state)
    if kind == "field_step":
        return _optimise_field(state)
    return _infer(state) if state["op"] == "infer" else _train(state)


# ---- what a pass cannot do without --------------------------------------------------------------------------------------------

def _level_entries(case):
    """Entries of each level of the grid's table."""
    for level in range(case["levels"]):
        resolution = math.ceil(case["base"] * case["scale"] ** level - 1) + 1
        yield min(-(-resolution ** case["dims"] // 8) * 8, 2 ** case["log2"])


def _network_flops(case, n_in, n_out):
    """Of a forward pass over the batch; a backward pass costs a product for each weight gradient and one for each delta."""
    w, hidden = case["width"], case["hidden"]
    first, rest = n_in * w, (hidden - 1) * w * w + w * n_out
    return 2 * case["batch"] * first, 2 * case["batch"] * rest


def work(case):
    n, kind = case["batch"], case["kind"]
    train = case.get("op", "train") == "train"
    size = flops = 0
    if kind in ("field", "encoding", "field_step"):
        entry = case["features"] * (2 if kind == "field_step" else 4)
        corners = n * 2 ** case["dims"]
        table = sum(case["features"] * e for e in _level_entries(case))
        touched = sum(min(e, corners) * entry for e in _level_entries(case))
        size += n * case["dims"] * 4 + touched  # positions and the table's entries
        flops += 2 * corners * case["levels"] * case["features"] * (2 if train else 1)
        if train:
            size += table * 4  # the table's gradient
        if kind == "encoding":
            size += n * case["levels"] * case["features"] * 4 * (2 if train else 1)
    if kind == "field_step":
        size += table * (6 * 4 + 2)  # the table's gradient, masters and moments read and written, the half-precision table written
    if kind != "encoding":
        n_in = case["n_in"] if kind == "network" else case["width"] if kind == "step" else case["levels"] * case["features"]
        n_out = case["n_out"] if "n_out" in case else case["width"]
        n_weights = (case["hidden"] + 1) * case["width"] ** 2
        first, rest = _network_flops(case, n_in, n_out)
        wants_dx = case.get("dx", False) or kind in ("field", "field_step")
        flops += (3 if train and wants_dx else 2 if train else 1) * first + (3 if train else 1) * rest
        size += n_weights * 4
        if kind in ("network", "step"):
            given = 4 if case.get("given") == "float32" else 2
            size += n * n_in * given * (2 if case["dx"] else 1)
        if kind in ("step", "field_step"):
            size += n * n_out * 4 + n_weights * (5 * 4 + 2)  # targets; masters, moments and the copy in the network's type
        else:
            size += n * n_out * 2 * (2 if train else 1) + (n_weights * 4 if train else 0)  # y, dL/dy, weight gradients
    return {"bytes": size, "flops": flops}


def tolerance(case):
    # a table's gradient is an fp32 sum over the batch in no fixed order; everything else is rounded to the network's type between
    # the layers and at the end (8 and 11 significant bits)
    if case["kind"] == "encoding":
        return {"rel": 2e-5}
    return {"rel": 1e-2 if case["dtype"] == "bf16" else 5e-3}
