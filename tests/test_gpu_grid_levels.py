"""The grid encoding level by level (tnn_grid_forward_by_level, and tnn_grid_forward on small batches): the rows of the kernel that walks all
levels of a point, bit for bit, which is checked against the oracle elsewhere (tests/test_gpu_grid.py, here through the larger batch)."""
import ctypes

import numpy as np
import pytest
import torch

from gpu_harness import BF16, FP16, FP32, ptr
from tiny_dpcpp_nn import _lib

pytestmark = pytest.mark.gpu
DIRECT = 2 ** 14  # the most points whose rows tnn_grid_forward writes level by level
TORCH = {FP32: torch.float32, BF16: torch.bfloat16, FP16: torch.float16}
BASE = dict(n_dims=3, n_levels=16, n_features_per_level=2, log2_hashmap_size=15, base_resolution=16, per_level_scale=1.447)


def bits(t):
    return t.contiguous().view(torch.int32 if t.element_size() == 4 else torch.int16)


def by_level(tnn, d, x, order, table, width, out_dtype):
    M = x.shape[0]
    need = (d.n_levels * d.n_features_per_level + 15) // 16 * 16 * TORCH[out_dtype].itemsize * ((M + 63) // 64 * 64) + 256
    work = torch.empty(need, dtype=torch.uint8, device=tnn.dev)
    out = torch.full((M, width), 7.0, dtype=TORCH[out_dtype], device=tnn.dev)
    args = (ctypes.byref(d), ptr(x) if order is None else None, ptr(order) if order is not None else None, ptr(table), ptr(out), out_dtype, width, M, ptr(work))
    assert tnn.lib.tnn_grid_forward_by_level(*args, need - 300, tnn.stream()) == _lib.TNN_ERR_WORKSPACE
    _lib.check(tnn.lib.tnn_grid_forward_by_level(*args, need, tnn.stream()))
    return out


@pytest.mark.parametrize("cfg,param_dtype,out_dtype,width", [
    (BASE, FP32, FP32, 32), (BASE, FP16, FP16, 64), (BASE, FP32, BF16, 36), (dict(BASE, n_dims=2, per_level_scale=1.5), FP32, FP32, 33),
    (dict(BASE, n_dims=2, log2_hashmap_size=19, per_level_scale=1.5), FP16, BF16, 32), (dict(BASE, n_features_per_level=1), FP32, FP32, 17),
    (dict(BASE, n_features_per_level=4), FP32, FP32, 64), (dict(BASE, n_features_per_level=8, n_levels=3, n_dims=2), FP16, FP16, 24),
    (dict(BASE, n_features_per_level=8, n_levels=7), FP32, FP32, 60), (dict(BASE, n_levels=1), FP32, FP32, 2), (dict(BASE, n_levels=5, interpolation="Smoothstep"), FP32, FP32, 10),
    (dict(BASE, interpolation="Nearest"), FP32, FP32, 32), (dict(BASE, hash="Prime"), FP32, FP32, 32), (dict(BASE, hash="ReversedPrime", n_dims=2), FP16, FP16, 32),
    (dict(BASE, n_dims=2, n_features_per_level=1), FP32, FP32, 17), (dict(BASE, n_dims=2, n_features_per_level=1, interpolation="Smoothstep"), FP16, FP16, 16),
    (dict(BASE, n_dims=2, n_features_per_level=4), FP16, FP32, 64), (dict(BASE, n_dims=2, n_features_per_level=4, grid_type="Tiled"), FP16, BF16, 70),
    (dict(BASE, n_dims=2, n_features_per_level=4, n_levels=6), FP32, FP32, 24), (dict(BASE, n_dims=2, grid_type="Tiled", base_resolution=5), FP32, FP32, 32),
    (dict(BASE, n_dims=2, n_features_per_level=1, grid_type="Dense", n_levels=5), FP32, BF16, 5),
    (dict(BASE, hash="Rng"), FP32, FP32, 32), (dict(BASE, grid_type="Dense", n_levels=5), FP32, FP32, 12), (dict(BASE, grid_type="Tiled"), FP32, FP32, 32)])
def test_levels_are_the_rows_of_the_points(tnn, cfg, param_dtype, out_dtype, width):
    d = tnn.grid_desc(cfg, param_dtype)
    gen = torch.Generator(device=tnn.dev).manual_seed(5)
    table = (torch.rand(tnn.grid_n_params(d), device=tnn.dev, generator=gen) * 2 - 1).to(TORCH[param_dtype])
    M = DIRECT + 77
    x = torch.rand((M, cfg["n_dims"]), device=tnn.dev, generator=gen)
    x[:6] = torch.tensor([0.0, 1.0, -0.25, 1.75, float("nan"), 0.999999], device=tnn.dev)[:, None]
    expected = tnn.grid_forward(d, x, table, width, out_dtype)
    assert torch.equal(bits(by_level(tnn, d, x, None, table, width, out_dtype)), bits(expected))
    assert torch.equal(bits(by_level(tnn, d, x, tnn.grid_order(d, x), table, width, out_dtype)), bits(expected))
    for m in (1, 2, 63, 129, 4097, DIRECT):  # written directly, odd numbers of lanes among them
        part = x[:m].contiguous()
        assert torch.equal(bits(tnn.grid_forward(d, part, table, width, out_dtype)), bits(expected[:m]))
        assert torch.equal(bits(tnn.grid_forward_ordered(d, tnn.grid_order(d, part), table, width, m, out_dtype)), bits(expected[:m]))


@pytest.mark.parametrize("levels,features", [(1, 1), (4, 2), (5, 4), (16, 2)])
@pytest.mark.parametrize("padding", [1, 2, 3, 31, 32, 33, 63, 64, 65, 200])
def test_padding_of_small_batches(tnn, levels, features, padding):
    """The columns behind the encoding's: on both sides of each number of lanes that write a row's."""
    d = tnn.grid_desc(dict(BASE, n_dims=2, n_levels=levels, n_features_per_level=features))
    table = torch.rand(tnn.grid_n_params(d), device=tnn.dev)
    for M, dtype in ((1, FP32), (67, BF16), (DIRECT, FP32), (DIRECT - 1, FP16)):
        x = torch.rand((M, 2), device=tnn.dev)
        y = tnn.grid_forward(d, x, table, levels * features + padding, dtype)
        assert torch.equal(bits(y[:, :levels * features]), bits(tnn.grid_forward(d, x, table, levels * features, dtype))) and not bool(y[:, levels * features:].any())


def test_padding_costs_little(tnn):
    """128 columns for the 8 of four levels: measured 4 us for either; 36 for the 128 where the last level's threads wrote the others."""
    d, M = tnn.grid_desc(dict(BASE, n_dims=2, n_levels=4)), 5000
    table, x, y = torch.rand(tnn.grid_n_params(d), device=tnn.dev), torch.rand((M, 2), device=tnn.dev), torch.empty((M, 128), device=tnn.dev)

    def time(width):
        times = []
        for _ in range(9):
            ev = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
            ev[0].record()
            for _ in range(20):
                assert tnn.lib.tnn_grid_forward(ctypes.byref(d), ptr(x), ptr(table), ptr(y), FP32, width, M, tnn.stream()) == 0
            ev[1].record()
            ev[1].synchronize()
            times.append(ev[0].elapsed_time(ev[1]))
        return sorted(times)[3]

    time(8)
    assert time(128) <= 3 * time(8)


@pytest.mark.parametrize("features,param_dtype,out_dtype,M", [(1, FP32, FP32, 2 ** 19), (1, FP16, BF16, 2 ** 19 + 77), (4, FP32, FP16, 2 ** 19 + 1), (4, FP16, FP32, 2 ** 19 - 1),
                                                              (8, FP32, BF16, 2 ** 19 + 513), (8, FP16, FP16, 2 ** 19), (2, FP32, FP32, 2 ** 19 - 1)])
def test_large_batches_of_three_dimensions(tnn, features, param_dtype, out_dtype, M):
    """On both sides of the size from which a thread takes two points."""
    cfg = dict(BASE, n_levels=5, n_features_per_level=features, log2_hashmap_size=13, base_resolution=13, interpolation="Smoothstep")
    d = tnn.grid_desc(cfg, param_dtype)
    gen = torch.Generator(device=tnn.dev).manual_seed(12)
    table = (torch.rand(tnn.grid_n_params(d), device=tnn.dev, generator=gen) * 2 - 1).to(TORCH[param_dtype])
    x = torch.rand((M, 3), device=tnn.dev, generator=gen)
    width = 5 * features
    expected = bits(tnn.grid_forward(d, x, table, width, out_dtype))
    assert torch.equal(bits(by_level(tnn, d, x, None, table, width, out_dtype)), expected)
    assert torch.equal(bits(by_level(tnn, d, x, tnn.grid_order(d, x), table, width, out_dtype)), expected)


@pytest.mark.parametrize("dims,log2,features,levels,M", [
    (3, 22, 2, 16, 1), (3, 22, 2, 16, 300), (3, 22, 2, 12, 5001), (3, 22, 2, 16, 20000), (2, 22, 2, 16, 5001), (3, 21, 2, 16, 2 ** 18), (3, 21, 2, 16, 2 ** 18 - 1),
    (3, 20, 2, 16, 2 ** 19 + 77), (3, 20, 4, 9, 4097), (3, 16, 2, 16, 3 * 2 ** 18), (3, 19, 2, 16, 2 ** 20 + 511)])
def test_levels_that_all_xcds_share(tnn, dims, log2, features, levels, M):
    """All levels shared, none, and the large ones behind coarse ones that are not; batches of fewer chunks than XCDs, and that are no whole eighths."""
    d = tnn.grid_desc(dict(BASE, n_dims=dims, n_levels=levels, n_features_per_level=features, log2_hashmap_size=log2))
    gen = torch.Generator(device=tnn.dev).manual_seed(7)
    table = torch.rand(tnn.grid_n_params(d), device=tnn.dev, generator=gen) * 2 - 1
    x = torch.rand((M, dims), device=tnn.dev, generator=gen)
    width = levels * features
    x2 = torch.cat([x, torch.rand((DIRECT + 1, dims), device=tnn.dev)])[: max(M, DIRECT + 1)]  # (a batch beyond those that are written by levels)
    expected = bits(tnn.grid_forward(d, x2, table, width, FP32)[:M])
    assert torch.equal(bits(by_level(tnn, d, x, None, table, width, FP32)), expected)
    assert torch.equal(bits(by_level(tnn, d, x, tnn.grid_order(d, x), table, width, FP32)), expected)


@pytest.mark.parametrize("features,levels,log2,M", [(2, 16, 21, 2 ** 20 + 8), (1, 16, 22, 2 ** 20 + 1)])
def test_a_large_field_by_levels(tnn, features, levels, log2, M):
    """Beyond the size from which large levels pay in inference: the rows of the same points in batches that one kernel takes."""
    import tiny_dpcpp_nn
    tiny_dpcpp_nn.manual_seed(3)
    model = tiny_dpcpp_nn.NetworkWithInputEncoding(
        3, 3, {"otype": "FullyFusedMLP", "activation": "ReLU", "output_activation": "None", "n_neurons": 32, "n_hidden_layers": 2},
        {"otype": "HashGrid", "type": "Hash", "n_levels": levels, "n_features_per_level": features, "log2_hashmap_size": log2, "base_resolution": 16, "per_level_scale": 1.5},
        dtype=torch.float16, use_bias=False)
    d = tnn.grid_desc(dict(BASE, n_levels=levels, n_features_per_level=features, log2_hashmap_size=log2, per_level_scale=1.5))
    assert [tnn.lib.tnn_grid_mlp_width_wants_levels(ctypes.byref(d), 32, m) for m in (2 ** 20, M, 2 ** 19)] == [0, 1, 0]
    x = torch.rand((M, 3), device=tnn.dev)
    with torch.no_grad():
        model.encoding.params.copy_(torch.rand(model.encoding.params.shape, device=tnn.dev) - 0.5)
        y = model(x)
        for rows in (slice(0, 2 ** 19), slice(2 ** 19, 2 ** 20), slice(M - 100000, M)):
            assert torch.equal(bits(y[rows]), bits(model(x[rows].contiguous())))


@pytest.mark.parametrize("ordered", [False, True])
def test_a_batch_of_several_launches(tnn, ordered):
    """32 levels: a launch takes 65535 chunks of 512 points; a batch with more, its last chunk and last 64 points not full."""
    cfg = dict(BASE, n_levels=32, n_features_per_level=1, log2_hashmap_size=12, per_level_scale=1.2)
    d = tnn.grid_desc(cfg)
    gen = torch.Generator(device=tnn.dev).manual_seed(9)
    table = torch.rand(tnn.grid_n_params(d), device=tnn.dev, generator=gen)
    M = 65535 * 512 + 5 * 512 + 77
    x = torch.rand((M, 3), device=tnn.dev, generator=gen)
    got = by_level(tnn, d, x, tnn.grid_order(d, x) if ordered else None, table, 32, BF16)
    assert torch.equal(bits(got), bits(tnn.grid_forward(d, x, table, 32, BF16)))


@pytest.mark.parametrize("dims,log2,M,levels", [
    (3, 16, DIRECT, 16), (3, 16, DIRECT + 1, 16), (3, 19, 2 ** 19 + 3, 16), (2, 16, 2 ** 19 - 1, 16), (2, 16, 2 ** 19, 16), (3, 22, 2 ** 17 - 1, 16), (3, 22, 2 ** 17, 16),
    (3, 14, 2 ** 19 - 1, 16), (2, 19, 2 ** 18 - 1, 8), (2, 19, 2 ** 18, 8), (2, 14, 3 * 2 ** 17 - 1, 12), (2, 14, 3 * 2 ** 17, 12), (2, 22, 2 ** 15 - 1, 16), (2, 22, 2 ** 15, 16),
    (3, 14, 2 ** 16, 8), (3, 14, 2 ** 16 + 1, 8), (3, 17, 7 * 2 ** 16 - 1, 8), (3, 17, 7 * 2 ** 16, 8), (3, 19, 2 ** 18 - 1, 4), (3, 19, 2 ** 18, 4)])
def test_encoding_module_on_both_sides_of_each_rule(tnn, dims, log2, M, levels):
    """The Python encoding takes whichever route its size says; the C ABI in two calls of half the points, or by points, gives the same rows."""
    import tiny_dpcpp_nn
    cfg = dict(BASE, n_dims=dims, log2_hashmap_size=log2, n_levels=levels)
    enc = tiny_dpcpp_nn.Encoding(dims, {"otype": "HashGrid", "type": "Hash", "n_levels": levels, "n_features_per_level": 2, "log2_hashmap_size": log2, "base_resolution": 16,
                                        "per_level_scale": 1.447})
    gen = torch.Generator(device=tnn.dev).manual_seed(6)
    with torch.no_grad():
        enc.params.copy_(torch.rand(enc.params.shape, device=tnn.dev, generator=gen) - 0.5)
        x = torch.rand((M, dims), device=tnn.dev, generator=gen)
        y = enc(x)
    d = tnn.grid_desc(cfg)
    x2 = torch.cat([x, x[: DIRECT + 1]]) if M <= DIRECT else x  # (a batch beyond the small ones)
    assert torch.equal(bits(y), bits(tnn.grid_forward(d, x2, enc.params.detach().reshape(-1), 2 * levels, FP32)[:M]))


# (dimensions, levels, log2 of a level's entries, points, whether inference goes by levels, whether in cell order): both sides of each rule
FIELD_SIDES = [
    (2, 16, 19, 2 ** 13 - 1, 0, 0), (2, 16, 19, 2 ** 13, 1, 0), (2, 13, 19, 23999, 1, 0), (2, 13, 19, 24000, 0, 0), (2, 12, 19, 2 ** 13, 0, 0), (2, 16, 14, 2 ** 13, 0, 0),
    (2, 16, 14, 2 ** 18 - 1, 0, 0), (2, 16, 14, 2 ** 18, 1, 0), (2, 16, 14, 2 ** 19, 1, 0), (2, 16, 14, 2 ** 19 + 1, 0, 0), (2, 8, 14, 2 ** 20, 1, 0), (2, 16, 19, 2 ** 19 - 1, 1, 0),
    (2, 16, 19, 2 ** 19, 0, 0), (2, 16, 21, 2 ** 18, 0, 0), (3, 16, 14, 1, 1, 0), (3, 11, 14, 2 ** 15 - 1, 1, 0), (3, 10, 14, 2 ** 15 - 1, 0, 0), (3, 16, 22, 23999, 1, 0),
    (3, 16, 22, 24000, 0, 0), (3, 16, 22, 2 ** 20, 0, 0), (3, 8, 14, 2 ** 16 - 1, 0, 0), (3, 8, 14, 2 ** 16, 1, 0), (3, 11, 14, 2 ** 15, 1, 0), (3, 2, 14, 2 ** 17 - 1, 0, 0),
    (3, 2, 14, 2 ** 17, 1, 0), (3, 16, 19, 5 * 2 ** 17 - 1, 1, 0), (3, 16, 19, 5 * 2 ** 17, 1, 1)]


@pytest.mark.parametrize("dims,levels,log2,M,by_levels,ordered", FIELD_SIDES)
def test_field_module_on_both_sides_of_each_rule(tnn, dims, levels, log2, M, by_levels, ordered):
    """NetworkWithInputEncoding without autograd takes the route its size says, with autograd the one that keeps the encoded batch: the rows of the network on a batch
    that one kernel encoded, all levels of a point."""
    import tiny_dpcpp_nn
    tiny_dpcpp_nn.manual_seed(3)
    model = tiny_dpcpp_nn.NetworkWithInputEncoding(
        dims, 3, {"otype": "FullyFusedMLP", "activation": "ReLU", "output_activation": "None", "n_neurons": 64, "n_hidden_layers": 2},
        {"otype": "HashGrid", "type": "Hash", "n_levels": levels, "n_features_per_level": 2, "log2_hashmap_size": log2, "base_resolution": 16, "per_level_scale": 1.5},
        dtype=torch.float16, use_bias=False)
    d = tnn.grid_desc(dict(BASE, n_dims=dims, n_levels=levels, log2_hashmap_size=log2, per_level_scale=1.5))
    assert tnn.lib.tnn_grid_mlp_wants_levels(ctypes.byref(d), M) == by_levels
    x = torch.rand((M, dims), device=tnn.dev)
    with torch.no_grad():
        model.encoding.params.copy_(torch.rand(model.encoding.params.shape, device=tnn.dev) - 0.5)
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        y = model(x)
        scratch = torch.cuda.max_memory_allocated() - before - 6 * M
        if M >= 2 ** 11:  # 2 bytes of 16 or 32 features a point, and 16 bytes and the histograms of an order
            assert (scratch >= 64 * M * (levels > 8) + 32 * M * (levels <= 8)) == bool(by_levels) and (scratch >= (64 + 16) * M) == bool(ordered)
        x2 = torch.cat([x, torch.rand((DIRECT, dims), device=tnn.dev)])[: max(M, DIRECT + 1)]  # (a batch beyond those that are written by levels)
        walked = tnn.grid_forward(d, x2, model.encoding.params.detach().reshape(-1), 64, FP32)[:M]
        assert torch.equal(bits(y), bits(model.network(walked)))
    assert torch.equal(bits(y), bits(model(x).detach()))


def test_a_small_batch_in_a_graph_replays(tnn):
    d = tnn.grid_desc(BASE)
    table = torch.rand(tnn.grid_n_params(d), device=tnn.dev)
    x = torch.rand((1000, 3), device=tnn.dev)
    out = torch.empty((1000, 32), device=tnn.dev)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        tnn.grid_forward(d, x, table, 32, out=out)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        tnn.grid_forward(d, x, table, 32, out=out)
    for seed in range(4):
        x.copy_(torch.rand(x.shape, device=tnn.dev, generator=torch.Generator(device=tnn.dev).manual_seed(seed)))
        out.fill_(float(seed))
        graph.replay()
        torch.cuda.synchronize()
        got = out.clone()
        assert np.isfinite(got.cpu().numpy()).all() and torch.equal(got, tnn.grid_forward(d, x, table, 32))


@pytest.mark.parametrize("W,F,n_levels,dims,dtype,n_hidden,M,y_cols", [
    (64, 2, 16, 3, FP16, 2, 1001, 3), (64, 2, 12, 2, BF16, 4, 4096, 64), (64, 2, 32, 3, FP16, 3, 33, 16), (64, 2, 1, 2, FP16, 2, 31, 1), (16, 1, 16, 3, BF16, 2, 500, 5),
    (32, 4, 5, 2, FP16, 3, 777, 32), (64, 8, 8, 3, BF16, 2, 2050, 24), (64, 8, 3, 3, FP16, 1, 65, 7), (128, 2, 20, 3, FP16, 2, 300, 128), (128, 1, 9, 2, BF16, 1, 1, 2)])
@pytest.mark.parametrize("ordered", [False, True])
def test_network_behind_levels(tnn, W, F, n_levels, dims, dtype, n_hidden, M, y_cols, ordered):
    """tnn_grid_mlp_forward_levels against the kernel that evaluates the encoding itself, and the backward pass on the levels it leaves against the one that forms
    them from the table: the same values, whatever the buffers held before."""
    cfg = dict(BASE, n_dims=dims, n_levels=n_levels, n_features_per_level=F, log2_hashmap_size=12)
    L, gd, md = tnn.lib, tnn.grid_desc(cfg), tnn.mlp_desc(dtype, W, n_hidden, "relu", "sigmoid" if M % 2 else "none")
    g, m = ctypes.byref(gd), ctypes.byref(md)
    rng = np.random.default_rng(M)
    gen = torch.Generator(device=tnn.dev).manual_seed(M)
    x = torch.rand((M, dims), device=tnn.dev, generator=gen)
    table = torch.rand(tnn.grid_n_params(gd), device=tnn.dev, generator=gen) - 0.5
    _, pf, pb = tnn.prepare(md, rng.uniform(-0.3, 0.3, (n_hidden + 1, W, W)).astype(np.float32))
    order = tnn.grid_order(gd, x) if ordered else None
    o = ptr(order) if ordered else None
    y, expected = (torch.full((M, y_cols), float("nan"), dtype=TORCH[dtype], device=tnn.dev) for _ in range(2))
    levels = torch.full((L.tnn_grid_levels_bytes(g, M) // 2,), float("nan"), dtype=TORCH[dtype], device=tnn.dev)
    _lib.check(L.tnn_grid_mlp_inference_rows(g, m, ptr(x), o, ptr(table), ptr(pf), ptr(expected), y_cols, M, tnn.stream()))
    _lib.check(L.tnn_grid_mlp_forward_levels(g, m, None, W, W, 0, None, None, ptr(pf), None, ptr(x), o, ptr(table), ptr(levels), ptr(y), y_cols, M, tnn.stream()))
    assert torch.equal(bits(y), bits(expected))
    assert bool(torch.isfinite(levels).all())  # nothing of it is left unwritten: the kernels read whole groups of levels, of whole tiles
    if L.tnn_grid_mlp_train_supported(g, m) != _lib.TNN_OK:
        return
    dy = (torch.randn((M, y_cols), device=tnn.dev, generator=gen) * 1e-2).to(TORCH[dtype])
    dy_full = dy if y_cols <= 16 or y_cols == W else torch.nn.functional.pad(dy, (0, W - y_cols))
    size = L.tnn_grid_mlp_train_step_workspace_bytes(g, m, M)
    results = []
    for call, source in ((L.tnn_grid_mlp_backward_rows, table), (L.tnn_grid_mlp_backward_levels_rows, levels)):
        work = torch.full((size,), 255, dtype=torch.uint8, device=tnn.dev)
        dW, dtable = torch.full(((n_hidden + 1) * W * W,), float("nan"), device=tnn.dev), torch.full_like(table, float("nan"))
        _lib.check(call(g, m, ptr(x), o, ptr(source), ptr(pf), ptr(pb), ptr(dy_full), dy_full.shape[1], 8.0, 0.125, ptr(dW), FP32, ptr(dtable), 1, M, ptr(work), size,
                        tnn.stream()))
        results.append((dW, dtable))
    assert torch.equal(results[0][0], results[1][0])
    scale = float(results[0][1].abs().max())  # (sums of fp32 atomics in no defined order: the bar of tnn_grid_backward)
    assert scale > 0 and float((results[0][1] - results[1][1]).abs().max()) <= 1e-5 * scale


@pytest.mark.parametrize("dims,log2,M,interpolation", [(3, 19, 2 ** 19 + 5, "Linear"), (3, 16, 2 ** 19 + 5, "Smoothstep"), (3, 16, 2 ** 19, "Nearest"), (3, 22, 2 ** 18, "Linear"), (2, 16, 2 ** 19, "Linear")])
def test_backward_takes_its_own_forward_passes_order(tnn, dims, log2, M, interpolation):
    """Two forward passes on other points, then their backward passes in either order, one of them twice: the gradients of the plain scatter."""
    import tiny_dpcpp_nn
    cfg = dict(BASE, n_dims=dims, log2_hashmap_size=log2, interpolation=interpolation)
    enc = tiny_dpcpp_nn.Encoding(dims, {"otype": "HashGrid", "type": "Hash", "n_levels": 16, "n_features_per_level": 2, "log2_hashmap_size": log2, "base_resolution": 16,
                                        "per_level_scale": 1.447, "interpolation": interpolation})
    d = tnn.grid_desc(cfg)
    gen = torch.Generator(device=tnn.dev).manual_seed(8)
    xs = [torch.rand((M, dims), device=tnn.dev, generator=gen) for _ in range(2)]
    dys = [torch.randn((M, 32), device=tnn.dev, generator=gen) for _ in range(2)]
    ys = [enc(x) for x in xs]
    for i in (0, 1, 0):
        enc.params.grad = None
        ys[i].backward(dys[i], retain_graph=True)
        expected = tnn.grid_backward(d, xs[i], dys[i], FP32)
        scale = float(expected.abs().max())
        assert float((enc.params.grad.reshape(-1) - expected.reshape(-1)).abs().max()) <= 1e-5 * scale  # (fp32 sums in another order: the bar of tnn_grid_backward)


@pytest.mark.parametrize("dims,config,M,kept", [
    (2, dict(n_levels=16, log2_hashmap_size=16), 2 ** 19, False), (3, dict(n_levels=16, log2_hashmap_size=16, interpolation="Nearest"), 2 ** 19, False),
    (3, dict(n_levels=16, log2_hashmap_size=16), 2 ** 19, True), (2, dict(n_levels=1, n_features_per_level=8, log2_hashmap_size=22, base_resolution=2100), 2 ** 18, True)])
def test_an_order_is_kept_where_the_backward_pass_reads_it(tnn, dims, config, M, kept):
    """Between its passes an encoding holds a batch's cell order only where the backward pass takes it: in three dimensions and, in two, where bins refuse levels."""
    import tiny_dpcpp_nn
    cfg = dict(BASE, n_dims=dims, **config)
    enc = tiny_dpcpp_nn.Encoding(dims, {"otype": "HashGrid", "type": "Hash", **{k: v for k, v in cfg.items() if k != "n_dims"}})
    d = tnn.grid_desc(cfg)
    gen = torch.Generator(device=tnn.dev).manual_seed(10)
    x = torch.rand((M, dims), device=tnn.dev, generator=gen)
    dy = torch.randn((M, enc.n_output_dims), device=tnn.dev, generator=gen)
    before = torch.cuda.memory_allocated()
    y = enc(x)
    extra = torch.cuda.memory_allocated() - before - y.numel() * 4
    assert (extra >= 16 * M) if kept else (extra < 16 * M)
    y.backward(dy)
    expected = tnn.grid_backward(d, x, dy, FP32)
    scale = float(expected.abs().max())
    assert float((enc.params.grad.reshape(-1) - expected.reshape(-1)).abs().max()) <= 1e-5 * scale  # (fp32 sums in another order: the bar of tnn_grid_backward)


class MemoryFor:
    """PyTorch's allocator gives out about `spare` bytes more than are in use, and no more."""

    def __init__(self, spare):
        self.spare = spare

    def limit(self, spare):
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + spare) / torch.cuda.get_device_properties(0).total_memory)

    def __enter__(self):
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        self.limit(0)
        self.held = []
        while True:  # (what is left of the blocks it has)
            try:
                self.held.append(torch.empty(2 ** 21, dtype=torch.uint8, device="cuda"))
            except torch.cuda.OutOfMemoryError:
                break
        self.limit(self.spare)

    def __exit__(self, *_):
        del self.held
        torch.cuda.set_per_process_memory_fraction(1.0)


def test_passes_run_where_memory_is_short(tnn):
    """Without memory for the encoded batch by levels the passes run as they do without it: the same values (a batch that is not put in cell order)."""
    import tiny_dpcpp_nn
    M, grid = 131000, {"otype": "HashGrid", "type": "Hash", "n_levels": 16, "n_features_per_level": 2, "log2_hashmap_size": 14, "base_resolution": 16, "per_level_scale": 1.447}
    tiny_dpcpp_nn.manual_seed(4)
    gen = torch.Generator(device=tnn.dev).manual_seed(11)
    model = tiny_dpcpp_nn.NetworkWithInputEncoding(3, 3, {"otype": "FullyFusedMLP", "activation": "ReLU", "output_activation": "None", "n_neurons": 64, "n_hidden_layers": 2}, grid,
                                                   dtype=torch.float16, use_bias=False)
    enc = tiny_dpcpp_nn.Encoding(3, grid)
    x = torch.rand((M, 3), device=tnn.dev, generator=gen)
    dy = (torch.randn((M, 3), device=tnn.dev, generator=gen) * 1e-3).half()
    with torch.no_grad():
        model.encoding.params.copy_(torch.rand(model.encoding.params.shape, device=tnn.dev, generator=gen) - 0.5)
        enc.params.copy_(model.encoding.params)
        encoded = enc(x)
    y = model(x)
    assert torch.cuda.memory_allocated() > 64 * M  # (the levels that this pass keeps)
    y.backward(dy)
    expected = [p.grad.clone() for p in model.parameters()]
    model.zero_grad()
    y = y.detach()
    with torch.no_grad(), MemoryFor(128 * M + 8 * 2 ** 20):  # a result of 128 bytes a point, and not as much again beside it
        again = enc(x)
    assert torch.equal(bits(again), bits(encoded))
    del again, encoded
    with MemoryFor(6 * 2 ** 20):  # not 64 bytes a point
        with torch.no_grad():
            w = model(x)
        kept = torch.cuda.memory_allocated()
        z = model(x)
        assert torch.cuda.memory_allocated() - kept < 16 * M
    assert torch.equal(bits(z.detach()), bits(y)) and torch.equal(bits(w), bits(y))
    z.backward(dy)
    (dtable, dW), (expected_dtable, expected_dW) = [p.grad for p in model.parameters()], expected
    assert dW.numel() < dtable.numel() and torch.equal(dW, expected_dW)
    assert float((dtable - expected_dtable).abs().max()) <= 1e-5 * float(expected_dtable.abs().max())  # (fp32 atomics in no defined order: the bar of tnn_grid_backward)
