"""The scatter that sorts its contributions by destination (tnn_grid_backward_binned) against the oracle and the plain scatter."""
import ctypes

import numpy as np
import pytest
import torch

from tolerances import BF16, FP16, FP32

pytestmark = pytest.mark.gpu

CFG2 = dict(n_dims=2, n_levels=16, n_features_per_level=2, log2_hashmap_size=15, base_resolution=16, per_level_scale=1.5)
CFG3 = dict(n_dims=3, n_levels=16, n_features_per_level=2, log2_hashmap_size=19, base_resolution=16, per_level_scale=1.447)
DT = {FP32: torch.float32, FP16: torch.float16, BF16: torch.bfloat16}


def binned(tnn, d, x, g, dtype, ordered=False, grad=None, overwrite=True, short=0, both=False):
    from tiny_dpcpp_nn import _lib
    M = x.shape[0]
    p = lambda t: ctypes.c_void_p(t.data_ptr()) if t is not None else None  # noqa: E731
    need = tnn.lib.tnn_grid_backward_workspace_bytes(ctypes.byref(d), M)
    work = torch.full((max(need - short, 1),), 0xA5, dtype=torch.uint8, device=tnn.dev)  # nothing in it has to be cleared
    order = tnn.grid_order(d, x) if ordered or both else None
    if grad is None:
        grad = torch.full((tnn.grid_n_params(d),), 0.123, dtype=torch.float32, device=tnn.dev)
    _lib.check(tnn.lib.tnn_grid_backward_binned(ctypes.byref(d), None if ordered else p(x), p(order), p(g), dtype, g.shape[1], p(grad), int(overwrite), M,
                                                p(work), work.numel(), tnn.stream()))
    return grad


@pytest.mark.parametrize("cfg", [CFG2, CFG3, dict(CFG3, log2_hashmap_size=22, n_levels=12), dict(CFG2, n_features_per_level=1, hash="Prime"),
                                 dict(CFG3, n_features_per_level=4, n_levels=8, interpolation="Smoothstep"), dict(CFG2, n_features_per_level=8, n_levels=7),
                                 dict(CFG3, interpolation="Nearest"), dict(CFG2, grid_type="Dense", n_levels=9), dict(CFG2, grid_type="Tiled"),
                                 dict(CFG2, n_levels=34, per_level_scale=1.2)])
@pytest.mark.parametrize("M,ordered,kind", [(1, False, "uniform"), (513, False, "uniform"), (40007, True, "uniform"), (40007, False, "few"), (2 ** 19 + 9, False, "uniform")])
def test_binned_scatter_matches_the_oracle(tnn, oracle, cfg, M, ordered, kind):
    """Bins of very different lengths ("few": all points on some twenty cells), a batch of more than one part, edges of bins, every kind of level. fp32 sums
    in another order against the oracle's double sum, at the plain scatter's bar; accumulate mode adds on top."""
    rng = np.random.default_rng(M + cfg["n_dims"])
    x = rng.uniform(0, 1, (M, cfg["n_dims"])).astype(np.float32)
    if kind == "few":
        x = x[rng.integers(0, 20, M)]
    x[0] = 1.0
    pw = cfg["n_levels"] * cfg["n_features_per_level"] + 4
    d = tnn.grid_desc(cfg)
    g = torch.from_numpy(rng.standard_normal((M, pw)).astype(np.float32)).to(tnn.dev)
    xt = torch.from_numpy(x).to(tnn.dev)
    for dtype in (FP32, BF16, FP16) if M == 40007 else (FP32,):
        gt = g.to(DT[dtype]).contiguous()
        grad = binned(tnn, d, xt, gt, dtype, ordered)
        ref = oracle.grid_backward(cfg, x, gt.float().cpu().numpy(), tnn.grid_n_params(d))
        bar = 1e-5 * max(1.0, np.abs(ref).max())
        assert np.abs(grad.cpu().numpy() - ref).max() <= bar
        twice = binned(tnn, d, xt, gt, dtype, ordered, grad=grad.clone(), overwrite=False)
        assert np.abs(twice.cpu().numpy() - 2 * ref).max() <= 2 * bar


def crowded(kind, cfg, M, rng):
    """Points of a training batch that leaves most of the unit cube empty."""
    D = cfg["n_dims"]
    u = rng.uniform(0, 1, (M, D))
    if kind == "inner":
        u = 0.05 + 0.9 * u
    elif kind == "quarter":
        u = 0.25 + 0.5 * u
    elif kind == "small":
        u = 0.4 + 0.05 * u
    elif kind == "shell":
        v = rng.standard_normal((M, D))
        u = np.clip(0.5 + 0.35 * v / np.linalg.norm(v, axis=1, keepdims=True) + 0.01 * rng.standard_normal((M, D)), 0, 1)
    elif kind == "one cell":
        u = 0.7 + 1e-6 * u
    elif kind == "line":  # the far corner along x in another run of 16 entries than the near one, at one level after the other
        scales = cfg["base_resolution"] * cfg["per_level_scale"] ** np.arange(cfg["n_levels"]) - 1
        u[:, 0] = (15 / scales)[rng.integers(1, cfg["n_levels"], M)]
    return u.astype(np.float32)


@pytest.mark.parametrize("cfg", [CFG2, CFG3, dict(CFG3, per_level_scale=2.0, log2_hashmap_size=15), dict(CFG2, n_features_per_level=1, n_levels=12),
                                 dict(CFG3, n_features_per_level=4, n_levels=8), dict(CFG2, n_features_per_level=8, n_levels=7), dict(CFG3, hash="Prime")])
@pytest.mark.parametrize("kind", ["inner", "quarter", "small", "shell", "one cell", "line"])
def test_crowded_points_match_the_oracle(tnn, oracle, cfg, kind):
    """The bar of the test above: products and sums of fp32 values, whatever the bins' lengths."""
    rng = np.random.default_rng(7)
    M = 70001
    x = crowded(kind, cfg, M, rng)
    d = tnn.grid_desc(cfg)
    g = torch.from_numpy(rng.standard_normal((M, cfg["n_levels"] * cfg["n_features_per_level"])).astype(np.float32)).to(tnn.dev)
    grad = binned(tnn, d, torch.from_numpy(x).to(tnn.dev), g, FP32)
    ref = oracle.grid_backward(cfg, x, g.cpu().numpy(), tnn.grid_n_params(d))
    assert np.abs(grad.cpu().numpy() - ref).max() <= 1e-5 * max(1.0, np.abs(ref).max())


@pytest.mark.parametrize("M", [33003, 50001, 2 ** 18 + 1])
def test_as_many_bins_as_a_level_may_have(tnn, oracle, M):
    """1024 bins a level (eight features, 2^21 entries), dealt out by the smallest workgroups and by the largest."""
    cfg = dict(n_dims=3, n_levels=3, n_features_per_level=8, log2_hashmap_size=21, base_resolution=128, per_level_scale=1.2)
    rng = np.random.default_rng(M)
    x = rng.uniform(0, 1, (M, 3)).astype(np.float32)
    d = tnn.grid_desc(cfg)
    g = torch.from_numpy(rng.standard_normal((M, 24)).astype(np.float32)).to(tnn.dev)
    grad = binned(tnn, d, torch.from_numpy(x).to(tnn.dev), g, FP32)
    ref = oracle.grid_backward(cfg, x, g.cpu().numpy(), tnn.grid_n_params(d))
    assert np.abs(grad.cpu().numpy() - ref).max() <= 1e-5 * max(1.0, np.abs(ref).max())


@pytest.mark.parametrize("cfg", [dict(CFG2, log2_hashmap_size=19), CFG3])
def test_crowded_points_take_about_as_long_as_even_ones(tnn, cfg):
    """No distribution of an ordinary batch falls off the fast path: measured 0.95 to 1.05 of the time for evenly spread points, where one
    that overfills bins of a fixed size took four to six times as long."""
    M, rng = 2 ** 18, np.random.default_rng(3)
    d = tnn.grid_desc(cfg)
    g = torch.randn((M, 32), device=tnn.dev)
    grad = torch.empty(tnn.grid_n_params(d), device=tnn.dev)

    def time(kind):
        x = torch.from_numpy(crowded(kind, cfg, M, rng)).to(tnn.dev)
        times = []
        for _ in range(8):
            ev = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
            ev[0].record()
            binned(tnn, d, x, g, FP32, grad=grad)
            ev[1].record()
            ev[1].synchronize()
            times.append(ev[0].elapsed_time(ev[1]))
        return sorted(times)[2]

    even = time("even")
    for kind in ("inner", "quarter", "shell"):
        assert time(kind) <= 2 * even, kind


def scatter_time(tnn, cfg, x):
    """Of nine samples of ten calls, the third."""
    d, M = tnn.grid_desc(cfg), x.shape[0]
    g = torch.randn((M, cfg["n_levels"] * cfg["n_features_per_level"]), device=tnn.dev)
    grad = torch.empty(tnn.grid_n_params(d), device=tnn.dev)
    work = torch.empty(tnn.lib.tnn_grid_backward_workspace_bytes(ctypes.byref(d), M), dtype=torch.uint8, device=tnn.dev)
    times = []
    for _ in range(9):
        ev = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        ev[0].record()
        for _ in range(10):
            assert tnn.lib.tnn_grid_backward_binned(ctypes.byref(d), x.data_ptr(), None, g.data_ptr(), FP32, g.shape[1], grad.data_ptr(), 1, M, work.data_ptr(), work.numel(), tnn.stream()) == 0
        ev[1].record()
        ev[1].synchronize()
        times.append(ev[0].elapsed_time(ev[1]))
    return sorted(times)[2]


@pytest.mark.parametrize("cfg,most", [(CFG2, 2.7), (dict(CFG2, log2_hashmap_size=19), 2.3)])
def test_points_in_a_corner_of_coarse_levels(tnn, cfg, most):
    """All points in a square of 5 % of the side, where the coarse levels are binned: 2.1 and 1.8 times as long as even ones, and 3.3 and 2.6 to 3.1 without copies of the sums."""
    M, rng = 2 ** 16, np.random.default_rng(3)
    even, small = (scatter_time(tnn, cfg, torch.from_numpy(crowded(kind, cfg, M, rng)).to(tnn.dev)) for kind in ("even", "small"))
    assert small <= most * even


@pytest.mark.parametrize("seed", [2, 3])
def test_long_bins_do_not_wait_for_each_other(tnn, seed):
    """All of 2^18 points are one of twenty: 4.0 and 4.4 times as long as even ones, and 6.1 and 6.2 where a workgroup takes the second of its long bins after the first."""
    cfg, M, rng = dict(CFG2, log2_hashmap_size=19), 2 ** 18, np.random.default_rng(seed)
    twenty = rng.uniform(0, 1, (20, 2))[rng.integers(0, 20, M)]
    few, even = (scatter_time(tnn, cfg, torch.from_numpy(x.astype(np.float32)).to(tnn.dev)) for x in (twenty, rng.uniform(0, 1, (M, 2))))
    assert few <= 5.2 * even


@pytest.mark.parametrize("features", [1, 2, 4, 8])
@pytest.mark.parametrize("cfg", [CFG2, CFG3, dict(CFG3, grid_type="Tiled", base_resolution=15)])
@pytest.mark.parametrize("crowd", [1500, 3000, 6000, 12000, 40007])
def test_bins_with_copies_of_their_sums(tnn, oracle, cfg, features, crowd):
    """So many points of 40007 in one cell: a bin has copies from eight records a lane on, which are one or more of such a point and 256, 512 or 1024 lanes. Every bin's
    sums are followed by others', with and without copies, in the same LDS; levels of an odd number of entries (tiled) take the other store. The bar of even points."""
    cfg = dict(cfg, n_features_per_level=features, n_levels=16 if features <= 2 else 10)
    M, rng = 40007, np.random.default_rng(crowd + features)
    x = rng.uniform(0, 1, (M, cfg["n_dims"])).astype(np.float32)
    x[rng.permutation(M)[:crowd]] = 0.4321
    d = tnn.grid_desc(cfg)
    g = rng.standard_normal((M, cfg["n_levels"] * features)).astype(np.float32)
    ref = oracle.grid_backward(cfg, x, g, tnn.grid_n_params(d))
    table = np.full(tnn.grid_n_params(d), 0.5, np.float32)
    for overwrite in (True, False):
        grad = binned(tnn, d, torch.from_numpy(x).to(tnn.dev), torch.from_numpy(g).to(tnn.dev), FP32, grad=torch.from_numpy(table).to(tnn.dev), overwrite=overwrite)
        assert np.abs(grad.cpu().numpy() - (0 if overwrite else 0.5) - ref).max() <= 1e-5 * max(1.0, np.abs(ref).max())


@pytest.mark.parametrize("cfg", [CFG2, CFG3, dict(CFG3, log2_hashmap_size=22, n_levels=12), dict(CFG3, n_features_per_level=8, n_levels=6, per_level_scale=2.0),
                                 dict(CFG2, interpolation="Nearest"), dict(CFG2, n_features_per_level=1, grid_type="Dense", n_levels=9)])
@pytest.mark.parametrize("kind", ["even", "small"])
def test_points_in_both_orders(tnn, oracle, cfg, kind):
    """Boxes and atomics take the cell order and the bins the caller's, where a call is given both: the contributions are the same."""
    rng = np.random.default_rng(11)
    M = 40007
    x = crowded(kind, cfg, M, rng)
    d = tnn.grid_desc(cfg)
    for dtype in (FP32, FP16):
        g = torch.from_numpy(rng.standard_normal((M, cfg["n_levels"] * cfg["n_features_per_level"])).astype(np.float32)).to(tnn.dev).to(DT[dtype])
        grad = binned(tnn, d, torch.from_numpy(x).to(tnn.dev), g, dtype, both=True)
        ref = oracle.grid_backward(cfg, x, g.float().cpu().numpy(), tnn.grid_n_params(d))
        assert np.abs(grad.cpu().numpy() - ref).max() <= 1e-5 * max(1.0, np.abs(ref).max())


def test_encoding_orders_a_batch_whose_finest_levels_are_not_binned(tnn):
    """Eight features in 2^22 entries are beyond what the bins hold in LDS: the encoding's backward pass hands both orders over from 2^18 points on."""
    import tiny_dpcpp_nn
    cfg = dict(CFG3, n_levels=5, n_features_per_level=8, log2_hashmap_size=22, per_level_scale=2.6)
    d = tnn.grid_desc(cfg)
    wants = lambda M, **kw: tnn.lib.tnn_grid_backward_wants_order(ctypes.byref(tnn.grid_desc(dict(cfg, **kw))), M)  # noqa: E731
    assert wants(2 ** 18) == 1 and wants(2 ** 18 - 1) == 0 and wants(2 ** 20, interpolation="Nearest") == 0 and wants(2 ** 20, log2_hashmap_size=19) == 0
    enc = tiny_dpcpp_nn.Encoding(3, {"otype": "HashGrid", "type": "Hash", "n_levels": 5, "n_features_per_level": 8, "log2_hashmap_size": 22,
                                     "base_resolution": 16, "per_level_scale": 2.6})
    x = torch.rand((2 ** 18 + 5, 3), device=tnn.dev)
    dy = torch.randn((x.shape[0], 40), device=tnn.dev)
    got, = torch.autograd.grad(enc(x), [enc.params], dy)
    ref = tnn.grid_backward(d, x, dy, FP32)
    assert float((got.reshape(-1) - ref.reshape(-1)).abs().max()) <= 1e-5 * float(ref.abs().max())


@pytest.mark.parametrize("cfg,M", [(CFG3, 16384), (dict(CFG3, n_levels=8, log2_hashmap_size=20), 32768), (dict(CFG2, n_levels=12, log2_hashmap_size=16), 65536), (CFG3, 2 ** 17)])
def test_workspace_of_a_batch_holds_a_smaller_one(tnn, cfg, M):
    """Just below these sizes the scatter has twice as many workgroups or bins more levels, and needs more."""
    from tiny_dpcpp_nn import _lib
    d = tnn.grid_desc(cfg)
    work = torch.empty(tnn.lib.tnn_grid_backward_workspace_bytes(ctypes.byref(d), M), dtype=torch.uint8, device=tnn.dev)
    for m in (M, M - 1, M * 15 // 16, M * 14 // 15):
        x, g = torch.rand((m, cfg["n_dims"]), device=tnn.dev), torch.randn((m, 2 * cfg["n_levels"]), device=tnn.dev)
        grad = torch.empty(tnn.grid_n_params(d), device=tnn.dev)
        _lib.check(tnn.lib.tnn_grid_backward_binned(ctypes.byref(d), x.data_ptr(), None, g.data_ptr(), FP32, g.shape[1], grad.data_ptr(), 1, m, work.data_ptr(), work.numel(), tnn.stream()))
        ref = tnn.grid_backward(d, x, g, FP32)
        assert float((grad - ref).abs().max()) <= 1e-5 * max(1.0, float(ref.abs().max()))


@pytest.mark.parametrize("features,levels,base,M", [(2, 16, 16, 122880), (2, 16, 16, 122881), (2, 6, 12, 14358), (2, 6, 12, 14359), (2, 8, 16, 5000), (1, 16, 16, 40000), (4, 6, 16, 20000), (2, 16, 8, 40000), (8, 3, 16, 16384)])
def test_batches_in_cell_order_without_boxes(tnn, oracle, features, levels, base, M):
    """Three dimensions, on both sides of the size up to which all levels are binned (2^17 points less what copies save, or two points a cell on the mean of the levels), and with boxes: larger batches, four and eight features, and levels that are
    copied (base 8), whose launch boxes share. The bar of the plain scatter."""
    cfg = dict(CFG3, n_features_per_level=features, n_levels=levels, base_resolution=base)
    rng = np.random.default_rng(M + features)
    x = rng.uniform(0, 1, (M, 3)).astype(np.float32)
    x[: M // 8] = x[0] * 0.9 + 0.01 * x[: M // 8]  # (some points crowd)
    d = tnn.grid_desc(cfg)
    g = rng.standard_normal((M, levels * features)).astype(np.float32)
    ref = oracle.grid_backward(cfg, x, g, tnn.grid_n_params(d))
    xt, gt = torch.from_numpy(x).to(tnn.dev), torch.from_numpy(g).to(tnn.dev)
    order = tnn.grid_order(d, xt)
    for rows in (None, xt):  # from the order alone, and with the points beside it
        grad = torch.full((tnn.grid_n_params(d),), float("nan"), device=tnn.dev)
        need = tnn.lib.tnn_grid_backward_workspace_bytes(ctypes.byref(d), M)
        work = torch.empty(max(need, 1), dtype=torch.uint8, device=tnn.dev)
        assert tnn.lib.tnn_grid_backward_binned(ctypes.byref(d), None if rows is None else rows.data_ptr(), order.data_ptr(), gt.data_ptr(), FP32, gt.shape[1], grad.data_ptr(), 1, M,
                                                work.data_ptr(), work.numel(), tnn.stream()) == 0, tnn.lib.tnn_last_error()
        assert np.abs(grad.cpu().numpy() - ref).max() <= 1e-5 * max(1.0, np.abs(ref).max())


def test_binned_workspace_is_checked(tnn):
    from tiny_dpcpp_nn import _lib
    d = tnn.grid_desc(CFG3)
    x = torch.rand((40960, 3), device=tnn.dev)
    with pytest.raises(_lib.TnnError):
        binned(tnn, d, x, torch.rand((40960, 32), device=tnn.dev), FP32, short=4096)
    assert tnn.lib.tnn_grid_backward_workspace_bytes(ctypes.byref(d), 0) == 0


@pytest.mark.parametrize("M", [28001, 32003, 60001, 64007, 80009])
@pytest.mark.parametrize("features", [1, 2, 8])
def test_sums_with_few_and_many_records_a_lane(tnn, oracle, M, features):
    """Two to six rounds of records of an even spread, which choose how many a lane has in flight, and levels whose last entries fill a bin's last pair or not. fp32 results
    of double sums: the bar of the plain scatter."""
    cfg = dict(CFG2, n_features_per_level=features, n_levels=16 if features <= 2 else 10)
    rng = np.random.default_rng(M + features)
    x = rng.uniform(0, 1, (M, 2)).astype(np.float32)
    d = tnn.grid_desc(cfg)
    g = rng.standard_normal((M, cfg["n_levels"] * features)).astype(np.float32)
    ref = oracle.grid_backward(cfg, x, g, tnn.grid_n_params(d))
    grad = binned(tnn, d, torch.from_numpy(x).to(tnn.dev), torch.from_numpy(g).to(tnn.dev), FP32)
    assert np.abs(grad.cpu().numpy() - ref).max() <= 1e-5 * max(1.0, np.abs(ref).max())


@pytest.mark.parametrize("features,log2,levels,M", [(1, 19, 16, 8192), (2, 19, 16, 8209), (2, 19, 16, 16384), (4, 17, 16, 8191), (8, 17, 12, 8191)])
@pytest.mark.parametrize("crowd", [0, 5000])
def test_workgroups_that_stay_for_several_bins(tnn, oracle, features, log2, levels, M, crowd):
    """Bins of 256 records at most, 128 with eight features, and 1500 to 3000 of them, 32 KB each, where 256 CUs hold four workgroups: the sums start from zero for each, also behind a
    long bin, with copies, of points in one cell. The bar of the plain scatter."""
    cfg = dict(CFG3, n_features_per_level=features, log2_hashmap_size=log2, n_levels=levels)
    rng = np.random.default_rng(M + features)
    x = rng.uniform(0, 1, (M, 3)).astype(np.float32)
    x[rng.permutation(M)[:crowd]] = 0.4321
    d = tnn.grid_desc(cfg)
    g = rng.standard_normal((M, levels * features)).astype(np.float32)
    ref = oracle.grid_backward(cfg, x, g, tnn.grid_n_params(d))
    table = torch.full((tnn.grid_n_params(d),), 0.5, device=tnn.dev)
    for overwrite in (True, False):
        grad = binned(tnn, d, torch.from_numpy(x).to(tnn.dev), torch.from_numpy(g).to(tnn.dev), FP32, grad=table.clone(), overwrite=overwrite)
        assert np.abs(grad.cpu().numpy() - (0 if overwrite else 0.5) - ref).max() <= 1e-5 * max(1.0, np.abs(ref).max())


@pytest.mark.parametrize("features", [1, 2, 4])
def test_tiled_levels_of_an_odd_number_of_entries(tnn, oracle, features):
    """A tiled level has base_resolution^3 entries, 29791 here: the next level begins in the middle of a pair of entries, and the last entry is half of one."""
    cfg = dict(CFG3, grid_type="Tiled", base_resolution=31, n_features_per_level=features, n_levels=5)
    rng = np.random.default_rng(features)
    M = 40007
    x = rng.uniform(0, 1, (M, 3)).astype(np.float32)
    d = tnn.grid_desc(cfg)
    assert d.offsets[1] % 2 == 1
    g = rng.standard_normal((M, cfg["n_levels"] * features)).astype(np.float32)
    ref = oracle.grid_backward(cfg, x, g, tnn.grid_n_params(d))
    grad = binned(tnn, d, torch.from_numpy(x).to(tnn.dev), torch.from_numpy(g).to(tnn.dev), FP32)
    assert np.abs(grad.cpu().numpy() - ref).max() <= 1e-5 * max(1.0, np.abs(ref).max())
