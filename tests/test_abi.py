"""CPU-side checks of the C-ABI library: it loads, exports every symbol include/tnn_hip.h declares,
and its pure host entry points (descriptor validation, size queries) behave. No kernel is launched."""
import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_symbols():
    txt = open(os.path.join(ROOT, "include", "tnn_hip.h")).read()
    txt = re.sub(r"/\*.*?\*/", "", txt, flags=re.S)
    return sorted(set(re.findall(r"\b(tnn_[a-z0-9_]+)\s*\(", txt)))


@pytest.fixture(scope="module")
def lib():
    from tiny_dpcpp_nn import _lib
    return _lib.load()


def test_exports_every_declared_symbol(lib):
    from tiny_dpcpp_nn import _lib
    names = declared_symbols()
    assert len(names) >= 20
    for n in names:
        assert hasattr(lib, n), f"{n} is declared in include/tnn_hip.h but not exported"
        assert n in _lib.SIGNATURES, f"{n} has no ctypes prototype"
    assert lib.tnn_abi_version() == 1


def test_descriptor_validation_is_host_only(lib):
    from tiny_dpcpp_nn import _lib
    good = _lib.MlpDesc(_lib.TNN_BF16, 64, 4, _lib.ACT_RELU, _lib.ACT_NONE)
    # (4+1) matrices * 2 tiles * 4 k-blocks * 512 elements * 2 bytes
    assert lib.tnn_mlp_prepared_bytes(ctypes.byref(good)) == 5 * 2 * 4 * 512 * 2
    assert lib.tnn_mlp_prepared_bytes(ctypes.byref(_lib.MlpDesc(_lib.TNN_FP16, 16, 2, 0, 8))) == 3 * 1 * 1 * 512 * 2
    for bad in (_lib.MlpDesc(_lib.TNN_BF16, 48, 4, 0, 8), _lib.MlpDesc(_lib.TNN_BF16, 64, 0, 0, 8), _lib.MlpDesc(_lib.TNN_FP32, 64, 4, 0, 8),
                _lib.MlpDesc(_lib.TNN_BF16, 64, 4, _lib.ACT_TANH, 8)):
        assert lib.tnn_mlp_prepared_bytes(ctypes.byref(bad)) == 0
        assert lib.tnn_mlp_backward_workspace_bytes(ctypes.byref(bad), 1024) == 0
    assert lib.tnn_mlp_backward_workspace_bytes(ctypes.byref(good), 1 << 18) > 0
    # the fused training step only needs room for per-workgroup partial weight gradients ...
    assert 0 < lib.tnn_mlp_train_step_workspace_bytes(ctypes.byref(good), 1 << 18) < 64 << 20
    # ... wider networks stage activations and deltas in the workspace
    wide = _lib.MlpDesc(_lib.TNN_FP16, 128, 8, _lib.ACT_RELU, _lib.ACT_NONE)
    assert lib.tnn_mlp_train_step_workspace_bytes(ctypes.byref(wide), 1 << 18) > lib.tnn_mlp_backward_workspace_bytes(ctypes.byref(wide), 1 << 18)


def test_grid_descriptor_host_side(lib):
    from tiny_dpcpp_nn import _lib
    d = _lib.GridDesc()
    assert lib.tnn_grid_desc_init(ctypes.byref(d), 2, 16, 2, 19, 16, 1.5, 0, 1, 1, _lib.TNN_FP16) == 0
    assert d.offsets[16] == 3829192 and lib.tnn_grid_n_params(ctypes.byref(d)) == 7658384
    assert lib.tnn_grid_desc_init(ctypes.byref(d), 3, 16, 2, 22, 16, 1.447, 0, 1, 1, _lib.TNN_FP16) == 0
    assert d.offsets[16] == 42519264
    assert lib.tnn_grid_desc_init(ctypes.byref(d), 3, 200, 2, 22, 16, 1.447, 0, 1, 1, _lib.TNN_FP16) == _lib.TNN_ERR_INVALID_ARGUMENT
    assert b"MAX_N_LEVELS" in lib.tnn_last_error()
    assert lib.tnn_grid_desc_init(ctypes.byref(d), 5, 16, 2, 22, 16, 1.447, 0, 1, 1, _lib.TNN_FP16) == _lib.TNN_ERR_UNSUPPORTED


def test_scatter_workspace_is_as_large_as_the_header_says(lib):
    """The sizes given at tnn_grid_backward_binned and tnn_grid_mlp_train_step_l2_adam, in MiB, and that they stop growing at 2^19 points."""
    from tiny_dpcpp_nn import _lib
    d = _lib.GridDesc()
    header = open(os.path.join(ROOT, "include", "tnn_hip.h")).read()
    for dims, features, sizes in ((2, 2, (183, 366)), (3, 2, (500, 1000)), (3, 4, (829, 1658)), (3, 8, (1377, 2754))):
        assert lib.tnn_grid_desc_init(ctypes.byref(d), dims, 16, features, 19, 16, 1.5 if dims == 2 else 1.447, 0, 1, 1, _lib.TNN_FP32) == 0
        got = [lib.tnn_grid_backward_workspace_bytes(ctypes.byref(d), 2 ** k) / 2 ** 20 for k in (18, 19, 20, 22)]
        assert [int(g) for g in got] == [sizes[0], sizes[1], sizes[1], sizes[1]]
        assert all(f"{size} " in header for size in sizes)
    mlp = _lib.MlpDesc(_lib.TNN_FP16, 64, 2, _lib.ACT_RELU, _lib.ACT_NONE)
    assert lib.tnn_grid_desc_init(ctypes.byref(d), 2, 16, 2, 19, 16, 1.5, 0, 1, 1, _lib.TNN_FP16) == 0
    step = int(lib.tnn_grid_mlp_train_step_workspace_bytes(ctypes.byref(d), ctypes.byref(mlp), 2 ** 18) / 2 ** 20)
    assert f"({step} MiB for 2^18 points" in header


@pytest.mark.parametrize("dims,features,levels,log2,scale,base,grid_type", [
    (2, 2, 16, 15, 1.5, 16, 0), (2, 2, 16, 19, 1.5, 16, 0), (2, 2, 12, 16, 1.5, 16, 0), (2, 2, 16, 22, 1.5, 16, 0), (2, 1, 16, 12, 1.3, 16, 0), (2, 8, 8, 17, 2.0, 16, 0), (2, 2, 40, 19, 1.2, 16, 0),
    (3, 2, 16, 19, 1.447, 16, 0), (3, 2, 8, 20, 1.447, 16, 0), (3, 2, 4, 19, 1.3, 16, 1), (3, 2, 16, 19, 1.447, 16, 2), (3, 4, 12, 14, 1.6, 16, 0), (3, 8, 3, 21, 1.2, 128, 0), (3, 1, 2, 23, 1.5, 300, 0)])
def test_scatter_workspace_of_a_batch_holds_smaller_ones(lib, dims, features, levels, log2, scale, base, grid_type):
    """Over the sizes where the binning's workgroups are halved, levels leave the bins for boxes, and coarse levels are binned or not. From 2^17 points on the size is the points' share of that for 2^18."""
    from tiny_dpcpp_nn import _lib
    d, mlp = _lib.GridDesc(), _lib.MlpDesc(_lib.TNN_FP16, 64, 2, _lib.ACT_RELU, _lib.ACT_NONE)
    assert lib.tnn_grid_desc_init(ctypes.byref(d), dims, levels, features, log2, base, scale, grid_type, 1, 1, _lib.TNN_FP32) == 0
    sizes = {2 ** k + e for k in range(8, 22) for e in (-1, 0, 1)} | {int(2 ** (8 + i / 12)) for i in range(156)}
    for halved in (2 ** 18, 2 ** 19, 2 ** 17):  # points times levels
        sizes |= {halved // n + e for n in range(1, levels + 1) for e in (-1, 0, 1)}
    for l in range(levels):
        sizes |= {min(2 ** 21, d.resolutions[l] ** dims // 2) + e for e in (-1, 0, 1)}
    sizes = sorted(m for m in sizes if m > 0)
    for query in (lambda m: lib.tnn_grid_backward_workspace_bytes(ctypes.byref(d), m), lambda m: lib.tnn_grid_mlp_train_step_workspace_bytes(ctypes.byref(d), ctypes.byref(mlp), m)):
        needs = [query(m) for m in sizes]
        assert needs == sorted(needs), [m for m, a, b in zip(sizes, needs, needs[1:]) if b < a]
    half, whole = (lib.tnn_grid_backward_workspace_bytes(ctypes.byref(d), m) for m in (2 ** 17, 2 ** 18))
    if levels > 2 and (log2, grid_type) not in ((12, 0), (14, 0), (19, 2)):  # (2^17 points of two levels have the smaller workgroups; levels of small tables are in boxes at 2^18, in cell order)
        assert half <= whole * 0.51


def scatter_need(lib, d, M, ordered):
    """Bytes that the scatter of M points says it needs where it has none to speak of, 0 where it needs none. Planned on the host and then refused: for the workspace, or
    for its table's alignment."""
    from tiny_dpcpp_nn import _lib
    rc = lib.tnn_grid_backward_binned(ctypes.byref(d), None if ordered else 4096, 4096 if ordered else None, 4096, _lib.TNN_FP32, d.n_levels * d.n_features_per_level, 4100, 1, M, 4096, 1, None)
    if rc == _lib.TNN_ERR_INVALID_ARGUMENT:
        return 0
    assert rc == _lib.TNN_ERR_WORKSPACE
    return int(lib.tnn_last_error().decode().rsplit(", ", 1)[1].split()[0])


@pytest.mark.parametrize("dims,features,levels,log2,scale,base,sides", [
    # (points in cell order, whether all levels are binned)
    (3, 2, 16, 19, 1.447, 16, ((4096, 0), (8192, 1), (122880, 1), (122881, 0))), (3, 1, 8, 19, 2.0, 16, ((8192, 1), (114688, 1), (114689, 0))), (3, 2, 8, 16, 1.3, 16, ((8192, 1), (109817, 1), (109818, 0))),
    (3, 2, 16, 17, 1.3, 32, ((5000, 1), (131071, 1), (131072, 0))), (3, 2, 7, 19, 2.0, 16, ((16384, 1), (50176, 1), (50177, 0))), (3, 2, 16, 17, 1.3, 15, ((5000, 1), (60489, 1), (60490, 0))), (3, 2, 8, 16, 1.25, 11, ((8192, 1), (10828, 1), (10829, 0))), (2, 2, 16, 19, 1.447, 16, ((65536, 0),)), (3, 2, 16, 17, 1.447, 8, ((16384, 0),)),
    (3, 4, 8, 19, 2.0, 16, ((8192, 0), (32768, 0))), (3, 8, 8, 19, 2.0, 16, ((8192, 0), (32768, 0))), (3, 8, 6, 16, 1.25, 8, ((16387, 0), (65536, 0)))])
def test_batches_have_boxes_where_a_cell_has_many_points(lib, dims, features, levels, log2, scale, base, sides):
    """Up to two points a cell on the mean of the levels, six of eight levels and more from 16 cells a side on, and for one and two features. Boxes take levels away from the bins, which have room for two records of every pair of corners of each level."""
    from tiny_dpcpp_nn import _lib
    d = _lib.GridDesc()
    assert lib.tnn_grid_desc_init(ctypes.byref(d), dims, levels, features, log2, base, scale, 0, 1, 1, _lib.TNN_FP32) == 0
    for M, binned in sides:
        assert (scatter_need(lib, d, M, True) >= 2 * (M << (dims - 1)) * levels * (8 + 4 * features)) == binned, M


@pytest.mark.parametrize("features,levels,log2,scale,base", [(2, 16, 19, 1.447, 16), (2, 16, 15, 1.5, 16), (2, 8, 17, 2.0, 16), (2, 16, 17, 1.3, 32), (1, 16, 19, 1.3, 16), (1, 4, 20, 2.0, 14), (2, 12, 14, 1.25, 11), (4, 8, 19, 2.0, 16),
                                                         (8, 6, 16, 1.25, 8)])
def test_scatter_workspace_holds_every_smaller_plan_in_either_order(lib, features, levels, log2, scale, base):
    """Around the sizes between which batches have no boxes, and the powers of two from which the bins take a level."""
    from tiny_dpcpp_nn import _lib
    d = _lib.GridDesc()
    assert lib.tnn_grid_desc_init(ctypes.byref(d), 3, levels, features, log2, base, scale, 0, 1, 1, _lib.TNN_FP32) == 0
    dense = int(2 * levels / sum(float(d.resolutions[l]) ** -3 for l in range(levels)))
    sizes = sorted({2 ** k + e for k in range(8, 19) for e in (-1, 0, 1)} | {int(2 ** (8 + i / 6)) for i in range(60)} | {n * dense + e for n in (1, 3) for e in (-1, 0, 1, 2, 3)} | {2 ** 17 * n // levels + e for n in range(1, levels + 1) for e in (-1, 0, 1)})
    most = 0
    for M in sizes:
        if M < 1:
            continue
        most = max([most] + [scatter_need(lib, d, M, ordered) for ordered in (False, True)])
        assert lib.tnn_grid_backward_workspace_bytes(ctypes.byref(d), M) >= most, M


def test_order_buffer_has_what_its_route_needs(lib):
    """16 bytes a point; up to 8192 points where the 4096 coarse cells start, beyond a histogram for 4096 points (256 at most) and the cells' totals. A buffer holds every smaller batch."""
    from tiny_dpcpp_nn import _lib
    d = _lib.GridDesc()
    assert lib.tnn_grid_desc_init(ctypes.byref(d), 3, 16, 2, 19, 16, 1.447, 0, 1, 1, _lib.TNN_FP32) == 0
    sizes = [1, 16, 17, 4096, 4097, 8192, 8193, 12288, 12289, 2 ** 18, 2 ** 20, 2 ** 20 + 1, 2 ** 22]
    needs = [lib.tnn_grid_order_bytes(ctypes.byref(d), M) for M in sizes]
    assert needs == [(16 * M + 255) // 256 * 256 + 16384 * (1 if M <= 8192 else min(256, (M + 4095) // 4096) + 1) + 256 for M in sizes]
    assert needs == sorted(needs)


def test_workspace_of_8192_rows_of_width_128_holds_fewer(lib):
    """From 8192 rows on a workgroup takes 128 rows instead of 64 and leaves half as many partial sums."""
    from tiny_dpcpp_nn import _lib
    wide = _lib.MlpDesc(_lib.TNN_FP16, 128, 8, _lib.ACT_RELU, _lib.ACT_NONE)
    for query in (lib.tnn_mlp_backward_workspace_bytes, lib.tnn_mlp_train_step_workspace_bytes):
        sizes = [query(ctypes.byref(wide), m) for m in (4096, 8128, 8184, 8192, 8256, 16384)]
        assert sizes == sorted(sizes)


@pytest.mark.parametrize("width,hidden", [(16, 9), (32, 2), (64, 4), (64, 9), (128, 1), (128, 8)])
def test_workspace_of_a_batch_holds_fewer_rows(lib, width, hidden):
    """The partial sums become fewer where a workgroup takes 64 rows more: behind 16384, 32768, ... rows."""
    from tiny_dpcpp_nn import _lib
    desc = _lib.MlpDesc(_lib.TNN_FP16, width, hidden, _lib.ACT_RELU, _lib.ACT_NONE)
    rows = sorted({8, 64, 4096, 24576, 200000} | {k * 8192 + e for k in range(1, 33) for e in (-8, 0, 8)})
    for query in (lib.tnn_mlp_backward_workspace_bytes, lib.tnn_mlp_train_step_workspace_bytes):
        sizes = [query(ctypes.byref(desc), m) for m in rows]
        assert sizes == sorted(sizes), [m for m, a, b in zip(rows, sizes, sizes[1:]) if b < a]
    if (width, hidden) == (128, 8):  # as many partial sums as there are: 128 of nine matrices, and nine of deltas
        assert lib.tnn_mlp_backward_workspace_bytes(ctypes.byref(desc), 16384) == 9 * 128 * 128 * 4 * 128 + 9 * 16384 * 128 * 2 + 512


@pytest.mark.parametrize("dims,features,levels,scale,log2,sides", [
    # the sizes on both sides of each rule of tnn_grid_forward_workspace_bytes: (points, whether by levels)
    (2, 2, 8, 1.5, 19, ((2 ** 14, 0), (2 ** 14 + 1, 0), (2 ** 17, 0), (2 ** 18 - 1, 0), (2 ** 18, 1), (2 ** 19 - 1, 1), (2 ** 19, 0))),
    (2, 2, 8, 2.0, 19, ((2 ** 16, 0), (2 ** 16 + 1, 1), (2 ** 18, 1))),
    (2, 2, 12, 1.5, 14, ((2 ** 15, 0), (2 ** 18 - 1, 0), (2 ** 18, 1), (3 * 2 ** 17 - 1, 1), (3 * 2 ** 17, 0))),
    (2, 2, 12, 1.5, 19, ((2 ** 14, 0), (2 ** 14 + 1, 1), (2 ** 18, 1), (3 * 2 ** 17, 0))),
    (2, 2, 12, 2.0, 19, ((3 * 2 ** 17, 1), (2 ** 19 - 1, 1), (2 ** 19, 0))),
    (2, 2, 13, 1.5, 14, ((2 ** 14 + 1, 1),)), (2, 2, 16, 1.3, 19, ((3 * 2 ** 17 - 1, 1), (3 * 2 ** 17, 0))), (2, 2, 16, 1.5, 19, ((2 ** 14 + 1, 1), (2 ** 19 - 1, 1), (2 ** 19, 0))),
    (2, 2, 16, 1.5, 22, ((2 ** 14 + 1, 1), (2 ** 15 - 1, 1), (2 ** 15, 0))), (2, 8, 16, 1.447, 14, ((2 ** 15, 1), (2 ** 15 + 1, 0), (2 ** 18, 0))), (2, 8, 8, 1.447, 14, ((2 ** 15, 0),)),
    (3, 2, 8, 1.447, 14, ((2 ** 14 + 1, 0), (2 ** 16, 0), (2 ** 16 + 1, 1), (7 * 2 ** 16 - 1, 1), (7 * 2 ** 16, 0))),
    (3, 2, 8, 1.447, 17, ((2 ** 14 + 1, 1), (7 * 2 ** 16, 0))), (3, 2, 8, 2.0, 17, ((7 * 2 ** 16, 1), (2 ** 20, 1))),
    (3, 2, 4, 1.447, 19, ((2 ** 16, 0), (2 ** 18 - 1, 0), (2 ** 18, 1), (7 * 2 ** 16, 0))), (3, 2, 16, 1.447, 19, ((2 ** 14, 0), (2 ** 14 + 1, 1), (2 ** 20, 1), (2 ** 24, 1))),
    (3, 2, 16, 1.447, 22, ((2 ** 17 - 1, 1), (2 ** 17, 0))), (3, 2, 12, 1.447, 22, ((2 ** 16 - 1, 1), (2 ** 16, 0))), (3, 2, 16, 1.447, 21, ((7 * 2 ** 16 - 1, 1), (7 * 2 ** 16, 0))),
    (3, 8, 16, 1.447, 19, ((2 ** 15, 1), (2 ** 15 + 1, 0), (2 ** 16, 0), (2 ** 16 + 1, 1), (2 ** 18, 0))), (3, 8, 8, 1.447, 19, ((2 ** 17, 0),))])
def test_encodings_go_by_level_where_that_was_measured_to_be_faster(lib, dims, features, levels, scale, log2, sides):
    from tiny_dpcpp_nn import _lib
    d = _lib.GridDesc()
    assert lib.tnn_grid_desc_init(ctypes.byref(d), dims, levels, features, log2, 16, scale, 0, 1, 1, _lib.TNN_FP32) == 0
    for M, by_level in sides:
        need = (levels * features + 15) // 16 * 16 * 4 * ((M + 63) // 64 * 64) + 256
        assert lib.tnn_grid_forward_workspace_bytes(ctypes.byref(d), _lib.TNN_FP32, M) == by_level * need, M


@pytest.mark.parametrize("dims,features,levels,log2,width,sides", [
    # on both sides of each rule of tnn_grid_mlp_width_wants_levels: (points, whether by levels)
    (3, 2, 1, 14, 128, ((1, 1), (2 ** 21, 1))), (3, 4, 1, 14, 128, ((1, 0),)), (2, 1, 1, 14, 128, ((1, 1),)), (2, 2, 8, 14, 128, ((2 ** 14, 0),)), (2, 2, 11, 14, 128, ((2 ** 14, 1), (2 ** 18 - 1, 1))),
    (3, 1, 1, 14, 64, ((1, 1),)), (2, 1, 8, 14, 64, ((1, 0),)), (3, 1, 8, 14, 32, ((1, 0),)), (2, 4, 9, 14, 64, ((2 ** 18, 1),)), (2, 4, 10, 14, 64, ((2 ** 18, 0),)),
    (2, 2, 8, 14, 64, ((2 ** 18 - 1, 0), (2 ** 18, 1), (2 ** 20, 1), (2 ** 20 + 1, 0))), (2, 2, 16, 20, 64, ((2 ** 18, 1), (2 ** 19 - 1, 1), (2 ** 19, 0))), (2, 2, 16, 21, 64, ((2 ** 18, 0),)),
    (3, 2, 11, 14, 32, ((2 ** 15 - 1, 1),)), (3, 1, 11, 14, 16, ((2 ** 15 - 1, 0), (2 ** 18, 1))), (3, 4, 11, 14, 64, ((23999, 1), (24000, 0))), (3, 2, 11, 20, 32, ((2 ** 15 - 1, 1), (2 ** 17, 1))),
    (3, 2, 11, 21, 32, ((23999, 1), (24000, 0), (2 ** 20, 0))), (3, 2, 8, 16, 16, ((2 ** 18 - 1, 0), (2 ** 18, 1))), (3, 2, 8, 18, 16, ((2 ** 18, 0),)), (3, 8, 6, 14, 64, ((2 ** 18, 1), (2 ** 19, 0))),
    (3, 8, 7, 14, 64, ((2 ** 18, 0),)), (3, 4, 4, 14, 64, ((2 ** 18 - 1, 0), (2 ** 19, 1))), (3, 4, 5, 14, 64, ((2 ** 19, 0),)), (3, 2, 8, 14, 64, ((2 ** 16 - 1, 0), (2 ** 16, 1))),
    (3, 2, 2, 14, 64, ((2 ** 17 - 1, 0), (2 ** 17, 1))), (3, 2, 8, 14, 32, ((2 ** 18 - 1, 0), (2 ** 18, 1)))])
def test_networks_go_by_level_where_that_was_measured_to_be_faster(lib, dims, features, levels, log2, width, sides):
    from tiny_dpcpp_nn import _lib
    d = _lib.GridDesc()
    assert lib.tnn_grid_desc_init(ctypes.byref(d), dims, levels, features, log2, 16, 2.0, 0, 1, 1, _lib.TNN_FP32) == 0
    for M, by_level in sides:
        assert lib.tnn_grid_mlp_width_wants_levels(ctypes.byref(d), width, M) == by_level, M
        assert width != 64 or lib.tnn_grid_mlp_wants_levels(ctypes.byref(d), M) == by_level
    assert lib.tnn_grid_mlp_width_wants_levels(ctypes.byref(d), width, 0) == 0


@pytest.mark.parametrize("features,levels,log2,base,scale,width,beyond", [
    # 3-D, levels of more than 8 MB: whether by levels beyond 2^20 points
    (2, 16, 22, 16, 1.447, 64, 1), (2, 3, 22, 64, 2.0, 64, 1), (2, 3, 22, 64, 2.0, 32, 1), (2, 1, 22, 256, 2.0, 32, 1),  # two features, width 32 and more: all;
    (2, 7, 22, 16, 2.0, 16, 1), (2, 6, 22, 16, 2.0, 16, 0), (2, 2, 22, 256, 2.0, 16, 0), (2, 3, 22, 256, 2.0, 16, 1), (2, 1, 22, 128, 2.0, 16, 0),  # at width 16 and of one feature by how many are
    (1, 7, 22, 16, 2.0, 32, 1), (1, 6, 22, 16, 2.0, 32, 0), (1, 7, 22, 16, 2.0, 16, 1), (1, 6, 22, 16, 2.0, 16, 0), (4, 8, 21, 16, 2.0, 64, 0), (4, 4, 20, 64, 2.0, 16, 0)])  # as large as the largest
def test_large_fields_go_by_level_where_that_was_measured_to_be_faster(lib, features, levels, log2, base, scale, width, beyond):
    from tiny_dpcpp_nn import _lib
    d = _lib.GridDesc()
    assert lib.tnn_grid_desc_init(ctypes.byref(d), 3, levels, features, log2, base, scale, 0, 1, 1, _lib.TNN_FP32) == 0
    assert max(d.offsets[l + 1] - d.offsets[l] for l in range(levels)) * features * 4 > 2 ** 23
    assert [lib.tnn_grid_mlp_width_wants_levels(ctypes.byref(d), width, M) for M in (2 ** 18, 2 ** 20, 2 ** 20 + 1, 2 ** 22)] == [0, 0, beyond, beyond]
