"""The passes on a caller's own rows: row counts, column counts and types where padding, conversion and scaling inside the kernels can
go wrong, against the passes on whole matrices (which the oracle tests cover)."""
import ctypes

import numpy as np
import pytest
import torch

from tolerances import BF16, FP16, FP32

pytestmark = pytest.mark.gpu
DT = {FP32: torch.float32, FP16: torch.float16, BF16: torch.bfloat16}


def p(t):
    return ctypes.c_void_p(t.data_ptr()) if t is not None else None


def network(tnn, oracle, dtype, W, hidden, out_act="none"):
    rng = np.random.default_rng(W + hidden)
    desc = tnn.mlp_desc(dtype, W, hidden, "relu", out_act)
    w = oracle.round(rng.uniform(-1, 1, (hidden + 1, W, W)) * np.sqrt(3.0 / W), dtype)
    return desc, tnn.prepare(desc, w)


@pytest.mark.parametrize("dtype", [BF16, FP16])
@pytest.mark.parametrize("W,hidden", [(16, 2), (32, 4), (64, 4), (128, 3), (128, 8)])
@pytest.mark.parametrize("M,x_cols,y_cols,x_fp32", [(1, 1, 1, True), (31, 3, 3, True), (33, 16, 16, False), (100, 8, 9, True), (70001, 5, 4, False), (66000, 0, 0, False)])
def test_inference_rows(tnn, oracle, dtype, W, hidden, M, x_cols, y_cols, x_fp32):
    from tiny_dpcpp_nn import _lib
    desc, (_, fwd, _) = network(tnn, oracle, dtype, W, hidden)
    x_cols, y_cols = x_cols or W, y_cols or W
    x = torch.rand((M, x_cols), device=tnn.dev) * 2 - 1
    x = x if x_fp32 else x.to(DT[dtype])
    y = torch.full((M, y_cols), float("nan"), dtype=DT[dtype], device=tnn.dev)
    whole = torch.full((-(-M // 8) * 8, W), 0.5, dtype=DT[dtype], device=tnn.dev)
    whole[:M, :x_cols] = x.to(DT[dtype])
    ref = tnn.inference(desc, fwd, whole)[:M, :y_cols]
    rc = tnn.lib.tnn_mlp_inference_rows(ctypes.byref(desc), p(fwd), p(x), FP32 if x_fp32 else dtype, x_cols, 0.5, p(y), y_cols, M, tnn.stream())
    if rc == _lib.TNN_ERR_UNSUPPORTED:  # the width-128 kernel that takes whole rows
        assert W == 128 and (hidden == 8 or M >= 65536)
        padded = torch.empty((M, W), dtype=DT[dtype], device=tnn.dev)
        _lib.check(tnn.lib.tnn_resize_rows(dtype, p(padded), W, M, FP32 if x_fp32 else dtype, p(x), x_cols, x_cols, 1, M, 0.5, 1.0, tnn.stream()))
        rc = tnn.lib.tnn_mlp_inference_rows(ctypes.byref(desc), p(fwd), p(padded), dtype, W, 0.0, p(y), y_cols, M, tnn.stream())
    _lib.check(rc)
    assert torch.equal(y.view(torch.int16), ref.contiguous().view(torch.int16))


@pytest.mark.parametrize("src,dst", [(FP32, BF16), (BF16, FP32), (FP16, FP16)])
@pytest.mark.parametrize("rows,cols,to_rows,to_cols", [(5, 3, 8, 16), (1, 64, 1, 64), (1000, 64, 1000, 7), (33, 17, 40, 32)])
def test_resize_rows(tnn, src, dst, rows, cols, to_rows, to_cols):
    from tiny_dpcpp_nn import _lib
    x = (torch.rand((rows, cols, 2), device=tnn.dev) - 0.5).to(DT[src])[:, :, 0]  # strided columns
    out = torch.empty((to_rows, to_cols), dtype=DT[dst], device=tnn.dev)
    _lib.check(tnn.lib.tnn_resize_rows(dst, p(out), to_cols, to_rows, src, p(x), cols, x.stride(0), x.stride(1), rows, 0.25, 128.0, tnn.stream()))
    ref = torch.full((to_rows, to_cols), 0.25, device=tnn.dev)
    ref[:, :cols] = 0
    ref[:rows, : min(cols, to_cols)] = (x.float() * 128.0)[:, :to_cols]
    assert torch.equal(out, ref.to(DT[dst]))


@pytest.mark.parametrize("dtype", [BF16, FP16])
@pytest.mark.parametrize("W,hidden,M,dy_cols", [(16, 2, 5, 16), (32, 4, 5001, 3), (64, 2, 257, 16), (64, 4, 70003, 1), (64, 4, 4099, 64), (128, 3, 1001, 128), (128, 8, 300, 128)])
def test_backward_rows(tnn, oracle, dtype, W, hidden, M, dy_cols):
    """Scales are powers of two: dL/dx equals the unscaled pass bit for bit where nothing underflows, weight gradients to fp32 sums in the same order."""
    from tiny_dpcpp_nn import _lib
    desc, (_, fwd, bwd) = network(tnn, oracle, dtype, W, hidden)
    n_mats, padded = hidden + 1, -(-M // 8) * 8
    x = torch.zeros((padded, W), dtype=DT[dtype], device=tnn.dev)
    x[:M] = (torch.rand((M, W), device=tnn.dev) * 2 - 1).to(DT[dtype])
    dy = (torch.randn((M, dy_cols), device=tnn.dev) * 0.1).to(DT[dtype])
    whole = torch.zeros((padded, W), dtype=DT[dtype], device=tnn.dev)
    whole[:M, :dy_cols] = dy
    packed = torch.full((n_mats * W * W,), float("nan"), device=tnn.dev)
    dx = torch.full((M, W), float("nan"), dtype=DT[dtype], device=tnn.dev)
    if W == 128:
        interm = tnn.forward(desc, fwd, x)
        _, dW, dX = tnn.backward(desc, bwd, whole, interm, want_interm=False)
        hid = torch.empty((hidden, M, W), dtype=DT[dtype], device=tnn.dev)
        y = torch.empty((M, 5), dtype=DT[dtype], device=tnn.dev)
        _lib.check(tnn.lib.tnn_mlp_forward_rows(ctypes.byref(desc), p(fwd), p(x), p(hid), p(y), 5, M, tnn.stream()))
        assert torch.equal(y, interm[-1][:M, :5]) and torch.equal(hid, interm[1:-1, :M])
        need = tnn.lib.tnn_mlp_backward_workspace_bytes(ctypes.byref(desc), M)
        ws = torch.empty(need, dtype=torch.uint8, device=tnn.dev)
        _lib.check(tnn.lib.tnn_mlp_backward_rows(ctypes.byref(desc), p(bwd), p(x), p(hid), None, p(dy), 4.0, 0.25, p(packed), FP32, p(dx), M, p(ws), need, tnn.stream()))
    else:
        dW, dX = tnn.backward_recompute(desc, fwd, bwd, x, whole, dw_fp32=False)
        need = tnn.lib.tnn_mlp_train_step_workspace_bytes(ctypes.byref(desc), M)
        ws = torch.empty(need, dtype=torch.uint8, device=tnn.dev)
        _lib.check(tnn.lib.tnn_mlp_backward_recompute_rows(ctypes.byref(desc), p(fwd), p(bwd), p(x), p(dy), dy_cols, 4.0, 0.25, p(packed), FP32, p(dx), M,
                                                           p(ws), need, tnn.stream()))
    ref = torch.empty((n_mats, W, W), dtype=DT[dtype], device=tnn.dev)
    _lib.check(tnn.lib.tnn_pack_and_transpose(dtype, W, n_mats, p(dW.contiguous()), p(ref), tnn.stream()))
    ref = ref.float().reshape(-1)
    step = 2.0 ** (-8 if dtype == BF16 else -10)  # one rounding of a sum taken from values four times as large
    assert float((packed - ref).abs().max()) <= 2 * step * float(ref.abs().max())
    assert float((dx.float() - dX[:M].float()).norm()) <= step * float(dX.float().norm())


@pytest.mark.parametrize("dtype", [BF16, FP16])
@pytest.mark.parametrize("W,hidden,n_in,n_out,bias,M", [(16, 2, 16, 16, 0, 31), (32, 4, 5, 7, 1, 9001), (64, 4, 64, 64, 0, 70001), (64, 18, 3, 1, 1, 500), (64, 2, 40, 16, 1, 2 ** 18),
                                                        (128, 2, 100, 128, 0, 3000)])
def test_push_and_inference_in_one_launch(tnn, dtype, W, hidden, n_in, n_out, bias, M):
    """The copies that a push leaves and the pass on them, bit for bit those of the two calls: few workgroups (others write the copies), many
    (those that compute do), depths whose weights do not fit LDS, padding weights."""
    from tiny_dpcpp_nn import _lib
    desc = tnn.mlp_desc(dtype, W, hidden, "relu", "none")
    n = (hidden + 1) * W * W
    nb = tnn.lib.tnn_mlp_prepared_bytes(ctypes.byref(desc)) // 2
    params = torch.randn(n, device=tnn.dev) * W ** -0.5
    sizes = (n, n, nb, nb)
    one, two = ([torch.full((k,), 7.0, dtype=DT[dtype], device=tnn.dev) for k in sizes] for _ in range(2))
    x = torch.rand((M, n_in), device=tnn.dev)
    if W == 128:
        x = torch.nn.functional.pad(x, [0, W - n_in], value=float(bias)).to(DT[dtype])
    xd, xc = (FP32, n_in) if W < 128 else (dtype, W)
    y1, y2 = (torch.empty((M, n_out), dtype=DT[dtype], device=tnn.dev) for _ in range(2))
    _lib.check(tnn.lib.tnn_mlp_push_inference_rows(ctypes.byref(desc), p(params), n_in, n_out, bias, *[p(t) for t in one], p(x), xd, xc, float(bias), p(y1), n_out, M,
                                                   tnn.stream()))
    _lib.check(tnn.lib.tnn_mlp_set_packed_weights(ctypes.byref(desc), p(params), FP32, n_in, n_out, bias, *[p(t) for t in two], tnn.stream()))
    _lib.check(tnn.lib.tnn_mlp_inference_rows(ctypes.byref(desc), p(two[2]), p(x), xd, xc, float(bias), p(y2), n_out, M, tnn.stream()))
    for a, b in zip(one + [y1], two + [y2]):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))


@pytest.mark.parametrize("M", [40, 20000])
def test_grid_push_and_inference_in_one_launch(tnn, M):
    from tiny_dpcpp_nn import _lib
    d = tnn.grid_desc(dict(n_dims=2, n_levels=16, n_features_per_level=2, log2_hashmap_size=12, base_resolution=16, per_level_scale=1.5))
    desc = tnn.mlp_desc(BF16, 64, 2, "relu", "none")
    n, nb = 3 * 64 * 64, tnn.lib.tnn_mlp_prepared_bytes(ctypes.byref(desc)) // 2
    params, table, x = torch.randn(n, device=tnn.dev) * 0.1, torch.randn(tnn.grid_n_params(d), device=tnn.dev), torch.rand((M, 2), device=tnn.dev)
    one, two = ([torch.full((k,), 7.0, dtype=torch.bfloat16, device=tnn.dev) for k in (n, n, nb, nb)] for _ in range(2))
    y1, y2 = (torch.empty((M, 3), dtype=torch.bfloat16, device=tnn.dev) for _ in range(2))
    g, m = ctypes.byref(d), ctypes.byref(desc)
    _lib.check(tnn.lib.tnn_grid_mlp_push_inference_rows(g, m, p(params), 64, 3, 0, *[p(t) for t in one], p(x), None, p(table), p(y1), 3, M, tnn.stream()))
    _lib.check(tnn.lib.tnn_mlp_set_packed_weights(m, p(params), FP32, 64, 3, 0, *[p(t) for t in two], tnn.stream()))
    _lib.check(tnn.lib.tnn_grid_mlp_inference_rows(g, m, p(x), None, p(table), p(two[2]), p(y2), 3, M, tnn.stream()))
    for a, b in zip(one + [y1], two + [y2]):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))
