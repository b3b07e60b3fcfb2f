"""GPU: which calls of nh_q8_0_mul_mat write the caller's workspace, and that the form which may write it gives the same values."""
import numpy as np
import pytest
import torch

from helpers import rel_l2, to_dev, to_host

pytestmark = pytest.mark.gpu


# (m, n, k, untouched): the edges of 16 rows, 40 MB and (4 rows) 80 MB, and shapes that run as two launches where the workspace is the call's own
@pytest.mark.parametrize("m,n,k,untouched", [(4, 1024, 4096, True), (16, 4096, 8192, True), (9, 4128, 4096, True), (16, 28672, 1024, True), (13, 9000, 2048, True), (8, 8192, 4096, True), (7, 1037, 16640, True),
                                             (16, 9634, 4096, True), (16, 9639, 4096, False), (4, 19269, 4096, True), (4, 19281, 4096, False), (17, 1024, 4096, False)])
def test_the_workspace_is_left_alone_where_promised(q8, m, n, k, untouched):
    assert q8.plan_mul_mat(m, n, k, own_workspace=True)["quantize_launch"] != untouched
    lib = q8._lib.lib()
    w = q8.tile(q8.fill_weight_blocks(m, n, k), n, k)
    x, res = q8.fill_activations(n, m * k).reshape(m, k), q8.fill_activations(k, m * n).reshape(m, n)
    need = lib.nh_q8_0_mul_mat_workspace_bytes(m, k)
    pattern = torch.arange(need, device="cuda").to(torch.uint8)
    want = to_host(q8.mul_mat(w, x, n, k))
    for add in (None, res):
        ws = pattern.clone()
        y = to_host(q8.mul_mat(w, x, n, k, workspace=ws, residual=add))
        assert torch.equal(ws, pattern) == untouched
        assert rel_l2(y if add is None else y - to_host(res), want) <= 2e-6
    op = (q8._lib.MulMatOp * 1)(q8._lib.MulMatOp(w.data_ptr(), x.data_ptr(), res.data_ptr(), m, n, k, 0, 0))
    ws = pattern.clone()
    q8._lib.check("batch", lib.nh_q8_0_mul_mat_batch(op, 1, ws.data_ptr(), need, torch.cuda.current_stream().cuda_stream))
    assert torch.equal(ws, pattern) == untouched and rel_l2(to_host(res), want) <= 2e-6


@pytest.mark.parametrize("m,n,k", [(16, 1024, 28672), (8, 2500, 11008), (16, 28672, 1024)])
def test_a_captured_call_needs_no_hand_off(q8, oracle, m, n, k):
    # a shape whose two launches hand K parts over is captured as the form that does not; one that has no K parts gives the eager bits
    split = q8.plan_mul_mat(m, n, k)["k_splits"] > 1
    wb, xb = oracle.fill_weights(m + n, n, k), oracle.fill_activations(m + k, m * k).reshape(m, k)
    w, x = q8.tile(to_dev(wb), n, k), to_dev(xb)
    q8._lib.check("nh_q8_0_prepare", q8._lib.lib().nh_q8_0_prepare())
    ws = torch.empty(q8._lib.lib().nh_q8_0_mul_mat_workspace_bytes(m, k), dtype=torch.uint8, device="cuda")
    eager, kept = to_host(q8.mul_mat(w, x, n, k)), to_host(q8.mul_mat(w, x, n, k, workspace=ws))
    assert rel_l2(eager, kept) <= 2e-6
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = q8.mul_mat(w, x, n, k)
        z = q8.mul_mat(w, x, n, k, workspace=ws)
    for _ in range(2):
        y.zero_()
        z.zero_()
        graph.replay()
        torch.cuda.synchronize()
        got = to_host(y)
        assert rel_l2(got, eager) <= 2e-6
        assert np.array_equal(got.view(np.uint32), (to_host(z) if split else eager).view(np.uint32))
