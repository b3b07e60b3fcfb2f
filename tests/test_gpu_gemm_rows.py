"""GPU parity: the streaming MFMA kernel for up to 32 quantized rows, and its fused gate / up form, at the edges of its tiles."""
import numpy as np
import pytest

from helpers import REL_L2_TOL, rel_l2, to_dev, to_host

pytestmark = pytest.mark.gpu


def _gemm(oracle, w, aq, m, n, k):  # the threaded checker takes block counts that are multiples of 16
    return oracle.gemm(w, aq, m, n, k, threads=8) if (k // 32) % 16 == 0 else oracle.gemm(w, aq, m, n, k)


# rows at either side of the 8-, 16- and 32-row operands; N with a ragged last strip; K of one group, fewer groups than waves, a last chunk
# of one group, and long enough for two and four workgroups per strip
@pytest.mark.parametrize("m", [1, 2, 8, 9, 16, 17, 31, 32])
# ... and for two sets of shares per workgroup (129 to 255 strips, or more than 128 groups), evenly shared and not
@pytest.mark.parametrize("n,k", [(33, 128), (100, 128 * 7), (8200, 128 * 17), (257, 128 * 35), (1024, 4096), (4096, 128 * 21), (4100, 4096), (5120, 128 * 37), (8200, 128 * 131)])
def test_gemm_rows(q8, oracle, m, n, k):
    assert q8.plan_mul_mat(m, n, k)["gemm_rows"]
    w = oracle.fill_weights(m + n, n, k)
    x = oracle.fill_activations(m + k, m * k).reshape(m, k)
    aq = oracle.quantize_rows(x)
    want = _gemm(oracle, w, aq, m, n, k)
    wt, at = q8.tile(to_dev(w), n, k), q8.quantize_row_q8_0(to_dev(x), tiled=True)
    got = to_host(q8.gemm(wt, at, m, n, k, tiled=True))
    for i in range(m):
        assert rel_l2(got[i], want[i]) <= REL_L2_TOL, i
    res = oracle.fill_activations(5, m * n).reshape(m, n)
    acc = to_dev(res.copy())
    q8.gemm_residual(wt, at, acc, m, n, k, out=acc)
    assert np.array_equal(to_host(acc), got + res)  # one fp32 add after the sum, in place; the sum itself is bit-stable


# [2 x n_ff x k] with a strip's K uncut (>= 129 strips, or a short K), several chunks per wave and ragged rows
@pytest.mark.parametrize("m", [1, 8, 11, 16, 23, 32])
@pytest.mark.parametrize("n_ff,k", [(128, 128), (4224, 128 * 9), (8192, 2048), (4224, 128 * 34)])
def test_gate_up_rows(q8, oracle, m, n_ff, k):
    lib = q8._lib.lib()
    assert lib.nh_q8_0_gate_up_silu_workspace_bytes(m, n_ff, k) == 0
    wg, wu = oracle.fill_weights(1 + m, n_ff, k), oracle.fill_weights(2 + m, n_ff, k)
    x = oracle.fill_activations(m + k, m * k).reshape(m, k)
    aq = oracle.quantize_rows(x)
    tg, tu = q8.tile(to_dev(wg), n_ff, k), q8.tile(to_dev(wu), n_ff, k)
    at = q8.quantize_row_q8_0(to_dev(x), tiled=True)
    act, gate, up = q8.gate_up_silu(tg, tu, at, m, n_ff, k, debug=True)
    gate, up = to_host(gate), to_host(up)
    assert rel_l2(gate, _gemm(oracle, wg, aq, m, n_ff, k)) <= REL_L2_TOL
    assert rel_l2(up, _gemm(oracle, wu, aq, m, n_ff, k)) <= REL_L2_TOL
    # the quantizer on the launch's own sums, byte for byte, and zero blocks in the rows past M
    whole = to_host(q8.untile(act, 32, n_ff)).reshape(32, -1)
    assert np.array_equal(whole[:m], oracle.silu_mul_quantize_rows(gate, up))
    assert not whole[m:].any()
    assert np.array_equal(to_host(q8.gate_up_silu(tg, tu, at, m, n_ff, k)), to_host(act))


# A captured call, whose hand-off cannot be the eager call's, runs the streaming kernel: the same sums in the same order, so the same bits.
# Two and four workgroups per strip, K shared unevenly, ragged strips; 100 strips with two sets of shares in each of two workgroups; and one workgroup.
@pytest.mark.parametrize("m", [3, 16, 17])
@pytest.mark.parametrize("n,k,splits,waves", [(4096, 4096, 2, 8), (1024, 4096, 4, 8), (257, 128 * 35, 4, 8), (4090, 128 * 21, 2, 8), (3200, 8192, 2, 16), (5120, 5120, 1, 16)])
def test_captured_and_eager_calls_have_the_same_bits(q8, oracle, m, n, k, splits, waves):
    import torch

    plan = q8.plan_mul_mat(17, n, k)  # (fewer rows would report the kernel that mul_mat quantizes in)
    assert plan["kernel"] == "gemm_skinny" and (plan["k_splits"], plan["waves"]) == (splits, waves) and q8.plan_mul_mat(m, n, k)["gemm_rows"]
    wt = q8.tile(q8.fill_weight_blocks(n + m, n, k), n, k)
    xs = [q8.fill_activations(30 + i, m * k).reshape(m, k) for i in range(3)]
    at = q8.quantize_row_q8_0(xs[0], tiled=True)
    c = torch.empty((m, n), dtype=torch.float32, device="cuda")
    q8._lib.check("nh_q8_0_prepare", q8._lib.lib().nh_q8_0_prepare())
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        q8._lib.check("gemm", q8._lib.lib().nh_q8_0_gemm_tiled(wt.data_ptr(), at.data_ptr(), c.data_ptr(), m, n, k, torch.cuda.current_stream().cuda_stream))
    for x in xs:
        at.copy_(q8.quantize_row_q8_0(x, tiled=True))
        c.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(to_host(c).view(np.uint32), to_host(q8.gemm(wt, at, m, n, k, tiled=True)).view(np.uint32))


def test_gemm_rows_in_a_graph(q8, oracle):
    # a captured launch takes no form whose hand-off is tagged by a number that a replay could not renew
    import torch

    m, n, k = 12, 1024, 4096
    w = oracle.fill_weights(3, n, k)
    wt = q8.tile(to_dev(w), n, k)
    xs = [oracle.fill_activations(20 + i, m * k).reshape(m, k) for i in range(3)]
    at = q8.quantize_row_q8_0(to_dev(xs[0]), tiled=True)
    lib, c = q8._lib.lib(), torch.empty((m, n), dtype=torch.float32, device="cuda")
    q8._lib.check("nh_q8_0_prepare", lib.nh_q8_0_prepare())
    q8.gemm(wt, at, m, n, k, tiled=True)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        q8._lib.check("gemm", lib.nh_q8_0_gemm_tiled(wt.data_ptr(), at.data_ptr(), c.data_ptr(), m, n, k, torch.cuda.current_stream().cuda_stream))
    for x in xs:
        at.copy_(q8.quantize_row_q8_0(to_dev(x), tiled=True))
        graph.replay()
        torch.cuda.synchronize()
        eager = to_host(q8.gemm(wt, at, m, n, k, tiled=True))
        assert rel_l2(to_host(c), eager) < 2e-6
        assert rel_l2(eager, oracle.gemm(w, oracle.quantize_rows(x), m, n, k, threads=8)) <= REL_L2_TOL


# 18 to 24 rows: the 24-row operand (its 48 (k half, row) units do not divide a transfer), at its edges and the edges of the other sizes
@pytest.mark.parametrize("m", [18, 24, 25])
@pytest.mark.parametrize("n,k", [(33, 128), (257, 128 * 35), (4100, 4096), (5120, 128 * 37)])
def test_the_24_row_operand(q8, oracle, m, n, k):
    test_gemm_rows(q8, oracle, m, n, k)


@pytest.mark.parametrize("n_ff,k", [(128, 128), (4224, 128 * 9), (4224, 128 * 34)])
def test_gate_up_of_24_rows(q8, oracle, n_ff, k):
    test_gate_up_rows(q8, oracle, 24, n_ff, k)


# 17 to 32 rows against 64 to 191 column blocks and 64 Mi weights and more: as many shares of K as the tile kernel, which had these shapes,
# where those are sixteen in two sets of eight waves' (or, captured, sixteen waves of the streaming kernel: the same bits); between 257 and 447 strips still the tile kernel
@pytest.mark.parametrize("m", [17, 24, 32])
@pytest.mark.parametrize("n,k,waves", [(8161, 10240, 16), (16384, 4096, 8)])
def test_rows_kernel_in_the_tile_kernels_place(q8, oracle, m, n, k, waves):
    plan = q8.plan_mul_mat(m, n, k)
    assert plan["kernel"] == "gemm_skinny" and plan["gemm_rows"] and (plan["k_splits"], plan["waves"]) == (1, waves)
    assert q8.plan_mul_mat(m, 10240, 8192)["kernel"] == "gemm_tile_stream" and q8.plan_mul_mat(33, n, k)["kernel"] != "gemm_skinny"
    w = oracle.fill_weights(m + n, n, k)
    x = oracle.fill_activations(m + k, m * k).reshape(m, k)
    want = _gemm(oracle, w, oracle.quantize_rows(x), m, n, k)
    got = to_host(q8.mul_mat(q8.tile(to_dev(w), n, k), to_dev(x), n, k))
    assert max(rel_l2(got[i], want[i]) for i in range(m)) <= REL_L2_TOL


@pytest.mark.parametrize("m", [20, 32])
def test_captured_call_in_the_tile_kernels_place(q8, oracle, m):
    test_captured_and_eager_calls_have_the_same_bits(q8, oracle, m, 8161, 10240, splits=1, waves=16)
