"""GPU parity: the tile kernel with several K sets where K does not divide over them -- the sets' shares differ by a 128-quant group, and the
shorter ones walk their last trip with zero scales."""
import numpy as np
import pytest
import torch

from helpers import REL_L2_TOL, rel_l2, to_dev, to_host

pytestmark = pytest.mark.gpu


def _gemm(oracle, w, aq, m, n, k):  # the threaded checker takes block counts that are multiples of 16
    return oracle.gemm(w, aq, m, n, k, threads=8) if (k // 32) % 16 == 0 else oracle.gemm(w, aq, m, n, k)


# (m, n, groups, kernel, K sets, workgroups along K): two and four sets, one and two activation strips, streamed weights or not, ragged rows and
# columns, the fewest groups that are cut, and one, two and three sets with the longer share; then K over two and four workgroups as well
SHAPES = [(700, 1536, 13, "gemm_tile", 2, 1), (700, 1500, 17, "gemm_tile", 4, 1), (701, 1536, 42, "gemm_tile", 4, 1), (300, 3400, 19, "gemm_tile", 4, 1), (24, 24577, 9, "gemm_tile_stream", 2, 1),
          (40, 24577, 17, "gemm_tile_stream", 4, 1), (200, 4090, 47, "gemm_tile", 4, 2), (120, 3840, 104 + 1, "gemm_tile", 4, 4)]


@pytest.mark.parametrize("m,n,groups,kernel,sets,splits", SHAPES)
def test_uneven_k_sets(q8, oracle, m, n, groups, kernel, sets, splits):
    k = 128 * groups
    plan = q8.plan_mul_mat(m, n, k)
    assert (plan["kernel"], plan["k_sets"], plan["k_splits"]) == (kernel, sets, splits) and groups % (sets * splits)
    w, x = oracle.fill_weights(m + n, n, k), oracle.fill_activations(m + k, m * k).reshape(m, k)
    want = _gemm(oracle, w, oracle.quantize_rows(x), m, n, k)
    wt, at = q8.tile(to_dev(w), n, k), q8.quantize_row_q8_0(to_dev(x), tiled=True)
    got = to_host(q8.gemm(wt, at, m, n, k, tiled=True))
    assert max(rel_l2(got[i], want[i]) for i in range(m)) <= REL_L2_TOL
    acc = q8.fill_activations(5, m * n).reshape(m, n)
    res = to_host(acc).copy()
    q8.gemm_residual(wt, at, acc, m, n, k, out=acc)
    assert np.array_equal(to_host(acc), got + res)  # one fp32 add after the sum, in place; the sum itself is bit-stable
    if splits > 1 and m > 64:  # captured, the streaming kernel stands in: the same shares, added in the same order
        q8._lib.check("nh_q8_0_prepare", q8._lib.lib().nh_q8_0_prepare())
        c = torch.zeros((m, n), dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            q8._lib.check("gemm", q8._lib.lib().nh_q8_0_gemm_tiled(wt.data_ptr(), at.data_ptr(), c.data_ptr(), m, n, k, torch.cuda.current_stream().cuda_stream))
        for _ in range(2):
            c.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert np.array_equal(to_host(c).view(np.uint32), got.view(np.uint32))


def test_the_zero_scales_hide_an_infinity(q8, oracle):
    # the last trip of a shorter share multiplies its last group again, by zero scales on both sides: an infinite scale there stays in its own column
    m, n, k = 700, 1536, 128 * 13
    w_d, a_d = np.full((n, k // 32), 0x3C00, dtype=np.uint16), np.full((m, k // 32), 0x3C00, dtype=np.uint16)
    w_d[5, -1], w_d[9, 4 * 7 - 1], a_d[3, -1] = 0x7C00, 0xFC00, 0x7C00
    want = np.full((m, n), k, dtype=np.float32)
    want[3], want[:, 5], want[:, 9] = np.inf, np.inf, -np.inf
    want[3, 9] = np.nan  # inf - inf
    wt = q8.tile(to_dev(oracle.pack_blocks(w_d, np.ones((n, k // 32, 32), dtype=np.int8))), n, k)
    at = q8.tile(to_dev(oracle.pack_blocks(a_d, np.ones((m, k // 32, 32), dtype=np.int8))), m, k)
    assert np.array_equal(to_host(q8.gemm(wt, at, m, n, k, tiled=True)), want, equal_nan=True)


# the fused gate / up, (m, n_ff, groups, activation strips, K sets, passes): two sets in one pass, of one and two strips, streamed weights or not, and
# one set where the mat-mats have two uneven ones; four sets in two passes, and two in four
@pytest.mark.parametrize("m,n_ff,groups,strips,sets,passes", [(100, 11008, 33, 2, 2, 1), (48, 5504, 33, 2, 4, 2), (40, 5504, 21, 2, 4, 2), (24, 24576, 33, 1, 2, 1), (40, 24576, 33, 2, 2, 1), (24, 24576, 15, 1, 2, 1),
                                                              (40, 24576, 15, 2, 2, 1), (24, 33024, 9, 1, 1, 1), (58, 9216, 18, 2, 2, 4)])
def test_uneven_k_sets_of_gate_up(q8, oracle, m, n_ff, groups, strips, sets, passes):
    k = 128 * groups
    plan = q8.plan_gate_up_silu(m, n_ff, k)
    assert (plan["form"], plan["activation_strips"], plan["k_sets"], plan["passes"]) == ("tile", strips, sets, passes) and (groups % (sets * passes) or sets == 1)
    assert q8._lib.lib().nh_q8_0_gate_up_silu_workspace_bytes(m, n_ff, k) == 0
    wg, wu = oracle.fill_weights(1 + m, n_ff, k), oracle.fill_weights(2 + m, n_ff, k)
    x = oracle.fill_activations(m + k, m * k).reshape(m, k)
    aq = oracle.quantize_rows(x)
    tg, tu, at = q8.tile(to_dev(wg), n_ff, k), q8.tile(to_dev(wu), n_ff, k), q8.quantize_row_q8_0(to_dev(x), tiled=True)
    act, gate, up = q8.gate_up_silu(tg, tu, at, m, n_ff, k, debug=True)
    gate, up = to_host(gate), to_host(up)
    assert rel_l2(gate, _gemm(oracle, wg, aq, m, n_ff, k)) <= REL_L2_TOL and rel_l2(up, _gemm(oracle, wu, aq, m, n_ff, k)) <= REL_L2_TOL
    assert np.array_equal(to_host(q8.untile(act, m, n_ff)).reshape(m, -1), oracle.silu_mul_quantize_rows(gate, up))
    assert np.array_equal(to_host(q8.gate_up_silu(tg, tu, at, m, n_ff, k)), to_host(act))
