"""GPU parity: the MFMA tile kernel on matrices wide enough that it goes through their column blocks in bands, where the launch is large enough."""
import numpy as np
import pytest

from helpers import REL_L2_TOL, rel_l2, to_dev, to_host

pytestmark = pytest.mark.gpu


# As the grid has them: 120 column blocks and more, three row groups and more; ragged rows and columns; one and two strips per wave, one K set and two.
@pytest.mark.parametrize(
    "m,n,k,grid",
    [(129, 128 * 128, 256, (128, 5)), (129, 128 * 120, 256, (120, 5)), (385, 128 * 128 - 127, 128, (128, 7)), (257, 128 * 136, 256, (136, 9)), (321, 128 * 144 - 70, 256, (144, 6)), (500, 128 * 152, 128, (152, 8)),
     (70, 128 * 168, 512, (168, 3)), (192, 128 * 128, 1024, (128, 6)), (100, 128 * 136, 256, (136, 2))],
)
def test_wide_as_the_grid_has_it(q8, oracle, m, n, k, grid):
    p = q8.plan_mul_mat(m, n, k)
    assert p["kernel"] == "gemm_tile" and p["grid"] == grid and p["k_splits"] == 1 and p["order"] == "grid", p
    w = oracle.fill_weights(m + n, n, k)
    x = oracle.fill_activations(m + k, m * k).reshape(m, k)
    aq = oracle.quantize_rows(x)
    want = oracle.gemm(w, aq, m, n, k, threads=8) if (k // 32) % 16 == 0 else oracle.gemm(w, aq, m, n, k)
    wt, at = q8.tile(to_dev(w), n, k), q8.quantize_row_q8_0(to_dev(x), tiled=True)
    got = to_host(q8.gemm(wt, at, m, n, k, tiled=True))
    for i in range(m):
        assert rel_l2(got[i], want[i]) <= REL_L2_TOL, i


def edge_rows(m):
    return sorted({i for i in (0, 31, 32, 63, 64, 95, 96, 127, 128, 159, 160, 255, 256, m // 2, m - 2, m - 1) if i < m})


# In bands: whole ones (the narrowest matrix that has them, 128 column blocks) and a last one of 8, 16 and 24; one strip per wave and two, one K set and two; ragged rows and columns.
# The rows on both sides of the strips' and row groups' edges, all columns.
@pytest.mark.parametrize("m,n,k,cut", [(129, 128 * 128, 2432, (1, 1)), (140, 128 * 152 - 127, 2176, (1, 1)), (70, 128 * 168, 2048, (1, 2)), (500, 128 * 144 - 70, 2304, (2, 1)), (1030, 128 * 136, 1152, (2, 1))])
def test_bands(q8, oracle, m, n, k, cut):
    p = q8.plan_mul_mat(m, n, k)
    assert p["kernel"] == "gemm_tile" and p["order"] == "bands_of_32" and (p["activation_strips"], p["k_sets"]) == cut, p
    w = oracle.fill_weights(m + n, n, k)
    x = oracle.fill_activations(m + k, m * k).reshape(m, k)
    rows = edge_rows(m)
    aq = oracle.quantize_rows(x[rows])
    want = oracle.gemm(w, aq, len(rows), n, k, threads=8) if (k // 32) % 16 == 0 else oracle.gemm(w, aq, len(rows), n, k)
    got = q8.gemm(q8.tile(to_dev(w), n, k), q8.quantize_row_q8_0(to_dev(x), tiled=True), m, n, k, tiled=True)
    for i, row in enumerate(rows):
        assert rel_l2(to_host(got[row]), want[i]) <= REL_L2_TOL, row


# The fused gate/up launch: two row groups too; one K set, two, and two in passes.
@pytest.mark.parametrize("m,n_ff,k,grid", [(100, 8192, 1024, (128, 2)), (100, 8704, 2048, (136, 2)), (193, 8192, 1024, (128, 4)), (290, 9216, 256, (144, 5)), (161, 9728, 128, (152, 3)), (385, 8704, 256, (136, 13))])
def test_gate_up_bands(q8, oracle, m, n_ff, k, grid):
    p = q8.plan_gate_up_silu(m, n_ff, k)
    assert p["form"] == "tile" and p["grid"] == grid and p["order"] == "bands_of_32", p
    wg, wu = oracle.fill_weights(21 + m, n_ff, k), oracle.fill_weights(22 + m, n_ff, k)
    x = oracle.fill_activations(m + k, m * k).reshape(m, k)
    aq_cpu = oracle.quantize_rows(x)
    tg, tu = q8.tile(to_dev(wg), n_ff, k), q8.tile(to_dev(wu), n_ff, k)
    aq = q8.quantize_row_q8_0(to_dev(x), tiled=True)
    act, gate, up = q8.gate_up_silu(tg, tu, aq, m, n_ff, k, debug=True)
    gate, up = to_host(gate), to_host(up)
    for got, w in ((gate, wg), (up, wu)):
        want = oracle.gemm(w, aq_cpu, m, n_ff, k, threads=8) if (k // 32) % 16 == 0 else oracle.gemm(w, aq_cpu, m, n_ff, k)
        for i in range(m):
            assert rel_l2(got[i], want[i]) <= REL_L2_TOL, i
    padded = (m + 31) // 32 * 32
    whole = to_host(q8.untile(act, padded, n_ff)).reshape(padded, -1)
    assert np.array_equal(whole[:m], oracle.silu_mul_quantize_rows(gate, up)) and not whole[m:].any()
