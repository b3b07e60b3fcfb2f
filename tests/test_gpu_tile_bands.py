"""GPU parity: the MFMA tile kernel on matrices wide enough that it goes through their column blocks in bands."""
import numpy as np
import pytest

from helpers import REL_L2_TOL, rel_l2, to_dev, to_host

pytestmark = pytest.mark.gpu


# The narrowest matrices that have bands (128 column blocks), whole bands and a last one of 8, 16 and 24; three row groups and more; ragged rows and columns; one and two strips
# per wave, one K set and two; both sides of the line.
@pytest.mark.parametrize(
    "m,n,k,grid",
    [(129, 128 * 128, 256, (128, 5)), (129, 128 * 120, 256, (120, 5)), (385, 128 * 128 - 127, 128, (128, 7)), (257, 128 * 136, 256, (136, 9)), (321, 128 * 144 - 70, 256, (144, 6)), (500, 128 * 152, 128, (152, 8)),
     (70, 128 * 168, 512, (168, 3)), (192, 128 * 128, 1024, (128, 6)), (100, 128 * 136, 256, (136, 2))],
)
def test_bands(q8, oracle, m, n, k, grid):
    p = q8.plan_mul_mat(m, n, k)
    assert p["kernel"] == "gemm_tile" and p["grid"] == grid and p["k_splits"] == 1 and p["order"] == ("bands_of_32" if grid[0] >= 128 and grid[1] > 2 else "grid"), p
    w = oracle.fill_weights(m + n, n, k)
    x = oracle.fill_activations(m + k, m * k).reshape(m, k)
    aq = oracle.quantize_rows(x)
    want = oracle.gemm(w, aq, m, n, k, threads=8) if (k // 32) % 16 == 0 else oracle.gemm(w, aq, m, n, k)
    wt, at = q8.tile(to_dev(w), n, k), q8.quantize_row_q8_0(to_dev(x), tiled=True)
    got = to_host(q8.gemm(wt, at, m, n, k, tiled=True))
    for i in range(m):
        assert rel_l2(got[i], want[i]) <= REL_L2_TOL, i


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
