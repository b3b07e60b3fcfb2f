"""GPU parity: the MFMA tile kernel with one activation strip per wave, where two would leave the last round of workgroups mostly idle."""
import numpy as np
import pytest

from helpers import REL_L2_TOL, rel_l2, to_dev, to_host

pytestmark = pytest.mark.gpu


# Both sides of the lines: workgroups of two strips just over one round and two, of one strip up to three and five (with two sets of K there, from 24 groups and above four rounds on); three strips, four and five; a last strip of one row, ragged
# columns, a number of column blocks that eight divides and others; one K set and two, even and uneven.
@pytest.mark.parametrize(
    "m,n,k,cut",
    [(161, 11008, 1024, (1, 2)), (161, 10960, 128 * 9, (1, 1)), (192, 16384, 512, (1, 1)), (192, 16385, 512, (2, 1)), (129, 12000, 1024, (1, 2)), (128, 24576, 512, (2, 1)), (1000, 2900, 1024, (1, 2)),
     (161, 21860, 1024, (1, 1)), (161, 21888, 128 * 9, (1, 1)), (161, 21860, 3072, (1, 2)), (161, 21860, 128 * 22, (1, 1)), (200, 18688, 3072, (1, 1)), (200, 18689, 3072, (1, 2)), (180, 21760, 512, (2, 1)), (256, 20480, 1024, (1, 1)), (256, 20480, 3072, (1, 2)), (256, 20481, 1024, (2, 1)), (96, 21760, 512, (1, 1)), (65, 16500, 1024, (1, 2)), (160, 12000, 128 * 25, (1, 2))],
)
def test_one_strip_per_wave(q8, oracle, m, n, k, cut):
    p = q8.plan_mul_mat(m, n, k)
    assert p["kernel"] == "gemm_tile" and (p["activation_strips"], p["k_sets"], p["k_splits"]) == (*cut, 1), p
    w = oracle.fill_weights(m + n, n, k)
    x = oracle.fill_activations(m + k, m * k).reshape(m, k)
    aq = oracle.quantize_rows(x)
    want = oracle.gemm(w, aq, m, n, k, threads=8) if (k // 32) % 16 == 0 else oracle.gemm(w, aq, m, n, k)
    wt, at = q8.tile(to_dev(w), n, k), q8.quantize_row_q8_0(to_dev(x), tiled=True)
    got = to_host(q8.gemm(wt, at, m, n, k, tiled=True))
    for i in range(m):
        assert rel_l2(got[i], want[i]) <= REL_L2_TOL, i
    res = oracle.fill_activations(5, m * n).reshape(m, n)
    acc = to_dev(res.copy())
    q8.gemm_residual(wt, at, acc, m, n, k, out=acc)
    assert np.array_equal(to_host(acc), got + res)  # one fp32 add after the sum, in place; the sum itself is bit-stable


# The fused gate/up launch in the same form: one K set, two in one pass, two and four, uneven ones; three strips and more; ragged rows.
@pytest.mark.parametrize("m,n_ff,k,cut", [(129, 11264, 512, (1, 1)), (129, 5632, 1024, (2, 1)), (72, 8960, 2048, (2, 4)), (290, 3968, 128 * 12, (2, 1)), (290, 6912, 128 * 9, (1, 1)), (161, 5504, 128 * 25, (2, 1)), (96, 14336, 256, (1, 1))])
def test_gate_up_one_strip_per_wave(q8, oracle, m, n_ff, k, cut):
    p = q8.plan_gate_up_silu(m, n_ff, k)
    assert p["form"] == "tile" and (p["activation_strips"], p["k_sets"], p["passes"]) == (1, *cut), p
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
    assert np.array_equal(to_host(q8.gate_up_silu(tg, tu, aq, m, n_ff, k)), to_host(act))
