"""GPU parity: the MFMA tile kernel with one activation strip per wave, where two would leave the last round of workgroups mostly idle."""
import numpy as np
import pytest

from helpers import REL_L2_TOL, rel_l2, to_dev, to_host

pytestmark = pytest.mark.gpu


# Both ends of the two ranges of workgroups (257 to 384, 513 to 608), four strips and five, a last strip of one row, ragged columns; one K set and two, even and uneven.
@pytest.mark.parametrize(
    "m,n,k,cut",
    [(161, 11008, 1024, (1, 2)), (161, 10960, 128 * 9, (1, 1)), (192, 16384, 512, (1, 1)), (192, 16385, 512, (2, 1)), (129, 12000, 1024, (1, 2)), (128, 24576, 512, (2, 1)), (1000, 2900, 1024, (1, 2)),
     (161, 21860, 1024, (1, 2)), (161, 21888, 128 * 9, (1, 1)), (180, 21760, 512, (2, 1)), (256, 19456, 1024, (1, 2)), (256, 19457, 1024, (2, 1)), (160, 12000, 128 * 25, (1, 2))],
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
