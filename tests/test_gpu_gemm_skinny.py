"""GPU parity: the streaming MFMA kernel above 32 rows, weights past the caches and through them, at the edges of its tiles."""
import numpy as np
import pytest

from helpers import REL_L2_TOL, rel_l2, to_dev, to_host

pytestmark = pytest.mark.gpu


def check(q8, oracle, m, n, k):
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


# One, two and more groups of rows; a number of strips that is a multiple of eight and one that is not (which decides how two groups load their
# weights); one and two activation strips per workgroup, the second one missing in the last group; ragged strips; K over workgroups.
@pytest.mark.parametrize(
    "m,n,k",
    [(33, 8192, 1024), (64, 8170, 128 * 9), (40, 4096, 1024), (33, 4105, 1024), (64, 256, 128), (64, 250, 128 * 7), (97, 8192, 1024), (161, 4200, 128 * 11), (300, 1000, 128 * 17), (65, 33, 128 * 33),
     (224, 1024, 4096), (130, 700, 128 * 35), (316, 896, 128 * 50), (1000, 256, 1024)],
)
def test_gemm_skinny(q8, oracle, m, n, k):
    assert q8.plan_mul_mat(m, n, k)["kernel"] == "gemm_skinny"
    check(q8, oracle, m, n, k)


# Both sides of each line between the cuts: one activation strip per workgroup and two, eight waves and sixteen, K over workgroups.
@pytest.mark.parametrize(
    "m,n,k,cut",
    [(65, 2752, 256, (1, 8, 1)), (96, 6816, 256, (1, 8, 1)), (65, 6880, 256, (2, 8, 1)), (100, 4096, 256, (2, 8, 1)), (129, 3264, 256, (1, 8, 1)), (160, 3300, 256, (2, 8, 1)), (250, 2048, 256, (1, 8, 1)),
     (34, 4128, 128 * 41, (2, 16, 1)), (34, 4128, 128 * 40, (1, 8, 1)), (34, 4096, 128 * 41, (1, 8, 1)), (190, 1910, 128 * 41, (2, 16, 1)), (193, 1910, 128 * 41, (1, 8, 1)),
     (64, 1056, 128 * 11, (1, 16, 1)), (64, 1024, 128 * 11, (1, 8, 1)), (64, 1056, 128 * 10, (1, 8, 1)), (33, 2570, 128 * 31, (1, 8, 1)), (256, 1000, 128 * 17, (1, 16, 1)), (256, 1000, 128 * 18, (1, 8, 1)),
     (97, 1000, 128 * 31, (1, 16, 1)), (97, 1000, 128 * 32, (1, 8, 2)), (97, 1000, 128 * 41, (1, 8, 2)), (33, 1056, 128 * 33, (1, 8, 2)), (64, 1000, 128 * 34, (1, 8, 4)), (64, 1000, 128 * 33, (1, 8, 2))],
)
def test_cuts(q8, oracle, m, n, k, cut):
    p = q8.plan_mul_mat(m, n, k)
    assert p["kernel"] == "gemm_skinny" and (p["activation_strips"], p["waves"], p["k_splits"]) == cut, p
    check(q8, oracle, m, n, k)
