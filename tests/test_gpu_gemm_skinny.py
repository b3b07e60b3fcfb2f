"""GPU parity: the streaming MFMA kernel above 32 rows, weights past the caches and through them, at the edges of its tiles."""
import numpy as np
import pytest

from helpers import REL_L2_TOL, rel_l2, to_dev, to_host

pytestmark = pytest.mark.gpu


# One, two and more groups of rows; a number of strips that is a multiple of eight and one that is not (which decides how two groups load their
# weights); one and two activation strips per workgroup, the second one missing in the last group; ragged strips; K over workgroups.
@pytest.mark.parametrize(
    "m,n,k",
    [(33, 8192, 1024), (64, 8170, 128 * 9), (40, 4096, 1024), (33, 4105, 1024), (64, 256, 128), (64, 250, 128 * 7), (97, 8192, 1024), (161, 4200, 128 * 11), (300, 1000, 128 * 17), (65, 33, 128 * 33),
     (224, 1024, 4096), (130, 700, 128 * 35), (316, 896, 128 * 50), (1000, 256, 1024)],
)
def test_gemm_skinny(q8, oracle, m, n, k):
    assert q8.plan_mul_mat(m, n, k)["kernel"] == "gemm_skinny"
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
