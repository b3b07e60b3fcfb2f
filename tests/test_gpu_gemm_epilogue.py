"""GPU parity: what the mat-mat kernels do behind their K loop -- the sum over waves, K sets and workgroups, and the residual."""
import numpy as np
import pytest

from helpers import REL_L2_TOL, rel_l2, to_dev, to_host

pytestmark = pytest.mark.gpu


# streaming kernel: two strips per workgroup (even and odd number of strips), one strip, K over workgroups, ragged rows and columns; tile kernel: one, two and four K sets
@pytest.mark.parametrize("m,n,k", [(117, 4096, 4096), (77, 8200, 4096), (117, 1000, 4096), (512, 1024, 4096), (40, 1030, 14336), (1500, 1030, 512), (700, 4100, 1024), (512, 4096, 2048)])
def test_residual_is_one_add(q8, oracle, m, n, k):
    w, x = oracle.fill_weights(m + n, n, k), oracle.fill_activations(k, m * k).reshape(m, k)
    res = oracle.fill_activations(m + n, m * n).reshape(m, n)
    aq = oracle.quantize_rows(x)
    wt, at = q8.tile(to_dev(w), n, k), q8.tile(to_dev(aq.reshape(-1)), m, k)
    plain = to_host(q8.gemm(wt, at, m, n, k, tiled=True))
    rows = sorted({0, 31, 32, m // 2, m - 1})
    want = oracle.gemm(w, np.ascontiguousarray(aq[rows]), len(rows), n, k)
    for i, row in enumerate(rows):
        assert rel_l2(plain[row], want[i]) <= REL_L2_TOL, row
    assert np.array_equal(to_host(q8.gemm_residual(wt, at, to_dev(res), m, n, k)), plain + res)
    acc = to_dev(res.copy())
    q8.gemm_residual(wt, at, acc, m, n, k, out=acc)
    assert np.array_equal(to_host(acc), plain + res)
