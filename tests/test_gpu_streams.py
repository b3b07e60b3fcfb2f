"""GPU: mat-mats that split K over workgroups beside work on other streams, where a form without that hand-off is left: not refused, not
wrong, and the same bits.  (Which calls are refused, and that a refused one launches nothing: tests/test_scratch_hand_out.py, on the CPU.)"""
import numpy as np
import pytest
import torch

from helpers import REL_L2_TOL, rel_l2, to_dev, to_host

pytestmark = pytest.mark.gpu

# the kernel for up to 32 rows, K over two workgroups per strip; the tile kernel for more than 64, K over two and over four per tile (the
# streaming kernel, with its own cut, would have had to hand sums over for the last one too)
SHAPES = [(4, 4096, 4096), (66, 4224, 5120), (66, 8192, 18432)]
NV, KV = 4096, 14336  # a mat-vec with K over four


def _busy(stream, call):
    """Enqueues a batch of call() on `stream`, long enough that it is still running afterwards; False if that never happened."""
    batch = 1000
    while batch <= 30000:
        stream.synchronize()
        for _ in range(batch):
            assert call() == 0
        if not stream.query():
            return True
        batch *= 10
    return False


# the stream that is kept busy: mat-vecs or mat-mats on a side stream, mat-mats on the null stream
@pytest.mark.parametrize("M,N,K", SHAPES, ids=["4 rows", "66 rows", "66 rows, long K"])
@pytest.mark.parametrize("busy_with", ["mat-vec", "mat-mat", "mat-mat on the null stream"])
def test_mat_mat_beside_another_stream(q8, oracle, busy_with, M, N, K):
    lib = q8._lib.lib()
    assert lib.nh_q8_0_prepare() == 0
    w, wv = oracle.fill_weights(1, N, K), q8.fill_weight_blocks(2, NV, KV)
    x = oracle.fill_activations(3, M * K).reshape(M, K)
    wt, wvt = q8.tile(to_dev(w), N, K), q8.tile(wv, NV, KV)
    at, xv = q8.quantize_row_q8_0(to_dev(x), tiled=True), q8.fill_activations(4, KV)
    want = oracle.gemm(w, oracle.quantize_rows(x), M, N, K, threads=8)
    c, c_busy, y, y_busy = (torch.zeros(s, device="cuda") for s in [(M, N), (M, N), NV, NV])
    q8._lib.check("mat-vec", lib.nh_q8_0_gemv_tiled_f32(wvt.data_ptr(), xv.data_ptr(), y.data_ptr(), NV, KV, None))
    torch.cuda.synchronize()
    y_want = to_host(y)
    a = torch.cuda.default_stream() if "null" in busy_with else torch.cuda.Stream()
    b = torch.cuda.Stream()

    def mat_mat(out, s):
        return lib.nh_q8_0_gemm_tiled(wt.data_ptr(), at.data_ptr(), out.data_ptr(), M, N, K, s.cuda_stream)

    def mat_vec(out, s):
        return lib.nh_q8_0_gemv_tiled_f32(wvt.data_ptr(), xv.data_ptr(), out.data_ptr(), NV, KV, s.cuda_stream)

    for s in (a, b):  # a stream's first launch sets its queue up: not while the other's batch drains
        assert mat_mat(c, s) == 0
        torch.cuda.synchronize()
    outs = [torch.empty_like(c) for _ in range(20)]
    running = _busy(a, (lambda: mat_vec(y_busy, a)) if busy_with == "mat-vec" else (lambda: mat_mat(c_busy, a)))
    for o in outs:
        assert mat_mat(o, b) == 0
    if busy_with != "mat-vec":
        assert mat_vec(y, b) == 0  # the mat-mat's hand-off is not the mat-vec's
    running = running and not a.query()
    torch.cuda.synchronize()
    for o in outs + ([c_busy] if busy_with != "mat-vec" else []):
        assert rel_l2(to_host(o), want) <= REL_L2_TOL
        assert np.array_equal(to_host(o), to_host(c))  # c: computed with nothing else running
    assert np.array_equal(to_host(y), y_want)
    if not running:
        pytest.skip("the busy stream drained before the others were tried: nothing overlapped")


def test_current_stream_handle(q8):
    # the handle the wrappers pass on is torch's, on the default stream and on another, by the short way and by the public one
    for s in (torch.cuda.default_stream(), torch.cuda.Stream()):
        with torch.cuda.stream(s):
            assert q8._stream() == q8._public_stream() == s.cuda_stream
