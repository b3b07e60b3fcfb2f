"""CPU: the kernel each mul_mat shape runs is decided by one host-side plan function, exposed through the C ABI
(nh_q8_0_debug_plan_mul_mat).  The launchers execute that plan, so pinning it here pins the route of every benchmark shape:
a change of a threshold that moves one of them shows up as a failure of this file, not as a silent change of what a parity
test covers.  No GPU needed."""
import pytest

from nihilus_amd import q8_0

L8B = {"q_o": (4096, 4096), "k_v": (1024, 4096), "gate_up": (14336, 4096), "down": (4096, 14336), "lm_head": (128256, 4096)}
L70B = {"q_o": (8192, 8192), "k_v": (1024, 8192), "gate_up": (28672, 8192), "down": (8192, 28672), "lm_head": (128256, 8192)}


def kernel(m, n, k):
    return q8_0.plan_mul_mat(m, n, k)["kernel"]


def test_decode_rows_never_leave_the_mat_vec_kernel():
    for n, k in list(L8B.values()) + list(L70B.values()):
        p = q8_0.plan_mul_mat(1, n, k)
        assert p["kernel"] == "gemv" and not p["quantize_launch"], (n, k)
        for m in (2, 3):
            p = q8_0.plan_mul_mat(m, n, k)
            assert p["kernel"] == "gemv_rows" and not p["quantize_launch"], (m, n, k)


def test_mat_vec_cut_of_the_decode_shapes():
    # (K splits, groups per wave, row parts): long K goes over several workgroups, few strips are cut by rows, never both
    want = {(4096, 4096): (1, 2, 2), (1024, 4096): (1, 2, 4), (14336, 4096): (1, 2, 1), (4096, 14336): (4, 2, 1), (128256, 4096): (1, 2, 1),
            (8192, 8192): (1, 4, 1), (1024, 8192): (1, 4, 4), (28672, 8192): (1, 4, 1), (8192, 28672): (8, 2, 1), (128256, 8192): (1, 4, 1),
            (6144, 4096): (1, 2, 1)}
    for (n, k), (splits, tiles, parts) in want.items():
        p = q8_0.plan_mul_mat(1, n, k)
        assert (p["k_splits"], p["groups_per_wave"], p["row_parts"]) == (splits, tiles, parts), (n, k, p)


def test_four_to_sixteen_rows_on_small_matrices_take_the_mfma_mat_vec():
    # no quantize launch, nothing in the workspace: 4 rows on matrices of up to 80 MB, 5 to 16 rows up to 40 MB while every workgroup has a CU (all of
    # them with a workspace of the caller's); beyond that the quantize launch and the MFMA kernels (every strip's workgroup quantizing the rows again
    # would cost more than the launch)
    for n, k in (L8B["q_o"], L8B["k_v"], L70B["k_v"]):
        for m in (4, 5, 8, 9, 16):
            p = q8_0.plan_mul_mat(m, n, k)
            assert p["kernel"] == "gemv_rows_mfma" and not p["quantize_launch"], (m, n, k)
        assert kernel(17, n, k) == "gemm_skinny"
    for n, k in (L8B["gate_up"], L8B["down"], L70B["q_o"]):
        assert kernel(4, n, k) == "gemv_rows_mfma" and kernel(5, n, k) != "gemv_rows_mfma" and kernel(8, n, k) != "gemv_rows_mfma"
    for n, k in (L70B["gate_up"], L70B["down"], L70B["lm_head"], L8B["lm_head"]):
        assert kernel(4, n, k) not in ("gemv_rows", "gemv_rows_mfma")
    # its cut: a workgroup per CU where K allows it, a wave at most two groups
    assert q8_0.plan_mul_mat(8, 4096, 4096)["k_splits"] == 2 and q8_0.plan_mul_mat(8, 4096, 4096)["groups_per_wave"] == 1
    assert q8_0.plan_mul_mat(4, 1024, 8192)["k_splits"] == 4
    assert q8_0.plan_mul_mat(4, 14336, 4096)["k_splits"] == 1 and q8_0.plan_mul_mat(4, 14336, 4096)["groups_per_wave"] == 2
    # nine to sixteen rows: one group per wave at a time (the rows' fp32 slices share the registers with the weight tiles)
    assert q8_0.plan_mul_mat(16, 4096, 4096)["k_splits"] == 2 and q8_0.plan_mul_mat(16, 4096, 4096)["groups_per_wave"] == 1
    assert q8_0.plan_mul_mat(16, 1024, 8192)["k_splits"] == 4


def test_crossover_shapes():
    # M in {1, 8, 32, 128, 512} on [4096 x 4096] and [14336 x 4096]
    assert [kernel(m, 4096, 4096) for m in (1, 8, 32, 128, 512)] == ["gemv", "gemv_rows_mfma", "gemm_skinny", "gemm_skinny", "gemm_tile"]
    assert [kernel(m, 14336, 4096) for m in (1, 8, 32, 128, 512)] == ["gemv", "gemm_skinny", "gemm_skinny", "gemm_tile", "gemm_tile"]
    p = q8_0.plan_mul_mat(512, 4096, 4096)  # a grid short of four waves per SIMD: four K sets per workgroup
    assert (p["activation_strips"], p["k_sets"], p["k_splits"], p["grid"]) == (2, 4, 1, (32, 8))
    p = q8_0.plan_mul_mat(512, 14336, 4096)
    assert (p["activation_strips"], p["k_sets"], p["k_splits"], p["grid"]) == (2, 1, 1, (112, 8))


def test_batched_decode_at_the_70b_shapes():
    # M in {4, 16, 64}
    want = {
        "q_o": ["gemv_rows_mfma", "gemm_tile_stream", "gemm_tile_stream"],
        "k_v": ["gemv_rows_mfma", "gemv_rows_mfma", "gemm_skinny"],
        "gate_up": ["gemm_tile_stream"] * 3,
        "down": ["gemm_skinny", "gemm_tile_stream", "gemm_tile_stream"],
        "lm_head": ["gemm_tile_stream"] * 3,
    }
    for name, (n, k) in L70B.items():
        assert [kernel(m, n, k) for m in (4, 16, 64)] == want[name], name
    # matrices with few column blocks reach every CU through a K split over workgroups
    for name in ("q_o", "down"):
        p = q8_0.plan_mul_mat(64, *L70B[name])
        assert p["k_sets"] == 4 and p["k_splits"] == 4 and p["grid"] == (64, 1), p
    assert q8_0.plan_mul_mat(64, *L70B["gate_up"])["k_splits"] == 1


def test_tile_kernel_is_not_chosen_where_its_k_split_cannot_be_made():
    # 33..64 rows, 32..191 column blocks, >= 48 Mi weights: the tile kernel only with K over several workgroups; a shape whose
    # K does not divide that way keeps the weight-streaming kernel (an unsplit tile grid of 160 workgroups on 256 CUs is the
    # form measured slower)
    assert kernel(64, 20480, 4096) == "gemm_skinny"
    assert kernel(64, 14336, 4096) == "gemm_tile_stream" and q8_0.plan_mul_mat(64, 14336, 4096)["k_splits"] == 2
    # K = 4096 + 128: 33 groups, no K set divides them
    assert kernel(64, 14336, 4224) == "gemm_skinny"


def test_empty_and_rejected_shapes():
    assert kernel(0, 4096, 4096) == "nothing" and kernel(4, 0, 4096) == "nothing" and kernel(4, 4096, 0) == "nothing"
    with pytest.raises(q8_0._lib.Q8Error):
        q8_0.plan_mul_mat(4, 4096, 100)
    with pytest.raises(q8_0._lib.Q8Error):
        q8_0.plan_mul_mat(-1, 4096, 4096)


def test_up_to_32_rows_every_wave_keeps_its_share_of_the_sums():
    # sets of eight waves that K goes over, in one workgroup or several: what bounds the additions in a row, and so the rounding error.
    # 129 to 255 strips and long K: two sets in one workgroup
    for (m, n, k), sets in {(4, 8192, 28672): 2, (24, 5120, 5120): 2, (24, 6144, 6144): 2, (24, 3200, 8192): 4, (32, 4096, 14336): 2, (8, 14336, 4096): 1, (24, 1024, 4096): 4}.items():
        p = q8_0.plan_mul_mat(m, n, k)
        assert p["kernel"] == "gemm_skinny" and p["gemm_rows"] and p["k_splits"] * p["waves"] == 8 * sets, (m, n, k, p)
    assert not q8_0.plan_mul_mat(33, 5120, 5120)["gemm_rows"] and not q8_0.plan_mul_mat(24, 28672, 8192)["gemm_rows"]


@pytest.mark.parametrize("m,n_ff,k", [(26, 9600, 36864), (29, 8320, 45056), (18, 9088, 176128), (32, 16128, 160768)])
def test_gate_up_of_one_strip_never_asks_for_four_k_sets(m, n_ff, k):
    # the fused kernel for one strip of rows has one and two K sets; K above 32768, which the kernel for up to 32 rows would have to hand over,
    # asks for more on grids this small: three launches, through the workspace
    assert q8_0._lib.lib().nh_q8_0_gate_up_silu_workspace_bytes(m, n_ff, k) == 2 * m * n_ff * 4


def test_k_that_no_number_of_sets_divides():
    # an odd number of 128-quant groups: the tile kernel takes as many K sets as for an even one, gate and up stay one launch
    for k in (4096 - 128, 4096, 4096 + 128):
        assert q8_0.plan_mul_mat(512, 4096, k)["k_sets"] == 4
    size = q8_0._lib.lib().nh_q8_0_gate_up_silu_workspace_bytes
    assert size(48, 11008, 4224) == 0 and size(100, 11008, 4224) == 0
    # ... and three launches where the mat-mats have K over workgroups and the fused form would have one set, or ragged passes
    assert size(65, 3712, 11648) > 0 and size(58, 6400, 2304) > 0


def test_gate_up_in_one_launch_has_the_shares_of_the_streaming_mat_mats():
    # where the mat-mats run on the streaming kernel, one launch adds as many shares of K as they do (K above 1024: below, one pass is enough)
    seen = 0
    for m in (33, 48, 57, 64, 69, 75, 92, 98, 115, 128, 135, 148, 160, 186, 270):
        for n_ff in range(896, 4993, 128):
            for k in (1152, 1408, 2048, 2176, 3072, 4096, 5248, 5632, 6144, 6656, 7680, 8192, 9728):
                gate_up, mat_mat = q8_0.plan_gate_up_silu(m, n_ff, k), q8_0.plan_mul_mat(m, n_ff, k)
                if gate_up["form"] == "tile" and mat_mat["kernel"] == "gemm_skinny":
                    assert mat_mat["k_splits"] * mat_mat["waves"] == gate_up["k_sets"] * gate_up["passes"], (m, n_ff, k)
                    seen += 1
    assert seen > 500


@pytest.mark.parametrize(
    "m,n,k,strips,order",
    [(129, 128 * 127, 256, 1, "by_xcd"), (1000, 128 * 129, 4096, 2, "by_xcd"), (117, 128 * 137, 256, 2, "by_xcd"),  # a number of column blocks that eight does not divide
     (129, 128 * 128, 2432, 1, "bands_of_32"), (129, 128 * 128, 2304, 1, "grid"), (140, 128 * 120, 8192, 1, "grid"),  # one strip per wave: 40 MiB of weights, 128 column blocks
     (512, 128 * 144, 2176, 2, "bands_of_32"), (512, 128 * 144, 2048, 2, "grid"), (3001, 14336, 4096, 2, "grid"), (128, 128 * 136, 40960, 2, "grid")],  # two: 2e10 products, three row groups
)
def test_order_of_the_tiles(m, n, k, strips, order):
    p = q8_0.plan_mul_mat(m, n, k)
    assert (p["kernel"], p["activation_strips"], p["order"]) == ("gemm_tile", strips, order), p


@pytest.mark.parametrize(
    "m,n_ff,k,strips,order",
    [(385, 8704, 256, 1, "bands_of_32"), (193, 8192, 1024, 2, "bands_of_32"), (100, 8192, 1024, 2, "bands_of_32"), (512, 14336, 4096, 2, "bands_of_32"), (512, 7680, 4096, 2, "grid"), (60, 9216, 4096, 2, "grid"),
     (512, 11008, 4096, 2, "by_xcd")],
)
def test_order_of_the_gate_up_tiles(m, n_ff, k, strips, order):
    p = q8_0.plan_gate_up_silu(m, n_ff, k)
    assert (p["form"], p["activation_strips"], p["order"]) == ("tile", strips, order), p


@pytest.mark.parametrize("m,n,k,past", [(64, 8192, 1024, True), (33, 4096, 1024, True), (33, 4128, 1024, False), (97, 1024, 256, False), (40, 128, 128 * 33, True), (64, 480, 128 * 33, False)])
def test_weights_past_the_caches(m, n, k, past):
    # streaming kernel: one group of rows; two whose workgroups are on one XCD, and not; more
    p = q8_0.plan_mul_mat(m, n, k)
    assert p["kernel"] == "gemm_skinny" and p["past_caches"] == past, p


@pytest.mark.parametrize(
    "n_embd,n_ff,splits,by_rows,held",
    [(4096, 14336, 2, True, 63), (3200, 10880, 2, True, 171), (4096, 20480, 4, False, 127), (4096, 15872, 2, True, 0), (4096, 15744, 2, True, 19),  # cut by rows, along K; a handful
     (4096, 10752, 2, True, 175), (4096, 10624, 2, True, 0), (2048, 11008, 2, True, 0), (3200, 17408, 4, False, 0), (4096, 8192, 1, False, 0),  # more than 176; most of the stage; a part of a second round; no round left
     (4224, 20480, 4, False, 0), (5760, 21248, 4, False, 0), (8192, 22016, 4, False, 0), (8192, 28672, 4, False, 0)],  # above 4096 values
)
def test_decode_layer_holds(n_embd, n_ff, splits, by_rows, held):
    assert q8_0.plan_decode_layer(n_embd, n_ff) == {"one_launch": True, "down_splits": splits, "down_by_rows": by_rows, "down_held": held}


def test_decode_layer_beyond_the_one_launch():
    assert not q8_0.plan_decode_layer(8320, 16384)["one_launch"]
    with pytest.raises(q8_0._lib.Q8Error):
        q8_0.plan_decode_layer(4096, 14400)


def test_what_leaves_a_callers_workspace_untouched():
    # nh_q8_0_mul_mat's promise: 4 to 16 rows on matrices of up to 40 MB, 4 rows up to 80 MB.  Without a workspace of the caller's the faster way
    moved = 0
    for n in (32, 1000, 1024, 2560, 4096, 4500, 5120, 6144, 8192, 14336, 28672, 128256):
        for k in (128, 1024, 2048, 4096, 5120, 8192, 14336, 28672):
            for m in range(4, 18):
                promised = m <= 16 and n * (k // 32) * 34 <= (80 if m == 4 else 40) << 20
                kept = q8_0.plan_mul_mat(m, n, k, own_workspace=True)
                assert kept["quantize_launch"] != promised and (kept["kernel"] == "gemv_rows_mfma") == promised, (m, n, k)
                moved += kept != q8_0.plan_mul_mat(m, n, k)
                assert promised or kept == q8_0.plan_mul_mat(m, n, k)
    assert moved > 100
    assert q8_0.plan_mul_mat(16, 4096, 8192)["quantize_launch"] and not q8_0.plan_mul_mat(16, 4096, 8192, own_workspace=True)["quantize_launch"]


@pytest.mark.parametrize("m,n,k", [(24, 8192, 36864), (32, 8192, 36864), (20, 14336, 40960), (17, 8096, 45056)])
def test_k_too_long_for_the_rows_kernel_stays_with_the_tile_kernel(m, n, k):
    # the rows kernel's hand-off does not hold two sets of K of so many strips; the streaming kernel in its place is the slowest of the three
    assert kernel(m, n, k) == "gemm_tile_stream"


@pytest.mark.parametrize("m,n,k,rows", [(20, 14656, 15360, True), (20, 14656, 17408, False), (17, 16128, 27648, False), (24, 8192, 32768, True), (28, 8192, 24576, True), (26, 8192, 27648, True),
                                        (28, 8192, 32768, False), (28, 8084, 26624, False)])
def test_long_k_of_17_to_32_rows(m, n, k, rows):
    # the rows kernel's line to the tile kernel with K over workgroups: two workgroups per CU with long K, and 25 rows and more where the tile
    # kernel has a workgroup per CU, are faster there
    assert q8_0.plan_mul_mat(m, n, k)["gemm_rows"] == rows and (kernel(m, n, k) == "gemm_tile_stream") != rows


@pytest.mark.parametrize("m,n_ff,groups,form", [(40, 24832, 54, (2, 2, 1)), (24, 29568, 38, (1, 2, 1)), (58, 25600, 18, (2, 2, 1)), (21, 41856, 103, (1, 1, 1)), (59, 40832, 103, (2, 1, 1)), (24, 33024, 9, (1, 1, 1))])
def test_gate_up_takes_no_pass_for_uneven_sets_of_the_mat_mats(m, n_ff, groups, form):
    # where the mat-mats' sets of K differ by a group, the one launch keeps its own number of sets and one pass
    p = q8_0.plan_gate_up_silu(m, n_ff, 128 * groups)
    assert (p["activation_strips"], p["k_sets"], p["passes"]) == form
    assert q8_0._lib.lib().nh_q8_0_gate_up_silu_workspace_bytes(m, n_ff, 128 * groups) == 0


@pytest.mark.parametrize("m,n_ff,groups", [(484, 768, 88), (331, 1024, 92), (902, 384, 120), (176, 1792, 108)])
def test_gate_up_stays_one_launch_where_the_mat_mats_have_sixteen_uneven_shares(m, n_ff, groups):
    assert q8_0.plan_mul_mat(m, n_ff, 128 * groups)["k_splits"] == 4 and groups % 16
    p = q8_0.plan_gate_up_silu(m, n_ff, 128 * groups)
    assert (p["form"], p["k_sets"], p["passes"], p["tree"]) == ("tile", 4, 2, True)
    assert q8_0._lib.lib().nh_q8_0_gate_up_silu_workspace_bytes(m, n_ff, 128 * groups) == 0


@pytest.mark.parametrize("m,n_ff,groups,form", [(67, 4096, 43, "three_launches"), (254, 2048, 114, "three_launches"), (131, 1536, 27, "three_launches"), (126, 4224, 43, "tile"), (354, 1536, 35, "tile"), (48, 5504, 33, "tile")])
def test_uneven_passes_of_gate_up_need_more_than_half_the_cus(m, n_ff, groups, form):
    p = q8_0.plan_gate_up_silu(m, n_ff, 128 * groups)
    assert p["form"] == form and (form != "tile" or p["passes"] == 2)


@pytest.mark.parametrize("m,n,groups,sets", [(701, 1536, 18, 2), (512, 4096, 38, 2), (512, 4096, 42, 4), (512, 4096, 17, 4), (24, 24832, 30, 2), (64, 24832, 30, 2), (64, 24832, 42, 4), (24, 24832, 58, 2),
                                             (24, 24832, 33, 4), (64, 60032, 9, 1), (117, 16640, 15, 1), (117, 28672, 25, 2), (24, 60032, 57, 1), (24, 60032, 56, 2)])
def test_short_uneven_sets_of_the_mat_mats(m, n, groups, sets):
    # two even sets stay two while four uneven ones would be short; with more workgroups than CUs one set stays one
    p = q8_0.plan_mul_mat(m, n, 128 * groups)
    assert p["kernel"].startswith("gemm_tile") and (p["k_sets"], p["k_splits"]) == (sets, 1)


@pytest.mark.parametrize("m,n,groups,splits", [(200, 4096, 87, 2), (120, 3840, 105, 4), (74, 9712, 46, 0), (358, 1636, 241, 0), (330, 1389, 242, 0), (86, 6255, 252, 4), (159, 1380, 88, 0), (96, 2139, 91, 0), (512, 4096, 33, 1)])
def test_uneven_k_over_workgroups_has_no_second_round_of_few(m, n, groups, splits):
    # more than 64 rows, K that the shares do not divide: over workgroups (splits) while they fit the CUs once or fill them nearly twice; else the streaming kernel (0)
    p = q8_0.plan_mul_mat(m, n, 128 * groups)
    assert (p["kernel"], p["k_splits"]) == ("gemm_tile", splits) if splits else p["kernel"] == "gemm_skinny"
