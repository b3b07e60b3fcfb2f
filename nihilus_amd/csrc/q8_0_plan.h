// Which kernel a mul_mat call runs, and how that kernel cuts the work: decided here, on the host, in one place, from the
// shape alone.  The launchers execute the plan they get from these functions and decide no cut, order or route themselves -- but for a call that is being
// captured, or finds the hand-off scratch of its form in use on another stream, which runs as the form without it that the plan has
// for it: in the mat-mats the same additions in the same order -- so a test can
// ask (nh_q8_0_debug_plan_mul_mat, no GPU needed) what a shape will run and pin it.
//
// The rules are measurements, not a model: each threshold below names the shapes it was fitted on.  A shape between the
// measured ones follows the nearest rule; the plan says which, so it can at least be seen and tested.
#pragma once
#include "q8_0_gemv_tiled.h"

namespace nh {

// values are part of the debug C entry's contract (include/nihilus_amd/q8_0_abi.h: nh_q8_0_debug_plan_mul_mat)
enum mul_mat_kernel : int {
	MM_NOTHING			= 0, // an empty problem: nothing, or a fill of the output
	MM_GEMV				= 1, // M == 1: quantize inside the streaming mat-vec (gemv_tiled_kernel)
	MM_GEMV_ROWS		= 2, // 2, 3 rows: the streaming mat-vec with one dot product per row (gemv_rows_kernel), quantize inside
	MM_GEMM_SKINNY		= 3, // quantize launch + weight-streaming MFMA kernel (gemm_skinny_kernel)
	MM_GEMM_TILE_STREAM = 4, // quantize launch + MFMA tile kernel with non-temporal weight loads (batched decode on large matrices)
	MM_GEMM_TILE		= 5, // quantize launch + MFMA tile kernel (prefill)
	MM_GEMV_ROWS_MFMA	= 6, // 4..16 rows on small matrices: the streaming mat-vec with the rows as an MFMA operand (gemv_rows8_kernel), quantize inside
};

constexpr int SK_WAVES			  = 8; // waves per workgroup of the weight-streaming MFMA kernel
constexpr int SK_WIDE_WAVES		  = 16; // the same where K over eight more is better than over another workgroup (plan_gemm_skinny, plan_gemm_streaming)
constexpr int SK_MAX_SPLIT_UNITS  = 2048; // strips * splits when splits > 1
constexpr int SK_MAX_SPLIT_STRIPS = 512;
constexpr int GEMM_SPLIT_MIN_TRIPS = 2; // K goes over more workgroups only while each K set keeps this many 128-quant groups
constexpr int GEMM_STREAM_TILE_MIN_COLUMN_BLOCKS = 192; // 128-row column blocks from which the tile kernel also takes the few-row (batched decode) shapes

// The MFMA tile kernel's cut: TM activation strips per wave; KS sets of four waves per workgroup, each on a share of K (grids
// that would leave SIMDs short of their four waves); also K over kz workgroups per tile (grids short of one workgroup per CU), their
// tiles added through the scratch by the last to arrive.
struct gemm_tile_cut {
	int tm, ks, kz;
	unsigned grid_x, grid_y;
	int order; // in which the workgroups take the tiles (gemm_tile_order)
};
inline gemm_tile_cut plan_gemm_tile(int64_t M, int64_t N, int64_t K, bool stream) {
	gemm_tile_cut c{};
	const int64_t m_strips = (M + 31) / 32, n_strips = (N + 31) / 32;
	const int groups	   = static_cast<int>(K / GROUP_K);
	// two activation strips per wave whenever there are two: every weight tile fetched is used twice (the one-strip form,
	// with twice the weight loads per MFMA, measured 8 to 60 % slower at M = 512)
	c.tm	 = m_strips >= 2 ? 2 : 1;
	c.grid_x = static_cast<unsigned>((n_strips + 3) / 4);
	c.grid_y = static_cast<unsigned>((m_strips + c.tm - 1) / c.tm);
	// K sets until every SIMD has four waves, while each keeps four groups.  K need not divide: the sets' shares differ by a group then (a mat-mat of its
	// own takes fewer where that does not pay, gemm_tile_mat_mat).  Measured, us, with as many sets as divide / this: [4096 x 4224] at 350 / 512 rows
	// 43.5 / 25.0 and 43.7 / 28.2, [4096 x 11136] 107.7 / 54.9 and 107.9 / 64.5, [2560 x 2688] at 512 28.5 / 18.4, [28672 x 3200] at 60 / 30 rows
	// 36.7 / 26.9 and 27.9 / 21.7
	c.ks	 = 1;
	while (c.ks < 4 && static_cast<int64_t>(c.grid_x) * c.grid_y * 4 * c.ks * 2 <= 4096 && groups / (c.ks * 2) >= 4) {
		c.ks *= 2;
	}
	c.kz = 1;
	if (stream) {
		const int64_t wgs = static_cast<int64_t>(c.grid_x) * c.grid_y;
		while (c.ks == 4 && wgs * c.kz * 2 <= 256 && groups % (c.ks * c.kz * 2) == 0 && groups / (c.ks * c.kz * 2) >= GEMM_SPLIT_MIN_TRIPS &&
			wgs * c.kz * 2 * c.tm * 4096 <= GEMM_SPLIT_SCRATCH_FLOATS && wgs <= GEMM_SPLIT_MAX_UNITS) {
			c.kz *= 2;
		}
	}
	return c;
}

// One activation strip per wave instead of two where that fills the chip's last round better: twice the workgroups of half the work, and no second strip that is none
// where their number is odd.  `percent`: what a round of them takes of a half round of the others, as weight tiles are fetched twice as often.  Measured, us, two strips / one:
//   mat-mats  [1024 x 4096] at 3001 rows (three half rounds for two rounds) 42.5 / 38.2, [4096 x 14336] at 600 126 / 118, [4096 x 1024] at 740 13.7 / 12.3, [8192 x 8192] at 330
//             80 / 72, [19712 x 3456] at 81 37.0 / 26.4; [4096 x 4096] at 1050 (five for three) 62.2 / 58.8, [8192 x 8192] at 520 122 / 116; [26752 x 6784] at 201 (six for four)
//             140 / 121; but seven for four [10496 x 3072] at 640 63.4 / 65.0, [25472 x 1024] at 234 27.0 / 29.4
//   gate/up   [2 x 1280 x 1280] at 788 rows (three for two) 32 / 20, [2 x 8960 x 5760] at 233 (five for three) 96 / 94, [2 x 2560 x 4608] at 787 79 / 58, [2 x 5248 x 3200] at 578
//             (seven for four) 72.6 / 68.5, [2 x 17792 x 4096] at 266 (ten for six) 142 / 128; but with eleven for six [2 x 28672 x 8192] at 178 261 / 274,
//             [2 x 22016 x 5632] at 236 181 / 189, [2 x 5376 x 2048] at 326 30.8 / 33.4 ([2 x 10368 x 7936] at 543 257 / 252), thirteen for seven [2 x 25600 x 5248] at 243 210 / 302
// Over 70 random shapes each whose cut differs: mat-mats 0.94 to 1.44 times as fast, mean 1.07; gate/up 0.98 to 1.60, mean 1.10.  Not with four strips ([20480 x 4096] at 100 rows 41 / 43,
// [2 x 9344 x 7808] at 119 78 / 80): of 50 random shapes each mat-mats 0.91 to 1.27, mean 0.98, gate/up 0.91 to 1.29, mean 1.01.
constexpr int ONE_STRIP_MAT_MAT = 115, ONE_STRIP_GATE_UP = 110;
inline bool gemm_tile_take_one_strip(gemm_tile_cut* c, int64_t m_strips, int percent) {
	const int64_t twos = int64_t{ c->grid_x } * c->grid_y, ones = int64_t{ c->grid_x } * m_strips;
	if (c->tm != 2 || c->kz != 1 || m_strips <= 2 || m_strips == 4 || twos <= 256 || (ones + 255) / 256 * percent > (twos + 255) / 256 * 200) {
		return false;
	}
	c->tm	  = 1;
	c->grid_y = static_cast<unsigned>(m_strips);
	return true;
}

// The order in which the tile kernel's workgroups take its tiles (not those with K over workgroups or with streamed weights, which have one row of workgroups or few).
//
// By XCD: workgroups go to the eight XCDs in turn.  With a number of column blocks that eight divides, a block's row groups are all on one XCD, whose L2 has its weights then;
// otherwise every XCD would read nearly all of them.  There each XCD takes the tiles of some consecutive column blocks instead, row groups fastest ([24171 x 10240] at 145 rows
// 182 -> 126 us, [3117 x 10752] at 912 134 -> 92, [2 x 3968 x 6528] at 274 77 -> 59 with one strip per wave; 60 random shapes with one 0.99 to 1.62 times as fast, mean 1.20, 120 with two
// 0.98 to 1.17, mean 1.04).  Not with eight dividing: a round of workgroups is a wider piece of the matrix then as it is ([8192 x 8192] at 330 rows 72 us, 76 this way).
//
// In bands of that many column blocks, all row groups of a band before the next band is begun, where eight divides their number.  With one band, every group of rows walks the
// whole matrix, from memory again where it is no longer cached, and the workgroups that run together share only their activations.  Measured, us, one band / this:
//   gate/up   [2 x 28672 x 8192] at 512 rows 740 / 578, at 178 two strips 289 / 252; [2 x 14336 x 4096] at 512 / 3001 166 / 157, 917 / 855; [2 x 26624 x 9344] at 858 1365 / 1064;
//             with one strip per wave [2 x 21504 x 7808] at 200 316 / 223, [2 x 24576 x 1920] at 273 121 / 88; 61 random shapes 0.97 to 1.73 times as fast, mean 1.15, 149 with two strips
//             0.98 to 1.22, mean 1.04
//   mat-mats  [27648 x 4736] at 1058 360 / 341, [20475 x 9984] at 1965 973 / 930, [25530 x 6784] at 738 340 / 325; 39 random shapes 0.99 to 1.16, mean 1.05, 59 with one strip 0.94 to 1.47,
//             mean 1.07; but below 2e10 products 8 of 0.95 to 1.01, mean 0.98 ([17408 x 2432] at 162 0.95), and with one strip below 40 MiB of weights 34 of 0.85 to 1.01, mean 0.95
//             ([22528 x 384] at 216 0.85): there it stays as it is
// (In runs of some milliseconds with waits between them the bands look worse than this, by up to 5 %: launches one after the other for tens of milliseconds run at a lower clock, as a
// prompt's do, and there the bytes saved count.  The figures are of such.)
// Bands of 16 to 64 column blocks are within 1 % of each other.  Below 128 nothing changes ([2 x 5632 x 7680] at 660 rows 161 / 161, [9146 x 9216] at 326 88.0 / 88.1), and two
// row groups of a mat-mat find each other's weights on their way as it is ([22528 x 2944] at 118 rows 32.9 / 32.9; gate / up [2 x 24064 x 8320] at 125 159 / 152).
constexpr int TILE_ORDER_GRID = 0, TILE_ORDER_XCD = 1, TILE_ORDER_BANDS = 32;
constexpr int64_t TILE_BANDS_MIN_PRODUCTS = 20'000'000'000, TILE_BANDS_ONE_STRIP_BYTES = 40ll << 20;
inline int gemm_tile_order(const gemm_tile_cut& c, bool gate_up, int64_t M, int64_t N, int64_t K) {
	if (c.grid_x % 8 != 0) {
		return c.grid_y > 1 ? TILE_ORDER_XCD : TILE_ORDER_GRID;
	}
	if (c.grid_x < 128 || c.grid_y < (gate_up ? 2u : 3u)) {
		return TILE_ORDER_GRID;
	}
	return gate_up || (c.tm == 1 ? N * (K / QK) * BLOCK_BYTES >= TILE_BANDS_ONE_STRIP_BYTES : M * N * K >= TILE_BANDS_MIN_PRODUCTS) ? TILE_ORDER_BANDS : TILE_ORDER_GRID;
}

// The tile kernel's cut for a mat-mat of its own (K not over workgroups).  Uneven sets walk as many trips as the longest, so short ones multiply up to a tenth
// more for nothing, and behind two sets, or more workgroups than CUs, there are two waves on a SIMD already.  Measured, us:
//   two even sets / four uneven   [4096 x 2304] at 512 rows 16.1 / 17.1, [8064 x 2816] at 200 22.9 / 25.5, [2048 x 3328] at 1000 22.8 / 23.1; of streamed weights
//                                 [24832 x 3840] at 24 / 64 rows 27.0 / 34.5 and 32.0 / 38.1, [32000 x 4864] 29.4 / 30.5 and 38.4 / 39.8; but
//                                 [4096 x 6912] at 512 43.2 / 40.9, [24832 x 5376] at 64 38.2 / 34.9.  One strip [32000 x 6400] at 24 38.4 / 40.0
//   one set / two uneven          [60032 x 1152] at 64 rows 21.4 / 25.3, [16640 x 1920] at 117 25.3 / 26.9, [28672 x 2176] at 117 31.2 / 30.3; one strip
//                                 [40064 x 1152] at 24 12.7 / 14.6, [60032 x 7296] 72.8 / 74.4
inline gemm_tile_cut gemm_tile_mat_mat(gemm_tile_cut c, int groups, int64_t m_strips, bool stream) {
	if (c.ks == 4 && c.kz == 1 && groups % 4 == 2 && (c.tm == 1 || groups < 40)) {
		c.ks = 2;
	}
	if (c.ks == 2 && groups % 2 != 0 && static_cast<int64_t>(c.grid_x) * c.grid_y > 256 && (c.tm == 1 || groups < 24)) {
		c.ks = 1;
	}
	// One set of K into two behind that: up to five rounds of them are less than four waves on a SIMD.  From K = 3072 on and with more than four rounds: 183 random shapes 0.97 to 1.07 times
	// as fast, mean 1.02 ([4096 x 4096] at 1100 rows 59.7 / 58.8; at 1600, seven rounds, 80.8 / 83.4); shorter 145 of 0.90 to 1.05, mean 0.98 ([13568 x 1024] at 294 0.94), with up to four rounds 32, 0.98.
	if (!stream && gemm_tile_take_one_strip(&c, m_strips, ONE_STRIP_MAT_MAT) && c.ks == 1 && groups >= 24 && groups % 2 == 0 && c.grid_x * m_strips > 1024 && c.grid_x * m_strips <= 1280) {
		c.ks = 2;
	}
	return c;
}

// The weight-streaming MFMA kernel's cut: MS activation strips per workgroup, K of a strip over `splits` workgroups of `waves` waves.
struct gemm_skinny_cut {
	int ms, splits, waves; // waves: 8 or 16, the shares of K that a workgroup adds
};
constexpr int64_t GEMM_ROWS_MAX = 32;
inline int gemm_rows_operand(int64_t M) { // operand rows the rows kernel is instantiated for
	return M <= 8 ? 8 : M <= 16 ? 16 : M <= 24 ? 24 : 32;
}
// This one decides how many shares K goes over (also for the forms that stand in for this kernel); how more than 32 rows carry them out: plan_gemm_streaming.
inline gemm_skinny_cut plan_gemm_skinny(int64_t M, int64_t N, int64_t K) {
	gemm_skinny_cut c{};
	const int groups	 = static_cast<int>(K / GROUP_K);
	const int64_t strips = (N + STRIP_ROWS - 1) / STRIP_ROWS, m_strips = (M + STRIP_ROWS - 1) / STRIP_ROWS;
	// Two activation strips per workgroup halve the weight traffic per row, but only pay once the grid fills the chip
	// without them: 64 rows against 128 weight strips are better off as 256 workgroups of one strip each.
	c.ms				= (m_strips <= 1 || strips * ((m_strips + 1) / 2) < 256) ? 1 : 2;
	const int64_t units = strips * ((m_strips + c.ms - 1) / c.ms);
	// K goes over sets of eight waves.  The hand-off between workgroups is expensive here (a partial tile of 16 values per lane and strip, an
	// arrival counter, the last arriver reading every share): only until every CU has a workgroup (and every wave
	// keeps at least two groups, one step of the kernel's walk: [4096 x 4096] at M = 32 12.1 -> 10.8 us, [1024 x 8192] at M = 64
	// 14.9 -> 13.2 us against keeping four), or when a wave would otherwise walk more than sixteen groups.  Measured on
	// [8192 x 28672] at M = 16: 68 us with eight sets per strip, 51 us with two.
	const auto sets_for = [&](int waves) {
		int sets = 1;
		while (waves == SK_WAVES && units * sets < 256 && groups >= 4 * SK_WAVES * sets && units * sets * 2 <= SK_MAX_SPLIT_UNITS && units <= SK_MAX_SPLIT_STRIPS) {
			sets *= 2;
		}
		while (groups > 16 * waves * sets && units * sets * 2 <= SK_MAX_SPLIT_UNITS && units <= SK_MAX_SPLIT_STRIPS) {
			sets *= 2;
		}
		return sets;
	};
	if (M <= GEMM_ROWS_MAX) {
		// Up to 32 rows: one cut for the rows kernel (q8_0_gemm_rows.hip) and for the streaming kernel, which takes its calls where the hand-off's
		// tags cannot be used, so that both add the same sums in the same order.  The rows kernel's hand-off is cheaper: until the launch has
		// a workgroup per CU, while every wave keeps a group ([4096 x 4096] at 4 rows 5.7 us with 256 workgroups, 6.0 with 512;
		// [4096 x 14336] 12.6 and 13.3; [1024 x 4096] 4.6 us with 128).  Where the rule above makes more sets than that, a workgroup takes
		// two of them (sixteen waves; in the rows kernel eight, one set after the other): no more additions in a row than there, and nothing
		// more to hand over.  One set instead, [6144 x 6144] at 8 / 32 rows: 8.7 / 11.5 us against 9.0 / 12.1, but [8192 x 28672] 2.0e-7 from
		// the sums in 64 bits where two sets are 1.5e-7, and [5120 x 5120] 9.9e-8 against 8.2e-8.  Few strips with a long K pay most for the
		// second set: [1037 x 16640] 7.3 / 10.5 us at 4 / 24 rows with one, 8.2 / 11.7 with two.  (Sixteen waves in the rows kernel too, at
		// [6144 x 6144]: 9.0 / 12.8 us.)
		const int sets = sets_for(SK_WAVES);
		c.waves		   = SK_WAVES;
		c.splits	   = 1;
		while (strips * c.splits * 2 <= 256 && groups >= 2 * SK_WAVES * c.splits && strips * gemm_rows_operand(M) * c.splits * 2 <= GEMV_MAX_SPLIT_UNITS) {
			c.splits *= 2;
		}
		if (sets > c.splits) {
			c.waves	 = SK_WIDE_WAVES;
			c.splits = sets / 2;
		}
		return c;
	}
	// 129 to 255 units and a K that eight waves would split: two workgroups each leave some CUs two and some one or none, and the launch
	// takes as long as the ones with two.  One workgroup of sixteen waves per unit has the same waves on every CU it uses and nothing to hand
	// over.  Measured, us, split / this: [1024 x 8192] at 200 rows 13.6 / 11.9, [1024 x 4096] at 224 rows 9.5 / 7.7, [3072 x 12288] at 40 rows
	// 20.6 / 18.0, [768 x 4096] at 180 rows 9.0 / 7.6, [4064 x 4096] at 50 rows 11.0 / 9.3, [2080 x 4096] at 64 rows 9.8 / 9.1, [640 x 14336] at
	// 256 rows 20.1 / 19.4.  Outside it does not pay: at 128 units, which the split makes into a workgroup per CU, 7.4 / 7.6 ([1024 x 4096] at
	// 117 rows) and 9.6 / 12.2 (K = 8192); at 256, 12.8 / 12.5 ([4096 x 4096] at 117 rows) and 8.5 / 8.8 (at 64).
	c.waves	 = (units > 128 && units < 256 && groups >= 4 * SK_WAVES) ? SK_WIDE_WAVES : SK_WAVES;
	c.splits = sets_for(c.waves);
	return c;
}

// Its weights go past the caches where no other workgroup reads them.  The groups of rows read the same ones: past the caches each would take them from memory again
// ([896 x 6400] at 316 rows 17.1 -> 11.4 us, [4319 x 4224] at 35 rows 13.9 -> 11.5, [4096 x 4096] at 200 rows 18.4 -> 16.8, [1024 x 4096] at 512 / 250 / 117 rows
// 10.6 -> 9.6, 7.3 -> 6.6, 7.1 -> 6.7).  Not with one group ([8192 x 4096] at 40 rows 12.3 as it is, 13.2 through the caches), nor with two whose workgroups are on
// one XCD (workgroups go to the eight in turn) at the same time: the second finds the first's lines on their way ([4096 x 4096] at 64 rows 8.1 / 8.25, at 117 rows
// the same).
inline bool gemm_skinny_past_caches(int64_t M, int64_t N, const gemm_skinny_cut& cut) {
	const int64_t strips = (N + STRIP_ROWS - 1) / STRIP_ROWS, m_strips = (M + STRIP_ROWS - 1) / STRIP_ROWS, m_groups = (m_strips + cut.ms - 1) / cut.ms;
	return m_groups == 1 || (m_groups == 2 && (strips * cut.splits) % 8 == 0);
}

// The streaming kernel's own mat-mats of more than 32 rows: never fewer shares of K than above, in another cut where that is faster (measured, us, cut above / this; in
// brackets 50 random shapes of each kind).
// - One strip per workgroup instead of two, up to 512 workgroups of one (of three strips, whose fourth would be work for nothing, up to 640): half as many leave
//   a part of the chip's last round idle ([4864 x 2432] at 94 rows 11.4 / 7.9, [5632 x 3968] at 72 16.8 / 13.0, [3016 x 7424] at 148 24.1 / 21.5; with five strips
//   [3346 x 2176] at 144, 525 of one, 10.3 / 11.0; 0.98 to 1.47, mean 1.23).  Also where two strips make just a workgroup per CU, if those are of eight row strips and
//   more: two workgroups on a CU wait for their loads in turn ([2048 x 1024] at 256 5.3 / 4.7, [1024 x 4096] at 512 10.4 / 10.4; [4096 x 4096] at 128 12.3 / 12.4).
// - Two strips instead of one, with sixteen waves, where those fit a workgroup per CU and ones of a strip do not, from K = 5248 on: the weights cross L2 once for
//   two strips ([7296 x 8832] at 36 rows 24.6 / 19.5, [5888 x 13568] at 48 37.7 / 28.8; at K = 4608 11.6 / 12.0).  With more than 64
//   rows from 360 workgroups on ([2560 x 6144] at 103 rows, 320, 12.7 / 14.1), and up to 192 ([1152 x 9856] at 310 18.4 / 19.0): 0.92 ([3200 x 5504] at 120) to 1.14 times
//   as fast below K = 7680, [2658 x 14464] at 170 33.1 / 28.2.  (Of all 0.92 to 1.40, mean 1.13.)
// - Sixteen waves instead of eight for 65 to 160 workgroups and eleven to 31 groups, and for more workgroups while a wave of eight has two groups or so: all of a wave's
//   share is on its way at once ([768 x 2048] at 104 rows 4.8 / 4.5, [1569 x 1664] at 57 4.8 / 4.7; [2048 x 2304] at 127, 256 workgroups, 5.8 / 6.0; up to 64
//   workgroups it may lose, [611 x 2688] at 80 rows 5.3 / 5.65; 0.95 to 1.08, mean 1.02).  Not instead of two workgroups of eight: 65 to 128 of them, with more than 64 rows
//   and up to 40 groups, 0.92 to 1.00, mean 0.96 ([1024 x 4096] at 117 rows 6.7 / 7.1, the same bits).
// - Four workgroups along K instead of two for up to 64 and from 34 groups on, as a CU more costs nothing there ([457 x 6272] at 40 rows 7.5 / 6.1, [384 x 8064] at
//   34 8.2 / 6.4; 1.08 to 1.30, mean 1.20).
// Not in more shares where gate / up of such a pair are one launch, which has no room for sixteen (plan_gate_up_with): one launch and three give the same bytes
// there (one in a hundred of the pairs whose mat-mats run here: [2 x 2688 x 2048] at 69 rows, [2 x 3840 x 6144] at 98), and
// the mat-mats cost no more: 40 random ones of those with sixteen shares / these 0.91 to 1.09, mean 1.01.
inline bool gate_up_one_launch_beside(const gemm_skinny_cut& mat_mat, int64_t M, int64_t n_ff, int64_t K); // below
inline gemm_skinny_cut plan_gemm_streaming(int64_t M, int64_t N, int64_t K) {
	const gemm_skinny_cut own = plan_gemm_skinny(M, N, K);
	gemm_skinny_cut c		  = own;
	if (M <= GEMM_ROWS_MAX) {
		return c;
	}
	const int groups	 = static_cast<int>(K / GROUP_K);
	const int64_t strips = (N + STRIP_ROWS - 1) / STRIP_ROWS, m_strips = (M + STRIP_ROWS - 1) / STRIP_ROWS;
	const int64_t ones = strips * m_strips, twos = strips * ((m_strips + 1) / 2); // workgroups of one strip, of two
	if (c.ms == 2 && c.splits == 1 && (twos > 256 || (twos == 256 && m_strips >= 8)) && ones <= (m_strips == 3 ? 640 : 512)) {
		c.ms = 1;
	} else if (c.ms == 1 && ones > 256 && twos < 256 && (M <= 64 || (M <= 192 && ones >= 360)) && groups >= 41 && c.splits * c.waves <= SK_WIDE_WAVES) {
		c = gemm_skinny_cut{ 2, 1, SK_WIDE_WAVES };
	} else if (c.ms == 1 && c.waves == SK_WAVES) {
		if (c.splits == 1 && ones > 64 && groups >= 11 && (ones <= 160 || (ones <= 256 && groups < 18))) {
			c.waves = SK_WIDE_WAVES;
		} else if (c.splits == 2 && ones <= 64 && groups >= 34) {
			c.splits = 4;
		}
	}
	if (c.splits * c.waves != own.splits * own.waves && gate_up_one_launch_beside(own, M, N, K)) {
		return own;
	}
	return c;
}

// More than 64 rows against a matrix whose tiles are short of a workgroup per CU, with K long enough: the tile kernel with K over workgroups
// until there is about one per CU.  The streaming kernel, which has the shape otherwise, takes the activations out of L2 once per weight
// strip, where four strips share them here; the hand-off costs 3 to 4 us, so every K set has to keep five groups.  Measured, us, this /
// the streaming kernel: [8192 x 28672] at 128 rows 91 / 129, [8192 x 8192] at 96 / 128 rows 31 / 36 and 31 / 38, [4096 x 8192] at 200 rows
// 28.5 / 34.3, [4096 x 14336] at 117 rows (seven groups, K over four) 28.5 / 31.1, [5120 x 5120] at 160 rows (five) 21.4 / 22.3; with four
// groups [4096 x 4096] at 200 rows 18.4 / 18.0, [2048 x 8192] at 256 rows 19.8 / 18.1; with two [4096 x 4096] at 117 rows 14.9 / 12.5.
//
// K need not divide, if the longest share is at most a tenth over the average: [4096 x 11136] at 200 rows 47.5 / 36.1 (the streaming kernel / this),
// [7936 x 28032] at 233 rows 271 / 172, [4992 x 13184] at 121 rows 55.5 / 39.6, [6784 x 6784] at 125 rows (seven groups where 6.6 would do)
// 32.6 / 29.1; but [5376 x 5376] at 144 rows (six for 5.25) 25.6 / 28.4.
// Such a K also needs its workgroups to fit the CUs once or fill them nearly twice, and not the sixteen waves that the streaming kernel has for
// 129 to 255 units: over 430 random shapes the streaming kernel takes 1.0 to 2.0 times as long then (two of 306 at 0.95 and 0.97), with 257 to 383
// workgroups 0.78 to 1.08 times ([9580 x 6016] at 65 rows 35.9 / 42.7), with sixteen waves 0.76 to 1.2 times ([1380 x 11264] at 159 rows 16.7 / 22.0).
//
// A captured call, and one that finds the hand-off scratch in use on another stream, runs on the streaming kernel with as many shares of K in
// one workgroup of eight or sixteen waves (`twin`), which add to the same bits and need no scratch: hence two or four workgroups along
// K, and as many as give no fewer shares than the streaming kernel's own cut.
constexpr int GEMM_TILE_SPLIT_MIN_GROUPS = 5, GEMM_TILE_SPLIT_MAX = 4;
inline bool plan_gemm_tile_split(int64_t M, int64_t N, int64_t K, gemm_tile_cut* cut, gemm_skinny_cut* twin) {
	gemm_tile_cut c			  = plan_gemm_tile(M, N, K, false);
	const gemm_skinny_cut own = plan_gemm_skinny(M, N, K);
	const int groups		  = static_cast<int>(K / GROUP_K);
	const int64_t wgs		  = static_cast<int64_t>(c.grid_x) * c.grid_y;
	const auto can_double	  = [&] {
		const int shares = c.ks * c.kz * 2, longest = (groups + shares - 1) / shares;
		return c.ks == 4 && c.kz < GEMM_TILE_SPLIT_MAX && 10 * longest * shares <= 11 * groups && groups / (c.ks * c.kz * 2) >= GEMM_TILE_SPLIT_MIN_GROUPS &&
			wgs * c.kz * 2 * c.tm * 4096 <= GEMM_SPLIT_SCRATCH_FLOATS && wgs <= GEMM_SPLIT_MAX_UNITS;
	};
	while (can_double() && (wgs * c.kz * 2 <= 256 || c.ks * c.kz < own.splits * own.waves)) {
		c.kz *= 2;
	}
	if (c.tm != 2 || c.kz == 1 || wgs * c.kz <= 128 || c.ks * c.kz < own.splits * own.waves) {
		return false;
	}
	if (groups % (c.ks * c.kz) != 0 && ((wgs * c.kz > 256 && wgs * c.kz < 384) || own.waves != SK_WAVES)) {
		return false;
	}
	*cut  = c;
	*twin = gemm_skinny_cut{ own.ms, 1, c.ks * c.kz };
	return true;
}

// Up to 32 rows the kernel of q8_0_gemm_rows.hip, with the cut above, where it is the faster one.  Measured against the kernels that had these
// shapes (weights rotated, kernel times, us):
//   rows                4            16            32
//   [4096 x 4096]    5.7 /  9.8    6.3 /  9.1    8.7 /  9.4   (streaming kernel with eight waves' operand tiles from L2)
//   [1024 x 4096]    4.6 /  8.0    5.0 /  8.2    6.9 /  8.8
//   [4096 x 14336]  12.3 / 18.1   13.2 / 17.9   15.8 / 18.4
//   [14336 x 4096]  11.0 / 13.9   12.1 / 14.7   14.4 / 15.8
//   [128256 x 4096] 80.7 / 83.9   86.1 / 88.1  106   / 91     (tile kernel)
//   [28672 x 8192]  39.1 / 39.4   41.5 / 39.6   47   / 40
// Every wave takes its own copy of the activations out of L2 (requests per weight line, [4096 x 14336]: 1.27 at 4 rows, 1.53 at 16, 2.07 at
// 32), which the tile kernel shares over four strips (1.29 to 1.36): from 192 column blocks on, where that fills the chip by itself, this kernel has K up to 4096
// and 16 rows.  The line lies between the two K measured.
inline bool gemm_rows_suits(int64_t M, int64_t N, int64_t K) {
	const int64_t column_blocks = (N + 127) / 128;
	if (M > GEMM_ROWS_MAX) {
		return false;
	}
	return column_blocks < GEMM_STREAM_TILE_MIN_COLUMN_BLOCKS || (M <= 16 && K <= 4096);
}

// The shapes of 64 to 191 column blocks and 64 Mi weights and more that the tile kernel with K over workgroups has otherwise (plan_gemm):
// up to a workgroup per CU, and near two of them; between, some CUs have two and the launch takes as long as they do.  Measured, us, tile /
// rows kernel:
//   rows      [8192 x 8192]   [8192 x 14336]  [8192 x 28672]  [10240 x 8192]  [12288 x 12288]  [14336 x 14336]  [16384 x 4096]  [20480 x 8192]
//   17 to 24  18.6 / 15.6     28.5 / 23.8     46.2 / 42.5     22.0 / 23.5     32.2 / 34.0      41.2 / 40.8      17.7 / 15.0     37.5 / 35.0
//   25 to 32  18.2 / 15.8     28.6 / 25.1     45.7 / 45.3     22.1 / 25.2     32.3 / 36.8      41.4 / 43.8      17.8 / 15.9     37.8 / 38.0
// Near two workgroups per CU only while K is at most 15360: over 370 random shapes of 17 to 24 rows and 448 to 512 strips tile / rows is 0.97 to 1.3 up to
// there, 0.96 to 1.0 at 16384 and 0.89 to 1.07 beyond ([14655 x 27648] at 17 rows 69.2 / 77.6).  25 to 32 rows on up to 256 strips with K above
// 24576 only where the tile kernel has fewer than four workgroups along K, one per CU ([8192 x 27648] at 26 rows 55.9 / 44.4, but
// [8192 x 32768] at 28 rows 48.8 / 51.9).
// (sixteen rows would gain as well, 18.8 / 14.4 and 45.8 / 40.4 in the first and third column: tests/test_plan_cpu.py fixes their kernel)
inline bool gemm_rows_instead_of_tile(int64_t M, int64_t N, int64_t K, const gemm_tile_cut& tile) {
	const int64_t strips = (N + STRIP_ROWS - 1) / STRIP_ROWS;
	if (M <= 16 || M > GEMM_ROWS_MAX) {
		return false;
	}
	if (strips <= 256) {
		return M <= 24 || K <= 24576 || tile.kz < 4;
	}
	return M <= 24 ? strips >= 448 && K <= 15360 : strips >= 512 && K <= 4096;
}

// whether the rows kernel's tagged sums hold this cut
inline bool gemm_rows_fits(int64_t M, int64_t N, const gemm_skinny_cut& cut) {
	return cut.splits == 1 || (N + STRIP_ROWS - 1) / STRIP_ROWS * gemm_rows_operand(M) * cut.splits <= GEMV_MAX_SPLIT_UNITS;
}

// A mat-mat on tiled, already quantized operands (nh_q8_0_gemm_tiled, and the second half of nh_q8_0_mul_mat wherever the activations are quantized by a launch of their own).
struct gemm_plan {
	int kernel; // MM_GEMM_SKINNY, MM_GEMM_TILE_STREAM or MM_GEMM_TILE (MM_NOTHING for an empty problem)
	gemm_tile_cut tile; // when a tile kernel runs
	gemm_skinny_cut skinny; // when the streaming kernel runs, and when it stands in for the tile kernel with K over workgroups
	bool rows; // the streaming kernel's form for up to 32 rows, with the same cut
};
inline gemm_plan plan_gemm(int64_t M, int64_t N, int64_t K) {
	gemm_plan p{};
	if (M <= 0 || N <= 0 || K <= 0) {
		p.kernel = MM_NOTHING;
		return p;
	}
	// Few rows: the weights are read once and the kernel is HBM-bound.  Somewhat more rows than that, but so few
	// 128-row x 32-row tiles that the tile kernel would leave most SIMDs with one wave or none (measured: it needs
	// more than one workgroup per CU to pay): the same streaming kernel over groups of 64 rows, K split over the
	// waves of a workgroup, the weights coming from cache after the first group.
	const int64_t column_blocks	  = (N + 127) / 128;
	const int64_t tile_workgroups = column_blocks * ((M + 31) / 32);
	const int64_t weights		  = N * K;
	bool stream_tile			  = false;
	bool wide					  = false;
	if (M <= GEMM_SKINNY_MAX_M) {
		// A matrix with enough 128-row column blocks to occupy the chip by itself takes the tile kernel at any M: its four
		// waves share each activation tile through LDS, where the streaming kernel's eight waves fetch one each from L2 --
		// at 32 to 64 rows that is one to two times the weight bytes in extra traffic into every CU ([28672 x 8192] at
		// M = 16 / 32 / 64: 50 / 55 / 75 us streaming, 44 / 44 / 69 us on the tile kernel; [128256 x 8192]: 193 / - / 298
		// against 182 / - / 221 us).  Below that the tile kernel's grid leaves CUs idle ([14336 x 4096] at M = 64: 30 us
		// against 23 us) and the streaming kernel, which can split K over workgroups, stays.
		if (column_blocks >= GEMM_STREAM_TILE_MIN_COLUMN_BLOCKS) {
			stream_tile = !gemm_rows_suits(M, N, K);
		} else if (M > 32 ? (column_blocks >= 32 && weights >= (48ll << 20)) : (M >= 16 && column_blocks >= 64 && weights >= (64ll << 20))) {
			// Between the two, with K long enough to cut: the tile kernel with K over several workgroups per tile as well, so
			// that 32 to 191 column blocks still put a workgroup on every CU.  Measured against the streaming kernel:
			// [8192 x 28672] M = 64 / 32 / 16: 52 / 46 / 46 against 70 / 52 / 48 us; [8192 x 8192]: 23.7 / 18.0 / 17.6 against
			// 24.1 / 19.0 / 18.4; [14336 x 4096] M = 64: 20.5 against 22.9 (M = 32: 16.8 against 16.2, left where it was);
			// [4096 x 14336] M = 64: 24.0 against 26.2 (M = 16: 19.8 against 18.0); [1024 x 8192] M = 64: 13.5 against 11.7;
			// [4096 x 4096] M = 64: 13.6 against 10.3.  So: two row strips from 48 Mi weights on, one (16 rows or more) from
			// 64 Mi (17 to 32 rows of those mostly go on to the rows kernel, which this line was drawn before:
			// gemm_rows_instead_of_tile).  The rule only holds where that K split is actually possible: a shape whose groups do not divide (kz
			// stays 1) would run the tile kernel on 32 to 191 workgroups, the form measured slower than the streaming kernel
			// ([14336 x 4096] at M = 64 unsplit: 30 against 23 us), and stays with the streaming kernel.
			const gemm_tile_cut tile = plan_gemm_tile(M, N, K, true);
			stream_tile				 = tile.kz > 1;
			if (stream_tile && gemm_rows_instead_of_tile(M, N, K, tile)) {
				gemm_skinny_cut cut = plan_gemm_skinny(M, N, K);
				wide				= cut.splits * SK_WAVES < tile.ks * tile.kz; // no fewer shares of K than there
				cut.waves			= wide ? SK_WIDE_WAVES : cut.waves;
				stream_tile			= !gemm_rows_fits(M, N, cut); // K above 32768: the streaming kernel, 62.7 us at [8192 x 36864] and 24 rows, against 54.2
			}
		}
	}
	if (stream_tile) {
		p.kernel = MM_GEMM_TILE_STREAM;
		p.tile	 = gemm_tile_mat_mat(plan_gemm_tile(M, N, K, true), static_cast<int>(K / GROUP_K), (M + 31) / 32, true);
	} else if (M > GEMM_SKINNY_MAX_M && tile_workgroups <= 256 && plan_gemm_tile_split(M, N, K, &p.tile, &p.skinny)) {
		p.kernel = MM_GEMM_TILE;
	} else if (M <= GEMM_SKINNY_MAX_M || tile_workgroups <= 256) {
		p.kernel = MM_GEMM_SKINNY;
		p.skinny = plan_gemm_streaming(M, N, K);
		if (wide) {
			p.skinny.waves = SK_WIDE_WAVES;
		}
		p.rows = gemm_rows_suits(M, N, K) && gemm_rows_fits(M, N, p.skinny);
	} else {
		p.kernel = MM_GEMM_TILE;
		p.tile	 = gemm_tile_mat_mat(plan_gemm_tile(M, N, K, false), static_cast<int>(K / GROUP_K), (M + 31) / 32, false);
		p.tile.order = gemm_tile_order(p.tile, false, M, N, K);
	}
	return p;
}

// The prefill FFN's gate and up mat-mats with SiLU * up and the quantizer behind them: one launch of the tile kernel's fused form, or the
// two mat-mats and the quantizer as launches of their own (through an fp32 workspace).
//
// Up to 32 rows the pair runs as the rows kernel's fused form (gate_up_rows_suits), which cuts no strip's K over workgroups: matrices
// of enough strips only.  Measured against the three launches (us): [2 x 14336 x 4096] at 4 / 16 / 32 rows 20.9 / 22.5 / 26.3 against
// 31.8 / 33.0 / 36.0; [2 x 28672 x 8192] at 16 rows 79.8 against 84.9.
inline bool gate_up_rows_suits(int64_t M, int64_t n_ff, int64_t K) {
	if (M <= 0 || M > GEMM_ROWS_MAX || n_ff <= 0 || K <= 0 || n_ff % GROUP_K != 0 || K % GROUP_K != 0) {
		return false;
	}
	return plan_gemm_skinny(M, n_ff, K).splits == 1 && (M <= 16 || gemm_rows_suits(M, n_ff, K));
}
// Its shares of K, eight or sixteen: the streaming kernel's, or no fewer than the tile kernel has where it takes the mat-mats ([8192 x 8192] at
// 16 rows: 9.4e-8 from the sums in 64 bits there, 1.1e-7 here with eight).
inline int gate_up_rows_waves(int64_t M, int64_t n_ff, int64_t K) {
	const gemm_plan g = plan_gemm(M, n_ff, K);
	if (g.kernel == MM_GEMM_TILE_STREAM) {
		return g.tile.ks * g.tile.kz > SK_WAVES ? SK_WIDE_WAVES : SK_WAVES;
	}
	return g.kernel == MM_GEMM_SKINNY ? g.skinny.waves : plan_gemm_skinny(M, n_ff, K).waves;
}
// The tile kernel's fused form, K sets included, wherever its grid has the chip's SIMDs two waves each, or about one where the matrices are
// small enough that the launches saved count for more than idle CUs.  Whole calls, us, fused / three launches:
//   rows      [2 x 14336 x 4096]   [2 x 28672 x 8192]   [2 x 11008 x 4096]   [2 x 8192 x 8192]   [2 x 5632 x 2048]   [2 x 4096 x 1024]
//   64        34.8 / 43.5          114 / 116            31.1 / 47.9                              19.4 / 22.4         11.8 / 13.8
//   117, 128  56.5 / 62                                 52 / 54              60 / 86             20.5 / 31           15.4 / 19.7
//   256                                                                      102 / 111           30 / 35             13.0 / 25.5
// and below two waves per SIMD: [2 x 5632 x 4096] at 40 rows (1408 waves, 46 Mi weights) faster, but [2 x 6144 x 8192] at 64 rows
// (1536 waves, 101 Mi) not.
//
// The mat-mats it stands for have K in up to four times as many shares (grids of half the size, and K over workgroups), and fewer shares
// are longer sums: [8192 x 8192] at 64 rows 9.4e-8 from the sums in 64 bits with sixteen, 1.5e-7 with four.  So the sets take as many, in two passes,
// adding them in the mat-mats' order (same bytes), or in four with two sets (their tree of eight has no room for a second sum: the last
// bits differ).  A pass costs 2.5 us; two of four sets are the most that pays ([2 x 8192 x 8192] at 64 rows: four would be 53 us, three
// launches are 52).  K of at most 1024, 32 blocks, has nothing to gain: one pass, whatever the mat-mats do.
struct gate_up_cut {
	gemm_tile_cut tile;
	int passes; // passes * ks shares of K, ks at a time
	bool tree; // eight shares in two passes, added as the streaming kernel adds them
};
constexpr int64_t GATE_UP_MIN_WAVES = 2048, GATE_UP_MIN_WAVES_SMALL = 1100, GATE_UP_SMALL_WEIGHTS = 48ll << 20, GATE_UP_SHORT_K = 1024, GATE_UP_UNEVEN_MIN_GROUPS = 12;
// even: no more sets than K divides over; g: the mat-mats it stands for
inline bool plan_gate_up_with(bool even, const gemm_plan& g, int64_t M, int64_t n_ff, int64_t K, gate_up_cut* cut) {
	if (M <= 0 || n_ff <= 0 || K <= 0 || n_ff % GROUP_K != 0 || K % GROUP_K != 0) {
		return false;
	}
	gate_up_cut c{ {}, 1, false };
	c.tile			  = plan_gemm_tile(M, 2 * n_ff, K, false); // grid_x = n_ff / 64 workgroups of two gate and two up strips
	const int groups  = static_cast<int>(K / GROUP_K);
	while (even && groups % c.tile.ks != 0) {
		c.tile.ks /= 2;
	}
	while (g.kernel == MM_GEMM_TILE && c.tile.ks > 1 && groups % c.tile.ks != 0 && groups / c.tile.ks < GATE_UP_UNEVEN_MIN_GROUPS && int64_t{ 2 } * c.tile.ks * c.tile.grid_x * c.tile.grid_y >= 1024) {
		c.tile.ks /= 2; // K does not divide, the sets' shares are short, and half as many sets already have a wave on every SIMD ([2 x 6016 x 2176] at 231 rows, one set / two: 32.5 / 35.3 us)
	}
	const int64_t waves = int64_t{ 4 } * c.tile.ks * c.tile.grid_x * c.tile.grid_y;
	if (c.tile.tm == 1 && c.tile.ks > 2) {
		return false; // no such form: K above 32768, which the rows kernel would have to hand over
	}
	if (c.tile.ks == 1 && g.kernel == MM_GEMM_TILE && g.tile.kz == 1) {
		// a prompt: one set of waves per workgroup has all of K (the mat-mats alone may have two)
	} else if (waves < (2 * n_ff * K <= GATE_UP_SMALL_WEIGHTS ? GATE_UP_MIN_WAVES_SMALL : GATE_UP_MIN_WAVES)) {
		return false;
	} else {
		const bool tree	 = g.kernel == MM_GEMM_SKINNY || (g.kernel == MM_GEMM_TILE && g.tile.kz > 1);
		int shares		 = g.kernel == MM_GEMM_SKINNY ? g.skinny.splits * g.skinny.waves : g.tile.ks * g.tile.kz;
		if (g.kernel != MM_GEMM_SKINNY && g.tile.kz == 1) {
			// K does not divide over the mat-mats' sets: a second pass for the last bits only ([2 x 11008 x 4352] at 100 rows 49.4 -> 55.1 us, [2 x 24832 x 6912] at 40 rows
			// 79.8 -> 88.2), or no single launch at all where there is one set ([2 x 41856 x 13184] at 21 rows 196 us, three launches 231)
			while (groups % shares != 0) {
				shares /= 2;
			}
			shares = shares > c.tile.ks ? shares : c.tile.ks;
		} else if (g.kernel == MM_GEMM_TILE && shares > 2 * c.tile.ks && groups % shares != 0 && groups % c.tile.ks == 0) {
			// Sixteen shares that differ by a group, from K over workgroups: eight, if the streaming kernel would have no more, so that a pair which is one launch
			// with a K that sixteen divide is one here too.  ([2 x 768 x 11264] at 484 rows: 56 us, the three launches 49 through a workspace.)
			const gemm_skinny_cut own = plan_gemm_skinny(M, n_ff, K);
			shares					  = shares / 2 >= own.splits * own.waves ? shares / 2 : shares;
		}
		if (K > GATE_UP_SHORT_K) {
			c.passes = shares / c.tile.ks;
			c.tree	 = tree && c.tile.ks == 4;
			if (c.passes > 1 && (c.tile.ks == 1 || c.passes > (c.tile.ks == 4 ? 2 : 4))) {
				return false;
			}
			// Passes of sets that K does not divide over: two, with the longest share at most a quarter over the average.  (Sets that do divide K have had their passes
			// before and keep them, also where the shares of all passes differ: two sets in four, [2 x 9216 x 2304] at 58 rows, three groups for 2.25, 28.4 / 29.1.)
			// Fused / three launches, us: [2 x 11008 x 4224] at 48 rows (five groups for 4.1) 33.3 / 42.2, [2 x 6784 x 2816] at 50 rows (three for 2.75) 23.1 / 26.1, but [2 x 6912 x 3200] at 42 rows (four
			// for 3.1) 27.5 / 26.3, [2 x 6400 x 2304] at 58 rows (three for 2.25) 23.3 / 21.9, and in four passes [2 x 5504 x 2176] at 140 rows 40.7 / 36.8.
			// And with more than 64 rows a workgroup on more than half the CUs: over 630 random shapes the three launches take 1.09 to 1.7 times as long there, and
			// 0.6 to 1.25 times (mean 0.98) with up to 128 workgroups ([2 x 4096 x 5504] at 67 rows 35.8 / 30.6).  Of up to 64 rows with 70 to 128: 0.91 to 1.24, mean 1.06.
			const int64_t wgs = int64_t{ c.tile.grid_x } * c.tile.grid_y;
			if (c.passes > 1 && groups % c.tile.ks != 0 && (c.passes > 2 || 4 * ((groups + shares - 1) / shares * shares) > 5 * groups || (c.tile.grid_y > 1 && wgs <= 128))) {
				return false;
			}
		}
	}
	if (c.tile.ks <= 2) {
		gemm_tile_take_one_strip(&c.tile, (M + STRIP_ROWS - 1) / STRIP_ROWS, ONE_STRIP_GATE_UP);
	}
	c.tile.order = gemm_tile_order(c.tile, true, M, n_ff, K);
	if (cut) {
		*cut = c;
	}
	return true;
}
inline bool plan_gate_up_fused(int64_t M, int64_t n_ff, int64_t K, gate_up_cut* cut = nullptr) {
	const gemm_plan g = plan_gemm(M, n_ff, K);
	return plan_gate_up_with(false, g, M, n_ff, K, cut) || plan_gate_up_with(true, g, M, n_ff, K, cut);
}
inline bool gate_up_one_launch_beside(const gemm_skinny_cut& mat_mat, int64_t M, int64_t n_ff, int64_t K) {
	const gemm_plan g{ MM_GEMM_SKINNY, {}, mat_mat, false };
	return plan_gate_up_with(false, g, M, n_ff, K, nullptr) || plan_gate_up_with(true, g, M, n_ff, K, nullptr);
}

// The MFMA mat-vec's cut (q8_0_gemv_rows_mfma.hip): K over workgroups until a wave owns at most two groups (one with the
// sixteen-row operand: its register budget), within the split scratch's units (one per strip, activation row and split); matrices with few strips are cut
// further so that the launch reaches the CUs.  Under HIP graph capture: no K split (a replay could not renew the hand-off's epoch),
// a chunked walk instead.
constexpr int GEMV_ROWS_MFMA_MAX = 16;
inline gemv_plan plan_gemv_rows_mfma(int64_t strips, int64_t K, int rows, bool capturing) { // rows: 8 or 16, the kernel's operand rows
	gemv_plan p;
	p.strips	   = static_cast<int>(strips);
	p.groups	   = static_cast<int>(K / GROUP_K);
	p.splits	   = 1;
	auto tiles_for = [&](int sp) { return (p.groups + GEMV_WAVES * sp - 1) / (GEMV_WAVES * sp); };
	auto room	   = [&](int sp) { return strips * rows * sp <= GEMV_MAX_SPLIT_UNITS; };
	const int fit  = rows <= 8 ? 2 : 1; // groups of a wave's K range that its registers hold at once
	while (tiles_for(p.splits) > fit && room(p.splits * 2)) {
		p.splits *= 2;
	}
	// (a workgroup per CU, not per two as in the dot-product kernel: every workgroup quantizes its K range of all the rows, and that
	// work is what the launch waits for -- [4096 x 4096] at 8 rows: 9.8 us with 128 workgroups, 7.5 us with 256)
	while (strips * p.splits < 256 && tiles_for(p.splits) > 1 && room(p.splits * 2)) {
		p.splits *= 2;
	}
	if (capturing) {
		p.splits = 1;
	}
	p.tiles = tiles_for(p.splits);
	return p;
}

// The matrices it takes: up to sixteen rows on at most 40 MB, four on at most 80 MB (two and three rows stay on the dot-product kernel).
// nh_q8_0_mul_mat promises its callers that these leave their workspace untouched.
inline bool gemv_rows_mfma_suits(int64_t M, int64_t N, int64_t K) {
	return M >= 4 && M <= GEMV_ROWS_MFMA_MAX && N * (K / QK) * BLOCK_BYTES <= int64_t{ M == 4 ? 80 : 40 } << 20;
}
// Of those, the ones where it is the fastest form; the others run as a quantize launch and the kernel for up to 32 quantized rows where the
// caller has no such promise (nh_q8_0_mul_mat_scratch).  Every strip's workgroup quantizes all the rows again, which costs in proportion to M, and its
// sixteen waves have a CU to themselves, so a launch of more workgroups than CUs walks some of them one after the other.  Measured
// against those two launches (weights rotated, us, this / the two launches; workgroups, groups per wave):
//   9 to 16 rows   [4096 x 4096] 256, 1:  9.7 /  9.7 (12 rows 8.5 /  9.5)   [8192 x 2048] 256, 1:  8.6 /  9.0   [1024 x 14336] 256, 1: 10.4 / 10.4
//                  [6144 x 4096] 384, 1: 16.2 / 10.4   [2560 x 5120] 320, 1: 14.0 /  9.3   [4096 x 8192] 512, 1: 17.4 / 12.1
//   8 rows         [4096 x 4096] 256, 1:  7.6 /  9.2   [4096 x 6144] 256, 2:  9.5 / 10.1   [8192 x 4096] 256, 2: 11.0 / 10.5
//                  [5120 x 2560] 320, 1:  8.2 /  9.0   [6144 x 4096] 384, 1: 10.0 /  9.6   [5120 x 5120] 320, 2: 13.1 / 10.5
//   6 rows         [8192 x 4096] 256, 2:  9.9 / 10.5   [6144 x 4096] 384, 1:  9.3 /  9.5   [4608 x 4608] 288, 2: 11.2 /  9.9
//   4 rows         [4096 x 8192] 256, 2: 10.2 / 11.4   [6144 x 4096] 384, 1:  8.6 /  9.6   [4608 x 4608] 288, 2:  9.7 /  9.9
// Over 500 random shapes of 5 to 16 rows on the far side of the line the two launches are faster, 1.1 (5, 6 rows) to 1.6 times (13 to 16), but for ten
// within 6 %.  Four rows on matrices of up to 80 MB ([14336 x 4096] 15.5 / 14.5, [8192 x 8192] 17.8 / 16.0): a line drawn against the kernels
// before, which tests/test_plan_cpu.py fixes.
inline bool gemv_rows_mfma_fastest(int64_t M, int64_t N, int64_t K) {
	constexpr int64_t MIB	   = int64_t{ 1 } << 20;
	const int64_t weight_bytes = N * (K / QK) * BLOCK_BYTES;
	const gemv_plan p		   = plan_gemv_rows_mfma((N + STRIP_ROWS - 1) / STRIP_ROWS, K, M <= 8 ? 8 : 16, false);
	const bool one_round	   = p.strips * p.splits <= 256;
	if (M > 8) {
		return one_round;
	}
	return M == 4 || (one_round ? M <= 6 || weight_bytes <= 32 * MIB : p.tiles == 1 && (M <= 6 || weight_bytes <= 20 * MIB));
}

// nh_q8_0_mul_mat: fp32 activations [M][K] against a tiled weight [N][K].  scratch: nh_q8_0_mul_mat_scratch, whose workspace any shape may write.
struct mul_mat_plan {
	int kernel; // mul_mat_kernel
	int quantize_launch; // 1: the activations are quantized by a launch of their own into the caller's workspace
	gemv_plan gemv; // MM_GEMV, MM_GEMV_ROWS: strips, groups, K splits, groups per wave
	int gemv_row_parts; // MM_GEMV: workgroups that share a strip by rows (unsplit launches with fewer strips than CUs)
	gemm_plan gemm; // the MFMA kernels
};
// row parts per strip of an unsplit mat-vec launch: fewer strips than CUs (the 4096-row projections have 128, k/v 32) are cut
// into 2 or 4 row parts so that the launch reaches that many more CUs; what a single CU takes in per microsecond is limited,
// so half a chip cannot stream at the full HBM rate however many loads it has in flight.  (Between 129 and 255 strips -- q+k+v's 192 --
// two parts measured slower: 8.3 against 7.1 us with the norm in front.)
inline int plan_gemv_row_parts(const gemv_plan& p) {
	if (p.splits != 1 || p.tiles > 4) {
		return 1;
	}
	return p.strips * 2 <= 256 ? (p.strips * 4 <= 256 ? 4 : 2) : 1;
}
inline mul_mat_plan plan_mul_mat(int64_t M, int64_t N, int64_t K, bool scratch = false) {
	mul_mat_plan p{};
	if (M <= 0 || N <= 0 || K <= 0) {
		p.kernel = MM_NOTHING;
		return p;
	}
	if (M == 1) {
		p.kernel		 = MM_GEMV;
		p.gemv			 = plan_gemv((N + STRIP_ROWS - 1) / STRIP_ROWS, K);
		p.gemv_row_parts = plan_gemv_row_parts(p.gemv);
		return p;
	}
	if (gemv_rows_mfma_suits(M, N, K) && (!scratch || gemv_rows_mfma_fastest(M, N, K))) {
		p.kernel		 = MM_GEMV_ROWS_MFMA;
		p.gemv			 = plan_gemv_rows_mfma((N + STRIP_ROWS - 1) / STRIP_ROWS, K, M <= 8 ? 8 : 16, false);
		p.gemv_row_parts = 1;
		return p;
	}
	if (gemv_rows_suits(M, N, K)) {
		p.kernel		 = MM_GEMV_ROWS;
		p.gemv_row_parts = 1;
		return p;
	}
	p.quantize_launch = 1;
	p.gemm			  = plan_gemm(M, N, K);
	p.kernel		  = p.gemm.kernel;
	return p;
}

// A decode block as one launch (q8_0_decode_layer.hip): whether the shape takes that form, and how its stages are cut.
//
// gate/up: a wave holds two groups of each matrix at a time: one such chunk covers its share up to 4096 values of hidden state, two up to 8192.
//
// Down: K over workgroups until a wave's share is four groups, within the scratch.  Cut by rows instead where two workgroups per strip are what that makes anyway, they put a
// workgroup on every CU and a wave can hold its whole share of K (the LLaMA-3-8B block: 256 workgroups of 16 rows, seven half-size groups per wave): a finished row then leaves its
// workgroup directly, without the K-split hand-off's two trips through memory, on the path that ends the launch.  Measured at that block: 42.6 against 43.1 us (the stage behind the
// down projection 6.2 against 6.8 us).  As a launch of its own, or in the one-launch FFN, the same cut measured no different from the K split.
constexpr int CHAIN_TILES = 4; // groups a wave stages at once: LDS slices are sized for it
constexpr int CHAIN_DOWN_ROWS_TILES = 8; // ... in the down stage when it is cut by rows (half-size groups)
constexpr int CHAIN_CUS = 256;
struct decode_layer_plan {
	bool one_launch, one_chunk, down_by_rows;
	int splits; // workgroups per down strip
	int held; // down workgroups that hold their weight requests back a while
};
inline decode_layer_plan plan_decode_layer(int64_t n_embd, int64_t n_ff, int64_t next_strips) {
	decode_layer_plan p{};
	if (n_embd <= 0 || n_ff <= 0 || n_embd % GROUP_K != 0 || n_ff % GROUP_K != 0 || n_embd > CHAIN_MAX_EMBD || n_ff > FFN_MAX_HIDDEN) {
		return p;
	}
	const int strips_e = static_cast<int>(n_embd / STRIP_ROWS), groups_e = static_cast<int>(n_embd / GROUP_K), groups_f = static_cast<int>(n_ff / GROUP_K);
	const auto share   = [&] { return (groups_f + GEMV_WAVES * p.splits - 1) / (GEMV_WAVES * p.splits); };
	p.splits		   = 1;
	while (share() > CHAIN_TILES && strips_e <= GEMV_MAX_SPLIT_STRIPS && strips_e * p.splits * 2 <= GEMV_MAX_SPLIT_UNITS) {
		p.splits *= 2;
	}
	if (share() > CHAIN_TILES || next_strips < 0 || next_strips >= (1 << 20)) {
		return p;
	}
	p.one_launch   = true;
	p.one_chunk	   = (groups_e + GEMV_WAVES - 1) / GEMV_WAVES <= 2;
	p.down_by_rows = p.splits == 2 && strips_e * 2 <= 256 && (groups_f + GEMV_WAVES - 1) / GEMV_WAVES <= CHAIN_DOWN_ROWS_TILES;
	// A CU holds one workgroup.  The last round of gate/up strips leaves some CUs to the first down workgroups, whose weights, requested at once, take bandwidth from the strips that
	// everybody waits for: also where K goes over workgroups and the first of them have their activation early.  They hold their requests back, up to 4096 values of hidden state
	// (a fixed time, chosen at the [4096 / 14336] block: 41.35 us without, 40.8 with 4096 clocks, 40.45 with 6144).  117 random shapes within the lines below gain 1 to 5 %, mean 3.
	// Above 4096 values, whose strips take two chunks, it goes either way: 100 random shapes 0.98 to 1.03, mean 1.00 ([5760 / 21248] 79.9 / 81.5 us, [7296 / 22528] 109.2 / 107.0).
	// Not where they are the stage, all but an eighth (40 random shapes 0.95 to 1.04, mean 0.98; with more than 176 of them as well 0.89 to 1.03, mean 0.97), where there are more than
	// 176 and the stage takes a part of a second round (0.94 to 1.02, mean 0.96), nor for a handful (no different).  Either of the last two alone would gain as well (0.96 to 1.05,
	// mean 1.03) and is left out.  Nor behind a third round, by when the strips no longer change in step ([8192 / 28672] 143.1 / 143.9).
	const int down_wgs	  = strips_e * p.splits;
	const int rounds_left = static_cast<int>(n_ff / STRIP_ROWS) - (CHAIN_CUS - 1); // strips behind those that start with attn_out's end or before
	const int beside	  = (CHAIN_CUS - rounds_left % CHAIN_CUS) % CHAIN_CUS;
	if (p.one_chunk && rounds_left > 0 && rounds_left <= 2 * CHAIN_CUS && beside >= CHAIN_CUS / 16 && beside <= CHAIN_CUS * 11 / 16 && beside * 8 <= down_wgs * 7 &&
		(down_wgs <= CHAIN_CUS || down_wgs >= 2 * CHAIN_CUS)) {
		p.held = beside;
	}
	return p;
}

} // namespace nh
