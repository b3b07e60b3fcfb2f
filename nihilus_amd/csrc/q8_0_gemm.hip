// Prefill mat-mat C[m][n] = dot(W row n, Aq row m) for Q8_0 operands, gfx950, int8 MFMA.
//
// Same arithmetic as the mat-vec (reference vec_dot_q8_0_q8_0, cpu/avx_2.hpp:4534-4747) for M activation
// rows; output is [M][N] with n fastest (reference cpu/avx_2.hpp:4934; dims [ne0 = N, ne1 = M],
// common/kernel_traits.hpp:393-417).
//
// One v_mfma_i32_32x32x32_i8 covers exactly one 32-quant block of 32 activation rows x 32 weight rows, so its
// int32 result is the exact per-block sum for 1024 (m, n) pairs.  Because both operands carry a scale per
// block, the accumulator cannot run across blocks: every MFMA result is converted and folded into an fp32
// accumulator with the factor f32(dA[m][b]) * f32(dW[n][b]) (exact in fp32: two 11-bit significands).
//
// Operand lanes: lane l supplies row (l % 32), quants 16*(l/32)..+15 of the block -- the tiled layout stores
// tiles in exactly that order, so operands go from memory to the MFMA with one 16-byte load per lane and no
// shuffle.  Result lanes: register i of lane l is C[m = 8*(i/4) + 4*(l/32) + i%4][n = l % 32].
#include "q8_0_plan.h"

#include <type_traits>

namespace nh {

constexpr int GEMM_WAVES_M = 2; // waves along M in a workgroup
constexpr int GEMM_WAVES_N = 2; // waves along N
constexpr int GEMM_TM	   = 2; // 32-row MFMA tiles per wave along M
constexpr int GEMM_TN	   = 2; // along N
constexpr int GEMM_BM	   = GEMM_WAVES_M * GEMM_TM * 32; // 128
constexpr int GEMM_BN	   = GEMM_WAVES_N * GEMM_TN * 32; // 128
constexpr int GEMM_THREADS = GEMM_WAVES_M * GEMM_WAVES_N * 64;

// 16 operand bytes for (row strip, block b): lane supplies row strip*32 + lane%32, half lane/32.
template<bool TILED> __device__ __forceinline__ v4i load_operand(const uint8_t* base, int rows, int nb, int strip, int b, int lane) {
	if constexpr (TILED) {
		return *reinterpret_cast<const v4i*>(base + macro_offset(strip, b / GROUP_BLOCKS, nb / GROUP_BLOCKS) + (b % GROUP_BLOCKS) * TILE_BYTES + 16 * lane);
	} else {
		const int row = min(strip * STRIP_ROWS + (lane & 31), rows - 1); // padding rows re-read the last row; dropped at the store
		return load16_unaligned(base + (static_cast<int64_t>(row) * nb + b) * BLOCK_BYTES + 2 + 16 * (lane >> 5));
	}
}
template<bool TILED> __device__ __forceinline__ float load_scale(const uint8_t* base, int rows, int nb, int row, int b) {
	if constexpr (TILED) {
		return half_bits_to_float(load_u16(base + macro_offset(row / STRIP_ROWS, b / GROUP_BLOCKS, nb / GROUP_BLOCKS) + MACRO_D_OFFSET + 8 * (row % STRIP_ROWS) + 2 * (b % GROUP_BLOCKS)));
	} else {
		return half_bits_to_float(load_u16(base + (static_cast<int64_t>(min(row, rows - 1)) * nb + b) * BLOCK_BYTES));
	}
}

template<bool TILED, bool DUMP>
__global__ __launch_bounds__(GEMM_THREADS) void gemm_kernel(const uint8_t* __restrict__ W, const uint8_t* __restrict__ A, float* __restrict__ C, int32_t* __restrict__ sums, int M, int N, int K) {
	__shared__ float a_scale[GROUP_BLOCKS][GEMM_BM]; // f32(dA) for this workgroup's rows, current 4 blocks
	__shared__ float w_scale[GROUP_BLOCKS][GEMM_BN];

	const int nb	   = K / QK;
	const int m_strips = (M + 31) / 32;
	const int n_strips = (N + 31) / 32;
	const int tid	   = threadIdx.x;
	const int lane	   = tid & 63;
	const int wave	   = tid >> 6;
	const int wm	   = wave / GEMM_WAVES_N;
	const int wn	   = wave % GEMM_WAVES_N;
	const int half	   = lane >> 5;
	const int m0	   = blockIdx.y * GEMM_BM; // first activation row of the workgroup
	const int n0	   = blockIdx.x * GEMM_BN;

	float acc[GEMM_TM][GEMM_TN][16];
#pragma unroll
	for (int i = 0; i < GEMM_TM; ++i) {
#pragma unroll
		for (int j = 0; j < GEMM_TN; ++j) {
#pragma unroll
			for (int e = 0; e < 16; ++e) {
				acc[i][j][e] = 0.0f;
			}
		}
	}

	for (int b0 = 0; b0 < nb; b0 += GROUP_BLOCKS) {
		// ---- scales of the next four blocks for all rows of the workgroup tile, as fp32, via LDS ----
		__syncthreads();
		for (int i = tid; i < GROUP_BLOCKS * GEMM_BM; i += GEMM_THREADS) {
			const int t = i / GEMM_BM, rr = i % GEMM_BM;
			const int b = b0 + t, row = m0 + rr;
			a_scale[t][rr] = (b < nb && row < m_strips * 32 && (TILED || row < M)) ? load_scale<TILED>(A, M, nb, row, b) : 0.0f;
		}
		for (int i = tid; i < GROUP_BLOCKS * GEMM_BN; i += GEMM_THREADS) {
			const int t = i / GEMM_BN, rr = i % GEMM_BN;
			const int b = b0 + t, row = n0 + rr;
			w_scale[t][rr] = (b < nb && row < n_strips * 32 && (TILED || row < N)) ? load_scale<TILED>(W, N, nb, row, b) : 0.0f;
		}
		__syncthreads();

#pragma unroll
		for (int t = 0; t < GROUP_BLOCKS; ++t) {
			const int b = b0 + t;
			if (b >= nb) {
				break;
			}
			v4i a[GEMM_TM], w[GEMM_TN];
#pragma unroll
			for (int i = 0; i < GEMM_TM; ++i) {
				const int strip = m0 / 32 + wm * GEMM_TM + i;
				a[i]			= strip < m_strips ? load_operand<TILED>(A, M, nb, strip, b, lane) : v4i{ 0, 0, 0, 0 };
			}
#pragma unroll
			for (int j = 0; j < GEMM_TN; ++j) {
				const int strip = n0 / 32 + wn * GEMM_TN + j;
				w[j]			= strip < n_strips ? load_operand<TILED>(W, N, nb, strip, b, lane) : v4i{ 0, 0, 0, 0 };
			}
#pragma unroll
			for (int i = 0; i < GEMM_TM; ++i) {
#pragma unroll
				for (int j = 0; j < GEMM_TN; ++j) {
					const v16i zero = { 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0 };
					const v16i s	= __builtin_amdgcn_mfma_i32_32x32x32_i8(a[i], w[j], zero, 0, 0, 0);
					const int ml	= (wm * GEMM_TM + i) * 32; // tile's first row inside the workgroup tile
					const int nl	= (wn * GEMM_TN + j) * 32 + (lane & 31);
					const float dw	= w_scale[t][nl];
#pragma unroll
					for (int e = 0; e < 16; ++e) {
						const int mr = ml + 8 * (e >> 2) + 4 * half + (e & 3);
						if constexpr (DUMP) {
							const int m = m0 + mr, n = n0 + nl;
							if (m < M && n < N) {
								sums[(static_cast<int64_t>(m) * N + n) * nb + b] = s[e];
							}
						} else {
							acc[i][j][e] = fmaf(static_cast<float>(s[e]), a_scale[t][mr] * dw, acc[i][j][e]);
						}
					}
				}
			}
		}
	}

	if constexpr (!DUMP) {
#pragma unroll
		for (int i = 0; i < GEMM_TM; ++i) {
#pragma unroll
			for (int j = 0; j < GEMM_TN; ++j) {
				const int n = n0 + (wn * GEMM_TN + j) * 32 + (lane & 31);
#pragma unroll
				for (int e = 0; e < 16; ++e) {
					const int m = m0 + (wm * GEMM_TM + i) * 32 + 8 * (e >> 2) + 4 * half + (e & 3);
					if (m < M && n < N) {
						C[static_cast<int64_t>(m) * N + n] = acc[i][j][e];
					}
				}
			}
		}
	}
}

// ---------------------------------------------------------------------------------------------------------
// The prefill kernel for the tiled layout.
//
// Both operands carry a scale per 32-quant block, so each 32x32x32 int8 MFMA result (1024 exact block sums, 16 per
// lane) has to be converted and folded into the fp32 accumulator before the next block: 16 conversions + 16
// multiply-adds per lane per MFMA.  Measured on this part, a SIMD retires one wave64 VALU instruction per ~2.5 cycles
// once it holds two or more waves (a lone wave issues one per ~4-5), and MFMA and VALU time add on a SIMD, also across
// waves: a (tile, block) costs 32 + 32 matrix-pipe cycles plus 32 x 2.5 VALU cycles, ~145 cycles against the 32 of the int8
// MFMA alone.  That is the ceiling (~22 % of the int8 MFMA peak); the kernel is shaped to add as little as possible:
//   * the scale products f32(dA[m][b]) * f32(dW[n][b]) are formed on the matrix pipe: one v_mfma_f32_32x32x8_f16 whose
//     operands are the two blocks' fp16 scales as stored, each in the k = 0 slot ({d, 0, 0, 0}; lanes 32..63 supply
//     the k = 4..7 slots = 0).  The product of two fp16 values is exact in fp32 (fp16 subnormals included) and lands
//     in the int8 MFMA's own accumulator layout: no conversion, broadcast or cross-lane move of a scale, ever;
//   * only the operand that is shared goes through LDS.  A workgroup is four waves; wave w owns weight strip
//     4*blockIdx.x + w and loads its tiles straight from global memory into registers (one coalesced 16-byte-per-lane
//     load per tile, already an MFMA operand, a whole 128-quant group ahead of use); all four waves share the same
//     TM activation strips, copied global -> LDS one group ahead (double-buffered, one barrier per group, the copy
//     spread over the four waves) and read back as conflict-free 16-byte-per-lane operand images plus one 8-byte read of a
//     group's four scales per strip;
//   * every global address is a wave-uniform base in scalar registers plus a 32-bit lane offset (the addressing mode of
//     global_load with a scalar base): no 64-bit address arithmetic on the VALU, which is the pipe the fold saturates,
//     and ~10 fewer registers than per-lane pointers (the difference between spilling and not at two activation strips);
//   * latency is hidden by occupancy, not by a software pipeline: one result-register set per tile keeps the kernel
//     at <= 128 VGPRs, four workgroups per CU, four waves per SIMD.  (A two-result-set, software-pipelined variant
//     at two waves per SIMD measured 8 % slower: with so few waves the SIMD falls back to the lone-wave issue rate
//     whenever one of them waits.)
// a 64-bit offset that the compiler may keep in scalar registers (it is the same for every lane of the wave)
__device__ __forceinline__ int64_t uniform_i64(int64_t v) {
	const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v)), hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(static_cast<uint64_t>(v) >> 32));
	return static_cast<int64_t>((static_cast<uint64_t>(hi) << 32) | lo);
}

typedef const __attribute__((address_space(1))) uint8_t* gptr_u8;
// base + wave-uniform offset as a pointer the compiler must keep in scalar registers (and cannot fold the lane offset into)
__device__ __forceinline__ gptr_u8 scalar_base(const uint8_t* base, int64_t uniform_off) {
	gptr_u8 p = (gptr_u8)(base) + uniform_off;
	asm volatile("" : "+s"(p));
	return p;
}
template<typename T, bool NT> __device__ __forceinline__ T load_sv(gptr_u8 p, uint32_t lane_off) {
	typedef const __attribute__((address_space(1))) T* gp;
	if constexpr (NT) {
		return __builtin_nontemporal_load(reinterpret_cast<gp>(p + lane_off));
	} else {
		return *reinterpret_cast<gp>(p + lane_off);
	}
}

// GATE_UP: the prefill FFN's first half as ONE launch (the reference's mega_ffn composite: ffn_gate and ffn_up mul_mat -> silu ->
// mul -> activation operand of ffn_down, infra/core_traits.hpp:976-989).  Waves 0, 1 of a workgroup take strips 2 * blockIdx.x + {0, 1}
// of W (gate), waves 2, 3 the SAME strips of W2 (up), all four against the one activation image in LDS; the loop is the plain
// kernel's.  Behind it the up waves hand their tiles to the gate waves through LDS, and those apply silu(g) * u and quantize: a
// 32-value block of the down projection's activation is one activation row against one 32-row weight strip, i.e. one (register,
// half-wave) of an MFMA result tile -- 32 lanes hold it, its maximum is five cross-lane steps, and the quants go out in the tiled
// operand layout (through an LDS image of the tile, one 16-byte store per lane).  With several K sets the sets' tiles are summed first, as
// in the plain kernel, and each set finishes the rows it has summed.  The two fp32 [M x N] intermediates are never
// written, the activation is read once for both matrices, and two launches (the second mat-mat and the SiLU * up quantizer) are gone.
// The arithmetic per value is that of the stand-alone kernels (silu_mul, quantize_row_q8_0), and where they add up K in more shares than
// the launch has sets, the sets take the shares in PASSES, each ending in the sum over the sets (gate_up_cut in q8_0_plan.h: 2.5 us a pass,
// with the next pass's first group on its way meanwhile; fetched behind the sum it was 4).
// C / C2 (optional, inspection): the fp32 gate / up tiles as the launch computed them.
template<int TM, bool DUMP, int KS, bool STREAM, bool SPLIT, bool GATE_UP, bool PASSES = false>
__device__ __forceinline__ void gemm_tiled_body(const uint8_t* __restrict__ W, const uint8_t* __restrict__ A, float* C, const float* R, int32_t* __restrict__ sums, int M, int N, int groups,
	float* __restrict__ partials, unsigned* __restrict__ counters, const uint8_t* __restrict__ W2, uint8_t* __restrict__ act_out, float* __restrict__ C2, int order, int passes = 1, bool tree = false) {
	static_assert(!SPLIT || (KS > 1 && !DUMP), "K over several workgroups continues the K sets' sum");
	static_assert(!GATE_UP || (!DUMP && !SPLIT), "the fused gate/up form leaves a workgroup's tile quantized");
	constexpr int STAGE_BYTES = TM * MACRO_BYTES; // the activation strips' macro-tiles of a group, as in memory
	constexpr int SET_BYTES	  = 2 * STAGE_BYTES + 256; // + 256: where waves that copy no scale table put theirs
	constexpr int PARK_BYTES   = KS > 1 ? KS * 4 * (KS - 1) * (16 * TM / KS) * 64 * 4 : 0; // the final sum over the K sets, below
	// GATE_UP epilogue: two up tiles per activation strip as fp32, then per gate wave TM tile images and TM x 32 scales
	constexpr int XCH_BYTES	   = GATE_UP ? 2 * TM * 16 * 64 * 4 : 0;
	constexpr int FUSE_BYTES   = GATE_UP ? XCH_BYTES + 2 * TM * (TILE_BYTES + 64) : 0;
	constexpr int LDS_BASE	   = KS * SET_BYTES > PARK_BYTES ? KS * SET_BYTES : PARK_BYTES;
	constexpr int SAVE_AT	   = LDS_BASE > FUSE_BYTES ? LDS_BASE : FUSE_BYTES; // the passes' sums so far, every value where its lane put it
	constexpr int LDS_BYTES	   = SAVE_AT + (PASSES ? 4 * TM * 16 * 64 * 4 : 0);
	static_assert(!PASSES || (GATE_UP && KS > 1));
	__shared__ __align__(16) uint8_t lds_raw[LDS_BYTES];
	typedef _Float16 v4h __attribute__((ext_vector_type(4)));

	const int tid	   = threadIdx.x;
	const int lane	   = tid & 63;
	const int wave_all = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int wave	   = wave_all & 3; // which of the workgroup's four weight strips
	const int kr	   = wave_all >> 2; // which K range
	uint8_t* lds	   = lds_raw + kr * SET_BYTES;
	// Which share of K a set has, of KS * gridDim.z (or, in PASSES, KS in each pass).  With K over workgroups in the shapes that the streaming kernel
	// can take too, the one that makes the sums below the tree that kernel adds its eight or sixteen waves' shares in (0 4 2 6 / 1 5 3 7,
	// then the same of 8 to 15), and its cut of K.  The shares differ by a group where K does not divide: every set of a workgroup walks as
	// many groups as the longest (they meet at a barrier behind each), the last of a shorter one with zero scales.
	constexpr bool TREE = SPLIT && !STREAM;
	static_assert(!TREE || KS == 4);
	const int z	= SPLIT ? static_cast<int>(blockIdx.z) : 0;
	const int zs = SPLIT ? static_cast<int>(gridDim.z) : 1;
	// this set's first group and number of groups (in this pass), and its first group in the next pass; g_len: the most groups any set has
	int g0 = 0, live = groups, g_len = groups, after = 0;
	auto begin_pass = [&](int pass) {
		const int shares	= KS * (PASSES ? passes : zs);
		const auto share_of = [&](int p) {
			if (TREE) {
				return 8 * (z >> 1) + (z & 1) + 4 * (kr & 1) + 2 * (kr >> 1);
			}
			return PASSES && tree ? p + 4 * (kr & 1) + 2 * (kr >> 1) : (PASSES ? p : z) * KS + kr;
		};
		const auto range = [&](int share, int& from, int& to) {
			if (TREE) {
				wave_k_range(groups, shares >> 4, share >> 3, 8, share & 7, from, to);
			} else {
				wave_k_range(groups, 0, 0, shares, share, from, to);
			}
		};
		int g1, unused;
		range(share_of(pass), g0, g1);
		live  = g1 - g0;
		g_len = (groups + shares - 1) / shares;
		after = g1 - 1;
		if (PASSES && pass + 1 < passes) {
			range(share_of(pass + 1), after, unused);
		}
	};
	if constexpr (KS > 1) {
		begin_pass(0);
	}
	const int half	   = lane >> 5;
	const int m_strips = (M + 31) / 32;
	const int n_strips = (N + 31) / 32;
	int bx = blockIdx.x, by = blockIdx.y; // block of weight strips, group of activation strips
	if constexpr (!SPLIT && !STREAM) {
		// three permutations of the grid; which one, and why: gemm_tile_order in q8_0_plan.h
		const unsigned gx = static_cast<unsigned>(GATE_UP ? (n_strips + 1) / 2 : (n_strips + 3) / 4), gy = static_cast<unsigned>(m_strips + TM - 1) / TM;
		if (order > TILE_ORDER_XCD) { // bands of that many column blocks
			const unsigned b = static_cast<unsigned>(order), id = by * gx + bx, first = id / (b * gy) * b;
			const unsigned r = id - first * gy, width = min(b, gx - first); // the last band may be narrower
			by				 = __builtin_amdgcn_readfirstlane(static_cast<int>(r / width));
			bx				 = __builtin_amdgcn_readfirstlane(static_cast<int>(first + r % width));
		} else if (order == TILE_ORDER_XCD) {
			const unsigned total = gx * gy, id = by * gx + bx, xcd = id % 8;
			const unsigned t	 = xcd * (total / 8) + min(xcd, total % 8) + id / 8; // XCDs 0 .. total % 8 - 1 have one more
			bx					 = __builtin_amdgcn_readfirstlane(static_cast<int>(t / gy));
			by					 = __builtin_amdgcn_readfirstlane(static_cast<int>(t % gy));
		}
	}
	const int ms0	   = by * TM;
	const int ns	   = GATE_UP ? bx * 2 + (wave & 1) : bx * 4 + wave;
	const uint8_t* Wm  = (GATE_UP && wave >= 2) ? W2 : W; // wave-uniform
	// every address below is a wave-uniform part (scalar registers, advanced by scalar adds) plus one of three lane constants
	uint32_t lane16 = 16u * lane;
	const int64_t w_off	  = uniform_i64(macro_offset(min(ns, n_strips - 1), 0, groups));
	struct w_regs {
		v4i q[GROUP_BLOCKS];
		v2u d;
	};
	// activations: global -> registers -> LDS, shared out over the four waves: wave w moves tiles TM*w .. TM*w+TM-1 of the
	// TM*4 tiles of a group, waves 0..TM-1 also the 256-byte scale table of strip w
	int64_t a_off[TM];
	uint32_t a_dst[TM];
#pragma unroll
	for (int j = 0; j < TM; ++j) {
		const int u = TM * wave + j;
		a_off[j]	= uniform_i64(macro_offset(min(ms0 + u / 4, m_strips - 1), 0, groups) + (u % 4) * TILE_BYTES);
		a_dst[j]	= (u / 4) * MACRO_BYTES + (u % 4) * TILE_BYTES; // + 16 * lane at the store
	}
	// every wave copies a dword per lane of a scale table (waves >= TM: strip TM-1's again, stored nowhere), so that all waves
	// issue the same loads
	const int64_t sc_off  = uniform_i64(macro_offset(min(ms0 + min(wave, TM - 1), m_strips - 1), 0, groups) + MACRO_D_OFFSET);
	const uint32_t sc_dst = wave < TM ? wave * MACRO_BYTES + MACRO_D_OFFSET : 2 * STAGE_BYTES; // + 4 * lane at the store
	const uint32_t sc_stage = wave < TM ? STAGE_BYTES : 0; // the spare area is not staged
	struct a_regs {
		v4i q[TM];
		uint32_t d;
	};
	auto fetch_a = [&](int g, a_regs& r) {
		const int64_t adv = static_cast<int64_t>(g0 + g) * MACRO_BYTES;
		asm volatile("" : "+v"(lane16));
		const uint32_t l4 = lane16 >> 2;
#pragma unroll
		for (int j = 0; j < TM; ++j) {
			r.q[j] = load_sv<v4i, false>(scalar_base(A, a_off[j] + adv), lane16);
		}
		r.d = load_sv<uint32_t, false>(scalar_base(A, sc_off + adv), l4);
	};
	auto stash_a = [&](int stage, const a_regs& r) {
		uint8_t* p	 = lds + stage * STAGE_BYTES;
		asm volatile("" : "+v"(lane16)); // wave-uniform offsets stay in scalar registers, added here, instead of one more lane constant each
#pragma unroll
		for (int j = 0; j < TM; ++j) {
			*reinterpret_cast<v4i*>(p + a_dst[j] + lane16) = r.q[j];
		}
		*reinterpret_cast<uint32_t*>(lds + stage * sc_stage + sc_dst + (lane16 >> 2)) = r.d;
	};
	auto fetch_w = [&](int g, w_regs& r) {
		const int64_t at = w_off + static_cast<int64_t>(g0 + g) * MACRO_BYTES;
		const gptr_u8 p	 = scalar_base(Wm, at);
		asm volatile("" : "+v"(lane16));
		const uint32_t l8 = (lane16 & 0x1F0u) >> 1; // the widening of a lane offset has to stay beside its loads for scalar base + 32-bit lane offset to be picked as the addressing mode
		r.d = load_sv<v2u, STREAM>(scalar_base(Wm, at + MACRO_D_OFFSET), l8);
		__builtin_amdgcn_sched_barrier(0); // in the trips' order: their waits are counts of what was requested behind
#pragma unroll
		for (int k = 0; k < GROUP_BLOCKS; ++k) {
			r.q[k] = load_sv<v4i, STREAM>(p + k * TILE_BYTES, lane16);
		}
	};
	// load number p of a group's set (PIECES of them: TM activation tiles, their scale dword, the weights' scales, four weight tiles);
	// the same loads as fetch_a and fetch_w, which the prologue issues in one go
	constexpr int PIECES = TM + 2 + GROUP_BLOCKS;
	constexpr int UNITS	 = GROUP_BLOCKS * TM; // of a trip: (block t, activation strip i) in the order u = TM * t + i
	// (The next trip's weights go to a second set of registers.  Into those of the tile each follows, once its last MFMA is issued, was 112 registers instead of 126
	// and no faster: [14336 x 4096] at 3001 rows 426.1 us against 424.3, [4096 x 14336] at 512 rows 78.5 / 78.1, [128256 x 4096] at 24 rows
	// 93.2 / 91.4, gate / up [2 x 41856 x 13184] at 21 rows 195.4 / 190.6; launches in random order.)
	auto fetch_piece = [&](int p, int in_pass, a_regs& ra, w_regs& rw) {
		const int g = g0 + in_pass;
		asm volatile("" : "+v"(lane16)); // in place: a copy for every load was one VALU instruction each
		if (p < TM) {
			ra.q[p] = load_sv<v4i, false>(scalar_base(A, a_off[p] + static_cast<int64_t>(g) * MACRO_BYTES), lane16);
		} else if (p == TM) {
			ra.d = load_sv<uint32_t, false>(scalar_base(A, sc_off + static_cast<int64_t>(g) * MACRO_BYTES), lane16 >> 2);
		} else if (p == TM + 1) { // in front of the tiles: the trip's first unit needs it, and waits for what was requested before it
			rw.d = load_sv<v2u, STREAM>(scalar_base(Wm, w_off + static_cast<int64_t>(g) * MACRO_BYTES + MACRO_D_OFFSET), (lane16 & 0x1F0u) >> 1);
		} else {
			const int k = p - TM - 2;
			rw.q[k] = load_sv<v4i, STREAM>(scalar_base(Wm, w_off + static_cast<int64_t>(g) * MACRO_BYTES + k * TILE_BYTES), lane16);
		}
	};
	v16f acc[TM];
#pragma unroll
	for (int i = 0; i < TM; ++i) {
		acc[i] = v16f{ 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0 };
	}
	int last = live - 1;

	w_regs wa, wb;
	a_regs pre;
	fetch_a(0, pre);
	fetch_w(0, wa);
	stash_a(0, pre);
	__syncthreads();
	// One trip = one 128-quant group.  Requested during it: the next group's activation tiles, then its weight tiles -- in
	// that order, because loads return in issue order: the (cached) activations are needed at the trip's end, for the barrier,
	// and must not queue behind weights that have until the next trip to arrive.  The requests are spread over the trip's
	// units, one or two behind each unit's LDS read: issued together at the trip's start, the sixteen waves of a CU that
	// leave the barrier at the same moment queue at the memory pipeline (0.4 to 2 k cycles per wave and trip before its first
	// MFMA).  Past the end the last group is requested again (a cache hit that nobody uses): every trip issues the same
	// loads, so every wait the compiler places is a count (a load under a condition makes it wait for everything
	// outstanding instead).
	auto trip = [&](int g, w_regs& cur, w_regs& nxt) {
		// (with another pass to come: its first group, on its way while this pass is summed)
		const int gn = PASSES ? (g < last ? g + 1 : after - g0) : min(g + 1, last);
		// (past the end of a set's share, where another set has one group more: zero scales on both sides add nothing)
		const bool zero = KS > 1 ? half || g >= live : half;
		const v2u wd = zero ? v2u{ 0u, 0u } : cur.d;
		const uint8_t* stage = lds + (g & 1) * STAGE_BYTES;
		asm volatile("" : "+v"(lane16));
		const uint8_t* a_at = stage + lane16;
		// the rows' scales of the group's four blocks, one 8-byte read per strip and trip (a half-word read per unit was eight: [8192 x 8192] at 512 rows
		// 94.4 -> 92.3 us, [4096 x 14336] at 117 rows 30.4 -> 29.4, one strip [128256 x 4096] at 24 rows 90.8 -> 91.8)
		v2u a_sc[TM];
#pragma unroll
		for (int i = 0; i < TM; ++i) {
			const v2u d = *reinterpret_cast<const v2u*>(stage + i * MACRO_BYTES + MACRO_D_OFFSET + ((lane16 >> 1) & 0xF8u));
			a_sc[i]		= zero ? v2u{ 0u, 0u } : d;
		}
		// the operand of unit u + 1 is read from LDS before unit u's arithmetic starts: one exposed LDS latency per trip, not eight
		auto read_a = [&](int u) { return *reinterpret_cast<const v4i*>(a_at + (u % TM) * MACRO_BYTES + (u / TM) * TILE_BYTES); };
		v4i a_cur = read_a(0);
#pragma unroll
		for (int u = 0; u < UNITS; ++u) {
			const int t = u / TM, i = u % TM;
			v4i a_nxt		= a_cur;
			if (u + 1 < UNITS) {
				a_nxt = read_a(u + 1);
			}
			__builtin_amdgcn_sched_barrier(0);
#pragma unroll
			for (int pc = u * PIECES / UNITS; pc < (u + 1) * PIECES / UNITS; ++pc) {
				fetch_piece(pc, gn, pre, nxt);
			}
			__builtin_amdgcn_sched_barrier(0);
			const v2u w_slot  = scale_slot(wd, t), a_slot = scale_slot(a_sc[i], t);
			const v16i zi	  = { 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0 };
			const v16f zf	  = { 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0 };
			const v16i sv	  = __builtin_amdgcn_mfma_i32_32x32x32_i8(a_cur, cur.q[t], zi, 0, 0, 0);
			if constexpr (DUMP) {
				const int n = ns * 32 + (lane & 31);
#pragma unroll
				for (int e = 0; e < 16; ++e) {
					const int m = (ms0 + i) * 32 + 8 * (e >> 2) + 4 * half + (e & 3);
					if (m < M && n < N) {
						sums[(static_cast<int64_t>(m) * N + n) * (groups * GROUP_BLOCKS) + g * GROUP_BLOCKS + t] = sv[e];
					}
				}
			} else {
				const v16f pv = __builtin_amdgcn_mfma_f32_32x32x8f16(__builtin_bit_cast(v4h, a_slot), __builtin_bit_cast(v4h, w_slot), zf, 0, 0, 0);
#pragma unroll
				for (int e = 0; e < 16; ++e) {
					acc[i][e] = fmaf(static_cast<float>(sv[e]), pv[e], acc[i][e]);
				}
				asm volatile("" : "+v"(acc[i]));
			}
			__builtin_amdgcn_sched_barrier(0);
			a_cur = a_nxt;
		}
		stash_a((g + 1) & 1, pre);
		__syncthreads();
	};
	constexpr int PER = 16 / KS; // values of a lane's 16 per strip that a K set finishes: registers PER * kr .. PER * kr + PER - 1
	float mine[TM * PER]; // this wave's share of the workgroup's tile (SPLIT: of its part of K)
	for (int pass = 0;; ++pass) {
		for (int g = 0; g < g_len; g += 2) {
			trip(g, wa, wb);
			if (g + 1 < g_len) {
				trip(g + 1, wb, wa);
			}
		}
		if constexpr (KS > 1 && !DUMP) {
			// The K sets' tiles are summed by all of them at once: set q keeps PER = 16 / KS of a lane's 16 values per strip (with
			// four sets: rows 8q .. 8q+7 of every 32-row strip), parks the other sets' shares in LDS, and after one barrier adds what
			// the others parked for it, in set order (s0 + s1 + s2 + s3 whatever q is, so the result does not depend on who adds),
			// and stores its own rows.  One set adding the others' whole tiles in turn took 12 % of the launch at M=512, N=K=4096.
			__syncthreads(); // every set is through with its stages
			float* park = reinterpret_cast<float*>(lds_raw);
			int own		= lane;
			if constexpr (PASSES) {
				asm volatile("" : "+v"(own)); // the addresses are worked out here, not kept in registers that the trips need
			}
			auto slot	= [&](int q, int src) { // where set src parks its share of part q (src != q), this wave's strip
				return park + ((((q * 4 + wave) * (KS - 1)) + (src < q ? src : src - 1)) * (PER * TM)) * 64 + own;
			};
#pragma unroll
			for (int q = 0; q < KS; ++q) {
				if (q != kr) {
					float* dst = slot(q, kr);
#pragma unroll
					for (int i = 0; i < TM; ++i) {
#pragma unroll
						for (int e = 0; e < PER; ++e) {
							dst[(i * PER + e) * 64] = acc[i][q * PER + e];
						}
					}
				}
			}
			float* save = reinterpret_cast<float*>(lds_raw + (PASSES ? SAVE_AT : 0)) + wave_all * (TM * PER * 64) + own;
			const int n = ns * 32 + (lane & 31);
			// the residual of this wave's rows, requested together and before the sums are: R may be C, every element is read here and written
			// below by the same thread
			float add[TM * PER];
			if (!GATE_UP && R) {
#pragma unroll
				for (int j = 0; j < TM * PER; ++j) {
					const int ee = kr * PER + j % PER;
					const int m	 = (ms0 + j / PER) * 32 + 8 * (ee >> 2) + 4 * half + (ee & 3);
					add[j]		 = (m < M && n < N) ? R[static_cast<int64_t>(m) * N + n] : 0.0f;
				}
			}
			__syncthreads();
			if constexpr (PASSES) { // (an earlier pass's are in LDS: nothing for the compiler to keep through the trips)
#pragma unroll
				for (int j = 0; j < TM * PER; ++j) {
					mine[j] = 0.0f;
				}
			}
#pragma unroll
			for (int q = 0; q < KS; ++q) {
				if (q == kr) {
#pragma unroll
					for (int i = 0; i < TM; ++i) {
#pragma unroll
						for (int e = 0; e < PER; ++e) {
							float part[KS], v;
#pragma unroll
							for (int src = 0; src < KS; ++src) {
								part[src] = src == q ? acc[i][q * PER + e] : slot(q, src)[(i * PER + e) * 64];
							}
							if constexpr (PASSES && KS == 2) { // one set after the other, two of them in each pass
								if (pass > 0) {
									part[0] = save[(i * PER + e) * 64] + part[0];
								}
							}
							v = part[0];
#pragma unroll
							for (int src = 1; src < KS; ++src) {
								v += part[src];
							}
							if constexpr (KS == 4) {
								if (TREE || (PASSES && tree)) {
									v = (part[0] + part[1]) + (part[2] + part[3]);
								}
							}
							if constexpr (PASSES && KS == 4) { // two workgroups' sums, or the two halves of the tree
								if (pass > 0) {
									v = save[(i * PER + e) * 64] + v;
								}
							}
							mine[i * PER + e] = v;
						}
					}
				}
			}
			if constexpr (SPLIT) {
				// K over gridDim.z workgroups: every one leaves its tile in the scratch (each wave its own rows, as it holds them),
				// counts itself in, and the last to arrive adds the tiles in z order -- whoever that is -- and stores
				__shared__ int last_flag;
				const int kz_count = static_cast<int>(gridDim.z);
				const int unit	   = static_cast<int>(by * gridDim.x + bx);
				constexpr int TILE_FLOATS = 4 * KS * TM * PER * 64; // = TM * 4096: a workgroup's tile
				float* tile = partials + (static_cast<int64_t>(unit) * kz_count) * TILE_FLOATS + wave_all * (TM * PER * 64) + lane;
				float* dst	= tile + static_cast<int64_t>(blockIdx.z) * TILE_FLOATS;
#pragma unroll
				for (int j = 0; j < TM * PER; ++j) {
					__hip_atomic_store(&dst[j * 64], mine[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
				}
				wait_stores_acknowledged();
				__syncthreads();
				if (tid == 0) {
					const unsigned prev = __hip_atomic_fetch_add(&counters[unit], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
					const int last		= (prev == static_cast<unsigned>(kz_count - 1));
					if (last) {
						__hip_atomic_store(&counters[unit], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); // ready for the next launch
					}
					last_flag = last;
				}
				__syncthreads();
				if (!last_flag) {
					return;
				}
#pragma unroll
				for (int j = 0; j < TM * PER; ++j) {
					mine[j] = 0.0f;
				}
				constexpr int STEP = TREE ? 2 : 1; // (an even number of workgroups)
				for (int z0 = 0; z0 < kz_count; z0 += STEP) {
					float got[STEP][TM * PER];
#pragma unroll
					for (int u = 0; u < STEP; ++u) {
#pragma unroll
						for (int j = 0; j < TM * PER; ++j) {
							got[u][j] = __hip_atomic_load(&tile[static_cast<int64_t>(z0 + u) * TILE_FLOATS + j * 64], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
						}
					}
#pragma unroll
					for (int j = 0; j < TM * PER; ++j) {
						const float v = TREE ? got[0][j] + got[STEP - 1][j] : got[0][j];
						mine[j]		  = z0 == 0 ? v : mine[j] + v;
					}
				}
			}
			if constexpr (!GATE_UP) {
				if (R) {
#pragma unroll
					for (int j = 0; j < TM * PER; ++j) {
						mine[j] += add[j];
					}
				}
#pragma unroll
				for (int j = 0; j < TM * PER; ++j) {
					const int ee = kr * PER + j % PER;
					const int m	 = (ms0 + j / PER) * 32 + 8 * (ee >> 2) + 4 * half + (ee & 3);
					if (m < M && n < N) {
						C[static_cast<int64_t>(m) * N + n] = mine[j];
					}
				}
				return;
			}
			__syncthreads(); // the sets have read each other's sums: the exchange below (or the next pass's stages) goes to the same place
			if constexpr (PASSES) {
				if (pass + 1 < passes) {
#pragma unroll
					for (int j = 0; j < TM * PER; ++j) {
						save[j * 64] = mine[j];
					}
#pragma unroll
					for (int i = 0; i < TM; ++i) {
						acc[i] = v16f{ 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0 };
					}
					if (g_len & 1) {
						wa = wb;
					}
					stash_a(0, pre);
					begin_pass(pass + 1);
					last = live - 1;
					__syncthreads();
					continue;
				}
			}
		} else {
#pragma unroll
			for (int j = 0; j < TM * PER; ++j) {
				mine[j] = acc[j / PER][j % PER];
			}
		}
		break;
	}
	if constexpr (GATE_UP) {
		// Every wave is through with the stages (the last trip ended in a barrier).  The gate wave and the up wave of a strip (and K set)
		// share the work behind the loop: the first half of their PER registers of every tile is finished by the gate wave, the second by
		// the up wave, each handing the other the half it does not finish (the exp and the divides of SiLU and of the quantizer are a
		// quarter of the loop's VALU work; on the gate waves alone they cost the launch 6 %).
		const int pair	 = wave & 1;
		const bool is_up = wave >= 2;
		float* xch		 = reinterpret_cast<float*>(lds_raw); // [pair][TM][16][64]: slot (i, e) holds the value of the wave that does not finish it
#pragma unroll
		for (int i = 0; i < TM; ++i) {
#pragma unroll
			for (int x = 0; x < PER / 2; ++x) {
				const int give															   = kr * PER + (is_up ? x : x + PER / 2);
				xch[((pair * TM + i) * 16 + give) * 64 + lane] = is_up ? mine[i * PER + x] : mine[i * PER + x + PER / 2];
			}
		}
		float* dbg = is_up ? C2 : C; // inspection copies of the fp32 tiles
		if (dbg) {
			const int n = ns * 32 + (lane & 31);
#pragma unroll
			for (int j = 0; j < TM * PER; ++j) {
				const int e = kr * PER + j % PER;
				const int m = (ms0 + j / PER) * 32 + 8 * (e >> 2) + 4 * half + (e & 3);
				if (m < M && n < N) {
					dbg[static_cast<int64_t>(m) * N + n] = mine[j];
				}
			}
		}
		__syncthreads();
		uint8_t* image = lds_raw + XCH_BYTES + pair * TM * (TILE_BYTES + 64); // the pair's TM tile images, each followed by its 32 scales
		const int j	   = lane & 31; // the lane's weight row = quant j of the block
#pragma unroll
		for (int i = 0; i < TM; ++i) {
			uint8_t* tile	 = image + i * (TILE_BYTES + 64);
			uint16_t* scales = reinterpret_cast<uint16_t*>(tile + TILE_BYTES);
#pragma unroll
			for (int x = 0; x < PER / 2; ++x) {
				const int e		  = kr * PER + (is_up ? x + PER / 2 : x);
				const float own	  = is_up ? mine[i * PER + x + PER / 2] : mine[i * PER + x];
				const float other = xch[((pair * TM + i) * 16 + e) * 64 + lane];
				const float v	  = is_up ? silu_mul(other, own) : silu_mul(own, other);
				// the block = this register over the 32 lanes of the half-wave: quantize_row_q8_0 on it
				float amax = fabsf(v);
#pragma unroll
				for (int off = 16; off >= 1; off >>= 1) {
					amax = fmaxf(amax, __shfl_xor(amax, off));
				}
				const float d  = __fdiv_rn(amax, 127.0f);
				const float id = (amax != 0.0f) ? __fdiv_rn(127.0f, amax) : 0.0f;
				const int r	   = 8 * (e >> 2) + 4 * half + (e & 3); // row within the activation strip
				tile[16 * (r + 32 * (j >> 4)) + (j & 15)] = static_cast<uint8_t>(quantize_value(v, id));
				if (j == 0) {
					scales[r] = float_to_half_bits(d);
				}
			}
		}
		__syncthreads(); // the waves of a pair have filled its images
		// tile i of the pair goes out through the first K set's gate wave (even i) or up wave (odd i): one 16-byte store per lane
		const int out_groups = N / GROUP_K; // the activation is [M x N]: N / 128 groups per strip, this strip's block is ns
		if (ns < n_strips && kr == 0) {
#pragma unroll
			for (int i = 0; i < TM; ++i) {
				if ((i & 1) == (is_up ? 1 : 0) && ms0 + i < m_strips) {
					const uint8_t* tile = image + i * (TILE_BYTES + 64);
					uint8_t* macro		= act_out + macro_offset(ms0 + i, ns / GROUP_BLOCKS, out_groups);
					*reinterpret_cast<v4i*>(macro + (ns % GROUP_BLOCKS) * TILE_BYTES + 16 * lane) = *reinterpret_cast<const v4i*>(tile + 16 * lane);
					if (lane < STRIP_ROWS) {
						*reinterpret_cast<uint16_t*>(macro + MACRO_D_OFFSET + 8 * lane + 2 * (ns % GROUP_BLOCKS)) = reinterpret_cast<const uint16_t*>(tile + TILE_BYTES)[lane];
					}
				}
			}
		}
		return;
	}
	if constexpr (!DUMP) {
#pragma unroll
		for (int i = 0; i < TM; ++i) {
			store_tile(acc[i], (ms0 + i) * 32, ns * 32, half, lane & 31, C, R, M, N);
		}
	}
}

template<int TM, bool DUMP, int KS = 1, bool STREAM = false, bool SPLIT = false>
__global__ __launch_bounds__(256 * KS, 4) void gemm_tiled_kernel(const uint8_t* __restrict__ W, const uint8_t* __restrict__ A, int M, int N, int groups, int order, float* C, const float* R,
	int32_t* __restrict__ sums, float* __restrict__ partials, unsigned* __restrict__ counters) {
	gemm_tiled_body<TM, DUMP, KS, STREAM, SPLIT, false>(W, A, C, R, sums, M, N, groups, partials, counters, nullptr, nullptr, nullptr, order);
}

// the fused gate / up form (GATE_UP above): N = rows of each of the two matrices; gate_out / up_out optional
template<int TM, int KS, bool STREAM, bool PASSES>
__global__ __launch_bounds__(256 * KS, 4) void gemm_gate_up_kernel(const uint8_t* __restrict__ W_gate, const uint8_t* __restrict__ W_up, const uint8_t* __restrict__ A, int M, int N, int groups,
	int order, int passes, bool tree, uint8_t* __restrict__ act_out, float* __restrict__ gate_out, float* __restrict__ up_out) {
	gemm_tiled_body<TM, false, KS, STREAM, false, true, PASSES>(W_gate, A, gate_out, nullptr, nullptr, M, N, groups, nullptr, nullptr, W_up, act_out, up_out, order, passes, tree);
}

// Executes a cut made by plan_gemm_tile (q8_0_plan.h): TM activation strips per wave, KS sets of four waves per workgroup,
// and K over kz workgroups per tile whose tiles are added through the scratch.
template<int TM, bool STREAM> static hipError_t launch_gemm_tiled_t(const gemm_tile_cut& cut, const uint8_t* w, const uint8_t* a, float* C, const float* R, int32_t* sums, int m, int n, int k, hipStream_t s) {
	const int groups = k / GROUP_K;
	const dim3 grid(cut.grid_x, cut.grid_y);
	if (sums) {
		gemm_tiled_kernel<TM, true><<<grid, dim3(256), 0, s>>>(w, a, m, n, groups, cut.order, C, R, sums, nullptr, nullptr);
		return hipGetLastError();
	}
	const int ks = cut.ks;
	if constexpr (STREAM || TM == 2) {
		if (cut.kz > 1) {
			float* partials	   = nullptr;
			unsigned* counters = nullptr;
			scratch_hold hold;
			const hipError_t e = acquire_gemm_split_scratch(&partials, &counters, STREAM, &hold, s);
			if (e != hipSuccess) {
				return e;
			}
			return launch_kernel(KIND_GEMM, gemm_tiled_kernel<TM, false, 4, STREAM, true>, dim3(grid.x, grid.y, static_cast<unsigned>(cut.kz)), dim3(1024), 0, s, w, a, m, n, groups, cut.order, C, R, sums, partials,
				counters);
		}
	}
	if (ks == 4) {
		return launch_kernel(KIND_GEMM, gemm_tiled_kernel<TM, false, 4, STREAM>, grid, dim3(1024), 0, s, w, a, m, n, groups, cut.order, C, R, sums, static_cast<float*>(nullptr), static_cast<unsigned*>(nullptr));
	}
	if (ks == 2) {
		return launch_kernel(KIND_GEMM, gemm_tiled_kernel<TM, false, 2, STREAM>, grid, dim3(512), 0, s, w, a, m, n, groups, cut.order, C, R, sums, static_cast<float*>(nullptr), static_cast<unsigned*>(nullptr));
	}
	return launch_kernel(KIND_GEMM, gemm_tiled_kernel<TM, false, 1, STREAM>, grid, dim3(256), 0, s, w, a, m, n, groups, cut.order, C, R, sums, static_cast<float*>(nullptr), static_cast<unsigned*>(nullptr));
}

// stream: the weights are read once and not again (a batch of decode rows against a large matrix), so their loads bypass the caches.
static hipError_t launch_gemm_tiled(const gemm_tile_cut& cut, const uint8_t* w, const uint8_t* a, float* C, const float* R, int32_t* sums, int m, int n, int k, hipStream_t s, bool stream) {
	if (stream) {
		return cut.tm == 2 ? launch_gemm_tiled_t<2, true>(cut, w, a, C, R, sums, m, n, k, s) : launch_gemm_tiled_t<1, true>(cut, w, a, C, R, sums, m, n, k, s);
	}
	return cut.tm == 2 ? launch_gemm_tiled_t<2, false>(cut, w, a, C, R, sums, m, n, k, s) : launch_gemm_tiled_t<1, false>(cut, w, a, C, R, sums, m, n, k, s);
}

// act_out (tiled, [M x n_ff]) = quantize_row_q8_0(silu(W_gate . Aq) * (W_up . Aq)); gate_dbg / up_dbg: optional fp32 copies of the two
// mat-mats' outputs.  workspace: 2 * M * n_ff floats for shapes the fused form does not take (plan_gate_up_fused), else unused.
hipError_t launch_gemm_gate_up_silu(const void* w_gate, const void* w_up, const void* aq, void* act_out, float* gate_dbg, float* up_dbg, float* workspace, int64_t M, int64_t n_ff, int64_t K,
	hipStream_t s) {
	if (M == 0 || n_ff == 0) {
		return hipSuccess;
	}
	if (gate_up_rows_suits(M, n_ff, K)) {
		return launch_gemm_rows_gate_up(w_gate, w_up, aq, act_out, gate_dbg, up_dbg, M, n_ff, K, gate_up_rows_waves(M, n_ff, K), s);
	}
	gate_up_cut cut{};
	if (plan_gate_up_fused(M, n_ff, K, &cut)) {
		const gemm_tile_cut& t = cut.tile;
		const dim3 grid(t.grid_x, t.grid_y);
		auto launch = [&](auto kernel) {
			return launch_kernel(KIND_GEMM, kernel, grid, dim3(static_cast<unsigned>(256 * t.ks)), 0, s, static_cast<const uint8_t*>(w_gate), static_cast<const uint8_t*>(w_up), static_cast<const uint8_t*>(aq),
				static_cast<int>(M), static_cast<int>(n_ff), static_cast<int>(K / GROUP_K), t.order, cut.passes, cut.tree, static_cast<uint8_t*>(act_out), gate_dbg, up_dbg);
		};
		if (t.tm == 1 && t.grid_y > 1) {
			return t.ks == 1 ? launch(gemm_gate_up_kernel<1, 1, false, false>) : cut.passes > 1 ? launch(gemm_gate_up_kernel<1, 2, false, true>) : launch(gemm_gate_up_kernel<1, 2, false, false>);
		}
		if (t.tm == 1) { // 17 to 32 rows on matrices of 192 column blocks and more (the rows kernel has the others)
			return t.ks == 1 ? launch(gemm_gate_up_kernel<1, 1, true, false>) : cut.passes > 1 ? launch(gemm_gate_up_kernel<1, 2, true, true>) : launch(gemm_gate_up_kernel<1, 2, true, false>);
		}
		auto launch_t = [&](auto stream) { // up to 64 rows the weights are read once
			constexpr bool STREAM = decltype(stream)::value;
			if (t.ks == 1) {
				return launch(gemm_gate_up_kernel<2, 1, STREAM, false>);
			}
			if (t.ks == 2) {
				return cut.passes > 1 ? launch(gemm_gate_up_kernel<2, 2, STREAM, true>) : launch(gemm_gate_up_kernel<2, 2, STREAM, false>);
			}
			return cut.passes > 1 ? launch(gemm_gate_up_kernel<2, 4, STREAM, true>) : launch(gemm_gate_up_kernel<2, 4, STREAM, false>);
		};
		return t.grid_y == 1 ? launch_t(std::true_type{}) : launch_t(std::false_type{});
	}
	float* gate = gate_dbg ? gate_dbg : workspace;
	float* up	= up_dbg ? up_dbg : workspace + M * n_ff;
	hipError_t e = launch_gemm(w_gate, aq, gate, nullptr, M, n_ff, K, true, s);
	if (e != hipSuccess) {
		return e;
	}
	e = launch_gemm(w_up, aq, up, nullptr, M, n_ff, K, true, s);
	if (e != hipSuccess) {
		return e;
	}
	return launch_silu_mul_quantize(gate, up, act_out, M, n_ff, true, s);
}

__global__ void zero_c_kernel(float* c, const float* src, int64_t n) {
	const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
	if (i < n) {
		c[i] = src ? src[i] : 0.0f;
	}
}

hipError_t launch_gemm(const void* W, const void* Aq, float* C, int32_t* sums, int64_t M, int64_t N, int64_t K, bool tiled, hipStream_t s, const float* residual) {
	if (M == 0 || N == 0) {
		return hipSuccess;
	}
	if (K == 0) { // empty dot products: C = residual, or 0
		if (!sums) {
			zero_c_kernel<<<dim3(static_cast<unsigned>((M * N + 255) / 256)), dim3(256), 0, s>>>(C, residual, M * N);
		}
		return hipGetLastError();
	}
	const dim3 grid(static_cast<unsigned>((N + GEMM_BN - 1) / GEMM_BN), static_cast<unsigned>((M + GEMM_BM - 1) / GEMM_BM));
	const uint8_t* w = static_cast<const uint8_t*>(W);
	const uint8_t* a = static_cast<const uint8_t*>(Aq);
	const int m = static_cast<int>(M), n = static_cast<int>(N), k = static_cast<int>(K);
	if (tiled) {
		if (sums) { // the inspection variant runs on the plain tile kernel, whatever the shape
			return launch_gemm_tiled(plan_gemm_tile(M, N, K, false), w, a, C, residual, sums, m, n, k, s, false);
		}
		const gemm_plan plan = plan_gemm(M, N, K); // which kernel and how it cuts the work: q8_0_plan.h
		if (plan.kernel == MM_GEMM_SKINNY) {
			// (a launch that hands K parts' sums over by epoch cannot be replayed from a graph, and is refused while another stream's is
			// under way: the streaming kernel, whose cut and order of additions are the same, takes those calls)
			if (plan.rows && (plan.skinny.splits == 1 || !stream_is_capturing(s))) {
				const hipError_t e = launch_gemm_rows(W, Aq, C, residual, M, N, K, plan.skinny, s);
				if (e != hipErrorNotReady) {
					return e;
				}
			}
			return launch_gemm_skinny(W, Aq, C, M, N, K, plan.skinny, s, residual);
		}
		// K over workgroups with more than 64 rows: where the scratch is another stream's for now, or the launch goes into a graph that may be
		// replayed beside another (the scratch would be both's), the streaming kernel, which gives the same bits without any
		const bool split_rows = plan.kernel == MM_GEMM_TILE && plan.tile.kz > 1;
		if (!split_rows || !stream_is_capturing(s)) {
			const hipError_t e = launch_gemm_tiled(plan.tile, w, a, C, residual, sums, m, n, k, s, plan.kernel == MM_GEMM_TILE_STREAM);
			if (!split_rows || e != hipErrorNotReady) {
				return e;
			}
		}
		return launch_gemm_skinny(W, Aq, C, M, N, K, plan.skinny, s, residual);
	} else {
		if (sums) {
			gemm_kernel<false, true><<<grid, dim3(GEMM_THREADS), 0, s>>>(w, a, C, sums, m, n, k);
		} else {
			return launch_kernel(KIND_GEMM, gemm_kernel<false, false>, grid, dim3(GEMM_THREADS), 0, s, w, a, C, sums, m, n, k);
		}
	}
	return hipGetLastError();
}

} // namespace nh
