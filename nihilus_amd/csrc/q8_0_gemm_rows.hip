// Batched decode with 2 ... 32 already quantized activation rows: C[m][n] = dot(W row n, Aq row m), and the FFN's gate / up pair with
// SiLU * up and the quantizer behind it in the same launch, gfx950.
//
// What bounds it is HBM and, at these sizes, latency: the weights are read once, so the kernel is the streaming mat-vec again -- a
// workgroup per (32-row weight strip, K part), its waves splitting the K range, a chunk of two groups (one of each matrix in the gate /
// up form) at a time with every load of it in flight before anything is waited for, one reduction at the end -- with the int8 MFMA as the
// inner product.  The weight tile as loaded is the B operand; the activation rows are the A operand.  Eight waves per workgroup and at
// most 128 registers: two workgroups per CU, so that one streams while the other reduces and leaves.
//
// K is cut, and the sums are added, as in the streaming kernel (q8_0_gemm_skinny.hip), which runs a call that is being captured or finds
// the hand-off's scratch in use on another stream: the result does not depend on which of the two ran.
//
// The activations come memory -> LDS without registers, and only the rows that exist: a 128-quant group of R rows (R = 8, 16, 24 or 32) is
// R / 8 transfers of 1 KiB (lane l fetches the 16 bytes of one (block, k half, row)), so that eight rows cost a quarter of the weight
// tile's requests; operand rows past R repeat them and their sums are never looked at.
#include "q8_0_plan.h"

#include <mutex>

namespace nh {

namespace {

// memory -> LDS, 16 bytes per lane: base (wave-uniform) + lane_off to LDS byte address lds_addr + 16 * lane
__device__ __forceinline__ void dma_b128(const uint8_t* base, uint32_t lane_off, uint32_t lds_addr) {
	uint32_t saved_m0;
	asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0" : "=&s"(saved_m0) : "v"(lane_off), "s"(base), "s"(lds_addr) : "memory");
}

typedef _Float16 rq_v4h __attribute__((ext_vector_type(4)));
typedef float rq_v16f __attribute__((ext_vector_type(16)));

// With 8 or 16 rows a lane multiplies the two scales of its 4 or 8 sums itself; with 24 or 32 (12 or 16 sums per lane) the products come from
// an f16 MFMA (measured at 32 rows, [14336 x 4096] 14.9 -> 14.4 us, [8192 x 8192] 15.6 -> 14.9; at 24 rows 14.9 -> 14.1 and 16.2 -> 15.8; at
// 16 rows 12.2 -> 12.8).
template<int R> constexpr bool rows_scale_mfma = R >= 24;
template<int R> constexpr int rows_group_bytes = R / 8 * 1024; // a group's operand rows in LDS: [block][k half][row][16 bytes]
template<int R> __device__ __forceinline__ int rows_operand_row(int r) { // of operand row r (0..31) in LDS: past R one that exists
	return R == 24 ? min(r, R - 1) : r & (R - 1);
}

// Groups [gc, gc + CNT) of a wave's K range, against MATS weight strips that share the activations.  CNT is a template parameter so
// that every wait is a count of younger loads.
template<int R, int T, int MATS, int CNT>
__device__ __forceinline__ void rows_chunk_n(const uint8_t* __restrict__ w_strip, const uint8_t* __restrict__ w_strip2, const uint8_t* __restrict__ a_strip, uint8_t* a_tiles, uint8_t* a_scales, int gc,
	int lane, float (&acc)[MATS][R / 2]) {
	static_assert(R * T <= 64, "one scale load per lane covers the chunk");
	const int r	   = lane & 31;
	const int half = lane >> 5;
	// ---- 1. the activation rows, requested first: memory -> LDS, then the scales of (group lane / R, row lane % R) through a
	// register; loads return in issue order, so whoever has the scales has the rows too ----
	const uint32_t lds_addr = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint8_t*)a_tiles));
#pragma unroll
	for (int c = 0; c < CNT; ++c) {
		const uint8_t* macro = a_strip + static_cast<int64_t>(gc + c) * MACRO_BYTES;
#pragma unroll
		for (int d = 0; d < R / 8; ++d) {
			// lane l of transfer d: byte 1024 d + 16 l of the group's LDS image = block u / (2 R), half u / R % 2, row u % R of unit u = 64 d + l
			// (64 units are whole blocks but for R = 24)
			constexpr bool WHOLE = 64 % (2 * R) == 0;
			const int unit = WHOLE ? lane : 64 * d + lane;
			const int off  = unit / (2 * R) * TILE_BYTES + (unit / R) % 2 * (TILE_BYTES / 2) + unit % R * 16;
			dma_b128(macro + (WHOLE ? d * (64 / (2 * R)) * TILE_BYTES : 0), off, lds_addr + c * rows_group_bytes<R> + d * 1024);
		}
	}
	const int sg = min(lane / R, CNT - 1), sr = lane % R;
	uint32_t sc_off = sg * MACRO_BYTES + MACRO_D_OFFSET + 8 * sr;
	asm volatile("" : "+v"(sc_off)::"memory"); // the load below takes its address from behind the transfers: it cannot be issued ahead of them
	const v2u sc = *reinterpret_cast<const v2u*>(a_strip + static_cast<int64_t>(gc) * MACRO_BYTES + sc_off);
	asm volatile("" ::: "memory");
	// ---- 2. every weight byte of the chunk ----
	v4i q[MATS][T][GROUP_BLOCKS];
	v2u dd[MATS][T];
#pragma unroll
	for (int c = 0; c < CNT; ++c) {
#pragma unroll
		for (int k = 0; k < MATS; ++k) {
			const uint8_t* macro = (k == 0 ? w_strip : w_strip2) + static_cast<int64_t>(gc + c) * MACRO_BYTES;
#pragma unroll
			for (int j = 0; j < GROUP_BLOCKS; ++j) {
				q[k][c][j] = __builtin_nontemporal_load(reinterpret_cast<const v4i*>(macro + j * TILE_BYTES + 16 * lane));
			}
			dd[k][c] = __builtin_nontemporal_load(reinterpret_cast<const v2u*>(macro + MACRO_D_OFFSET + 8 * r));
		}
	}
	__builtin_amdgcn_sched_barrier(0);
	// ---- 3. the scales, [block][row]: as fp32, or (24 and 32 rows) as the fp16 bits that the scale MFMA takes ----
	if (lane / R < CNT) {
		if constexpr (rows_scale_mfma<R>) {
			uint32_t* out = reinterpret_cast<uint32_t*>(a_scales) + (lane / R) * GROUP_BLOCKS * R + sr;
			out[0]		  = sc.x & 0xFFFFu;
			out[R]		  = sc.x >> 16;
			out[2 * R]	  = sc.y & 0xFFFFu;
			out[3 * R]	  = sc.y >> 16;
		} else {
			float* out = reinterpret_cast<float*>(a_scales) + (lane / R) * GROUP_BLOCKS * R + sr;
			out[0]	   = half_bits_to_float(static_cast<uint16_t>(sc.x & 0xFFFFu));
			out[R]	   = half_bits_to_float(static_cast<uint16_t>(sc.x >> 16));
			out[2 * R] = half_bits_to_float(static_cast<uint16_t>(sc.y & 0xFFFFu));
			out[3 * R] = half_bits_to_float(static_cast<uint16_t>(sc.y >> 16));
		}
	}
	asm volatile("" ::"v"(sc) : "memory"); // the rows have landed (issue order): no LDS read of them above this point
	__builtin_amdgcn_wave_barrier();
	// ---- 4. one MFMA per block and matrix; lane (r, half) gets column r's sums for rows 8 i + 4 half + (0..3) in s[4 i .. 4 i + 3] ----
#pragma unroll
	for (int c = 0; c < CNT; ++c) {
#pragma unroll
		for (int j = 0; j < GROUP_BLOCKS; ++j) {
			const v4i a = *reinterpret_cast<const v4i*>(a_tiles + c * rows_group_bytes<R> + j * (32 * R) + half * (16 * R) + rows_operand_row<R>(r) * 16);
			if constexpr (rows_scale_mfma<R>) {
				// the products d_x * d_w on the matrix pipe, block j's scales in the k = 0 slot.  Both operands are zero in every other slot
				// (k = 4..7: lanes 32..63): a zero on one side only would make a NaN of the other side's infinity.
				const uint32_t d = reinterpret_cast<const uint32_t*>(a_scales)[(c * GROUP_BLOCKS + j) * R + rows_operand_row<R>(r)];
				const v2u dx	 = v2u{ half ? 0u : d, 0u };
#pragma unroll
				for (int k = 0; k < MATS; ++k) {
					const v16i zi	 = { 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0 };
					const rq_v16f zf = { 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0 };
					const v2u dw	 = scale_slot(half ? v2u{ 0u, 0u } : dd[k][c], j);
					const v16i s	 = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, q[k][c][j], zi, 0, 0, 0);
					const rq_v16f p	 = __builtin_amdgcn_mfma_f32_32x32x8f16(__builtin_bit_cast(rq_v4h, dx), __builtin_bit_cast(rq_v4h, dw), zf, 0, 0, 0);
#pragma unroll
					for (int e = 0; e < R / 2; ++e) {
						acc[k][e] = fmaf(static_cast<float>(s[e]), p[e], acc[k][e]);
					}
				}
				__builtin_amdgcn_sched_barrier(0); // left alone the compiler forms every block's operands at once and spills
				continue;
			}
#pragma unroll
			for (int k = 0; k < MATS; ++k) {
				const uint32_t dp = (j & 2) ? dd[k][c].y : dd[k][c].x;
				const float dw	  = half_bits_to_float(static_cast<uint16_t>((j & 1) ? (dp >> 16) : (dp & 0xFFFFu)));
				const v16i zi	  = { 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0 };
				const v16i s	  = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, q[k][c][j], zi, 0, 0, 0);
#pragma unroll
				for (int e4 = 0; e4 < R / 8; ++e4) {
					const float4 dx	   = *reinterpret_cast<const float4*>(reinterpret_cast<const float*>(a_scales) + (c * GROUP_BLOCKS + j) * R + 8 * e4 + 4 * half);
					acc[k][4 * e4 + 0] = fmaf(static_cast<float>(s[4 * e4 + 0]), dw * dx.x, acc[k][4 * e4 + 0]);
					acc[k][4 * e4 + 1] = fmaf(static_cast<float>(s[4 * e4 + 1]), dw * dx.y, acc[k][4 * e4 + 1]);
					acc[k][4 * e4 + 2] = fmaf(static_cast<float>(s[4 * e4 + 2]), dw * dx.z, acc[k][4 * e4 + 2]);
					acc[k][4 * e4 + 3] = fmaf(static_cast<float>(s[4 * e4 + 3]), dw * dx.w, acc[k][4 * e4 + 3]);
				}
			}
		}
	}
}

template<int R, int T, int MATS>
__device__ __forceinline__ void rows_chunk(const uint8_t* __restrict__ w_strip, const uint8_t* __restrict__ w_strip2, const uint8_t* __restrict__ a_strip, uint8_t* a_tiles, uint8_t* a_scales, int gc,
	int cnt, int lane, float (&acc)[MATS][R / 2]) {
	static_assert(T == 1 || T == 2);
	switch (cnt) { // wave-uniform (an if with an else instead: 4.16 -> 4.23 us at [8123 x 1280], 5.29 -> 5.50 at 24 rows)
		case 1:
			rows_chunk_n<R, T, MATS, 1>(w_strip, w_strip2, a_strip, a_tiles, a_scales, gc, lane, acc);
			break;
		case 2:
			if constexpr (T == 2) {
				rows_chunk_n<R, T, MATS, 2>(w_strip, w_strip2, a_strip, a_tiles, a_scales, gc, lane, acc);
			}
			break;
		default:
			break;
	}
}

// The workgroup's LDS: the waves' activation tiles and scales, then (behind a barrier) the last set's partial sums in the same place; the
// first of two sets' behind them.
template<int R, int T, int MATS, int SETS> struct rows_lds {
	static constexpr int TILES	= T * rows_group_bytes<R>; // per wave
	static constexpr int SCALES = T * GROUP_BLOCKS * R * 4; // per wave
	static constexpr int STAGE	= SK_WAVES * (TILES + SCALES);
	static constexpr int RED	= MATS * (R / 2) * SK_WAVES * 64 * 4;
	static constexpr int FIRST	= STAGE > RED ? STAGE : RED;
	static constexpr int BYTES	= FIRST + (SETS - 1) * RED;
	static_assert(SK_WAVES * TILES <= 65536, "the memory -> LDS transfers address the tiles with 16 bits");
	static_assert(SETS == 1 || SETS == 2);
};

// A workgroup's K part of a strip, all waves' partial sums left in LDS: [matrix][value][wave][lane].  With two sets the eight waves walk
// the ranges that sixteen would have, one after the other: as many additions in a row as sixteen waves make, with no more than eight
// waves' registers, LDS or launch.
template<int R, int T, int MATS, int SETS>
__device__ __forceinline__ void rows_strip(const uint8_t* __restrict__ w_strip, const uint8_t* __restrict__ w_strip2, const uint8_t* __restrict__ A, uint8_t* lds, int groups, int split_shift, int split,
	int lane, int wave) {
	using L = rows_lds<R, T, MATS, SETS>;
	uint8_t* a_tiles = lds + wave * L::TILES;
	uint8_t* a_scales = lds + SK_WAVES * L::TILES + wave * L::SCALES;
	for (int set = 0; set < SETS; ++set) {
		int g0, g1;
		wave_k_range(groups, split_shift + (SETS - 1), split * SETS + set, SK_WAVES, wave, g0, g1);
		float acc[MATS][R / 2];
#pragma unroll
		for (int k = 0; k < MATS; ++k) {
#pragma unroll
			for (int e = 0; e < R / 2; ++e) {
				acc[k][e] = 0.0f;
			}
		}
		for (int gc = g0; gc < g1; gc += T) {
			rows_chunk<R, T, MATS>(w_strip, w_strip2, A, a_tiles, a_scales, gc, min(T, g1 - gc), lane, acc);
			__builtin_amdgcn_wave_barrier(); // the next chunk overwrites this wave's tiles
		}
		const bool last = set == SETS - 1;
		if (last) {
			__syncthreads(); // everybody is through with the tiles
		}
		float* red = reinterpret_cast<float*>(lds + (last ? 0 : L::FIRST));
#pragma unroll
		for (int k = 0; k < MATS; ++k) {
#pragma unroll
			for (int e = 0; e < R / 2; ++e) {
				red[((k * (R / 2) + e) * SK_WAVES + wave) * 64 + lane] = acc[k][e];
			}
		}
	}
	__syncthreads();
}
// output (row m, strip column l) of matrix k: the waves' partial sums in the streaming kernel's order (q8_0_gemm_skinny.hip), of which this
// is the form for few rows: the same cut, the same chains of additions, the same tree over them, so the same bits.  (One wave after the
// other, and longer chains, were also up to 35 % further from the sums in 64 bits.)
template<int R, int T, int MATS, int SETS> __device__ __forceinline__ float rows_total(const uint8_t* lds, int k, int m, int l) {
	const int e = 4 * (m >> 3) + (m & 3), at = 32 * ((m >> 2) & 1) + l;
	const auto eight = [&](const uint8_t* red) {
		const float* p = reinterpret_cast<const float*>(red) + (k * (R / 2) + e) * (SK_WAVES * 64) + at;
		return ((p[64 * 0] + p[64 * 4]) + (p[64 * 2] + p[64 * 6])) + ((p[64 * 1] + p[64 * 5]) + (p[64 * 3] + p[64 * 7]));
	};
	return SETS == 1 ? eight(lds) : eight(lds + rows_lds<R, T, MATS, SETS>::FIRST) + eight(lds);
}

} // namespace

template<int R, int T, int SETS>
__global__ __launch_bounds__(SK_WAVES * 64, 4) void gemm_rows_kernel(const uint8_t* __restrict__ W, const uint8_t* __restrict__ A, int groups, int split_shift, int M, int N, const float* residual, float* C,
	uint64_t* __restrict__ tagged, unsigned epoch) {
	__shared__ __align__(16) uint8_t lds[rows_lds<R, T, 1, SETS>::BYTES];
	const int tid	= threadIdx.x;
	const int lane	= tid & 63;
	const int wave	= __builtin_amdgcn_readfirstlane(tid >> 6);
	const int strip = static_cast<int>(blockIdx.x >> split_shift);
	const int split = static_cast<int>(blockIdx.x) & ((1 << split_shift) - 1);
	// thread t finishes outputs (row t / 32 + 16 i, strip column t % 32); their residuals (which may be those outputs) are requested here, a memory
	// latency ahead of their use (100 random shapes, half of them with one: as fast as with the read behind the reduction, 0.98 to 1.04)
	constexpr int OWN = (R + 15) / 16;
	const int m0 = tid >> 5, l = tid & 31, n = strip * STRIP_ROWS + l;
	const int rows = min(M, R);
	float res[OWN];
#pragma unroll
	for (int i = 0; i < OWN; ++i) {
		res[i] = 0.0f;
		if (residual && m0 + 16 * i < rows && n < N) {
			res[i] = residual[static_cast<int64_t>(m0 + 16 * i) * N + n];
		}
	}
	rows_strip<R, T, 1, SETS>(W + macro_offset(strip, 0, groups), nullptr, A, lds, groups, split_shift, split, lane, wave);
	float total[OWN];
#pragma unroll
	for (int i = 0; i < OWN; ++i) {
		if (m0 + 16 * i < rows) {
			total[i] = rows_total<R, T, 1, SETS>(lds, 0, m0 + 16 * i, l);
		}
	}
	if (split_shift == 0) {
#pragma unroll
		for (int i = 0; i < OWN; ++i) {
			if (m0 + 16 * i < rows && n < N) {
				C[static_cast<int64_t>(m0 + 16 * i) * N + n] = residual ? total[i] + res[i] : total[i];
			}
		}
		return;
	}
#pragma unroll
	for (int i = 0; i < OWN; ++i) {
		if (m0 + 16 * i < rows) {
			split_k_publish(tagged, epoch, strip * R + m0 + 16 * i, 1 << split_shift, split, l, total[i], res[i]);
		}
	}
	wait_stores_acknowledged();
#pragma unroll
	for (int i = 0; i < OWN; ++i) {
		if (m0 + 16 * i < rows) {
			split_k_collect(tagged, epoch, strip * R + m0 + 16 * i, 1 << split_shift, l, C + static_cast<int64_t>(m0 + 16 * i) * N, n, N, residual != nullptr, res[i]);
		}
	}
}

// The gate and up strips of the same 32 rows against one activation, then silu(g) * u and quantize_row_q8_0: the 32 values of an
// activation row are one block of the down projection's operand and sit in one half-wave.
template<int R, int T, int SETS>
__global__ __launch_bounds__(SK_WAVES * 64, 4) void gemm_rows_gate_up_kernel(const uint8_t* __restrict__ W_gate, const uint8_t* __restrict__ W_up, const uint8_t* __restrict__ A,
	int groups, int M, int N, uint8_t* __restrict__ act_out, float* __restrict__ gate_out, float* __restrict__ up_out) {
	__shared__ __align__(16) uint8_t lds[rows_lds<R, T, 2, SETS>::BYTES];
	const int tid	= threadIdx.x;
	const int lane	= tid & 63;
	const int wave	= __builtin_amdgcn_readfirstlane(tid >> 6);
	const int strip = static_cast<int>(blockIdx.x);
	rows_strip<R, T, 2, SETS>(W_gate + macro_offset(strip, 0, groups), W_up + macro_offset(strip, 0, groups), A, lds, groups, 0, 0, lane, wave);
	uint8_t* macro = act_out + macro_offset(0, strip / GROUP_BLOCKS, N / GROUP_K);
	const int t	   = strip % GROUP_BLOCKS;
#pragma unroll
	for (int o = 0; o < STRIP_ROWS * STRIP_ROWS; o += SK_WAVES * 64) {
		const int m = (o + tid) >> 5, l = tid & 31;
		float v = 0.0f; // rows past M are the operand's padding: zero blocks
		if (m < M && m < R) {
			const float g = rows_total<R, T, 2, SETS>(lds, 0, m, l), u = rows_total<R, T, 2, SETS>(lds, 1, m, l);
			v = silu_mul(g, u);
			if (gate_out) {
				gate_out[static_cast<int64_t>(m) * N + strip * STRIP_ROWS + l] = g;
				up_out[static_cast<int64_t>(m) * N + strip * STRIP_ROWS + l]   = u;
			}
		}
		float amax = fabsf(v);
#pragma unroll
		for (int off = 16; off >= 1; off >>= 1) {
			amax = fmaxf(amax, __shfl_xor(amax, off));
		}
		const float d  = __fdiv_rn(amax, 127.0f);
		const float id = (amax != 0.0f) ? __fdiv_rn(127.0f, amax) : 0.0f;
		macro[t * TILE_BYTES + 16 * (m + 32 * (l >> 4)) + (l & 15)] = static_cast<uint8_t>(quantize_value(v, id));
		if (l == 0) {
			*reinterpret_cast<uint16_t*>(macro + MACRO_D_OFFSET + 8 * m + 2 * t) = float_to_half_bits(d);
		}
	}
}

// The tagged partial sums of a K split: this kernel's own (shared with the mat-vecs' scratch, a mat-mat on one stream and a mat-vec on
// another refused each other), one allocation per device on first use, in two parts: the null stream's, which may not be queried while
// some other stream is being captured and so never shares, and one that serves the other streams one at a time.
namespace {
	struct rows_scratch {
		uint64_t* tagged = nullptr; // [GEMV_MAX_SPLIT_UNITS][32] {epoch, partial sum}
		unsigned epoch	 = 0;
		hipStream_t user = nullptr; // stream of the last launch that used this part
	};
	constexpr size_t ROWS_SCRATCH_WORDS = static_cast<size_t>(GEMV_MAX_SPLIT_UNITS) * STRIP_ROWS;
	// hold == nullptr: make it if need be; otherwise a launch on `s` is about to use it, and the caller keeps *hold until it is enqueued
	hipError_t get_rows_scratch(rows_scratch* out, scratch_hold* hold, hipStream_t s) {
		static std::recursive_mutex locks[64];
		static rows_scratch per_device[64][2];
		int dev		 = 0;
		hipError_t e = hipGetDevice(&dev);
		if (e != hipSuccess) {
			return e;
		}
		if (dev < 0 || dev >= 64) {
			return hipErrorInvalidDevice;
		}
		scratch_hold g(locks[dev]);
		if (!per_device[dev][0].tagged) {
			void* p = nullptr;
			e		= hipMalloc(&p, 2 * ROWS_SCRATCH_WORDS * 8);
			if (e != hipSuccess) {
				return e;
			}
			e = hipMemset(p, 0, 2 * ROWS_SCRATCH_WORDS * 8); // synchronous, once: every tag starts at epoch 0, which no launch uses
			if (e != hipSuccess) {
				(void)hipFree(p);
				return e;
			}
			per_device[dev][0].tagged = static_cast<uint64_t*>(p);
			per_device[dev][1].tagged = static_cast<uint64_t*>(p) + ROWS_SCRATCH_WORDS;
		}
		rows_scratch& sc = per_device[dev][s != nullptr];
		if (hold) {
			if (sc.user != s && sc.user != nullptr) {
				e = stream_drained(sc.user);
				if (e != hipSuccess) {
					return e;
				}
			}
			sc.user = s;
			if (++sc.epoch == 0) {
				++sc.epoch;
			}
		}
		*out = sc;
		if (hold) {
			*hold = std::move(g);
		}
		return hipSuccess;
	}
} // namespace

hipError_t prepare_gemm_rows_scratch() {
	rows_scratch sc;
	return get_rows_scratch(&sc, nullptr, nullptr);
}

template<int SETS> static hipError_t launch_rows_t(const uint8_t* w, const uint8_t* a, float* C, const float* residual, int m, int n, int groups, int splits, const rows_scratch& sc, hipStream_t s) {
	int shift = 0;
	while ((1 << shift) < splits) {
		++shift;
	}
	const dim3 grid(static_cast<unsigned>((n + STRIP_ROWS - 1) / STRIP_ROWS * splits)), block(SK_WAVES * 64);
	auto launch = [&](auto kernel) { return launch_kernel(KIND_GEMM, kernel, grid, block, 0, s, w, a, groups, shift, m, n, residual, C, sc.tagged, sc.epoch); };
	return m <= 8 ? launch(gemm_rows_kernel<8, 2, SETS>) : m <= 16 ? launch(gemm_rows_kernel<16, 2, SETS>) : m <= 24 ? launch(gemm_rows_kernel<24, 2, SETS>) : launch(gemm_rows_kernel<32, 2, SETS>);
}

// 1 <= M <= 32, K > 0; cut: plan_gemm_skinny, where gemm_rows_fits
hipError_t launch_gemm_rows(const void* W, const void* Aq, float* C, const float* residual, int64_t M, int64_t N, int64_t K, const gemm_skinny_cut& cut, hipStream_t s) {
	rows_scratch sc;
	scratch_hold hold;
	if (cut.splits > 1) {
		const hipError_t e = get_rows_scratch(&sc, &hold, s);
		if (e != hipSuccess) {
			return e;
		}
	}
	const uint8_t *w = static_cast<const uint8_t*>(W), *a = static_cast<const uint8_t*>(Aq);
	const int m = static_cast<int>(M), n = static_cast<int>(N), groups = static_cast<int>(K / GROUP_K);
	return cut.waves == SK_WAVES ? launch_rows_t<1>(w, a, C, residual, m, n, groups, cut.splits, sc, s) : launch_rows_t<2>(w, a, C, residual, m, n, groups, cut.splits, sc, s);
}

template<int SETS> static hipError_t launch_rows_gate_up_t(const uint8_t* wg, const uint8_t* wu, const uint8_t* a, uint8_t* out, float* gate_dbg, float* up_dbg, int m, int n, int groups, hipStream_t s) {
	auto launch = [&](auto kernel) { return launch_kernel(KIND_GEMM, kernel, dim3(static_cast<unsigned>(n / STRIP_ROWS)), dim3(SK_WAVES * 64), 0, s, wg, wu, a, groups, m, n, out, gate_dbg, up_dbg); };
	return m <= 8 ? launch(gemm_rows_gate_up_kernel<8, 1, SETS>) : m <= 16 ? launch(gemm_rows_gate_up_kernel<16, 1, SETS>) : m <= 24 ? launch(gemm_rows_gate_up_kernel<24, 1, SETS>) : launch(gemm_rows_gate_up_kernel<32, 1, SETS>);
}

hipError_t launch_gemm_rows_gate_up(const void* w_gate, const void* w_up, const void* aq, void* act_out, float* gate_dbg, float* up_dbg, int64_t M, int64_t n_ff, int64_t K, int waves, hipStream_t s) {
	const uint8_t *wg = static_cast<const uint8_t*>(w_gate), *wu = static_cast<const uint8_t*>(w_up), *a = static_cast<const uint8_t*>(aq);
	uint8_t* out = static_cast<uint8_t*>(act_out);
	const int m = static_cast<int>(M), n = static_cast<int>(n_ff), groups = static_cast<int>(K / GROUP_K);
	return waves == SK_WAVES ? launch_rows_gate_up_t<1>(wg, wu, a, out, gate_dbg, up_dbg, m, n, groups, s) : launch_rows_gate_up_t<2>(wg, wu, a, out, gate_dbg, up_dbg, m, n, groups, s);
}

} // namespace nh
