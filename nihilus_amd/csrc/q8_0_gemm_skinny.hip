// Batched-decode mat-mat for some dozens of activation rows, and for more on small grids: C[m][n] = dot(W row n, Aq row m), gfx950.  (Up to 32
// rows the kernel of q8_0_gemm_rows.hip has the shapes; this one runs those of its calls that cannot use its hand-off, to the same bits.)
//
// With so few rows the weights are read once and nothing is reused enough to leave the HBM roofline, so this is the
// streaming mat-vec again -- one workgroup per (32-row weight strip, K split), waves splitting the strip's K range,
// all of a chunk's loads issued before anything is waited for, one fixed-order reduction at the end -- with the
// v_dot4 inner product replaced by the int8 MFMA: the weight tile a wave fetches (one coalesced 16-byte-per-lane load
// in the tiled layout) is the B operand as it stands, the matching activation tile (served by L2: the activations
// are M*K bytes) is the A operand, and one v_mfma_i32_32x32x32_i8 yields the exact block sums of 32 rows x 32
// columns.  Scale products come from a v_mfma_f32_32x32x8_f16 on the blocks' fp16 scales (exact, same register layout),
// then one convert + one multiply-add per value.  Same arithmetic as the prefill kernel (reference
// vec_dot_q8_0_q8_0, cpu/avx_2.hpp:4534-4747; output [M][N], n fastest, cpu/avx_2.hpp:4934).
#include "q8_0_plan.h"

#include <mutex>

namespace nh {

typedef _Float16 sk_v4h __attribute__((ext_vector_type(4)));
typedef float sk_v16f __attribute__((ext_vector_type(16)));

// NT: past the caches, for weights that no other workgroup reads
template<bool NT, typename T> __device__ __forceinline__ T load_weights(const T* p) {
	if constexpr (NT) {
		return __builtin_nontemporal_load(p);
	} else {
		return *p;
	}
}

template<int MS, int GC, int WAVES, bool NT>
__global__ __launch_bounds__(WAVES * 64, 4) void gemm_skinny_kernel(const uint8_t* __restrict__ W, const uint8_t* __restrict__ A, int groups, int split_shift, int M, int N,
	float* C, const float* R, float* __restrict__ partials, unsigned* __restrict__ counters) {
	__shared__ float red[MS * 16][WAVES][64];
	__shared__ int last_flag;

	const int tid	 = threadIdx.x;
	const int lane	 = tid & 63;
	const int wave	 = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int splits = 1 << split_shift;
	const int strip	 = static_cast<int>(blockIdx.x >> split_shift);
	const int split	 = static_cast<int>(blockIdx.x) & (splits - 1);
	const int mg	 = static_cast<int>(blockIdx.y); // group of MS activation strips (more than 32 * MS rows: the weights are read once per group, from cache after the first)
	const int unit	 = mg * static_cast<int>(gridDim.x >> split_shift) + strip; // index of this (row group, weight strip) in the split scratch
	int g0, g1; // this wave's share of the strip's K range
	// sixteen waves: the shares that two workgroups of eight would have
	if constexpr (WAVES == SK_WIDE_WAVES) {
		wave_k_range(groups, split_shift + 1, 2 * split + (wave >> 3), SK_WAVES, wave & 7, g0, g1);
	} else {
		wave_k_range(groups, split_shift, split, WAVES, wave, g0, g1);
	}
	const int r		 = lane & 31;
	const int half	 = lane >> 5;

	sk_v16f acc[MS];
#pragma unroll
	for (int i = 0; i < MS; ++i) {
		acc[i] = sk_v16f{ 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0 };
	}

	const uint8_t* w_strip = W + macro_offset(strip, 0, groups);
	struct w_regs {
		v4i q[GROUP_BLOCKS];
		v2u d;
	};
	struct a_regs {
		v4i q[MS][GROUP_BLOCKS];
		v2u d[MS];
	};
	auto issue_w = [&](int g, w_regs& b) {
		const uint8_t* macro = w_strip + static_cast<int64_t>(g) * MACRO_BYTES;
#pragma unroll
		for (int j = 0; j < GROUP_BLOCKS; ++j) {
			b.q[j] = load_weights<NT>(reinterpret_cast<const v4i*>(macro + j * TILE_BYTES + 16 * lane));
		}
		b.d = load_weights<NT>(reinterpret_cast<const v2u*>(macro + MACRO_D_OFFSET + 8 * r));
	};
	// Activation rows beyond M are zero padding in the tiled operand.  Their lanes all read the strip's last row instead of
	// their own (zeros as well, since a strip with any padding ends in it): one cache line per load instead of one per four
	// lanes, so a batch of 4 rows costs a fraction of the cache traffic of a full strip, with no extra registers or branches.
	int a_q_off[MS], a_d_off[MS];
#pragma unroll
	for (int i = 0; i < MS; ++i) {
		const bool real = (mg * MS + i) * STRIP_ROWS + r < M;
		a_q_off[i]		= real ? 16 * lane : 16 * (STRIP_ROWS - 1);
		a_d_off[i]		= real ? 8 * r : 8 * (STRIP_ROWS - 1);
	}
	// With an odd number of activation strips the last group of two has only one: its second strip's loads go to the last strip that
	// exists (its results belong to no row and are dropped at the store).
	const int last_m_strip = (M + STRIP_ROWS - 1) / STRIP_ROWS - 1;
	auto issue_a = [&](int g, a_regs& b) {
#pragma unroll
		for (int i = 0; i < MS; ++i) {
			const uint8_t* am = A + macro_offset(min(mg * MS + i, last_m_strip), g, groups);
#pragma unroll
			for (int j = 0; j < GROUP_BLOCKS; ++j) {
				b.q[i][j] = *reinterpret_cast<const v4i*>(am + j * TILE_BYTES + a_q_off[i]);
			}
			b.d[i] = *reinterpret_cast<const v2u*>(am + MACRO_D_OFFSET + a_d_off[i]);
		}
	};
	auto compute = [&](const w_regs& w, const a_regs& a) {
		// lanes 32..63 feed the k = 4..7 slots of the scale MFMA: zero
		const v2u wdz = half ? v2u{ 0u, 0u } : w.d;
#pragma unroll
		for (int j = 0; j < GROUP_BLOCKS; ++j) {
			const v2u ws = scale_slot(wdz, j);
#pragma unroll
			for (int i = 0; i < MS; ++i) {
				const sk_v16f zf = { 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0 };
				const v16i zi	 = { 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0 };
				const v16i s	 = __builtin_amdgcn_mfma_i32_32x32x32_i8(a.q[i][j], w.q[j], zi, 0, 0, 0);
				const v2u as	 = scale_slot(half ? v2u{ 0u, 0u } : a.d[i], j);
				const sk_v16f p	 = __builtin_amdgcn_mfma_f32_32x32x8f16(__builtin_bit_cast(sk_v4h, as), __builtin_bit_cast(sk_v4h, ws), zf, 0, 0, 0);
#pragma unroll
				for (int e = 0; e < 16; ++e) {
					acc[i][e] = fmaf(static_cast<float>(s[e]), p[e], acc[i][e]);
				}
			}
		}
	};
	// GC groups per step: their loads are issued, then waited for together (loads complete in issue order, so a
	// short-latency activation load queued behind a weight load returns no earlier than it: prefetching one kind deeper
	// than the other buys nothing), then computed.  (The compiler sinks the second group's loads into the branch that
	// uses them, behind the first group's MFMAs; holding them in front, and one group per step, both measured the same
	// within 0.3 us on every shape of the crossover and 70B tables: the eight waves of two workgroups per CU are what
	// keeps bytes in flight, not the depth of one wave.)
	for (int g = g0; g < g1; g += GC) {
		w_regs w[GC];
		a_regs a[GC];
#pragma unroll
		for (int c = 0; c < GC; ++c) {
			issue_w(min(g + c, g1 - 1), w[c]); // past the end: the last group again (a cache hit, never used) so that the waits stay countable
		}
#pragma unroll
		for (int c = 0; c < GC; ++c) {
			issue_a(min(g + c, g1 - 1), a[c]);
		}
		__builtin_amdgcn_sched_barrier(0); // every load of the step before the first MFMA (left alone, the compiler interleaves them: measured slower)
#pragma unroll
		for (int c = 0; c < GC; ++c) {
			if (c == 0 || g + c < g1) {
				compute(w[c], a[c]);
			}
		}
	}
	// ---- the waves' partial sums through LDS; a wave finishes OWN of every lane's MS * 16 values ----
	// (One wave finishing them all, behind a tree of barriers, and reading the residual value by value behind its own stores was a chain
	// of 16 * MS memory latencies: [4096 x 4096] at 117 rows 17.2 us with a residual and 14.6 without; now 12.3 and 12.2.)
	constexpr int OWN = MS * 16 / WAVES;
	const int n		  = strip * STRIP_ROWS + r;
	const auto row_of = [&](int v) { return (mg * MS + (v >> 4)) * STRIP_ROWS + 8 * ((v & 15) >> 2) + 4 * half + (v & 3); };
	float add[OWN]; // R may be C: every element is read here and written below by the same thread
	if (R) {
#pragma unroll
		for (int o = 0; o < OWN; ++o) {
			const int m = row_of(wave * OWN + o);
			add[o]		= (m < M && n < N) ? R[static_cast<int64_t>(m) * N + n] : 0.0f;
		}
	}
#pragma unroll
	for (int i = 0; i < MS; ++i) {
#pragma unroll
		for (int e = 0; e < 16; ++e) {
			red[i * 16 + e][wave][lane] = acc[i][e];
		}
	}
	__syncthreads();
	float own[OWN];
#pragma unroll
	for (int o = 0; o < OWN; ++o) {
		const auto& p = red[wave * OWN + o];
		static_assert(WAVES == 8 || WAVES == 16, "a fixed tree over the waves' partial sums");
		const auto eight = [&](int w) {
			return ((p[w + 0][lane] + p[w + 4][lane]) + (p[w + 2][lane] + p[w + 6][lane])) + ((p[w + 1][lane] + p[w + 5][lane]) + (p[w + 3][lane] + p[w + 7][lane]));
		};
		own[o] = eight(0);
		if constexpr (WAVES == 16) {
			own[o] += eight(8);
		}
	}
	auto store = [&](float (&v)[OWN]) {
		if (R) {
#pragma unroll
			for (int o = 0; o < OWN; ++o) {
				v[o] += add[o];
			}
		}
#pragma unroll
		for (int o = 0; o < OWN; ++o) {
			const int m = row_of(wave * OWN + o);
			if (m < M && n < N) {
				C[static_cast<int64_t>(m) * N + n] = v[o];
			}
		}
	};
	if (splits == 1) {
		store(own);
		return;
	}

	// ---- K split over several workgroups: partial tiles through device-scope atomics, last arriver adds in split order ----
	float* tile = partials + static_cast<int64_t>(unit) * splits * (MS * 16 * 64) + wave * (OWN * 64) + lane;
#pragma unroll
	for (int o = 0; o < OWN; ++o) {
		__hip_atomic_store(&tile[static_cast<int64_t>(split) * (MS * 16 * 64) + o * 64], own[o], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
	}
	wait_stores_acknowledged();
	__syncthreads();
	if (tid == 0) {
		const unsigned prev = __hip_atomic_fetch_add(&counters[unit], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
		const int last		= (prev == static_cast<unsigned>(splits - 1));
		if (last) {
			__hip_atomic_store(&counters[unit], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
		}
		last_flag = last;
	}
	__syncthreads();
	if (!last_flag) {
		return;
	}
	// four splits' worth of partial sums requested at a time, added in split order
	float sum[OWN];
#pragma unroll
	for (int o = 0; o < OWN; ++o) {
		sum[o] = 0.0f;
	}
	for (int sp0 = 0; sp0 < splits; sp0 += 4) {
		float v[4][OWN];
#pragma unroll
		for (int u = 0; u < 4; ++u) {
#pragma unroll
			for (int o = 0; o < OWN; ++o) {
				v[u][o] = (sp0 + u < splits) ? __hip_atomic_load(&tile[static_cast<int64_t>(sp0 + u) * (MS * 16 * 64) + o * 64], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0.0f;
			}
		}
#pragma unroll
		for (int u = 0; u < 4; ++u) {
			if (sp0 + u < splits) {
#pragma unroll
				for (int o = 0; o < OWN; ++o) {
					sum[o] += v[u][o];
				}
			}
		}
	}
	store(sum);
}

// Scratch of the K-split paths (partial tiles and arrival counters): one allocation per device on first use, in two pairs: one for the
// launches of this kernel and of the tile kernel for up to 64 rows, one for the tile kernel's with more rows (which need no scratch if they
// must: they would have the others refused).  Of a pair one is the null stream's, which may not be queried while some other stream is
// being captured and so never shares, and one serves the other streams one at a time.
static_assert(GEMM_SPLIT_SCRATCH_FLOATS == SK_MAX_SPLIT_UNITS * 2 * 16 * 64 && GEMM_SPLIT_MAX_UNITS == SK_MAX_SPLIT_STRIPS, "scratch of one size");
struct skinny_scratch {
	float* partials	   = nullptr;
	unsigned* counters = nullptr;
	hipStream_t user   = nullptr; // stream of the last K-split launch
};
// hold == nullptr: make it if need be.  Otherwise a K-split launch on `s` is about to use it, and the caller keeps *hold until it is
// enqueued.  If the previous such launch of its part went to another stream that has not drained, hipErrorNotReady comes back.  Not
// checked for capturing streams.
static hipError_t get_skinny_scratch(skinny_scratch* out, bool few_rows = true, scratch_hold* hold = nullptr, hipStream_t s = nullptr) {
	constexpr int PARTS = 4;
	static std::recursive_mutex locks[64];
	static skinny_scratch per_device[64][PARTS];
	int dev		 = 0;
	hipError_t e = hipGetDevice(&dev);
	if (e != hipSuccess) {
		return e;
	}
	if (dev < 0 || dev >= 64) {
		return hipErrorInvalidDevice;
	}
	scratch_hold g(locks[dev]);
	if (!per_device[dev][0].partials) {
		void* p			   = nullptr;
		const size_t tiles = static_cast<size_t>(SK_MAX_SPLIT_UNITS) * 2 * 16 * 64 * 4; // two 32-row activation strips at most
		const size_t part  = tiles + SK_MAX_SPLIT_STRIPS * 4;
		e				   = hipMalloc(&p, PARTS * part);
		if (e != hipSuccess) {
			return e;
		}
		e = hipMemset(p, 0, PARTS * part);
		if (e != hipSuccess) {
			(void)hipFree(p);
			return e;
		}
		for (int i = 0; i < PARTS; ++i) {
			uint8_t* base				= static_cast<uint8_t*>(p) + i * part;
			per_device[dev][i].partials = reinterpret_cast<float*>(base);
			per_device[dev][i].counters = reinterpret_cast<unsigned*>(base + tiles);
		}
	}
	skinny_scratch& sc = per_device[dev][2 * !few_rows + (s != nullptr)];
	if (hold && !stream_is_capturing(s)) {
		if (sc.user != s && sc.user != nullptr) {
			e = stream_drained(sc.user);
			if (e != hipSuccess) {
				return e;
			}
		}
		sc.user = s;
	}
	*out = sc;
	if (hold) {
		*hold = std::move(g);
	}
	return hipSuccess;
}

// The same scratch for the tile kernel's K split over workgroups (GEMM_SPLIT_SCRATCH_FLOATS floats of tiles, GEMM_SPLIT_MAX_UNITS
// counters that every launch leaves at zero); same one-stream rule.
hipError_t acquire_gemm_split_scratch(float** partials, unsigned** counters, bool few_rows, scratch_hold* hold, hipStream_t s) {
	skinny_scratch sc;
	const hipError_t e = get_skinny_scratch(&sc, few_rows, hold, s);
	if (e != hipSuccess) {
		return e;
	}
	*partials = sc.partials;
	*counters = sc.counters;
	return hipSuccess;
}

hipError_t prepare_gemm_scratch() {
	skinny_scratch sc;
	const hipError_t e = get_skinny_scratch(&sc);
	return e != hipSuccess ? e : prepare_gemm_rows_scratch();
}

template<int MS> static hipError_t launch_skinny_t(int splits, int waves, const uint8_t* w, const uint8_t* a, float* C, const float* R, int m, int n, int groups, hipStream_t s) {
	const int strips   = (n + STRIP_ROWS - 1) / STRIP_ROWS;
	const int m_groups = ((m + STRIP_ROWS - 1) / STRIP_ROWS + MS - 1) / MS;
	skinny_scratch sc;
	scratch_hold hold;
	if (splits > 1) {
		const hipError_t e = get_skinny_scratch(&sc, true, &hold, s);
		if (e != hipSuccess) {
			return e;
		}
	}
	int shift = 0;
	while ((1 << shift) < splits) {
		++shift;
	}
	const dim3 grid(static_cast<unsigned>(strips * splits), static_cast<unsigned>(m_groups)), block(static_cast<unsigned>(64 * waves));
	const bool nt	  = gemm_skinny_past_caches(m, n, gemm_skinny_cut{ MS, splits, waves });
	const auto launch = [&](auto kernel) { return launch_kernel(KIND_GEMM, kernel, grid, block, 0, s, w, a, groups, shift, m, n, C, R, sc.partials, sc.counters); };
	if (waves == SK_WIDE_WAVES) {
		return nt ? launch(gemm_skinny_kernel<MS, 2, SK_WIDE_WAVES, true>) : launch(gemm_skinny_kernel<MS, 2, SK_WIDE_WAVES, false>);
	}
	return nt ? launch(gemm_skinny_kernel<MS, 2, SK_WAVES, true>) : launch(gemm_skinny_kernel<MS, 2, SK_WAVES, false>);
}

// cut: plan_gemm_streaming, or the stand-in for the rows kernel's or the tile kernel's (q8_0_plan.h)
hipError_t launch_gemm_skinny(const void* W, const void* Aq, float* C, int64_t M, int64_t N, int64_t K, const gemm_skinny_cut& cut, hipStream_t s, const float* residual) {
	const uint8_t* w = static_cast<const uint8_t*>(W);
	const uint8_t* a = static_cast<const uint8_t*>(Aq);
	const int groups = static_cast<int>(K / GROUP_K);
	if (cut.ms == 1) {
		return launch_skinny_t<1>(cut.splits, cut.waves, w, a, C, residual, static_cast<int>(M), static_cast<int>(N), groups, s);
	}
	return launch_skinny_t<2>(cut.splits, cut.waves, w, a, C, residual, static_cast<int>(M), static_cast<int>(N), groups, s);
}

} // namespace nh
