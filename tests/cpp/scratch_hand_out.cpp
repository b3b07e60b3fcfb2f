// The library's per-GPU hand-off scratch, two host threads and two streams -- on the CPU.
//
// The program defines the HIP runtime functions that the library calls and exports them (-rdynamic: the dynamic linker finds a program's own
// definitions first), so nothing here reaches a GPU: a launch is a record, a launch of the first thread takes as long as the test wants,
// and a stream is busy from the end of the first launch on it until reset().  The library itself is the built one.
//
// Per entry point: thread 1 is inside the runtime's launch call on stream A when thread 2 makes the same call on stream B.  Whatever B's
// call does (wait, refuse, take a form without scratch), it must not launch the kernel that A's call launches: both would hand partial
// sums over through the same words.
#define __HIP_PLATFORM_AMD__
#include <hip/hip_runtime_api.h>

#include <chrono>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "nihilus_amd/q8_0_abi.h"

namespace {
struct launch_record {
	const void* kernel;
	hipStream_t stream;
};
std::mutex state_lock;
std::condition_variable state_changed;
std::vector<launch_record> launches;
std::map<hipStream_t, bool> busy;
bool first_in_launch = false, second_done = false;
thread_local bool slow_launches = false;

hipError_t record_launch(const void* kernel, hipStream_t s) {
	std::unique_lock<std::mutex> g(state_lock);
	if (slow_launches) { // the launch call has begun and nothing is enqueued yet
		first_in_launch = true;
		state_changed.notify_all();
		state_changed.wait_for(g, std::chrono::milliseconds(200), [] { return second_done; });
	}
	launches.push_back({ kernel, s });
	busy[s] = true;
	return hipSuccess;
}
struct call_configuration {
	dim3 grid, block;
	size_t shmem;
	hipStream_t stream;
};
thread_local call_configuration pending;
} // namespace

extern "C" {
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shmem, hipStream_t s) {
	pending = { grid, block, shmem, s };
	return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shmem, hipStream_t* s) {
	*grid  = pending.grid;
	*block = pending.block;
	*shmem = pending.shmem;
	*s	   = pending.stream;
	return hipSuccess;
}
void** __hipRegisterFatBinary(const void*) {
	static void* handle = nullptr;
	return &handle;
}
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, dim3*, dim3*, int*) {
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {
}
void __hipUnregisterFatBinary(void**) {
}
hipError_t hipLaunchKernel(const void* kernel, dim3, dim3, void**, size_t, hipStream_t s) {
	return record_launch(kernel, s);
}
hipError_t hipExtLaunchKernel(const void* kernel, dim3, dim3, void**, size_t, hipStream_t s, hipEvent_t, hipEvent_t, int) {
	return record_launch(kernel, s);
}
hipError_t hipGetDevice(int* device) {
	*device = 0;
	return hipSuccess;
}
hipError_t hipGetDeviceCount(int* count) {
	*count = 1;
	return hipSuccess;
}
hipError_t hipGetDeviceProperties(hipDeviceProp_t* prop, int) { // (the header's macro gives it its versioned name)
	std::memset(prop, 0, sizeof(*prop));
	std::strcpy(prop->gcnArchName, "gfx950");
	prop->multiProcessorCount = 256;
	return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t bytes) {
	*p = std::aligned_alloc(4096, (bytes + 4095) / 4096 * 4096);
	return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) {
	return hipMalloc(p, bytes);
}
hipError_t hipFree(void* p) {
	std::free(p);
	return hipSuccess;
}
hipError_t hipMemset(void*, int, size_t) {
	return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void* symbol) {
	*p = const_cast<void*>(symbol);
	return hipSuccess;
}
hipError_t hipGetLastError() {
	return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* status) {
	*status = hipStreamCaptureStatusNone;
	return hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode*) {
	return hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t s) {
	std::lock_guard<std::mutex> g(state_lock);
	return busy[s] ? hipErrorNotReady : hipSuccess;
}
} // extern "C"

namespace {
void reset() {
	std::lock_guard<std::mutex> g(state_lock);
	launches.clear();
	busy.clear();
	first_in_launch = second_done = false;
}

// never looked at on the host: any 16-byte aligned addresses that do not overlap
template<typename T> T* operand(int i) {
	return reinterpret_cast<T*>(uintptr_t{ 0x100000000 } * static_cast<unsigned>(i + 1));
}

struct entry_point {
	std::string name;
	std::function<int(void*)> call;
};

std::vector<entry_point> entry_points() {
	std::vector<entry_point> all;
	const auto gemm = [&all](int64_t m, int64_t n, int64_t k) {
		all.push_back({ "gemm_tiled " + std::to_string(m) + " rows [" + std::to_string(n) + " x " + std::to_string(k) + "]",
			[=](void* s) { return nh_q8_0_gemm_tiled(operand<void>(0), operand<void>(1), operand<float>(2), m, n, k, s); } });
	};
	const auto mul_mat = [&all](int64_t m, int64_t n, int64_t k) {
		all.push_back({ "mul_mat " + std::to_string(m) + " rows [" + std::to_string(n) + " x " + std::to_string(k) + "]",
			[=](void* s) { return nh_q8_0_mul_mat(operand<void>(0), operand<float>(1), operand<float>(2), m, n, k, operand<void>(3), int64_t{ 1 } << 30, s); } });
	};
	gemm(4, 4096, 4096); // the rows kernel, two workgroups per strip
	gemm(24, 1024, 4096);
	gemm(40, 1024, 4096); // the streaming kernel
	gemm(64, 8192, 28672); // the tile kernel with streamed weights
	gemm(96, 8192, 8192); // the tile kernel, K over workgroups
	mul_mat(1, 4096, 14336);
	mul_mat(2, 4096, 14336);
	mul_mat(8, 4096, 4096);
	all.push_back({ "gemv_tiled_f32_noalloc", [](void* s) { return nh_q8_0_gemv_tiled_f32_noalloc(operand<void>(0), operand<float>(1), operand<float>(2), 4096, 14336, s); } });
	all.push_back({ "mul_mat_f32_activations", [](void* s) { return nh_q8_0_mul_mat_f32_activations(operand<void>(0), operand<float>(1), operand<float>(2), 1, 4096, 14336, s); } });
	all.push_back({ "gemv_tiled_group_f32", [](void* s) {
		const void* w[2]  = { operand<void>(0), operand<void>(1) };
		const float* x[2] = { operand<float>(2), operand<float>(3) };
		float* y[2]		  = { operand<float>(4), operand<float>(5) };
		const int64_t n[2] = { 4096, 4096 }, k[2] = { 14336, 14336 };
		return nh_q8_0_gemv_tiled_group_f32(w, x, y, nullptr, n, k, 2, s);
	} });
	all.push_back({ "a normalised row shared by a large mat-vec's workgroups", [](void* s) {
		const void* w[1]   = { operand<void>(0) };
		float* y[1]		   = { operand<float>(1) };
		const int64_t n[1] = { 128256 };
		return nh_q8_0_gemv_tiled_multi_norm_f32(w, y, n, 1, operand<float>(2), operand<float>(3), 1e-5f, 4096, s);
	} });
	all.push_back({ "ffn_f32", [](void* s) {
		return nh_q8_0_ffn_f32(operand<void>(0), operand<void>(1), operand<void>(2), operand<float>(3), operand<float>(4), 1e-5f, nullptr, operand<float>(5), 14336, 4096, 4096, s);
	} });
	all.push_back({ "decode_layer_f32", [](void* s) {
		const void* w[1]   = { operand<void>(0) };
		float* y[1]		   = { operand<float>(1) };
		const int64_t n[1] = { 6144 };
		return nh_q8_0_decode_layer_f32(operand<void>(2), operand<float>(3), operand<float>(4), operand<float>(5), operand<void>(6), operand<void>(7), operand<void>(8), operand<float>(9),
			operand<float>(10), w, y, n, 1, operand<float>(11), 1e-5f, 4096, 14336, s);
	} });
	return all;
}

// A mat-mat on one stream never has the mat-mat on another one refused where their scratch is not the same: (rows, N, K) running, (rows, N, K) called.
struct shape {
	int64_t m, n, k;
};
const std::pair<shape, shape> side_by_side[] = {
	{ { 96, 8192, 8192 }, { 64, 1024, 8192 } }, // the tile kernel with K over workgroups beside the streaming kernel with K over workgroups
	{ { 96, 8192, 8192 }, { 40, 1024, 4096 } },
	{ { 96, 8192, 8192 }, { 96, 8192, 8192 } }, // the second one takes a form without scratch
	{ { 128, 8192, 28672 }, { 128, 8192, 28672 } },
	{ { 66, 4096, 10240 }, { 66, 4096, 10240 } },
	{ { 4, 4096, 4096 }, { 40, 1024, 4096 } }, // the rows kernel beside the streaming kernel
	{ { 4, 4096, 4096 }, { 4, 4096, 4096 } }, // the second one runs on the streaming kernel
	{ { 40, 1024, 4096 }, { 96, 8192, 8192 } },
};

int failures = 0;
void expect(bool ok, const std::string& name, const char* what) {
	if (!ok) {
		std::printf("FAILED %s: %s\n", name.c_str(), what);
		++failures;
	}
}
} // namespace

int main() {
	const hipStream_t a = reinterpret_cast<hipStream_t>(0x10), b = reinterpret_cast<hipStream_t>(0x20);
	for (const entry_point& e : entry_points()) {
		reset();
		expect(e.call(a) == NH_OK, e.name, "refused on an idle GPU"); // sets the scratch up
		reset();
		int rc_a = -1, rc_b = -1;
		std::thread first([&] {
			slow_launches = true;
			rc_a		  = e.call(a);
		});
		{
			std::unique_lock<std::mutex> g(state_lock);
			state_changed.wait_for(g, std::chrono::seconds(10), [] { return first_in_launch; });
			expect(first_in_launch, e.name, "the first call launched nothing");
		}
		rc_b = e.call(b);
		{
			std::lock_guard<std::mutex> g(state_lock);
			second_done = true;
			state_changed.notify_all();
		}
		first.join();
		expect(rc_a == NH_OK, e.name, "the first call failed");
		expect(rc_b == NH_OK || rc_b == NH_ERR_BUSY, e.name, "the second call failed");
		std::vector<const void*> on_a, on_b;
		for (const launch_record& l : launches) {
			(l.stream == a ? on_a : on_b).push_back(l.kernel);
		}
		expect(rc_b == NH_ERR_BUSY ? on_b.empty() : !on_b.empty(), e.name, "a refused call launched, or an accepted one did not");
		for (const void* k : on_b) {
			for (const void* l : on_a) {
				expect(k != l, e.name, "both streams run the kernel that hands over through one scratch");
			}
		}
		// once A has drained, B is served by the same kernel
		const std::vector<const void*> want = on_a;
		reset();
		expect(e.call(b) == NH_OK, e.name, "refused on an idle GPU");
		expect(launches.size() == want.size() && !launches.empty() && launches.back().kernel == want.back(), e.name, "another form on an idle GPU");
		reset();
	}
	uintptr_t next_stream = 0x100; // streams that no earlier call has used: the library asks whether a stream is idle, not what it runs
	for (const auto& [one, two] : side_by_side) {
		const hipStream_t s1 = reinterpret_cast<hipStream_t>(next_stream += 0x10), s2 = reinterpret_cast<hipStream_t>(next_stream += 0x10);
		const auto call = [](const shape& x, void* s) { return nh_q8_0_gemm_tiled(operand<void>(0), operand<void>(1), operand<float>(2), x.m, x.n, x.k, s); };
		const std::string name = std::to_string(two.m) + " rows [" + std::to_string(two.n) + " x " + std::to_string(two.k) + "] beside " + std::to_string(one.m) + " rows [" + std::to_string(one.n) + " x " +
			std::to_string(one.k) + "]";
		reset();
		expect(call(one, s1) == NH_OK, name, "the first call failed");
		expect(call(two, s2) == NH_OK, name, "the second call failed");
		reset();
	}
	// ... and is refused, with nothing launched, where the form that is left needs scratch that a third stream is using
	reset();
	const hipStream_t s1 = reinterpret_cast<hipStream_t>(next_stream += 0x10), s2 = reinterpret_cast<hipStream_t>(next_stream += 0x10), s3 = reinterpret_cast<hipStream_t>(next_stream += 0x10);
	const auto four_rows = [](void* s) { return nh_q8_0_gemm_tiled(operand<void>(0), operand<void>(1), operand<float>(2), 4, 4096, 4096, s); };
	expect(four_rows(s1) == NH_OK && four_rows(s2) == NH_OK, "4 rows on three streams", "the first two are served");
	const size_t before = launches.size();
	expect(four_rows(s3) == NH_ERR_BUSY && launches.size() == before, "4 rows on three streams", "the third is refused");
	if (failures == 0) {
		std::printf("scratch hand-out ok\n");
	}
	return failures == 0 ? 0 : 1;
}
