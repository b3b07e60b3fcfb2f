// The calls of a model step on several rows (mul_mat, gemm, gemm_residual, rms_norm_quantize, gate_up_silu) as one native function each,
// for nihilus_amd/q8_0.py: the checks, the output's allocation, the current stream and the call through the C ABI.
//
// What bounds a small projection is the host.  A launch costs it 2.4 us; the same call from Python through ctypes took 7.9 us ([1024 x 4096]
// against one row): 1.3 us for the ctypes call itself, 1.5 us for each tensor that Python allocates, 2.4 us for checks, sizes and the
// stream, against 0.5 us, 0.6 us and 0.1 us here.
//
// A function returns the result tensor, or a non-zero status of the library as a number, or None for anything but plain tensors of the
// right kinds and sizes (subclasses, modes that intercept torch calls, wrong shapes, ...): the caller then goes the Python way, which
// also makes the error messages.  Nothing is enqueued before None is returned.
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/ops/empty.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include "nihilus_amd/q8_0_abi.h"

namespace {

// the arguments of a call, read one after the other; ok() once all have been
struct args {
	PyObject* const* at;
	Py_ssize_t left;
	bool good;

	args(PyObject* const* a, Py_ssize_t n, Py_ssize_t want) : at(a), left(n), good(n == want && !at::impl::torch_function_mode_enabled() && !c10::impl::TorchDispatchModeTLS::any_modes_set()) {
	}
	const at::Tensor* tensor(at::ScalarType type) {
		PyObject* o = good ? *at++ : nullptr;
		if (!o || !THPVariable_CheckExact(o)) {
			good = false;
			return nullptr;
		}
		const at::Tensor& t = THPVariable_Unpack(o);
		good				= t.defined() && t.is_cuda() && t.scalar_type() == type && t.has_storage() && t.is_contiguous();
		return good ? &t : nullptr;
	}
	const at::Tensor* tensor_or_none(at::ScalarType type) {
		if (good && *at == Py_None) {
			++at;
			return nullptr;
		}
		return tensor(type);
	}
	int64_t integer() {
		PyObject* o = good ? *at++ : nullptr;
		if (!o || !PyLong_CheckExact(o)) {
			good = false;
			return 0;
		}
		int overflow	= 0;
		const int64_t v = PyLong_AsLongLongAndOverflow(o, &overflow);
		good			= overflow == 0;
		return v;
	}
	float number() {
		PyObject* o = good ? *at++ : nullptr;
		if (!o || !PyFloat_CheckExact(o)) {
			good = false;
			return 0.0f;
		}
		return static_cast<float>(PyFloat_AS_DOUBLE(o));
	}
};

const float* floats(const at::Tensor& t) {
	return static_cast<const float*>(t.const_data_ptr());
}
at::Tensor bytes_like(const at::Tensor& t, int64_t n) {
	return at::empty({ n }, t.options().dtype(at::kByte));
}
void* stream() { // the current device's, as nihilus_amd/q8_0.py has it
	return c10::hip::getCurrentHIPStream().stream();
}
// rows of a [M, K] or [K] activation; -1 for any other shape
int64_t rows_of(const at::Tensor& x, int64_t k) {
	if (x.dim() == 1) {
		return x.size(0) == k ? 1 : -1;
	}
	return x.dim() == 2 && x.size(1) == k ? x.size(0) : -1;
}

// runs `call` without the interpreter's lock (a full queue makes a launch wait) and hands its output, or its status, to Python
template<typename Call> PyObject* finish(const at::Tensor& out, Call call) {
	int status;
	Py_BEGIN_ALLOW_THREADS
	status = call();
	Py_END_ALLOW_THREADS
	return status == 0 ? THPVariable_Wrap(out) : PyLong_FromLong(status);
}

// any exception of torch's (an allocation that fails, a tensor without memory): the Python way raises it
template<PyObject* (*F)(args&)> PyObject* guarded(PyObject* const* a, Py_ssize_t n, Py_ssize_t want) {
	try {
		args in(a, n, want);
		if (PyObject* out = in.good ? F(in) : nullptr) {
			return out;
		}
	} catch (const std::exception&) {
	}
	PyErr_Clear();
	Py_RETURN_NONE;
}
template<PyObject* (*F)(args&), int WANT> PyObject* entry(PyObject*, PyObject* const* a, Py_ssize_t n) {
	return guarded<F>(a, n, WANT);
}

// mul_mat(w_tiled, x, n, k, residual or None)
PyObject* mul_mat(args& in) {
	const at::Tensor* w = in.tensor(at::kByte);
	const at::Tensor* x = in.tensor(at::kFloat);
	const int64_t n = in.integer(), k = in.integer();
	const at::Tensor* residual = in.tensor_or_none(at::kFloat);
	const int64_t m			   = in.good ? rows_of(*x, k) : -1;
	if (m < 0 || w->numel() != nh_q8_0_tiled_bytes(n, k) || (residual && residual->numel() != m * n)) {
		return nullptr;
	}
	const int64_t need = nh_q8_0_mul_mat_workspace_bytes(m, k);
	if (need < 0) {
		return nullptr;
	}
	at::Tensor workspace;
	if (need > 0) {
		workspace = bytes_like(*x, need);
	}
	const at::Tensor y = at::empty({ m, n }, x->options());
	const void* wp	   = w->const_data_ptr();
	const float* xp	   = floats(*x);
	const float* rp	   = residual ? floats(*residual) : nullptr;
	float* yp		   = static_cast<float*>(y.mutable_data_ptr());
	void* ws		   = need > 0 ? workspace.mutable_data_ptr() : nullptr;
	void* s			   = stream();
	return finish(y, [&] { return nh_q8_0_mul_mat_scratch(wp, xp, rp, yp, m, n, k, ws, need, s); });
}

// gemm(w_tiled, aq_tiled, m, n, k, residual or None)
PyObject* gemm(args& in) {
	const at::Tensor* w = in.tensor(at::kByte);
	const at::Tensor* a = in.tensor(at::kByte);
	const int64_t m = in.integer(), n = in.integer(), k = in.integer();
	const at::Tensor* residual = in.tensor_or_none(at::kFloat);
	if (!in.good || w->numel() != nh_q8_0_tiled_bytes(n, k) || a->numel() != nh_q8_0_tiled_bytes(m, k) || (residual && residual->numel() != m * n)) {
		return nullptr;
	}
	const at::Tensor c = at::empty({ m, n }, w->options().dtype(at::kFloat));
	const void *wp = w->const_data_ptr(), *ap = a->const_data_ptr();
	const float* rp = residual ? floats(*residual) : nullptr;
	float* cp		= static_cast<float*>(c.mutable_data_ptr());
	void* s			= stream();
	return finish(c, [&] { return residual ? nh_q8_0_gemm_tiled_residual(wp, ap, rp, cp, m, n, k, s) : nh_q8_0_gemm_tiled(wp, ap, cp, m, n, k, s); });
}

// rms_norm_quantize(x, norm_weight, eps), tiled output
PyObject* rms_norm_quantize(args& in) {
	const at::Tensor* x	 = in.tensor(at::kFloat);
	const at::Tensor* nw = in.tensor(at::kFloat);
	const float eps		 = in.number();
	if (!in.good || x->dim() < 1 || x->dim() > 2) {
		return nullptr;
	}
	const int64_t k = x->size(x->dim() - 1), m = x->dim() == 2 ? x->size(0) : 1, size = nh_q8_0_tiled_bytes(m, k);
	if (nw->numel() != k || size < 0) {
		return nullptr;
	}
	const at::Tensor out = bytes_like(*x, size);
	const float *xp = floats(*x), *np = floats(*nw);
	void *op = out.mutable_data_ptr(), *s = stream();
	return finish(out, [&] { return nh_q8_0_rms_norm_quantize_tiled(xp, np, eps, op, m, k, s); });
}

// gate_up_silu(w_gate, w_up, aq_tiled, m, n_ff, k)
PyObject* gate_up_silu(args& in) {
	const at::Tensor* g = in.tensor(at::kByte);
	const at::Tensor* u = in.tensor(at::kByte);
	const at::Tensor* a = in.tensor(at::kByte);
	const int64_t m = in.integer(), n_ff = in.integer(), k = in.integer();
	if (!in.good) {
		return nullptr;
	}
	const int64_t size = nh_q8_0_tiled_bytes(m, n_ff), need = nh_q8_0_gate_up_silu_workspace_bytes(m, n_ff, k);
	if (size < 0 || need < 0) {
		return nullptr;
	}
	const int64_t w_size = nh_q8_0_tiled_bytes(n_ff, k);
	if (size > 0 && (g->numel() < w_size || u->numel() < w_size || a->numel() < nh_q8_0_tiled_bytes(m, k))) {
		return nullptr; // larger buffers than the operands are taken, as by the Python way
	}
	const at::Tensor out = bytes_like(*a, size);
	at::Tensor workspace;
	if (need > 0) {
		workspace = bytes_like(*a, need);
	}
	const void *gp = g->const_data_ptr(), *up = u->const_data_ptr(), *ap = a->const_data_ptr();
	void *op = out.mutable_data_ptr(), *ws = need > 0 ? workspace.mutable_data_ptr() : nullptr, *s = stream();
	return finish(out, [&] { return nh_q8_0_gemm_tiled_gate_up_silu(gp, up, ap, op, ws, need, m, n_ff, k, s); });
}

template<PyObject* (*F)(args&), int WANT> constexpr PyMethodDef method(const char* name) {
	return { name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&entry<F, WANT>)), METH_FASTCALL, nullptr };
}
PyMethodDef methods[] = { method<mul_mat, 5>("mul_mat"), method<gemm, 6>("gemm"), method<rms_norm_quantize, 3>("rms_norm_quantize"), method<gate_up_silu, 6>("gate_up_silu"),
	{ nullptr, nullptr, 0, nullptr } };
PyModuleDef module = { PyModuleDef_HEAD_INIT, "_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr };

} // namespace

PyMODINIT_FUNC PyInit__calls() {
	PyObject* m = PyModule_Create(&module);
	if (m && PyModule_AddStringConstant(m, "built_for", NH_BUILT_FOR) != 0) { // nihilus_amd/build.py
		Py_CLEAR(m);
	}
	return m;
}
