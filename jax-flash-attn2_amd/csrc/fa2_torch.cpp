// Calls of the torch operator as a Python extension: the parameter block, the outputs and the scratch of an ordinary call are made here
// instead of in Python, where a decoding step on a short cache spent more time on them than its kernels take (B1 Hq32 Hkv8 D128, one row
// over 1029 keys 24.4 -> 11.2 us a call on the host, of which the two launches are 5; B2 H16 S512 D64 causal 19.7 -> 7.9; forward and
// backward of B1 H4 S64 137 -> 87).  Entry points are the same ones of include/fa2.h, given as addresses by whoever has opened
// libfa2_hip.so (_lib.py).
//
// Nothing depends on it but time: where it is not built, or for another torch or Python, the Python code makes every call.
//
// A call that needs anything else - a copy of an operand for its alignment, a padded head dim, a bias of another type, a tensor
// subclass - is left to the Python code (None is returned before anything has been launched), and so is every error of an argument's form.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <math.h>
#include <string.h>

#include "../../include/fa2.h"

namespace {

struct Library {
	int (*fwd)(const fa2_params*, void*);
	int (*bwd)(const fa2_params*, void*);
	int (*validate)(const fa2_params*, int);
	size_t (*fwd_scratch)(const fa2_params*);
	size_t (*bwd_scratch)(const fa2_params*);
	size_t (*bwd_split_scratch)(const fa2_params*);
};

// A call that this file does not serve.
struct Other {};

// Only plain tensors: a subclass may intercept what the Python code asks of it.
const at::Tensor& tensor(PyObject* o) {
	if (!THPVariable_CheckExact(o)) throw Other();
	return THPVariable_Unpack(o);
}

// (a number that a float cannot hold is Python's to refuse)
float number(PyObject* o) {
	double x;
	if (PyFloat_CheckExact(o)) {
		x = PyFloat_AS_DOUBLE(o);
	} else {
		if (!PyLong_CheckExact(o)) throw Other();
		x = PyLong_AsDouble(o);
		if (x == -1.0 && PyErr_Occurred()) throw python_error();
	}
	if (isfinite(x) && !isfinite((float)x)) throw Other();
	return (float)x;
}

// An operand in other memory than q's is Python's to refuse (or to let pass: pinned host memory).
const at::Tensor& beside(const at::Tensor& x, const at::Tensor& q) {
	if (x.device() != q.device()) throw Other();
	return x;
}

const int32_t* lengths(const at::Tensor& x, const at::Tensor& q, bool exact) {
	if (beside(x, q).scalar_type() != at::kInt || !x.is_contiguous() || (exact ? x.numel() != q.size(0) : x.numel() < q.size(0))) throw Other();
	return (const int32_t*)x.data_ptr();
}

// The kernels read 16 bytes at a time along the rows; anything else is copied first, by the Python code.
fa2_tensor rows(const at::Tensor& x) {
	const int64_t sb = x.stride(0), ss = x.stride(1), sh = x.stride(2);
	void* p = x.data_ptr();
	if (x.stride(3) != 1 || ((sb | ss | sh) & 7) || ((uintptr_t)p & 15)) throw Other();
	return fa2_tensor{p, sb, ss, sh};
}

int bias_dtype(at::ScalarType t) {
	switch (t) {
		case at::kHalf: return FA2_FP16;
		case at::kBFloat16: return FA2_BF16;
		case at::kFloat: return FA2_FP32;
		case at::kByte:
		case at::kBool: return FA2_MASK_U8;  // (one byte per position, 0 = masked)
		default: throw Other();
	}
}

int window_bound(PyObject* o) {
	if (!PyLong_CheckExact(o)) throw Other();
	int overflow = 0;
	const long long w = PyLong_AsLongLongAndOverflow(o, &overflow);
	if (overflow) return overflow < 0 ? -1 : 1 << 30;
	return w < -1 ? -1 : w > (1 << 30) ? 1 << 30 : (int)w;
}

// What a forward and a backward call share: (bias, seqlens, scale, p_drop, causal, seed, kv_lens, window, softcap) at `arg`.
void fill(fa2_params& p, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, PyObject* const* arg) {
	if (q.dim() != 4 || k.dim() != 4 || v.dim() != 4) throw Other();
	memset(&p, 0, sizeof(p));
	p.struct_size = sizeof(p);
	p.dtype = q.scalar_type() == at::kHalf ? FA2_FP16 : q.scalar_type() == at::kBFloat16 ? FA2_BF16 : throw Other();
	int64_t limit = 0;
	for (int i = 0; i < 4; ++i) limit |= q.size(i) | k.size(i);
	if (limit > INT32_MAX) throw Other();
	p.B = (int32_t)q.size(0);
	p.Sq = (int32_t)q.size(1);
	p.Hq = (int32_t)q.size(2);
	p.Sk = (int32_t)k.size(1);
	p.Hkv = (int32_t)k.size(2);
	const int64_t D = q.size(3);
	if (D <= 0 || D > 256) throw Other();
	p.D = D <= 64 ? 64 : D <= 128 ? 128 : 256;
	p.head_dim = (int32_t)D;
	p.q = rows(q);
	p.k = rows(beside(k, q));
	p.v = rows(beside(v, q));

	if (arg[0] != Py_None) {
		const at::Tensor& bias = beside(tensor(arg[0]), q);
		if (bias.dim() != 4 || bias.stride(3) != 1) throw Other();
		p.bias = bias.data_ptr();
		p.bias_dtype = bias_dtype(bias.scalar_type());
		p.bias_group = bias.size(1) == p.Hkv && p.Hkv != p.Hq && bias.size(1) != 1;
		p.bias_stride_b = bias.size(0) == 1 ? 0 : bias.stride(0);
		p.bias_stride_h = bias.size(1) == 1 ? 0 : bias.stride(1);
		p.bias_stride_m = bias.stride(2);
	}
	if (arg[1] != Py_None) p.seqlens = lengths(tensor(arg[1]), q, false);
	p.scale = arg[2] == Py_None ? (float)(1.0 / sqrt((double)D)) : number(arg[2]);
	p.p_drop = number(arg[3]);
	if (arg[4] != Py_True && arg[4] != Py_False) throw Other();
	p.causal = arg[4] == Py_True;
	if (arg[5] == Py_None) {
	} else if (PyLong_CheckExact(arg[5])) {
		p.seed = PyLong_AsUnsignedLongLongMask(arg[5]);
	} else {
		const at::Tensor& seed = beside(tensor(arg[5]), q);
		if (seed.scalar_type() != at::kLong || seed.numel() != 1) throw Other();
		p.seed_dev = (const uint64_t*)seed.data_ptr();
	}
	if (arg[6] != Py_None) p.kv_lens = lengths(tensor(arg[6]), q, true);
	if (arg[7] != Py_None) {
		if (!PyTuple_CheckExact(arg[7]) || PyTuple_GET_SIZE(arg[7]) != 2) throw Other();
		p.has_window = 1;
		p.window_left = window_bound(PyTuple_GET_ITEM(arg[7], 0));
		p.window_right = window_bound(PyTuple_GET_ITEM(arg[7], 1));
	}
	p.softcap = arg[8] == Py_None ? 0.f : number(arg[8]);
}

at::Tensor like(const at::Tensor& x) { return at::empty(x.sizes(), x.options().memory_format(at::MemoryFormat::Contiguous)); }
at::Tensor bytes(size_t n, const at::Tensor& x) { return at::empty({(int64_t)n}, x.options().dtype(at::kByte)); }

// Rows of fewer columns than the head dim of the kernels are served where the library takes them as they are.
void check_rows(const Library& lib, const fa2_params& p, int which) {
	if (p.head_dim == p.D) return;
	if (lib.validate(&p, which) == FA2_EUNSUPPORTED) throw Other();
	// (rows too far apart are copied, by the Python code)
	for (const fa2_tensor* t : {&p.q, &p.k, &p.v, &p.o, &p.dout})
		if (t->stride_s > 0x7fffffff / 256) throw Other();
}

// Other threads run Python while outputs and scratch are allocated (which may be a hipMalloc) and the kernels are launched.
struct NoGil {
	PyThreadState* state = PyEval_SaveThread();
	~NoGil() { PyEval_RestoreThread(state); }
};

const Library& library(PyObject* capsule) {
	const Library* lib = (const Library*)PyCapsule_GetPointer(capsule, "fa2");
	if (!lib) throw python_error();
	return *lib;
}

PyObject* none() { Py_RETURN_NONE; }

// forward(library, q, k, v, bias, seqlens, scale, p_drop, causal, seed, kv_lens, window, softcap, stream) -> (out, lse), the code of an
// error, or None (not served)
PyObject* forward(PyObject*, PyObject* const* arg, Py_ssize_t n) {
	HANDLE_TH_ERRORS
	if (n != 14) {
		PyErr_SetString(PyExc_TypeError, "forward takes 14 arguments");
		return nullptr;
	}
	try {
		const Library& lib = library(arg[0]);
		const at::Tensor &q = tensor(arg[1]), &k = tensor(arg[2]), &v = tensor(arg[3]);
		fa2_params p;
		fill(p, q, k, v, arg + 4);
		void* stream = PyLong_AsVoidPtr(arg[13]);
		if (!stream && PyErr_Occurred()) throw python_error();
		at::Tensor out, lse, scratch;
		int rc;
		{
			NoGil released;
			check_rows(lib, p, 0);
			out = like(q);
			lse = at::empty({p.B, p.Hq, p.Sq}, q.options().dtype(at::kFloat));
			p.o = rows(out);
			p.lse = (float*)lse.data_ptr();
			if (size_t need = lib.fwd_scratch(&p)) {
				scratch = bytes(need, q);
				p.scratch = scratch.data_ptr();
				p.scratch_bytes = need;
			}
			rc = lib.fwd(&p, stream);
		}
		if (rc) return PyLong_FromLong(rc);
		return Py_BuildValue("(NN)", THPVariable_Wrap(std::move(out)), THPVariable_Wrap(std::move(lse)));
	} catch (const Other&) {
		return none();
	}
	END_HANDLE_TH_ERRORS
}

// backward(library, q, k, v, <as forward, from bias to softcap>, out, lse, dout, stream) -> (dq, dk, dv), the code of an error, or None
PyObject* backward(PyObject*, PyObject* const* arg, Py_ssize_t n) {
	HANDLE_TH_ERRORS
	if (n != 17) {
		PyErr_SetString(PyExc_TypeError, "backward takes 17 arguments");
		return nullptr;
	}
	try {
		const Library& lib = library(arg[0]);
		const at::Tensor &q = tensor(arg[1]), &k = tensor(arg[2]), &v = tensor(arg[3]), &out = tensor(arg[13]), &lse = tensor(arg[14]),
		                 &dout = tensor(arg[15]);
		fa2_params p;
		fill(p, q, k, v, arg + 4);
		void* stream = PyLong_AsVoidPtr(arg[16]);
		if (!stream && PyErr_Occurred()) throw python_error();
		if (out.dim() != 4 || dout.dim() != 4) throw Other();
		p.o = rows(beside(out, q));
		p.dout = rows(beside(dout, q));
		if (beside(lse, q).scalar_type() != at::kFloat || !lse.is_contiguous() || lse.numel() < (int64_t)p.B * p.Hq * p.Sq) throw Other();
		p.lse = (float*)lse.data_ptr();
		at::Tensor dq, dk, dv, scratch;
		int rc;
		{
			NoGil released;
			check_rows(lib, p, 1);
			dq = like(q);
			dk = like(k);
			dv = like(v);
			p.dq = rows(dq);
			p.dk = rows(dk);
			p.dv = rows(dv);
			const size_t least = lib.bwd_scratch(&p), split = lib.bwd_split_scratch(&p);
			const size_t need = least > split ? least : split;
			scratch = bytes(need > 256 ? need : 256, q);
			p.scratch = scratch.data_ptr();
			p.scratch_bytes = need > 256 ? need : 256;
			rc = lib.bwd(&p, stream);
		}
		if (rc) return PyLong_FromLong(rc);
		return Py_BuildValue("(NNN)", THPVariable_Wrap(std::move(dq)), THPVariable_Wrap(std::move(dk)), THPVariable_Wrap(std::move(dv)));
	} catch (const Other&) {
		return none();
	}
	END_HANDLE_TH_ERRORS
}

// checked(q, k, v, bias, attention_mask, *numbers) -> 1: the shapes and types are in order (0: the Python code says what is not, or
// looks at what this does not); + 2: nothing differentiates, batches or traces the call, so that no autograd function has to stand around
// it.  (`numbers`: the further arguments that may be tensors with a gradient.)
PyObject* checked(PyObject*, PyObject* const* arg, Py_ssize_t n) {
	HANDLE_TH_ERRORS
	if (n < 5) {
		PyErr_SetString(PyExc_TypeError, "checked takes 5 arguments or more");
		return nullptr;
	}
	try {
		const at::Tensor &q = tensor(arg[0]), &k = tensor(arg[1]), &v = tensor(arg[2]);
		if (q.dim() != 4 || k.dim() != 4 || v.dim() != 4 || k.sizes() != v.sizes()) throw Other();
		const int64_t B = q.size(0), Hq = q.size(2), Hkv = k.size(2);
		if (k.size(0) != B || k.size(3) != q.size(3) || Hkv <= 0 || Hq % Hkv) throw Other();
		if (q.scalar_type() != k.scalar_type() || q.scalar_type() != v.scalar_type()) throw Other();
		if (q.scalar_type() != at::kHalf && q.scalar_type() != at::kBFloat16) throw Other();
		bool grad = q.requires_grad() || k.requires_grad() || v.requires_grad();
		bool forward_ad = q._fw_grad(0).defined() || k._fw_grad(0).defined() || v._fw_grad(0).defined();
		if (arg[4] != Py_None && (arg[3] != Py_None || q.size(1) != k.size(1))) throw Other();
		if (arg[3] != Py_None) {
			const at::Tensor& bias = tensor(arg[3]);
			if (bias.dim() != 4 || bias.size(2) != q.size(1) || bias.size(3) != k.size(1)) throw Other();
			if (bias.size(0) != 1 && bias.size(0) != B) throw Other();
			if (bias.size(1) != 1 && bias.size(1) != Hq && bias.size(1) != Hkv) throw Other();
			grad = grad || bias.requires_grad();
			forward_ad = forward_ad || bias._fw_grad(0).defined();
		}
		const bool transformed = c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) ||
		                         c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerBackMode);
		bool numbers = true;
		for (Py_ssize_t i = 5; i < n; ++i) numbers = numbers && (arg[i] == Py_None || PyFloat_CheckExact(arg[i]) || PyLong_CheckExact(arg[i]));
		const bool plain = numbers && !(grad && c10::GradMode::is_enabled()) && !forward_ad && !transformed && !torch::jit::tracer::isTracing();
		return PyLong_FromLong(plain ? 3 : 1);
	} catch (const Other&) {
		return PyLong_FromLong(0);
	}
	END_HANDLE_TH_ERRORS
}

// bind(addresses of fa2_fwd, fa2_bwd, fa2_validate, fa2_fwd_scratch_bytes, fa2_bwd_scratch_bytes, fa2_bwd_split_scratch_bytes)
PyObject* bind(PyObject*, PyObject* const* arg, Py_ssize_t n) {
	static_assert(sizeof(Library) == 6 * sizeof(void*), "");
	if (n != 6) {
		PyErr_SetString(PyExc_TypeError, "bind takes 6 addresses");
		return nullptr;
	}
	void* at[6];
	for (int i = 0; i < 6; ++i) {
		at[i] = PyLong_AsVoidPtr(arg[i]);
		if (!at[i]) {
			if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "an address is 0");
			return nullptr;
		}
	}
	Library* lib = new Library;
	memcpy((void*)lib, at, sizeof(at));
	PyObject* capsule = PyCapsule_New(lib, "fa2", [](PyObject* c) { delete (Library*)PyCapsule_GetPointer(c, "fa2"); });
	if (!capsule) delete lib;
	return capsule;
}

PyMethodDef methods[] = {{"bind", (PyCFunction)(void (*)(void))bind, METH_FASTCALL, nullptr},
                         {"checked", (PyCFunction)(void (*)(void))checked, METH_FASTCALL, nullptr},
                         {"forward", (PyCFunction)(void (*)(void))forward, METH_FASTCALL, nullptr},
                         {"backward", (PyCFunction)(void (*)(void))backward, METH_FASTCALL, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fa2_torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

#define FA2_STRING_(x) #x
#define FA2_STRING(x) FA2_STRING_(x)

PyMODINIT_FUNC PyInit__fa2_torch() {
	PyObject* m = PyModule_Create(&module);
	// (FA2_TORCH_VERSION: from the Makefile.  Another torch may lay its tensors out otherwise and load this file all the same.)
	if (m && PyModule_AddObject(m, "built_for", PyUnicode_FromFormat("%s %d.%d", FA2_STRING(FA2_TORCH_VERSION), PY_MAJOR_VERSION, PY_MINOR_VERSION))) Py_CLEAR(m);
	return m;
}
