// The callers of ops.py for the common case, native: argument checks on the tensors themselves, the result's allocation, the C ABI call.
//
// What bounds a small call is the host: with the checks and the ctypes call in Python 6.5 - 7.5 us for kernels of 2 - 5 us, here 4.4 - 5, of which
// 3.5 are the runtime's launch (a convolution step and a gated norm of four tokens: 15.5 -> 9.8 us the pair; float32 256 x 512 . 512 x 1024
// 8.8 -> 6.1, what its kernel takes).  Every function returns None for anything but plain dense device
// tensors of one type with fitting shapes: the caller in ops.py then goes through its own checks, which raise or take the call.
// Nothing is kept from one call to the next.
#include "anygpu_hip.h"

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

namespace {

PyObject* raise_for = nullptr;      // capi.check(name, code)

// A tensor whose memory is what it says: no subclass, no functorch wrapper, no lazy conjugation or negation.
const at::Tensor* plain(PyObject* obj)
{
	static const c10::DispatchKeySet foreign({c10::DispatchKey::Python, c10::DispatchKey::PythonDispatcher, c10::DispatchKey::FuncTorchBatched,
	                                          c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::BatchedNestedTensor,
	                                          c10::DispatchKey::Functionalize, c10::DispatchKey::Conjugate, c10::DispatchKey::Negative,
	                                          c10::DispatchKey::ZeroTensor});
	if (!THPVariable_CheckExact(obj)) return nullptr;
	const at::Tensor& t = THPVariable_Unpack(obj);
	if (!t.defined() || !t.is_cuda() || t.layout() != c10::kStrided || t.key_set().has_any(foreign)) return nullptr;
	return &t;
}

// A result tensor that the caller brings: the operands' type and device.
bool fits(const at::Tensor& out, const at::Tensor& like) { return out.scalar_type() == like.scalar_type() && out.device() == like.device(); }

bool half_or_float(const at::Tensor& t) { return t.scalar_type() == at::kHalf || t.scalar_type() == at::kFloat; }

bool as_int(PyObject* obj, int64_t* out)
{
	if (!PyLong_Check(obj)) return false;
	int overflow = 0;
	*out = PyLong_AsLongLongAndOverflow(obj, &overflow);
	return overflow == 0;
}

bool as_float(PyObject* obj, float* out)
{
	if (!PyFloat_Check(obj) && !PyLong_CheckExact(obj)) return false;
	const double v = PyFloat_AsDouble(obj);
	if (v == -1.0 && PyErr_Occurred())
	{
		PyErr_Clear();
		return false;
	}
	*out = (float)v;
	return true;
}

// Under a dispatch mode the allocation belongs to the mode: ops.py makes it.
bool no_modes() { return !c10::impl::TorchDispatchModeTLS::any_modes_set(); }

at::Tensor result(at::IntArrayRef sizes, const at::Tensor& like)
{
	return at::empty(sizes, at::TensorOptions().dtype(like.dtype()).device(like.device()));
}

void* stream() { return c10::hip::getCurrentHIPStream(c10::hip::current_device()).stream(); }

const void* in(const at::Tensor& t) { return t.numel() ? t.const_data_ptr() : nullptr; }

// (the launch without the interpreter lock, as through ctypes)
template <typename F>
int launch(F&& call)
{
	void* const on = stream();
	PyThreadState* const held = PyEval_SaveThread();
	const int rc = call(on);
	PyEval_RestoreThread(held);
	return rc;
}

PyObject* finish(const char* name, int rc, const at::Tensor& out)
{
	if (rc != ANYGPU_OK)
	{
		PyObject* const done = raise_for ? PyObject_CallFunction(raise_for, "si", name, rc) : nullptr;
		Py_XDECREF(done);
		if (!PyErr_Occurred()) PyErr_Format(PyExc_RuntimeError, "%s failed with code %d", name, rc);
		return nullptr;
	}
	return THPVariable_Wrap(out);
}

int64_t at_least_one(int64_t v) { return v > 1 ? v : 1; }

#define DECLINE_UNLESS(cond) \
	if (!(cond)) Py_RETURN_NONE

// tensor_mm: lhs, rhs, out or None, b_layout, a_layout
PyObject* mm(PyObject*, PyObject* const* args, Py_ssize_t n_args)
{
	HANDLE_TH_ERRORS
	int64_t b_layout, a_layout;
	DECLINE_UNLESS(n_args == 5 && as_int(args[3], &b_layout) && as_int(args[4], &a_layout) && no_modes());
	const at::Tensor *a = plain(args[0]), *b = plain(args[1]);
	DECLINE_UNLESS(a && b && a->dim() == 2 && b->dim() == 2 && half_or_float(*a) && a->scalar_type() == b->scalar_type());
	DECLINE_UNLESS(a->stride(1) == 1 && b->stride(1) == 1);
	DECLINE_UNLESS((a_layout == ANYGPU_A_ROW_MAJOR || (a_layout == ANYGPU_A_COL_MAJOR && a->scalar_type() == at::kFloat)) &&
	               (b_layout == ANYGPU_B_ROW_MAJOR || b_layout == ANYGPU_B_COL_MAJOR));
	const bool a_row = a_layout == ANYGPU_A_ROW_MAJOR, b_row = b_layout == ANYGPU_B_ROW_MAJOR;
	const int64_t m = a->size(a_row ? 0 : 1), k = a->size(a_row ? 1 : 0), n = b->size(b_row ? 1 : 0);
	DECLINE_UNLESS(b->size(b_row ? 0 : 1) == k);
	at::Tensor out;
	if (args[2] == Py_None) out = result({m, n}, *a);
	else
	{
		const at::Tensor* given = plain(args[2]);
		DECLINE_UNLESS(given && fits(*given, *a) && given->dim() == 2 && given->size(0) == m && given->size(1) == n && given->stride(1) == 1);
		out = *given;
	}
	const int64_t lda = a->size(0) > 1 ? a->stride(0) : at_least_one(a->size(1));
	const int64_t ldb = b->size(0) > 1 ? b->stride(0) : at_least_one(b->size(1));
	const int64_t ldc = m > 1 ? out.stride(0) : at_least_one(n);
	const void *ap = in(*a), *bp = in(*b);
	void* cp = out.mutable_data_ptr();
	if (a->scalar_type() == at::kHalf)
		return finish("anygpu_gemm_f16_f32acc", launch([&](void* s) { return anygpu_gemm_f16_f32acc(ap, bp, cp, m, n, k, lda, ldb, ldc, (int)b_layout, s); }), out);
	return finish("anygpu_gemm_f32", launch([&](void* s) {
		return anygpu_gemm_f32((const float*)ap, (const float*)bp, nullptr, (float*)cp, m, n, k, lda, ldb, ldc, (int)a_layout, (int)b_layout, s); }), out);
	END_HANDLE_TH_ERRORS
}

// tensor_gemm: xt, wt, bt, b_layout
PyObject* gemm(PyObject*, PyObject* const* args, Py_ssize_t n_args)
{
	HANDLE_TH_ERRORS
	int64_t b_layout;
	DECLINE_UNLESS(n_args == 4 && as_int(args[3], &b_layout) && no_modes());
	const at::Tensor *x = plain(args[0]), *w = plain(args[1]), *b = plain(args[2]);
	DECLINE_UNLESS(x && w && b && x->dim() == 2 && w->dim() == 2 && half_or_float(*x));
	DECLINE_UNLESS(w->scalar_type() == x->scalar_type() && b->scalar_type() == x->scalar_type());
	DECLINE_UNLESS(x->is_contiguous() && w->is_contiguous() && b->is_contiguous() && (b_layout == ANYGPU_B_ROW_MAJOR || b_layout == ANYGPU_B_COL_MAJOR));
	const bool b_row = b_layout == ANYGPU_B_ROW_MAJOR;
	const int64_t m = x->size(0), k = x->size(1), n = w->size(b_row ? 1 : 0);
	DECLINE_UNLESS(w->size(b_row ? 0 : 1) == k && b->numel() == n);
	const at::Tensor out = result({m, n}, *x);
	const int64_t lda = at_least_one(k), ldb = at_least_one(w->size(1)), ldc = at_least_one(n);
	const void *xp = in(*x), *wp = in(*w), *bp = in(*b);
	void* cp = out.mutable_data_ptr();
	if (x->scalar_type() == at::kHalf)
		return finish("anygpu_gemm_f16_f32acc_bias", launch([&](void* s) { return anygpu_gemm_f16_f32acc_bias(xp, wp, bp, cp, m, n, k, lda, ldb, ldc, (int)b_layout, s); }), out);
	return finish("anygpu_gemm_f32", launch([&](void* s) {
		return anygpu_gemm_f32((const float*)xp, (const float*)wp, (const float*)bp, (float*)cp, m, n, k, lda, ldb, ldc, ANYGPU_A_ROW_MAJOR, (int)b_layout, s); }), out);
	END_HANDLE_TH_ERRORS
}

// tensor_gemma_linear_softcap: xt, wt, softcap
PyObject* linear_softcap(PyObject*, PyObject* const* args, Py_ssize_t n_args)
{
	HANDLE_TH_ERRORS
	float cap;
	DECLINE_UNLESS(n_args == 3 && as_float(args[2], &cap) && no_modes());
	const at::Tensor *x = plain(args[0]), *w = plain(args[1]);
	DECLINE_UNLESS(x && w && x->dim() == 3 && w->dim() == 2 && x->size(2) == w->size(1) && half_or_float(*x) && w->scalar_type() == x->scalar_type());
	DECLINE_UNLESS(x->is_contiguous() && w->is_contiguous());
	const int64_t m = x->size(0) * x->size(1), k = x->size(2), n = w->size(0), ld = at_least_one(k), ldc = at_least_one(n);
	const at::Tensor out = result({x->size(0), x->size(1), n}, *x);
	const void *xp = in(*x), *wp = in(*w);
	void* cp = out.mutable_data_ptr();
	if (x->scalar_type() == at::kHalf)
		return finish("anygpu_gemm_f16_f32acc_softcap", launch([&](void* s) { return anygpu_gemm_f16_f32acc_softcap(xp, wp, cp, m, n, k, ld, ld, ldc, ANYGPU_B_COL_MAJOR, cap, s); }), out);
	return finish("anygpu_gemm_f32_softcap", launch([&](void* s) {
		return anygpu_gemm_f32_softcap((const float*)xp, (const float*)wp, (float*)cp, m, n, k, ld, ld, ldc, ANYGPU_B_COL_MAJOR, cap, s); }), out);
	END_HANDLE_TH_ERRORS
}

// mlp_gemma2_fused_upproj: xt, wt_gp, wt_up, b_layout
PyObject* upproj(PyObject*, PyObject* const* args, Py_ssize_t n_args)
{
	HANDLE_TH_ERRORS
	int64_t b_layout;
	DECLINE_UNLESS(n_args == 4 && as_int(args[3], &b_layout) && no_modes());
	const at::Tensor *x = plain(args[0]), *g = plain(args[1]), *u = plain(args[2]);
	DECLINE_UNLESS(x && g && u && g->dim() == 2 && g->sizes() == u->sizes() && x->dim() >= 1 && half_or_float(*x));
	DECLINE_UNLESS(g->scalar_type() == x->scalar_type() && u->scalar_type() == x->scalar_type());
	DECLINE_UNLESS(x->is_contiguous() && g->is_contiguous() && u->is_contiguous() && (b_layout == ANYGPU_B_ROW_MAJOR || b_layout == ANYGPU_B_COL_MAJOR));
	const bool b_row = b_layout == ANYGPU_B_ROW_MAJOR;
	const int64_t k = g->size(b_row ? 0 : 1), n = g->size(b_row ? 1 : 0);
	DECLINE_UNLESS(x->size(-1) == k);
	const int64_t m = k ? x->numel() / k : 0, lda = at_least_one(k), ldb = at_least_one(g->size(1)), ldc = at_least_one(n);
	c10::SmallVector<int64_t, 5> sizes(x->sizes().begin(), x->sizes().end());
	sizes.back() = n;
	const at::Tensor out = result(sizes, *x);
	const void *xp = in(*x), *gp = in(*g), *up = in(*u);
	void* cp = out.mutable_data_ptr();
	if (x->scalar_type() == at::kHalf)
		return finish("anygpu_gemm_f16_f32acc_gelu_mul", launch([&](void* s) { return anygpu_gemm_f16_f32acc_gelu_mul(xp, gp, up, cp, m, n, k, lda, ldb, ldc, (int)b_layout, s); }), out);
	return finish("anygpu_gemm_f32_gelu_mul", launch([&](void* s) {
		return anygpu_gemm_f32_gelu_mul((const float*)xp, (const float*)gp, (const float*)up, (float*)cp, m, n, k, lda, ldb, ldc, (int)b_layout, s); }), out);
	END_HANDLE_TH_ERRORS
}

// tensor_softmax: x, out or None, alpha, softcap, causal, window, q_len, diag
PyObject* softmax(PyObject*, PyObject* const* args, Py_ssize_t n_args)
{
	HANDLE_TH_ERRORS
	float alpha, cap;
	int64_t causal, window, q_len, diag;
	DECLINE_UNLESS(n_args == 8 && as_float(args[2], &alpha) && as_float(args[3], &cap) && as_int(args[4], &causal) && as_int(args[5], &window) &&
	               as_int(args[6], &q_len) && as_int(args[7], &diag) && no_modes());
	const at::Tensor* x = plain(args[0]);
	DECLINE_UNLESS(x && x->dim() == 2 && (x->stride(1) == 1 || x->size(1) <= 1) && half_or_float(*x));
	const int64_t rows = x->size(0), cols = x->size(1);
	at::Tensor out;
	if (args[1] == Py_None) out = result({rows, cols}, *x);
	else
	{
		const at::Tensor* given = plain(args[1]);
		DECLINE_UNLESS(given && fits(*given, *x) && given->dim() == 2 && given->size(0) == rows && given->size(1) == cols && (given->stride(1) == 1 || cols <= 1));
		out = *given;
	}
	const int64_t xs = rows > 1 ? x->stride(0) : at_least_one(cols), ys = rows > 1 ? out.stride(0) : at_least_one(cols);
	const void* xp = in(*x);
	void* yp = out.mutable_data_ptr();
	const int on = causal != 0;
	if (x->scalar_type() == at::kHalf)
		return finish("anygpu_softmax_rows_f16", launch([&](void* s) { return anygpu_softmax_rows_f16(xp, yp, rows, cols, xs, ys, q_len, diag, alpha, cap, on, window, s); }), out);
	return finish("anygpu_softmax_rows_f32", launch([&](void* s) {
		return anygpu_softmax_rows_f32((const float*)xp, (float*)yp, rows, cols, xs, ys, q_len, diag, alpha, cap, on, window, s); }), out);
	END_HANDLE_TH_ERRORS
}

// tensor_causal_conv1d: xt, wt, bt, out or None
PyObject* conv1d(PyObject*, PyObject* const* args, Py_ssize_t n_args)
{
	HANDLE_TH_ERRORS
	// (a result that the caller brings goes through ops.py)
	DECLINE_UNLESS(n_args == 4 && args[3] == Py_None && no_modes());
	const at::Tensor *x = plain(args[0]), *w = plain(args[1]), *b = plain(args[2]);
	DECLINE_UNLESS(x && w && b && x->dim() == 3 && w->dim() == 2 && b->dim() == 1 && half_or_float(*x));
	DECLINE_UNLESS(x->size(1) == w->size(0) && w->size(0) == b->size(0) && w->size(1) <= 4);
	DECLINE_UNLESS(w->scalar_type() == x->scalar_type() && b->scalar_type() == x->scalar_type() && x->is_contiguous() && w->is_contiguous() && b->is_contiguous());
	const at::Tensor out = result(x->sizes(), *x);
	const int64_t batch = x->size(0), chan = x->size(1), len = x->size(2), width = w->size(1);
	const void *xp = in(*x), *wp = in(*w), *bp = in(*b);
	void* yp = out.mutable_data_ptr();
	if (x->scalar_type() == at::kHalf)
		return finish("anygpu_causal_conv1d_silu_f16", launch([&](void* s) { return anygpu_causal_conv1d_silu_f16(xp, wp, bp, yp, batch, chan, len, width, s); }), out);
	return finish("anygpu_causal_conv1d_silu_f32", launch([&](void* s) {
		return anygpu_causal_conv1d_silu_f32((const float*)xp, (const float*)wp, (const float*)bp, (float*)yp, batch, chan, len, width, s); }), out);
	END_HANDLE_TH_ERRORS
}

// tensor_causal_conv1d_update: xt, state, wt, bt
PyObject* conv1d_update(PyObject*, PyObject* const* args, Py_ssize_t n_args)
{
	HANDLE_TH_ERRORS
	DECLINE_UNLESS(n_args == 4 && no_modes());
	const at::Tensor *x = plain(args[0]), *state = plain(args[1]), *w = plain(args[2]), *b = plain(args[3]);
	DECLINE_UNLESS(x && state && w && b && x->dim() == 2 && state->dim() == 3 && w->dim() == 2 && b->dim() == 1 && half_or_float(*x));
	DECLINE_UNLESS(x->size(1) == w->size(0) && w->size(0) == b->size(0) && w->size(1) <= 4);
	DECLINE_UNLESS(state->size(0) == x->size(0) && state->size(1) == x->size(1) && state->size(2) == w->size(1) - 1);
	DECLINE_UNLESS(w->scalar_type() == x->scalar_type() && b->scalar_type() == x->scalar_type() && state->scalar_type() == x->scalar_type());
	DECLINE_UNLESS(x->is_contiguous() && state->is_contiguous() && w->is_contiguous() && b->is_contiguous());
	const at::Tensor out = result(x->sizes(), *x);
	const int64_t batch = x->size(0), chan = x->size(1), width = w->size(1);
	const void *xp = in(*x), *wp = in(*w), *bp = in(*b);
	void *sp = state->numel() ? state->mutable_data_ptr() : nullptr, *yp = out.mutable_data_ptr();
	if (x->scalar_type() == at::kHalf)
		return finish("anygpu_causal_conv1d_silu_update_f16", launch([&](void* s) { return anygpu_causal_conv1d_silu_update_f16(xp, sp, wp, bp, yp, batch, chan, width, s); }), out);
	return finish("anygpu_causal_conv1d_silu_update_f32", launch([&](void* s) {
		return anygpu_causal_conv1d_silu_update_f32((const float*)xp, (float*)sp, (const float*)wp, (const float*)bp, (float*)yp, batch, chan, width, s); }), out);
	END_HANDLE_TH_ERRORS
}

// tensor_rms_norm: xt, wt, eps, zero_centered, gate or None
PyObject* rms_norm(PyObject*, PyObject* const* args, Py_ssize_t n_args)
{
	HANDLE_TH_ERRORS
	float eps;
	int64_t centered;
	DECLINE_UNLESS(n_args == 5 && as_float(args[2], &eps) && as_int(args[3], &centered) && no_modes());
	const at::Tensor *x = plain(args[0]), *w = plain(args[1]), *z = args[4] == Py_None ? nullptr : plain(args[4]);
	DECLINE_UNLESS(x && w && (z || args[4] == Py_None) && w->dim() == 1 && x->dim() >= 1 && x->size(-1) == w->size(0) && half_or_float(*x));
	DECLINE_UNLESS(w->scalar_type() == x->scalar_type() && x->is_contiguous() && w->is_contiguous());
	DECLINE_UNLESS(!z || (z->sizes() == x->sizes() && z->scalar_type() == x->scalar_type() && z->is_contiguous()));
	const int64_t cols = w->size(0), rows = cols ? x->numel() / cols : 0;
	const at::Tensor out = result(x->sizes(), *x);
	const void *xp = in(*x), *wp = in(*w), *zp = z ? in(*z) : nullptr;
	void* yp = out.mutable_data_ptr();
	if (x->scalar_type() == at::kHalf)
		return finish("anygpu_gated_rmsnorm_f16", launch([&](void* s) { return anygpu_gated_rmsnorm_f16(xp, zp, wp, yp, rows, cols, eps, (int)centered, s); }), out);
	return finish("anygpu_gated_rmsnorm_f32", launch([&](void* s) {
		return anygpu_gated_rmsnorm_f32((const float*)xp, (const float*)zp, (const float*)wp, (float*)yp, rows, cols, eps, (int)centered, s); }), out);
	END_HANDLE_TH_ERRORS
}

// sdp_attention_masked_scaled_fwd, the fused form: q, k, v, mask, alpha
PyObject* attention_masked(PyObject*, PyObject* const* args, Py_ssize_t n_args)
{
	HANDLE_TH_ERRORS
	float alpha;
	DECLINE_UNLESS(n_args == 5 && as_float(args[4], &alpha) && no_modes());
	const at::Tensor *q = plain(args[0]), *k = plain(args[1]), *v = plain(args[2]), *mask = plain(args[3]);
	DECLINE_UNLESS(q && k && v && mask && half_or_float(*q) && k->scalar_type() == q->scalar_type() && v->scalar_type() == q->scalar_type() && mask->scalar_type() == q->scalar_type());
	const int64_t dims = q->dim();
	DECLINE_UNLESS(dims >= 2 && k->dim() == dims && mask->dim() == dims && k->sizes() == v->sizes());
	const int64_t n_q = q->size(-2), d = q->size(-1), n_k = k->size(-2);
	DECLINE_UNLESS(k->size(-1) == d && (d == 64 || d == 128 || d == 256) && n_q > 0 && n_k > 0 && q->numel() > 0);
	DECLINE_UNLESS(mask->size(-2) == n_q && mask->size(-1) == n_k);
	for (int64_t i = 0; i < dims - 2; ++i) DECLINE_UNLESS(k->size(i) == q->size(i) && mask->size(i) == 1);
	// (what is not dense is made so by ops.py)
	DECLINE_UNLESS(q->is_contiguous() && k->is_contiguous() && v->is_contiguous() && mask->is_contiguous());
	const at::Tensor out = result(q->sizes(), *q);
	const int64_t heads = q->numel() / (n_q * d);
	const void *qp = in(*q), *kp = in(*k), *vp = in(*v), *mp = in(*mask);
	void* yp = out.mutable_data_ptr();
	if (q->scalar_type() == at::kHalf)
		return finish("anygpu_sdp_attention_fwd_masked_f16", launch([&](void* s) { return anygpu_sdp_attention_fwd_masked_f16(qp, kp, vp, mp, yp, heads, 1, n_q, n_k, d, n_k, alpha, 0.0f, s); }), out);
	return finish("anygpu_sdp_attention_fwd_masked_f32", launch([&](void* s) {
		return anygpu_sdp_attention_fwd_masked_f32((const float*)qp, (const float*)kp, (const float*)vp, (const float*)mp, (float*)yp, heads, 1, n_q, n_k, d, n_k, alpha, 0.0f, s); }), out);
	END_HANDLE_TH_ERRORS
}

// sdp_attention_fwd: q, k, v, alpha, softcap, causal, window, decode or None
PyObject* attention(PyObject*, PyObject* const* args, Py_ssize_t n_args)
{
	HANDLE_TH_ERRORS
	float alpha, cap;
	int64_t causal, window, decode = 0;
	DECLINE_UNLESS(n_args == 8 && as_float(args[3], &alpha) && as_float(args[4], &cap) && as_int(args[5], &causal) && as_int(args[6], &window) &&
	               (args[7] == Py_None || as_int(args[7], &decode)) && no_modes());
	const at::Tensor *q = plain(args[0]), *k = plain(args[1]), *v = plain(args[2]);
	DECLINE_UNLESS(q && k && v && half_or_float(*q) && k->scalar_type() == q->scalar_type() && v->scalar_type() == q->scalar_type());
	const int64_t dims = q->dim();
	DECLINE_UNLESS(dims >= 3 && k->dim() == dims && k->sizes() == v->sizes() && k->size(-1) == q->size(-1) && k->size(-3) > 0 && q->size(-3) % k->size(-3) == 0);
	for (int64_t i = 0; i < dims - 3; ++i) DECLINE_UNLESS(k->size(i) == q->size(i));
	DECLINE_UNLESS(q->is_contiguous() && k->is_contiguous() && v->is_contiguous());
	const int64_t n_q = q->size(-2), d = q->size(-1), n_k = k->size(-2), q_per_kv = q->size(-3) / k->size(-3);
	const int64_t heads = n_q * d ? q->numel() / (n_q * d) : 0;
	if (args[7] == Py_None)
	{
		// (the rule of ops.sdp_attention_fwd, which explains it)
		const int64_t rows = q_per_kv * n_q;
		decode = n_k >= 256 && (d == 64 || d == 128 || d == 256) && ((0 < rows && rows <= 16) || (rows <= 128 && n_q <= 16 && heads <= 128));
	}
	const at::Tensor out = result(q->sizes(), *q);
	const void *qp = in(*q), *kp = in(*k), *vp = in(*v);
	void* yp = out.mutable_data_ptr();
	const bool half = q->scalar_type() == at::kHalf;
	const int on = causal != 0;
	if (decode)
	{
		const char* const name = half ? "anygpu_sdp_attention_decode_workspace_bytes" : "anygpu_sdp_attention_decode_f32_workspace_bytes";
		const int64_t need = half ? anygpu_sdp_attention_decode_workspace_bytes(heads, q_per_kv, n_q, n_k, d, on, window)
		                          : anygpu_sdp_attention_decode_f32_workspace_bytes(heads, q_per_kv, n_q, n_k, d, on, window);
		if (need < 0) return finish(name, (int)need, out);
		const int64_t bytes = need > 16 ? need : 16;
		const at::Tensor workspace = at::empty({bytes}, at::TensorOptions().dtype(at::kByte).device(q->device()));
		void* wp = workspace.mutable_data_ptr();
		if (half)
			return finish("anygpu_sdp_attention_decode_f16", launch([&](void* s) {
				return anygpu_sdp_attention_decode_f16(qp, kp, vp, yp, wp, bytes, heads, q_per_kv, n_q, n_k, d, alpha, cap, on, window, s); }), out);
		return finish("anygpu_sdp_attention_decode_f32", launch([&](void* s) {
			return anygpu_sdp_attention_decode_f32((const float*)qp, (const float*)kp, (const float*)vp, (float*)yp, wp, bytes, heads, q_per_kv, n_q, n_k, d, alpha, cap, on, window, s); }), out);
	}
	if (half)
		return finish("anygpu_sdp_attention_fwd_f16", launch([&](void* s) { return anygpu_sdp_attention_fwd_f16(qp, kp, vp, yp, heads, q_per_kv, n_q, n_k, d, alpha, cap, on, window, s); }), out);
	return finish("anygpu_sdp_attention_fwd_f32", launch([&](void* s) {
		return anygpu_sdp_attention_fwd_f32((const float*)qp, (const float*)kp, (const float*)vp, (float*)yp, heads, q_per_kv, n_q, n_k, d, alpha, cap, on, window, s); }), out);
	END_HANDLE_TH_ERRORS
}

PyObject* set_check(PyObject*, PyObject* callable)
{
	Py_INCREF(callable);
	Py_XDECREF(raise_for);
	raise_for = callable;
	Py_RETURN_NONE;
}

#define FAST(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {FAST(mm), FAST(gemm), FAST(linear_softcap), FAST(upproj), FAST(softmax), FAST(conv1d), FAST(conv1d_update), FAST(rms_norm),
                         FAST(attention_masked), FAST(attention), {"set_check", set_check, METH_O, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_torch_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

extern "C" __attribute__((visibility("default"))) PyObject* PyInit__torch_calls() { return PyModule_Create(&module); }
