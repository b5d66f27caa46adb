// The per-call host work of the Python entry points in native code: checks, output and scratch allocation, the argument
// block and the call into libaf3_dpa.so.  A small call's kernels run for 5 us; the same work in Python took 13 to 45 us.
//
// Every function takes the plain case of its entry point -- ordinary device tensors of matching types on the current
// device, innermost stride 1 -- and answers None for anything else (and for every malformed call), which sends the caller
// to the Python implementation with its conversions and error messages.  A negative number is an af3_status.
#include <Python.h>

#include <array>
#include <cmath>
#include <mutex>
#include <unordered_map>
#include <vector>

#include <ATen/core/Tensor.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/ops/clone.h>
#include <ATen/ops/linear.h>
#include <ATen/ops/matmul.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/af3_dpa.h"

extern "C" int64_t af3_dpa_workspace_used(const af3_dpa_params*);   // (api.hip; not part of the ABI)
extern "C" int     af3_dpa_log2_domain(const af3_dpa_params*);            // (likewise)
extern "C" int af3_project_suits(int64_t, int64_t, int64_t);              // (projection.hip, likewise)
extern "C" int af3_grid_project(const void*, const int64_t*, const void*, const void*, float, const void*, const void*, const void*, const void*, const void*, int64_t, int64_t, int32_t, float, void*,
								void*, void*, void*, void*, void*);        // (grid_project.hip, likewise)
extern "C" int af3_project(const void*, const void*, const void*, void*, int64_t, int64_t, int64_t, int32_t, void*);

namespace {

using at::Tensor;

// ---- plain tensors ----------------------------------------------------------------------------------------------------
const Tensor* tensor_of(PyObject* o) { return THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr; }

bool on_device(const Tensor& t, int dev) { return t.is_cuda() && t.get_device() == dev; }
bool inner_1(const Tensor& t) { return t.stride(-1) == 1; }
int  dtype_code(const Tensor& t) { return t.scalar_type() == at::kBFloat16 ? AF3_BF16 : t.scalar_type() == at::kFloat ? AF3_F32 : -1; }
// the current device when the (first) tensor is on it, -1 otherwise; asks the runtime only about device tensors
int device_of(const Tensor* t) {
	if(!t || !t->is_cuda()) return -1;
	const int dev = (int)c10::hip::current_device();
	return t->get_device() == dev ? dev : -1;
}
void* current_stream(int dev) { return (void*)c10::hip::getCurrentHIPStream((c10::DeviceIndex)dev).stream(); }
Tensor new_tensor(at::IntArrayRef sizes, at::ScalarType type, int dev) {
	return Tensor(at::detail::empty_cuda(sizes, type, at::Device(at::kCUDA, (c10::DeviceIndex)dev), std::nullopt));
}
// scratch of one call: the caching allocator hands the block to later work of the same stream only
at::DataPtr new_scratch(int64_t bytes) { return c10::hip::HIPCachingAllocator::get()->allocate((size_t)bytes); }
PyObject* none() { Py_RETURN_NONE; }
PyObject* wrap(Tensor&& t) { return THPVariable_Wrap(std::move(t)); }

struct without_gil {
	PyThreadState* s = PyEval_SaveThread();
	~without_gil() { PyEval_RestoreThread(s); }
};

// key mask in any of its shapes ([L], [B|1, L], [B|1, 1, 1, L], bool): pointer and batch stride (0: one row for all)
struct key_mask {
	const uint8_t* ptr = nullptr;
	int64_t        stride = 0;
};
bool mask_of(PyObject* o, int64_t B, int64_t L, int dev, key_mask& m) {
	if(o == Py_None) return true;
	const Tensor* t = tensor_of(o);
	if(!t || !on_device(*t, dev) || t->scalar_type() != at::kBool) return false;
	const int64_t d = t->dim();
	if(d != 1 && d != 2 && d != 4) return false;
	if(t->size(-1) != L || !inner_1(*t)) return false;
	if(d == 4 && (t->size(1) != 1 || t->size(2) != 1)) return false;
	if(d > 1 && t->size(0) != 1 && t->size(0) != B) return false;
	m.ptr    = static_cast<const uint8_t*>(t->const_data_ptr());
	m.stride = d > 1 && t->size(0) != 1 ? t->stride(0) : 0;
	return true;
}
bool bias_of(PyObject* o, int64_t H, int64_t L, int dev, const Tensor*& t) {
	t = nullptr;
	if(o == Py_None) return true;
	t = tensor_of(o);
	return t && on_device(*t, dev) && t->dim() == 3 && t->size(0) == H && t->size(1) >= L && t->size(2) >= L && inner_1(*t);
}

void put_strides(int64_t (&dst)[3], const Tensor& t) { dst[0] = t.stride(0), dst[1] = t.stride(1), dst[2] = t.stride(2); }
void put_bias(af3_dpa_params& p, const Tensor& b) {
	p.bias = b.const_data_ptr(), p.bias_stride[0] = b.stride(0), p.bias_stride[1] = b.stride(1), p.bias_dtype = dtype_code(b);
}
af3_dpa_params block(int64_t B, int64_t H, int64_t L, int64_t D, int code, int64_t hint) {
	af3_dpa_params p{};
	p.B = B, p.H = H, p.L = L, p.D = D;
	p.io_dtype = p.out_dtype = p.mma_dtype = code;
	p.softmax_scale = (float)std::pow((double)D, -0.5);
	p.q_descale = p.k_descale = p.v_descale = 1.f;
	p.reserved = (int32_t)hint;
	return p;
}
at::DataPtr workspace_for(af3_dpa_params& p, bool exact_bias) {
	at::DataPtr   ws;
	if(!exact_bias) p.reserved |= 4;
	const int64_t bytes = exact_bias ? 0 : af3_dpa_workspace_used(&p);
	if(bytes > 0) ws = new_scratch(bytes), p.workspace = ws.get(), p.workspace_bytes = bytes;
	return ws;
}
int forward(af3_dpa_params& p, bool exact_bias, int dev) {
	const at::DataPtr ws = workspace_for(p, exact_bias);
	return af3_dpa_forward(&p, current_stream(dev));
}
PyObject* answer(int rc, Tensor&& out) { return rc == AF3_OK ? wrap(std::move(out)) : PyLong_FromLong(rc); }

// ---- matrices derived from weights ------------------------------------------------------------------------------------
// Remembered for as long as their sources are the same live tensors at the same version, address and layout.  The weak
// reference keeps a source's address from being handed to another tensor, so the address alone identifies it.  An entry goes with
// its first source (fused.py hears of that and calls forget_source); past MAX_DERIVED entries all go.  Guarded by the GIL.
constexpr size_t MAX_DERIVED = 1024;
using derived_key = std::array<uintptr_t, 5>;   // what (tag), up to four sources
struct key_hash {
	size_t operator()(const derived_key& k) const {
		size_t h = 0;
		for(uintptr_t v : k) h = (h ^ (size_t)(v >> 4)) * 0x9E3779B97F4A7C15ull + (v & 15);
		return h;
	}
};
struct source {
	c10::weak_intrusive_ptr<c10::TensorImpl> ref;
	const void*      ptr;
	int64_t          version;
	at::ScalarType   type;
	std::vector<int64_t> sizes, strides;
};
struct derived {
	std::vector<source> sources;
	Tensor              value;
};
std::unordered_map<derived_key, derived, key_hash>* g_derived = new std::unordered_map<derived_key, derived, key_hash>();   // (never destroyed: tensors must not be freed after the runtime)

bool make_key(int64_t tag, PyObject* const* o, Py_ssize_t n, derived_key& k) {
	k.fill(0);
	k[0] = (uintptr_t)tag;
	if(n < 1 || n > 4) return false;
	for(Py_ssize_t i = 0; i < n; i++) {
		const Tensor* t = tensor_of(o[i]);
		if(!t || t->is_inference()) return false;
		k[1 + i] = reinterpret_cast<uintptr_t>(t->unsafeGetTensorImpl());
	}
	return true;
}
const Tensor* derived_of(int64_t tag, PyObject* const* o, Py_ssize_t n) {
	derived_key k;
	if(!make_key(tag, o, n, k)) return nullptr;
	const auto it = g_derived->find(k);
	if(it == g_derived->end()) return nullptr;
	for(Py_ssize_t i = 0; i < n; i++) {
		const Tensor& t = *tensor_of(o[i]);
		const source& s = it->second.sources[i];
		if(s.ptr != t.const_data_ptr() || s.version != (int64_t)t._version() || s.type != t.scalar_type() || t.sizes() != s.sizes || t.strides() != s.strides) return nullptr;
	}
	return &it->second.value;
}
// remember(tag, value, source...): True for a new entry, None where it is there already or the tensors cannot be remembered
PyObject* py_remember(PyObject*, PyObject* const* a, Py_ssize_t n) {
	HANDLE_TH_ERRORS
	derived_key   k;
	const Tensor* value = n >= 3 ? tensor_of(a[1]) : nullptr;
	if(!value || !make_key(PyLong_AsLongLong(a[0]), a + 2, n - 2, k)) return none();
	const Tensor* known = derived_of(PyLong_AsLongLong(a[0]), a + 2, n - 2);
	if(known && known->is_same(*value)) return none();
	for(auto it = g_derived->begin(); it != g_derived->end();) {
		bool dead = false;
		for(const source& s : it->second.sources) dead = dead || s.ref.expired();
		it = dead ? g_derived->erase(it) : std::next(it);
	}
	if(g_derived->size() >= MAX_DERIVED) g_derived->clear();
	derived d;
	d.value = *value;
	for(Py_ssize_t i = 2; i < n; i++) {
		const Tensor& t = *tensor_of(a[i]);
		d.sources.push_back(source{c10::weak_intrusive_ptr<c10::TensorImpl>(t.getIntrusivePtr()), t.const_data_ptr(), (int64_t)t._version(), t.scalar_type(), t.sizes().vec(), t.strides().vec()});
	}
	(*g_derived)[k] = std::move(d);
	Py_RETURN_TRUE;
	END_HANDLE_TH_ERRORS
}
// recalls(tag, source...): whether a matrix is remembered for these
PyObject* py_recalls(PyObject*, PyObject* const* a, Py_ssize_t n) {
	HANDLE_TH_ERRORS
	return PyBool_FromLong(n >= 2 && derived_of(PyLong_AsLongLong(a[0]), a + 1, n - 1) != nullptr);
	END_HANDLE_TH_ERRORS
}
// forget_source(address of a source's TensorImpl, as Tensor._cdata gives it)
PyObject* py_forget_source(PyObject*, PyObject* const* a, Py_ssize_t n) {
	const uintptr_t source = n == 1 ? (uintptr_t)PyLong_AsUnsignedLongLong(a[0]) : 0;
	if(PyErr_Occurred()) return nullptr;
	for(auto it = g_derived->begin(); it != g_derived->end();) {
		bool uses = false;
		for(size_t i = 1; i < it->first.size(); i++) uses = uses || it->first[i] == source;
		it = source && uses ? g_derived->erase(it) : std::next(it);
	}
	return none();
}
PyObject* py_forget(PyObject*, PyObject*) {
	g_derived->clear();
	return none();
}
// the tags fused.py remembers its matrices under
enum : int64_t { FUSED_WEIGHT = 1, Q_BIAS_ROW = 2, OUT_PROJ_T = 3, GLU_T = 4 };
int64_t tag_of(int64_t what, int64_t head, int code) { return what | (head << 8) | ((int64_t)code << 40); }

// ---- attention --------------------------------------------------------------------------------------------------------
// attention(q, k, v, mask, bias, kernel hint, exact bias)
PyObject* py_attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
	HANDLE_TH_ERRORS
	if(n != 7) return none();
	const Tensor *q = tensor_of(a[0]), *k = tensor_of(a[1]), *v = tensor_of(a[2]), *bias;
	if(!q || !k || !v || q->dim() != 4 || q->numel() == 0) return none();
	const int dev = device_of(q), code = dtype_code(*q);
	if(dev < 0 || code < 0 || k->scalar_type() != q->scalar_type() || v->scalar_type() != q->scalar_type() || k->sizes() != q->sizes() || v->sizes() != q->sizes()) return none();
	if(!on_device(*k, dev) || !on_device(*v, dev) || !inner_1(*q) || !inner_1(*k) || !inner_1(*v)) return none();
	const int64_t B = q->size(0), H = q->size(1), L = q->size(2), D = q->size(3);
	key_mask m;
	if(!mask_of(a[3], B, L, dev, m) || !bias_of(a[4], H, L, dev, bias) || (bias && bias->scalar_type() != q->scalar_type())) return none();
	af3_dpa_params p = block(B, H, L, D, code, PyLong_AsLong(a[5]));
	const bool     exact = a[6] == Py_True;
	Tensor         out;
	int            rc;
	{
		without_gil g;
		out = new_tensor(q->sizes(), q->scalar_type(), dev);
		p.q = q->const_data_ptr(), p.k = k->const_data_ptr(), p.v = v->const_data_ptr(), p.out = out.data_ptr();
		put_strides(p.q_stride, *q), put_strides(p.k_stride, *k), put_strides(p.v_stride, *v), put_strides(p.out_stride, out);
		if(bias) put_bias(p, *bias);
		p.key_mask = m.ptr, p.key_mask_stride_b = m.stride;
		rc = forward(p, exact, dev);
	}
	return answer(rc, std::move(out));
	END_HANDLE_TH_ERRORS
}

// attention_fp8(q, k, v, mask, bias, compensated): quantise (two launches), attend
PyObject* py_attention_fp8(PyObject*, PyObject* const* a, Py_ssize_t n) {
	HANDLE_TH_ERRORS
	if(n != 6) return none();
	const Tensor *q = tensor_of(a[0]), *k = tensor_of(a[1]), *v = tensor_of(a[2]), *bias;
	if(!q || !k || !v || q->dim() != 4 || q->numel() == 0) return none();
	const int dev = device_of(q), code = dtype_code(*q);
	if(dev < 0 || code < 0 || k->scalar_type() != q->scalar_type() || v->scalar_type() != q->scalar_type() || k->sizes() != q->sizes() || v->sizes() != q->sizes()) return none();
	if(!on_device(*k, dev) || !on_device(*v, dev) || !q->is_contiguous() || !k->is_contiguous() || !v->is_contiguous()) return none();
	const int64_t B = q->size(0), H = q->size(1), L = q->size(2), D = q->size(3);
	key_mask m;
	if(D % 4 != 0 || !mask_of(a[3], B, L, dev, m) || !bias_of(a[4], H, L, dev, bias) || (bias && bias->scalar_type() != at::kBFloat16)) return none();
	const bool comp = a[5] == Py_True;
	Tensor     out;
	int        rc;
	{
		without_gil g;
		out = new_tensor(q->sizes(), q->scalar_type(), dev);
		// one block: q8, k8, their residuals, v8t (rows padded to 16 keys), the quantiser's floats
		const int64_t each = (q->numel() + 255) & ~255ll, lpad = (L + 15) / 16 * 16, vt = (B * H * D * lpad + 255) & ~255ll;
		at::DataPtr   mem  = new_scratch((comp ? 4 : 2) * each + vt + 256 + AF3_QKV_SCRATCH_FLOATS * 4);
		uint8_t*      at8  = static_cast<uint8_t*>(mem.get());
		uint8_t *q8 = at8, *k8 = q8 + each, *qlo = comp ? k8 + each : nullptr, *klo = comp ? qlo + each : nullptr, *v8 = k8 + (comp ? 3 : 1) * each;
		float *descales = reinterpret_cast<float*>(v8 + vt), *scratch = descales + 64;
		rc = af3_quantize_qkv_fp8_e4m3(q->const_data_ptr(), k->const_data_ptr(), v->const_data_ptr(), code, B, H, L, D, (float)std::pow((double)D, -0.5), q8, k8, v8, lpad, qlo, klo, descales, scratch,
									   current_stream(dev));
		if(rc == AF3_OK) {
			af3_dpa_params p = block(B, H, L, D, AF3_FP8_E4M3, 0);
			p.softmax_scale = 1.f, p.out_dtype = code;
			p.q = q8, p.k = k8, p.v = v8, p.q_lo = qlo, p.k_lo = klo, p.out = out.data_ptr(), p.device_descales = descales;
			put_strides(p.q_stride, *q), put_strides(p.k_stride, *q), put_strides(p.out_stride, out);
			p.v_stride[0] = H * D * lpad, p.v_stride[1] = D * lpad, p.v_stride[2] = lpad;
			if(bias) put_bias(p, *bias);
			p.key_mask = m.ptr, p.key_mask_stride_b = m.stride;
			rc = af3_dpa_forward(&p, current_stream(dev));
		}
	}
	return answer(rc, std::move(out));
	END_HANDLE_TH_ERRORS
}

// the attention launch on the projections y [B*N, 4C] -- per token and head (k | v | q | gate) -- into out [B, N, C]
int attend(const Tensor& y, int64_t B, int64_t N, int64_t head, const key_mask& m, const Tensor* bias, Tensor& out, int64_t hint, bool exact, int dev) {
	const int64_t C = y.size(1) / 4, K = C / head, esz = (int64_t)y.element_size();
	af3_dpa_params p = block(B, head, N, K, dtype_code(y), hint);
	const auto* base = static_cast<const uint8_t*>(y.const_data_ptr());
	p.k = base, p.v = base + K * esz, p.q = base + 2 * K * esz, p.gate = base + 3 * K * esz, p.out = out.data_ptr();
	const int64_t st[3] = {N * 4 * C, 4 * K, 4 * C}, so[3] = {N * C, K, C};
	for(int i = 0; i < 3; i++) p.q_stride[i] = p.k_stride[i] = p.v_stride[i] = p.gate_stride[i] = st[i], p.out_stride[i] = so[i];
	p.bias_dtype = p.io_dtype;
	if(bias) put_bias(p, *bias);
	p.key_mask = m.ptr, p.key_mask_stride_b = m.stride;
	return forward(p, exact, dev);
}

// rows of x [.., C] times the fused projection weight [4C, C], plus the row: this library's kernel where it suits, a library GEMM otherwise
Tensor project(const Tensor& x, int64_t M, const Tensor& weight, const Tensor* row, int dev, int& rc) {
	const int64_t K = weight.size(1), N = weight.size(0);
	rc = AF3_OK;
	if(x.scalar_type() == at::kBFloat16 && weight.is_contiguous() && af3_project_suits(M, N, K)) {
		const Tensor rows = reinterpret_cast<uintptr_t>(x.const_data_ptr()) % 16 == 0 ? x : x.clone();
		Tensor       y    = new_tensor({M, N}, at::kBFloat16, dev);
		rc = af3_project(rows.const_data_ptr(), weight.const_data_ptr(), row ? row->const_data_ptr() : nullptr, y.data_ptr(), M, N, K, 0, current_stream(dev));
		return y;
	}
	return at::linear(x.dim() == 2 ? x : x.reshape({M, K}), weight, row ? *row : Tensor());
}

// self_attention(x [N, C] or [S, N, C], mask, bias, wq, wk, wv, wg, q_bias, head, kernel hint, exact bias)
PyObject* py_self_attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
	HANDLE_TH_ERRORS
	if(n != 11) return none();
	const Tensor *x = tensor_of(a[0]), *bias;
	const int64_t head = PyLong_AsLongLong(a[8]);
	const int     dev = device_of(x);
	if(dev < 0 || (x->dim() != 2 && x->dim() != 3) || !x->is_contiguous() || x->numel() == 0 || head < 1) return none();
	const int     code = dtype_code(*x);
	const int64_t C = x->size(-1), N = x->size(-2), S = x->dim() == 3 ? x->size(0) : 1;
	key_mask      m;
	if(code < 0 || C % head != 0 || !mask_of(a[1], S, N, dev, m) || !bias_of(a[2], head, N, dev, bias) || (bias && bias->scalar_type() != x->scalar_type())) return none();
	// (both were derived from checked weights; a call with other ones finds nothing here)
	const Tensor* w  = derived_of(tag_of(FUSED_WEIGHT, head, code), a + 3, 4);
	const Tensor* qb = derived_of(tag_of(Q_BIAS_ROW, head, code), a + 7, 1);
	if(!w || !qb || w->size(1) != C || qb->size(0) != 4 * C || !on_device(*w, dev) || !on_device(*qb, dev)) return none();
	const Tensor weight = *w, row = *qb;
	const int64_t hint = PyLong_AsLongLong(a[9]);
	const bool    exact = a[10] == Py_True;
	Tensor out;
	int    rc;
	{
		without_gil g;
		const Tensor y = project(*x, S * N, weight, &row, dev, rc);
		if(rc != AF3_OK) {
		} else if(y.scalar_type() != x->scalar_type() || !y.is_contiguous()) rc = 1;  // (autocast)
		else {
			out = new_tensor(x->sizes(), x->scalar_type(), dev);
			rc  = attend(y, S, N, head, m, bias, out, hint, exact, dev);
		}
	}
	return rc == 1 ? none() : answer(rc, std::move(out));
	END_HANDLE_TH_ERRORS
}

// ---- grid attention ---------------------------------------------------------------------------------------------------
// The one-kernel form into `out` [B, N, C]: 0, an af3_status, or 1 where the library does not take the shape.
int grid_kernel(const Tensor& pair, const key_mask& m, const Tensor* bias, const Tensor* const (&ws)[4], int64_t head, Tensor& out, int dev) {
	af3_grid_attention_params g{};
	const int64_t B = pair.size(0), N = pair.size(1), C = pair.size(2);
	g.pair = pair.const_data_ptr(), g.pair_stride[0] = pair.stride(0), g.pair_stride[1] = pair.stride(1);
	g.q_proj = ws[0]->const_data_ptr(), g.k_proj = ws[1]->const_data_ptr(), g.v_proj = ws[2]->const_data_ptr(), g.gating_query = ws[3]->const_data_ptr();
	g.B = B, g.N = N, g.C = C, g.head = head, g.dtype = dtype_code(pair);
	if(bias) g.bias = bias->const_data_ptr(), g.bias_stride[0] = bias->stride(0), g.bias_stride[1] = bias->stride(1), g.bias_dtype = dtype_code(*bias);
	g.key_mask = m.ptr, g.key_mask_stride_b = m.stride;
	out   = new_tensor({B, N, C}, pair.scalar_type(), dev);
	g.out = out.data_ptr(), g.out_stride[0] = N * C, g.out_stride[1] = C;
	if(!af3_grid_attention_supported(&g)) return 1;
	at::DataPtr   mem;
	const int64_t bytes = af3_grid_attention_workspace_bytes(&g);
	if(bytes > 0) mem = new_scratch(bytes), g.workspace = mem.get(), g.workspace_bytes = bytes;
	return af3_grid_attention_forward(&g, current_stream(dev));
}
bool grid_weights(PyObject* const* o, const Tensor& pair, int64_t head, int dev, const Tensor* (&ws)[4]) {
	const int64_t C = pair.size(2);
	for(int i = 0; i < 4; i++) {
		ws[i] = tensor_of(o[i]);
		if(!ws[i] || !on_device(*ws[i], dev) || ws[i]->scalar_type() != pair.scalar_type() || ws[i]->dim() != 2 || ws[i]->size(0) != C || ws[i]->size(1) != C || !ws[i]->is_contiguous()) return false;
	}
	return head > 0 && C % head == 0;
}

// grid_kernel(pair, mask, bias, wq, wk, wv, wg, head)
PyObject* py_grid_kernel(PyObject*, PyObject* const* a, Py_ssize_t n) {
	HANDLE_TH_ERRORS
	if(n != 8) return none();
	const Tensor *pair = tensor_of(a[0]), *bias, *ws[4];
	const int64_t head = PyLong_AsLongLong(a[7]);
	const int     dev = device_of(pair);
	key_mask      m;
	if(dev < 0 || pair->dim() != 3 || pair->numel() == 0 || dtype_code(*pair) < 0 || !inner_1(*pair)) return none();
	if(!grid_weights(a + 3, *pair, head, dev, ws) || !mask_of(a[1], pair->size(0), pair->size(1), dev, m) || !bias_of(a[2], head, pair->size(1), dev, bias) || (bias && dtype_code(*bias) < 0)) return none();
	Tensor out;
	int    rc;
	{
		without_gil g;
		rc = grid_kernel(*pair, m, bias, ws, head, out, dev);
	}
	return rc == 1 ? none() : answer(rc, std::move(out));
	END_HANDLE_TH_ERRORS
}

// shapes for which af3_linear beats the library GEMM (measured): bfloat16, 64 or 128 input channels, at most 128 outputs
bool narrow(const Tensor& rows, int64_t n_out) {
	return rows.scalar_type() == at::kBFloat16 && (rows.size(-1) == 64 || rows.size(-1) == 128) && n_out % 32 == 0 && n_out <= 128 && n_out > 0 && rows.numel() > 0 && rows.is_contiguous() &&
		   reinterpret_cast<uintptr_t>(rows.const_data_ptr()) % 16 == 0;
}
int narrow_linear(const Tensor& rows, const Tensor& weight, Tensor& out, int dev) {
	const int64_t K = rows.size(-1), M = rows.numel() / K, N = weight.size(0);
	auto sizes = rows.sizes().vec();
	sizes.back() = N;
	out = new_tensor(sizes, rows.scalar_type(), dev);
	return af3_linear(rows.const_data_ptr(), weight.const_data_ptr(), out.data_ptr(), M, K, N, AF3_BF16, current_stream(dev));
}

// out_projection(rows [.., C], out_proj [C, C] = weight^T)
PyObject* py_out_projection(PyObject*, PyObject* const* a, Py_ssize_t n) {
	HANDLE_TH_ERRORS
	if(n != 2) return none();
	const Tensor *rows = tensor_of(a[0]), *wt = derived_of(OUT_PROJ_T, a + 1, 1);
	const int     dev = device_of(rows);
	if(dev < 0 || !wt || !on_device(*wt, dev) || wt->scalar_type() != rows->scalar_type() || wt->size(1) != rows->size(-1) || !narrow(*rows, wt->size(0))) return none();
	const Tensor weight = *wt;
	Tensor       out;
	int          rc;
	{
		without_gil g;
		rc = narrow_linear(*rows, weight, out, dev);
	}
	return answer(rc, std::move(out));
	END_HANDLE_TH_ERRORS
}

// linear(x [.., K], weight [N, K])
PyObject* py_linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
	HANDLE_TH_ERRORS
	if(n != 2) return none();
	const Tensor *x = tensor_of(a[0]), *w = tensor_of(a[1]);
	const int     dev = device_of(x);
	if(dev < 0 || !w || x->dim() < 1 || w->dim() != 2 || !on_device(*w, dev) || w->scalar_type() != x->scalar_type() || w->size(1) != x->size(-1) || !w->is_contiguous() ||
	   !narrow(*x, w->size(0)))
		return none();
	Tensor out;
	int    rc;
	{
		without_gil g;
		rc = narrow_linear(*x, *w, out, dev);
	}
	return answer(rc, std::move(out));
	END_HANDLE_TH_ERRORS
}

// ---- LayerNorm + pair bias ----------------------------------------------------------------------------------------------
struct ln_args {
	const Tensor *pair, *gamma, *beta, *proj;
	float         eps;
};
bool ln_of(PyObject* const* a, int& dev, ln_args& r) {   // a: pair, ln_weight, ln_bias, eps, proj_weight
	r = {tensor_of(a[0]), tensor_of(a[1]), tensor_of(a[2]), tensor_of(a[4]), 0.f};
	dev = device_of(r.pair);
	if(dev < 0 || !r.gamma || !r.beta || !r.proj || r.pair->dim() != 3 || r.proj->dim() != 2 || r.pair->numel() == 0 || dtype_code(*r.pair) < 0 || !inner_1(*r.pair)) return false;
	const int64_t C = r.pair->size(2), head = r.proj->size(0);
	if(r.proj->size(1) != C || r.gamma->numel() != C || r.beta->numel() != C || C > 2048 || head < 1 || head > 64 || (2 + head) * C * 4 > 160 * 1024 - 1024) return false;
	for(const Tensor* t : {r.pair, r.gamma, r.beta, r.proj})
		if(!on_device(*t, dev) || t->scalar_type() != r.pair->scalar_type() || (t != r.pair && !t->is_contiguous())) return false;
	const double eps = PyFloat_AsDouble(a[3]);
	if(eps == -1.0 && PyErr_Occurred()) {
		PyErr_Clear();
		return false;
	}
	r.eps = (float)eps;
	return true;
}
int ln_pair_bias(const ln_args& r, Tensor& normed, Tensor& bias, int dev) {
	const int64_t n_i = r.pair->size(0), n_j = r.pair->size(1), C = r.pair->size(2), head = r.proj->size(0);
	normed = new_tensor({n_i, n_j, C}, r.pair->scalar_type(), dev);
	bias   = new_tensor({head, n_i, n_j}, r.pair->scalar_type(), dev);
	const int64_t ps[2] = {r.pair->stride(0), r.pair->stride(1)}, bs[2] = {n_i * n_j, n_j};
	return af3_layernorm_pair_bias(r.pair->const_data_ptr(), ps, r.gamma->const_data_ptr(), r.beta->const_data_ptr(), r.eps, r.proj->const_data_ptr(), normed.data_ptr(), bias.data_ptr(), bs, n_i, n_j, C,
								   head, dtype_code(*r.pair), current_stream(dev));
}

// layernorm_pair_bias(pair, ln_weight, ln_bias, eps, proj_weight)
PyObject* py_layernorm_pair_bias(PyObject*, PyObject* const* a, Py_ssize_t n) {
	HANDLE_TH_ERRORS
	ln_args   r;
	int       dev = -1;
	if(n != 5 || !ln_of(a, dev, r)) return none();
	Tensor normed, bias;
	int    rc;
	{
		without_gil g;
		rc = ln_pair_bias(r, normed, bias, dev);
	}
	if(rc != AF3_OK) return PyLong_FromLong(rc);
	PyObject *x = wrap(std::move(normed)), *y = x ? wrap(std::move(bias)) : nullptr;
	if(!y) {
		Py_XDECREF(x);
		return nullptr;
	}
	PyObject* both = PyTuple_Pack(2, x, y);
	Py_DECREF(x), Py_DECREF(y);
	return both;
	END_HANDLE_TH_ERRORS
}

// LayerNorm, pair bias and projections in one kernel (128 channels in 4 heads, bfloat16), then the attention launch on q, k, v and the
// gate [B, 4, N, 32] and the output projection.
bool grid_projected_ok(const ln_args& r, const Tensor* const (&ws)[4]) {
	const auto odd = [](const Tensor* t, int to) { return reinterpret_cast<uintptr_t>(t->const_data_ptr()) % to != 0; };
	return r.pair->size(2) == 128 && r.proj->size(0) == 4 && r.pair->scalar_type() == at::kBFloat16 && r.pair->stride(0) % 8 == 0 && r.pair->stride(1) % 8 == 0 && !odd(r.pair, 16) &&
		   !odd(r.gamma, 16) && !odd(r.beta, 16) && !odd(r.proj, 16) && !odd(ws[0], 4) && !odd(ws[1], 4) && !odd(ws[2], 4) && !odd(ws[3], 4);
}
// Where the memory for q, k, v and the gate of the whole call is not there, they go in slabs of batch rows of at most 256 MB, after a
// pass over the whole pair tensor for the bias, which every slab needs (N = 640 414 -> 488 us, 1024 1316 -> 1450).
constexpr int64_t GRID_SLAB_BYTES = (int64_t)256 << 20;
int grid_projected_rows(const ln_args& r, const key_mask& m, const Tensor* const (&ws)[4], bool turned, int64_t hint, bool exact, const Tensor& out_weight, int64_t rows, Tensor& out, int dev) {
	const int64_t n_i = r.pair->size(0), n_j = r.pair->size(1), B = turned ? n_j : n_i, N = turned ? n_i : n_j, each = rows * N * 128;
	const bool    whole = rows == B;
	at::DataPtr   mem = new_scratch((4 * each + 4 * n_i * n_j) * 2), rows_out = new_scratch(each * 2);
	auto* const     q = static_cast<uint16_t*>(mem.get());
	uint16_t *const k = q + each, *const v = k + each, *const gate = v + each, *const bias = gate + each;
	if(!whole) out = new_tensor({B, N, 128}, at::kBFloat16, dev);
	const int64_t ps[2] = {r.pair->stride(0), r.pair->stride(1)};
	const auto project_rows = [&](int64_t b0, int64_t count, float q_scale, bool with_rows, bool with_bias) {
		const auto* x = static_cast<const uint16_t*>(r.pair->const_data_ptr()) + b0 * ps[turned ? 1 : 0];
		return af3_grid_project(x, ps, r.gamma->const_data_ptr(), r.beta->const_data_ptr(), r.eps, r.proj->const_data_ptr(), ws[0]->const_data_ptr(), ws[1]->const_data_ptr(), ws[2]->const_data_ptr(),
								ws[3]->const_data_ptr(), turned ? N : count, turned ? count : N, turned, q_scale, with_rows ? q : nullptr, with_rows ? k : nullptr, with_rows ? v : nullptr,
								with_rows ? gate : nullptr, with_bias ? bias : nullptr, current_stream(dev));
	};
	int rc = whole ? AF3_OK : project_rows(0, B, 1.f, false, true);
	for(int64_t b0 = 0; b0 < B && rc == AF3_OK; b0 += rows) {
		const int64_t  count = B - b0 < rows ? B - b0 : rows;
		af3_dpa_params p = block(count, 4, N, 32, AF3_BF16, hint);
		p.q = q, p.k = k, p.v = v, p.gate = gate, p.out = rows_out.get(), p.bias = bias;
		const int64_t st[3] = {4 * N * 32, N * 32, 32}, so[3] = {N * 128, 32, 128};
		for(int i = 0; i < 3; i++) p.q_stride[i] = p.k_stride[i] = p.v_stride[i] = p.gate_stride[i] = st[i], p.out_stride[i] = so[i];
		p.bias_stride[0] = n_i * n_j, p.bias_stride[1] = n_j, p.bias_dtype = AF3_BF16;
		p.key_mask = m.ptr ? m.ptr + b0 * m.stride : nullptr, p.key_mask_stride_b = m.stride;
		{
			const at::DataPtr work = workspace_for(p, exact);
			// The whole scale of the logits goes into q where it is projected, in fp32: one rounding.  What is left for the attention
			// kernel is 1 in its own units (a product with it gives the same bits back).
			const float log2e = 1.4426950408889634f, q_scale = af3_dpa_log2_domain(&p) ? p.softmax_scale * log2e : p.softmax_scale;
			p.softmax_scale = q_scale == p.softmax_scale ? 1.f : 1.f / log2e;
			rc = project_rows(b0, count, q_scale, true, whole);
			if(rc == AF3_OK) rc = af3_dpa_forward(&p, current_stream(dev));
		}
		if(rc != AF3_OK) break;
		if(whole) mem = at::DataPtr(), out = new_tensor({B, N, 128}, at::kBFloat16, dev);   // (the result may take the place of what is no longer needed)
		rc = af3_linear(rows_out.get(), out_weight.const_data_ptr(), static_cast<uint16_t*>(out.data_ptr()) + b0 * N * 128, count * N, 128, out_weight.size(0), AF3_BF16, current_stream(dev));
	}
	return rc;
}
int grid_projected(const ln_args& r, const key_mask& m, const Tensor* const (&ws)[4], bool turned, int64_t hint, bool exact, const Tensor& out_weight, Tensor& out, int dev) {
	const int64_t B = r.pair->size(turned ? 1 : 0), N = r.pair->size(turned ? 0 : 1), fit = GRID_SLAB_BYTES / (N * 1024) / 32 * 32;
	const int64_t rows = fit < 32 ? 32 : fit;
	if(rows < B) {
		try {
			return grid_projected_rows(r, m, ws, turned, hint, exact, out_weight, B, out, dev);
		} catch(const c10::OutOfMemoryError&) {
		}
	}
	return grid_projected_rows(r, m, ws, turned, hint, exact, out_weight, rows < B ? rows : B, out, dev);
}

// grid_block(pair, ln_weight, ln_bias, eps, proj_weight, mask, wq, wk, wv, wg, out_proj, head, transpose, least (batch row, head) pairs of
// the one-kernel form, kernel hint, exact bias): the whole block of GridSelfAttentionCpp.forward
PyObject* py_grid_block(PyObject*, PyObject* const* a, Py_ssize_t n) {
	HANDLE_TH_ERRORS
	ln_args       r;
	int           dev = -1;
	const Tensor* ws[4];
	key_mask      m;
	if(n != 16 || !ln_of(a, dev, r)) return none();
	const int64_t head = PyLong_AsLongLong(a[11]), least = PyLong_AsLongLong(a[13]), hint = PyLong_AsLongLong(a[14]);
	const bool    turned = a[12] == Py_True, exact = a[15] == Py_True;
	const int64_t B = r.pair->size(turned ? 1 : 0), N = r.pair->size(turned ? 0 : 1), C = r.pair->size(2);
	// (the closing projection is af3_linear: 64 or 128 channels in bfloat16)
	if(B != N || r.pair->scalar_type() != at::kBFloat16 || (C != 64 && C != 128) || r.proj->size(0) != head || !grid_weights(a + 6, *r.pair, head, dev, ws) || !mask_of(a[5], B, N, dev, m)) return none();
	const Tensor* wt = derived_of(OUT_PROJ_T, a + 10, 1);
	const Tensor* wf = derived_of(tag_of(FUSED_WEIGHT, head, dtype_code(*r.pair)), a + 6, 4);  // (three launches only)
	if(!wt || !on_device(*wt, dev) || wt->scalar_type() != r.pair->scalar_type() || wt->size(0) != C || wt->size(1) != C) return none();
	const Tensor out_weight = *wt, fused = wf ? *wf : Tensor();
	Tensor out;
	int    rc;
	{
		without_gil g;
		if(grid_projected_ok(r, ws)) rc = grid_projected(r, m, ws, turned, hint, exact, out_weight, out, dev);
		else {
			Tensor normed, bias, gated;
			rc = ln_pair_bias(r, normed, bias, dev);
			if(rc == AF3_OK) {
				const Tensor rows = turned ? normed.transpose(0, 1) : normed;
				rc = B * head >= least && !exact ? grid_kernel(rows, m, &bias, ws, head, gated, dev) : 1;
				if(rc == 1 && fused.defined()) {
					const Tensor y = at::linear(rows.reshape({B * N, C}), fused);
					if(y.scalar_type() == normed.scalar_type() && y.is_contiguous()) {
						gated = new_tensor({B, N, C}, y.scalar_type(), dev);
						rc    = attend(y, B, N, head, m, &bias, gated, hint, exact, dev);
					}
				}
			}
			if(rc == AF3_OK) rc = narrow_linear(gated, out_weight, out, dev);
		}
		if(turned && rc == AF3_OK) out = out.transpose(0, 1);
	}
	return rc == 1 ? none() : answer(rc, std::move(out));
	END_HANDLE_TH_ERRORS
}

// ---- gated linear unit --------------------------------------------------------------------------------------------------
// gated_linear_unit(x [.., K], weight [K, 2N], tag of its transposed form)
PyObject* py_gated_linear_unit(PyObject*, PyObject* const* a, Py_ssize_t n) {
	HANDLE_TH_ERRORS
	if(n != 3) return none();
	const Tensor *x = tensor_of(a[0]), *wt = derived_of(PyLong_AsLongLong(a[2]), a + 1, 1);
	const int     dev = device_of(x);
	if(dev < 0 || !wt || x->dim() < 1 || x->numel() == 0 || x->scalar_type() != at::kBFloat16 || wt->scalar_type() != at::kBFloat16 || !on_device(*wt, dev) || !x->is_contiguous() ||
	   reinterpret_cast<uintptr_t>(x->const_data_ptr()) % 16 || x->size(-1) != wt->size(1))
		return none();
	const Tensor weight = *wt;
	Tensor       out;
	int          rc;
	{
		without_gil g;
		const int64_t K = weight.size(1), N = weight.size(0) / 2;
		auto sizes = x->sizes().vec();
		sizes.back() = N;
		out = new_tensor(sizes, at::kBFloat16, dev);
		rc  = af3_gated_linear_unit(x->const_data_ptr(), weight.const_data_ptr(), out.data_ptr(), x->numel() / K, K, N, AF3_BF16, current_stream(dev));
	}
	return answer(rc, std::move(out));
	END_HANDLE_TH_ERRORS
}

#define AF3_FN(name, doc) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(py_##name)), METH_FASTCALL, doc}
PyMethodDef methods[] = {
	AF3_FN(attention, "attention(q, k, v, mask, bias, kernel_hint, exact_bias)"),
	AF3_FN(attention_fp8, "attention_fp8(q, k, v, mask, bias, compensated)"),
	AF3_FN(self_attention, "self_attention(x, mask, bias, wq, wk, wv, wg, q_bias, head, kernel_hint, exact_bias)"),
	AF3_FN(grid_kernel, "grid_kernel(pair, mask, bias, wq, wk, wv, wg, head)"),
	AF3_FN(grid_block, "grid_block(pair, ln_weight, ln_bias, eps, proj_weight, mask, wq, wk, wv, wg, out_proj, head, transpose, least_groups, kernel_hint, exact_bias)"),
	AF3_FN(out_projection, "out_projection(rows, out_proj)"),
	AF3_FN(linear, "linear(x, weight)"),
	AF3_FN(layernorm_pair_bias, "layernorm_pair_bias(pair, ln_weight, ln_bias, eps, proj_weight)"),
	AF3_FN(gated_linear_unit, "gated_linear_unit(x, weight, tag)"),
	AF3_FN(remember, "remember(tag, value, source...): a matrix derived from weights"),
	AF3_FN(recalls, "recalls(tag, source...): whether one is remembered for these"),
	AF3_FN(forget_source, "forget_source(address): drops what was derived from this tensor"),
	{"forget", py_forget, METH_NOARGS, "forget(): drops every remembered matrix"},
	{nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", "native host side of the entry points", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) {
	PyObject* m = PyModule_Create(&module);
	if(!m) return nullptr;
	for(auto& [name, value] : {std::pair<const char*, long>{"FUSED_WEIGHT", FUSED_WEIGHT}, {"Q_BIAS_ROW", Q_BIAS_ROW}, {"OUT_PROJ_T", OUT_PROJ_T}, {"GLU_T", GLU_T}}) PyModule_AddIntConstant(m, name, value);
	return m;
}
