// The wrappers' calls on plain arguments, in native code.
//
// A call of the Python wrappers spends 12 to 25 us of host time on argument
// checks, allocations and a ctypes call of some twenty arguments, which is what
// a small kernel's call costs in all (4 rows of 1000 scores: 14.5 us for a 10 us
// kernel); the wrappers that read lengths from the device spend 65 to 110 us,
// most of it in small tensor operations around the copies.  The functions here
// do the same for arguments in their plain form -- exact torch.Tensor objects
// on one HIP device, contiguous, lengths and tables int32 on that device -- and
// return None for everything else: other types, layouts and devices, empty
// calls, and every argument the wrapper would refuse.  The wrapper then runs its
// own checks and raises or converts as it always did.  Outputs come from ATen's
// caching allocator and work goes to the current stream, as there.
//
// The C entry points are those of the library the package has loaded: bind()
// receives their addresses.  A non-zero return code is handed back as an int,
// which the wrapper turns into its error.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <vector>

#include "../../include/dsa_mi355x.h"

namespace {

struct Entries {
  decltype(&dsa_topk_select_workspace_size) topk_ws;
  decltype(&dsa_topk_select_ws) topk;
  decltype(&dsa_act_quant) act_quant;
  decltype(&dsa_sparse_mla_workspace_size) mla_ws;
  decltype(&dsa_sparse_mla_fwd) mla;
  decltype(&dsa_sparse_mla_decode_parts_applies) parts_applies;
  decltype(&dsa_sparse_mla_decode_parts) parts;
  decltype(&dsa_sparse_attention_fwd) attention;
  decltype(&dsa_lightning_indexer_workspace_size) idx_ws;
  decltype(&dsa_lightning_indexer) idx;
  decltype(&dsa_lightning_indexer_fused_workspace_size) idxf_ws;
  decltype(&dsa_lightning_indexer_fused) idxf;
  decltype(&dsa_lightning_indexer_tnd_workspace_size) tnd_ws;
  decltype(&dsa_lightning_indexer_tnd) tnd;
  decltype(&dsa_lightning_indexer_tnd_fused_workspace_size) tndf_ws;
  decltype(&dsa_lightning_indexer_tnd_fused) tndf;
  decltype(&dsa_sparse_flash_mla_workspace_size) v4_ws;
  decltype(&dsa_sparse_flash_mla) v4;
} E;
bool bound = false;

constexpr int64_t kAlign = 256;
int64_t aligned(int64_t n) { return (n + kAlign - 1) / kAlign * kAlign; }

// An argument: an exact torch.Tensor, None, or neither (`other`).
struct Arg {
  const at::Tensor* t = nullptr;
  bool other = false;
  explicit Arg(PyObject* o) {
    if (o == Py_None) return;
    if (THPVariable_CheckExact(o)) t = &THPVariable_Unpack(o);
    else other = true;
  }
  explicit operator bool() const { return t != nullptr; }
  template <class T>
  const T* ptr() const { return t ? static_cast<const T*>(t->data_ptr()) : nullptr; }
};

// An exact int that fits 64 bits.
bool int_of(PyObject* o, int64_t& v) {
  if (!PyLong_CheckExact(o)) return false;
  int overflow = 0;
  v = PyLong_AsLongLongAndOverflow(o, &overflow);
  return overflow == 0;
}

// Contiguous, on `dev`, of dtype `st`.
bool plain(const at::Tensor& t, c10::Device dev, at::ScalarType st) {
  return t.device() == dev && t.scalar_type() == st && t.is_contiguous();
}
// None, or plain int32 of n elements.
bool lens_ok(const Arg& a, c10::Device dev, int64_t n) {
  return !a.other && (!a || (plain(*a.t, dev, at::kInt) && a.t->numel() == n));
}

at::Tensor make(at::IntArrayRef sizes, at::ScalarType st, c10::Device dev) {
  return at::empty(sizes, at::TensorOptions().dtype(st).device(dev));
}
void* stream(c10::Device dev) { return c10::hip::getCurrentHIPStream(dev.index()).stream(); }
int kind16(at::ScalarType st) { return st == at::kBFloat16 ? DSA_KIND_BF16 : st == at::kHalf ? DSA_KIND_FP16 : -1; }
int kind_idx(at::ScalarType st) { return st == at::kFloat8_e4m3fn ? DSA_KIND_FP8_E4M3 : kind16(st); }

PyObject* wrap(at::Tensor t) { return THPVariable_Wrap(std::move(t)); }
PyObject* pair(at::Tensor a, at::Tensor b) {
  PyObject* r = PyTuple_New(2);
  if (!r) return nullptr;
  PyTuple_SET_ITEM(r, 0, wrap(std::move(a)));
  PyTuple_SET_ITEM(r, 1, wrap(std::move(b)));
  return r;
}
#define DSA_RC(rc) \
  if (const int rc_ = (rc); rc_ != 0) return PyLong_FromLong(rc_)
#define DSA_PLAIN(cond) \
  if (!(cond)) Py_RETURN_NONE

// Other Python threads run while this one allocates, launches or waits for the device.
struct NoGil {
  PyThreadState* state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};

// Device int32 values on the host.
std::vector<int32_t> host_values(const at::Tensor& t) {
  const NoGil unlocked;
  const at::Tensor h = t.cpu();
  const int32_t* p = h.data_ptr<int32_t>();
  return std::vector<int32_t>(p, p + h.numel());
}

// (x, top_k, sorted, row_len, return_values)
PyObject* topk(PyObject*, PyObject* const* v, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  int64_t k = 0;
  DSA_PLAIN(bound && n == 5 && THPVariable_CheckExact(v[0]) && int_of(v[1], k) && PyBool_Check(v[2]) &&
            PyBool_Check(v[4]));
  const at::Tensor& x = THPVariable_Unpack(v[0]);
  const Arg len(v[3]);
  DSA_PLAIN(x.is_cuda() && x.dim() >= 1 && x.numel() > 0 && plain(x, x.device(), at::kFloat) && k >= 1 && k <= 8192);
  const c10::Device dev = x.device();
  const int64_t cols = x.size(-1), rows = x.numel() / cols;
  DSA_PLAIN(lens_ok(len, dev, rows));
  std::vector<int64_t> sizes(x.sizes().begin(), x.sizes().end());
  sizes.back() = k;
  const bool sorted = v[2] == Py_True, values = v[4] == Py_True;
  at::Tensor idx, val, ws;
  int rc;
  {
    const NoGil unlocked;
    idx = make(sizes, at::kInt, dev);
    if (values) val = make(sizes, at::kFloat, dev);
    const size_t bytes = E.topk_ws(rows, cols, k);
    if (bytes) ws = make({(int64_t)bytes}, at::kByte, dev);
    rc = E.topk(x.data_ptr<float>(), cols, rows, cols, k, len.ptr<int32_t>(), sorted, idx.data_ptr<int32_t>(),
                values ? val.data_ptr<float>() : nullptr, bytes ? ws.data_ptr() : nullptr, bytes, stream(dev));
  }
  DSA_RC(rc);
  return values ? pair(std::move(idx), std::move(val)) : wrap(std::move(idx));
  END_HANDLE_TH_ERRORS
}

// (x, round_scale, out kind)
PyObject* act_quant(PyObject*, PyObject* const* v, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  int64_t out = 0;
  DSA_PLAIN(bound && n == 3 && THPVariable_CheckExact(v[0]) && PyBool_Check(v[1]) && int_of(v[2], out));
  const at::Tensor& x = THPVariable_Unpack(v[0]);
  const int in = x.scalar_type() == at::kFloat ? DSA_KIND_FP32 : kind16(x.scalar_type());
  DSA_PLAIN(x.is_cuda() && in >= 0 && (x.dim() == 2 || x.dim() == 3) && x.is_contiguous() && x.numel() > 0);
  DSA_PLAIN(out == DSA_KIND_INT8 || out == DSA_KIND_FP8_E4M3);
  const int64_t cols = x.size(-1), rows = x.numel() / cols;
  std::vector<int64_t> sizes(x.sizes().begin(), x.sizes().end());
  const bool round = v[1] == Py_True;
  at::Tensor y, s;
  int rc;
  {
    const NoGil unlocked;
    y = make(sizes, out == DSA_KIND_INT8 ? at::kChar : at::kFloat8_e4m3fn, x.device());
    sizes.back() = 1;
    s = make(sizes, at::kFloat, x.device());
    rc = E.act_quant(in, x.data_ptr(), rows, cols, (int)out, y.data_ptr(), s.data_ptr<float>(), round,
                     stream(x.device()));
  }
  DSA_RC(rc);
  return pair(std::move(y), std::move(s));
  END_HANDLE_TH_ERRORS
}

// Block table of B rows, or none.
bool table_ok(const Arg& bt, c10::Device dev, int64_t B) {
  return !bt.other && (!bt || (bt.t->dim() == 2 && bt.t->size(0) == B && bt.t->size(1) > 0 &&
                               plain(*bt.t, dev, at::kInt)));
}

// (q, kv, indices, sm_scale, block_table, q lengths, kv lengths, is_causal): one KV head
PyObject* sparse_mla(PyObject*, PyObject* const* v, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  DSA_PLAIN(bound && n == 8 && THPVariable_CheckExact(v[0]) && THPVariable_CheckExact(v[1]) &&
            THPVariable_CheckExact(v[2]) && PyFloat_CheckExact(v[3]) && PyBool_Check(v[7]));
  const at::Tensor &q = THPVariable_Unpack(v[0]), &kv = THPVariable_Unpack(v[1]), &ix = THPVariable_Unpack(v[2]);
  const Arg bt(v[4]), ql(v[5]), kl(v[6]);
  DSA_PLAIN(q.is_cuda() && q.dim() == 4 && kv.dim() == 4 && ix.dim() >= 3 && ix.dim() <= 4);
  const c10::Device dev = q.device();
  const int kind = kind16(q.scalar_type());
  DSA_PLAIN(kind >= 0 && plain(q, dev, q.scalar_type()) && plain(kv, dev, q.scalar_type()) && plain(ix, dev, at::kInt));
  const int64_t B = q.size(0), S = q.size(1), H = q.size(2), topk = ix.size(-1);
  DSA_PLAIN(B > 0 && S > 0 && topk > 0 && q.size(3) == 576 && kv.size(3) == 576 && kv.size(2) == 1 && H >= 16 &&
            H % 16 == 0 && H <= 1024 && ix.size(0) == B && ix.size(1) == S && (ix.dim() == 3 || ix.size(2) == 1));
  DSA_PLAIN(table_ok(bt, dev, B) && lens_ok(ql, dev, B) && lens_ok(kl, dev, B) && (bt || kv.size(0) == B));
  const int64_t bs = bt ? kv.size(1) : 0, mb = bt ? bt.t->size(1) : 0, skv = bt ? bs * mb : kv.size(1);
  const float scale = (float)PyFloat_AS_DOUBLE(v[3]);
  const bool causal = v[7] == Py_True;
  at::Tensor out, lse, ws;
  int rc;
  {
    const NoGil unlocked;
    out = make({B, S, H, 512}, q.scalar_type(), dev);
    lse = make({B, S, H}, at::kFloat, dev);
    const size_t bytes = E.mla_ws(B, S, H, topk);
    if (bytes) ws = make({(int64_t)bytes}, at::kByte, dev);
    rc = E.mla(kind, q.data_ptr(), kv.data_ptr(), ix.data_ptr<int32_t>(), bt.ptr<int32_t>(), ql.ptr<int32_t>(),
               kl.ptr<int32_t>(), B, S, H, 576, 512, skv, bs, mb, topk, scale, causal, out.data_ptr(),
               lse.data_ptr<float>(), bytes ? ws.data_ptr() : nullptr, bytes, stream(dev));
  }
  DSA_RC(rc);
  return pair(std::move(out), std::move(lse));
  END_HANDLE_TH_ERRORS
}

// (q, kv, indices, sm_scale, q lengths, kv lengths, is_causal): 128-wide grouped heads
PyObject* sparse_gqa(PyObject*, PyObject* const* v, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  DSA_PLAIN(bound && n == 7 && THPVariable_CheckExact(v[0]) && THPVariable_CheckExact(v[1]) &&
            THPVariable_CheckExact(v[2]) && PyFloat_CheckExact(v[3]) && PyBool_Check(v[6]));
  const at::Tensor &q = THPVariable_Unpack(v[0]), &kv = THPVariable_Unpack(v[1]), &ix = THPVariable_Unpack(v[2]);
  const Arg ql(v[4]), kl(v[5]);
  DSA_PLAIN(q.is_cuda() && q.dim() == 4 && kv.dim() == 4 && ix.dim() == 4);
  const c10::Device dev = q.device();
  const int kind = kind16(q.scalar_type());
  DSA_PLAIN(kind >= 0 && plain(q, dev, q.scalar_type()) && plain(kv, dev, q.scalar_type()) && plain(ix, dev, at::kInt));
  const int64_t B = q.size(0), S = q.size(1), H = q.size(2), G = kv.size(2), topk = ix.size(3);
  DSA_PLAIN(B > 0 && S > 0 && H > 0 && topk > 0 && q.size(3) == 128 && kv.size(0) == B && kv.size(3) == 128 && G > 0 &&
            H % G == 0 && H / G <= 1024 && ix.size(0) == B && ix.size(1) == S && ix.size(2) == G);
  DSA_PLAIN(lens_ok(ql, dev, B) && lens_ok(kl, dev, B));
  const float scale = (float)PyFloat_AS_DOUBLE(v[3]);
  const bool causal = v[6] == Py_True;
  at::Tensor out, lse;
  int rc;
  {
    const NoGil unlocked;
    out = make({B, S, H, 128}, q.scalar_type(), dev);
    lse = make({B, S, H}, at::kFloat, dev);
    rc = E.attention(kind, q.data_ptr(), kv.data_ptr(), ix.data_ptr<int32_t>(), nullptr, ql.ptr<int32_t>(),
                     kl.ptr<int32_t>(), B, S, H, G, 128, 128, kv.size(1), 0, 0, topk, scale, causal, out.data_ptr(),
                     lse.data_ptr<float>(), nullptr, 0, stream(dev));
  }
  DSA_RC(rc);
  return pair(std::move(out), std::move(lse));
  END_HANDLE_TH_ERRORS
}

// (query, key, query_rope, key_rope, indices, scale, q lengths, kv lengths, is_causal, block_table)
PyObject* decode_parts(PyObject*, PyObject* const* v, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  DSA_PLAIN(bound && n == 10 && PyFloat_CheckExact(v[5]) && PyBool_Check(v[8]));
  for (int i = 0; i < 5; ++i) DSA_PLAIN(THPVariable_CheckExact(v[i]));
  const at::Tensor &q = THPVariable_Unpack(v[0]), &k = THPVariable_Unpack(v[1]), &qr = THPVariable_Unpack(v[2]),
                   &kr = THPVariable_Unpack(v[3]), &ix = THPVariable_Unpack(v[4]);
  const Arg ql(v[6]), kl(v[7]), bt(v[9]);
  DSA_PLAIN(q.is_cuda() && q.dim() == 3 && qr.dim() == 3 && k.dim() == 4 && kr.dim() == 4);
  const c10::Device dev = q.device();
  const at::ScalarType st = q.scalar_type();
  const int kind = kind16(st);
  DSA_PLAIN(kind >= 0 && plain(q, dev, st) && plain(k, dev, st) && plain(qr, dev, st) && plain(kr, dev, st) &&
            plain(ix, dev, at::kInt));
  const int64_t T = q.size(0), N = q.size(1);
  DSA_PLAIN(T > 0 && N > 0 && q.size(2) == 512 && qr.size(0) == T && qr.size(1) == N && qr.size(2) == 64 &&
            k.size(2) == 1 && k.size(3) == 512 && kr.size(0) == k.size(0) && kr.size(1) == k.size(1) &&
            kr.size(2) == 1 && kr.size(3) == 64 && ix.numel() % T == 0);
  for (const at::Tensor* t : {&q, &k, &qr, &kr})  // read by 16-byte loads; joining them would have moved them
    DSA_PLAIN((reinterpret_cast<uintptr_t>(t->data_ptr()) & 15) == 0);
  const int64_t topk = ix.numel() / T;
  DSA_PLAIN(E.parts_applies(1, T, N, topk) && table_ok(bt, dev, 1) && lens_ok(ql, dev, 1) && lens_ok(kl, dev, 1) &&
            (bt || k.size(0) == 1));
  const int64_t bs = bt ? k.size(1) : 0, mb = bt ? bt.t->size(1) : 0, skv = bt ? bs * mb : k.size(1);
  const float scale = (float)PyFloat_AS_DOUBLE(v[5]);
  const bool causal = v[8] == Py_True;
  at::Tensor out, ws;
  int rc;
  {
    const NoGil unlocked;
    const int64_t lse_bytes = aligned(T * N * 4);  // the LSE (not returned) and the workspace in one allocation
    const size_t bytes = E.mla_ws(1, T, N, topk);
    out = make({T, N, 512}, st, dev);
    ws = make({lse_bytes + (int64_t)bytes}, at::kByte, dev);
    uint8_t* p = ws.data_ptr<uint8_t>();
    rc = E.parts(kind, q.data_ptr(), qr.data_ptr(), k.data_ptr(), kr.data_ptr(), ix.data_ptr<int32_t>(),
                 bt.ptr<int32_t>(), ql.ptr<int32_t>(), kl.ptr<int32_t>(), 1, T, N, skv, bs, mb, topk, scale, causal,
                 out.data_ptr(), reinterpret_cast<float*>(p), p + lse_bytes, bytes, stream(dev));
  }
  DSA_RC(rc);
  return wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// The streamed top-k is the default past 32768 keys with at least 2048 rows (see the wrapper).
bool fuse(PyObject* o, int64_t rows, int64_t S2) { return o == Py_None ? S2 > 32768 && rows >= 2048 : o == Py_True; }

// Values in the wrapper's dtype: fp32 for fp8 queries, else the query's.
PyObject* idx_result(at::Tensor idx, at::Tensor val, bool values, at::ScalarType st, c10::Device dev) {
  const at::ScalarType vt = st == at::kFloat8_e4m3fn ? at::kFloat : st;
  if (!values) return pair(std::move(idx), make({0}, vt, dev));
  return pair(std::move(idx), vt == at::kFloat ? std::move(val) : val.to(vt));
}

// (query, key, weights, q lengths, k lengths, block_table, packed, sparse_count, sparse_mode, return_value,
//  key_scale, fuse_topk); packed: TND queries, lengths as prefix sums (keys too, unless paged)
PyObject* indexer(PyObject*, PyObject* const* v, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  int64_t K = 0, mode = 0;
  DSA_PLAIN(bound && n == 12 && THPVariable_CheckExact(v[0]) && THPVariable_CheckExact(v[1]) &&
            THPVariable_CheckExact(v[2]) && int_of(v[7], K) && int_of(v[8], mode) && PyBool_Check(v[9]));
  const at::Tensor &q = THPVariable_Unpack(v[0]), &k = THPVariable_Unpack(v[1]), &w = THPVariable_Unpack(v[2]);
  const Arg aq(v[3]), ak(v[4]), bt(v[5]), ks(v[10]);
  const bool packed = v[6] == Py_True, values = v[9] == Py_True;
  DSA_PLAIN(q.is_cuda() && q.dim() == (packed ? 3 : 4) && !aq.other && !ak.other && !ks.other);
  const c10::Device dev = q.device();
  const at::ScalarType st = q.scalar_type();
  const int kind = kind_idx(st);
  const int64_t H = q.size(-2), D = q.size(-1);
  DSA_PLAIN(kind >= 0 && plain(q, dev, st) && plain(k, dev, st) && plain(w, dev, at::kFloat) &&
            (D == 64 || D == 128) && H >= 1 && H <= 64 && (mode == 0 || mode == 3) && k.size(-1) == D &&
            (v[11] == Py_None || v[11] == Py_True || v[11] == Py_False) && (!bt || !values));
  DSA_PLAIN((K >= 1 && K <= 2048) || (K % 1024 == 0 && K > 0 && K <= 8192));
  if (packed) DSA_PLAIN(aq && plain(*aq.t, dev, at::kInt) && aq.t->dim() == 1 && aq.t->numel() > 0);
  const int64_t B = packed ? aq.t->numel() : q.size(0), T = packed ? q.size(0) : B * q.size(1);
  DSA_PLAIN(B > 0 && T > 0 && w.numel() == T * H && w.dim() >= (packed ? 2 : 3) && w.size(0) == q.size(0) &&
            w.size(1) == q.size(1) && (packed || w.size(2) == H) && table_ok(bt, dev, B) &&
            lens_ok(aq, dev, B) && lens_ok(ak, dev, B));
  // Keys: [B, S2, 1, D], [T_k, 1, D] packed, or a paged pool [blocks, block_size, 1, D].
  const int64_t key_rows = k.numel() / D;
  int64_t bs = 0, mb = 0;
  if (bt) {
    bs = k.dim() == 4 ? k.size(1) : 0;
    mb = bt.t->size(1);
    DSA_PLAIN(ak && k.dim() == 4 && k.size(2) == 1 && bs > 0 && bs % 16 == 0 && bs <= 1024);
  } else if (packed) {
    DSA_PLAIN(ak && k.dim() == 3 && k.size(1) == 1);
  } else {
    DSA_PLAIN(k.dim() == 4 && k.size(0) == B && k.size(2) == 1);
  }
  if (ks) DSA_PLAIN(plain(*ks.t, dev, at::kFloat) && ks.t->numel() == key_rows);
  // Lengths the launch needs, or the wrapper checks, on the host.
  int64_t S1 = packed ? 0 : q.size(1), S2 = packed || bt ? 0 : k.size(1), rows = T;
  if (packed) {
    const std::vector<int32_t> cu = host_values(*aq.t);
    for (int64_t b = 0; b < B; ++b) {
      const int64_t len = (int64_t)cu[b] - (b ? cu[b - 1] : 0);
      DSA_PLAIN(len >= 0);
      S1 = std::max(S1, len);
    }
    rows = cu[B - 1];
    DSA_PLAIN(rows <= T);
  } else if (aq) {
    for (const int32_t x : host_values(*aq.t)) DSA_PLAIN(x <= S1);
  }
  if (ak) {
    const std::vector<int32_t> kl = host_values(*ak.t);
    if (packed && !bt) {
      for (int64_t b = 0; b < B; ++b) {
        const int64_t len = (int64_t)kl[b] - (b ? kl[b - 1] : 0);
        DSA_PLAIN(len >= 0);
        S2 = std::max(S2, len);
      }
      DSA_PLAIN(kl[B - 1] <= key_rows);
    } else {
      const int64_t most = *std::max_element(kl.begin(), kl.end());
      DSA_PLAIN(most <= (bt ? mb * bs : S2));
      if (bt) S2 = most;
    }
  }
  DSA_PLAIN(S1 > 0 && S2 > 0 && rows > 0);
  const bool f = fuse(v[11], rows, S2);
  at::Tensor idx, val;
  int rc;
  {
    const NoGil unlocked;
    idx = packed ? make({rows, 1, K}, at::kInt, dev) : make({B, S1, 1, K}, at::kInt, dev);
    if (values) val = make(idx.sizes(), at::kFloat, dev);
    float* vp = values ? val.data_ptr<float>() : nullptr;
    const size_t bytes = packed ? (f ? E.tndf_ws(B, rows, S1, S2, K) : E.tnd_ws(rows, S2, K))
                                : (f ? E.idxf_ws : E.idx_ws)(B, S1, S2, K);
    at::Tensor ws = make({(int64_t)bytes}, at::kByte, dev);
    if (packed) {
      rc = (f ? E.tndf : E.tnd)(kind, q.data_ptr(), k.data_ptr(), ks.ptr<float>(), w.data_ptr<float>(), B, rows, S1, S2,
                                H, D, aq.ptr<int32_t>(), bt ? nullptr : ak.ptr<int32_t>(),
                                bt ? ak.ptr<int32_t>() : nullptr, bt.ptr<int32_t>(), bs, mb, (int)mode, K,
                                idx.data_ptr<int32_t>(), vp, ws.data_ptr(), bytes, stream(dev));
    } else {
      rc = (f ? E.idxf : E.idx)(kind, q.data_ptr(), k.data_ptr(), ks.ptr<float>(), w.data_ptr<float>(), B, S1, S2, H, D,
                                aq.ptr<int32_t>(), ak.ptr<int32_t>(), bt.ptr<int32_t>(), bs, mb, (int)mode, K,
                                idx.data_ptr<int32_t>(), vp, ws.data_ptr(), bytes, stream(dev));
    }
  }
  DSA_RC(rc);
  return idx_result(std::move(idx), std::move(val), values, st, dev);
  END_HANDLE_TH_ERRORS
}

// (q, ori_kv, cmp_kv, cmp_sparse_indices, ori_block_table, cmp_block_table, cu_seqlens_q, seqused_kv, sinks,
//  softmax_scale, cmp_ratio, ori_win_left, return lse): packed (TND) queries
PyObject* flash_mla(PyObject*, PyObject* const* v, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  int64_t win = 0, ratio = 4;
  DSA_PLAIN(bound && n == 13 && THPVariable_CheckExact(v[0]) && THPVariable_CheckExact(v[1]) &&
            PyFloat_CheckExact(v[9]) && (v[10] == Py_None || int_of(v[10], ratio)) && int_of(v[11], win) &&
            PyBool_Check(v[12]));
  const at::Tensor &q = THPVariable_Unpack(v[0]), &ori = THPVariable_Unpack(v[1]);
  const Arg cmp(v[2]), sel(v[3]), obt(v[4]), cbt(v[5]), cu(v[6]), kvl(v[7]), sinks(v[8]);
  DSA_PLAIN(q.is_cuda() && q.dim() == 3 && ori.dim() == 4 && cu && kvl && obt && !cmp.other && !sel.other &&
            !sinks.other && !cbt.other);
  const c10::Device dev = q.device();
  const at::ScalarType st = q.scalar_type();
  const int kind = kind16(st);
  const int64_t T = q.size(0), H = q.size(1), B = cu.t->numel() - 1;
  DSA_PLAIN(kind >= 0 && plain(q, dev, st) && plain(ori, dev, st) && T > 0 && H >= 16 && H % 16 == 0 && H <= 1024 &&
            q.size(2) == 512 && ori.size(2) == 1 && ori.size(3) == 512 && B >= 1 && cu.t->dim() == 1 &&
            plain(*cu.t, dev, at::kInt) && plain(*kvl.t, dev, at::kInt) && kvl.t->numel() == B &&
            table_ok(obt, dev, B));
  if (sinks) DSA_PLAIN(plain(*sinks.t, dev, at::kFloat) && sinks.t->numel() == H);
  int64_t K = 0, cmp_blocks = 0, cmp_bs = 0, cmp_tl = 0;
  if (cmp) {
    DSA_PLAIN(cmp.t->dim() == 4 && plain(*cmp.t, dev, st) && cmp.t->size(2) == 1 && cmp.t->size(3) == 512 && cbt &&
              table_ok(cbt, dev, B) && ratio >= 1 && (sel || v[10] != Py_None));
    cmp_blocks = cmp.t->size(0);
    cmp_bs = cmp.t->size(1);
    cmp_tl = cbt.t->size(1);
    if (sel) {
      DSA_PLAIN(sel.t->dim() == 3 && sel.t->size(0) == T && sel.t->size(1) == 1 && sel.t->size(2) > 0 &&
                plain(*sel.t, dev, at::kInt));
      K = sel.t->size(2);
    }
  }
  const std::vector<int32_t> starts = host_values(*cu.t);
  DSA_PLAIN(starts[0] >= 0 && starts[B] <= T);
  for (int64_t b = 0; b < B; ++b) DSA_PLAIN(starts[b + 1] >= starts[b]);
  int64_t max_cmp = 0;
  if (cmp && !sel) {
    const std::vector<int32_t> kl = host_values(*kvl.t);
    const int32_t most = *std::max_element(kl.begin(), kl.end());
    DSA_PLAIN(most >= 0);
    max_cmp = most / ratio;
  }
  const float scale = (float)PyFloat_AS_DOUBLE(v[9]);
  at::Tensor out, lse;
  int rc;
  {
    const NoGil unlocked;
    const at::Tensor qlen = at::sub(cu.t->narrow(0, 1, B), cu.t->narrow(0, 0, B));
    out = make({T, H, 512}, st, dev);
    lse = make({T, H}, at::kFloat, dev);
    const size_t bytes = E.v4_ws(T, H, win, cmp && !sel ? max_cmp : K);
    at::Tensor ws = make({std::max<int64_t>((int64_t)bytes, 1)}, at::kByte, dev);
    rc = E.v4(kind, q.data_ptr(), T, H, 512, B, cu.ptr<int32_t>(), qlen.data_ptr<int32_t>(), kvl.ptr<int32_t>(),
              ori.data_ptr(), ori.size(0), ori.size(1), obt.ptr<int32_t>(), obt.t->size(1), cmp.ptr<void>(), cmp_blocks,
              cmp_bs, cmp ? cbt.ptr<int32_t>() : nullptr, cmp_tl, cmp ? sel.ptr<int32_t>() : nullptr, K, ratio, win,
              max_cmp, sinks.ptr<float>(), scale, out.data_ptr(), lse.data_ptr<float>(), ws.data_ptr(), bytes,
              stream(dev));
  }
  DSA_RC(rc);
  return v[12] == Py_True ? pair(std::move(out), std::move(lse)) : wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// ({entry name: address})
PyObject* bind(PyObject*, PyObject* d) {
  struct Slot {
    const char* name;
    void* slot;
  } slots[] = {{"dsa_topk_select_workspace_size", &E.topk_ws},
               {"dsa_topk_select_ws", &E.topk},
               {"dsa_act_quant", &E.act_quant},
               {"dsa_sparse_mla_workspace_size", &E.mla_ws},
               {"dsa_sparse_mla_fwd", &E.mla},
               {"dsa_sparse_mla_decode_parts_applies", &E.parts_applies},
               {"dsa_sparse_mla_decode_parts", &E.parts},
               {"dsa_sparse_attention_fwd", &E.attention},
               {"dsa_lightning_indexer_workspace_size", &E.idx_ws},
               {"dsa_lightning_indexer", &E.idx},
               {"dsa_lightning_indexer_fused_workspace_size", &E.idxf_ws},
               {"dsa_lightning_indexer_fused", &E.idxf},
               {"dsa_lightning_indexer_tnd_workspace_size", &E.tnd_ws},
               {"dsa_lightning_indexer_tnd", &E.tnd},
               {"dsa_lightning_indexer_tnd_fused_workspace_size", &E.tndf_ws},
               {"dsa_lightning_indexer_tnd_fused", &E.tndf},
               {"dsa_sparse_flash_mla_workspace_size", &E.v4_ws},
               {"dsa_sparse_flash_mla", &E.v4}};
  for (const Slot& s : slots) {
    PyObject* o = PyDict_Check(d) ? PyDict_GetItemString(d, s.name) : nullptr;
    void* p = o ? PyLong_AsVoidPtr(o) : nullptr;
    if (!p) {
      if (!PyErr_Occurred()) PyErr_Format(PyExc_ValueError, "no address for %s", s.name);
      return nullptr;
    }
    *static_cast<void**>(s.slot) = p;
  }
  bound = true;
  Py_RETURN_NONE;
}

template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyMethodDef fast(const char* name) {
  return {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(F)), METH_FASTCALL, nullptr};
}

PyMethodDef methods[] = {fast<topk>("topk"),
                         fast<act_quant>("act_quant"),
                         fast<sparse_mla>("sparse_mla"),
                         fast<sparse_gqa>("sparse_gqa"),
                         fast<decode_parts>("decode_parts"),
                         fast<indexer>("indexer"),
                         fast<flash_mla>("flash_mla"),
                         {"bind", bind, METH_O, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "dsa_host_path", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_dsa_host_path() { return PyModule_Create(&module); }
