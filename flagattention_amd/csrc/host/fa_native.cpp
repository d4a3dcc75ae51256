// Host path of the operators, native: the checks, allocations and launches of a usual call.
//
// A decode step of a few short sequences takes about 15 us on the GPU and took about 47 us
// of Python (attribute reads of seven tensors, an argument block built field by field, six
// allocations, three foreign calls).  Each function here takes an operator's arguments,
// checks everything that the operator's Python checks, and runs the call through the C ABI
// of libflagattention_amd.so.  A call that fails any check, or is of a form not handled here
// (tensor subclasses and wrapped tensors, layouts that need a copy, empty inputs), gets None
// back before anything has been allocated or launched, and the Python path then handles it:
// it raises the error, or runs the general form.
//
// Nothing is kept between calls but the CU count of each device.  Launches run without the
// GIL, as foreign calls do.
#include <Python.h>

#include <ATen/TensorSubclassLikeUtils.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/empty_like.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdint>
#include <stdexcept>
#include <string>

#include "flagattention_amd.h"

namespace {

constexpr int64_t kFixedOverheadBlocks = 4;  // dense scheduler cost per sequence
constexpr int64_t kRowsPerTile = FA_MLA_ROWS_PER_TILE;
constexpr int64_t kPage = FA_MLA_PAGE_SIZE;
constexpr int64_t kTopkMaxLen = 65536;

PyObject* g_sig_name = nullptr;  // interned "_fa_mla_sig"

PyObject* none() { Py_RETURN_NONE; }

struct NoGil {
  PyThreadState* state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};

int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

// A plain strided GPU tensor of Python type torch.Tensor (or Parameter), else nullptr.
const at::Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !t.has_storage() ||
      at::isTensorSubclassLike(t))
    return nullptr;
  return &t;
}

bool aligned16(const at::Tensor& t) {
  return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0;
}
// 16-byte aligned rows: the base and the strides (in elements of 2 bytes) of the first dims
bool rows16(const at::Tensor& t, int dims) {
  for (int i = 0; i < dims; ++i)
    if (t.stride(i) % 8 != 0) return false;
  return aligned16(t);
}

bool to_int(PyObject* o, int64_t* v) {
  if (!PyLong_CheckExact(o)) return false;
  int overflow = 0;
  const long long x = PyLong_AsLongLongAndOverflow(o, &overflow);
  if (overflow != 0 || (x == -1 && PyErr_Occurred())) {
    PyErr_Clear();
    return false;
  }
  *v = x;
  return true;
}
bool to_double(PyObject* o, double* v) {
  if (PyFloat_CheckExact(o)) {
    *v = PyFloat_AS_DOUBLE(o);
    return true;
  }
  int64_t i;
  if (!to_int(o, &i)) return false;
  *v = static_cast<double>(i);
  return true;
}
bool to_bool(PyObject* o, bool* v) {
  if (!PyBool_Check(o)) return false;
  *v = o == Py_True;
  return true;
}

int cu_count(int device) {
  static std::atomic<int> counts[64];
  if (device < 0 || device >= 64) return 0;
  int n = counts[device].load(std::memory_order_relaxed);
  if (n == 0) {
    int32_t v = 0;
    if (fa_device_cu_count(device, &v) != FA_OK) return 0;
    n = v;
    counts[device].store(n, std::memory_order_relaxed);
  }
  return n;
}

void* stream_of(const c10::Device& d) { return c10::hip::getCurrentHIPStream(d.index()).stream(); }

at::Tensor make(at::IntArrayRef sizes, at::ScalarType dt, const c10::Device& d) {
  return at::empty(sizes, at::TensorOptions().dtype(dt).device(d));
}

void check(int rc) {
  if (rc == FA_OK) return;
  const char* msg = fa_last_error();
  throw std::runtime_error("flagattention_amd error " + std::to_string(rc) + ": " +
                           (msg ? msg : ""));
}

// ---- get_mla_metadata(cache_seqlens, rows, heads_k, heads_q, topk, num_sm_parts) ----
PyObject* mla_metadata(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 6) return none();
  const at::Tensor* lens = plain(args[0]);
  int64_t rows, heads_k, heads_q = 0, topk = 0, parts = 0;
  if (!lens || !to_int(args[1], &rows) || !to_int(args[2], &heads_k)) return none();
  const bool has_q = args[3] != Py_None, has_topk = args[4] != Py_None;
  const bool has_parts = args[5] != Py_None;
  if ((has_q && !to_int(args[3], &heads_q)) || (has_topk && !to_int(args[4], &topk)) ||
      (has_parts && !to_int(args[5], &parts)))
    return none();
  if (lens->scalar_type() != at::kInt || lens->dim() != 1 || !lens->is_contiguous()) return none();
  const int64_t batch = lens->size(0);
  if (batch < 1 || batch > FA_MLA_MAX_BATCH || heads_k != 1 || rows < 1) return none();
  if ((has_q && heads_q < 1) || (has_topk && (topk < 1 || !has_q)) || topk > INT32_MAX)
    return none();
  const c10::Device device = lens->device();
  if (!has_parts) {
    const int64_t blocks = has_topk ? std::max<int64_t>(1, rows / heads_q) * cdiv(heads_q, kRowsPerTile)
                                    : cdiv(rows, kRowsPerTile);
    const int cus = cu_count(device.index());
    if (cus == 0) return none();
    parts = std::max<int64_t>(1, std::min<int64_t>(FA_MLA_MAX_PARTS, cus / blocks));
  }
  if (parts < 1 || parts > FA_MLA_MAX_PARTS) return none();
  at::Tensor md, ns;
  {
    NoGil nogil;
    c10::DeviceGuard guard(device);
    md = make({parts, FA_MLA_MD_STRIDE}, at::kInt, device);
    ns = make({batch + 1}, at::kInt, device);
    check(fa_mla_get_metadata(lens->data_ptr<int32_t>(), static_cast<int32_t>(batch),
                              static_cast<int32_t>(topk), static_cast<int32_t>(parts),
                              has_topk ? 0 : static_cast<int32_t>(kFixedOverheadBlocks),
                              md.data_ptr<int32_t>(), ns.data_ptr<int32_t>(), stream_of(device)));
  }
  PyObject* const sig = Py_BuildValue("(LL)", static_cast<long long>(batch),
                                      static_cast<long long>(topk));
  PyObject* const a = THPVariable_Wrap(std::move(md));
  PyObject* const b = THPVariable_Wrap(std::move(ns));
  PyObject* out = nullptr;
  if (sig && a && b && PyObject_SetAttr(a, g_sig_name, sig) == 0 &&
      PyObject_SetAttr(b, g_sig_name, sig) == 0)
    out = PyTuple_Pack(2, a, b);
  Py_XDECREF(sig);
  Py_XDECREF(a);
  Py_XDECREF(b);
  return out;
  END_HANDLE_TH_ERRORS
}

// Whether scheduler metadata is untagged or was built for (batch, topk).
bool sig_matches(PyObject* t, int64_t batch, int64_t topk) {
  PyObject* sig = PyObject_GetAttr(t, g_sig_name);
  if (!sig) {
    PyErr_Clear();
    return true;
  }
  int64_t b, k;
  const bool ok = PyTuple_CheckExact(sig) && PyTuple_GET_SIZE(sig) == 2 &&
                  to_int(PyTuple_GET_ITEM(sig, 0), &b) && to_int(PyTuple_GET_ITEM(sig, 1), &k) &&
                  b == batch && k == topk;
  Py_DECREF(sig);
  return ok;
}

// ---- flash_mla_with_kvcache(q, k_cache, block_table, cache_seqlens, head_dim_v, tile_md,
//                             num_splits, softmax_scale, causal, is_fp8_kvcache, indices) ----
PyObject* mla_decode(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 11) return none();
  const at::Tensor *q = plain(args[0]), *kc = plain(args[1]), *bt = plain(args[2]),
                   *lens = plain(args[3]), *md = plain(args[5]), *ns = plain(args[6]);
  const bool sparse = args[10] != Py_None;
  const at::Tensor* idx = sparse ? plain(args[10]) : nullptr;
  if (!q || !kc || !bt || !lens || !md || !ns || (sparse && !idx)) return none();
  int64_t dv;
  double scale = 1.0 / std::sqrt(static_cast<double>(FA_MLA_D_QK));
  bool causal, fp8;
  if (!to_int(args[4], &dv) || (args[7] != Py_None && !to_double(args[7], &scale)) ||
      !to_bool(args[8], &causal) || !to_bool(args[9], &fp8) || !std::isfinite(scale))
    return none();
  if (q->dim() != 4 || kc->dim() != 4 || bt->dim() != 2 || md->dim() != 2) return none();
  const int64_t batch = q->size(0), s_q = q->size(1), h_q = q->size(2);
  if (q->scalar_type() != at::kBFloat16 || q->size(3) != FA_MLA_D_QK || dv != FA_MLA_D_V ||
      batch < 1 || batch > FA_MLA_MAX_BATCH || s_q < 1 || h_q < 1 || q->stride(3) != 1 ||
      !rows16(*q, 3))
    return none();
  const int64_t esz = kc->element_size();
  if (kc->size(0) < 1 || kc->size(1) != kPage || kc->size(2) != 1 || kc->stride(3) != 1 ||
      (kc->stride(0) * esz) % 16 != 0 || (kc->stride(1) * esz) % 16 != 0 || !aligned16(*kc))
    return none();
  if (fp8) {
    if ((kc->scalar_type() != at::kByte && kc->scalar_type() != at::kFloat8_e4m3fn) ||
        kc->size(3) != FA_MLA_FP8_ROW_BYTES || !sparse)
      return none();
  } else if (kc->scalar_type() != at::kBFloat16 || kc->size(3) != FA_MLA_D_QK) {
    return none();
  }
  if (bt->scalar_type() != at::kInt || bt->size(0) != batch || bt->size(1) < 1 ||
      bt->stride(1) != 1 || lens->scalar_type() != at::kInt || lens->dim() != 1 ||
      lens->size(0) != batch || !lens->is_contiguous())
    return none();
  const int64_t parts = md->size(0);
  if (md->scalar_type() != at::kInt || md->size(1) != FA_MLA_MD_STRIDE || !md->is_contiguous() ||
      parts < 1 || parts > FA_MLA_MAX_PARTS || ns->scalar_type() != at::kInt || ns->dim() != 1 ||
      ns->size(0) != batch + 1 || !ns->is_contiguous())
    return none();
  int64_t topk = 0;
  if (sparse) {
    if (idx->scalar_type() != at::kInt || idx->dim() != 3 || idx->size(0) != batch ||
        idx->size(1) != s_q || idx->size(2) < 1 || idx->size(2) > INT32_MAX ||
        idx->stride(2) != 1 || causal)
      return none();
    topk = idx->size(2);
  }
  if (!sig_matches(args[5], batch, topk) || !sig_matches(args[6], batch, topk)) return none();
  const c10::Device device = q->device();
  for (const at::Tensor* t : {kc, bt, lens, md, ns})
    if (t->device() != device) return none();
  if (sparse && idx->device() != device) return none();

  at::Tensor out, lse;
  {
    NoGil nogil;
    c10::DeviceGuard guard(device);
    const int64_t rows = s_q * h_q;
    out = make({batch, s_q, h_q, FA_MLA_D_V}, at::kBFloat16, device);
    lse = make({batch, h_q, s_q}, at::kFloat, device);
    // one workspace: partial outputs (bf16), their lse (fp32), gather rows (int32)
    const int64_t o_bytes = (batch + parts) * rows * FA_MLA_D_V * 2;
    const int64_t lse_bytes = cdiv((batch + parts) * rows * 4, 256) * 256;
    // row ids only where the decode does not translate its slots itself
    const int64_t row_bytes = topk > FA_MLA_FOLD_TOPK ? batch * s_q * cdiv(topk, kPage) * kPage * 4 : 0;
    const at::Tensor ws = make({o_bytes + lse_bytes + row_bytes}, at::kByte, device);
    uint8_t* const w = ws.data_ptr<uint8_t>();
    fa_mla_decode_args a = {};
    a.q = q->data_ptr();
    a.q_stride_b = q->stride(0);
    a.q_stride_s = q->stride(1);
    a.q_stride_h = q->stride(2);
    a.kv = kc->data_ptr();
    a.kv_block_stride = kc->stride(0) * esz;
    a.kv_row_stride = kc->stride(1) * esz;
    a.num_kv_blocks = kc->size(0);
    a.block_table = bt->data_ptr<int32_t>();
    a.bt_stride_b = bt->stride(0);
    a.max_blocks_per_seq = static_cast<int32_t>(bt->size(1));
    a.cache_seqlens = lens->data_ptr<int32_t>();
    a.tile_md = md->data_ptr<int32_t>();
    a.num_splits = ns->data_ptr<int32_t>();
    a.num_parts = static_cast<int32_t>(parts);
    a.out = out.data_ptr();
    a.lse = lse.data_ptr<float>();
    a.o_accum = w;
    a.lse_accum = reinterpret_cast<float*>(w + o_bytes);
    a.batch = static_cast<int32_t>(batch);
    a.s_q = static_cast<int32_t>(s_q);
    a.h_q = static_cast<int32_t>(h_q);
    a.softmax_scale = static_cast<float>(scale);
    a.causal = causal;
    void* const stream = stream_of(device);
    if (sparse) {
      a.indices = idx->data_ptr<int32_t>();
      a.idx_stride_b = idx->stride(0);
      a.idx_stride_s = idx->stride(1);
      a.topk = static_cast<int32_t>(topk);
      if (topk > FA_MLA_FOLD_TOPK) {
        a.sparse_rows = reinterpret_cast<int32_t*>(w + o_bytes + lse_bytes);
        check(fa_mla_sparse_rows(&a, stream));
      }
      check(fa_mla_decode_sparse(&a, fp8, stream));
    } else {
      check(fa_mla_decode_dense(&a, stream));
    }
    check(fa_mla_combine(&a, stream));
  }
  PyObject* const o = THPVariable_Wrap(std::move(out));
  PyObject* const l = THPVariable_Wrap(std::move(lse));
  PyObject* const both = o && l ? PyTuple_Pack(2, o, l) : nullptr;
  Py_XDECREF(o);
  Py_XDECREF(l);
  return both;
  END_HANDLE_TH_ERRORS
}

// ---- grouped-query decode ----
bool gqa_dim(int64_t d) {
  return d == 16 || d == 32 || d == 64 || d == 128 || d == 256 || d == 512;
}
bool gqa_dtype(const at::Tensor& t) {
  return t.scalar_type() == at::kHalf || t.scalar_type() == at::kBFloat16;
}

// The split rule of gqa.py, whose comments say why its lines lie there; its constants have the
// same names there, and tests/test_native_host.py compares the two rules.
constexpr int64_t kRowsPerWg = 16;
constexpr int64_t kMinSplitTokens = 256;
constexpr int64_t kShortSplitTokens = 128;
constexpr int64_t kMaxShortSplits = 64, kMaxShortSplitsSmallDim = 16;
constexpr int64_t kMaxShortPartials = int64_t{1} << 21;
constexpr int64_t kPrefillMinRows = 16;
constexpr int64_t kPrefillRowsPerWg = 128;
constexpr int64_t kPrefillUnsplitTokens = 512;
constexpr int64_t kPrefillMaxPartials = int64_t{1} << 20;

// rows = query rows per KV head, pairs = batch x KV heads.
int64_t choose_splits(int64_t pairs, int64_t rows, int64_t rows_per_wg, int64_t d, int64_t max_len,
                      int64_t cus) {
  const int64_t base = pairs * cdiv(rows, rows_per_wg);
  if (base >= cus || max_len <= kMinSplitTokens) return 1;
  const int64_t s = std::min(cdiv(2 * cus, base), cdiv(max_len, kMinSplitTokens));
  const bool one_wg_per_cu = rows_per_wg == kRowsPerWg && d >= 256;
  const int64_t few =
      std::min(one_wg_per_cu ? cus / base : cdiv(cus, base), cdiv(max_len, kShortSplitTokens));
  if (few > (d > 64 ? kMaxShortSplits : kMaxShortSplitsSmallDim) ||
      pairs * rows * few * d > kMaxShortPartials)
    return s;
  return std::max(s, few);
}

// Whether a many-row call of few keys runs unsplit.
bool prefill_unsplit(int64_t pairs, int64_t rows, int64_t d, int64_t n, int64_t cus) {
  if (n > kPrefillUnsplitTokens) return false;
  const int64_t few =
      std::min(cdiv(cus, pairs * cdiv(rows, kPrefillRowsPerWg)), cdiv(n, kShortSplitTokens));
  return n <= (d == 256 ? 256 : 384) || few < 3 || pairs * rows * few * d > kPrefillMaxPartials;
}

// Splits of a contiguous call.
int64_t contiguous_splits(int64_t pairs, int64_t rows, int64_t d, int64_t n, int64_t cus) {
  const bool many = (d == 64 || d == 128 || d == 256) && rows > kPrefillMinRows;
  if (many && prefill_unsplit(pairs, rows, d, n, cus)) return 1;
  return choose_splits(pairs, rows, many ? kPrefillRowsPerWg : kRowsPerWg, d, n, cus);
}

// whole 32-key tiles (gqa.py)
int64_t whole_tiles(int64_t tokens) { return cdiv(tokens, 32) * 32; }

void run_gqa(fa_gqa_decode_args& a, int64_t rows, const c10::Device& device) {
  at::Tensor part;
  if (a.num_splits > 1) {
    const int64_t n = rows * a.num_splits;
    part = make({n * (a.d + 1)}, at::kFloat, device);
    a.o_part = part.data_ptr<float>();
    a.lse_part = a.o_part + n * a.d;
  }
  void* const stream = stream_of(device);
  check(fa_gqa_decode(&a, stream));
  if (a.num_splits > 1) check(fa_gqa_combine(&a, stream));
}

// paged_attention(query, key_cache, value_cache, context_lens, block_tables, attn_scale,
//                 max_context_len, num_splits)
PyObject* paged(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 8) return none();
  const at::Tensor *q = plain(args[0]), *k = plain(args[1]), *v = plain(args[2]),
                   *lens = plain(args[3]), *bt = plain(args[4]);
  double scale;
  int64_t max_len, num_splits;
  if (!q || !k || !v || !lens || !bt || !to_double(args[5], &scale) ||
      !to_int(args[6], &max_len) || !to_int(args[7], &num_splits))
    return none();
  if (q->dim() != 3 || k->dim() != 4 || !v->sizes().equals(k->sizes()) ||
      !v->strides().equals(k->strides()))
    return none();
  const int64_t seqs = q->size(0), h_q = q->size(1), d = q->size(2);
  const int64_t nblk = k->size(0), h_kv = k->size(1), block = k->size(2);
  if (seqs < 1 || k->size(3) != d || !gqa_dim(d) || h_kv < 1 || h_q < 1 || h_q % h_kv != 0 ||
      block < 1 || nblk < 1 || !gqa_dtype(*q) || k->scalar_type() != q->scalar_type() ||
      v->scalar_type() != q->scalar_type() || q->stride(2) != 1 || k->stride(3) != 1 ||
      !rows16(*q, 2) || !rows16(*k, 3) || !rows16(*v, 3))
    return none();
  if (lens->scalar_type() != at::kInt || lens->dim() != 1 || lens->size(0) != seqs ||
      !lens->is_contiguous() || bt->scalar_type() != at::kInt || bt->dim() != 2 ||
      bt->size(0) != seqs || bt->size(1) < 1 || bt->stride(1) != 1)
    return none();
  if (num_splits < 0 || max_len < 1 || max_len > (1 << 30)) return none();
  const c10::Device device = q->device();
  for (const at::Tensor* t : {k, v, lens, bt})
    if (t->device() != device) return none();
  int64_t split_tokens;
  if (num_splits == 0) {
    const int cus = cu_count(device.index());
    if (cus == 0) return none();
    split_tokens = whole_tiles(
        cdiv(max_len, choose_splits(seqs * h_kv, h_q / h_kv, kRowsPerWg, d, max_len, cus)));
  } else if (num_splits == 1) {
    split_tokens = max_len;
  } else {
    const int64_t each = cdiv(max_len, num_splits);
    split_tokens = 1;
    while (split_tokens < each) split_tokens *= 2;
  }
  const int64_t s = cdiv(max_len, split_tokens);
  if (s == 1) split_tokens = 1 << 30;  // one split sees every key of its sequence
  at::Tensor out;
  {
    NoGil nogil;
    c10::DeviceGuard guard(device);
    out = at::empty_like(*q);
    fa_gqa_decode_args a = {};
    a.q = q->data_ptr();
    a.q_stride_b = q->stride(0);
    a.q_stride_h = q->stride(1);
    a.k = k->data_ptr();
    a.v = v->data_ptr();
    a.k_stride_0 = k->stride(0);
    a.k_stride_h = k->stride(1);
    a.k_stride_t = k->stride(2);
    a.v_stride_0 = v->stride(0);
    a.v_stride_h = v->stride(1);
    a.v_stride_t = v->stride(2);
    a.block_table = bt->data_ptr<int32_t>();
    a.bt_stride_b = bt->stride(0);
    a.max_blocks_per_seq = static_cast<int32_t>(bt->size(1));
    a.block_size = static_cast<int32_t>(block);
    a.num_blocks = nblk;
    a.seqlens = lens->data_ptr<int32_t>();
    a.out = out.data_ptr();
    a.o_stride_b = out.stride(0);
    a.o_stride_h = out.stride(1);
    a.batch = static_cast<int32_t>(seqs);
    a.h_q = static_cast<int32_t>(h_q);
    a.h_kv = static_cast<int32_t>(h_kv);
    a.m = 1;
    a.d = static_cast<int32_t>(d);
    a.num_splits = static_cast<int32_t>(s);
    a.split_tokens = static_cast<int32_t>(split_tokens);
    a.scale = static_cast<float>(scale);
    a.dtype = q->scalar_type() == at::kBFloat16;
    run_gqa(a, seqs * h_q, device);
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// _dense_decode(q, k, v, causal, sm_scale, want_lse): (o, lse or None)
PyObject* contiguous(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 6) return none();
  const at::Tensor *q = plain(args[0]), *k = plain(args[1]), *v = plain(args[2]);
  bool causal, want_lse;
  if (!q || !k || !v || !to_bool(args[3], &causal) || !to_bool(args[5], &want_lse)) return none();
  if (q->dim() != 4 || k->dim() != 4 || v->dim() != 4) return none();
  const int64_t batch = q->size(0), h_q = q->size(1), m = q->size(2), d = q->size(3);
  const int64_t h_kv = k->size(1), n = k->size(2);
  double scale = 1.0 / std::sqrt(static_cast<double>(d));
  if (args[4] != Py_None && !to_double(args[4], &scale)) return none();
  if (batch < 1 || h_q < 1 || m < 1 || n < 1 || n > (1 << 30) || !gqa_dim(d) ||
      k->size(0) != batch || k->size(3) != d || !v->sizes().equals(k->sizes()) || h_kv < 1 ||
      h_q % h_kv != 0 || !gqa_dtype(*q) || k->scalar_type() != q->scalar_type() ||
      v->scalar_type() != q->scalar_type() || !std::isfinite(scale))
    return none();
  if (q->stride(3) != 1 || k->stride(3) != 1 || v->stride(3) != 1 || !rows16(*q, 3) ||
      !rows16(*k, 3) || !rows16(*v, 3))
    return none();
  const c10::Device device = q->device();
  if (k->device() != device || v->device() != device) return none();
  const int cus = cu_count(device.index());
  if (cus == 0) return none();
  int64_t s = contiguous_splits(batch * h_kv, h_q / h_kv * m, d, n, cus);
  int64_t split_tokens = whole_tiles(cdiv(n, s));
  s = cdiv(n, split_tokens);
  if (s == 1) split_tokens = 1 << 30;
  at::Tensor out, lse;
  {
    NoGil nogil;
    c10::DeviceGuard guard(device);
    out = at::empty_like(*q);
    if (out.stride(3) != 1 || !rows16(out, 3)) out = make(q->sizes(), q->scalar_type(), device);
    if (want_lse) lse = make({batch, h_q, m}, at::kFloat, device);
    fa_gqa_decode_args a = {};
    a.q = q->data_ptr();
    a.q_stride_b = q->stride(0);
    a.q_stride_h = q->stride(1);
    a.q_stride_m = q->stride(2);
    a.k = k->data_ptr();
    a.v = v->data_ptr();
    a.k_stride_0 = k->stride(0);
    a.k_stride_h = k->stride(1);
    a.k_stride_t = k->stride(2);
    a.v_stride_0 = v->stride(0);
    a.v_stride_h = v->stride(1);
    a.v_stride_t = v->stride(2);
    a.n = static_cast<int32_t>(n);
    a.out = out.data_ptr();
    a.o_stride_b = out.stride(0);
    a.o_stride_h = out.stride(1);
    a.o_stride_m = out.stride(2);
    a.lse = want_lse ? lse.data_ptr<float>() : nullptr;
    a.batch = static_cast<int32_t>(batch);
    a.h_q = static_cast<int32_t>(h_q);
    a.h_kv = static_cast<int32_t>(h_kv);
    a.m = static_cast<int32_t>(m);
    a.d = static_cast<int32_t>(d);
    a.num_splits = static_cast<int32_t>(s);
    a.split_tokens = static_cast<int32_t>(split_tokens);
    a.scale = static_cast<float>(scale);
    a.causal = causal;
    a.dtype = q->scalar_type() == at::kBFloat16;
    run_gqa(a, batch * h_q * m, device);
  }
  PyObject* const o = THPVariable_Wrap(std::move(out));
  PyObject* l = Py_None;
  if (want_lse)
    l = THPVariable_Wrap(std::move(lse));
  else
    Py_INCREF(l);
  PyObject* const both = o && l ? PyTuple_Pack(2, o, l) : nullptr;
  Py_XDECREF(o);
  Py_XDECREF(l);
  return both;
  END_HANDLE_TH_ERRORS
}

// split_counts(pairs, rows, d, n, cus): the split counts that the rule gives a paged and a
// contiguous call (1 or more of each extent), for the comparison with gqa.py.
PyObject* split_counts(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  int64_t x[5];
  if (nargs != 5) return none();
  for (int i = 0; i < 5; ++i)
    if (!to_int(args[i], &x[i]) || x[i] < 1) return none();
  return Py_BuildValue(
      "(LL)", static_cast<long long>(choose_splits(x[0], x[1], kRowsPerWg, x[2], x[3], x[4])),
      static_cast<long long>(contiguous_splits(x[0], x[1], x[2], x[3], x[4])));
}

// ---- topk_indices(scores, cache_seqlens, topk, causal), result allocated here ----
PyObject* topk_indices(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 4) return none();
  const at::Tensor *scores = plain(args[0]), *lens = plain(args[1]);
  int64_t topk;
  bool causal;
  if (!scores || !lens || !to_int(args[2], &topk) || !to_bool(args[3], &causal)) return none();
  if (scores->dim() != 3 || scores->scalar_type() != at::kFloat || lens->dim() != 1 ||
      lens->scalar_type() != at::kInt || !lens->is_contiguous())
    return none();
  const int64_t batch = scores->size(0), s_q = scores->size(1), len = scores->size(2);
  if (batch < 1 || s_q < 1 || len < 1 || len > kTopkMaxLen || topk < 1 || topk > kTopkMaxLen ||
      scores->stride(2) != 1 || lens->size(0) != batch || lens->device() != scores->device() ||
      batch > INT32_MAX || s_q > INT32_MAX)
    return none();
  const int64_t ws_bytes =
      fa_mla_topk_workspace_bytes(static_cast<int32_t>(batch), static_cast<int32_t>(s_q),
                                  static_cast<int32_t>(len), static_cast<int32_t>(topk));
  if (ws_bytes < 0) return none();
  at::Tensor out;
  {
    NoGil nogil;
    const c10::Device device = scores->device();
    c10::DeviceGuard guard(device);
    out = make({batch, s_q, topk}, at::kInt, device);
    at::Tensor ws;
    if (ws_bytes > 0) ws = make({ws_bytes}, at::kByte, device);
    check(fa_mla_topk_indices(scores->data_ptr<float>(), scores->stride(0), scores->stride(1),
                              lens->data_ptr<int32_t>(), static_cast<int32_t>(batch),
                              static_cast<int32_t>(s_q), static_cast<int32_t>(len),
                              static_cast<int32_t>(topk), causal, out.data_ptr<int32_t>(),
                              ws_bytes > 0 ? ws.data_ptr() : nullptr, ws_bytes,
                              stream_of(device)));
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// ---- concat_and_cache_mla(kv_c, k_pe, kv_cache, slot_mapping, is_fp8): True when done ----
PyObject* cache_write(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 5) return none();
  const at::Tensor *kv = plain(args[0]), *pe = plain(args[1]), *cache = plain(args[2]),
                   *slots = plain(args[3]);
  bool fp8;
  if (!kv || !pe || !cache || !slots || !to_bool(args[4], &fp8)) return none();
  if (kv->dim() != 2 || pe->dim() != 2 || cache->dim() != 4 || slots->dim() != 1) return none();
  const int64_t t = kv->size(0);
  if (t < 1 || t > INT32_MAX || kv->scalar_type() != at::kBFloat16 || kv->size(1) != FA_MLA_D_V ||
      pe->scalar_type() != at::kBFloat16 || pe->size(0) != t ||
      pe->size(1) != FA_MLA_D_QK - FA_MLA_D_V || kv->stride(1) != 1 || pe->stride(1) != 1 ||
      !rows16(*kv, 1) || !rows16(*pe, 1))
    return none();
  const int64_t esz = cache->element_size();
  if (cache->size(0) < 1 || cache->size(1) != kPage || cache->size(2) != 1 ||
      cache->stride(3) != 1 || (cache->stride(0) * esz) % 16 != 0 ||
      (cache->stride(1) * esz) % 16 != 0 || !aligned16(*cache))
    return none();
  if (fp8 ? (cache->size(3) != FA_MLA_FP8_ROW_BYTES ||
             (cache->scalar_type() != at::kByte && cache->scalar_type() != at::kFloat8_e4m3fn))
          : (cache->size(3) != FA_MLA_D_QK || cache->scalar_type() != at::kBFloat16))
    return none();
  if ((slots->scalar_type() != at::kLong && slots->scalar_type() != at::kInt) ||
      slots->size(0) != t)
    return none();
  const c10::Device device = kv->device();
  for (const at::Tensor* x : {pe, cache, slots})
    if (x->device() != device) return none();
  {
    NoGil nogil;
    c10::DeviceGuard guard(device);
    const at::Tensor wide = slots->to(at::kLong).contiguous();
    check(fa_mla_kvcache_write(kv->data_ptr(), kv->stride(0), pe->data_ptr(), pe->stride(0),
                               wide.data_ptr<int64_t>(), static_cast<int32_t>(t),
                               cache->data_ptr(), cache->stride(0) * esz, cache->stride(1) * esz,
                               cache->size(0), fp8, stream_of(device)));
  }
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

#define FA_METHOD(name)                                                                     \
  {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(name)), METH_FASTCALL, \
   nullptr}
PyMethodDef g_methods[] = {FA_METHOD(mla_metadata), FA_METHOD(mla_decode),   FA_METHOD(paged),
                           FA_METHOD(contiguous),   FA_METHOD(topk_indices), FA_METHOD(cache_write),
                           FA_METHOD(split_counts), {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, g_methods};

}  // namespace

PyMODINIT_FUNC PyInit__native() {
  g_sig_name = PyUnicode_InternFromString("_fa_mla_sig");
  PyObject* const m = g_sig_name ? PyModule_Create(&g_module) : nullptr;
  if (m && PyModule_AddIntConstant(m, "ABI_VERSION", FA_ABI_VERSION) != 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
