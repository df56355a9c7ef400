// Native call path of the Python launchers: reads the tensors of one call,
// fills the C-ABI argument structs and launches, in a few microseconds where
// the same steps in Python take 15 to 25 (about 45 struct fields, 40 tensor
// attributes), longer than the small kernels they launch.
//
// A call takes this path only when everything about it is ordinary: plain
// torch.Tensor arguments on one GPU in the shapes, dtypes, strides and sizes
// that the Python launcher accepts, launched on the current stream, not under
// stream capture.  Anything else returns None before anything is launched, and
// the Python launcher (flydsl_amd/*.py) then does the call, or raises what it
// raises.  Which schedule a decode takes is the Python launcher's decision
// too (`plan` below).
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstring>

#include "pa_fp8.h"

namespace {

struct Entry {
  decltype(&pa_fp8_decode_partition) partition;
  decltype(&pa_fp8_decode_reduce) reduce;
  decltype(&pa_fp8_decode_split) split;
  decltype(&pa_fp8_decode_team) team;
  decltype(&pa_fp8_split_slot_bytes) split_bytes;
  decltype(&pa_fp8_team_slot_bytes) team_bytes;
  decltype(&pa_fp8_decode_balanced) balanced;
  decltype(&pa_fp8_merge_balanced) merge;
  decltype(&pa_fp8_balanced_workspace_bytes) balanced_bytes;
  decltype(&pa_fp8_decode_worklist) worklist;
  decltype(&pa_fp8_reduce_worklist) reduce_worklist;
  decltype(&pa_fp8_recommended_splits) splits;
  decltype(&pa_fp8_rope_cache) rope;
  decltype(&pa_fp8_qk_norm_rope_quant) qknr;
  decltype(&pa_fp8_mla_decode) mla_decode;
  decltype(&pa_fp8_mla_reduce) mla_reduce;
} fn;
bool ready = false;
PyObject* check_fn = nullptr;  // _lib.check(rc, name): raises

#define NOT_HERE Py_RETURN_NONE

// Launches `call` without the GIL, as ctypes does.
template <typename F>
int launch(F&& call) {
  int rc;
  Py_BEGIN_ALLOW_THREADS;
  rc = call();
  Py_END_ALLOW_THREADS;
  return rc;
}

// A plain tensor on GPU `dev` (-1: any, then set), or nullptr.
struct Reader {
  int dev = -1;
  bool ok = true;
  const at::Tensor* operator()(PyObject* o) {
    if (!ok || !THPVariable_CheckExact(o)) {
      ok = false;
      return nullptr;
    }
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided) {
      ok = false;
      return nullptr;
    }
    const int d = t.device().index();
    if (dev < 0) dev = d;
    if (d != dev) ok = false;
    return &t;
  }
};

bool is(const at::Tensor& t, at::ScalarType s) { return t.scalar_type() == s; }
bool one_byte(const at::Tensor& t) { return t.element_size() == 1; }
bool shape_is(const at::Tensor& t, std::initializer_list<int64_t> s) {
  return t.sizes() == at::IntArrayRef(s.begin(), s.size());
}
bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// Stream of the call: the device's current one, unless it is capturing.
bool current(int dev, hipStream_t* s, int64_t* id) {
  const c10::hip::HIPStream st = c10::hip::getCurrentHIPStream((c10::DeviceIndex)dev);
  *s = st.stream();
  *id = (int64_t)st.id();
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  return hipStreamIsCapturing(*s, &cap) == hipSuccess && cap == hipStreamCaptureStatusNone;
}

PyObject* failed(int rc, const char* name) {
  PyObject* r = PyObject_CallFunction(check_fn, "is", rc, name);
  if (r) {
    Py_DECREF(r);
    PyErr_Format(PyExc_RuntimeError, "%s failed: %d", name, rc);
  }
  return nullptr;
}

at::Tensor device_bytes(int64_t n, int dev) {
  return at::empty({n}, at::TensorOptions().dtype(at::kByte).device(at::Device(at::kCUDA, (c10::DeviceIndex)dev)));
}

// Errors of torch calls end the native attempt; nothing has been launched
// where they can occur.
template <typename F>
PyObject* guarded(F&& f) {
  if (!ready) NOT_HERE;
  try {
    return f();
  } catch (const std::exception&) {
    if (PyErr_Occurred()) return nullptr;
    NOT_HERE;
  }
}

// ---------------------------------------------------------------------------
// Paged decode
// ---------------------------------------------------------------------------

bool md_tensor(PyObject* md, const char* key, Reader& rd, const at::Tensor** out) {
  PyObject* o = PyDict_GetItemString(md, key);
  if (!o) return false;
  *out = rd(o);
  return rd.ok;
}
bool md_int(PyObject* md, const char* key, int64_t* out) {
  PyObject* o = PyDict_GetItemString(md, key);
  if (!o || !PyLong_CheckExact(o)) return false;
  *out = PyLong_AsLongLong(o);
  return !PyErr_Occurred();
}

// pa_decode(output, query, key_cache, value_cache, context_lengths, kv_page_indices, kv_indptr, softmax_scale,
//           key_scale, value_scale, sliding_window, metadata, block_tables, max_context_partition_num,
//           exp_sums, max_logits, temporary_output, plan, workspace)
//   plan(route, batch, kv_heads, P, eqgs, head_size, block_size, capacity, tokens, user_partials, have_partials,
//        False, one_launch, per_token, device index) -> (kind, n, P)
//   workspace(device, stream id, pairs, bytes) -> (slots, bytes, counters, count, holder)
PyObject* pa_decode(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 19) NOT_HERE;
  return guarded([&]() -> PyObject* {
    Reader rd;
    const at::Tensor *out = rd(a[0]), *q = rd(a[1]), *kc = rd(a[2]), *vc = rd(a[3]), *cl = rd(a[4]), *ks = rd(a[8]),
                     *vs = rd(a[9]);
    if (!rd.ok || !PyFloat_CheckExact(a[7]) || !PyLong_CheckExact(a[10]) || !PyLong_CheckExact(a[13])) NOT_HERE;
    const double scale = PyFloat_AS_DOUBLE(a[7]);
    const int64_t window = PyLong_AsLongLong(a[10]);
    int64_t P = PyLong_AsLongLong(a[13]);
    if (PyErr_Occurred() || window < 0 || window > 0x7fffffff || P < 0 || P > 0xffff) return PyErr_Clear(), Py_NewRef(Py_None);
    if (q->dim() != 3 || out->dim() != 3 || kc->dim() != 5 || cl->dim() != 1 || cl->size(0) == 0) NOT_HERE;
    const bool bf16 = is(*q, at::kBFloat16);
    if (!bf16 && !is(*q, at::kHalf)) NOT_HERE;
    int od;
    if (is(*out, at::kBFloat16)) od = PA_DTYPE_BF16;
    else if (is(*out, at::kHalf)) od = PA_DTYPE_F16;
    else if (is(*out, at::kFloat)) od = PA_DTYPE_F32;
    else NOT_HERE;
    const int64_t B = cl->size(0), rows = q->size(0), Hq = q->size(1), D = q->size(2);
    const int64_t NB = kc->size(0), H = kc->size(1), bs = kc->size(3);
    if (H <= 0 || rows % B || rows == 0 || Hq % H || D % 64 || D < 64 || D > 512 || NB <= 0 || bs <= 0) NOT_HERE;
    const int64_t ql = rows / B, gqa = Hq / H, eq = ql * gqa;
    if (kc->size(2) != D / 16 || kc->size(4) != 16 || !one_byte(*kc) || !one_byte(*vc)) NOT_HERE;
    const bool trans = vc->dim() == 5;
    if (trans ? !(vc->size(2) == bs / 16 && vc->size(3) == D && vc->size(4) == 16)
              : !(vc->dim() == 4 && vc->size(2) == D && vc->size(3) == bs))
      NOT_HERE;
    if (q->stride(2) != 1 || out->stride(2) != 1 || kc->stride(4) != 1 || vc->stride(-1) != 1) NOT_HERE;
    if (out->sizes() != q->sizes()) NOT_HERE;
    const bool pt = ks->dim() > 1;
    if (!is(*ks, at::kFloat) || !is(*vs, at::kFloat)) NOT_HERE;
    if (pt) {
      if (ks->dim() != 4 || vs->dim() != 4 || ks->size(0) != NB || ks->size(1) != H || ks->size(2) != bs ||
          ks->strides() != vs->strides() || ks->stride(2) != 1)
        NOT_HERE;
    }
    if (!is(*cl, at::kInt)) NOT_HERE;
    const int64_t lim = 0x7fffffff;
    if (B > lim || NB > lim || H > lim || bs > lim || Hq > lim) NOT_HERE;

    PyObject* md = a[11];
    const char* route;
    const at::Tensor* pages = nullptr;
    const at::Tensor* indptr = nullptr;
    if (window > 0) {
      route = "sw";
      const int need = fn.splits((int)B, (int)H, 1, (int)window, 256, (int)ql, 1);
      if (P == 0) P = need;
      if (1 < P && P < need) NOT_HERE;
    } else if (bs == 16 || bs == 64) {
      route = "small";
    } else {
      route = "flat";
    }
    const bool flat = route[0] == 'f';
    if (flat) {
      pages = rd(a[5]);
      indptr = rd(a[6]);
      if (!rd.ok || !is(*pages, at::kInt) || !is(*indptr, at::kInt)) NOT_HERE;
    } else {
      pages = rd(a[12]);
      if (!rd.ok || !is(*pages, at::kInt) || pages->dim() != 2 || pages->stride(1) != 1 || pages->size(0) < B) NOT_HERE;
    }
    if (!flat && md != Py_None) NOT_HERE;
    if (pages->numel() > lim) NOT_HERE;

    hipStream_t s;
    int64_t sid;
    if (!current(rd.dev, &s, &sid)) NOT_HERE;

    const at::Tensor* part[3] = {nullptr, nullptr, nullptr};
    int given = 0;
    for (int i = 0; i < 3; ++i)
      if (a[14 + i] != Py_None) {
        part[i] = rd(a[14 + i]);
        ++given;
      }
    if (!rd.ok) NOT_HERE;

    pa_fp8_stream_args sa;
    std::memset(&sa, 0, sizeof sa);
    sa.abi_version = PA_FP8_ABI_VERSION;
    sa.output = out->data_ptr();
    sa.query = q->data_ptr();
    sa.key_cache = kc->data_ptr();
    sa.value_cache = vc->data_ptr();
    sa.block_tables = (const int32_t*)pages->data_ptr();
    sa.context_lengths = (const int32_t*)cl->data_ptr();
    sa.key_scale = (const float*)ks->data_ptr();
    sa.value_scale = (const float*)vs->data_ptr();
    if (flat) {
      sa.kv_indptr = (const int32_t*)indptr->data_ptr();
      sa.max_blocks_per_seq = (int32_t)std::max<int64_t>(1, pages->numel());
    } else {
      sa.stride_bt_seq = pages->stride(0);
      sa.max_blocks_per_seq = (int32_t)pages->size(1);
    }
    sa.stride_q_tok = q->stride(0);
    sa.stride_q_head = q->stride(1);
    sa.stride_k_block = kc->stride(0);
    sa.stride_k_head = kc->stride(1);
    sa.stride_v_block = vc->stride(0);
    sa.stride_v_head = vc->stride(1);
    if (pt) {
      sa.stride_ks_block = ks->stride(0);
      sa.stride_ks_head = ks->stride(1);
    }
    sa.stride_out_tok = out->stride(0);
    sa.stride_out_head = out->stride(1);
    sa.num_seqs = (int32_t)B;
    sa.num_kv_heads = (int32_t)H;
    sa.query_length = (int32_t)ql;
    sa.query_group_size = (int32_t)gqa;
    sa.head_size = (int32_t)D;
    sa.block_size = (int32_t)bs;
    sa.num_blocks = (int32_t)NB;
    sa.sliding_window = (int32_t)window;
    sa.per_token_kv = pt;
    sa.trans_v = trans;
    sa.query_dtype = bf16 ? PA_DTYPE_BF16 : PA_DTYPE_F16;
    sa.output_dtype = od;
    sa.softmax_scale = (float)scale;
    int rc;

    if (flat && md != Py_None) {
      if (!PyDict_CheckExact(md)) NOT_HERE;
      const at::Tensor *wi, *wf, *pi, *ri, *rf, *rp, *po, *pl;
      int64_t num_sm, psize, mql;
      if (!md_tensor(md, "work_indptr", rd, &wi) || !md_tensor(md, "work_info_flat", rd, &wf) ||
          !md_tensor(md, "partition_indptr", rd, &pi) || !md_tensor(md, "reduce_indptr", rd, &ri) ||
          !md_tensor(md, "reduce_final_map", rd, &rf) || !md_tensor(md, "reduce_partial_map", rd, &rp) ||
          !md_tensor(md, "partial_output", rd, &po) || !md_tensor(md, "partial_lse", rd, &pl) ||
          !md_int(md, "num_sm", &num_sm) || !md_int(md, "partition_size", &psize) ||
          !md_int(md, "query_length", &mql) || !md_int(md, "stride_po_ql", &sa.stride_po_row) ||
          !md_int(md, "stride_pl_ql", &sa.stride_pl_row)) {
        PyErr_Clear();
        NOT_HERE;
      }
      if (psize != 256 || mql != ql || pi->size(0) != B + 1 || !is(*po, at::kFloat) || !is(*pl, at::kFloat) ||
          !is(*wi, at::kInt) || !is(*wf, at::kInt) || !is(*pi, at::kInt) || !is(*ri, at::kInt) ||
          !is(*rf, at::kInt) || !is(*rp, at::kInt))
        NOT_HERE;
      sa.work_indptr = (const int32_t*)wi->data_ptr();
      sa.work_info = (const int32_t*)wf->data_ptr();
      sa.partition_indptr = (const int32_t*)pi->data_ptr();
      sa.partial_output = (float*)po->data_ptr();
      sa.partial_lse = (float*)pl->data_ptr();
      sa.num_workers = (int32_t)num_sm;
      pa_fp8_worklist_reduce_args r;
      std::memset(&r, 0, sizeof r);
      r.abi_version = PA_FP8_ABI_VERSION;
      r.output = out->data_ptr();
      // the reduce reads partial rows from row query_length on
      r.partial_output = sa.partial_output + ql * sa.stride_po_row;
      r.partial_lse = sa.partial_lse + ql * sa.stride_pl_row;
      r.reduce_indptr = (const int32_t*)ri->data_ptr();
      r.reduce_final_map = (const int32_t*)rf->data_ptr();
      r.reduce_partial_map = (const int32_t*)rp->data_ptr();
      r.stride_out_tok = sa.stride_out_tok;
      r.stride_out_head = sa.stride_out_head;
      r.stride_po_row = sa.stride_po_row;
      r.stride_pl_row = sa.stride_pl_row;
      r.num_groups = (int32_t)B;
      r.num_query_heads = (int32_t)Hq;
      r.head_size = (int32_t)D;
      r.max_query_length = (int32_t)ql;
      r.output_dtype = od;
      if ((rc = launch([&] { return fn.worklist(&sa, s); })) != 0) return failed(rc, "pa_fp8_decode_worklist");
      if ((rc = launch([&] { return fn.reduce_worklist(&r, s); })) != 0) return failed(rc, "pa_fp8_reduce_worklist");
      return PyUnicode_FromString("ps_split_reduce");
    }

    // ---- the schedule ----
    auto in31 = [&](int64_t x) { return x >= 0 && x <= lim; };
    const bool one_launch = aligned16(sa.output) && sa.stride_out_tok % 8 == 0 && sa.stride_out_head % 8 == 0 &&
                            in31(sa.stride_k_block) && in31(sa.stride_v_block) && (!pt || in31(sa.stride_ks_block));
    const int64_t capacity = flat ? -1 : pages->size(1) * bs;
    int64_t tokens = flat ? pages->numel() * bs : capacity;
    if (window > 0) tokens = std::min<int64_t>(tokens, window + ql + 32);
    auto truth = [](bool x) { return x ? Py_True : Py_False; };
    PyObject* cap = flat ? Py_NewRef(Py_None) : PyLong_FromLongLong(capacity);
    if (!cap) return nullptr;
    PyObject* plan = PyObject_CallFunction(
        a[17], "sLLLLLLOLOOOOOi", route, (long long)B, (long long)H, (long long)P, (long long)eq, (long long)D,
        (long long)bs, cap, (long long)tokens, truth(given > 0), truth(given == 3), Py_False, truth(one_launch),
        truth(pt), rd.dev);
    Py_DECREF(cap);
    if (!plan) return nullptr;
    const char* kind_s;
    int spw = 0, slots = 0;
    char kind = 0;
    if (PyArg_ParseTuple(plan, "sii", &kind_s, &spw, &slots))
      kind = kind_s[0] == 's' && kind_s[1] == 'p' ? 'p' : kind_s[0];  // owner, slots, sPlit, team, balanced
    Py_DECREF(plan);
    if (!kind) return nullptr;
    P = slots;
    const char* name = window > 0 ? (P <= 1 ? "ps_sw_fused_partitioned" : "ps_sw_partitioned")
                                  : (flat ? "ps_split_reduce" : "ps_small_block");
    if (kind == 'p' || kind == 't') {
      sa.num_workers = spw;
      const int64_t bytes = kind == 't' ? fn.team_bytes(spw) : fn.split_bytes((int)B, (int)H, spw);
      // (w holds the workspace until the launch is issued)
      PyObject* w = PyObject_CallFunction(a[18], "iLLL", rd.dev, (long long)sid, (long long)(B * H), (long long)bytes);
      if (!w) return nullptr;
      unsigned long long sp = 0, sn = 0, cp = 0, cn = 0;
      PyObject* holder;
      if (!PyArg_ParseTuple(w, "KKKKO", &sp, &sn, &cp, &cn, &holder)) {
        Py_DECREF(w);
        return nullptr;
      }
      rc = launch([&] {
        return kind == 't' ? fn.team(&sa, (void*)sp, (int64_t)sn, (int32_t*)cp, (int64_t)cn, s)
                           : fn.split(&sa, (void*)sp, (int64_t)sn, (int32_t*)cp, (int64_t)cn, s);
      });
      Py_DECREF(w);
      if (rc != 0) return failed(rc, kind == 't' ? "pa_fp8_decode_team" : "pa_fp8_decode_split");
      return PyUnicode_FromString(name);
    }
    if (kind == 'b') {
      sa.num_workers = spw;
      const int64_t bytes = fn.balanced_bytes((int)B, (int)H, (int)ql, (int)gqa, sa.num_workers);
      if (bytes <= 0) NOT_HERE;
      const at::Tensor ws = device_bytes(bytes, rd.dev);
      if ((rc = launch([&] { return fn.balanced(&sa, ws.data_ptr(), bytes, s); })) != 0) return failed(rc, "pa_fp8_decode_balanced");
      if ((rc = launch([&] { return fn.merge(&sa, ws.data_ptr(), bytes, s); })) != 0) return failed(rc, "pa_fp8_merge_balanced");
      return PyUnicode_FromString(name);
    }

    // ---- owner launch, or slots and their reduce ----
    const bool owner = kind == 'o';
    if (!owner && kind != 's') NOT_HERE;
    auto partial_shapes = [&]() {
      return shape_is(*part[0], {B, H, P, eq}) && shape_is(*part[1], {B, H, P, eq}) &&
             shape_is(*part[2], {B, H, P, eq, D}) && is(*part[0], at::kFloat) && is(*part[1], at::kFloat) &&
             part[0]->strides() == part[1]->strides() && part[0]->stride(3) == 1 && part[2]->stride(4) == 1 &&
             (is(*part[2], at::kBFloat16) || is(*part[2], at::kFloat));
    };
    if (given == 3 && !partial_shapes()) NOT_HERE;
    if (!owner && given != 0 && given != 3) NOT_HERE;
    if (owner && window == 0) P = spw = (int)std::min<int64_t>(P, 4);
    pa_fp8_partition_args pa;
    std::memset(&pa, 0, sizeof pa);
    pa.abi_version = PA_FP8_ABI_VERSION;
    pa.query = sa.query;
    pa.key_cache = sa.key_cache;
    pa.value_cache = sa.value_cache;
    pa.block_tables = sa.block_tables;
    pa.kv_indptr = sa.kv_indptr;
    pa.stride_bt_seq = sa.stride_bt_seq;
    pa.max_blocks_per_seq = sa.max_blocks_per_seq;
    pa.context_lengths = sa.context_lengths;
    pa.key_scale = sa.key_scale;
    pa.value_scale = sa.value_scale;
    pa.stride_q_tok = sa.stride_q_tok;
    pa.stride_q_head = sa.stride_q_head;
    pa.stride_k_block = sa.stride_k_block;
    pa.stride_k_head = sa.stride_k_head;
    pa.stride_v_block = sa.stride_v_block;
    pa.stride_v_head = sa.stride_v_head;
    pa.stride_ks_block = sa.stride_ks_block;
    pa.stride_ks_head = sa.stride_ks_head;
    pa.num_seqs = sa.num_seqs;
    pa.num_kv_heads = sa.num_kv_heads;
    pa.num_partitions = (int32_t)P;
    pa.query_length = sa.query_length;
    pa.query_group_size = sa.query_group_size;
    pa.head_size = sa.head_size;
    pa.block_size = sa.block_size;
    pa.num_blocks = sa.num_blocks;
    pa.sliding_window = sa.sliding_window;
    pa.per_token_kv = sa.per_token_kv;
    pa.trans_v = sa.trans_v;
    pa.query_dtype = sa.query_dtype;
    pa.softmax_scale = sa.softmax_scale;
    pa.slots_per_workgroup = spw;
    if (owner) {
      pa.output = sa.output;
      pa.output_dtype = od;
      pa.stride_out_tok = sa.stride_out_tok;
      pa.stride_out_head = sa.stride_out_head;
      pa.tmp_dtype = PA_DTYPE_BF16;
      if ((rc = launch([&] { return fn.partition(&pa, s); })) != 0) return failed(rc, "pa_fp8_decode_partition");
      return PyUnicode_FromString(name);
    }
    at::Tensor own[3];
    if (given == 0) {
      const auto f32 = out->options().dtype(at::kFloat);
      own[0] = at::empty({B, H, P, eq}, f32);
      own[1] = at::empty({B, H, P, eq}, f32);
      own[2] = at::empty({B, H, P, eq, D}, f32.dtype(at::kBFloat16));
      for (int i = 0; i < 3; ++i) part[i] = &own[i];
    }
    pa.exp_sums = (float*)part[0]->data_ptr();
    pa.max_logits = (float*)part[1]->data_ptr();
    pa.tmp_out = part[2]->data_ptr();
    pa.stride_es_seq = part[0]->stride(0);
    pa.stride_es_head = part[0]->stride(1);
    pa.stride_es_part = part[0]->stride(2);
    pa.stride_to_seq = part[2]->stride(0);
    pa.stride_to_head = part[2]->stride(1);
    pa.stride_to_part = part[2]->stride(2);
    pa.stride_to_group = part[2]->stride(3);
    pa.tmp_dtype = is(*part[2], at::kFloat) ? PA_DTYPE_F32 : PA_DTYPE_BF16;
    pa_fp8_reduce_args r;
    std::memset(&r, 0, sizeof r);
    r.abi_version = PA_FP8_ABI_VERSION;
    r.output = sa.output;
    r.exp_sums = pa.exp_sums;
    r.max_logits = pa.max_logits;
    r.tmp_out = pa.tmp_out;
    // output [B*ql, Hq, D] addressed as [B, ql, Hkv, gqa, D]
    r.stride_out_seq = ql * sa.stride_out_tok;
    r.stride_out_ql = sa.stride_out_tok;
    r.stride_out_kv_head = gqa * sa.stride_out_head;
    r.stride_out_group = sa.stride_out_head;
    r.stride_es_seq = pa.stride_es_seq;
    r.stride_es_head = pa.stride_es_head;
    r.stride_es_part = pa.stride_es_part;
    r.stride_to_seq = pa.stride_to_seq;
    r.stride_to_head = pa.stride_to_head;
    r.stride_to_part = pa.stride_to_part;
    r.stride_to_group = pa.stride_to_group;
    r.num_seqs = sa.num_seqs;
    r.num_kv_heads = sa.num_kv_heads;
    r.num_partitions = (int32_t)P;
    r.query_length = sa.query_length;
    r.query_group_size = sa.query_group_size;
    r.head_size = sa.head_size;
    r.output_dtype = od;
    r.tmp_dtype = pa.tmp_dtype;
    if ((rc = launch([&] { return fn.partition(&pa, s); })) != 0) return failed(rc, "pa_fp8_decode_partition");
    if ((rc = launch([&] { return fn.reduce(&r, s); })) != 0) return failed(rc, "pa_fp8_decode_reduce");
    return PyUnicode_FromString(name);
  });
}

// ---------------------------------------------------------------------------
// KV-cache writer
// ---------------------------------------------------------------------------

// rope(config, Q, K, V, Positions, CosCache, SinCache, SlotMapping, KeyCache, ValueCache, Q_out, K_out, num_tokens,
//      KScale, VScale); config: (head_dim, q heads, kv heads, block size, flash, bf16, apply_scale, reuse, i64)
PyObject* rope(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 15) NOT_HERE;
  return guarded([&]() -> PyObject* {
    int D, QH, KH, bs, flash, bf16, scaled, reuse, i64;
    if (!PyArg_ParseTuple(a[0], "iiiiiiiii", &D, &QH, &KH, &bs, &flash, &bf16, &scaled, &reuse, &i64)) return nullptr;
    Reader rd;
    const at::Tensor* t[11];
    for (int i = 0; i < 11; ++i) t[i] = rd(a[1 + i]);
    if (!rd.ok || !PyLong_CheckExact(a[12])) NOT_HERE;
    const int64_t T = PyLong_AsLongLong(a[12]);
    if (PyErr_Occurred() || T <= 0 || T > 0x7fffffff) return PyErr_Clear(), Py_NewRef(Py_None);
    const at::Tensor *ks = nullptr, *vs = nullptr;
    if (scaled) {
      ks = rd(a[13]);
      vs = rd(a[14]);
      if (!rd.ok || !is(*ks, at::kFloat) || !is(*vs, at::kFloat) || ks->numel() < 1 || vs->numel() < 1) NOT_HERE;
    }
    const at::Tensor &q = *t[0], &k = *t[1], &v = *t[2], &pos = *t[3], &cos = *t[4], &sin = *t[5], &slot = *t[6],
                     &kc = *t[7], &vc = *t[8], &qo = *t[9], &ko = *t[10];
    const at::ScalarType dt = bf16 ? at::kBFloat16 : at::kHalf, it = i64 ? at::kLong : at::kInt;
    for (const at::Tensor* x : {&q, &qo})
      if (!shape_is(*x, {T, QH, D}) || !is(*x, dt) || x->stride(2) != 1) NOT_HERE;
    for (const at::Tensor* x : {&k, &v, &ko})
      if (!shape_is(*x, {T, KH, D}) || !is(*x, dt) || x->stride(2) != 1) NOT_HERE;
    for (const at::Tensor* x : {&pos, &slot})
      if (!is(*x, it) || x->dim() != 1 || x->size(0) < T || x->stride(0) != 1) NOT_HERE;
    const int64_t cols = reuse ? D / 2 : D;
    for (const at::Tensor* x : {&cos, &sin})
      if (x->dim() != 2 || x->size(1) != cols || !is(*x, dt) || x->stride(1) != 1) NOT_HERE;
    if (cos.size(0) != sin.size(0) || cos.size(0) > 0x7fffffff) NOT_HERE;
    auto cache_dtype = [&](const at::Tensor& x) {
      return scaled ? (is(x, at::kFloat8_e4m3fn) || is(x, at::kByte)) : is(x, dt);
    };
    if (!cache_dtype(kc) || !cache_dtype(vc) || !kc.is_contiguous() || !vc.is_contiguous()) NOT_HERE;
    const int64_t nb = kc.size(0);
    int layout;
    if (flash) {
      if (!shape_is(kc, {nb, bs, KH, D}) || !shape_is(vc, {nb, bs, KH, D})) NOT_HERE;
      layout = PA_CACHE_FLASH;
    } else {
      if (!shape_is(kc, {nb, KH, D / 16, bs, 16})) NOT_HERE;
      if (vc.dim() == 5) {
        if (bs % 16 || !shape_is(vc, {nb, KH, bs / 16, D, 16})) NOT_HERE;
        layout = PA_CACHE_ATOM_TRANS_V;
      } else {
        if (!shape_is(vc, {nb, KH, D, bs})) NOT_HERE;
        layout = PA_CACHE_ATOM;
      }
    }
    if (nb > 0x7fffffff) NOT_HERE;
    hipStream_t s;
    int64_t sid;
    if (!current(rd.dev, &s, &sid)) NOT_HERE;
    pa_fp8_rope_cache_args r;
    std::memset(&r, 0, sizeof r);
    r.abi_version = PA_FP8_ABI_VERSION;
    r.q = q.data_ptr();
    r.k = k.data_ptr();
    r.v = v.data_ptr();
    r.positions = pos.data_ptr();
    r.slot_mapping = slot.data_ptr();
    r.cos_cache = cos.data_ptr();
    r.sin_cache = sin.data_ptr();
    r.key_cache = kc.data_ptr();
    r.value_cache = vc.data_ptr();
    r.q_out = qo.data_ptr();
    r.k_out = ko.data_ptr();
    if (scaled) {
      r.k_scale = (const float*)ks->data_ptr();
      r.v_scale = (const float*)vs->data_ptr();
    }
    r.stride_q_tok = q.stride(0);
    r.stride_q_head = q.stride(1);
    r.stride_k_tok = k.stride(0);
    r.stride_k_head = k.stride(1);
    r.stride_v_tok = v.stride(0);
    r.stride_v_head = v.stride(1);
    r.stride_qo_tok = qo.stride(0);
    r.stride_qo_head = qo.stride(1);
    r.stride_ko_tok = ko.stride(0);
    r.stride_ko_head = ko.stride(1);
    r.stride_cos_pos = cos.stride(0);
    r.stride_sin_pos = sin.stride(0);
    r.num_tokens = (int32_t)T;
    r.num_q_heads = QH;
    r.num_kv_heads = KH;
    r.head_dim = D;
    r.block_size = bs;
    r.num_blocks = (int32_t)nb;
    r.max_pos = (int32_t)cos.size(0);
    r.dtype = bf16 ? PA_DTYPE_BF16 : PA_DTYPE_F16;
    r.cache_layout = layout;
    r.apply_scale = scaled;
    r.reuse_freqs_front_part = reuse;
    r.index_i64 = i64;
    const int rc = launch([&] { return fn.rope(&r, s); });
    if (rc != 0) return failed(rc, "pa_fp8_rope_cache");
    Py_RETURN_TRUE;
  });
}

// ---------------------------------------------------------------------------
// Fused RMSNorm + RoPE + fp8 quant
// ---------------------------------------------------------------------------

// qknr(q, kv, kv_weight, cos, sin, positions, num_q_heads, head_dim, rope_head_dim, q_weight, quant, group, e8m0)
// -> (q_out, kv_out, q_scale, kv_scale); the caller has checked the configuration.
PyObject* qknr(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 13) NOT_HERE;
  return guarded([&]() -> PyObject* {
    Reader rd;
    const at::Tensor *q = rd(a[0]), *kv = rd(a[1]), *kw = rd(a[2]), *cos = rd(a[3]), *sin = rd(a[4]), *pos = rd(a[5]);
    const at::Tensor* qw = a[9] == Py_None ? nullptr : rd(a[9]);
    if (!rd.ok) NOT_HERE;
    int64_t v[5];
    const int at_[5] = {6, 7, 8, 11, 12};
    for (int i = 0; i < 5; ++i) {
      if (!PyLong_CheckExact(a[at_[i]])) NOT_HERE;
      v[i] = PyLong_AsLongLong(a[at_[i]]);
      if (PyErr_Occurred()) return PyErr_Clear(), Py_NewRef(Py_None);
    }
    const int64_t H = v[0], D = v[1], RD = v[2], G = v[3];
    const bool e8 = v[4] != 0, quant = a[10] == Py_True;
    if (H < 0 || D <= 0 || RD < 0 || G <= 0 || D % G) NOT_HERE;
    for (const at::Tensor* x : {q, kv, kw, cos, sin})
      if (!is(*x, at::kBFloat16)) NOT_HERE;
    const int64_t T = q->dim() ? q->size(0) : 0;
    if (T <= 0 || T > 0x7fffffff) NOT_HERE;
    int64_t qstride;
    if (q->dim() == 2) {
      if (q->size(1) != H * D || !q->is_contiguous()) NOT_HERE;
      qstride = H * D;
    } else {
      if (!shape_is(*q, {T, H, D}) || q->stride(2) != 1 || q->stride(1) != D) NOT_HERE;
      qstride = q->stride(0);
    }
    if (kv->dim() != 2 || kv->size(1) != D || kv->size(0) < T || kv->stride(1) != 1 || kv->stride(0) % 2) NOT_HERE;
    if (!is(*pos, at::kLong) || pos->dim() != 1 || pos->size(0) < T || !pos->is_contiguous()) NOT_HERE;
    if (cos->dim() != 2 || cos->size(1) != RD / 2 || cos->sizes() != sin->sizes() || !cos->is_contiguous() ||
        !sin->is_contiguous() || cos->size(0) > 0x7fffffff)
      NOT_HERE;
    if (kw->numel() != D || !kw->is_contiguous()) NOT_HERE;
    if (qw && (!is(*qw, at::kBFloat16) || qw->numel() != D || !qw->is_contiguous())) NOT_HERE;
    hipStream_t s;
    int64_t sid;
    if (!current(rd.dev, &s, &sid)) NOT_HERE;
    const auto opt = q->options();
    const auto od = opt.dtype(quant ? at::kFloat8_e4m3fn : at::kBFloat16);
    const at::Tensor qo = at::empty({T, H, D}, od), ko = at::empty({T, D}, od);
    at::Tensor qs, ks;
    if (quant) {
      const auto sd = opt.dtype(e8 ? at::kByte : at::kFloat);
      qs = at::empty({T, H, D / G}, sd);
      ks = at::empty({T, D / G}, sd);
    }
    pa_qk_norm_rope_args r;
    std::memset(&r, 0, sizeof r);
    r.abi_version = PA_FP8_ABI_VERSION;
    r.q = q->data_ptr();
    r.kv = kv->data_ptr();
    r.q_weight = qw ? qw->data_ptr() : nullptr;
    r.kv_weight = kw->data_ptr();
    r.cos_cache = cos->data_ptr();
    r.sin_cache = sin->data_ptr();
    r.positions = (decltype(r.positions))pos->data_ptr();
    r.q_out = qo.data_ptr();
    r.kv_out = ko.data_ptr();
    if (quant) {
      r.q_scale = qs.data_ptr();
      r.kv_scale = ks.data_ptr();
    }
    r.stride_q_tok = qstride;
    r.stride_kv_tok = kv->stride(0);
    r.num_tokens = (int32_t)T;
    r.num_q_heads = (int32_t)H;
    r.head_dim = (int32_t)D;
    r.rope_head_dim = (int32_t)RD;
    r.max_pos = (int32_t)cos->size(0);
    r.quant = quant;
    r.group_size = (int32_t)G;
    r.scale_e8m0 = quant && e8;
    const int rc = launch([&] { return fn.qknr(&r, s); });
    if (rc != 0) return failed(rc, "pa_fp8_qk_norm_rope_quant");
    PyObject* out = PyTuple_New(4);
    if (!out) return nullptr;
    PyTuple_SET_ITEM(out, 0, THPVariable_Wrap(qo));
    PyTuple_SET_ITEM(out, 1, THPVariable_Wrap(ko));
    PyTuple_SET_ITEM(out, 2, quant ? THPVariable_Wrap(qs) : Py_NewRef(Py_None));
    PyTuple_SET_ITEM(out, 3, quant ? THPVariable_Wrap(ks) : Py_NewRef(Py_None));
    return out;
  });
}

// ---------------------------------------------------------------------------
// MLA decode and reduce
// ---------------------------------------------------------------------------

constexpr int64_t kMlaHeads = 128, kMlaQk = 576, kMlaV = 512;

// mla_decode(query, kv_buffer, kv_page_indices, work_indptr, work_info_set, final_output, split_output, split_lse,
//            softmax_scale, precise)
PyObject* mla_decode(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 10) NOT_HERE;
  return guarded([&]() -> PyObject* {
    Reader rd;
    const at::Tensor* t[8];
    for (int i = 0; i < 8; ++i) t[i] = rd(a[i]);
    if (!rd.ok || !PyFloat_CheckExact(a[8])) NOT_HERE;
    const at::Tensor &q = *t[0], &kv = *t[1], &idx = *t[2], &wp = *t[3], &wi = *t[4], &fo = *t[5], &so = *t[6],
                     &sl = *t[7];
    if (q.dim() != 3 || !is(q, at::kFloat8_e4m3fn) || !is(kv, at::kFloat8_e4m3fn) || q.size(0) == 0) NOT_HERE;
    const int64_t R = q.size(0), np = so.dim() ? so.size(0) : 0;
    if (!shape_is(q, {R, kMlaHeads, kMlaQk}) || kv.dim() != 4 || kv.size(1) * kv.size(2) != 1 || kv.size(3) != kMlaQk ||
        !shape_is(fo, {R, kMlaHeads, kMlaV}) || !shape_is(so, {np, 1, kMlaHeads, kMlaV}) ||
        !shape_is(sl, {np, 1, kMlaHeads, 1}))
      NOT_HERE;
    for (int i = 0; i < 8; ++i)
      if (!t[i]->is_contiguous()) NOT_HERE;
    if (!is(fo, at::kBFloat16) || !is(so, at::kFloat) || !is(sl, at::kFloat) || !is(idx, at::kInt) ||
        !is(wp, at::kInt) || !is(wi, at::kInt))
      NOT_HERE;
    const int64_t lim = 0x7fffffff;
    if (R > lim || np > lim || idx.numel() > lim || wi.numel() > lim || wp.numel() < 1) NOT_HERE;
    hipStream_t s;
    int64_t sid;
    if (!current(rd.dev, &s, &sid)) NOT_HERE;
    pa_mla_decode_args r;
    std::memset(&r, 0, sizeof r);
    r.abi_version = PA_FP8_ABI_VERSION;
    r.query = q.data_ptr();
    r.kv_buffer = kv.data_ptr();
    r.kv_page_indices = (const int32_t*)idx.data_ptr();
    r.work_indptr = (const int32_t*)wp.data_ptr();
    r.work_info = (const int32_t*)wi.data_ptr();
    r.final_output = fo.data_ptr();
    r.split_output = np > 0 ? (float*)so.data_ptr() : nullptr;
    r.split_lse = np > 0 ? (float*)sl.data_ptr() : nullptr;
    r.num_pages = kv.size(0);
    r.num_page_indices = (int32_t)idx.numel();
    r.num_rows = (int32_t)R;
    r.num_workers = (int32_t)(wp.numel() - 1);
    r.num_works = (int32_t)(wi.numel() / 8);
    r.num_partial = (int32_t)np;
    r.softmax_scale = (float)PyFloat_AS_DOUBLE(a[8]);
    r.precise_p = a[9] == Py_True;
    const int rc = launch([&] { return fn.mla_decode(&r, s); });
    if (rc != 0) return failed(rc, "pa_fp8_mla_decode");
    Py_RETURN_TRUE;
  });
}

// mla_reduce(partial_output, partial_lse, reduce_indptr, reduce_final_map, reduce_partial_map, final_output)
PyObject* mla_reduce(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 6) NOT_HERE;
  return guarded([&]() -> PyObject* {
    Reader rd;
    const at::Tensor* t[6];
    for (int i = 0; i < 6; ++i) {
      t[i] = rd(a[i]);
      if (!rd.ok || !t[i]->is_contiguous()) NOT_HERE;
    }
    const at::Tensor &po = *t[0], &pl = *t[1], &ri = *t[2], &rf = *t[3], &rp = *t[4], &fo = *t[5];
    if (!is(po, at::kFloat) || !is(pl, at::kFloat) || !is(fo, at::kBFloat16) || !is(ri, at::kInt) ||
        !is(rf, at::kInt) || !is(rp, at::kInt))
      NOT_HERE;
    const int64_t lim = 0x7fffffff;
    if (fo.dim() < 2 || fo.size(-1) != kMlaV || fo.size(-2) != kMlaHeads || ri.numel() < 1 ||
        rf.numel() < 2 * (ri.numel() - 1) || po.numel() / (kMlaHeads * kMlaV) > lim || rp.numel() > lim)
      NOT_HERE;
    hipStream_t s;
    int64_t sid;
    if (!current(rd.dev, &s, &sid)) NOT_HERE;
    pa_mla_reduce_args r;
    std::memset(&r, 0, sizeof r);
    r.abi_version = PA_FP8_ABI_VERSION;
    r.split_output = (const float*)po.data_ptr();
    r.split_lse = (const float*)pl.data_ptr();
    r.reduce_indptr = (const int32_t*)ri.data_ptr();
    r.reduce_final_map = (const int32_t*)rf.data_ptr();
    r.reduce_partial_map = (const int32_t*)rp.data_ptr();
    r.final_output = fo.data_ptr();
    r.num_groups = (int32_t)(ri.numel() - 1);
    r.num_partial = (int32_t)(po.numel() / (kMlaHeads * kMlaV));
    r.num_partial_map = (int32_t)rp.numel();
    r.num_rows = (int32_t)(fo.numel() / (kMlaHeads * kMlaV));
    const int rc = launch([&] { return fn.mla_reduce(&r, s); });
    if (rc != 0) return failed(rc, "pa_fp8_mla_reduce");
    Py_RETURN_TRUE;
  });
}

// init(addresses in the order of Entry's fields, check): the entry points of
// the loaded library.
PyObject* init(PyObject*, PyObject* args) {
  PyObject *addrs, *check;
  if (!PyArg_ParseTuple(args, "O!O", &PyTuple_Type, &addrs, &check)) return nullptr;
  constexpr Py_ssize_t kEntries = sizeof(Entry) / sizeof(void*);
  if (PyTuple_GET_SIZE(addrs) != kEntries) {
    PyErr_SetString(PyExc_ValueError, "one address per entry point");
    return nullptr;
  }
  void** at = reinterpret_cast<void**>(&fn);
  for (Py_ssize_t i = 0; i < kEntries; ++i) {
    at[i] = PyLong_AsVoidPtr(PyTuple_GET_ITEM(addrs, i));
    if (!at[i]) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "null entry point");
      return nullptr;
    }
  }
  Py_XDECREF(check_fn);
  check_fn = Py_NewRef(check);
  ready = true;
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"init", init, METH_VARARGS, nullptr},
    {"pa_decode", (PyCFunction)(void (*)(void))pa_decode, METH_FASTCALL, nullptr},
    {"rope", (PyCFunction)(void (*)(void))rope, METH_FASTCALL, nullptr},
    {"qknr", (PyCFunction)(void (*)(void))qknr, METH_FASTCALL, nullptr},
    {"mla_decode", (PyCFunction)(void (*)(void))mla_decode, METH_FASTCALL, nullptr},
    {"mla_reduce", (PyCFunction)(void (*)(void))mla_reduce, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) { return PyModule_Create(&module); }
