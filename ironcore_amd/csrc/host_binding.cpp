// The call path of the attention layer and of the tensor-level wrappers, native:
// shape checks, strides, output and workspace allocation and the C-ABI calls,
// without the interpreter in between.  A cached decode step of a small model is
// bound by this path (three launches of a few microseconds each behind 33 us of
// Python on one core); the functions here leave 2-3 us of it.
//
// Each function handles the ordinary case completely, or returns None: the Python
// wrapper (paged_ops.py, layers/attention.py) then takes its own path, which makes
// tensors contiguous, switches the device or names what is wrong with the arguments.
// What a layer call's attention does not take is looked for before its append is
// launched; where only the library's own limits refuse it (2^31 rows, a 4 GiB block),
// the append has been made, and the wrapper makes it again, the same rows into the
// same slots.  Nothing is kept between calls: outputs and
// workspaces come from torch's allocator, which orders their reuse on the stream
// and serves a capturing stream from the graph's own pool.
#include <torch/extension.h>

#include <ATen/TensorSubclassLikeUtils.h>
#include <ATen/autocast_mode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>

#include <algorithm>
#include <atomic>
#include <climits>

#include "../../include/ironcore_paged.h"

namespace {

using at::Tensor;
using OptTensor = c10::optional<Tensor>;
namespace py = pybind11;

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kBFloat16: return IC_DTYPE_BF16;
    case at::kHalf: return IC_DTYPE_F16;
    case at::kFloat: return IC_DTYPE_F32;
    default: return -1;
  }
}

// Whether a library call was made: false for arguments that it does not take, which the Python wrapper then handles
// or refuses by name.  A launch that failed is raised from here, as _lib.PagedLibraryError: the library has read (and
// so cleared) HIP's last error, and a second try by the wrapper would hide it.
bool made(const char *func, int rc) {
  if (rc == IC_ERR_LAUNCH) {
    py::gil_scoped_acquire gil;
    py::module_::import("ironcore_amd._lib").attr("check")(func, rc);
  }
  return rc == IC_OK;
}

bool on(const Tensor &t, int64_t device) { return t.is_cuda() && t.get_device() == device; }

struct Pool {
  int64_t nb, gn, bs, hd, sb, sh, st;
  int dtype;
  const void *k, *v;
  bool ok = false;
  Pool(const Tensor &kp, const Tensor &vp, int64_t device) {
    if (kp.dim() != 4 || !on(kp, device) || !on(vp, device) || kp.scalar_type() != vp.scalar_type() ||
        kp.sizes() != vp.sizes() || kp.strides() != vp.strides() || kp.stride(3) != 1)
      return;
    nb = kp.size(0), gn = kp.size(1), bs = kp.size(2), hd = kp.size(3);
    sb = kp.stride(0), sh = kp.stride(1), st = kp.stride(2);
    dtype = dtype_code(kp.scalar_type());
    k = kp.data_ptr(), v = vp.data_ptr();
    ok = dtype >= 0 && gn > 0;
  }
  bool attends() const { return hd == 32 || hd == 64 || hd == 128; }
};

bool index_vector(const Tensor &t, at::ScalarType type, int64_t n, int64_t device) {
  return on(t, device) && t.scalar_type() == type && t.numel() == n && t.is_contiguous();
}
bool table(const Tensor &t, int64_t rows, int64_t device) {
  return on(t, device) && t.scalar_type() == at::kInt && t.dim() == 2 && t.size(0) == rows && t.stride(1) == 1;
}

// [n, heads, hd] rows, heads contiguous within a row.
bool rows3(const Tensor &t, int64_t heads, int64_t hd) {
  return t.dim() == 3 && t.size(1) == heads && t.size(2) == hd && t.stride(2) == 1 && t.stride(1) == hd;
}
// [b, s, heads, hd] that is [b*s, heads, hd] rows at one stride.
bool rows4(const Tensor &t, int64_t b, int64_t s, int64_t heads, int64_t hd) {
  return t.dim() == 4 && t.size(0) == b && t.size(1) == s && t.size(2) == heads && t.size(3) == hd &&
         t.stride(3) == 1 && t.stride(2) == hd && (b == 1 || t.stride(0) == s * t.stride(1));
}
// The same where one row a sequence may come at any stride.  With s == 1 the stride of that dimension says nothing (half of a
// projection's row, as a decode step hands it over, keeps the half's length there).
bool step_rows4(const Tensor &t, int64_t b, int64_t s, int64_t heads, int64_t hd) {
  return rows4(t, b, s, heads, hd) || (s == 1 && t.dim() == 4 && t.size(0) == b && t.size(1) == 1 && t.size(2) == heads &&
                                       t.size(3) == hd && t.stride(3) == 1 && t.stride(2) == hd);
}
int64_t row_stride4(const Tensor &t) { return t.size(1) > 1 ? t.stride(1) : t.stride(0); }

// Rows that a kernel reads in 16-byte pieces, `row` elements each.
bool rows16(const void *p, int64_t stride, int64_t row, int64_t element_size) {
  return reinterpret_cast<uintptr_t>(p) % 16 == 0 && (stride * element_size) % 16 == 0 && stride >= row;
}

bool append_rows(const void *k, const void *v, int64_t stride, const Pool &p, const Tensor &slots, int64_t n,
                 void *stream) {
  return made("ic_kv_append",
              ic_kv_append(k, v, stride, const_cast<void *>(p.k), const_cast<void *>(p.v), p.sb, p.sh, p.st,
                           slots.data_ptr<int64_t>(), n, (int)p.gn, (int)p.hd, (int)p.bs, p.nb, p.dtype, stream));
}

struct Decode {
  const Tensor &tables, &lens;
  int64_t max_ctx, min_chunk, cohort;
  const OptTensor &shared;
  double scale;
};

bool decode_fits(const Pool &p, int64_t b, int64_t hn, const Decode &d, int64_t device) {
  if (!p.attends() || hn % p.gn != 0 || b == 0 || !table(d.tables, b, device) ||
      !index_vector(d.lens, at::kInt, b, device) || d.max_ctx > d.tables.size(1) * p.bs || d.cohort < 1 ||
      p.bs % 16 != 0 ||
      ic_paged_decode_shared_workspace_bytes((int)b, (int)hn, (int)p.gn, (int)p.hd, (int)d.cohort) == 0)
    return false;
  return d.cohort == 1 ||
         (d.shared.has_value() && index_vector(*d.shared, at::kInt, (b + d.cohort - 1) / d.cohort, device));
}

// Whether a cohort's shared blocks are worth reading once.  What its members read again then comes from the cache while all
// of it fits there (256 MB, beside other data), and without cohorts there is no second phase, the grid fits the rows and small
// batches take one launch with the append.  us of a layer call with cohorts / without, prompts x samples, prefix + suffix:
//   16 / 4 heads of 128    22 x 16, 80 + 232       225 MB    40.4 / 29.5        21 x 16, 1 680 + 120     1 239    45.8 / 87.2
//                          4 x 4, 160 + 41           7       20.4 / 9.9         10 x 16, 816 + 467         420    40.2 / 34.3
//   32 / 8 of 128          12 x 4, 80 + 55          27       24.3 / 17.7        30 x 8, 240 + 451          679    68.1 / 64.9
//   12 / 12 of 128         3 x 8, 384 + 289         99       30.4 / 13.3        4 x 4, 2 256 + 55          227    35.1 / 42.6
//                          14 x 4, 240 + 672       313       41.7 / 31.1        29 x 4, 736 + 43           555    41.4 / 47.0
//   28 / 4 of 128          29 x 4, 80 + 62          34       26.1 / 19.7        32 x 16, 1 024 + 1 024   2 147    153 / 197
//   28 / 4 of 64           32 x 16, 160 + 45       107       28.9 / 28.4        3 x 16, 80 + 753            41    26.7 / 27.0
// Between 200 and 700 MB either may be faster; the line is where none of 64 was slower by more than a percent.  (Passes over one
// layer's pools, which stay in that cache.  With 1.2 GB of pools in turn: 138 MB 36.4 / 28.2, 251 MB 34.3 / 31.4, 7 MB 25.1 / 17.2, and
// in a model's step, us a layer, 147 MB 127 / 119, 21 MB 69 / 62: the line stays.)
// At head dim 64 a cohort of more than 64 query rows is the exception: it fills both of the kernel's column tiles and all eight waves,
// while the plain call, where it is not the pair kernel (decode_takes_pairs), streams grouped heads of 64 at half its rate.
// Hot and cold, from three quarters of the CUs in pairs on (fewer leave CUs for the plain call's splits):
//   28 / 4 of 64           10 x 16, 576 + 36    100 MB    25.6 / 28.5   27.4 / 30.1       3 x 16, 912 + 40    47    25.6 / 27.8   27.0 / 28.8
//                          5 x 10, 576 + 36      31       23.4 / 27.8   24.7 / 28.8       5 x 16, 160 + 400   46    27.4 / 25.4   29.1 / 27.1
//                          2 x 16, 576 + 36      20       26.0 / 25.1   27.4 / 25.8       2 x 16, 1 504 + 100 53    29.2 / 20.0   30.3 / 21.0
//                          30 x 8, 400 + 40     108       36.1 / 28.0   38.2 / 30.7       20 x 4, 304 + 60    30    36.0 / 24.5   38.3 / 25.7
//   64 / 8 of 64           2 x 16, 576 + 36      40       24.4 / 29.8   25.4 / 30.9       2 x 10, 912 + 36    39    28.4 / 26.8   29.4 / 28.0
//   32 / 8 of 64           3 x 24, 576 + 36      90       23.7 / 27.1   25.2 / 28.5       2 x 32, 576 + 36    80    24.7 / 19.4   26.2 / 19.6
//   12 / 4 of 64           6 x 24, 576 + 36      90       23.7 / 26.9   25.0 / 28.3       3 x 24, 576 + 36    45    24.2 / 18.9   25.6 / 18.8
//   16 / 8 of 64           3 x 64, 320 + 36     140       26.6 / 18.8   28.0 / 20.6
//   28 / 4 of 32           10 x 16, 304 + 36     28       34.7 / 24.3   36.4 / 25.0
bool cohorts_pay(int64_t b, int64_t hn, int64_t gn, int64_t hd, int64_t max_ctx, int64_t cohort, int64_t element_size) {
  if (cohort <= 1 || gn < 1) return false;
  if (b * max_ctx * gn * hd * 2 * element_size > 192000000) return true;
  const int64_t group = hn / gn, pairs = b * gn;
  const bool pair_kernel = group <= 2 ? max_ctx <= 2048 : group <= 4 && max_ctx <= 1024 && pairs <= 512;
  return hd == 64 && cohort * group > 64 && pairs >= 192 && !pair_kernel;
}

bool decode(const Tensor &out, const void *q, int64_t q_stride, const Pool &p, int64_t b, int64_t hn, const Decode &d,
            void *stream) {
  const size_t need = ic_paged_decode_shared_workspace_bytes((int)b, (int)hn, (int)p.gn, (int)p.hd, (int)d.cohort);
  const Tensor ws = at::empty({(int64_t)need}, out.options().dtype(at::kByte));
  return made("ic_paged_decode_shared",
              ic_paged_decode_shared(out.data_ptr(), out.stride(0), q, q_stride, p.k, p.v, p.sb, p.sh, p.st,
                                     d.tables.data_ptr<int32_t>(), d.tables.stride(0), d.lens.data_ptr<int32_t>(),
                                     (int)b, (int)hn, (int)p.gn, (int)p.hd, (int)p.bs, p.nb, (int)d.max_ctx,
                                     (float)d.scale, (int)d.min_chunk, (int)d.cohort,
                                     d.cohort > 1 ? d.shared->data_ptr<int32_t>() : nullptr, ws.data_ptr(), need,
                                     p.dtype, stream));
}

// ---- tensor-level calls (paged_ops) ----------------------------------------------------------

bool kv_append(const Tensor &k_new, const Tensor &v_new, const Tensor &k_pool, const Tensor &v_pool,
               const Tensor &slots, int64_t device, int64_t stream) {
  const Pool p(k_pool, v_pool, device);
  if (!p.ok || !rows3(k_new, p.gn, p.hd) || !rows3(v_new, p.gn, p.hd) || k_new.size(0) != v_new.size(0) ||
      k_new.stride(0) != v_new.stride(0) || k_new.scalar_type() != k_pool.scalar_type() ||
      v_new.scalar_type() != k_pool.scalar_type() || !on(k_new, device) || !on(v_new, device) ||
      !index_vector(slots, at::kLong, k_new.size(0), device))
    return false;
  return append_rows(k_new.data_ptr(), v_new.data_ptr(), k_new.stride(0), p, slots, k_new.size(0), (void *)stream);
}

OptTensor paged_decode(const Tensor &query, const Tensor &k_pool, const Tensor &v_pool, const Tensor &tables,
                       const Tensor &lens, int64_t max_ctx, double scale, const OptTensor &out_given,
                       int64_t min_chunk, int64_t cohort, const OptTensor &shared, int64_t device, int64_t stream) {
  const Pool p(k_pool, v_pool, device);
  if (!p.ok || query.dim() != 3 || !rows3(query, query.size(1), p.hd) || !on(query, device) ||
      query.scalar_type() != k_pool.scalar_type())
    return c10::nullopt;
  const int64_t b = query.size(0), hn = query.size(1);
  const Decode d{tables, lens, max_ctx, min_chunk, cohort, shared, scale};
  if (!decode_fits(p, b, hn, d, device)) return c10::nullopt;
  if (out_given.has_value() &&
      (out_given->dim() != 2 || out_given->size(0) != b || out_given->size(1) != hn * p.hd ||
       out_given->scalar_type() != query.scalar_type() || out_given->stride(1) != 1 || !on(*out_given, device)))
    return c10::nullopt;
  const Tensor out = out_given.has_value() ? *out_given : at::empty({b, hn * p.hd}, query.options());
  if (!decode(out, query.data_ptr(), query.stride(0), p, b, hn, d, (void *)stream)) return c10::nullopt;
  return out;
}

// ---- the layer -----------------------------------------------------------------------------

// Rotary tables and the table row of each of n tokens; `on` is false without rotary embeddings.
struct Rope {
  bool used = false, ok = true;
  const int32_t *positions = nullptr;
  const float *cos = nullptr, *sin = nullptr;
  int64_t rows = 0;
  Rope(const OptTensor &pos, const OptTensor &c, const OptTensor &s, int64_t n, int64_t hd, int64_t device) {
    if (!c.has_value()) return;
    used = true;
    ok = pos.has_value() && s.has_value() && index_vector(*pos, at::kInt, n, device) && c->dim() == 2 &&
         c->size(1) == hd / 2 && c->sizes() == s->sizes() && index_vector(*c, at::kFloat, c->numel(), device) &&
         index_vector(*s, at::kFloat, c->numel(), device);
    if (!ok) return;
    positions = pos->data_ptr<int32_t>();
    cos = c->data_ptr<float>(), sin = s->data_ptr<float>();
    rows = c->size(0);
  }
};

// The new rows of a layer call: query [b, s, hn, hd], key and value [b, s, gn, hd], a slot for each.
struct NewRows {
  int64_t b = 0, s = 0, hn = 0;
  bool ok = false;
  NewRows(const Tensor &query, const Tensor &key, const Tensor &value, const Pool &p, at::ScalarType type,
          int64_t device) {
    if (query.dim() != 4) return;
    b = query.size(0), s = query.size(1), hn = query.size(2);
    ok = step_rows4(query, b, s, hn, p.hd) && step_rows4(key, b, s, p.gn, p.hd) && step_rows4(value, b, s, p.gn, p.hd) &&
         row_stride4(key) == row_stride4(value) && query.scalar_type() == type && key.scalar_type() == type &&
         value.scalar_type() == type && on(query, device) && on(key, device) && on(value, device) && b * s > 0;
  }
};

// Append with the keys rotated on their way, the query into a tensor of its own.
bool rope_append(const Tensor &key, const Tensor &value, const Pool &p, const Tensor &slots, const Rope &r, int64_t n,
                 void *q_out, const void *q, int64_t q_stride, int64_t hn, void *stream) {
  return made("ic_rope_kv_append_to",
              ic_rope_kv_append_to(q_out, hn * p.hd, q, q_stride, (int)hn, key.data_ptr(),
                                   value.data_ptr(), row_stride4(key), const_cast<void *>(p.k),
                                   const_cast<void *>(p.v), p.sb, p.sh, p.st, slots.data_ptr<int64_t>(), r.positions,
                                   r.cos, r.sin, r.rows, n, (int)p.gn, (int)p.hd, (int)p.bs, p.nb, p.dtype, stream));
}

// One cached decode step of a layer (sq == 1): append and attention in one launch where the library takes both together
// (small batches of short contexts), else one after the other, with rotary tables the query rotated into a tensor of its
// own and the keys on their way into the pool.
OptTensor decode_step(const Tensor &query, const Tensor &key, const Tensor &value, const Tensor &k_pool,
                      const Tensor &v_pool, const Tensor &tables, const Tensor &lens, const Tensor &slots,
                      int64_t max_ctx, double scale, int64_t cohort, const OptTensor &shared,
                      const OptTensor &positions, const OptTensor &cos, const OptTensor &sin, int64_t device,
                      int64_t stream) {
  const Pool p(k_pool, v_pool, device);
  if (!p.ok) return c10::nullopt;
  const NewRows in(query, key, value, p, k_pool.scalar_type(), device);
  if (!in.ok || in.s != 1 || !index_vector(slots, at::kLong, in.b, device)) return c10::nullopt;
  const Decode asked{tables, lens, max_ctx, 0, cohort, shared, scale};
  const Rope rope(positions, cos, sin, in.b, p.hd, device);
  if (!rope.ok || !decode_fits(p, in.b, in.hn, asked, device)) return c10::nullopt;
  if (!cohorts_pay(in.b, in.hn, p.gn, p.hd, max_ctx, cohort, query.element_size())) cohort = 1;
  const Decode d{tables, lens, max_ctx, 0, cohort, shared, scale};
  const void *q = query.data_ptr();
  int64_t q_stride = row_stride4(query);
  if (!rows16(q, q_stride, in.hn * p.hd, query.element_size())) return c10::nullopt;
  const Tensor out = at::empty({in.b, 1, in.hn * p.hd}, query.options());
  if (cohort == 1 && rows16(key.data_ptr(), row_stride4(key), p.gn * p.hd, key.element_size()) &&
      rows16(value.data_ptr(), row_stride4(value), p.gn * p.hd, key.element_size())) {
    ic_decode_append_call c = {};
    c.out = out.data_ptr(), c.out_stride_seq = in.hn * p.hd;
    c.q = q, c.q_stride_seq = q_stride;
    c.k_new = key.data_ptr(), c.v_new = value.data_ptr(), c.new_stride_token = row_stride4(key);
    c.k_pool = const_cast<void *>(p.k), c.v_pool = const_cast<void *>(p.v);
    c.pool_stride_block = p.sb, c.pool_stride_head = p.sh, c.pool_stride_token = p.st, c.num_blocks = p.nb;
    c.block_tables = tables.data_ptr<int32_t>(), c.block_table_stride = tables.stride(0);
    c.context_lens = lens.data_ptr<int32_t>(), c.slot_mapping = slots.data_ptr<int64_t>();
    c.positions = rope.positions, c.cos_table = rope.cos, c.sin_table = rope.sin, c.table_rows = rope.rows;
    c.n_seqs = (int)in.b, c.hn = (int)in.hn, c.gn = (int)p.gn, c.hd = (int)p.hd, c.block_size = (int)p.bs;
    c.max_context_len = (int)max_ctx, c.scale = (float)scale, c.dtype = p.dtype;
    if (made("ic_paged_decode_append", ic_paged_decode_append(&c, (void *)stream))) return out;
  }
  Tensor rotated;
  if (rope.used) {
    rotated = at::empty({in.b, in.hn * p.hd}, query.options());
    if (!rope_append(key, value, p, slots, rope, in.b, rotated.data_ptr(), q, q_stride, in.hn, (void *)stream))
      return c10::nullopt;
    q = rotated.data_ptr();
    q_stride = in.hn * p.hd;
  } else if (!append_rows(key.data_ptr(), value.data_ptr(), row_stride4(key), p, slots, in.b, (void *)stream)) {
    return c10::nullopt;
  }
  if (!decode(out, q, q_stride, p, in.b, in.hn, d, (void *)stream)) return c10::nullopt;
  return out;
}

ic_prefill_call prefill_call(const Tensor &out, const Tensor &query, const Pool &p, int64_t b, int64_t s, int64_t hn,
                             double scale, bool causal) {
  ic_prefill_call c = {};
  c.out = out.data_ptr();
  c.out_stride_token = hn * p.hd;
  c.q = query.data_ptr();
  c.q_stride_token = row_stride4(query);
  c.k_pool = p.k, c.v_pool = p.v;
  c.pool_stride_block = p.sb, c.pool_stride_head = p.sh, c.pool_stride_token = p.st;
  c.n_seqs = (int)b, c.max_chunk_len = (int)s;
  c.hn = (int)hn, c.gn = (int)p.gn, c.hd = (int)p.hd;
  c.block_size = (int)p.bs, c.num_blocks = p.nb;
  c.scale = (float)scale, c.causal = causal, c.dtype = p.dtype;
  return c;
}

// A chunk of new tokens per sequence: append, then attend.  `bounds` int32 [b + 1] holds the bounds of the
// packed chunks; chunks of unequal length come with the rows of the padded tensors they are (int64, any
// placement), whose other rows are padding: slot -1, output zero.  The query is rotated inside the attention
// kernel.  `max_ctx`: no context is longer (0: not known).
OptTensor prefill_step(const Tensor &query, const Tensor &key, const Tensor &value, const Tensor &k_pool,
                       const Tensor &v_pool, const Tensor &tables, const Tensor &lens, const Tensor &slots,
                       const OptTensor &bounds, const OptTensor &rows, int64_t longest, double scale,
                       const OptTensor &positions, const OptTensor &cos, const OptTensor &sin, int64_t device,
                       int64_t stream, int64_t max_ctx) {
  const Pool p(k_pool, v_pool, device);
  if (!p.ok || !p.attends()) return c10::nullopt;
  const NewRows in(query, key, value, p, k_pool.scalar_type(), device);
  if (!in.ok || in.hn % p.gn != 0 || !index_vector(slots, at::kLong, in.b * in.s, device) ||
      !table(tables, in.b, device) || !index_vector(lens, at::kInt, in.b, device) ||
      (bounds.has_value() ? !index_vector(*bounds, at::kInt, in.b + 1, device) : rows.has_value() || longest != in.s) ||
      longest > in.s || in.b * in.s > INT_MAX ||
      !rows16(query.data_ptr(), row_stride4(query), in.hn * p.hd, query.element_size()) ||
      (p.dtype != IC_DTYPE_F32 && p.bs % 16 != 0 && tables.stride(0) != 1) ||  // 16 bits: whole groups of 16 rows
      (rows.has_value() && (rows->numel() == 0 || !index_vector(*rows, at::kLong, rows->numel(), device))))
    return c10::nullopt;
  const Rope rope(positions, cos, sin, in.b * in.s, p.hd, device);
  if (!rope.ok) return c10::nullopt;
  const Tensor out = at::empty({in.b, in.s, in.hn * p.hd}, query.options());
  ic_prefill_call c = prefill_call(out, query, p, in.b, longest, in.hn, scale, true);
  ic_append_call ap = {};
  ap.k_new = key.data_ptr(), ap.v_new = value.data_ptr(), ap.new_stride_token = row_stride4(key);
  ap.k_pool = const_cast<void *>(p.k), ap.v_pool = const_cast<void *>(p.v);
  ap.pool_stride_block = p.sb, ap.pool_stride_head = p.sh, ap.pool_stride_token = p.st, ap.num_blocks = p.nb;
  ap.slot_mapping = slots.data_ptr<int64_t>(), ap.n_tokens = in.b * in.s;
  ap.gn = (int)p.gn, ap.hd = (int)p.hd, ap.block_size = (int)p.bs, ap.dtype = p.dtype;
  ap.positions = rope.positions, ap.cos_table = rope.cos, ap.sin_table = rope.sin, ap.table_rows = rope.rows;
  if (rows.has_value()) {  // the rows that no chunk holds become zeros beside the append
    c.rows = ap.rows = rows->data_ptr<int64_t>();
    c.n_rows = ap.n_rows = rows->numel(), c.q_rows = in.b * in.s;
    ap.zero_out = out.data_ptr();
    ap.zero_row_bytes = (int)(in.hn * p.hd * query.element_size()), ap.zero_stride_bytes = ap.zero_row_bytes;
    ap.bounds = bounds->data_ptr<int32_t>(), ap.n_seqs = (int)in.b, ap.row_pitch = (int)in.s;
  }
  if (!made("ic_append_chunks", ic_append_chunks(&ap, (void *)stream))) return c10::nullopt;
  c.block_tables = tables.data_ptr<int32_t>();
  c.block_table_stride = tables.stride(0);
  c.context_lens = lens.data_ptr<int32_t>();
  c.uniform_context = (int)std::clamp<int64_t>(max_ctx, 0, INT_MAX);
  if (bounds.has_value())
    c.cu_seqlens_q = bounds->data_ptr<int32_t>();
  else
    c.row_pitch = in.s;  // chunks of one length
  c.positions = rope.positions;
  c.cos_table = rope.cos, c.sin_table = rope.sin, c.table_rows = rope.rows;
  if (!made("ic_paged_prefill_ex", ic_paged_prefill_ex(&c, (void *)stream))) return c10::nullopt;
  return out;
}

// A byte mask [1 or b, 1 or hn, sq, sk] (nonzero = visible) packed for the prefill kernels: (bits, lists,
// flags), see ic_mask_pack.  The flags are still on the device.
c10::optional<std::tuple<Tensor, Tensor, Tensor>> pack_mask(const Tensor &mask, int64_t device, int64_t stream) {
  if (mask.dim() != 4 || mask.scalar_type() != at::kByte || !on(mask, device) || mask.numel() == 0 ||
      mask.stride(3) != 1)
    return c10::nullopt;
  const int64_t n = mask.size(0), heads = mask.size(1), rows = mask.size(2), keys = mask.size(3);
  const int64_t qtiles = (rows + 127) / 128, tiles = (keys + 63) / 64;
  const Tensor bits = at::empty({n * heads, qtiles * 4, tiles, 32}, mask.options().dtype(at::kLong));
  const Tensor lists = at::empty({n * heads, qtiles, tiles + 1}, mask.options().dtype(at::kInt));
  const Tensor flags = at::ones({2}, mask.options().dtype(at::kInt));
  if (!made("ic_mask_pack",
            ic_mask_pack(mask.data_ptr<uint8_t>(), mask.stride(0), mask.stride(1), mask.stride(2), (int)n, (int)heads,
                         (int)rows, (int)keys, reinterpret_cast<uint64_t *>(bits.data_ptr<int64_t>()),
                         lists.data_ptr<int32_t>(), flags.data_ptr<int32_t>(), (void *)stream)))
    return c10::nullopt;
  return std::make_tuple(bits, lists, flags);
}

// [b, s, heads, hd] row by row, the strides of size-1 dimensions included (is_contiguous() lets those be anything).
Tensor row_major(const Tensor &t) {
  const auto s = t.sizes(), st = t.strides();
  if (st[3] == 1 && st[2] == s[3] && st[1] == s[2] * s[3] && st[0] == s[1] * s[2] * s[3]) return t;
  return t.clone(at::MemoryFormat::Contiguous);
}

struct DenseMask {
  bool causal;
  const OptTensor &bits, &lists;  // packed: seqs x heads planes (1 or b, 1 or hn)
  int64_t seqs, heads;
};

// The dense call on tensors as they lie: the kernel walks key and value as a pool of one block per sequence, at
// whatever strides they share.
OptTensor dense_as_laid(const Tensor &query, const Tensor &key, const Tensor &value, const DenseMask &m, double scale,
                        int64_t device, void *stream) {
  const Pool p(key.permute({0, 2, 1, 3}), value.permute({0, 2, 1, 3}), device);
  const int64_t b = query.size(0), s = query.size(1), hn = query.size(2);
  if (!p.ok || !p.attends() || p.nb != b || hn % p.gn != 0 || !step_rows4(query, b, s, hn, p.hd) || !on(query, device) ||
      query.scalar_type() != key.scalar_type() || (b == 1 && p.sb < p.bs * p.st))
    return c10::nullopt;
  const Tensor out = at::empty({b, s, hn * p.hd}, query.options());
  ic_prefill_call c = prefill_call(out, query, p, b, s, hn, scale, m.causal);
  c.row_pitch = s;
  c.uniform_context = (int)p.bs;
  if (m.bits.has_value()) {
    const int64_t planes = m.seqs * m.heads, qtiles = (s + 127) / 128, tiles = (p.bs + 63) / 64;
    if (m.causal || !m.lists.has_value() || (m.seqs != 1 && m.seqs != b) || (m.heads != 1 && m.heads != hn) ||
        !index_vector(*m.bits, at::kLong, planes * qtiles * 4 * tiles * 32, device) ||
        !index_vector(*m.lists, at::kInt, planes * qtiles * (tiles + 1), device))
      return c10::nullopt;
    c.mask_bits = reinterpret_cast<const uint64_t *>(m.bits->data_ptr<int64_t>());
    c.mask_lists = m.lists->data_ptr<int32_t>();
    c.mask_plane_head = m.heads > 1 ? 1 : 0;
    c.mask_plane_seq = m.seqs > 1 ? (int)m.heads : 0;
  }
  if (!made("ic_paged_prefill_ex", ic_paged_prefill_ex(&c, stream))) return c10::nullopt;
  return out;
}

// The dense call: query [b, sq, hn, hd] on key / value [b, sk, gn, hd].  Tensors that do not lie as the kernel walks
// them are copied: a query whose rows are not one stride apart, or, one row a sequence, at a stride that the kernel does
// not take (one row for the whole batch, rows at an odd distance), keys and values with strides of their own (a rotary
// model rotates the keys into a tensor of their own and leaves the values a slice of the projection).
OptTensor dense(const Tensor &query, const Tensor &key, const Tensor &value, bool causal, const OptTensor &bits,
                const OptTensor &lists, int64_t mask_seqs, int64_t mask_heads, double scale, int64_t device,
                int64_t stream) {
  if (query.dim() != 4 || key.dim() != 4 || value.dim() != 4 || key.size(1) == 0 || query.size(1) == 0)
    return c10::nullopt;
  const DenseMask m{causal, bits, lists, mask_seqs, mask_heads};
  const int64_t b = query.size(0), s = query.size(1), hn = query.size(2), hd = query.size(3);
  const bool laid = rows4(query, b, s, hn, hd) ||
                    (step_rows4(query, b, s, hn, hd) &&
                     rows16(query.data_ptr(), row_stride4(query), hn * hd, query.element_size()));
  const Tensor q = laid ? query : row_major(query);
  OptTensor out = dense_as_laid(q, key, value, m, scale, device, (void *)stream);
  if (!out.has_value()) {
    const Tensor k = row_major(key), v = row_major(value);
    if (!k.is_same(key) || !v.is_same(value)) out = dense_as_laid(q, k, v, m, scale, device, (void *)stream);
  }
  return out;
}

// ---- the model's linears --------------------------------------------------------------------

// Nothing but values: no subclass, no functorch or forward-mode wrapper, no view that a kernel would misread.
bool plain(const Tensor &t) {
  return !at::isTensorSubclassLike(t) && !t.is_conj() && !t.is_neg() && !t._fw_grad(0).defined();
}

// Whether torch's product, and its addition of the bias, is as fast or faster for m rows, the weights read from memory.
// (splits: what the kernel would take; a tile is a workgroup's 64 columns in fp32, 128 in 16 bits.)  Library / kernel, us:
//  * more columns than the CUs hold tiles of at once, so that a second, short wave of workgroups runs alone: 1 024 x
//    50 304 fp32 39 / 47, 4 096 x 50 304 bf16 68 / 74; x 32 000 28 / 26 and 53 / 47;
//  * fp32, more than 16 rows, one split (each workgroup reads all of x twice over): 4 096 x 11 008 46 / 58, with the
//    bias 48 / 57; short columns have a bias's launch to gain: 512 x 2 048 11 / 8;
//  * two splits of 113 to 128 tiles: 4 096 x 8 192 fp32 26 / 29, 4 096 x 16 384 bf16 26 / 28, while 8 192 x 8 192 is
//    57 / 53, 1 536 x 8 192 fp32 16 / 14 and 1 088 x 16 384 bf16 13 / 11;
//  * short columns, whose split pays for its second launch only by a bias: fp32, 8 rows 640 x 4 096 7.0 / 7.6, 768 x
//    3 072 8.0 / 7.5, 17 rows 1 024 x 4 096 9.1 / 10.3, 3 072 x 3 072 18 / 17; bf16, 16 rows 1 536 x 1 536 7 / 8, x
//    6 144 12 / 10, 2 048 x 2 048 9 / 8, 17 rows 1 792 x 2 048 8 / 9; without a split, 1 024 x 1 024 6.0 / 6.8.
bool library_as_fast(int64_t m, int64_t n, int64_t k, bool fp32, int64_t splits, bool bias) {
  const int64_t tiles = (n + (fp32 ? 63 : 127)) / (fp32 ? 64 : 128);
  const bool many = m > 16;
  if (tiles > (fp32 ? 512 : 256) && (fp32 || !bias)) return true;
  const bool two_splits = splits == 2 && tiles > 112 && k < 8192 && k >= (fp32 ? 2048 : 1280);
  if (bias) return fp32 && many && (splits == 1 ? k > 768 || n > 16384 : two_splits);
  if (splits == 1) return many || k * (fp32 ? 4 : 2) <= 2048;
  if (two_splits) return true;
  if (many) return fp32 ? splits < 8 && k < 3072 : k < 2048;
  return fp32 ? k < (m > 8 ? 1024 : 768) : k < 2048 && n < 5120;
}

// y = x W (+ bias) for the few rows of a decode step; x [..., k] contiguous, W [k, n].  What a dispatched product
// would do beside it (autograd, autocast, tracing, dispatch modes) is left to that.
OptTensor linear_rows(const Tensor &x, const Tensor &w, const OptTensor &bias, int64_t device, int64_t stream) {
  if (x.dim() < 2 || w.dim() != 2 || !on(x, device) || !on(w, device) || x.scalar_type() != w.scalar_type() ||
      x.size(-1) != w.size(0) || x.numel() == 0 || !x.is_contiguous() || w.stride(1) != 1 || !plain(x) || !plain(w) ||
      c10::impl::dispatch_mode_enabled() || at::autocast::is_autocast_enabled(at::kCUDA))
    return c10::nullopt;
  const int dtype = dtype_code(x.scalar_type());
  const int64_t k = w.size(0), n = w.size(1), m = x.numel() / k;
  if (dtype < 0 || m > IC_LINEAR_ROWS_MAX || n > INT_MAX || k > INT_MAX) return c10::nullopt;
  if (bias.has_value() && (!index_vector(*bias, x.scalar_type(), n, device) || bias->dim() != 1 || !plain(*bias)))
    return c10::nullopt;
  if (at::GradMode::is_enabled() &&
      (x.requires_grad() || w.requires_grad() || (bias.has_value() && bias->requires_grad())))
    return c10::nullopt;
  const int es = (int)x.element_size();
  if (n % (16 / es) != 0 || k % (64 / es) != 0 || (w.stride(0) * es) % 16 != 0 || w.stride(0) < n) return c10::nullopt;
  const size_t need = ic_linear_rows_workspace_bytes((int)m, (int)n, (int)k, 0, dtype);
  const int64_t splits = need > 0 ? (int64_t)need / (4 * m * n) : 1;
  if (library_as_fast(m, n, k, dtype == IC_DTYPE_F32, splits, bias.has_value())) return c10::nullopt;
  auto sizes = x.sizes().vec();
  sizes.back() = n;
  const Tensor out = at::empty(sizes, x.options());
  Tensor ws;
  if (need > 0) ws = at::empty({(int64_t)need}, x.options().dtype(at::kByte));
  if (!made("ic_linear_rows",
            ic_linear_rows(out.data_ptr(), n, x.data_ptr(), k, w.data_ptr(), w.stride(0),
                           bias.has_value() ? bias->data_ptr() : nullptr, (int)m, (int)n, (int)k, 0,
                           need > 0 ? ws.data_ptr() : nullptr, need, dtype, (void *)stream)))
    return c10::nullopt;
  return out;
}

// ---- a transformer layer's decode step -------------------------------------------------------

// A parameter or activation of a step: plain values of one type on the device, rows of 16-byte pieces.
bool step_tensor(const Tensor &t, at::ScalarType type, int64_t device) {
  return on(t, device) && t.scalar_type() == type && plain(t) && !(at::GradMode::is_enabled() && t.requires_grad());
}
bool step_vector(const OptTensor &t, int64_t n, at::ScalarType type, int64_t device) {
  return !t.has_value() || (step_tensor(*t, type, device) && t->dim() == 1 && t->numel() == n && t->is_contiguous() &&
                            reinterpret_cast<uintptr_t>(t->data_ptr()) % 16 == 0);
}
bool step_matrix(const OptTensor &t, int64_t k, int64_t n, at::ScalarType type, int64_t device) {
  return t.has_value() && step_tensor(*t, type, device) && t->dim() == 2 && t->size(0) == k && t->size(1) == n &&
         t->stride(1) == 1 && n * t->element_size() % 16 == 0 && k * t->element_size() % 64 == 0 &&
         rows16(t->data_ptr(), t->stride(0), n, t->element_size());
}
const void *data(const OptTensor &t) { return t.has_value() ? t->data_ptr() : nullptr; }

// Whether a step may go past the dispatcher at all.
bool step_outside_torch() { return c10::impl::dispatch_mode_enabled() || at::autocast::is_autocast_enabled(at::kCUDA); }

// The norm of up to 32 rows [b, 1, n].
OptTensor norm_rows(const Tensor &x, const Tensor &weight, const OptTensor &bias, int64_t norm, double eps,
                    int64_t device, int64_t stream) {
  const at::ScalarType type = x.scalar_type();
  const int dtype = dtype_code(type);
  const int64_t n = x.size(-1), m = n > 0 ? x.numel() / n : 0;
  if (dtype < 0 || m < 1 || m > IC_LINEAR_ROWS_MAX || n > IC_STEP_LINEAR_ROW_MAX || !step_tensor(x, type, device) ||
      !x.is_contiguous() || !rows16(x.data_ptr(), n, n, x.element_size()) || !step_vector(weight, n, type, device) ||
      !step_vector(bias, n, type, device) || step_outside_torch())
    return c10::nullopt;
  const Tensor out = at::empty(x.sizes(), x.options());
  ic_step_linear_call c = {};
  c.norm_out = out.data_ptr(), c.norm_out_stride = n;
  c.residual = x.data_ptr(), c.residual_stride = n;
  c.norm_weight = weight.data_ptr(), c.norm_bias = data(bias);
  c.m = (int)m, c.n = (int)n, c.norm = (int)norm, c.eps = (float)eps, c.dtype = dtype;
  if (!made("ic_step_linear", ic_step_linear(&c, (void *)stream))) return c10::nullopt;
  return out;
}

// One layer of a decode step: hidden [b, 1, d] and its input norm in, the layer's output and the norm that follows it
// (the next layer's, or the model's last) out.  `w`: q, kv, attention output, post-attention norm, up, down, next norm, a
// weight and a bias each.  Seven launches and more: projections with the append, attention (one or two), output projection
// with residual and norm (two), up-projection with the activation, down-projection with residual and norm (two).
c10::optional<std::tuple<Tensor, Tensor>> decoder_layer(
    const Tensor &hidden, const Tensor &normed, const std::vector<OptTensor> &w, int64_t hn, int64_t gn, int64_t hd,
    int64_t act, int64_t norm, double eps, int64_t next_norm, double next_eps, bool post_ln, const Tensor &k_pool, const Tensor &v_pool,
    const Tensor &tables, const Tensor &lens, const Tensor &slots, int64_t max_ctx, double scale, int64_t cohort,
    const OptTensor &shared, const OptTensor &positions, const OptTensor &cos, const OptTensor &sin, int64_t device,
    int64_t stream) {
  const Pool p(k_pool, v_pool, device);
  const at::ScalarType type = hidden.scalar_type();
  if (w.size() != 14 || !p.ok || p.gn != gn || p.hd != hd || hidden.dim() != 3 || hidden.size(1) != 1 || k_pool.scalar_type() != type ||
      normed.sizes() != hidden.sizes() || !step_tensor(hidden, type, device) || !step_tensor(normed, type, device) ||
      !hidden.is_contiguous() || !normed.is_contiguous() || step_outside_torch())
    return c10::nullopt;
  const int64_t b = hidden.size(0), d = hidden.size(2), q_cols = hn * p.hd, kv_cols = p.gn * p.hd;
  if (b < 1 || b > IC_LINEAR_ROWS_MAX || d > IC_STEP_LINEAR_ROW_MAX || !w[8].has_value() || w[8]->dim() != 2)
    return c10::nullopt;
  const int64_t up_cols = w[8]->size(1), f = act >= IC_ACT_GLU ? up_cols / 2 : up_cols;
  const int es = (int)hidden.element_size();
  if (!rows16(hidden.data_ptr(), d, d, es) || !rows16(normed.data_ptr(), d, d, es) ||
      !step_matrix(w[0], d, q_cols, type, device) || !step_vector(w[1], q_cols, type, device) ||
      !step_matrix(w[2], d, 2 * kv_cols, type, device) || !step_vector(w[3], 2 * kv_cols, type, device) ||
      !step_matrix(w[4], q_cols, d, type, device) || !step_vector(w[5], d, type, device) || !w[6].has_value() ||
      !step_vector(w[6], d, type, device) || !step_vector(w[7], d, type, device) ||
      !step_matrix(w[8], d, up_cols, type, device) || !step_vector(w[9], up_cols, type, device) ||
      up_cols > (1 << 30) || (act >= IC_ACT_GLU && (up_cols * es) % 32 != 0) || !step_matrix(w[10], f, d, type, device) ||
      !step_vector(w[11], d, type, device) || !w[12].has_value() || !step_vector(w[12], d, type, device) ||
      !step_vector(w[13], d, type, device) || !index_vector(slots, at::kLong, b, device))
    return c10::nullopt;
  const Decode dec{tables, lens, max_ctx, 0, cohort, shared, scale};
  const Rope rope(positions, cos, sin, b, p.hd, device);
  if (!rope.ok || !decode_fits(p, b, hn, dec, device) ||
      !rows16(p.k, p.sb, 1, es) || !rows16(p.v, p.sb, 1, es) || (p.sh * es) % 16 != 0 || (p.st * es) % 16 != 0)
    return c10::nullopt;
  if (!cohorts_pay(b, hn, p.gn, p.hd, max_ctx, cohort, es)) cohort = 1;

  ic_step_linear_call qkv = {}, proj = {}, up = {}, down = {};
  qkv.m = proj.m = up.m = down.m = (int)b;
  qkv.dtype = proj.dtype = up.dtype = down.dtype = p.dtype;
  qkv.x = normed.data_ptr(), qkv.x_stride = d, qkv.k = (int)d;
  qkv.w = data(w[0]), qkv.bias = data(w[1]), qkv.w_stride = w[0]->stride(0), qkv.n = (int)q_cols;
  qkv.w2 = data(w[2]), qkv.bias2 = data(w[3]), qkv.w2_stride = w[2]->stride(0), qkv.n2 = (int)(2 * kv_cols);
  qkv.out_stride = q_cols;
  qkv.k_pool = const_cast<void *>(p.k), qkv.v_pool = const_cast<void *>(p.v);
  qkv.pool_stride_block = p.sb, qkv.pool_stride_head = p.sh, qkv.pool_stride_token = p.st, qkv.num_blocks = p.nb;
  qkv.hn = (int)hn, qkv.gn = (int)p.gn, qkv.hd = (int)p.hd, qkv.block_size = (int)p.bs;
  qkv.slot_mapping = slots.data_ptr<int64_t>();
  qkv.positions = rope.positions, qkv.cos_table = rope.cos, qkv.sin_table = rope.sin, qkv.table_rows = rope.rows;
  proj.x_stride = q_cols, proj.k = (int)q_cols;
  proj.w = data(w[4]), proj.bias = data(w[5]), proj.w_stride = w[4]->stride(0), proj.n = (int)d;
  proj.residual = post_ln ? normed.data_ptr() : hidden.data_ptr(), proj.residual_stride = d;
  proj.norm = (int)norm, proj.eps = (float)eps, proj.norm_weight = data(w[6]), proj.norm_bias = data(w[7]);
  proj.out_stride = proj.norm_out_stride = d;
  up.x_stride = d, up.k = (int)d;
  up.w = data(w[8]), up.bias = data(w[9]), up.w_stride = w[8]->stride(0), up.n = (int)up_cols;
  up.act = (int)act, up.out_stride = f;
  down.x_stride = f, down.k = (int)f;
  down.w = data(w[10]), down.bias = data(w[11]), down.w_stride = w[10]->stride(0), down.n = (int)d;
  down.norm = (int)next_norm, down.eps = (float)next_eps, down.norm_weight = data(w[12]), down.norm_bias = data(w[13]);
  down.residual_stride = down.out_stride = down.norm_out_stride = d;

  // one allocation for what the layer's launches hand to each other
  const Tensor out = at::empty({b, 1, d}, hidden.options()), out_normed = at::empty({b, 1, d}, hidden.options());
  down.residual = out.data_ptr();  // (any address: what the workspace depends on)
  size_t work = 0;
  for (const ic_step_linear_call *c : {&qkv, &proj, &up, &down}) work = std::max(work, ic_step_linear_workspace_bytes(c));
  const size_t decode_work =
      ic_paged_decode_shared_workspace_bytes((int)b, (int)hn, (int)p.gn, (int)p.hd, (int)cohort);
  size_t total = 0;
  auto take = [&](size_t bytes) {
    const size_t at = total;
    total += (bytes + 255) & ~(size_t)255;
    return at;
  };
  const size_t at_q = take(b * q_cols * es), at_att = take(b * q_cols * es), at_mid = take(b * d * es),
               at_mid_normed = take(b * d * es), at_act = take(b * f * es), at_work = take(std::max(work, decode_work));
  const Tensor scratch = at::empty({(int64_t)total}, hidden.options().dtype(at::kByte));
  char *base = static_cast<char *>(scratch.data_ptr());
  qkv.out = base + at_q;
  proj.x = base + at_att, proj.out = base + at_mid, proj.norm_out = base + at_mid_normed;
  up.x = base + at_mid_normed, up.out = base + at_act;
  down.x = base + at_act, down.residual = post_ln ? proj.norm_out : proj.out;
  down.out = out.data_ptr(), down.norm_out = out_normed.data_ptr();
  for (ic_step_linear_call *c : {&qkv, &proj, &up, &down}) c->workspace = base + at_work, c->workspace_bytes = work;

  auto linear = [&](const ic_step_linear_call &c) { return made("ic_step_linear", ic_step_linear(&c, (void *)stream)); };
  if (!linear(qkv) ||
      !made("ic_paged_decode_shared",
            ic_paged_decode_shared(base + at_att, q_cols, qkv.out, q_cols, p.k, p.v, p.sb, p.sh, p.st,
                                   tables.data_ptr<int32_t>(), tables.stride(0), lens.data_ptr<int32_t>(), (int)b,
                                   (int)hn, (int)p.gn, (int)p.hd, (int)p.bs, p.nb, (int)max_ctx, (float)scale, 0,
                                   (int)cohort, cohort > 1 ? shared->data_ptr<int32_t>() : nullptr, base + at_work,
                                   decode_work, p.dtype, (void *)stream)) ||
      !linear(proj) || !linear(up) || !linear(down))
    return c10::nullopt;
  return std::make_tuple(out, out_normed);
}

// All layers of a decode step and the norm behind them in one launch (ic_step_stack; more layers than one call holds: in
// equal parts).  `w`: a layer's weights and biases as decoder_layer takes them, but for the next norm; `norms`: its input
// norm and its post-attention norm as (kind, eps, weight, bias).  None for what the call does not take, and where the
// layers' own launches are as fast (stack_takes).
using Norm = std::tuple<int64_t, double, Tensor, OptTensor>;

// us a layer and token of a replayed step, layers' launches / stack (8 layers; heads / KV heads, ffn, context, rows):
//   fp32 d 768     12 / 12 of 64   3 072     300    1  34 / 25     4  38 / 28     5  38 / 33    16  46 / 40
//                                           1 700    4  54 / 42    16  69 / 61
//                                  4 096     300    16  47 / 45    gated, 4  50 / 43    gated, 16  55 / 56
//                                  8 192     300     4  50 / 47    16  55 / 61
//                  12 / 3 of 64    3 072     250     4  37 / 31     6  37 / 36    16  40 / 40      500   16  47 / 45
//                  12 / 6 of 64    3 072     250     4  35 / 32    16  42 / 42      128   16  39 / 40
//                  6 / 6 of 128    2 304     380     4  39 / 38    16  49 / 51    1 000    4  54 / 63
//                  6 / 3 of 128    2 304     250     4  36 / 48
//        d 512     8 / 8 of 64     2 048     300     4  31 / 24    16  35 / 31
//        d 832     13 / 13 of 64   3 328     300     4  40 / 43    16  47 / 56
//        d 1 024   8 / 8 of 128    4 096     300     4  48 / 56    16  53 / 69
//   bf16 d 1 024   8 / 8 of 128    2 752     300    16  45 / 37    2 000   16  67 / 58;   8 192   300   16  59 / 51
//                  16 / 4 of 64    2 752     500     2  40 / 32    16  45 / 41
//                  16 / 8 of 64    2 752     128    16  39 / 38      500   16  46 / 42
//                  8 / 2 of 128    2 752     380     1  42 / 40     4  45 / 43    10  47 / 49      450    2  42 / 43
//                  8 / 4 of 128    2 752     380     2  37 / 42    16  45 / 53
//   fp16           8 / 2 of 128    2 752     250     2  39 / 41     4  39 / 42     8  40 / 47
// In fp32 a row of more than 768 (the product keeps eight steps of weights and not six) and heads of 128 do not fit the registers,
// nor do the four query rows of grouped heads of 128 (bf16 spills less); above four rows the fp32 product takes 16x16 instructions,
// mostly for rows that are not there, and long columns weigh more.  A pair's rows are walked by one workgroup, which bounds the
// contexts of grouped heads.  Below 2 MB of weights a layer (fp32 d 256, ffn 352 24.4 / 20.6) there is little to prefetch, and
// the layers stay calls of their own, any of which may be a module's.
bool stack_pays(at::ScalarType type, int64_t b, int64_t d, int64_t f, int64_t group, int64_t hd, int64_t max_ctx, int64_t layer_bytes) {
  const int64_t rounds = (max_ctx + 127) / 128;
  if (layer_bytes < 2000000 || f > 8192 || group > 4 || rounds > (group == 1 ? 16 : 4)) return false;
  if (type == at::kFloat) return d <= 768 && hd == 64 && (b <= 4 || (f <= 4096 && group != 2));
  return group == 1 || hd == 64 || (type == at::kBFloat16 && group > 2 && b <= 4 && rounds <= 3);
}

// Whether a step of these sizes goes to decoder_stack: asked by itself before the caller gathers the layers' tensors (25 us of
// the host for four layers, which a step bound by the host would lose for nothing).
bool stack_takes(at::ScalarType type, int64_t b, int64_t d, int64_t f, int64_t hn, int64_t gn, int64_t hd, int64_t act,
                 int64_t max_ctx) {
  if (dtype_code(type) < 0 || b < 1 || b > IC_STEP_STACK_ROWS || d < 1 || d > 1024 || f < 1 || gn < 1 || hn < gn || hn % gn != 0 ||
      (hd != 64 && hd != 128))
    return false;
  const int64_t columns = 2 * hn * hd + 2 * gn * hd + (act >= IC_ACT_GLU ? 3 : 2) * f;
  return stack_pays(type, b, d, f, hn / gn, hd, max_ctx, d * columns * (int64_t)c10::elementSize(type));
}

// Where launches say that they gave up a wait (ic_step_stack), and whether one has since the last time this was asked.
std::atomic<int32_t *> step_status{nullptr};
bool step_given_up() {
  int32_t *const word = step_status.load(std::memory_order_acquire);
  return word != nullptr && __atomic_load_n(word, __ATOMIC_RELAXED) != 0 && __atomic_exchange_n(word, 0, __ATOMIC_RELAXED) != 0;
}

OptTensor decoder_stack(const Tensor &x, const std::vector<std::vector<OptTensor>> &w,
                        const std::vector<std::tuple<Norm, Norm>> &norms, const Norm &last, int64_t hn, int64_t gn,
                        int64_t hd, int64_t act, const std::vector<std::tuple<Tensor, Tensor>> &pools, const Tensor &tables,
                        const Tensor &lens, const Tensor &slots, int64_t max_ctx, double scale, const OptTensor &positions,
                        const OptTensor &cos, const OptTensor &sin, int64_t device, int64_t stream) {
  const at::ScalarType type = x.scalar_type();
  const size_t layers = w.size();
  if (layers == 0 || norms.size() != layers || pools.size() != layers || x.dim() != 3 || x.size(1) != 1 ||
      !step_tensor(x, type, device) || !x.is_contiguous() || dtype_code(type) < 0 || step_outside_torch())
    return c10::nullopt;
  const int64_t b = x.size(0), d = x.size(2), q_cols = hn * hd, kv_cols = gn * hd;
  const int es = (int)x.element_size();
  if (!rows16(x.data_ptr(), d, d, es) || w[0].size() != 12 || !w[0][8].has_value() || w[0][8]->dim() != 2 ||
      !index_vector(slots, at::kLong, b, device))
    return c10::nullopt;
  const int64_t up_cols = w[0][8]->size(1), f = act >= IC_ACT_GLU ? up_cols / 2 : up_cols;
  if (up_cols > (1 << 20) || (act >= IC_ACT_GLU && up_cols % 2 != 0) || !stack_takes(type, b, d, f, hn, gn, hd, act, max_ctx))
    return c10::nullopt;
  const Pool first(std::get<0>(pools[0]), std::get<1>(pools[0]), device);
  const OptTensor none;
  const Decode dec{tables, lens, max_ctx, 0, 1, none, scale};
  const Rope rope(positions, cos, sin, b, hd, device);
  if (!first.ok || !rope.ok || first.gn != gn || first.hd != hd || std::get<0>(pools[0]).scalar_type() != type ||
      !decode_fits(first, b, hn, dec, device))
    return c10::nullopt;
  auto matrix = [&](const OptTensor &t, int64_t k, int64_t n) {
    return step_matrix(t, k, n, type, device) && t->stride(0) == n;
  };
  auto norm_fits = [&](const Norm &n) {
    return step_vector(std::get<2>(n), d, type, device) && step_vector(std::get<3>(n), d, type, device);
  };
  if (!norm_fits(last)) return c10::nullopt;
  std::vector<ic_step_layer> table(layers);
  for (size_t i = 0; i < layers; ++i) {
    const auto &t = w[i];
    const Norm &in = std::get<0>(norms[i]), &post = std::get<1>(norms[i]);
    const Pool p(std::get<0>(pools[i]), std::get<1>(pools[i]), device);
    if (t.size() != 12 || !matrix(t[0], d, q_cols) || !step_vector(t[1], q_cols, type, device) || !matrix(t[2], d, 2 * kv_cols) ||
        !step_vector(t[3], 2 * kv_cols, type, device) || !matrix(t[4], q_cols, d) || !step_vector(t[5], d, type, device) ||
        !matrix(t[8], d, up_cols) || !step_vector(t[9], up_cols, type, device) || !matrix(t[10], f, d) ||
        !step_vector(t[11], d, type, device) || !norm_fits(in) || !norm_fits(post) || !p.ok || p.gn != gn || p.hd != hd ||
        p.bs != first.bs || p.nb != first.nb || p.sb != first.sb || p.sh != first.sh || p.st != first.st ||
        p.dtype != first.dtype)
      return c10::nullopt;
    ic_step_layer &l = table[i];
    l.input_norm_weight = std::get<2>(in).data_ptr(), l.input_norm_bias = data(std::get<3>(in));
    l.q_weight = data(t[0]), l.q_bias = data(t[1]), l.kv_weight = data(t[2]), l.kv_bias = data(t[3]);
    l.proj_weight = data(t[4]), l.proj_bias = data(t[5]);
    l.post_norm_weight = std::get<2>(post).data_ptr(), l.post_norm_bias = data(std::get<3>(post));
    l.up_weight = data(t[8]), l.up_bias = data(t[9]), l.down_weight = data(t[10]), l.down_bias = data(t[11]);
    l.k_pool = const_cast<void *>(p.k), l.v_pool = const_cast<void *>(p.v);
    l.input_norm = (int)std::get<0>(in), l.post_norm = (int)std::get<0>(post);
    l.input_norm_eps = (float)std::get<1>(in), l.post_norm_eps = (float)std::get<1>(post);
  }
  ic_step_stack_call c = {};
  c.m = (int)b, c.d = (int)d, c.f = (int)f, c.hn = (int)hn, c.gn = (int)gn, c.hd = (int)hd, c.act = (int)act;
  c.pool_stride_block = first.sb, c.pool_stride_head = first.sh, c.pool_stride_token = first.st, c.num_blocks = first.nb;
  c.block_tables = tables.data_ptr<int32_t>(), c.block_table_stride = tables.stride(0);
  c.context_lens = lens.data_ptr<int32_t>(), c.slot_mapping = slots.data_ptr<int64_t>();
  c.positions = rope.positions, c.cos_table = rope.cos, c.sin_table = rope.sin, c.table_rows = rope.rows;
  c.block_size = (int)first.bs, c.max_context_len = (int)max_ctx, c.scale = (float)scale, c.dtype = first.dtype;
  c.status = ic_step_status();
  step_status.store(c.status, std::memory_order_release);
  const size_t parts = (layers + IC_STEP_STACK_LAYERS - 1) / IC_STEP_STACK_LAYERS;
  Tensor in = x, out, ws;
  for (size_t part = 0, from = 0; part < parts; ++part) {
    const size_t to = layers * (part + 1) / parts;
    const bool end = part + 1 == parts;
    c.layers = table.data() + from, c.num_layers = (int)(to - from);
    out = at::empty({b, 1, d}, x.options());
    c.x = in.data_ptr();
    c.out = end ? nullptr : out.data_ptr(), c.norm_out = end ? out.data_ptr() : nullptr;
    if (end) {
      c.norm = (int)std::get<0>(last), c.eps = (float)std::get<1>(last);
      c.norm_weight = std::get<2>(last).data_ptr(), c.norm_bias = data(std::get<3>(last));
    }
    c.workspace_bytes = ic_step_stack_workspace_bytes(&c);
    if (c.workspace_bytes == 0) return c10::nullopt;
    ws = at::empty({(int64_t)c.workspace_bytes}, x.options().dtype(at::kByte));
    c.workspace = ws.data_ptr();
    if (!made("ic_step_stack", ic_step_stack(&c, (void *)stream))) return c10::nullopt;
    in = out, from = to;
  }
  return out;
}

// ---- greedy decoding --------------------------------------------------------------------------

// The next token of each row of logits [b, n] and, wanted, how far it is ahead: stored into column `*column` of `tokens`
// [b, columns] and `margins`, and into `next` [b, 1].  `finished` comes with an eos token.
bool greedy(const Tensor &logits, const OptTensor &column, const OptTensor &tokens, const OptTensor &margins,
            const OptTensor &next, const OptTensor &finished, int64_t eos, int64_t device, int64_t stream) {
  const int dtype = dtype_code(logits.scalar_type());
  if (dtype < 0 || logits.dim() != 2 || logits.size(0) == 0 || logits.size(1) < 2 || logits.size(0) > INT_MAX / 64 ||
      logits.size(1) > INT_MAX / 2 || logits.stride(1) != 1 || !on(logits, device) || !plain(logits) ||
      c10::impl::dispatch_mode_enabled())
    return false;
  const int64_t b = logits.size(0), n = logits.size(1), es = logits.element_size();
  const int64_t stride = b > 1 ? logits.stride(0) : n;
  auto table = [&](const OptTensor &t, at::ScalarType type) {
    return !t.has_value() || (on(*t, device) && t->scalar_type() == type && t->dim() == 2 && t->size(0) == b &&
                              t->size(1) > 0 && t->is_contiguous());
  };
  if (!rows16(logits.data_ptr(), stride, n, es) || (n * es) % 16 != 0 || !table(tokens, at::kLong) ||
      !table(margins, at::kFloat) || (tokens.has_value() && margins.has_value() && tokens->size(1) != margins->size(1)) ||
      (column.has_value() && !index_vector(*column, at::kLong, 1, device)) ||
      (next.has_value() && !index_vector(*next, at::kLong, b, device)) ||
      (finished.has_value() && !index_vector(*finished, at::kBool, b, device)))
    return false;
  ic_greedy_call c = {};
  c.logits = logits.data_ptr(), c.stride = stride;
  c.rows = (int)b, c.n = (int)n, c.dtype = dtype;
  if (tokens.has_value()) c.tokens = tokens->data_ptr<int64_t>(), c.token_stride = c.columns = tokens->size(1);
  if (margins.has_value()) c.margins = margins->data_ptr<float>(), c.margin_stride = c.columns = margins->size(1);
  if (column.has_value()) c.column = column->data_ptr<int64_t>();
  if (next.has_value()) c.next = next->data_ptr<int64_t>();
  if (finished.has_value()) c.finished = reinterpret_cast<uint8_t *>(finished->data_ptr<bool>()), c.eos = eos;
  c.workspace_bytes = ic_greedy_workspace_bytes(c.rows, c.n);
  const Tensor ws = at::empty({(int64_t)c.workspace_bytes}, logits.options().dtype(at::kByte));
  c.workspace = ws.data_ptr();
  return made("ic_greedy", ic_greedy(&c, (void *)stream));
}

// Position, slot and context length of the next token of each row (see ic_advance).
bool advance(const Tensor &lens, const Tensor &tables, int64_t block_size, const Tensor &positions,
             const Tensor &token_positions, const Tensor &slots, const Tensor &column, int64_t device, int64_t stream) {
  const int64_t b = lens.numel();
  if (b == 0 || b > INT_MAX / 512 || !index_vector(lens, at::kInt, b, device) || !table(tables, b, device) ||
      tables.size(1) > INT_MAX || block_size > INT_MAX || !index_vector(positions, at::kInt, b, device) ||
      !index_vector(token_positions, at::kLong, b, device) || !index_vector(slots, at::kLong, b, device) ||
      !index_vector(column, at::kLong, 1, device))
    return false;
  ic_advance_call c = {};
  c.context_lens = lens.data_ptr<int32_t>();
  c.block_tables = tables.data_ptr<int32_t>(), c.block_table_stride = tables.stride(0);
  c.rows = (int)b, c.table_width = (int)tables.size(1), c.block_size = (int)block_size;
  c.positions = positions.data_ptr<int32_t>(), c.token_positions = token_positions.data_ptr<int64_t>();
  c.slot_mapping = slots.data_ptr<int64_t>(), c.column = column.data_ptr<int64_t>();
  return made("ic_advance", ic_advance(&c, (void *)stream));
}

}  // namespace

// (wrapped, so that torch's exceptions keep their Python types: an allocation that does not fit raises
// torch.OutOfMemoryError.  The GIL is given up for the call: a launch may wait on a full queue and an allocation on the
// GPU, and other threads go on meanwhile.)
PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("cohorts_pay", &cohorts_pay);
  m.def("kv_append", torch::wrap_pybind_function_no_gil(kv_append));
  m.def("paged_decode", torch::wrap_pybind_function_no_gil(paged_decode));
  m.def("decode_step", torch::wrap_pybind_function_no_gil(decode_step));
  m.def("prefill_step", torch::wrap_pybind_function_no_gil(prefill_step), py::arg("query"), py::arg("key"), py::arg("value"),
        py::arg("k_pool"), py::arg("v_pool"), py::arg("tables"), py::arg("lens"), py::arg("slots"), py::arg("bounds"),
        py::arg("rows"), py::arg("longest"), py::arg("scale"), py::arg("positions"), py::arg("cos"), py::arg("sin"),
        py::arg("device"), py::arg("stream"), py::arg("max_ctx") = 0);
  m.def("dense", torch::wrap_pybind_function_no_gil(dense));
  m.def("linear_rows", torch::wrap_pybind_function_no_gil(linear_rows));
  m.def("norm_rows", torch::wrap_pybind_function_no_gil(norm_rows));
  m.def("decoder_layer", torch::wrap_pybind_function_no_gil(decoder_layer));
  m.attr("STEP_ROWS") = IC_LINEAR_ROWS_MAX;
  m.def("stack_takes", &stack_takes);
  m.def("step_given_up", &step_given_up);
  m.def("decoder_stack", torch::wrap_pybind_function_no_gil(decoder_stack));
  m.def("greedy", torch::wrap_pybind_function_no_gil(greedy));
  m.def("advance", torch::wrap_pybind_function_no_gil(advance));
  m.def("pack_mask", torch::wrap_pybind_function_no_gil(pack_mask));
}
