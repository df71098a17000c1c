// Host side of the launches: a Python extension module that checks tensors, allocates results and fills the argument
// tables of the C ABI (include/ditango_hip.h), which it calls.  A layer call of a small problem lasts about as long on
// the GPU as the checks of its two dozen tensors in Python did: with 4 KV chunks of 512 keys 59 us a call through
// ctypes, of which 20 are kernels.
//
// Nothing here reads device memory, synchronises or keeps state between calls.  Errors are raised as the exception class
// that ditango_amd._hip hands over (DitangoHipError).
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/core/CachingDeviceAllocator.h>
#include <torch/csrc/utils/pybind.h>

#include <algorithm>
#include <optional>
#include <string>
#include <utility>
#include <vector>

#include "ditango_hip.h"

namespace py = pybind11;
using at::Tensor;

namespace {

py::handle g_error;   // the exception class (kept alive by the module that set it)

[[noreturn]] void fail(const std::string& msg) {
  PyErr_SetString(g_error ? g_error.ptr() : PyExc_RuntimeError, msg.c_str());
  throw py::error_already_set();
}
template <typename... Parts>
std::string text(const Parts&... parts) {
  std::string s;
  (s.append(parts), ...);
  return s;
}
// name[i], spelled only when a check fails
struct Name {
  const char* base;
  int64_t i = -1;
  std::string str() const { return i < 0 ? std::string(base) : text(base, "[", std::to_string(i), "]"); }
};
#define REQUIRE(cond, ...)              \
  do {                                  \
    if (!(cond)) [[unlikely]]           \
      fail(text(__VA_ARGS__));          \
  } while (0)

// A call of the C ABI, without the interpreter lock: a launch that waits for room in the GPU's queue must not stop the other
// Python threads.  (The arguments are evaluated, and checked, before it is given up.)
template <typename... P, typename... A>
void call(const char* what, int (*fn)(P...), A... args) {
  int rc;
  {
    py::gil_scoped_release unlocked;
    rc = fn(args...);
  }
  if (rc != 0) fail(text(what, " failed with code ", std::to_string(rc), ": ", dt_last_error()));
}
#define CALL(fn, ...) call(#fn, fn, __VA_ARGS__)
// Uninitialised memory; without the lock as well, the allocator may wait for the device.
Tensor empty(at::IntArrayRef sizes, at::TensorOptions options) {
  py::gil_scoped_release unlocked;
  return at::empty(sizes, options);
}

bool is_half(const Tensor& t) { return t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kHalf; }

int dtype_code(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kBFloat16: return DT_BF16;
    case at::kFloat: return DT_FP32;
    case at::kHalf: return DT_FP16;
    default: fail("unsupported state dtype (bf16, fp16 or fp32)");
  }
}

bool shape_is(const Tensor& t, std::initializer_list<int64_t> want) { return t.sizes() == at::IntArrayRef(want); }

struct Dims {
  int64_t B, S, H, D;
};

Dims check_bshd(const Tensor& t, const Name& name) {
  REQUIRE(t.is_cuda(), name.str(), " must live on the GPU");
  REQUIRE(is_half(t), name.str(), " must be bf16 or fp16");
  REQUIRE(t.dim() == 4 && t.stride(3) == 1, name.str(), " must be [B,S,H,D] with contiguous D");
  return {t.size(0), t.size(1), t.size(2), t.size(3)};
}

// DT_LSE_BHS or DT_LSE_BSH of a dense lse tensor of (B, S, H) rows.  Where the shape alone cannot tell (S == H), a 4-D
// tensor is read as the running layout [B,S,H,1] (utils.py:49) and a 3-D one as flash-attn's [B,H,S].
int lse_layout(const Tensor& lse, int64_t B, int64_t S, int64_t H) {
  const auto sizes = lse.sizes();
  const auto strides = lse.strides();
  const bool four = lse.dim() == 4 && sizes[3] == 1;
  REQUIRE((lse.dim() == 3 || four) && lse.scalar_type() == at::kFloat, "lse must be fp32 with 3 (or 4, last=1) dims");
  // dense in the order (d0, d1, d2) of its first three dimensions (strides of dimensions of size 1 do not matter)
  auto dense = [&](int a, int b, int c) {
    return (sizes[c] == 1 || strides[c] == 1) && (sizes[b] == 1 || strides[b] == sizes[c]) &&
           (sizes[a] == 1 || strides[a] == sizes[b] * sizes[c]);
  };
  const bool empty = lse.numel() == 0;
  for (int pass = 0; pass < 2; ++pass) {
    const bool bsh = four == (pass == 0);
    if (!(sizes[0] == B && sizes[1] == (bsh ? S : H) && sizes[2] == (bsh ? H : S))) continue;
    if (empty || dense(0, 1, 2)) return bsh ? DT_LSE_BSH : DT_LSE_BHS;
    if (dense(0, 2, 1)) return bsh ? DT_LSE_BHS : DT_LSE_BSH;
  }
  fail("lse is not a dense [B,H,S] or [B,S,H] of the state's rows");
}

void* ptr(const Tensor& t) { return t.data_ptr(); }
void* ptr(const std::optional<Tensor>& t) { return t ? t->data_ptr() : nullptr; }
void* stream_of(uint64_t s) { return reinterpret_cast<void*>(s); }

void check_state(const Tensor& o, const Tensor& l, const Dims& d, at::ScalarType dtype, const Name& on, const Name& ln) {
  REQUIRE(o.scalar_type() == dtype && o.is_contiguous() && shape_is(o, {d.B, d.S, d.H, d.D}), on.str(),
          " must be contiguous [B,Sq,H,D] in q's dtype");
  REQUIRE(l.scalar_type() == at::kFloat && l.is_contiguous() && shape_is(l, {d.B, d.H, d.S}), ln.str(),
          " must be contiguous fp32 [B,H,Sq]");
}

// ---- KV chunks ---------------------------------------------------------------------------------------------

// The KV chunks one layer call can touch: pointers, lengths, strides.
struct ChunkTable {
  std::vector<Tensor> keep;   // alive while the pointers are in use
  std::vector<const void*> k, v;
  std::vector<int32_t> len;
  std::vector<int64_t> sb;
  int64_t n = 0, B = 0, H = 0, D = 0, ss = 0, sh = 0;
  at::ScalarType dtype = at::kBFloat16;

  // batch > 0: 3-D chunks are packed [batch * S, H, D] (the variable-length entry's layout); `convert` is called on
  // chunks that are neither bf16 nor fp16
  ChunkTable(const std::vector<Tensor>& ks, const std::vector<Tensor>& vs, int64_t batch, const py::object& convert) {
    n = (int64_t)ks.size();
    REQUIRE(n > 0 && ks.size() == vs.size(), "need at least one KV chunk and as many V as K chunks");
    keep.reserve(2 * n);
    k.reserve(n); v.reserve(n); len.reserve(n); sb.reserve(n);
    bool any = false;
    for (int64_t i = 0; i < n; ++i) {
      Tensor kt = ks[i], vt = vs[i];
      if (!convert.is_none()) {
        if (!is_half(kt)) kt = py::cast<Tensor>(convert(kt));
        if (!is_half(vt)) vt = py::cast<Tensor>(convert(vt));
      }
      if (batch > 0 && kt.dim() == 3) kt = kt.view({batch, kt.size(0) / batch, kt.size(1), kt.size(2)});
      if (batch > 0 && vt.dim() == 3) vt = vt.view({batch, vt.size(0) / batch, vt.size(1), vt.size(2)});
      if (i == 0) dtype = kt.scalar_type();
      const Dims d = check_bshd(kt, {"k", i});
      check_bshd(vt, {"v", i});
      REQUIRE(kt.scalar_type() == dtype && vt.scalar_type() == dtype, Name{"k", i}.str(),
              " / v must have one dtype with the other attention inputs");
      REQUIRE(kt.sizes() == vt.sizes() && kt.strides() == vt.strides(), Name{"k", i}.str(), " / v mismatch");
      if (d.S > 0) {
        if (!any) {
          ss = kt.stride(1); sh = kt.stride(2);
          B = d.B; H = d.H; D = d.D;
          any = true;
        }
        REQUIRE(kt.stride(1) == ss && kt.stride(2) == sh, "all chunks must share token/head strides");
        REQUIRE(d.B == B && d.H == H && d.D == D, "chunk B/H/D mismatch");
      }
      k.push_back(kt.data_ptr());
      v.push_back(vt.data_ptr());
      len.push_back((int32_t)d.S);
      sb.push_back(kt.stride(0));
      keep.push_back(std::move(kt));
      keep.push_back(std::move(vt));
    }
    REQUIRE(any, "all KV chunks are empty");
  }
};

Dims check_query(const Tensor& q, const ChunkTable& t) {
  const Dims d = check_bshd(q, {"q"});
  REQUIRE(q.scalar_type() == t.dtype, "q must have the dtype of the KV chunks");
  REQUIRE(d.B == t.B && d.H == t.H && d.D == t.D, "q and KV chunks disagree on B/H/D");
  return d;
}

// Segment boundaries in device memory (see ditango_amd._hip.DeviceSegments).
struct Segments {
  Tensor cu_q;
  std::vector<std::optional<Tensor>> cu_kv;
  int64_t max_q = 0;
  int32_t n_seg() const { return (int32_t)cu_q.numel() - 1; }
};
void check_boundaries(const Tensor& t, const Name& name) {
  REQUIRE(t.is_cuda() && t.scalar_type() == at::kInt && t.dim() == 1 && t.is_contiguous(), name.str(),
          " must be a contiguous int32 vector on the GPU");
}
Segments make_segments(const Tensor& cu_q, std::vector<std::optional<Tensor>> cu_kv, int64_t max_q) {
  check_boundaries(cu_q, {"cu_seqlens_q"});
  for (size_t i = 0; i < cu_kv.size(); ++i)
    if (cu_kv[i]) {
      check_boundaries(*cu_kv[i], {"cu_seqlens_kv", (int64_t)i});
      REQUIRE(cu_kv[i]->numel() == cu_q.numel(), Name{"cu_seqlens_kv", (int64_t)i}.str(),
              " must have as many entries as cu_seqlens_q");
    }
  REQUIRE(cu_q.numel() >= 2, "cu_seqlens_q needs at least two entries");
  REQUIRE(max_q > 0, "max_seqlen_q must be positive");
  return {cu_q, std::move(cu_kv), max_q};
}

typedef std::pair<int32_t, int32_t> Range;   // (begin, length)

int64_t bytes_of(const std::optional<Tensor>& t) { return t ? (int64_t)t->nbytes() : 0; }

// One launch or, where the jobs exceed the limits of one, several (ditango_amd._hip.attn_jobs_fwd).
void attn_jobs(const Tensor& q, const ChunkTable& table, const std::vector<std::vector<int32_t>>& jobs,
               const std::vector<Tensor>& outs, const std::vector<Tensor>& lses, double scale,
               const std::optional<std::vector<Range>>& q_ranges,
               const std::optional<std::vector<std::vector<Range>>>& kv_ranges, const std::optional<Tensor>& workspace,
               int32_t flags, bool no_alloc, const Segments* seg, const std::optional<std::vector<int32_t>>& job_segments,
               uint64_t stream, const dt_merge_result* merge = nullptr) {
  const Dims d = check_query(q, table);
  const size_t nj = jobs.size();
  REQUIRE(!(no_alloc && workspace), "no_alloc launches take no workspace");
  if (seg) {
    REQUIRE(!q_ranges && !kv_ranges && !no_alloc, "device segment boundaries replace the host ranges");
    REQUIRE(job_segments && job_segments->size() == nj, "one segment index per job");
    REQUIRE((int64_t)seg->cu_kv.size() == table.n, "one cu_seqlens_kv per chunk of the table");
  }
  REQUIRE(nj == outs.size() && nj == lses.size(), "one destination per job");
  REQUIRE(!q_ranges || q_ranges->size() == nj, "one query range per job");
  REQUIRE(!kv_ranges || kv_ranges->size() == nj, "one list of key ranges per job");
  for (size_t j = 0; j < nj; ++j) {
    check_state(outs[j], lses[j], d, q.scalar_type(), {"outs", (int64_t)j}, {"lses", (int64_t)j});
    REQUIRE(jobs[j].size() <= DT_MAX_JOB_ENTRIES, "a job references more than ", std::to_string(DT_MAX_JOB_ENTRIES), " chunks");
    REQUIRE(!kv_ranges || (*kv_ranges)[j].size() >= jobs[j].size(), "one key range per chunk reference");
    for (int32_t c : jobs[j])
      REQUIRE(c >= 0 && c < table.n, "job ", std::to_string(j), " references chunk ", std::to_string(c), " outside the table of ",
              std::to_string(table.n));
  }
  const bool whole = table.n <= DT_MAX_CHUNKS;   // every chunk is in the launch's table under its own number
  std::vector<int32_t> local(whole ? 0 : table.n);
  size_t start = 0;
  while (start < nj) {
    // the jobs of this launch: within the limits on jobs, chunk references and (a larger table) distinct chunks
    size_t end = start, entries = 0;
    std::vector<int32_t> ids;
    if (!whole) std::fill(local.begin(), local.end(), -1);
    while (end < nj && end - start < DT_MAX_JOBS && entries + jobs[end].size() <= DT_MAX_JOB_ENTRIES) {
      if (!whole) {
        const size_t before = ids.size();
        for (int32_t c : jobs[end])
          if (local[c] < 0) {
            local[c] = (int32_t)ids.size();
            ids.push_back(c);
          }
        if (ids.size() > DT_MAX_CHUNKS) {
          for (size_t i = before; i < ids.size(); ++i) local[ids[i]] = -1;
          ids.resize(before);
          break;
        }
      }
      entries += jobs[end].size();
      ++end;
    }
    REQUIRE(end > start, "job ", std::to_string(start), " references more than ", std::to_string(DT_MAX_CHUNKS),
            " distinct chunks: split it and merge the parts");
    if (!whole && ids.empty()) ids.push_back(0);
    const void *kp[DT_MAX_CHUNKS], *vp[DT_MAX_CHUNKS];
    int32_t lens[DT_MAX_CHUNKS];
    int64_t sbs[DT_MAX_CHUNKS];
    const int32_t* cu_kv[DT_MAX_CHUNKS];
    const int32_t nc = whole ? (int32_t)table.n : (int32_t)ids.size();
    for (int32_t i = 0; i < nc; ++i) {
      const int32_t c = whole ? i : ids[i];
      kp[i] = table.k[c]; vp[i] = table.v[c];
      lens[i] = table.len[c]; sbs[i] = table.sb[c];
      if (seg) cu_kv[i] = static_cast<const int32_t*>(ptr(seg->cu_kv[c]));
    }
    int32_t begin[DT_MAX_JOBS + 1], chunks[DT_MAX_JOB_ENTRIES], kb[DT_MAX_JOB_ENTRIES], kl[DT_MAX_JOB_ENTRIES];
    int32_t qb[DT_MAX_JOBS], ql[DT_MAX_JOBS], segs[DT_MAX_JOBS];
    void* op[DT_MAX_JOBS];
    float* lp[DT_MAX_JOBS];
    const int32_t n = (int32_t)(end - start);
    int32_t e = 0;
    for (int32_t jj = 0; jj < n; ++jj) {
      const size_t j = start + jj;
      begin[jj] = e;
      for (size_t i = 0; i < jobs[j].size(); ++i, ++e) {
        chunks[e] = whole ? jobs[j][i] : local[jobs[j][i]];
        if (kv_ranges) { kb[e] = (*kv_ranges)[j][i].first; kl[e] = (*kv_ranges)[j][i].second; }
      }
      if (q_ranges) { qb[jj] = (*q_ranges)[j].first; ql[jj] = (*q_ranges)[j].second; }
      if (seg) segs[jj] = (*job_segments)[j];
      op[jj] = outs[j].data_ptr();
      lp[jj] = static_cast<float*>(lses[j].data_ptr());
    }
    begin[n] = e;
    const auto sq = q.strides();
    if (merge)   // (the caller has seen to it that there is one launch, without ranges)
      CALL(dt_attn_jobs_merge_fwd, ptr(q), d.B, d.S, d.H, d.D, sq[0], sq[1], sq[2], nc, kp, vp, lens, sbs, table.ss, table.sh, n,
           begin, chunks, op, lp, merge, (float)scale, flags, ptr(workspace), bytes_of(workspace), stream_of(stream));
    else if (seg)
      CALL(dt_attn_varlen_jobs_ws_fwd, ptr(q), d.B, d.S, d.H, d.D, sq[0], sq[1], sq[2], nc, kp, vp, lens, sbs, table.ss,
           table.sh, n, begin, chunks, segs, seg->n_seg(), static_cast<const int32_t*>(ptr(seg->cu_q)), cu_kv,
           (int32_t)seg->max_q, op, lp, (float)scale, flags, ptr(workspace), bytes_of(workspace), stream_of(stream));
    else if (no_alloc)
      CALL(dt_attn_seg_jobs_noalloc_fwd, ptr(q), d.B, d.S, d.H, d.D, sq[0], sq[1], sq[2], nc, kp, vp, lens, sbs, table.ss,
           table.sh, n, begin, chunks, kv_ranges ? kb : nullptr, kv_ranges ? kl : nullptr, q_ranges ? qb : nullptr,
           q_ranges ? ql : nullptr, op, lp, (float)scale, flags, stream_of(stream));
    else
      CALL(dt_attn_seg_jobs_ws_fwd, ptr(q), d.B, d.S, d.H, d.D, sq[0], sq[1], sq[2], nc, kp, vp, lens, sbs, table.ss,
           table.sh, n, begin, chunks, kv_ranges ? kb : nullptr, kv_ranges ? kl : nullptr, q_ranges ? qb : nullptr,
           q_ranges ? ql : nullptr, op, lp, (float)scale, flags, ptr(workspace), bytes_of(workspace), stream_of(stream));
    start = end;
  }
}

Tensor new_out(const Dims& d, at::ScalarType dtype, const Tensor& like) {
  return empty({d.B, d.S, d.H, d.D}, like.options().dtype(dtype));
}
Tensor new_lse(const Dims& d, bool bsh, const Tensor& like) {
  const auto opt = like.options().dtype(at::kFloat);
  return bsh ? empty({d.B, d.S, d.H, 1}, opt) : empty({d.B, d.H, d.S}, opt);
}
typedef std::vector<std::pair<Tensor, Tensor>> States;

std::pair<Tensor, Tensor> merge(const std::vector<Tensor>& outs, const std::vector<Tensor>& lses, std::optional<Tensor> dst_out,
                                std::optional<Tensor> dst_lse, at::ScalarType dst_dtype, bool dst_bsh, uint64_t stream);

// The counters of a launch that merges n_states states into one of dst_dtype (see dt_merge_result); none where it cannot, or where its
// sizes are better served by the merge kernel behind it.  Only a launch that merges asks for them, with counters(how many): host work, and
// memory of the stream's.  `counters` may be the stream's set itself.
std::optional<Tensor> merge_counters(const Tensor& q, const Dims& d, at::ScalarType dst_dtype, int32_t flags, int64_t n_jobs,
                                     bool host_listed, int64_t key_tiles, int64_t n_states, const py::object& counters) {
  if (counters.is_none() || (flags & DT_ATTN_Q_PRESCALED) || (dst_dtype != at::kFloat && dst_dtype != q.scalar_type()) ||
      d.H * d.D * 32 * 4 >= (1ll << 31))
    return std::nullopt;
  const int need = dt_attn_merges_in_launch(d.B, d.S, d.H, d.D, n_jobs, host_listed, key_tiles, n_states);
  if (need == 0) return std::nullopt;
  // (a set that is kept already, or who is asked for one; a set too small for this launch: as if there were none)
  const bool kept = !PyCallable_Check(counters.ptr());
  auto c = py::cast<std::optional<Tensor>>(kept ? counters : counters(need));
  if (kept && c->numel() < need) return std::nullopt;
  REQUIRE(!c || (c->is_cuda() && c->scalar_type() == at::kInt && c->is_contiguous()), "counters must be int32 on the GPU");
  return c;   // (their number is checked with the launch)
}
int64_t tiles_of(const ChunkTable& table, int32_t c) { return (table.len[c] + 63) / 64; }
dt_merge_result merge_into(const Tensor& out, const Tensor& lse, const Tensor& counters) {
  return {ptr(out), static_cast<float*>(ptr(lse)), dtype_code(out), 0, nullptr, nullptr, static_cast<uint32_t*>(ptr(counters)), counters.numel()};
}

// What attn_states merges behind its launch, or with it: `outs`, `lses` and then states[which[..]].
struct StatesMerge {
  std::vector<Tensor> outs, lses;
  std::vector<int32_t> which;
  at::ScalarType dtype;
  py::object counters;
  std::pair<Tensor, Tensor> result;
};

// The fresh states (out in q's dtype, lse [B,H,Sq]) of q against the concatenations of the chunks jobs[j]
// (ditango_amd._hip.attn_states): one launch, unless the jobs exceed its limits; a job of more than max_chunks chunks is
// computed in pieces that are folded into its state.
States attn_states(const Tensor& q, const std::vector<Tensor>& ks, const std::vector<Tensor>& vs,
                   const std::vector<std::vector<int32_t>>& jobs, int64_t max_chunks, const std::optional<std::vector<int32_t>>& cu_q,
                   const std::optional<std::vector<std::vector<int32_t>>>& cu_kv, const std::optional<Tensor>& workspace,
                   int32_t flags, const Segments* seg, const py::object& convert, uint64_t stream, StatesMerge* m = nullptr) {
  REQUIRE(q.dim() == 4, "q must be [B,S,H,D] with contiguous D");
  const Dims d{q.size(0), q.size(1), q.size(2), q.size(3)};
  const ChunkTable table(ks, vs, d.B, convert);
  States states, pieces;
  std::vector<std::vector<int32_t>> lists;
  std::vector<Tensor> outs, lses;
  std::vector<int32_t> segs;
  std::vector<Range> q_ranges;
  std::vector<std::vector<Range>> kv_ranges;
  std::vector<std::pair<size_t, size_t>> folds;   // (first piece, number of pieces) of the states computed in pieces
  REQUIRE(max_chunks > 0, "a piece of a job needs at least one chunk");
  REQUIRE(!cu_q || !cu_q->empty(), "cu_seqlens_q needs at least one entry");
  REQUIRE(!cu_q || (cu_kv && cu_kv->size() == ks.size()), "one cu_seqlens_kv per chunk");
  const size_t n_seg = seg ? seg->n_seg() : cu_q ? cu_q->size() - 1 : 1;
  for (const auto& job : jobs) {
    for (int32_t c : job)
      REQUIRE(c >= 0 && c < table.n, "a job references chunk ", std::to_string(c), " outside the table of ", std::to_string(table.n));
    states.emplace_back(new_out(d, q.scalar_type(), q), new_lse(d, false, q));
    const size_t first = pieces.size();
    for (size_t at = 0; at == 0 || at < job.size(); at += max_chunks) {
      pieces.push_back(at == 0 ? states.back() : std::make_pair(new_out(d, q.scalar_type(), q), new_lse(d, false, q)));
      const std::vector<int32_t> piece(job.begin() + at, job.begin() + std::min(job.size(), at + (size_t)max_chunks));
      for (size_t s = 0; s < n_seg; ++s) {   // a segment of a packed batch is a job of its own on the state's rows
        lists.push_back(piece);
        outs.push_back(pieces.back().first);
        lses.push_back(pieces.back().second);
        if (seg) segs.push_back((int32_t)s);
        if (cu_q) {
          q_ranges.emplace_back((*cu_q)[s], (*cu_q)[s + 1] - (*cu_q)[s]);
          auto& r = kv_ranges.emplace_back();
          for (int32_t c : piece) {
            REQUIRE((*cu_kv)[c].size() >= cu_q->size(), "cu_seqlens_kv must have at least as many entries as cu_seqlens_q");
            r.emplace_back((*cu_kv)[c][s], (*cu_kv)[c][s + 1] - (*cu_kv)[c][s]);
          }
        }
      }
    }
    if (pieces.size() - first > 1) folds.emplace_back(first, pieces.size() - first);
  }
  if (m) {
    for (int32_t i : m->which) {
      REQUIRE(i >= 0 && (size_t)i < states.size(), "merge of a state that is not computed");
      m->outs.push_back(states[i].first);
      m->lses.push_back(states[i].second);
    }
    // one launch of whole jobs, and states in the form that it reads
    size_t entries = 0;
    for (const auto& list : lists) entries += list.size();
    bool whole = !seg && !cu_q && folds.empty() && !lists.empty() && lists.size() <= DT_MAX_JOBS && entries <= DT_MAX_JOB_ENTRIES &&
                 table.n <= DT_MAX_CHUNKS && m->outs.size() <= DT_MAX_MERGE_LIST;
    const void* state_outs[DT_MAX_MERGE_LIST];
    const float* state_lses[DT_MAX_MERGE_LIST];
    for (size_t i = 0; whole && i < m->outs.size(); ++i) {
      const Tensor &o = m->outs[i], &l = m->lses[i];
      whole = o.scalar_type() == q.scalar_type() && o.is_cuda() && o.is_contiguous() && shape_is(o, {d.B, d.S, d.H, d.D}) &&
              lse_layout(l, d.B, d.S, d.H) == DT_LSE_BHS && (reinterpret_cast<uintptr_t>(ptr(o)) & 15) == 0;
      state_outs[i] = ptr(o);
      state_lses[i] = static_cast<const float*>(ptr(l));
    }
    std::optional<Tensor> counters;
    if (whole) {
      int64_t longest = 0;
      for (const auto& list : lists) {
        int64_t tiles = 0;
        for (int32_t c : list) tiles += tiles_of(table, c);
        longest = std::max(longest, tiles);
      }
      counters = merge_counters(q, d, m->dtype, flags, (int64_t)lists.size(), true, longest, (int64_t)m->outs.size(), m->counters);
    }
    if (counters) {
      m->result = {new_out(d, m->dtype, q), new_lse(d, true, q)};
      dt_merge_result into = merge_into(m->result.first, m->result.second, *counters);
      into.n_states = (int32_t)m->outs.size();
      into.state_outs = state_outs;
      into.state_lses = state_lses;
      attn_jobs(q, table, lists, outs, lses, 0.0, std::nullopt, std::nullopt, workspace, flags, false, nullptr, std::nullopt, stream, &into);
      return states;
    }
  }
  if (lists.empty() && !m) return states;
  if (!lists.empty()) attn_jobs(q, table, lists, outs, lses, 0.0, cu_q ? std::optional(std::move(q_ranges)) : std::nullopt,
            cu_q ? std::optional(std::move(kv_ranges)) : std::nullopt, workspace, flags, false, seg,
            seg ? std::optional(std::move(segs)) : std::nullopt, stream);
  for (const auto& [first, n] : folds) {
    std::vector<Tensor> o, l;
    for (size_t i = 0; i < n; ++i) {
      o.push_back(pieces[first + i].first);
      l.push_back(pieces[first + i].second);
    }
    merge(o, l, o[0], l[0], q.scalar_type(), false, stream);
  }
  if (m) m->result = merge(m->outs, m->lses, std::nullopt, std::nullopt, m->dtype, true, stream);
  return states;
}

// attn_states, and the merge of (outs, lses) and states[which[..]], in the same launch where it can (ditango_amd._hip.attn_states_merge).
std::tuple<States, Tensor, Tensor> attn_states_merge(
    const Tensor& q, const std::vector<Tensor>& ks, const std::vector<Tensor>& vs, const std::vector<std::vector<int32_t>>& jobs,
    int64_t max_chunks, const std::optional<std::vector<int32_t>>& cu_q, const std::optional<std::vector<std::vector<int32_t>>>& cu_kv,
    const std::optional<Tensor>& workspace, int32_t flags, const Segments* seg, const py::object& convert, std::vector<Tensor> outs,
    std::vector<Tensor> lses, std::vector<int32_t> which, at::ScalarType dst_dtype, const py::object& counters, uint64_t stream) {
  REQUIRE(outs.size() == lses.size(), "one lse per state");
  StatesMerge m{std::move(outs), std::move(lses), std::move(which), dst_dtype, counters, {}};
  States states = attn_states(q, ks, vs, jobs, max_chunks, cu_q, cu_kv, workspace, flags, seg, convert, stream, &m);
  return {std::move(states), m.result.first, m.result.second};
}

// The fp32 states of fp32 q against the concatenations of the fp32 chunks jobs[j] (ditango_amd._hip.attn_jobs_f32_fwd); every
// chunk may have strides of its own.  bsh: lse as [B,Sq,H,1].
States attn_states_f32(const Tensor& q, const std::vector<Tensor>& ks, const std::vector<Tensor>& vs,
                       const std::vector<std::vector<int32_t>>& jobs, double scale, uint64_t stream, bool bsh,
                       const std::optional<Tensor>& workspace, const std::optional<Tensor>& counters) {
  REQUIRE(!counters || (counters->is_cuda() && counters->scalar_type() == at::kInt && counters->is_contiguous()),
          "counters must be int32 on the GPU");
  auto check_f32 = [](const Tensor& t, const Name& name) {
    REQUIRE(t.is_cuda() && t.scalar_type() == at::kFloat && t.dim() == 4 && t.stride(3) == 1, name.str(),
            " must be fp32 [B,S,H,D] on the GPU with contiguous D");
  };
  check_f32(q, {"q"});
  const Dims d{q.size(0), q.size(1), q.size(2), q.size(3)};
  REQUIRE(ks.size() == vs.size(), "need as many V as K chunks");
  for (size_t i = 0; i < ks.size(); ++i) {
    check_f32(ks[i], {"k", (int64_t)i});
    check_f32(vs[i], {"v", (int64_t)i});
    REQUIRE(ks[i].sizes() == vs[i].sizes() && ks[i].size(0) == d.B && ks[i].size(2) == d.H && ks[i].size(3) == d.D, "k/v shape mismatch");
    REQUIRE(ks[i].strides() == vs[i].strides(), "k and v must share strides");
  }
  States states;
  for (size_t j = 0; j < jobs.size(); ++j) {
    states.emplace_back(new_out(d, at::kFloat, q), new_lse(d, bsh, q));
    for (int32_t c : jobs[j]) REQUIRE(c >= 0 && (size_t)c < ks.size(), "job ", std::to_string(j), " references a chunk outside the table");
  }
  for (size_t start = 0; start < jobs.size();) {
    std::vector<int32_t> local(ks.size(), -1);
    const float *kp[DT_MAX_CHUNKS], *vp[DT_MAX_CHUNKS];
    int32_t lens[DT_MAX_CHUNKS], begin[DT_MAX_JOBS + 1], chunks[DT_MAX_JOB_ENTRIES];
    int64_t sb[DT_MAX_CHUNKS], ss[DT_MAX_CHUNKS], sh[DT_MAX_CHUNKS];
    float *op[DT_MAX_JOBS], *lp[DT_MAX_JOBS];
    int32_t nc = 0, e = 0, n = 0;
    begin[0] = 0;
    for (; start + n < jobs.size() && n < DT_MAX_JOBS; ++n) {
      const auto& job = jobs[start + n];
      int32_t fresh = 0;
      for (size_t i = 0; i < job.size(); ++i)
        if (local[job[i]] < 0 && std::find(job.begin(), job.begin() + i, job[i]) == job.begin() + i) ++fresh;
      if (nc + fresh > DT_MAX_CHUNKS || e + job.size() > DT_MAX_JOB_ENTRIES) break;
      for (int32_t c : job) {
        if (local[c] < 0) {
          local[c] = nc;
          kp[nc] = static_cast<const float*>(ptr(ks[c]));
          vp[nc] = static_cast<const float*>(ptr(vs[c]));
          lens[nc] = (int32_t)ks[c].size(1);
          sb[nc] = ks[c].stride(0); ss[nc] = ks[c].stride(1); sh[nc] = ks[c].stride(2);
          ++nc;
        }
        chunks[e++] = local[c];
      }
      begin[n + 1] = e;
      op[n] = static_cast<float*>(ptr(states[start + n].first));
      lp[n] = static_cast<float*>(ptr(states[start + n].second));
    }
    REQUIRE(n > 0, "job ", std::to_string(start), " references more chunks than one launch addresses: split it and merge the parts");
    CALL(dt_attn_jobs_f32_ws_fwd, static_cast<const float*>(ptr(q)), d.B, d.S, d.H, d.D, q.stride(0), q.stride(1), q.stride(2),
         nc, kp, vp, lens, sb, ss, sh, n, begin, chunks, op, lp, bsh ? DT_LSE_BSH : DT_LSE_BHS, (float)scale, ptr(workspace),
         bytes_of(workspace), static_cast<uint32_t*>(ptr(counters)), counters ? counters->numel() : 0, stream_of(stream));
    start += n;
  }
  return states;
}

// Device-scheduled launch over a table that fits one launch (ditango_amd._hip.attn_sched_fwd).  The schedule is row `row`
// of ids [rows, C] and counts [rows, 2] (or the tensors themselves, row 0).
void attn_sched(const Tensor& q, const ChunkTable& table, const Tensor& ids, const Tensor& count, int64_t row, int32_t max_jobs,
                const Tensor& slot_out, const Tensor& slot_lse, int32_t diag, const std::optional<Tensor>& diag_out,
                const std::optional<Tensor>& diag_lse, double scale, const std::optional<std::vector<Range>>& seg_q,
                const std::optional<std::vector<std::vector<Range>>>& seg_kv, const std::optional<Tensor>& workspace,
                int32_t flags, const Segments* seg, uint64_t stream, const dt_merge_result* merge = nullptr) {
  const Dims d = check_query(q, table);
  REQUIRE(table.n <= DT_MAX_CHUNKS, "the table holds ", std::to_string(table.n), " chunks, one launch addresses ",
          std::to_string(DT_MAX_CHUNKS));
  REQUIRE(ids.scalar_type() == at::kInt && count.scalar_type() == at::kInt && ids.is_cuda() && count.is_cuda(),
          "schedule tensors must be int32 on the GPU");
  const int64_t per_row = ids.dim() > 1 ? ids.size(-1) : ids.numel(), per_count = count.dim() > 1 ? count.size(-1) : count.numel();
  // (row 0 is the tensors themselves: a list of any shape, a count that may be an element of a strided view)
  REQUIRE(ids.is_contiguous() && count.numel() >= 1 &&
              (row == 0 ? ids.numel() >= max_jobs
                        : count.is_contiguous() && per_row >= max_jobs && row > 0 && (row + 1) * per_row <= ids.numel() &&
                              (row + 1) * per_count <= count.numel()),
          "compute id list shorter than max_jobs");
  REQUIRE(slot_out.scalar_type() == q.scalar_type() && slot_out.is_contiguous() && slot_out.dim() == 5 &&
              slot_out.sizes().slice(1) == at::IntArrayRef({d.B, d.S, d.H, d.D}) && slot_out.size(0) >= table.n,
          "slot_out must be contiguous [C,B,Sq,H,D] in q's dtype");
  REQUIRE(slot_lse.scalar_type() == at::kFloat && slot_lse.is_contiguous() && slot_lse.dim() == 4 &&
              slot_lse.sizes().slice(1) == at::IntArrayRef({d.B, d.H, d.S}) && slot_lse.size(0) >= table.n,
          "slot_lse must be contiguous fp32 [C,B,H,Sq]");
  if (diag >= 0 && diag < table.n) {
    REQUIRE(diag_out && diag_lse, "a diag chunk needs (diag_out, diag_lse)");
    check_state(*diag_out, *diag_lse, d, q.scalar_type(), {"diag_out"}, {"diag_lse"});
  }
  const auto sq = q.strides();
  const int32_t* dev_ids = static_cast<const int32_t*>(ptr(ids)) + row * per_row;
  const int32_t* dev_count = static_cast<const int32_t*>(ptr(count)) + row * per_count;
  float* sl = static_cast<float*>(ptr(slot_lse));
  float* dl = static_cast<float*>(ptr(diag_lse));
  if (merge) {   // (whole queries)
    CALL(dt_attn_sched_merge_fwd, ptr(q), d.B, d.S, d.H, d.D, sq[0], sq[1], sq[2], (int32_t)table.n, table.k.data(),
         table.v.data(), table.len.data(), table.sb.data(), table.ss, table.sh, dev_ids, dev_count, max_jobs, ptr(slot_out),
         slot_out.stride(0), sl, slot_lse.stride(0), diag, ptr(diag_out), dl, merge, (float)scale, flags, ptr(workspace),
         bytes_of(workspace), stream_of(stream));
    return;
  }
  if (seg) {
    REQUIRE(!seg_q && !seg_kv, "device segment boundaries replace the host ranges");
    REQUIRE((int64_t)seg->cu_kv.size() == table.n, "one cu_seqlens_kv per chunk of the table");
    const int32_t* cu_kv[DT_MAX_CHUNKS];
    for (int64_t c = 0; c < table.n; ++c) cu_kv[c] = static_cast<const int32_t*>(ptr(seg->cu_kv[c]));
    CALL(dt_attn_sched_varlen_ws_fwd, ptr(q), d.B, d.S, d.H, d.D, sq[0], sq[1], sq[2], (int32_t)table.n, table.k.data(),
         table.v.data(), table.len.data(), table.sb.data(), table.ss, table.sh, dev_ids, dev_count, max_jobs, ptr(slot_out),
         slot_out.stride(0), sl, slot_lse.stride(0), diag, ptr(diag_out), dl, seg->n_seg(),
         static_cast<const int32_t*>(ptr(seg->cu_q)), cu_kv, (int32_t)seg->max_q, (float)scale, flags, ptr(workspace),
         bytes_of(workspace), stream_of(stream));
    return;
  }
  int32_t n_seg = 0, qb[DT_MAX_SEGMENTS], ql[DT_MAX_SEGMENTS], kb[DT_MAX_JOB_ENTRIES], kl[DT_MAX_JOB_ENTRIES];
  if (seg_q) {
    n_seg = (int32_t)seg_q->size();
    REQUIRE(seg_kv && (int64_t)seg_kv->size() == table.n, "seg_kv needs one (begin, length) per chunk and segment");
    REQUIRE(n_seg > 0 && n_seg <= DT_MAX_SEGMENTS && n_seg * table.n <= DT_MAX_JOB_ENTRIES, "need 1..",
            std::to_string(DT_MAX_SEGMENTS), " segments and at most ", std::to_string(DT_MAX_JOB_ENTRIES), " (chunk, segment) pairs");
    for (int32_t s = 0; s < n_seg; ++s) { qb[s] = (*seg_q)[s].first; ql[s] = (*seg_q)[s].second; }
    int32_t e = 0;
    for (const auto& r : *seg_kv) {
      REQUIRE((int32_t)r.size() == n_seg, "seg_kv needs one (begin, length) per chunk and segment");
      for (const Range& x : r) { kb[e] = x.first; kl[e++] = x.second; }
    }
  }
  CALL(dt_attn_sched_seg_ws_fwd, ptr(q), d.B, d.S, d.H, d.D, sq[0], sq[1], sq[2], (int32_t)table.n, table.k.data(),
       table.v.data(), table.len.data(), table.sb.data(), table.ss, table.sh, dev_ids, dev_count, max_jobs, ptr(slot_out),
       slot_out.stride(0), sl, slot_lse.stride(0), diag, ptr(diag_out), dl, n_seg, n_seg ? qb : nullptr, n_seg ? ql : nullptr,
       n_seg ? kb : nullptr, n_seg ? kl : nullptr, (float)scale, flags, ptr(workspace), bytes_of(workspace),
       stream_of(stream));
}

// ---- states ------------------------------------------------------------------------------------------------

struct StateList {   // the states of one merge launch
  int32_t n = 0;
  const void* out[DT_MAX_MERGE];
  const float* lse[DT_MAX_MERGE];
  int32_t dtype[DT_MAX_MERGE], layout[DT_MAX_MERGE];
  void add(const void* o, const void* l, int32_t dt, int32_t lay) {
    out[n] = o;
    lse[n] = static_cast<const float*>(l);
    dtype[n] = dt;
    layout[n++] = lay;
  }
  void launch(const Tensor& dst_out, const Tensor& dst_lse, const Dims& d, uint64_t stream) const {
    CALL(dt_merge_states, n, out, lse, dtype, layout, ptr(dst_out), dtype_code(dst_out), static_cast<float*>(ptr(dst_lse)),
         lse_layout(dst_lse, d.B, d.S, d.H), d.B, d.S, d.H, d.D, stream_of(stream));
  }
};

// N-way merge; more states than one launch folds run in rounds through a running fp32 state (ditango_amd._hip.merge_states).
std::pair<Tensor, Tensor> merge(const std::vector<Tensor>& outs, const std::vector<Tensor>& lses, std::optional<Tensor> dst_out,
                                std::optional<Tensor> dst_lse, at::ScalarType dst_dtype, bool dst_bsh, uint64_t stream) {
  const size_t n = outs.size();
  REQUIRE(n > 0 && n == lses.size(), "need at least one state and one lse per state");
  REQUIRE(outs[0].dim() == 4, "outs[0] must be contiguous [B,Sq,H,D] on the GPU");
  const Dims d{outs[0].size(0), outs[0].size(1), outs[0].size(2), outs[0].size(3)};
  if (!dst_out) dst_out = new_out(d, dst_dtype, outs[0]);
  if (!dst_lse) dst_lse = new_lse(d, dst_bsh, outs[0]);
  REQUIRE(dst_out->is_contiguous() && shape_is(*dst_out, {d.B, d.S, d.H, d.D}), "dst_out must be contiguous [B,Sq,H,D]");
  StateList s;
  Tensor run_out, run_lse;
  for (size_t i = 0; i < n; ++i) {
    const Tensor &o = outs[i], &l = lses[i];
    REQUIRE(o.is_cuda() && o.is_contiguous() && shape_is(o, {d.B, d.S, d.H, d.D}), Name{"outs", (int64_t)i}.str(),
            " must be contiguous [B,Sq,H,D] on the GPU");
    if (s.n == DT_MAX_MERGE) {
      if (!run_out.defined()) {
        run_out = new_out(d, at::kFloat, outs[0]);
        run_lse = new_lse(d, false, outs[0]);
      }
      s.launch(run_out, run_lse, d, stream);
      s.n = 0;
      s.add(ptr(run_out), ptr(run_lse), DT_FP32, DT_LSE_BHS);
    }
    s.add(ptr(o), ptr(l), dtype_code(o), lse_layout(l, d.B, d.S, d.H));
  }
  s.launch(*dst_out, *dst_lse, d, stream);
  return {*dst_out, *dst_lse};
}

// Merge of every slot of an arena ([C,B,Sq,H,D] / [C,B,H,Sq]), slot `diag` replaced by (diag_out, diag_lse).
std::pair<Tensor, Tensor> merge_arena(const Tensor& arena_out, const Tensor& arena_lse, int64_t diag, const Tensor& diag_out,
                                      const Tensor& diag_lse, at::ScalarType dst_dtype, uint64_t stream) {
  REQUIRE(arena_out.dim() == 5 && arena_out.is_cuda() && arena_out.is_contiguous(), "the arena must be contiguous [C,B,Sq,H,D]");
  const int64_t C = arena_out.size(0);
  const Dims d{arena_out.size(1), arena_out.size(2), arena_out.size(3), arena_out.size(4)};
  REQUIRE(arena_lse.scalar_type() == at::kFloat && arena_lse.is_contiguous() && shape_is(arena_lse, {C, d.B, d.H, d.S}),
          "the arena's lse must be contiguous fp32 [C,B,H,Sq]");
  if (diag >= 0 && diag < C) check_state(diag_out, diag_lse, d, arena_out.scalar_type(), {"diag_out"}, {"diag_lse"});
  const Tensor dst_out = new_out(d, dst_dtype, arena_out), dst_lse = new_lse(d, true, arena_out);
  const int32_t dt = dtype_code(arena_out);
  const int64_t out_bytes = arena_out.stride(0) * arena_out.element_size(), lse_bytes = arena_lse.stride(0) * 4;
  StateList s;
  Tensor run_out, run_lse;
  for (int64_t c = 0; c < C; ++c) {
    if (s.n == DT_MAX_MERGE) {
      if (!run_out.defined()) {
        run_out = new_out(d, at::kFloat, arena_out);
        run_lse = new_lse(d, false, arena_out);
      }
      s.launch(run_out, run_lse, d, stream);
      s.n = 0;
      s.add(ptr(run_out), ptr(run_lse), DT_FP32, DT_LSE_BHS);
    }
    if (c == diag) s.add(ptr(diag_out), ptr(diag_lse), dt, DT_LSE_BHS);
    else s.add(static_cast<const char*>(ptr(arena_out)) + c * out_bytes, static_cast<const char*>(ptr(arena_lse)) + c * lse_bytes, dt, DT_LSE_BHS);
  }
  s.launch(dst_out, dst_lse, d, stream);
  return {dst_out, dst_lse};
}

// attn_sched on whole queries and the merge of the arena, in the same launch where it can (ditango_amd._hip.attn_sched_merge).
std::pair<Tensor, Tensor> attn_sched_merge(const Tensor& q, const ChunkTable& table, const Tensor& ids, const Tensor& count, int64_t row,
                                           int32_t max_jobs, const Tensor& slot_out, const Tensor& slot_lse, int32_t diag,
                                           const Tensor& diag_out, const Tensor& diag_lse, at::ScalarType dst_dtype,
                                           const std::optional<Tensor>& workspace, const py::object& counters,
                                           int32_t flags, uint64_t stream) {
  const Dims d = check_query(q, table);
  std::optional<Tensor> arrive;
  if (max_jobs > 0 && slot_out.dim() == 5 && slot_out.size(0) == table.n) {
    int64_t longest = 0;
    for (int32_t c = 0; c < table.n; ++c) longest = std::max(longest, tiles_of(table, c));
    arrive = merge_counters(q, d, dst_dtype, flags, max_jobs, false, longest, table.n, counters);
  }
  if (arrive) {
    const Tensor out = new_out(d, dst_dtype, q), lse = new_lse(d, true, q);
    const dt_merge_result into = merge_into(out, lse, *arrive);
    attn_sched(q, table, ids, count, row, max_jobs, slot_out, slot_lse, diag, diag_out, diag_lse, 0.0, std::nullopt, std::nullopt,
               workspace, flags, nullptr, stream, &into);
    return {out, lse};
  }
  attn_sched(q, table, ids, count, row, max_jobs, slot_out, slot_lse, diag, diag_out, diag_lse, 0.0, std::nullopt, std::nullopt,
             workspace, flags, nullptr, stream);
  return merge_arena(slot_out, slot_lse, diag, diag_out, diag_lse, dst_dtype, stream);
}

// One pass from (src_out, src_lse) into (dst_out, dst_lse), any dtypes and lse layouts.
void copy_state(const Tensor& src_out, const Tensor& src_lse, const Tensor& dst_out, const Tensor& dst_lse, uint64_t stream) {
  REQUIRE(src_out.dim() == 4 && src_out.is_cuda() && src_out.is_contiguous(), "the source must be contiguous [B,Sq,H,D] on the GPU");
  const Dims d{src_out.size(0), src_out.size(1), src_out.size(2), src_out.size(3)};
  REQUIRE(dst_out.is_cuda() && dst_out.is_contiguous() && shape_is(dst_out, {d.B, d.S, d.H, d.D}),
          "the destination must be contiguous [B,Sq,H,D] on the GPU");
  CALL(dt_state_copy, ptr(src_out), dtype_code(src_out), static_cast<const float*>(ptr(src_lse)),
       lse_layout(src_lse, d.B, d.S, d.H), ptr(dst_out), dtype_code(dst_out), static_cast<float*>(ptr(dst_lse)),
       lse_layout(dst_lse, d.B, d.S, d.H), d.B, d.S, d.H, d.D, stream_of(stream));
}
void cache_store(const Tensor& src_out, const Tensor& src_lse, const Tensor& slot_out, const Tensor& slot_lse, uint64_t stream) {
  REQUIRE(is_half(slot_out), "slot_out must be contiguous bf16 or fp16 [B,Sq,H,D]");
  REQUIRE(slot_lse.is_contiguous() && src_out.dim() == 4 && shape_is(slot_lse, {src_out.size(0), src_out.size(2), src_out.size(1)}),
          "slot_lse must be contiguous fp32 [B,H,Sq]");
  copy_state(src_out, src_lse, slot_out, slot_lse, stream);
}
std::pair<Tensor, Tensor> cache_load(const Tensor& slot_out, const Tensor& slot_lse, at::ScalarType dst_dtype, bool dst_bsh,
                                     std::optional<Tensor> dst_out, std::optional<Tensor> dst_lse, uint64_t stream) {
  REQUIRE(is_half(slot_out) && slot_out.dim() == 4, "slot_out must be contiguous bf16 or fp16");
  const Dims d{slot_out.size(0), slot_out.size(1), slot_out.size(2), slot_out.size(3)};
  REQUIRE(slot_lse.is_contiguous() && shape_is(slot_lse, {d.B, d.H, d.S}), "slot_lse must be contiguous fp32 [B,H,Sq]");
  if (!dst_out) dst_out = new_out(d, dst_dtype, slot_out);
  if (!dst_lse) dst_lse = new_lse(d, dst_bsh, slot_out);
  copy_state(slot_out, slot_lse, *dst_out, *dst_lse, stream);
  return {*dst_out, *dst_lse};
}

void zero_rows_from(const Tensor& t, const Tensor& first_row, uint64_t stream) {
  REQUIRE(t.is_cuda() && t.is_contiguous() && t.dim() >= 1, "t must be a contiguous device tensor");
  REQUIRE(first_row.is_cuda() && first_row.scalar_type() == at::kInt && first_row.numel() >= 1, "first_row must be int32 on the GPU");
  const int64_t n = t.size(0);
  CALL(dt_zero_rows_from, ptr(t), n, t.numel() / (n > 0 ? n : 1) * t.element_size(),
       static_cast<const int32_t*>(ptr(first_row)), stream_of(stream));
}

// ---- producer ------------------------------------------------------------------------------------------------

// ditango_amd._hip.qk_norm_rope
Tensor qk_norm_rope(const Tensor& x, int32_t norm, const std::optional<Tensor>& weight, const std::optional<Tensor>& bias, double eps,
                    int32_t rope, const std::optional<Tensor>& cos, const std::optional<Tensor>& sin, int32_t rope_begin,
                    std::optional<int32_t> rope_end, const std::vector<int32_t>& sections, int32_t rounding, std::optional<Tensor> out,
                    double out_scale, uint64_t stream) {
  REQUIRE(x.is_cuda() && is_half(x) && x.dim() == 4 && x.stride(3) == 1, "x must be bf16 or fp16 [B,S,H,D] on the GPU");
  const Dims d{x.size(0), x.size(1), x.size(2), x.size(3)};
  if (!out) out = new_out(d, x.scalar_type(), x);
  REQUIRE(out->is_cuda() && out->scalar_type() == x.scalar_type() && out->is_contiguous() && shape_is(*out, {d.B, d.S, d.H, d.D}),
          "out must be a contiguous [B,S,H,D] in x's dtype");
  if (x.scalar_type() == at::kHalf) rounding |= DT_IO_FP16;
  const bool narrow = rounding & DT_WEIGHTS_16;
  for (const auto* t : {&weight, &bias})
    REQUIRE(!*t || ((*t)->is_cuda() && (*t)->scalar_type() == (narrow ? x.scalar_type() : at::kFloat) && (*t)->is_contiguous() &&
                    (*t)->numel() == d.D),
            t == &weight ? "weight" : "bias", " must be ", narrow ? "of the dtype of x" : "fp32", ", [D] on the GPU");
  const int64_t end = rope_end ? *rope_end : d.S, rows = end - rope_begin;
  int64_t table_stride = 0;
  if (rope != DT_ROPE_NONE && rows > 0) {
    for (const auto* t : {&cos, &sin})
      REQUIRE(*t && (*t)->is_cuda() && (*t)->scalar_type() == at::kFloat && (*t)->is_contiguous() && ((*t)->dim() == 2 || (*t)->dim() == 3) &&
                  (*t)->size(-1) == d.D && (*t)->size(-2) == rows,
              t == &cos ? "cos" : "sin", " must be a contiguous fp32 [rows, D] or [B, rows, D] table on the GPU");
    REQUIRE(cos->sizes() == sin->sizes(), "cos and sin must have one shape");
    if (cos->dim() == 3) {
      REQUIRE(cos->size(0) == d.B, "batched tables need B leading entries");
      table_stride = rows * d.D;
    }
  }
  CALL(dt_qk_norm_rope, ptr(x), x.stride(0), x.stride(1), x.stride(2), ptr(*out), d.B, d.S, d.H, d.D, norm, ptr(weight), ptr(bias), (float)eps,
       rope, static_cast<const float*>(ptr(cos)), static_cast<const float*>(ptr(sin)), table_stride, rope_begin, (int32_t)end,
       sections.data(), (int32_t)sections.size(), rounding, (float)out_scale, stream_of(stream));
  return *out;
}

// ditango_amd._hip.qkv_project.  A projection: (weight, bias, norm, norm weight, norm bias, eps, rope).
using Projection = std::tuple<Tensor, std::optional<Tensor>, int32_t, std::optional<Tensor>, std::optional<Tensor>, double, bool>;
std::vector<Tensor> qkv_project(const Tensor& text_rows, const Tensor& video, int64_t heads, const std::vector<Projection>& projections,
                                const std::optional<Tensor>& cos, const std::optional<Tensor>& sin, uint64_t stream) {
  for (const auto* t : {&text_rows, &video})
    REQUIRE(t->is_cuda() && is_half(*t) && t->dim() == 3 && t->stride(2) == 1 && t->scalar_type() == video.scalar_type() && t->size(0) == video.size(0) &&
                t->size(2) == video.size(2),
            "text and video must be bf16 or fp16 [B,tokens,channels] on the GPU, of one dtype");
  REQUIRE(projections.size() == 3 && heads > 0, "three projections and a positive number of heads are needed");
  const int64_t B = video.size(0), T = text_rows.size(1), V = video.size(1), K = video.size(2), D = std::get<0>(projections[0]).size(0) / heads;
  dt_projection table[3] = {};
  std::vector<Tensor> outs;
  for (int i = 0; i < 3; ++i) {
    const auto& [w, bias, norm, norm_w, norm_b, eps, rope] = projections[i];
    REQUIRE(w.is_cuda() && w.scalar_type() == video.scalar_type() && w.is_contiguous() && shape_is(w, {heads * D, K}),
            "weights must be contiguous [heads D, channels] in the tokens' dtype");
    REQUIRE(!bias || (bias->is_cuda() && bias->scalar_type() == video.scalar_type() && bias->is_contiguous() && bias->numel() == heads * D),
            "biases must be [heads D] in the tokens' dtype");
    for (const auto* t : {&norm_w, &norm_b})
      REQUIRE(!*t || ((*t)->is_cuda() && (*t)->scalar_type() == video.scalar_type() && (*t)->is_contiguous() && (*t)->numel() == D),
              "norm parameters must be [D] in the tokens' dtype");
    if (rope)
      for (const auto* t : {&cos, &sin})
        REQUIRE(*t && (*t)->is_cuda() && (*t)->scalar_type() == at::kFloat && (*t)->is_contiguous() && shape_is(**t, {V, D}),
                "cos and sin must be contiguous fp32 [video tokens, D] tables on the GPU");
    outs.push_back(new_out(Dims{B, T + V, heads, D}, video.scalar_type(), video));
    table[i] = {ptr(w), ptr(bias), ptr(outs.back()), ptr(norm_w), ptr(norm_b), norm, rope, (float)eps};
  }
  const int32_t rounding = video.scalar_type() == at::kHalf ? DT_IO_FP16 : 0;
  CALL(dt_qkv_project, ptr(text_rows), text_rows.stride(0), text_rows.stride(1), (int32_t)T, ptr(video), video.stride(0), video.stride(1), (int32_t)V, (int32_t)B,
       (int32_t)K, (int32_t)heads, (int32_t)D, table, static_cast<const float*>(ptr(cos)), static_cast<const float*>(ptr(sin)), rounding,
       stream_of(stream));
  return outs;
}

// ---- host state of a call -------------------------------------------------------------------------------------

// Element [row, col] of a 2-D int64 tensor in host memory, or nothing where it is another one or the place is not there.
std::optional<int64_t> element(const Tensor& t, int64_t row, int64_t col) {
  if (!t.device().is_cpu() || t.layout() != at::kStrided || t.scalar_type() != at::kLong || t.is_neg() || t.dim() != 2 || row < 0 || row >= t.size(0) ||
      col < 0 || col >= t.size(1))
    return std::nullopt;
  return t.const_data_ptr<int64_t>()[row * t.stride(0) + col * t.stride(1)];
}
// Bytes that PyTorch's allocator has handed out on a device.
int64_t allocated_bytes(int64_t device) {
  return c10::getDeviceAllocator(at::kCUDA)->getDeviceStats((c10::DeviceIndex)device).allocated_bytes[0].current;
}

}  // namespace

PYBIND11_MODULE(_ditango_host, m) {
  m.def("set_error_class", [](py::object cls) { g_error = cls.release(); });
  m.def("lse_layout", &lse_layout);
  py::class_<ChunkTable>(m, "ChunkTable")
      .def(py::init<const std::vector<Tensor>&, const std::vector<Tensor>&, int64_t, const py::object&>())
      .def_readonly("n", &ChunkTable::n)
      .def_readonly("B", &ChunkTable::B)
      .def_readonly("H", &ChunkTable::H)
      .def_readonly("D", &ChunkTable::D)
      .def_readonly("ss", &ChunkTable::ss)
      .def_readonly("sh", &ChunkTable::sh)
      .def_property_readonly("arrays", [](const ChunkTable& t) {
        std::vector<uint64_t> k, v;
        for (int64_t i = 0; i < t.n; ++i) {
          k.push_back(reinterpret_cast<uint64_t>(t.k[i]));
          v.push_back(reinterpret_cast<uint64_t>(t.v[i]));
        }
        return py::make_tuple(k, v, t.len, t.sb);
      });
  py::class_<Segments>(m, "Segments").def(py::init(&make_segments)).def_property_readonly("n_seg", &Segments::n_seg);
  m.def("attn_jobs", [](const Tensor& q, const ChunkTable& table, const std::vector<std::vector<int32_t>>& jobs,
                        const std::vector<Tensor>& outs, const std::vector<Tensor>& lses, double scale,
                        const std::optional<std::vector<Range>>& q_ranges, const std::optional<std::vector<std::vector<Range>>>& kv_ranges,
                        const std::optional<Tensor>& workspace, int32_t flags, bool no_alloc, const Segments* seg,
                        const std::optional<std::vector<int32_t>>& job_segments, uint64_t stream) {
    attn_jobs(q, table, jobs, outs, lses, scale, q_ranges, kv_ranges, workspace, flags, no_alloc, seg, job_segments, stream);
  });
  m.def("attn_states", [](const Tensor& q, const std::vector<Tensor>& ks, const std::vector<Tensor>& vs,
                          const std::vector<std::vector<int32_t>>& jobs, int64_t max_chunks, const std::optional<std::vector<int32_t>>& cu_q,
                          const std::optional<std::vector<std::vector<int32_t>>>& cu_kv, const std::optional<Tensor>& workspace,
                          int32_t flags, const Segments* seg, const py::object& convert, uint64_t stream) {
    return attn_states(q, ks, vs, jobs, max_chunks, cu_q, cu_kv, workspace, flags, seg, convert, stream);
  });
  m.def("attn_states_merge", &attn_states_merge);
  m.def("attn_states_f32", &attn_states_f32, py::arg("q"), py::arg("ks"), py::arg("vs"), py::arg("jobs"), py::arg("scale"), py::arg("stream"),
        py::arg("bsh") = false, py::arg("workspace") = py::none(), py::arg("counters") = py::none());
  m.def("attn_sched", [](const Tensor& q, const ChunkTable& table, const Tensor& ids, const Tensor& count, int64_t row, int32_t max_jobs,
                         const Tensor& slot_out, const Tensor& slot_lse, int32_t diag, const std::optional<Tensor>& diag_out,
                         const std::optional<Tensor>& diag_lse, double scale, const std::optional<std::vector<Range>>& seg_q,
                         const std::optional<std::vector<std::vector<Range>>>& seg_kv, const std::optional<Tensor>& workspace,
                         int32_t flags, const Segments* seg, uint64_t stream) {
    attn_sched(q, table, ids, count, row, max_jobs, slot_out, slot_lse, diag, diag_out, diag_lse, scale, seg_q, seg_kv, workspace, flags,
               seg, stream);
  });
  m.def("attn_sched_merge", &attn_sched_merge);
  m.def("merge", &merge);
  m.def("merge_arena", &merge_arena);
  m.def("cache_store", &cache_store);
  m.def("cache_load", &cache_load);
  m.def("zero_rows_from", &zero_rows_from);
  m.def("qk_norm_rope", &qk_norm_rope);
  m.def("qkv_project", &qkv_project);
  m.def("element", &element);
  m.def("allocated_bytes", &allocated_bytes);
}
