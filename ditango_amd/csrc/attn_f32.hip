// Chunk attention in fp32 from fp32 inputs: out = softmax(q k^T * scale) v and the natural-log lse.
//
// The 16-bit MFMA kernel (attn_fwd.hip) is the path of the model-sized configurations; this one exists
// for callers that hold fp32 tensors and want the attention of THOSE numbers, not of their bf16
// roundings -- the reference's CPU-runnable configuration (fp32, 512 queries x 4 chunks of 512 keys,
// 4 heads, d = 64, which the reference runs on its torch math path because flash_attn_func takes no
// fp32).  Products and sums are fp32 throughout (v_mfma_f32_32x32x2_f32 multiplies and adds in fp32), so
// results agree with an fp32 or fp64 closed form to rounding error.
//
// What bounds it: the fp32 matrix pipe, 64 cycles per v_mfma_f32_32x32x2_f32 = 157 TFLOP/s.  In that time a
// wavefront only needs one new value per lane of the A operand, so the operands come straight from global
// memory (L1 / L2) into registers: no LDS, no barrier, every wavefront runs on its own.
//   * A wavefront owns 32 queries and walks key tiles of 32.  Scores are computed transposed, S^T = K Q^T: a
//     lane owns ONE query (column lane % 32) and 16 of the tile's keys, so the row maximum is an in-register
//     reduction plus one exchange with lane ^ 32.
//   * An MFMA contracts two values, one per half of the wavefront.  Which two is free as long as both operands
//     agree: halves 0 and 1 take d = 8 j + t and 8 j + 4 + t, so one 16-byte load of K (and of Q) feeds four
//     MFMAs; for O^T += V^T P^T the pair is the two keys whose probabilities the two halves already hold in the
//     same accumulator register, so P goes from the softmax into the MFMA without moving.  The rows of V^T are
//     permuted (row i of block b is d = i * D/32 + b), so one load of V feeds D / 32 MFMAs.
//   * One tile's V is loaded before the score MFMAs, the next tile's K before the P V ones: each has the other
//     product's time (64 to 128 MFMAs) to arrive, with single buffers.
//   * The four wavefronts of a workgroup are four query tiles (KW = 1) or split the keys of one (KW = 4, every
//     fourth tile each, folded through the LDS at the end).
//   * Measured: 12 heads x 2048 queries x 4 chunks of 2048 keys 103 TFLOP/s at d = 64 and 114 at d = 128 (a plain
//     fp32 library GEMM of 8192^3 reaches 154 on the same part); the configuration above, one launch for its four
//     chunks: 18 us against 4 x 220 us on the vector ALU (1.2 TFLOP/s).
#include <cfloat>
#include <cmath>

#include "dt_common.h"

namespace dt {
namespace {

constexpr int kThreadsF32 = 256;
constexpr int kWavesF32 = kThreadsF32 / 64;
constexpr int kTile = 32;   // queries per wavefront, keys per tile

typedef float f32x16 __attribute__((ext_vector_type(16)));
// rows need no more than the 4-byte alignment of their elements
typedef float f32x4 __attribute__((ext_vector_type(4), aligned(4)));
typedef float f32x2 __attribute__((ext_vector_type(2), aligned(4)));

// What stands in for a row of V past the end of a chunk.
__device__ const float kZeroRow[4] = {};

struct AttnF32Args {
  const float* q;
  int64_t q_sb, q_ss, q_sh;
  int32_t B, H, Sq;
  int32_t n_qg;      // query groups (workgroups) per (batch, head)
  int32_t total;     // B * H * n_qg
  int32_t per_xcd;
  float scale, scale_log2;
  // job j attends to the concatenation of the chunks job_chunks[job_begin[j] .. job_begin[j + 1])
  const float* k[DT_MAX_CHUNKS];
  const float* v[DT_MAX_CHUNKS];
  int64_t kv_sb[DT_MAX_CHUNKS], kv_ss[DT_MAX_CHUNKS], kv_sh[DT_MAX_CHUNKS];
  int32_t kv_len[DT_MAX_CHUNKS];
  float* out[DT_MAX_JOBS];
  float* lse[DT_MAX_JOBS];
  int32_t job_begin[DT_MAX_JOBS + 1];
  int32_t job_chunks[DT_MAX_JOB_ENTRIES];
};
static_assert(sizeof(AttnF32Args) <= 4096, "the kernel arguments travel in the 4 KB kernarg segment");

template <int D>
struct F32Lds {
  static constexpr int kPitch = D + 4;             // floats per query row of a wavefront's partial output
  static constexpr int kFloatsPerWave = kTile * kPitch + 2 * kTile;   // + maximum and sum of every query
  static constexpr int kBytes = kWavesF32 * kFloatsPerWave * 4;
};

// D = 64: two wavefronts per SIMD.  D = 128: the operands of a tile (K, V, Q, O: 64
// registers each) leave room for one.
template <int D, int KW>
__global__ __launch_bounds__(kThreadsF32, D == 64 ? 2 : 1) void attn_f32_kernel(const AttnF32Args args_by_value) {
  using L = F32Lds<D>;
  constexpr int kNB = D / 32;      // blocks of 32 output elements
  constexpr int kKL = D / 8;       // 16-byte K loads of a lane per tile
  typedef float vvec __attribute__((ext_vector_type(kNB), aligned(4)));
  // read in place, in the kernarg segment (the struct is the only parameter)
  typedef const AttnF32Args __attribute__((address_space(4))) KernArgs;
  KernArgs& a = *(KernArgs*)__builtin_amdgcn_kernarg_segment_ptr();
  (void)args_by_value;
  extern __shared__ __attribute__((aligned(16))) float lds_f32[];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int col = lane & 31, hh = lane >> 5;
  const int job = blockIdx.y;
  // every XCD works through a contiguous range of heads: its L2 then holds few K / V streams
  const int idx = blockIdx.x >> 3;
  const int item = (int)(blockIdx.x & 7) * a.per_xcd + idx;
  if (idx >= a.per_xcd || item >= a.total) return;
  const int bh = item / a.n_qg;
  const int qg = item - bh * a.n_qg;
  const int b = bh / a.H, h = bh - b * a.H;
  const int q0 = (qg * (kWavesF32 / KW) + wave / KW) * kTile;
  const int kpart = wave % KW;
  if (KW == 1 && q0 >= a.Sq) return;   // (no barrier follows in this variant)

  // Q: B operand, d = 8 j + 4 hh + t (rows past Sq repeat the last one; their results are not stored)
  f32x4 qf[kKL];
  {
    const float* qp = a.q + (int64_t)b * a.q_sb + (int64_t)min(q0 + col, a.Sq - 1) * a.q_ss + (int64_t)h * a.q_sh + 4 * hh;
#pragma unroll
    for (int j = 0; j < kKL; ++j) qf[j] = *reinterpret_cast<const f32x4*>(qp + 8 * j);
  }

  f32x16 o[kNB];
#pragma unroll
  for (int i = 0; i < kNB; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[i][r] = 0.f;
  // The maximum starts at the lowest finite value: a row that has met nothing but scores of -inf then gets weights of
  // exp2(-inf) = 0 and no sum, without a test for it (a test per tile: +1 % at d = 128).
  float m = -FLT_MAX, l = 0.f;
  const float c = a.scale_log2;

  // The cursor: this wavefront's tiles are every KW-th of the job's, counted through its chunks.  Behind the last
  // tile it stays on a chunk with keys, so that the loads below need no branch.
  int seg = a.job_begin[job] - 1;
  const int seg_end = a.job_begin[job + 1];
  int k0 = 0, len = 0;          // first key of the tile, keys of the chunk
  const float *kb = nullptr, *vb = nullptr;   // K / V of the chunk for this batch and head
  int64_t ss = 0;               // its token stride
  int whole = 0;                // its keys, where a lane's offset in a tile of V fits 32 bits
  auto advance = [&](int tiles) __attribute__((always_inline)) -> bool {
    k0 += tiles * kTile;
    while (k0 >= len) {
      int cid = 0, n = 0;
      while (n == 0) {
        if (++seg >= seg_end) return false;
        cid = a.job_chunks[seg];
        n = a.kv_len[cid];
      }
      k0 -= (len + kTile - 1) / kTile * kTile;   // tiles that reach into this chunk
      len = n;
      const int64_t off = (int64_t)b * a.kv_sb[cid] + (int64_t)h * a.kv_sh[cid];
      kb = a.k[cid] + off;
      vb = a.v[cid] + off;
      ss = a.kv_ss[cid];
      whole = (uint64_t)ss < (1u << 28) ? n : 0;
    }
    return true;
  };

  f32x4 kf[kKL];
  vvec vf[16];
  auto load_k = [&]() __attribute__((always_inline)) {
    const float* p = kb + (int64_t)min(k0 + col, len - 1) * ss + 4 * hh;
#pragma unroll
    for (int j = 0; j < kKL; ++j) kf[j] = *reinterpret_cast<const f32x4*>(p + 8 * j);
  };
  // Keys 8 (r / 4) + 4 hh + r % 4 of the tile; past the end zeros, not some key: their probability is 0, and 0 times an
  // infinity would be NaN.  The zeros are loaded, and chunks of a larger stride take the branch of 64-bit offsets: with the
  // loaded rows zeroed behind a test, or 64-bit offsets in whole tiles, every tile takes 1 to 4 % longer (12 heads x 1742 queries
  // x 3484 keys: 405 us at d = 128 and 218 at d = 64 with both, 402 and 211 as it is, and with neither zeros nor large strides).
  auto load_v = [&]() __attribute__((always_inline)) {
    if (k0 + kTile <= whole) {
      const float* p = vb + (int64_t)k0 * ss;
      const uint32_t lane_off = (uint32_t)(4 * hh) * (uint32_t)ss + (uint32_t)(kNB * col);
#pragma unroll
      for (int r = 0; r < 16; ++r)
        vf[r] = *reinterpret_cast<const vvec*>(p + (int64_t)(8 * (r >> 2) + (r & 3)) * ss + lane_off);
    } else {
      // (both pointers in the global address space, or the loads become flat ones)
      typedef const __attribute__((address_space(1))) vvec* Row;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = k0 + 8 * (r >> 2) + 4 * hh + (r & 3);
        const Row row = (Row)(vb + (int64_t)min(key, len - 1) * ss + kNB * col);
        vf[r] = *(key < len ? row : (Row)kZeroRow);
      }
    }
  };

  bool more = advance(kpart);
  if (more) load_k();
  while (more) {
    load_v();
    __builtin_amdgcn_sched_barrier(0);   // V is on its way before the score MFMAs start
    const int valid = len - k0;
    f32x16 s, s_odd;   // two chains: an MFMA that waits for the one before it leaves the pipe idle (D = 64: +12 %)
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = s_odd[r] = 0.f;
#pragma unroll
    for (int j = 0; j < kKL; ++j)
#pragma unroll
      for (int t = 0; t < 4; t += 2) {
        s = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[j][t], qf[j][t], s, 0, 0, 0);
        s_odd = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[j][t + 1], qf[j][t + 1], s_odd, 0, 0, 0);
      }
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] += s_odd[r];
    __builtin_amdgcn_sched_barrier(0);
    more = advance(KW);
    // The next tile's K is on its way before the P V MFMAs (behind the last tile: some K again).  Without a branch:
    // with one, V could only be awaited together with this K.
    load_k();
    __builtin_amdgcn_sched_barrier(0);
    if (valid < kTile) {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (8 * (r >> 2) + 4 * hh + (r & 3) >= valid) s[r] = -INFINITY;
    }
    float mx = s[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    if (__any(mx > m)) {
      const float m_new = fmaxf(m, mx);
      const float alpha = __builtin_amdgcn_exp2f((m - m_new) * c);   // (0 on the first tile, or 1 with nothing to rescale)
      l *= alpha;
#pragma unroll
      for (int i = 0; i < kNB; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[i][r] *= alpha;
      m = m_new;
    }
    // the difference first, then the scale: the exponent is exact to its own rounding however large the scores are
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = __builtin_amdgcn_exp2f((s[r] - m) * c);
      l += s[r];
    }
#pragma unroll
    for (int r = 0; r < 16; ++r)
#pragma unroll
      for (int i = 0; i < kNB; ++i) {
        float vi;
        if constexpr (kNB == 2) vi = i == 0 ? vf[r].x : vf[r].y;
        else vi = vf[r][i];
        o[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(vi, s[r], o[i], 0, 0, 0);
      }
  }
  l += __shfl_xor(l, 32);

  // ---- epilogue: O^T -> LDS as [query][d], then whole rows to memory; with KW > 1 the parts are folded on the way
  float* mine = lds_f32 + wave * L::kFloatsPerWave;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    vvec row;
#pragma unroll
    for (int i = 0; i < kNB; ++i) row[i] = o[i][r];
    *reinterpret_cast<vvec*>(mine + col * L::kPitch + (8 * (r >> 2) + 4 * hh + (r & 3)) * kNB) = row;
  }
  if (hh == 0) {
    mine[kTile * L::kPitch + col] = m;
    mine[kTile * L::kPitch + kTile + col] = l;
  }
  if constexpr (KW > 1) __syncthreads();
  else asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // a wavefront reads back only what it wrote itself
  const float* parts = lds_f32 + (wave - kpart) * L::kFloatsPerWave;
  constexpr int kLanesPerRow = D / 4;
  constexpr int kRowsPerPass = 64 / kLanesPerRow;
  constexpr int kRowsPerWave = kTile / KW;
  float* out = a.out[job];
  float* lse = a.lse[job];
#pragma unroll
  for (int p = 0; p < kRowsPerWave; p += kRowsPerPass) {
    const int row = kpart * kRowsPerWave + p + lane / kLanesPerRow;
    const int d = (lane % kLanesPerRow) * 4;
    float mm = -INFINITY;
#pragma unroll
    for (int w = 0; w < KW; ++w) mm = fmaxf(mm, parts[w * L::kFloatsPerWave + kTile * L::kPitch + row]);
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    float den = 0.f;
#pragma unroll
    for (int w = 0; w < KW; ++w) {
      const float* pw = parts + w * L::kFloatsPerWave;
      const float lw = pw[kTile * L::kPitch + kTile + row];
      const float ww = KW == 1 ? 1.f : (lw == 0.f ? 0.f : __builtin_amdgcn_exp2f((pw[kTile * L::kPitch + row] - mm) * c));
      const f32x4 x = *reinterpret_cast<const f32x4*>(pw + row * L::kPitch + d);
      den = fmaf(ww, lw, den);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] = fmaf(ww, x[e], acc[e]);
    }
    if (q0 + row < a.Sq) {
      const float inv = den > 0.f ? 1.f / den : 0.f;
      f32x4 y;
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = acc[e] * inv;
      *reinterpret_cast<f32x4*>(out + (((int64_t)b * a.Sq + q0 + row) * a.H + h) * D + d) = y;
      if (d == 0) lse[((int64_t)b * a.H + h) * a.Sq + q0 + row] = den > 0.f ? mm * a.scale + logf(den) : -INFINITY;
    }
  }
}

template <int D, int KW>
int launch_f32(AttnF32Args& a, int n_jobs, hipStream_t stream) {
  // more than 64 KB of dynamic LDS has to be allowed once per kernel and device
  static thread_local int allowed_dev = -1;
  int dev = 0;
  if (int rc = hip_fail(hipGetDevice(&dev), "hipGetDevice")) return rc;
  if (allowed_dev != dev) {
    if (int rc = hip_fail(hipFuncSetAttribute(reinterpret_cast<const void*>(&attn_f32_kernel<D, KW>),
                                              hipFuncAttributeMaxDynamicSharedMemorySize, F32Lds<D>::kBytes),
                          "hipFuncSetAttribute"))
      return rc;
    allowed_dev = dev;
  }
  constexpr int kQueries = kTile * kWavesF32 / KW;
  a.n_qg = (a.Sq + kQueries - 1) / kQueries;
  a.total = a.B * a.H * a.n_qg;
  a.per_xcd = (a.total + 7) / 8;
  hipLaunchKernelGGL((attn_f32_kernel<D, KW>), dim3((unsigned)a.per_xcd * 8u, (unsigned)n_jobs, 1), dim3(kThreadsF32),
                     F32Lds<D>::kBytes, stream, a);
  return hip_fail(hipGetLastError(), "attn_f32 launch");
}

}  // namespace
}  // namespace dt

using namespace dt;

extern "C" int dt_attn_jobs_f32_fwd(const float* q, int32_t B, int32_t Sq, int32_t H, int32_t D, int64_t q_sb, int64_t q_ss,
                                    int64_t q_sh, int32_t n_chunks, const float* const* k_ptrs,
                                    const float* const* v_ptrs, const int32_t* kv_lens, const int64_t* kv_sb,
                                    const int64_t* kv_ss, const int64_t* kv_sh, int32_t n_jobs, const int32_t* job_begin,
                                    const int32_t* job_chunks, float* const* out_ptrs, float* const* lse_ptrs,
                                    float softmax_scale, void* stream) {
  if (B <= 0 || Sq <= 0 || H <= 0) {
    set_error("B, Sq, H must be positive (got %d, %d, %d)", B, Sq, H);
    return DT_ERR_INVALID;
  }
  if (D != 64 && D != 128) {
    set_error("head dim %d not built (64 and 128 are)", D);
    return DT_ERR_UNSUPPORTED;
  }
  if (n_chunks < 0 || n_chunks > DT_MAX_CHUNKS || (n_chunks > 0 && (!k_ptrs || !v_ptrs || !kv_lens || !kv_sb || !kv_ss || !kv_sh))) {
    set_error("%d KV chunks: need 0..%d and a chunk table", n_chunks, DT_MAX_CHUNKS);
    return DT_ERR_INVALID;
  }
  if (n_jobs == 0) return DT_OK;
  if (!q || n_jobs < 0 || n_jobs > DT_MAX_JOBS || !job_begin || !job_chunks || !out_ptrs || !lse_ptrs) {
    set_error("%d jobs: need 0..%d, a query tensor and non-null job tables", n_jobs, DT_MAX_JOBS);
    return DT_ERR_INVALID;
  }
  const int64_t units = (int64_t)B * H * ((Sq + kTile - 1) / kTile);   // query tiles of a job
  if (units > (1 << 28)) {
    set_error("too many query tiles (%lld)", (long long)units);
    return DT_ERR_INVALID;
  }
  AttnF32Args a{};
  a.q = q;
  a.q_sb = q_sb; a.q_ss = q_ss; a.q_sh = q_sh;
  a.B = B; a.H = H; a.Sq = Sq;
  a.scale = softmax_scale > 0.f ? softmax_scale : 1.0f / std::sqrt((float)D);
  a.scale_log2 = a.scale * 1.4426950408889634f;
  for (int i = 0; i < n_chunks; ++i) {
    if (kv_lens[i] < 0 || (kv_lens[i] > 0 && (!k_ptrs[i] || !v_ptrs[i]))) {
      set_error("chunk %d: negative length or null k/v", i);
      return DT_ERR_INVALID;
    }
    a.k[i] = k_ptrs[i]; a.v[i] = v_ptrs[i];
    a.kv_len[i] = kv_lens[i]; a.kv_sb[i] = kv_sb[i]; a.kv_ss[i] = kv_ss[i]; a.kv_sh[i] = kv_sh[i];
  }
  if (job_begin[0] != 0) {
    set_error("job_begin must start at 0");
    return DT_ERR_INVALID;
  }
  for (int j = 0; j < n_jobs; ++j) {
    if (job_begin[j + 1] < job_begin[j] || job_begin[j + 1] > DT_MAX_JOB_ENTRIES) {
      set_error("job_begin must be monotone and end at most at %d (job %d)", DT_MAX_JOB_ENTRIES, j);
      return DT_ERR_INVALID;
    }
    if (!out_ptrs[j] || !lse_ptrs[j]) {
      set_error("job %d: null destination", j);
      return DT_ERR_INVALID;
    }
    a.out[j] = out_ptrs[j]; a.lse[j] = lse_ptrs[j];
    a.job_begin[j] = job_begin[j];
  }
  a.job_begin[n_jobs] = job_begin[n_jobs];
  for (int e = 0; e < job_begin[n_jobs]; ++e) {
    if (job_chunks[e] < 0 || job_chunks[e] >= n_chunks) {
      set_error("job chunk reference %d is outside the chunk table", job_chunks[e]);
      return DT_ERR_INVALID;
    }
    a.job_chunks[e] = job_chunks[e];
  }
  // One wavefront per SIMD takes 1024 query tiles.  Below three such rounds the last one is rarely full and splitting
  // the keys four ways fills it (12 heads x 2048 queries x 2 chunks, 1536 tiles: 270 instead of 346 us at d = 64, 479
  // instead of 601 at d = 128; 256 tiles: 40 instead of 110 us); from there on four query tiles that read the same keys
  // are the better neighbours in a workgroup (3072 tiles: 500 each at d = 64, 908 instead of 954 us at d = 128).
  // The line holds for chunks of 256 keys and more.  A wavefront with a tile or less pays for the exchange of the parts without a
  // shorter loop: 24 heads x 2048 queries x 512 keys 79 split, 96 us unsplit at d = 64, 153 and 165 at d = 128, but x 64 keys 27 and 21,
  // 60 and 39.  Short chunks are launches of tens of us either way and up to 512 query tiles split well too (4 heads x 512 x 64 keys
  // 6.8 and 10.7 us), so the number of keys is left out of the rule.
  const bool split = units * n_jobs < 3 * 1024;
  if (D == 128)
    return split ? launch_f32<128, 4>(a, n_jobs, (hipStream_t)stream) : launch_f32<128, 1>(a, n_jobs, (hipStream_t)stream);
  return split ? launch_f32<64, 4>(a, n_jobs, (hipStream_t)stream) : launch_f32<64, 1>(a, n_jobs, (hipStream_t)stream);
}

extern "C" int dt_attn_chunk_f32_fwd(const float* q, const float* k, const float* v, float* out, float* lse, int32_t B,
                                     int32_t Sq, int32_t Sk, int32_t H, int32_t D, int64_t q_sb, int64_t q_ss,
                                     int64_t q_sh, int64_t kv_sb, int64_t kv_ss, int64_t kv_sh, float softmax_scale,
                                     void* stream) {
  if (Sk < 0) {
    set_error("Sk must be non-negative (got %d)", Sk);
    return DT_ERR_INVALID;
  }
  const int32_t begin[2] = {0, 1}, chunk = 0;
  return dt_attn_jobs_f32_fwd(q, B, Sq, H, D, q_sb, q_ss, q_sh, 1, &k, &v, &Sk, &kv_sb, &kv_ss, &kv_sh, 1, begin, &chunk, &out,
                              &lse, softmax_scale, stream);
}
