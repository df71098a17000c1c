// Chunk attention in fp32 from fp32 inputs: out = softmax(q k^T * scale) v and the natural-log lse.
//
// The 16-bit MFMA kernel (attn_fwd.hip) is the path of the model-sized configurations; this one exists
// for callers that hold fp32 tensors and want the attention of THOSE numbers, not of their bf16
// roundings -- the reference's CPU-runnable configuration (fp32, 512 queries x 4 chunks of 512 keys,
// 4 heads, d = 64, which the reference runs on its torch math path because flash_attn_func takes no
// fp32).
//
// The products run on the bf16 matrix pipe, 16 times the rate of the fp32 one: every fp32 operand is split into three bf16 values h + m +
// l, 3 x 8 bits, which leaves nothing out, and a product is the sum of the six terms hh, hm, mh, mm, hl, lh; what is dropped (ml, lm, ll) is
// below 2^-25 of the product, less than the one rounding of an fp32 multiply-add.  Small terms are added first, and a tile's share of O^T is
// summed for itself and then added once.  Against fp64, over 22 launches of 96 ... 1680 queries x 190 ... 9560 keys: relative error (2-norm)
// 1.6 ... 2.4e-7, where v_mfma_f32_32x32x2_f32 (64 cycles for two values a lane) gave 2.9 ... 4.6e-7 of the same numbers.
// Numbers that do not split -- infinities, NaN, what ends below the exponent range -- show in Q or in the result (NaN, or less than
// 2^-100); a wavefront that sees them walks its keys once more with fp32 products and takes the elements or rows concerned from there.
// What does not show: a weight below 2^-110 loses up to 2^-126, which counts where its V is more than 2^100 times the result, and an element
// of K below 2^-110 as much, which with |Q| <= 2^90 is 2^-36 of a score.
//
// What bounds it: a wavefront issues in order, and an MFMA holds it up (24 MFMAs with 88 vector instructions between them take about as
// long as one behind the other), so a tile takes 48 MFMAs x 32 cycles + 330 vector instructions x 4 at d = 64 (twice the MFMAs at 128), less what
// the other wavefront of the SIMD hides of it: counters of 8 heads x 1195 queries x 9560 keys, MFMA pipe busy 46 % of the SIMDs' cycles, vector
// ALU 49 %, both at once in a third of the former.  So the split of K and V, half of the vector instructions where every wavefront does its
// own (7 of them per MFMA against 15), is shared:
//   * QW (2 or 4) wavefronts of a workgroup own 32 queries each and walk the same key tiles of 32.  Each loads its share of a tile in whole
//     lines, a turn ahead, splits it and puts the three parts into the LDS, from where all read operands (16-byte reads of K,
//     transposing reads of V, as in attn_fwd.hip).  The KW = 4 / QW groups of a workgroup take every KW-th tile.
//   * Scores are computed transposed, S^T = K Q^T: a lane owns ONE query (column lane % 32) and 16 of the tile's keys, the row maximum is an
//     in-register reduction plus one exchange with lane ^ 32, and with the rows of K permuted the probabilities are where the
//     second product needs them.
//   * In a small launch nothing is shared (QW = 1): a wavefront splits all of its tiles from memory to registers, and nobody waits for anybody.
//   * Where the queries alone leave the chip idle, `parts` workgroups share the keys of a work item (plan_f32).
//   * Measured (us per call with the GPU kept busy, kernel of fp32 products and merge kernel behind it -> this, which needs no other):
//     4 heads x 512 queries x 2048 keys, d = 64 30 -> 19; 12 x 1053 x 4212 163 -> 101; 8 x 1195 x 9560 258 -> 153 (157 TFLOP/s, as much as
//     the fp32 pipe has); d = 128 12 x 355 x 2840 107 -> 72, 10 x 847 x 1694 120 -> 72.
#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstddef>
#include <mutex>
#include <type_traits>

#include "dt_common.h"

namespace dt {
namespace {

constexpr int kThreadsF32 = 256;
constexpr int kWavesF32 = kThreadsF32 / 64;
constexpr int kTile = 32;   // queries per wavefront, keys per tile
constexpr int kMaxParts = 16;   // workgroups that share the key tiles of a work item

typedef float f32x16 __attribute__((ext_vector_type(16)));
// rows need no more than the 4-byte alignment of their elements
typedef float f32x4 __attribute__((ext_vector_type(4), aligned(4)));
typedef float f32x2 __attribute__((ext_vector_type(2), aligned(4)));

constexpr int kDevice = 16;   // cache-policy bit of a raw buffer access: device scope (sc1)
typedef __amdgpu_buffer_rsrc_t Rsrc;
__device__ __forceinline__ Rsrc buffer_of(const void* base, uint32_t valid_bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, valid_bytes, 0x00020000);
}
__device__ __forceinline__ f32x4 load4(Rsrc r, uint32_t off, uint32_t uniform_off) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, uniform_off, 0));
}
__device__ __forceinline__ f32x2 load2(Rsrc r, uint32_t off, uint32_t uniform_off) {
  return __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(r, off, uniform_off, 0));
}

struct F32Chunk {
  const float *k, *v;
  int64_t sb, ss, sh;   // element strides
  int64_t len;
};
struct F32Job {
  float *out, *lse;
  int32_t begin, end;
};
struct AttnF32Args {
  const float* q;
  int64_t q_sb, q_ss, q_sh;
  int32_t B, H, Sq, D;
  int32_t parts;     // workgroups that share the key tiles of a work item
  int32_t lse_bsh;   // lse as [B,Sq,H] instead of [B,H,Sq]
  // parts > 1: sums, relative to the part's maximum, [part][job][item][32 QW queries][D], and behind them (maximum, sum of weights) of
  // every query; arrival counters, one per job and item, zero between launches
  float* ws;
  uint32_t* arrive;
  int32_t n_qg;      // query groups (workgroups) per (batch, head)
  int32_t total;     // B * H * n_qg
  int32_t per_xcd;
  float scale, scale_log2;
  float grid, inv_grid;
  // job j attends to the concatenation of the chunks refs[job[j].begin .. job[j].end)
  int32_t refs[DT_MAX_JOB_ENTRIES];
  F32Job job[DT_MAX_JOBS];
  F32Chunk chunk[DT_MAX_CHUNKS];
};
static_assert(sizeof(AttnF32Args) <= 4096, "the kernel arguments travel in the 4 KB kernarg segment");

typedef const AttnF32Args __attribute__((address_space(4))) KernArgsF32;
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kJob = (int)offsetof(AttnF32Args, job), kChunk = (int)offsetof(AttnF32Args, chunk), kRefs = (int)offsetof(AttnF32Args, refs);
// Brings the argument lines that a workgroup is about to read into the scalar cache, all at once (see attn_fwd.hip).
__device__ __forceinline__ void prefetch_args(uint64_t args) {
  uint32_t t0, t1, t2, t3, t4, t5, t6, t7, t8, t9, t10;
  asm volatile(
      "s_load_dword %0, %11, 0x0\n\ts_load_dword %1, %11, 0x40\n\ts_load_dword %2, %11, %12\n\ts_load_dword %3, %11, %13\n\t"
      "s_load_dword %4, %11, %14\n\ts_load_dword %5, %11, %15\n\ts_load_dword %6, %11, %16\n\ts_load_dword %7, %11, %17\n\t"
      "s_load_dword %8, %11, %18\n\ts_load_dword %9, %11, %19\n\ts_load_dword %10, %11, %20\n\ts_waitcnt lgkmcnt(0)"
      : "=&s"(t0), "=&s"(t1), "=&s"(t2), "=&s"(t3), "=&s"(t4), "=&s"(t5), "=&s"(t6), "=&s"(t7), "=&s"(t8), "=&s"(t9), "=&s"(t10)
      : "s"(args), "i"(kRefs), "i"(kRefs + 64), "i"(kJob), "i"(kJob + 64), "i"(kChunk), "i"(kChunk + 64), "i"(kChunk + 128),
        "i"(kChunk + 192), "i"(kChunk + 256)
      : "memory");
}

template <int D, int QW>
struct F32Lds {
  // while the keys are walked: three parts of K and of V per group of wavefronts, [32 keys][D] of 16 bits each
  static constexpr int kPlane = kTile * D * 2;
  static constexpr int kGroupBytes = 6 * kPlane;
  __device__ static constexpr int swz_k(int row) { return D == 128 ? (row & 15) : ((row >> 1) & 7); }
  __device__ static constexpr int swz_v(int row) { return D == 128 ? (row & 3) : ((row >> 1) & 1); }
  // behind that: the output rows of every wavefront
  static constexpr int kPitch = D + 4;             // floats per query row of a wavefront's partial output
  static constexpr int kFloatsPerWave = kTile * kPitch + 2 * kTile;   // + maximum and sum of every query
  static constexpr int kWalk = QW == 1 ? 0 : kWavesF32 / QW * kGroupBytes, kEnd = kWavesF32 * kFloatsPerWave * 4;
  // behind both: a flag of every wavefront, and the largest of every column of V in the keys that a lane looked through
  static constexpr int kFlags = kWalk > kEnd ? kWalk : kEnd, kColumns = kFlags + 64;
  static constexpr int kBytes = kColumns + kThreadsF32 * 16;
};
// Transposing LDS read, see attn_fwd.hip.
typedef short s16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ s16x4 lds_read_tr(const uint8_t* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(p));
}

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float pair32 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef short s16x8 __attribute__((ext_vector_type(8)));

// Two fp32 values as the sum of three bf16 ones each: h, the 8 leading bits of the significand rounded to nearest, m the same of
// what is left, l the rest.  24 bits are three times 8: nothing is left behind l.
struct Split2 {
  uint32_t h, m, l;
};
__device__ __forceinline__ Split2 split2(float a, float b) {
  auto round = [](pair32 r) { return __builtin_bit_cast(uint32_t, __builtin_convertvector(r, bf16x2)); };
  auto less = [](pair32 r, uint32_t w) {
    return pair32{r.x - __builtin_bit_cast(float, w << 16), r.y - __builtin_bit_cast(float, w & 0xffff0000u)};
  };
  Split2 s;
  pair32 r = {a, b};
  s.h = round(r);
  r = less(r, s.h);
  s.m = round(r);
  r = less(r, s.m);
  s.l = round(r);
  return s;
}
// Eight values, as an operand of the MFMA.
struct Split8 {
  bf16x8 h, m, l;
};
__device__ __forceinline__ Split8 split8(const float (&x)[8]) {
  u32x4 h, m, l;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const Split2 s = split2(x[2 * i], x[2 * i + 1]);
    h[i] = s.h; m[i] = s.m; l[i] = s.l;
  }
  return {__builtin_bit_cast(bf16x8, h), __builtin_bit_cast(bf16x8, m), __builtin_bit_cast(bf16x8, l)};
}
__device__ __forceinline__ f32x16 mfma16(const bf16x8& a, const bf16x8& b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// Workgroup barrier that waits for this wavefront's LDS traffic only: loads of later tiles stay in flight across it.
__device__ __forceinline__ void tile_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// Magnitudes of an element of Q for which three bf16 values hold what counts of an fp32 one: below 2^-110 the last of them loses bits to
// the end of the exponent range, which 2^90 times as large a K would bring back.
constexpr uint32_t kTiny = (uint32_t)(127 - 100) << 23, kHuge = (uint32_t)(127 + 90) << 23;
struct QRange {
  float most = 0.f;
  uint32_t least = ~0u;   // twice the bits, less one: zero, which is three times zero, is the largest
  __device__ __forceinline__ void add(float x, float y) {
    // (in assembly: fmaxf would first quiet what was loaded)
    asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(most) : "v"(x), "v"(y));
    least = min(least, min((__builtin_bit_cast(uint32_t, x) << 1) - 1, (__builtin_bit_cast(uint32_t, y) << 1) - 1));
  }
  __device__ __forceinline__ bool odd() const { return __builtin_bit_cast(uint32_t, most) > kHuge || least < 2 * kTiny - 1; }
};
// Whether an element of O^T is one that the split products may have got wrong: not finite (an infinity leaves NaN behind where
// it is split), or so small that its terms may have ended below the exponent range, zero among them.  A zero is also what terms of ordinary
// size leave now and then (once in some million elements of random numbers), or a column of V that is zero.
constexpr uint32_t kOddFrom = 0xff000000u - 2 * kTiny;
__device__ __forceinline__ uint32_t oddity(float x) { return (__builtin_bit_cast(uint32_t, x) << 1) - 2 * kTiny; }

// m scale + log(den), rounded about once: the logarithm of den's exponent and of its significand, and the two large terms' sum
// with its error.  ln 2 in two parts after Cody and Waite: 355 / 512, its nearest with ten bits, and what is left of it; the significand between
// the square roots of 1/2 and 2, where its logarithm is smallest.  (Plainly, the rounding of a logarithm of 2 to 5 comes on top: 2-norm error of the lse against fp64, 4 heads x 512
// queries x 2048 keys, 5.2e-8 -> 3.44e-8; the rounding of the exact value to fp32 alone is 3.38e-8.)
__device__ __forceinline__ float lse_of(float m, float den, float scale) {
  if (!(den > 0.f)) return -INFINITY;
  float f = __builtin_amdgcn_frexp_mantf(den);
  float k = (float)__builtin_amdgcn_frexp_expf(den);
  if (f < 0.70710678f) {
    f *= 2.f;
    k -= 1.f;
  }
  constexpr float kLn2Hi = 355.f / 512.f, kLn2Lo = (float)(0.693147180559945309 - 355.0 / 512.0);   // (10 bits: k kLn2Hi is exact)
  const float a = m * scale, b = k * kLn2Hi, sum = a + b;
  if (!(__builtin_fabsf(sum) < INFINITY)) return sum;
  const float back = sum - a;
  const float rest = __builtin_fmaf(m, scale, -a) + ((a - (sum - back)) + (b - back));
  return sum + (rest + __builtin_fmaf(k, kLn2Lo, logf(f)));
}

// The walk through the key tiles of a job that one group of wavefronts works on: `left` tiles, counted through the job's chunks.
template <bool kFar>
struct Cursor {
  int seg, seg_end, left;
  int k0 = 0, len = 0;          // first key of the tile, keys of the chunk
  const float *kb = nullptr, *vb = nullptr;   // K / V of the chunk for this batch and head
  int64_t ss = 0;               // its token stride
  uint32_t plane = 0;           // (!kFar) bytes of the chunk's K (and V) as a buffer, behind which keys read as zeros

  __device__ __forceinline__ Cursor(KernArgsF32& a, int job, int n) : seg(a.job[job].begin - 1), seg_end(a.job[job].end), left(n) {}
  // False behind the last tile: the buffers are then empty, loads touch no memory and return zeros.
  __device__ __forceinline__ bool advance(KernArgsF32& a, int b, int h, int tiles) {
    if (--left < 0) {
      k0 = len = 0;
      plane = 0;
      return false;
    }
    k0 += tiles * kTile;
    while (k0 >= len) {
      int cid = 0, n = 0;
      while (n == 0 && ++seg < seg_end) {   // (there is a chunk: `left` tiles are)
        cid = a.refs[seg];
        n = (int)a.chunk[cid].len;
      }
      k0 -= (len + kTile - 1) / kTile * kTile;   // tiles that reach into this chunk
      len = n;
      const auto& chunk = a.chunk[cid];
      const int64_t off = (int64_t)b * chunk.sb + (int64_t)h * chunk.sh;
      kb = chunk.k + off;
      vb = chunk.v + off;
      ss = chunk.ss;
      plane = ((uint32_t)(n - 1) * (uint32_t)ss + (uint32_t)a.D) * 4u;
    }
    return true;
  }
};

// O^T of 32 queries against the cursor's tiles with fp32 products (v_mfma_f32_32x32x2_f32), straight from global memory, and which half rows of Q
// do not split: for the few wavefronts that have such numbers.  An MFMA contracts two values, one per half of the wavefront; which two is free as long
// as both operands agree: halves 0 and 1 take d = 8 j + t and 8 j + 4 + t, and of P V the two keys whose probabilities they hold in
// the same accumulator register.  Register r of block i is d = (8 (r / 4) + 4 hh + r % 4) D/32 + i.
template <int D, bool kFar>
__device__ __forceinline__ void walk_fp32(KernArgsF32& a, int b, int h, int job, int q0, int first, int step, int n, f32x16 (&o)[D / 32],
                                          float& m, float& l, bool& odd_q) {
  constexpr int kNB = D / 32;
  constexpr int kKL = D / 8;       // 16-byte K loads of a lane per tile
  typedef float vvec __attribute__((ext_vector_type(kNB), aligned(4)));
  const int lane = threadIdx.x & 63, col = lane & 31, hh = lane >> 5;
  const float c = a.scale_log2;
  f32x4 qf[kKL];
  const float* qp = a.q + (int64_t)b * a.q_sb + (int64_t)min(q0 + col, a.Sq - 1) * a.q_ss + (int64_t)h * a.q_sh + 4 * hh;
#pragma unroll
  for (int j = 0; j < kKL; ++j) qf[j] = *reinterpret_cast<const f32x4*>(qp + 8 * j);
  QRange range;
#pragma unroll
  for (int j = 0; j < kKL; ++j)
#pragma unroll
    for (int t = 0; t < 4; t += 2) range.add(qf[j][t], qf[j][t + 1]);
  odd_q = range.odd();
#pragma unroll
  for (int i = 0; i < kNB; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[i][r] = 0.f;
  m = -FLT_MAX;
  l = 0.f;
  Cursor<kFar> at(a, job, n);
  for (bool more = at.advance(a, b, h, first); more; more = at.advance(a, b, h, step)) {
    f32x16 s;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = 0.f;
    const float* p = at.kb + (int64_t)min(at.k0 + col, at.len - 1) * at.ss + 4 * hh;
#pragma unroll
    for (int j = 0; j < kKL; ++j) {
      const f32x4 k = *reinterpret_cast<const f32x4*>(p + 8 * j);
#pragma unroll
      for (int t = 0; t < 4; ++t) s = __builtin_amdgcn_mfma_f32_32x32x2f32(k[t], qf[j][t], s, 0, 0, 0);
    }
    const int valid = at.len - at.k0;
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      if (8 * (r >> 2) + 4 * hh + (r & 3) >= valid) s[r] = -INFINITY;
      mx = fmaxf(mx, s[r]);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    const float m_new = fmaxf(m, mx);
    const float alpha = __builtin_amdgcn_exp2f((m - m_new) * c);
    l *= alpha;
    m = m_new;
#pragma unroll
    for (int i = 0; i < kNB; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[i][r] *= alpha;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = __builtin_amdgcn_exp2f((s[r] - m) * c);
      l += s[r];
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      // (past the end zeros, not some key: 0 times an infinity would be NaN)
      const int key = at.k0 + 8 * (r >> 2) + 4 * hh + (r & 3);
      vvec v = *reinterpret_cast<const vvec*>(at.vb + (int64_t)min(key, at.len - 1) * at.ss + kNB * col);
      if (key >= at.len) v = 0.f;
#pragma unroll
      for (int i = 0; i < kNB; ++i) {
        float vi;
        if constexpr (kNB == 2) vi = i == 0 ? v.x : v.y;
        else vi = v[i];
        o[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(vi, s[r], o[i], 0, 0, 0);
      }
    }
  }
  l += __shfl_xor(l, 32);
}

// QW query tiles of 32 and KW groups of key tiles: wavefront w works on query tile w % QW of the workgroup and on every KW-th key
// tile of the workgroup's part.  The QW wavefronts of a group share what they split; with QW = 1 there is nothing to share, and operands go from
// memory to the registers that the MFMAs read.
template <int D, int QW, bool kFar>
__global__ __launch_bounds__(kThreadsF32, D == 64 ? 2 : 1) void attn_f32_kernel(const AttnF32Args args_by_value) {
  constexpr int KW = kWavesF32 / QW;
  using L = F32Lds<D, QW>;
  constexpr int kNB = D / 32;                 // blocks of 32 output elements
  constexpr int kRowLanes = D / 4;            // lanes that load a key, 16 bytes each
  constexpr int kRowsPer = 64 / kRowLanes;    // keys of a load instruction
  constexpr int kLoads = kTile / (kRowsPer * QW);   // loads of a wavefront per tile and operand
  // read in place, in the kernarg segment (the struct is the only parameter)
  KernArgsF32& a = *(KernArgsF32*)__builtin_amdgcn_kernarg_segment_ptr();
  (void)args_by_value;
  prefetch_args((uint64_t)__builtin_amdgcn_kernarg_segment_ptr());
  extern __shared__ __attribute__((aligned(16))) uint8_t lds_f32[];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int member = wave % QW, group = wave / QW;
  const int col = lane & 31, hh = lane >> 5;
  const int job = blockIdx.y / a.parts, part = blockIdx.y - job * a.parts;
  // every XCD works through a contiguous range of heads: its L2 then holds few K / V streams
  const int idx = blockIdx.x >> 3;
  const int item = (int)(blockIdx.x & 7) * a.per_xcd + idx;
  if (idx >= a.per_xcd || item >= a.total) return;
  const int bh = item / a.n_qg;
  const int qg = item - bh * a.n_qg;
  const int b = bh / a.H, h = bh - b * a.H;
  const int q0 = (qg * QW + member) * kTile;
  const float c = a.scale_log2;

  // key tiles of the job, of which this workgroup takes `turns` times KW from `first` on (the groups in turn)
  int tiles = 0;
  for (int s = a.job[job].begin; s < a.job[job].end; ++s) tiles += ((int)a.chunk[a.refs[s]].len + kTile - 1) / kTile;
  const int per_part = (tiles + a.parts * KW - 1) / (a.parts * KW);
  const int begin = part * per_part * KW, mine_of = min(tiles, begin + per_part * KW) - begin;
  const int turns = mine_of > 0 ? (mine_of + KW - 1) / KW : 0;
  const int n_tiles = mine_of > group ? (mine_of - group + KW - 1) / KW : 0;

  // ---- K and V: a wavefront loads its share of a tile with whole lines, splits it and puts the three parts into the LDS
  Cursor<kFar> at_k(a, job, n_tiles), at_v(a, job, n_tiles);   // K runs two tiles ahead, V one: a load has a whole turn to arrive
  const int d_mine = 4 * (lane % kRowLanes);
  auto row_mine = [&](int i) { return (i * QW + member) * kRowsPer + lane / kRowLanes; };
  f32x4 kreg[kLoads], vreg[kLoads];
  // 16 bytes (or 8) of a row of a tile; zeros past the end of the chunk
  auto load_row = [&](const Cursor<kFar>& at, const float* base, int row, int d, auto x) __attribute__((always_inline)) {
    x = 0.f;
    if constexpr (kFar) {
      const int key = at.k0 + row;
      if (key < at.len) x = *reinterpret_cast<const decltype(x)*>(base + (int64_t)key * at.ss + d);
      return x;
    } else {
      // (the tile's offset is the scalar one: inside the buffer, as the range check subtracts it from the length)
      const uint32_t off = ((uint32_t)row * (uint32_t)at.ss + d) * 4u, tile_off = (uint32_t)at.k0 * (uint32_t)at.ss * 4u;
      if constexpr (sizeof(x) == 16) return load4(buffer_of(base, at.plane), off, tile_off);
      else return load2(buffer_of(base, at.plane), off, tile_off);
    }
  };
  auto load_tile = [&](const Cursor<kFar>& at, const float* base, f32x4 (&reg)[kLoads]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) reg[i] = load_row(at, base, row_mine(i), d_mine, f32x4());
  };
  uint8_t* planes = lds_f32 + group * L::kGroupBytes;
  auto put = [&](uint8_t* to, const f32x4& x) __attribute__((always_inline)) {
    const Split2 lo = split2(x[0], x[1]), hi = split2(x[2], x[3]);
    *reinterpret_cast<u32x2*>(to) = u32x2{lo.h, hi.h};
    *reinterpret_cast<u32x2*>(to + L::kPlane) = u32x2{lo.m, hi.m};
    *reinterpret_cast<u32x2*>(to + 2 * L::kPlane) = u32x2{lo.l, hi.l};
  };
  // rows of 16-bit elements; 16-byte chunks (K) and 64-byte segments (V) are stored permuted by the row, so that neither the reads of
  // 16 bytes a row nor the transposing ones meet in a bank
  auto put_k = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int r = row_mine(i);
      put(planes + r * (2 * D) + 16 * ((d_mine >> 3) ^ L::swz_k(r)) + 2 * (d_mine & 7), kreg[i]);
    }
  };
  auto put_v = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int r = row_mine(i);
      put(planes + 3 * L::kPlane + r * (2 * D) + 64 * ((d_mine >> 5) ^ L::swz_v(r)) + 2 * (d_mine & 31), vreg[i]);
    }
  };
  const int krow = (col & 19) | ((col & 4) << 1) | ((col & 8) >> 1);
  auto k_frag = [&](int plane, int s) __attribute__((always_inline)) {
    return *reinterpret_cast<const bf16x8*>(planes + plane * L::kPlane + krow * (2 * D) + 16 * ((2 * s + hh) ^ L::swz_k(krow)));
  };
  const int vrow = 8 * hh + ((lane & 15) >> 2);
  auto v_frag = [&](int plane, int i, int half) __attribute__((always_inline)) {
    const uint8_t* p = planes + (3 + plane) * L::kPlane + (vrow + 16 * half) * (2 * D) + 64 * (i ^ L::swz_v(vrow)) +
                       (16 * ((lane >> 4) & 1) + 4 * (lane & 3)) * 2;
    const s16x4 lo = lds_read_tr(p), hi = lds_read_tr(p + 4 * (2 * D));
    return __builtin_bit_cast(bf16x8, (s16x8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  };

  // The instructions that split the next operand go between the MFMAs, for the other wavefront's to fall into (left to the compiler 0.3 to
  // 1.4 % longer: 12 heads x 1053 queries x 4212 keys 109.4 -> 111.4 us, 24 x 2048 x 4096 288 -> 291, d = 128 614 -> 616).
  auto interleave = [](auto reads, auto products) __attribute__((always_inline)) {
    constexpr int kValu = (44 * kLoads / 2 + decltype(products)::value - 1) / decltype(products)::value;
    __builtin_amdgcn_sched_group_barrier(0x100, decltype(reads)::value, 0);
#pragma unroll
    for (int i = 0; i < decltype(products)::value; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, kValu, 0);
      __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
    }
  };

  const bool any = at_k.advance(a, b, h, begin + group);
  bool more = at_v.advance(a, b, h, begin + group);
  // QW = 1: the elements of a lane's operands, key krow of K and keys 16 (r / 8) + 8 hh + r % 8 of V, d = col D/32 + i
  typedef float vvec __attribute__((ext_vector_type(kNB), aligned(4)));
  f32x4 k1[QW == 1 ? D / 8 : 1];
  auto load_k1 = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < D / 8; ++j) k1[j] = load_row(at_k, at_k.kb, krow, 16 * (j >> 1) + 8 * hh + 4 * (j & 1), f32x4());
  };
  if constexpr (QW == 1) {
    load_k1();
  } else {
    load_tile(at_k, at_k.kb, kreg);
    load_tile(at_v, at_v.vb, vreg);
  }

  // Q: B operand, d = 16 s + 8 hh + e (rows past Sq repeat the last one; their results are not stored)
  Split8 qs[D / 16];
  bool odd_q;   // a row of the wavefront's is outside the magnitudes that can be split
  {
    // Whole rows through the LDS (the output rows' place): as loads of 16 bytes of 32 different rows 0.2 to 1 us longer (us per call, 12 heads
    // x 280 queries x 560 keys, d = 128 27.9 -> 26.9, 10 x 114 x 456 22.7 -> 22.3; 4 x 512 x 2048, d = 64 21.7 -> 21.4).
    const float* qp = a.q + (int64_t)b * a.q_sb + (int64_t)h * a.q_sh + d_mine;
    float* rows = reinterpret_cast<float*>(lds_f32) + wave * L::kFloatsPerWave;
    f32x4 qv[kTile / kRowsPer];
#pragma unroll
    for (int i = 0; i < kTile / kRowsPer; ++i)
      qv[i] = *reinterpret_cast<const f32x4*>(qp + (int64_t)min(q0 + i * kRowsPer + lane / kRowLanes, a.Sq - 1) * a.q_ss);
#pragma unroll
    for (int i = 0; i < kTile / kRowsPer; ++i)
      *reinterpret_cast<f32x4*>(rows + (i * kRowsPer + lane / kRowLanes) * L::kPitch + d_mine) = qv[i];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int i = 0; i < D / 8; ++i) qv[i] = *reinterpret_cast<const f32x4*>(rows + col * L::kPitch + 16 * (i >> 1) + 8 * hh + 4 * (i & 1));
    QRange range;
#pragma unroll
    for (int s = 0; s < D / 16; ++s) {
      float x[8];
#pragma unroll
      for (int t = 0; t < 8; ++t) x[t] = qv[2 * s + (t >> 2)][t & 3];
#pragma unroll
      for (int t = 0; t < 8; t += 2) range.add(x[t], x[t + 1]);
      qs[s] = split8(x);
    }
    odd_q = __builtin_amdgcn_readfirstlane(__any(range.odd())) != 0;
  }

  f32x16 o[kNB];   // O^T: register r of block i is d = 32 i + 8 (r / 4) + 4 hh + r % 4
#pragma unroll
  for (int i = 0; i < kNB; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[i][r] = 0.f;
  // The maximum starts at the lowest finite value: a row that has met nothing but scores of -inf then gets weights of
  // exp2(-inf) = 0 and no sum, without a test for it.
  float m = -FLT_MAX, l = 0.f;

  // (the small terms for themselves: D / 16 sums at the magnitude of the score are rounded, not six times as many)
  auto scores = [&](const bf16x8& kh, const bf16x8& km, const bf16x8& kl, const Split8& q, f32x16& s, f32x16& small) __attribute__((always_inline)) {
    small = mfma16(kl, q.h, small);
    small = mfma16(kh, q.l, small);
    small = mfma16(km, q.m, small);
    small = mfma16(km, q.h, small);
    small = mfma16(kh, q.m, small);
    s = mfma16(kh, q.h, s);
  };
  // weights of a tile's scores, as operands; the factor of what was summed before
  auto weigh = [&](f32x16& s, int valid, float& alpha, Split8 (&ps)[2]) __attribute__((always_inline)) {
    if (__builtin_expect(valid < kTile, 0)) {
      asm volatile("" ::: "memory");   // keeps this a real branch
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (16 * (r >> 3) + 8 * hh + (r & 7) >= valid) s[r] = -INFINITY;
    }
    float mx = s[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    // The reference is the next multiple of a.grid (a power of two, 2 to 4 in the exponent): rows, groups and parts of one magnitude have
    // the same one, and their sums meet with weights that are exactly 1.
    const float m_new = fmaxf(m, ceilf(mx * a.inv_grid) * a.grid);
    alpha = __builtin_amdgcn_exp2f((m - m_new) * c);   // (0 on the first tile, or 1 with nothing to rescale)
    m = m_new;
    // the difference first, then the scale: the exponent is exact to its own rounding however large the scores are
    float sum[2] = {0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = __builtin_amdgcn_exp2f((s[r] - m) * c);
      sum[r & 1] += s[r];
    }
    l = fmaf(l, alpha, sum[0] + sum[1]);
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      float p[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) p[e] = s[8 * g + e];
      ps[g] = split8(p);
    }
  };
  if constexpr (QW == 1) {
    while (more) {
      const int valid = at_v.len - at_v.k0;
      vvec v1[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) v1[r] = load_row(at_v, at_v.vb, 16 * (r >> 3) + 8 * hh + (r & 7), kNB * col, vvec());
      __builtin_amdgcn_sched_barrier(0);   // V is on its way before the scores are computed
      f32x16 s, small;
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = small[r] = 0.f;
#pragma unroll
      for (int j = 0; j < D / 16; ++j) {
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = k1[2 * j + (e >> 2)][e & 3];
        const Split8 ks = split8(x);
        scores(ks.h, ks.m, ks.l, qs[j], s, small);
      }
      at_k.advance(a, b, h, KW);
      load_k1();
      __builtin_amdgcn_sched_barrier(0);
      more = at_v.advance(a, b, h, KW);
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] += small[r];
      float alpha;
      Split8 ps[2];
      weigh(s, valid, alpha, ps);
#pragma unroll
      for (int i = 0; i < kNB; ++i) {
        Split8 vs[2];
#pragma unroll
        for (int g = 0; g < 2; ++g) {
          float x[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) x[e] = v1[8 * g + e][i];
          vs[g] = split8(x);
        }
        f32x16 t;
#pragma unroll
        for (int r = 0; r < 16; ++r) t[r] = 0.f;
        t = mfma16(vs[0].l, ps[0].h, t);
        t = mfma16(vs[1].l, ps[1].h, t);
        t = mfma16(vs[0].h, ps[0].l, t);
        t = mfma16(vs[1].h, ps[1].l, t);
        t = mfma16(vs[0].m, ps[0].m, t);
        t = mfma16(vs[1].m, ps[1].m, t);
        t = mfma16(vs[0].m, ps[0].h, t);
        t = mfma16(vs[1].m, ps[1].h, t);
        t = mfma16(vs[0].h, ps[0].m, t);
        t = mfma16(vs[1].h, ps[1].m, t);
        t = mfma16(vs[0].h, ps[0].h, t);
        t = mfma16(vs[1].h, ps[1].h, t);
#pragma unroll
        for (int r = 0; r < 16; ++r) o[i][r] = fmaf(o[i][r], alpha, t[r]);
      }
    }
  } else {
  tile_barrier();   // (everybody has Q)
  if (turns > 0) {
    put_k();
    at_k.advance(a, b, h, KW);
    load_tile(at_k, at_k.kb, kreg);
  }
  tile_barrier();
  for (int turn = 0; turn < turns; ++turn) {
    // K of this tile is in the LDS
    const int valid = more ? at_v.len - at_v.k0 : 0;   // (none: the group's tiles are over, another's are not)
    bf16x8 kf[D / 16][3];   // read before the split of V, whose instructions hide the wait for them
#pragma unroll
    for (int j = 0; j < D / 16; ++j)
#pragma unroll
      for (int p = 0; p < 3; ++p) kf[j][p] = k_frag(p, j);
    put_v();
    f32x16 s, small;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = small[r] = 0.f;
#pragma unroll
    for (int j = 0; j < D / 16; ++j) scores(kf[j][0], kf[j][1], kf[j][2], qs[j], s, small);
    interleave(std::integral_constant<int, 3 * D / 16>(), std::integral_constant<int, 6 * D / 16>());
    more = at_v.advance(a, b, h, KW);
    load_tile(at_v, at_v.vb, vreg);
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] += small[r];
    float alpha;
    Split8 ps[2];
    weigh(s, valid, alpha, ps);
    tile_barrier();
    // V of this tile is in the LDS, and nobody reads its K any more
    // The tile's share of O^T is summed for itself, the small terms first: one rounding at the magnitude of O^T per tile.
#pragma unroll
    for (int i = 0; i < kNB; i += 2) {
      bf16x8 vf[3][2][2];   // (as K: before the split of the next K)
#pragma unroll
      for (int p = 0; p < 3; ++p)
#pragma unroll
        for (int g = 0; g < 2; ++g)
#pragma unroll
          for (int e = 0; e < 2; ++e) vf[p][g][e] = v_frag(p, i + e, g);
      if (i == 0) put_k();
      f32x16 t[2];
#pragma unroll
      for (int r = 0; r < 16; ++r) t[0][r] = t[1][r] = 0.f;
      auto term = [&](int plane, const bf16x8 (&p)[2]) __attribute__((always_inline)) {
#pragma unroll
        for (int g = 0; g < 2; ++g)
#pragma unroll
          for (int e = 0; e < 2; ++e) t[e] = mfma16(vf[plane][g][e], p[g], t[e]);
      };
      const bf16x8 ph[2] = {ps[0].h, ps[1].h}, pm[2] = {ps[0].m, ps[1].m}, pl[2] = {ps[0].l, ps[1].l};
      term(2, ph);
      term(0, pl);
      term(1, pm);
      term(1, ph);
      term(0, pm);
      term(0, ph);
      if (i == 0) interleave(std::integral_constant<int, 24>(), std::integral_constant<int, 24>());
#pragma unroll
      for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[i + e][r] = fmaf(o[i + e][r], alpha, t[e][r]);
    }
    at_k.advance(a, b, h, KW);
    load_tile(at_k, at_k.kb, kreg);
    tile_barrier();
  }
  }
  l += __shfl_xor(l, 32);

  // ---- epilogue: O^T -> LDS as [query][d] (the tiles' place), then whole rows to memory; the groups are folded on the way
  float* mine = reinterpret_cast<float*>(lds_f32) + wave * L::kFloatsPerWave;
  uint32_t worst = 0;
  if constexpr (QW == 1) {   // (register r of block i is d = (8 (r / 4) + 4 hh + r % 4) D/32 + i)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      vvec x;
#pragma unroll
      for (int i = 0; i < kNB; ++i) {
        x[i] = o[i][r];
        worst = max(worst, oddity(x[i]));
      }
      *reinterpret_cast<vvec*>(mine + col * L::kPitch + (8 * (r >> 2) + 4 * hh + (r & 3)) * kNB) = x;
    }
  } else {
#pragma unroll
    for (int i = 0; i < kNB; ++i)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        f32x4 x;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          x[e] = o[i][4 * g + e];
          worst = max(worst, oddity(x[e]));
        }
        *reinterpret_cast<f32x4*>(mine + col * L::kPitch + 32 * i + 8 * g + 4 * hh) = x;
      }
  }
  if (hh == 0) {
    mine[kTile * L::kPitch + col] = m;
    mine[kTile * L::kPitch + kTile + col] = l;
  }
  const bool odd_sum = !(l > 0.f && l < INFINITY);   // (no sum: a maximum whose reference is past the exponent range, or scores of -inf only)
  const bool suspect = any && (odd_q || __any(odd_sum || worst >= kOddFrom));
  uint32_t* flags = reinterpret_cast<uint32_t*>(lds_f32 + L::kFlags);
  if (lane == 0) flags[wave] = suspect;
  tile_barrier();
  const u32x4 flag = *reinterpret_cast<const u32x4*>(flags);
  if (__builtin_expect(__builtin_amdgcn_readfirstlane(flag.x | flag.y | flag.z | flag.w) != 0, 0)) {
    // A zero below a column of V that is zero (a narrower head's padding, keys that are padding) is exact.  Below one with an element of
    // ordinary size it is what terms leave that cancel; what small elements beside that one lost is below 2^-126.  So the group's V is looked
    // through once more for the largest of every column, each wavefront its rows.  us, no zeros / a zero column computed once more /
    // looked through: 12 heads x 1053 queries x 4212 keys, d = 64 105 / 260 / 106; 10 x 847 x 1694, d = 128 72 / 222 / 76; 12 x 355 x 2840
    // 69 / 199 / 76.  (The maxima taken while V is split cost every launch at d = 64 3 %.)
    constexpr int kAtOnce = D / 4 / kLoads;   // tiles on their way together
    // (a lane number of its own: with the loop's, the loop's addresses stay in registers until here and its schedule is 2 % longer)
    int here = threadIdx.x & 63;
    asm volatile("" : "+v"(here));
    const int quad = here % kRowLanes, first_row = member * kRowsPer + here / kRowLanes;
    u32x4 most = {0, 0, 0, 0};   // (twice the bits: the order of magnitudes)
    Cursor<kFar> at(a, job, n_tiles);
    bool left = at.advance(a, b, h, begin + group);
    while (left) {
      f32x4 x[kAtOnce][kLoads];
#pragma unroll
      for (int t = 0; t < kAtOnce; ++t) {   // (behind the last tile: zeros)
#pragma unroll
        for (int i = 0; i < kLoads; ++i) x[t][i] = load_row(at, at.vb, first_row + i * QW * kRowsPer, 4 * quad, f32x4());
        left = at.advance(a, b, h, KW);
      }
#pragma unroll
      for (int t = 0; t < kAtOnce; ++t)
#pragma unroll
        for (int i = 0; i < kLoads; ++i) most = __builtin_elementwise_max(most, __builtin_bit_cast(u32x4, x[t][i]) << 1);
    }
    uint8_t* columns = lds_f32 + L::kColumns + 1024 * group * QW + 16 * here;
    *reinterpret_cast<u32x4*>(columns + 1024 * member) = most;
    tile_barrier();
    columns += 16 * (quad - here);
    most = u32x4{0, 0, 0, 0};
#pragma unroll
    for (int w = 0; w < QW * kRowsPer; ++w) most = __builtin_elementwise_max(most, *reinterpret_cast<const u32x4*>(columns + 16 * kRowLanes * w));
    bool odd = false;
#pragma unroll
    for (int i = 0; i < D / 8; ++i) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(mine + (here & 31) * L::kPitch + 8 * i + 4 * (here >> 5));
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t column = (uint32_t)__shfl((int)most[e], 2 * i + (here >> 5));   // (by all lanes)
        odd |= oddity(x[e]) >= kOddFrom && column != 0 && (x[e] != 0.f || column < 2 * kTiny);
      }
    }
    if (any && (odd_q || __any(odd_sum || odd))) {
      // Once more with fp32 products, for the elements and rows that need it; the others stay what they are.
      float m2, l2;
      bool odd_half;   // (of the lane's half of its row of Q)
      walk_fp32<D, kFar>(a, b, h, job, q0, begin + group, KW, n_tiles, o, m2, l2, odd_half);
      const bool other_half = __shfl_xor((int)odd_half, 32) != 0;   // (exchanged by all lanes)
      const bool whole_row = odd_sum || odd_half || other_half;
      const float f = __builtin_amdgcn_exp2f((m2 - m) * c);
#pragma unroll
      for (int r = 0; r < 16; ++r)
#pragma unroll
        for (int i = 0; i < kNB; ++i) {
          float* x = mine + col * L::kPitch + (8 * (r >> 2) + 4 * hh + (r & 3)) * kNB + i;
          if (whole_row) *x = o[i][r];
          else if (oddity(*x) >= kOddFrom) *x = o[i][r] * f;
        }
      if (whole_row && hh == 0) {
        mine[kTile * L::kPitch + col] = m2;
        mine[kTile * L::kPitch + kTile + col] = l2;
      }
    }
    tile_barrier();
  }
  const float* halves = reinterpret_cast<float*>(lds_f32) + member * L::kFloatsPerWave;   // group g: QW wavefronts on
  constexpr int kRowsPerWave = kTile / KW;
  // `row` of the workgroup's 32 QW
  auto store_row = [&](int row, const float (&acc)[4], float den, float mm) __attribute__((always_inline)) {
    const int q = qg * QW * kTile + row;
    if (q >= a.Sq) return;
    const float inv = den > 0.f ? 1.f / den : 0.f;
    f32x4 y;
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = acc[e] * inv;
    *reinterpret_cast<f32x4*>(a.job[job].out + (((int64_t)b * a.Sq + q) * a.H + h) * D + d_mine) = y;
    if (d_mine == 0)
      a.job[job].lse[a.lse_bsh ? ((int64_t)b * a.Sq + q) * a.H + h : ((int64_t)b * a.H + h) * a.Sq + q] =
          lse_of(mm, den, a.scale);
  };
  const int64_t n_rows = (int64_t)(gridDim.y / a.parts) * a.total * (QW * kTile);   // of a part, all jobs
  const int64_t sums = n_rows * a.parts * D;
  auto part_row = [&](int p) { return p * n_rows + ((int64_t)job * a.total + item) * (QW * kTile); };
#pragma unroll 1
  for (int p = 0; p < kRowsPerWave; p += kRowsPer) {
    const int row = group * kRowsPerWave + p + lane / kRowLanes;
    float mm = -INFINITY;
#pragma unroll
    for (int w = 0; w < KW; ++w) mm = fmaxf(mm, halves[w * QW * L::kFloatsPerWave + kTile * L::kPitch + row]);
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    float den = 0.f;
#pragma unroll
    for (int w = 0; w < KW; ++w) {
      const float* pw = halves + w * QW * L::kFloatsPerWave;
      const float lw = pw[kTile * L::kPitch + kTile + row];
      const float ww = KW == 1 ? 1.f : (lw == 0.f ? 0.f : __builtin_amdgcn_exp2f((pw[kTile * L::kPitch + row] - mm) * c));
      const f32x4 x = *reinterpret_cast<const f32x4*>(pw + row * L::kPitch + d_mine);
      den = fmaf(ww, lw, den);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] = fmaf(ww, x[e], acc[e]);
    }
    if (a.parts == 1) {
      store_row(row + member * kTile, acc, den, mm);
    } else {
      // past the L2, for the workgroup that folds (see attn_fwd.hip, "states that meet inside a launch")
      const int at = member * kTile + row;
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, f32x4{acc[0], acc[1], acc[2], acc[3]}),
                                             buffer_of(a.ws + part_row(part) * D, QW * kTile * D * 4), (at * D + d_mine) * 4, 0, kDevice);
      if (d_mine == 0) {
        float* ml = a.ws + sums + 2 * (part_row(part) + at);
        __hip_atomic_store(ml, mm, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(ml + 1, den, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  }
  if (a.parts == 1) return;

  // ---- the workgroup that is the last of its item to get here folds the parts
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  uint32_t* last = reinterpret_cast<uint32_t*>(lds_f32);
  if (threadIdx.x == 0) {
    uint32_t* counter = a.arrive + (int64_t)job * a.total + item;
    const bool mine_is = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 == (uint32_t)a.parts;
    if (mine_is) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *last = mine_is;
  }
  __syncthreads();
  if (*last == 0) return;
  __syncthreads();
  constexpr int kRows = kTile * QW;
  constexpr int kSteps = kRows / (kWavesF32 * kRowsPer);   // rows of a lane
  constexpr int kBatch = 16 / kSteps;                      // parts whose sums are on their way together
  auto row_of = [&](int i) { return (i * kWavesF32 + wave) * kRowsPer + lane / kRowLanes; };
  f32x4 x[kBatch][kSteps];
  auto load_sums = [&](int p) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < kBatch; ++j) {
      // (behind the last part an empty buffer: zeros, no memory is touched)
      const Rsrc src = buffer_of(a.ws + part_row(min(p + j, a.parts - 1)) * D, p + j < a.parts ? kRows * D * 4 : 0);
#pragma unroll
      for (int i = 0; i < kSteps; ++i)
        x[j][i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(src, (row_of(i) * D + d_mine) * 4, 0, kDevice));
    }
  };
  float* weights = reinterpret_cast<float*>(lds_f32) + 2 * kRows;   // [part][query]; in front of them (maximum, sum) of every query
  load_sums(0);
  if (threadIdx.x < kRows) {   // a thread, a query
    f32x2 ml[kMaxParts];
#pragma unroll
    for (int p = 0; p < kMaxParts; ++p)
      ml[p] = __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(
                                            buffer_of(a.ws + sums + 2 * part_row(min(p, a.parts - 1)), p < a.parts ? kRows * 8 : 0),
                                            threadIdx.x * 8, 0, kDevice));
    float mm = -INFINITY, den = 0.f;
#pragma unroll
    for (int p = 0; p < kMaxParts; ++p) mm = p < a.parts ? fmaxf(mm, ml[p].x) : mm;
#pragma unroll
    for (int p = 0; p < kMaxParts; ++p) {
      const float w = ml[p].y == 0.f ? 0.f : __builtin_amdgcn_exp2f((ml[p].x - mm) * c);   // (no part, no sum)
      den = fmaf(w, ml[p].y, den);
      weights[p * kRows + threadIdx.x] = w;
    }
    weights[(int)threadIdx.x - 2 * kRows] = mm;
    weights[(int)threadIdx.x - kRows] = den;
  }
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  float acc[kSteps][4];
#pragma unroll
  for (int i = 0; i < kSteps; ++i) acc[i][0] = acc[i][1] = acc[i][2] = acc[i][3] = 0.f;
  for (int p = 0; p < a.parts; p += kBatch) {
#pragma unroll
    for (int j = 0; j < kBatch; ++j)
#pragma unroll
      for (int i = 0; i < kSteps; ++i) {
        const float w = weights[(p + j) * kRows + row_of(i)];
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[i][e] = fmaf(w, x[j][i][e], acc[i][e]);
      }
    if (p + kBatch < a.parts) load_sums(p + kBatch);
  }
#pragma unroll
  for (int i = 0; i < kSteps; ++i)
    store_row(row_of(i), acc[i], weights[row_of(i) - kRows], weights[row_of(i) - 2 * kRows]);
}

template <int D, int QW, bool kFar>
int launch_f32(AttnF32Args& a, int n_jobs, hipStream_t stream) {
  // more than 64 KB of dynamic LDS has to be allowed once per kernel and device
  static thread_local int allowed_dev = -1;
  constexpr int kLds = F32Lds<D, QW>::kBytes;
  int dev = 0;
  if (int rc = hip_fail(hipGetDevice(&dev), "hipGetDevice")) return rc;
  if (allowed_dev != dev) {
    if (int rc = hip_fail(hipFuncSetAttribute(reinterpret_cast<const void*>(&attn_f32_kernel<D, QW, kFar>),
                                              hipFuncAttributeMaxDynamicSharedMemorySize, kLds),
                          "hipFuncSetAttribute"))
      return rc;
    allowed_dev = dev;
  }
  hipLaunchKernelGGL((attn_f32_kernel<D, QW, kFar>), dim3((unsigned)a.per_xcd * 8u, (unsigned)(n_jobs * a.parts), 1), dim3(kThreadsF32),
                     kLds, stream, a);
  return hip_fail(hipGetLastError(), "attn_f32 launch");
}

// Query tiles of a workgroup and workgroups that share the keys of a work item.  What a launch takes, in us: its rounds of workgroups
// times the turns of one times what a turn takes (one workgroup on a CU, and at d = 64 two), and what a launch, a round, a second workgroup on a CU and
// the fold of the parts cost on top.  Four query tiles a workgroup split K and V half as often as two, but fold twice the bytes and leave a
// small launch fewer workgroups; one query tile splits everything itself, and starts and ends sooner, with four groups of keys and no barriers
// in between.  The constants are fitted to 190 shapes of 1 ... 24 heads x 32 ... 4096 queries against 1 ... 8 chunks of 64 ... 2048 keys, as one
// job and a job a chunk, in every form and split (7300 timings, errors 5 to 8 %); in launches of several rounds, where the forms are close, a
// split or one query tile has to gain more than 3 %.  The plan takes 0.5 % more than the best form on average with scratch and 0.1 %
// without, at most 14 % (6 heads x 1005 queries x 8 jobs of 24 tiles, d = 64).
// us unsplit -> as planned, two query tiles or more -> one too: 4 heads x 512 queries x 2048 keys, d = 64 67 -> 22 -> 19 (4 parts);
// 2 x 553 x 4424 134 -> 30 -> 22, d = 128 245 -> 48 -> 39; 1 x 32 x 64, d = 128 13.8 -> 11.1 (1 part); without scratch, which parts
// need, 4 x 512 x 2048, d = 64 67 -> 37, d = 128 119 -> 66.
struct F32Plan {
  int qw = 2, parts = 1;
};
struct F32Cost {
  double one, two;      // a turn alone, beside another workgroup's
  double launch, parts, part;
  double round, pair;   // a further round; a second workgroup on a CU
};
F32Plan plan_f32(int D, int heads, int Sq, int n_jobs, int tiles, bool far, int64_t workspace_bytes, int64_t n_counters) {
  constexpr F32Cost kCost[2][3] = {{{1.84, 3.18, 5.8, 3.2, 0.15, 2.1, 1.5}, {1.87, 2.95, 7.3, 2.7, 0.42, 2.1, 1.0}, {1.58, 2.57, 7.9, 2.8, 0.57, 1.1, 2.9}},
                                   {{3.7, 0, 8.5, 3.2, 0.36, 5.2, 0}, {3.49, 0, 10.9, 2.9, 0.6, 6.3, 0}, {2.92, 0, 12.4, 3.1, 0.86, 6.0, 0}}};
  constexpr int64_t kCus = 32;   // of an XCD
  F32Plan best;
  double least = 1e30;
  for (int qw = 1; qw <= (far ? 2 : 4); qw *= 2) {
    const F32Cost& t = kCost[D == 128][qw >> 1];
    const int64_t items = (int64_t)heads * ((Sq + kTile * qw - 1) / (kTile * qw)), per_xcd = (items + 7) / 8 * n_jobs;
    const int kw = kWavesF32 / qw;
    for (int parts = 1; parts <= kMaxParts; ++parts) {
      if (parts > 1 && (parts * kw > tiles || items * n_jobs > n_counters || items * n_jobs * parts * (kTile * qw) * (D + 2) * 4 > workspace_bytes)) break;
      const double turns = (tiles + kw * parts - 1) / (kw * parts);
      const int64_t groups = per_xcd * parts;
      double time = t.launch + (parts > 1 ? t.parts + t.part * parts : 0.0);
      if (D == 128) {
        const int64_t rounds = (groups + kCus - 1) / kCus;
        time += rounds * turns * t.one + (rounds - 1) * t.round;
      } else {
        const int64_t full = groups / (2 * kCus), rest = groups % (2 * kCus);
        time += full * turns * t.two + (rest == 0 ? 0.0 : rest <= kCus ? turns * t.one : turns * t.two);
        time += (full + (rest > 0) - 1) * t.round + (groups > kCus ? t.pair : 0.0);
      }
      if (parts > 1 && per_xcd > kCus) time *= 1.03;
      if (qw == 1 && groups > 2 * kCus) time *= 1.03;
      if (time < least) {
        least = time;
        best.qw = qw;
        best.parts = parts;
      }
    }
  }
  return best;
}

}  // namespace
}  // namespace dt

using namespace dt;

extern "C" int dt_attn_jobs_f32_ws_fwd(const float* q, int32_t B, int32_t Sq, int32_t H, int32_t D, int64_t q_sb, int64_t q_ss,
                                    int64_t q_sh, int32_t n_chunks, const float* const* k_ptrs,
                                    const float* const* v_ptrs, const int32_t* kv_lens, const int64_t* kv_sb,
                                    const int64_t* kv_ss, const int64_t* kv_sh, int32_t n_jobs, const int32_t* job_begin,
                                    const int32_t* job_chunks, float* const* out_ptrs, float* const* lse_ptrs,
                                    int32_t lse_layout, float softmax_scale, void* workspace, int64_t workspace_bytes, uint32_t* counters,
                                    int64_t n_counters, void* stream) {
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
  a.B = B; a.H = H; a.Sq = Sq; a.D = D;
  a.parts = 1;
  a.scale = softmax_scale > 0.f ? softmax_scale : 1.0f / std::sqrt((float)D);
  a.scale_log2 = a.scale * 1.4426950408889634f;
  a.grid = std::exp2(std::floor(std::log2(4.f / a.scale_log2)));
  a.inv_grid = 1.f / a.grid;
  bool far = false;
  for (int i = 0; i < n_chunks; ++i) {
    if (kv_lens[i] < 0 || (kv_lens[i] > 0 && (!k_ptrs[i] || !v_ptrs[i]))) {
      set_error("chunk %d: negative length or null k/v", i);
      return DT_ERR_INVALID;
    }
    a.chunk[i] = {k_ptrs[i], v_ptrs[i], kv_sb[i], kv_ss[i], kv_sh[i], kv_lens[i]};
    // (a chunk's keys of one batch and head beyond 2 GiB, or in falling order: 64-bit offsets.  us, 32 -> 64 bits: 4 heads x 512 queries x 2048
    // keys, d = 64 20 -> 23; 24 x 2048 x 4096 286 -> 338, d = 128 613 -> 755)
    far = far || kv_ss[i] < 0 || (kv_lens[i] > 0 && (uint64_t)kv_ss[i] > (1ull << 29) / ((uint64_t)kv_lens[i] + kTile));
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
    a.job[j] = {out_ptrs[j], lse_ptrs[j], job_begin[j], job_begin[j + 1]};
  }
  for (int e = 0; e < job_begin[n_jobs]; ++e) {
    if (job_chunks[e] < 0 || job_chunks[e] >= n_chunks) {
      set_error("job chunk reference %d is outside the chunk table", job_chunks[e]);
      return DT_ERR_INVALID;
    }
    a.refs[e] = job_chunks[e];
  }
  if (lse_layout != DT_LSE_BHS && lse_layout != DT_LSE_BSH) {
    set_error("unknown lse layout %d", lse_layout);
    return DT_ERR_INVALID;
  }
  a.lse_bsh = lse_layout == DT_LSE_BSH;
  int tiles = 0;
  for (int j = 0; j < n_jobs; ++j) {
    int64_t n = 0;
    for (int e = job_begin[j]; e < job_begin[j + 1]; ++e) n += ((int64_t)kv_lens[job_chunks[e]] + kTile - 1) / kTile;
    tiles = std::max(tiles, (int)std::min<int64_t>(n, INT32_MAX / 2));
  }
  const bool scratch = workspace && counters;
  const F32Plan plan = plan_f32(D, B * H, Sq, n_jobs, tiles, far, scratch ? workspace_bytes : 0, scratch ? n_counters : 0);
  const int qw = plan.qw;
  a.parts = plan.parts;
  a.n_qg = (Sq + kTile * qw - 1) / (kTile * qw);
  a.total = B * H * a.n_qg;
  a.per_xcd = (a.total + 7) / 8;
  a.ws = static_cast<float*>(workspace);
  a.arrive = counters;
  hipStream_t s = (hipStream_t)stream;
  std::unique_lock<std::mutex> lock;   // (another thread's parts, on the same stream and workspace, may wait for a fold kernel)
  if (a.parts > 1) lock = std::unique_lock<std::mutex>(workspace_lock(workspace));
  auto launch = [&](auto d, auto w, auto f) { return launch_f32<decltype(d)::value, decltype(w)::value, decltype(f)::value>(a, n_jobs, s); };
  auto launch_d = [&](auto d) {
    const std::integral_constant<int, 1> one;
    const std::integral_constant<int, 2> two;
    if (far) return qw == 1 ? launch(d, one, std::true_type()) : launch(d, two, std::true_type());
    if (qw == 4) return launch(d, std::integral_constant<int, 4>(), std::false_type());
    return qw == 1 ? launch(d, one, std::false_type()) : launch(d, two, std::false_type());
  };
  return D == 128 ? launch_d(std::integral_constant<int, 128>()) : launch_d(std::integral_constant<int, 64>());
}

extern "C" int dt_attn_jobs_f32_fwd(const float* q, int32_t B, int32_t Sq, int32_t H, int32_t D, int64_t q_sb, int64_t q_ss,
                                    int64_t q_sh, int32_t n_chunks, const float* const* k_ptrs,
                                    const float* const* v_ptrs, const int32_t* kv_lens, const int64_t* kv_sb,
                                    const int64_t* kv_ss, const int64_t* kv_sh, int32_t n_jobs, const int32_t* job_begin,
                                    const int32_t* job_chunks, float* const* out_ptrs, float* const* lse_ptrs,
                                    float softmax_scale, void* stream) {
  return dt_attn_jobs_f32_ws_fwd(q, B, Sq, H, D, q_sb, q_ss, q_sh, n_chunks, k_ptrs, v_ptrs, kv_lens, kv_sb, kv_ss, kv_sh, n_jobs, job_begin,
                                 job_chunks, out_ptrs, lse_ptrs, DT_LSE_BHS, softmax_scale, nullptr, 0, nullptr, 0, stream);
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
