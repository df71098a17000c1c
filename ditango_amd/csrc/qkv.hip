// The q, k and v of a layer in one launch: three linear projections of the text and video tokens, with LayerNorm over the head
// dimension and interleaved RoPE on q and k before they are written, as the [B,S,H,64] tensors the attention kernel reads.
// Replaces the concatenation, the three library products and the two producer launches of
// executor/cogvideox/attention_processor.py:39-71.
//
// What bounds it: loads and MFMAs, which overlap only in part.  48 heads x 2222 tokens x 3072 channels (126 GFLOP), us per call, timed with work
// left out: all 122, without the loads of the loop 103, without its MFMAs 84, four steps of 96 27 (41 MB of results leave at once; tables
// and norm); MFMAs alone hold 1.8 GHz and take 67.  The loads are some 37 KB a CU and step, which come at 58 GB/s a CU whatever their rows and
// however far ahead they are issued.  In a loop of calls, modules and producer -> this: the same 153 -> 122 us (1030 TFLOP/s), 16 heads x 602 x
// 1024 42 -> 17.  From 200 GFLOP on the library's products take less (48 x 8016 429 -> 458), and the adapter calls the modules.
// out^T = W X^T with v_mfma_f32_32x32x16, accumulated in fp32.  A wavefront owns one head (64 output columns) of 32 MB tokens; with
// the product transposed a lane holds 32 of the 64 columns of ONE token, four neighbouring ones at a time.
//   * A workgroup of 8 wavefronts takes BM = 32 MB WM tokens x BN = 64 (8 / WM) columns of the three outputs side by side.
//   * Steps of 64 input channels with two LDS buffers, of 32 with three where the tile is 320 x 256: tiles go from memory straight into the
//     LDS (global_load_lds, one or two steps ahead) as rows of 128 or 64 bytes, their 16-byte pieces permuted by the row so that operand
//     reads meet in no bank.
//   * The two wavefronts of a SIMD issue their loads at different halves of the step (an M0 write and a load each 20 cycles or so,
//     in which a wavefront issues no MFMA; together with the epilogue's tables through the LDS 140 -> 128 us), and an operand read follows
//     each MFMA (128 -> 125).
//   * One barrier a step, in its middle: in front of it a wavefront has read the last operands it needs of the step's buffer and
//     waited for its own loads of the next one; behind it come the first operands of the next step, half a step before the MFMAs
//     that take them.
//   * The accumulators go through the LDS as rows of 16-bit projections, and norm and rotation follow with eight lanes a row, in the order
//     of sums of qk_norm_rope_kernel: q, k and v are bit for bit those of the modules and the producer wherever the library adds up a
//     product in one chain.
#include <algorithm>
#include <type_traits>

#include "producer_math.h"

namespace dt {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

constexpr int kThreads = 512;
constexpr int kWaves = 8;
constexpr int kHead = 64;
constexpr int kXcds = 8;
constexpr int kStageBytes = kWaves * 32 * kHead * 2;   // output rows on their way

constexpr int kLds = 163840;                           // of a CU
constexpr int table_pieces(int MB, int WM) { return std::min(MB, (kLds - kStageBytes) / (2 * 32 * WM * kHead * 4)); }   // that fit beside the rows

struct QkvProj {
  const uint16_t* w;          // [N, K]
  const uint16_t* bias;       // [N] or null
  uint16_t* y;                // [M, N]
  const uint16_t *nw, *nb;    // LayerNorm weight and bias over the head dimension, or null
  int32_t norm, rope;
  float eps;
};
struct QkvArgs {
  const uint16_t *text, *video;
  int64_t text_sb, text_ss, video_sb, video_ss;   // elements
  int32_t T, S, M;            // text tokens, all tokens of a sample, of the batch
  int32_t N, K;               // output columns of one projection, input channels
  int32_t m_tiles, tiles, per_xcd;
  Quotient by_s;              // tokens by S
  const float *cos, *sin;     // [S - T, 64]
  QkvProj proj[3];
};
typedef const QkvArgs __attribute__((address_space(4))) KernArgs;

template <bool kHalf>
struct Elem {
  typedef bf16x8 x8;
  typedef bf16x2 x2;
  __device__ static __forceinline__ f32x16 mfma(x8 a, x8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }
};
template <>
struct Elem<true> {
  typedef f16x8 x8;
  typedef f16x2 x2;
  __device__ static __forceinline__ f32x16 mfma(x8 a, x8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0); }
};
template <bool kHalf>
__device__ __forceinline__ f32x2 unpack2(uint32_t w) {
  if constexpr (kHalf) return __builtin_convertvector(__builtin_bit_cast(f16x2, w), f32x2);
  else return f32x2{__builtin_bit_cast(float, w << 16), __builtin_bit_cast(float, w & 0xffff0000u)};
}
// 64 x 16 bytes from the lanes' addresses to consecutive LDS bytes (see load_block_to_lds in attn_fwd.hip for why in assembly).
__device__ __forceinline__ void load_block_to_lds(const uint16_t* from, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
               :
               : "v"(from), "s"(__builtin_amdgcn_readfirstlane(lds_addr))
               : "memory", "m0");
}
template <int N>
__device__ __forceinline__ void wait_loads() {
  static_assert(N >= 0 && N <= 63, "an immediate of the wait");
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt vmcnt(%0)" : : "i"(N) : "memory");
}
__device__ __forceinline__ void step_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

template <int MB, int WM, int KH, int NBUF, bool kHalf>
__global__ __launch_bounds__(kThreads, 2) void qkv_kernel(const QkvArgs args_by_value) {
  typedef Elem<kHalf> E;
  constexpr int WN = kWaves / WM;
  constexpr int BM = 32 * MB * WM, BN = kHead * WN;
  constexpr int kStep = 16 * KH, kRowBytes = kStep * 2;   // input channels of a step
  constexpr int kPieces = kRowBytes / 16, kRowsPer = 64 / kPieces;   // 16-byte pieces of a row, rows of a load
  constexpr int kSwzShift = KH == 2 ? 2 : 1;
  constexpr int kGroups = (BM + BN) / kRowsPer;           // 1 KB loads of a step
  constexpr int kMost = (kGroups + kWaves - 1) / kWaves;  // of a wavefront
  constexpr int kFull = kGroups % kWaves ? kGroups % kWaves : kWaves;   // wavefronts that have so many; the others one less
  constexpr int kBufBytes = (BM + BN) * kRowBytes;
  KernArgs& a = *(KernArgs*)__builtin_amdgcn_kernarg_segment_ptr();
  (void)args_by_value;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>((uint8_t __attribute__((address_space(3)))*)lds);

  // tiles of an XCD are neighbours: all token tiles of a column tile, then the next column tile
  const int idx = blockIdx.x >> 3;
  const int tile = (int)(blockIdx.x & (kXcds - 1)) * a.per_xcd + idx;
  if (idx >= a.per_xcd || tile >= a.tiles) return;
  const int n_tile = tile / a.m_tiles;
  const int m0 = (tile - n_tile * a.m_tiles) * BM, n0 = n_tile * BN;
  const int lane = threadIdx.x & 63, col = lane & 31, hh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int wm = wave / WN, wn = wave - wm * WN;
  const int steps = a.K / kStep;

  // (a division by a variable is some 30 instructions)
  auto batch_of = [&](int m) __attribute__((always_inline)) { return (int)quotient((uint32_t)m, Quotient{a.by_s.mul, a.by_s.shift}); };
  // ---- this lane's place in the tiles it loads: rows past the end are the last one's again
  const uint16_t* from[kMost];
#pragma unroll
  for (int i = 0; i < kMost; ++i) {
    const int row = (i * kWaves + wave) * kRowsPer + lane / kPieces;
    const int piece = (lane % kPieces) ^ ((row >> kSwzShift) & (kPieces - 1));
    if (row < BM) {
      const int m = min(m0 + row, a.M - 1), b = batch_of(m), s = m - b * a.S;
      from[i] = s < a.T ? a.text + b * a.text_sb + s * a.text_ss : a.video + b * a.video_sb + (int64_t)(s - a.T) * a.video_ss;
    } else {
      const int n = min(n0 + row - BM, 3 * a.N - 1), p = (n >= a.N) + (n >= 2 * a.N);
      const uint16_t* w = p == 0 ? a.proj[0].w : p == 1 ? a.proj[1].w : a.proj[2].w;
      from[i] = w + (int64_t)(n - p * a.N) * a.K;
    }
    from[i] += 8 * piece;
  }
  auto load_step = [&](int buffer) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kMost; ++i) {
      if (i + 1 < kMost || wave < kFull) load_block_to_lds(from[i], lds0 + buffer * kBufBytes + (i * kWaves + wave) * 1024);
      from[i] += kStep;
    }
  };
  // all but the loads of the kAhead newest steps
  auto wait_steps = [&](auto ahead) __attribute__((always_inline)) {
    constexpr int kAhead = decltype(ahead)::value;
    if constexpr (kFull == kWaves || kAhead == 0) wait_loads<kAhead * kMost>();
    else if (wave < kFull) wait_loads<kAhead * kMost>();
    else wait_loads<kAhead * (kMost - 1)>();
  };

  f32x16 acc[2][MB];
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[j][i][r] = 0.f;

  struct Operands {
    typename E::x8 w[2], x[MB];
  };
  // operands of half a step: 16 input channels
  auto read = [&](Operands& o, int buffer, int half) __attribute__((always_inline)) {
    const uint8_t* at = lds + buffer * kBufBytes + col * kRowBytes + (((2 * half + hh) ^ ((col >> kSwzShift) & (kPieces - 1))) << 4);
#pragma unroll
    for (int j = 0; j < 2; ++j) o.w[j] = *reinterpret_cast<const typename E::x8*>(at + (BM + wn * kHead + 32 * j) * kRowBytes);
#pragma unroll
    for (int i = 0; i < MB; ++i) o.x[i] = *reinterpret_cast<const typename E::x8*>(at + (wm * 32 * MB + 32 * i) * kRowBytes);
  };
  auto multiply = [&](const Operands& o) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[j][i] = E::mfma(o.w[j], o.x[i], acc[j][i]);
    // the reads in front of them, one behind each: in front of all, the first MFMA waits until the LDS has taken every one
    constexpr int kReads = MB + 2, kMfmas = 2 * MB;
#pragma unroll
    for (int i = 0; i < kReads; ++i) {
      if (i < kMfmas) __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    if (kMfmas > kReads) __builtin_amdgcn_sched_group_barrier(0x008, kMfmas - kReads, 0);
    __builtin_amdgcn_sched_barrier(0);
  };
  load_step(0);
#pragma unroll
  for (int t = 1; t < NBUF; ++t)
    if (t < steps) load_step(t);
  if (steps >= NBUF) wait_steps(std::integral_constant<int, NBUF - 1>());
  else wait_steps(std::integral_constant<int, 0>());
  step_barrier();
  Operands operands[2];
  read(operands[0], 0, 0);
  int buffer = 0;
  const bool late = wave >= kWaves / 2;
  for (int t = 0; t < steps; ++t) {
    if (late && t > 0 && t + NBUF - 1 < steps) load_step(buffer == 0 ? NBUF - 1 : buffer - 1);
#pragma unroll
    for (int h = 0; h < KH - 1; ++h) {
      read(operands[(h + 1) & 1], buffer, h + 1);
      multiply(operands[h & 1]);
    }
    // the next step's tile has landed, for everybody; nobody reads this one's any more
    if (t + NBUF - 1 < steps) wait_steps(std::integral_constant<int, NBUF - 2>());
    else wait_steps(std::integral_constant<int, 0>());
    step_barrier();
    if (!late && t + NBUF < steps) load_step(buffer);
    buffer = buffer == NBUF - 1 ? 0 : buffer + 1;
    read(operands[0], buffer, 0);   // (behind the last step: some operands nobody uses)
    multiply(operands[(KH - 1) & 1]);
  }

  // ---- bias, LayerNorm, RoPE; a wavefront's rows go through LDS of its own, so that stores are whole rows.  The tables of the
  // workgroup's tokens come into the LDS once for all of its heads (from memory for each, the launch took 25 us longer).
  // They come in pieces, 32 rows for each of the WM wavefronts along the tokens, as many at a time as the LDS holds.
  constexpr int kTable = 32 * WM * kHead * 4, kPieces32 = table_pieces(MB, WM);
  bool rotates = false;   // a projection of the workgroup's columns
#pragma unroll
  for (int p = 0; p < 3; ++p) rotates |= a.proj[p].rope && n0 < (p + 1) * a.N && n0 + BN > p * a.N;
  auto tables = [&](int piece) __attribute__((always_inline)) { return (uint32_t)(kStageBytes + piece % kPieces32 * 2 * kTable); };
  auto load_tables = [&](int piece) __attribute__((always_inline)) {
    if (!rotates) return;
#pragma unroll
    for (int i = 0; i < WM; ++i) {
      const int row = (i * kWaves + wave) * 4 + (lane >> 4);
      const int m = min(m0 + (row / 32 * MB + piece) * 32 + row % 32, a.M - 1), s = m - batch_of(m) * a.S;
      const int64_t at = (int64_t)max(s - a.T, 0) * kHead + 4 * (lane & 15);
      const uint32_t to = lds0 + tables(piece) + (i * kWaves + wave) * 1024;
      load_block_to_lds(reinterpret_cast<const uint16_t*>(a.cos + at), to);
      load_block_to_lds(reinterpret_cast<const uint16_t*>(a.sin + at), to + kTable);
    }
  };
#pragma unroll
  for (int piece = 0; piece < kPieces32; ++piece) load_tables(piece);
  const int n_wave = n0 + wn * kHead;
  const bool mine = n_wave < 3 * a.N;
  const int p = mine ? n_wave / a.N : 0, n_proj = mine ? n_wave - p * a.N : 0;
  const auto& pr = a.proj[p];
  u32x2 bias[2][4];
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      bias[j][g] = pr.bias ? *reinterpret_cast<const u32x2*>(pr.bias + n_proj + 32 * j + 8 * g + 4 * hh) : u32x2{0, 0};
  const int d = 8 * (lane & 7);   // of a row that comes back from the stage
  const uint32_t one = pack2<kHalf>(1.f, 1.f);
  const u32x4 nw = pr.nw ? *reinterpret_cast<const u32x4*>(pr.nw + d) : u32x4{one, one, one, one};
  const u32x4 nb = pr.nb ? *reinterpret_cast<const u32x4*>(pr.nb + d) : u32x4{0, 0, 0, 0};
  wait_loads<0>();
  step_barrier();
  uint8_t* stage = lds + wave * (32 * kHead * 2);
#pragma unroll
  for (int i = 0; i < MB; ++i) {
    if (i >= kPieces32) {   // its tables have come into the place of an earlier piece's
      wait_loads<0>();
      step_barrier();
    }
    const int m_first = m0 + (wm * MB + i) * 32;
    if (mine && m_first < a.M) {
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g) {   // rounded as the projection's output is
          u32x2 x;
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            const f32x2 b = unpack2<kHalf>(bias[j][g][e]);
            x[e] = pack2<kHalf>(acc[j][i][4 * g + 2 * e] + b.x, acc[j][i][4 * g + 2 * e + 1] + b.y);
          }
          *reinterpret_cast<u32x2*>(stage + col * (kHead * 2) + (((4 * j + g) ^ ((col >> 1) & 7)) << 4) + 8 * hh) = x;
        }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      // eight lanes a row, as in qk_norm_rope_kernel
      u32x4 raw[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 8 * r + (lane >> 3);
        raw[r] = *reinterpret_cast<const u32x4*>(stage + row * (kHead * 2) + (((lane & 7) ^ ((row >> 1) & 7)) << 4));
      }
      if (pr.norm != DT_NORM_NONE) {
        float mean[4], ss[4], rs[4], w[8], b[8];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float v[8];
          unpack8<kHalf>(raw[r], v);
          mean[r] = row_sum<8>(v) * (1.0f / kHead);
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] -= mean[r];
          ss[r] = row_squares<8>(v);
        }
        inverse_rms4<kHead>(ss[0], ss[1], ss[2], ss[3], pr.eps, rs);
        unpack8<kHalf>(nw, w);
        unpack8<kHalf>(nb, b);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float v[8];
          unpack8<kHalf>(raw[r], v);
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = layer_norm16<kHalf>(v[e], mean[r], rs[r], w[e], b[e]);
#pragma unroll
          for (int e = 0; e < 4; ++e) raw[r][e] = pack2<kHalf>(v[2 * e], v[2 * e + 1]);
        }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 8 * r + (lane >> 3), m = m_first + row;
        if (pr.rope) {
          const float* c = reinterpret_cast<const float*>(lds + tables(i)) + (32 * wm + row) * kHead + d;
          const bool video = m - batch_of(m) * a.S >= a.T;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const f32x2 z = unpack2<kHalf>(raw[r][e]);
            const f32x2 cs = *reinterpret_cast<const f32x2*>(c + 2 * e), sn = *reinterpret_cast<const f32x2*>(c + kTable / 4 + 2 * e);
            const uint32_t y = pack2<kHalf>(rotated(z.x, -z.y, cs.x, sn.x), rotated(z.y, z.x, cs.y, sn.y));
            raw[r][e] = video ? y : raw[r][e];
          }
        }
        if (m < a.M) *reinterpret_cast<u32x4*>(pr.y + (int64_t)m * a.N + n_proj + d) = raw[r];
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    if (i + kPieces32 < MB) {   // everybody is done with this piece's tables
      step_barrier();
      load_tables(i + kPieces32);
    }
  }
}

template <int MB, int WM, int KH, int NBUF>
constexpr int lds_bytes() {
  return std::max(NBUF * (32 * MB * WM + kHead * (kWaves / WM)) * KH * 32, kStageBytes + table_pieces(MB, WM) * 2 * 32 * WM * kHead * 4);
}

template <int MB, int WM, int KH, int NBUF, bool kHalf>
int launch_t(QkvArgs& a, hipStream_t stream) {
  constexpr int BM = 32 * MB * WM, BN = kHead * (kWaves / WM), kBytes = lds_bytes<MB, WM, KH, NBUF>();
  static_assert(kBytes <= kLds, "the LDS of a CU");
  static thread_local int allowed_dev = -1;   // more than 64 KB of dynamic LDS has to be allowed once per kernel and device
  int dev = 0;
  if (int rc = hip_fail(hipGetDevice(&dev), "hipGetDevice")) return rc;
  if (allowed_dev != dev) {
    if (int rc = hip_fail(hipFuncSetAttribute(reinterpret_cast<const void*>(&qkv_kernel<MB, WM, KH, NBUF, kHalf>), hipFuncAttributeMaxDynamicSharedMemorySize, kBytes),
                          "hipFuncSetAttribute"))
      return rc;
    allowed_dev = dev;
  }
  a.m_tiles = (a.M + BM - 1) / BM;
  a.tiles = a.m_tiles * ((3 * a.N + BN - 1) / BN);
  a.per_xcd = (a.tiles + kXcds - 1) / kXcds;
  a.by_s = quotient_by(a.S);
  hipLaunchKernelGGL((qkv_kernel<MB, WM, KH, NBUF, kHalf>), dim3((unsigned)a.per_xcd * kXcds), dim3(kThreads), kBytes, stream, a);
  return hip_fail(hipGetLastError(), "qkv launch");
}
template <int MB, int WM, int KH, int NBUF>
int launch(QkvArgs& a, bool half, hipStream_t stream) {
  return half ? launch_t<MB, WM, KH, NBUF, true>(a, stream) : launch_t<MB, WM, KH, NBUF, false>(a, stream);
}

// Which tile a launch takes: 64 x 256, two workgroups a CU, 192 x 256, 256 x 256 or 320 x 256.  The time of each in us is its rounds of the
// 256 CUs times the 64-channel steps of one, and what a round and the launch cost on top; constants fitted in loops of calls, those of the last one with
// tiles of 160 x 512, whose place it has taken.  Over 77 launches of 8 ... 48 heads (8 ... 48 steps) x 280 ... 12 000 tokens with the GPU kept busy the
// choice takes 0.04 % more than the best of the four on average and 2.7 % at most (24 x 11 853: 206 us, 320 x 256 200); the times are 11 to 17 % above
// the measured ones, those of each tile alike.  us, 64 x 256 / 192 x 256 / 256 x 256 / 320 x 256: 16 heads x 602 tokens 15 / 27 / 33 / 42; 24 x 4330
// 93 / 81 / 95 / 70; 48 x 2222 162 / 129 / 157 / 120 (252 workgroups of 320 x 256, one round); 48 x 3328 241 / 194 / 172 / 207 (468 of 256 x 256, two).
enum Tiles { kFew, kSome, kMore, kMany };
Tiles plan(int M, int N, int K) {
  constexpr int kCus = 32;   // of an XCD
  const double steps = K / 64.0;
  auto per_xcd = [&](int bm, int bn) { return ((int64_t)((M + bm - 1) / bm) * ((3 * N + bn - 1) / bn) + kXcds - 1) / kXcds; };
  auto time = [&](int bm, int bn, double launch, double step, double round) {
    const double rounds = (double)((per_xcd(bm, bn) + kCus - 1) / kCus);
    return launch + rounds * step * steps + (rounds - 1) * round;
  };
  const int64_t pairs = per_xcd(64, 256) / (2 * kCus), rest = per_xcd(64, 256) % (2 * kCus);
  const double shared = (double)(pairs + (rest > kCus ? 1 : 0)), alone = rest > 0 && rest <= kCus ? 1 : 0;
  const double of[4] = {4.2 + alone * (2.7 + 0.80 * steps) + shared * (9.1 + 1.08 * steps), time(192, 256, 15.4, 1.18, 16.0),
                        time(256, 256, 17.0, 1.45, 16.0), time(320, 256, 19.8, 1.96, 24.9)};
  return (Tiles)(std::min_element(of, of + 4) - of);
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace
}  // namespace dt

using namespace dt;

extern "C" int dt_qkv_project(const void* text, int64_t text_stride_b, int64_t text_stride_s, int32_t T, const void* video,
                              int64_t video_stride_b, int64_t video_stride_s, int32_t V, int32_t B, int32_t K, int32_t H, int32_t D,
                              const dt_projection* proj, const float* cos, const float* sin, int32_t rounding, void* stream) {
  if (B <= 0 || T < 0 || V < 0 || T > INT32_MAX - V || T + V <= 0 || H <= 0 || K <= 0) {
    set_error("B, T + V, H and K must be positive (got %d, %d + %d, %d, %d)", B, T, V, H, K);
    return DT_ERR_INVALID;
  }
  if (D != kHead || K % 64) {
    set_error("head dim %d and %d input channels not built (64, and multiples of 64, are)", D, K);
    return DT_ERR_UNSUPPORTED;
  }
  if ((int64_t)B * (T + V) > (1 << 24) || H > (1 << 16) || K > (1 << 20)) {
    set_error("too many tokens, heads or channels (%lld, %d, %d)", (long long)B * (T + V), H, K);
    return DT_ERR_INVALID;
  }
  if ((T > 0 && (!text || !aligned16(text))) || (V > 0 && (!video || !aligned16(video))) || (text_stride_b & 7) || (text_stride_s & 7) ||
      (video_stride_b & 7) || (video_stride_s & 7) || !proj) {
    set_error("tokens must be non-null, 16-byte aligned, with strides that are multiples of 8 elements; three projections are needed");
    return DT_ERR_INVALID;
  }
  if (rounding & ~DT_IO_FP16) {
    set_error("bad rounding code %d", rounding);
    return DT_ERR_INVALID;
  }
  QkvArgs a{};
  a.text = static_cast<const uint16_t*>(text); a.video = static_cast<const uint16_t*>(video);
  a.text_sb = text_stride_b; a.text_ss = text_stride_s; a.video_sb = video_stride_b; a.video_ss = video_stride_s;
  a.T = T; a.S = T + V; a.M = B * (T + V);
  a.N = H * kHead; a.K = K;
  a.cos = cos; a.sin = sin;
  for (int i = 0; i < 3; ++i) {
    const dt_projection& p = proj[i];
    if (!p.weight || !p.out || !aligned16(p.weight) || !aligned16(p.out) || !aligned16(p.bias) || !aligned16(p.norm_weight) || !aligned16(p.norm_bias)) {
      set_error("projection %d: null weight or output, or a pointer that is not 16-byte aligned", i);
      return DT_ERR_INVALID;
    }
    if (p.norm != DT_NORM_NONE && p.norm != DT_NORM_LAYER) {
      set_error("projection %d: bad norm code %d", i, p.norm);
      return DT_ERR_INVALID;
    }
    if (p.rope && V > 0 && (!cos || !sin || !aligned16(cos) || !aligned16(sin))) {
      set_error("cos/sin tables must be non-null and 16-byte aligned");
      return DT_ERR_INVALID;
    }
    a.proj[i] = {static_cast<const uint16_t*>(p.weight), static_cast<const uint16_t*>(p.bias), static_cast<uint16_t*>(p.out),
                 static_cast<const uint16_t*>(p.norm_weight), static_cast<const uint16_t*>(p.norm_bias), p.norm, p.rope != 0 && V > 0, p.eps};
  }
  const bool half = (rounding & DT_IO_FP16) != 0;
  const hipStream_t s = (hipStream_t)stream;
  switch (plan(a.M, a.N, K)) {
    case kFew: return launch<1, 2, 4, 2>(a, half, s);
    case kSome: return launch<3, 2, 4, 2>(a, half, s);
    case kMore: return launch<4, 2, 4, 2>(a, half, s);
    default: return launch<5, 2, 2, 3>(a, half, s);
  }
}
