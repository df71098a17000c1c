// Chunk attention forward for gfx950 (MI355X): out = softmax(q k^T * scale) v and
// the natural-log lse of one query shard against one or several KV chunks.
//
// Stands in for flash_attn_func as called at core/attention.py:137-143,185-191
// of the reference.
//
// Shape of the computation
//   * One workgroup = 8 wavefronts = 256 queries of one (batch, head); each
//     wavefront owns 32 queries.  D = 128: one workgroup per CU, two wavefronts per
//     SIMD (256 VGPRs each); D = 64: two workgroups per CU (128 VGPRs each).
//     (Launches too small to fill the chip with those: 32 queries, whose keys
//     the wavefronts share, see attn_rows32.)
//   * The 8 wavefronts form two groups of 4 that run the same loop ONE PHASE
//     APART ("ping-pong"): while group A issues the MFMAs of a tile
//     (O^T += V^T P^T of the previous tile, then S^T = K Q^T of this one), group B
//     runs the VALU half (online softmax of its tile, issuing the loads of a later
//     K/V tile), and vice versa; a workgroup barrier separates the
//     phases.  Each SIMD holds one wavefront of either group, so its matrix pipe
//     and its vector ALU are busy at the same time instead of taking turns.
//   * KV is consumed in tiles of 64 keys, staged in LDS as they come, [key][d],
//     four buffers per operand.  A tile goes from global memory STRAIGHT into
//     LDS (buffer loads with the LDS as destination: no registers, no LDS write
//     instructions, no wait for them in the softmax), issued three (K) and two
//     (V) tiles ahead of their first use.  Staging through registers cost a
//     fifth of the loop's cycles: the fill's LDS writes queue up in front of the
//     operand reads of the wavefronts that are issuing MFMAs.  Such a load writes
//     1 KB of consecutive LDS bytes, so rows are not padded but XOR-swizzled (the
//     lane picks which 16 bytes of global memory it fetches); operand reads stay
//     bank-conflict free and use immediate offsets from a few per-lane address
//     registers.  The second MFMA needs V^T; the transposition is done by the
//     LDS read itself (ds_read_b64_tr_b16).  The buffer descriptor lives in
//     scalar registers, and rows past the end of a chunk arrive as zeros.
//   * Scores are computed TRANSPOSED, S^T = K Q^T, with v_mfma_f32_32x32x16_bf16:
//     in the accumulator layout a lane then owns ONE query (column lane%32) and
//     16 of the 32 keys of the tile, so the online-softmax max/sum are
//     in-register reductions plus a single exchange with lane^32.
//   * The rows of the K operand are permuted (bits 2 and 3 of the row index
//     swapped) so that the 8 accumulator registers a lane holds for a half tile
//     are 8 CONSECUTIVE keys.  Rounded to bf16 they are directly the B operand
//     of the second MFMA, O^T += V^T P^T, whose A operand (8 consecutive keys of
//     one d column) is two transposing reads of 4 keys each.
//   * O^T stays in registers as [d][query]: a rescale is a multiply by a per-lane
//     scalar.  The reference maximum the accumulators are scaled to may lag behind
//     the true row maximum (the lse stays exact): the common path computes no row
//     maximum at all, the fp32 row sum it needs anyway is the overflow detector,
//     and only a tile whose sum exceeds 2^12 is redone with its exact maximum.  The epilogue
//     transposes through LDS so that the global stores are 16 bytes per lane.
//   * Workgroups are mapped to (head, query tile) so that the 8 XCDs each work
//     through a contiguous range of heads: the workgroups that share an XCD's
//     L2 stream the same K/V.
#include <algorithm>
#include <cmath>
#include <cstddef>
#include <mutex>
#include <type_traits>

#include "attn_schedule.h"
#include "dt_common.h"

namespace dt {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// The 16-bit element type of q, K, V, P and the output states: bfloat16, or IEEE half (kHalf).  Loads, LDS
// layout, swizzles and the transposing reads only see 16-bit elements; the type decides the MFMA and the
// roundings of P and of the output.
template <bool kHalf>
struct Elem {
  typedef __bf16 t;
  typedef __bf16 x8 __attribute__((ext_vector_type(8)));
  typedef __bf16 x4 __attribute__((ext_vector_type(4)));
  typedef __bf16 x2 __attribute__((ext_vector_type(2)));
  __device__ static __forceinline__ f32x16 mfma(x8 a, x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
  // two packed elements of a 32-bit word, widened
  __device__ static __forceinline__ f32x2 widen(uint32_t w) {
    f32x2 f;
    f.x = __builtin_bit_cast(float, w << 16);
    f.y = __builtin_bit_cast(float, w & 0xffff0000u);
    return f;
  }
};
template <>
struct Elem<true> {
  typedef _Float16 t;
  typedef _Float16 x8 __attribute__((ext_vector_type(8)));
  typedef _Float16 x4 __attribute__((ext_vector_type(4)));
  typedef _Float16 x2 __attribute__((ext_vector_type(2)));
  __device__ static __forceinline__ f32x16 mfma(x8 a, x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
  __device__ static __forceinline__ f32x2 widen(uint32_t w) {
    return __builtin_convertvector(__builtin_bit_cast(x2, w), f32x2);
  }
};

constexpr int kWaves = 8;
constexpr int kThreads = kWaves * 64;
constexpr int kBQ = kWaves * 32;  // queries per workgroup
constexpr int kBK = 64;           // keys per tile
constexpr int kXcds = 8;
constexpr int kNumBuf = DT_SCHED_NUM_BUF;  // LDS buffers per operand; a tile uses buffer (tile & 3)
static_assert(kNumBuf == 4, "buffer indices are computed with & 3 and the loop is unrolled by four");
constexpr int kRingDepth = 4;     // operand fragments the LDS reads of a matrix phase run ahead of its MFMAs (2 and 6 measured: no gain)
// Row permutation of the K operand: MFMA row i -> key (within a 32-key half tile).
__device__ __forceinline__ int key_of_row(int i) {
  return (i & 19) | ((i & 4) << 1) | ((i & 8) >> 1);
}

// Raw buffer descriptor word 3 for gfx9-family targets (32-bit data format, no swizzle).
constexpr int kRsrcFlags = 0x00020000;

// Workgroup barrier between the phases.  Waits for this wavefront's LDS traffic only:
// global loads issued for a later tile stay in flight across it.
__device__ __forceinline__ void phase_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}
// Waits until at most N of this wavefront's tile loads are still in flight.  N comes from attn_schedule.h.
template <int N>
__device__ __forceinline__ void wait_tile_loads() {
#define DT_WAIT_VMCNT(K) asm volatile("s_waitcnt vmcnt(" #K ")" ::: "memory")
  if constexpr (N == 0) DT_WAIT_VMCNT(0);
  else if constexpr (N == 3) DT_WAIT_VMCNT(3);
  else if constexpr (N == 4) DT_WAIT_VMCNT(4);
  else if constexpr (N == 5) DT_WAIT_VMCNT(5);
  else if constexpr (N == 6) DT_WAIT_VMCNT(6);
  else if constexpr (N == 8) DT_WAIT_VMCNT(8);
  else {
    static_assert(N == 10, "add the immediate for this wait count");
    DT_WAIT_VMCNT(10);
  }
#undef DT_WAIT_VMCNT
}
// The same barrier with the results of the finished phase routed through it as in/out
// operands.  Register-only code may otherwise migrate across an asm statement; tied to it,
// the phase's work stays on its own side (the vector phase produces P^T, the matrix phase
// produces S^T and updates O^T).
// After a vector phase the wavefront also waits for the direct-to-LDS tile loads it issued earlier,
// all but the kInFlight newest: behind the barrier they are visible to every wavefront.
template <int kInFlight, typename V, int NK>
__device__ __forceinline__ void phase_barrier_after_vector(V (&p)[NK][2]) {
  __builtin_amdgcn_sched_barrier(0);
#define DT_VECTOR_BARRIER(N)                                                      \
  if constexpr (NK == 2)                                                          \
    asm volatile("s_waitcnt vmcnt(" #N ") lgkmcnt(0)\n\ts_barrier"                 \
                 : "+v"(p[0][0]), "+v"(p[0][1]), "+v"(p[1][0]), "+v"(p[1][1])     \
                 :                                                                \
                 : "memory");                                                     \
  else                                                                            \
    asm volatile("s_waitcnt vmcnt(" #N ") lgkmcnt(0)\n\ts_barrier" : "+v"(p[0][0]), "+v"(p[0][1]) : : "memory")
  if constexpr (kInFlight == 6) { DT_VECTOR_BARRIER(6); }
  else if constexpr (kInFlight == 3) { DT_VECTOR_BARRIER(3); }
  else if constexpr (kInFlight == 2) { DT_VECTOR_BARRIER(2); }
  else {
    static_assert(kInFlight == 1, "loads in flight across the barrier: 1, 2, 3 or 6");
    DT_VECTOR_BARRIER(1);
  }
#undef DT_VECTOR_BARRIER
  __builtin_amdgcn_sched_barrier(0);
}
template <typename V, int NK, int NO>
__device__ __forceinline__ void phase_barrier_after_matrix(V (&sa)[NK], V (&oa)[NO]) {
  __builtin_amdgcn_sched_barrier(0);
  // (two statements: the operands are tied to the first, the barrier follows it)
  if constexpr (NK == 2) asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(sa[0]), "+v"(sa[1]) : : "memory");
  else asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(sa[0]) : : "memory");
  if constexpr (NO == 4) asm volatile("s_barrier" : "+v"(oa[0]), "+v"(oa[1]), "+v"(oa[2]), "+v"(oa[3]) : : "memory");
  else asm volatile("s_barrier" : "+v"(oa[0]), "+v"(oa[1]) : : "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// A tile's per-lane sum of probabilities (32 of them) above which the tile is redone with an
// exact row maximum.  Below it every probability is at most 2^12: harmless for the bf16
// operand (same relative precision at any exponent), inside the range of the fp16 operand (largest
// finite value 65504; the reference never exceeds the row's true maximum, so a probability is at least its
// true softmax weight and loses no more to fp16's small end than under an exact maximum) and for the fp32
// accumulators.
constexpr float kSumLimit = 4096.0f;
// The same for queries that come with softmax_scale * log2(e) folded in (kPre): rows keep the
// reference 0 while the maximum of their first tile lies in [kBandLo, kBandHi] (powers of two;
// 2^-40 .. 2^24 neither underflows nor overflows anything downstream), so a probability is then
// simply exp2(score), and a tile is redone when its sum exceeds 2^40.
constexpr float kSumLimitPre = 1099511627776.0f;
constexpr float kBandLo = -40.f, kBandHi = 24.f;
// References of up to this many log2 units are taken off by the MFMAs themselves (see kRefInC).  A score near 0 then keeps the
// roundings of D / 16 MFMAs at the size of the reference: 8 times 2^-18 at most, 2^-15 log2 units, for references of 64.  (Where the reference is
// above it, its weight is 2^-64; one below it is a first tile's, which a later one leaves.)  Beyond that the scores stay whole and their
// maximum comes off in the exponent.
constexpr float kRefInCMost = 64.f;

template <int D>
struct Tile {
  // Both tiles sit in LDS as [key][d] rows WITHOUT padding: a tile arrives through direct-to-LDS
  // buffer loads, and one such instruction writes 1 KB of consecutive LDS bytes (lane L -> bytes
  // 16 L .. 16 L + 15), so rows cannot be padded.  Bank conflicts are avoided by swizzling instead:
  // which 16 bytes of global memory a lane fetches is free, so a row's 16-byte chunks (K) or
  // 64-byte segments (V) are stored XOR-permuted by a function of the row.
  //   K: chunk c of row r sits at chunk position c ^ swz_k(r); the 16 lanes of a ds_read_b128 pass
  //      read 16 rows at the same c and land in 16 distinct 16-byte bank groups.
  //   V: segment g of row r sits at segment position g ^ swz_v(r); a transposing 8-byte read pass
  //      touches 4 rows x one 64-byte segment, which land in the four quarters of the banks.
  // swz_v only depends on row bits that the immediate row steps of the operand reads (multiples
  // of 4 rows) leave alone; the per-lane part of the swizzle is folded into a few precomputed
  // address registers (one per k-step for K, one per 32 columns for V).
  static constexpr int kRowBytes = D * 2;
  static constexpr int kChunks = D / 8;               // 16-byte chunks per row
  static constexpr int kSegs = D / 32;                // 64-byte segments per row
  static constexpr int kBytesK = kBK * kRowBytes;
  static constexpr int kBytesV = kBK * kRowBytes;
  static constexpr int kOffV = kNumBuf * kBytesK;     // V buffers follow the K buffers
  static constexpr int kBlocks = kBytesK / 1024;      // direct-load instructions per tile and operand
  static constexpr int kLoads = kBlocks / kWaves;     // ... per wavefront (2 or 1)
  static constexpr int kRowsPerBlock = 1024 / kRowBytes;
  static constexpr int kLdsTiles = kNumBuf * (kBytesK + kBytesV);
  static constexpr int kStageBytes = 32 * D;          // epilogue: 32 rows x half the columns of a wavefront's output
  static constexpr int kLdsBytes = kLdsTiles + kWaves * kStageBytes;   // all of a CU's 160 KB: one workgroup at 128, two at 64
  static_assert(D == 128 || D == 64, "swizzles are written for these two head dimensions");
  __device__ static constexpr int swz_k(int row) { return D == 128 ? (row & 15) : ((row >> 1) & 7); }
  // staging rows are written 8 bytes per lane, 32 rows side by side: 16 of them in distinct banks
  __device__ static constexpr int swz_o(int row) { return D == 128 ? ((row >> 1) & 7) : ((row >> 2) & 3); }
  __device__ static constexpr int swz_v(int row) { return D == 128 ? (row & 3) : ((row >> 1) & 1); }
};

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
// Transposing LDS read (ds_read_b64_tr_b16).  Within each block of 16 lanes the 16 x 4 matrix of
// 16-bit elements [source lane][element] is read as 4 rows of 16 (source lane 4j+m supplies
// row j, columns 4m..4m+3) and lane i receives column i: element j = row j, column i.
__device__ __forceinline__ s16x4 lds_read_tr(const uint8_t* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (s16x4 __attribute__((address_space(3)))*)(p));
}

// Raw buffer descriptor: base address, stride 0, number of valid bytes, flags.
__device__ __forceinline__ u32x4 make_rsrc(const void* base, uint32_t valid_bytes) {
  const uint64_t p = reinterpret_cast<uint64_t>(base);
  u32x4 r;   // uniform by construction; say so, the descriptor then lives in scalar registers
  r.x = __builtin_amdgcn_readfirstlane((uint32_t)p);
  r.y = __builtin_amdgcn_readfirstlane((uint32_t)(p >> 32) & 0xffffu);
  r.z = __builtin_amdgcn_readfirstlane(valid_bytes);
  r.w = (uint32_t)kRsrcFlags;
  return r;
}
// One 16-byte-per-lane buffer load whose destination is the LDS: lane L's bytes land at
// lds_addr + 16 L (lds_addr, through M0, is uniform).  Written as inline assembly on purpose: the
// compiler, when it sees such a load, makes every later LDS read of the wavefront wait for ALL
// outstanding loads (it cannot tell that the reads touch other buffers), which turns a prefetch
// several phases deep into one that must land within the phase.  Here the waits are the explicit
// vmcnt in front of the barriers.  (Loads the compiler does not know of only make its own vmcnt
// waits for other loads stricter, never too weak: the counter retires in order.)
__device__ __forceinline__ void load_block_to_lds(u32x4 rsrc, uint32_t lane_off, uint32_t uniform_off, uint32_t lds_addr) {
  // (the uniform operands are uniform by construction; say so, or a value the compiler happens to
  // hold in a vector register ends up in the instruction as one)
  u32x4 r;
  r.x = __builtin_amdgcn_readfirstlane(rsrc.x);
  r.y = __builtin_amdgcn_readfirstlane(rsrc.y);
  r.z = __builtin_amdgcn_readfirstlane(rsrc.z);
  r.w = __builtin_amdgcn_readfirstlane(rsrc.w);
  asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds"
               :
               : "v"(lane_off), "s"(r), "s"(__builtin_amdgcn_readfirstlane(uniform_off)),
                 "s"(__builtin_amdgcn_readfirstlane(lds_addr))
               : "memory", "m0");
}
// The wavefront's next 1 KB block of the same tile: same M0, the instruction's immediate offset moves both the LDS
// address and the global address on by 1 KB (lane_off is reduced by as much where the global side should not move).
// Rewriting M0 between two such loads costs about 17 cycles each time: the write waits until the load before it
// has read the register.
__device__ __forceinline__ void load_next_block_to_lds(u32x4 rsrc, uint32_t lane_off, uint32_t uniform_off) {
  u32x4 r;
  r.x = __builtin_amdgcn_readfirstlane(rsrc.x);
  r.y = __builtin_amdgcn_readfirstlane(rsrc.y);
  r.z = __builtin_amdgcn_readfirstlane(rsrc.z);
  r.w = __builtin_amdgcn_readfirstlane(rsrc.w);
  asm volatile("buffer_load_dwordx4 %0, %1, %2 offen offset:1024 lds"
               :
               : "v"(lane_off), "s"(r), "s"(__builtin_amdgcn_readfirstlane(uniform_off))
               : "memory");
}
// The same from an address of each lane's own.
__device__ __forceinline__ void load_rows_to_lds(const uint16_t* from, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
               :
               : "v"(from), "s"(__builtin_amdgcn_readfirstlane(lds_addr))
               : "memory", "m0");
}

// Segment boundaries are read through the constant address space, i.e. with scalar loads: the lists were
// written before the launch and the address is uniform.  (As a vector load the compiler follows it with
// vmcnt(0), which inside the loop would also wait for every tile load in flight.)
typedef const int32_t __attribute__((address_space(4))) ConstI32;
__device__ __forceinline__ int boundary(const int32_t* list, int i) { return ((ConstI32*)list)[i]; }

// What launch job `job` is: its chunk references, its query rows, its destination.
struct JobView {
  int seg_begin, seg_end, single;   // chunk references [seg_begin, seg_end), or the one chunk `single` >= 0
  int q_begin, q_end;
  int vseg;                         // segment of a packed variable-length batch (device-listed jobs only)
  int dseg;                         // segment whose boundaries are read from device memory (a.cu_q != nullptr)
  uint16_t* out;
  float* lse;
};
template <typename Args>
__device__ __forceinline__ bool view_job(Args& a, int job, JobView& v) {
  v.single = -1;
  v.q_begin = 0;
  v.q_end = a.Sq;
  v.vseg = -1;
  v.dseg = -1;
  if (a.dev_ids != nullptr) {
    int slot = job;
    if (a.n_seg > 0) {
      const int r = job / a.n_slots;
      slot = job - r * a.n_slots;
      v.vseg = a.n_seg - 1 - r;
    }
    if (slot >= *a.dev_count) return false;
    v.single = __builtin_amdgcn_readfirstlane(a.dev_ids[slot]);  // uniform by construction; tell the compiler
    if (v.single < 0 || v.single >= a.n_chunks) return false;  // never index the tables with a bad id
    v.seg_begin = 0;
    v.seg_end = 1;
    if (v.single == a.diag) {
      v.out = a.diag_out;
      v.lse = a.diag_lse;
    } else {
      v.out = a.slot_out + (int64_t)v.single * a.slot_out_stride;
      v.lse = a.slot_lse + (int64_t)v.single * a.slot_lse_stride;
    }
    if (v.vseg >= 0) {
      if (a.cu_q != nullptr) {
        v.dseg = v.vseg;
      } else {
        v.q_begin = a.seg_q_begin[v.vseg];
        v.q_end = v.q_begin + a.seg_q_len[v.vseg];
      }
    }
  } else {
    v.seg_begin = a.job[job].begin;
    v.seg_end = a.job[job].end;
    v.out = a.job[job].out;
    v.lse = a.job[job].lse;
    if (a.cu_q != nullptr) {
      v.dseg = a.job[job].q_begin;
    } else {
      v.q_begin = a.job[job].q_begin;
      v.q_end = v.q_begin + a.job[job].q_len;
    }
  }
  if (v.dseg >= 0) {
    // boundaries from device memory: nothing on the host has looked at them, so they are clamped
    // to the rows that exist (a malformed list then yields wrong rows, never a stray access)
    v.q_begin = min(max(boundary(a.cu_q, v.dseg), 0), a.Sq);
    v.q_end = min(max(boundary(a.cu_q, v.dseg + 1), v.q_begin), a.Sq);
  }
  return true;
}

// The arguments where they arrive (see attn_fwd_kernel), as a reference that the compiler cannot relate to another.
typedef const AttnArgs __attribute__((address_space(4))) KernArgs;
__device__ __forceinline__ KernArgs& kernel_args() {
  uint64_t p = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return *(KernArgs*)p;
}

// Chunk reference `seg` of a job: keys [begin, begin + len) of chunk cid.
struct KeyRef {
  int cid, begin, len;
};
__device__ __forceinline__ KeyRef key_ref(const JobView& v, int seg) {
  KernArgs& a = kernel_args();
  KeyRef r;
  if (v.single < 0) {
    r.cid = a.entry[seg].chunk;
    r.begin = a.entry[seg].kv_begin;
    r.len = a.entry[seg].kv_len;
  } else {
    r.cid = v.single;
    r.begin = 0;
    // (with boundaries in device memory the table holds no ranges, and (chunk, segment) pairs are not bounded by its size)
    if (v.vseg >= 0 && v.dseg < 0) {
      r.begin = a.entry[v.single * a.n_seg + v.vseg].kv_begin;
      r.len = a.entry[v.single * a.n_seg + v.vseg].kv_len;
    } else {
      r.len = a.chunk[v.single].len;
    }
  }
  if (v.dseg >= 0) {
    const int keys = a.chunk[r.cid].len;
    r.begin = min(max(boundary(a.cu_kv[r.cid], v.dseg), 0), keys);
    r.len = min(max(boundary(a.cu_kv[r.cid], v.dseg + 1), r.begin), keys) - r.begin;
  }
  return r;
}

// Work items of fewer key tiles than this are never cut along the keys or the rows: an item costs about four tiles on top of its
// own, and a segment of a few padding tokens keeps the sums of one pass.  us per launch uncut -> cut, 4 heads x 512 queries at
// D = 64 and 24 x 1000 at D = 128: 8 tiles 13.2 -> 10.7, 17.3 -> 15.3; 6 tiles 11.4 -> 9.7, 15.3 -> 13.8; up to 5 tiles the planner
// does not cut.  Tiles of at most 128 rows (always cut from here on), 30 heads x 128, D = 128: 8 tiles 15.6 -> 14.1, 4 tiles 11.4 ->
// 11.4, 2 tiles 9.3 -> 10.0.
constexpr int kMinSplitTiles = 8;

// Wavefronts per SIMD the register budget is set for.  D = 128: two (one workgroup per CU: its LDS
// tiles fill the CU).  D = 64: four, i.e. TWO workgroups per CU (80 KB of LDS and at most 128
// registers each): the second workgroup's wavefronts issue into the barrier waits, the start-up and
// the epilogue of the first, which at 35 key tiles per work item are a tenth of its time (+10 %).
constexpr int kWavesPerSimdD64 = 4;
// Brings the cache lines of the arguments that a workgroup is about to read into the scalar cache, all at once: the
// header, the first jobs, chunks and chunk references.  Read one after the other as the control flow gets to them, each
// line is a cache miss of 0.5 us of its own when a launch starts (stamps of a launch of 4 heads x 512 queries: 2.9 us
// for the argument reads in front of the first tile load, 1.4 with them prefetched; the launch against one key tile 9.5 -> 7.9 us at
// D = 64, 10.3 -> 9.4 at D = 128, together with the wait for Q behind the first tile loads).  The loads and their wait are one asm statement, so no register is pending behind it.
constexpr int kArgLine = 64;
constexpr int kJobAt = (int)offsetof(AttnArgs, job), kChunkAt = (int)offsetof(AttnArgs, chunk), kEntryAt = (int)offsetof(AttnArgs, entry);
__device__ __forceinline__ void prefetch_args(uint64_t args) {
  uint32_t t0, t1, t2, t3, t4, t5, t6, t7, t8, t9, t10, t11, t12, t13;
  asm volatile(
      "s_load_dword %0, %14, 0x0\n\ts_load_dword %1, %14, 0x40\n\ts_load_dword %2, %14, 0x80\n\ts_load_dword %3, %14, 0xc0\n\t"
      "s_load_dword %4, %14, %15\n\ts_load_dword %5, %14, %16\n\ts_load_dword %6, %14, %17\n\ts_load_dword %7, %14, %18\n\t"
      "s_load_dword %8, %14, %19\n\ts_load_dword %9, %14, %20\n\ts_load_dword %10, %14, %21\n\ts_load_dword %11, %14, %22\n\t"
      "s_load_dword %12, %14, %23\n\ts_load_dword %13, %14, %24\n\ts_waitcnt lgkmcnt(0)"
      : "=&s"(t0), "=&s"(t1), "=&s"(t2), "=&s"(t3), "=&s"(t4), "=&s"(t5), "=&s"(t6), "=&s"(t7), "=&s"(t8), "=&s"(t9), "=&s"(t10),
        "=&s"(t11), "=&s"(t12), "=&s"(t13)
      : "s"(args), "i"(kJobAt), "i"(kJobAt + kArgLine), "i"(kJobAt + 2 * kArgLine), "i"(kJobAt + 3 * kArgLine), "i"(kChunkAt),
        "i"(kChunkAt + kArgLine), "i"(kChunkAt + 2 * kArgLine), "i"(kChunkAt + 3 * kArgLine), "i"(kEntryAt), "i"(kEntryAt + kArgLine)
      : "memory");
}

// ---- states that meet inside a launch ----------------------------------------------------------
// What another workgroup of the launch reads (states and partial states of a merging launch) is stored and loaded with the
// device-scope bit: past the L1 and the XCD's L2, so that behind the writer's s_waitcnt vmcnt(0) it is where every XCD finds
// it.  The fences of an acquire and release at device scope do the same to whole caches: the invalidation alone, executed by
// one wavefront per merge, took the keys and values of the XCD's other workgroups out of its L2 and cost 4 us per work
// item (two samples of 24 heads x 1861 queries x 3 of 8 chunks 242 -> 261 us); counting and waiting cost nothing that shows.
constexpr int kNt = 2, kDevice = 16, kDeviceNt = kDevice | kNt;   // cache-policy bits of a raw buffer access: nt, sc1
typedef __amdgpu_buffer_rsrc_t Rsrc;
__device__ __forceinline__ Rsrc buffer_of(const void* base, uint32_t valid_bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, valid_bytes, kRsrcFlags);
}
__device__ __forceinline__ void store_device(float* p, float x) {
  __hip_atomic_store(p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float load_device(const float* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// This wavefront's contribution (device-scope stores) is complete: counts it.  True for the last of `expected`, whose
// device-scope loads then see the contributions of the others, and for which the counter is back at zero.
__device__ __forceinline__ bool arrive_last(uint32_t* counter, int expected) {
  wait_tile_loads<0>();   // (stores as well)
  if (expected > 1) {
    uint32_t before = 0;
    if ((threadIdx.x & 63) == 0) before = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if ((int)__builtin_amdgcn_readfirstlane(before) + 1 != expected) return false;
    if ((threadIdx.x & 63) == 0) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  asm volatile("" ::: "memory");   // no load moves up in front of this
  return true;
}

// Merges the states there are of the 32 query rows from row0 on (one batch and head): out = sum_i w_i out_i / sum_i w_i with
// w_i = exp(lse_i - max), all in fp32.  One wavefront, which needs nobody else: `stage` is LDS of its own.
//
// HBM-bound in large launches: the workgroups run in step, so the last job's all merge at the end of a round, at 5.3 TB/s.
// Against a merge kernel behind the launch: 24 heads x 119 056 queries, 3 of 32 chunks computed 17.79 -> 16.07 ms; 48 heads x
// 2222, D = 64, 5 of 8 340 -> 336 us; 4 heads x 512, D = 64, 2 of 4 19.0 -> 16.3.  Tried without success: the jobs side by side,
// each some items behind the one before it, so that a part of the workgroups merges while the others compute (they fall out of
// step and no longer share keys and values in the L2: 24 heads x 14 882, 4 of 8 8.53 -> 8.75 ms); adjacent heads on the 8 XCDs
// (16.1 -> 16.6 ms).
//
// In small ones a chain of waits at the end of the launch: one wavefront reads 32 rows of all states.  Up to 8 states
// (kOneBatch) every weight is known before the first row, so rows are finished one after the other, without accumulators for
// all of them, and the registers hold loads instead: 128 at D = 128 (4 steps of 8 states or all 8 steps of 4), 64 at D = 64.
// How many steps are in flight decides little at the sizes that merge here (us per call with the GPU kept busy, two -> this: 24
// heads x 96 queries, two states, D = 64 12.8 -> 12.6, D = 128 15.3 -> 15.2, 4 states 15.9 -> 16.4; 12 x 700, D = 64 17.3 -> 17.2; 24 x 4000,
// 3 of 8 chunks 540 -> 540).  More states keep 32 rows of sums in registers and two steps in flight (three make no difference to 29
// states of 743 MB).
template <int D, bool kHalf, int kStates, bool kOneBatch, int kRows = 32>
__device__ __forceinline__ void merge_rows(uint8_t* stage, int b, int h, int row0) {
  typedef Elem<kHalf> E;
  constexpr int kLoads = D == 128 ? kStates : 4;        // states of a step
  constexpr int kParts = kStates / kLoads;              // steps of the same rows
  constexpr int kRowLanes = D / 8;                      // a lane holds 8 columns of a row
  constexpr int kRowsPer = 64 / kRowLanes;              // rows of a load instruction
  constexpr int kRowSteps = kRows / kRowsPer;
  constexpr int kSteps = kRowSteps * kParts;            // steps of a batch of states
  constexpr int kDepthMost = (kOneBatch ? D / 4 : D / 8) / kLoads;
  constexpr int kDepth = kDepthMost < kSteps ? kDepthMost : kSteps;   // steps in flight
  static_assert(kMergeBatch % kStates == 0, "the lists are filled up to whole batches");
  static_assert(kSteps % kDepth == 0, "a step's registers are known at compile time");
  KernArgs& a = kernel_args();
  typedef const AttnState __attribute__((address_space(4))) KernState;
  KernState* states = a.dev_ids ? a.arena : a.state;
  const int lane = threadIdx.x & 63, col = lane & 31;
  const int n = a.merge_n, H = a.H, Sq = a.Sq;
  const int rows = min(kRows, Sq - row0);
  const int64_t lse_at = ((int64_t)b * H + h) * Sq + row0;
  const int64_t out_at = (((int64_t)b * Sq + row0) * H + h) * D;
  const uint32_t row_bytes = (uint32_t)H * D * 2u;
  const uint32_t valid = (uint32_t)(rows - 1) * row_bytes + D * 2u;
  const int my_row = min(col, rows - 1);
  const uint32_t lane_off = (uint32_t)(lane / kRowLanes) * row_bytes + 16u * (uint32_t)(lane % kRowLanes);
  // The batch under the load cursor.  States that are not there (behind the last one, and everything once i0 < 0) are empty
  // descriptors: their loads touch no memory and return zeros.  So do those of rows that are not there.  (The row is part of the
  // lane's offset, as in the stores: the scalar offset stays 0, below the length of every descriptor that is not empty.)
  int i0 = (n - 1) / kStates * kStates;
  u32x4 r[kStates];
  auto open = [&]() __attribute__((always_inline)) {
    KernState* st = states + max(i0, 0);
#pragma unroll
    for (int j = 0; j < kStates; ++j) r[j] = make_rsrc(st[j].out + out_at, i0 >= 0 && i0 + j < n ? valid : 0u);
  };
  u32x4 x[kDepth][kLoads];
  auto load = [&](int s) __attribute__((always_inline)) {
    const uint32_t off = lane_off + (uint32_t)(s / kParts * kRowsPer) * row_bytes;
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      const u32x4& d = r[s % kParts * kLoads + j];
      x[s % kDepth][j] = __builtin_amdgcn_raw_buffer_load_b128(
          __builtin_amdgcn_make_buffer_rsrc((void*)((uint64_t)d.y << 32 | d.x), 0, d.z, kRsrcFlags), off, 0, kDeviceNt);
    }
  };
  float l[kStates];
  auto load_lse = [&](int i0) __attribute__((always_inline)) {   // (the lists go on behind the last state with copies of it)
    KernState* st = states + max(i0, 0);
#pragma unroll
    for (int j = 0; j < kStates; ++j) l[j] = load_device(st[j].lse + lse_at + my_row);
  };
  if (kOneBatch) load_lse(0);
  open();
#pragma unroll
  for (int s = 0; s < kDepth; ++s) load(s);
  float m = -INFINITY, den = 0.f;
  for (int i = 0; i < n; i += kStates) {   // (the last batch, which comes first below, stays in l)
    if (!kOneBatch) load_lse(i);
#pragma unroll
    for (int j = 0; j < kStates; ++j) m = fmaxf(m, l[j]);
    if (kOneBatch) break;
  }
  const bool wide = a.merge_dtype == DT_FP32;
  const Rsrc dst = buffer_of(static_cast<uint8_t*>(a.merge_out) + out_at * (wide ? 4 : 2), wide ? 2 * valid : valid);
  // 1 / sum of the weights of row `col`; -1 for a row whose states are all empty, whose result is 0, whatever the states hold
  float norm;
  auto finish_row = [&]() __attribute__((always_inline)) {
    norm = !(m > -INFINITY) ? -1.f : den > 0.f ? 1.f / den : 0.f;
    if (lane < rows) a.merge_lse[((int64_t)b * Sq + row0 + lane) * H + h] = den > 0.f ? m + __logf(den) : -INFINITY;
  };
  float* weights = reinterpret_cast<float*>(stage);   // [32 rows][kStates]
  auto store_rows = [&](int rs, float f, const float (&sum)[8]) __attribute__((always_inline)) {
    float o[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = f < 0.f ? 0.f : sum[e] * f;
    if (wide) {
      // A lane's 32 bytes as two stores would write every other 16 bytes of a line: through the LDS, so that a store covers
      // whole rows (24 heads x 14 882 queries against one key tile, 8 states merged: 250 -> 232 us; stores of half lines, exchanged
      // in the registers of four lanes, lose as much).
      constexpr int kWeightBytes = kOneBatch ? 32 * kStates * 4 : 0;
      constexpr int kTurns = kWeightBytes + 2048 <= Tile<D>::kStageBytes ? 1 : 2;   // all rows at once, or half of them
      static_assert(kWeightBytes + 2048 / kTurns <= Tile<D>::kStageBytes, "a wavefront's own staging rows");
      uint8_t* rows_at = stage + kWeightBytes;
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        if (kTurns == 1 ? q == 0 : lane / 32 == q) {
#pragma unroll
          for (int e = 0; e < 8; e += 4)
            *reinterpret_cast<f32x4*>(rows_at + (kTurns == 1 ? lane : col) * 32 + 4 * e) = f32x4{o[e], o[e + 1], o[e + 2], o[e + 3]};
        }
        asm volatile("" ::: "memory");   // (a lane that stores nothing would keep what it has read before)
        const u32x4 v = *reinterpret_cast<const u32x4*>(rows_at + (kTurns == 1 ? q * 1024 : 0) + lane * 16);
        asm volatile("" ::: "memory");
        const uint32_t row = (uint32_t)(rs * kRowsPer + q * (kRowsPer / 2)) + (uint32_t)lane / (2 * kRowLanes);
        __builtin_amdgcn_raw_buffer_store_b128(v, dst, 2 * row * row_bytes + 16u * ((uint32_t)lane % (2 * kRowLanes)), 0, kNt);
      }
    } else {
      u32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        f32x2 pair;
        pair.x = o[2 * e];
        pair.y = o[2 * e + 1];
        v[e] = __builtin_bit_cast(uint32_t, __builtin_convertvector(pair, typename E::x2));
      }
      __builtin_amdgcn_raw_buffer_store_b128(v, dst, lane_off + (uint32_t)(rs * kRowsPer) * row_bytes, 0, kNt);
    }
  };
  float acc[kOneBatch ? 1 : kRowSteps][8];
#pragma unroll
  for (auto& row : acc)
#pragma unroll
    for (int e = 0; e < 8; ++e) row[e] = 0.f;
  while (i0 >= 0) {
#pragma unroll
    for (int j = 0; j < kStates; ++j) {
      l[j] = i0 + j < n && m > -INFINITY ? __expf(l[j] - m) : 0.f;
      den += l[j];
    }
    if constexpr (kOneBatch) finish_row();
#pragma unroll
    for (int j = 0; j < kStates; j += 4) *reinterpret_cast<f32x4*>(weights + col * kStates + j) = f32x4{l[j], l[j + 1], l[j + 2], l[j + 3]};
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
      const int rs = s / kParts;
      float (&sum)[8] = acc[kOneBatch ? 0 : rs];
      float f = 0.f;
      if (kOneBatch && s % kParts == kParts - 1) f = __shfl(norm, rs * kRowsPer + lane / kRowLanes);
      const float* ws = weights + (rs * kRowsPer + lane / kRowLanes) * kStates + s % kParts * kLoads;
      f32x4 wv[kLoads / 4];
#pragma unroll
      for (int j = 0; j < kLoads / 4; ++j) wv[j] = *reinterpret_cast<const f32x4*>(ws + 4 * j);
#pragma unroll
      for (int j = 0; j < kLoads; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const f32x2 v = E::widen(x[s % kDepth][j][e]);
          sum[2 * e] = __builtin_fmaf(wv[j / 4][j % 4], v.x, sum[2 * e]);
          sum[2 * e + 1] = __builtin_fmaf(wv[j / 4][j % 4], v.y, sum[2 * e + 1]);
        }
      if (!kOneBatch && s + kDepth == kSteps) {   // the next batch
        i0 -= kStates;
        open();
        load_lse(i0);
      }
      if (!kOneBatch || s + kDepth < kSteps) load((s + kDepth) % kSteps);
      __builtin_amdgcn_sched_barrier(0);   // the loads stay behind the step that frees their registers
      if (kOneBatch && s % kParts == kParts - 1) {
        store_rows(rs, f, sum);
#pragma unroll
        for (int e = 0; e < 8; ++e) sum[e] = 0.f;
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if constexpr (kOneBatch) return;
  }
  finish_row();
  if constexpr (!kOneBatch) {
#pragma unroll
    for (int s = 0; s < kRowSteps; ++s) store_rows(s, __shfl(norm, s * kRowsPer + lane / kRowLanes), acc[s]);
  }
}

// The work of one workgroup: query rows from row0 on of one job, batch and head.  `slice` is
// set to the 32-row slice of the tile whose rows this wavefront has stored, -1 for none.
//
// kSplitKeys: no more than half of the 256 rows exist, or another workgroup has the other half.  Wavefronts w and w + 4 --
// one of either group -- then share 32 queries: the leading group's takes the first 32 keys of every tile, the trailing
// group's the others, and the two states meet in fp32 through the LDS at the end.  Loads, buffers, barriers and waits are
// those of the other form, a wavefront's phases have half the MFMAs and half the softmax.  A tile then takes 0.60 of the
// time of a full one (one round of items of 32 key tiles: D = 128 79 -> 49 us, D = 64 87 -> 52), not half: the load
// instructions and barriers stay.  That much is saved on the last query tile of a head where up to 128 of its rows exist
// (24 heads x 1400 queries x 4 chunks, D = 128: 121 -> 118 us), and by cutting the items of the last round in two (plan_tail).
template <int D, bool kPre, bool kHalf, bool kMerge, bool kSplitKeys>
__device__ __forceinline__ void attn_item(const JobView& view, int b, int h, int row0, bool is_part, int part, int unit, int xcd, int& slice) {
  slice = -1;
  using T = Tile<D>;
  using E = Elem<kHalf>;
  typedef typename E::x8 ex8;
  typedef typename E::x4 ex4;
  typedef typename E::x2 ex2;
  // The scores of a tile start from minus the reference instead of from zero: C of a product's first MFMA, 16 registers of one value
  // since a lane owns one query.  What is left to the softmax is a multiplication in place of the multiply-add: an instruction of
  // half the bytes and operands, which is power the matrix pipe can use.  us per call: 24 heads x 14 882 queries, 4 of 8 chunks 8198 -> 8036, 24 x
  // 119 056, 3 of 32 15 503 -> 15 256, 24 x 4001, 2 of 4 338.4 -> 332.8, 2 x 24 x 1861, 3 of 8 272 -> 269.  (At D = 64 the registers
  // are not there: 56 spilled.)
  constexpr bool kRefInC = D == 128 && !kPre;
  constexpr int kKeyBlocks = kSplitKeys ? 1 : 2;   // 32-key blocks of a tile that a wavefront works on
  // A reference of its own for every place that reads arguments, unrelated to the others as far as the compiler can see:
  // it otherwise reads whole lines at the top and holds what later places need in spilled scalar registers (119 at D = 128 and
  // 116 at D = 64 instead of 109 and 103).
  auto args = []() __attribute__((always_inline)) -> KernArgs& { return kernel_args(); };
  KernArgs& a = args();
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int seg_begin = view.seg_begin, seg_end = view.seg_end;
  const int q_begin = view.q_begin, q_end = view.q_end;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: keeps group/buffer arithmetic scalar
  const int group = wave >> 2;  // 0: leads, 1: runs one phase behind
  const int col = lane & 31;    // query column (B operand) / operand row (A operand)
  const int hh = lane >> 5;     // which half of the contraction dimension this lane feeds
  const int q0 = q_begin + row0 + (kSplitKeys ? wave & 3 : wave) * 32;
  const int key0 = kSplitKeys ? 32 * group : 0;  // first key of a tile that this wavefront works on

  typedef __attribute__((address_space(3))) uint8_t* lds_ptr_t;
  const uint32_t lds_base = (uint32_t)(uintptr_t)(lds_ptr_t)lds;

  // ---- Q: B operand of S^T = K Q^T, kept in registers --------------------------------
  // The wavefront's 32 rows come as whole lines, through the LDS: half of them through its staging rows, a quarter each through
  // its own shares of V buffers 3 and 2, which nothing but its own later tile loads writes.  Read from memory as fragments, a load
  // instruction touched 32 lines for 32 bytes each, in front of all tile loads: from the start of a work item to its first scores 5.4 ->
  // 4.2 us (stamps of 24 heads x 119 056 queries, D = 128), of 98.  us per call, together with the addresses in the epilogue (2.1 -> 1.4 us
  // an item): 16 heads x 300 queries, 2 of 4 chunks, D = 128 19.7 -> 18.0, 24 x 1000, 4 of 8 67.5 -> 65.1, 2 x 24 x 1861, 3 of 8 283.3 ->
  // 278.7; D = 64 4 x 512, 2 of 4 15.4 -> 14.7, 48 x 2222, 5 of 8 340 -> 336; launches at the power cap (24 x 14 882) stay as they are.
  ex8 qf[D / 16];
  constexpr int kQuarter = T::kLoads;   // 1 KB blocks of 8 rows
  const uint32_t q_quarter[4] = {(uint32_t)(T::kLdsTiles + wave * T::kStageBytes), (uint32_t)(T::kLdsTiles + wave * T::kStageBytes + kQuarter * 1024),
                                 (uint32_t)(T::kOffV + 3 * T::kBytesV + wave * kQuarter * 1024),
                                 (uint32_t)(T::kOffV + 2 * T::kBytesV + wave * kQuarter * 1024)};
  {
    const uint16_t* qp = a.q + (int64_t)b * a.q_sb + (int64_t)h * a.q_sh;
#pragma unroll
    for (int i = 0; i < 4 * kQuarter; ++i) {
      const int row = i * T::kRowsPerBlock + lane / T::kChunks;
      const uint32_t chunk = (uint32_t)(lane % T::kChunks) ^ T::swz_k(row);
      load_rows_to_lds(qp + (int64_t)min(q0 + row, q_end - 1) * a.q_ss + 8 * chunk, lds_base + q_quarter[i / kQuarter] + i % kQuarter * 1024);
    }
  }
  // ---- tile bookkeeping -----------------------------------------------------------------
  // Two cursors walk the job's chunks tile by tile, all in scalar registers: the load cursor
  // (ahead of the compute cursor: base pointers of the tile and keys left in its chunk) and
  // the compute cursor (keys left in the chunk of the tile whose scores are being computed).
  // The load cursor addresses a tile as (buffer descriptor of its chunk, byte offset of its first key from the
  // chunk's first key).  The descriptors (base of the chunk's keys for this batch and head, number of valid
  // bytes) only change with the chunk; per tile the cursor moves one scalar offset.  A chunk's (batch, head)
  // plane is below 2 GiB (checked on the host), so offsets fit 32 bits with room for the lane's part.
  const uint32_t row_bytes = (uint32_t)a.kv_ss * 2u;
  const uint32_t tile_bytes = (uint32_t)kBK * row_bytes;
  u32x4 rk, rv;   // K and V of the chunk under the load cursor
  uint32_t k_off = 0u;
  int ld_seg = seg_begin, ld_left = 0;
  int cp_seg = seg_begin, cp_left = 0;
  auto ld_open = [&](const KeyRef& r) __attribute__((always_inline)) {
    k_off = 0u;
    ld_left = r.len;
    if (r.len > 0) {
      KernArgs& a = args();
      const int64_t head_off = (int64_t)b * a.chunk[r.cid].sb + (int64_t)h * a.kv_sh + (int64_t)r.begin * a.kv_ss;
      const uint32_t valid = (uint32_t)(r.len - 1) * row_bytes + (uint32_t)(D * 2);
      rk = make_rsrc(a.chunk[r.cid].k + head_off, valid);
      rv = make_rsrc(a.chunk[r.cid].v + head_off, valid);
    } else {
      // past the last chunk: an empty descriptor, loads store zeros without touching memory
      rk = make_rsrc(nullptr, 0u);
      rv = rk;
    }
  };
  auto ld_next_chunk = [&]() __attribute__((always_inline)) {
    KeyRef r;
    r.len = 0;
    while (r.len == 0 && ++ld_seg < seg_end) r = key_ref(view, ld_seg);
    ld_open(r);
  };
  auto cp_next_chunk = [&]() __attribute__((always_inline)) {
    cp_left = 0;
    while (cp_left == 0 && ++cp_seg < seg_end) cp_left = key_ref(view, cp_seg).len;
  };
  // the first reference opens both cursors (most jobs have no other)
  KeyRef first;
  first.len = 0;
  if (seg_begin < seg_end) first = key_ref(view, seg_begin);
  int n_tiles = (first.len + kBK - 1) / kBK;
  for (int s = seg_begin + 1; s < seg_end; ++s) n_tiles += (key_ref(view, s).len + kBK - 1) / kBK;
  if (__builtin_expect(first.len > 0, 1)) {
    ld_open(first);
    cp_left = first.len;
  } else {
    ld_next_chunk();
    cp_next_chunk();
  }
  if (is_part) {
    // this workgroup covers key tiles [t0, t1) of the item: walk both cursors to t0
    const int ways = n_tiles < kMinSplitTiles ? 1 : a.part_ways;   // (then part 0 covers all, the others nothing)
    const int t0 = min((int)((int64_t)n_tiles * part / ways), n_tiles);
    const int t1 = min((int)((int64_t)n_tiles * (part + 1) / ways), n_tiles);
    int skip = t0;
    while (skip > 0 && ld_seg < seg_end) {
      const int in_chunk = (ld_left + kBK - 1) / kBK;
      if (skip >= in_chunk) {
        skip -= in_chunk;
        ld_next_chunk();
      } else {
        k_off += (uint32_t)skip * tile_bytes;
        ld_left -= skip * kBK;
        skip = 0;
      }
    }
    skip = t0;
    while (skip > 0 && cp_seg < seg_end) {
      const int in_chunk = (cp_left + kBK - 1) / kBK;
      if (skip >= in_chunk) {
        skip -= in_chunk;
        cp_next_chunk();
      } else {
        cp_left -= skip * kBK;
        skip = 0;
      }
    }
    n_tiles = t1 - t0;
  }

  // ---- tile loads: global memory -> LDS without passing through registers ---------------
  // A wavefront brings in kLoads consecutive 1 KB blocks of every K tile and of every V tile (blocks
  // kLoads * wave + i = rows kRowsPerBlock * (kLoads * wave + i) ...; consecutive, so that one M0 value serves
  // all of them).  Lane L of a load lands at LDS bytes
  // 16 L .. 16 L + 15 of the block, i.e. at row L / kChunks, chunk position L % kChunks; it
  // therefore fetches the chunk of global memory that the swizzle assigns to that position.
  // Raw buffer loads: the descriptor (base of the chunk's first key for this batch and head,
  // number of valid bytes) lives in scalar registers, the tile's offset from there travels as the
  // load's scalar offset (which the range check includes), and rows past the end of the chunk fail
  // the hardware bounds check and arrive as zeros (their scores are masked to -inf; zero V rows
  // add nothing).
  // this lane's byte offset from the tile's first key for its i-th block, loop invariant; less the 1 KB per block
  // that the immediate offset of load_next_block_to_lds adds back (a block's rows start at least that far in)
  uint32_t k_goff[T::kLoads], v_goff[T::kLoads];
#pragma unroll
  for (int i = 0; i < T::kLoads; ++i) {
    const int lrow = T::kRowsPerBlock * (T::kLoads * wave + i) + lane / T::kChunks;
    const int pos = lane % T::kChunks;
    k_goff[i] = (uint32_t)lrow * row_bytes + 16u * (uint32_t)(pos ^ T::swz_k(lrow)) - 1024u * i;
    v_goff[i] = (uint32_t)lrow * row_bytes + 16u * (uint32_t)((((pos >> 2) ^ T::swz_v(lrow)) << 2) | (pos & 3)) - 1024u * i;
  }
  static_assert(T::kLoads <= 2 && T::kRowsPerBlock * T::kRowBytes == 1024, "one immediate offset of 1 KB, whole rows per block");
  // Issues this wavefront's loads of V of the tile before the one under the load cursor and of
  // K of the tile under it (tile X, into K buffer X & 3; V is needed two phases later than K, so
  // its loads run one tile behind), and moves the cursor on.  Past the last tile the loads are still
  // issued, against an empty descriptor (they store zeros without touching memory): with the same
  // number of loads in every iteration the counter the barrier waits on is static.
  // V of the previous tile: its offset, and -- only in the call after the cursor changed chunks -- the
  // descriptor of the chunk it belongs to.
  uint32_t v_off = 0u;
  u32x4 rv_old;
  bool v_lags = false, no_v = true;   // the very first call has no previous tile: its share of the V buffer holds rows of Q
  auto load_tile = [&](int kbuf) __attribute__((always_inline)) {
    const int vbuf = (kbuf + kNumBuf - 1) & (kNumBuf - 1);
    const uint32_t kdst = lds_base + kbuf * T::kBytesK + wave * (1024 * T::kLoads);
    const uint32_t vdst = lds_base + T::kOffV + vbuf * T::kBytesV + wave * (1024 * T::kLoads);
    auto load_blocks = [&](const u32x4& rsrc, const uint32_t (&goff)[T::kLoads], uint32_t off, uint32_t dst) __attribute__((always_inline)) {
      load_block_to_lds(rsrc, goff[0], off, dst);
      if constexpr (T::kLoads == 2) load_next_block_to_lds(rsrc, goff[1], off);
    };
    // V first: the barrier waits let the K half of a call stay in flight one vector phase longer
    if (no_v) {
      no_v = false;
    } else if (__builtin_expect(v_lags, 0)) {
      load_blocks(rv_old, v_goff, v_off, vdst);
      v_lags = false;
    } else {
      load_blocks(rv, v_goff, v_off, vdst);
    }
    load_blocks(rk, k_goff, k_off, kdst);
    v_off = k_off;
    k_off += tile_bytes;
    ld_left -= kBK;
    if (__builtin_expect(ld_left <= 0 && ld_seg < seg_end, 0)) {
      rv_old = rv;
      v_lags = true;
      ld_next_chunk();
    }
  };

  // ---- accumulators ---------------------------------------------------------------------
  f32x16 o_acc[D / 32];
#pragma unroll
  for (int i = 0; i < D / 32; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) o_acc[i][r] = 0.f;
  // reference (raw scores; kPre: log2 units) the accumulators are scaled to
  float m_ref = kPre ? 0.f : -INFINITY;
  float rs_bias = kPre ? INFINITY : 0.f;  // kPre: inf until the row has seen a key (forces the exact path)
  bool any_off = kRefInC;                 // some row of this wavefront has a reference that the scores do not start from (kPre: other than 0)
  float limit = kSumLimit;                // kRefInC: -1, below every sum, while some row of this wavefront has no reference
  f32x16 neg_ref;                         // kRefInC: what the scores start from
#pragma unroll
  for (int r = 0; r < 16; ++r) neg_ref[r] = 0.f;
  if constexpr (kRefInC) asm volatile("" : "+v"(neg_ref));   // registers, not a constant to be built for every product
  float l_run = 0.f;        // running sum over THIS lane's keys (halves combined at the end)
  const float c = kPre ? 1.f : a.scale_log2;

  // operand read addresses of this lane within a K / V buffer (the lane's part of the swizzle)
  uint32_t kld[D / 16];  // K fragment of k-step s: row key_of_row(col) (+32 for the second half tile)
  {
    const int krow = key0 + key_of_row(col);
#pragma unroll
    for (int s = 0; s < D / 16; ++s) kld[s] = krow * T::kRowBytes + 16 * ((2 * s + hh) ^ T::swz_k(krow));
  }
  // V operand: this lane is source lane 4j+m of its 16-lane block and supplies keys 8*hh + j,
  // d columns 16*(block parity) + 4m .. +3 of the fragment's 32-column segment
  uint32_t vld[T::kSegs];
  {
    const int vrow = key0 + 8 * hh + ((lane & 15) >> 2);
#pragma unroll
    for (int g = 0; g < T::kSegs; ++g)
      vld[g] = T::kOffV + vrow * T::kRowBytes + 64 * (g ^ T::swz_v(vrow)) + (16 * ((lane >> 4) & 1) + 4 * (lane & 3)) * 2;
  }

  f32x16 s_acc[kKeyBlocks];    // S^T of the tile whose softmax comes next
  ex8 p_frag[kKeyBlocks][2];   // P^T of the tile whose P V product comes next
  int cp_valid = 0;      // keys that exist in the tile held in s_acc

  // S^T = K Q^T for tile 0 only (first matrix phase)
  auto qk_only = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int kb = 0; kb < kKeyBlocks; ++kb) {
#pragma unroll
      for (int r = 0; r < 16; ++r) s_acc[kb][r] = 0.f;
#pragma unroll
      for (int s = 0; s < D / 16; ++s) {
        const ex8 ka = *reinterpret_cast<const ex8*>(lds + kld[s] + kb * 32 * T::kRowBytes);
        s_acc[kb] = E::mfma(ka, qf[s], s_acc[kb]);
      }
    }
  };

  // One matrix phase: O^T += V^T P^T for tile `tile`, then S^T = K Q^T for tile `tile + 1`,
  // as ONE stream of MFMAs fed by a ring of LDS reads kept kRing fragments ahead, so that the
  // single wavefront of this SIMD that is in its matrix phase never waits for LDS latency.
  // (After the last tile the second half recomputes scores on a stale K buffer; they are unused.)
  // U = tile & 3 picks the buffers at compile time: all operand reads use immediate offsets.
  constexpr int kPV = D / 32 * 2 * kKeyBlocks;   // fragments of the P V product
  constexpr int kQK = kKeyBlocks * (D / 16);     // fragments of the score product
  constexpr int kFrags = kPV + kQK;
  constexpr int kRing = kRingDepth;
  // Where a wavefront issues its tile loads: at the start of its vector phase, or behind the
  // MFMAs of its matrix phase (one phase later, and then awaited one call earlier).  At D = 64
  // the vector phase is the longer one (half the MFMAs per softmax element) and the matrix
  // phase has the room (measured +16 %); at D = 128 it is the other way round (+1.5 %).
  constexpr bool kLoadAfterMatrix = (D == 64 ? DT_SCHED_LOAD_AFTER_MATRIX_D64 : DT_SCHED_LOAD_AFTER_MATRIX_D128) != 0;
  static_assert(T::kLoads == (D == 64 ? DT_SCHED_LOADS_D64 : DT_SCHED_LOADS_D128),
                "attn_schedule.h states how many load instructions a wavefront issues per tile and operand");
  // shares of tile loads that may stay in flight across the barrier that ends a vector phase
  constexpr int kVectorInFlight = D == 64 ? DT_SCHED_VECTOR_BARRIER_INFLIGHT_D64 : DT_SCHED_VECTOR_BARRIER_INFLIGHT_D128;
  static_assert(DT_SCHED_PROLOGUE_CALLS_LEADING == DT_SCHED_CALL_AHEAD && DT_SCHED_PROLOGUE_CALLS_TRAILING == DT_SCHED_CALL_AHEAD + 1,
                "the prologue issues exactly the calls the loop's first phase pair assumes: tiles 0 .. 2 + group");
  // The operand ring lives across the barrier in front of a matrix phase: its first kRing
  // fragments (V fragments of a tile completed at least a phase ago) are read at the END of the
  // preceding vector phase, so their LDS latency passes while the wavefront waits at the barrier
  // instead of in front of the first MFMA.
  ex8 ring[kRing];
  auto v_frag = [&](int vbuf, int i) __attribute__((always_inline)) -> ex8 {
    // 8 consecutive keys of one d column = two transposing reads of 4 keys each
    const int db = i % (D / 32), kb = (i / (D / 32)) >> 1, half = (i / (D / 32)) & 1;
    const uint8_t* p = lds + vld[db] + vbuf * T::kBytesV + (32 * kb + 16 * half) * T::kRowBytes;
    const s16x4 lo = lds_read_tr(p);
    const s16x4 hi = lds_read_tr(p + 4 * T::kRowBytes);
    const s16x8 both = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    return __builtin_bit_cast(ex8, both);
  };
  auto ring_prefill = [&](auto u_tag) __attribute__((always_inline)) {
    constexpr int kU = decltype(u_tag)::value;
#pragma unroll
    for (int i = 0; i < kRing; ++i) ring[i] = v_frag(kU, i);
  };
  auto matrix_phase = [&](auto u_tag) __attribute__((always_inline)) {
    constexpr int kU = decltype(u_tag)::value;         // V buffer of this tile
    constexpr int kUK = (kU + 1) & (kNumBuf - 1);      // K buffer of the next tile
    auto frag = [&](int i) -> ex8 {
      if (i < kPV) return v_frag(kU, i);
      const int j = i - kPV;
      const int kb = j % kKeyBlocks, sidx = j / kKeyBlocks;
      return *reinterpret_cast<const ex8*>(lds + kld[sidx] + kUK * T::kBytesK + kb * 32 * T::kRowBytes);
    };
#pragma unroll
    for (int i = 0; i < kFrags; ++i) {
      const ex8 cur = ring[i % kRing];
      if (i + kRing < kFrags) ring[i % kRing] = frag(i + kRing);
      if (i < kPV) {
        const int db = i % (D / 32), kb = (i / (D / 32)) >> 1, half = (i / (D / 32)) & 1;
        o_acc[db] = E::mfma(cur, p_frag[kb][half], o_acc[db]);
      } else {
        const int j = i - kPV;
        const int kb = j % kKeyBlocks, sidx = j / kKeyBlocks;
        if (sidx == 0) {
          f32x16 zero;
#pragma unroll
          for (int r = 0; r < 16; ++r) zero[r] = 0.f;
          s_acc[kb] = E::mfma(cur, qf[sidx], kRefInC ? neg_ref : zero);
        } else {
          s_acc[kb] = E::mfma(cur, qf[sidx], s_acc[kb]);
        }
      }
    }
    // pin the order: the reads of kRing fragments up front (a V fragment is two reads), then the
    // reads of one more fragment behind every MFMA
    static_assert(kRing <= kPV, "the prefill is assumed to consist of V fragments");
#pragma unroll
    for (int i = 0; i < kPV - kRing; ++i) {   // MFMAs whose refill is a V fragment
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
    }
#pragma unroll
    for (int i = 0; i < kQK; ++i) {           // MFMAs whose refill is a K fragment
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, kRing, 0);
  };

  // ---- prologue ---------------------------------------------------------------------------
  // Schedule of the loads (phases are separated by workgroup barriers; group g runs the vector
  // phase of tile t in phase 2t + g and its matrix phase in phase 2t + g + 1):
  //   * K of tile X is read in phases 2X-1 and 2X (scores, matrix phases of tile X-1), V of tile X
  //     at the end of phases 2X and 2X+1 (the operand ring's prefill) and in phases 2X+1 and 2X+2.
  //   * A call of load_tile issues V of tile Y-1 and then K of tile Y.  In the vector phase of
  //     tile t a wavefront of group g makes the call Y = t+3+g: with four buffers per operand the
  //     slot a load overwrites (K of tile Y-4: last read in phase 2Y-8; V of tile Y-5: phase 2Y-8)
  //     is free since the barrier before the phase the load is issued in (2Y-6 or 2Y-7).
  //   * The barrier that ends a vector phase waits for all of the wavefront's loads but the newest
  //     call and the K half of the call before: V of tile t+1+g and K of tile t+1+g are then in
  //     the LDS for everybody, i.e. V one barrier before its first reader (the prefill in phase
  //     2(t+1) + g at the earliest) after three phases in flight, K after five.
  //   * At D = 64 the calls are made behind the MFMAs of the matrix phase instead (see
  //     kLoadAfterMatrix); the barrier of the next vector phase then lets only the K half of the
  //     newest call stay in flight.
  // Here: the calls Y = 0..2 -- the V half of the first has no tile, the wavefront's share of that
  // buffer holds rows of Q -- of which K of tile 0 (first scores) and V of tile 0 (first prefill) are
  // awaited, and Q with them.  The trailing group makes the call Y = 3 once its rows of Q are out of
  // the buffer that it fills, and waits one phase, which staggers the two groups.
  using U0 = std::integral_constant<int, 0>;
  using U1 = std::integral_constant<int, 1>;
  using U2 = std::integral_constant<int, 2>;
  using U3 = std::integral_constant<int, 3>;
#pragma unroll
  for (int y = 0; y < DT_SCHED_PROLOGUE_CALLS_LEADING; ++y) load_tile(y);
  // in flight behind this wait: K of tile 1 and the two shares of the call behind it
  static_assert(DT_SCHED_PROLOGUE_INFLIGHT_TRAILING - 2 * (DT_SCHED_PROLOGUE_CALLS_TRAILING - DT_SCHED_PROLOGUE_CALLS_LEADING) ==
                    DT_SCHED_PROLOGUE_INFLIGHT_LEADING, "the trailing group's last call comes behind the wait: two shares fewer in flight");
  wait_tile_loads<DT_SCHED_PROLOGUE_INFLIGHT_LEADING * T::kLoads>();
  {
    const uint32_t at = q_quarter[0] + col * T::kRowBytes;
    const uint32_t row_at = col < 16 ? at : (col < 24 ? q_quarter[2] : q_quarter[3]) + (col & 7) * T::kRowBytes;
#pragma unroll
    for (int s = 0; s < D / 16; ++s) qf[s] = *reinterpret_cast<const ex8*>(lds + row_at + 16 * ((2 * s + hh) ^ T::swz_k(col)));
  }
  // Route the fragments through an empty asm: they are then defined by it, not by loads that the compiler could repeat.
#pragma unroll
  for (int s = 0; s < D / 16; ++s) asm volatile("" : "+v"(qf[s]));
  phase_barrier();
  if (group == 1) {
#pragma unroll
    for (int y = DT_SCHED_PROLOGUE_CALLS_LEADING; y < DT_SCHED_PROLOGUE_CALLS_TRAILING; ++y) load_tile(y);   // (over rows of Q)
    phase_barrier();
  }
  // first matrix phase: scores of tile 0
  if (n_tiles > 0) {
    qk_only();
    cp_valid = cp_left;
    cp_left -= kBK;
    if (cp_left <= 0) cp_next_chunk();
  }
  // Behind this barrier the leading group computes the scores of tile 1, so K of tile 1 has to be in
  // the LDS from ALL wavefronts.  The leading group waits for its share at the end of its vector
  // phase; the trailing group is in its score-only phase here and has no vector phase in between,
  // so it waits for its share now (of the 7 shares of its four calls, the 3 oldest: K0, V0, K1).
  // From tile 2 on, the wait that ends a group's vector phase covers the tile the other group
  // reads next.
  if (group == 1) wait_tile_loads<DT_SCHED_TRAILING_K1_INFLIGHT * T::kLoads>();
  phase_barrier_after_matrix(s_acc, o_acc);

  // one iteration = vector phase of tile t, then matrix phase (P V of tile t, scores of t+1)
  auto iteration = [&](int t, auto u_tag) __attribute__((always_inline)) -> bool {
    constexpr int kU = decltype(u_tag)::value;  // t & 3
    // ======== vector phase: tile loads for later, online softmax of tile t ========
    // The vector phase runs at raised wave priority: where the two wavefronts of a SIMD compete for
    // the vector issue port, the one doing the softmax goes first.  With equal priorities the older
    // wavefront wins in either role and the phases of the two groups come out unequal (measured
    // 1.43k vs 1.24k cycles of vector work), so every other barrier waits for a squeezed softmax.
    // (D = 64: four wavefronts of two workgroups share the SIMD and the raised priority only gets in
    // the way of the other workgroup's matrix phase: measured -3 %, so it is left at 0 there)
    __builtin_amdgcn_s_setprio(D == 64 ? 0 : 1);
    if constexpr (!kLoadAfterMatrix) load_tile((kU + DT_SCHED_CALL_AHEAD + group) & (kNumBuf - 1));
    // (kPre: the same rare branch takes the reference off the scores of a wavefront in which some
    // row has left the band; everywhere else the reference is 0 and there is nothing to subtract)
    if (__builtin_expect(cp_valid < kBK || (kPre && any_off), 0)) {
      // the empty asm has side effects as far as the compiler knows, which keeps this a real
      // branch: otherwise the selects below are hoisted out and run for every tile
      asm volatile("" ::: "memory");
      const int lim = cp_valid - key0;
#pragma unroll
      for (int kb = 0; kb < kKeyBlocks; ++kb)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = 32 * kb + 16 * (r >> 3) + 8 * hh + (r & 7);
          if (key >= lim) s_acc[kb][r] = -INFINITY;
          if constexpr (kPre) s_acc[kb][r] -= m_ref;
          if constexpr (kRefInC) asm volatile("" : "+v"(s_acc[kb][r]));   // one compare and select after the other: 115 spilled scalars otherwise
        }
    }
    // Probabilities relative to the reference maximum the accumulators are scaled to.  The
    // maximum of the tile is NOT computed on this path: the row sum, needed anyway, doubles as
    // the overflow detector.  While it stays below kSumLimit every probability is bounded and a
    // lagging reference is harmless (the lse stays exact); otherwise -- including the first tile,
    // where the reference is -inf and the sum comes out inf or NaN -- the tile is redone below
    // with its exact maximum.
    float mc = m_ref * c;
    float rs0 = rs_bias, rs1 = 0.f;
    // The first tile of a work item always takes the exact path below (its reference is still -inf), so its pass
    // through the common path is thrown away: skip it.  Results are bit-identical; +0.4-0.5 % at D = 128.  (At
    // D = 64 the extra branch costs registers the kernel does not have: 36 spills, -18 %; it keeps the plain form.)
    // So do all tiles of a wavefront with a reference beyond what the MFMAs take (any_off, which stands for the first tile as well): its scores
    // are whole, and their maximum comes off in the exponent.  With the reference taken off the scores themselves, those behind a first
    // tile far below them lost their last bits: behind 64 keys at scores of -1e5 a score of 1 was off by 6e-3.  us per call, off the scores ->
    // this: 24 heads x 4001 queries, 2 chunks, logits of sigma 16 433 -> 386; 24 x 14 882, 4 chunks 10 500 -> 9780, of sigma 1 (no such row)
    // 8034 -> 8063.  A branch of its own for these tiles, without the maximum, was faster with them (8910) and slower without (8090).
    if (D == 128 && __builtin_expect(kRefInC ? any_off : t == 0, 0)) {
      asm volatile("" ::: "memory");   // keeps this a real branch
      rs0 = INFINITY;
    } else
#pragma unroll
    for (int kb = 0; kb < kKeyBlocks; ++kb)
#pragma unroll
      for (int r = 0; r < 16; r += 2) {
        f32x2 p;
        if constexpr (kPre) {
          p.x = __builtin_amdgcn_exp2f(s_acc[kb][r]);
          p.y = __builtin_amdgcn_exp2f(s_acc[kb][r + 1]);
        } else if constexpr (kRefInC) {
          p.x = __builtin_amdgcn_exp2f(s_acc[kb][r] * c);
          p.y = __builtin_amdgcn_exp2f(s_acc[kb][r + 1] * c);
        } else {
          p.x = __builtin_amdgcn_exp2f(__builtin_fmaf(s_acc[kb][r], c, -mc));
          p.y = __builtin_amdgcn_exp2f(__builtin_fmaf(s_acc[kb][r + 1], c, -mc));
        }
        if (!kPre && kb == 0 && r == 0) {   // the sums start from these two (0 + p is not folded: it would turn -0 into +0)
          rs0 = p.x;
          rs1 = p.y;
        } else {
          rs0 += p.x;
          rs1 += p.y;
        }
        const ex2 pb = __builtin_convertvector(p, ex2);
        p_frag[kb][r >> 3][r & 7] = pb.x;
        p_frag[kb][r >> 3][(r & 7) + 1] = pb.y;
      }
    if (__builtin_expect(__any(!(rs0 + rs1 <= (kPre ? kSumLimitPre : kRefInC ? limit : kSumLimit))), 0)) {
      float mx = s_acc[0][0];
#pragma unroll
      for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s_acc[0][r]);
      if constexpr (kKeyBlocks == 2) {
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s_acc[1][r]);
      }
      mx = fmaxf(mx, __shfl_xor(mx, 32));
      float m_new, alpha;
      if constexpr (kPre) {
        float rs_tot = rs0 + rs1;
        rs_tot += __shfl_xor(rs_tot, 32);
        const bool first = rs_bias != 0.f;
        const float mx_true = mx + m_ref;
        if (first) m_new = (mx_true >= kBandLo && mx_true <= kBandHi) || !(mx_true > -INFINITY) ? 0.f : mx_true;
        else m_new = !(rs_tot <= kSumLimitPre) ? fmaxf(m_ref, mx_true) : m_ref;
        alpha = first ? 1.f : __builtin_amdgcn_exp2f(m_ref - m_new);
        rs_bias = first && !(mx > -INFINITY) ? INFINITY : 0.f;
        mx = m_new - m_ref;  // what the scores in s_acc still have to lose
      } else {
        const float taken = kRefInC ? -neg_ref[0] : 0.f;   // off the scores already
        m_new = fmaxf(m_ref, mx + taken);
        mx = m_new - taken;
        alpha = m_new > -INFINITY ? __builtin_amdgcn_exp2f((m_ref - m_new) * c) : 1.f;
      }
      m_ref = m_new;
      if (t > 0 && (!kRefInC || __any(alpha != 1.f))) {   // (nothing to scale yet, or nothing that changes)
        if constexpr (kRefInC) asm volatile("" ::: "memory");
        l_run *= alpha;
#pragma unroll
        for (int i = 0; i < D / 32; ++i)
#pragma unroll
          for (int r = 0; r < 16; ++r) o_acc[i][r] *= alpha;
      }
      // a row whose keys are all masked so far keeps m_ref = -inf: use 0 so that exp2(-inf - 0) = 0
      mc = kPre ? mx : (m_new > -INFINITY ? mx * c : 0.f);
      if constexpr (kRefInC) {
        const bool in_c = __builtin_fabsf(m_new * c) <= kRefInCMost;
#pragma unroll
        for (int r = 0; r < 16; ++r) neg_ref[r] = in_c ? -m_new : 0.f;
        asm volatile("" : "+v"(neg_ref));
        any_off = __any(!in_c && m_new > -INFINITY);
        limit = __any(!(m_new > -INFINITY)) ? -1.f : kSumLimit;
      }
      if constexpr (kPre) any_off = any_off || __any(m_ref != 0.f);
      rs0 = 0.f;
      rs1 = 0.f;
#pragma unroll
      for (int kb = 0; kb < kKeyBlocks; ++kb)
#pragma unroll
        for (int r = 0; r < 16; r += 2) {
          f32x2 p;
          p.x = __builtin_amdgcn_exp2f(__builtin_fmaf(s_acc[kb][r], c, -mc));
          p.y = __builtin_amdgcn_exp2f(__builtin_fmaf(s_acc[kb][r + 1], c, -mc));
          rs0 += p.x;
          rs1 += p.y;
          const ex2 pb = __builtin_convertvector(p, ex2);
          p_frag[kb][r >> 3][r & 7] = pb.x;
          p_frag[kb][r >> 3][(r & 7) + 1] = pb.y;
        }
    }
    l_run += rs0 + rs1;
    ring_prefill(u_tag);
    phase_barrier_after_vector<kVectorInFlight * T::kLoads>(p_frag);

    // ======== matrix phase: O^T += V^T P^T (tile t), S^T = K Q^T (tile t+1) ========
    __builtin_amdgcn_s_setprio(0);
    matrix_phase(u_tag);
    if constexpr (kLoadAfterMatrix) load_tile((kU + DT_SCHED_CALL_AHEAD + group) & (kNumBuf - 1));
    // the tile after the last one of this workgroup's range has no keys for it (its scores are
    // computed on whatever the buffer holds and never used; it may belong to the next part of a
    // split item)
    cp_valid = t + 1 < n_tiles ? cp_left : 0;
    cp_left -= kBK;
    if (cp_left <= 0) cp_next_chunk();
    if (__builtin_expect(t + 1 >= n_tiles, 0)) return false;
    phase_barrier_after_matrix(s_acc, o_acc);
    return true;
  };
  // Iterations come in fours (one per LDS buffer, so that buffer offsets are immediates); the last
  // round stops after the last tile.
  for (int t = 0; t < n_tiles; t += 4)
    if (!iteration(t, U0{}) || !iteration(t + 1, U1{}) || !iteration(t + 2, U2{}) || !iteration(t + 3, U3{})) break;
  // The trailing group waits for the end of the leading group's last matrix phase; its own is the last thing that
  // happens to the tile buffers, nobody waits for it.  (Without a tile the trailing group is one barrier ahead.)
  if (group == 0) phase_barrier_after_matrix(s_acc, o_acc);
  // tile loads issued for tiles past the end are still on their way (they store zeros): let them land before the
  // workgroup ends and its LDS becomes another's
  wait_tile_loads<0>();

  if constexpr (kSplitKeys) {
    // The trailing group's accumulators, as they lie in the registers, through the tile buffers (everybody is past its
    // last read of them and its last load behind the first barrier); reference and sum through its staging rows.
    phase_barrier();
    const int pair = wave & 3;
    uint8_t* slot = lds + pair * (32 * D * 4) + lane * 16;
    float* ml = reinterpret_cast<float*>(lds + T::kLdsTiles + (pair + 4) * T::kStageBytes) + lane;
    if (group == 1) {
#pragma unroll
      for (int i = 0; i < D / 32; ++i)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          f32x4 x;
#pragma unroll
          for (int e = 0; e < 4; ++e) x[e] = o_acc[i][4 * g + e];
          *reinterpret_cast<f32x4*>(slot + (4 * i + g) * 1024) = x;
        }
      ml[0] = m_ref;
      ml[64] = l_run;
    }
    phase_barrier();
    if (group == 1) return;
    const float m_other = ml[0], m_new = fmaxf(m_ref, m_other);
    // (neither half has seen a key: both sums are 0 and stay so)
    const float mine = m_new > -INFINITY ? __builtin_amdgcn_exp2f((m_ref - m_new) * c) : 0.f;
    const float theirs = m_new > -INFINITY ? __builtin_amdgcn_exp2f((m_other - m_new) * c) : 0.f;
    l_run = l_run * mine + ml[64] * theirs;
    m_ref = m_new;
#pragma unroll
    for (int i = 0; i < D / 32; ++i)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4 x = *reinterpret_cast<const f32x4*>(slot + (4 * i + g) * 1024);
#pragma unroll
        for (int e = 0; e < 4; ++e) o_acc[i][4 * g + e] = o_acc[i][4 * g + e] * mine + x[e] * theirs;
      }
  }

  // ---- epilogue -------------------------------------------------------------------------
  const float l_tot = l_run + __shfl_xor(l_run, 32);
  float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
  float lse = l_tot > 0.f ? (m_ref * c + __builtin_amdgcn_logf(l_tot)) * 0.6931471805599453f : -INFINITY;
  const int qrow = q0 + col;
  KernArgs& e = args();
  if (is_part) {
    // A part's state goes to the workspace as it lies in the registers, in fp32: whole kilobytes per store, no rounding.
    const int ways = e.part_ways;
    const int64_t item = (int64_t)unit * kXcds + xcd, slot = item * ways + part;
    float* dst_lse = e.ws_lse + slot * kBQ + wave * 32 + col;
    const uint32_t slice_bytes = 32 * D * 4;
    float* dst = e.ws_out + (slot * kWaves + wave) * (32 * D);
    // (a NaN among the scores leaves no sum: the fold has to see that, an lse of -inf would be an empty part)
    const float part_lse = l_tot == l_tot ? lse : l_tot;
    if (hh == 0) {
      if constexpr (kMerge) store_device(dst_lse, part_lse);
      else *dst_lse = part_lse;
    }
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        f32x4 val;
#pragma unroll
        for (int e = 0; e < 4; ++e) val[e] = o_acc[db][4 * g + e] * inv;
        if constexpr (kMerge)
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, val), buffer_of(dst, slice_bytes),
                                                 (4 * db + g) * 1024 + lane * 16, 0, kDevice);
        else *reinterpret_cast<f32x4*>(dst + (4 * db + g) * 256 + lane * 4) = val;
      }
    if constexpr (!kMerge) {
      return;
    } else {
      // The wavefront that completes the last part of these 32 rows folds them all; the rest is as if it had computed the
      // whole item.
      if (!arrive_last(e.arrive + item * kWaves + wave, ways)) return;
      const int64_t slot0 = item * ways;
      const float* lses = e.ws_lse + slot0 * kBQ + wave * 32 + col;
      const float* parts = e.ws_out + (slot0 * kWaves + wave) * (32 * D);
      // Two parts are under way while one is added (behind the last one, empty descriptors: no memory is touched).  At the sizes that
      // fold themselves -- long launches, and short ones in two parts -- it decides little (us per call, one after the other -> this: D =
      // 128 24 heads x 8903 queries, 4 of 8 chunks, 8 parts 3050 -> 3043; D = 64 12 x 7844, 10 of 16, 16 parts 3433 -> 3442).
      f32x4 x[2][D / 8];
      float l[2];
      auto load = [&](int p, int buf) __attribute__((always_inline)) {
        const int at = min(p, ways - 1);
        const Rsrc src = buffer_of(parts + (int64_t)at * (kBQ * D), p < ways ? slice_bytes : 0u);
        l[buf] = load_device(lses + at * kBQ);
#pragma unroll
        for (int g = 0; g < D / 8; ++g)
          x[buf][g] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(src, g * 1024 + lane * 16, 0, kDevice));
      };
      load(0, 0);
      load(1, 1);
      float m = -INFINITY, den = 0.f;
      for (int p = 0; p < ways; p += 8) {
        float some[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) some[j] = load_device(lses + min(p + j, ways - 1) * kBQ);
#pragma unroll
        for (int j = 0; j < 8; ++j) m = fmaxf(m, some[j]);
      }
#pragma unroll
      for (int i = 0; i < D / 32; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) o_acc[i][r] = 0.f;
      for (int p0 = 0; p0 < ways; p0 += 2) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const float w = p0 + j >= ways || l[j] == -INFINITY ? 0.f : __expf(l[j] - m);   // (NaN stays NaN, and with it the row's sum)
          den += w;
#pragma unroll
          for (int g = 0; g < D / 8; ++g)
#pragma unroll
            for (int k = 0; k < 4; ++k) o_acc[g / 4][4 * (g % 4) + k] = __builtin_fmaf(w, x[j][g][k], o_acc[g / 4][4 * (g % 4) + k]);
          load(p0 + j + 2, j);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      inv = den > 0.f ? 1.f / den : 0.f;
      lse = den > 0.f ? m + __logf(den) : -INFINITY;
    }
  }
  if (hh == 0 && qrow < q_end) {
    float* dst = view.lse + ((int64_t)b * e.H + h) * e.Sq + qrow;
    if constexpr (kMerge) store_device(dst, lse);
    else *dst = lse;
  }

  // O^T (registers, [d][query]) -> LDS [query][d] in the element type -> coalesced 16-byte stores, half of the columns at
  // a time through this wavefront's own staging rows.  No barrier: the staging rows are nobody else's and no part of the
  // tile buffers, so the leading group writes its output while the trailing group is still in its last matrix phase.
  uint8_t* stage = lds + T::kLdsTiles + wave * T::kStageBytes;
  constexpr int kHalfChunks = D / 16;                 // 16-byte chunks in half a row
  constexpr int kRowsPerPass = 64 / kHalfChunks;
  const int rr = lane / kHalfChunks, cc = lane % kHalfChunks;
  // (a lane's rows by steps from its first: with a product of 64 bits for each row the epilogue took 2.1 us, 1.4 without)
  uint16_t* const out0 = view.out + (((int64_t)b * e.Sq + q0) * e.H + h) * D;
  const uint32_t row_elems = (uint32_t)e.H * D;
  uint16_t* const out_lane = out0 + (int64_t)rr * row_elems + cc * 8;
  const int64_t out_step = (int64_t)kRowsPerPass * row_elems;
#pragma unroll
  for (int half = 0; half < 2; ++half) {
#pragma unroll
    for (int i = 0; i < D / 64; ++i)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x16& o = o_acc[half * (D / 64) + i];
        f32x2 lo, hi;
        lo.x = o[4 * g + 0] * inv;
        lo.y = o[4 * g + 1] * inv;
        hi.x = o[4 * g + 2] * inv;
        hi.y = o[4 * g + 3] * inv;
        const ex2 l2 = __builtin_convertvector(lo, ex2);
        const ex2 h2 = __builtin_convertvector(hi, ex2);
        ex4 pk;
        pk.x = l2.x; pk.y = l2.y; pk.z = h2.x; pk.w = h2.y;
        *reinterpret_cast<ex4*>(stage + col * D + (((4 * i + g) ^ T::swz_o(col)) << 4) + 8 * hh) = pk;
      }
#pragma unroll
    for (int p = 0; p < 32 / kRowsPerPass; ++p) {
      const int row = p * kRowsPerPass + rr;
      const u32x4 val = *reinterpret_cast<const u32x4*>(stage + row * D + ((cc ^ T::swz_o(row)) << 4));
      if (q0 + row < q_end) {
        if constexpr (kMerge)
          __builtin_amdgcn_raw_buffer_store_b128(val, buffer_of(out0, 64u * row_elems),
                                                 (uint32_t)rr * row_elems * 2u + half * D + cc * 16 + (uint32_t)(2 * p * kRowsPerPass) * row_elems, 0, kDeviceNt);
        else __builtin_nontemporal_store(val, reinterpret_cast<u32x4*>(out_lane + p * out_step + half * (D / 2)));
      }
    }
  }
  slice = ((row0 & (kBQ - 1)) >> 5) + (kSplitKeys ? wave & 3 : wave);
}

// The work item (batch, head, query tile) of this workgroup, from its place in the grid alone.
__device__ __forceinline__ int item_of_block(KernArgs& a) {
  uint32_t x = blockIdx.x, y = blockIdx.y;
  asm volatile("" : "+s"(x), "+s"(y));   // (worked out where it is needed, not kept from the start of the kernel)
  int idx = x >> 3;
  if ((int)y >= a.job_planes) {
    const int unit = (((int)y - a.job_planes) * (int)(gridDim.x >> 3) + idx) / a.part_ways;
    idx = (a.tail_start + unit) % a.per_xcd;
  }
  return (int)(x & (kXcds - 1)) * a.per_xcd + idx;
}

// kMerge: a launch that merges (see AttnArgs::arrive).
template <int D, bool kPre, bool kHalf, bool kMerge>
__global__ __launch_bounds__(kThreads, D == 64 ? kWavesPerSimdD64 : 2) void attn_fwd_kernel(const AttnArgs args_by_value) {
  static_assert(!(kMerge && kPre), "prescaled launches do not merge");
  static_assert(!(kPre && kHalf), "the prescaled softmax keeps probabilities up to 2^40: bf16 only");
  // The arguments are read where they arrive: in the kernarg segment (constant address space, scalar loads),
  // through its base pointer -- AttnArgs is the kernel's only parameter, so it sits at offset 0.  Going through the
  // by-value parameter instead leaves it to the optimiser to prove that its private copy of the 3.6 KB struct is
  // never needed; with the tables indexed at run time from several branches it sometimes cannot, and every lane
  // then copies the whole struct into scratch memory before it starts (seven times the run time of a short launch).
  (void)args_by_value;
  prefetch_args((uint64_t)__builtin_amdgcn_kernarg_segment_ptr());
  KernArgs& a = kernel_args();

  // ---- which (job, batch, head, query tile) ------------------------------------------
  int job = blockIdx.y;
  const int xcd = blockIdx.x & (kXcds - 1);
  int idx = blockIdx.x >> 3;
  int part = 0, unit = 0;  // which of the part_ways key-tile ranges of which split item (counted per XCD)
  bool is_part = false;    // this workgroup computes one part of a split item
  int row0 = 0;            // first query row of the tile that this workgroup computes
  bool half_rows = false;  // ... and no more than half of the tile's rows
  if (job >= a.job_planes) {
    // planes behind the jobs hold the parts of the split items, in dispatch order
    const int pi = (job - a.job_planes) * (int)(gridDim.x >> 3) + idx;
    if (pi >= a.tail_items * a.part_ways) return;
    unit = pi / a.part_ways;
    part = pi - unit * a.part_ways;
    const int flat = a.tail_start + unit;
    job = flat / a.per_xcd;
    idx = flat - job * a.per_xcd;
    if (a.row_split) {
      row0 = part * (kBQ / 2);
      half_rows = true;
    } else {
      is_part = true;
    }
  } else if ((int64_t)job * a.per_xcd + idx >= a.tail_start) {
    return;  // runs as parts
  }
  const int item = xcd * a.per_xcd + idx;
  if (idx >= a.per_xcd || item >= a.total) return;
  const int bh = item / a.nqt;
  const int qt = item - bh * a.nqt;
  const int b = bh / a.H;
  const int h = bh - b * a.H;

  JobView view;
  const bool there = view_job(a, job, view);
  if (!kMerge && !there) return;
  row0 += qt * kBQ;
  // (the grid is sized for the longest job / segment; a launch that merges has whole jobs only)
  const int rows = there ? view.q_end - view.q_begin - row0 : 0;
  if (!kMerge && rows <= 0) return;
  // what this wavefront stores; of a job that is not there, its first workgroup says that nothing will come
  int slice = part > 0 ? -1 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (!kMerge || rows > 0) {
    bool split_keys = false;
    if (!kPre && !is_part && (half_rows || rows <= kBQ / 2)) {
      int n_tiles = 0;
      for (int s = view.seg_begin; s < view.seg_end; ++s) n_tiles += (key_ref(view, s).len + kBK - 1) / kBK;
      split_keys = n_tiles >= kMinSplitTiles;
      if (!split_keys && half_rows && part > 0) return;   // part 0 does the whole tile
    }
    if (split_keys) attn_item<D, kPre, kHalf, kMerge, !kPre>(view, b, h, row0, false, 0, 0, 0, slice);
    else attn_item<D, kPre, kHalf, kMerge, false>(view, b, h, row0, is_part, part, unit, xcd, slice);
  }
  if constexpr (kMerge) {
    slice = __builtin_amdgcn_readfirstlane(slice);   // uniform by construction
    if (slice < 0) return;
    KernArgs& m = kernel_args();
    const int at = item_of_block(m);
    const int bh = at / m.nqt;
    const int first = (at - bh * m.nqt) * kBQ + 32 * slice;
    if (first >= m.Sq || !arrive_last(m.arrive + kPartCounters + (int64_t)at * kWaves + slice, m.merge_jobs)) return;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int b = bh / m.H;
    uint8_t* stage = lds + Tile<D>::kLdsTiles + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) * Tile<D>::kStageBytes;
    const int n = m.merge_n;
    if (n <= 4) merge_rows<D, kHalf, 4, true>(stage, b, bh - b * m.H, first);
    else if (n <= kMergeBatch) merge_rows<D, kHalf, kMergeBatch, true>(stage, b, bh - b * m.H, first);
    else merge_rows<D, kHalf, D == 128 ? 8 : 4, false>(stage, b, bh - b * m.H, first);
  }
}

// ---- launches of few query rows -----------------------------------------------------------------
// A launch that leaves CUs idle is a chain of waits: start, tiles one after the other at the pace of two groups that meet at
// barriers (0.7 us a tile where nothing else runs: 4 heads x 512 queries, D = 64), result, merge.  Here a workgroup has 32
// queries instead of 256, and its eight wavefronts share the KEYS: wavefront w takes the tiles w, w + 8 ..., by itself, from
// registers and LDS of its own, with no barrier; their states meet once, in fp32 through the LDS.  A chunk of 512 keys is one
// tile deep.  Four wavefronts do the same where there are more slices than CUs, or fewer tiles than wavefronts.  The keys and values
// are read by eight times as many workgroups: 110 GB/s a CU out of the L2 is what long items are bound by, and why short_rows
// ends at 32 tiles, or earlier (most_tiles).
// us per call, workgroups of 256 (128) queries -> this: D = 64 4 heads x 512 queries, 2 of 4 chunks 15.1 -> 9.2, 8 x 1024, 1 of 4 18.9 ->
// 10.9, 16 x 300, 2 of 4 17.8 -> 10.3, 16 x 64 10.4 -> 7.1; D = 128 4 x 512 17.7 -> 13.5, 4 x 128 14.7 -> 8.8, 24 x 128 15.3 -> 9.9,
// 8 x 1024 24.1 -> 18.7.
// K and V of a tile take the same 8 (16) KB of LDS in turn.  K read from memory as fragments, beside V, was 1.2 ... 4 us longer at
// the sizes above: an instruction then touches 32 lines for 32 bytes each, and what the L1 holds of them is gone before the
// next one asks for the rest of the line.
// (They name the kernel, by its wavefronts; part_ways: slices of 32 rows of a head, tail_items: slices of an XCD.)
struct AttnRows8 : AttnArgs {};
struct AttnRows4 : AttnArgs {};
constexpr int kRowsStates = 4;    // states that a short launch merges itself, at most (short_launch_merges)
// LDS: the tile of each wavefront (afterwards its share of the state), references and sums, 32 result rows.
template <int D, int W>
struct Rows32 {
  static constexpr int kOffRef = W * Tile<D>::kBytesV;                // [wavefront][reference, sum][32 queries]
  static constexpr int kOffRows = kOffRef + W * 2 * 32 * 4;
  static constexpr int kOffFlag = kOffRows + 32 * Tile<D>::kRowBytes;
  static constexpr int kLdsBytes = kOffFlag + 16;
  static constexpr int kGroups = D / 8;                               // 4-element groups of a lane's accumulators
  static_assert(kGroups * 1024 == Tile<D>::kBytesV, "a wavefront's accumulators take the place of its V tile");
};

// 32 queries of one job, batch and head: of W wavefronts, w works on the key tiles w, w + W ... on its own.
template <int D, bool kHalf, bool kMerge, int W>
__device__ __forceinline__ void attn_rows32(const JobView& view, int b, int h, int row0) {
  using T = Tile<D>;
  using R = Rows32<D, W>;
  using E = Elem<kHalf>;
  typedef typename E::x8 ex8;
  typedef typename E::x4 ex4;
  typedef typename E::x2 ex2;
  KernArgs& a = kernel_args();
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  typedef __attribute__((address_space(3))) uint8_t* lds_ptr_t;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, hh = lane >> 5;
  const int q0 = view.q_begin + row0;
  uint8_t* const v_tile = lds + wave * T::kBytesV;
  const uint32_t v_addr = (uint32_t)(uintptr_t)(lds_ptr_t)lds + wave * T::kBytesV;

  // ---- the cursor: tile `tile` of the chunk reference `seg`
  const uint32_t row_bytes = (uint32_t)a.kv_ss * 2u;
  int seg = view.seg_begin, tile = wave;
  u32x4 rk, rv;
  int keys = 0;
  bool opened = false;
  // Finds the tile; false behind the last one.
  auto seek = [&]() __attribute__((always_inline)) -> bool {
    while (seg < view.seg_end) {
      if (!opened) {
        const KeyRef r = key_ref(view, seg);
        keys = r.len;
        if (keys > 0) {
          const int64_t head_off = (int64_t)b * a.chunk[r.cid].sb + (int64_t)h * a.kv_sh + (int64_t)r.begin * a.kv_ss;
          const uint32_t valid = (uint32_t)(keys - 1) * row_bytes + (uint32_t)(D * 2);
          rk = make_rsrc(a.chunk[r.cid].k + head_off, valid);
          rv = make_rsrc(a.chunk[r.cid].v + head_off, valid);
        }
        opened = true;
      }
      const int tiles = (keys + kBK - 1) / kBK;
      if (tile < tiles) return true;
      tile -= tiles;
      ++seg;
      opened = false;
    }
    return false;
  };
  // K is read into registers, then V is loaded over it.  The swizzles are those of the other form.
  uint32_t k_row, k_chunk, kld;
  {
    const int lrow = lane / T::kChunks, pos = lane % T::kChunks, krow = key_of_row(col);
    k_row = (uint32_t)lrow * row_bytes;
    k_chunk = 16u * (uint32_t)(pos ^ T::swz_k(lrow));
    kld = krow * T::kRowBytes + 16 * (hh ^ T::swz_k(krow));
  }
  auto load_k = [&]() __attribute__((always_inline)) {
    const uint32_t off = (uint32_t)(tile * kBK) * row_bytes;
    uint32_t block = T::kRowsPerBlock * row_bytes;
    asm volatile("" : "+s"(block));   // (added where it is used: the sums would be held in registers)
#pragma unroll
    for (int i = 0; i < T::kBlocks; ++i)
      load_block_to_lds(rk, k_row + (k_chunk ^ (16 * T::swz_k(T::kRowsPerBlock * i))) + i * block, off, v_addr + i * 1024);
  };
  uint32_t v_lane;
  {
    const int lrow = lane / T::kChunks, pos = lane % T::kChunks;
    v_lane = (uint32_t)lrow * row_bytes + 16u * (uint32_t)((((pos >> 2) ^ T::swz_v(lrow)) << 2) | (pos & 3));
    static_assert(T::swz_v(T::kRowsPerBlock) == T::swz_v(0), "the swizzle of a block's rows is that of the first block's");
  }
  auto load_v = [&]() __attribute__((always_inline)) {
    const uint32_t off = (uint32_t)(tile * kBK) * row_bytes;
    uint32_t block = T::kRowsPerBlock * row_bytes;
    asm volatile("" : "+s"(block));
#pragma unroll
    for (int i = 0; i < T::kBlocks; ++i) load_block_to_lds(rv, v_lane + i * block, off, v_addr + i * 1024);
  };

  bool more = seek();
  ex8 qf[D / 16];
  {
    const uint16_t* qp = a.q + (int64_t)b * a.q_sb + (int64_t)h * a.q_sh + (int64_t)min(q0 + col, view.q_end - 1) * a.q_ss + 8 * hh;
#pragma unroll
    for (int s = 0; s < D / 16; ++s) qf[s] = *reinterpret_cast<const ex8*>(qp + 16 * s);
  }
  f32x16 o_acc[D / 32];
#pragma unroll
  for (int i = 0; i < D / 32; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) o_acc[i][r] = 0.f;
  float m_ref = -INFINITY, l_run = 0.f;
  const float c = a.scale_log2;
  uint32_t vld[T::kSegs];
  {
    const int vrow = 8 * hh + ((lane & 15) >> 2);
#pragma unroll
    for (int g = 0; g < T::kSegs; ++g)
      vld[g] = vrow * T::kRowBytes + 64 * (g ^ T::swz_v(vrow)) + (16 * ((lane >> 4) & 1) + 4 * (lane & 3)) * 2;
  }
  if (more) load_k();
  while (more) {
    ex8 kf[2][D / 16];
    wait_tile_loads<0>();
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int s = 0; s < D / 16; ++s) kf[kb][s] = *reinterpret_cast<const ex8*>(v_tile + (kld ^ (32 * s)) + kb * 32 * T::kRowBytes);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // nothing is read from the tile any more
    load_v();
    const int lim = keys - tile * kBK;
    f32x16 s_acc[2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
      for (int r = 0; r < 16; ++r) s_acc[kb][r] = 0.f;
#pragma unroll
      for (int s = 0; s < D / 16; ++s) s_acc[kb] = E::mfma(kf[kb][s], qf[s], s_acc[kb]);
    }
    tile += W;
    more = seek();
    if (lim < kBK) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (32 * kb + 16 * (r >> 3) + 8 * hh + (r & 7) >= lim) s_acc[kb][r] = -INFINITY;
    }
    float mx = s_acc[0][0];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s_acc[kb][r]);
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    // (the reference in log2 units, rounded once: what the probabilities lose and what the states are weighted by is then the same number)
    const float m_new = fmaxf(m_ref, mx * c);
    const float alpha = m_new > -INFINITY ? __builtin_amdgcn_exp2f(m_ref - m_new) : 1.f;
    m_ref = m_new;
    l_run *= alpha;
#pragma unroll
    for (int i = 0; i < D / 32; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) o_acc[i][r] *= alpha;
    const float mc = m_new > -INFINITY ? m_new : 0.f;
    float rs0 = 0.f, rs1 = 0.f;
    ex8 p_frag[2][2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int r = 0; r < 16; r += 2) {
        f32x2 p;
        p.x = __builtin_amdgcn_exp2f(__builtin_fmaf(s_acc[kb][r], c, -mc));
        p.y = __builtin_amdgcn_exp2f(__builtin_fmaf(s_acc[kb][r + 1], c, -mc));
        rs0 += p.x;
        rs1 += p.y;
        const ex2 pb = __builtin_convertvector(p, ex2);
        p_frag[kb][r >> 3][r & 7] = pb.x;
        p_frag[kb][r >> 3][(r & 7) + 1] = pb.y;
      }
    l_run += rs0 + rs1;
    wait_tile_loads<0>();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        if (kb + half > 0) __builtin_amdgcn_sched_barrier(0x40f);   // no more than the operands of a step at a time
#pragma unroll
        for (int db = 0; db < D / 32; ++db) {
          const uint8_t* p = v_tile + vld[db] + (32 * kb + 16 * half) * T::kRowBytes;
          const s16x4 lo = lds_read_tr(p);
          const s16x4 hi = lds_read_tr(p + 4 * T::kRowBytes);
          const s16x8 both = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
          o_acc[db] = E::mfma(__builtin_bit_cast(ex8, both), p_frag[kb][half], o_acc[db]);
        }
      }
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // nothing is read from the tile any more
    if (more) load_k();
  }

  // ---- the states meet in the LDS: every wavefront adds up its share of the columns
  float* const refs = reinterpret_cast<float*>(lds + R::kOffRef);
  l_run += __shfl_xor(l_run, 32);
  if (hh == 0) {
    refs[wave * 64 + col] = m_ref;
    refs[wave * 64 + 32 + col] = l_run;
  }
#pragma unroll
  for (int i = 0; i < D / 32; ++i)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<f32x4*>(v_tile + (4 * i + g) * 1024 + lane * 16) =
          f32x4{o_acc[i][4 * g], o_acc[i][4 * g + 1], o_acc[i][4 * g + 2], o_acc[i][4 * g + 3]};
  phase_barrier();
  float w[W], l_tot = 0.f, m = -INFINITY;
#pragma unroll
  for (int j = 0; j < W; ++j) {
    w[j] = refs[j * 64 + col];
    m = fmaxf(m, w[j]);
  }
#pragma unroll
  for (int j = 0; j < W; ++j) {
    w[j] = m > -INFINITY ? __builtin_amdgcn_exp2f(w[j] - m) : 0.f;
    l_tot = __builtin_fmaf(refs[j * 64 + 32 + col], w[j], l_tot);
  }
  const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
  uint8_t* const rows = lds + R::kOffRows;
#pragma unroll
  for (int k = 0; k < R::kGroups / W; ++k) {
    const int g = wave * (R::kGroups / W) + k;
    f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < W; ++j) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(lds + j * T::kBytesV + g * 1024 + lane * 16);
#pragma unroll
      for (int e = 0; e < 4; ++e) sum[e] = __builtin_fmaf(x[e], w[j], sum[e]);
    }
    f32x2 lo, hi;
    lo.x = sum[0] * inv; lo.y = sum[1] * inv;
    hi.x = sum[2] * inv; hi.y = sum[3] * inv;
    const ex2 l2 = __builtin_convertvector(lo, ex2);
    const ex2 h2 = __builtin_convertvector(hi, ex2);
    ex4 pk;
    pk.x = l2.x; pk.y = l2.y; pk.z = h2.x; pk.w = h2.y;
    *reinterpret_cast<ex4*>(rows + col * T::kRowBytes + ((g ^ T::swz_k(col)) << 4) + 8 * hh) = pk;
  }
  if (wave == 0 && hh == 0 && q0 + col < view.q_end) {
    // log(2^m * sum), the sum by its exponent and mantissa: what the logarithm's last bits are worth does not grow with the number of keys
    constexpr float kLn2 = 0.6931471805599453f;
    const float fraction = __builtin_amdgcn_logf(__builtin_amdgcn_frexp_mantf(l_tot)) * kLn2;
    const float log_sum = __builtin_fmaf((float)__builtin_amdgcn_frexp_expf(l_tot), kLn2, __builtin_fmaf(m, kLn2, fraction));
    const float lse = l_tot > 0.f ? log_sum : -INFINITY;
    float* dst = view.lse + ((int64_t)b * a.H + h) * a.Sq + q0 + col;
    if constexpr (kMerge) store_device(dst, lse);
    else *dst = lse;
  }
  phase_barrier();
  constexpr int kRowsPerPass = 64 * W / T::kChunks;
  uint16_t* const out0 = view.out + (((int64_t)b * a.Sq + q0) * a.H + h) * D;
  const uint32_t row_elems = (uint32_t)a.H * D;
#pragma unroll
  for (int pass = 0; pass < 32; pass += kRowsPerPass) {
    const int row = pass + tid / T::kChunks, cc = tid % T::kChunks;
    if (row >= 32 || q0 + row >= view.q_end) break;
    const u32x4 val = *reinterpret_cast<const u32x4*>(rows + row * T::kRowBytes + ((cc ^ T::swz_k(row)) << 4));
    if constexpr (kMerge)
      __builtin_amdgcn_raw_buffer_store_b128(val, buffer_of(out0, 64u * row_elems), 2u * row * row_elems + 16u * cc, 0, kDeviceNt);
    else __builtin_nontemporal_store(val, reinterpret_cast<u32x4*>(out0 + (int64_t)row * row_elems + 8 * cc));
  }
}

// A launch of few query rows (see short_rows): a workgroup of W wavefronts for every 32 rows of a job.
template <int D, bool kHalf, bool kMerge, int W>
__device__ __forceinline__ void attn_rows32_kernel() {
  using R = Rows32<D, W>;
  prefetch_args((uint64_t)__builtin_amdgcn_kernarg_segment_ptr());
  KernArgs& a = kernel_args();
  // the slices of 32 rows of all (batch, head): part_ways a head, tail_items an XCD
  const int at = (int)(blockIdx.x & (kXcds - 1)) * a.tail_items + (int)(blockIdx.x >> 3);
  const int bh = at / a.part_ways;
  const int slice = at - bh * a.part_ways;
  const int b = bh / a.H;
  const int h = bh - b * a.H;
  if (b >= a.B) return;
  const int row0 = 32 * slice;
  JobView view;
  const bool there = view_job(a, blockIdx.y, view);
  const int rows = there ? view.q_end - view.q_begin - row0 : 0;
  if (rows > 0) attn_rows32<D, kHalf, kMerge, W>(view, b, h, row0);
  if constexpr (kMerge) {
    KernArgs& m = kernel_args();
    if (row0 >= m.Sq) return;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int* const flag = reinterpret_cast<int*>(lds + R::kOffFlag);
    wait_tile_loads<0>();   // this wavefront's stores
    phase_barrier();        // everybody's
    if (wave == 0) {
      const bool last = arrive_last(m.arrive + kPartCounters + (int64_t)bh * m.nqt * kWaves + slice, m.merge_jobs);
      if ((threadIdx.x & 63) == 0) *flag = last;
    }
    phase_barrier();
    if (!__builtin_amdgcn_readfirstlane(*flag)) return;
    constexpr int kOfLoad = 64 / Tile<D>::kChunks, kMine = kOfLoad * W < 32 ? 32 / W : kOfLoad;   // rows of a wavefront
    const int first = row0 + kMine * wave;
    if (kMine * wave >= 32 || first >= m.Sq) return;
    uint8_t* const stage = lds + wave * Tile<D>::kBytesV;
    merge_rows<D, kHalf, kRowsStates, true, kMine>(stage, b, h, first);
  }
}
template <int D, bool kPre, bool kHalf, bool kMerge>
__global__ __launch_bounds__(512, D == 64 ? 4 : 2) void attn_fwd_kernel(const AttnRows8 args_by_value) {
  (void)args_by_value;
  attn_rows32_kernel<D, kHalf, kMerge, 8>();
}
template <int D, bool kPre, bool kHalf, bool kMerge>
__global__ __launch_bounds__(256, D == 64 ? 4 : 2) void attn_fwd_kernel(const AttnRows4 args_by_value) {
  (void)args_by_value;
  attn_rows32_kernel<D, kHalf, kMerge, 4>();
}

// Folds the part_ways partial states of every split item into the item's rows of its destination.  A workgroup takes 64
// columns of the 32 query rows of one wavefront of the item's workgroup: its four wavefronts share the 4-element groups
// of a row, lane L of a group holds query L % 32 as in the attention kernel, and the rows go through the LDS so that
// the stores are 128 contiguous bytes.  Latency-bound (a few hundred KB per CU): many small workgroups with the loads of
// four parts in flight.
constexpr int kFoldThreads = 256;
template <int D, bool kHalf>
__global__ __launch_bounds__(kFoldThreads) void attn_tail_fold_kernel(const AttnArgs args_by_value) {
  typedef const AttnArgs __attribute__((address_space(4))) KernArgs;
  KernArgs& a = *(KernArgs*)__builtin_amdgcn_kernarg_segment_ptr();
  (void)args_by_value;
  prefetch_args((uint64_t)__builtin_amdgcn_kernarg_segment_ptr());
  typedef typename Elem<kHalf>::x2 ex2;
  typedef typename Elem<kHalf>::x4 ex4;
  constexpr int kHalves = D / 64;
  constexpr int kMine = 8 / (kFoldThreads / 64);       // 4-element groups of a lane
  constexpr int kPitch = 64 * 2 + 16;
  constexpr int kInFlight = 4;
  __shared__ __attribute__((aligned(16))) uint8_t rows[32 * kPitch];
  const int xcd = blockIdx.x & (kXcds - 1);   // the XCD the parts ran on: what is left of them in its L2 is read from there
  const int half = (blockIdx.x >> 3) % kHalves;
  const int rest = (blockIdx.x >> 3) / kHalves;
  const int slice = rest & (kWaves - 1);
  const int unit = rest >> 3;
  const int flat = a.tail_start + unit;
  const int job = flat / a.per_xcd;
  const int item = xcd * a.per_xcd + flat - job * a.per_xcd;
  if (item >= a.total) return;
  const int bh = item / a.nqt;
  const int qt = item - bh * a.nqt;
  const int b = bh / a.H;
  const int h = bh - b * a.H;
  JobView view;
  if (!view_job(a, job, view)) return;
  const int q0 = view.q_begin + qt * kBQ + slice * 32;
  if (q0 >= view.q_end) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = lane & 31, hh = lane >> 5;
  const int ways = a.part_ways;
  const int64_t slot0 = ((int64_t)unit * kXcds + xcd) * ways;
  const float* lses = a.ws_lse + slot0 * kBQ + slice * 32 + col;
  const float* parts = a.ws_out + (slot0 * kWaves + slice) * (32 * D) + (8 * half + wave * kMine) * 256 + lane * 4;
  float m = -INFINITY, den = 0.f;
  f32x4 acc[kMine];
#pragma unroll
  for (int g = 0; g < kMine; ++g) acc[g] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int p0 = 0; p0 < ways; p0 += kInFlight) {
    float l[kInFlight];
    f32x4 x[kInFlight][kMine];
#pragma unroll
    for (int i = 0; i < kInFlight; ++i) {
      const int p = min(p0 + i, ways - 1);
      l[i] = lses[p * kBQ];
#pragma unroll
      for (int g = 0; g < kMine; ++g) x[i][g] = *reinterpret_cast<const f32x4*>(parts + (int64_t)p * (kBQ * D) + g * 256);
    }
    float m_new = m;
#pragma unroll
    for (int i = 0; i < kInFlight; ++i) {
      // Behind the last part the loads repeat it, and nothing of that may be left: 0 times an infinity would be NaN.  (Masked,
      // not assigned in a branch: the compiler would move the loads into it, and they would no longer be in flight together.)
      const bool there = p0 + i < ways;
      const uint32_t mask = there ? 0xffffffffu : 0u;
      if (!there) l[i] = -INFINITY;
#pragma unroll
      for (int g = 0; g < kMine; ++g) {
        u32x4 bits = __builtin_bit_cast(u32x4, x[i][g]);
        bits &= mask;
        x[i][g] = __builtin_bit_cast(f32x4, bits);
      }
      m_new = fmaxf(m_new, l[i]);
    }
    const float alpha = m > -INFINITY ? __expf(m - m_new) : 0.f;
    m = m_new;
    den *= alpha;
#pragma unroll
    for (int g = 0; g < kMine; ++g)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[g][e] *= alpha;
#pragma unroll
    for (int i = 0; i < kInFlight; ++i) {
      const float w = l[i] == -INFINITY ? 0.f : __expf(l[i] - m);   // (NaN stays NaN, and with it the row's sum)
      den += w;
#pragma unroll
      for (int g = 0; g < kMine; ++g)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[g][e] = __builtin_fmaf(w, x[i][g][e], acc[g][e]);
    }
  }
  const float inv = den > 0.f ? 1.f / den : 0.f;
#pragma unroll
  for (int g = 0; g < kMine; ++g) {
    f32x2 lo, hi;
    lo.x = acc[g][0] * inv; lo.y = acc[g][1] * inv;
    hi.x = acc[g][2] * inv; hi.y = acc[g][3] * inv;
    const ex2 l2 = __builtin_convertvector(lo, ex2);
    const ex2 h2 = __builtin_convertvector(hi, ex2);
    ex4 pk;
    pk.x = l2.x; pk.y = l2.y; pk.z = h2.x; pk.w = h2.y;
    *reinterpret_cast<ex4*>(rows + col * kPitch + (8 * (wave * kMine + g) + 4 * hh) * 2) = pk;
  }
  if (half == 0 && wave == 0 && hh == 0 && q0 + col < view.q_end)
    view.lse[((int64_t)b * a.H + h) * a.Sq + q0 + col] = den > 0.f ? m + __logf(den) : -INFINITY;
  __syncthreads();
  const int row = threadIdx.x >> 3, cc = threadIdx.x & 7;
  if (q0 + row < view.q_end)
    __builtin_nontemporal_store(*reinterpret_cast<const u32x4*>(rows + row * kPitch + cc * 16),
                                reinterpret_cast<u32x4*>(view.out + (((int64_t)b * a.Sq + q0 + row) * a.H + h) * D + 64 * half + cc * 8));
}

static_assert(Tile<128>::kLdsBytes == kAttnLdsBytes128 && Tile<64>::kLdsBytes == kAttnLdsBytes64,
              "dt_common.h states the LDS footprint of the attention kernel");

// Args: AttnArgs, or what names another form of the kernel.
template <int D, bool kPre, bool kHalf, bool kMerge, typename Args>
static int launch_one(const Args& a, dim3 grid, hipStream_t stream) {
  constexpr int kLdsBytes = std::is_same_v<Args, AttnRows8> ? Rows32<D, 8>::kLdsBytes
                            : std::is_same_v<Args, AttnRows4> ? Rows32<D, 4>::kLdsBytes : Tile<D>::kLdsBytes;
  constexpr int kThreadsOf = std::is_same_v<Args, AttnRows4> ? 256 : kThreads;
  void (*const kernel)(const Args) = attn_fwd_kernel<D, kPre, kHalf, kMerge>;
  // more than 64 KB of dynamic LDS has to be allowed once per kernel and device
  static thread_local int allowed_dev = -1;
  int dev = 0;
  if (int rc = hip_fail(hipGetDevice(&dev), "hipGetDevice")) return rc;
  if (allowed_dev != dev) {
    if (int rc = hip_fail(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes),
                          "hipFuncSetAttribute"))
      return rc;
    allowed_dev = dev;
  }
  hipLaunchKernelGGL(kernel, grid, dim3(kThreadsOf), kLdsBytes, stream, a);
  return hip_fail(hipGetLastError(), "attn_fwd launch");
}

template <typename Args>
static int launch_dim(const Args& a, int D, dim3 grid, hipStream_t stream) {
  if (a.arrive) {
    // (eight wavefronts are for more than 4 key tiles, and at D = 128 a launch of so few rows merges up to 4: this cannot fire; it guards later
    // edits to either rule)
    constexpr bool kBuilt128 = !std::is_same_v<Args, AttnRows8>;
    if (D == 128 && !kBuilt128) {
      set_error("internal: no merging launch of eight wavefronts a workgroup is built for head dim 128");
      return DT_ERR_INVALID;
    }
    if constexpr (kBuilt128)
      if (D == 128) return a.elem_f16 ? launch_one<128, false, true, true>(a, grid, stream) : launch_one<128, false, false, true>(a, grid, stream);
    return a.elem_f16 ? launch_one<64, false, true, true>(a, grid, stream) : launch_one<64, false, false, true>(a, grid, stream);
  }
  if (a.elem_f16) return D == 128 ? launch_one<128, false, true, false>(a, grid, stream) : launch_one<64, false, true, false>(a, grid, stream);
  if constexpr (std::is_same_v<Args, AttnArgs>)
    if (a.q_prescaled) return D == 128 ? launch_one<128, true, false, false>(a, grid, stream) : launch_one<64, true, false, false>(a, grid, stream);
  return D == 128 ? launch_one<128, false, false, false>(a, grid, stream) : launch_one<64, false, false, false>(a, grid, stream);
}

// Number of CUs of the current device (one workgroup of the attention kernel per CU at a time).
static int cu_count() {
  static thread_local int cached_dev = -1, cached = 0;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 0;
  if (dev != cached_dev) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    cached = n;
    cached_dev = dev;
  }
  return cached;
}

// Scratch of the allocation-free entry point: the tail-balancing workspace as a device array that
// lives as long as the code object (one copy per GPU, at that GPU's own address).  Host code never
// uses the array's name as an address: static_tail_scratch() asks the runtime for the device
// address once per device and hands that out.
static __device__ __align__(256) uint8_t g_tail_scratch[kStaticTailBytes];

int static_tail_scratch(void** ptr, int64_t* bytes) {
  constexpr int kMaxDevices = 64;
  static std::mutex mu;
  static void* addr[kMaxDevices] = {};
  int dev = 0;
  if (int rc = hip_fail(hipGetDevice(&dev), "hipGetDevice")) return rc;
  if (dev < 0 || dev >= kMaxDevices) {
    set_error("device ordinal %d outside the %d the static scratch table covers", dev, kMaxDevices);
    return DT_ERR_UNSUPPORTED;
  }
  std::lock_guard<std::mutex> lock(mu);
  if (addr[dev] == nullptr) {
    void* p = nullptr;
    if (int rc = hip_fail(hipGetSymbolAddress(&p, HIP_SYMBOL(g_tail_scratch)), "hipGetSymbolAddress(tail scratch)"))
      return rc;
    if (p == nullptr || (reinterpret_cast<uintptr_t>(p) & 255) != 0) {
      set_error("the runtime returned an unusable address for the static tail scratch");
      return DT_ERR_HIP;
    }
    addr[dev] = p;
  }
  *ptr = addr[dev];
  *bytes = kStaticTailBytes;
  return DT_OK;
}

// What the planner knows about a launch job: key tiles of one of its work items, query rows.
struct JobSize {
  int32_t tiles, rows;
};

// The order of host-listed jobs by falling length, those with few query rows first (they are gone in no time).  False where
// the jobs already come like that.
static bool longest_first(const JobSize* size, int n_jobs, int* order) {
  for (int j = 0; j < n_jobs; ++j) order[j] = j;
  auto before = [&](int x, int y) {
    return size[x].rows != size[y].rows ? size[x].rows < size[y].rows : size[x].tiles > size[y].tiles;
  };
  bool sorted = true;
  for (int j = 1; j < n_jobs; ++j) sorted = sorted && !before(j, j - 1);
  if (!sorted) std::stable_sort(order, order + n_jobs, before);
  return !sorted;
}

static void reorder_jobs(AttnArgs& a, int n_jobs, const int* order) {
  const AttnArgs o = a;
  int e = 0;
  for (int j = 0; j < n_jobs; ++j) {
    const int from = order[j];
    a.job[j] = o.job[from];
    a.job[j].begin = e;
    for (int x = o.job[from].begin; x < o.job[from].end; ++x, ++e) a.entry[e] = o.entry[x];
    a.job[j].end = e;
  }
}

// Sizes of the launch's jobs.  Device-listed jobs count as the longest chunk.  Where the boundaries are in device memory
// a job counts with its whole chunks, and the query rows are taken to belong to the first segment (max_seqlen_q of them;
// the model passes the valid tokens and, behind them, one padding segment).
static void job_sizes(const AttnArgs& a, int n_jobs, JobSize* size) {
  auto tiles_of = [](int keys) { return (keys + kBK - 1) / kBK; };
  const int rows_first = std::min(a.nqt * kBQ, a.Sq), rows_other = std::max(0, std::min(rows_first, a.Sq - rows_first));
  int longest = 0;
  for (int c = 0; c < a.n_chunks; ++c) longest = std::max(longest, tiles_of(a.chunk[c].len));
  for (int j = 0; j < n_jobs; ++j) {
    const bool listed = a.dev_ids == nullptr;
    int seg = listed ? a.job[j].q_begin : a.n_seg > 0 ? a.n_seg - 1 - j / a.n_slots : -1;
    size[j].tiles = 0;
    if (!listed) size[j].tiles = longest;
    else
      for (int e = a.job[j].begin; e < a.job[j].end; ++e)
        size[j].tiles += tiles_of(a.cu_q ? a.chunk[a.entry[e].chunk].len : a.entry[e].kv_len);
    if (a.cu_q) size[j].rows = seg == 0 ? rows_first : rows_other;
    else if (listed) size[j].rows = a.job[j].q_len;
    else size[j].rows = seg >= 0 ? a.seg_q_len[seg] : a.Sq;
  }
}

// Which work items at the end of the launch run as how many parts each.
struct TailPlan {
  int32_t items = 0, ways = 0;   // per XCD; parts of an item
  bool rows = false;             // the parts are halves of the rows
};

// Time is counted in key tiles, on one XCD (workgroups go to the XCDs in turn, so each works through its own share of
// every job).  Jobs by falling length: the short ones behind fill the gaps that the long ones leave, so the
// launch ends as if it consisted of items of the last job's length T only, in ceil(units / cus) rounds of them.  Or
// (`by_count`) the items are counted as they are, whatever their lengths: launch_time says which of the two is right.  The
// items of the last, partly filled round are cut into w parts each, which are handed to CUs as they come free: they take
// ceil(rem * w / cus) rounds of (T / w + overhead) instead of one of T, plus the fold kernel.  A launch of less than one
// round is split as a whole.
// Measured on the HunyuanVideo, Step-Video and CogVideoX shares: a part costs about 6 tiles on top of its own (start-up,
// epilogue, partial state) when all parts run at once and about 10 when they take several rounds, so many small parts
// only pay in the first case; the fold kernel and the parts' stores cost about 4 (D = 128: 6, twice the bytes).
// The other way to end a launch early: the items of the last round as two workgroups of half the query rows each, 0.6 of
// an item's time (see attn_item) with no partial states and no fold kernel, where they fit the round side by side.  It
// wins over the cut along the keys while items are short (about 70 key tiles at half a round) and needs no 16 tiles: us
// per layer call, cut along the keys or not at all -> along the rows: 24 heads x 1000 queries x 4 chunks, D = 64 44.0 ->
// 39.3; 30 heads x 1100 x 2, D = 128 73.2 -> 65.2, D = 64 44.4 -> 40.4; 10 heads x 1100 x 2, D = 64 30.2 -> 23.5; two samples of
// 24 heads x 1861 x 3, D = 128 297 -> 287.  The planner counts short last query tiles as whole ones: counting them as 0.6
// moved the cut of the last round by half an item and lost 1 ... 6 % (24 heads x 3700 x 4, D = 128 583 against 607).
// Launches of less than a round that used to run unsplit (us, before -> now): 1 head x 8000 queries x 8000 keys, D = 128
// 140 -> 49; 3 heads x 2048 x 4096 77 -> 36; 10 heads x 1154 queries, two states over 1 and 2 chunks of 1154 keys 53 -> 45;
// 4 heads x 5777 queries x 4 chunks of 5777 keys (368 work items, 23 per head) 270 -> 250.
static TailPlan plan_tail(const AttnArgs& a, int D, int n_jobs, const JobSize* size, int cus, int64_t slots_cap, bool by_count) {
  TailPlan plan;
  constexpr double kPartOverheadOneRound = 6.0, kPartOverheadRounds = 10.0, kHalfItem = 0.6;
  const double fold_overhead = D == 128 ? 6.0 : 4.0;
  const int last = size[n_jobs - 1].tiles, last_rows = size[n_jobs - 1].rows;
  if (last < 1 || (int64_t)n_jobs * a.per_xcd >= INT32_MAX) return plan;
  double units = 0;
  int same = 0, longest = 0;   // jobs at the end that are like the last one
  for (int j = 0; j < n_jobs; ++j) {
    const double r = (double)size[j].tiles / last;
    const int items = a.B * a.H * ((size[j].rows + kBQ - 1) / kBQ);
    units += (double)((items + kXcds - 1) / kXcds) * (r < 0.75 ? r : std::floor(r + 0.5));
    same = size[j].rows == last_rows && r > 0.9 && r < 1.1 ? same + 1 : 0;
    longest = std::max(longest, size[j].tiles);
  }
  int rem, T;
  if (n_jobs * a.per_xcd <= cus) {   // less than one round
    rem = n_jobs * a.per_xcd;
    T = longest;
  } else {
    // (with boundaries that only the device knows the last round may be full for all the host can tell)
    rem = a.cu_q ? 0 : by_count ? n_jobs * a.per_xcd % cus : (int)std::ceil(units - 1e-9) % cus;
    T = last;
    if (rem > (by_count ? 1 : same) * a.per_xcd) return plan;
  }
  if (rem <= 0) return plan;
  double best = 0.1 * T;   // least gain worth the extra kernel
  for (int w = 2; T >= 16 && w <= 16; ++w) {
    if ((int64_t)rem * kXcds * w > slots_cap || T / w < 6) break;
    const int rounds = (rem * w + cus - 1) / cus;
    const double part = (double)T / w, overhead = rounds == 1 ? kPartOverheadOneRound : kPartOverheadRounds;
    const double gain = T - rounds * (part + overhead) - fold_overhead;
    if (gain > best) {
      best = gain;
      plan.items = rem;
      plan.ways = w;
    }
  }
  const double gain_rows = (1.0 - kHalfItem) * T - 2.0;
  if (!a.q_prescaled && 2 * rem <= cus && last_rows > kBQ / 2 && T >= kMinSplitTiles && gain_rows > (plan.items > 0 ? best : 0.0)) {
    plan.items = rem;
    plan.ways = 2;
    plan.rows = true;
  }
  return plan;
}

// What a launch with jobs of unequal length takes, in key tiles.  An XCD hands its workgroups to its four shader engines in
// turn, whether an engine has a CU free or not, so each engine works through every fourth workgroup on eight CUs: 42 items
// of 210 and 105 tiles in this order, which would fill 32 CUs evenly, leave one engine with a third item for a CU.
// (Differences between two orders and splits of a launch correlate with the measured ones at 0.87 in this model, at 0.63
// in one that gives every item to the CU that is free first; 55 launches at D = 128.)  The clock rises where CUs are idle,
// so that about 0.6 of a difference in the end times is seen: the rest of the price is the work done.
static double launch_time(const AttnArgs& a, int n_jobs, const JobSize* size, int cus, const TailPlan& plan) {
  constexpr int kEngines = 4, kMaxCus = 16;
  constexpr double kItem = 4.0, kPart = 10.0, kHalfItem = 0.6, kFold = 6.0, kEndShare = 0.6;
  const int per_engine = std::min(kMaxCus, cus / kEngines);
  double busy[kEngines][kMaxCus] = {}, work = 0, end = 0;
  int wg = 0;
  auto run = [&](double tiles) {
    double* cu = std::min_element(busy[wg % kEngines], busy[wg % kEngines] + per_engine);
    *cu += tiles;
    work += tiles;
    end = std::max(end, *cu);
    ++wg;
  };
  const int n = n_jobs * a.per_xcd, whole = n - plan.items;
  auto exists = [&](int flat) { return flat % a.per_xcd % a.nqt * kBQ < size[flat / a.per_xcd].rows; };
  for (int flat = 0; flat < n; ++flat) {
    if (flat < whole && exists(flat)) run(size[flat / a.per_xcd].tiles + kItem);
    else ++wg;
  }
  for (int flat = whole; flat < n; ++flat) {
    const double tiles = size[flat / a.per_xcd].tiles;
    for (int p = 0; p < plan.ways; ++p) {
      if (exists(flat)) run(plan.rows ? kHalfItem * tiles + kItem : tiles / plan.ways + kPart);
      else ++wg;
    }
  }
  const double fold = plan.items > 0 && !plan.rows ? kFold : 0.0;
  return kEndShare * (end + fold) + (1.0 - kEndShare) * work / (kEngines * per_engine);
}

// Order of the jobs and split of the last round (slots_cap < 0: no split).  Jobs of one length: there is one order, and the
// items are counted.  Of several, in a launch of more than one round: the order of the caller with the remainder by count, or
// the longest first with the remainder in units of the last job or by count, whatever takes least by launch_time.  Of two that
// take the same, D = 128 keeps the caller's order (the shorter job in front, whose long items then run alone at a higher clock:
// 24 heads x 3721 queries, 1 + 2 chunks 468 -> 463 us), D = 64 the longest first (30 heads x 2001 103 -> 99).
// Over 318 launches of 4 ... 48 heads x 1200 ... 14 882 queries, 2 or 3 jobs of 1 ... 7 chunks: 2.3 % less time on average than
// always the longest first in units (40 heads x 1596, D = 64, 1 + 7 chunks 309 -> 238 us; 48 x 6851, D = 128, 1 + 2 2896 -> 2826;
// most lost 3.6 %, 24 x 3641, D = 128, 1 + 2 413 -> 426) and 3.0 % less than always the caller's order by count (D = 128: never
// more; D = 64: up to 12 % more in launches of two or three rounds, where the two workgroups of a CU share it, which is not
// modelled: 12 heads x 6902, 1 + 3 593 -> 656).
static TailPlan plan_launch(AttnArgs& a, int D, int n_jobs, JobSize* size, int cus, int64_t slots_cap) {
  constexpr int kMaxItems = 2048;   // of an XCD, 64 rounds: the end of a longer launch is nothing, and pricing it takes time
  int order[DT_MAX_JOBS * DT_MAX_SEGMENTS];
  JobSize sorted[DT_MAX_JOBS * DT_MAX_SEGMENTS];
  const bool changes = a.dev_ids == nullptr && longest_first(size, n_jobs, order);
  for (int j = 0; j < n_jobs; ++j) sorted[j] = size[changes ? order[j] : j];
  const bool split = slots_cap >= 0;
  bool uneven = false;
  for (int j = 1; j < n_jobs; ++j) uneven = uneven || size[j].tiles != size[0].tiles;
  TailPlan best = split ? plan_tail(a, D, n_jobs, sorted, cus, slots_cap, false) : TailPlan();
  const int64_t items = (int64_t)n_jobs * a.per_xcd;
  bool given = false;
  if (a.dev_ids == nullptr && uneven && cus > 0 && items > cus && items <= kMaxItems) {
    double least = launch_time(a, n_jobs, sorted, cus, best);
    auto consider = [&](const JobSize* s, bool as_given) {
      const TailPlan plan = split ? plan_tail(a, D, n_jobs, s, cus, slots_cap, true) : TailPlan();
      const double time = launch_time(a, n_jobs, s, cus, plan);
      if (as_given && D == 128 ? time < 1.001 * least : time < least) {
        least = time;
        best = plan;
        given = as_given;
      }
    };
    if (split) consider(sorted, false);
    if (changes) consider(size, true);
  }
  if (changes && !given) reorder_jobs(a, n_jobs, order);
  return best;
}

std::mutex& workspace_lock(const void* workspace) {
  constexpr int kBits = 6;
  static std::mutex locks[1 << kBits];
  return locks[(reinterpret_cast<uintptr_t>(workspace) >> 4) * 0x9e3779b97f4a7c15ull >> (64 - kBits)];
}

// How a launch runs as workgroups of 32 query rows (see attn_rows32): wavefronts of one (0: it does not), slices of 32 rows of a head,
// slices of an XCD.
struct ShortRows {
  int waves = 0, slices = 0;
  int64_t per_xcd = 0;
};
// Like the other ways to split, for launches with a workspace (without one the items stay whole), though it needs none.
// The workgroups have to be resident together: of eight wavefronts one a CU at D = 128 and two at D = 64, of four twice as many.
// us per call, workgroups of 256 rows -> of 32 with eight wavefronts, with four, by workgroups and key tiles:
//   * D = 64 128 workgroups, 3 tiles 15.2 -> 8.0, 7.8; 6 17.6 -> 8.8, 9.2; 16 19.5 -> 10.9, 11.8; 32 22.7 -> 16.5, 19.0; (256, 48 tiles 24.6 -> 21.6;
//     16, 48 tiles 20.4 -> 18.7, 96 in up to 16 parts 21.7 -> 27.7);
//     512, 1 tile 13.9 -> 8.8, 7.8; 10 17.2 -> 13.6, 13.2; 32 28.5 -> 25.2, 25.2; 768, 1 tile 15.5 -> 14.6, 9.5; 10 18.6 -> 21.8, 17.1; 32 30.3 -> 31.7, 29.4;
//     1024, 6 tiles 20.6 -> 23.6, 19.8; 10 21.8 -> 27.1, 23.7; 1536, 1 tile 16.3 -> 22.8, 17.9;
//   * D = 128 128 workgroups, 3 tiles 14.4 -> 11.0, 10.8; 6 17.7 -> 12.5, 12.8; 32 24.6 -> 23.4, 27.2; (16, 32 tiles 22.4 -> 20.5; 128, 48 tiles
//     27.6 -> 29.8); 384, 1 tile 13.8 -> 15.9, 11.7; 6 19.1 -> 20.8, 17.3; 10 21.0 -> 25.0, 21.4; 512, 6 tiles 21.3 -> 23.4, 19.6; 768, 1 tile
//     15.5 -> 22.5, 18.2.
// At D = 64 with more workgroups than CUs, long jobs come back to workgroups of 256 rows.  A job's keys are then read by several workgroups
// that share CUs with others (time of 32 rows against 256, some 600 launches of 1 ... 384 heads x 8 ... 4000 queries, batch and jobs in all splits):
//   * a head's rows in one slice: 0.77 ... 1.00 up to 32 tiles, however many heads there are;
//   * in two: up to 2 workgroups a CU 0.88 ... 1.00 for 16 tiles, 0.94 ... 1.21 for 22 and more (8 x 24 heads x 48, 30 tiles 29.6 -> 36.0); up to 3 1.01 ... 1.14
//     from 14 tiles on (16 x 24 x 64, 17 tiles 30.3 -> 34.6), but 0.82 ... 0.97 where a head's keys lie within 256 bytes of each other (two heads
//     of a contiguous tensor: 192 x 2 x 33, 32 tiles 51.7 -> 42.7);
//   * in more: up to 2 workgroups a CU 0.77 ... 1.05, 0.88 on average; up to 3 0.93 ... 1.03 for 10 tiles, 0.96 ... 1.07 for 13, to 1.5 for more (4 x 48 x 109, 29 tiles
//     29.5 -> 44.1; 24 x 969, 31 tiles 24.2 -> 26.1; 1 x 48 x 254, two jobs of 32 24.6 -> 27.4).
static int most_tiles(const AttnArgs& a, int D, int slices, int64_t units, int cus) {
  if (units <= cus) return 32;
  if (D == 128) return 8;
  if (slices == 1 || (slices == 2 && a.kv_ss <= 2 * D)) return 32;
  return units > 2 * cus ? 10 : slices == 2 ? 16 : 32;
}
static ShortRows short_rows(const AttnArgs& a, int D, int n_jobs, const JobSize* size, int cus) {
  const int rows_most = std::min(a.nqt * kBQ, a.Sq);
  int rows = 0, tiles = 0;
  for (int j = 0; j < n_jobs; ++j) {
    rows = std::max(rows, a.cu_q ? rows_most : size[j].rows);
    tiles = std::max(tiles, size[j].tiles);
  }
  ShortRows s;
  s.slices = (rows + 31) / 32;
  s.per_xcd = ((int64_t)a.B * a.H * s.slices + kXcds - 1) / kXcds;
  if (a.q_prescaled) return {};
  const int64_t units = s.per_xcd * n_jobs;
  if (units > (D == 128 ? 2 : tiles <= 6 ? 4 : 3) * cus || tiles > most_tiles(a, D, s.slices, units, cus)) return {};
  s.waves = units <= cus && tiles > 4 ? 8 : 4;
  return s;
}

// The launch as it is planned (and the fold kernel behind it).
static int launch_planned(AttnArgs& a, int D, int n_jobs, const ShortRows& rows, hipStream_t stream, void* workspace, int64_t workspace_bytes) {
  const int64_t slot_bytes = partial_state_bytes(D);
  const unsigned planes_x = (unsigned)a.per_xcd * kXcds;
  if (rows.waves > 0) {
    a.part_ways = rows.slices;
    a.tail_items = (int)rows.per_xcd;
    const dim3 grid((unsigned)rows.per_xcd * kXcds, (unsigned)n_jobs, 1);
    return rows.waves == 8 ? launch_dim(AttnRows8{a}, D, grid, stream) : launch_dim(AttnRows4{a}, D, grid, stream);
  }
  if (a.tail_items == 0) return launch_dim(a, D, dim3(planes_x, (unsigned)n_jobs, 1), stream);
  const int64_t slots = (int64_t)a.tail_items * kXcds * a.part_ways;
  if (a.arrive && !a.row_split && (int64_t)a.tail_items * kXcds * kWaves > kPartCounters) {
    set_error("internal: %d split items per XCD exceed the part counters", a.tail_items);
    return DT_ERR_INVALID;
  }
  // (the planner only considers splits that fit, so this cannot fire; it guards later edits to it)
  if (!a.row_split && slots * slot_bytes > workspace_bytes) {
    set_error("internal: tail split of %lld parts needs %lld bytes of scratch, %lld are there", (long long)slots,
              (long long)(slots * slot_bytes), (long long)workspace_bytes);
    return DT_ERR_INVALID;
  }
  if (!a.row_split) {
    a.ws_out = static_cast<float*>(workspace);
    a.ws_lse = a.ws_out + slots * kBQ * D;
  }
  if (a.tail_start <= 0) {   // every item is split: no job planes
    a.tail_start = 0;
    a.job_planes = 0;
  }
  // parts per XCD, spread over planes of per_xcd entries
  const int part_planes = (a.tail_items * a.part_ways + a.per_xcd - 1) / a.per_xcd;
  const dim3 grid(planes_x, (unsigned)(a.job_planes + part_planes), 1);
  if (a.row_split) return launch_dim(a, D, grid, stream);   // (no partial states)
  std::lock_guard<std::mutex> pair(workspace_lock(workspace));
  if (int rc = launch_dim(a, D, grid, stream)) return rc;
  if (a.arrive) return DT_OK;   // folded by the launch itself
  const dim3 fold_grid((unsigned)a.tail_items * kXcds * kWaves * (D / 64)), fold_block(kFoldThreads);
  if (D == 128) {
    if (a.elem_f16) hipLaunchKernelGGL((attn_tail_fold_kernel<128, true>), fold_grid, fold_block, 0, stream, a);
    else hipLaunchKernelGGL((attn_tail_fold_kernel<128, false>), fold_grid, fold_block, 0, stream, a);
  } else {
    if (a.elem_f16) hipLaunchKernelGGL((attn_tail_fold_kernel<64, true>), fold_grid, fold_block, 0, stream, a);
    else hipLaunchKernelGGL((attn_tail_fold_kernel<64, false>), fold_grid, fold_block, 0, stream, a);
  }
  return hip_fail(hipGetLastError(), "attn tail fold launch");
}

// Whether a launch that merges does so itself, or the fold and merge kernels behind it; `tiles` is the key tiles of the longest
// item, `cus` the CUs of an XCD.  What an item pays is its states' way past the L2, the wait for them and the count; what the
// launch gains is the merge of one round beside the keys of another.  us per call through proAttention.attn, kernels behind -> own:
//   * only the last job's items merge, so there have to be more of them than run at a time, 1.5 a CU: D = 128 24 heads x 1861 queries, 15 of 16
//     chunks computed (24 a XCD) 643 -> 664, 24 x 4000, 3 of 8 (48) 543 -> 536; D = 64 24 x 1861 377 -> 382, 24 x 4000, 15 of 16 1463 ->
//     1450;
//   * an item has to be long beside what it pays, 10 key tiles at D = 64 (24 x 6000 against chunks of 6 tiles 229 -> 246, 16 x 8000, 8 tiles
//     142 -> 142, 32 x 5157, 11 tiles 318 -> 311) and 20 at D = 128, whose states are twice the bytes (24 x 6000, 6 tiles 429 -> 449, 16 x
//     8000, 8 tiles 266 -> 281, 24 x 6510, 13 tiles 605 -> 605, 32 x 8979, 24 tiles 1292 -> 1281);
//   * with 8 items a CU in all both head dimensions gain or are even (24 x 119 056, 3 of 32 17.2 -> 15.9 ms, 30 x 8713, 2 of 3 1877 -> 1863); with
//     fewer D = 128 may lose (48 x 2222, 1 of 8, 1.7 a CU 162 -> 167; 4 of 16, 6.8 a CU 512 -> 514), D = 64 does not (101 -> 102, 301 -> 295).
static bool long_launch_merges(int D, int n_jobs, int per_xcd, int tiles, int cus) {
  return cus > 0 && (int64_t)n_jobs * per_xcd >= 8 * cus && 2 * per_xcd >= 3 * cus && tiles >= (D == 64 ? 10 : 20);
}
// In a short launch the merge is one wavefront's chain of waits per 32 rows, against kernels that spread over the chip, and the GPU mostly
// loses by it; what is gained is one launch less for the host, 2.5 us.  Through proAttention.attn a call whose jobs are listed on the device
// (reuse mask) takes the host 16 us, one with jobs listed by the host (stride schedule) 30; a launch that is over by then merges itself
// (us per call in a loop of calls, kernels behind -> own; in brackets the same with the GPU kept busy):
//   * D = 64 up to 128 queries (24 x 96, 2 states 18.7 -> 15.9 [13.3 -> 12.9]) and beyond them up to 12 items an XCD (4 x 512, 2 of 4
//     19.0 -> 16.3 [16.4 -> 15.8], 24 x 200 18.4 -> 17.0 [15.7 -> 16.9]), 48 where the host lists the jobs (48 x 400, steps of 1 and 4 chunks
//     33.0 -> 30.4 [25.0 -> 26.1]); 24 items on the device's list are too many (48 x 512, two states 20.5 -> 23.0 [22.0 -> 24.3], 24 x 512, 4
//     states 20.6 -> 23.4) and 72 on the host's (48 x 600, 2 chunks 36.2 -> 37.9);
//   * D = 64 in launches that the GPU gains by: one job of 24 key tiles and more, whose items all merge (30 x 1952, 1 of 3 1.06, 12 x 4154,
//     1 of 4 77.5 -> 75.4; 32 x 1479, 24 tiles 1.00, 32 x 1068, 5 tiles 0.96), and an item a CU of one job, of 10 key tiles (12 x 7732,
//     steps of up to 4 chunks 2964 -> 2941, 48 x 2222 148 -> 146; 16 x 1968, 11 tiles 1.00; 24 x 1735 and 48 x 1000, 0.7 a CU, 0.98, 0.96);
//   * D = 128 up to 12 items and either 128 queries and 4 key tiles (24 x 96, 2 states 18.7 -> 16.7 [14.3 -> 15.7]; 30 x 99, 4 tiles 1.00) or
//     160 and 2 (8 x 147, 2 tiles 1.16, 20 x 156, one 1.11; 3 tiles are even: 12 x 142 1.01, 24 x 156 0.95); 48 x 119, 18 items 0.95, 24 x
//     103, 7 tiles 0.94, 12 x 200, 4 tiles 18.4 -> 20.8 [17.9 -> 20.7], 24 x 200, one tile 0.98, 12 x 253, one tile 0.94.  With the host's
//     list up to 24 items of 4 key tiles (48 x 254, 24 items 32.1 -> 29.8 [20.8 -> 25.0]; 48 x 400, 48 items 32.3 -> 36.4);
//   * measured with workgroups of 256 rows, and kept for those of 32, whose wavefronts merge 4 or 8 rows each;
//   * up to 4 states: 8 are twice the loads of the chain (D = 64 24 x 269 17.0 -> 21.7, D = 128 20 x 200 19 -> 25);
//   * items in up to two parts: three and more are folded one after the other (3 x 1706, D = 64, 4 parts 0.91).  The parts are those of
//     workgroups of 256 rows also where the launch takes 32, which has none: such a launch of 17 to 32 key tiles at D = 64 leaves its merge to the
//     kernel behind it and would be shorter with its own (3 x 1706, 1 of 4 chunks 16.5 -> 13.7 [15.0 -> 12.6], 24 x 96, 1 of 2 of 2048 keys 16.1 -> 14.0
//     [15.5 -> 13.8], 12 x 900, 1 of 2 of 1600 20.5 -> 18.2 [20.2 -> 18.1]).
static bool short_launch_merges(int D, int Sq, int n_states, int n_jobs, bool host_listed, int per_xcd, int tiles, int cus) {
  const int64_t items = (int64_t)n_jobs * per_xcd;
  const bool small = Sq <= kBQ / 2;
  if (n_states > kRowsStates) return false;
  if (D == 64) return small || items <= (host_listed ? 48 : 12) || (n_jobs == 1 && tiles >= 24) || (cus > 0 && per_xcd >= cus && tiles >= 10);
  return (items <= (host_listed ? 24 : 12) && (small || host_listed) && tiles <= 4) || (items <= 12 && Sq <= 160 && tiles <= 2);
}
// CUs of an XCD of the current device; 0: not known.
static int xcd_cus() {
  const int cus = cu_count();
  return cus >= 64 && cus % kXcds == 0 ? cus / kXcds : 0;
}
bool may_merge_in_launch(int D, int Sq, int n_states, int n_jobs, bool host_listed, int per_xcd, int tiles) {
  const int cus = xcd_cus();
  return long_launch_merges(D, n_jobs, per_xcd, tiles, cus) || short_launch_merges(D, Sq, n_states, n_jobs, host_listed, per_xcd, tiles, cus);
}
static bool merges_in_launch(const AttnArgs& a, int D, int n_jobs, int tiles, int cus, const TailPlan& plan) {
  if (long_launch_merges(D, n_jobs, a.per_xcd, tiles, cus)) return true;
  return short_launch_merges(D, a.Sq, a.merge_n, n_jobs, a.dev_ids == nullptr, a.per_xcd, tiles, cus) &&
         (plan.items == 0 || plan.rows || plan.ways <= 2);
}

// The merge of such a launch, by the merge kernel.
static int merge_behind(const AttnArgs& a, int D, hipStream_t stream) {
  const AttnState* states = a.dev_ids ? a.arena : a.state;
  const void* outs[DT_MAX_CHUNKS];
  const float* lses[DT_MAX_CHUNKS];
  int32_t dtypes[DT_MAX_CHUNKS];
  for (int i = 0; i < a.merge_n; ++i) {
    outs[i] = states[i].out;
    lses[i] = states[i].lse;
    dtypes[i] = a.elem_f16 ? DT_FP16 : DT_BF16;
  }
  return dt_merge_states(a.merge_n, outs, lses, dtypes, nullptr, a.merge_out, a.merge_dtype, a.merge_lse, DT_LSE_BSH, a.B, a.Sq, a.H,
                         D, stream);
}
static_assert(DT_MAX_MERGE_LIST <= DT_MAX_CHUNKS && DT_MAX_CHUNKS <= DT_MAX_MERGE, "any list of states is one merge launch");

int launch_attn(const AttnArgs& a_in, int D, int n_jobs, hipStream_t stream, void* workspace, int64_t workspace_bytes) {
  if (n_jobs <= 0 || a_in.total <= 0) return DT_OK;
  if (D != 128 && D != 64) {
    set_error("head dim %d not built (64 and 128 are)", D);
    return DT_ERR_UNSUPPORTED;
  }
  if (a_in.elem_f16 && a_in.q_prescaled) {
    set_error("fp16 tensors and a prescaled q do not combine (the prescaled softmax keeps probabilities beyond fp16's range)");
    return DT_ERR_UNSUPPORTED;
  }
  AttnArgs a = a_in;
  a.job_planes = n_jobs;
  a.tail_start = INT32_MAX;
  a.tail_items = 0;
  a.part_ways = 0;
  a.row_split = 0;
  constexpr int kMaxLaunchJobs = DT_MAX_JOBS * DT_MAX_SEGMENTS;   // (more: no planning)
  bool merge_after = false;
  ShortRows rows;
  if (n_jobs <= kMaxLaunchJobs) {
    JobSize size[kMaxLaunchJobs];
    job_sizes(a, n_jobs, size);
    const int cus = xcd_cus();
    const bool split = cus > 0 && workspace;
    if (split) rows = short_rows(a, D, n_jobs, size, cus);
    const TailPlan plan = plan_launch(a, D, n_jobs, size, cus, split ? std::min(workspace_bytes, kWorkspaceBytes) / partial_state_bytes(D) : -1);
    a.tail_items = plan.items;
    a.part_ways = plan.ways;
    a.row_split = plan.rows ? 1 : 0;
    if (plan.items > 0) a.tail_start = n_jobs * a.per_xcd - plan.items;
    if (a.arrive) {
      int longest = 0;
      for (int j = 0; j < n_jobs; ++j) longest = std::max(longest, size[j].tiles);
      merge_after = !merges_in_launch(a, D, n_jobs, longest, cus, plan);
    }
  }
  if (!merge_after) return launch_planned(a, D, n_jobs, rows, stream, workspace, workspace_bytes);
  a.arrive = nullptr;
  if (int rc = launch_planned(a, D, n_jobs, rows, stream, workspace, workspace_bytes)) return rc;
  return merge_behind(a, D, stream);
}

}  // namespace dt
