// Shared declarations of the kernel translation units (not part of the public ABI).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "ditango_hip.h"

#include <mutex>

namespace dt {

void set_error(const char* fmt, ...);
int hip_fail(hipError_t e, const char* what);

// n / d for n < 2^31, with mul = ceil(2^(31 + L) / d) and shift = L - 1 for the smallest L with d <= 2^L: the error of mul, less
// than d, times n stays below 2^(31 + L).  d = 1: shift -1.
struct Quotient {
  uint32_t mul;
  int32_t shift;
};
static inline Quotient quotient_by(int32_t d) {
  int L = 0;
  while ((1ll << L) < d) ++L;
  return {L == 0 ? 0u : (uint32_t)(((1ull << (31 + L)) + (uint64_t)d - 1) / (uint64_t)d), L - 1};
}
__device__ __forceinline__ uint32_t quotient(uint32_t n, const Quotient& by) {
  return by.shift < 0 ? n : __umulhi(n, by.mul) >> by.shift;
}

// One KV chunk, one reference of a job to a chunk, one job of an attention launch: a record each, so that a workgroup finds
// what it needs in one or two cache lines.
struct AttnChunk {
  const uint16_t* k;
  const uint16_t* v;
  int64_t sb;       // batch stride, elements
  int32_t len;      // keys
};
struct AttnEntry {
  int32_t chunk;
  int32_t kv_begin, kv_len;   // keys [kv_begin, kv_begin + kv_len) of the chunk
};
struct AttnJob {
  uint16_t* out;
  float* lse;
  int32_t begin, end;         // chunk references
  // query rows [q_begin, q_begin + q_len): a segment of a packed variable-length batch is a job on sub-ranges (with
  // boundaries in device memory q_begin names the segment)
  int32_t q_begin, q_len;
};

struct AttnState {
  const uint16_t* out;        // [B,Sq,H,D]
  const float* lse;           // [B,H,Sq]
};

// Kernel arguments of the chunk-attention kernel.  Passed by value, so the
// chunk and job tables travel in the kernarg segment: no device-side table,
// no host-to-device copy per call.  q, K, V and the output states are 16-bit elements: bfloat16, or IEEE half when
// elem_f16 is set.
struct AttnArgs {
  // ---- what the workgroups read: three cache lines and the head of the fourth
  const uint16_t* q;
  int64_t q_sb, q_ss, q_sh;
  int32_t H, Sq;
  int32_t nqt;        // query tiles per (batch, head)
  int32_t total;      // B*H*nqt work items per job
  int32_t per_xcd;    // work items handed to each of the 8 XCDs
  // Tail balancing (workspace launches only).  The work items of a launch, in dispatch order: those of an XCD are
  // numbered flat = job * per_xcd + idx (idx: position in the XCD's share of the job).  Items with flat < tail_start run
  // as one workgroup each; the tail_items behind them run as part_ways workgroups over disjoint ranges of key
  // tiles, in grid planes of their own behind the job planes (same launch, so a part starts as soon as a CU is
  // free).  The parts write fp32 partial states into the workspace and a small second kernel folds them into the destination.
  // With row_split the two parts of an item are its two halves of the query rows instead: no partial states, no fold.
  int32_t job_planes;  // grid planes (blockIdx.y) that are jobs (0: every item is split); planes behind them hold parts
  int32_t tail_start;  // INT32_MAX: nothing is split
  int32_t tail_items;  // per XCD
  int32_t part_ways;
  int32_t n_chunks;
  int32_t n_seg;
  float scale_log2;    // softmax scale * log2(e)
  int64_t kv_ss, kv_sh;
  // Device-listed jobs (dev_ids != nullptr): job j computes chunk dev_ids[j] if j < *dev_count.  On a packed
  // variable-length batch (n_seg > 0) they come segment-major, the first segment last: launch job j is slot
  // j % n_slots of the schedule, and the keys of segment s inside chunk c are those of entry[c * n_seg + s].
  const int32_t* dev_ids;
  const int32_t* dev_count;
  // Segment boundaries that live in DEVICE memory (cu_q != nullptr), the calling convention of
  // flash_attn_varlen_func: cu_q[s], cu_q[s + 1] bound the query rows of segment s and cu_kv[c][s],
  // cu_kv[c][s + 1] its keys inside chunk c (every chunk brings its own boundaries).  The host never
  // reads them; the kernel clamps them to the tensors' extents.
  const int32_t* cu_q;
  int32_t n_slots;
  int32_t diag;
  uint16_t* slot_out;
  float* slot_lse;
  int64_t slot_out_stride, slot_lse_stride;
  uint16_t* diag_out;
  float* diag_lse;
  float* ws_out;    // [slot][8 wavefronts][D / 8 groups of 4 elements][64 lanes][4], the accumulators as they lie in registers
  float* ws_lse;    // [slot][256]
  int32_t row_split;    // the tail items are cut in two along the query rows instead of along the keys (no partial states)
  // Launches that merge (arrive != nullptr): whoever completes the last of the launch's merge_jobs states of 32 query rows
  // merges the merge_n states there are of these rows (`arena` or `state` below) into merge_out and merge_lse ([B,Sq,H]).
  // The parts of a split item meet in the same way; there is no fold kernel.  Counters: kPartCounters for the parts, then 8 per work item of a job.
  int32_t merge_n;
  uint32_t* arrive;
  void* merge_out;
  float* merge_lse;
  int32_t merge_jobs;
  int32_t merge_dtype;  // DT_FP32, or the states' own 16-bit type
  // ---- the host's own
  int32_t B;
  int32_t q_prescaled;  // the caller folded scale_log2 into q: scores are already in log2 units
  int32_t elem_f16;     // the 16-bit tensors are IEEE half instead of bfloat16
  // ---- tables
  union {
    AttnJob job[DT_MAX_JOBS];
    AttnState arena[DT_MAX_CHUNKS];       // merging launches with device-listed jobs: what they merge
  };
  AttnChunk chunk[DT_MAX_CHUNKS];
  AttnEntry entry[DT_MAX_JOB_ENTRIES];
  int32_t seg_q_begin[DT_MAX_SEGMENTS];
  int32_t seg_q_len[DT_MAX_SEGMENTS];
  union {
    const int32_t* cu_kv[DT_MAX_CHUNKS];
    AttnState state[DT_MAX_MERGE_LIST];   // ... with host-listed jobs
  };
};

// Dynamic LDS of one attention workgroup by head dimension (four 64-key buffers per operand and the epilogue's
// staging rows).  The
// occupancy of a CU follows from it: one workgroup at 128, two at 64.
constexpr int kAttnLdsBytes128 = 163840;
constexpr int kAttnLdsBytes64 = 81920;

// Bytes of one partial state of a split item: 256 queries in fp32 and their lse.
constexpr int64_t partial_state_bytes(int D) { return 256ll * D * 4 + 256 * 4; }

// Workspace bytes the tail balancing can use at most (what dt_attn_workspace_bytes reports).
constexpr int64_t kWorkspaceBytes = 1536 * partial_state_bytes(64);
static_assert(kWorkspaceBytes / partial_state_bytes(64) == 1536 && kWorkspaceBytes / partial_state_bytes(128) == 773);

// The allocation-free entry point splits tails inside a device array of this many bytes.  At D = 128 a tail of 17 ... 31 items
// per XCD takes two or three parts an item, up to 500 in all: with half the array it runs unsplit (24 heads x 14882 x one
// chunk, D = 128 2156 -> 2145 us; D = 64, 1008 parts, 1271 -> 1253).
constexpr int64_t kStaticTailBytes = DT_NOALLOC_TAIL_SLOTS * partial_state_bytes(64);
static_assert(kStaticTailBytes / partial_state_bytes(64) == 1024 && kStaticTailBytes / partial_state_bytes(128) == 515);
// Arrival counters of the parts of split items in a merging launch: one per 32-row slice of an item; a launch splits fewer
// items than the chip has CUs.
constexpr int kPartCounters = 2048;

// Device address and size of that array on the current device (looked up once per device).
int static_tail_scratch(void** ptr, int64_t* bytes);

constexpr int kMergeBatch = 8;   // the lists of states are filled up to multiples of this with the last one
static_assert(DT_MAX_CHUNKS % kMergeBatch == 0 && DT_MAX_MERGE_LIST % kMergeBatch == 0, "filled lists stay in their place");
static_assert(DT_MAX_MERGE_LIST * sizeof(AttnState) <= DT_MAX_CHUNKS * sizeof(int32_t*), "the list shares the boundaries' place");
static_assert(sizeof(AttnArgs) <= 4096, "the kernel arguments travel in the 4 KB kernarg segment");

// Held while a launch that writes partial states, and the fold kernel where there is one, go into the queue: two threads may
// launch on one stream, with the workspace that belongs to it, and no parts of the other's may come between the parts and their
// fold.  (One of a few locks, chosen by the workspace: a thread that waits for room in its stream's queue holds up few others.)
std::mutex& workspace_lock(const void* workspace);
// Whether a merging launch of these sizes may merge itself (see merges_in_launch).
bool may_merge_in_launch(int D, int Sq, int n_states, int n_jobs, bool host_listed, int per_xcd, int tiles);
int launch_attn(const AttnArgs& a, int D, int n_jobs, hipStream_t stream, void* workspace = nullptr,
                int64_t workspace_bytes = 0);

}  // namespace dt
