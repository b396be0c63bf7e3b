// wp_plan.hip -- once-per-step segment plan, built on the GPU (gfx950).
//
// Input: token_lora_indices[T] (int64 or int32) in HBM.  One workgroup builds,
// with every intermediate held in LDS (gfx950: 160 KB per workgroup):
//
//   1. the exported segment table, bit-exact with the reference's
//      build_seg_bounds_kernel (csrc/kernels/warp_pipe_r32.cu:461-512):
//      maximal runs of equal ids in token order, ids < 0 skipped, every run
//      split into pieces of 32 tokens (the last one takes the remainder),
//      slots assigned in token-start order by an exclusive scan;
//   2. the grouping the apply kernels run on (no reference counterpart): the
//      tokens of ids >= 0 in a stable counting sort by adapter id (`perm`), each
//      adapter's tokens cut into blocks of `bt` tokens.  Every touched adapter's
//      weights are then streamed once per block instead of once per run (about
//      232 runs vs 49 adapters for 256 Zipf-routed decode tokens).
//
// The reference uses one 256-thread block with a serial per-run scan and a
// Hillis-Steele scan over shared memory, writing over PCIe into mapped host
// memory.  Here the kernel is bound by latency alone (a few KB of traffic, one
// workgroup), so it is built to pass few workgroup barriers: 64 consecutive
// tokens are one wave's lanes, a run table is a 64-bit ballot per 64 tokens,
// ranks among equal ids come from ballots and popcounts, and every wave scans
// the per-wave counts by itself instead of waiting for another to do it.  A
// step whose ids are below 256 takes two barriers in all; larger ids take the
// same counting pass once per further 8 bits.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "wp_apply.h"
#include "wp_sync.h"

namespace wp {
namespace {


// Traced builds (-DWP_TRACE): thread 0 records the 100 MHz real-time counter
// at the plan build's phase boundaries into m.trace[0..7], after waiting for
// its memory operations: 0 entry, 1 ids loaded, 2 run masks exchanged (first
// barrier, maintenance done), 3 segment pieces and digit counts exchanged
// (second barrier), 4 segment table stored, 5 digit bases known, 6 perm and
// block token lists stored, 7 block table and header stored.
#ifdef WP_TRACE
__device__ __forceinline__ void plan_stamp(const Maint& m, int i) {
  if (m.trace != nullptr && threadIdx.x == 0) {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    m.trace[i] = wall_clock64();
  }
}
#else
__device__ __forceinline__ void plan_stamp(const Maint&, int) {}
#endif

// ---------------------------------------------------------- maintenance ----

__device__ __forceinline__ uint64_t agent_load64(const void* p) {
  return __hip_atomic_load(static_cast<const uint64_t*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void agent_store64(void* p, uint64_t v) {
  __hip_atomic_store(static_cast<uint64_t*>(p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// What a plan build does first (every thread of the workgroup takes part):
//   * each ready staging-slot publication is written into the adapter table,
//     so that every kernel of the step that follows sees the same table (a
//     publication read while its writer is at work -- odd or changed sequence
//     -- is left for the next build);
//   * after a give-up (kHdrPoison), the partial buffer is refilled with
//     kPartialEmpty and the per-block counters cleared, then the word reset.
// Ends with a workgroup barrier.
__device__ void maintain(uint32_t* header, const Maint& m, int* s_flag) {
  const int tid = threadIdx.x;
  if (m.table != nullptr && tid < m.n_pubs) {
    const SlotPub* p = m.pubs + tid;
    const uint32_t s1 = __hip_atomic_load(&p->seq, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT);
    if ((s1 & 1u) == 0u) {
      const int32_t id = __hip_atomic_load(&p->id, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const uint32_t gen = __hip_atomic_load(&p->gen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const uint32_t retired = __hip_atomic_load(m.retired + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      uint64_t w[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) w[i] = agent_load64(reinterpret_cast<const uint64_t*>(&p->entry) + i);
      // The payload loads complete before the sequence is read again.
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      const uint32_t s2 = __hip_atomic_load(&p->seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      // A fill whose release has been enqueued before this build is not
      // installed again, whichever landed first.
      if (s1 == s2 && id >= 0 && id < m.table_cap && gen > retired) {
        uint64_t* dst = reinterpret_cast<uint64_t*>(m.table + id);
#pragma unroll
        for (int i = 0; i < 4; ++i) dst[i] = w[i];
        __hip_atomic_fetch_add(&header[kHdrTableVer], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  }
  if (tid == 0) *s_flag = m.part != nullptr ? static_cast<int>(
                              __hip_atomic_load(&header[kHdrPoison], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) : 0;
  __syncthreads();
  if (*s_flag != 0) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    const u32x4 e = u32x4{kPartialEmpty, kPartialEmpty, kPartialEmpty, kPartialEmpty};
    u32x4* part4 = reinterpret_cast<u32x4*>(m.part);
    for (uint64_t i = tid; i < m.part_words / 4; i += blockDim.x) part4[i] = e;
    for (uint64_t i = tid; i < m.consumed_words; i += blockDim.x) m.consumed[i] = 0u;
    __syncthreads();
    if (tid == 0) __hip_atomic_store(&header[kHdrPoison], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

__global__ __launch_bounds__(256) void maintain_kernel(uint32_t* header, Maint m) {
  __shared__ int s_flag;
  maintain(header, m, &s_flag);
}

// A publication under its sequence lock: odd sequence, payload, even
// sequence, with agent-scope release fences between, so a reader that saw
// the same even value before and after its payload loads has a whole payload.
// One thread.
__device__ void publish(SlotPub* pub, int32_t id, uint32_t gen, const Entry& en) {
  const uint32_t base = __hip_atomic_load(&pub->seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & ~1u;
  __hip_atomic_store(&pub->seq, base + 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
  __hip_atomic_store(&pub->id, id, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(&pub->gen, gen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
  for (int i = 0; i < 4; ++i)
    agent_store64(reinterpret_cast<uint64_t*>(&pub->entry) + i, reinterpret_cast<const uint64_t*>(&en)[i]);
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
  __hip_atomic_store(&pub->seq, base + 2u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// One wave; thread 0 writes.
__global__ __launch_bounds__(64) void entry_writes_kernel(EntryWrites w) {
  if (threadIdx.x != 0) return;
  if (w.pub != nullptr) publish(w.pub, w.pub_id, w.pub_gen, w.pub_entry);
  for (int i = 0; i < w.n_retire; ++i)
    __hip_atomic_fetch_max(w.retire[i], w.retire_gen[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  for (int i = 0; i < w.n; ++i) *w.dst[i] = w.val[i];
  if (w.header != nullptr && w.n > 0)
    __hip_atomic_fetch_add(&w.header[kHdrTableVer], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Workgroup (job, part) copies its share of the job's A and B in 16-byte
// units; every workgroup's stores complete before it counts itself done, and
// the job's last workgroup publishes the slot.
__global__ __launch_bounds__(256) void stage_copy_kernel(StageJobs jobs) {
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  const int j = blockIdx.x / kStageWorkgroups;
  const int part = blockIdx.x - j * kStageWorkgroups;
  const StageJob& job = jobs.job[j];
  const uint64_t stride = static_cast<uint64_t>(kStageWorkgroups) * blockDim.x;
  const uint64_t first = static_cast<uint64_t>(part) * blockDim.x + threadIdx.x;
  for (int m = 0; m < 2; ++m) {
    const u32x4* src = static_cast<const u32x4*>(m == 0 ? job.src_a : job.src_b);
    u32x4* dst = static_cast<u32x4*>(m == 0 ? job.dst_a : job.dst_b);
    const uint64_t n = (m == 0 ? job.a_bytes : job.b_bytes) / 16;
    // Four loads in flight per thread.
    uint64_t i = first;
    for (; i + 3 * stride < n; i += 4 * stride) {
      const u32x4 v0 = src[i], v1 = src[i + stride], v2 = src[i + 2 * stride], v3 = src[i + 3 * stride];
      dst[i] = v0;
      dst[i + stride] = v1;
      dst[i + 2 * stride] = v2;
      dst[i + 3 * stride] = v3;
    }
    for (; i < n; i += stride) dst[i] = src[i];
  }
  __shared__ int s_last;
  // Release: this workgroup's stores are visible device-wide before its count.
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
  __syncthreads();
  if (threadIdx.x == 0) {
    const uint32_t done = __hip_atomic_fetch_add(&job.pub->copies, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
    s_last = done == kStageWorkgroups - 1 ? 1 : 0;
  }
  __syncthreads();
  if (s_last != 0 && threadIdx.x == 0) {
    __hip_atomic_store(&job.pub->copies, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    publish(job.pub, job.pub_id, job.pub_gen, job.pub_entry);
  }
}

// plan_kernel's explicit arguments, as laid out in its kernel-argument
// segment: touch_kernel_args reads below this size only.
struct PlanKernelArgs {
  const void* idx;
  int idx_is_int64, T;
  uint32_t* header;
  Segment* segments;
  Block* blocks;
  int32_t* perm;
  int32_t* bperm;
  Entry* bentries;
  FinePlan fine;
  int seg_cap, block_cap, bt;
  Maint m;
};
static_assert(offsetof(PlanKernelArgs, m) == 104 && sizeof(PlanKernelArgs) == 104 + sizeof(Maint),
              "plan_kernel's argument size as passed to touch_kernel_args");

// ------------------------------------------------------------- plan build ----

// Digits of one counting pass (8 bits).
constexpr int kDigits = 256;

__device__ __forceinline__ uint64_t lanes_below(int lane) { return (1ull << lane) - 1ull; }
__device__ __forceinline__ int last_bit(uint64_t m) { return 63 - __builtin_clzll(m); }

template <typename V, typename Op>
__device__ __forceinline__ V wave_all_reduce(V v, Op op) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = op(v, __shfl_xor(v, off, 64));
  return v;
}

// Position of the last start bit in the words before `first`, or -1.
template <int NWORDS>
__device__ __forceinline__ int last_start_before(const uint64_t* s_start, int first) {
  if (first == 0) return -1;
  const int lane = threadIdx.x & 63;
  int v = -1;
#pragma unroll
  for (int k = 0; k < (NWORDS + 63) / 64; ++k) {
    const int wi = lane + 64 * k;
    if (wi < first) {
      const uint64_t m = s_start[wi];
      if (m != 0) v = wi * 64 + last_bit(m);
    }
  }
  return wave_all_reduce(v, [](int a, int b) { return a > b ? a : b; });
}

// Set bits of the words before `first` (low half) and of all words (high half).
template <int NWORDS>
__device__ __forceinline__ uint32_t count_words(const uint64_t* s_words, int first) {
  const int lane = threadIdx.x & 63;
  uint32_t v = 0;
#pragma unroll
  for (int k = 0; k < (NWORDS + 63) / 64; ++k) {
    const int wi = lane + 64 * k;
    if (wi < NWORDS) {
      const uint32_t c = static_cast<uint32_t>(__popcll(s_words[wi]));
      v += (c << 16) + (wi < first ? c : 0u);
    }
  }
  return wave_all_reduce(v, [](uint32_t a, uint32_t b) { return a + b; });
}

// Pieces of runs.  start[e] marks the first item of each run among the 64
// items of this wave's word e (word index first + e, item i = 64 * word +
// lane); `carry` is the last run start before the wave's words.  piece[e]
// marks the items of `live` at a multiple of P from their run's start, and
// rs[e] is the lane's run start.
template <int E>
__device__ __forceinline__ void mark_pieces(const uint64_t (&start)[E], const uint64_t (&live)[E], int first, int carry,
                                            int P, uint64_t (&piece)[E], int (&rs)[E]) {
  const int lane = threadIdx.x & 63;
  const uint64_t le = (lanes_below(lane) << 1) | 1ull;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int w0 = (first + e) * 64;
    const uint64_t below = start[e] & le;
    rs[e] = below != 0 ? w0 + last_bit(below) : carry;
    const bool p = ((live[e] >> lane) & 1ull) != 0 && ((w0 + lane - rs[e]) & (P - 1)) == 0;
    piece[e] = __ballot(p);
    if (start[e] != 0) carry = w0 + last_bit(start[e]);
  }
}

// Rank of each item among the wave's earlier items of the same digit (in item
// order), and the wave's count per digit left in cnt[] (zeroed by the caller).
// `bits`: digit bits that can be set.  The row is this wave's own and LDS
// accesses of one wave complete in order; volatile keeps the compiler from
// carrying a count across words.
template <int E>
__device__ __forceinline__ void rank_digits(const uint32_t (&dig)[E], const uint64_t (&live)[E], int bits,
                                            volatile uint32_t* cnt, uint32_t (&rank)[E]) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    rank[e] = 0;
    if (live[e] == 0) continue;
    uint64_t m = live[e];
    for (int b = 0; b < bits; ++b) {
      const bool one = ((dig[e] >> b) & 1u) != 0;
      const uint64_t ones = __ballot(one);
      m &= one ? ones : ~ones;
    }
    if ((live[e] >> lane) & 1ull) {
      const uint32_t base = cnt[dig[e]];
      rank[e] = base + static_cast<uint32_t>(__popcll(m & lanes_below(lane)));
      if ((m & lanes_below(lane)) == 0) cnt[dig[e]] = base + static_cast<uint32_t>(__popcll(m));
    }
  }
}

// One wave's view of every wave's digit counts: digits 4 * lane .. + 3.
struct Digits {
  uint32_t tot[4];  // items of the digit
  uint32_t pre[4];  // ... in the waves before this one
  uint32_t off[4];  // items of all digits below
  uint32_t blk[4];  // blocks of all digits below
  uint32_t fblk[4]; // kFineTokens-token blocks of all digits below (fine only)
  uint32_t n_items, n_blocks, n_fine, n_digits;
};
template <int NW>
__device__ __forceinline__ Digits scan_digits(const uint32_t (*s_cnt)[kDigits], int wave, int max_digit, int bt_log2,
                                              bool fine) {
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  const int lane = threadIdx.x & 63;
  Digits r;
#pragma unroll
  for (int j = 0; j < 4; ++j) r.tot[j] = r.pre[j] = 0;
  if (4 * lane <= max_digit) {
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const u32x4 c = *reinterpret_cast<const u32x4*>(&s_cnt[w][4 * lane]);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        r.tot[j] += c[j];
        r.pre[j] += w < wave ? c[j] : 0u;
      }
    }
  }
  // Items (at most 8192) and blocks (at most as many) in one scan.
  const uint32_t round = (1u << bt_log2) - 1u;
  uint32_t own[4], sum = 0;
  r.n_digits = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    own[j] = r.tot[j] | (((r.tot[j] + round) >> bt_log2) << 16);
    sum += own[j];
    r.n_digits += static_cast<uint32_t>(__popcll(__ballot(r.tot[j] != 0)));
  }
  uint32_t inc = sum;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t y = __shfl_up(inc, off, 64);
    if (lane >= off) inc += y;
  }
  const uint32_t all = __shfl(inc, 63, 64);
  r.n_items = all & 0xffffu;
  r.n_blocks = all >> 16;
  uint32_t ex = inc - sum;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    r.off[j] = ex & 0xffffu;
    r.blk[j] = ex >> 16;
    ex += own[j];
    r.fblk[j] = 0;
  }
  r.n_fine = r.n_blocks;
  if (fine) {
    sum = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      own[j] = (r.tot[j] + kFineTokens - 1) / kFineTokens;
      sum += own[j];
    }
    inc = sum;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t y = __shfl_up(inc, off, 64);
      if (lane >= off) inc += y;
    }
    r.n_fine = __shfl(inc, 63, 64);
    ex = inc - sum;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      r.fblk[j] = ex;
      ex += own[j];
    }
  }
  return r;
}

// An adapter's table entry as of this build (agent-scope loads: the maintenance
// may have installed it from another wave), or an empty one.
struct EntryWords {
  uint64_t w[4];
};
__device__ __forceinline__ EntryWords read_entry(const Maint& m, int32_t id, bool wanted) {
  EntryWords en{{0, 0, 0, 0}};
  if (wanted && m.table != nullptr && id >= 0 && id < m.table_cap) {
#pragma unroll
    for (int i = 0; i < 4; ++i) en.w[i] = agent_load64(reinterpret_cast<const uint64_t*>(m.table + id) + i);
  }
  return en;
}
__device__ __forceinline__ void put_block(Block* blocks, Entry* bentries, int q, int32_t id, int first, int count,
                                          const EntryWords& en) {
  Block b;
  b.adapter_id = id;
  b.first = first;
  b.count = count;
  b.entry = id;
  blocks[q] = b;
  if (bentries != nullptr) {
    uint64_t* dst = reinterpret_cast<uint64_t*>(bentries + q);
#pragma unroll
    for (int i = 0; i < 4; ++i) dst[i] = en.w[i];
  }
}

// Measured on MI355X, build_seg_bounds per launch in a graph of 40 (launch
// included), against a run table sorted by counting or by a bitonic sort
// (Zipf(1.1) routing over 64 ids, before -> now, us; past 512 tokens both
// tables of blocks): T=64 8.8 -> 4.1, 256 12.6 -> 4.5, 512 20.1 -> 6.2, 1024
// 27.0 -> 7.6, 2048 41.7 -> 8.1, 4096 80.5 -> 11.8, 8192 152.7 -> 20.5; 16
// contiguous prompts, T=8192 24.2 -> 16.9; ids up to 1e6, T=256 15.2 -> 7.4,
// T=8192 198.7 -> 46.4.
template <int NT, int E>
__global__ __launch_bounds__(NT) void plan_kernel(const void* __restrict__ idx, int idx_is_int64, int T,
                                                  uint32_t* __restrict__ header, Segment* __restrict__ segments,
                                                  Block* __restrict__ blocks, int32_t* __restrict__ perm,
                                                  int32_t* __restrict__ bperm, Entry* __restrict__ bentries,
                                                  FinePlan fine, int seg_cap, int block_cap, int bt, Maint m) {
  touch_kernel_args<static_cast<int>(sizeof(PlanKernelArgs))>();
  constexpr int CAP = NT * E;
  constexpr int NW = NT / 64;
  constexpr int NWORDS = NW * E;
  static_assert(NW % 4 == 0 && CAP <= 65536 / 2, "digit columns per wave; 16-bit token positions");
  __shared__ uint64_t s_start[NWORDS];  // run starts, one bit per item
  __shared__ uint64_t s_piece[NWORDS];  // piece starts
  __shared__ uint64_t s_fpiece[NWORDS]; // ... of the fine table (ids of 256 and more)
  __shared__ alignas(16) uint32_t s_cnt[NW][kDigits];
  // Each wave's own digit bases: {items below | items of earlier waves << 16,
  // blocks below | fine blocks below << 16}.
  __shared__ uint2 s_base[NW][kDigits];
  __shared__ uint32_t s_wmax[NW];
  __shared__ uint32_t s_wflag[NW];
  // Ids of 256 and more only: the keys by token, and the order of each pass.
  __shared__ uint32_t s_key[CAP];
  __shared__ uint16_t s_ord[2][CAP];
  __shared__ int s_flag;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int first = wave * E;  // this wave's first word
  const int bt_log2 = 31 - __builtin_clz(static_cast<unsigned>(bt));
  plan_stamp(m, 0);

  // 1. ids: lane l of word w holds token 64 w + l.  The id before the wave's
  //    first token, the publications' state, the poison word and the table
  //    version load beside them (the routing does not depend on the table).
  const auto load_id = [&](int i) {
    return idx_is_int64 ? static_cast<const long long*>(idx)[i]
                        : static_cast<long long>(static_cast<const int*>(idx)[i]);
  };
  long long ids[E];
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int i = (first + e) * 64 + lane;
    ids[e] = i < T ? load_id(i) : -1;
  }
  long long before = 0;
  if (first > 0 && first * 64 - 1 < T) before = load_id(first * 64 - 1);
  // A slot whose publication is absent or retired needs no maintenance.  The
  // words are read unordered: a publication that was complete before this
  // launch is seen whole, one still being written may wait for the next build
  // (maintain() itself reads under the sequence lock).
  uint32_t todo = 0;
  if (m.table != nullptr && tid < m.n_pubs) {
    const SlotPub* p = m.pubs + tid;
    const int32_t id = __hip_atomic_load(&p->id, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint32_t gen = __hip_atomic_load(&p->gen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint32_t retired = __hip_atomic_load(m.retired + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    todo = id >= 0 && gen > retired ? 1u : 0u;
  }
  uint32_t table_ver = 0;
  if (tid == 0) {
    if (m.part != nullptr)
      todo |= __hip_atomic_load(&header[kHdrPoison], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u ? 1u : 0u;
    // The table version the block entry copies below are taken at.  A build
    // without copies records a version that no table write produces (the
    // complement of the current one), so copies left by an earlier build can
    // never pass for current ones.
    table_ver = __hip_atomic_load(&header[kHdrTableVer], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  plan_stamp(m, 1);

  // 2. Run starts in token order (reference :484) and the largest key.
  uint64_t start[E], live[E];
  uint32_t key[E];
  uint32_t kmax = 0;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int i = (first + e) * 64 + lane;
    long long prev = __shfl_up(ids[e], 1, 64);
    if (lane == 0) prev = before;
    start[e] = __ballot(i < T && (i == 0 || prev != ids[e]));
    before = __shfl(ids[e], 63, 64);
    const bool ok = i < T && ids[e] >= 0;
    live[e] = __ballot(ok);
    key[e] = static_cast<uint32_t>(static_cast<int>(ids[e]));
    if (ok && key[e] > kmax) kmax = key[e];
    if (lane == 0) {
      s_start[first + e] = start[e];
      if (i < T) reinterpret_cast<uint64_t*>(header + kHdrMask)[first + e] = live[e];
    }
  }
  kmax = wave_all_reduce(kmax, [](uint32_t a, uint32_t b) { return a > b ? a : b; });
  const uint64_t any_todo = __ballot(todo != 0);
  if (lane == 0) {
    s_wmax[wave] = kmax;
    s_wflag[wave] = any_todo != 0 ? 1u : 0u;
  }
  // This wave's digit counts (a row only it writes and, until the second
  // barrier, reads).
#pragma unroll
  for (int j = 0; j < kDigits / 64; ++j) s_cnt[wave][lane + 64 * j] = 0u;
  lds_barrier();

  uint32_t flag = 0;
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    kmax = s_wmax[w] > kmax ? s_wmax[w] : kmax;
    flag |= s_wflag[w];
  }
  if (flag != 0) {
    // Publications into the adapter table, the partial buffer's repair.
    maintain(header, m, &s_flag);
    __syncthreads();
    if (tid == 0) table_ver = __hip_atomic_load(&header[kHdrTableVer], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  plan_stamp(m, 2);

  // 3. The exported table's pieces: a run of id >= 0 starts one every 32
  //    tokens (reference :485-489).  The first counting pass over the ids.
  uint64_t piece[E];
  int rs[E];
  mark_pieces<E>(start, live, first, last_start_before<NWORDS>(s_start, first), kMaxSegmentTokens, piece, rs);
#pragma unroll
  for (int e = 0; e < E; ++e)
    if (lane == 0) s_piece[first + e] = piece[e];
  const bool small_ids = kmax < static_cast<uint32_t>(kDigits);
  const int max_digit = small_ids ? static_cast<int>(kmax) : kDigits - 1;
  uint32_t dig[E], rank[E];
#pragma unroll
  for (int e = 0; e < E; ++e) {
    dig[e] = key[e] & (kDigits - 1);
    if (!small_ids) s_key[(first + e) * 64 + lane] = key[e];
  }
  rank_digits<E>(dig, live, small_ids ? 32 - __builtin_clz(kmax | 1u) : 8, s_cnt[wave], rank);
  lds_barrier();
  plan_stamp(m, 3);

  // 4. Segment table: slots by token order (reference :494-503).
  const uint32_t nseg = count_words<NWORDS>(s_piece, first);
  const int n_segs = static_cast<int>(nseg >> 16);
  int slot0 = static_cast<int>(nseg & 0xffffu);
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int w = first + e;
    const int i = w * 64 + lane;
    const int slot = slot0 + __popcll(piece[e] & lanes_below(lane));
    slot0 += __popcll(piece[e]);
    if (!((piece[e] >> lane) & 1ull) || slot >= seg_cap) continue;
    // The piece ends at the next run or piece start (at most 32 tokens on), or at T.
    const uint64_t up = ((start[e] | piece[e]) >> lane) >> 1;
    int end = T;
    if (up != 0) {
      end = i + 1 + __builtin_ctzll(up);
    } else if (w + 1 < NWORDS) {
      const uint64_t nx = s_start[w + 1] | s_piece[w + 1];
      if (nx != 0) end = (w + 1) * 64 + __builtin_ctzll(nx);
    }
    Segment s;
    s.adapter_id = static_cast<int>(key[e]);
    s.token_start = i;
    s.token_count = end - i;
    s.pad = 0;
    segments[slot] = s;
  }
  plan_stamp(m, 4);

  // 5. Tokens grouped by adapter, token order kept inside an adapter.
  const bool has_fine = fine.blocks != nullptr;
  const bool want_entry = bentries != nullptr;
  int n_tok, n_groups, n_blocks, n_fine;
  if (small_ids) {
    const Digits g = scan_digits<NW>(s_cnt, wave, max_digit, bt_log2, has_fine);
    n_tok = static_cast<int>(g.n_items);
    n_groups = static_cast<int>(g.n_digits);
    n_blocks = static_cast<int>(g.n_blocks);
    n_fine = static_cast<int>(g.n_fine);
    if (4 * lane <= max_digit) {
#pragma unroll
      for (int j = 0; j < 4; ++j) s_base[wave][4 * lane + j] = uint2{g.off[j] | (g.pre[j] << 16), g.blk[j] | (g.fblk[j] << 16)};
    }
    plan_stamp(m, 5);
#pragma unroll
    for (int e = 0; e < E; ++e) {
      if (!((live[e] >> lane) & 1ull)) continue;
      const int i = (first + e) * 64 + lane;
      const uint2 bs = s_base[wave][dig[e]];
      const int pos = static_cast<int>((bs.x >> 16) + rank[e]);  // inside the adapter's group
      perm[static_cast<int>(bs.x & 0xffffu) + pos] = i;
      const int q = static_cast<int>(bs.y & 0xffffu) + (pos >> bt_log2);
      if (q < block_cap) bperm[static_cast<int64_t>(q) * kBlockTokens + (pos & (bt - 1))] = i;
      if (has_fine) {
        const int f = static_cast<int>(bs.y >> 16) + pos / kFineTokens;
        if (f < block_cap) fine.bperm[static_cast<int64_t>(f) * kBlockTokens + pos % kFineTokens] = i;
      }
    }
    plan_stamp(m, 6);
    if constexpr (E == 1) {
      // Block tables: wave w writes the blocks w / 4, w / 4 + NW / 4, ... of
      // the digits 4 * lane + w % 4.
      const int j = wave & 3;
      const auto pick = [&](const uint32_t(&v)[4]) {
        return static_cast<int>(j == 0 ? v[0] : j == 1 ? v[1] : j == 2 ? v[2] : v[3]);
      };
      const int id = 4 * lane + j;
      const int tot = pick(g.tot), off = pick(g.off), blk0 = pick(g.blk), fblk0 = pick(g.fblk);
      const EntryWords en = read_entry(m, id, want_entry && tot > 0);
      for (int k = wave >> 2; k << bt_log2 < tot; k += NW / 4)
        if (blk0 + k < block_cap) put_block(blocks, bentries, blk0 + k, id, off + k * bt, min(bt, tot - k * bt), en);
      if (has_fine) {
        for (int k = wave >> 2; k * kFineTokens < tot; k += NW / 4)
          if (fblk0 + k < block_cap)
            put_block(fine.blocks, fine.bentries, fblk0 + k, id, off + k * kFineTokens,
                      min(kFineTokens, tot - k * kFineTokens), en);
      }
    } else {
      // Larger plans: a thread per block finds its digit in the wave's bases
      // (one adapter may own every block).
      const auto table = [&](Block* out, Entry* oent, int n, int size_log2, int half) {
        for (int q = tid; q < min(n, block_cap); q += NT) {
          int lo = 0, hi = max_digit;
          while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (static_cast<int>((s_base[wave][mid].y >> half) & 0xffffu) <= q) {
              lo = mid;
            } else {
              hi = mid - 1;
            }
          }
          const uint2 bs = s_base[wave][lo];
          const int k = q - static_cast<int>((bs.y >> half) & 0xffffu);
          const int at = static_cast<int>(bs.x & 0xffffu) + (k << size_log2);
          const int end = lo < max_digit ? static_cast<int>(s_base[wave][lo + 1].x & 0xffffu) : n_tok;
          put_block(out, oent, q, lo, at, min(1 << size_log2, end - at), read_entry(m, lo, want_entry));
        }
      };
      table(blocks, bentries, n_blocks, bt_log2, 0);
      if (has_fine) table(fine.blocks, fine.bentries, n_fine, 4, 16);
    }
  } else {
    // Larger ids: the counting pass again over the next 8 bits of the order
    // so far, then the groups' blocks from the sorted order the way the
    // segments came from the token order.
    n_tok = 0;
    int cur = 0;
    uint64_t lv[E];
    uint32_t tok[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
      lv[e] = live[e];
      tok[e] = static_cast<uint32_t>((first + e) * 64 + lane);
    }
    for (int shift = 0;; shift += 8) {
      const Digits g = scan_digits<NW>(s_cnt, wave, kDigits - 1, bt_log2, false);
      n_tok = static_cast<int>(g.n_items);
#pragma unroll
      for (int j = 0; j < 4; ++j) s_base[wave][4 * lane + j].x = g.off[j] + g.pre[j];
#pragma unroll
      for (int e = 0; e < E; ++e)
        if ((lv[e] >> lane) & 1ull) s_ord[cur][s_base[wave][dig[e]].x + rank[e]] = static_cast<uint16_t>(tok[e]);
      lds_barrier();
      if (shift + 8 >= 32 || (kmax >> (shift + 8)) == 0) break;
#pragma unroll
      for (int j = 0; j < kDigits / 64; ++j) s_cnt[wave][lane + 64 * j] = 0u;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int q = (first + e) * 64 + lane;
        lv[e] = __ballot(q < n_tok);
        tok[e] = q < n_tok ? s_ord[cur][q] : 0u;
        dig[e] = (s_key[tok[e]] >> (shift + 8)) & (kDigits - 1);
      }
      rank_digits<E>(dig, lv, 8, s_cnt[wave], rank);
      cur ^= 1;
      lds_barrier();
    }
    plan_stamp(m, 5);
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int q = (first + e) * 64 + lane;
      lv[e] = __ballot(q < n_tok);
      tok[e] = q < n_tok ? s_ord[cur][q] : 0u;
      dig[e] = s_key[tok[e]];
      uint32_t prev = __shfl_up(dig[e], 1, 64);
      if (lane == 0 && q > 0 && q < n_tok) prev = s_key[s_ord[cur][q - 1]];
      start[e] = __ballot(q < n_tok && (q == 0 || prev != dig[e]));
      if (lane == 0) s_start[first + e] = start[e];
    }
    lds_barrier();
    n_groups = static_cast<int>(count_words<NWORDS>(s_start, first) >> 16);
    mark_pieces<E>(start, lv, first, last_start_before<NWORDS>(s_start, first), bt, piece, rs);
    uint64_t fpiece[E];
    if (has_fine) {
      int unused[E];
      mark_pieces<E>(start, lv, first, last_start_before<NWORDS>(s_start, first), kFineTokens, fpiece, unused);
    }
#pragma unroll
    for (int e = 0; e < E; ++e) {
      if (lane != 0) continue;
      s_piece[first + e] = piece[e];
      if (has_fine) s_fpiece[first + e] = fpiece[e];
    }
    lds_barrier();
    const auto table = [&](const uint64_t(&pc)[E], const uint64_t* s_pc, int size, Block* out, int32_t* operm,
                           Entry* oent) {
      const uint32_t nblk = count_words<NWORDS>(s_pc, first);
      int blk0 = static_cast<int>(nblk & 0xffffu);
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int w = first + e;
        const int q = w * 64 + lane;
        const uint64_t le = (lanes_below(lane) << 1) | 1ull;
        const int b = blk0 + __popcll(pc[e] & le) - 1;  // this position's block
        blk0 += __popcll(pc[e]);
        if (q >= n_tok || b >= block_cap) continue;
        operm[static_cast<int64_t>(b) * kBlockTokens + ((q - rs[e]) & (size - 1))] = static_cast<int>(tok[e]);
        if (!((pc[e] >> lane) & 1ull)) continue;
        const uint64_t up = ((start[e] | pc[e]) >> lane) >> 1;
        int end = n_tok;
        if (up != 0) {
          end = q + 1 + __builtin_ctzll(up);
        } else if (w + 1 < NWORDS) {
          const uint64_t nx = s_start[w + 1] | s_pc[w + 1];
          if (nx != 0) end = (w + 1) * 64 + __builtin_ctzll(nx);
        }
        const int id = static_cast<int>(dig[e]);
        put_block(out, oent, b, id, q, end - q, read_entry(m, id, want_entry));
      }
      return static_cast<int>(nblk >> 16);
    };
    n_blocks = table(piece, s_piece, bt, blocks, bperm, bentries);
    n_fine = has_fine ? table(fpiece, s_fpiece, kFineTokens, fine.blocks, fine.bperm, fine.bentries) : n_blocks;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int q = (first + e) * 64 + lane;
      if (q < n_tok) perm[q] = static_cast<int>(tok[e]);
    }
    plan_stamp(m, 6);
  }

  if (tid == 0) {
    header[kHdrNumSegments] = static_cast<uint32_t>(n_segs);
    header[kHdrNumBlocks] = static_cast<uint32_t>(min(n_blocks, block_cap));
    header[kHdrNumFine] = static_cast<uint32_t>(min(n_fine, block_cap));
    header[kHdrNumGroups] = static_cast<uint32_t>(n_groups);
    header[kHdrNumValid] = static_cast<uint32_t>(n_tok);
    header[kHdrT] = static_cast<uint32_t>(T);
    header[kHdrBlockTokens] = static_cast<uint32_t>(bt);
    header[kHdrPlanVer] = bentries != nullptr ? table_ver : ~table_ver;
  }
  plan_stamp(m, 7);
}

}  // namespace

// Host launcher: the smallest capacity variant that holds T.
hipError_t launch_plan(const void* idx, int idx_is_int64, int T, uint32_t* header, Segment* segments, Block* blocks,
                       int32_t* perm, int32_t* bperm, Entry* bentries, const FinePlan* fine, int seg_cap, int block_cap,
                       int bt, const Maint* m, hipStream_t stream) {
  if (T < 0 || bt < 1 || bt > kBlockTokens || (bt & (bt - 1)) != 0) return hipErrorInvalidValue;
  Maint mm{};
  if (m != nullptr) mm = *m;
  FinePlan ff{};
  if (fine != nullptr && bt > kFineTokens) ff = *fine;
  // Both tables carry entries, or neither.
  if (ff.blocks != nullptr && (ff.bperm == nullptr || (ff.bentries == nullptr) != (bentries == nullptr)))
    return hipErrorInvalidValue;
  // Publications are applied by threads 0..n_pubs-1 of the smallest variant.
  if (mm.n_pubs < 0 || mm.n_pubs > 256) return hipErrorInvalidValue;
  // The smallest capacity that holds T: a wave's words are consecutive, so a
  // larger one would leave waves idle while others work their words in turn.
  auto run = [&](auto nt, auto e) {
    plan_kernel<decltype(nt)::value, decltype(e)::value><<<1, decltype(nt)::value, 0, stream>>>(
        idx, idx_is_int64, T, header, segments, blocks, perm, bperm, bentries, ff, seg_cap, block_cap, bt, mm);
  };
  if (T <= 256) {
    run(std::integral_constant<int, 256>{}, std::integral_constant<int, 1>{});
  } else if (T <= 1024) {
    run(std::integral_constant<int, 1024>{}, std::integral_constant<int, 1>{});
  } else if (T <= 2048) {
    run(std::integral_constant<int, 1024>{}, std::integral_constant<int, 2>{});
  } else if (T <= 4096) {
    run(std::integral_constant<int, 1024>{}, std::integral_constant<int, 4>{});
  } else if (T <= kPlanMaxTokens) {
    run(std::integral_constant<int, 1024>{}, std::integral_constant<int, 8>{});
  } else {
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_maintain(uint32_t* header, const Maint& m, hipStream_t stream) {
  if (m.n_pubs < 0 || m.n_pubs > 256) return hipErrorInvalidValue;
  maintain_kernel<<<1, 256, 0, stream>>>(header, m);
  return hipGetLastError();
}

hipError_t launch_entry_writes(const EntryWrites& w, hipStream_t stream) {
  if (w.n < 0 || w.n > kMaxEntryWrites || w.n_retire < 0 || w.n_retire > kMaxEntryWrites) return hipErrorInvalidValue;
  entry_writes_kernel<<<1, 64, 0, stream>>>(w);
  return hipGetLastError();
}

hipError_t launch_stage_copies(const StageJobs& jobs, hipStream_t stream) {
  if (jobs.n < 0 || jobs.n > kMaxStageJobs) return hipErrorInvalidValue;
  for (int j = 0; j < jobs.n; ++j)
    if (jobs.job[j].pub == nullptr || jobs.job[j].a_bytes % 16 != 0 || jobs.job[j].b_bytes % 16 != 0)
      return hipErrorInvalidValue;
  if (jobs.n == 0) return hipSuccess;
  stage_copy_kernel<<<jobs.n * kStageWorkgroups, 256, 0, stream>>>(jobs);
  return hipGetLastError();
}

}  // namespace wp
