// Slot allocator of the KV pool for gfx950: the device-side searches and reference counting that the reference
// does with torch.nonzero over the whole pool on every call (loongserve/common/longserve_mem_manager.py:32-88).
//   take the first `need` free slots, in ascending order          (alloc, :37-40)
//   find the first run of `need` consecutive free slots           (alloc_contiguous, :50-55)
//   add / drop one reference on a list of slots and count          (add_refs :73-79, decrease_refs :82-88)
// `mem_state` is int32 per slot, 0 = free.  All of it is integer work on a few MB, bound by launch latency and
// by one pass over the state array; two short launches replace the reference's nonzero / slice / compare chains (three for
// pools of more than 8 million slots, one for small allocs from up to 65536), one for the reference counts of up to 4096 slots.
#include "common.hip.h"

namespace lsattn {

constexpr int kPoolThreads = 256;
constexpr int kPoolPieces = 4;                                 // 16-byte pieces per thread
constexpr int kPoolBlockSlots = kPoolThreads * 4 * kPoolPieces;  // 4096 slots per workgroup
constexpr int kPoolWaves = kPoolThreads / 64;

typedef int i32x4 __attribute__((ext_vector_type(4)));

// Slots of one workgroup, coalesced: piece j of thread t covers slots base + 1024 j + 4 t .. + 3; the scan order of
// the (piece, thread) pairs is j-major, which is ascending slot order.  Slots past `size` read as in use.
struct PoolTile {
  int64_t base;
  i32x4 s[kPoolPieces];
  __device__ __forceinline__ void load(const int32_t* __restrict__ state, int64_t size) {
    base = (int64_t)blockIdx.x * kPoolBlockSlots;
#pragma unroll
    for (int j = 0; j < kPoolPieces; j++) {
      const int64_t p = base + j * (kPoolThreads * 4) + threadIdx.x * 4;
      if (p + 3 < size) {
        s[j] = *(const i32x4*)(state + p);
      } else {
#pragma unroll
        for (int e = 0; e < 4; e++) s[j][e] = p + e < size ? state[p + e] : 1;
      }
    }
  }
  __device__ __forceinline__ int64_t pos(int j, int e) const { return base + j * (kPoolThreads * 4) + threadIdx.x * 4 + e; }
};

__device__ __forceinline__ int wave_incl_sum(int v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int o = __shfl_up(v, d);
    if (lane >= d) v += o;
  }
  return v;
}
__device__ __forceinline__ int64_t wave_incl_max(int64_t v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int64_t o = __shfl_up(v, d);
    if (lane >= d) v = o > v ? o : v;
  }
  return v;
}

// ---------------------------------------------------------------------------------------------------
// Pass 1: per workgroup of 4096 slots, the number of free slots and the position of the last slot in use (-1: none).
// ---------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(kPoolThreads) void pool_summarise_kernel(const int32_t* __restrict__ state, int64_t size,
                                                                      int32_t* __restrict__ blk_free,
                                                                      int64_t* __restrict__ blk_last_used,
                                                                      int64_t* __restrict__ first_fit) {
  if (first_fit && blockIdx.x == 0 && threadIdx.x == 0) *first_fit = -1;  // "no run", until pass 3 finds one
  __shared__ int sh_cnt[kPoolWaves];
  __shared__ int64_t sh_last[kPoolWaves];
  PoolTile t;
  t.load(state, size);
  int cnt = 0;
  int64_t last = -1;
#pragma unroll
  for (int j = 0; j < kPoolPieces; j++)
#pragma unroll
    for (int e = 0; e < 4; e++) {
      cnt += t.s[j][e] == 0;
      if (t.s[j][e] != 0 && t.pos(j, e) < size) last = t.pos(j, e);  // ascending within the thread's pieces
    }
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) {
    cnt += __shfl_xor(cnt, d);
    const int64_t o = __shfl_xor(last, d);
    last = o > last ? o : last;
  }
  if ((threadIdx.x & 63) == 0) {
    sh_cnt[threadIdx.x >> 6] = cnt;
    sh_last[threadIdx.x >> 6] = last;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int c = 0;
    int64_t l = -1;
    for (int w = 0; w < kPoolWaves; w++) {
      c += sh_cnt[w];
      l = sh_last[w] > l ? sh_last[w] : l;
    }
    blk_free[blockIdx.x] = c;
    blk_last_used[blockIdx.x] = l;
  }
}

// ---------------------------------------------------------------------------------------------------
// Pass 2 (one workgroup), for pools of more than kPoolDirectBlocks workgroups of pass 1: exclusive prefix sum of their
// free counts and exclusive prefix maximum of their last-used positions.  Smaller pools do without it: there each workgroup of
// pass 3 adds up the summaries in front of it itself (at most eight per thread, from the L2), which costs less than
// a launch: alloc of 64 slots of 2.5 million 10 -> 6 us on the device.
// ---------------------------------------------------------------------------------------------------
constexpr int64_t kPoolDirectBlocks = 2048;
__global__ __launch_bounds__(1024) void pool_scan_summaries_kernel(const int32_t* __restrict__ blk_free,
                                                                   const int64_t* __restrict__ blk_last_used, int64_t nb,
                                                                   int64_t* __restrict__ free_before,
                                                                   int64_t* __restrict__ last_used_before) {
  __shared__ int64_t sh_sum[1024];
  __shared__ int64_t sh_max[1024];
  const int64_t per = (nb + 1023) / 1024;
  const int64_t b0 = (int64_t)threadIdx.x * per, b1 = b0 + per < nb ? b0 + per : nb;
  int64_t sum = 0, mx = -1;
  for (int64_t b = b0; b < b1; b++) {
    sum += blk_free[b];
    mx = blk_last_used[b] > mx ? blk_last_used[b] : mx;
  }
  sh_sum[threadIdx.x] = sum;
  sh_max[threadIdx.x] = mx;
  __syncthreads();
  // Hillis-Steele over the 1024 thread totals
  for (int d = 1; d < 1024; d <<= 1) {
    int64_t s = 0, m = -1;
    if ((int)threadIdx.x >= d) {
      s = sh_sum[threadIdx.x - d];
      m = sh_max[threadIdx.x - d];
    }
    __syncthreads();
    sh_sum[threadIdx.x] += s;
    sh_max[threadIdx.x] = m > sh_max[threadIdx.x] ? m : sh_max[threadIdx.x];
    __syncthreads();
  }
  int64_t run_sum = threadIdx.x ? sh_sum[threadIdx.x - 1] : 0;
  int64_t run_max = threadIdx.x ? sh_max[threadIdx.x - 1] : -1;
  for (int64_t b = b0; b < b1; b++) {
    free_before[b] = run_sum;
    last_used_before[b] = run_max;
    run_sum += blk_free[b];
    run_max = blk_last_used[b] > run_max ? blk_last_used[b] : run_max;
  }
}

// The sum of blk_free (MAX: the maximum of blk_last_used) over the workgroups in front of this one, by all its threads.
template <bool MAX>
__device__ __forceinline__ int64_t pool_before(const int32_t* __restrict__ blk_free, const int64_t* __restrict__ blk_last_used) {
  __shared__ int64_t sh[kPoolWaves];
  int64_t v = MAX ? -1 : 0;
  for (int64_t b = threadIdx.x; b < blockIdx.x; b += kPoolThreads) {
    if (MAX) v = blk_last_used[b] > v ? blk_last_used[b] : v;
    else v += blk_free[b];
  }
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) {
    const int64_t o = __shfl_xor(v, d);
    v = MAX ? (o > v ? o : v) : v + o;
  }
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  v = sh[0];
#pragma unroll
  for (int w = 1; w < kPoolWaves; w++) v = MAX ? (sh[w] > v ? sh[w] : v) : v + sh[w];
  return v;
}

// ---------------------------------------------------------------------------------------------------
// Pass 3 of alloc: the free slot with rank r < need (ranks count free slots in ascending slot order) is written to
// out_index[r] and marked in use.  Workgroups whose first rank is already >= need leave at once.  When fewer than `need` slots
// are free, the last workgroup fills the rest of out_index with -1, so the result is defined.
// ---------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(kPoolThreads) void pool_take_kernel(int32_t* __restrict__ state, int64_t size,
                                                                 const int64_t* __restrict__ free_before,
                                                                 const int32_t* __restrict__ blk_free, int64_t need,
                                                                 int64_t* __restrict__ out_index, int64_t* __restrict__ cells) {
  __shared__ int sh[kPoolPieces][kPoolWaves];
  PoolTile t;
  if (!free_before) t.load(state, size);  // (asked for beside the summaries)
  const int64_t first_rank = free_before ? free_before[blockIdx.x] : pool_before<false>(blk_free, nullptr);
  if (blockIdx.x == gridDim.x - 1) {
    const int64_t total = first_rank + blk_free[blockIdx.x];
    if (threadIdx.x == 0) cells[0] = total;
    for (int64_t i = total + threadIdx.x; i < need; i += kPoolThreads) out_index[i] = -1;
  }
  if (first_rank >= need) return;
  // (behind pass 2 by those that take something only: 64 of 42 million slots, with the free after it, 86 us when all read, 66 so)
  if (free_before) t.load(state, size);
  const int wave = threadIdx.x >> 6;
  int incl[kPoolPieces], mine[kPoolPieces];
#pragma unroll
  for (int j = 0; j < kPoolPieces; j++) {
    mine[j] = (t.s[j][0] == 0) + (t.s[j][1] == 0) + (t.s[j][2] == 0) + (t.s[j][3] == 0);
    incl[j] = wave_incl_sum(mine[j]);
    if ((threadIdx.x & 63) == 63) sh[j][wave] = incl[j];
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kPoolPieces; j++) {
    int before = 0;  // free slots of the (piece, wave) pairs that come earlier in slot order
    for (int jj = 0; jj < kPoolPieces; jj++)
      for (int w = 0; w < kPoolWaves; w++)
        if (jj < j || (jj == j && w < wave)) before += sh[jj][w];
    int64_t rank = first_rank + before + incl[j] - mine[j];
    if (rank >= need) continue;
    i32x4 ns = t.s[j];
    bool any = false;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      if (t.s[j][e] == 0 && rank < need) {
        out_index[rank++] = t.pos(j, e);
        ns[e] = 1;
        any = true;
      }
    }
    if (any) {
      const int64_t p = t.pos(j, 0);
      if (p + 3 < size) {
        *(i32x4*)(state + p) = ns;
      } else {
#pragma unroll
        for (int e = 0; e < 4; e++)
          if (p + e < size) state[p + e] = ns[e];
      }
    }
  }
}

// ---------------------------------------------------------------------------------------------------
// alloc of a few slots of a pool of up to 65536 in one launch (pool_is_one_group): one workgroup walks it from the front, kScanSlots at a time with the next
// two lots under way, and stops behind the last slot it takes.  Every wave has 1024 slots in a row of a lot, so that ranks need one count
// per wave.  Bound by the latency of its first load and, past that, by issue: 0.8 us for a lot without a free slot, 1.5 for one that has some.
// The host has one launch less, 3.4 us of a call (15.6 -> 12.2 with a fill in front).  Device time, the two launches above | this one, by where the free slots
// lie (at the front, every second one, as many as are asked for and scattered over the whole pool, those at its end):
//   24 of 65536 6.8 | 4.9, 6.2 | 4.3, 7.1 | 8.6, 7.2 | 7.1     64 of 65536 6.7 | 4.9, 6.4 | 4.4, 7.2 | 9.5, 7.2 | 7.1    256 of 65536 6.6 | 4.9, 6.4 | 4.4, 7.3 | 11.7, 7.2 | 7.1
//   64 of 32768 6.5 | 4.0, 6.2 | 4.6, 7.2 | 6.8, 7.2 | 5.2     256 of 32768 6.5 | 4.1, 6.3 | 4.6, 7.3 | 7.8, 7.3 | 5.3   1024 of 32768 6.6 | 4.7, 6.5 | 4.8, 7.5 | 9.1, 7.2 | 5.9
//   64 of 16384 6.3 | 3.9, 6.2 | 4.4, 6.9 | 4.8, 6.8 | 4.1     1024 of 16384 6.4 | 4.5, 6.5 | 4.7, 7.2 | 6.0, 7.0 | 4.7  4096 of 16384 7.2 | 4.6, 7.0 | 4.8, 7.2 | 6.0, 7.2 | 4.8
// So pools of one lot whatever is asked for (all 16384 of 16384 7.3 | 7.7), of two for up to 256 slots, and of four for up to 64: a full pool's few
// scattered slots then cost the device 2.3 us more at most, less than the host saves, and the other states up to 2.5 less.  Past four lots
// the walk to the end alone takes as long as the two launches, which read the pool on all CUs.
// (All lots read and counted before the first is taken from, so that no store stands between them: slower everywhere, 4.3 -> 7.1 and 8.6 -> 10.2.)
// ---------------------------------------------------------------------------------------------------
constexpr int kScanPieces = 4, kScanSlots = 1024 * 4 * kScanPieces;
constexpr bool pool_is_one_group(int64_t size, int64_t need) { return size <= kScanSlots || (size <= 2 * kScanSlots ? need <= 256 : size <= 4 * kScanSlots && need <= 64); }
__global__ __launch_bounds__(1024) void pool_alloc_one_group_kernel(int32_t* __restrict__ state, int size, int64_t need, int64_t* __restrict__ out_index,
                                                                    int64_t* __restrict__ cells) {
  __shared__ __attribute__((aligned(16))) int sh[2][16];  // (two sets in turn: one barrier per lot)
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  struct Lot {
    i32x4 s[kScanPieces];
  };
  auto pos = [&](int base, int j) { return base + wave * (256 * kScanPieces) + j * 256 + lane * 4; };
  auto load = [&](int base) {  // (slots past the end read as in use)
    Lot l;
#pragma unroll
    for (int j = 0; j < kScanPieces; j++) {
      const int p = pos(base, j);
      if (p + 3 < size) {
        l.s[j] = *(const i32x4*)(state + p);
      } else {
#pragma unroll
        for (int e = 0; e < 4; e++) l.s[j][e] = p + e < size ? state[p + e] : 1;
      }
    }
    return l;
  };
  const int wanted = need < size ? (int)need : size;
  int taken = 0;  // free slots in front of the lot: the rank of its first one
  int set = 0;
  // takes what is free of the lot at `base`; true if the walk goes on
  auto take = [&](const Lot& cur, int base) __attribute__((always_inline)) {
    set ^= 1;
    int mine = 0;  // of this wave
#pragma unroll
    for (int j = 0; j < kScanPieces; j++)
#pragma unroll
      for (int e = 0; e < 4; e++) mine += __builtin_popcountll(__builtin_amdgcn_ballot_w64(cur.s[j][e] == 0));
    if (lane == 0) sh[set][wave] = mine;
    __syncthreads();
    int before = 0, all = 0;  // of the waves in front, of all
#pragma unroll
    for (int w = 0; w < 16; w += 4) {
      const i32x4 n = *(const i32x4*)&sh[set][w];
#pragma unroll
      for (int e = 0; e < 4; e++) {
        before += w + e < wave ? n[e] : 0;
        all += n[e];
      }
    }
    int first = taken + __builtin_amdgcn_readfirstlane(before);  // the rank of the wave's first free slot
    taken += __builtin_amdgcn_readfirstlane(all);
    if (mine > 0 && first < wanted) {  // (wave-uniform)
#pragma unroll
      for (int j = 0; j < kScanPieces; j++) {
        int below = 0, piece = 0;
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const uint64_t lanes = __builtin_amdgcn_ballot_w64(cur.s[j][e] == 0);
          below += __builtin_amdgcn_mbcnt_hi((uint32_t)(lanes >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)lanes, 0u));
          piece += __builtin_popcountll(lanes);
        }
        int rank = first + below;
        first += piece;
        if (piece == 0) continue;
        i32x4 ns = cur.s[j];
        bool any = false;
        const int p = pos(base, j);
#pragma unroll
        for (int e = 0; e < 4; e++)
          if (cur.s[j][e] == 0 && rank < wanted) {
            out_index[rank++] = p + e;
            ns[e] = 1;
            any = true;
          }
        if (any) {
          if (p + 3 < size) {
            *(i32x4*)(state + p) = ns;
          } else {
#pragma unroll
            for (int e = 0; e < 4; e++)
              if (p + e < size) state[p + e] = ns[e];
          }
        }
      }
    }
    return taken < wanted && base + kScanSlots < size;
  };
  Lot a = load(0), b = load(kScanSlots), c = load(2 * kScanSlots);
  for (int base = 0; need > 0; base += 3 * kScanSlots) {
    if (!take(a, base)) break;
    a = load(base + 3 * kScanSlots);
    if (!take(b, base + kScanSlots)) break;
    b = load(base + 4 * kScanSlots);
    if (!take(c, base + 2 * kScanSlots)) break;
    c = load(base + 5 * kScanSlots);
  }
  for (int64_t i = (int64_t)taken + threadIdx.x; i < need; i += 1024) out_index[i] = -1;
  if (threadIdx.x == 0) cells[0] = taken;
}

// ---------------------------------------------------------------------------------------------------
// Pass 3 of alloc_contiguous: with u(p) = position of the last slot in use at or before p, a run of free slots
// reaches length `need` exactly at the one p with p - u(p) == need, and starts at p - need + 1.  The smallest
// such start over the pool is the reference's can_use_index[...][0] (longserve_mem_manager.py:52-55).  The minimum is
// taken on the unsigned value, so the preset -1 stands for "none" and loses to every real start.
// ---------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(kPoolThreads) void pool_first_fit_kernel(const int32_t* __restrict__ state, int64_t size,
                                                                      const int64_t* __restrict__ last_used_before,
                                                                      const int64_t* __restrict__ blk_last_used,
                                                                      int64_t need, int64_t* __restrict__ first_fit) {
  __shared__ int64_t sh[kPoolPieces][kPoolWaves];
  PoolTile t;
  t.load(state, size);
  const int64_t u_before = last_used_before ? last_used_before[blockIdx.x] : pool_before<true>(nullptr, blk_last_used);
  const int wave = threadIdx.x >> 6;
  int64_t own[kPoolPieces], incl[kPoolPieces];
#pragma unroll
  for (int j = 0; j < kPoolPieces; j++) {
    own[j] = -1;
#pragma unroll
    for (int e = 0; e < 4; e++)
      if (t.s[j][e] != 0) own[j] = t.pos(j, e);  // slots past the end count as in use: runs stop there
    incl[j] = wave_incl_max(own[j]);
    if ((threadIdx.x & 63) == 63) sh[j][wave] = incl[j];
  }
  __syncthreads();
  int64_t best = INT64_MAX;
#pragma unroll
  for (int j = 0; j < kPoolPieces; j++) {
    int64_t u = u_before;
    for (int jj = 0; jj < kPoolPieces; jj++)
      for (int w = 0; w < kPoolWaves; w++)
        if (jj < j || (jj == j && w < wave)) u = sh[jj][w] > u ? sh[jj][w] : u;
    const int64_t prev = __shfl_up(incl[j], 1);  // lanes before this one in the wave
    if ((threadIdx.x & 63) != 0) u = prev > u ? prev : u;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int64_t p = t.pos(j, e);
      if (t.s[j][e] != 0) {
        u = p;
      } else if (p - u == need && p - need + 1 < best) {
        best = p - need + 1;
      }
    }
  }
  if (best != INT64_MAX) atomicMin((unsigned long long*)first_fit, (unsigned long long)best);
}

// ---------------------------------------------------------------------------------------------------
// Reference counting on a list of slots.  torch's `mem_state[index] += d` gathers, adds and writes back, so a slot
// named k times still changes by d once; both kernels keep that: the first reads every old value, the second
// writes old + d.  counted[0] = entries whose slot is non-zero before (+1: has_used_tokens, :75) or after
// (-1: used_tokens, :85) the update; counted[1] = entries outside the pool (skipped).  Negative entries wrap
// once, as in torch indexing.
// ---------------------------------------------------------------------------------------------------
// The counts may be asked for in pinned host memory, where the caller looks for them while the kernel ends: whole words, written
// through to the system.
__device__ __forceinline__ void put_counts(int64_t* counted, int64_t used, int64_t bad) {
  __hip_atomic_store(counted, used, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  __hip_atomic_store(counted + 1, bad, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Up to kRefsOneGroup entries by one workgroup: every old value is in a register before the barrier, every new one is
// written behind it.  (bound by its three dependent loads and two stores: 3 us, where the two launches below take 4 and a gap)
constexpr int kRefsPer = 4;
constexpr int64_t kRefsOneGroup = 1024 * kRefsPer;
static_assert(kRefsOneGroup == LSATTN_POOL_REFS_ORDERED, "counts behind the state: the one-workgroup launch");
__global__ __launch_bounds__(1024) void pool_refs_small_kernel(int32_t* __restrict__ state, int64_t size,
                                                               const int64_t* __restrict__ index, int64_t n, int delta,
                                                               int64_t* __restrict__ counted) {
  __shared__ int sh[2][16];
  int64_t slot[kRefsPer];
  int32_t old[kRefsPer];
#pragma unroll
  for (int k = 0; k < kRefsPer; k++) {
    const int64_t i = threadIdx.x + 1024 * k;
    slot[k] = i < n ? index[i] : 0;
  }
  int used = 0, bad = 0;
#pragma unroll
  for (int k = 0; k < kRefsPer; k++) {
    const bool listed = threadIdx.x + 1024 * k < n;
    if (slot[k] < 0) slot[k] += size;
    const bool inside = slot[k] >= 0 && slot[k] < size;
    bad += listed && !inside;
    if (!listed || !inside) slot[k] = -1;
    old[k] = slot[k] >= 0 ? state[slot[k]] : 0;
  }
#pragma unroll
  for (int k = 0; k < kRefsPer; k++) used += slot[k] >= 0 && (delta > 0 ? old[k] : old[k] + delta) != 0;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kRefsPer; k++)
    if (slot[k] >= 0) __hip_atomic_store(state + slot[k], old[k] + delta, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  // Whoever sees the counts (the host, which may go on to another stream) finds the state written: the stores go through to
  // memory and have arrived in front of the barrier below (a fence of the device writes the whole L2 back, 3 us more).
  // (from inline assembly that names memory: no store may be moved past it, as past the builtin, which names none)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) {
    used += __shfl_xor(used, d);
    bad += __shfl_xor(bad, d);
  }
  if ((threadIdx.x & 63) == 0) {
    sh[0][threadIdx.x >> 6] = used;
    sh[1][threadIdx.x >> 6] = bad;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    used = bad = 0;
    for (int w = 0; w < 16; w++) {
      used += sh[0][w];
      bad += sh[1][w];
    }
    put_counts(counted, used, bad);
  }
}

__global__ __launch_bounds__(256) void pool_refs_gather_kernel(const int32_t* __restrict__ state, int64_t size,
                                                               const int64_t* __restrict__ index, int64_t n, int delta,
                                                               int32_t* __restrict__ old_state, int64_t* __restrict__ blk_counts) {
  __shared__ int sh[2][4];
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  int used = 0, bad = 0;
  if (i < n) {
    int64_t s = index[i];
    if (s < 0) s += size;
    if (s < 0 || s >= size) {
      bad = 1;
    } else {
      const int32_t o = state[s];
      old_state[i] = o;
      used = (delta > 0 ? o : o + delta) != 0;
    }
  }
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) {
    used += __shfl_xor(used, d);
    bad += __shfl_xor(bad, d);
  }
  if ((threadIdx.x & 63) == 0) {
    sh[0][threadIdx.x >> 6] = used;
    sh[1][threadIdx.x >> 6] = bad;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    blk_counts[2 * blockIdx.x] = sh[0][0] + sh[0][1] + sh[0][2] + sh[0][3];
    blk_counts[2 * blockIdx.x + 1] = sh[1][0] + sh[1][1] + sh[1][2] + sh[1][3];
  }
}

__global__ __launch_bounds__(256) void pool_refs_apply_kernel(int32_t* __restrict__ state, int64_t size,
                                                              const int64_t* __restrict__ index, int64_t n, int delta,
                                                              const int32_t* __restrict__ old_state,
                                                              const int64_t* __restrict__ blk_counts, int64_t nblk,
                                                              int64_t* __restrict__ counted) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) {
    int64_t s = index[i];
    if (s < 0) s += size;
    if (s >= 0 && s < size) state[s] = old_state[i] + delta;
  }
  if (blockIdx.x == 0) {  // the per-workgroup counts are complete: the gather launch precedes this one on the stream
    __shared__ int64_t sh[2][4];
    int64_t used = 0, bad = 0;
    for (int64_t b = threadIdx.x; b < nblk; b += 256) {
      used += blk_counts[2 * b];
      bad += blk_counts[2 * b + 1];
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
      used += __shfl_xor(used, d);
      bad += __shfl_xor(bad, d);
    }
    if ((threadIdx.x & 63) == 0) {
      sh[0][threadIdx.x >> 6] = used;
      sh[1][threadIdx.x >> 6] = bad;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      put_counts(counted, sh[0][0] + sh[0][1] + sh[0][2] + sh[0][3], sh[1][0] + sh[1][1] + sh[1][2] + sh[1][3]);
    }
  }
}

// Workspace layout of the searches: int64 cells[2] (cells[0] = free slots an alloc has come across: all of the pool unless the one-workgroup launch had enough before its end) | int64 free_before[nb] | int64 last_used_before[nb] |
// int64 blk_last_used[nb] | int32 blk_free[nb]
struct PoolWorkspace {
  int64_t nb;
  int64_t *cells, *free_before, *last_used_before, *blk_last_used;
  int32_t* blk_free;
};
inline int64_t pool_blocks(int64_t size) { return (size + kPoolBlockSlots - 1) / kPoolBlockSlots; }
inline size_t pool_search_bytes(int64_t size) { return (size_t)(16 + pool_blocks(size) * 28 + 15) & ~(size_t)15; }
inline PoolWorkspace pool_carve(void* ws, int64_t size) {
  PoolWorkspace w;
  w.nb = pool_blocks(size);
  w.cells = (int64_t*)ws;
  w.free_before = w.cells + 2;
  w.last_used_before = w.free_before + w.nb;
  w.blk_last_used = w.last_used_before + w.nb;
  w.blk_free = (int32_t*)(w.blk_last_used + w.nb);
  return w;
}
inline int64_t refs_blocks(int64_t n) { return (n + 255) / 256; }

}  // namespace lsattn

using namespace lsattn;

extern "C" size_t lsattn_pool_search_workspace_bytes(int64_t pool_size) { return pool_size > 0 ? pool_search_bytes(pool_size) : 0; }

extern "C" size_t lsattn_pool_refs_workspace_bytes(int64_t n) {
  return n > 0 ? (size_t)(refs_blocks(n) * 16 + ((n * 4 + 15) & ~(int64_t)15)) : 0;
}

static int pool_search_checks(const void* mem_state, int64_t size, int64_t need, const void* ws, size_t ws_bytes) {
  if (!mem_state || !ws || size <= 0 || need < 0) return LSATTN_ERR_INVALID_ARG;
  if (((uintptr_t)mem_state & 15) || ((uintptr_t)ws & 15)) return LSATTN_ERR_INVALID_ARG;
  if (ws_bytes < pool_search_bytes(size)) return LSATTN_ERR_WORKSPACE;
  if (pool_blocks(size) > 0x7fffffff) return LSATTN_ERR_INVALID_ARG;
  return LSATTN_OK;
}

// Passes 1 and, for a large pool, 2; true if pass 2 has run.
static bool pool_summarise(const PoolWorkspace& w, const int32_t* mem_state, int64_t pool_size, int64_t* first_fit, hipStream_t st) {
  LSATTN_LAUNCH_KERNEL(pool_summarise_kernel, dim3((unsigned)w.nb), dim3(kPoolThreads), 0, st, mem_state, pool_size, w.blk_free,
                     w.blk_last_used, first_fit);
  if (w.nb <= kPoolDirectBlocks) return false;
  LSATTN_LAUNCH_KERNEL(pool_scan_summaries_kernel, dim3(1), dim3(1024), 0, st, w.blk_free, w.blk_last_used, w.nb, w.free_before,
                     w.last_used_before);
  return true;
}

extern "C" int lsattn_pool_alloc(int32_t* mem_state, int64_t pool_size, int64_t need, int64_t* out_index, void* workspace,
                                 size_t workspace_bytes, void* stream) {
  const int rc = pool_search_checks(mem_state, pool_size, need, workspace, workspace_bytes);
  if (rc != LSATTN_OK) return rc;
  if (need > 0 && !out_index) return LSATTN_ERR_INVALID_ARG;
  hipStream_t st = (hipStream_t)stream;
  const PoolWorkspace w = pool_carve(workspace, pool_size);
  if (pool_is_one_group(pool_size, need)) {
    LSATTN_LAUNCH_KERNEL(pool_alloc_one_group_kernel, dim3(1), dim3(1024), 0, st, mem_state, (int)pool_size, need, out_index, w.cells);
    return check_launch();
  }
  const bool scan = pool_summarise(w, mem_state, pool_size, nullptr, st);
  LSATTN_LAUNCH_KERNEL(pool_take_kernel, dim3((unsigned)w.nb), dim3(kPoolThreads), 0, st, mem_state, pool_size,
                     scan ? w.free_before : nullptr, w.blk_free, need, out_index, w.cells);
  return check_launch();
}

extern "C" int lsattn_pool_find_contiguous(const int32_t* mem_state, int64_t pool_size, int64_t need, int64_t* out_start,
                                           void* workspace, size_t workspace_bytes, void* stream) {
  const int rc = pool_search_checks(mem_state, pool_size, need, workspace, workspace_bytes);
  if (rc != LSATTN_OK) return rc;
  if (!out_start || need <= 0) return LSATTN_ERR_INVALID_ARG;
  hipStream_t st = (hipStream_t)stream;
  const PoolWorkspace w = pool_carve(workspace, pool_size);
  const bool scan = pool_summarise(w, mem_state, pool_size, out_start, st);
  LSATTN_LAUNCH_KERNEL(pool_first_fit_kernel, dim3((unsigned)w.nb), dim3(kPoolThreads), 0, st, mem_state, pool_size,
                     scan ? w.last_used_before : nullptr, w.blk_last_used, need, out_start);
  return check_launch();
}

extern "C" int lsattn_pool_update_refs(int32_t* mem_state, int64_t pool_size, const int64_t* index, int64_t n, int delta,
                                       int64_t* counted, void* workspace, size_t workspace_bytes, void* stream) {
  if (!mem_state || pool_size <= 0 || n < 0 || (delta != 1 && delta != -1) || !counted) return LSATTN_ERR_INVALID_ARG;
  if (n > 0 && (!index || !workspace)) return LSATTN_ERR_INVALID_ARG;
  if ((uintptr_t)workspace & 15) return LSATTN_ERR_INVALID_ARG;
  if (workspace_bytes < lsattn_pool_refs_workspace_bytes(n)) return LSATTN_ERR_WORKSPACE;
  const int64_t nblk = refs_blocks(n);
  if (nblk > 0x7fffffff) return LSATTN_ERR_INVALID_ARG;
  hipStream_t st = (hipStream_t)stream;
  int64_t* blk_counts = (int64_t*)workspace;
  int32_t* old_state = (int32_t*)(blk_counts + 2 * nblk);
  if (n <= kRefsOneGroup) {  // (n = 0 too: counted = {0, 0})
    LSATTN_LAUNCH_KERNEL(pool_refs_small_kernel, dim3(1), dim3(1024), 0, st, mem_state, pool_size, index, n, delta, counted);
    return check_launch();
  }
  LSATTN_LAUNCH_KERNEL(pool_refs_gather_kernel, dim3((unsigned)nblk), dim3(256), 0, st, mem_state, pool_size, index, n, delta,
                     old_state, blk_counts);
  LSATTN_LAUNCH_KERNEL(pool_refs_apply_kernel, dim3((unsigned)nblk), dim3(256), 0, st, mem_state, pool_size, index,
                     n, delta, old_state, blk_counts, nblk, counted);
  return check_launch();
}
