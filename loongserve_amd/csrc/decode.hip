// Token-indexed flash decoding for gfx950: stage 1 (gather + split-K partials) and
// stage 2 (LSE merge over the block axis).
//
// Stage 1 replaces flash_decoding_stage1_kernel
// (longserve_cuda_kernels/src/flash_decoding_stage1.cu:25-143).  Differences by design:
//   * one wave64 serves one KV head and up to eight query heads of its GQA group (four at a time, in
//     up to two rounds over the rows it has loaded; larger groups take several waves), so a K/V row is
//     fetched once per group instead of once per query head;
//   * a K/V row of 128 16-bit elements is read by 16 lanes x 16 bytes; a wave has four
//     such lane groups and every group keeps 8 K rows and 8 V rows in flight;
//   * each lane group runs its own online softmax; groups are merged once per block with
//     an LSE merge, and the partial is written with plain stores (no atomics), so the
//     result is deterministic;
//   * a workgroup walks several consecutive blocks, so the launch is sized for the chip
//     and not for block_seq.
// Short contexts in the fused call are one launch without partials (decode_direct_kernel).
#include <atomic>
#include <chrono>
#include <type_traits>

#include "common.hip.h"

namespace lsattn {

struct Stage1Params {
  float* mid_o;
  float* mid_lse;
  const void* q;
  const void* k;
  const void* v;
  int64_t k_s0, k_s1, v_s0, v_s1;
  float scale_log2;  // sm_scale * log2(e)
  const int32_t* req_to_tokens;
  const int32_t* b_req_idx;
  const int32_t* b_seqlen;
  int64_t batch, hq, hkv, num_blocks, max_seq_len, block_seq, grid_blocks;  // block_seq: tokens per partial computed
  int64_t row_mul, fine_block_seq;  // partial of coarse block i goes to row i * row_mul; rows in between are marked empty
  int64_t blk_rows, req_rows;       // rows of mid_o between consecutive blocks / requests: (batch * hq, hq) in the reference's layout
  int32_t blocks_per_wg;  // consecutive blocks walked by one workgroup
  int32_t tasks;          // hkv * (group / GT) wave tasks
  int32_t tasks_on_x;     // grid = (task groups, chunks, batch) instead of (chunks, task groups, batch)
  int32_t max_shares, share_units;  // equal shares: at most so many, of at least so many units each
  void* o;                          // (DIRECT, JOIN) the result [batch, hq, 128] and its log-sum-exps
  float* out_lse;
  int32_t o_dtype;                  // (JOIN)
  uint64_t arrivals;                // (JOIN) where this launch's counts of arrivals start
};

constexpr int kTok = 8;  // K/V rows in flight per 16-lane group

// f(integral_constant<int, 0>) ... f(integral_constant<int, N-1>): loop indices that must be constant expressions
template <int N, typename F> __device__ __forceinline__ void static_for(F&& f) {
  if constexpr (N > 0) {
    static_for<N - 1>(f);
    f(std::integral_constant<int, N - 1>{});
  }
}

template <typename OT> __device__ __forceinline__ void store4(void* base, int64_t elem, const f32x4& v);
template <> __device__ __forceinline__ void store4<float>(void* base, int64_t elem, const f32x4& v) {
  *(f32x4*)((float*)base + elem) = v;
}
template <> __device__ __forceinline__ void store4<F16>(void* base, int64_t elem, const f32x4& v) {
  *(u32x2*)((uint16_t*)base + elem) = u32x2{pack2<F16>(v[0], v[1]), pack2<F16>(v[2], v[3])};
}
template <> __device__ __forceinline__ void store4<BF16>(void* base, int64_t elem, const f32x4& v) {
  *(u32x2*)((uint16_t*)base + elem) = u32x2{pack2<BF16>(v[0], v[1]), pack2<BF16>(v[2], v[3])};
}

// ------------------------------------------------------------------------------------
// Stage 1 and the merge in one launch (JOIN): the workgroup, or wave, of a (request, task) that is the last to have stored its partial
// merges all of them into the result.  Nobody waits for anybody.  What it takes is a count of arrivals in memory that the caller
// does not clear: the first eight bytes of the task's rows of the result, which the merge overwrites.  They hold anything at first.
// Whoever finds no count of this launch there puts the launch's start in (one of them succeeds), before it counts itself; the start
// is 64 bits that no other launch has, so nothing else is taken for a count, and a replay from a graph finds the last replay's result.
// Partials go through to memory and are read past the L2s (each XCD has its own).
// ------------------------------------------------------------------------------------
constexpr int64_t kJoinMaxPartials = 64;
constexpr int64_t kCUs = 256;  // compute units of the MI355X
__device__ __forceinline__ void store_through(float* dst, const f32x4& v) {
  asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1\n\ts_nop 1" : : "v"(dst), "v"(v) : "memory");  // (the s_nop: as in store_partial_row)
}
template <typename V> __device__ __forceinline__ V load_past_l2(const V* src) {
  return __hip_atomic_load(src, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t* arrivals_of(const Stage1Params& p, int64_t out_row0) {
  return (uint64_t*)((char*)p.o + out_row0 * 128 * (p.o_dtype == LSATTN_F32 ? 4 : 2));
}
__device__ __forceinline__ void store_result(const Stage1Params& p, int64_t elem, const f32x4& v) {
  if (p.o_dtype == LSATTN_F32) store4<float>(p.o, elem, v);
  else if (p.o_dtype == LSATTN_F16) store4<F16>(p.o, elem, v);
  else store4<BF16>(p.o, elem, v);
}
// `seen`: what the word held when the workgroup (wave) started; n: partials, one of them each.  Returns what the word held when the start was put in, or `seen` if it is a count already;
// nobody waits for it before arrive.
__device__ __forceinline__ uint64_t start_arrivals(uint64_t* word, uint64_t seen, uint64_t start, int n) {
  uint64_t held = seen;
  if (seen - start > (uint64_t)n) __hip_atomic_compare_exchange_strong(word, &held, start, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return held;
}
// Behind a wait for the stores of the partial.  If the word was neither what was seen nor a count of this launch, the start is put in over what it was then: once at most in memory
// that nobody else writes, and never without end.
constexpr int kStartTries = 64;
__device__ __forceinline__ bool arrive(uint64_t* word, uint64_t seen, uint64_t held, uint64_t start, int n) {
  for (int i = 0; i < kStartTries && held != seen && held - start > (uint64_t)n; i++) {
    seen = held;
    __hip_atomic_compare_exchange_strong(word, &held, start, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  return __hip_atomic_fetch_add(word, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) - start == (uint64_t)(n - 1);
}
// The merge of `n` <= kJoinMaxPartials partials of up to 16 query heads, by the four waves of a workgroup.
// Half a wave reads a row, 16 bytes a lane; a head's rows are dealt to S half waves, which meet in LDS.  Sixteen rows of a
// half wave are asked for at once, beside the log-sum-exps, of which lane e holds those of partials e and 32 + e.
__device__ __forceinline__ void join_partials(const Stage1Params& p, char* lds, const int lane, const int wave, const int64_t out_row0, const int nh,
                                              const int64_t row0, const int n) {
  const int c = lane & 31, half = wave * 2 + (lane >> 5);
  const int S = nh == 1 ? 8 : nh == 2 ? 4 : nh <= 4 ? 2 : 1, slice = half & (S - 1);
  const int rows_here = (n + S - 1) / S;  // (the same for all half waves; positions past the last partial repeat it and weigh nothing)
  const float* const lse_at = p.mid_lse + row0;
  const float* const rows_at = p.mid_o + row0 * 128;
  const uint32_t blk_rows = (uint32_t)p.blk_rows;  // (offsets below 2^31 bytes, checked on the host)
  for (int h0 = 0; h0 < nh; h0 += 8 / S) {
    const int h = h0 + half / S;
    const bool live = h < nh;
    const uint32_t hh = live ? h : nh - 1;
    float lse0 = -INFINITY, lse1 = -INFINITY;
    if (c < n) lse0 = load_past_l2(lse_at + (hh + c * blk_rows));
    if (32 + c < n) lse1 = load_past_l2(lse_at + (hh + (32 + c) * blk_rows));
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    float M = 0.f, L = 0.f, w0 = 0.f, w1 = 0.f;
    for (int i = 0; i < rows_here; i += 16) {
      f32x4 row[16];
#pragma unroll
      for (int q = 0; q < 16; q += 4) {
        if (i + q < rows_here) {
#pragma unroll
          for (int u = q; u < q + 4; u++) {
            const int e = (i + u) * S + slice;
            const uint32_t at = (hh + (e < n ? e : n - 1) * blk_rows) * 512u + c * 16u;
            asm volatile("global_load_dwordx4 %0, %1, %2 sc1" : "=v"(row[u]) : "v"(at), "s"(rows_at) : "memory");
          }
        }
      }
      if (i == 0) {
        M = fmaxf(lse0, lse1);
#pragma unroll
        for (int d = 16; d > 0; d >>= 1) M = fmaxf(M, __shfl_xor(M, d, 64));
        w0 = exp2_diff(lse0 * kLog2e, M * kLog2e);  // (0 past the last partial)
        w1 = exp2_diff(lse1 * kLog2e, M * kLog2e);
        L = w0 + w1;
#pragma unroll
        for (int d = 16; d > 0; d >>= 1) L += __shfl_xor(L, d, 64);
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
      for (int q = 0; q < 16; q += 4) {
        if (i + q < rows_here) {
#pragma unroll
          for (int u = q; u < q + 4; u++) {
            asm volatile("" : "+v"(row[u]));
            const int e = (i + u) * S + slice;
            const float w = e < n ? __shfl(e < 32 ? w0 : w1, (lane & 32) | (e & 31), 64) : 0.f;
            if (w != 0.f) acc += row[u] * w;  // (what has no weight may be infinite)
          }
        }
      }
    }
    if (S > 1) {
      f32x4* part = (f32x4*)(lds + 16);
      part[half * 32 + c] = acc;
      __syncthreads();
      if (slice == 0)
        for (int w = 1; w < S; w++) acc += part[(half + w) * 32 + c];
    }
    if (slice == 0 && live) {
      const float inv = L > 0.f ? 1.f / L : 0.f;
      store_result(p, (out_row0 + h) * 128 + c * 4, acc * inv);
      if (c == 0) p.out_lse[out_row0 + h] = L > 0.f ? M + __builtin_amdgcn_logf(L) * kLn2 : -INFINITY;
    }
  }
}

// sum over two packed 16-bit products with fp32 accumulation (v_dot2c_f32_f16 / v_dot2c_f32_bf16)
template <typename T> __device__ __forceinline__ float dot2acc(uint32_t a, uint32_t b, float c);
template <> __device__ __forceinline__ float dot2acc<F16>(uint32_t a, uint32_t b, float c) {
  return __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, a), __builtin_bit_cast(f16x2, b), c, false);
}
template <> __device__ __forceinline__ float dot2acc<BF16>(uint32_t a, uint32_t b, float c) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, a), __builtin_bit_cast(bf16x2, b), c, false);
}
// the same as volatile inline assembly, for sequences whose instruction order is fixed by hand
template <typename T> struct Dot;
template <> struct Dot<F16> {
  static __device__ __forceinline__ void first(float& d, uint32_t a, uint32_t b) { asm volatile("v_dot2_f32_f16 %0, %1, %2, 0" : "=v"(d) : "v"(a), "v"(b)); }
  static __device__ __forceinline__ void next(float& d, uint32_t a, uint32_t b) { asm volatile("v_dot2c_f32_f16 %0, %1, %2" : "+v"(d) : "v"(a), "v"(b)); }
};
template <> struct Dot<BF16> {
  static __device__ __forceinline__ void first(float& d, uint32_t a, uint32_t b) { asm volatile("v_dot2_f32_bf16 %0, %1, %2, 0" : "=v"(d) : "v"(a), "v"(b)); }
  static __device__ __forceinline__ void next(float& d, uint32_t a, uint32_t b) { asm volatile("v_dot2c_f32_bf16 %0, %1, %2" : "+v"(d) : "v"(a), "v"(b)); }
};

// SPLIT: the NW waves of a workgroup share one task and take every NW-th batch of 32 tokens of a block; their partials
// meet in LDS.  For launches too small to fill the chip otherwise (short contexts at small batch): NW times as many rows
// in flight.
// ONCE: every K/V row is read by one wave only (at most GT query heads per KV head), so the rows are loaded
// non-temporally; otherwise the waves that take the other query heads of the group read them again and ordinary loads let
// those find the rows in L2.
template <typename T, int GT, int NW, bool SPLIT, bool ONCE, int HR, bool JOIN = false>
__global__ __launch_bounds__(NW * 64, JOIN ? (GT == 1 ? 4 : 3) : 1) void decode_stage1_kernel(Stage1Params p) {
  static_assert(!JOIN || (SPLIT && NW == 4), "join_partials takes the four waves of a workgroup");
  constexpr int GH = GT * HR;  // query heads per task
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int grp = lane >> 4;   // which of the 4 row slots of the wave
  const int sub = lane & 15;   // 16-byte column slot: elements sub*8 .. sub*8+7
  const int jbase = (sub >> 2) * 2;  // first of the two rows whose scores this lane finishes (see the reduction)
  const int64_t b = blockIdx.z;
  // The workgroups that read the other KV heads of the same tokens are next to this one in dispatch order when the
  // task index is the fastest grid dimension: the pieces of a token's K (and V) span are then fetched close together in
  // time (measured 2 % faster on GQA 32/8, two task groups per chunk).
  const int task = SPLIT ? (int)(p.tasks_on_x ? blockIdx.x : blockIdx.y) : (int)(p.tasks_on_x ? blockIdx.x : blockIdx.y) * NW + wave;
  if (task >= p.tasks) return;  // (SPLIT: the same for every wave of the workgroup, like the block range below)
  // a task = one KV head and up to GT query heads of its group; the last task of a group whose size is not a multiple of
  // GT has fewer (nh): its spare accumulators repeat the last query head and are not written
  const int group = (int)(p.hq / p.hkv);
  const int sub_groups = (group + GH - 1) / GH;
  const int kvh = task / sub_groups;
  const int sg = task % sub_groups;
  const int qh0 = kvh * group + sg * GH;
  const int nh = group - sg * GH < GH ? group - sg * GH : GH;

  const int len = p.b_seqlen[b];  // positions inside a request are 32-bit (max_seq_len is checked on the host)
  int64_t nblk = len <= 0 ? 0 : ((int64_t)len + p.block_seq - 1) / p.block_seq;
  if (nblk > p.grid_blocks) nblk = p.grid_blocks;
  if (nblk > (p.num_blocks + p.row_mul - 1) / p.row_mul) nblk = (p.num_blocks + p.row_mul - 1) / p.row_mul;
  int64_t fine_nblk = len <= 0 ? 0 : ((int64_t)len + p.fine_block_seq - 1) / p.fine_block_seq;  // rows the request reaches
  if (fine_nblk > p.num_blocks) fine_nblk = p.num_blocks;
  // Workgroups go to the 8 XCDs round-robin in linear id order, so a fixed chunk index always lands on the same XCDs and
  // the first chunks (all that short requests have) would load some XCDs more than others; the chunk index is rotated by
  // the request index to spread them (batch 64 with lengths 4096..32768: 5.62 -> 5.9 TB/s).
  const unsigned n_chunks = p.tasks_on_x ? gridDim.y : gridDim.x;
  const unsigned chunk = ((p.tasks_on_x ? blockIdx.y : blockIdx.x) + (unsigned)b) % n_chunks;
  const int64_t blk_begin = (int64_t)chunk * p.blocks_per_wg;
  int64_t blk_end = blk_begin + p.blocks_per_wg;
  if (blk_end > nblk) blk_end = nblk;
  if (JOIN && nblk <= 0 && blk_begin == 0) {  // a request without tokens
    for (int i = wave * 64 + lane; i < nh * 32; i += NW * 64) store_result(p, (b * p.hq + qh0) * 128 + i * 4, f32x4{0.f, 0.f, 0.f, 0.f});
    if (wave == 0 && lane < nh) p.out_lse[b * p.hq + qh0 + lane] = -INFINITY;
  }
  if (blk_begin >= blk_end) return;
  // (JOIN) workgroups that store partials of this request and task, of one block each or of several
  const int arrivals = JOIN ? (int)((nblk + p.blocks_per_wg - 1) / p.blocks_per_wg) : 0;
  uint64_t* const word = JOIN ? arrivals_of(p, b * p.hq + qh0) : nullptr;
  uint64_t seen = 0;
  if (JOIN) seen = load_past_l2(word);  // (by every wave: no branch, and so no wait here)

  const int32_t* table = p.req_to_tokens + (int64_t)p.b_req_idx[b] * p.max_seq_len;
  const char* kbase = (const char*)p.k + ((int64_t)kvh * p.k_s1 + sub * 8) * 2;
  const char* vbase = (const char*)p.v + ((int64_t)kvh * p.v_s1 + sub * 8) * 2;
  const int64_t k_row_bytes = p.k_s0 * 2, v_row_bytes = p.v_s0 * 2;

  // q stays packed (8 elements = 4 words per head and lane); the scale is applied to the reduced dot
  u32x4 qw[GH];
#pragma unroll
  for (int h = 0; h < GH; h++) qw[h] = *(const u32x4*)((const char*)p.q + ((b * p.hq + qh0 + (h < nh ? h : nh - 1)) * 128 + sub * 8) * 2);

  for (int64_t blk = blk_begin; blk < blk_end; blk++) {
    const int t0 = (int)(blk * p.block_seq);
    const int64_t t1_64 = (int64_t)t0 + p.block_seq;
    const int t1 = t1_64 > len ? len : (int)t1_64;
    const int t_last = t1 - 1;

    float m[GH], l[GH], o[GH][8];
#pragma unroll
    for (int h = 0; h < GH; h++) {
      m[h] = -INFINITY;
      l[h] = 0.f;
#pragma unroll
      for (int i = 0; i < 8; i++) o[h][i] = 0.f;
    }

    // Slot indices of the first batch of rows.  A row position past the block repeats the block's
    // last row (always a real slot): it is loaded like any other and dropped by the validity mask,
    // so the loop body has no divergent control flow.
    constexpr int kStep = 4 * kTok * (SPLIT ? NW : 1);
    const int it0 = t0 + (SPLIT ? wave * 4 * kTok : 0);
    int32_t slot[kTok];
#pragma unroll
    for (int j = 0; j < kTok; j++) {
      const int tok = it0 + j * 4 + grp;
      slot[j] = table[tok < t1 ? tok : t_last];
    }

    for (int it = it0; it < t1; it += kStep) {
      u32x4 kr[kTok], vr[kTok];
      // (the empty statements keep each 64-bit address next to its load instead of sixteen of them live at once)
#pragma unroll
      for (int j = 0; j < kTok; j++) {
        asm volatile("" : "+v"(slot[j]));
        kr[j] = ONCE ? __builtin_nontemporal_load((const u32x4*)(kbase + (int64_t)slot[j] * k_row_bytes))
                     : *(const u32x4*)(kbase + (int64_t)slot[j] * k_row_bytes);
      }
#pragma unroll
      for (int j = 0; j < kTok; j++) {
        asm volatile("" : "+v"(slot[j]));
        vr[j] = ONCE ? __builtin_nontemporal_load((const u32x4*)(vbase + (int64_t)slot[j] * v_row_bytes))
                     : *(const u32x4*)(vbase + (int64_t)slot[j] * v_row_bytes);
      }
      // The rows are read once: non-temporal loads.  As ordinary loads they push the block partials (which stage 2
      // reads back) out of the caches early, and the trickle of write-backs between the reads costs the gather 5 %.
      // all 16 row loads are issued before anything else happens (the scheduler would otherwise sink
      // each load next to its first use and expose its latency)
      __builtin_amdgcn_sched_barrier(0);
      // slot indices of the next batch while the rows are in flight
#pragma unroll
      for (int j = 0; j < kTok; j++) {
        const int tok = it + kStep + j * 4 + grp;
        slot[j] = table[tok < t1 ? tok : t_last];
      }
      __builtin_amdgcn_sched_barrier(0);

      // HR rounds of GT query heads each over the rows just loaded (HR = 2: groups of 5 to 8 query heads per KV head
      // fetch every row once, not once per four heads)
      static_for<HR>([&](auto hr_tag) {
        constexpr int HB = decltype(hr_tag)::value * GT;
        // Partial dots over this lane's 8 elements for the 8 rows x GT heads of the group (value index
        // v = GT*j + h), then a transposing reduction over the 16 lanes of the row group: two halving steps
        // with bank-masked DPP adds (lanes with sub bits (3,2) = (B3,B2) keep values [NV/2*B3 + NV/4*B2, +NV/4))
        // and a sum over the quad.  Every lane ends with the finished raw scores of two rows,
        // jbase = 4*B3 + 2*B2 and jbase + 1, for all GT heads: w[GT*r + h].  The softmax scale is folded
        // into the exp2 argument.
        constexpr int NV = kTok * GT;
        float u[NV / 2], w[NV / 4];
        // Everything up to the quad sums is volatile inline assembly in a fixed order: a DPP read needs two
        // wait states after the write of its source, the compiler's hazard recogniser does not look into inline
        // assembly, and it would otherwise move the dots between the DPP adds.  The first halving step of a
        // value pair (v, v + NV/2) follows the dots of the next pair, so only two partial dots are live at a time.
        float lo_prev = 0.f, hi_prev = 0.f;
  #pragma unroll
        for (int i = 0; i < NV / 2; i++) {
          const int j = i / GT, h = i % GT;
          float lo, hi;
          Dot<T>::first(lo, qw[HB + h][0], kr[j][0]);
          Dot<T>::first(hi, qw[HB + h][0], kr[j + kTok / 2][0]);
  #pragma unroll
          for (int c = 1; c < 4; c++) {
            Dot<T>::next(lo, qw[HB + h][c], kr[j][c]);
            Dot<T>::next(hi, qw[HB + h][c], kr[j + kTok / 2][c]);
          }
          if (i > 0) {
            asm volatile("v_add_f32_dpp %0, %1, %1 row_ror:8 row_mask:0xf bank_mask:0x3" : "=v"(u[i - 1]) : "v"(lo_prev));
            asm volatile("v_add_f32_dpp %0, %1, %1 row_ror:8 row_mask:0xf bank_mask:0xc" : "+v"(u[i - 1]) : "v"(hi_prev));
          }
          lo_prev = lo;
          hi_prev = hi;
        }
        asm volatile("s_nop 1");
        asm volatile("v_add_f32_dpp %0, %1, %1 row_ror:8 row_mask:0xf bank_mask:0x3" : "=v"(u[NV / 2 - 1]) : "v"(lo_prev));
        asm volatile("v_add_f32_dpp %0, %1, %1 row_ror:8 row_mask:0xf bank_mask:0xc" : "+v"(u[NV / 2 - 1]) : "v"(hi_prev));
        asm volatile("s_nop 1");
  #pragma unroll
        for (int i = 0; i < NV / 4; i++) asm volatile("v_add_f32_dpp %0, %1, %1 row_ror:12 row_mask:0xf bank_mask:0x5" : "=v"(w[i]) : "v"(u[i]));
        asm volatile("s_nop 1");
  #pragma unroll
        for (int i = 0; i < NV / 4; i++) asm volatile("v_add_f32_dpp %0, %1, %1 row_ror:4 row_mask:0xf bank_mask:0xa" : "+v"(w[i]) : "v"(u[i + NV / 4]));
        asm volatile("s_nop 1");
  #pragma unroll
        for (int i = 0; i < NV / 4; i++) {
          w[i] += dpp_mov<0xB1>(w[i]);  // quad_perm [1,0,3,2]
          w[i] += dpp_mov<0x4E>(w[i]);  // quad_perm [2,3,0,1]
        }
        // rows past the block only exist in its last batch and are masked there
        const bool tail = it + 4 * kTok > t1;
        if (tail) {
  #pragma unroll
          for (int r = 0; r < 2; r++) {
            const bool valid = it + (jbase + r) * 4 + grp < t1;
  #pragma unroll
            for (int h = 0; h < GT; h++) w[GT * r + h] = valid ? w[GT * r + h] : -INFINITY;
          }
        }
        float pw[2 * GT];
        float alpha[GT];
        bool grow = false;
  #pragma unroll
        for (int h = 0; h < GT; h++) {
          float mx = fmaxf(w[h], w[GT + h]);
          mx = fmaxf(mx, dpp_mov<0x124>(mx));  // row_ror:4
          mx = fmaxf(mx, dpp_mov<0x128>(mx));  // row_ror:8: now the maximum over the 8 rows, in every lane
          const float m_new = fmaxf(m[HB + h], mx * p.scale_log2);  // scale > 0
          const float m_safe = (m_new == -INFINITY) ? 0.f : m_new;
          alpha[h] = __builtin_amdgcn_exp2f(m[HB + h] - m_safe);
          grow |= m_new != m[HB + h];
          pw[h] = __builtin_amdgcn_exp2f(__builtin_fmaf(w[h], p.scale_log2, -m_safe));
          pw[GT + h] = __builtin_amdgcn_exp2f(__builtin_fmaf(w[GT + h], p.scale_log2, -m_safe));
          float ps = pw[h] + pw[GT + h];
          ps += dpp_mov<0x124>(ps);
          ps += dpp_mov<0x128>(ps);
          l[HB + h] = l[HB + h] * alpha[h] + ps;
          m[HB + h] = m_new;
        }
        // the accumulators only need rescaling when some running max moved (rare once warmed up)
        if (__builtin_amdgcn_ballot_w64(grow) != 0) {
  #pragma unroll
          for (int h = 0; h < GT; h++)
  #pragma unroll
            for (int i = 0; i < 8; i++) o[HB + h][i] *= alpha[h];
        }
        if (std::is_same<T, F16>::value) {
          // O += P V on pairs of rows: the owners pack (p[2q], p[2q+1]) to fp16 (p <= 1), row pair q is
          // broadcast from lane 4q of the group, the two V rows are interleaved element by element
          uint32_t pp[GT];
  #pragma unroll
          for (int h = 0; h < GT; h++) pp[h] = pack2<F16>(pw[h], pw[GT + h]);
          static_for<kTok / 2>([&](auto q_tag) {
            constexpr int q = decltype(q_tag)::value;
            uint32_t bq[GT];
  #pragma unroll
            for (int h = 0; h < GT; h++) bq[h] = __builtin_bit_cast(uint32_t, dpp_mov<0x150 + 4 * q>(__builtin_bit_cast(float, pp[h])));  // row_newbcast
  #pragma unroll
            for (int w4 = 0; w4 < 4; w4++) {
              const uint32_t lo = __builtin_amdgcn_perm(vr[2 * q + 1][w4], vr[2 * q][w4], 0x05040100u);
              const uint32_t hi = __builtin_amdgcn_perm(vr[2 * q + 1][w4], vr[2 * q][w4], 0x07060302u);
  #pragma unroll
              for (int h = 0; h < GT; h++) {
                o[HB + h][2 * w4] = dot2acc<F16>(bq[h], lo, o[HB + h][2 * w4]);
                o[HB + h][2 * w4 + 1] = dot2acc<F16>(bq[h], hi, o[HB + h][2 * w4 + 1]);
              }
            }
          });
        } else {
          // bf16: a bf16 P would cost ~1e-3 relative error, so P stays fp32 and is broadcast row by row
          static_for<kTok>([&](auto j_tag) {
            constexpr int j = decltype(j_tag)::value;
            float vf[8];
            unpack8<T>(vr[j], vf);
  #pragma unroll
            for (int h = 0; h < GT; h++) {
              const float pb = dpp_mov<0x150 + 4 * (j >> 1)>(pw[GT * (j & 1) + h]);  // row_newbcast
  #pragma unroll
              for (int i = 0; i < 8; i++) o[HB + h][i] = __builtin_fmaf(pb, vf[i], o[HB + h][i]);
            }
          });
        }
      });
    }

    // merge the four lane groups (and, SPLIT, the waves) and write the block's partial
    __shared__ float xw[SPLIT ? NW : 1][GH][16][10];  // per wave, head and column slot: 8 sums, running max, row sum
    auto write_partial = [&](int h, float M, float L, const float (&ov)[8]) {
      if (h >= nh) return;
      const float inv = 1.f / L;
      if constexpr (JOIN) {
        const f32x4 lo = f32x4{ov[0] * inv, ov[1] * inv, ov[2] * inv, ov[3] * inv}, hi = f32x4{ov[4] * inv, ov[5] * inv, ov[6] * inv, ov[7] * inv};
        const float lse = (M + __builtin_amdgcn_logf(L)) * kLn2;
        const int64_t row = blk * p.blk_rows + b * p.req_rows + qh0 + h;
        store_through(p.mid_o + row * 128 + sub * 8, lo);
        store_through(p.mid_o + row * 128 + sub * 8 + 4, hi);
        if (sub == 0) __hip_atomic_store(p.mid_lse + row, lse, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        return;
      }
      const int64_t row = blk * p.row_mul * p.blk_rows + b * p.req_rows + qh0 + h;
      f32x4* dst = (f32x4*)(p.mid_o + row * 128 + sub * 8);
      dst[0] = f32x4{ov[0] * inv, ov[1] * inv, ov[2] * inv, ov[3] * inv};
      dst[1] = f32x4{ov[4] * inv, ov[5] * inv, ov[6] * inv, ov[7] * inv};
      if (sub == 0) p.mid_lse[row] = (M + __builtin_amdgcn_logf(L)) * kLn2;
      // the rows of the blocks merged into this partial (row_mul <= 16: lane `sub` takes the sub-th of them)
      if (sub >= 1 && sub < p.row_mul && blk * p.row_mul + sub < fine_nblk)
        p.mid_lse[(blk * p.row_mul + sub) * p.blk_rows + b * p.req_rows + qh0 + h] = -INFINITY;
    };
#pragma unroll
    for (int h = 0; h < GH; h++) {
      float M = fmaxf(m[h], __shfl_xor(m[h], 16));
      M = fmaxf(M, __shfl_xor(M, 32));
      const float w = exp2_diff(m[h], M);  // 0 for a group (or, SPLIT, a whole wave) that saw no row
      float L = l[h] * w;
      L += __shfl_xor(L, 16);
      L += __shfl_xor(L, 32);
      float ov[8];
#pragma unroll
      for (int i = 0; i < 8; i++) {
        float x = o[h][i] * w;
        x += __shfl_xor(x, 16);
        x += __shfl_xor(x, 32);
        ov[i] = x;
      }
      if (grp == 0) {
        if (SPLIT) {
          float* dst = xw[wave][h][sub];
#pragma unroll
          for (int i = 0; i < 8; i++) dst[i] = ov[i];
          dst[8] = M;
          dst[9] = L;
        } else {
          write_partial(h, M, L, ov);  // the block holds >= 1 row, so M is finite and L > 0
        }
      }
    }
    if (SPLIT) {
      __syncthreads();
      if (wave == 0 && grp == 0) {
#pragma unroll
        for (int h = 0; h < GH; h++) {
          float M = xw[0][h][sub][8];
#pragma unroll
          for (int w = 1; w < NW; w++) M = fmaxf(M, xw[w][h][sub][8]);
          float L = 0.f, ov[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int w = 0; w < NW; w++) {
            const float* src = xw[w][h][sub];
            const float f = exp2_diff(src[8], M);
            L += src[9] * f;
#pragma unroll
            for (int i = 0; i < 8; i++) ov[i] += src[i] * f;
          }
          write_partial(h, M, L, ov);
        }
      }
      __syncthreads();  // the next block of this workgroup writes the same LDS
    }
  }
  if constexpr (JOIN) {
    __shared__ __attribute__((aligned(16))) char meet[16 + 8 * 32 * 16];
    if (wave == 0 && lane == 0) {
      const uint64_t held = start_arrivals(word, seen, p.arrivals, arrivals);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (wave 0 has stored the partials)
      *(uint32_t*)meet = arrive(word, seen, held, p.arrivals, arrivals);
    }
    __syncthreads();
    if (*(const uint32_t*)meet) join_partials(p, meet, lane, wave, b * p.hq + qh0, nh, b * p.req_rows + qh0, (int)nblk);
  }
}

// ------------------------------------------------------------------------------------
// Stage 1 for large launches (any group size): both products on the matrix pipe.
// One wave64 = one KV head, up to 16 query heads of its group (the 16 columns of a 16x16x32 MFMA) and a run of
// consecutive blocks; the waves of a workgroup are independent (no barrier) and take neighbouring KV heads over the same
// tokens, whose rows lie side by side in memory.  A batch is 32 tokens:
//   the K and V rows are loaded the way the other stage-1 kernels load them, a whole 256-byte row per 16 lanes (loading the
//     MFMA operand layout straight from memory, 16 rows x 64 bytes per instruction, ran 20 % slower), double-buffered in
//     registers so that the rows of batch j + 1 are in flight while batch j is computed;
//   at compute time the wave turns its rows into operand layout through its own 17.5 KB of LDS (rows padded to 272 and
//     288 bytes, so that the sixteen rows of a K read and the eight rows of a transposing V read fall into different banks
//     and every address is one register plus an immediate): K rows are read back as the A operand of S = K Q^T (Q^T, the B operand, stays in registers), V rows are
//     read back transposed (ds_read_b64_tr_b16) as the A operand of O^T += V^T P^T;
//   the softmax runs on the accumulators (a lane holds one query head's scores of eight tokens), and P, converted in
//     place, is the B operand of the second product.  A bfloat16 P would cost about 1e-3 relative error, so bfloat16
//     inputs multiply V by the high and by the low part of P.
// All global loads are issued from inline assembly, so that the hand-placed waits leave exactly the next batch's rows
// outstanding; tests/test_prefill_isa_hazards.py checks that no register of a load in flight is touched before its wait.
// ------------------------------------------------------------------------------------
__device__ __forceinline__ float xlane16(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_ds_swizzle(__builtin_bit_cast(int, v), 0x401F));  // lane ^ 16
}
__device__ __forceinline__ float xlane32(float v) {
  const unsigned u = __builtin_bit_cast(unsigned, v);
  auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return __builtin_bit_cast(float, (threadIdx.x & 32) ? r[0] : r[1]);
}
template <typename T> struct Mfma16;
template <> struct Mfma16<F16> {
  static __device__ __forceinline__ f32x4 run(const u32x4& a, const u32x4& b, const f32x4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
};
template <> struct Mfma16<BF16> {
  static __device__ __forceinline__ f32x4 run(const u32x4& a, const u32x4& b, const f32x4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
};

constexpr int kMfmaWaves = 4;        // waves per workgroup (independent)
constexpr int kMfmaBatch = 32;       // tokens per batch
constexpr int kMfmaKRow = 272, kMfmaVRow = 288;  // padded row lengths in LDS (bytes)
constexpr int kMfmaStage = kMfmaBatch * (kMfmaKRow + kMfmaVRow);  // LDS bytes per wave: the K rows and the V rows of one batch

// WS (small launches with fewer than four tasks): the four waves of a workgroup share one task and one block, take every
// fourth batch of its tokens and merge their partials through LDS: four times the waves of the plain shape, each short.
// One unit of work of a workgroup: request b, task group bid_t, chunk group bid_c (of n_cgroups in the grid; LISTED: the
// unit comes from a list of the units that exist, and its chunk group is taken as it is).
// RANGE: the wave walks a share of the line of all requests' tokens instead (ShareWalk): batch after batch without a break
// where one request ends and the next begins (the loads run ahead of the arithmetic across that point: they need only the
// slot numbers, which come from the table row of whatever request the share has reached), one partial per request it
// touches, number v + request of the launch (mid_o as [partial, Hq, 128]; the merge behind it knows whose partial that is).
// The lane's eight 16-byte pieces of a partial's row, 64 bytes apart, each scaled by `inv`.  The stores carry the
// system-scope bits: such a store goes through to memory as it is issued instead of waiting in the L2 as a dirty line
// that is written back later, alone, between the reads of a gather that keeps every memory channel busy.  Measured on
// a plain streaming read of 4 GiB with 8 KB stores mixed in: 67 MB of them (1.6 % of the bytes, what config 3 writes at
// one partial per 256 tokens) take the read from 6.47 to 5.65 TB/s as ordinary stores, to 5.94 with these bits; 4 MB
// (0.1 %) to 6.28 and 6.42.  Issued from inline assembly (the compiler has no store of this kind that is not atomic);
// a vector instruction may not overwrite the data registers of a store of more than 64 bits in the two cycles behind
// it, which the compiler knows of its own stores only: hence the s_nop.
__device__ __forceinline__ void store_partial_row(float* dst, const f32x4 (&acc)[8], const float inv) {
#define LSATTN_STORE_ROW_PIECE(db)                                                                                                  \
  {                                                                                                                                \
    const f32x4 piece = acc[db] * inv;                                                                                             \
    asm volatile("global_store_dwordx4 %0, %1, off offset:%2 sc0 sc1\n\ts_nop 1" : : "v"(dst), "v"(piece), "n"(64 * db) : "memory"); \
  }
  LSATTN_STORE_ROW_PIECE(0) LSATTN_STORE_ROW_PIECE(1) LSATTN_STORE_ROW_PIECE(2) LSATTN_STORE_ROW_PIECE(3)
  LSATTN_STORE_ROW_PIECE(4) LSATTN_STORE_ROW_PIECE(5) LSATTN_STORE_ROW_PIECE(6) LSATTN_STORE_ROW_PIECE(7)
#undef LSATTN_STORE_ROW_PIECE
}

__device__ __forceinline__ uint32_t share_units_of(const int len, const int64_t block_seq, const int64_t grid_blocks) {
  const uint32_t n = len <= 0 ? 0u : ((uint32_t)len + (uint32_t)block_seq - 1u) / (uint32_t)block_seq;
  return n > (uint32_t)grid_blocks ? (uint32_t)grid_blocks : n;
}
// A share of the line of units (kMfmaBatch tokens of a request each): units [x, end) of it, x in request r.
struct ShareWalk {
  uint32_t v, x, end;
  int r;
  // units of requests 0 .. r, length and table row of request r: lane r's (up to 64 requests) or in LDS and memory
  bool in_registers;
  uint32_t incl;
  int len, req;
  const uint32_t* first_unit;
};
// One request's part of the share: tokens [t, t_end) of request r.
struct ShareSegment {
  int r, t, t_end;
  uint32_t x_end;  // where on the line it ends
  int req;
};
__device__ __forceinline__ ShareSegment share_segment(const Stage1Params& p, const ShareWalk& w, int r, uint32_t x) {
  uint32_t r0, r1;
  int len;
  ShareSegment s;
  for (;; r++) {  // (requests without units are skipped; x is below the line's end, so one is found)
    if (w.in_registers) {
      r1 = __builtin_amdgcn_readlane(w.incl, r);
      if (r1 > x) {
        r0 = r > 0 ? __builtin_amdgcn_readlane(w.incl, r - 1) : 0u;
        len = __builtin_amdgcn_readlane(w.len, r);
        s.req = __builtin_amdgcn_readlane(w.req, r);
        break;
      }
    } else {
      r1 = __builtin_amdgcn_readfirstlane(w.first_unit[r + 1]);
      if (r1 > x) {
        r0 = __builtin_amdgcn_readfirstlane(w.first_unit[r]);
        len = p.b_seqlen[r];
        s.req = p.b_req_idx[r];
        break;
      }
    }
  }
  s.r = r;
  s.x_end = r1 < w.end ? r1 : w.end;
  s.t = (int)(x - r0) * kMfmaBatch;
  s.t_end = (int)(s.x_end - r0) * kMfmaBatch;
  if (s.t_end > len) s.t_end = len;
  return s;
}

// OT (WS): the workgroup takes all tokens of its request and writes the result, in this type; void: partials.
// JOIN (WS): partials, and the workgroup of a (request, task) that is the last to have written its own merges them into the result.
template <typename T, bool WS, bool LISTED, bool RANGE = false, typename OT = void, bool JOIN = false>
__device__ __forceinline__ void stage1_mfma_unit(const Stage1Params& p, char* lds, const int lane, const int wave, const int64_t b,
                                                 const unsigned bid_t, const unsigned bid_c, const unsigned n_cgroups,
                                                 const ShareWalk& walk = ShareWalk{}) {
  constexpr bool DIRECT = !std::is_same<OT, void>::value;
  static_assert(!(DIRECT || JOIN) || (WS && DIRECT != JOIN), "the waves of a workgroup share the request");
  constexpr float kUp = DIRECT && std::is_same<T, F16>::value ? 16384.f : 1.f;  // the weights in O are so many times those in l
  const int n = lane & 15, g = lane >> 4;  // query head (column) or 16-byte chunk of a row / token group or row of four
  // The waves of a workgroup: tw of them on neighbouring tasks (KV heads: their rows of a token lie side by side in memory
  // and are then fetched at about the same time), the rest on consecutive chunks of tokens.
  const int tw = WS ? 1 : (p.tasks_on_x & 7), cw = WS ? 1 : kMfmaWaves / tw;
  const int task = WS ? (int)bid_t : bid_t * tw + (wave & (tw - 1));
  if (task >= p.tasks) return;
  const int group = (int)(p.hq / p.hkv);
  const int sub_groups = (group + 15) / 16;
  const int kvh = task / sub_groups;
  const int sg = task % sub_groups;
  const int qh0 = kvh * group + sg * 16;
  const int nh = group - sg * 16 < 16 ? group - sg * 16 : 16;

  constexpr int kStep = WS ? kMfmaWaves * kMfmaBatch : kMfmaBatch;  // tokens from one of the wave's batches to its next
  const int bs = (int)p.block_seq;  // a multiple of 32 where blocks end within the walk (checked on the host); DIRECT walks a request whole, whatever it is
  int64_t fine_nblk = 0, blk_begin = 0;
  int t_begin, t_end, n_batches;
  int join_n = 0;  // (JOIN) partials of the request
  const int32_t* table;
  ShareSegment sl_seg, co_seg;  // (RANGE) where the slot numbers requested next and the batch computed next stand
  if constexpr (RANGE) {
    sl_seg = co_seg = share_segment(p, walk, walk.r, walk.x);
    t_begin = co_seg.t;
    t_end = co_seg.t_end;
    n_batches = (int)(walk.end - walk.x);
    table = p.req_to_tokens + (int64_t)co_seg.req * p.max_seq_len;
  } else {
    const int len = p.b_seqlen[b], req = p.b_req_idx[b];  // (both before anything is stored: scalar loads)
    int64_t nblk = len <= 0 ? 0 : ((int64_t)len + p.block_seq - 1) / p.block_seq;
    if (nblk > p.grid_blocks) nblk = p.grid_blocks;
    if (nblk > (p.num_blocks + p.row_mul - 1) / p.row_mul) nblk = (p.num_blocks + p.row_mul - 1) / p.row_mul;
    fine_nblk = len <= 0 ? 0 : ((int64_t)len + p.fine_block_seq - 1) / p.fine_block_seq;
    if (fine_nblk > p.num_blocks) fine_nblk = p.num_blocks;
    const unsigned n_chunks = n_cgroups * cw;
    const unsigned wave_chunk = bid_c * cw + (WS ? 0 : wave >> (tw == 4 ? 2 : tw == 2 ? 1 : 0));
    const unsigned chunk = LISTED ? wave_chunk : (wave_chunk + (unsigned)b) % n_chunks;  // (rotated by the request, as above)
    blk_begin = DIRECT ? 0 : (int64_t)chunk * p.blocks_per_wg;  // (WS: one block per workgroup)
    int64_t blk_end = blk_begin + p.blocks_per_wg;
    if (DIRECT || blk_end > nblk) blk_end = nblk;
    join_n = (int)nblk;
    if constexpr (DIRECT || JOIN) {
      if (nblk <= 0 && blk_begin == 0) {  // a request without tokens (the same for all waves)
        for (int i = wave * 64 + lane; i < nh * 32; i += kMfmaWaves * 64) {
          const int64_t elem = (b * p.hq + qh0) * 128 + i * 4;
          if constexpr (DIRECT) store4<OT>(p.o, elem, f32x4{0.f, 0.f, 0.f, 0.f});
          else store_result(p, elem, f32x4{0.f, 0.f, 0.f, 0.f});
        }
        if (wave == 0 && lane < nh) p.out_lse[b * p.hq + qh0 + lane] = -INFINITY;
        return;
      }
    }
    if (blk_begin >= blk_end) return;  // (WS: the same for the waves, which meet at a barrier below)
    t_begin = (int)(blk_begin * bs) + (WS ? wave * kMfmaBatch : 0);
    t_end = blk_end * bs > len ? len : (int)(blk_end * bs);
    n_batches = t_begin < t_end ? (t_end - t_begin + kStep - 1) / kStep : 0;
    table = p.req_to_tokens + (int64_t)req * p.max_seq_len;
  }
  int t_last = t_end - 1;

  const char* kbase = (const char*)p.k + ((int64_t)kvh * p.k_s1) * 2 + n * 16;
  const char* vbase = (const char*)p.v + ((int64_t)kvh * p.v_s1) * 2 + n * 16;
  const int64_t k_row_bytes = p.k_s0 * 2, v_row_bytes = p.v_s0 * 2;

  // Q^T as B operands: qb[ks] = Q[head n][32 ks + 8 g .. + 7] (zero for the spare columns)
  u32x4 qb[4];
  auto load_q = [&](const int64_t req) __attribute__((always_inline)) {
    const char* qrow = (const char*)p.q + ((req * p.hq + qh0 + (n < nh ? n : 0)) * 128 + 8 * g) * 2;
#pragma unroll
    for (int ks = 0; ks < 4; ks++) qb[ks] = n < nh ? *(const u32x4*)(qrow + ks * 64) : u32x4{0, 0, 0, 0};
  };
  load_q(RANGE ? co_seg.r : b);
  char* lds_k = lds + wave * kMfmaStage;
  char* lds_v = lds_k + kMfmaBatch * kMfmaKRow;
  // the lane writes chunk n of row 4 i + g (one register + 4 i rows as immediate), reads K row n (and 16 + n), chunk
  // 4 ks + g, and V through the transposing read: lane n of a group points at row 4 g + n / 4, elements 4 (n % 4) .. + 3 of a d-block
  char* kwrite0 = lds_k + g * kMfmaKRow + n * 16;
  char* vwrite0 = lds_v + g * kMfmaVRow + n * 16;
  const char* kread0 = lds_k + n * kMfmaKRow + g * 16;
  const int vread0 = (int)(uintptr_t)(__attribute__((address_space(3))) char*)lds_v + (4 * g + (n >> 2)) * kMfmaVRow + 8 * (n & 3);
  // Slot numbers of a batch: the lane loads chunk n of the rows of tokens 4 i + g; positions past the end repeat the last
  // row.  Issued from inline assembly like the data loads (one hand-kept count of outstanding loads).
  struct Slots {
    int v[8];
  };
  auto load_slots = [&](int t0, Slots& sl) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const int tok = t0 + 4 * i + g;
      const uint32_t off = (uint32_t)(tok < t_last ? tok : t_last) * 4u;  // (a row of the table is shorter than 2^31 entries)
      asm volatile("global_load_dword %0, %1, %2" : "=v"(sl.v[i]) : "v"(off), "s"(table) : "memory");
    }
  };
  // waits until at most N loads are outstanding and makes the slot numbers of `sl` usable
  auto wait_slots = [&](auto n_tag, Slots& sl) __attribute__((always_inline)) {
    constexpr int N = decltype(n_tag)::value;
    asm volatile("s_waitcnt vmcnt(%8)"
                 : "+v"(sl.v[0]), "+v"(sl.v[1]), "+v"(sl.v[2]), "+v"(sl.v[3]), "+v"(sl.v[4]), "+v"(sl.v[5]), "+v"(sl.v[6]), "+v"(sl.v[7])
                 : "n"(N)
                 : "memory");
  };
  // the 16 row loads of a batch: K rows into kr, V rows into vr (rows are read once: non-temporal)
  auto issue = [&](const Slots& sl, u32x4 (&kr)[8], u32x4 (&vr)[8]) __attribute__((always_inline)) {
    // (the 64-bit row address is formed next to its load, in a scratch register pair that dies with it: sixteen addresses
    // formed ahead of their loads would not fit the register file beside two batches of rows)
    const uint32_t krb = (uint32_t)k_row_bytes, vrb = (uint32_t)v_row_bytes;
#pragma unroll
    for (int i = 0; i < 8; i++) {
      uint64_t addr;
      asm volatile("v_mad_u64_u32 %1, vcc, %2, %3, %4\n\tglobal_load_dwordx4 %0, %1, off nt"
                   : "=v"(kr[i]), "=&v"(addr) : "v"(sl.v[i]), "s"(krb), "v"(kbase) : "vcc", "memory");
    }
#pragma unroll
    for (int i = 0; i < 8; i++) {
      uint64_t addr;
      asm volatile("v_mad_u64_u32 %1, vcc, %2, %3, %4\n\tglobal_load_dwordx4 %0, %1, off nt"
                   : "=v"(vr[i]), "=&v"(addr) : "v"(sl.v[i]), "s"(vrb), "v"(vbase) : "vcc", "memory");
    }
  };
  // waits until at most 24 loads (the slot numbers requested last and the next batch's rows) are outstanding and makes
  // kr / vr usable
  auto wait_rows = [&](u32x4 (&kr)[8], u32x4 (&vr)[8]) __attribute__((always_inline)) {
    asm volatile("s_waitcnt vmcnt(24)"
                 : "+v"(kr[0]), "+v"(kr[1]), "+v"(kr[2]), "+v"(kr[3]), "+v"(kr[4]), "+v"(kr[5]), "+v"(kr[6]), "+v"(kr[7]), "+v"(vr[0]),
                   "+v"(vr[1]), "+v"(vr[2]), "+v"(vr[3]), "+v"(vr[4]), "+v"(vr[5]), "+v"(vr[6]), "+v"(vr[7])
                 :
                 : "memory");
  };

  f32x4 oacc[8];
  float m = -INFINITY, l = 0.f;  // running maximum (log2 domain, the same in the four lanes of a head) / the lane's part of the sum
  auto reset = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int db = 0; db < 8; db++) oacc[db] = f32x4{0.f, 0.f, 0.f, 0.f};
    m = -INFINITY;
    l = 0.f;
  };
  reset();
  auto flush = [&](int64_t blk) __attribute__((always_inline)) {
    float lt = l + xlane16(l);
    lt += xlane32(lt);
    if (n < nh) {
      const float inv = 1.f / lt;  // a block holds at least one token
      const int64_t row = RANGE ? ((int64_t)walk.v + co_seg.r) * p.hq + qh0 + n : blk * p.row_mul * p.blk_rows + b * p.req_rows + qh0 + n;
      float* dst = p.mid_o + row * 128 + 4 * g;
      store_partial_row(dst, oacc, inv);
      if (g == 0) p.mid_lse[row] = (m + __builtin_amdgcn_logf(lt)) * kLn2;
      if (!RANGE) {
        // the rows of the blocks merged into this partial (row_mul <= 16: lane group g takes every fourth of them)
        for (int r = 1 + g; r < p.row_mul; r += 4)
          if (blk * p.row_mul + r < fine_nblk) p.mid_lse[(blk * p.row_mul + r) * p.blk_rows + b * p.req_rows + qh0 + n] = -INFINITY;
      }
    }
  };
  // one batch whose rows have arrived in kr / vr
  auto compute = [&](int t0, const u32x4 (&kr)[8], const u32x4 (&vr)[8]) __attribute__((always_inline)) {
    // rows into operand layout through the wave's LDS (the reads of the previous batch were consumed by its MFMAs)
#pragma unroll
    for (int i = 0; i < 8; i++) {
      *(u32x4*)(kwrite0 + 4 * i * kMfmaKRow) = kr[i];
      *(u32x4*)(vwrite0 + 4 * i * kMfmaVRow) = vr[i];
    }
    f32x4 s[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
      s[h] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 4; ks++) {
        const u32x4 ka = *(const u32x4*)(kread0 + h * 16 * kMfmaKRow + ks * 64);
        s[h] = Mfma16<T>::run(ka, qb[ks], s[h]);
      }
    }
    // s[h][r] = score of token t0 + 16 h + 4 g + r for head n
    float mx = -INFINITY;
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const bool valid = t0 + 16 * h + 4 * g + r < t_end;
        s[h][r] = valid ? s[h][r] * p.scale_log2 : -INFINITY;
        mx = fmaxf(mx, s[h][r]);
      }
    mx = fmaxf(mx, xlane16(mx));
    mx = fmaxf(mx, xlane32(mx));            // over the batch's 32 tokens (at least one is valid)
    const float m_new = fmaxf(m, mx);
    const float alpha = exp2_diff(m, m_new);
    if (__builtin_amdgcn_ballot_w64(m_new != m) != 0) {
#pragma unroll
      for (int db = 0; db < 8; db++) oacc[db] *= alpha;
      l *= alpha;
    }
    m = m_new;
    const float m_ref = DIRECT && m_new == -INFINITY ? 0.f : m_new;  // (scores of -inf weigh nothing, as in the lane kernel)
    float pv[8];
    float ps = 0.f;
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        pv[4 * h + r] = __builtin_amdgcn_exp2f(s[h][r] - m_ref);
        ps += pv[4 * h + r];
      }
    l += ps;
    // P^T as B operand: the lane's eight tokens are the contraction slots 8 g .. 8 g + 7, the order the V^T operand uses
    u32x4 phi, plo, prest;
    if (DIRECT && std::is_same<T, F16>::value) {
      // P in two parts of eleven bits, 2^14 times as large (which the result is divided by), so that a small weight keeps its bits too.
      // The parts are cut off and so none is below zero; nor is the second one zero beside a first one (but at least 2^-38 of the largest weight), or an
      // infinite V would turn into a NaN at it.  A weight of zero has no parts.  (Weights below 2^-38 have no first part, as those below
      // 2^-25 have none in the kernels of two launches.)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const float x0 = pv[2 * e] * kUp, x1 = pv[2 * e + 1] * kUp;
        phi[e] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(x0, x1));
        float h0, h1;
        unpack2<F16>(phi[e], h0, h1);
        plo[e] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(fmaxf(x0 - h0, fminf(x0, 0x1p-24f)), fmaxf(x1 - h1, fminf(x1, 0x1p-24f))));
      }
    } else if (std::is_same<T, F16>::value) {
#pragma unroll
      for (int e = 0; e < 4; e++) phi[e] = pack2<F16>(pv[2 * e], pv[2 * e + 1]);
    } else if (DIRECT) {
      // P in full, as the lane kernel has it for the launches that were its own: three parts of eight bits, cut off likewise
#pragma unroll
      for (int e = 0; e < 4; e++) {
        uint32_t hi[2], lo[2];
        float rest[2];
#pragma unroll
        for (int i = 0; i < 2; i++) {
          const float x = pv[2 * e + i];
          hi[i] = __builtin_bit_cast(uint32_t, x) & 0xffff0000u;
          const float least = fminf(x, 0x1p-126f), x1 = fmaxf(x - __builtin_bit_cast(float, hi[i]), least);
          lo[i] = __builtin_bit_cast(uint32_t, x1) & 0xffff0000u;
          rest[i] = fmaxf(x1 - __builtin_bit_cast(float, lo[i]), least);
        }
        phi[e] = (hi[0] >> 16) | hi[1];
        plo[e] = (lo[0] >> 16) | lo[1];
        prest[e] = pack2<BF16>(rest[0], rest[1]);
      }
    } else {
#pragma unroll
      for (int e = 0; e < 4; e++) {
        // high part: P truncated to bfloat16; low part: the rest, rounded
        const uint32_t h0 = __builtin_bit_cast(uint32_t, pv[2 * e]) & 0xffff0000u, h1 = __builtin_bit_cast(uint32_t, pv[2 * e + 1]) & 0xffff0000u;
        phi[e] = (h0 >> 16) | h1;
        plo[e] = pack2<BF16>(pv[2 * e] - __builtin_bit_cast(float, h0), pv[2 * e + 1] - __builtin_bit_cast(float, h1));
      }
    }
#pragma unroll
    for (int db = 0; db < 8; db++) {
      const i16x4 xa = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4*)(vread0 + db * 32));
      const i16x4 xb = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4*)(vread0 + db * 32 + 16 * kMfmaVRow));
      const u32x2 wa = __builtin_bit_cast(u32x2, xa), wb = __builtin_bit_cast(u32x2, xb);
      const u32x4 va = u32x4{wa[0], wa[1], wb[0], wb[1]};
      oacc[db] = Mfma16<T>::run(va, phi, oacc[db]);
      if (DIRECT || !std::is_same<T, F16>::value) oacc[db] = Mfma16<T>::run(va, plo, oacc[db]);
      if (DIRECT && !std::is_same<T, F16>::value) oacc[db] = Mfma16<T>::run(va, prest, oacc[db]);
    }
  };
  auto finish_batch = [&](int t0) __attribute__((always_inline)) {
    if (WS) return;  // (the block's partial is merged from the four waves after the loop)
    if constexpr (RANGE) {
      co_seg.t += kMfmaBatch;
      if (co_seg.t >= co_seg.t_end) {  // the share's part of this request is done
        flush(0);
        if (co_seg.x_end < walk.end) {
          reset();
          co_seg = share_segment(p, walk, co_seg.r + 1, co_seg.x_end);
          t_end = co_seg.t_end;
          load_q(co_seg.r);
          // the query has landed here, not at its first use in the loop, where the wait would be for the rows in flight in every trip
          asm volatile("" : "+v"(qb[0]), "+v"(qb[1]), "+v"(qb[2]), "+v"(qb[3]));
        }
      }
      return;
    }
    if ((t0 + kMfmaBatch - t_begin) % bs == 0 || t0 + kMfmaBatch >= t_end) {
      flush(blk_begin + (t0 - t_begin) / bs);
      reset();
    }
  };

  // Order of the loads, oldest first, when batch j is about to be computed:  rows(j) | slots(j+2) | rows(j+1).  Loads return
  // in order, so the wait for vmcnt(24) ends when rows(j) have landed and leaves the other two groups in flight (a partial's
  // stores in between count too and only make a wait longer); slots(j+1), which rows(j+1) were addressed with, were the
  // oldest group one wait earlier (that vmcnt(24), in front of an issue, is a no-op except in the first trip).
  u32x4 kr0[8], vr0[8], kr1[8], vr1[8];
  Slots s_even, s_odd;
  // the slot numbers of batch j, j counting up by one from call to call
  auto next_slots = [&](int j, Slots& sl) __attribute__((always_inline)) {
    if constexpr (RANGE) {
      load_slots(sl_seg.t, sl);  // (past the share's end: the last batch again, never used)
      if (sl_seg.t + kMfmaBatch < sl_seg.t_end) {
        sl_seg.t += kMfmaBatch;
      } else if (sl_seg.x_end < walk.end) {
        sl_seg = share_segment(p, walk, sl_seg.r + 1, sl_seg.x_end);
        t_last = sl_seg.t_end - 1;
        table = p.req_to_tokens + (int64_t)sl_seg.req * p.max_seq_len;
      }
    } else {
      load_slots(t_begin + j * kStep, sl);
    }
  };
  uint64_t* const word = JOIN ? arrivals_of(p, b * p.hq + qh0) : nullptr;
  uint64_t seen = 0;
  if (JOIN) seen = load_past_l2(word);
  next_slots(0, s_even);
  next_slots(1, s_odd);
  wait_slots(std::integral_constant<int, 8>{}, s_even);
  issue(s_even, kr0, vr0);
  // two batches per trip, so that the register set of a batch is a compile-time choice
  for (int j = 0; j < n_batches; j += 2) {
    next_slots(j + 2, s_even);                              // slots(j+2): rows(j) have been addressed
    wait_slots(std::integral_constant<int, 24>{}, s_odd);   // slots(j+1) usable
    issue(s_odd, kr1, vr1);                                 // rows(j+1) (past the end: the last row again, never used)
    wait_rows(kr0, vr0);
    {
      const int t0 = RANGE ? co_seg.t : t_begin + j * kStep;
      compute(t0, kr0, vr0);
      finish_batch(t0);
    }
    next_slots(j + 3, s_odd);                               // slots(j+3)
    wait_slots(std::integral_constant<int, 24>{}, s_even);  // slots(j+2) usable
    issue(s_even, kr0, vr0);                                // rows(j+2)
    wait_rows(kr1, vr1);
    if (j + 1 < n_batches) {
      const int t0 = RANGE ? co_seg.t : t_begin + (j + 1) * kStep;
      compute(t0, kr1, vr1);
      finish_batch(t0);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (rows requested past the end land before the registers are given back)
  uint64_t held = seen;
  if (JOIN && wave == 0 && lane == 0) held = start_arrivals(word, seen, p.arrivals, join_n);
  if constexpr (WS) {
    // The four partials of the block meet in LDS (each wave's own 17.5 KB: its last batch's operands have been consumed);
    // every wave then finishes two of the eight d-blocks.  A wave without a batch of its own brings m = -inf, l = 0.
    float lt = l + xlane16(l);
    lt += xlane32(lt);
    f32x4* mine = (f32x4*)(lds + wave * kMfmaStage);
#pragma unroll
    for (int db = 0; db < 8; db++) mine[db * 64 + lane] = oacc[db];
    // (as a float vector: __builtin_bit_cast applied to an element of an integer vector, bit_cast(float, v[1]), compiled to a
    // read of element 0 with this compiler)
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    *(f32x2*)(lds + wave * kMfmaStage + 8192 + lane * 8) = f32x2{m, lt};
    __syncthreads();
    float mi[kMfmaWaves], li[kMfmaWaves], M = -INFINITY;
#pragma unroll
    for (int w = 0; w < kMfmaWaves; w++) {
      const f32x2 ml = *(const f32x2*)(lds + w * kMfmaStage + 8192 + lane * 8);
      mi[w] = ml[0];
      li[w] = ml[1];
      M = fmaxf(M, mi[w]);
    }
    float L = 0.f;
#pragma unroll
    for (int w = 0; w < kMfmaWaves; w++) {
      mi[w] = exp2_diff(mi[w], M);  // (the weight of wave w's partial; 0 for one that saw no token)
      L += li[w] * mi[w];
    }
    if (n < nh) {
      const float inv = DIRECT && L == 0.f ? 0.f : 1.f / L * (1.f / kUp);  // a block holds at least one token (whose score may be -inf)
      const int64_t row = DIRECT ? b * p.hq + qh0 + n : blk_begin * p.row_mul * p.blk_rows + b * p.req_rows + qh0 + n;
#pragma unroll
      for (int d = 0; d < 2; d++) {
        const int db = 2 * wave + d;
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < kMfmaWaves; w++) acc += ((const f32x4*)(lds + w * kMfmaStage))[db * 64 + lane] * mi[w];
        if constexpr (DIRECT) store4<OT>(p.o, row * 128 + 16 * db + 4 * g, acc * inv);
        else if (JOIN) store_through(p.mid_o + row * 128 + 16 * db + 4 * g, acc * inv);
        else *(f32x4*)(p.mid_o + row * 128 + 16 * db + 4 * g) = acc * inv;
      }
      if (wave == 0) {
        float* lse = DIRECT ? p.out_lse : p.mid_lse;
        const float value = (M + __builtin_amdgcn_logf(L)) * kLn2;
        if (JOIN && g == 0) __hip_atomic_store(lse + row, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        else if (g == 0) lse[row] = value;
        if (!DIRECT && !JOIN)
          for (int r = 1 + g; r < p.row_mul; r += 4)
            if (blk_begin * p.row_mul + r < fine_nblk) p.mid_lse[(blk_begin * p.row_mul + r) * p.blk_rows + b * p.req_rows + qh0 + n] = -INFINITY;
      }
    }
    if constexpr (JOIN) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's part of the partial is in memory
      __syncthreads();                                  // ... and so are the others'
      uint32_t* const last = (uint32_t*)lds;
      if (wave == 0 && lane == 0) *last = arrive(word, seen, held, p.arrivals, join_n);
      __syncthreads();
      if (*last) join_partials(p, lds, lane, wave, b * p.hq + qh0, nh, b * p.req_rows + qh0, join_n);
    }
  }
}

template <typename T, bool WS>
__global__ __launch_bounds__(kMfmaWaves * 64, 2) void decode_stage1_mfma_kernel(Stage1Params p) {
  __shared__ __attribute__((aligned(1024))) char lds[kMfmaWaves * kMfmaStage];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool tasks_first = !WS && (p.tasks_on_x & 8) != 0;  // grid = (task groups, chunk groups, batch): a chunk's task groups are dispatched together
  stage1_mfma_unit<T, WS, false>(p, lds, lane, wave, blockIdx.z, tasks_first ? blockIdx.x : blockIdx.y, tasks_first ? blockIdx.y : blockIdx.x,
                                 tasks_first ? gridDim.y : gridDim.x);
}

// Short contexts in one launch: a workgroup takes all tokens of a (request, task), as the shape whose waves split a block does with a
// block's, and writes the result itself; no partials, no merge behind.  Bound by latency: request, slot numbers, rows, the four waves' parts,
// each behind the other; 128 tokens take 5.9 us, where two launches take 8.8 (4.4 each, whatever they do; replayed from a graph).
// The weights go to the matrix pipe in two (f16) or three (bf16) parts, as good as fp32: the error against 64 bits of the fp32 result
// is 1e-7 to 5e-7, where one f16 part leaves 2e-4, and two bf16 parts 5e-6.  The parts cost no time that shows: loads are waited for.
template <typename T, typename OT>
__global__ __launch_bounds__(kMfmaWaves * 64, 2) void decode_direct_kernel(Stage1Params p) {
  __shared__ __attribute__((aligned(1024))) char lds[kMfmaWaves * kMfmaStage];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  stage1_mfma_unit<T, true, false, false, OT>(p, lds, lane, wave, blockIdx.y, blockIdx.x, 0, 1);
}

// The shape whose waves split a block, with the merge in the launch (JOIN).
template <typename T>
__global__ __launch_bounds__(kMfmaWaves * 64, 2) void decode_joined_kernel(Stage1Params p) {
  __shared__ __attribute__((aligned(1024))) char lds[kMfmaWaves * kMfmaStage];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  stage1_mfma_unit<T, true, false, false, void, true>(p, lds, lane, wave, blockIdx.z, blockIdx.y, blockIdx.x, gridDim.x);
}

// The plain shape over a list of the units that exist.  The grid above has a workgroup for every (chunk group, task group)
// of the longest request times the batch, and the host does not know the lengths: a batch of one long request and many
// short ones is mostly workgroups that find nothing to do (one request of 131072 tokens with 255 of 512, 256 tokens per
// partial: a million workgroups for 5000 units; starting and ending them takes three times as long as the reads).  Here
// a fixed grid of two workgroups per CU walks the units: every workgroup first numbers the units of all requests (the
// first unit of each request, a prefix sum over the batch, in LDS), then takes units blockIdx.x, blockIdx.x + gridDim.x,
// ...; the request of a unit is found by bisection.  Within a request the task groups of a chunk group are
// neighbouring units, which run at the same time on neighbouring workgroups (all KV heads of a token are fetched together).
constexpr int kListedMaxBatch = 1024;
constexpr int64_t kListedFromWorkgroups = 32768;  // launches of the plain grid from which the list is walked instead
// ... and from a quarter of that when a partial covers 1024 tokens and more (the fused call's splits): with units that long
// a skewed batch has few of them, one to a CU at best, and the plain grid's empty workgroups stand in their way (131072 +
// 63 x 2048 tokens at 2048 per partial, 8192 workgroups: 0.217 -> 0.167 ms; at 1024, 16384 workgroups: 0.207 -> 0.176);
// batches of one length lose under one percent (64 x 65536 at 1024: 2.777 -> 2.80 ms).  At 256 tokens per partial the
// list costs an even batch more than that (config 3, 16384 workgroups: 947 -> 962 us) and stays with the larger grids.
constexpr int64_t kListedFromWorkgroupsCoarse = 8192;
constexpr int64_t kListedCoarseTokens = 1024;
// Equal shares from eight requests on wherever the plain shape would run, and for fewer from 2048 waves of 256 tokens on, two workgroups per CU.  Of less than two,
// where the CUs that hold two set the grid's time, those that gain whatever the lengths are (of the time of the grids, 3400 launches on four and more KV heads):
//   four to seven requests, 1345 to 1536 waves: of one length 0.87 to 1.01, of others 0.58 to 0.97 (us, 32/8: 5 x 8860 40.0 | 38.1, 4 of at most 11264 31.4 | 24.5).  Below that one length gains more (0.81 to 0.95)
//     but ragged ones of which few enough workgroups find tokens take up to 1.13 (6 of at most 6044 16/8 22.3 | 24.3), as two or three do there (3 of at most 15516 24/8 22.6 | 24.9); above it one length takes up to
//     1.09 (4 x 13569 8/8 42.5 | 44.8)
//   one request from 1025 waves on 0.74 to 0.99 (35000 tokens 32/8 36 | 30, 66000 64/8 67 | 52), except where the grid has nearly two workgroups per CU, to 1.12 (groups below four
//     from one and a half on), and there also nearly four, to 1.04
// Fewer than four KV heads, where a grid of the shape whose waves split a block stands against it, from more than 3072 waves on, and past whole rounds of that grid: one or two KV heads
// and eight requests and more 2049 to 2304 waves 0.52 to 1.02, 0.95 in the mean (past that, or of fewer requests, to 1.13: 3 of at most 205825 16/1 39.2 | 44.1; three KV heads, which leave a
// wave of a workgroup idle, to 1.12), with one KV head and 24 to a hundred requests also 1025 to 1280, 0.50 to 1.02, 0.74
// (fewer requests of different lengths to 1.28: 5 of at most 61952 16/1 23.4 | 30.0, 16 of at most 16896 22.2 | 23.7; four hundred of a block each to 1.19: 768 tokens 8/1 35.8 | 42.6); in between one length loses up to 16 %.
constexpr int64_t kSharesMinBatch = 8;
// Not where the rows of the partials' buffers hold less than half of the shares the chip has waves for: 256 requests of 256 tokens,
// GQA 32/8, are one share (2.9 ms) or a grid (57 us).  And not in place of a grid that one round of workgroups, one per CU, walks,
// if the rows hold fewer shares than the chip has waves for (24 requests of 1024 tokens, GQA 32/8, 73 shares: 30.1 us against 22.6; 33 of
// 512: 32.2 against 20.6), or if the requests are few and the longest one's blocks about equal (8 of 8000 GQA 32/8: 48.4 against 45.7, 32 of
// 384 MHA 32: 38.9 against 35.4, ragged 27.9 against 27.1; with unequal blocks shares win, 16 ragged ones up to 1500 in blocks of 1024, MHA 32:
// 45.7 against 55.7, and so they do for 128 ragged requests up to 1024: 56.7 against 65.1).  Past one round the shares win also where the
// rows cut them (65 requests of 257 tokens, GQA 32/8, 66 shares: 26.5 against 32.1; of 512 between 5 % slower and 2 % faster,
// ragged 27.6 against 31.2).
constexpr int64_t kSharesOneRoundBatch = 32;
constexpr int kShareUnits = 4;                    // a share holds at least so many units of kMfmaBatch tokens
template <typename T>
__global__ __launch_bounds__(kMfmaWaves * 64, 2) void decode_stage1_mfma_listed_kernel(Stage1Params p) {
  __shared__ __attribute__((aligned(1024))) char lds[kMfmaWaves * kMfmaStage];
  __shared__ uint32_t first_unit[kListedMaxBatch + 1];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tw = p.tasks_on_x & 7, cw = kMfmaWaves / tw;
  const uint32_t task_groups = (uint32_t)((p.tasks + tw - 1) / tw);
  const int batch = (int)p.batch;  // <= kListedMaxBatch (checked on the host)
  if (wave == 0) {
    const int64_t rows_avail = (p.num_blocks + p.row_mul - 1) / p.row_mul;
    uint32_t carry = 0;
    for (int b0 = 0; b0 < batch; b0 += 64) {
      const int bb = b0 + lane;
      uint32_t units = 0;
      if (bb < batch) {
        const int len = p.b_seqlen[bb];
        int64_t nblk = len <= 0 ? 0 : ((int64_t)len + p.block_seq - 1) / p.block_seq;  // (the same clamps as in the unit)
        if (nblk > p.grid_blocks) nblk = p.grid_blocks;
        if (nblk > rows_avail) nblk = rows_avail;
        const int64_t per_group = (int64_t)p.blocks_per_wg * cw;
        units = (uint32_t)((nblk + per_group - 1) / per_group) * task_groups;
      }
      uint32_t incl = units;  // inclusive prefix sum over the 64 lanes
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const uint32_t up = __shfl_up(incl, d, 64);
        if (lane >= d) incl += up;
      }
      if (bb < batch) first_unit[bb] = carry + incl - units;
      carry += __builtin_amdgcn_readlane(incl, 63);
    }
    if (lane == 0) first_unit[batch] = carry;
  }
  __syncthreads();
  const uint32_t total = first_unit[batch];
  for (uint32_t unit = blockIdx.x; unit < total; unit += gridDim.x) {
    // the request that holds the unit: first_unit[lo] <= unit < first_unit[hi] throughout (requests without units are skipped)
    int lo = 0, hi = batch;
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      const uint32_t f = __builtin_amdgcn_readfirstlane(first_unit[mid]);
      if (f <= unit) lo = mid;
      else hi = mid;
    }
    const uint32_t local = unit - __builtin_amdgcn_readfirstlane(first_unit[lo]);
    const uint32_t cgroup = local / task_groups;
    stage1_mfma_unit<T, false, true>(p, lds, lane, wave, lo, local - cgroup * task_groups, cgroup, 0);
  }
}

// The plain shape with the work dealt in equal shares (the fused call, whose partials are scratch).  All units of
// kMfmaBatch tokens of all requests, request after request, form one line, which the workgroups of a task group cut into V
// contiguous shares, one per wave that walks tokens; a wave computes its share of every request it touches into ONE
// partial.  Every wave gets the same number of tokens to within one batch whatever the lengths are, a request long or
// short costs one partial per share it touches instead of one per block (the partials, written while the gather
// saturates the memory system, cost eight times their bytes), and no split size has to be guessed from the longest request.
// V is worked out from the tokens that exist: a share per wave that walks tokens of a grid of one workgroup per CU, but none
// shorter than share_units units.  A launch costs about 7 us of start-up and finish plus its bytes at 6 to 6.6 TB/s; one
// workgroup per CU (four waves with two batches of rows in flight each, 128 KB) keeps HBM as busy as two do and leaves half as
// many partials: 24 requests of 200 to 4000 tokens, GQA 32/8, both launches 45.5 -> 39.3 us (56.4 with grids split by the
// longest request), 64 of 512 to 8192 150 -> 146, 64 of 4000 to 30000 588 -> 582.  Share v of request r leaves partial
// number v + r (the partials of a request lie side by side, and all of them are below V + batch: mid_o has a row per 256
// tokens of the longest request and request, which bounds V).
// Shares are handed to the workgroups first and to the waves of a workgroup that walk tokens second: few shares then sit on
// as many CUs.  Neighbouring workgroups hold the task groups of the same share (all KV heads of a token are fetched at
// about the same time).  The merge that follows (decode_merge_shares_kernel) works out the same shares.
struct Shares {
  uint32_t total, V;
  __device__ __forceinline__ Shares(uint32_t total_, uint32_t max_shares, uint32_t share_units) {
    total = total_;
    V = total / share_units;
    V = V > max_shares ? max_shares : V < 1 ? 1 : V;
  }
  // quotients of integers below 2^38 by integers below 2^27 are exact through a double: the fraction is 0 or at least 2^-27
  __device__ __forceinline__ uint32_t begin(uint32_t v) const { return (uint32_t)((double)v * (double)total / (double)V); }
  __device__ __forceinline__ uint32_t of(uint32_t unit) const { return (uint32_t)(((double)(unit + 1) * (double)V - 1.0) / (double)total); }
};
template <typename T>
__global__ __launch_bounds__(kMfmaWaves * 64, 2) void decode_stage1_mfma_range_kernel(Stage1Params p) {
  __shared__ __attribute__((aligned(1024))) char lds[kMfmaWaves * kMfmaStage];
  __shared__ uint32_t first_unit[kListedMaxBatch + 1];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tw = p.tasks_on_x & 7;
  const uint32_t task_groups = (uint32_t)((p.tasks + tw - 1) / tw);
  const int batch = (int)p.batch;  // <= kListedMaxBatch (checked on the host)
  // units in front of each request: a wave counts up to 64 requests in its registers, more go through LDS
  ShareWalk w;
  w.first_unit = first_unit;
  w.incl = 0;
  w.len = w.req = 0;
  uint32_t total;
  auto scan64 = [&](int len) __attribute__((always_inline)) {
    uint32_t s = share_units_of(len, kMfmaBatch, p.grid_blocks);
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const uint32_t up = __shfl_up(s, d, 64);
      if (lane >= d) s += up;
    }
    return s;
  };
  w.in_registers = batch <= 64;
  if (w.in_registers) {
    if (lane < batch) {
      w.len = p.b_seqlen[lane];
      w.req = p.b_req_idx[lane];
    }
    w.incl = scan64(w.len);
    total = __builtin_amdgcn_readlane(w.incl, 63);
  } else {
    if (wave == 0) {
      uint32_t carry = 0;
      if (lane == 0) first_unit[0] = 0;
      for (int b0 = 0; b0 < batch; b0 += 64) {
        const uint32_t s = scan64(b0 + lane < batch ? p.b_seqlen[b0 + lane] : 0);
        if (b0 + lane < batch) first_unit[b0 + lane + 1] = carry + s;
        carry += __builtin_amdgcn_readlane(s, 63);
      }
    }
    __syncthreads();
    total = first_unit[batch];
  }
  const Shares shares(total, (uint32_t)p.max_shares, (uint32_t)p.share_units);
  const uint32_t tg = blockIdx.x % task_groups;
  w.v = (uint32_t)(wave / tw) * (gridDim.x / task_groups) + blockIdx.x / task_groups;
  if (w.v >= shares.V) return;
  w.x = __builtin_amdgcn_readfirstlane(shares.begin(w.v));
  w.end = __builtin_amdgcn_readfirstlane(shares.begin(w.v + 1));
  if (w.x >= w.end) return;
  // the request that holds unit x: the last one whose first unit is not past it
  if (w.in_registers) {
    w.r = __builtin_popcountll(__builtin_amdgcn_ballot_w64(w.incl <= w.x));
  } else {
    int lo = 0, hi = batch;
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      const uint32_t f = __builtin_amdgcn_readfirstlane(first_unit[mid]);
      if (f <= w.x) lo = mid;
      else hi = mid;
    }
    w.r = lo;
  }
  stage1_mfma_unit<T, false, true, true>(p, lds, lane, wave, 0, tg, 0, 0, w);
}

// ------------------------------------------------------------------------------------
// Stage 2: one workgroup per (request, head), the heads of a request next to each other in the grid (a request much
// longer than the others then has all its workgroups start together, wherever it stands in the batch, instead of its
// last head at the very end of the launch); SL slices of D/4 lanes walk the block axis in parallel (the reference walks
// it serially, flash_decoding_stage2.cu:38-48), then merge through LDS.
// ------------------------------------------------------------------------------------
struct Stage2Params {
  void* o;
  float* out_lse;
  const int32_t* b_seqlen;
  const float* mid_o;
  const float* mid_lse;
  int64_t batch, heads, num_seq_blocks, block_seq;
  int64_t blk_rows, req_rows;  // rows of mid_o between consecutive blocks / requests
  int64_t grid_blocks;         // (SHARES) stage 1's bound on a request's units, from the longest request
  int64_t max_shares, share_units;  // (SHARES) as in Stage1Params
  int64_t lead_rows;                // rows in front of every request's blocks
};

template <typename OT, int D, int NT>
__global__ __launch_bounds__(NT) void decode_stage2_kernel(Stage2Params p) {
  constexpr int LPR = D / 4;      // lanes per row (float4 each)
  constexpr int SL = NT / LPR;    // slices walking the block axis
  const int64_t b = blockIdx.x / (uint32_t)p.heads, h = blockIdx.x % (uint32_t)p.heads;
  const int slice = threadIdx.x / LPR, c = threadIdx.x % LPR;
  const int len = p.b_seqlen[b];
  int64_t n = p.lead_rows + (len <= 0 ? 0 : ((int64_t)len + p.block_seq - 1) / p.block_seq);
  if (n > p.num_seq_blocks) n = p.num_seq_blocks;
  const int64_t row_stride = p.blk_rows;
  const int64_t row0 = b * p.req_rows + h;
  const int64_t out_row = b * p.heads + h;

  float M = -INFINITY, L = 0.f;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  auto fold = [&](float lse, const f32x4& tv) {
    if (lse == -INFINITY) return;  // an empty partial contributes nothing
    const float Mn = fmaxf(M, lse);
    const float so = exp2_diff(M * kLog2e, Mn * kLog2e);
    const float sn = __builtin_amdgcn_exp2f((lse - Mn) * kLog2e);
    acc = acc * so + tv * sn;
    L = L * so + sn;
    M = Mn;
  };
  // U rows and their log-sum-exps requested together, none waiting for another: with many requests in the batch the
  // partials of one request lie batch x heads rows apart (a megabyte and more) and every load pays the full latency; a
  // long request's merge is a chain of them.  Positions past the request's last block repeat that block and are
  // dropped; an empty partial's row is loaded like any other (it may hold anything: stage 1 leaves the rows it merged
  // into another one untouched) and dropped by its log-sum-exp.
  constexpr int U = 8;  // rows a slice has in flight (sixteen measured slower: the many short requests of a batch then ask for rows they drop)
  for (int64_t i = slice; i < n; i += U * SL) {
    float lse[U];
    f32x4 tv[U];
    bool holds[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int64_t e = i + u * SL < n ? i + u * SL : n - 1;
      holds[u] = i + u * SL < n;
      const int64_t row = e * row_stride + row0;
      lse[u] = p.mid_lse[row];
      tv[u] = *(const f32x4*)(p.mid_o + row * D + c * 4);
    }
#pragma unroll
    for (int u = 0; u < U; u++)
      if (holds[u]) fold(lse[u], tv[u]);
  }
  __shared__ float sM[SL], sL[SL];
  __shared__ f32x4 sAcc[SL][LPR];
  if (c == 0) {
    sM[slice] = M;
    sL[slice] = L;
  }
  sAcc[slice][c] = acc;
  __syncthreads();
  if (slice == 0) {
    float Mt = -INFINITY;
#pragma unroll
    for (int s = 0; s < SL; s++) Mt = fmaxf(Mt, sM[s]);
    float Lt = 0.f;
    f32x4 a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < SL; s++) {
      const float w = exp2_diff(sM[s] * kLog2e, Mt * kLog2e);
      Lt += sL[s] * w;
      a += sAcc[s][c] * w;
    }
    const float inv = Lt > 0.f ? 1.f / Lt : 0.f;
    store4<OT>(p.o, out_row * D + c * 4, a * inv);
    if (c == 0) p.out_lse[out_row] = Lt > 0.f ? Mt + __builtin_amdgcn_logf(Lt) * kLn2 : -INFINITY;
  }
}

// The merge behind decode_stage1_mfma_range_kernel: W waves per (request, head), 4 / W pairs per workgroup (heads of one
// request; sixteen waves: one pair).  Every wave counts the units in front of its request and in all and knows from them the first and the last
// share that reach into the request: their partials are consecutive rows.  Half a wave reads a row (16 bytes a lane), eight
// rows and their log-sum-exps in flight per half wave.  Bound by its chain of dependent loads (the argument block, the lengths, the rows)
// and, from a few thousand pairs on, by the workgroups' turn-over: with a whole workgroup of eight slices per pair, as in
// decode_stage2_kernel, 128 requests with 32 heads took 10.2 us for one to three rows each.
template <typename OT, int W>
__global__ __launch_bounds__(W > 4 ? W * 64 : 256) void decode_merge_shares_kernel(Stage2Params p) {
  constexpr int D = 128, U = 8;
  constexpr int PAIRS = W > 4 ? 1 : 4 / W;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t head_groups = ((uint32_t)p.heads + PAIRS - 1) / PAIRS;
  const int b = blockIdx.x / head_groups;
  const int h = (int)(blockIdx.x % head_groups) * PAIRS + wave / W;
  uint32_t pre = 0, tot = 0;
  for (int i = lane; i < (int)p.batch; i += 64) {
    const uint32_t u = share_units_of(p.b_seqlen[i], kMfmaBatch, p.grid_blocks);
    tot += u;
    pre += i < b ? u : 0u;
  }
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) {
    pre += __shfl_xor(pre, d, 64);
    tot += __shfl_xor(tot, d, 64);
  }
  const uint32_t units = share_units_of(p.b_seqlen[b], kMfmaBatch, p.grid_blocks);
  const bool live = h < (int)p.heads;  // (the last group of heads may be short)
  int n = 0;
  int64_t row0 = 0;
  if (units > 0 && live) {
    const Shares shares(tot, (uint32_t)p.max_shares, (uint32_t)p.share_units);
    const uint32_t v0 = shares.of(pre), v1 = shares.of(pre + units - 1);
    n = (int)(v1 - v0) + 1;
    row0 = ((int64_t)v0 + b) * p.heads + h;
  }
  const int half = lane >> 5, c = lane & 31;
  const int slice = (wave % W) * 2 + half;
  float M = -INFINITY, L = 0.f;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int i = 0; i < n; i += U * 2 * W) {  // (i and n are the same for the whole wave)
    float lse[U];
    f32x4 tv[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int e = i + u * 2 * W + slice;
      const int64_t row = row0 + (int64_t)(e < n ? e : n - 1) * p.heads;
      lse[u] = e < n ? p.mid_lse[row] : -INFINITY;
      tv[u] = *(const f32x4*)(p.mid_o + row * D + c * 4);
    }
    float Mn = M;
#pragma unroll
    for (int u = 0; u < U; u++) Mn = fmaxf(Mn, lse[u]);
    const float so = exp2_diff(M * kLog2e, Mn * kLog2e);
    acc *= so;
    L *= so;
#pragma unroll
    for (int u = 0; u < U; u++) {
      const float w = exp2_diff(lse[u] * kLog2e, Mn * kLog2e);  // (0 past the last row)
      acc += tv[u] * w;
      L += w;
    }
    M = Mn;
  }
  auto join = [&](float Mo, float Lo, const f32x4& ao) {
    const float Mn = fmaxf(M, Mo);
    const float a = exp2_diff(M * kLog2e, Mn * kLog2e), o = exp2_diff(Mo * kLog2e, Mn * kLog2e);
    acc = acc * a + ao * o;
    L = L * a + Lo * o;
    M = Mn;
  };
  {
    f32x4 ao;
#pragma unroll
    for (int e = 0; e < 4; e++) ao[e] = __shfl_xor(acc[e], 32, 64);
    const float Mo = __shfl_xor(M, 32, 64), Lo = __shfl_xor(L, 32, 64);
    join(Mo, Lo, ao);
  }
  if constexpr (W > 1) {
    __shared__ float sM[W], sL[W];
    __shared__ f32x4 sAcc[W][32];
    if (half == 0) sAcc[wave][c] = acc;
    if (lane == 0) {
      sM[wave] = M;
      sL[wave] = L;
    }
    __syncthreads();
    if (wave != 0) return;
    if constexpr (W <= 4) {
#pragma unroll
      for (int w = 1; w < W; w++) join(sM[w], sL[w], sAcc[w][c]);
    } else {  // (none of the sixteen waits for another)
#pragma unroll
      for (int w = 1; w < W; w++) M = fmaxf(M, sM[w]);
      acc = f32x4{0.f, 0.f, 0.f, 0.f};
      L = 0.f;
#pragma unroll
      for (int w = 0; w < W; w++) {
        const float x = exp2_diff(sM[w] * kLog2e, M * kLog2e);
        acc += sAcc[w][c] * x;
        L += sL[w] * x;
      }
    }
  }
  if (half == 0 && live) {
    const int64_t out_row = (int64_t)b * p.heads + h;
    const float inv = L > 0.f ? 1.f / L : 0.f;
    store4<OT>(p.o, out_row * D + c * 4, acc * inv);
    if (c == 0) p.out_lse[out_row] = L > 0.f ? M + __builtin_amdgcn_logf(L) * kLn2 : -INFINITY;
  }
}

constexpr uint32_t kWideMergePairs = 64;
// What the fused call allows stage 1 to do beside it: merge its partials itself (JOIN), which leaves `done` set.
struct JoinPlan {
  const lsattn_decode_stage2_args* s2;
  bool done = false;
};
// Where a launch's counts of arrivals start: 64 bits that another launch does not have, far from any other's in all likelihood.
static uint64_t next_arrivals() {
  static std::atomic<uint64_t> launches{(uint64_t)std::chrono::steady_clock::now().time_since_epoch().count()};
  uint64_t x = launches.fetch_add(1, std::memory_order_relaxed) * 0x9e3779b97f4a7c15ull;  // (splitmix64, Steele et al. 2014)
  x = (x ^ (x >> 30)) * 0xbf58476d1ce4e5b9ull;
  x = (x ^ (x >> 27)) * 0x94d049bb133111ebull;
  return x ^ (x >> 31);
}
// Which launches merge their own partials.  `partials` per request at most, of `heads` query heads per task; workgroups of the grid.  The last
// workgroup reads the partials alone, at some 50 GB/s: up to max_rows of them (one memory latency, 2 to 2.5 us behind the kernel's
// work, where a second launch takes 3.5 and more), half of that where two workgroups per CU are busy with rows of their own.
// Measured over 108 launches (two launches | one, us a call, eager; and replayed from a graph), GQA 32/8:
//   1 x 2048 11.9 | 10.9 (9.5 | 9.3)   4 x 1500 12.7 | 10.6 (11.2 | 10.2)   6 of 87..700 12.5 | 11.2 (10.7 | 10.0)   16 x 900 18.4 | 16.7 (17.9 | 17.2)
//   1 x 8192, 32 partials, 13.4 | 12.3 (13.1 | 12.5)   1 x 16384, 64, 20.3 | 20.3 (20.3 | 21.0, not taken)   2 x 8000 19.0 | 18.6 (18.7 | 19.0, not taken)
// eight heads per task: 1 x 2048 8/1 10.5 | 9.6   1 x 3000 8/1, 96 rows, 11.1 | 10.8 (10.4 | 10.6, not taken)   1 x 8000 8/1, 256, 11.4 | 13.0 (not taken)
// the lane kernel: 1 x 2048 32/32 10.6 | 9.5   10 x 400 24/8 14.0 | 13.1   4 x 5000 24/8, 60 rows, 640 workgroups, 24.8 | 25.4 (not taken)
// sixteen heads: 1 x 1500 64/4, 96 rows in two turns, 12.0 | 12.8 (not taken).
// Launches of more than a workgroup per CU, replayed from a graph (3000 launches): up to two per CU in blocks of up to 512 tokens and 64 rows 0.83 to 1.03; not taken: 65 to 128 rows (8 of at most 7935
// 8/2 14.8 | 15.5), blocks of 1024 (40 x 10140 4/1 40.0 | 41.8), more workgroups (40 x 4608 8/2 36.7 | 42.6, 64 x 1535 8/2 24.5 | 28.0), and a request's only partial (400 x 768 8/1 35.7 | 42.6): partials are
// stored through to memory, which the other workgroups' reads wait behind.  65 to 128 rows of few workgroups: eager 0.90 to 1.01, replayed 0.95 to 1.08 (3 of at most 8092 4/1 10.8 | 11.6).
// Whether the runtime knows p as memory of the current GPU's own: not the host's, managed, or another GPU's, where the counts' 64-bit atomics at the scope of
// one GPU are not sure to work.  (0.2 us, of launches that would merge only; a tensor labelled with this GPU may wrap any of them.)
static bool is_memory_of_this_gpu(const void* p) {
  hipPointerAttribute_t at = {};
  int device = -1;
  if (hipPointerGetAttributes(&at, p) != hipSuccess || hipGetDevice(&device) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return at.type == hipMemoryTypeDevice && !at.isManaged && at.device == device;
}
static bool join_takes(JoinPlan* join, Stage1Params& p, int64_t partials, int64_t heads, int64_t max_rows, int64_t workgroups) {
  if (workgroups > kCUs && max_rows > 64) max_rows = 64;
  if (workgroups >= 2 * kCUs) max_rows /= 2;
  if (partials < 2 || workgroups > 2 * kCUs || (workgroups > kCUs && p.block_seq > 512)) return false;
  if (!join || p.row_mul != 1 || partials > kJoinMaxPartials || heads > 8 || partials * heads > max_rows || (partials * p.blk_rows + heads) * 512 > 0x7fffffff) return false;
  if (!is_memory_of_this_gpu(join->s2->o)) return false;
  join->done = true;
  p.o = join->s2->o;
  p.out_lse = join->s2->out_logexpsum;
  p.o_dtype = join->s2->o_dtype;
  p.arrivals = next_arrivals();
  return true;
}

template <typename T, int GT, int HR>
static int launch_stage1(const lsattn_decode_stage1_args* a, hipStream_t st, JoinPlan* join) {
  constexpr int NW = 4;  // waves (tasks) per workgroup; 8 measured no faster
  Stage1Params p;
  p.mid_o = a->mid_o;
  p.mid_lse = a->mid_o_logexpsum;
  p.q = a->q;
  p.k = a->k;
  p.v = a->v;
  p.k_s0 = a->k_stride_0;
  p.k_s1 = a->k_stride_1;
  p.v_s0 = a->v_stride_0;
  p.v_s1 = a->v_stride_1;
  p.scale_log2 = a->sm_scale * kLog2e;
  p.req_to_tokens = a->req_to_tokens;
  p.b_req_idx = a->b_req_idx;
  p.b_seqlen = a->b_seqlen;
  p.batch = a->batch;
  p.hq = a->num_q_heads;
  p.hkv = a->num_kv_heads;
  p.num_blocks = a->num_blocks;
  p.blk_rows = a->partials_by_request ? a->num_q_heads : a->batch * a->num_q_heads;
  p.req_rows = a->partials_by_request ? a->num_blocks * a->num_q_heads : a->num_q_heads;
  p.max_seq_len = a->max_seq_len;
  p.row_mul = a->merge_blocks > 1 ? a->merge_blocks : 1;
  p.fine_block_seq = a->seq_block_size;
  p.block_seq = a->seq_block_size * p.row_mul;
  p.grid_blocks = (a->max_len_in_batch + p.block_seq - 1) / p.block_seq;  // stage1.cu:211, in partials computed
  const int group = (int)(a->num_q_heads / a->num_kv_heads);
  p.tasks = (int)a->num_kv_heads * ((group + GT * HR - 1) / (GT * HR));
  const int wgs_y = (p.tasks + NW - 1) / NW;
  // a workgroup walks consecutive blocks until it has covered at least 256 tokens (smaller units measured slower for
  // short blocks, larger ones lose to tail imbalance)
  constexpr int64_t kTokensPerWorkgroup = 256;
  int64_t per_wg = (kTokensPerWorkgroup + p.block_seq - 1) / p.block_seq;
  if (per_wg < 1) per_wg = 1;
  const int64_t rows_avail = (a->num_blocks + p.row_mul - 1) / p.row_mul;
  int64_t nblk = p.grid_blocks < rows_avail ? p.grid_blocks : rows_avail;
  if (nblk < 1) return LSATTN_OK;
  p.blocks_per_wg = (int32_t)per_wg;
  const int64_t chunks = (nblk + per_wg - 1) / per_wg;
  if (chunks > 0x7fffffff || a->batch > 65535 || wgs_y > 65535) return LSATTN_ERR_INVALID_ARG;
  // A launch of less than one workgroup per CU leaves most of the chip's load slots empty: the waves of a workgroup then
  // share one task and split each block's tokens (measured: 64 workgroups, one request of 8192 tokens with 8 KV heads,
  // 19.9 -> 10.0 us; from 256 workgroups on it gains nothing; blocks shorter than 32 tokens per wave cannot use it).
  const bool once = group <= GT * HR;
  // ... and so does a launch with fewer tasks than a workgroup has waves (one or two KV heads: the other waves would idle)
  const bool split = (chunks * wgs_y * a->batch < 256 || p.tasks < NW) && p.block_seq >= 32 * NW && p.tasks <= 65535;
  if (split) {
    p.tasks_on_x = chunks <= 65535;
    dim3 grid = p.tasks_on_x ? dim3((unsigned)p.tasks, (unsigned)chunks, (unsigned)a->batch)
                             : dim3((unsigned)chunks, (unsigned)p.tasks, (unsigned)a->batch);
    if constexpr (HR == 1) {
      if (once && join_takes(join, p, nblk, group, 64, chunks * p.tasks * a->batch)) {
        LSATTN_LAUNCH_KERNEL((decode_stage1_kernel<T, GT, NW, true, true, 1, true>), grid, dim3(NW * 64), 0, st, p);
        return check_launch();
      }
    }
    if (once) LSATTN_LAUNCH_KERNEL((decode_stage1_kernel<T, GT, NW, true, true, HR>), grid, dim3(NW * 64), 0, st, p);
    else LSATTN_LAUNCH_KERNEL((decode_stage1_kernel<T, GT, NW, true, false, HR>), grid, dim3(NW * 64), 0, st, p);
    return check_launch();
  }
  p.tasks_on_x = wgs_y <= 2 && chunks <= 65535;  // with more task groups per chunk (MHA, 32 KV heads) it measured 2 % slower
  dim3 grid = p.tasks_on_x ? dim3((unsigned)wgs_y, (unsigned)chunks, (unsigned)a->batch)
                           : dim3((unsigned)chunks, (unsigned)wgs_y, (unsigned)a->batch);
  if (once) LSATTN_LAUNCH_KERNEL((decode_stage1_kernel<T, GT, NW, false, true, HR>), grid, dim3(NW * 64), 0, st, p);
  else LSATTN_LAUNCH_KERNEL((decode_stage1_kernel<T, GT, NW, false, false, HR>), grid, dim3(NW * 64), 0, st, p);
  return check_launch();
}

// Waves of the plain shape up to which the shape whose waves split a block runs instead, on four and more KV heads.  Of the plain shape's time, 1700 launches:
// 513 to 544 waves 0.66 to 0.99 where the lengths differ, 0.94 to 1.02 where they do not (12 of at most 2716 16/4 20.0 | 16.7 us); 545 to 576 0.67 to 1.02, 0.99 to 1.09 (12 of 1281 32/8
// 21.1 | 22.6), not taken.
constexpr int64_t kSplitMaxWaves = 544;
// Large launches: the matrix-pipe kernel, when its conditions hold (blocks a multiple of 32 tokens, enough waves to fill
// the chip); lsattn_set_tuning forces the choice where the conditions allow it (tuning, tests).
// What the fused call hands to stage 1 and on to the merge behind it.
struct SharesPlan {
  int64_t units;           // in: kMfmaBatch-token units of the longest request, in whole blocks of 256 tokens
  int64_t rows;            // in: rows of the partials' buffers per request, as far as the longest request goes
  int64_t max_shares = 0;  // out: 0 if the launch was none for equal shares
};

// `shares`: deal the blocks in equal shares (decode_stage1_mfma_range_kernel) or launch nothing (*taken stays false).
template <typename T> static int launch_stage1_mfma(const lsattn_decode_stage1_args* a, hipStream_t st, bool* taken, SharesPlan* shares = nullptr,
                                                    JoinPlan* join = nullptr) {
  *taken = false;
  const int group = (int)(a->num_q_heads / a->num_kv_heads);
  Stage1Params p;
  p.mid_o = a->mid_o;
  p.mid_lse = a->mid_o_logexpsum;
  p.q = a->q;
  p.k = a->k;
  p.v = a->v;
  p.k_s0 = a->k_stride_0;
  p.k_s1 = a->k_stride_1;
  p.v_s0 = a->v_stride_0;
  p.v_s1 = a->v_stride_1;
  p.scale_log2 = a->sm_scale * kLog2e;
  p.req_to_tokens = a->req_to_tokens;
  p.b_req_idx = a->b_req_idx;
  p.b_seqlen = a->b_seqlen;
  p.batch = a->batch;
  p.hq = a->num_q_heads;
  p.hkv = a->num_kv_heads;
  p.num_blocks = a->num_blocks;
  p.blk_rows = a->partials_by_request ? a->num_q_heads : a->batch * a->num_q_heads;
  p.req_rows = a->partials_by_request ? a->num_blocks * a->num_q_heads : a->num_q_heads;
  p.max_seq_len = a->max_seq_len;
  p.row_mul = a->merge_blocks > 1 ? a->merge_blocks : 1;
  p.fine_block_seq = a->seq_block_size;
  p.block_seq = a->seq_block_size * p.row_mul;
  p.grid_blocks = (a->max_len_in_batch + p.block_seq - 1) / p.block_seq;
  if (p.block_seq % kMfmaBatch || a->k_stride_0 >= (1 << 30) || a->v_stride_0 >= (1 << 30)) return LSATTN_OK;
  p.tasks = (int)a->num_kv_heads * ((group + 15) / 16);
  int64_t per_wave = (256 + p.block_seq - 1) / p.block_seq;  // a wave walks at least 256 tokens
  if (per_wave < 1) per_wave = 1;
  const int64_t rows_avail = (a->num_blocks + p.row_mul - 1) / p.row_mul;
  const int64_t nblk = p.grid_blocks < rows_avail ? p.grid_blocks : rows_avail;
  if (nblk < 1) return LSATTN_OK;
  p.blocks_per_wg = (int32_t)per_wave;
  const int64_t chunks = (nblk + per_wave - 1) / per_wave;
  const int tw = p.tasks >= 4 ? 4 : p.tasks >= 2 ? 2 : 1, cw = kMfmaWaves / tw;
  const int64_t wgs_x = (chunks + cw - 1) / cw, wgs_y = (p.tasks + tw - 1) / tw;
  if (wgs_x > 0x7fffffff || a->batch > 65535 || wgs_y > 65535) return LSATTN_OK;
  // Which shape, by the launch's size in waves of the plain shape (256 tokens x task x request; measured):
  //   groups of four and more query heads per KV head: up to kSplitMaxWaves waves (3072 on fewer than four KV heads, where the plain
  //     shape has no neighbouring heads to put side by side) the shape whose four waves split a block (a launch of 8 to 512
  //     plain waves runs 30-45 % shorter with it than with either other kernel), above that the plain shape;
  //   smaller groups (most of an MFMA's sixteen columns idle): the plain shape from 768 waves, below that the lane kernel.
  const int64_t waves = chunks * p.tasks * a->batch;
  const bool can_split = p.block_seq % (kMfmaWaves * kMfmaBatch) == 0 && nblk <= 0x7fffffff;
  //   (A few more of the plain shape's workgroups than one per CU, 1025 to 1536 waves on four and more KV heads, split among a block's waves, 1200 launches of both stages
  //     at 256 tokens a block: 0.53 to 1.0 of the time where the lengths differ and some CUs held two, but up to 1.23 where few enough workgroups found tokens, and 1.06 to 1.21 for one
  //     request on 16 or 32 KV heads.  The host cannot tell them apart: not taken.)
  bool split_waves = group >= 4 && can_split && waves <= (p.tasks < 4 ? 3072 : kSplitMaxWaves);
  bool use = !split_waves && waves >= (group >= 4 ? 513 : 768);
  const Tuning tn = tuning();  // (lsattn_set_tuning: tuning and tests)
  if (tn.decode_stage1 == LSATTN_DECODE_STAGE1_LANE) use = split_waves = false;
  if (tn.decode_stage1 == LSATTN_DECODE_STAGE1_MFMA) use = true, split_waves = false;
  if (tn.decode_stage1 == LSATTN_DECODE_STAGE1_SPLIT && can_split) use = false, split_waves = true;
  if (shares) {
    const int64_t task_groups = (p.tasks + tw - 1) / tw;
    const bool forced = tn.decode_listed == LSATTN_DECODE_LISTED_SHARES;  // (tests: whatever the launch's size)
    if (tn.decode_listed == LSATTN_DECODE_LISTED_OFF || tn.decode_listed == LSATTN_DECODE_LISTED_ON) return LSATTN_OK;
    int64_t per_group = kCUs / task_groups;  // workgroups per task group: one workgroup per CU in all
    if (per_group < 1 || p.row_mul != 1 || a->batch > kListedMaxBatch || shares->units * a->batch > 0x7ffffff) return LSATTN_OK;
    int64_t max_shares = per_group * cw;
    const int64_t by_tokens = shares->units * a->batch / kShareUnits;
    if (max_shares > by_tokens) max_shares = by_tokens > 0 ? by_tokens : 1;
    // partials are numbered below V + batch - 1: the rows of the buffers that the longest request can reach
    const int64_t wanted = max_shares, by_rows = a->batch * (shares->rows - 1) + 1;
    if (max_shares > by_rows) max_shares = by_rows;
    if (!forced && tn.decode_stage1 != 0) return LSATTN_OK;
    // (waves of the plain shape at 256 tokens each, whatever the split asked for; the shape whose waves split a block keeps its launches)
    const int64_t waves256 = (shares->units * kMfmaBatch + 255) / 256 * p.tasks * a->batch;
    const bool past_rounds = group >= 4 && p.tasks < 3 && a->batch >= 8 && ((waves256 > 8 * kCUs && waves256 <= 9 * kCUs) ||
                                                          (p.tasks == 1 && a->batch >= 24 && a->batch <= 100 && waves256 > 4 * kCUs && waves256 <= 5 * kCUs));
    const bool large = past_rounds || waves256 >= (group < 4 ? 768 : p.tasks < 4 ? 12 * kCUs + 1 : kSplitMaxWaves + 1);
    const bool few = a->batch > 1 && a->batch < kSharesMinBatch && waves256 < 8 * kCUs && (a->batch < 4 || 4 * waves256 <= 21 * kCUs || waves256 > 6 * kCUs);
    // (one request by the blocks it fills: a last block of a few tokens makes no round of its own, 1 x 32769 tokens 32/8 29.4 | 30.6)
    const int64_t full = a->max_len_in_batch / 256 * p.tasks;
    const bool nearly_two = full > (group < 4 ? 6 : 7) * kCUs && full <= 8 * kCUs, nearly_four = group < 4 && full > 13 * kCUs && full <= 16 * kCUs;
    const bool one = a->batch < 2 && (p.tasks < 4 || full <= 4 * kCUs || nearly_two || nearly_four);
    if (!forced && (!large || few || one)) return LSATTN_OK;
    // Launches that the lane kernel would take (in blocks as coarse as the split asked for they may be few waves): it multiplies V by fp32 weights where V is bf16, this kernel by two bf16
    // parts of them (error against 64 bits 4e-7 | 4.8e-6: two of 131870 tokens, 2/1 heads; one of 65936, 10/5), and f16 weights round a little worse here (eight launches, in the mean
    // 1.92e-4 | 2.01e-4).  So only the large ones.
    const bool lane = !use && !split_waves;
    if (!forced && lane && (a->batch < 2 || (a->batch < kSharesMinBatch && waves256 < 8 * kCUs) || (group >= 4 && p.tasks < 4 && waves256 <= 12 * kCUs))) return LSATTN_OK;
    // Short contexts, whose rows hold too few shares (a longest request of up to 256 tokens one share, whatever the batch),
    // and grids of one round of workgroups, see kSharesOneRoundBatch.
    const int64_t wgs = wgs_x * wgs_y * a->batch;
    const bool one_round = wgs > kCUs / 2 && wgs <= kCUs;
    const bool even = nblk == 1 || a->max_len_in_batch * 8 >= nblk * p.block_seq * 7;
    if (!forced && (by_rows * 2 < wanted || (one_round && (by_rows < wanted || (even && a->batch <= kSharesOneRoundBatch))))) return LSATTN_OK;
    if (per_group > max_shares) per_group = max_shares;
    *taken = true;
    shares->max_shares = max_shares;
    p.max_shares = (int32_t)max_shares;
    p.share_units = kShareUnits;
    p.block_seq = p.fine_block_seq = kMfmaBatch;
    p.grid_blocks = shares->units;
    p.tasks_on_x = tw;
    LSATTN_LAUNCH_KERNEL((decode_stage1_mfma_range_kernel<T>), dim3((unsigned)(per_group * task_groups)), dim3(kMfmaWaves * 64), 0, st, p);
    return check_launch();
  }
  if (split_waves) {
    *taken = true;
    p.blocks_per_wg = 1;
    p.tasks_on_x = 1;
    if (join_takes(join, p, nblk, group, group <= 4 ? 128 : 64, nblk * p.tasks * a->batch)) {
      LSATTN_LAUNCH_KERNEL((decode_joined_kernel<T>), dim3((unsigned)nblk, (unsigned)p.tasks, (unsigned)a->batch), dim3(kMfmaWaves * 64), 0, st, p);
      return check_launch();
    }
    LSATTN_LAUNCH_KERNEL((decode_stage1_mfma_kernel<T, true>), dim3((unsigned)nblk, (unsigned)p.tasks, (unsigned)a->batch), dim3(kMfmaWaves * 64),
                       0, st, p);
    return check_launch();
  }
  if (!use) return LSATTN_OK;
  *taken = true;
  // The task groups of a chunk are dispatched one after the other (x runs fastest), so that all KV heads of a token are
  // fetched at about the same time: config 3's shape 6.03 -> 6.17 TB/s, 32 KV heads 6.0 -> 6.5.
  const bool tasks_first = wgs_y > 1 && wgs_x <= 65535;
  p.tasks_on_x = tw | (tasks_first ? 8 : 0);  // (this kernel: waves of a workgroup on neighbouring tasks; the grid's order)
  // Launches of very many workgroups walk a list of the units that exist instead (see the kernel): most of such a grid
  // is empty whenever the batch mixes long and short requests, which the host cannot see.
  // lsattn_set_tuning overrides the choice (tuning and tests).
  const int64_t wgs_total = wgs_x * wgs_y * a->batch;
  bool listed = wgs_total >= kListedFromWorkgroups || (a->seq_block_size >= kListedCoarseTokens && wgs_total >= kListedFromWorkgroupsCoarse);
  if (tn.decode_listed == LSATTN_DECODE_LISTED_OFF) listed = false;
  if (tn.decode_listed == LSATTN_DECODE_LISTED_ON) listed = true;
  if (listed && a->batch <= kListedMaxBatch && wgs_total <= 0x7fffffff) {
    const int64_t resident = 2 * kCUs;  // two workgroups of this kernel per CU
    LSATTN_LAUNCH_KERNEL((decode_stage1_mfma_listed_kernel<T>), dim3((unsigned)(wgs_total < resident ? wgs_total : resident)),
                       dim3(kMfmaWaves * 64), 0, st, p);
    return check_launch();
  }
  const dim3 grid = tasks_first ? dim3((unsigned)wgs_y, (unsigned)wgs_x, (unsigned)a->batch) : dim3((unsigned)wgs_x, (unsigned)wgs_y, (unsigned)a->batch);
  LSATTN_LAUNCH_KERNEL((decode_stage1_mfma_kernel<T, false>), grid, dim3(kMfmaWaves * 64), 0, st, p);
  return check_launch();
}

// The result is written while other workgroups still read.  Whether it lies over the pool's rows or the table only the caller knows (their
// extents are not in the arguments).  Not where it lies over the queries, unless row by row and each workgroup reads its own first
// (`rows_may_match`), or over the lengths and rows of the requests.
static bool result_is_apart(const lsattn_decode_stage1_args* a, const lsattn_decode_stage2_args* s2, bool rows_may_match) {
  if (s2->o_is_apart != 1 && s2->o_is_apart != 2) return false;
  const int64_t pairs = a->batch * a->num_q_heads;
  auto apart = [](const void* x, int64_t nx, const void* y, int64_t ny) { return (const char*)x + nx <= (const char*)y || (const char*)y + ny <= (const char*)x; };
  const int64_t o_bytes = pairs * 128 * (s2->o_dtype == LSATTN_F32 ? 4 : 2), q_bytes = pairs * 256;
  const bool rows_match = rows_may_match && s2->o == a->q && o_bytes == q_bytes;
  return (rows_match || apart(s2->o, o_bytes, a->q, q_bytes)) && apart(s2->out_logexpsum, pairs * 4, a->q, q_bytes) &&
         apart(s2->o, o_bytes, a->b_seqlen, a->batch * 4) && apart(s2->o, o_bytes, a->b_req_idx, a->batch * 4) &&
         apart(s2->out_logexpsum, pairs * 4, a->b_seqlen, a->batch * 4) && apart(s2->out_logexpsum, pairs * 4, a->b_req_idx, a->batch * 4);
}

// Which launches of the fused call are one (decode_direct_kernel).  A workgroup walks its request in turns of 128 tokens, some 0.8 us each;
// two launches take some 4 us more than one for their starts and ends, and the longer the request the more workgroups share it.  The launch
// lasts as long as its longest request, whatever the others are, so the rule takes what is no slower with one long request among short
// ones, with a mild spread and with equal lengths.  Measured over 2700 launches (the longest 192 to 768 tokens, the others as long, a quarter or
// 16; 16 to 4096 workgroups; 32/8, 8/1, 64/8, 64/4, 24/8, 16/8 and 32/32 heads, f16 and bf16; two launches | one, us, replayed from a graph):
//   8 x 320 32/8 10.1 | 9.4    16 x 384 8/1 9.4 | 8.8      16 x 512 32/8 12.8 | 13.7 (not taken)   32, one of 640, the others 160, 32/8 17.5 | 13.7
//   64 x 640 64/8 37.6 | 32.6  256 x 512 32/8 100 | 95     48 x 512 16/8 22.5 | 24.3 (not taken)   48, one of 1024, the others 128, 32/8 15.0 | 20.3 (not taken)
//   4 x 320 32/32 9.6 | 9.7    2048 of 80 8/1 49.6 | 29.3  512, one of 320, the others 16, 32/8 36.8 | 39.5 (not taken)
// So up to 384 tokens, and up to 640 where there is a workgroup per CU (the two launches too walk more than a turn each then); with groups of
// four to seven query heads up to eight workgroups per CU, of more without a bound (at 16 per CU 0.49 to 0.95); with two or three (most of an
// MFMA's columns idle) up to 384 tokens below four per CU; with one, where the lane kernel stands against it, up to 320 below two.  The launches
// taken: 0.71 in the mean, 1.02 at most.
static bool decode_is_direct(const lsattn_decode_stage1_args* a, const lsattn_decode_stage2_args* s2) {
  const Tuning tn = tuning();
  if (tn.decode_stage1 != 0 || tn.decode_listed != 0) return false;  // (choices among the shapes of two launches)
  if (a->merge_blocks > 1 || a->batch > 65535 || a->k_stride_0 >= (1 << 30) || a->v_stride_0 >= (1 << 30)) return false;
  const int64_t group = a->num_q_heads / a->num_kv_heads, wgs = a->batch * a->num_kv_heads * ((group + 15) / 16), longest = a->max_len_in_batch;
  if (group == 1 ? longest > 320 || wgs >= 2 * kCUs
      : group < 4 ? longest > 384 || wgs >= 4 * kCUs
                  : longest > (wgs < kCUs ? 384 : 640) || (group < 8 && wgs > 8 * kCUs))
    return false;
  return result_is_apart(a, s2, true);
}
template <typename T> static int launch_direct(const lsattn_decode_stage1_args* a, const lsattn_decode_stage2_args* s2, hipStream_t st) {
  Stage1Params p = {};
  p.q = a->q;
  p.k = a->k;
  p.v = a->v;
  p.k_s0 = a->k_stride_0;
  p.k_s1 = a->k_stride_1;
  p.v_s0 = a->v_stride_0;
  p.v_s1 = a->v_stride_1;
  p.scale_log2 = a->sm_scale * kLog2e;
  p.req_to_tokens = a->req_to_tokens;
  p.b_req_idx = a->b_req_idx;
  p.b_seqlen = a->b_seqlen;
  p.batch = a->batch;
  p.hq = a->num_q_heads;
  p.hkv = a->num_kv_heads;
  p.num_blocks = a->num_blocks;  // (the tokens attended to are those that blocks and rows of partials would have covered)
  p.max_seq_len = a->max_seq_len;
  p.row_mul = 1;
  p.fine_block_seq = p.block_seq = a->seq_block_size;
  p.grid_blocks = (a->max_len_in_batch + p.block_seq - 1) / p.block_seq;
  p.tasks = (int)(a->num_kv_heads * ((a->num_q_heads / a->num_kv_heads + 15) / 16));
  p.tasks_on_x = 1;
  p.o = s2->o;
  p.out_lse = s2->out_logexpsum;
  const dim3 grid((unsigned)p.tasks, (unsigned)a->batch), block(kMfmaWaves * 64);
  switch (s2->o_dtype) {
    case LSATTN_F32: LSATTN_LAUNCH_KERNEL((decode_direct_kernel<T, float>), grid, block, 0, st, p); break;
    case LSATTN_F16: LSATTN_LAUNCH_KERNEL((decode_direct_kernel<T, F16>), grid, block, 0, st, p); break;
    case LSATTN_BF16: LSATTN_LAUNCH_KERNEL((decode_direct_kernel<T, BF16>), grid, block, 0, st, p); break;
    default: return LSATTN_ERR_UNSUPPORTED;
  }
  return check_launch();
}

template <typename T> static int dispatch_stage1(const lsattn_decode_stage1_args* a, hipStream_t st, SharesPlan* shares = nullptr, JoinPlan* join = nullptr) {
  const int group = (int)(a->num_q_heads / a->num_kv_heads);
  if (shares) {  // (in equal shares or not at all: shares->max_shares stays 0 then)
    bool taken;
    return launch_stage1_mfma<T>(a, st, &taken, shares);
  }
  {
    bool taken;
    const int rc = launch_stage1_mfma<T>(a, st, &taken, nullptr, join);
    if (taken) return rc;
  }
  // groups of 3 and 4 take four query heads per task (3: one spare): fetching a K/V row once per group matters more than
  // the spare accumulators cost
  // groups of more than four: eight query heads per task in two rounds of four over the same rows
  if (group >= 5) return launch_stage1<T, 4, 2>(a, st, join);
  if (group >= 3) return launch_stage1<T, 4, 1>(a, st, join);
  if (group == 2) return launch_stage1<T, 2, 1>(a, st, join);
  return launch_stage1<T, 1, 1>(a, st, join);
}

}  // namespace lsattn

using namespace lsattn;

static int validate_stage1(const lsattn_decode_stage1_args* a) {
  if (!a || !a->mid_o || !a->mid_o_logexpsum || !a->q || !a->k || !a->v || !a->req_to_tokens || !a->b_req_idx ||
      !a->b_seqlen)
    return LSATTN_ERR_INVALID_ARG;
  if (a->merge_blocks < 0 || a->merge_blocks > 16 || a->seq_block_size * (a->merge_blocks > 1 ? a->merge_blocks : 1) > 0x40000000)
    return LSATTN_ERR_INVALID_ARG;
  if (a->batch < 0 || a->num_q_heads <= 0 || a->num_kv_heads <= 0 || a->num_blocks < 0 || a->seq_block_size < 1 ||
      a->max_len_in_batch < 0 || a->max_seq_len < 0 || a->max_seq_len > 0x7fffff00)  // 32-bit token positions in the kernel
    return LSATTN_ERR_INVALID_ARG;
  if (a->num_q_heads % a->num_kv_heads != 0) return LSATTN_ERR_INVALID_ARG;
  // 16-byte row loads: strides must keep every row 16-byte aligned
  if (a->k_stride_0 % 8 || a->k_stride_1 % 8 || a->v_stride_0 % 8 || a->v_stride_1 % 8) return LSATTN_ERR_INVALID_ARG;
  if (((uintptr_t)a->k | (uintptr_t)a->v | (uintptr_t)a->q | (uintptr_t)a->mid_o) & 15) return LSATTN_ERR_INVALID_ARG;
  if (a->head_dim != 128) return LSATTN_ERR_UNSUPPORTED;  // as flash_decoding_stage1.cu:210
  return LSATTN_OK;
}

// `shares` (the fused call): launch stage 1 in equal shares if the launch is one for them (max_shares > 0 then) or nothing.
static int decode_stage1(const lsattn_decode_stage1_args* a, void* stream, SharesPlan* shares, JoinPlan* join = nullptr) {
  const int rc = validate_stage1(a);
  if (rc != LSATTN_OK) return rc;
  if (a->batch == 0 || a->num_blocks == 0 || a->max_len_in_batch == 0) return LSATTN_OK;
  hipStream_t st = (hipStream_t)stream;
  if (a->dtype == LSATTN_F16) return dispatch_stage1<F16>(a, st, shares, join);
  if (a->dtype == LSATTN_BF16) return dispatch_stage1<BF16>(a, st, shares, join);
  return LSATTN_ERR_UNSUPPORTED;
}

extern "C" int lsattn_decode_stage1(const lsattn_decode_stage1_args* a, void* stream) { return decode_stage1(a, stream, nullptr); }

// `live_blocks`: an upper bound of the partial rows any request has (the rows of the buffer, or fewer when the caller
// knows the longest request); it picks the shape of the merge, which decides the order of its additions.
template <typename OT> static int dispatch_stage2(const Stage2Params& p, int64_t D, dim3 grid, int64_t live_blocks, hipStream_t st) {
  if (p.max_shares > 0) {
    if (D != 128) return LSATTN_ERR_UNSUPPORTED;
    // four waves per pair while that keeps every pair resident at once (sixteen waves per CU)
    // (sixteen for the few pairs of one or two requests, which may have hundreds of rows each: both launches 0.84 to 1.03, in the mean 0.97 with one long
    // request; with more pairs 0.99 to 1.17, and of more requests, whose rows are fewer, to 1.09: 16, one of 5120, 4/4 heads 15.3 | 16.7 us)
    if (p.batch <= 2 && grid.x <= kWideMergePairs && p.max_shares >= 128) LSATTN_LAUNCH_KERNEL((decode_merge_shares_kernel<OT, 16>), grid, dim3(1024), 0, st, p);
    else if ((int64_t)grid.x <= 4 * kCUs) LSATTN_LAUNCH_KERNEL((decode_merge_shares_kernel<OT, 4>), grid, dim3(256), 0, st, p);
    else LSATTN_LAUNCH_KERNEL((decode_merge_shares_kernel<OT, 1>), dim3((unsigned)(p.batch * ((p.heads + 3) / 4))), dim3(256), 0, st, p);
    return check_launch();
  }
  // few (batch, head) pairs with many partials each (long contexts at small batch): 1024 threads walk the block axis in 32
  // slices instead of 8, or the merge takes a fifth of the time of the gather it follows
  const bool wide = D == 128 && live_blocks >= 64 && ((int64_t)grid.x < 2048 || (live_blocks >= 1024 && (int64_t)grid.x < 8192));
  switch (D) {
    case 32: LSATTN_LAUNCH_KERNEL((decode_stage2_kernel<OT, 32, 256>), grid, dim3(256), 0, st, p); break;
    case 64: LSATTN_LAUNCH_KERNEL((decode_stage2_kernel<OT, 64, 256>), grid, dim3(256), 0, st, p); break;
    case 128:
      if (wide) LSATTN_LAUNCH_KERNEL((decode_stage2_kernel<OT, 128, 1024>), grid, dim3(1024), 0, st, p);
      else LSATTN_LAUNCH_KERNEL((decode_stage2_kernel<OT, 128, 256>), grid, dim3(256), 0, st, p);
      break;
    default: return LSATTN_ERR_UNSUPPORTED;
  }
  return check_launch();
}

static int validate_stage2(const lsattn_decode_stage2_args* a) {
  if (!a || !a->o || !a->out_logexpsum || !a->b_seqlen || !a->mid_o || !a->mid_o_logexpsum) return LSATTN_ERR_INVALID_ARG;
  if (a->batch < 0 || a->num_heads <= 0 || a->num_seq_blocks < 0 || a->block_seq < 1 || a->lead_rows < 0) return LSATTN_ERR_INVALID_ARG;
  if (((uintptr_t)a->o | (uintptr_t)a->mid_o) & 15) return LSATTN_ERR_INVALID_ARG;
  if (a->head_dim != 32 && a->head_dim != 64 && a->head_dim != 128) return LSATTN_ERR_UNSUPPORTED;
  return a->batch * a->num_heads > 0x7fffffff ? LSATTN_ERR_INVALID_ARG : LSATTN_OK;
}

static int decode_stage2(const lsattn_decode_stage2_args* a, int64_t live_blocks, void* stream, const SharesPlan* shares = nullptr) {
  const int rc = validate_stage2(a);
  if (rc != LSATTN_OK) return rc;
  if (a->batch == 0) return LSATTN_OK;
  Stage2Params p{a->o, a->out_logexpsum, a->b_seqlen, a->mid_o, a->mid_o_logexpsum,
                 a->batch, a->num_heads, a->num_seq_blocks, a->block_seq,
                 a->partials_by_request ? a->num_heads : a->batch * a->num_heads,
                 a->partials_by_request ? a->num_seq_blocks * a->num_heads : a->num_heads, shares ? shares->units : 0,
                 shares ? shares->max_shares : 0, kShareUnits, a->lead_rows < a->num_seq_blocks ? a->lead_rows : a->num_seq_blocks};
  dim3 grid((unsigned)(a->batch * a->num_heads));
  hipStream_t st = (hipStream_t)stream;
  switch (a->o_dtype) {
    case LSATTN_F32: return dispatch_stage2<float>(p, a->head_dim, grid, live_blocks, st);
    case LSATTN_F16: return dispatch_stage2<F16>(p, a->head_dim, grid, live_blocks, st);
    case LSATTN_BF16: return dispatch_stage2<BF16>(p, a->head_dim, grid, live_blocks, st);
    default: return LSATTN_ERR_UNSUPPORTED;
  }
}

extern "C" int lsattn_decode_stage2(const lsattn_decode_stage2_args* a, void* stream) {
  return decode_stage2(a, a ? a->num_seq_blocks : 0, stream);
}

extern "C" int lsattn_decode_attention(const lsattn_decode_stage1_args* s1, const lsattn_decode_stage2_args* s2, void* stream) {
  if (!s1 || !s2) return LSATTN_ERR_INVALID_ARG;
  // the two stages must describe the same partials
  if (s1->mid_o != s2->mid_o || s1->mid_o_logexpsum != s2->mid_o_logexpsum || s1->b_seqlen != s2->b_seqlen ||
      s1->batch != s2->batch || s1->num_q_heads != s2->num_heads || s1->num_blocks != s2->num_seq_blocks ||
      s1->head_dim != s2->head_dim || s1->seq_block_size != s2->block_seq || s2->lead_rows != 0 || !s1->partials_by_request != !s2->partials_by_request)
    return LSATTN_ERR_INVALID_ARG;
  // (anything that either stage would refuse goes the way of two launches, which refuses it)
  if (validate_stage1(s1) == LSATTN_OK && validate_stage2(s2) == LSATTN_OK && s1->batch > 0 && s1->num_blocks > 0 && s1->max_len_in_batch > 0 &&
      (s1->dtype == LSATTN_F16 || s1->dtype == LSATTN_BF16) && (s2->o_dtype == LSATTN_F32 || s2->o_dtype == LSATTN_F16 || s2->o_dtype == LSATTN_BF16) &&
      decode_is_direct(s1, s2))
    return s1->dtype == LSATTN_F16 ? launch_direct<F16>(s1, s2, (hipStream_t)stream) : launch_direct<BF16>(s1, s2, (hipStream_t)stream);
  // Most launches deal the tokens in equal shares (decode_stage1_mfma_range_kernel), however coarse the split asked for: the
  // partials are scratch here.  The rows the shares may fill are counted from the longest request, at most one per 256
  // of its tokens, so that the result does not depend on the height of the buffers where they are tall enough for that.
  if (s1->merge_blocks <= 1 && s1->seq_block_size >= 256 && s1->max_len_in_batch > 0 && s1->num_blocks > 0 &&
      s1->max_len_in_batch < 0x7fffff00) {
    SharesPlan shares;
    // (in whole blocks of 256 tokens, as the grids count: a request a little longer than the bound is attended to the end)
    shares.rows = (s1->max_len_in_batch + 255) / 256;
    shares.units = shares.rows * (256 / kMfmaBatch);
    if (shares.rows > s1->num_blocks) shares.rows = s1->num_blocks;
    const int rc1 = decode_stage1(s1, stream, &shares);
    if (rc1 != LSATTN_OK) return rc1;
    if (shares.max_shares > 0) {
      lsattn_decode_stage2_args a2 = *s2;
      a2.block_seq = kMfmaBatch;
      return decode_stage2(&a2, 0, stream, &shares);
    }
  }
  // (the merge in stage 1's launch counts in o, see is_memory_of_this_gpu; launches of forced shapes are two)
  JoinPlan join{s2};
  const Tuning tn = tuning();
  const bool may_join = s2->o_is_apart == 2 && tn.decode_stage1 == 0 && tn.decode_listed == 0 && validate_stage2(s2) == LSATTN_OK && (s2->o_dtype == LSATTN_F32 || s2->o_dtype == LSATTN_F16 || s2->o_dtype == LSATTN_BF16) &&
                        result_is_apart(s1, s2, false);
  const int rc = decode_stage1(s1, stream, nullptr, may_join ? &join : nullptr);
  if (rc != LSATTN_OK || join.done) return rc;
  // the merge's shape from the rows the longest request can reach, not from the rows the buffer happens to have: the
  // same call gives the same bits whatever the buffer's height (lsattn_decode_attention_static passes its own)
  int64_t live = s1->seq_block_size > 0 ? (s1->max_len_in_batch + s1->seq_block_size - 1) / s1->seq_block_size : 0;
  if (live > s2->num_seq_blocks) live = s2->num_seq_blocks;
  return decode_stage2(s2, live, stream);
}

// ------------------------------------------------------------------------------------
// lsattn_decode_attention with the split-K partials in a file-scope device array instead of caller memory, for callers
// that cannot allocate.  Every device the library runs on holds its own copy of the array at its own address; the name
// below is only the host-side handle of it, so host code uses the address hipGetSymbolAddress returns for the current
// device (looked up once per device) and nothing else.
// ------------------------------------------------------------------------------------
static __device__ __align__(256) unsigned char scratch[LSATTN_STATIC_SCRATCH_BYTES];

namespace {
constexpr int kMaxDevices = 64;
std::atomic<void*> g_scratch_ptr[kMaxDevices];  // zero-initialised: not looked up yet

// device address of `scratch` on the current device, or nullptr
void* scratch_on_current_device() {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return nullptr;
  void* ptr = g_scratch_ptr[dev].load(std::memory_order_acquire);
  if (ptr) return ptr;
  // two threads that race here look the same address up twice; either store is right
  if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) {
    (void)hipGetLastError();
    return nullptr;
  }
  g_scratch_ptr[dev].store(ptr, std::memory_order_release);
  return ptr;
}
}  // namespace

extern "C" int lsattn_decode_attention_static(const lsattn_decode_stage1_args* s1, const lsattn_decode_stage2_args* s2,
                                              void* stream) {
  if (!s1 || !s2) return LSATTN_ERR_INVALID_ARG;
  // the partials are the library's here: the caller names none
  if (s1->mid_o || s1->mid_o_logexpsum || s2->mid_o || s2->mid_o_logexpsum) return LSATTN_ERR_INVALID_ARG;
  if (s1->b_seqlen != s2->b_seqlen || s1->batch != s2->batch || s1->num_q_heads != s2->num_heads ||
      s1->num_blocks != s2->num_seq_blocks || s1->head_dim != s2->head_dim || s1->seq_block_size != s2->block_seq || s2->lead_rows != 0)
    return LSATTN_ERR_INVALID_ARG;
  if (s1->batch < 0 || s1->num_q_heads <= 0 || s1->num_blocks < 0 || s1->seq_block_size < 1 || s1->max_len_in_batch < 0 ||
      s1->merge_blocks > 1)
    return LSATTN_ERR_INVALID_ARG;
  if (s1->head_dim != 128) return LSATTN_ERR_UNSUPPORTED;
  // Rows of partials this call can touch: stage 1 writes block i of a request only for i below both bounds, and stage 2
  // is told the same count, so it reads no row that this call has not written (the array keeps the last call's bytes).
  int64_t rows = (s1->max_len_in_batch + s1->seq_block_size - 1) / s1->seq_block_size;
  if (rows > s1->num_blocks) rows = s1->num_blocks;
  const int64_t per_row = s1->batch * s1->num_q_heads;  // (request, head) pairs per block row
  if (per_row > 0 && rows > (int64_t)LSATTN_STATIC_SCRATCH_BYTES / 4 / 129 / per_row) return LSATTN_ERR_WORKSPACE;
  if ((uint64_t)(rows * per_row * 129) * 4 > (uint64_t)LSATTN_STATIC_SCRATCH_BYTES) return LSATTN_ERR_WORKSPACE;
  // The array is laid out for as many rows as it holds for this batch, up to one per 256 tokens of the longest request: the
  // rows bound the number of equal shares in the fused call below.
  int64_t rows_laid = (s1->max_len_in_batch + 255) / 256;
  if (per_row > 0 && rows_laid > (int64_t)LSATTN_STATIC_SCRATCH_BYTES / 4 / 129 / per_row) rows_laid = (int64_t)LSATTN_STATIC_SCRATCH_BYTES / 4 / 129 / per_row;
  if (rows_laid < rows) rows_laid = rows;
  rows = rows_laid;
  const int64_t o_floats = rows * per_row * 128;         // a multiple of 128 floats: the LSE part stays 16-byte aligned
  float* base = (float*)scratch_on_current_device();
  if (!base) return LSATTN_ERR_LAUNCH;
  lsattn_decode_stage1_args a1 = *s1;
  lsattn_decode_stage2_args a2 = *s2;
  a1.mid_o = base;
  a1.mid_o_logexpsum = base + o_floats;
  a1.num_blocks = rows;
  a1.partials_by_request = a2.partials_by_request = 1;  // (the layout is nobody's but the library's here)
  a2.mid_o = a1.mid_o;
  a2.mid_o_logexpsum = a1.mid_o_logexpsum;
  a2.num_seq_blocks = rows;
  return lsattn_decode_attention(&a1, &a2, stream);
}
