// The prefill attention step for head sizes 16, 32 and 64 (the reference's Triton kernel takes them beside 128:
// loongserve/models/llama/triton_kernel/ring_context_flashattention_nopad.py:248-250) and, for batches of short prompts, 128
// (prefill_short_blocks), gfx950, wave64.
//
// What bounds it is vector work: a 32 x 32 block of scores takes a wave 16 exponentials, 16 multiply-adds, 16 additions and
// some 15 conversions and checks against 16 (D = 64) to 6 (D = 16) MFMAs, and the time falls only a third from D = 64 to 16.
// Hence no work beside those in the common path, and four waves per SIMD whose phases mix freely:
//   * a workgroup of four waves; a wave owns 32 (small launches: 16) query positions of one head.  With grouped-query
//     heads up to four heads of a KV head sit side by side in a workgroup, which then ends sooner on the diagonal;
//   * K and V tiles of 64 keys go to LDS by direct loads, two stages, one barrier per tile, chunks XOR-swizzled (bfloat16 V
//     passes through registers and becomes fp16 there);
//   * scores transposed, S^T = K Q^T with v_mfma_f32_16x16x32 (a head of 16 fills half of the contraction with
//     zeros), 32 keys per step, so a lane owns one query column: the fp32 scores turn into the B operand of O^T += V^T P^T in
//     place (P and V as fp16, sums of P in fp32), V^T operands through ds_read_b64_tr_b16; a wave skips the steps none of its
//     rows sees;
//   * the running maximum of a row is raised only when a P of 2 or more shows up; no exchange between lanes otherwise;
//   * the three epilogues of the 128-wide kernel: 0 the step's fp32 partial (O, LSE), 1 the reference's in-place
//     (o, m, l) update (ring_context_flashattention_nopad.py:171-188), 2 the LSE merge into a running fp32 (O, LSE).
// Against 16 positions per wave, eight waves, tiles staged through registers and the maximum exchanged in every step
// (fp16, causal): D = 64, 8 x 2048 tokens GQA 32/8 380 -> 183 us (0.75 PFLOP/s), 1 x 8192 MHA 640 -> 310, 16 x 512 73 -> 47,
// 1 x 100 7.4 -> 6.0; D = 32, 8 x 2048 283 -> 135; D = 16 278 -> 121.
#include <type_traits>

#include "common.hip.h"

namespace lsattn {
namespace {

typedef __attribute__((address_space(3))) i16x4* lds_i16x4_ptr;

template <typename T> struct MfmaS;
template <> struct MfmaS<F16> {
  static __device__ __forceinline__ f32x4 run(const u32x4& a, const u32x4& b, const f32x4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
};
template <> struct MfmaS<BF16> {
  static __device__ __forceinline__ f32x4 run(const u32x4& a, const u32x4& b, const f32x4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
};

// bfloat16 -> fp16, round toward zero: exact in fp16's normal range, larger magnitudes become +-65504
__device__ __forceinline__ u32x4 bf16_to_f16(const u32x4& w) {
  u32x4 r;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    float lo, hi;
    unpack2<BF16>(w[i], lo, hi);
    r[i] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(lo, hi));
  }
  return r;
}

// lanes c, c + 16, c + 32, c + 48 hold the four parts of query column c
__device__ __forceinline__ float xor16(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_ds_swizzle(__builtin_bit_cast(int, v), 0x401F));
}
__device__ __forceinline__ float xor32(float v) {
  const unsigned u = __builtin_bit_cast(unsigned, v);
  auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return __builtin_bit_cast(float, (threadIdx.x & 32) ? r[0] : r[1]);
}
__device__ __forceinline__ float col_max(float v) {
  v = fmaxf(v, xor16(v));
  return fmaxf(v, xor32(v));
}
__device__ __forceinline__ float col_sum(float v) {
  v += xor16(v);
  return v + xor32(v);
}

struct SmallParams {
  const void* q;
  const void* k;
  const void* v;
  int64_t q_st, q_sh, k_st, k_sh, v_st, v_sh;
  const int32_t* q_start;
  const int32_t* q_len;
  const int32_t* q_first;
  const int32_t* kv_start;
  const int32_t* kv_len;
  const int32_t* kv_first;
  const int32_t* o_start;
  int32_t hq, hkv, heads_per_kv, peers;
  int32_t group, pack_shift;  // groups of 1 << pack_shift heads side by side per KV head
  int32_t last_tile;          // of query positions, the first one of the launch
  FastDiv d_hkv, d_peers;
  float scale_log2;
  void* o;
  int64_t o_st, o_sh;
  float* lse;
  float* m;
  float* l;
  int64_t ml_st, ml_sh;
  int32_t batch;  // (TURN: a request's place among the ids moves on by one from tile to tile)
  FastDiv d_batch;
};

constexpr int kWaves = 4;   // waves per workgroup
constexpr int kTile = 64;   // keys per LDS tile
constexpr uint32_t kOnes = 0x3C003C00u;  // two ones in fp16
constexpr int64_t kCUs = 256;
constexpr int32_t kShortMaxRows = 768;    // 128-wide heads: the longest query chunk this kernel takes
constexpr int64_t kShortMaxKeys = 1024;   // and the keys up to which it does, of the longest request
constexpr int64_t kMaxTiles = 65535;  // tiles of one launch (the third index of a grid)

// s_waitcnt vmcnt(0) (expcnt / lgkmcnt fields left at their maximum)
__device__ __forceinline__ void wait_loads() { __builtin_amdgcn_s_waitcnt(0x0F70); }

// 16 bytes per lane from tile + off into LDS at dst (wave-uniform) + 16 * lane.  From inline assembly, or the compiler would
// wait for the load before every later LDS read; the s_nop is the wait state between a write of m0 and its use.
__device__ __forceinline__ void load_to_lds(int dst, const char* tile, uint32_t off) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst), "v"(off), "s"(tile) : "m0", "memory");
}
__device__ __forceinline__ const char* uniform_ptr(const char* ptr) {
  const uint64_t u = (uint64_t)ptr;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)u), hi = __builtin_amdgcn_readfirstlane((uint32_t)(u >> 32));
  return (const char*)(((uint64_t)hi << 32) | lo);
}

// DV: the V tiles are fp16 in memory and go straight into LDS as the K tiles do; otherwise (bfloat16 V) they pass through
// registers and are converted on the way.  QB: blocks of 16 query positions per wave.
template <typename T, int D, int MODE, bool DV, int QB, bool TURN = false>
__global__ __launch_bounds__(kWaves * 64, D == 128 ? 2 : QB == 2 && D == 64 && !DV ? 3 : 4) void prefill_small_kernel(SmallParams p) {
  constexpr int KS = D >= 32 ? D / 32 : 1;  // contraction steps of Q K^T (32 elements each; D = 16 fills half of one)
  constexpr int NDB = D / 16;               // 16-wide blocks of the head
  constexpr int CPR = D / 8;                // 16-byte chunks per K or V row
  constexpr int RB = D * 2;                 // bytes per row in LDS
  constexpr int TB = kTile * RB;            // bytes per tile
  constexpr int RPI = 64 / CPR;             // rows per load instruction (a wave's 64 lanes, 16 bytes each)
  constexpr int NI = (kTile + kWaves * RPI - 1) / (kWaves * RPI);  // load instructions per wave and tile: four for D = 128, two for 64, else one
  constexpr int RPB = 256 / RB;             // rows that pass all 64 LDS banks once
  // two stages of (K tile, V tile): the next tile is written while the present one is read.  Rows are not padded (a load to
  // LDS writes 1 KB in a row); instead the 16-byte chunks of a row are XORed with a function of the row: K so that a
  // column of chunks of sixteen rows, which one read takes, lies in sixteen different sets of four banks, V so that 32 bytes of
  // each of eight rows (half a transposing read) cover the banks once.  Rows sixteen apart share their XOR.
  __shared__ __attribute__((aligned(1024))) char lds[2 * 2 * TB];
  auto swz_k = [](int row) { return (row / RPB) & (CPR - 1); };
  auto swz_v = [](int row) { return ((row / RPB) & (CPR / 2 - 1)) << 1; };

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;
  // grid: (KV head, heads side by side), request, tile from the last one down: the heaviest tiles of all requests start
  // first, and with a multiple of eight KV heads the workgroups of one run on one XCD (ids are dealt round-robin)
  const int gq = (int)div_by(blockIdx.x, p.d_hkv), kvh = (int)blockIdx.x - gq * p.hkv;
  int b = blockIdx.y;
  if constexpr (TURN) {  // (requests_take_turns; a kernel of its own, so that the others stay as they are)
    const uint32_t place = blockIdx.y + blockIdx.z;
    b = (int)(place - div_by(place, p.d_batch) * (uint32_t)p.batch);
  }
  const int rows_wg = (kWaves * QB * 16) >> p.pack_shift;  // query positions of this workgroup
  const int m_wg = (p.last_tile - (int)blockIdx.z) * rows_wg;
  const int q_len = p.q_len[b];
  if (m_wg >= q_len) return;  // (the whole workgroup: the loop below holds barriers)
  const int wph_shift = 2 - p.pack_shift;  // log2 of the waves per head
  const int h = kvh * p.heads_per_kv + (gq << p.pack_shift) + (wave >> wph_shift);
  const int m0 = m_wg + (wave & ((1 << wph_shift) - 1)) * (QB * 16);  // the wave's first position
  const int kv_len = p.kv_len[b], qf = p.q_first[b], kf = p.kv_first[b], P = p.peers;
  const int64_t q_start = p.q_start[b], kv_start = p.kv_start[b];
  const int64_t o_start = p.o_start ? (int64_t)p.o_start[b] : q_start;

  // keys of this KV chunk visible to global query position qpos (ring_context_flashattention_nopad.py:156-159)
  auto visible_keys = [&](int qpos) -> int {
    const int dq = qpos - kf;
    const int n = dq >= 0 ? (int)div_by((uint32_t)dq, p.d_peers) + 1 : 0;
    return n > kv_len ? kv_len : n;
  };
  // per block qb of 16 positions: the lane's position m0 + 16 qb + c, whether it exists, the keys it sees
  bool in_range[QB];
  int cnt[QB];
  u32x4 qreg[QB][KS];  // Q^T as B operands: qreg[qb][ks] = Q[position][32 ks + 8 g .. + 7]
  f32x4 oacc[QB][NDB]; // O^T: oacc[qb][db][j] = O[position][16 db + 4 g + j]
  float m_run[QB], l_run[QB];  // log2-domain running max of the column; the lane's share of its running sum
  f32x4 l_pv[QB];  // the column's sum of the fp16 values that multiply V (all four elements)
#pragma unroll
  for (int qb = 0; qb < QB; qb++) {
    const int m = m0 + 16 * qb + c;
    in_range[qb] = m < q_len;
    cnt[qb] = in_range[qb] ? visible_keys(qf + m * P) : 0;
    const char* src = (const char*)p.q + ((q_start + (in_range[qb] ? m : m_wg)) * p.q_st + (int64_t)h * p.q_sh) * 2;
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      const int d0 = 32 * ks + 8 * g;
      qreg[qb][ks] = d0 < D ? *(const u32x4*)(src + d0 * 2) : u32x4{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int db = 0; db < NDB; db++) oacc[qb][db] = f32x4{0.f, 0.f, 0.f, 0.f};
    m_run[qb] = -INFINITY;
    l_run[qb] = 0.f;
    l_pv[qb] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // (positions ascend: a later row sees at least as many keys)
  auto last_seen = [&](int first, int rows) -> int {  // keys the last existing position of [first, first + rows) sees; 0 if none exists
    return first < q_len ? visible_keys(qf + (first + rows - 1 < q_len ? first + rows - 1 : q_len - 1) * P) : 0;
  };
  const int cnt_wave = __builtin_amdgcn_readfirstlane(last_seen(m0, QB * 16));
  // (rows past the end see nothing: a wave that holds some masks everywhere only where it has to, in their own columns,
  // which nothing reads; its first row sees the fewest keys of the others)
  const int cnt_first = __builtin_amdgcn_readfirstlane(m0 < q_len ? visible_keys(qf + m0 * P) : 0);
  const int cnt_wg = __builtin_amdgcn_readfirstlane(last_seen(m_wg, rows_wg));

  const char* kbase = (const char*)p.k + (kv_start * p.k_st + (int64_t)kvh * p.k_sh) * 2;
  const char* vbase = (const char*)p.v + (kv_start * p.v_st + (int64_t)kvh * p.v_sh) * 2;
  // staging: instruction i of a wave carries rows (wave + 4 i) * RPI .. of the K tile and of the V tile.  Tiles that lie inside the
  // chunk take a scalar tile address and the lane's 32-bit offset, no vector arithmetic.
  const bool stager = NI * kWaves * RPI == kTile || wave * RPI < kTile;  // (D = 16: two waves)
  const int st_row = wave * RPI + lane / CPR;
  const uint32_t k_row = (uint32_t)p.k_st * 2, v_row = (uint32_t)p.v_st * 2;  // (a tile's rows span less than 2^31 bytes)
  const uint32_t k_off = st_row * k_row + ((lane % CPR) ^ swz_k(st_row)) * 16, v_off = st_row * v_row + ((lane % CPR) ^ swz_v(st_row)) * 16;
  const int lds_base = (int)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
  u32x4 vst[NI];
  auto request = [&](int stage, int t) __attribute__((always_inline)) {
    if (!stager) return;
    const char* kt = uniform_ptr(kbase + (int64_t)t * kTile * k_row);
    const char* vt = uniform_ptr(vbase + (int64_t)t * kTile * v_row);
    const int dst = __builtin_amdgcn_readfirstlane(lds_base + stage * 2 * TB + wave * 1024);
    const int last = kv_len - 1 - t * kTile;
#pragma unroll
    for (int i = 0; i < NI; i++) {
      constexpr int STEP = kWaves * RPI;
      uint32_t ko = k_off, vo = v_off;
      if (last < kTile - 1) {  // (wave-uniform; rows past the end repeat the last one and are masked)
        int r0 = st_row;
        asm volatile("" : "+v"(r0));  // (worked out here and not kept in registers over the loop)
        int back = r0 + i * STEP - last;
        back = back < 0 ? 0 : back;
        ko -= (uint32_t)back * k_row;
        vo -= (uint32_t)back * v_row;
      }
      load_to_lds(dst + i * kWaves * 1024, kt, ko + (uint32_t)(i * STEP) * k_row);
      if (DV) load_to_lds(dst + TB + i * kWaves * 1024, vt, vo + (uint32_t)(i * STEP) * v_row);
      else vst[i] = *(const u32x4*)(vt + (vo + (uint32_t)(i * STEP) * v_row));
    }
  };
  // the tile that was requested, complete in LDS for this wave
  auto deposit = [&](int stage) __attribute__((always_inline)) {
    if (!DV && stager) {
#pragma unroll
      for (int i = 0; i < NI; i++) *(u32x4*)(lds + stage * 2 * TB + TB + (wave + i * kWaves) * 1024 + lane * 16) = bf16_to_f16(vst[i]);
    }
    wait_loads();
  };
  // transposing read: lane c of a 16-lane group points at row c >> 2, columns 4 (c & 3) .. + 3 of a 4 x 16 block and
  // receives column c of it; group g takes rows 4 g .. 4 g + 3 and, sixteen rows on, 16 + 4 g .. + 3: the eight keys
  // whose scores the lane holds
  int kaddr[KS], vaddr[NDB];
#pragma unroll
  for (int ks = 0; ks < KS; ks++) kaddr[ks] = lds_base + c * RB + (((4 * ks + g) & (CPR - 1)) ^ swz_k(c)) * 16;
#pragma unroll
  for (int db = 0; db < NDB; db++) {
    const int row = 4 * g + (c >> 2);
    vaddr[db] = lds_base + TB + row * RB + ((2 * db + ((c & 3) >> 1)) ^ swz_v(row)) * 16 + (c & 1) * 8;
  }
  const float scale = p.scale_log2;
  const int nt = (cnt_wg + kTile - 1) / kTile;  // the same for every wave of the workgroup

  u32x4 ka[2][KS];  // K operands of the next 32 keys
  auto load_ka = [&](int at) __attribute__((always_inline)) {
#pragma unroll
    for (int kb = 0; kb < 2; kb++)
#pragma unroll
      for (int ks = 0; ks < KS; ks++) {
        ka[kb][ks] = *(const __attribute__((address_space(3))) u32x4*)(kaddr[ks] + at + kb * 16 * RB);
        if (D == 16 && g >= 2) ka[kb][ks] = u32x4{0u, 0u, 0u, 0u};
      }
  };
  auto tile = [&](auto stage_tag, int t) __attribute__((always_inline)) {
    constexpr int S = decltype(stage_tag)::value;
    if (t + 1 < nt) request(S ^ 1, t + 1);
    if (t * kTile < cnt_wave) load_ka(S * 2 * TB);
#pragma unroll
    for (int half = 0; half < 2; half++) {
      const int k0 = t * kTile + 32 * half;
      if (k0 < cnt_wave) {  // (wave-uniform: else none of the wave's rows sees these keys)
        // S^T = K Q^T: s[qb][kb][j] = score of key k0 + 16 kb + 4 g + j for the lane's query of block qb; a K operand
        // serves all blocks
        f32x4 s[QB][2];
#pragma unroll
        for (int ks = 0; ks < KS; ks++)
#pragma unroll
          for (int kb = 0; kb < 2; kb++)
#pragma unroll
            for (int qb = 0; qb < QB; qb++) s[qb][kb] = MfmaS<T>::run(ka[kb][ks], qreg[qb][ks], ks == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : s[qb][kb]);
        if (k0 + 32 > cnt_first) {  // (wave-uniform: the wave's first row, which sees the fewest keys, does not see the whole step)
#pragma unroll
          for (int qb = 0; qb < QB; qb++) {
            const int rel = cnt[qb] - k0 - 4 * g;
#pragma unroll
            for (int kb = 0; kb < 2; kb++)
#pragma unroll
              for (int j = 0; j < 4; j++) s[qb][kb][j] = 16 * kb + j < rel ? s[qb][kb][j] : -INFINITY;
          }
        }
        // P = exp2(S * scale - m) with the running maxima as they are; they are raised, and the step done again, only if some
        // P comes out as 2 or more (or as inf or NaN, as for a row that has seen no key yet: m = -inf), which is bit 14 of
        // its fp16 form.  No exchange between lanes, no chain through the maximum in the common case.
        u32x4 pk[QB];  // P^T as B operands: the lane's eight keys are contraction slots 8 g .. 8 g + 7, the order the V^T operand uses
        float ps[QB];
        auto compute_p = [&](int qb, float neg_m) __attribute__((always_inline)) {
          float pv[8];
#pragma unroll
          for (int e = 0; e < 8; e++) pv[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[qb][e / 4][e % 4], scale, neg_m));
          ps[qb] = ((pv[0] + pv[1]) + (pv[2] + pv[3])) + ((pv[4] + pv[5]) + (pv[6] + pv[7]));
#pragma unroll
          for (int e = 0; e < 4; e++) pk[qb][e] = pack2<F16>(pv[2 * e], pv[2 * e + 1]);
        };
        uint32_t any = 0;
#pragma unroll
        for (int qb = 0; qb < QB; qb++) {
          compute_p(qb, -m_run[qb]);
          any |= (pk[qb][0] | pk[qb][1]) | (pk[qb][2] | pk[qb][3]);
        }
        if (__builtin_expect(__builtin_amdgcn_ballot_w64((any & 0x40004000u) != 0) != 0, 0)) {
#pragma unroll
          for (int qb = 0; qb < QB; qb++) {
            const float mx = fmaxf(fmaxf(fmaxf(s[qb][0][0], s[qb][0][1]), fmaxf(s[qb][0][2], s[qb][0][3])),
                                   fmaxf(fmaxf(s[qb][1][0], s[qb][1][1]), fmaxf(s[qb][1][2], s[qb][1][3])));
            const float m_new = fmaxf(m_run[qb], col_max(mx) * scale);  // (the scale is positive)
            const float alpha = exp2_diff(m_run[qb], m_new);
            l_run[qb] *= alpha;
            l_pv[qb] *= alpha;
#pragma unroll
            for (int db = 0; db < NDB; db++) oacc[qb][db] *= alpha;
            m_run[qb] = m_new;
            compute_p(qb, m_new == -INFINITY ? 0.f : -m_new);  // (a row that has seen no key: every P is 0)
          }
        }
#pragma unroll
        for (int qb = 0; qb < QB; qb++) l_run[qb] += ps[qb];
        // (the scores' registers are free now and take the next K operands; asked for any earlier, these or the V operands
        // below spill: 64-wide heads, 8 x 2048 tokens, 217 us instead of 168 (without l_pv) with the V operands read before the softmax)
        __builtin_amdgcn_sched_barrier(0);
        u32x4 va[NDB];
#pragma unroll
        for (int db = 0; db < NDB; db++) {
          const int at = vaddr[db] + S * 2 * TB + 32 * half * RB;
          const i16x4 xa = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_ptr)at);
          const i16x4 xb = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_ptr)(at + 16 * RB));
          const u32x2 wa = __builtin_bit_cast(u32x2, xa), wb = __builtin_bit_cast(u32x2, xb);
          va[db] = u32x4{wa[0], wa[1], wb[0], wb[1]};
        }
        if (half == 0) load_ka(S * 2 * TB + 32 * RB);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int db = 0; db < NDB; db++)
#pragma unroll
          for (int qb = 0; qb < QB; qb++) oacc[qb][db] = MfmaS<F16>::run(va[db], pk[qb], oacc[qb][db]);
#pragma unroll
        for (int qb = 0; qb < QB; qb++) l_pv[qb] = MfmaS<F16>::run(u32x4{kOnes, kOnes, kOnes, kOnes}, pk[qb], l_pv[qb]);
      }
    }
    // the next tile is in the other stage (last read one barrier ago), then everyone meets: that tile is complete and this
    // one is done with
    if (t + 1 < nt) deposit(S ^ 1);
    __syncthreads();
  };
  if (nt > 0) {
    request(0, 0);
    deposit(0);
    __syncthreads();
  }
  for (int t = 0; t < nt; t += 2) {  // (the stage is a constant of the code)
    tile(std::integral_constant<int, 0>{}, t);
    if (t + 1 < nt) tile(std::integral_constant<int, 1>{}, t + 1);
  }

  // ---- epilogues (the 128-wide kernel's), block by block of 16 positions ----
#pragma unroll
  for (int qb = 0; qb < QB; qb++) {
    const int mb = m0 + 16 * qb;
    if (mb >= q_len) break;  // (wave-uniform: a block without positions; it only helped to stage)
    const float l_tot = col_sum(l_run[qb]);
    // (0 exactly if the row saw no key.  A NaN score makes the sum NaN: it counts as a key, so that the row's outputs and its running
    // state become NaN, as they do in the reference, and no step before or after hides it)
    const bool seen = !(l_tot == 0.f);
    // O becomes a mean with the very weights it was summed with: a rounding that a row's weights share (one key that outweighs
    // the others) falls out of it, which makes up for maxima that lag (a P of 1 is exact in fp16, one of 1.4 is not).
    // Against 64 bits the fp32 partial of N(0, 1) * 0.5 inputs is off by 1.70e-4 to 1.72e-4 at 1000 to 3000 tokens of 64-wide heads,
    // 1.74e-4 to 1.75e-4 with maxima that never lag and 1.76e-4 with neither.  The sum that (m, l) and the LSE state stays the fp32 one.
    const float fix = l_pv[qb][0] == 0.f ? 0.f : l_tot / l_pv[qb][0];
#pragma unroll
    for (int db = 0; db < NDB; db++) oacc[qb][db] *= fix;
    const bool here = in_range[qb];
    const int64_t tok = o_start + (here ? mb + c : mb);
    if (MODE == 0) {
      if (here) {
        const float inv = seen ? 1.f / l_tot : 0.f;
        float* orow = (float*)p.o + tok * p.o_st + (int64_t)h * p.o_sh;
#pragma unroll
        for (int db = 0; db < NDB; db++) *(f32x4*)(orow + db * 16 + 4 * g) = oacc[qb][db] * inv;
        if (g == 0) p.lse[tok * p.hq + h] = seen ? (m_run[qb] + __builtin_amdgcn_logf(l_tot)) * kLn2 : -INFINITY;
      }
    }
    if (MODE == 1) {
      // the reference's update of (o, m, l); a row in its start state (m = -inf, l = 0) may hold anything in o
      const int64_t at = tok * p.ml_st + (int64_t)h * p.ml_sh;
      const float m_old = p.m[at], l_old = p.l[at];
      const float M = fmaxf(m_run[qb], m_old);
      const bool upd = here && seen;  // (a row that saw a key has a maximum, unless all its scores are NaN)
      float L = 0.f;
      if (upd) {
        const float w_old = l_old * exp2_diff(m_old, M);
        const float w_new = exp2_diff(m_run[qb], M);
        L = w_old + l_tot * w_new;
        const float inv = 1.f / L;
        uint16_t* orow = (uint16_t*)p.o + tok * p.o_st + (int64_t)h * p.o_sh;
#pragma unroll
        for (int db = 0; db < NDB; db++) {
          float o0 = 0.f, o1 = 0.f, o2 = 0.f, o3 = 0.f;
          if (w_old != 0.f) {
            const u32x2 old = *(const u32x2*)(orow + db * 16 + 4 * g);
            unpack2<T>(old[0], o0, o1);
            unpack2<T>(old[1], o2, o3);
          }
          const float r0 = (o0 * w_old + oacc[qb][db][0] * w_new) * inv, r1 = (o1 * w_old + oacc[qb][db][1] * w_new) * inv;
          const float r2 = (o2 * w_old + oacc[qb][db][2] * w_new) * inv, r3 = (o3 * w_old + oacc[qb][db][3] * w_new) * inv;
          *(u32x2*)(orow + db * 16 + 4 * g) = u32x2{pack2<T>(r0, r1), pack2<T>(r2, r3)};
        }
      }
      // (the four lanes of a column all read the old m and l above, in the same instruction as the one that writes them below)
      if (upd && g == 0) {
        p.m[at] = M;
        p.l[at] = L;
      }
    }
    if (MODE == 2) {
      // fold the step's partial into the running fp32 (O, LSE); a row that saw no key stays as it is
      const bool upd = here && seen;
      const float a_old = p.lse[tok * p.hq + h] * kLog2e;
      float new_lse = 0.f;
      if (upd) {
        const float a_new = m_run[qb] + __builtin_amdgcn_logf(l_tot);
        const float top = fmaxf(a_old, a_new);
        const float w_old = exp2_diff(a_old, top);
        const float w_new = __builtin_amdgcn_exp2f(a_new - top);
        const float W = w_old + w_new;
        const float c_old = w_old / W, c_new = w_new / (W * l_tot);
        float* orow = (float*)p.o + tok * p.o_st + (int64_t)h * p.o_sh;
#pragma unroll
        for (int db = 0; db < NDB; db++) {
          // an empty row (lse = -inf) may hold anything: its old values are dropped, not multiplied by zero
          const f32x4 keep = w_old != 0.f ? *(const f32x4*)(orow + db * 16 + 4 * g) : f32x4{0.f, 0.f, 0.f, 0.f};
          *(f32x4*)(orow + db * 16 + 4 * g) = keep * c_old + oacc[qb][db] * c_new;
        }
        new_lse = (top + __builtin_amdgcn_logf(W)) * kLn2;
      }
      if (upd && g == 0) p.lse[tok * p.hq + h] = new_lse;
    }
  }
}

// Whether a request's place among the ids moves on from tile to tile (TURN).  Ids go to the eight XCDs in turn and within one to its four
// shader engines.  If the ids of two tiles of a request are a multiple of 32 apart, all its workgroups share one shader engine of an
// XCD, and while only the longest requests have a tile left to start, the others idle: 8 sequences of 1000 to 3000 tokens, 32/8 heads
// of 64, had 2 workgroups on a CU until half of the launch was over, some 4 and some 1, where 8 x 2048 keep 3.9.  Turning places
// fill them evenly.  Measured over 60 ragged launches (2 to 32 sequences, 300 to 6000 tokens; microseconds, fixed | turning):
//   8 x 1000..3000 32/8 183 | 165   2 x 1206..3618 64/8 144 | 123   4 x 120..3615 64/8 bf16 87.9 | 61.8   4 x 688..2064 32/32 53.2 | 47.3
//   4 x 2582..5165 32/8 bf16 344 | 314   8 x 1304..2608 12/12 88.8 | 79.5   16 x 31..959 64/8 57.3 | 53.5
// At other distances (11 x 388..1166 32/8 44.8 | 47.1; distance 6 of the eights 9 % better to 4 % worse), with fewer than 16 tiles
// (8 x 280..842 32/32 31.5 | 33.3) and with equal lengths turning gains nothing: those keep the kernel without it.
bool requests_take_turns(const lsattn_prefill_args* a, int64_t ids_per_tile, int64_t tiles) {
  return ids_per_tile * a->batch % 32 == 0 && tiles >= 16 && a->total_q_rows > 0 && a->total_q_rows * 10 <= (int64_t)a->batch * a->max_q_len * 9;
}

template <typename T, int D, int MODE, bool DV, int QB, bool TURN = false> int launch_rows(SmallParams p, const lsattn_prefill_args* a, hipStream_t st) {
  const int64_t rows_wg = (kWaves * QB * 16) >> p.pack_shift;
  for (int64_t tiles = (a->max_q_len + rows_wg - 1) / rows_wg; tiles > 0; tiles -= kMaxTiles) {
    p.last_tile = (int32_t)(tiles - 1);
    LSATTN_LAUNCH_KERNEL((prefill_small_kernel<T, D, MODE, DV, QB, TURN>),
                         dim3((unsigned)(p.hkv * p.group), (unsigned)a->batch, (unsigned)(tiles < kMaxTiles ? tiles : kMaxTiles)),
                         dim3(kWaves * 64), 0, st, p);
    const int rc = check_launch();
    if (rc != LSATTN_OK) return rc;
  }
  return LSATTN_OK;
}

// query heads of a KV head side by side in a workgroup: as many (1, 2 or 4; the power of two) as the group divides by
int pack_shift_of(const lsattn_prefill_args* a) {
  const int32_t heads = a->num_q_heads / a->num_kv_heads;
  return heads % 4 == 0 ? 2 : heads % 2 == 0 ? 1 : 0;
}
// Workgroups that find rows, with `blocks` blocks of 16 positions per wave: the longest request's times the batch, or fewer if
// the caller bounds the rows of all requests together.
int64_t workgroups(const lsattn_prefill_args* a, int pack_shift, int blocks) {
  const int64_t rows = (kWaves * blocks * 16) >> pack_shift;
  const int64_t by_longest = a->batch * ((a->max_q_len + rows - 1) / rows);
  const int64_t by_total = a->total_q_rows > 0 ? (a->total_q_rows + rows - 1) / rows + a->batch : by_longest;
  return (by_total < by_longest ? by_total : by_longest) * (a->num_q_heads >> pack_shift);
}

// 32 positions per wave serve twice the rows with each K and V operand read, 16 make twice as many, shorter waves: these from
// three workgroups of the larger shape per CU down, where the launch is as long as its longest wave.  Measured at 64-wide heads
// (32 | 16 positions, without the sum of the fp16 weights, which costs both 4 to 8 %): 256 workgroups 21.5 | 16.2 us, 512 24.9 | 20.4 and 40.3 | 32.6, 768 30.4 | 31.4, 1024 36.6 | 35.7 and
// 92.8 | 99.3, 2048 43.9 | 48.6, 4096 170 | 200.
template <typename T, int D, int MODE, bool DV> int launch(const SmallParams& p, const lsattn_prefill_args* a, hipStream_t st) {
  if (a->num_q_heads > 65535 || a->batch > 65535) return LSATTN_ERR_INVALID_ARG;
  switch (prefill_small_route(a)) {
    case LSATTN_ROUTE_SMALL_16: return launch_rows<T, D, MODE, DV, 1>(p, a, st);
    case LSATTN_ROUTE_SMALL_TURNS: return launch_rows<T, D, MODE, DV, 2, true>(p, a, st);
    default: return launch_rows<T, D, MODE, DV, 2>(p, a, st);
  }
}

template <typename T, int MODE, bool DV> int launch_128(const SmallParams& p, const lsattn_prefill_args* a, hipStream_t st) {
  return prefill_small_route(a) == LSATTN_ROUTE_SMALL_16 ? launch_rows<T, 128, MODE, DV, 1>(p, a, st) : launch_rows<T, 128, MODE, DV, 2>(p, a, st);
}

template <typename T, int MODE, bool DV> int launch_d(const SmallParams& p, const lsattn_prefill_args* a, hipStream_t st) {
  switch (a->head_dim) {
    case 16: return launch<T, 16, MODE, DV>(p, a, st);
    case 32: return launch<T, 32, MODE, DV>(p, a, st);
    case 64: return launch<T, 64, MODE, DV>(p, a, st);
    case 128: return launch_128<T, MODE, DV>(p, a, st);
    default: return LSATTN_ERR_UNSUPPORTED;
  }
}

template <typename T, bool DV> int launch_mode(const SmallParams& p, const lsattn_prefill_args* a, int mode, hipStream_t st) {
  switch (mode) {
    case 0: return launch_d<T, 0, DV>(p, a, st);
    case 1: return launch_d<T, 1, DV>(p, a, st);
    case 2: return launch_d<T, 2, DV>(p, a, st);
    default: return LSATTN_ERR_INVALID_ARG;
  }
}

}  // namespace

// Short prompts of 128-wide heads: the kernel of prefill.hip spends 9 us on starting and ending whatever it computes (eight
// waves of 256 registers that fill 128 KB of rings and some 40 KB of code before the first product); this one has a
// quarter of the code, workgroups of 64 rows (128) and two of them per CU, converts a bfloat16 V on the way (no launch in front
// that copies it), but reads LDS four times (twice) as much per product, and a tile takes longer (below).  Measured over 472 launches (1 to
// 32 prompts of 32 to 2048 tokens, equal or log-uniform over a factor of 8, 32/32, 32/8, 64/8 and 8/1 heads; both epilogues;
// microseconds, the kernel of prefill.hip | 16 positions per wave | 32; bf16 with its copy of V):
//   1 x 100 MHA f16 10.9 | 5.5 | 7.8        1 x 512 32/8 f16 15.6 | 12.3 | 16.5    16 x 128 MHA f16 25.6 | 19.6 | 17.7
//   1 x 30 32/8 bf16 12.4 | 4.9 | 6.4       7 x 67..269 32/8 13.5 | 9.3 | 10.8      16 x 256 MHA f16 37.4 | 45.1 | 36.7
//   8 x 512 32/8 f16 36.6 | 43.6 | 37.9     1 x 1024 32/8 f16 20.8 | 21.5 | 26.9    (neither is taken)
// 16 positions per wave win up to two and a half workgroups per CU (with one head per workgroup, which leaves the other kernel
// four times the rows to mask, up to six, for prompts of up to 512 tokens), 32 up to six and 256 tokens; the geometric
// mean over the launches the rule takes is 25 to 35 % below the other kernel, the worst is 5 % above it.
// The keys: a tile of 64 costs a wave 0.95 us here (bf16 V 1.5) against 0.56 in the 128-row shape, which a launch with one long
// context waits for, so the longest request decides (whole call, 32/8 heads, the other kernel | this one, f16, then bf16):
//   8 x 64 rows behind 600 keys each 20.8 | 15.7, 28.0 | 18.7      4 x 100 behind 1000 each 24.9 | 21.7, 30.5 | 25.9      1 x 200 behind 1024 22.1 | 19.8, 25.2 | 24.0
//   2 x 100, one behind 1900 30.6 | 31.8, 34.5 | 39.8      8 x 64, one behind 7500 79.8 | 108.8, 88 | 169      16 x 64, one behind 15000 145 | 264, 155 | 352
// The host knows no lengths, only bounds: what total_kv_rows holds beyond the query rows may all belong to one request.
int prefill_short_blocks(const lsattn_prefill_args* a) {
  if (a->head_dim != 128 || a->kv_cuts > 1 || a->o_b_start_loc || a->max_q_len <= 0 || a->max_q_len > kShortMaxRows || a->batch <= 0 || a->num_kv_heads <= 0)
    return 0;
  int64_t longest = kShortMaxKeys + 1;
  if (a->total_kv_rows > 0) {
    longest = a->total_kv_rows;
    if (a->total_q_rows > 0) {
      const int64_t most = (int64_t)a->batch * a->max_q_len, rows = a->total_q_rows < most ? a->total_q_rows : most;
      const int64_t beyond = a->total_kv_rows > rows ? a->total_kv_rows - rows : 0;
      if (a->max_q_len + beyond < longest) longest = a->max_q_len + beyond;
    }
  }
  if (a->max_kv_len > 0 && a->max_kv_len < longest) longest = a->max_kv_len;
  if (longest > kShortMaxKeys) return 0;
  const Tuning tn = tuning();
  if (tn.prefill_rows || tn.prefill_order || tn.prefill_pack) return 0;  // (choices among the 128-wide kernel's shapes)
  const int pack = pack_shift_of(a);
  const int64_t one = workgroups(a, pack, 1), two = workgroups(a, pack, 2);
  if (one <= 5 * kCUs / 2 || (pack == 0 && a->max_q_len <= 512 && one <= 6 * kCUs)) return 1;
  return a->max_q_len <= 256 && two <= 6 * kCUs ? 2 : 0;
}

int prefill_small_route(const lsattn_prefill_args* a) {
  if (a->head_dim == 128) return prefill_short_blocks(a) == 1 ? LSATTN_ROUTE_SMALL_16 : LSATTN_ROUTE_SMALL_32;
  const int pack = pack_shift_of(a);
  if (workgroups(a, pack, 2) < 3 * kCUs) return LSATTN_ROUTE_SMALL_16;
  const int64_t rows_wg = (kWaves * 2 * 16) >> pack;
  return requests_take_turns(a, a->num_q_heads >> pack, (a->max_q_len + rows_wg - 1) / rows_wg) ? LSATTN_ROUTE_SMALL_TURNS : LSATTN_ROUTE_SMALL_32;
}

// One prefill step with head_dim 16, 32 or 64, or a short one with 128 (arguments already validated; epilogue `mode` as in the 128-wide kernel).
int launch_prefill_small(const lsattn_prefill_args* a, int mode, hipStream_t st) {
  SmallParams p;
  p.q = a->q;
  p.k = a->k;
  p.v = a->v;
  p.q_st = a->q_stride_t;
  p.q_sh = a->q_stride_h;
  p.k_st = a->k_stride_t;
  p.k_sh = a->k_stride_h;
  p.v_st = a->v_stride_t;
  p.v_sh = a->v_stride_h;
  p.q_start = a->q_b_start_loc;
  p.q_len = a->q_b_seq_len;
  p.q_first = a->q_first_token_global_idx;
  p.kv_start = a->kv_b_start_loc;
  p.kv_len = a->kv_b_seq_len;
  p.kv_first = a->kv_first_token_global_idx;
  p.o_start = a->o_b_start_loc;
  p.hq = (int32_t)a->num_q_heads;
  p.hkv = (int32_t)a->num_kv_heads;
  p.heads_per_kv = (int32_t)(a->num_q_heads / a->num_kv_heads);
  p.peers = (int32_t)a->sp_peers;
  p.pack_shift = pack_shift_of(a);
  p.group = p.heads_per_kv >> p.pack_shift;
  p.d_hkv = fast_div((uint32_t)p.hkv);
  p.d_peers = fast_div((uint32_t)p.peers);
  p.batch = (int32_t)a->batch;
  p.d_batch = fast_div((uint32_t)p.batch);
  p.scale_log2 = a->sm_scale * kLog2e;
  p.o = a->o;
  p.o_st = a->o_stride_t;
  p.o_sh = a->o_stride_h;
  p.lse = a->lse;
  p.m = a->m;
  p.l = a->l;
  p.ml_st = a->ml_stride_t;
  p.ml_sh = a->ml_stride_h;
  if (a->dtype == LSATTN_F16) return launch_mode<F16, true>(p, a, mode, st);
  return a->v_is_f16 ? launch_mode<BF16, true>(p, a, mode, st) : launch_mode<BF16, false>(p, a, mode, st);
}

}  // namespace lsattn

extern "C" int lsattn_prefill_converts_v(const lsattn_prefill_args* a) {
  if (!a || a->dtype != LSATTN_BF16) return 0;
  if (a->head_dim != 128) return 1;
  // (a V that the tile loads cannot read as it lies is copied: the copy lies straight)
  if (((uintptr_t)a->v & 15) || a->v_stride_t % 8 || a->v_stride_h % 8 || a->v_stride_t <= 0 || a->v_stride_t > (1 << 24)) return 0;
  return lsattn::prefill_short_blocks(a) != 0;
}
