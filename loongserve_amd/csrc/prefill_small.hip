// The prefill attention step for head sizes 16, 32 and 64 (the reference's Triton kernel takes them beside 128:
// loongserve/models/llama/triton_kernel/ring_context_flashattention_nopad.py:248-250) and, for batches of short prompts, 128
// (prefill_short_blocks), gfx950, wave64.
//
// What bounds it at 64 and below is vector work: a 32 x 32 block of scores takes a wave 16 exponentials, 16 multiply-adds, 16 additions and
// some 15 conversions and checks against 18 (D = 64) to 8 (D = 16) MFMAs, and the time falls only a third from D = 64 to 16.  At 128
// it is MFMA and LDS, and for short prompts the start and end of workgroups.
// Hence no work beside those in the common path, and three or four waves per SIMD whose phases mix freely:
//   * a workgroup of four waves; a wave owns 32 (small launches: 16) query positions of one head.  With grouped-query
//     heads up to four heads of a KV head sit side by side in a workgroup, which then ends sooner on the diagonal;
//   * K and V tiles of 64 keys (two stages), or 32 (128-wide heads, 32 positions: three), go to LDS by direct loads, one barrier per tile,
//     chunks XOR-swizzled (bfloat16 V passes through registers and becomes fp16 there);
//   * scores transposed, S^T = K Q^T with v_mfma_f32_16x16x32 (a head of 16 fills half of the contraction with
//     zeros), 32 keys per step, so a lane owns one query column: the fp32 scores turn into the B operand of O^T += V^T P^T in
//     place (P and V as fp16, sums of P in fp32), V^T operands through ds_read_b64_tr_b16; a wave skips the steps none of its
//     rows sees;
//   * the running maximum of a row is raised only when a P of 2 or more shows up; no exchange between lanes otherwise;
//   * the three epilogues of the 128-wide kernel: 0 the step's fp32 partial (O, LSE), 1 the reference's in-place
//     (o, m, l) update (ring_context_flashattention_nopad.py:171-188), 2 the LSE merge into a running fp32 (O, LSE); O is turned round
//     in LDS first, so that stores fill whole lines.
// Measured (fp16, causal, in place, whole calls): D = 64, 8 x 2048 tokens GQA 32/8 172 to 178 us (0.78 PFLOP/s), 16 x 512 43, 32 x 256 34,
// 16 x 1024 107; D = 128, 16 x 1024 191 us (0.72 PFLOP/s), 16 x 512 65, 1 x 100 8.7 replayed from a graph (of which 3.6 are the fills of m and l; 4.9 as a partial).
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
  int32_t batch, bunch, turns;  // the grid takes `bunch` requests at a time; whether their places move on by one from tile to tile
  FastDiv d_bunch;
};

constexpr int kWaves = 4;   // waves per workgroup
constexpr uint32_t kOnes = 0x3C003C00u;  // two ones in fp16
constexpr int64_t kCUs = 256;
constexpr int64_t kL2Bytes = 32 << 20;    // of the eight L2s together
constexpr int64_t kBunchWorkgroups = 512; // workgroups of a bunch of requests of about equal, short lengths
constexpr int64_t kShortMaxKeys = 1280;   // 128-wide heads: the keys of the longest request up to which this kernel may take a step,
constexpr int64_t kLoneMaxKeys = 1472;    // of a lone prompt folded in place,
constexpr int64_t kPartsMaxKeys = 2304, kPartsMaxKeysBf16 = 2048;  // and of one in up to a workgroup per CU, whose tiles two waves share
// Two waves per wave's positions (KP = 2) from so many keys on: one workgroup per CU and less of 16 positions per wave, 128-wide heads, one wave each |
// two (us, in place; 8/1 where nothing is said): 300 tokens 9.5 | 9.6, 32/32 9.1 | 9.5; 450 11.3 | 10.9, 32/32 11.8 | 11.7; 500 32/8 12.8 | 12.1; 600 13.6 | 12.7;
// 900 17.6 | 15.7; 1280 22.6 | 19.4; a full step of a ring of 900 18.7 | 16.5.
constexpr int64_t kPartsMinKeys = 512;
constexpr int64_t kMaxIds = 65535;  // of the second or third index of a grid

// s_waitcnt vmcnt(N) (expcnt / lgkmcnt fields left at their maximum)
template <int N> __device__ __forceinline__ void wait_loads() { __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14)); }

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

// A launch's shape by head size and positions per wave: keys per LDS tile, tiles in LDS (requested one fewer ahead), workgroups per CU.
// 128-wide heads, 32 positions per wave: three stages of 32 keys (48 KB) and at most 168 registers (158; 168 where V is bfloat16), so that three
// workgroups fit a CU.
template <int D, int WP> constexpr int kTileOf = D == 128 && WP == 32 ? 32 : 64;
template <int D, int WP> constexpr int kStagesOf = D == 128 && WP == 32 ? 3 : 2;
template <int D, int WP, bool DV> constexpr int kResident = D == 128 ? (WP == 32 ? 3 : 2) : WP == 32 && D == 64 && !DV ? 3 : 4;

// DV: the V tiles are fp16 in memory and go straight into LDS as the K tiles do; otherwise (bfloat16 V) they pass through
// registers and are converted on the way.  WP: query positions per wave, 16 or 32.  (Products of 32 x 32 x 16, which take a tenth fewer
// vector instructions, ran at 1.88 GHz where these run at 2.16: 8 ragged sequences of 64-wide heads 164 us against 161, 16 x 1024 tokens of
// 128-wide ones 199 against 194.)
// KP = 2: two waves share the positions of a wave and take the first and the second 32 keys of every tile (launches of up to a workgroup per CU, whose one
// wave per SIMD issues an instruction every five cycles or so); their parts are joined in LDS.  A tile takes 0.75 us of a lone workgroup instead of 0.96, the join and the start
// of twice the waves 1.1.
template <typename T, int D, int MODE, bool DV, int WP, int KP = 1>
__global__ __launch_bounds__(kWaves * KP * 64, (kResident<D, WP, DV>)) void prefill_small_kernel(SmallParams p) {
  static_assert(KP == 1 || (KP == 2 && WP == 16 && D >= 32), "the parts of a tile of 64 keys, the columns that each of two waves finishes");
  constexpr int NW = kWaves * KP;
  constexpr int QB = WP / 16;               // blocks of 16 positions per wave
  constexpr int KS = D >= 32 ? D / 32 : 1;  // contraction steps of Q K^T (32 elements each; D = 16 fills half of one)
  constexpr int NDB = D / 16;               // 16-wide blocks of the head
  constexpr int TK = kTileOf<D, WP>, NS = kStagesOf<D, WP>;
  constexpr int CPR = D / 8;                // 16-byte chunks per K or V row
  constexpr int RB = D * 2;                 // bytes per row in LDS
  constexpr int TB = TK * RB;               // bytes per tile
  constexpr int RPI = 64 / CPR;             // rows per load instruction (a wave's 64 lanes, 16 bytes each)
  constexpr int NI = (TK + NW * RPI - 1) / (NW * RPI);  // load instructions per wave and tile
  constexpr int RPB = 256 / RB;             // rows that pass all 64 LDS banks once
  // NS stages of (K tile, V tile): the next tiles are written while the present one is read.  Rows are not padded (a load to
  // LDS writes 1 KB in a row); instead the 16-byte chunks of a row are XORed with a function of the row: K so that a
  // column of chunks of sixteen rows, which one read takes, lies in sixteen different sets of four banks, V so that 32 bytes of
  // each of eight rows (half a transposing read) cover the banks once.  Rows sixteen apart share their XOR.
  // (behind them, for the epilogue that folds into (o, m, l): 256 bytes per wave for the old m and l of its rows)
  constexpr int kStateOff = NS * 2 * TB;
  constexpr int kJoinOff = kStateOff + (MODE == 1 ? NW * 256 : 0);  // (KP = 2: the waves' maxima and sums)
  __shared__ __attribute__((aligned(1024))) char lds[kJoinOff + (KP > 1 ? NW * 256 : 0)];
  auto swz_k = [](int row) { return (row / RPB) & (CPR - 1); };
  auto swz_v = [](int row) { return ((row / RPB) & (CPR / 2 - 1)) << 1; };

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;  // query column, lane group
  const int rw = KP > 1 ? wave & (kWaves - 1) : wave, kp = KP > 1 ? wave / kWaves : 0;  // whose positions; which part of the keys
  // grid: (KV head, heads side by side), (tile from the last one down, request of a bunch), bunch of requests: the heaviest tiles of
  // all requests of a bunch start first, and with a multiple of eight KV heads the workgroups of one run on one XCD (ids are dealt round-robin)
  const int gq = (int)div_by(blockIdx.x, p.d_hkv), kvh = (int)blockIdx.x - gq * p.hkv;
  const int tile_id = (int)div_by(blockIdx.y, p.d_bunch);
  int place = (int)blockIdx.y - tile_id * p.bunch;
  if (p.turns) place += tile_id, place -= (int)div_by((uint32_t)place, p.d_bunch) * p.bunch;
  const int b = (int)blockIdx.z * p.bunch + place;
  if (b >= p.batch) return;
  const int rows_wg = (kWaves * WP) >> p.pack_shift;  // query positions of this workgroup
  const int m_wg = (p.last_tile - tile_id) * rows_wg;
  // (the request's numbers are all asked for before the first of them is used)
  const int q_len = p.q_len[b], kv_len = p.kv_len[b], qf = p.q_first[b], kf = p.kv_first[b], P = p.peers;
  const int q_start32 = p.q_start[b], kv_start32 = p.kv_start[b], o_start32 = p.o_start ? p.o_start[b] : q_start32;
  asm volatile("" ::"s"(q_len), "s"(kv_len), "s"(qf), "s"(kf), "s"(q_start32), "s"(kv_start32), "s"(o_start32));
  if (m_wg >= q_len) return;  // (the whole workgroup: the loop below holds barriers)
  const int wph_shift = 2 - p.pack_shift;  // log2 of the waves per head
  const int h = kvh * p.heads_per_kv + (gq << p.pack_shift) + (rw >> wph_shift);
  const int m0 = m_wg + (rw & ((1 << wph_shift) - 1)) * WP;  // the wave's first position
  const int64_t q_start = q_start32, kv_start = kv_start32, o_start = o_start32;

  // keys of this KV chunk visible to global query position qpos (ring_context_flashattention_nopad.py:156-159)
  auto visible_keys = [&](int qpos) -> int {
    const int dq = qpos - kf;
    const int n = dq >= 0 ? (int)div_by((uint32_t)dq, p.d_peers) + 1 : 0;
    return n > kv_len ? kv_len : n;
  };
  const int lds_base = (int)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
  // The old m and l (MODE 1) are asked for first of all and go straight into LDS: no register is held over the loop, and the epilogue need
  // not go to memory to learn whether a row is still in its start state, whose old o is never read.
  if (MODE == 1) {  // (lanes 0 to 31 the m of a position each, the others the l)
    const int m = m0 + (lane & (WP - 1));
    const int64_t at = (o_start + (m < q_len ? m : m_wg)) * p.ml_st + (int64_t)h * p.ml_sh;
    const float* src = (lane < 32 ? p.m : p.l) + at;
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" ::"s"(lds_base + kStateOff + wave * 256), "v"(src) : "m0", "memory");
  }
  // per block qb of 16 positions, the lane's position m0 + 16 qb + c
  int cnt[QB];           // keys it sees (0 if it does not exist), from the lane's first key of a step
  u32x4 qreg[QB][KS];    // Q^T as B operands: qreg[qb][ks] = Q[position][32 ks + 8 g .. + 7]
  f32x4 oacc[QB][NDB];   // O^T: oacc[qb][db][j] = O[position][16 db + 4 g + j]
  float m_run[QB], l_run[QB];  // log2-domain running max of the column; the lane's share of its running sum
  f32x4 l_pv[QB];        // the column's sum of the fp16 values that multiply V (all four elements)
#pragma unroll
  for (int qb = 0; qb < QB; qb++) {
    const int m = m0 + 16 * qb + c;
    cnt[qb] = (m < q_len ? visible_keys(qf + m * P) : 0) - 4 * g;
    const char* src = (const char*)p.q + ((q_start + (m < q_len ? m : m_wg)) * p.q_st + (int64_t)h * p.q_sh) * 2;
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
  const int cnt_wave = __builtin_amdgcn_readfirstlane(last_seen(m0, WP));
  // (rows past the end see nothing: a wave that holds some masks everywhere only where it has to, in their own columns,
  // which nothing reads; its first row sees the fewest keys of the others)
  const int cnt_first = __builtin_amdgcn_readfirstlane(m0 < q_len ? visible_keys(qf + m0 * P) : 0);
  const int cnt_wg = __builtin_amdgcn_readfirstlane(last_seen(m_wg, rows_wg));

  const char* kbase = (const char*)p.k + (kv_start * p.k_st + (int64_t)kvh * p.k_sh) * 2;
  const char* vbase = (const char*)p.v + (kv_start * p.v_st + (int64_t)kvh * p.v_sh) * 2;
  // staging: instruction i of a wave carries rows (wave + 4 i) * RPI .. of the K tile and of the V tile.  Tiles that lie inside the
  // chunk take a scalar tile address and the lane's 32-bit offset, no vector arithmetic.
  const bool stager = NI * NW * RPI == TK || wave * RPI < TK;  // (D = 16: two waves)
  const int st_row = wave * RPI + lane / CPR;
  const uint32_t k_row = (uint32_t)p.k_st * 2, v_row = (uint32_t)p.v_st * 2;  // (a tile's rows span less than 2^31 bytes)
  const uint32_t k_off = st_row * k_row + ((lane % CPR) ^ swz_k(st_row)) * 16, v_off = st_row * v_row + ((lane % CPR) ^ swz_v(st_row)) * 16;
  constexpr int STEP = NW * RPI;  // rows between a wave's load instructions
  constexpr bool APART = !DV && NS > 2;  // K tiles are requested NS - 1 tiles ahead, V tiles that pass through registers one
  u32x4 vst[NI];
  // K and V of tile t (or one of them)
  auto request = [&](auto k_tag, auto v_tag, int stage, int t) __attribute__((always_inline)) {
    constexpr bool K = decltype(k_tag)::value, V = decltype(v_tag)::value;
    if (!stager) return;
    const char* kt = K ? uniform_ptr(kbase + (int64_t)t * TK * k_row) : nullptr;
    const char* vt = V ? uniform_ptr(vbase + (int64_t)t * TK * v_row) : nullptr;
    const int dst = __builtin_amdgcn_readfirstlane(lds_base + stage * 2 * TB + wave * 1024);
    const int last = kv_len - 1 - t * TK;
#pragma unroll
    for (int i = 0; i < NI; i++) {
      uint32_t ko = k_off, vo = v_off;
      if (last < TK - 1) {  // (wave-uniform; rows past the end repeat the last one and are masked)
        int r0 = st_row;
        asm volatile("" : "+v"(r0));  // (worked out here and not kept in registers over the loop)
        int back = r0 + i * STEP - last;
        back = back < 0 ? 0 : back;
        if (K) ko -= (uint32_t)back * k_row;
        if (V) vo -= (uint32_t)back * v_row;
      }
      if (K) load_to_lds(dst + i * NW * 1024, kt, ko + (uint32_t)(i * STEP) * k_row);
      if (V && DV) load_to_lds(dst + TB + i * NW * 1024, vt, vo + (uint32_t)(i * STEP) * v_row);
      if (V && !DV) vst[i] = *(const u32x4*)(vt + (vo + (uint32_t)(i * STEP) * v_row));
    }
  };
  constexpr std::true_type yes{};
  constexpr std::false_type no{};
  auto deposit_v = [&](int stage) __attribute__((always_inline)) {  // (bfloat16 V: the tile in the registers into LDS)
    if (!DV && stager) {
#pragma unroll
      for (int i = 0; i < NI; i++) *(u32x4*)(lds + stage * 2 * TB + TB + (wave + i * NW) * 1024 + lane * 16) = bf16_to_f16(vst[i]);
    }
  };
  // transposing read: lane c of a 16-lane group points at row c >> 2, columns 4 (c & 3) .. + 3 of a 4 x 16 block and
  // receives column c of it; group g takes rows 4 g .. 4 g + 3 and, sixteen rows on, 16 + 4 g .. + 3: the eight keys
  // whose scores the lane holds
  // (the contraction step and the block are bits of the chunk number that g and the lane leave free, so they are XORed into the address:
  // in registers of their own, or, where none are to spare (LEAN), next to each read)
  constexpr bool LEAN = D == 128 && WP == 32;
  constexpr bool LEAN_V = LEAN || (D == 64 && WP == 32);
  constexpr int NKA = LEAN ? 1 : KS, NVA = LEAN_V ? 1 : NDB;
  int kaddr[NKA], vaddr[NVA];
#pragma unroll
  for (int ks = 0; ks < NKA; ks++) kaddr[ks] = lds_base + c * RB + (((4 * ks + g) & (CPR - 1)) ^ swz_k(c)) * 16;
#pragma unroll
  for (int db = 0; db < NVA; db++) {
    const int row = 4 * g + (c >> 2);
    vaddr[db] = lds_base + TB + row * RB + ((2 * db + ((c & 3) >> 1)) ^ swz_v(row)) * 16 + (c & 1) * 8;
  }
  auto kaddr_of = [&](int ks) __attribute__((always_inline)) {
    if (!LEAN) return kaddr[LEAN ? 0 : ks];
    int a = kaddr[0];
    if (ks) asm volatile("v_xor_b32 %0, %1, %2" : "=v"(a) : "n"(ks * 64), "v"(kaddr[0]));
    return a;
  };
  auto vaddr_of = [&](int db) __attribute__((always_inline)) {
    if (!LEAN_V) return vaddr[LEAN_V ? 0 : db];
    int a = vaddr[0];
    if (db) asm volatile("v_xor_b32 %0, %1, %2" : "=v"(a) : "n"(db * 32), "v"(vaddr[0]));
    return a;
  };
  const float scale = p.scale_log2;
  const int nt = (cnt_wg + TK - 1) / TK;  // the same for every wave of the workgroup

  constexpr int VR = LEAN ? 4 : NDB;       // V operands
  u32x4 ka[2][KS];  // K operands of the next 32 keys
  auto load_ka = [&](int at) __attribute__((always_inline)) {
#pragma unroll
    for (int kb = 0; kb < 2; kb++)
#pragma unroll
      for (int ks = 0; ks < KS; ks++) {
        u32x4 x = *(const __attribute__((address_space(3))) u32x4*)(kaddr_of(ks) + at + kb * 16 * RB);
        if (D == 16 && g >= 2) x = u32x4{0u, 0u, 0u, 0u};
        ka[kb][ks] = x;
      }
  };
  auto tile = [&](auto stage_tag, int t) __attribute__((always_inline)) {
    constexpr int S = decltype(stage_tag)::value;
    // the wave's loads of this tile have landed (those of a tile behind it may be under way), then everyone meets: the tile is complete,
    // and the stage of the tile before it is done with and takes the next request
    if (DV && NS > 2 && t + 1 < nt) wait_loads<2 * NI * (NS - 2)>();
    else wait_loads<0>();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if constexpr (APART) {
      if (t + NS - 1 < nt) request(yes, no, (S + NS - 1) % NS, t + NS - 1);
      if (t + 1 < nt) request(no, yes, 0, t + 1);  // (into registers)
    } else {
      if (t + NS - 1 < nt) request(yes, yes, (S + NS - 1) % NS, t + NS - 1);
    }
    const int k_wave = 32 * kp, b_wave = k_wave * RB;  // (KP = 2) the wave's first key of the tile
    if (t * TK + k_wave < cnt_wave) load_ka(S * 2 * TB + b_wave);
#pragma unroll
    for (int part = 0; part < TK / 32 / KP; part++) {
      const int k0 = t * TK + k_wave + 32 * part;
      if (k0 < cnt_wave) {  // (wave-uniform: else none of the wave's rows sees these keys)
        // S^T = K Q^T: s[qb][kb][j] = score of key k0 + 16 kb + 4 g + j for the lane's query of block qb; a K operand serves all blocks
        // (starting from named zeros: with the zero written into the first product the 128-wide kernel spills 22 registers)
        f32x4 s[QB][2];
#pragma unroll
        for (int qb = 0; qb < QB; qb++) s[qb][0] = s[qb][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ks++)
#pragma unroll
          for (int kb = 0; kb < 2; kb++)
#pragma unroll
            for (int qb = 0; qb < QB; qb++) s[qb][kb] = MfmaS<T>::run(ka[kb][ks], qreg[qb][ks], s[qb][kb]);
        if (k0 + 32 > cnt_first) {  // (wave-uniform: the wave's first row, which sees the fewest keys, does not see the whole step)
#pragma unroll
          for (int qb = 0; qb < QB; qb++) {
            const int rel = cnt[qb] - k0;
#pragma unroll
            for (int e = 0; e < 8; e++) s[qb][e / 4][e % 4] = 16 * (e / 4) + e % 4 < rel ? s[qb][e / 4][e % 4] : -INFINITY;
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
        u32x4 va[VR];  // V operand of block db in va[db % VR]
        auto load_va = [&](int db) __attribute__((always_inline)) {
          const int at = vaddr_of(db) + b_wave + S * 2 * TB + 32 * part * RB;
          const i16x4 xa = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_ptr)at);
          const i16x4 xb = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_ptr)(at + 16 * RB));
          const u32x2 wa = __builtin_bit_cast(u32x2, xa), wb = __builtin_bit_cast(u32x2, xb);
          return u32x4{wa[0], wa[1], wb[0], wb[1]};
        };
#pragma unroll
        for (int db = 0; db < VR; db++) va[db] = load_va(db);
        if (part + 1 < TK / 32 / KP) load_ka(S * 2 * TB + 32 * (part + 1) * RB);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int db = 0; db < NDB; db++) {
#pragma unroll
          for (int qb = 0; qb < QB; qb++) oacc[qb][db] = MfmaS<F16>::run(va[db % VR], pk[qb], oacc[qb][db]);
          if (db + VR < NDB) {
            va[db % VR] = load_va(db + VR);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
#pragma unroll
        for (int qb = 0; qb < QB; qb++) l_pv[qb] = MfmaS<F16>::run(u32x4{kOnes, kOnes, kOnes, kOnes}, pk[qb], l_pv[qb]);
      }
    }
    if (!DV && t + 1 < nt) deposit_v((S + 1) % NS);
  };
#pragma unroll
  for (int t = 0; t < NS - 1; t++) {
    if (t < nt) {
      if (APART && t > 0) request(yes, no, t, t);
      else request(yes, yes, t, t);
    }
  }
  if (nt > 0) deposit_v(0);
  for (int t = 0; t < nt; t += NS) {  // (the stage is a constant of the code)
    tile(std::integral_constant<int, 0>{}, t);
    if (t + 1 < nt) tile(std::integral_constant<int, 1>{}, t + 1);
    if constexpr (NS == 3)
      if (t + 2 < nt) tile(std::integral_constant<int, 2>{}, t + 2);
  }

  // ---- epilogues (the 128-wide kernel's) ----
  // O leaves through LDS (MODE 0 and 1, 32 positions per wave): written as the lanes hold it, a store touches 16 rows with 32 or 64 bytes
  // each, a request per row to the L2s, and turned round whole lines of a few rows: 16 x 1024 tokens 32/8 199 -> 190 us in
  // place and 207 -> 201 as fp32, 16 x 512 bf16 72 -> 66 (128-wide heads).  The small launches of 16 positions write directly (turned round, 1 x 100 took 0.4 us more).
  constexpr bool TURNED = MODE != 2 && WP == 32;
  constexpr int ES = MODE == 1 ? 2 : 4;                // bytes per element of O
  constexpr int RBO = D * ES < 256 ? D * ES : 256;     // bytes of a row that are turned round at a time
  constexpr int CO = RBO / 16;                         // 16-byte chunks of them, XORed with a function of the row as the tiles' are
  static_assert(!TURNED || kWaves * WP * RBO <= kStateOff, "the tiles' LDS holds the waves' rows");
  auto o_chunk = [](int row, int chunk) { return row * RBO + ((chunk ^ (row / (256 / RBO) & (CO - 1))) << 4); };
  char* const o_lds = lds + wave * WP * RBO;
  if (MODE == 1 && nt == 0) wait_loads<0>();  // (else the loop has waited for the old m and l)
  if (TURNED) __syncthreads();                // (the last tile is done with)
  // KP = 2: every wave leaves the half of O that the other finishes in LDS (the tiles are done with), its maximum and its sums, and joins the
  // other's with its own half, EDB blocks that are oacc[0][0 .. EDB - 1] from here on, columns from col0.
  constexpr int EDB = NDB / KP;
  const int col0 = 16 * EDB * kp;
  float lse_old = 0.f;  // (MODE 2)
  if constexpr (KP > 1) {
    static_assert(NW * EDB * 1024 <= kStateOff, "the tiles' LDS holds the halves");
    if (MODE == 2) {  // (read before the wave that replaces it may write)
      lse_old = p.lse[(o_start + (m0 + c < q_len ? m0 + c : m_wg)) * p.hq + h];
      asm volatile("" ::"v"(lse_old));
    }
    const float l_wave = col_sum(l_run[0]);
    const int other = wave ^ kWaves;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < EDB; i++) {
      *(f32x4*)(lds + (wave * EDB + i) * 1024 + lane * 16) = kp ? oacc[0][i] : oacc[0][EDB + i];
      if (kp) oacc[0][i] = oacc[0][EDB + i];
    }
    if (g == 0) *(f32x4*)(lds + kJoinOff + wave * 256 + c * 16) = f32x4{m_run[0], l_wave, l_pv[0][0], 0.f};
    __syncthreads();
    const f32x4 st = *(const f32x4*)(lds + kJoinOff + other * 256 + c * 16);
    const float top = fmaxf(m_run[0], st[0]);
    const float w0 = exp2_diff(m_run[0], top), w1 = exp2_diff(st[0], top);  // (0 for a part that saw no key)
    l_run[0] = l_wave * w0 + st[1] * w1;
    l_pv[0][0] = l_pv[0][0] * w0 + st[2] * w1;
#pragma unroll
    for (int i = 0; i < EDB; i++) oacc[0][i] = oacc[0][i] * w0 + *(const f32x4*)(lds + (other * EDB + i) * 1024 + lane * 16) * w1;
    m_run[0] = top;
  }
  if (m0 >= q_len) return;                    // (wave-uniform: a wave without positions; it only helped to stage)
  // (the lane's numbers are worked out again and not kept over the loop)
  const int lane_e = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)), c_e = lane_e & 15, g_e = lane_e >> 4;
  uint32_t rows = 0;      // (MODE 1) which of the wave's rows are written
  float factor[QB];       // (MODE 0) of the row's O
#pragma unroll
  for (int qb = 0; qb < QB; qb++) {
    const int mb = m0 + 16 * qb;
    const float l_tot = KP > 1 ? l_run[qb] : col_sum(l_run[qb]);
    // (0 exactly if the row saw no key.  A NaN score makes the sum NaN: it counts as a key, so that the row's outputs and its running
    // state become NaN, as they do in the reference, and no step before or after hides it)
    const bool seen = !(l_tot == 0.f);
    // O becomes a mean with the very weights it was summed with: a rounding that a row's weights share (one key that outweighs
    // the others) falls out of it, which makes up for maxima that lag (a P of 1 is exact in fp16, one of 1.4 is not).
    // Against 64 bits the fp32 partial of N(0, 1) * 0.5 inputs is off by 1.70e-4 to 1.72e-4 at 1000 to 3000 tokens of 64-wide heads,
    // 1.74e-4 to 1.75e-4 with maxima that never lag and 1.76e-4 with neither.  The sum that (m, l) and the LSE state stays the fp32 one.
    const float fix = l_pv[qb][0] == 0.f ? 0.f : l_tot / l_pv[qb][0];
    const int m_e = mb + c_e;
    const bool here = m_e < q_len;
    const int64_t tok = o_start + (here ? m_e : m0);  // (a lane without a position: the wave's first, never written)
    if (MODE == 0) {
      factor[qb] = seen ? fix * (1.f / l_tot) : 0.f;
      if (here) {
        if (!TURNED) {
          float* orow = (float*)p.o + tok * p.o_st + (int64_t)h * p.o_sh + col0 + 4 * g_e;
#pragma unroll
          for (int db = 0; db < EDB; db++) *(f32x4*)(orow + 16 * db) = oacc[qb][db] * factor[qb];
        }
        if (g_e == 0 && kp == 0) p.lse[tok * p.hq + h] = seen ? (m_run[qb] + __builtin_amdgcn_logf(l_tot)) * kLn2 : -INFINITY;
      }
    }
    if (MODE == 1) {
      // the reference's update of (o, m, l); a row in its start state (m = -inf, l = 0) may hold anything in o
      const float m_old = *(const float*)(lds + kStateOff + wave * 256 + (16 * qb + c_e) * 4);
      const float l_old = *(const float*)(lds + kStateOff + wave * 256 + 128 + (16 * qb + c_e) * 4);
      const float M = fmaxf(m_run[qb], m_old);
      const bool upd = here && seen;  // (a row that saw a key has a maximum, unless all its scores are NaN)
      const float w_old = upd ? l_old * exp2_diff(m_old, M) : 0.f;
      const float w_new = exp2_diff(m_run[qb], M) * fix;
      const float L = w_old + l_tot * exp2_diff(m_run[qb], M);
      const float inv = 1.f / L;
      uint16_t* orow = (uint16_t*)p.o + tok * p.o_st + (int64_t)h * p.o_sh + col0 + 4 * g_e;
      u32x2 old[EDB];
#pragma unroll
      for (int db = 0; db < EDB; db++) old[db] = u32x2{0u, 0u};
      // (a wave none of whose rows carries an earlier step's result, as in the first step of a ring and in a prefill on one GPU, does not
      // read o; w_old is NaN if an old sum or maximum is)
      if (__builtin_amdgcn_ballot_w64(w_old != 0.f) != 0) {
        if (w_old != 0.f) {
#pragma unroll
          for (int db = 0; db < EDB; db++) old[db] = *(const u32x2*)(orow + 16 * db);
        }
      }
#pragma unroll
      for (int db = 0; db < EDB; db++) {
        float o0, o1, o2, o3;
        unpack2<T>(old[db][0], o0, o1);
        unpack2<T>(old[db][1], o2, o3);
        const f32x4& x = oacc[qb][db];
        const u32x2 res = u32x2{pack2<T>((o0 * w_old + x[0] * w_new) * inv, (o1 * w_old + x[1] * w_new) * inv),
                                pack2<T>((o2 * w_old + x[2] * w_new) * inv, (o3 * w_old + x[3] * w_new) * inv)};
        if (TURNED) *(u32x2*)(o_lds + o_chunk(16 * qb + c_e, 2 * db + (g_e >> 1)) + (g_e & 1) * 8) = res;
        else if (upd) *(u32x2*)(orow + 16 * db) = res;
      }
      rows |= (uint32_t)(__builtin_amdgcn_ballot_w64(upd) & 0xffffu) << 16 * qb;
      if (upd && g_e == 0 && kp == 0) {
        p.m[tok * p.ml_st + (int64_t)h * p.ml_sh] = M;
        p.l[tok * p.ml_st + (int64_t)h * p.ml_sh] = L;
      }
    }
    if (MODE == 2) {
      // fold the step's partial into the running fp32 (O, LSE); a row that saw no key stays as it is
      const bool upd = here && seen;
      const float a_old = (KP > 1 ? lse_old : p.lse[tok * p.hq + h]) * kLog2e;
      float new_lse = 0.f;
      if (upd) {
        const float a_new = m_run[qb] + __builtin_amdgcn_logf(l_tot);
        const float top = fmaxf(a_old, a_new);
        const float w_old = exp2_diff(a_old, top);
        const float w_new = __builtin_amdgcn_exp2f(a_new - top);
        const float W = w_old + w_new;
        const float c_old = w_old / W, c_new = w_new / (W * l_tot) * fix;
        float* orow = (float*)p.o + tok * p.o_st + (int64_t)h * p.o_sh + col0 + 4 * g_e;
#pragma unroll
        for (int db = 0; db < EDB; db++) {
          // an empty row (lse = -inf) may hold anything: its old values are dropped, not multiplied by zero
          const f32x4 keep = w_old != 0.f ? *(const f32x4*)(orow + 16 * db) : f32x4{0.f, 0.f, 0.f, 0.f};
          *(f32x4*)(orow + 16 * db) = keep * c_old + oacc[qb][db] * c_new;
        }
        new_lse = (top + __builtin_amdgcn_logf(W)) * kLn2;
      }
      if (upd && g_e == 0 && kp == 0) p.lse[tok * p.hq + h] = new_lse;
    }
  }
  if (TURNED) {
    // (four-byte words of a row's 16 bytes: o_stride_t and o_stride_h are multiples of four elements)
    typedef u32x4 ChunkAt8 __attribute__((aligned(8)));
    char* obase = (char*)p.o + ((o_start + m0) * p.o_st + (int64_t)h * p.o_sh) * ES;
    const int n_rows = q_len - m0 < WP ? q_len - m0 : WP;
#pragma unroll
    for (int half = 0; half < D * ES / RBO; half++) {
      if (MODE == 0) {
#pragma unroll
        for (int qb = 0; qb < QB; qb++)
#pragma unroll
          for (int db = half * RBO / 64; db < NDB && db < (half + 1) * RBO / 64; db++)
            *(f32x4*)(o_lds + o_chunk(16 * qb + c_e, 4 * db - half * CO + g_e)) = oacc[qb][db] * factor[qb];
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // (the wave's own rows: its LDS instructions keep their order)
#pragma unroll
      for (int it = 0; it < WP * CO / 64; it++) {
        const int r = it * (64 / CO) + lane_e / CO;
        const u32x4 v = *(const u32x4*)(o_lds + o_chunk(r, lane_e % CO));
        if (MODE == 1 ? (rows >> r & 1) != 0 : r < n_rows) *(ChunkAt8*)(obase + r * p.o_st * ES + half * RBO + lane_e % CO * 16) = v;
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
  }
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

// Rows of K that the requests read, as far as the host can tell: those of the prompts, and of contexts where the caller bounds them.  The K
// buffer may have more (a view with spare rows).
int64_t kv_rows_read(const lsattn_prefill_args* a) {
  const int64_t most = (int64_t)a->batch * a->max_q_len, prompts = a->total_q_rows > 0 && a->total_q_rows < most ? a->total_q_rows : most;
  const int64_t contexts = a->max_kv_len > a->max_q_len ? (int64_t)a->batch * (a->max_kv_len - a->max_q_len) : 0;
  int64_t rows = a->total_kv_rows;
  if (prompts + contexts < rows) rows = prompts + contexts;
  if (a->max_kv_len > 0 && (int64_t)a->batch * a->max_kv_len < rows) rows = (int64_t)a->batch * a->max_kv_len;
  return rows;
}

// Whether a request's place among the ids moves on from tile to tile.  Ids go to the eight XCDs in turn and within one to its four
// shader engines.  If the ids of two tiles of a request are a multiple of 32 apart, all its workgroups share one shader engine of an
// XCD, and while only the longest requests have a tile left to start, the others idle: 8 sequences of 1000 to 3000 tokens, 32/8 heads
// of 64, had 2 workgroups on a CU until half of the launch was over, some 4 and some 1, where 8 x 2048 keep 3.9.  Turning places
// fill them evenly.  Measured over 60 ragged launches (2 to 32 sequences, 300 to 6000 tokens; microseconds, fixed | turning):
//   8 x 1000..3000 32/8 183 | 165   2 x 1206..3618 64/8 144 | 123   4 x 120..3615 64/8 bf16 87.9 | 61.8   4 x 688..2064 32/32 53.2 | 47.3
//   4 x 2582..5165 32/8 bf16 344 | 314   8 x 1304..2608 12/12 88.8 | 79.5   16 x 31..959 64/8 57.3 | 53.5
// At other distances (11 x 388..1166 32/8 44.8 | 47.1; distance 6 of the eights 9 % better to 4 % worse), with fewer than 16 tiles
// (8 x 280..842 32/32 31.5 | 33.3) and with equal lengths turning gains nothing: there the places stay.
bool ragged(const lsattn_prefill_args* a) { return a->total_q_rows > 0 && a->total_q_rows * 10 <= (int64_t)a->batch * a->max_q_len * 9; }
bool requests_take_turns(const lsattn_prefill_args* a, int64_t ids_per_tile, int64_t tiles) {
  return ids_per_tile % 32 == 0 && tiles >= 16 && ragged(a);
}

// How many requests the grid takes at a time (a bunch), the heaviest tiles of all of them first.  All of the batch starts the heaviest work of the
// launch first, and is best for ragged batches; but every layer of tiles then reads the K/V of the whole batch again, which past the
// L2s' 32 MB comes from beyond them, so bunches hold about as much.  And short prompts of about equal length leave the CUs unevenly filled that
// way (their workgroups come in layers of equal length): in bunches of some 512 workgroups, light tiles of one run beside heavy
// ones of the next.  Measured (microseconds, 1, 2, 4, 8, 16 and 32 requests at a time up to the batch, 128-wide heads):
//   16 x 512 32/32 (8 MB each) 77 75 78 86 99   16 x 1024 32/32 (16 MB) 231 229 235 243 262   32 x 512 32/32 170 169 171 182 197 201
//   32 x 256 32/8 52.2 50.6 47.9 52.0 61.4 61.4   16 x 256 32/8 34.6 32.8 30.8 30.5 35.6   8 x 512 32/8 44.3 42.0 37.8 43.4   16 x 512 32/8 71 67 64 70 72
//   16 x 1024 32/8 216 207 204 201 206   4 x 1024 32/8 62.7 57.9 55.3   ragged: 8 x 100..2000 32/8 70.6 68.9 64.3 61.2, 20 x 200..800 32/8 81 78 72 80 80 71 (all 20)
// and 64-wide: 16 x 1024 32/32 119 120 125 128 140   8 x 2048 32/32 198 192 189 210   16 x 1024 32/8 117 112 112 108 108
// Short equal prompts over 3000 launches (2 to 60 of 60 to 512 tokens), in bunches of some 512 workgroups, of the time of all at once (the mean; 95 of 100
// stay below): 128-wide 0.97 (1.03); narrower heads, one per workgroup, from two rounds of the chip on 0.86 (0.99), below 0.99 (1.07); several
// side by side, whose prompts have up to four times the tiles, 1.02 (1.12), the worst 1.28 (11 x 333 64/8 16-wide 17.9 | 20.7).  Narrower heads thus
// only the first of these.
// The K/V bytes are those that the requests read (kv_rows_read), not those of the buffer: in bunches of one or two for a larger buffer's sake, requests
// of 16- to 64-wide heads took up to a third longer (14 x 1300 at most 16/16 against 65536 rows; 250 ragged batches 1.035 in the mean).  Ragged batches
// gain by bytes too, though they lose the heaviest-first order of the whole batch, but not where a bunch is about one round of workgroups, which then
// ends with the longest request's alone (16- to 64-wide heads, where one has 1024; 11 x 5345 at most 16/16 146 us whole, 193 in two).  Over launches of 300 to
// 6000 tokens whose K/V is 64 MB and more, of the time before the bunches (all at once | by bytes | by bytes from two rounds per bunch on; the mean, the worst):
//   16 to 64 wide, 540 ragged 0.944 1.05 | 0.899 1.33 | 0.910 1.05, 188 equal 0.950 1.06 | 0.888 1.19 | 0.913 1.06;  128 wide, 305 ragged 0.880 1.29 | 0.849 1.10, 143 equal 0.957 1.55 | 0.894 1.10
// (128-wide heads fill a bunch of 32 MB with half a round, and fare best so.)
int64_t requests_per_bunch(const lsattn_prefill_args* a, int64_t ids, int64_t tiles) {
  int64_t bunches = 1;
  const int64_t kv_bytes = kv_rows_read(a) * a->num_kv_heads * a->head_dim * 4;
  const int64_t wgs = ids * tiles * a->batch, resident = (a->head_dim == 128 ? 3 : 4) * kCUs;
  const int64_t by_kv = kv_bytes / kL2Bytes < a->batch ? kv_bytes / kL2Bytes : a->batch;
  if (by_kv > 1 && (a->head_dim == 128 || workgroups(a, pack_shift_of(a), 2) >= 2 * resident * by_kv)) bunches = by_kv;
  const bool layers = a->head_dim == 128 ? wgs > resident : pack_shift_of(a) == 0 && wgs >= 2 * resident;
  if (a->total_q_rows > 0 && !ragged(a) && a->max_q_len <= 512 && layers && wgs / kBunchWorkgroups > bunches) bunches = wgs / kBunchWorkgroups;
  if (bunches > a->batch) bunches = a->batch;
  return (a->batch + bunches - 1) / bunches;
}

struct Order {
  int64_t bunch;
  bool turns;
};
// (of the shape with 32 positions per wave; launches of the other are small)
Order order_of(const lsattn_prefill_args* a, int pack_shift) {
  const int64_t rows_wg = (kWaves * 32) >> pack_shift, tiles = (a->max_q_len + rows_wg - 1) / rows_wg, ids = a->num_q_heads >> pack_shift;
  const int64_t fits = tiles < kMaxIds ? kMaxIds / tiles : 1;  // (the grid's second index)
  int64_t bunch = requests_per_bunch(a, ids, tiles);
  bunch = bunch < fits ? bunch : fits;
  return {bunch, requests_take_turns(a, ids * bunch, tiles)};
}

template <typename T, int D, int MODE, bool DV, int WP, int KP = 1> int launch_rows(SmallParams p, const lsattn_prefill_args* a, hipStream_t st) {
  const int64_t rows_wg = (kWaves * WP) >> p.pack_shift;
  const Order order = WP == 32 ? order_of(a, p.pack_shift) : Order{p.batch, false};
  p.bunch = (int32_t)order.bunch;
  p.d_bunch = fast_div((uint32_t)p.bunch);
  p.turns = order.turns;
  const int64_t most = kMaxIds / p.bunch;  // tiles of one launch
  const unsigned bunches = (unsigned)((a->batch + p.bunch - 1) / p.bunch);
  for (int64_t tiles = (a->max_q_len + rows_wg - 1) / rows_wg; tiles > 0; tiles -= most) {
    p.last_tile = (int32_t)(tiles - 1);
    LSATTN_LAUNCH_KERNEL((prefill_small_kernel<T, D, MODE, DV, WP, KP>),
                         dim3((unsigned)(p.hkv * p.group), (unsigned)((tiles < most ? tiles : most) * p.bunch), bunches), dim3(kWaves * KP * 64), 0, st, p);
    const int rc = check_launch();
    if (rc != LSATTN_OK) return rc;
  }
  return LSATTN_OK;
}

// The most keys a request can have, as far as the host can tell: what the K buffer holds beyond the query rows may all belong to one request, unless the
// caller bounds the lengths.  kUnknownKeys: nothing is known.
constexpr int64_t kUnknownKeys = INT64_MAX;
int64_t longest_keys(const lsattn_prefill_args* a) {
  int64_t longest = kUnknownKeys;
  if (a->total_kv_rows > 0) {
    longest = a->total_kv_rows;
    if (a->total_q_rows > 0) {
      const int64_t most = (int64_t)a->batch * a->max_q_len, rows = a->total_q_rows < most ? a->total_q_rows : most;
      const int64_t beyond = a->total_kv_rows > rows ? a->total_kv_rows - rows : 0;
      if (a->max_q_len + beyond < longest) longest = a->max_q_len + beyond;
    }
  }
  if (a->max_kv_len > 0 && a->max_kv_len < longest) longest = a->max_kv_len;
  return longest;
}

// Whether two waves share a wave's positions (KP = 2) in a launch with 16 positions per wave.  Up to a workgroup per CU, and with 64-wide heads, whose waves have fewer products
// between their waits, up to three, the later the more there are.  Of the time of one wave each, 64 wide, over 270 launches (1 to 8 prompts of 150 to
// 2500 tokens; 32/32, 32/8, 64/8, 16/16 and 8/1 heads, f16 and bf16, partials and in place), by the longest prompt:
//   up to one per CU   below 300 1.01   300 to 450 0.97   to 600 0.93   to 800 0.90   to 1100 0.88   to 2500 0.84 (1700 tokens 32/8 bf16 27.4 -> 23.2 us)
//   up to two          below 300 1.11   300 to 600 1.00   to 800 0.93   to 1100 0.90   to 2500 0.85      up to three   below 1100 1.02 to 1.15   to 1500 0.93   to 2500 0.89
// and past that 0.99 to 1.21.  Per CU as if all requests were as long as the longest: of ragged ones the workgroups without rows leave early and the long ones meet on
// a few CUs, where twice the waves take up to 1.36 of the time (4, one of 742, full steps, 16/1 128 wide 39.6 | 45.4; 4 of at most 2075 8/8 64 wide 27.0 | 30.8); and of several requests by the
// keys of the mean one, or of the longest prompt: what the K buffer holds beyond the rows was taken for one request's context (6 of at most 61 rows behind 87 keys 40/8 7.7 | 8.7).
bool two_waves_share(const lsattn_prefill_args* a) {
  const int64_t rows = (kWaves * 16) >> pack_shift_of(a);
  const int64_t most = (int64_t)a->batch * ((a->max_q_len + rows - 1) / rows) * (a->num_q_heads >> pack_shift_of(a));
  int64_t keys = longest_keys(a);
  if (a->batch > 1 || keys == kUnknownKeys) {
    const int64_t mean = a->total_kv_rows / a->batch, likely = mean > a->max_q_len ? mean : a->max_q_len;
    if (likely < keys) keys = likely;
  }
  if (most <= kCUs) return keys >= (a->head_dim == 64 ? 448 : kPartsMinKeys);
  return a->head_dim == 64 && (most <= 2 * kCUs ? a->max_q_len >= 640 : most <= 3 * kCUs && a->max_q_len >= 1152);
}

// 32 positions per wave serve twice the rows with each K and V operand read, 16 make twice as many, shorter waves: these from
// three workgroups of the larger shape per CU down, where the launch is as long as its longest wave.  Measured at 64-wide heads
// (32 | 16 positions, without the sum of the fp16 weights, which costs both 4 to 8 %): 256 workgroups 21.5 | 16.2 us, 512 24.9 | 20.4 and 40.3 | 32.6, 768 30.4 | 31.4, 1024 36.6 | 35.7 and
// 92.8 | 99.3, 2048 43.9 | 48.6, 4096 170 | 200.
template <typename T, int D, int MODE, bool DV> int launch(const SmallParams& p, const lsattn_prefill_args* a, hipStream_t st) {
  if (a->num_q_heads > 65535 || a->batch > 65535) return LSATTN_ERR_INVALID_ARG;
  switch (prefill_small_route(a)) {
    case LSATTN_ROUTE_SMALL_16:
      if constexpr (D == 64)
        if (two_waves_share(a)) return launch_rows<T, 64, MODE, DV, 16, 2>(p, a, st);
      return launch_rows<T, D, MODE, DV, 16>(p, a, st);
    default: return launch_rows<T, D, MODE, DV, 32>(p, a, st);
  }
}

template <typename T, int MODE, bool DV> int launch_128(const SmallParams& p, const lsattn_prefill_args* a, hipStream_t st) {
  switch (prefill_small_route(a)) {
    case LSATTN_ROUTE_SMALL_16:
      if (two_waves_share(a)) return launch_rows<T, 128, MODE, DV, 16, 2>(p, a, st);
      return launch_rows<T, 128, MODE, DV, 16>(p, a, st);
    default: return launch_rows<T, 128, MODE, DV, 32>(p, a, st);
  }
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
// waves of 256 registers that fill 128 KB of rings and some 40 KB of code before the first product; its four-wave shape 12 us, two workgroups on a
// CU).  This one has a quarter of the code and, with 32 positions per wave, three workgroups on a CU, of which one starts or ends while the others
// compute, at the same rate per tile; it converts a bfloat16 V on the way (no launch in front that copies it).  16 positions
// per wave are for launches that do not fill the chip.  Measured over 10600 launches (1 to 40 prompts of 200 to 2048 tokens, equal or log-uniform
// over a factor of up to 20, some behind contexts; 32/32, 32/8, 64/8, 8/1, 16/16, 40/40, 24/8 and 16/8 heads; the three epilogues; calls with
// the fills of m and l; microseconds, the kernel of prefill.hip | 16 positions per wave | 32; bf16 with its copy of V):
//   3 x 560 32/32 bf16 45.6 | 28.1 | 29.0     10 x 306 32/8 35.3 | 32.6 | 26.9       19 x 566 32/8 bf16 104.4 | 118.4 | 83.8   3 x 386 at most 64/8 25.0 | 20.0 | 21.1
//   2 x 819 32/8 34.0 | 27.4 | 31.6           7 x 821 at most 32/8 bf16 52.6 | 51.4 | 39.9   6 x 999 64/8 141 | 164 | 127            16 x 853 at most 32/8 72.6 | 88.4 | 59.3
//   1 x 1113 32/8 29.0 | 26.9 | 35.9          6 x 1072 at most 64/8 81.7 | 89.5 | 63.9       3 x 1012 32/8 49.0 | 50.6 | 45.5, partial 41.1 | 44.8 | 41.2
//   2 x 1594 32/8 partial 49.0 | 62.9 | 59.1 (not taken)     19 x 1244 64/8 partial 594 | 846 | 621 (not taken)    2 x 1793 at most 32/8 partial 47.9 | 74.0 | 62.5 (not taken)
// A full step of a ring (all keys of the chunk seen by all rows, as in a ring over contiguous shards) gains less: twice the tiles for the same
// start and end.  The host cannot tell it from a batch of prompts, whose numbers are the same.  The launches taken come, in the geometric mean (95 of
// 100 stay below the figure in brackets), to so much of the time before this kernel, prompts, then full steps:
//   up to 768 rows 0.79 (0.97), 0.91 (1.16)     769 to 1024 0.85 (0.99), 1.03 (1.25)     1025 to 1280 0.88 (1.02), 1.01 (1.12)
// so the rule goes by the prompts up to 1024 rows and from there on takes what a ring's shards bear too; past 1280 that is one f16 prompt, up to
// 1472 rows, in the in-place epilogue, with 16 positions and one head per workgroup: the third workgroup per CU, 0.78 to 0.91 and full steps 0.97 to 1.08
// (1410 tokens 32/32 37.9 -> 31.3 us; 1536 rows 0.89 to 0.95 and 1.06 to 1.12, the partial 0.87 to 1.01 and 1.06 to 1.12: not taken).
//   One request folded in place in up to a workgroup per CU, where two waves share each tile: up to 2304 keys, bf16 2048, prompts, full steps and chunks
// behind a context alike 0.77 to 0.98 of the other kernel (us: 8/1 1450 tokens 28.5 | 21.5, 2040 32.3 | 27.2, bf16 1100 25.5 | 20.3, 1850 33.0 | 29.8; 200 rows behind 1024 keys 32/8
// 24.2 | 19.1, 300 behind 2000 36.0 | 31.2; past that f16 0.89 to 1.03, bf16 1.00 to 1.13).
//   16 positions: up to three workgroups per CU (two and a half of a ragged batch; with one head per workgroup, which leaves each wave fewer
// rows to mask, four and six), past 768 rows up to one, and the third, where workgroups of 128 rows would run a second round with a few of them (a ragged batch
// only with one head per workgroup: a lone long request between short ones came to up to 1.6 of the other kernel's time).  Past 1024 rows
// these only for one prompt, or for equal ones in the in-place epilogue, which lasts longer in the other kernel, and in bf16 with one
// head per workgroup.  (Four ring steps of 1120 rows 32/32 186 | 167, 32/8 184 | 169, 8/1 105 | 90.)
//   32 from there on: past 768 rows from three (ragged: three and a half) of its own per CU, past 1024 from four (five), where the other
// kernel's four-wave shape has more than one round; equal prompts past 1024 rows in more than ten per CU are for that kernel's faster loop.
//   Equal f16 requests in the in-place epilogue also fill the third workgroup of 32 positions per CU (workgroups of 128 rows split the launch into a full
// round and a thin one there): 769 to 1024 rows in 33/16 per CU and more 0.58 to 1.01 of the other kernel's time, full steps 0.73 to 0.88 (in fewer prompts to 1.05, 5 x 832 16/1 30.8 | 32.3); 1025 to 1280 in more than
// 2.6 0.75 to 0.87, full steps 0.83 to 0.96 (us: 11 x 929 8/1 62.3 | 40.4, 2 x 792 40/8 45.7 | 34.3, 9 x 1198 8/1 63.2 | 52.6, as a full step 9 x 1005 8/8 70.9 | 65.1; from 2 to 2.6 prompts up to 1.06; 1281 to 1408 up to 1.12, more than three per CU full steps to 1.22: not taken).
// The keys: a chunk behind a context waits for its longest request, and a tile of a lone workgroup takes longer here (0.95 us against 0.56 in the
// 128-row shape), so the longest request decides (whole call, 32/8 heads, the other kernel | this one with 16 positions, f16, then bf16):
//   8 x 64 rows behind 600 keys each 20.8 | 15.7, 28.0 | 18.7      4 x 100 behind 1000 each 24.9 | 21.7, 30.5 | 25.9      1 x 200 behind 1024 22.1 | 19.8, 25.2 | 24.0
//   2 x 100, one behind 1900 30.6 | 31.8, 34.5 | 39.8      8 x 64, one behind 7500 79.8 | 108.8, 88 | 169      16 x 64, one behind 15000 145 | 264, 155 | 352
// The host knows no lengths, only bounds: what total_kv_rows holds beyond the query rows may all belong to one request.
int prefill_short_blocks(const lsattn_prefill_args* a) {
  if (a->head_dim != 128 || a->kv_cuts > 1 || a->o_b_start_loc || a->max_q_len <= 0 || a->max_q_len > kPartsMaxKeys || a->batch <= 0 || a->batch > kMaxIds || a->num_kv_heads <= 0)
    return 0;
  const int64_t longest = longest_keys(a);
  if (longest > kPartsMaxKeys) return 0;
  const Tuning tn = tuning();
  if (tn.prefill_rows || tn.prefill_order || tn.prefill_pack) return 0;  // (choices among the 128-wide kernel's shapes)
  const int pack = pack_shift_of(a);
  const int64_t one = workgroups(a, pack, 1), two = workgroups(a, pack, 2);
  const bool f16 = a->dtype == LSATTN_F16, rag = ragged(a);
  // (m: of the three steps only the in-place one has it)
  if (a->batch == 1 && a->m && longest <= (f16 ? kPartsMaxKeys : kPartsMaxKeysBf16) && two_waves_share(a)) return 1;
  if (longest > kShortMaxKeys || a->max_q_len > kShortMaxKeys)
    return f16 && a->m && a->batch == 1 && a->max_q_len == longest && longest <= kLoneMaxKeys && pack == 0 && one > 2 * kCUs && one <= 3 * kCUs;
  if (a->max_q_len <= 768) return longest > 1024 ? 0 : 2 * one <= (pack ? rag ? 5 : 6 : rag ? 12 : 8) * kCUs ? 1 : 2;
  const bool past = longest > 1024;
  if (one <= kCUs) return !past || (f16 && a->batch == 1) ? 1 : 0;
  // (otherwise bf16 does not look at m: whether V is to be copied may be asked without it)
  if (one > 2 * kCUs && one <= 3 * kCUs && (past ? !rag && (f16 ? a->m != nullptr : pack == 0) : !rag || pack == 0)) return 1;
  if (f16 && a->m && a->batch > 1 && !rag && a->max_q_len == longest && two <= 3 * kCUs && (past ? 5 * two > 13 * kCUs : 16 * two >= 33 * kCUs)) return 2;
  if (past) return two > (rag ? 5 : 4) * kCUs && (rag || two <= 10 * kCUs) ? 2 : 0;
  return 2 * two >= (rag ? 7 : 6) * kCUs ? 2 : 0;
}

int prefill_small_route(const lsattn_prefill_args* a) {
  const int pack = pack_shift_of(a);
  if (a->head_dim == 128 ? prefill_short_blocks(a) == 1 : workgroups(a, pack, 2) < 3 * kCUs) return LSATTN_ROUTE_SMALL_16;
  return order_of(a, pack).turns ? LSATTN_ROUTE_SMALL_TURNS : LSATTN_ROUTE_SMALL_32;
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
