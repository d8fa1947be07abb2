// The element-wise steps around attention in the reference's extension module, for gfx950:
//   rms_norm              (longserve_cuda_kernels/src/rms_norm.cu:10-62)
//   silu_and_mul_inplace  (longserve_cuda_kernels/src/silu_and_mul.cu:12-49)
//   rotary_emb            (longserve_cuda_kernels/src/rotary_emb.cu:10-55)
// All three are HBM-bound fp16 streams: 16 bytes per lane and access, every input byte read once.
#include "common.hip.h"

namespace lsattn {
// Streams that are read and written back in place run with non-temporal accesses (NT) once they are larger than the caches:
// a line that is read, kept in the L2 as dirty and evicted later costs HBM more than one that passes through (activation
// of 16384 x 11008: 203 -> 177 us, 6.1 TB/s).  Out-of-place streams of that size (the norm, the pool rows) lose by it.
constexpr int64_t kStreamBytes = 64 << 20;
template <bool NT, typename V> __device__ __forceinline__ V stream_load(const V* p) { return NT ? __builtin_nontemporal_load(p) : *p; }
template <bool NT, typename V> __device__ __forceinline__ void stream_store(V* p, const V& v) {
  if (NT) __builtin_nontemporal_store(v, p);
  else *p = v;
}
// ---------------------------------------------------------------------------------------------------
// rms_norm: out[t, i] = half(float(x[t, i]) * float(w[i]) * inv_rms[t]),  inv_rms = rsqrt(sum x^2 / H + eps),
// the product in the reference's order (rms_norm.cu:42-45).  A row is a workgroup's (WPR = 4 waves) or, where it is
// narrow, a wave's (WPR = 1, four rows per workgroup).  Rows of up to WPR * 64 * CHUNKS pieces of 16 bytes stay in registers
// between the two passes, longer rows are read twice.  Bound by HBM for many rows and by the chain of its loads for few;
// in a wave per row there is a quarter of the loads of a row in flight beside each other (16384 rows of 4096 49.1 us against
// 43.7, 24 rows 4.9 against 2.9), but in a workgroup per row a narrow one leaves lanes idle and meets at a barrier for little: 262144 rows of
// 128 174 us against 64, of 512 199 against 96, of 1024 265 against 177 (5.9 to 6.1 TB/s from 512 on; below that the turn-over of the
// workgroups bounds it).  A wave per row up to 512 wide, and up to 1024 from 1024 rows on (fewer take 2.5 us instead of 2.4); at 1536
// the wave wins from 4096 rows on (87.8 against 78.9 at 65536) and loses 15 % below, at 2048 it loses throughout.
// ---------------------------------------------------------------------------------------------------
// The weights are asked for beside the row, not behind the barrier (24 rows of 4096 2.65 -> 2.56 us, one 2.55 -> 2.46).
// The result is stored non-temporally (NT) where it is no larger than the L2s are together: it does not wait there as dirty lines for the
// next kernel's reads (1000 rows of 4096 5.3 -> 4.7 us, 4000 13.9 -> 11.3; with a kernel that reads the result behind it 12.0 -> 11.1 and 24.7 -> 23.8,
// with a product by 4096 x 1024 31.6 -> 31.1 and 58.6 -> 58.1).  Past that the norm itself may gain, but whoever reads the result loses more: 8000 rows and
// the product 96 -> 98, 16384 rows and it 160 -> 165, and an addition 80 -> 86.
constexpr int64_t kRmsNarrow = 512, kRmsNarrowRows = 1024, kRmsStreamedBytes = 32 << 20;
constexpr int64_t kMaxGroups = (1 << 24) - 1;  // workgroups of 256 threads in one launch (fewer than 2^32 threads)

__device__ __forceinline__ float wave_sum(float v) {
  v = sum_row16(v);
  v += __shfl_xor(v, 16);
  v += __shfl_xor(v, 32);
  return v;
}

template <int WPR, int CHUNKS, bool NT>
__global__ __launch_bounds__(256) void rms_norm_kernel(uint16_t* __restrict__ out, const uint16_t* __restrict__ in,
                                                       const uint16_t* __restrict__ weight, int64_t rows, int64_t hidden, float eps) {
  constexpr int LANES = 64 * WPR;  // of a row
  const int64_t t = (int64_t)blockIdx.x * (4 / WPR) + threadIdx.x / LANES;
  if (WPR == 1 && t >= rows) return;  // (no barrier below then)
  const int lane = threadIdx.x % LANES;
  const int pieces = (int)(hidden / 8);  // 16-byte pieces in a row
  const u32x4* row = (const u32x4*)(in + t * hidden);
  const u32x4* wrow = (const u32x4*)weight;
  u32x4* orow = (u32x4*)(out + t * hidden);
  const bool cached = pieces <= LANES * CHUNKS;
  u32x4 keep[CHUNKS], weights[CHUNKS];
  float ss = 0.f;
  auto add_squares = [&](const u32x4& x) {
    float f[8];
    unpack8<F16>(x, f);
#pragma unroll
    for (int e = 0; e < 8; e++) ss = __builtin_fmaf(f[e], f[e], ss);
  };
  if (cached) {
#pragma unroll
    for (int c = 0; c < CHUNKS; c++) {
      const int i = lane + LANES * c;
      keep[c] = i < pieces ? row[i] : u32x4{0, 0, 0, 0};
      weights[c] = i < pieces ? wrow[i] : u32x4{0, 0, 0, 0};
    }
#pragma unroll
    for (int c = 0; c < CHUNKS; c++) add_squares(keep[c]);
#pragma unroll
    for (int c = 0; c < CHUNKS; c++) asm volatile("" : "+v"(weights[c]));  // (or the compiler moves their loads behind the barrier)
  } else {
    for (int i = lane; i < pieces; i += LANES) add_squares(row[i]);
  }
  ss = wave_sum(ss);
  if constexpr (WPR > 1) {
    __shared__ float part[4];
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = ss;
    __syncthreads();
    ss = (part[0] + part[1]) + (part[2] + part[3]);
  }
  const float inv_rms = __builtin_amdgcn_rsqf(ss / (float)hidden + eps);
  auto scale_piece = [&](const u32x4& x, const u32x4& w) {
    float a[8], b[8];
    unpack8<F16>(x, a);
    unpack8<F16>(w, b);
    u32x4 r;
#pragma unroll
    for (int e = 0; e < 4; e++) r[e] = pack2<F16>(a[2 * e] * b[2 * e] * inv_rms, a[2 * e + 1] * b[2 * e + 1] * inv_rms);
    return r;
  };
  if (cached) {
#pragma unroll
    for (int c = 0; c < CHUNKS; c++) {
      const int i = lane + LANES * c;
      if (i < pieces) stream_store<NT>(orow + i, scale_piece(keep[c], weights[c]));
    }
  } else {
    for (int i = lane; i < pieces; i += LANES) stream_store<NT>(orow + i, scale_piece(row[i], wrow[i]));
  }
}

// WPR waves per row, in slices of as many rows as a launch has workgroups for.
template <int WPR, int CHUNKS>
static int launch_rms_norm(uint16_t* out, const uint16_t* in, const uint16_t* weight, int64_t rows, int64_t hidden, float eps, hipStream_t st) {
  constexpr int64_t PER_WG = 4 / WPR;
  const bool nt = rows <= kRmsStreamedBytes / 2 / hidden;
  for (int64_t t0 = 0; t0 < rows; t0 += kMaxGroups * PER_WG) {
    const int64_t n = rows - t0 < kMaxGroups * PER_WG ? rows - t0 : kMaxGroups * PER_WG;
    const dim3 grid((unsigned)((n + PER_WG - 1) / PER_WG));
    if (nt) LSATTN_LAUNCH_KERNEL((rms_norm_kernel<WPR, CHUNKS, true>), grid, dim3(256), 0, st, out + t0 * hidden, in + t0 * hidden, weight, n, hidden, eps);
    else LSATTN_LAUNCH_KERNEL((rms_norm_kernel<WPR, CHUNKS, false>), grid, dim3(256), 0, st, out + t0 * hidden, in + t0 * hidden, weight, n, hidden, eps);
    const int rc = check_launch();
    if (rc != LSATTN_OK) return rc;
  }
  return LSATTN_OK;
}

// ---------------------------------------------------------------------------------------------------
// silu_and_mul_inplace: io[t, i] = half(silu(io[t, i])) * io[t, I + i] for i < I, the second half of the row untouched;
// silu in fp32, rounded to half, then a half multiply (silu_and_mul.cu:14-17, :30-33).
// ---------------------------------------------------------------------------------------------------
template <bool NT>
__global__ __launch_bounds__(256) void silu_and_mul_kernel(uint16_t* __restrict__ io, uint32_t units, int64_t inter, FastDiv by_row) {
  const uint32_t gid = blockIdx.x * 256 + threadIdx.x;
  if (gid >= units) return;
  const uint32_t t = div_by(gid, by_row), i = gid - t * (uint32_t)(inter / 8);
  // (whole rows of eight halves: picking 32-bit words out of an integer vector and bit-casting them to half
  // pairs made this compiler read word 0 every time)
  f16x8* gate = (f16x8*)(io + (int64_t)t * 2 * inter) + i;
  const f16x8 g = stream_load<NT>(gate);
  const f16x8 u = stream_load<NT>((const f16x8*)(io + (int64_t)t * 2 * inter + inter) + i);
  f16x8 r;
#pragma unroll
  for (int e = 0; e < 8; e++) {
    const float x = (float)g[e];
    const _Float16 sl = (_Float16)(x / (1.f + __builtin_amdgcn_exp2f(-x * kLog2e)));
    r[e] = sl * u[e];  // half multiply, round to nearest even
  }
  stream_store<NT>(gate, r);
}

// ---------------------------------------------------------------------------------------------------
// rotary_emb, in place on x[t, h, :] (last dimension contiguous), in the reference's half arithmetic (rotary_emb.cu:30-33):
//   new_x1 = fma(x1, cos, -(x2 * sin)),  new_x2 = fma(x1, sin, x2 * cos)   with x1 = x[..., :D/2], x2 = x[..., D/2:],
// every product and fma rounded to half once.  A lane owns 8 elements of x1 and the matching 8 of x2.
// ---------------------------------------------------------------------------------------------------
// The lane's 16 bytes of x1 and of x2 at p1 and p2, rotated in place; the rotated pieces in n1 and n2.
template <bool NT>
__device__ __forceinline__ void rotate_piece(f16x8* p1, f16x8* p2, const f16x8& co, const f16x8& si, f16x8& n1, f16x8& n2) {
  const f16x8 x1 = stream_load<NT>(p1), x2 = stream_load<NT>(p2);
  const f16x8 t1 = x2 * si, t2 = x2 * co;  // rounded to half (this file is compiled without contraction)
#pragma unroll
  for (int e = 0; e < 8; e++) {
    n1[e] = __builtin_fmaf16(x1[e], co[e], -t1[e]);
    n2[e] = __builtin_fmaf16(x1[e], si[e], t2[e]);
  }
  stream_store<NT>(p1, n1);
  stream_store<NT>(p2, n2);
}

// ---------------------------------------------------------------------------------------------------
// The write-back of a step's new tokens in one launch: rotary embedding of q and of the K heads in place (the arithmetic
// of rotate_piece), every token's rotated K heads and its V heads copied to the token's slot of the KV pool, and the
// slots entered in the request table.  A unit is 32 bytes of one (token, head): the two 16-byte halves a rotary lane
// owns, or two consecutive 16-byte pieces of a V head.  Blocks past the data units do the registration, one table entry
// per lane.
// ---------------------------------------------------------------------------------------------------
struct RotaryWriteParams {
  uint16_t* q;
  int64_t q_st, q_sh;
  uint16_t* kv;
  int64_t kv_st, kv_sh;
  const uint16_t* cos_t;
  const uint16_t* sin_t;
  uint16_t* pool;
  int64_t pool_stride;  // elements per slot
  const void* dest;     // int32 or int64 (dest_i64), of all tokens; this launch begins with token token0
  int64_t token0;
  int32_t* req_to_tokens;
  int64_t max_seq_len;
  const int32_t* b_req_idx;
  const int32_t* b_start_loc;
  const int32_t* b_seq_len;
  int64_t batch;
  uint32_t hq, hkv, head_dim, heads;  // heads: those of a token that are units of this launch (no V heads without a pool)
  uint32_t units, data_blocks, reg_blocks_per_req;
  FastDiv by_pieces, by_heads;
  int32_t reg_mode;  // 0 none, 1 every token of every request (prefill), 2 the last token of every request (decode)
  int32_t dest_i64;
};

template <bool NT> __global__ __launch_bounds__(256) void rotary_kv_write_kernel(RotaryWriteParams p) {
  auto slot = [&](int64_t i) -> int64_t { return p.dest_i64 ? ((const int64_t*)p.dest)[i] : (int64_t)((const int32_t*)p.dest)[i]; };
  if (blockIdx.x >= p.data_blocks) {
    const uint32_t rb = blockIdx.x - p.data_blocks;
    if (p.reg_mode == 1) {
      const int64_t b = rb / p.reg_blocks_per_req;
      const int64_t j = (int64_t)(rb % p.reg_blocks_per_req) * 256 + threadIdx.x;
      if (j >= p.b_seq_len[b] || j >= p.max_seq_len) return;
      p.req_to_tokens[(int64_t)p.b_req_idx[b] * p.max_seq_len + j] = (int32_t)slot((int64_t)p.b_start_loc[b] + j);
    } else {
      const int64_t i = (int64_t)rb * 256 + threadIdx.x;
      if (i >= p.batch) return;
      const int64_t pos = (int64_t)p.b_seq_len[i] - 1;
      if (pos < 0 || pos >= p.max_seq_len) return;
      p.req_to_tokens[(int64_t)p.b_req_idx[i] * p.max_seq_len + pos] = (int32_t)slot(i);
    }
    return;
  }
  const uint32_t gid = blockIdx.x * 256 + threadIdx.x;
  if (gid >= p.units) return;
  const uint32_t th = div_by(gid, p.by_pieces), c = gid - th * (p.head_dim / 16);  // unit of its head
  const int64_t t = div_by(th, p.by_heads);
  const uint32_t h = th - (uint32_t)t * p.heads;
  if (h >= p.hq + p.hkv) {
    // V head: 32 bytes to the pool
    const uint32_t hv = h - p.hq;  // head index inside the token's K/V row
    const f16x8* src = (const f16x8*)(p.kv + t * p.kv_st + hv * p.kv_sh) + 2 * c;
    f16x8* dst = (f16x8*)(p.pool + slot(p.token0 + t) * p.pool_stride + (int64_t)hv * p.head_dim) + 2 * c;
    const f16x8 a = src[0], b = src[1];
    dst[0] = a;
    dst[1] = b;
    return;
  }
  const bool is_k = h >= p.hq;
  uint16_t* base = is_k ? p.kv + t * p.kv_st + (h - p.hq) * p.kv_sh : p.q + t * p.q_st + h * p.q_sh;
  const f16x8 co = *((const f16x8*)(p.cos_t + t * (p.head_dim / 2)) + c);
  const f16x8 si = *((const f16x8*)(p.sin_t + t * (p.head_dim / 2)) + c);
  f16x8 n1, n2;
  rotate_piece<NT>((f16x8*)base + c, (f16x8*)(base + p.head_dim / 2) + c, co, si, n1, n2);
  if (is_k && p.pool) {
    uint16_t* prow = p.pool + slot(p.token0 + t) * p.pool_stride + (int64_t)(h - p.hq) * p.head_dim;
    *((f16x8*)prow + c) = n1;
    *((f16x8*)(prow + p.head_dim / 2) + c) = n2;
  }
}

// ---------------------------------------------------------------------------------------------------
// bf16 -> fp16 row copy, rounded toward zero (exact inside fp16's normal range, +-65504 beyond it): prepares a bf16 V
// for the prefill kernel, whose P V product runs in fp16.  One 16-byte piece per lane.
// ---------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void bf16_to_f16_rows_kernel(const uint16_t* __restrict__ src, int64_t src_stride,
                                                               uint16_t* __restrict__ dst, int64_t dst_stride, uint32_t pieces,
                                                               uint32_t pieces_per_row, FastDiv by_row) {
  const uint32_t gid = blockIdx.x * 256 + threadIdx.x;
  if (gid >= pieces) return;
  const int64_t r = div_by(gid, by_row);
  const uint32_t c = gid - (uint32_t)r * pieces_per_row;
  const u32x4 w = *((const u32x4*)(src + r * src_stride) + c);
  u32x4 o;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    float lo, hi;
    unpack2<BF16>(w[i], lo, hi);
    o[i] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(lo, hi));
  }
  *((u32x4*)(dst + r * dst_stride) + c) = o;
}

}  // namespace lsattn

using namespace lsattn;

extern "C" int lsattn_bf16_to_f16_rows(const void* src, int64_t src_stride, void* dst, int64_t dst_stride, int64_t n_rows,
                                       int64_t row_elems, void* stream) {
  if (!src || !dst || n_rows < 0 || row_elems <= 0) return LSATTN_ERR_INVALID_ARG;
  if (row_elems % 8 || src_stride % 8 || dst_stride % 8 || src_stride < row_elems || dst_stride < row_elems ||
      (((uintptr_t)src | (uintptr_t)dst) & 15))
    return LSATTN_ERR_INVALID_ARG;
  if (n_rows == 0) return LSATTN_OK;
  const int64_t per_row = row_elems / 8;
  if (per_row > kMaxUnits) return LSATTN_ERR_INVALID_ARG;
  for (int64_t r0 = 0, slice = kMaxUnits / per_row; r0 < n_rows; r0 += slice) {
    const int64_t pieces = (n_rows - r0 < slice ? n_rows - r0 : slice) * per_row;
    LSATTN_LAUNCH_KERNEL(bf16_to_f16_rows_kernel, dim3((unsigned)((pieces + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       (const uint16_t*)src + r0 * src_stride, src_stride, (uint16_t*)dst + r0 * dst_stride, dst_stride,
                       (uint32_t)pieces, (uint32_t)per_row, fast_div((uint32_t)per_row));
  }
  return check_launch();
}

extern "C" int lsattn_rms_norm(void* out, const void* in, const void* weight, int64_t num_tokens, int64_t hidden_size,
                               float eps, void* stream) {
  if (!out || !in || !weight || num_tokens < 0 || hidden_size <= 0) return LSATTN_ERR_INVALID_ARG;
  if (hidden_size % 8 || (((uintptr_t)out | (uintptr_t)in | (uintptr_t)weight) & 15)) return LSATTN_ERR_INVALID_ARG;
  if (num_tokens == 0) return LSATTN_OK;
  if (hidden_size > 0x7fffffff) return LSATTN_ERR_INVALID_ARG;
  uint16_t* o = (uint16_t*)out;
  const uint16_t *x = (const uint16_t*)in, *w = (const uint16_t*)weight;
  hipStream_t st = (hipStream_t)stream;
  if (hidden_size <= kRmsNarrow || (hidden_size <= 2 * kRmsNarrow && num_tokens >= kRmsNarrowRows))
    return launch_rms_norm<1, 2>(o, x, w, num_tokens, hidden_size, eps, st);
  return launch_rms_norm<4, 4>(o, x, w, num_tokens, hidden_size, eps, st);
}

extern "C" int lsattn_silu_and_mul_inplace(void* io, int64_t num_tokens, int64_t ffn_inter_dim, void* stream) {
  if (!io || num_tokens < 0 || ffn_inter_dim <= 0) return LSATTN_ERR_INVALID_ARG;
  if (ffn_inter_dim % 8 || ((uintptr_t)io & 15)) return LSATTN_ERR_INVALID_ARG;
  if (num_tokens == 0) return LSATTN_OK;
  const int64_t per_row = ffn_inter_dim / 8;
  if (per_row > kMaxUnits) return LSATTN_ERR_INVALID_ARG;
  const bool nt = num_tokens * ffn_inter_dim * 4 >= kStreamBytes;
  for (int64_t t0 = 0, slice = kMaxUnits / per_row; t0 < num_tokens; t0 += slice) {
    const int64_t units = (num_tokens - t0 < slice ? num_tokens - t0 : slice) * per_row;
    uint16_t* rows = (uint16_t*)io + t0 * 2 * ffn_inter_dim;
    const dim3 grid((unsigned)((units + 255) / 256));
    if (nt) LSATTN_LAUNCH_KERNEL(silu_and_mul_kernel<true>, grid, dim3(256), 0, (hipStream_t)stream, rows, (uint32_t)units, ffn_inter_dim, fast_div((uint32_t)per_row));
    else LSATTN_LAUNCH_KERNEL(silu_and_mul_kernel<false>, grid, dim3(256), 0, (hipStream_t)stream, rows, (uint32_t)units, ffn_inter_dim, fast_div((uint32_t)per_row));
  }
  return check_launch();
}

namespace lsattn {
// Launches of rotary_kv_write_kernel over whole tokens, as many as have at most kMaxUnits units; the table is entered with the last one.
static int launch_rotary(RotaryWriteParams p, int64_t num_tokens, int64_t max_len_in_batch, hipStream_t st) {
  const int64_t per_token = (int64_t)p.heads * (p.head_dim / 16);
  if (per_token > kMaxUnits) return LSATTN_ERR_INVALID_ARG;
  int64_t reg_blocks = 0;
  if (p.reg_mode == 1) {
    p.reg_blocks_per_req = (uint32_t)((max_len_in_batch + 255) / 256);
    reg_blocks = p.reg_blocks_per_req * p.batch;
  } else if (p.reg_mode == 2) {
    reg_blocks = (p.batch + 255) / 256;
  }
  if (reg_blocks > 0x40000000) return LSATTN_ERR_INVALID_ARG;
  p.by_pieces = fast_div(p.head_dim / 16);
  p.by_heads = fast_div(p.heads);
  const bool nt = num_tokens * (int64_t)(p.hq + p.hkv) * p.head_dim * 2 >= kStreamBytes;
  if (num_tokens == 0 && reg_blocks == 0) return LSATTN_OK;  // (no launch whose outcome there is to report)
  const int64_t slice = kMaxUnits / per_token;
  for (int64_t t0 = 0;; t0 += slice) {
    const bool last = num_tokens - t0 <= slice;
    RotaryWriteParams s = p;
    s.units = (uint32_t)((last ? num_tokens - t0 : slice) * per_token);
    s.data_blocks = (s.units + 255) / 256;
    s.q += t0 * p.q_st;
    s.kv += t0 * p.kv_st;
    s.cos_t += t0 * (p.head_dim / 2);
    s.sin_t += t0 * (p.head_dim / 2);
    if (!last) s.reg_mode = 0;
    s.token0 = t0;
    const int64_t blocks = s.data_blocks + (last ? reg_blocks : 0);
    if (blocks > 0x7fffffff) return LSATTN_ERR_INVALID_ARG;
    if (blocks > 0) {
      if (nt) LSATTN_LAUNCH_KERNEL(rotary_kv_write_kernel<true>, dim3((unsigned)blocks), dim3(256), 0, st, s);
      else LSATTN_LAUNCH_KERNEL(rotary_kv_write_kernel<false>, dim3((unsigned)blocks), dim3(256), 0, st, s);
    }
    if (last) break;
  }
  return check_launch();
}
}  // namespace lsattn

extern "C" int lsattn_rotary_emb(void* x, const void* cos, const void* sin, int64_t x_stride_t, int64_t x_stride_h,
                                 int64_t num_tokens, int64_t num_heads, int64_t head_dim, void* stream) {
  if (!x || !cos || !sin || num_tokens < 0 || num_heads <= 0 || head_dim <= 0) return LSATTN_ERR_INVALID_ARG;
  if (head_dim % 16 || x_stride_t % 8 || x_stride_h % 8 || (((uintptr_t)x | (uintptr_t)cos | (uintptr_t)sin) & 15))
    return LSATTN_ERR_INVALID_ARG;
  if (num_tokens == 0) return LSATTN_OK;
  if (num_heads > kMaxUnits || head_dim > kMaxUnits) return LSATTN_ERR_INVALID_ARG;
  RotaryWriteParams p = {};
  p.q = p.kv = (uint16_t*)x;
  p.q_st = x_stride_t;
  p.q_sh = x_stride_h;
  p.cos_t = (const uint16_t*)cos;
  p.sin_t = (const uint16_t*)sin;
  p.hq = p.heads = (uint32_t)num_heads;
  p.head_dim = (uint32_t)head_dim;
  return launch_rotary(p, num_tokens, 0, (hipStream_t)stream);
}

extern "C" int lsattn_rotary_kv_write(const lsattn_rotary_kv_write_args* a, void* stream) {
  if (!a || !a->q || !a->kv || !a->cos || !a->sin || a->num_tokens < 0 || a->num_q_heads <= 0 || a->num_kv_heads <= 0 ||
      a->head_dim <= 0 || a->batch < 0)
    return LSATTN_ERR_INVALID_ARG;
  if (a->head_dim % 16 || a->q_stride_t % 8 || a->q_stride_h % 8 || a->kv_stride_t % 8 || a->kv_stride_h % 8 ||
      (((uintptr_t)a->q | (uintptr_t)a->kv | (uintptr_t)a->cos | (uintptr_t)a->sin | (uintptr_t)a->pool) & 15))
    return LSATTN_ERR_INVALID_ARG;
  if (a->pool && (!a->dest_index || a->pool_slot_stride % 8 || a->pool_slot_stride < 2 * a->num_kv_heads * a->head_dim))
    return LSATTN_ERR_INVALID_ARG;
  if (a->register_mode < 0 || a->register_mode > 2) return LSATTN_ERR_INVALID_ARG;
  if (a->register_mode != 0 &&
      (!a->req_to_tokens || !a->dest_index || !a->b_req_idx || !a->b_seq_len || a->max_seq_len <= 0 ||
       (a->register_mode == 1 && (!a->b_start_loc || a->max_len_in_batch < 0 || a->max_len_in_batch > a->max_seq_len))))
    return LSATTN_ERR_INVALID_ARG;
  if (a->dest_index_is_i64 != 0 && a->dest_index_is_i64 != 1) return LSATTN_ERR_INVALID_ARG;
  const int64_t heads = a->num_q_heads + (a->pool ? 2 : 1) * a->num_kv_heads;
  if (heads > kMaxUnits || a->head_dim > kMaxUnits) return LSATTN_ERR_INVALID_ARG;
  RotaryWriteParams p = {};
  p.q = (uint16_t*)a->q;
  p.q_st = a->q_stride_t;
  p.q_sh = a->q_stride_h;
  p.hq = (uint32_t)a->num_q_heads;
  p.kv = (uint16_t*)a->kv;
  p.kv_st = a->kv_stride_t;
  p.kv_sh = a->kv_stride_h;
  p.hkv = (uint32_t)a->num_kv_heads;
  p.heads = (uint32_t)heads;
  p.cos_t = (const uint16_t*)a->cos;
  p.sin_t = (const uint16_t*)a->sin;
  p.head_dim = (uint32_t)a->head_dim;
  p.pool = (uint16_t*)a->pool;
  p.pool_stride = a->pool_slot_stride;
  p.dest = a->dest_index;
  p.dest_i64 = a->dest_index_is_i64;
  p.req_to_tokens = a->req_to_tokens;
  p.max_seq_len = a->max_seq_len;
  p.b_req_idx = a->b_req_idx;
  p.b_start_loc = a->b_start_loc;
  p.b_seq_len = a->b_seq_len;
  p.batch = a->batch;
  p.reg_mode = a->register_mode;
  return launch_rotary(p, a->num_tokens, a->max_len_in_batch, (hipStream_t)stream);
}
