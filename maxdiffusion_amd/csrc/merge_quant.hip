// HBM-bound helpers around the attention kernel: LSE-space chunk merge, f32->bf16 finalize,
// per-tensor absmax e4m3 quantisation.
#include "mdattn_common.h"
#include "mdattn_host.h"

namespace mdattn {

struct MergeArgs {
  float* o_run;
  float* lse_run;
  const void* o_cur;
  const float* lse_cur;
  int H, S;
  int64_t rows;  // B*H*S
  int h_fast;    // rows are walked with the head index fastest (what [B,S,H,D] storage wants) instead of the token index
  int64_t r_sb, r_ss, r_sh, c_sb, c_ss, c_sh;
};

// LPR = D/8 lanes per (b,h,s) row, all in one wave: every lane reads the row's two lse values
// in the same instruction, before lane 0 of the row overwrites lse_run.
template <int LPR, bool CUR_F32>
__global__ __launch_bounds__(256) void merge_kernel(MergeArgs a) {
  const int tid = threadIdx.x, lane = tid % LPR;
  const int64_t row = (int64_t)blockIdx.x * (256 / LPR) + tid / LPR;
  if (row >= a.rows) return;
  int s, h;
  int64_t b;
  if (a.h_fast) {  // consecutive rows of a workgroup are consecutive in memory
    h = (int)(row % a.H);
    const int64_t bs = row / a.H;
    s = (int)(bs % a.S);
    b = bs / a.S;
  } else {
    s = (int)(row % a.S);
    const int64_t bh = row / a.S;
    h = (int)(bh % a.H);
    b = bh / a.H;
  }
  const int64_t lidx = (b * a.H + h) * a.S + s;
  const float l1 = a.lse_run[lidx], l2 = a.lse_cur[lidx];
  float4* pr = reinterpret_cast<float4*>(a.o_run + b * a.r_sb + s * a.r_ss + h * a.r_sh) + 2 * lane;
  float4 r0 = pr[0], r1 = pr[1];
  float cur[8];
  if (CUR_F32) {
    const float4* pc = reinterpret_cast<const float4*>((const float*)a.o_cur + b * a.c_sb + s * a.c_ss + h * a.c_sh) + 2 * lane;
    float4 c0 = ld_nt(pc), c1 = ld_nt(pc + 1);
    cur[0] = c0.x; cur[1] = c0.y; cur[2] = c0.z; cur[3] = c0.w; cur[4] = c1.x; cur[5] = c1.y; cur[6] = c1.z; cur[7] = c1.w;
  } else {
    const uint4* pc = reinterpret_cast<const uint4*>((const unsigned short*)a.o_cur + b * a.c_sb + s * a.c_ss + h * a.c_sh) + lane;
    unpack8(ld_nt(pc), cur);
  }
  const float L = fmaxf(l1, l2);
  float w1 = 0.f, w2 = 0.f;
  if (L > -INFINITY) { w1 = expf(l1 - L); w2 = expf(l2 - L); }
  const float den = w1 + w2;
  const float inv = den > 0.f ? 1.0f / den : 0.f;
  w1 *= inv; w2 *= inv;
  r0.x = w1 * r0.x + w2 * cur[0]; r0.y = w1 * r0.y + w2 * cur[1]; r0.z = w1 * r0.z + w2 * cur[2]; r0.w = w1 * r0.w + w2 * cur[3];
  r1.x = w1 * r1.x + w2 * cur[4]; r1.y = w1 * r1.y + w2 * cur[5]; r1.z = w1 * r1.z + w2 * cur[6]; r1.w = w1 * r1.w + w2 * cur[7];
  pr[0] = r0; pr[1] = r1;
  if (lane == 0) a.lse_run[lidx] = den > 0.f ? L + logf(den) : L;
}

__global__ __launch_bounds__(256) void finalize_kernel(const float4* __restrict__ in, uint4* __restrict__ out, int64_t n8) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n8; i += (int64_t)gridDim.x * 256) {
    const float4 a = ld_nt(in + 2 * i), b = ld_nt(in + 2 * i + 1);
    const float f[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    st_nt(out + i, pack8(f));
  }
}

// Dense copies of one or two buffers (blockIdx.y), 16 bytes per lane.  A launch's own time rules it at the sizes of rotary tables and
// weights: 2 x 2.4 MB 5.4 us from memory and 2.8 from the caches, 2 x 8 KB 4.8 and 1.7, the runtime's copy of one of the two buffers 5.2
// and 2.3, 4.8 and 1.4.  Two planes in one launch save the second, on the stream and on the host.
__global__ __launch_bounds__(256) void copy_kernel(const uint4* src0, uint4* dst0, const uint4* src1, uint4* dst1, int64_t n16) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n16) (blockIdx.y ? dst1 : dst0)[i] = (blockIdx.y ? src1 : src0)[i];
}

__global__ void zero2_kernel(float* p) { if (threadIdx.x < 2) p[threadIdx.x] = 0.f; }

// |x| of a non-negative-masked bf16 orders like its bit pattern, so the absmax is an integer max.  Eight independent
// 16-byte loads in flight per lane and trip.  Returns the workgroup's maximum to its first lane.
__device__ __forceinline__ unsigned absmax_bits(const uint4* __restrict__ x, int64_t n8) {
  __shared__ unsigned wmax[4];
  unsigned m = 0;
  auto fold = [&](const uint4& u) {
    const unsigned w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const unsigned lo = (w[j] << 16) & 0x7FFF0000u, hi = w[j] & 0x7FFF0000u;
      m = max(m, max(lo, hi));
    }
  };
  const int64_t stride = (int64_t)gridDim.x * 256;
  int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  for (; i + 7 * stride < n8; i += 8 * stride) {
    uint4 u[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) u[j] = ld_nt(x + i + j * stride);
#pragma unroll
    for (int j = 0; j < 8; ++j) fold(u[j]);
  }
  for (; i < n8; i += stride) fold(x[i]);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = max(m, (unsigned)__shfl_xor((int)m, o));
  if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = m;
  __syncthreads();
  return max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3]));
}

// One atomic per workgroup (thousands of same-address atomics from every wave would cost as much as the read itself).
__global__ __launch_bounds__(256) void absmax_kernel(const uint4* __restrict__ x, int64_t n8, unsigned* amax_bits) {
  const unsigned m = absmax_bits(x, n8);
  if (threadIdx.x == 0 && m) atomicMax(amax_bits, m);
}

// x8 = e4m3(x * premul / s) with s = absmax(x * premul) / 448, or the next power of two above it (pow2): a
// power-of-two scale costs e4m3, a floating-point format, no precision, only up to one binade of its range.
__device__ __forceinline__ float quant_scale(float absmax, float premul, int pow2) {
  float amax = absmax * premul;
  amax = amax > 1e-12f ? amax : 1e-12f;
  float s = amax * (1.0f / 448.0f);
  if (pow2) {
    const unsigned b = __float_as_uint(s);
    s = __uint_as_float(((b & 0x007FFFFFu) ? b + 0x00800000u : b) & 0x7F800000u);
  }
  return s;
}
__device__ __forceinline__ uint4 quant16(const uint4& a, const uint4& b, float r) {
  float f[16];
  unpack8(a, f);
  unpack8(b, f + 8);
  unsigned o[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    float v[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) v[t] = fminf(fmaxf(f[4 * j + t] * r, -448.f), 448.f);
    int pk = 0;
    pk = __builtin_amdgcn_cvt_pk_fp8_f32(v[0], v[1], pk, false);
    pk = __builtin_amdgcn_cvt_pk_fp8_f32(v[2], v[3], pk, true);
    o[j] = (unsigned)pk;
  }
  return make_uint4(o[0], o[1], o[2], o[3]);
}
__global__ __launch_bounds__(256) void quant_kernel(const uint4* __restrict__ x, uint4* __restrict__ y, int64_t n16, float* scale,
                                                    float premul, int pow2) {
  const float s = quant_scale(scale[1], premul, pow2);
  const float r = premul / s;
  if (blockIdx.x == 0 && threadIdx.x == 0) scale[0] = s;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n16; i += (int64_t)gridDim.x * 256)
    y[i] = quant16(x[2 * i], x[2 * i + 1], r);
}

// The same for q, k and v of one attention call in two launches instead of nine.  Every workgroup of the first leaves its
// maximum in a slot of its own (same-address atomics take 14 ns each: 28 us for a tensor's 2,048 workgroups, whatever its
// size, and the slots need no clearing launch); every workgroup of the second folds its tensor's slots, one 16-byte load per
// lane, before it quantises.  The second walks tensors and rows backwards, over what the first read last.  4 x 1,080 tokens x 5
// heads: 78 us of kernels in nine launches -> 11; 11,232 x 4: 104 -> 19; 32,760 x 40 (bound by its 2.5 GB): 462 -> 452.
struct Quant3Args {
  const uint4* x[3];
  uint4* y[3];
  int64_t n16[3];
  unsigned* part;    // [3][kQuantSlots]
  float* scale;      // [3][2]
  float premul[3];
  int pow2[3];
  int slots;         // workgroups per tensor in the first kernel
};
constexpr int kQuantSlots = 1024;
__global__ __launch_bounds__(256) void absmax3_kernel(Quant3Args a) {
  const int t = blockIdx.y;
  const unsigned m = absmax_bits(a.x[t], 2 * a.n16[t]);
  if (threadIdx.x == 0) a.part[t * kQuantSlots + blockIdx.x] = m;
}
__global__ __launch_bounds__(256) void quant3_kernel(Quant3Args a) {
  __shared__ unsigned wmax[4];
  const int t = 2 - blockIdx.y, tid = threadIdx.x;
  const uint4 u = reinterpret_cast<const uint4*>(a.part + t * kQuantSlots)[tid];
  const int have = a.slots - 4 * tid;
  unsigned m = max(max(have > 0 ? u.x : 0u, have > 1 ? u.y : 0u), max(have > 2 ? u.z : 0u, have > 3 ? u.w : 0u));
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = max(m, (unsigned)__shfl_xor((int)m, o));
  if ((tid & 63) == 0) wmax[tid >> 6] = m;
  __syncthreads();
  const float absmax = __uint_as_float(max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3])));
  const float s = quant_scale(absmax, a.premul[t], a.pow2[t]);
  const float r = a.premul[t] / s;
  if (blockIdx.x == 0 && tid == 0) {
    a.scale[2 * t] = s;
    a.scale[2 * t + 1] = absmax;
  }
  const uint4* x = a.x[t];
  for (int64_t i = a.n16[t] - 1 - ((int64_t)blockIdx.x * 256 + tid); i >= 0; i -= (int64_t)gridDim.x * 256)
    a.y[t][i] = quant16(x[2 * i], x[2 * i + 1], r);
}

}  // namespace mdattn

using namespace mdattn;

extern "C" int mdattn_merge(void* stream, float* o_run, float* lse_run, const void* o_cur, const float* lse_cur,
                            int cur_is_f32, int B, int H, int S, int D,
                            const mdattn_strides* run_strides, const mdattn_strides* cur_strides) {
  if (!o_run || !lse_run || !o_cur || !lse_cur || B <= 0 || H <= 0 || S <= 0 || D <= 0) return MDATTN_E_BADARG;
  if (!run_strides || !cur_strides) return MDATTN_E_BADARG;
  if (D != 64 && D != 128 && D != 256) return MDATTN_E_UNSUPPORTED;
  if (!aligned16(o_run) || !aligned16(o_cur) || (reinterpret_cast<uintptr_t>(lse_run) & 3u) || (reinterpret_cast<uintptr_t>(lse_cur) & 3u))
    return MDATTN_E_ALIGN;
  if (!strides_ok(run_strides, 8) || !strides_ok(cur_strides, 8)) return MDATTN_E_ALIGN;
  MergeArgs a;
  a.o_run = o_run; a.lse_run = lse_run; a.o_cur = o_cur; a.lse_cur = lse_cur;
  a.H = H; a.S = S; a.rows = (int64_t)B * H * S;
  a.h_fast = run_strides->head < run_strides->seq;
  a.r_sb = run_strides->batch; a.r_ss = run_strides->seq; a.r_sh = run_strides->head;
  a.c_sb = cur_strides->batch; a.c_ss = cur_strides->seq; a.c_sh = cur_strides->head;
  const int lpr = D / 8;
  const int64_t nblocks = (a.rows + (256 / lpr) - 1) / (256 / lpr);
  if (nblocks > 0x7FFFFFFF) return MDATTN_E_UNSUPPORTED;
  dim3 grid((unsigned)nblocks), block(256);
  hipStream_t st = (hipStream_t)stream;
#define MDATTN_MERGE_CASE(L)                                                          \
  if (lpr == L) {                                                                     \
    if (cur_is_f32) MDATTN_LAUNCH((merge_kernel<L, true>), grid, block, 0, st, a); \
    else MDATTN_LAUNCH((merge_kernel<L, false>), grid, block, 0, st, a);           \
  }
  MDATTN_MERGE_CASE(8) MDATTN_MERGE_CASE(16) MDATTN_MERGE_CASE(32)
#undef MDATTN_MERGE_CASE
  return launch_status();
}

extern "C" int mdattn_finalize(void* stream, const float* o_run, void* out_bf16, int64_t n) {
  if (!o_run || !out_bf16 || n <= 0) return MDATTN_E_BADARG;
  if (n % 8) return MDATTN_E_UNSUPPORTED;
  if (!aligned16(o_run) || !aligned16(out_bf16)) return MDATTN_E_ALIGN;
  const int64_t n8 = n / 8;
  const unsigned grid = (unsigned)((n8 + 255) / 256 < 65536 ? (n8 + 255) / 256 : 65536);
  MDATTN_LAUNCH(finalize_kernel, dim3(grid), dim3(256), 0, (hipStream_t)stream, (const float4*)o_run, (uint4*)out_bf16, n8);
  return launch_status();
}

extern "C" int mdattn_quant_e4m3(void* stream, const void* x_bf16, void* x_fp8, float* scale_out, int64_t n,
                                 float premul, int pow2_scale) {
  if (!x_bf16 || !x_fp8 || !scale_out || n <= 0) return MDATTN_E_BADARG;
  if (!(premul > 0.f) || !(premul < 1e30f)) return MDATTN_E_BADARG;
  if (n % 16) return MDATTN_E_UNSUPPORTED;
  if (!aligned16(x_bf16) || !aligned16(x_fp8) || (reinterpret_cast<uintptr_t>(scale_out) & 7u)) return MDATTN_E_ALIGN;
  hipStream_t st = (hipStream_t)stream;
  const int64_t n8 = n / 8, n16 = n / 16;
  const unsigned g1 = (unsigned)((n8 + 255) / 256 < 2048 ? (n8 + 255) / 256 : 2048);
  const unsigned g2 = (unsigned)((n16 + 255) / 256 < 16384 ? (n16 + 255) / 256 : 16384);
  MDATTN_LAUNCH(zero2_kernel, dim3(1), dim3(64), 0, st, scale_out);
  if (launch_status() != MDATTN_OK) return MDATTN_E_LAUNCH;
  MDATTN_LAUNCH(absmax_kernel, dim3(g1), dim3(256), 0, st, (const uint4*)x_bf16, n8, (unsigned*)(scale_out + 1));
  if (launch_status() != MDATTN_OK) return MDATTN_E_LAUNCH;
  MDATTN_LAUNCH(quant_kernel, dim3(g2), dim3(256), 0, st, (const uint4*)x_bf16, (uint4*)x_fp8, n16, scale_out,
                     premul, pow2_scale);
  return launch_status();
}

extern "C" int mdattn_host_copy(void* stream, const void* src0, void* dst0, const void* src1, void* dst1, int64_t bytes) {
  if (!src0 || !dst0 || !src1 != !dst1 || bytes <= 0) return MDATTN_E_BADARG;
  if (bytes % 16 || !aligned16(src0) || !aligned16(dst0) || !aligned16(src1) || !aligned16(dst1)) return MDATTN_E_ALIGN;
  const int64_t n16 = bytes / 16, groups = (n16 + 255) / 256;
  if (groups > 0x7FFFFFFF) return MDATTN_E_UNSUPPORTED;
  MDATTN_LAUNCH(copy_kernel, dim3((unsigned)groups, src1 ? 2 : 1), dim3(256), 0, (hipStream_t)stream, (const uint4*)src0, (uint4*)dst0, (const uint4*)src1,
                (uint4*)dst1, n16);
  return launch_status();
}

extern "C" int64_t mdattn_host_quant3_floats(void) { return 8 + 3 * kQuantSlots; }

extern "C" int mdattn_host_quant3_e4m3(void* stream, const void* q, const void* k, const void* v, void* q8, void* k8, void* v8, float* ws, int64_t nq,
                                       int64_t nkv, float q_premul) {
  if (!q || !k || !v || !q8 || !k8 || !v8 || !ws || nq <= 0 || nkv <= 0) return MDATTN_E_BADARG;
  if (!(q_premul > 0.f) || !(q_premul < 1e30f)) return MDATTN_E_BADARG;
  if (nq % 16 || nkv % 16) return MDATTN_E_UNSUPPORTED;
  if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(q8) || !aligned16(k8) || !aligned16(v8) || !aligned16(ws)) return MDATTN_E_ALIGN;
  Quant3Args a;
  a.x[0] = (const uint4*)q; a.x[1] = (const uint4*)k; a.x[2] = (const uint4*)v;
  a.y[0] = (uint4*)q8; a.y[1] = (uint4*)k8; a.y[2] = (uint4*)v8;
  a.n16[0] = nq / 16; a.n16[1] = a.n16[2] = nkv / 16;
  a.scale = ws;
  a.part = reinterpret_cast<unsigned*>(ws + 8);
  a.premul[0] = q_premul; a.premul[1] = a.premul[2] = 1.0f;
  a.pow2[0] = a.pow2[1] = 1; a.pow2[2] = 0;
  const int64_t most = nq > nkv ? nq / 16 : nkv / 16;
  // at least 8 KB of the longer tensor per workgroup; a workgroup without rows of the shorter one leaves 0
  const int64_t want = (2 * most + 511) / 512;
  const unsigned g1 = (unsigned)(want < kQuantSlots ? want : kQuantSlots);
  a.slots = (int)g1;
  const int64_t want2 = (most + 255) / 256;
  const unsigned g2 = (unsigned)(want2 < 8192 ? want2 : 8192);
  MDATTN_LAUNCH(absmax3_kernel, dim3(g1, 3), dim3(256), 0, (hipStream_t)stream, a);
  if (launch_status() != MDATTN_OK) return MDATTN_E_LAUNCH;
  MDATTN_LAUNCH(quant3_kernel, dim3(g2, 3), dim3(256), 0, (hipStream_t)stream, a);
  return launch_status();
}

// ------------------------------------------------------------------------------------------- key mask -> bias
namespace mdattn {
__global__ __launch_bounds__(256) void key_mask_bias_kernel(const uint8_t* __restrict__ keep, float* __restrict__ bias,
                                                            int Skv, int64_t bias_stride, float masked_value) {
  const int b = blockIdx.y;
  for (int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x; j < bias_stride; j += (int64_t)gridDim.x * 256)
    bias[b * bias_stride + j] = (j < Skv && keep[(int64_t)b * Skv + j]) ? 0.f : masked_value;
}
}  // namespace mdattn

extern "C" int mdattn_key_mask_bias(void* stream, const void* keep, float* bias, int B, int Skv, int64_t bias_stride,
                                    float masked_value) {
  if (!keep || !bias || B <= 0 || Skv <= 0 || bias_stride < Skv) return MDATTN_E_BADARG;
  if (B > 65535) return MDATTN_E_UNSUPPORTED;
  const unsigned gx = (unsigned)((bias_stride + 255) / 256 < 1024 ? (bias_stride + 255) / 256 : 1024);
  MDATTN_LAUNCH(mdattn::key_mask_bias_kernel, dim3(gx, B), dim3(256), 0, (hipStream_t)stream,
                     (const uint8_t*)keep, bias, Skv, bias_stride, masked_value);
  return mdattn::launch_status();
}

// ------------------------------------------------------------------------------- key mask -> bias and tile lists
namespace mdattn {
// The bias of key_mask_bias_kernel (masked value -inf) together with the lists of key tiles that hold a kept key, for
// tiles of 32 and of 64 keys: a masked attention then costs what its kept keys cost.  A workgroup takes kTileSlice tiles of 64
// keys of one batch element, as many as its waves load in one trip; where its entries start it finds by counting the kept tiles
// of all the slices before it, 64 bytes per lane (one workgroup per element took one slice after the other: 42 us for 75,600
// keys, now 5.0; 4.9 and 5.0 us for 4,096).  Masked calls before (every tile visited, the bias added to every logit) and with the
// lists: 500 of 2,048 keys x 2,048 queries x 20 heads 61 -> 23 us; 3,900 of 4,096 keys 188 -> 171 us at head dim 128, 126 ->
// 107 us at 64 (x 2 x 10 heads).  With a dropped key in every tile the lists give nothing (attn_fwd_bf16.hip: kKeyMask).
constexpr int kTileSlice = 128;
__global__ __launch_bounds__(1024) void key_tiles_kernel(const uint8_t* __restrict__ keep, float* __restrict__ bias, int* __restrict__ tiles,
                                                         int Skv, int64_t bias_stride, int B, int slices, int sb32, int sb64) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int b = blockIdx.x / slices, slice = blockIdx.x - b * slices;
  const uint8_t* kb = keep + (int64_t)b * Skv;
  float* bb = bias + b * bias_stride;
  int* l32 = tiles + (int64_t)b * sb32;
  int* l64 = tiles + (int64_t)B * sb32 + (int64_t)b * sb64;
  __shared__ int kept[2][kTileSlice];  // keys kept in each half of a tile
  __shared__ int sums[2][16], mine[2][kTileSlice / 64];
  const int n64 = (Skv + 63) / 64, t0 = slice * kTileSlice, last = t0 + kTileSlice < n64 ? t0 + kTileSlice : n64;

  // this slice's keys, neighbouring lanes on neighbouring keys: a wave covers one tile per load, eight loads in flight
  // (the address of a key past the end is that of the last one: under a condition the loads would wait for one another)
  uint8_t k[kTileSlice / 16];
#pragma unroll
  for (int i = 0; i < kTileSlice / 16; ++i) {
    const int64_t key = (int64_t)(t0 + wave + 16 * i) * 64 + lane;
    k[i] = kb[key < Skv ? key : Skv - 1];
  }
  // the tiles in front of it, all of 64 keys
  typedef unsigned u32x4_any __attribute__((ext_vector_type(4), aligned(1)));
  int c32 = 0, c64 = 0;
  for (int t = tid; t - lane < t0; t += 1024) {
    unsigned h0 = 0, h1 = 0;
    if (t < t0) {
      const u32x4_any* p = reinterpret_cast<const u32x4_any*>(kb + (int64_t)t * 64);
      const u32x4_any w = p[0] | p[1], x = p[2] | p[3];
      h0 = w.x | w.y | w.z | w.w;
      h1 = x.x | x.y | x.z | x.w;
    }
    const unsigned long long b0 = __builtin_amdgcn_ballot_w64(h0 != 0), b1 = __builtin_amdgcn_ballot_w64(h1 != 0);
    c32 += __popcll(b0) + __popcll(b1);
    c64 += __popcll(b0 | b1);
  }
  if (lane == 0) { sums[0][wave] = c32; sums[1][wave] = c64; }
#pragma unroll
  for (int i = 0; i < kTileSlice / 16; ++i) {
    const int at = wave + 16 * i;
    const int64_t key = (int64_t)(t0 + at) * 64 + lane;
    const bool kp = key < Skv && k[i];
    if (key < bias_stride) bb[key] = kp ? 0.f : -INFINITY;
    const unsigned long long m = __builtin_amdgcn_ballot_w64(kp);
    if (lane == 0) {
      kept[0][at] = __popc((unsigned)m);
      kept[1][at] = __popc((unsigned)(m >> 32));
    }
  }
  __syncthreads();
  // a lane per tile.  Exclusive ranks: of the first / second half's tile among the 32-key tiles, of the tile among the 64-key tiles
  const int t = t0 + tid;
  const int k0 = tid < kTileSlice ? kept[0][tid] : 0, k1 = tid < kTileSlice ? kept[1][tid] : 0;
  const unsigned long long lt = (1ull << lane) - 1;
  const unsigned long long b0 = __builtin_amdgcn_ballot_w64(k0 > 0), b1 = __builtin_amdgcn_ballot_w64(k1 > 0);
  if (lane == 0 && wave < kTileSlice / 64) {
    mine[0][wave] = __popcll(b0) + __popcll(b1);
    mine[1][wave] = __popcll(b0 | b1);
  }
  __syncthreads();
  if (tid >= kTileSlice) return;
  int r32 = __popcll(b0 & lt) + __popcll(b1 & lt), r64 = __popcll((b0 | b1) & lt), n32 = 0, n = 0;
#pragma unroll
  for (int w = 0; w < 16; ++w) { n32 += sums[0][w]; n += sums[1][w]; }
  r32 += n32;
  r64 += n;
#pragma unroll
  for (int w = 0; w < kTileSlice / 64; ++w) {
    if (w < wave) { r32 += mine[0][w]; r64 += mine[1][w]; }
    n32 += mine[0][w];
    n += mine[1][w];
  }
  const int left = Skv - t * 64;  // keys of this tile that exist
  if (k0 + k1 > 0) {
    const int e0 = left < 32 ? left : 32, e1 = left - 32 < 32 ? left - 32 : 32;
    if (k0 > 0) l32[1 + r32] = 4 * t + (k0 < e0);
    if (k1 > 0) l32[1 + r32 + (k0 > 0)] = 4 * t + 2 + (k1 < e1);
    l64[1 + r64] = 2 * t + (k0 + k1 < (left < 64 ? left : 64));
  }
  if (last == n64 && tid == 0) {
    l32[0] = n32;
    l64[0] = n;
  }
}
}  // namespace mdattn

extern "C" int64_t mdattn_host_key_tiles_ints(int B, int Skv) {
  return (int64_t)B * (key_tiles_ints(Skv, 32) + key_tiles_ints(Skv, 64));
}

extern "C" int mdattn_host_key_tiles(void* stream, const void* keep, float* bias, int* tiles, int B, int Skv, int64_t bias_stride) {
  if (!keep || !bias || !tiles || B <= 0 || Skv <= 0 || bias_stride < Skv || bias_stride % 32) return MDATTN_E_BADARG;
  const int slices = (int)(((int64_t)Skv + 64 * mdattn::kTileSlice - 1) / (64 * mdattn::kTileSlice));
  if ((int64_t)B * slices > 0x7FFFFFFF) return MDATTN_E_UNSUPPORTED;
  MDATTN_LAUNCH(mdattn::key_tiles_kernel, dim3(B * slices), dim3(1024), 0, (hipStream_t)stream, (const uint8_t*)keep, bias, tiles, Skv, bias_stride, B,
                slices, key_tiles_ints(Skv, 32), key_tiles_ints(Skv, 64));
  return mdattn::launch_status();
}
