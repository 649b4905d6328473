// Backward of the non-causal attention forward for gfx950 (MI355X), bf16 MFMA, head_dim 128: dq, dk, dv from
// (q, k, v, out, dout, lse).  With logits s = scale*q.k, p = exp(s - lse), dp = dout.v^T, delta = rowsum(dout*out):
//   dv = p^T dout,   ds = p * (dp - delta),   dq = scale * ds k,   dk = scale * ds^T q.
//
// One kernel body, two passes, no atomics: every gradient is accumulated by the waves that own its rows.
//   dq pass:      "entity" rows = 32 q rows per wave (q and dout fragments in registers), "stream" rows = keys
//                 (k for the scores and for the accumulation, v for dP).
//   dk / dv pass: entity rows = 32 key rows per wave (k and v fragments in registers), stream rows = q rows (q for
//                 the scores and the dk accumulation, dout for dP and the dv accumulation).  S^T and dP^T are formed
//                 once per tile; P feeds the dv accumulators and dS the dk ones: seven matrix products per call
//                 where five are necessary (S and dP are formed in both passes).
// Stream rows are walked in tiles of 32 through a 2-slot LDS ring filled by direct global->LDS loads.
// Per tile, with the forward kernel's fragment orders:
//   S^T  = stream1 . entity1^T      (A = tile rows by ds_read_b128, B = entity fragments)   lane = entity row
//   dP^T = stream2 . entity2^T
//   W    = exp2(c*S - lse*log2e) [* (dP - delta)]     f32, packed to bf16 in B-operand order (the factor `scale` of
//                                                      dS is applied once, to the finished accumulators)
//   acc^T += stream3^T . W          (A = the tile through the transposing LDS read)
// lse and delta belong to the q rows: per-lane scalars for dq; for dk / dv sixteen values per lane and tile, which
// ride through the ring next to the tile (a register load inside the loop would be waited for in issue order, i.e.
// behind the next tile's loads).  The dq pass forms them and leaves them in a workspace for the dk / dv pass (-delta and
// -lse in log2 units, padded to a multiple of 32 rows with -lse = -inf so that padded q rows get p = 0).  Both are stored
// negated because they start the MFMA chains they are subtracted from: dP^T - delta comes out of the chain, and so does
// S^T - lse when the caller's q already carries scale * log2(e) (the factor c is then 1).
#include <atomic>
#include <mutex>
#include <type_traits>

#include "mdattn_common.h"
#include "mdattn_host.h"

namespace mdattn {
namespace {

constexpr int kBT = 32;                  // stream rows per tile
// A tile: 32 rows of HD elements, filled by loads of 1 KB (4 rows at head dim 128, 8 at 64, LTX-2's audio stream).  One copy serves the row
// reads (ds_read_b128, 16 rows x one 16-byte chunk at a time) and the transposing reads (ds_read_b64_tr_b16, 4 rows x 64
// bytes): chunk c of row r sits at position c ^ swizzle(r), whose upper part, distinct within 4 rows that follow each other, moves
// the 64-byte segment (the 4 rows x 64 bytes cover every bank once) and whose lower part makes all positions of 16 rows distinct.  With
// a copy in a layout for each kind of read every tensor that is read both ways went from the L2 to LDS twice.
template <int HD>
struct BwdTile {
  static constexpr int RPI = HD == 128 ? 4 : 8;        // rows one load instruction fills
  static constexpr int Row = HD * 2, Bytes = 32 * Row;
  static __device__ __forceinline__ int swizzle(int r) { return HD == 128 ? 4 * (r & 3) + ((r >> 2) & 3) : 4 * ((r >> 1) & 1) + ((r >> 2) & 3); }
};

// Per-row f32 values of a stream tile (lse and delta of its q rows, or the bias of its keys) travel through the ring as
// well: 64 floats behind the tiles of a slot.
constexpr int kAuxFloats = 64;
template <int MODE, int HD, bool BIAS>
constexpr int bwd_slot_bytes() { return 2 * BwdTile<HD>::Bytes + ((MODE != 0 || BIAS) ? 4 * kAuxFloats : 0); }

// Tensors whose entity rows go through LDS: of the dq pass's three, at head dim 128 two, whose areas of two workgroups of four waves fit
// a CU.
template <int MODE, int HD>
constexpr int bwd_staged() { return MODE != 0 ? 0 : HD == 64 ? 3 : 2; }

typedef s16x4 __attribute__((address_space(3))) * lds_s16x4_ptr_b;
typedef __attribute__((ext_vector_type(8))) short s16x8_b;

typedef const bf16x8 __attribute__((address_space(3))) * lds_bf16x8_ptr;
typedef const f32x4 __attribute__((address_space(3))) * lds_f32x4_ptr;

// LDS addresses
__device__ __forceinline__ bf16x8 read_row(unsigned at) { return *(lds_bf16x8_ptr)at; }
__device__ __forceinline__ bf16x8 read_vt_b(unsigned at0, unsigned at1) {
  s16x4 r0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr_b)at0);
  s16x4 r1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr_b)at1);
  s16x8_b r = __builtin_shufflevector(r0, r1, 0, 1, 2, 3, 4, 5, 6, 7);
  return __builtin_bit_cast(bf16x8, r);
}

struct BwdArgs {
  const __bf16* e1;  // entity tensor of the score contraction
  const __bf16* e2;  // entity tensor of the dP contraction
  const __bf16* s1;  // stream tensor of the score contraction, which the gradient (MODE 3: dk) accumulates with
  const __bf16* s2;  // stream tensor of the dP contraction; MODE 3: dv accumulates with it
  __bf16* out;       // gradient of the entity rows
  __bf16* out2;      // MODE 3: dv
  int64_t o2_sb, o2_ss, o2_sh;
  // Written by the dq pass for the dk / dv pass, both negated (they start the MFMA chains that they are subtracted from)
  float* lse2;         // [B,H,Sp] -lse * log2(e), -inf on padded rows
  float* delta;        // [B,H,Sp] -rowsum(dout * out), 0 on padded rows
  const __bf16* fwd;   // MODE 0: the forward's out, with the strides of dout (e2)
  const float* lse;    // MODE 0: the forward's lse [B,H,Se]
  int H, Se, Ss, Sp, D;
  int net, total, chunk;
  int64_t e1_sb, e1_ss, e1_sh, e2_sb, e2_ss, e2_sh;
  int64_t s1_sb, s1_ss, s1_sh, s2_sb, s2_ss, s2_sh;
  int64_t o_sb, o_ss, o_sh;
  float c, scale;
  const float* bias;   // BIAS: additive per-key bias [B, bias_sb] in natural-log units (mdattn_fwd_bf16_bias)
  int64_t bias_sb;
  const int* tiles;    // BIAS: TileLists of 32 keys, tiles_sb ints per batch element, or null (see AttnArgs)
  int tiles_sb;
  // stream split: the tiles of the stream are dealt to nsplit workgroups per entity tile, tps tiles each; with nsplit > 1
  // a workgroup leaves f32 partial sums [split][B*H][Se][D] (part: out's, part2: out2's) for bwd_reduce_kernel
  int nsplit, tps;
  float* part;
  float* part2;
  int waves;  // per workgroup (head dim 128: 8 or 4)
};

// A wave's 32 rows of a gradient, rounded to bf16 and stored as pieces of 128 bytes of a row (8 rows per instruction), 64 columns
// at a time through `stage` (kStageRows bytes of LDS that nobody else touches any more; 64 columns and not the row, so that
// eight waves fit the ring).  As the accumulators lie, an instruction wrote 16 bytes of each of 32 rows a whole token apart:
// a training pass with 32,760 queries x 512 keys x 12 heads 638 -> 622 us, Flux 24 x 4,608 1076 -> 1062, 2 x 1,337 x 32 heads of 64
// 214 -> 209 (the longer the stream, the smaller the share: 18,900 x 20 heads 13.28 ms both ways).
constexpr int kStageRowB = 64 * 2 + 16, kStageRows = 32 * kStageRowB;
template <int ND, bool PADDED>
__device__ __forceinline__ void store_rows(const f32x16 (&acc)[ND], float mul, __bf16* base, int64_t ss, int row0, int rows, int D, int lane,
                                           char* stage) {
  const int l32 = lane & 31, hh = lane >> 5, rr = lane >> 3, cc = lane & 7;
#pragma unroll
  for (int d0 = 0; d0 < ND; d0 += 2) {
    // LDS accesses of one wave execute in order: the reads see the writes above them, and the next round's writes follow
#pragma unroll
    for (int db = d0; db < (d0 + 2 < ND ? d0 + 2 : ND); ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        uint2 u;
        u.x = pack2(acc[db][4 * g] * mul, acc[db][4 * g + 1] * mul);
        u.y = pack2(acc[db][4 * g + 2] * mul, acc[db][4 * g + 3] * mul);
        *reinterpret_cast<uint2*>(stage + l32 * kStageRowB + ((db - d0) * 32 + 8 * g + 4 * hh) * 2) = u;
      }
    const int col = d0 * 32 + cc * 8;
    if (col >= (PADDED ? D : ND * 32)) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int row = row0 + 8 * j + rr;
      const uint4 v = *reinterpret_cast<const uint4*>(stage + (8 * j + rr) * kStageRowB + cc * 16);
      if (row < rows) *reinterpret_cast<uint4*>(base + (int64_t)row * ss + col) = v;
    }
  }
}

// The same for the f32 partial sums of a wave's rows [rows][D]: 32 columns at a time, 128 bytes of each of 8 rows per instruction
// instead of 32 bytes of each of 32 (dk / dv pass of 32,760 queries x 512 keys x 12 heads 236 -> 227 us).
template <int ND, bool PADDED>
__device__ __forceinline__ void store_partial_rows(const f32x16 (&acc)[ND], float mul, float* base, int row0, int rows, int D, int lane, char* stage) {
  const int l32 = lane & 31, hh = lane >> 5, rr = lane >> 3, cc = lane & 7;
#pragma unroll
  for (int db = 0; db < ND; ++db) {
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<f32x4*>(stage + l32 * kStageRowB + (8 * g + 4 * hh) * 4) =
          f32x4{acc[db][4 * g] * mul, acc[db][4 * g + 1] * mul, acc[db][4 * g + 2] * mul, acc[db][4 * g + 3] * mul};
    const int col = db * 32 + cc * 4;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int row = row0 + 8 * j + rr;
      const f32x4 v = *reinterpret_cast<const f32x4*>(stage + (8 * j + rr) * kStageRowB + cc * 16);
      if (row < rows && (!PADDED || col < D)) *reinterpret_cast<f32x4*>(base + (int64_t)row * (PADDED ? D : ND * 32) + col) = v;
    }
  }
}

// MODE 0: dq (entity = q rows, stream = keys); 3: dk and dv in one pass (entity = key rows, stream = q rows).
// DC != 0: head dims other than HD (a.D, a multiple of 8 up to DC), as in the forward's flat schedule: the layout of HD, the
// MFMAs that cover DC columns; chunks past a.D are zero in the entity fragments and in the tiles (written once, no load
// touches them), and not stored in the gradients.
template <int MODE, int HD, bool BIAS, bool PRE, int DC, int NW>
__device__ __forceinline__ void attn_bwd_body(const BwdArgs& a) {
  static_assert(!(PRE && BIAS), "a biased logit is touched after the MFMAs anyway");
  extern __shared__ __attribute__((aligned(1024))) char smem_raw_b[];  // (fragment addresses are formed by xor)
  static_assert(MODE == 0 || MODE == 3, "dq, or dk and dv");
  constexpr bool BOTH = MODE == 3;
  using T = BwdTile<HD>;
  constexpr bool PADDED = DC != 0;
  constexpr int NJ = (PADDED ? DC : HD) / 16;         // MFMAs per 32 x 32 block of a contraction over the head dim
  constexpr int ND = ((PADDED ? DC : HD) + 31) / 32;  // 32-wide slabs of d = accumulators
  constexpr int kSlot = bwd_slot_bytes<MODE, HD, BIAS>(), kAux = 2 * T::Bytes;  // a slot: two tiles, the f32 values
  constexpr bool AUX = MODE != 0 || BIAS;
#ifndef MDATTN_BWD_LA
#define MDATTN_BWD_LA 4
#endif
  // fragment look-ahead of the dq pass over its whole read stream (head dim 64, at three waves per SIMD, has room for
  // two: 1 % on one machine, A/B; not with a key mask's tile list); the merged pass windows its two MFMA phases separately, LA1 and LA3 below
  constexpr int LA = MODE == 0 ? (HD == 128 ? MDATTN_BWD_LA : BIAS ? 0 : 2) : 0;
  static_assert(LA == 0 || (!BOTH && LA <= 2 * ND), "the window covers the three-product pass");
#ifndef MDATTN_BWD_LA1
#define MDATTN_BWD_LA1 2
#endif
#ifndef MDATTN_BWD_LA3
#define MDATTN_BWD_LA3 6
#endif
  constexpr int LA3 = BOTH && HD == 128 ? (BIAS ? 4 : MDATTN_BWD_LA3) : 0;
  constexpr int LA1 = BOTH && HD == 128 ? MDATTN_BWD_LA1 : 0;  // merged pass: look-ahead over the chains' row reads only

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hh = lane >> 5;

  const int wg = blockIdx.x;
  const int w = (wg & 7) * a.chunk + (wg >> 3);
  if (w >= a.total) return;
  // entity tiles fastest: neighbouring workgroups walk the same piece of the stream
  const int bhs = w / a.net, et = w - bhs * a.net;
  const int bh = bhs / a.nsplit, sp = bhs - bh * a.nsplit;
  const int b = bh / a.H, h = bh - b * a.H;
  const int r0 = et * (NW * 32) + wave * 32;
  // this workgroup's stream: rows ss0 .. ss0 + Ss - 1 of the sequence (never empty); everything below counts from ss0
  const bool listed = BIAS && MODE == 0 && a.tiles;  // (its tiles are numbered from the sequence's start)
  const int ss0 = listed ? 0 : sp * a.tps * kBT;
  const int Ss = listed || a.Ss - ss0 < a.tps * kBT ? a.Ss - ss0 : a.tps * kBT;
  int nt = (Ss + kBT - 1) / kBT;
  const float c = a.c;
  // dq pass with a mask: the key tiles that hold a kept key, this workgroup's share of them (perhaps none)
  [[maybe_unused]] TileList tl{BIAS && MODE == 0 && a.tiles ? a.tiles + (int64_t)b * a.tiles_sb : nullptr};
  [[maybe_unused]] const int tl_n = tl.count(sp * a.tps + nt);
  if constexpr (BIAS && MODE == 0) {
    if (tl.list) {
      nt = tl_n - sp * a.tps < a.tps ? tl_n - sp * a.tps : a.tps;
      nt = nt > 0 ? nt : 0;
    }
  }

  float* lrow = a.lse2 + ((int64_t)b * a.H + h) * a.Sp + (MODE != 0 ? ss0 : 0);
  float* drow = a.delta + ((int64_t)b * a.H + h) * a.Sp + (MODE != 0 ? ss0 : 0);
  // a wave without rows, or with excluded keys only, brings its share of the tiles and computes nothing
  bool idle = r0 >= a.Se;
  // key bias in log2 units: a per-lane scalar when the keys are the entity rows, sixteen values per tile otherwise
  [[maybe_unused]] const float* bias_row = BIAS ? a.bias + b * a.bias_sb + (MODE == 0 ? ss0 : 0) : nullptr;
  [[maybe_unused]] float bias_e = 0.f;
  if constexpr (BIAS && MODE != 0) {
    bias_e = bias_row[r0 + l32 < a.Se ? r0 + l32 : a.Se - 1] * kLog2e;
    if (!__syncthreads_or(bias_e != -INFINITY)) nt = 0;  // only excluded keys in this workgroup: zero gradients (a NaN excludes none)
    idle = idle || __builtin_amdgcn_ballot_w64(bias_e != -INFINITY) == 0;
  }

  // ---- direct global -> LDS loads of one stream tile (layouts and lane maps of the forward kernel)
  const __bf16* s1p = a.s1 + b * a.s1_sb + h * a.s1_sh + ss0 * a.s1_ss;
  const __bf16* s2p = a.s2 + b * a.s2_sb + h * a.s2_sh + ss0 * a.s2_ss;
  constexpr int RPI = T::RPI;
  const int grow = HD == 128 ? lane >> 4 : lane >> 3;
  // lane -> logical 16-byte chunk stored at this lane's position of row group g (a wave fills the groups wave, wave + NW, ...: the
  // swizzle sees the same g)
  auto in_head = [&](int col) __attribute__((always_inline)) { return !PADDED || col < a.D ? col : 0; };
  auto chunk_col = [&](int g) __attribute__((always_inline)) { return ((lane & (HD / 8 - 1)) ^ T::swizzle(RPI * g + grow)) * 8; };
  const int acol0 = chunk_col(wave);
  const int acol = in_head(acol0);
  [[maybe_unused]] const bool ain = !PADDED || acol0 < a.D;
  const unsigned smem_addr = lds_addr_of(smem_raw_b);
  // byte offset of a lane's chunk from the first row of its row group: the same for every full tile (strides are below 2^23).  The
  // merged pass at head dim 128 has no registers to keep the two offsets in (spilled, every reload would wait for the load
  // issued before it): it forms them again per tile from the lane number, half a dozen full-rate instructions.
  constexpr bool REFORM = BOTH && HD == 128;
  auto chunk_ofs = [&](int ln, int64_t ss) __attribute__((always_inline)) {
    const int gr = HD == 128 ? ln >> 4 : ln >> 3;
    return (__umul24((unsigned)gr, (unsigned)ss) + (unsigned)in_head(((ln & (HD / 8 - 1)) ^ T::swizzle(RPI * wave + gr)) * 8)) * 2u;
  };
  [[maybe_unused]] const unsigned ofs1 = REFORM ? 0u : chunk_ofs(lane, a.s1_ss), ofs2 = REFORM ? 0u : chunk_ofs(lane, a.s2_ss);
  // wave 0 brings a tile's f32 values: lanes 0-31 the lse of its 32 q rows and lanes 32-63 their delta, or (dq pass)
  // every lane the bias of key lane % 32.  Through LDS because a register load here would be waited for in order
  // behind the next tile's loads.
  [[maybe_unused]] const unsigned ofs_aux =
      MODE != 0 ? (lane < 32 ? 0u : (unsigned)((a.delta - a.lse2) * 4)) + (unsigned)l32 * 4u : (unsigned)l32 * 4u;
  [[maybe_unused]] const uint64_t amask = __builtin_amdgcn_ballot_w64(ain);
  // a row group: the lanes whose chunk lies inside the head dim
  auto dma_a = [&](auto... at) __attribute__((always_inline)) {
    if constexpr (PADDED) lds_dma16(at..., amask);
    else lds_dma16(at...);
  };
  auto dma = [&](int slot, int t) __attribute__((always_inline)) {
    const unsigned A1 = smem_addr + (unsigned)(slot * kSlot), A2 = A1 + T::Bytes;
    if constexpr (AUX) {
      if (wave == 0) {
        unsigned oa = ofs_aux;
        if constexpr (REFORM) {
          int ln = lane;
          asm volatile("" : "+v"(ln));
          oa = (ln < 32 ? 0u : (unsigned)((a.delta - a.lse2) * 4)) + (unsigned)(ln & 31) * 4u;
        }
        lds_dma4((MODE != 0 ? lrow : bias_row) + t * kBT, oa, A1 + kAux);
      }
    }
    if (t * kBT + kBT <= Ss) {  // a full tile: uniform row-group bases, one per-lane offset per stream
      unsigned o1 = ofs1, o2 = ofs2;
      if constexpr (REFORM) {
        int ln = lane;
        asm volatile("" : "+v"(ln));  // opaque: keeps the two offsets from being hoisted out of the loop
        o1 = chunk_ofs(ln, a.s1_ss);
        o2 = chunk_ofs(ln, a.s2_ss);
      }
#pragma unroll
      for (int i = 0; i < (kBT / RPI) / NW; ++i) {
        const int g = wave + NW * i;
        const int64_t r = t * kBT + RPI * g;
        dma_a(s1p + r * a.s1_ss, o1, A1 + (unsigned)g * 1024u);
        dma_a(s2p + r * a.s2_ss, o2, A2 + (unsigned)g * 1024u);
      }
    } else {  // the ragged last tile: rows past the end repeat the last row
#pragma unroll
      for (int i = 0; i < (kBT / RPI) / NW; ++i) {
        const int g = wave + NW * i;
        int rr = t * kBT + RPI * g + grow;
        rr = rr < Ss ? rr : Ss - 1;
        dma_a(s1p + (int64_t)rr * a.s1_ss + acol, A1 + (unsigned)g * 1024u);
        dma_a(s2p + (int64_t)rr * a.s2_ss + acol, A2 + (unsigned)g * 1024u);
      }
    }
  };

  f32x16 acc[ND];
  [[maybe_unused]] f32x16 acc2[BOTH ? ND : 1];  // MODE 3: dv next to dk
#pragma unroll
  for (int db = 0; db < ND; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      acc[db][i] = 0.f;
      if constexpr (BOTH) acc2[db][i] = 0.f;
    }

  // Fragment addresses from the first byte of a tile, a multiple of 256: row read j (logical chunk 2 j + hh of row l32) at k_at ^ 32 j;
  // transposing read of 32-column slab sg at v_at ^ 64 sg for the rows 4 hh + 0..3 and, eight rows on, at that ^ 32.
  const int vxr = (lane & 15) >> 2;
  const unsigned k_at = (unsigned)(l32 * T::Row + ((hh ^ T::swizzle(l32)) * 16));
  const unsigned v_at = (unsigned)((4 * hh + vxr) * T::Row + ((2 * ((lane >> 4) & 1) + ((lane & 3) >> 1)) ^ T::swizzle(4 * hh + vxr)) * 16 + (lane & 1) * 8);
  // CONST, the dq pass with eight waves: the two copies of the loop body know their slot, and what the xors give is a lane constant plus
  // an immediate offset.  Elsewhere they are formed again for every tile: the merged pass at head dim 128 has no registers for
  // them, and a short stream walks two copies slower than one (32,760 queries x 512 keys x 12 heads 176 us, 199 with two copies;
  // 18,900 x 18,900 x 20 4,470 and 4,266).
  constexpr bool CONST = MODE == 0 && NW == 8;
  auto row_frag = [&](unsigned tile, int j, int ofs) __attribute__((always_inline)) {
    return (((CONST ? smem_addr : tile) + k_at) ^ (unsigned)(32 * j)) + (CONST ? tile - smem_addr + ofs : (unsigned)ofs);
  };
  auto vt_frag = [&](unsigned slot_at, int jv, int second) __attribute__((always_inline)) {  // second: of the slot's second tile
    const unsigned at = ((CONST ? smem_addr : slot_at) + v_at) ^ (unsigned)(64 * (jv % ND)), add = (CONST ? slot_at - smem_addr : 0u) + second * T::Bytes;
    return read_vt_b(at + (add + (jv / ND) * 16 * T::Row), (at ^ 32u) + (add + (8 + (jv / ND) * 16) * T::Row));
  };

  // ---- entity fragments.  As lanes hold them they are 16-byte pieces of one row: a load from global memory touches 32 bytes of each of
  // 32 rows.  The dq pass, which reads three rows for every one it writes, stages them instead: a wave's rows arrive like a
  // stream tile, whole rows per load, in an area that then becomes the ring, and the fragments are read with a row tile's offsets
  // (32,530 queries x 77 keys x 20 heads 172 -> 147 us, 69,319 x 512 x 40 1,231 -> 1,156, 18,900 x 18,900 x 20 4,235 -> 4,202).
  // The dk / dv pass, with two tensors and a long stream, would only see its first tile requested later (512 x 512 x 32 22.4 -> 23.2 us).
  constexpr int NST = bwd_staged<MODE, HD>();
  bf16x8 ef1[NJ], ef2[NJ];
  [[maybe_unused]] bf16x8 ef3[MODE == 0 ? NJ : 1];  // MODE 0: the forward's out, for delta
  const bf16x8 zero8 = __builtin_bit_cast(bf16x8, u32x4{0u, 0u, 0u, 0u});
  auto in_row = [&](int s) __attribute__((always_inline)) { return !PADDED || s * 16 + hh * 8 < a.D; };
  auto direct = [&](bf16x8 (&f)[NJ], const __bf16* p, int64_t ss) __attribute__((always_inline)) {
    p += (int64_t)(r0 + l32 < a.Se ? r0 + l32 : a.Se - 1) * ss + hh * 8;
#pragma unroll
    for (int s = 0; s < NJ; ++s) f[s] = in_row(s) ? *reinterpret_cast<const bf16x8*>(p + s * 16) : zero8;
  };
  if constexpr (NST == 0) {
    direct(ef1, a.e1 + b * a.e1_sb + h * a.e1_sh, a.e1_ss);
    direct(ef2, a.e2 + b * a.e2_sb + h * a.e2_sh, a.e2_ss);
  } else {
    const unsigned stage0 = smem_addr + (unsigned)(wave * NST * T::Bytes);
    const bool whole = r0 + 32 <= a.Se;
    auto stage = [&](const __bf16* p, int64_t ss, int n) __attribute__((always_inline)) {
#pragma unroll
      for (int g = 0; g < 32 / RPI; ++g) {
        const int col = in_head(chunk_col(g));
        const unsigned at = stage0 + (unsigned)(n * T::Bytes + g * 1024);
        if (whole) {
          lds_dma16(p + (int64_t)(r0 + RPI * g) * ss, (__umul24((unsigned)grow, (unsigned)ss) + (unsigned)col) * 2u, at);
        } else {
          const int row = r0 + RPI * g + grow;
          lds_dma16(p + (int64_t)(row < a.Se ? row : a.Se - 1) * ss + col, at);
        }
      }
    };
    const __bf16* po = a.fwd + b * a.e2_sb + h * a.e2_sh;
    if constexpr (NST < 3) direct(ef3, po, a.e2_ss);
    stage(a.e1 + b * a.e1_sb + h * a.e1_sh, a.e1_ss, 0);
    stage(a.e2 + b * a.e2_sb + h * a.e2_sh, a.e2_ss, 1);
    if constexpr (NST == 3) stage(po, a.e2_ss, 2);
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the wave's own rows
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      ef1[j] = in_row(j) ? read_row(row_frag(stage0, j, 0)) : zero8;
      ef2[j] = in_row(j) ? read_row(row_frag(stage0, j, T::Bytes)) : zero8;
      if constexpr (NST == 3) ef3[j] = in_row(j) ? read_row(row_frag(stage0, j, 2 * T::Bytes)) : zero8;
    }
    __syncthreads();  // every wave holds its fragments: the staging area is the ring now
  }

  if (!ain) {  // the chunks past the head dim of this wave's row groups (the loop's first barrier shows them to the others)
#pragma unroll
    for (int i = 0; i < 2 * ((kBT / RPI) / NW); ++i) {
      char* at = smem_raw_b + (i & 1) * kSlot + (wave + NW * (i >> 1)) * 1024 + lane * 16;
      *reinterpret_cast<uint4*>(at) = make_uint4(0u, 0u, 0u, 0u);
      *reinterpret_cast<uint4*>(at + T::Bytes) = make_uint4(0u, 0u, 0u, 0u);
    }
  }

  // LISTED: the tile at position t of this workgroup's share as tile * 2 + (it holds keys with a bias)
  constexpr bool LISTED = BIAS && MODE == 0;
  [[maybe_unused]] auto entry = [&](int t) __attribute__((always_inline)) {
    if (!tl.list) return 2 * t + 1;
    const int at = sp * a.tps + t;
    if (t == 0 && (at & 63)) tl.lane_entry = tl.list[1 + ((at & ~63) + lane < tl_n ? (at & ~63) + lane : tl_n - 1)];
    return tl.at(at, tl_n, lane);
  };
  [[maybe_unused]] int ec = 0;
  if constexpr (LISTED) {
    if (nt > 0) {
      ec = entry(0);
      dma(0, ec >> 1);
    }
  } else {
    if (!BIAS || nt > 0) dma(0, 0);
  }
  // Beside the first tile's way: rowsum(dout * out) from the dout fragments that the pass holds anyway.  In a launch in front of it
  // dout was read once more (40 us at 32,760 rows x 12 heads): a training pass there against 512 keys 656 -> 644 us, 24 x 4,608
  // 1094 -> 1076.
  float nlse_e = 0.f, ndelta_e = 0.f;  // both negated
  if constexpr (MODE == 0) {
#pragma unroll
    for (int s = 0; s < NJ; ++s)
#pragma unroll
      for (int e = 0; e < 8; ++e) ndelta_e = __builtin_fmaf(-(float)ef3[s][e], (float)ef2[s][e], ndelta_e);
    ndelta_e = xhalf_sum(ndelta_e);
    // rows whose keys were all masked (the forward wrote lse = -inf, out = 0) take no part: p = 0
    const int row = r0 + l32;
    const float lv = a.lse[(int64_t)bh * a.Se + (row < a.Se ? row : a.Se - 1)];
    nlse_e = lv > -INFINITY ? -lv * kLog2e : -INFINITY;
    if (sp == 0 && hh == 0 && row < a.Sp) {
      lrow[row] = row < a.Se ? nlse_e : -INFINITY;
      drow[row] = row < a.Se ? ndelta_e : 0.f;
    }
  }
  auto tile = [&](int t, auto slot) __attribute__((always_inline)) {  // slot: t & 1, an int or an integral_constant
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's share of tile t has landed
    __syncthreads();                      // ... and everyone's; the other slot (tile t-1) is free
    int kt = t;
    [[maybe_unused]] bool mixed = true;
    if constexpr (LISTED) {
      kt = ec >> 1;
      mixed = ec & 1;
      if (t + 1 < nt) {
        ec = entry(t + 1);
        dma(slot ^ 1, ec >> 1);
      }
    } else {
      if (t + 1 < nt) dma(slot ^ 1, t + 1);
    }
    if (idle) return;
    const unsigned base = smem_addr + (unsigned)(slot * kSlot);

    // Start values of the two MFMA chains: -delta for dP^T, so that the chain ends on dP - delta; and, when the
    // logits come out of the MFMAs in log2 units (PRE), -lse for S^T, so that exp2 applies to the chain's result
    // as it is.  Per-lane constants when the q rows are the entity rows, the tile's values from LDS otherwise.
    [[maybe_unused]] auto aux4 = [&](int i) __attribute__((always_inline)) { return *(lds_f32x4_ptr)(base + (unsigned)(kAux + 4 * i)); };
    f32x16 S, dP;
    if constexpr (MODE == 0) {
#pragma unroll
      for (int i = 0; i < 16; ++i) { S[i] = PRE ? nlse_e : 0.f; dP[i] = ndelta_e; }
    } else {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4 dv = aux4(32 + 8 * g + 4 * hh);
#pragma unroll
        for (int e = 0; e < 4; ++e) dP[4 * g + e] = dv[e];
        if constexpr (PRE) {
          const f32x4 lv = aux4(8 * g + 4 * hh);
#pragma unroll
          for (int e = 0; e < 4; ++e) S[4 * g + e] = lv[e];
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) S[4 * g + e] = 0.f;
        }
      }
    }
    // The tile's fragment reads as one stream: NJ row reads for S^T, NJ for dP^T, then the 2*ND transposing reads
    // of the accumulation.  With LA > 0 a window of LA fragments runs ahead of the MFMAs (pinned by scheduling
    // barriers: left to itself the compiler waits for every read right before its MFMA).
    auto frag = [&](int n) __attribute__((always_inline)) {
      if (n < NJ) return read_row(row_frag(base, n, 0));
      if (n < 2 * NJ) return read_row(row_frag(base, n - NJ, T::Bytes));
      return vt_frag(base, n - 2 * NJ, 0);
    };
    [[maybe_unused]] bf16x8 win[LA > 0 ? LA : 1];
    if constexpr (LA > 0) {
#pragma unroll
      for (int n = 0; n < LA; ++n) win[n] = frag(n);
#pragma unroll
      for (int n = 0; n < 2 * NJ; ++n) {
        if (n < NJ) S = __builtin_amdgcn_mfma_f32_32x32x16_bf16(win[n % LA], ef1[n % NJ], S, 0, 0, 0);
        else dP = __builtin_amdgcn_mfma_f32_32x32x16_bf16(win[n % LA], ef2[n % NJ], dP, 0, 0, 0);
        win[n % LA] = frag(n + LA);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else if constexpr (LA1 > 0) {  // a window over the row reads of the two chains only
      bf16x8 w1[LA1];
#pragma unroll
      for (int n = 0; n < LA1; ++n) w1[n] = frag(n);
#pragma unroll
      for (int n = 0; n < 2 * NJ; ++n) {
        if (n < NJ) S = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w1[n % LA1], ef1[n % NJ], S, 0, 0, 0);
        else dP = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w1[n % LA1], ef2[n % NJ], dP, 0, 0, 0);
        if (n + LA1 < 2 * NJ) w1[n % LA1] = frag(n + LA1);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
#pragma unroll
      for (int j = 0; j < NJ; ++j) S = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag(j), ef1[j], S, 0, 0, 0);
#pragma unroll
      for (int j = 0; j < NJ; ++j) dP = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag(NJ + j), ef2[j], dP, 0, 0, 0);
    }
    // W = P or dS, eight logits (one B operand) at a time
    if constexpr (MODE == 0) {
      if (t == nt - 1) {  // keys past the end of a ragged last tile take no part
        const int sbase = kt * kBT + 4 * hh;
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (sbase + 8 * (i >> 2) + (i & 3) >= Ss) S[i] = -INFINITY;
      }
    }
    bf16x8 W[2];
    [[maybe_unused]] bf16x8 Wp[2];  // MODE 3: the probabilities themselves, for dv
#pragma unroll
    for (int hb = 0; hb < 2; ++hb) {
      [[maybe_unused]] float nl[8];  // -lse (log2 units) of each logit's q row, with the key's bias added
      if constexpr (!PRE) {
        if constexpr (MODE == 0) {
#pragma unroll
          for (int e = 0; e < 8; ++e) nl[e] = nlse_e;
          if (BIAS && mixed) {
#pragma unroll
            for (int g = 0; g < 2; ++g) {
              const int col = kt * kBT + 8 * (2 * hb + g) + 4 * hh;
              const f32x4 bv = aux4(8 * (2 * hb + g) + 4 * hh);
#pragma unroll
              for (int e = 0; e < 4; ++e)
                nl[4 * g + e] = col + e < Ss ? __builtin_fmaf(bv[e], kLog2e, nlse_e) : -INFINITY;  // whatever the padding holds
            }
          }
        } else {
#pragma unroll
          for (int g = 0; g < 2; ++g) {
            const f32x4 lv = aux4(8 * (2 * hb + g) + 4 * hh);
#pragma unroll
            for (int e = 0; e < 4; ++e) nl[4 * g + e] = BIAS ? lv[e] + bias_e : lv[e];
          }
        }
      }
      unsigned wpk[4];
      [[maybe_unused]] unsigned ppk[4];
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        const float p0 = __builtin_amdgcn_exp2f(PRE ? S[8 * hb + e] : __builtin_fmaf(S[8 * hb + e], c, nl[e]));
        const float p1 = __builtin_amdgcn_exp2f(PRE ? S[8 * hb + e + 1] : __builtin_fmaf(S[8 * hb + e + 1], c, nl[e + 1]));
        // dS without its factor `scale`: applied once, to the accumulators
        wpk[e >> 1] = pack2(p0 * dP[8 * hb + e], p1 * dP[8 * hb + e + 1]);
        if constexpr (BOTH) ppk[e >> 1] = pack2(p0, p1);
      }
      W[hb] = __builtin_bit_cast(bf16x8, u32x4{wpk[0], wpk[1], wpk[2], wpk[3]});
      if constexpr (BOTH) Wp[hb] = __builtin_bit_cast(bf16x8, u32x4{ppk[0], ppk[1], ppk[2], ppk[3]});
    }
    if constexpr (LA3 > 0) {  // merged pass: a window over the transposing reads of both accumulations
      auto frag3 = [&](int n) __attribute__((always_inline)) {
        return vt_frag(base, n >> 1, n & 1);
      };
      bf16x8 w3[LA3];
#pragma unroll
      for (int n = 0; n < LA3; ++n) w3[n] = frag3(n);
#pragma unroll
      for (int n = 0; n < 4 * ND; ++n) {
        const int jv = n >> 1;
        if (n & 1) acc2[jv % ND] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w3[n % LA3], Wp[jv / ND], acc2[jv % ND], 0, 0, 0);
        else acc[jv % ND] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w3[n % LA3], W[jv / ND], acc[jv % ND], 0, 0, 0);
        if (n + LA3 < 4 * ND) w3[n % LA3] = frag3(n + LA3);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else
#pragma unroll
    for (int jv = 0; jv < 2 * ND; ++jv) {
      if constexpr (LA > 0) {
        acc[jv % ND] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(win[(2 * NJ + jv) % LA], W[jv / ND], acc[jv % ND], 0, 0, 0);
        if (jv + LA < 2 * ND) win[(2 * NJ + jv) % LA] = frag(2 * NJ + jv + LA);
        __builtin_amdgcn_sched_barrier(0);
        continue;
      }
      const bf16x8 f = vt_frag(base, jv, 0);
      acc[jv % ND] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f, W[jv / ND], acc[jv % ND], 0, 0, 0);
      if constexpr (BOTH) {
        const bf16x8 f2 = vt_frag(base, jv, 1);
        acc2[jv % ND] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f2, Wp[jv / ND], acc2[jv % ND], 0, 0, 0);
      }
    }
  };
  if constexpr (CONST) {
    for (int t = 0; t < nt; t += 2) {
      tile(t, std::integral_constant<int, 0>{});
      if (t + 1 >= nt) break;
      tile(t + 1, std::integral_constant<int, 1>{});
    }
  } else {
    for (int t = 0; t < nt; ++t) tile(t, t & 1);
  }

  const float osc = a.scale;  // dq = scale * dS k, dk = scale * dS^T q
  // the lane number once more: the loop has no register for it (spills at head dim 128)
  const int ln = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
  __syncthreads();  // every wave has finished reading the ring, and no load into it is in flight: it now stages the outputs
  char* stage = smem_raw_b + wave * kStageRows;
  if (a.nsplit > 1) {  // partial sums over this workgroup's share of the stream, in f32
    const int64_t nbh = a.total / (a.net * a.nsplit), o = ((int64_t)sp * nbh + bh) * a.Se * (PADDED ? a.D : HD);
    store_partial_rows<ND, PADDED>(acc, osc, a.part + o, r0, a.Se, a.D, ln, stage);
    if constexpr (BOTH) store_partial_rows<ND, PADDED>(acc2, 1.0f, a.part2 + o, r0, a.Se, a.D, ln, stage);
    return;
  }
  store_rows<ND, PADDED>(acc, osc, a.out + b * a.o_sb + h * a.o_sh, a.o_ss, r0, a.Se, a.D, ln, stage);
  if constexpr (BOTH) store_rows<ND, PADDED>(acc2, 1.0f, a.out2 + b * a.o2_sb + h * a.o2_sh, a.o2_ss, r0, a.Se, a.D, ln, stage);
}

template <int MODE, int HD, bool BIAS, bool PRE, int DC, int NW>
__global__ __launch_bounds__((NW * 64)) __attribute__((amdgpu_waves_per_eu(HD == 64 ? 3 : 2, HD == 64 ? 3 : 2))) void attn_bwd_kernel(BwdArgs a) {
  attn_bwd_body<MODE, HD, BIAS, PRE, DC, NW>(a);
}
// The dk / dv pass at head dim 128 wants a few registers more than half the register file (128 accumulators, 64 of
// entity fragments, 32 of S and dP): held to two waves per SIMD, which the schedule needs to overlap one wave's
// exponentials with the other's MFMAs; at one wave per SIMD it measured 28 % slower.  Head dim 64 fits three waves
// per SIMD (3 % faster than two).
template <int HD, bool BIAS, bool PRE, int DC, int NW>
__global__ __launch_bounds__((NW * 64)) __attribute__((amdgpu_waves_per_eu(HD == 64 ? 3 : 2, HD == 64 ? 3 : 2))) void attn_bwd_both_kernel(BwdArgs a) {
  attn_bwd_body<3, HD, BIAS, PRE, DC, NW>(a);
}

// Sums the partial gradients of a split pass in the order of the splits and rounds them to bf16: one 16-byte store per
// lane, blockIdx.y = tensor.  Bound by the partials' bytes: 12.8 us for 63 MB (4.9 TB/s).
struct BwdReduceArgs {
  const float* part[2];
  __bf16* out[2];
  int64_t sb[2], ss[2], sh[2];
  int H, S, nsplit;
  int cpr;         // 16-byte chunks per row, D/8
  int64_t chunks;  // B*H*S*cpr
};
__global__ __launch_bounds__(256) void bwd_reduce_kernel(BwdReduceArgs a) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= a.chunks) return;
  const int t = blockIdx.y;
  const int64_t row = i / a.cpr;
  const int c = (int)(i - row * a.cpr);
  const int s = (int)(row % a.S);
  const int64_t bh = row / a.S;
  const int64_t b = bh / a.H, h = bh - b * a.H;
  const float4* p = reinterpret_cast<const float4*>(a.part[t]) + 2 * i;
  float f[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int k = 0; k < a.nsplit; ++k, p += 2 * a.chunks) {
    const float4 u = ld_nt(p), v = ld_nt(p + 1);
    f[0] += u.x; f[1] += u.y; f[2] += u.z; f[3] += u.w; f[4] += v.x; f[5] += v.y; f[6] += v.z; f[7] += v.w;
  }
  *reinterpret_cast<uint4*>(a.out[t] + b * a.sb[t] + (int64_t)s * a.ss[t] + h * a.sh[t] + c * 8) = pack8(f);
}

// How a pass is launched: the waves of a workgroup and into how many pieces it cuts its stream, by the lowest cost in us of
//   rounds of workgroups x (stream tiles per workgroup x time per tile + a workgroup's start and end)
//   + for a cut stream the partials, read back at 5 TB/s, and the launch that sums them.
// Head dims above 64: eight waves (256 entity rows, one workgroup per CU) share each tile, which a full chip walks 4 % faster;
// four (128 rows, two workgroups per CU) leave less of a tile empty, and hide one workgroup's start behind the other's tiles, which
// in the dq pass, whose start reads three rows for every one it will write, counts against a few hundred keys; alone on a CU
// a workgroup of four is a third faster per tile.  Measured (dq / dk, dv pass, us, eight waves -> four): 69,319 queries x 512 keys x 40
// heads 1,421 / 1,259 -> 1,251 / 1,360, 512 x 512 x 32 24.8 / 28.5 -> 18.6 / 22.7, 2,000 x 2,000 x 40 153 / 201 -> 130 / 181, 18,900 x
// 18,900 x 20 4,345 / 6,039 -> 4,495 / 6,328.
// The stream is cut where its own rows leave a pass without workgroups: 12 heads x 32,760 queries x 512 keys: the dk / dv pass takes
// 1312 us in one piece (24 workgroups) and 201 us in ten, + 13 us of bwd_reduce_kernel.
constexpr int kMinSplitTiles = 8, kMaxSplit = 32;
// The rates were fitted at head dims 128 and 64 and serve 72 to 96 and up to 48 as they are.  Over 91 random shapes each pass as planned is 0.2 to
// 2.2 % behind the fastest of its plans on average, 17 % at most, at 80 and 96 as at 128; under a mask 1 to 6 %, and up to 1.9 times where the
// mask drops most keys: what it keeps is known on the device only.
using BwdPlan = mdattn_host_bwd_pass;
// A key bias or mask costs the dq pass 0.3 us per tile, whose sixteen bias values per lane stand between the products (measured 0.25 to 0.35 more
// with one, two and three workgroups on a CU, at head dims 40 to 128); the dk / dv pass has one per lane and call.  Without that 2 x 4 heads
// x 3,572 x 3,572 under a mask ran its dq pass whole, 125 us, 93 in three pieces, and 16 heads of 40 x 1,688 x 1,688 45 us, 33 in three.
inline double bwd_bias_us(int tensors, bool bias) { return bias && tensors == 1 ? 0.3 : 0.0; }
inline double bwd_pass_us(int D, int tensors, bool bias, int waves, int64_t wgs, int tps) {
  const double more = bwd_bias_us(tensors, bias);
  if (D <= 64) {  // workgroups of four waves, three per CU
    const double tile[3] = {more + (tensors == 2 ? 0.74 : 0.54), more + (tensors == 2 ? 1.15 : 0.8), more + (tensors == 2 ? 1.45 : 1.1)};  // with one, two, three of them
    const int64_t rest = wgs % 768;
    return (double)(wgs / 768) * (tps * tile[2] + 4.0) + (rest ? tps * tile[(rest - 1) / 256] + 4.0 : 0.0);
  }
  const int slots = waves == 8 ? 256 : 512;
  const int64_t rounds = waves == 8 ? wgs / 256 : wgs / 512, rest = wgs - rounds * slots;
  const double tile = more + (tensors == 2 ? (waves == 8 ? 1.65 : 1.75) : (waves == 8 ? 1.2 : 1.25));
  const double alone = waves == 8 ? tile : more + (tensors == 2 ? 1.3 : 0.8);       // with the CU to itself
  const double full = tensors == 2 ? 0.0 : waves == 8 ? 10.0 : 5.5;        // of a start, when every CU reads its rows at once
  double us = (double)rounds * (tps * tile + 4.0 + full);
  if (rest) us += tps * (rest <= 256 ? alone : tile) + 4.0 + full * (double)rest / slots;
  return us;
}
// entity rows Se, stream rows Ss; tensors: gradients the pass produces (2 in the dk / dv pass); room: floats for partials
inline BwdPlan bwd_plan(int64_t BH, int Se, int Ss, int D, int tensors, bool bias, int64_t room) {
  const int nt = (Ss + kBT - 1) / kBT;
  const int64_t floats = BH * Se * D;
  const double partial = 1.5 * tensors * (double)floats * 4 / 5e6;  // (writing them is half hidden)
  const int most = D > 64 ? 8 : 4;
  BwdPlan best{most, 1, nt, 0};
  double best_cost = 1e300;
  for (int waves = most; waves >= 4; waves -= 4) {
    const double cost = bwd_pass_us(D, tensors, bias, waves, BH * ((Se + waves * 32 - 1) / (waves * 32)), nt);
    if (cost < best_cost) { best_cost = cost; best.waves = waves; }
  }
  for (int waves = most; waves >= 4; waves -= 4) {
    const int64_t entities = BH * ((Se + waves * 32 - 1) / (waves * 32));
    // no cut is faster than its tiles on a full chip, the partials of two pieces and their launch
    const int slots = D <= 64 ? 768 : waves == 8 ? 256 : 512;
    const double full_tile = D <= 64 ? (tensors == 2 ? 1.45 : 1.1) : tensors == 2 ? (waves == 8 ? 1.65 : 1.75) : (waves == 8 ? 1.2 : 1.25);
    if ((double)entities * nt * (full_tile + bwd_bias_us(tensors, bias)) / slots + 2 * partial + 6.0 >= best_cost * 0.95) continue;
    for (int n = 2; n <= kMaxSplit && nt / n >= kMinSplitTiles; ++n) {
      const int tps = (nt + n - 1) / n, ns = (nt + tps - 1) / tps;
      if (ns * floats * tensors > room) break;
      const double cost = bwd_pass_us(D, tensors, bias, waves, entities * ns, tps) + partial * ns + 6.0;
      if (cost < best_cost * 0.95) { best_cost = cost; best = {waves, ns, tps, ns * floats}; }
    }
  }
  return best;
}
// The plan of a call without limits, and where a pass's partials do not fit, the best one for that pass that does.  Which cuts are
// looked at decides where two are within 5 %: with the limit in the first search a call with the workspace of this very plan was launched
// with another in one of forty shapes.
inline mdattn_host_bwd_plan bwd_plans(int64_t BH, int Sq, int Skv, int D, bool bias, int64_t room) {
  mdattn_host_bwd_plan p{bwd_plan(BH, Sq, Skv, D, 1, bias, INT64_MAX), bwd_plan(BH, Skv, Sq, D, 2, bias, INT64_MAX)};
  if (p.dq.floats > room) p.dq = bwd_plan(BH, Sq, Skv, D, 1, bias, room);
  if (2 * p.dkv.floats > room) p.dkv = bwd_plan(BH, Skv, Sq, D, 2, bias, room);
  return p;
}
// whether a pass of this plan covers its Ss stream rows, without an empty piece, and says the space it takes
inline bool bwd_plan_ok(const BwdPlan& p, int64_t BH, int Se, int Ss, int D) {
  const int64_t nt = ((int64_t)Ss + kBT - 1) / kBT;
  return (p.waves == 4 || (p.waves == 8 && D > 64)) && p.pieces >= 1 && p.tiles >= 1 && (int64_t)p.pieces * p.tiles >= nt &&
         (int64_t)(p.pieces - 1) * p.tiles < nt && p.floats == (p.pieces > 1 ? p.pieces * BH * Se * D : 0);
}

template <int MODE, int HD, bool BIAS, bool PRE, int DC, int NW>
int launch_bwd_nw(hipStream_t st, BwdArgs a, int B) {
  // the ring, or in front of it the waves' staged rows and behind it their staged outputs
  constexpr int ring = 2 * bwd_slot_bytes<MODE, HD, BIAS>(), staged = NW * bwd_staged<MODE, HD>() * BwdTile<HD>::Bytes, stored = NW * kStageRows;
  constexpr int lds_bytes = ring > staged ? (ring > stored ? ring : stored) : (staged > stored ? staged : stored);
  a.net = (a.Se + NW * 32 - 1) / (NW * 32);
  const int64_t total = (int64_t)B * a.H * a.net * a.nsplit;
  if (total > (int64_t)0x7FFFFFF0) return MDATTN_E_UNSUPPORTED;
  a.total = (int)total;
  a.chunk = (a.total + 7) / 8;
  void (*kern)(BwdArgs);
  if constexpr (MODE == 3) kern = attn_bwd_both_kernel<HD, BIAS, PRE, DC, NW>;
  else kern = attn_bwd_kernel<MODE, HD, BIAS, PRE, DC, NW>;
  static LdsOptIn opted;
  if (lds_opt_in(opted, reinterpret_cast<const void*>(kern), lds_bytes) != MDATTN_OK) return MDATTN_E_LAUNCH;
  MDATTN_LAUNCH(kern, dim3(a.chunk * 8), dim3(NW * 64), lds_bytes, st, a);
  return launch_status();
}

template <int MODE, int HD, bool BIAS, bool PRE, int DC = 0>
int launch_bwd_as(hipStream_t st, const BwdArgs& a, int B) {
  if constexpr (HD == 128) {
    if (a.waves == 8) return launch_bwd_nw<MODE, HD, BIAS, PRE, DC, 8>(st, a, B);
  }
  return launch_bwd_nw<MODE, HD, BIAS, PRE, DC, 4>(st, a, B);
}

// scale * log2(e) == 1 (to f32 round-off: the caller's q carries the factor, as for the forward): the logits leave the
// MFMAs in log2 units and take -lse as the chain's start value instead of a multiply-add each.
template <int MODE, int HD, bool BIAS>
int launch_bwd(hipStream_t st, const BwdArgs& a, int B) {
  // (not for the merged pass at head dim 128: there the start values come from LDS, a read that the chain's first
  // MFMA then waits for, and the multiply-add version measured 3 % faster)
  if constexpr (!BIAS && !(MODE == 3 && HD == 128)) {
    if (a.c > 1.0f - 1e-6f && a.c < 1.0f + 1e-6f) return launch_bwd_as<MODE, HD, false, true>(st, a, B);
  }
  return launch_bwd_as<MODE, HD, BIAS, false>(st, a, B);
}

template <int MODE, bool BIAS>
int launch_bwd_dim(hipStream_t st, const BwdArgs& a, int B) {
  if (a.D == 128) return launch_bwd<MODE, 128, BIAS>(st, a, B);
  if (a.D == 64) return launch_bwd<MODE, 64, BIAS>(st, a, B);
  if (a.D <= 48) return launch_bwd_as<MODE, 64, BIAS, false, 48>(st, a, B);
  if (a.D <= 80) return launch_bwd_as<MODE, 128, BIAS, false, 80>(st, a, B);
  return launch_bwd_as<MODE, 128, BIAS, false, 96>(st, a, B);
}
template <int MODE>
int launch_bwd_any(hipStream_t st, const BwdArgs& a, int B) {
  return a.bias ? launch_bwd_dim<MODE, true>(st, a, B) : launch_bwd_dim<MODE, false>(st, a, B);
}

int launch_bwd_reduce(hipStream_t st, const BwdArgs& a, int B) {
  BwdReduceArgs r;
  r.part[0] = a.part; r.part[1] = a.part2;
  r.out[0] = a.out; r.out[1] = a.part2 ? a.out2 : nullptr;
  r.sb[0] = a.o_sb; r.ss[0] = a.o_ss; r.sh[0] = a.o_sh;
  r.sb[1] = a.o2_sb; r.ss[1] = a.o2_ss; r.sh[1] = a.o2_sh;
  r.H = a.H; r.S = a.Se; r.nsplit = a.nsplit;
  r.cpr = a.D / 8;
  r.chunks = (int64_t)B * a.H * a.Se * r.cpr;
  const dim3 grid((unsigned)((r.chunks + 255) / 256), a.part2 ? 2 : 1);
  MDATTN_LAUNCH(bwd_reduce_kernel, grid, dim3(256), 0, st, r);
  return launch_status();
}

}  // namespace
}  // namespace mdattn

using namespace mdattn;

extern "C" int64_t mdattn_bwd_workspace_floats(int B, int H, int Sq) {
  if (B <= 0 || H <= 0 || Sq <= 0) return 0;
  return 2 * (int64_t)B * H * (((int64_t)Sq + 31) / 32 * 32);
}

// the two passes run one after the other and their partials share the space
static int64_t plan_floats(int B, int H, int Sq, const mdattn_host_bwd_plan& p) {
  return mdattn_bwd_workspace_floats(B, H, Sq) + (p.dq.floats > 2 * p.dkv.floats ? p.dq.floats : 2 * p.dkv.floats);
}

extern "C" int64_t mdattn_bwd_split_workspace_floats(int B, int H, int Sq, int Skv, int D) {
  if (B <= 0 || H <= 0 || Sq <= 0 || Skv <= 0 || !native_head_dim(D)) return 0;
  const int64_t BH = (int64_t)B * H;
  const int64_t plain = plan_floats(B, H, Sq, bwd_plans(BH, Sq, Skv, D, false, INT64_MAX)), biased = plan_floats(B, H, Sq, bwd_plans(BH, Sq, Skv, D, true, INT64_MAX));
  return plain > biased ? plain : biased;
}

extern "C" int64_t mdattn_host_bwd_plan_floats(int B, int H, int Sq, int Skv, int D, int key_bias, int64_t workspace_floats, mdattn_host_bwd_plan* plan) {
  const int64_t base = mdattn_bwd_workspace_floats(B, H, Sq);
  if (base == 0 || Skv <= 0 || !native_head_dim(D) || (workspace_floats >= 0 && workspace_floats < base)) return 0;
  const mdattn_host_bwd_plan p = bwd_plans((int64_t)B * H, Sq, Skv, D, key_bias != 0, workspace_floats < 0 ? INT64_MAX : workspace_floats - base);
  if (plan) *plan = p;
  return plan_floats(B, H, Sq, p);
}

// Shared body of mdattn_bwd_bf16 and mdattn_bwd_bf16_static: validation and the two passes.
static int bwd_run(hipStream_t st, const void* q, const void* k, const void* v, const void* out, const void* dout,
                   const float* lse, void* dq, void* dk, void* dv, float* workspace, int64_t workspace_floats,
                   int B, int H, int Sq, int Skv, int D,
                   const mdattn_strides* q_strides, const mdattn_strides* k_strides,
                   const mdattn_strides* v_strides, const mdattn_strides* o_strides, float scale,
                   const float* key_bias, int64_t bias_stride, bool any_head_dim = false, const int* tiles = nullptr,
                   const mdattn_host_bwd_plan* plan = nullptr) {
  if (!q || !k || !v || !out || !dout || !lse || !dq || !dk || !dv || !workspace) return MDATTN_E_BADARG;
  if (key_bias) {
    if (bias_stride < ((int64_t)Skv + 31) / 32 * 32 || bias_stride % 32 != 0) return MDATTN_E_BADARG;
    if (!aligned16(key_bias)) return MDATTN_E_ALIGN;
  }
  if (B <= 0 || H <= 0 || Sq <= 0 || Skv <= 0 || D <= 0) return MDATTN_E_BADARG;
  if (!q_strides || !k_strides || !v_strides || !o_strides) return MDATTN_E_BADARG;
  if (!(scale > 0.f) || !(scale < 1e30f)) return MDATTN_E_BADARG;
  if (D != 128 && D != 64 && !(any_head_dim && native_head_dim(D))) return MDATTN_E_UNSUPPORTED;
  if (workspace_floats < mdattn_bwd_workspace_floats(B, H, Sq)) return MDATTN_E_BADARG;
  if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(out) || !aligned16(dout) || !aligned16(dq) ||
      !aligned16(dk) || !aligned16(dv) || !aligned16(workspace) || (reinterpret_cast<uintptr_t>(lse) & 3u))
    return MDATTN_E_ALIGN;
  if (!strides_ok(q_strides, 8) || !strides_ok(k_strides, 8) || !strides_ok(v_strides, 8) || !strides_ok(o_strides, 8))
    return MDATTN_E_ALIGN;
  if (q_strides->seq < D || k_strides->seq < D || v_strides->seq < D || o_strides->seq < D) return MDATTN_E_BADARG;
  // every tensor is streamed by one of the passes with 32-bit byte offsets inside a row group
  if (q_strides->seq >= (1 << 23) || k_strides->seq >= (1 << 23) || v_strides->seq >= (1 << 23) || o_strides->seq >= (1 << 23))
    return MDATTN_E_UNSUPPORTED;

  const int Sp = (Sq + 31) / 32 * 32;
  float* lse2 = workspace;
  float* delta = workspace + (int64_t)B * H * Sp;
  const int64_t rows = (int64_t)B * H * Sp;
  if (rows >= (1 << 29)) return MDATTN_E_UNSUPPORTED;  // delta - lse2 as a 32-bit byte offset

  // a stream is cut as far as the caller's workspace holds the partials (it always holds lse2 and delta)
  const int64_t BH = (int64_t)B * H;
  if (plan && (!bwd_plan_ok(plan->dq, BH, Sq, Skv, D) || !bwd_plan_ok(plan->dkv, BH, Skv, Sq, D) || workspace_floats < plan_floats(B, H, Sq, *plan)))
    return MDATTN_E_BADARG;
  const mdattn_host_bwd_plan p = plan ? *plan : bwd_plans(BH, Sq, Skv, D, key_bias != nullptr, workspace_floats - 2 * rows);
  BwdArgs a;
  a.lse2 = lse2; a.delta = delta; a.fwd = (const __bf16*)out; a.lse = lse; a.H = H; a.Sp = Sp; a.D = D; a.c = scale * kLog2e; a.scale = scale;
  a.bias = key_bias; a.bias_sb = bias_stride;
  a.tiles = tiles; a.tiles_sb = key_tiles_ints(Skv, 32);
  auto set = [](int64_t& sb, int64_t& ss, int64_t& sh, const mdattn_strides* s) { sb = s->batch; ss = s->seq; sh = s->head; };
  // dq: entity q / dout, stream k (scores), v (dP), k (accumulate)
  a.e1 = (const __bf16*)q; a.e2 = (const __bf16*)dout; a.s1 = (const __bf16*)k; a.s2 = (const __bf16*)v;
  a.out = (__bf16*)dq; a.Se = Sq; a.Ss = Skv;
  set(a.e1_sb, a.e1_ss, a.e1_sh, q_strides); set(a.e2_sb, a.e2_ss, a.e2_sh, o_strides);
  set(a.s1_sb, a.s1_ss, a.s1_sh, k_strides); set(a.s2_sb, a.s2_ss, a.s2_sh, v_strides);
  set(a.o_sb, a.o_ss, a.o_sh, q_strides);
  a.waves = p.dq.waves; a.nsplit = p.dq.pieces; a.tps = p.dq.tiles; a.part = workspace + 2 * rows; a.part2 = nullptr;
  int rc = launch_bwd_any<0>(st, a, B);
  if (rc != MDATTN_OK) return rc;
  if (a.nsplit > 1 && (rc = launch_bwd_reduce(st, a, B)) != MDATTN_OK) return rc;
  // dk and dv in one pass: entity k / v, stream q (scores, and accumulate for dk), dout (dP, and accumulate for dv)
  a.e1 = (const __bf16*)k; a.e2 = (const __bf16*)v; a.s1 = (const __bf16*)q; a.s2 = (const __bf16*)dout;
  a.out = (__bf16*)dk; a.out2 = (__bf16*)dv; a.Se = Skv; a.Ss = Sq;
  set(a.e1_sb, a.e1_ss, a.e1_sh, k_strides); set(a.e2_sb, a.e2_ss, a.e2_sh, v_strides);
  set(a.s1_sb, a.s1_ss, a.s1_sh, q_strides); set(a.s2_sb, a.s2_ss, a.s2_sh, o_strides);
  set(a.o_sb, a.o_ss, a.o_sh, k_strides); set(a.o2_sb, a.o2_ss, a.o2_sh, v_strides);
  a.waves = p.dkv.waves; a.nsplit = p.dkv.pieces; a.tps = p.dkv.tiles; a.part2 = a.part + p.dkv.floats;
  rc = launch_bwd_any<3>(st, a, B);
  if (rc == MDATTN_OK && a.nsplit > 1) rc = launch_bwd_reduce(st, a, B);
  return rc;
}


extern "C" int mdattn_bwd_bf16(void* stream, const void* q, const void* k, const void* v, const void* out, const void* dout,
                               const float* lse, void* dq, void* dk, void* dv, float* workspace, int64_t workspace_floats,
                               int B, int H, int Sq, int Skv, int D,
                               const mdattn_strides* q_strides, const mdattn_strides* k_strides,
                               const mdattn_strides* v_strides, const mdattn_strides* o_strides, float scale) {
  return bwd_run((hipStream_t)stream, q, k, v, out, dout, lse, dq, dk, dv, workspace, workspace_floats, B, H, Sq, Skv, D,
                 q_strides, k_strides, v_strides, o_strides, scale, nullptr, 0);
}

extern "C" int mdattn_bwd_bf16_bias(void* stream, const void* q, const void* k, const void* v, const void* out, const void* dout,
                                    const float* lse, void* dq, void* dk, void* dv, float* workspace, int64_t workspace_floats,
                                    int B, int H, int Sq, int Skv, int D,
                                    const mdattn_strides* q_strides, const mdattn_strides* k_strides,
                                    const mdattn_strides* v_strides, const mdattn_strides* o_strides, float scale,
                                    const float* key_bias, int64_t bias_stride) {
  if (!key_bias) return MDATTN_E_BADARG;
  return bwd_run((hipStream_t)stream, q, k, v, out, dout, lse, dq, dk, dv, workspace, workspace_floats, B, H, Sq, Skv, D,
                 q_strides, k_strides, v_strides, o_strides, scale, key_bias, bias_stride);
}

extern "C" int mdattn_host_bwd_bf16(void* stream, const void* q, const void* k, const void* v, const void* out, const void* dout,
                                    const float* lse, void* dq, void* dk, void* dv, float* workspace, int64_t workspace_floats,
                                    int B, int H, int Sq, int Skv, int D,
                                    const mdattn_strides* q_strides, const mdattn_strides* k_strides,
                                    const mdattn_strides* v_strides, const mdattn_strides* o_strides, float scale,
                                    const float* key_bias, int64_t bias_stride, const int* tiles, const mdattn_host_bwd_plan* plan) {
  return bwd_run((hipStream_t)stream, q, k, v, out, dout, lse, dq, dk, dv, workspace, workspace_floats, B, H, Sq, Skv, D,
                 q_strides, k_strides, v_strides, o_strides, scale, key_bias, bias_stride, true, key_bias ? tiles : nullptr, plan);
}

// ---------------------------------------------------------------------------------------------------
// mdattn_bwd_bf16_static: the same backward for callers that cannot allocate (HIP graph capture, serving loops that
// forbid hipMalloc).  The workspace (-lse in log2 units and -delta, one float each per padded query row, and behind them the
// partial gradients of a split pass where the array has room) lives in a
// file-scope device array instead of a caller's buffer.  Every GPU holds its own copy of the array at its own
// address: that address is looked up once per device with hipGetSymbolAddress and kept; host code never uses the
// array's name as a pointer.  The dq pass writes every element of it that the dk / dv pass reads, so nothing has to be cleared
// between calls; calls that overlap on one GPU share the array and race.
static __device__ __align__(256) float scratch[MDATTN_BWD_STATIC_MAX_FLOATS];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
std::atomic<float*> g_scratch_ptr[kMaxDevices];

// Device address of `scratch` on the current device (looked up on the first call per device), or nullptr.
float* scratch_on_current_device() {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return nullptr;
  float* p = g_scratch_ptr[dev].load(std::memory_order_acquire);
  if (p) return p;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  p = g_scratch_ptr[dev].load(std::memory_order_relaxed);
  if (p) return p;
  void* sym = nullptr;
  if (hipGetSymbolAddress(&sym, HIP_SYMBOL(scratch)) != hipSuccess || !sym) {
    (void)hipGetLastError();
    return nullptr;
  }
  p = static_cast<float*>(sym);
  g_scratch_ptr[dev].store(p, std::memory_order_release);
  return p;
}
}  // namespace

// Also the warm-up of the static entry point: looks the array's address up for the current device (which may make the
// runtime load the code object and place the array), so that a later mdattn_bwd_bf16_static call -- under graph
// capture, say -- finds it resolved.  Without a GPU the lookup fails quietly.
extern "C" int64_t mdattn_bwd_static_max_floats(void) {
  (void)scratch_on_current_device();
  return MDATTN_BWD_STATIC_MAX_FLOATS;
}

extern "C" int mdattn_bwd_bf16_static(void* stream, const void* q, const void* k, const void* v, const void* out,
                                      const void* dout, const float* lse, void* dq, void* dk, void* dv,
                                      int B, int H, int Sq, int Skv, int D,
                                      const mdattn_strides* q_strides, const mdattn_strides* k_strides,
                                      const mdattn_strides* v_strides, const mdattn_strides* o_strides, float scale) {
  if (B <= 0 || H <= 0 || Sq <= 0) return MDATTN_E_BADARG;
  const int64_t need = mdattn_bwd_workspace_floats(B, H, Sq);
  if (need > (int64_t)MDATTN_BWD_STATIC_MAX_FLOATS) return MDATTN_E_TOOBIG;
  float* ws = scratch_on_current_device();
  if (!ws) return MDATTN_E_LAUNCH;
  return bwd_run((hipStream_t)stream, q, k, v, out, dout, lse, dq, dk, dv, ws, MDATTN_BWD_STATIC_MAX_FLOATS, B, H, Sq, Skv, D,
                 q_strides, k_strides, v_strides, o_strides, scale, nullptr, 0);
}
