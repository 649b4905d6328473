// Shared device/host helpers for the gfx950 kernels behind mdattn.h.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>

#include "mdattn.h"

namespace mdattn {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(4))) short s16x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(8))) float f32x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(2))) unsigned u32x2;
typedef __attribute__((ext_vector_type(4))) unsigned u32x4;
typedef __attribute__((ext_vector_type(8))) int i32x8;

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

// max over the two lanes l and l^32 (the two halves of a wave64).
__device__ __forceinline__ float xhalf_max(float x) {
  u32x2 r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float xhalf_sum(float x) {
  u32x2 r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Butterfly sum over each aligned group of 16 lanes, on the VALU's DPP path.
__device__ __forceinline__ float row16_sum(float x) {
  x += __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(x), 0xB1, 0xF, 0xF, true));   // quad_perm [1,0,3,2]
  x += __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(x), 0x4E, 0xF, 0xF, true));   // quad_perm [2,3,0,1]
  x += __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(x), 0x141, 0xF, 0xF, true));  // row_half_mirror
  x += __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(x), 0x140, 0xF, 0xF, true));  // row_mirror
  return x;
}

__device__ __forceinline__ float bf16_bits_to_f32(unsigned short b) { return __uint_as_float(((unsigned)b) << 16); }

// 8 bf16 packed in a uint4 -> 8 floats.
__device__ __forceinline__ void unpack8(const uint4& u, float* f) {
  f[0] = __uint_as_float(u.x << 16); f[1] = __uint_as_float(u.x & 0xFFFF0000u);
  f[2] = __uint_as_float(u.y << 16); f[3] = __uint_as_float(u.y & 0xFFFF0000u);
  f[4] = __uint_as_float(u.z << 16); f[5] = __uint_as_float(u.z & 0xFFFF0000u);
  f[6] = __uint_as_float(u.w << 16); f[7] = __uint_as_float(u.w & 0xFFFF0000u);
}

// two floats -> packed bf16 pair (round-to-nearest-even; gfx950 has a native convert).
__device__ __forceinline__ unsigned pack2(float a, float b) {
  f32x2 v = {a, b};
  bf16x2 r = __builtin_convertvector(v, bf16x2);
  return __builtin_bit_cast(unsigned, r);
}
__device__ __forceinline__ uint4 pack8(const float* f) {
  uint4 u;
  u.x = pack2(f[0], f[1]); u.y = pack2(f[2], f[3]); u.z = pack2(f[4], f[5]); u.w = pack2(f[6], f[7]);
  return u;
}

// streaming (non-temporal) 16-byte accesses for data touched exactly once
__device__ __forceinline__ uint4 ld_nt(const uint4* p) {
  const u32x4 v = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
  return make_uint4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ float4 ld_nt(const float4* p) {
  const f32x4 v = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p));
  return make_float4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ void st_nt(uint4* p, const uint4& u) {
  const u32x4 v = {u.x, u.y, u.z, u.w};
  __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(p));
}

// Four consecutive rotation angles' cos and sin, group i (of four) of a rotary table in one of the layouts of
// mdattn_host.h's MDATTN_TABLE_*: the table is read as the model made it (splitting a complex table into planes first was
// two strided copies, 10 us and two launches of a 160 us call at 4,680 tokens).
template <int TABLE>
__device__ __forceinline__ void load_rope4(const float4* cos, const float4* sin, int64_t i, float* cc, float* sv) {
  if constexpr (TABLE == 0) {  // planes [S, D/2]
    const float4 c = cos[i], s = sin[i];
    cc[0] = c.x; cc[1] = c.y; cc[2] = c.z; cc[3] = c.w;
    sv[0] = s.x; sv[1] = s.y; sv[2] = s.z; sv[3] = s.w;
  } else if constexpr (TABLE == 1) {  // complex [S, D/2]
    const float4 a = cos[2 * i], b = cos[2 * i + 1];
    cc[0] = a.x; cc[1] = a.z; cc[2] = b.x; cc[3] = b.z;
    sv[0] = a.y; sv[1] = a.w; sv[2] = b.y; sv[3] = b.w;
  } else if constexpr (TABLE == 2) {  // planes [S, D], each angle for both of its pair
    const float4 a = cos[2 * i], b = cos[2 * i + 1], c = sin[2 * i], d = sin[2 * i + 1];
    cc[0] = a.x; cc[1] = a.z; cc[2] = b.x; cc[3] = b.z;
    sv[0] = c.x; sv[1] = c.z; sv[2] = d.x; sv[3] = d.z;
  } else {  // matrices [S, D/2, 2, 2] = [[cos, -sin], [sin, cos]]
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float4 m = cos[4 * i + j];
      cc[j] = m.x;
      sv[j] = m.z;
    }
  }
}

// Direct global -> LDS load of 16 bytes per lane: lane i's bytes land at lds_addr + 16*i (the LDS base
// travels in M0).  Written as inline assembly so that the loads stay asynchronous: the compiler cannot
// tell which LDS bytes such a load writes and would otherwise wait for it before the next LDS read.
// The statement writes M0 and says so, so the compiler never keeps a value of its own in M0 across it.
// The kernels track these loads themselves with s_waitcnt vmcnt.
__device__ __forceinline__ void lds_dma16(const void* base, unsigned byte_off, unsigned lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(lds_addr), "v"(byte_off), "s"(base) : "memory", "m0");
}
__device__ __forceinline__ void lds_dma16(const void* addr, unsigned lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(lds_addr), "v"(addr) : "memory", "m0");
}
// The same for the lanes of `mask` (at least one).  The mask is applied inside the statement: under an `if` the compiler merges
// such loads across branches and with that takes the LDS address into a vector register.
__device__ __forceinline__ void lds_dma16(const void* base, unsigned byte_off, unsigned lds_addr, uint64_t mask) {
  uint64_t all;
  asm volatile("s_mov_b32 m0, %1\n\ts_and_saveexec_b64 %0, %4\n\tglobal_load_lds_dwordx4 %2, %3\n\ts_mov_b64 exec, %0"
               : "=&s"(all) : "s"(lds_addr), "v"(byte_off), "s"(base), "s"(mask) : "memory", "m0", "scc");
}
__device__ __forceinline__ void lds_dma16(const void* addr, unsigned lds_addr, uint64_t mask) {
  uint64_t all;
  asm volatile("s_mov_b32 m0, %1\n\ts_and_saveexec_b64 %0, %3\n\tglobal_load_lds_dwordx4 %2, off\n\ts_mov_b64 exec, %0"
               : "=&s"(all) : "s"(lds_addr), "v"(addr), "s"(mask) : "memory", "m0", "scc");
}
// The 4-byte form: lane i's dword lands at lds_addr + 4*i.
__device__ __forceinline__ void lds_dma4(const void* base, unsigned byte_off, unsigned lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dword %1, %2" : : "s"(lds_addr), "v"(byte_off), "s"(base) : "memory", "m0");
}
__device__ __forceinline__ unsigned lds_addr_of(const void* p) {
  return (unsigned)(uintptr_t)(const void __attribute__((address_space(3)))*)p;
}

// The key tiles that a masked pass visits (made by key_tiles_kernel): entry = tile * 2 + (1: the tile holds excluded keys).  A
// wave keeps 64 entries in a register, one per lane, and reads the wanted one into a scalar: a scalar load per tile would
// turn every LDS wait around it into a full one.
struct TileList {
  const int* list;  // [count, entry 0, entry 1, ..]; null: none, every tile is visited
  int lane_entry = 0;
  __device__ __forceinline__ int count(int all) const { return list ? __builtin_amdgcn_readfirstlane(list[0]) : all; }
  // entry t of n; successive calls go up by one, or repeat
  __device__ __forceinline__ int at(int t, int n, int lane) {
    if ((t & 63) == 0) {
      const int i = t + lane;
      lane_entry = list[1 + (i < n ? i : n - 1)];
      // waited for here, once in 64 tiles: a load still pending where the branch ends would be waited for at every tile, and with
      // it every tile that is on its way into LDS
      asm volatile("" : "+v"(lane_entry));
    }
    return __builtin_amdgcn_readlane(lane_entry, t & 63);
  }
};

// Arguments of the attention-forward kernels (element strides; head_dim contiguous).
struct AttnArgs {
  const __bf16* q;
  const __bf16* k;
  const __bf16* v;
  __bf16* out;
  float* lse;
  int H, Sq, Skv, D;
  int nqt, total, chunk;
  int64_t q_sb, q_ss, q_sh;
  int64_t k_sb, k_ss, k_sh;
  int64_t v_sb, v_ss, v_sh;
  int64_t o_sb, o_ss, o_sh;
  float c;  // scale * log2(e)
  const float* bias;   // optional additive per-key bias [B, bias_sb] (natural-log units), flat kernel only
  int64_t bias_sb;
  const int* tiles;    // kKeyMask: per batch element, the number of key tiles to visit and their entries (see key_tiles_kernel)
  int tiles_sb;
  float* o_run;    // when set: no `out`; the result is merged in LSE space into this f32 carry (strides o_s*, in floats)
  float* lse_run;  // ... and into its lse [B,H,Sq]
  // key split (flat kernel without a bias): the key tiles are dealt to nsplit workgroups per query tile, tps each; with part
  // set, each leaves its un-normalised f32 output [split][B*H][Sq][D] and (reference point, sum of P) per row for
  // fwd_combine_kernel
  int nsplit, tps, BH;
  int cached_out;  // flat kernel at head dims other than 64 and 128: the output by ordinary stores
  float* part;
  float2* ml;
};



inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
// ints per batch of a TileList for tiles of ts keys
inline int key_tiles_ints(int Skv, int ts) { return 1 + (Skv + ts - 1) / ts; }
// Head dims that the attention kernels walk as they are: 64 and 128, and, in the layout of the next of these two with the
// MFMAs that cover 48, 80 or 96 columns, multiples of 8 up to 48 and from 72 to 96.  (56 saves nothing against 64; 104 to 120
// save a column of MFMAs at most, spill in the backward, and lose the pipelined forward: they are padded by the caller.)
inline bool native_head_dim(int D) { return D == 64 || D == 128 || (D > 0 && D % 8 == 0 && (D <= 48 || (D > 64 && D <= 96))); }
// a rotary table of layout `table` (0: planes, cos and sin; 1: complex; 2: repeated planes; 3: matrices): both pointers or none
// for the planes, cos alone for the others
inline bool table_ok(const float* cos, const float* sin, int table) {
  if (table < 0 || table > 3) return false;
  return table == 0 || table == 2 ? (cos == nullptr) == (sin == nullptr) : sin == nullptr;
}
inline bool strides_ok(const mdattn_strides* s, int64_t mult) {
  return s && s->batch % mult == 0 && s->seq % mult == 0 && s->head % mult == 0 && s->seq > 0 && s->head > 0 && s->batch >= 0;
}
// Every kernel launch of the library goes through MDATTN_LAUNCH and is followed by launch_status().  hipGetLastError()
// returns (and clears) the last error of ANY earlier HIP call on the calling thread, so an error that the caller's own
// code left pending would otherwise surface here as MDATTN_E_LAUNCH of a launch that went fine: MDATTN_LAUNCH reads
// the pending error first.  That clears it: a caller who wants to see its own sticky error has to read it before
// calling into the library.
#define MDATTN_LAUNCH(...)         \
  do {                             \
    (void)hipGetLastError();       \
    hipLaunchKernelGGL(__VA_ARGS__); \
  } while (0)
inline int launch_status() { return hipGetLastError() == hipSuccess ? MDATTN_OK : MDATTN_E_LAUNCH; }

// A kernel that needs more dynamic LDS than the default limit has to opt in with hipFuncSetAttribute, once per
// kernel and device: one LdsOptIn per kernel instance remembers the devices that have been told.
struct LdsOptIn {
  std::atomic<uint64_t> devices{0};
};
inline int lds_opt_in(LdsOptIn& flag, const void* kernel, int lds_bytes) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return MDATTN_E_LAUNCH;
  const uint64_t bit = 1ull << dev;
  if (flag.devices.load(std::memory_order_acquire) & bit) return MDATTN_OK;
  if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes) != hipSuccess) return MDATTN_E_LAUNCH;
  flag.devices.fetch_or(bit, std::memory_order_release);
  return MDATTN_OK;
}

// Schedule forced by mdattn_set_fwd_schedule (0: chosen by shape).
int forced_fwd_schedule();

}  // namespace mdattn
