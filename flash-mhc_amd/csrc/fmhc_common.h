// Shared device helpers for the mHC-lite K1/K3/K4 HIP kernels (gfx950, wave64).
//
// Data conventions used by every kernel in this library:
//   * bf16 tensors arrive as uint16_t bit patterns, row-major and contiguous.
//   * fp32 accumulation everywhere; every bf16 output is rounded exactly once,
//     round-to-nearest-even, by the hardware v_cvt_pk_bf16_f32 conversion.
//   * A lane moves 16 bytes (8 bf16) per memory instruction, at any 2-byte
//     alignment; the up to 7 last elements of a row with C % 8 != 0 are moved
//     one per lane.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "../../include/flash_mhc_hip.h"

namespace fmhc {

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

constexpr int kWave = 64;

// 16 (8) bytes at any address that is a multiple of 2: gfx950 moves unaligned
// vectors in one instruction, so odd widths and operands off 16-byte
// alignment take the same kernels as aligned ones (the code for an aligned
// and an unaligned vector is the same global_load_dwordx4).
typedef unsigned int u32x4_any __attribute__((ext_vector_type(4), aligned(2)));
typedef unsigned int u32x2_any __attribute__((ext_vector_type(2), aligned(2)));
typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));

__device__ __forceinline__ u32x4 ld16(const void* p) { return *static_cast<const u32x4_any*>(p); }
__device__ __forceinline__ void st16(void* p, u32x4 v) { *static_cast<u32x4_any*>(p) = v; }
__device__ __forceinline__ f32x4 ld16f(const void* p) { return *static_cast<const f32x4_any*>(p); }

// Streaming loads/stores.  Data that is read or written exactly once per
// launch carries the nontemporal hint so it does not evict the small,
// reused operands (W, coefficients) from the caches.
#ifndef FMHC_NT_LOADS
#define FMHC_NT_LOADS 1
#endif
#ifndef FMHC_NT_STORES
#define FMHC_NT_STORES 1
#endif

template <typename V>
__device__ __forceinline__ V ld_stream(const V* p) {
#if FMHC_NT_LOADS
  return __builtin_nontemporal_load(p);
#else
  return *p;
#endif
}

template <typename V>
__device__ __forceinline__ void st_stream(V* p, V v) {
#if FMHC_NT_STORES
  __builtin_nontemporal_store(v, p);
#else
  *p = v;
#endif
}

__device__ __forceinline__ u32x4 ld16_stream(const void* p) {
#if FMHC_NT_LOADS
  return __builtin_nontemporal_load(static_cast<const u32x4_any*>(p));
#else
  return ld16(p);
#endif
}

__device__ __forceinline__ void st16_stream(void* p, u32x4 v) {
#if FMHC_NT_STORES
  __builtin_nontemporal_store(v, static_cast<u32x4_any*>(p));
#else
  st16(p, v);
#endif
}

__device__ __forceinline__ void st8_stream(void* p, u32x2 v) {
#if FMHC_NT_STORES
  __builtin_nontemporal_store(v, static_cast<u32x2_any*>(p));
#else
  *static_cast<u32x2_any*>(p) = v;
#endif
}

// Loads carry the hint at every size.  Without it launches that read up to 80
// MiB were faster where the same few tensors came round again and stayed in the
// memory-side cache (hint / none, us: forward of T = 1003, C = 2560 51.9 / 50.3,
// training step of T = 4096, C = 1024 163 / 160 replayed on one state), and
// slower on new tensors and inside a stack of blocks: T = 8192, C = 1024 K1
// forward 18.4 / 18.9, K3 forward 15.9 / 16.5, K3 backward 25.9 / 26.8, K4
// forward 25.6 / 26.6, K1 forward then backward 54.5 / 58.8; forward of T = 8192
// 77 / 80; per block of six in a captured training step T = 8192 261 / 268, T =
// 4096 155 / 158, T = 16384, C = 512 285 / 302, T = 1003, C = 2560 163 / 166, in
// an eval forward T = 8192 72.8 / 71.9, the others within 1%.  Kernels that read
// again what the launch before them or their own first pass has read take
// ordinary loads (premap.hip, k1.hip).

// bf16 bit pattern -> fp32 (exact).
__device__ __forceinline__ float bf_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
__device__ __forceinline__ float bf16_to_f32(uint16_t h) {
  return __uint_as_float(static_cast<uint32_t>(h) << 16);
}

// Two fp32 -> packed bf16 pair, round-to-nearest-even (v_cvt_pk_bf16_f32).
__device__ __forceinline__ uint32_t pack_bf16x2(float a, float b) {
  bf16x2 r = {static_cast<__bf16>(a), static_cast<__bf16>(b)};
  return __builtin_bit_cast(uint32_t, r);
}
__device__ __forceinline__ uint16_t f32_to_bf16(float a) {
  return __builtin_bit_cast(uint16_t, static_cast<__bf16>(a));
}

__device__ __forceinline__ void unpack8(const u32x4 v, float f[8]) {
  f[0] = bf_lo(v.x); f[1] = bf_hi(v.x);
  f[2] = bf_lo(v.y); f[3] = bf_hi(v.y);
  f[4] = bf_lo(v.z); f[5] = bf_hi(v.z);
  f[6] = bf_lo(v.w); f[7] = bf_hi(v.w);
}

__device__ __forceinline__ u32x4 pack8(const float f[8]) {
  u32x4 v;
  v.x = pack_bf16x2(f[0], f[1]);
  v.y = pack_bf16x2(f[2], f[3]);
  v.z = pack_bf16x2(f[4], f[5]);
  v.w = pack_bf16x2(f[6], f[7]);
  return v;
}

// Element group moved by one lane per step: VEC = 8 (one 16-byte vector) or,
// for the elements past a row's last whole group, VEC = 1 (one bf16 scalar).  `idx` counts groups, so the element offset is
// idx * VEC.  raw() issues the load and keeps the packed bf16 bits; unpack()
// widens them to fp32; load() does both.  NT: with the nontemporal hint.
template <int VEC, bool NT>
struct Lanes;
template <int VEC>
using Vec = std::integral_constant<int, VEC>;

template <bool NT>
struct Lanes<8, NT> {
  using Raw = u32x4;
  __device__ static __forceinline__ Raw raw(const uint16_t* __restrict__ row, int idx) {
    return NT ? ld16_stream(row + 8 * idx) : ld16(row + 8 * idx);
  }
  __device__ static __forceinline__ void unpack(const Raw v, float f[8]) { unpack8(v, f); }
  __device__ static __forceinline__ void load(const uint16_t* __restrict__ row, int idx, float f[8]) {
    unpack8(raw(row, idx), f);
  }
  __device__ static __forceinline__ void store(uint16_t* __restrict__ row, int idx, const float f[8]) {
    if constexpr (NT)
      st16_stream(row + 8 * idx, pack8(f));
    else
      st16(row + 8 * idx, pack8(f));
  }
};

template <bool NT>
struct Lanes<1, NT> {
  __device__ static __forceinline__ void load(const uint16_t* __restrict__ row, int idx, float f[1]) {
    f[0] = bf16_to_f32(row[idx]);
  }
  __device__ static __forceinline__ void store(uint16_t* __restrict__ row, int idx, const float f[1]) {
    row[idx] = f32_to_bf16(f[0]);
  }
};

// The elements past a row's last whole group of 8 (at most 7), one per lane:
// f(idx) in lane `first` of the row's lanes (8 or more).  WHOLE: there are
// none (C % 8 == 0), and the kernel carries no code for them.
template <bool WHOLE, typename F>
__device__ __forceinline__ void row_tail(int C, int first, F&& f) {
  if constexpr (!WHOLE) {
    const int c = (C & ~7) + first;
    if (c < C) f(c);
  }
}

// K3 forward of one element group of a token: out[c] = bf16(h0 x0[c] +
// h1 x1[c] + h2 x2[c] + h3 x3[c]), the products added in stream order with
// fused multiply-adds.  Shared by the K3 kernel and the pre-map's kernels,
// which must agree bit for bit.
// NT: x with the nontemporal hint; WHOLE: the output with it (rows of whole,
// aligned groups), and rows have no tail.
template <int VEC, bool WHOLE, bool NT = WHOLE>
__device__ __forceinline__ void k3_mix(const uint16_t* __restrict__ x0, const float h[4], uint16_t* __restrict__ orow,
                                       int g, int C) {
  const uint16_t* x1 = x0 + C;
  const uint16_t* x2 = x1 + C;
  const uint16_t* x3 = x2 + C;
  float a[VEC], b[VEC], c[VEC], d[VEC], o[VEC];
  Lanes<VEC, NT>::load(x0, g, a);
  Lanes<VEC, NT>::load(x1, g, b);
  Lanes<VEC, NT>::load(x2, g, c);
  Lanes<VEC, NT>::load(x3, g, d);
#pragma unroll
  for (int e = 0; e < VEC; ++e) {
    float acc = h[0] * a[e];
    acc = __builtin_fmaf(h[1], b[e], acc);
    acc = __builtin_fmaf(h[2], c[e], acc);
    o[e] = __builtin_fmaf(h[3], d[e], acc);
  }
  Lanes<VEC, WHOLE>::store(orow, g, o);
}

// A whole token: groups first, first + step, ... below C / 8, then the tail.
template <bool WHOLE, bool NT = WHOLE>
__device__ __forceinline__ void k3_token(const uint16_t* __restrict__ x0, const float h[4],
                                         uint16_t* __restrict__ orow, int first, int step, int C) {
  const int ng = C / 8;
#pragma unroll 2
  for (int g = first; g < ng; g += step) k3_mix<8, WHOLE, NT>(x0, h, orow, g, C);
  row_tail<WHOLE>(C, first, [&](int c) { k3_mix<1, WHOLE, NT>(x0, h, orow, c, C); });
}

// Residency caps.  K3's and K4's kernels use a few dozen VGPRs, so eight
// 4-wave workgroups could share a CU; they run faster with fewer, from 16
// workgroups per CU on (below, a cap adds a round of workgroups).  The host's
// launch reserves LDS the kernel does not use (cap_lds).  With one 16-byte
// group per lane the best residency found is about kCapLanes lanes with work
// per CU, 10 to 12 waves.  Swept over 0, 16, 20, ... 64 KiB per workgroup (us,
// no cap against this one): T = 65536, C = 1000 K3 forward 110 against 104,
// K3 backward 222 / 195, K4 forward 221 / 197, K4 backward 342 / 314; C = 1024
// 112 / 106, 190 / 189, 194 / 187, 303 / 298; C = 2048 222 / 210, 398 / 382,
// 398 / 378, 629 / 601; T = 32768, C = 2560 142 / 132, 247 / 236, 246 / 238,
// 374 / 374; T = 60000, C = 520 (65 of 128 lanes) K3 backward 105 / 97, K4
// backward 165 / 160.  K3 forward with a quarter of the lanes idle or more
// loses with any cap (C = 520 52 -> 54, 712 35 -> 37) and takes none.
// With several groups per lane (kLoopLpt): K3 forward six workgroups per CU
// (T = 262144, C = 4096 5.60-5.67 -> 5.88-5.93 TB/s), K4 forward five, the
// backwards none (K3 backward there 5.57 -> 5.35-5.41 with five).
// K1's backward dx likewise runs faster with one workgroup per CU (k1.hip).
#ifndef FMHC_LDS_CAP
#define FMHC_LDS_CAP 1
#endif
constexpr unsigned kLdsCapSix = 24 * 1024;
constexpr unsigned kLdsCapFive = 32 * 1024;
// One workgroup per CU (K1 backward dx, k1.hip).
constexpr unsigned kLdsCapOne = 96 * 1024;
constexpr unsigned kLdsPerCu = 160 * 1024;

// The reserve `dyn` for `kernel` if the kernel's own LDS plus dyn fit in a
// CU's LDS, else 0 (no cap): a launch asking for more LDS than the CU holds
// is not refused, and faults.  Callers keep the result in a static of the
// launch site's kernel instantiation.
inline unsigned lds_reserve(const void* kernel, unsigned dyn) {
  hipFuncAttributes a;
  if (dyn == 0 || hipFuncGetAttributes(&a, kernel) != hipSuccess) return 0u;
  return a.sharedSizeBytes + dyn <= kLdsPerCu ? dyn : 0u;
}

constexpr int kCapLanes = 680;
// Unaligned groups keep more waves in flight.  No cap against this one, us, K3
// backward, K4 forward: T = 30011, C = 1001 102 / 94, 104 / 97; T = 50000, C = 700
// off 16 bytes 122 / 119, 120 / 118; T = 40000, C = 777 105 / 100, 104 / 99, 900
// off 16 bytes 126 / 119, 123 / 118; T = 20011, C = 1535 107 / 100, 105 / 99; T =
// 16000, C = 2049 111 / 106, 109 / 106; T = 65536, C = 513 115 / 108, 117 / 108;
// C = 521, 601 (half the lanes idle) equal.  K4 backward is within 1.5%
// either way (C = 513 184 / 178).  680 lanes lost at C = 700 (137, 134).  K3
// forward takes none (C = 1001 alone 52 against 55).
constexpr int kCapLanesUnaligned = 1150;
constexpr unsigned kCapMinBlocks = 16u * 256u;

// A kernel's own LDS; callers keep it in a static of the launch site's
// instantiation.
inline unsigned own_lds(const void* kernel) {
  hipFuncAttributes a;
  return hipFuncGetAttributes(&a, kernel) == hipSuccess ? static_cast<unsigned>(a.sharedSizeBytes) : kLdsPerCu;
}

// The LDS reserve that leaves about `lanes` lanes with work resident on a CU, for
// `blocks` workgroups of a kernel with `own` bytes of LDS and `block` threads,
// lpt lanes per token and `groups` groups per row.  1280 bytes stay free per
// workgroup, the granularity of an allocation.
inline unsigned cap_lds(unsigned own, unsigned blocks, int block, int lpt, int groups, int lanes) {
  if (blocks < kCapMinBlocks || lpt < kWave) return 0u;
  const int busy = block * groups / lpt;  // lanes with work in a workgroup
  const int n = busy > 0 ? (lanes + busy / 2) / busy : 0;
  if (n < 1 || n >= 8) return 0u;
  const unsigned each = kLdsPerCu / static_cast<unsigned>(n);
  return each > own + 1280u ? each - own - 1280u : 0u;
}

// Sum over the wave's 64 lanes, every lane receiving the total, with the
// pairs of group_sum<64>'s butterfly (lanes 32 apart first, then 16, 8, 4,
// 2, 1), so the same bits, on the VALU's cross-lane moves instead of LDS
// permutes.  Lanes 32 apart (v_permlane32_swap, which exchanges the two
// halves of its operands) and 16 apart (v_permlane16_swap: odd rows of one
// operand with even rows of the other); every 16-lane row then holds the same
// values, so a rotation by 8 within the row pairs lane j with j ^ 8, and, the
// values now repeating every 8 lanes, a rotation by 4 pairs j with a lane
// holding j ^ 4's value; quad permutations pair j ^ 2 and j ^ 1.  Every lane
// of the wave must be active.
__device__ __forceinline__ float wave_sum(float v) {
  const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(h[0]) + __uint_as_float(h[1]);
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  // DPP controls: row_ror:8, row_ror:4, quad_perm [2,3,0,1], quad_perm [1,0,3,2].
  v += __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(v), 0x128, 0xf, 0xf, false));
  v += __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(v), 0x124, 0xf, 0xf, false));
  v += __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(v), 0x4e, 0xf, 0xf, false));
  v += __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(v), 0xb1, 0xf, 0xf, false));
  return v;
}

// Sum over the four lanes 16 apart (one per 16-lane row), in the order of the
// two shuffle steps v += v[lane ^ 16]; v += v[lane ^ 32]: v_permlane16_swap
// pairs each row with its neighbour, v_permlane32_swap the two halves.  Every
// lane of the wave must be active.
__device__ __forceinline__ float rows_sum(float v) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(h[0]) + __uint_as_float(h[1]);
}

// Sum over each 16-lane row, every lane of the row receiving the total: the
// butterfly lanes 1, 2, 4, 8 apart.  Quad permutations pair lane ^ 1 and
// lane ^ 2; the half-row mirror (lane j with 7 - j within each 8) then pairs
// the same values as lane ^ 4, since every quad holds one value by then, and
// the row mirror (j with 15 - j) those of lane ^ 8.  All 16 lanes of a row
// must be active.
__device__ __forceinline__ float row16_sum(float v) {
  // DPP controls: quad_perm [1,0,3,2], quad_perm [2,3,0,1], row_half_mirror, row_mirror.
  v += __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(v), 0xb1, 0xf, 0xf, false));
  v += __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(v), 0x4e, 0xf, 0xf, false));
  v += __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(v), 0x141, 0xf, 0xf, false));
  v += __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(v), 0x140, 0xf, 0xf, false));
  return v;
}

// Slice order of the per-token stream sums s_j = sum_c x[t, j, c] g[t, c]
// (K3's grad_h_pre) for rows with C a multiple of 128, shared by every kernel
// that produces them, so that each gives the same bits however it splits a
// row: each 8-element group's products as an FMA chain from zero, row16_sum
// over the 16 groups of each 128-column slice, then the C / 128 slice sums
// added in slice order (the first one taken as is).
constexpr int kSliceCols = 128;
constexpr int kMaxSlices = 64;  // C up to 8192 per stream
constexpr int kCanonRounds = 4;  // 16-byte groups per lane

// The slice order applies to a K3-backward layout of lpt lanes per token with
// 16-byte groups: C a multiple of 128, at most kMaxSlices slices, at least 16
// lanes per token and at most kCanonRounds groups per lane.
inline bool k3_canon(int64_t C, int lpt) {
  return C % kSliceCols == 0 && C / kSliceCols <= kMaxSlices && lpt >= 16 && C / 8 <= int64_t{kCanonRounds} * lpt;
}

// One round of a token held by LPT aligned lanes (16 <= LPT <= 64) whose lane
// sub holds group sub + k LPT of the row: e[j] is that group's FMA chain
// (zero past the row).  Adds slices k LPT / 16 ... of the round to s[j], in
// slice order; ns = C / 128.  Every lane of the token must be active.
template <int LPT>
__device__ __forceinline__ void slice_sums_add(float (&e)[4], float (&s)[4], int k, int ns, int lane) {
  static_assert(LPT >= 16 && LPT <= 64, "rows of 16 lanes within one wave");
#pragma unroll
  for (int j = 0; j < 4; ++j) e[j] = row16_sum(e[j]);
  const int tb = lane & ~(LPT - 1);
#pragma unroll
  for (int r = 0; r < LPT / 16; ++r) {
    const int sigma = k * (LPT / 16) + r;
    if (sigma < ns) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        // A whole wave per token: the row's sum is read as a scalar (no LDS).
        const float p = LPT == kWave ? __int_as_float(__builtin_amdgcn_readlane(__float_as_int(e[j]), 16 * r))
                                     : __shfl(e[j], tb + 16 * r, kWave);
        s[j] = sigma == 0 ? p : s[j] + p;
      }
    }
  }
}

// Sum over the LPT consecutive lanes that share one token (LPT a power of
// two <= 64): a butterfly, lanes LPT / 2 apart first.  Every lane of the
// group receives the total.  LPT = 64 runs wave_sum (same bits) and needs
// every lane of the wave active.
template <int LPT>
__device__ __forceinline__ float group_sum(float v) {
  if constexpr (LPT == kWave) {
    return wave_sum(v);
  } else {
#pragma unroll
    for (int m = LPT / 2; m >= 1; m >>= 1) v += __shfl_xor(v, m, kWave);
    return v;
  }
}

// Lanes per token of K3 and K4 for rows of C columns: one 16-byte group per
// lane, rounded up to 8, 16, 32 or whole waves up to kMaxLpt lanes; longer
// rows are walked by kLoopLpt lanes.  With one wave for all widths below 1024,
// and 256 lanes above, the last trip of a lane's loop was nearly empty for many
// widths, and every trip waited for its own loads.  K3 forward / backward, K4
// forward / backward with that rule against this one (and its residency caps),
// us: T = 65536, C = 1000 131 / 258 / 262 / 423 against 103 / 196 / 198 / 307;
// T = 60000, C = 520 79 / 139 / 146 / 249 against 52 / 100 / 100 / 162;
// T = 30000, C = 712 48 / 91 / 93 / 147 against 35 / 64 / 64 / 104, C = 1536
// 80 / 147 / 142 / 237 against 73 / 131 / 131 / 204, C = 3000 168 / 338 / 324 /
// 521 against 141 / 278 / 275 / 440; T = 16384, C = 2056 77 / 118 / 139 / 245
// against 59 / 105 / 107 / 170.  512 lanes lost at C = 4096 (T = 16384 108 /
// 203 / 193 / 315 against 124 / 227 / 206 / 351), which keeps 256 lanes with
// two groups each.
constexpr int kMaxLpt = 448;
constexpr int kLoopLpt = 256;
inline int lanes_per_token(int C) {
  const int groups = C / 8;
  if (groups > kMaxLpt) return kLoopLpt;
  if (groups > 32) return (groups + kWave - 1) / kWave * kWave;
  return groups > 16 ? 32 : groups > 8 ? 16 : 8;
}

constexpr int kBlock = 256;  // threads per workgroup, or one token's lanes where they do not divide it

// Threads per workgroup for LPT lanes per token.
template <int LPT>
constexpr int block_of() {
  return kBlock % LPT == 0 ? kBlock : LPT;
}

// Tokens per workgroup with lpt lanes per token.
inline int64_t tokens_per_block(int lpt) { return kBlock % lpt == 0 ? kBlock / lpt : 1; }

// f(first token, tokens) over pieces of T tokens whose launches, of `block`
// threads for per_block tokens, stay below 2^32 threads, the most a HIP launch
// takes: one piece but for the largest operands (T = 2^25 from C = 520 on, 174
// GB for K3 forward).  Pieces of whole eights of tokens, so that their rows are
// aligned as the operands are.
template <typename F>
void for_launches(int64_t T, int block, int64_t per_block, F&& f) {
  const int64_t most = (((int64_t{1} << 32) - 1) / block * per_block) & ~int64_t{7};
  for (int64_t t = 0; t < T; t += most) f(t, T - t < most ? T - t : most);
}

// How K3 and K4 walk a row, as compile-time constants: LPT lanes per token,
// LOOP: several groups per lane, WHOLE: whole, aligned groups, loaded and
// stored with the nontemporal hint.
template <int kLpt, bool kLoop, bool kWhole>
struct RowWalk {
  static constexpr int LPT = kLpt;
  static constexpr bool LOOP = kLoop;
  static constexpr bool WHOLE = kWhole;
  static constexpr int CAP = WHOLE ? kCapLanes : kCapLanesUnaligned;  // lanes of cap_lds
};

// f(RowWalk) for rows of C columns whose 16-byte groups are aligned or not.
// Unaligned groups (C % 8 != 0, or a base address off 16 bytes) leave out the
// nontemporal hint: neighbouring lanes' groups share lines, and the hint
// makes each access fetch or write its part on its own (K3 forward / backward,
// K4 forward / backward with the hint against without, us: T = 65536, C = 100
// 17.5 / 32.0 / 32.5 / 53.4 against 11.8 / 24.0 / 24.7 / 45.1; T = 20011,
// C = 300 14.3 / 24.0 / 23.8 / 42.5 against 12.1 / 19.3 / 19.9 / 38.3).
template <typename F>
void with_row_walk(int C, bool aligned, F&& f) {
  auto pick = [&](auto whole) {
    constexpr bool WHOLE = decltype(whole)::value;
    const int lpt = lanes_per_token(C);
    if (C / 8 > lpt) return f(RowWalk<kLoopLpt, true, WHOLE>{});
    switch (lpt) {
      case 448: return f(RowWalk<448, false, WHOLE>{});
      case 384: return f(RowWalk<384, false, WHOLE>{});
      case 320: return f(RowWalk<320, false, WHOLE>{});
      case 256: return f(RowWalk<256, false, WHOLE>{});
      case 192: return f(RowWalk<192, false, WHOLE>{});
      case 128: return f(RowWalk<128, false, WHOLE>{});
      case 64: return f(RowWalk<64, false, WHOLE>{});
      case 32: return f(RowWalk<32, false, WHOLE>{});
      case 16: return f(RowWalk<16, false, WHOLE>{});
      default: return f(RowWalk<8, false, WHOLE>{});
    }
  };
  if (!aligned || C % 8 != 0)
    pick(std::false_type{});
  else
    pick(std::true_type{});
}

// Token of a lane.  LPT <= 64: 64 / LPT tokens per wave; wider: LPT / 64 waves
// per token.
template <int LPT>
__device__ __forceinline__ int64_t token_of_lane(int lane) {
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  if constexpr (LPT > kWave) {
    return static_cast<int64_t>(blockIdx.x) * (block_of<LPT>() / LPT) + wave / (LPT / kWave);
  } else {
    constexpr int TPW = kWave / LPT;
    const int64_t first = (static_cast<int64_t>(blockIdx.x) * (kBlock / kWave) + wave) * TPW;
    return LPT == kWave ? first : first + lane / LPT;
  }
}

// Position of this lane among its token's LPT lanes.
template <int LPT>
__device__ __forceinline__ int sub_of_lane() {
  return static_cast<int>(threadIdx.x) % LPT;
}

// Status helpers shared by the C entry points.
inline int hip_status(hipError_t e) {
  return e == hipSuccess ? FMHC_OK : FMHC_ERR_HIP_BASE + static_cast<int>(e);
}

inline int launch_status() { return hip_status(hipGetLastError()); }

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

inline unsigned int blocks_for(int64_t items, int64_t per_block) {
  return static_cast<unsigned int>((items + per_block - 1) / per_block);
}

}  // namespace fmhc
