// K3: pre-map of the n = 4 residual streams into the layer input, and its
// backward.
//
//   forward   out[t,c]        = bf16(sum_j h_pre[t,j] * x[t,j,c])       j = 0..3 in order
//   backward  grad_x[t,j,c]   = bf16(h_pre[t,j] * go[t,c])
//             grad_h_pre[t,j] = sum_c x[t,j,c] * go[t,c]                 (fp32)
//
// Follows src/flash_mhc/kernels.py:673-717 (forward) and :720-853 (fused
// backward) of the reference, written for gfx950:
//   * a group of LPT consecutive lanes owns one token: a wave64 holds 64 / LPT
//     tokens, or a token spans LPT / 64 waves (lanes_per_token, fmhc_common.h).
//     Each lane moves 16-byte vectors of all four stream rows, so every x row
//     is read once and every output row written once;
//   * the four per-token coefficients are wave-uniform when LPT >= 64 and then
//     live in SGPRs;
//   * the backward's four reductions over C finish with an in-wave butterfly
//     and, when a token spans several waves, an LDS sum over them in wave
//     order (no atomics), so grad_h_pre is deterministic.
#include <type_traits>

#include "fmhc_common.h"

namespace fmhc {

namespace {

template <typename WALK>
__global__ __launch_bounds__(block_of<WALK::LPT>()) void k3_fwd_kernel(const uint16_t* __restrict__ x,
                                                        const float* __restrict__ h_pre,
                                                        uint16_t* __restrict__ out,
                                                        int64_t T, int C) {
  constexpr int LPT = WALK::LPT;
  constexpr bool LOOP = WALK::LOOP, WHOLE = WALK::WHOLE;
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t tok = token_of_lane<LPT>(lane);
  if (tok >= T) return;
  const int sub = sub_of_lane<LPT>();
  const float* hp = h_pre + tok * 4;
  const float h[4] = {hp[0], hp[1], hp[2], hp[3]};
  const uint16_t* x0 = x + tok * 4 * C;
  if constexpr (!LOOP) {
    if (sub < C / 8) k3_mix<8, WHOLE>(x0, h, out + tok * C, sub, C);
    row_tail<WHOLE>(C, sub, [&](int c) { k3_mix<1, WHOLE>(x0, h, out + tok * C, c, C); });
  } else {
    k3_token<WHOLE>(x0, h, out + tok * C, sub, LPT, C);
  }
}

// GX = false: grad_h_pre only (the pre-map backward adds h_pre * go into K1's
// grad_x store instead of writing it here).  CANON (C a multiple of 128, at
// most kMaxSlices slices): grad_h_pre in the slice order of slice_sums_add
// (fmhc_common.h), which the pre-map backward's split kernel reproduces;
// otherwise one FMA chain per lane over its groups and its elements of the
// row's tail, then group_sum.
template <typename WALK, bool GX, bool CANON>
__global__ __launch_bounds__(block_of<WALK::LPT>()) void k3_bwd_kernel(const uint16_t* __restrict__ x,
                                                        const float* __restrict__ h_pre,
                                                        const uint16_t* __restrict__ go,
                                                        uint16_t* __restrict__ grad_x,
                                                        float* __restrict__ grad_h_pre,
                                                        int64_t T, int C) {
  constexpr int LPT = WALK::LPT;
  constexpr bool LOOP = WALK::LOOP, WHOLE = WALK::WHOLE;
  static_assert(!CANON || LPT >= 16, "slice order: whole 16-lane rows");
  constexpr int WPT = LPT > kWave ? LPT / kWave : 1;  // waves per token
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t tok = token_of_lane<LPT>(lane);
  // With several waves per token every wave reaches the barrier below.
  if constexpr (WPT == 1) {
    if (tok >= T) return;
  }
  const bool live = tok < T;
  const int sub = sub_of_lane<LPT>();
  const int ng = C / 8;
  // CANON with several waves per token: the slice sums of each of the
  // workgroup's tokens.
  constexpr bool kSliceLds = CANON && WPT > 1;
  __shared__ float slices_of[kSliceLds ? block_of<LPT>() / LPT : 1]
                            [kSliceLds ? (LOOP ? kMaxSlices : LPT / 16) : 1][4];
  float(*slices)[4] = slices_of[kSliceLds ? static_cast<int>(threadIdx.x) / LPT : 0];

  float s[4] = {0.f, 0.f, 0.f, 0.f};
  if (live) {
  const float* hp = h_pre + tok * 4;
  const float h0 = hp[0], h1 = hp[1], h2 = hp[2], h3 = hp[3];
  const uint16_t* x0 = x + tok * 4 * C;
  const uint16_t* x1 = x0 + C;
  const uint16_t* x2 = x1 + C;
  const uint16_t* x3 = x2 + C;
  const uint16_t* grow = go + tok * C;
  uint16_t* gx0 = grad_x + tok * 4 * C;
  uint16_t* gx1 = gx0 + C;
  uint16_t* gx2 = gx1 + C;
  uint16_t* gx3 = gx2 + C;

  auto round = [&](auto vec, int g, float (&acc)[4]) __attribute__((always_inline)) {
    constexpr int VEC = decltype(vec)::value;
    float q[VEC], a[VEC], b[VEC], c[VEC], d[VEC], o[VEC];
    Lanes<VEC, WHOLE>::load(grow, g, q);
    Lanes<VEC, WHOLE>::load(x0, g, a);
    Lanes<VEC, WHOLE>::load(x1, g, b);
    Lanes<VEC, WHOLE>::load(x2, g, c);
    Lanes<VEC, WHOLE>::load(x3, g, d);
    if constexpr (GX) {
#pragma unroll
      for (int e = 0; e < VEC; ++e) o[e] = h0 * q[e];
      Lanes<VEC, WHOLE>::store(gx0, g, o);
#pragma unroll
      for (int e = 0; e < VEC; ++e) o[e] = h1 * q[e];
      Lanes<VEC, WHOLE>::store(gx1, g, o);
#pragma unroll
      for (int e = 0; e < VEC; ++e) o[e] = h2 * q[e];
      Lanes<VEC, WHOLE>::store(gx2, g, o);
#pragma unroll
      for (int e = 0; e < VEC; ++e) o[e] = h3 * q[e];
      Lanes<VEC, WHOLE>::store(gx3, g, o);
    }
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      acc[0] = __builtin_fmaf(a[e], q[e], acc[0]);
      acc[1] = __builtin_fmaf(b[e], q[e], acc[1]);
      acc[2] = __builtin_fmaf(c[e], q[e], acc[2]);
      acc[3] = __builtin_fmaf(d[e], q[e], acc[3]);
    }
  };
  if constexpr (CANON) {
    // Lane sub takes group sub + k LPT in round k (slice (sub + k LPT) / 16);
    // whole 16-lane rows are inside or past the row.  All rounds' loads
    // first, then the slice sums.
    constexpr int kRounds = !LOOP ? 1 : kCanonRounds;
    const int ns = ng / 16;
    float e[kRounds][4];
#pragma unroll
    for (int k = 0; k < kRounds; ++k) {
#pragma unroll
      for (int j = 0; j < 4; ++j) e[k][j] = 0.f;
      if (sub + k * LPT < ng) round(Vec<8>{}, sub + k * LPT, e[k]);
    }
#pragma unroll
    for (int k = 0; k < kRounds; ++k) {
      if (k * LPT >= ng) break;  // uniform
      if constexpr (WPT == 1) {
        slice_sums_add<LPT>(e[k], s, k, ns, lane);
      } else {
        const int g = sub + k * LPT;
#pragma unroll
        for (int j = 0; j < 4; ++j) e[k][j] = row16_sum(e[k][j]);
        if ((sub & 15) == 0 && g < ng) {
#pragma unroll
          for (int j = 0; j < 4; ++j) slices[g >> 4][j] = e[k][j];
        }
      }
    }
  } else {
    if constexpr (!LOOP) {
      if (sub < ng) round(Vec<8>{}, sub, s);
    } else {
#pragma unroll 2
      for (int g = sub; g < ng; g += LPT) round(Vec<8>{}, g, s);
    }
    row_tail<WHOLE>(C, sub, [&](int c) { round(Vec<1>{}, c, s); });
  }
  }
  if constexpr (!CANON) {
    constexpr int GS = LPT < kWave ? LPT : kWave;
#pragma unroll
    for (int j = 0; j < 4; ++j) s[j] = group_sum<GS>(s[j]);
  }
  if constexpr (WPT > 1) {
    // The token's waves add their sums in wave order (deterministic), or
    // with CANON its slices in slice order.
    __shared__ float red[block_of<LPT>() / kWave][4];
    const int wave = static_cast<int>(threadIdx.x) >> 6;
    if (!CANON && lane == 0) {
#pragma unroll
      for (int j = 0; j < 4; ++j) red[wave][j] = s[j];
    }
    __syncthreads();
    if (live && sub == 0) {
      float t[4] = {0.f, 0.f, 0.f, 0.f};
      if constexpr (CANON) {
        const int ns = ng / 16;
#pragma unroll
        for (int j = 0; j < 4; ++j) t[j] = slices[0][j];
        for (int sg = 1; sg < ns; ++sg)
#pragma unroll
          for (int j = 0; j < 4; ++j) t[j] += slices[sg][j];
      } else {
#pragma unroll
        for (int w = 0; w < WPT; ++w)
#pragma unroll
          for (int k = 0; k < 4; ++k) t[k] += red[wave + w][k];
      }
      float* dst = grad_h_pre + tok * 4;
#pragma unroll
      for (int k = 0; k < 4; ++k) dst[k] = t[k];
    }
  } else if (sub == 0) {
    float* dst = grad_h_pre + tok * 4;
#pragma unroll
    for (int j = 0; j < 4; ++j) dst[j] = s[j];
  }
}

// K3 forward's residency from 16 to 40 workgroups per CU, where fewer resident
// ones leave a longer last round: T = 16384, C = 512 14.5 us, with kCapLanes
// 15.8, with no cap 14.8; T = 24000 20.7 / 22.2 / 21.4; T = 16384, C = 448 13.0 /
// 14.5 / 13.0; T = 12000, C = 1024 20.9 / 21.9 / 21.3; T = 4096, C = 2048 14.6 /
// 15.7 / 14.9, C = 2560 17.9 / 19.5 / 18.0.  From 40 per CU on kCapLanes is equal
// or better (T = 65536, C = 512 54.5 against 55.3).  K3 backward and K4 keep
// kCapLanes there (T = 10000, C = 3000 K4 forward 89.8 against 92.6, C = 1400 K3
// backward 42.7 / 44.7, T = 12000, C = 1000 K4 backward 58.9 / 60.7).
constexpr unsigned kK3FewBlocks = 40u * 256u;
constexpr int kK3FewLanes = 1280;

int launch_k3_fwd(const uint16_t* x, const float* h_pre, uint16_t* out, int64_t T, int C,
                  hipStream_t s) {
  with_row_walk(C, aligned16(x) && aligned16(out), [&](auto w) {
    using Walk = decltype(w);
    constexpr int L = Walk::LPT;
    // Residency cap (fmhc_common.h).
    static const unsigned own = own_lds(reinterpret_cast<const void*>(&k3_fwd_kernel<Walk>));
    for_launches(T, block_of<L>(), tokens_per_block(L), [&](int64_t t, int64_t n) {
      const dim3 grid(blocks_for(n, tokens_per_block(L)));
      unsigned lds = 0;
      if (Walk::LOOP)
        lds = kLdsCapSix;
      else if (Walk::WHOLE && 4 * (C / 8) >= 3 * L)
        lds = cap_lds(own, grid.x, block_of<L>(), L, C / 8, grid.x < kK3FewBlocks ? kK3FewLanes : kCapLanes);
      k3_fwd_kernel<Walk><<<grid, block_of<L>(), FMHC_LDS_CAP ? lds : 0u, s>>>(x + t * 4 * C, h_pre + t * 4,
                                                                              out + t * C, n, C);
    });
  });
  return launch_status();
}

template <bool GX>
int launch_k3_bwd(const uint16_t* x, const float* h_pre, const uint16_t* go, uint16_t* grad_x,
                  float* grad_h_pre, int64_t T, int C, hipStream_t s) {
  const bool canon = k3_canon(C, lanes_per_token(C));
  with_row_walk(C, aligned16(x) && aligned16(go) && aligned16(grad_x), [&](auto w) {
    constexpr int L = decltype(w)::LPT;
    auto launch = [&](auto walk, auto canon_c) {
      using Walk = decltype(walk);
      constexpr bool CANON = decltype(canon_c)::value;
      // Residency cap (fmhc_common.h): with grad_x and one group per lane.
      static const unsigned own = own_lds(reinterpret_cast<const void*>(&k3_bwd_kernel<Walk, GX, CANON>));
      for_launches(T, block_of<L>(), tokens_per_block(L), [&](int64_t t, int64_t n) {
        const dim3 grid(blocks_for(n, tokens_per_block(L)));
        unsigned lds = 0;
        if (GX && FMHC_LDS_CAP && !Walk::LOOP) lds = cap_lds(own, grid.x, block_of<L>(), L, C / 8, Walk::CAP);
        k3_bwd_kernel<Walk, GX, CANON><<<grid, block_of<L>(), lds, s>>>(
            x + t * 4 * C, h_pre + t * 4, go + t * C, GX ? grad_x + t * 4 * C : nullptr, grad_h_pre + t * 4, n, C);
      });
    };
    if constexpr (L >= 16) {
      if (canon) return launch(w, std::true_type{});
    }
    // With grad_x, tokens narrower than a wave are equal or faster in the
    // loop's schedule (T = 65536, C = 100 25.7 -> 23.2 us, C = 250 51.2 -> 49.7,
    // T = 100000, C = 60 24.7 -> 23.3).
    if constexpr (GX && L < kWave)
      launch(RowWalk<L, true, decltype(w)::WHOLE>{}, std::false_type{});
    else
      launch(w, std::false_type{});
  });
  return launch_status();
}

bool bad_sizes(int64_t T, int64_t C, int64_t n) {
  return T < 0 || C <= 0 || C > (int64_t{1} << 30) || n != 4;
}

}  // namespace

}  // namespace fmhc

extern "C" int fmhc_k3_fwd(const uint16_t* x, const float* h_pre, uint16_t* out, int64_t T,
                           int64_t C, int64_t n, void* stream) {
  using namespace fmhc;
  if (bad_sizes(T, C, n)) return FMHC_ERR_INVALID_ARGUMENT;
  if (T == 0) return FMHC_OK;
  if (!x || !h_pre || !out) return FMHC_ERR_INVALID_ARGUMENT;
  hipStream_t s = static_cast<hipStream_t>(stream);
  return launch_k3_fwd(x, h_pre, out, T, static_cast<int>(C), s);
}

extern "C" int fmhc_k3_bwd(const uint16_t* x, const float* h_pre, const uint16_t* grad_out,
                           uint16_t* grad_x, float* grad_h_pre, int64_t T, int64_t C, int64_t n,
                           void* stream) {
  using namespace fmhc;
  if (bad_sizes(T, C, n)) return FMHC_ERR_INVALID_ARGUMENT;
  if (T == 0) return FMHC_OK;
  if (!x || !h_pre || !grad_out || !grad_h_pre) return FMHC_ERR_INVALID_ARGUMENT;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int c = static_cast<int>(C);
  return grad_x ? launch_k3_bwd<true>(x, h_pre, grad_out, grad_x, grad_h_pre, T, c, s)
                : launch_k3_bwd<false>(x, h_pre, grad_out, nullptr, grad_h_pre, T, c, s);  // grad_h_pre only
}
