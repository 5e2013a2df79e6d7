// K4: post-mixing (residual stream mix + post-weighted layer output) and its
// backward.
//
//   forward   out[t,i,c]    = bf16(h_post[t,i] * lo[t,c] + sum_j H[t,i,j] * x[t,j,c])
//   backward  grad_lo[t,c]  = bf16(sum_i h_post[t,i] * go[t,i,c])
//             grad_hp[t,i]  = sum_c go[t,i,c] * lo[t,c]           (fp32)
//             grad_H[t,i,j] = sum_c go[t,i,c] * x[t,j,c]          (fp32)
//             grad_x[t,j,c] = bf16(sum_i H[t,i,j] * go[t,i,c])
//
// Follows src/flash_mhc/kernels.py:384-481 (forward) and :487-665 (fused
// backward) of the reference, written for gfx950: a group of LPT consecutive
// lanes owns one token and streams 16-byte vectors of every row it touches, so
// each input row is read once and each output row written once per launch.
// The backward keeps its 20 per-token partial sums in registers and finishes
// them with an in-wave butterfly (and, when a token spans several waves, an
// LDS sum over them in wave order): no atomics, deterministic.
#include <type_traits>

#include "fmhc_common.h"

namespace fmhc {

namespace {

template <typename WALK>
__global__ __launch_bounds__(block_of<WALK::LPT>()) void k4_fwd_kernel(const uint16_t* __restrict__ x,
                                                        const uint16_t* __restrict__ lo,
                                                        const float* __restrict__ H,
                                                        const float* __restrict__ h_post,
                                                        uint16_t* __restrict__ out,
                                                        int64_t T, int C) {
  constexpr int LPT = WALK::LPT;
  constexpr bool LOOP = WALK::LOOP, WHOLE = WALK::WHOLE;
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t tok = token_of_lane<LPT>(lane);
  if (tok >= T) return;
  const int sub = sub_of_lane<LPT>();
  const int ng = C / 8;

  float h[4][4], p[4];
  {
    const float* Ht = H + tok * 16;
    const float* pt = h_post + tok * 4;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      p[i] = pt[i];
#pragma unroll
      for (int j = 0; j < 4; ++j) h[i][j] = Ht[i * 4 + j];
    }
  }
  const uint16_t* xr[4];
  uint16_t* orow[4];
  xr[0] = x + tok * 4 * C;
  orow[0] = out + tok * 4 * C;
#pragma unroll
  for (int j = 1; j < 4; ++j) {
    xr[j] = xr[j - 1] + C;
    orow[j] = orow[j - 1] + C;
  }
  const uint16_t* lrow = lo + tok * C;

  auto mix = [&](auto vec, int g) __attribute__((always_inline)) {
    constexpr int VEC = decltype(vec)::value;
    float l[VEC], xv[4][VEC];
    Lanes<VEC, WHOLE>::load(lrow, g, l);
#pragma unroll
    for (int j = 0; j < 4; ++j) Lanes<VEC, WHOLE>::load(xr[j], g, xv[j]);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float o[VEC];
#pragma unroll
      for (int e = 0; e < VEC; ++e) {
        float acc = p[i] * l[e];
#pragma unroll
        for (int j = 0; j < 4; ++j) acc = __builtin_fmaf(h[i][j], xv[j][e], acc);
        o[e] = acc;
      }
      Lanes<VEC, WHOLE>::store(orow[i], g, o);
    }
  };
  if constexpr (!LOOP) {
    if (sub < ng) mix(Vec<8>{}, sub);
  } else {
#pragma unroll 2
    for (int g = sub; g < ng; g += LPT) mix(Vec<8>{}, g);
  }
  row_tail<WHOLE>(C, sub, [&](int c) { mix(Vec<1>{}, c); });
}

template <typename WALK, bool EARLY>
__global__ __launch_bounds__(block_of<WALK::LPT>()) void k4_bwd_kernel(const uint16_t* __restrict__ x,
                                                        const uint16_t* __restrict__ lo,
                                                        const float* __restrict__ H,
                                                        const float* __restrict__ h_post,
                                                        const uint16_t* __restrict__ go,
                                                        uint16_t* __restrict__ grad_x,
                                                        uint16_t* __restrict__ grad_lo,
                                                        float* __restrict__ grad_H,
                                                        float* __restrict__ grad_hp,
                                                        int64_t T, int C) {
  constexpr int LPT = WALK::LPT;
  constexpr bool LOOP = WALK::LOOP, WHOLE = WALK::WHOLE;
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

  float shp[4] = {0.f, 0.f, 0.f, 0.f};
  float sH[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) sH[i][j] = 0.f;

  if (live) {
  float h[4][4], p[4];
  {
    const float* Ht = H + tok * 16;
    const float* pt = h_post + tok * 4;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      p[i] = pt[i];
#pragma unroll
      for (int j = 0; j < 4; ++j) h[i][j] = Ht[i * 4 + j];
    }
  }
  const uint16_t* xr[4];
  const uint16_t* gr[4];
  uint16_t* gxr[4];
  xr[0] = x + tok * 4 * C;
  gr[0] = go + tok * 4 * C;
  gxr[0] = grad_x + tok * 4 * C;
#pragma unroll
  for (int j = 1; j < 4; ++j) {
    xr[j] = xr[j - 1] + C;
    gr[j] = gr[j - 1] + C;
    gxr[j] = gxr[j - 1] + C;
  }
  const uint16_t* lrow = lo + tok * C;
  uint16_t* glrow = grad_lo + tok * C;

  auto round = [&](auto vec, int g) __attribute__((always_inline)) {
    constexpr int VEC = decltype(vec)::value;
    float q[4][VEC], l[VEC];
#pragma unroll
    for (int i = 0; i < 4; ++i) Lanes<VEC, WHOLE>::load(gr[i], g, q[i]);
    Lanes<VEC, WHOLE>::load(lrow, g, l);

    // EARLY: the iteration's x rows load with grad_out and lo, before its
    // first store (the compiler keeps a load behind an earlier store).
    float xs[EARLY ? 4 : 1][VEC];
    if constexpr (EARLY) {
#pragma unroll
      for (int j = 0; j < 4; ++j) Lanes<VEC, WHOLE>::load(xr[j], g, xs[j]);
    }
    // grad_lo and the grad_h_post partial sums.
    {
      float o[VEC];
#pragma unroll
      for (int e = 0; e < VEC; ++e) {
        float acc = p[0] * q[0][e];
        acc = __builtin_fmaf(p[1], q[1][e], acc);
        acc = __builtin_fmaf(p[2], q[2][e], acc);
        o[e] = __builtin_fmaf(p[3], q[3][e], acc);
      }
      Lanes<VEC, WHOLE>::store(glrow, g, o);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int e = 0; e < VEC; ++e) shp[i] = __builtin_fmaf(q[i][e], l[e], shp[i]);
    }

    // One x stream at a time: grad_H partial sums and grad_x.
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float xl[VEC], o[VEC];
      const float* xv = xl;
      if constexpr (EARLY)
        xv = xs[j];
      else
        Lanes<VEC, WHOLE>::load(xr[j], g, xl);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int e = 0; e < VEC; ++e) sH[i][j] = __builtin_fmaf(q[i][e], xv[e], sH[i][j]);
#pragma unroll
      for (int e = 0; e < VEC; ++e) {
        float acc = h[0][j] * q[0][e];
        acc = __builtin_fmaf(h[1][j], q[1][e], acc);
        acc = __builtin_fmaf(h[2][j], q[2][e], acc);
        o[e] = __builtin_fmaf(h[3][j], q[3][e], acc);
      }
      Lanes<VEC, WHOLE>::store(gxr[j], g, o);
    }
  };
  if constexpr (!LOOP) {
    if (sub < ng) round(Vec<8>{}, sub);
  } else {
#pragma unroll 2
    for (int g = sub; g < ng; g += LPT) round(Vec<8>{}, g);
  }
  row_tail<WHOLE>(C, sub, [&](int c) { round(Vec<1>{}, c); });
  }

  constexpr int GS = LPT < kWave ? LPT : kWave;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    shp[i] = group_sum<GS>(shp[i]);
#pragma unroll
    for (int j = 0; j < 4; ++j) sH[i][j] = group_sum<GS>(sH[i][j]);
  }
  if constexpr (WPT > 1) {
    // The token's waves add their 20 sums in wave order (deterministic).
    __shared__ float red[block_of<LPT>() / kWave][20];
    const int wave = static_cast<int>(threadIdx.x) >> 6;
    if (lane == 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        red[wave][16 + i] = shp[i];
#pragma unroll
        for (int j = 0; j < 4; ++j) red[wave][i * 4 + j] = sH[i][j];
      }
    }
    __syncthreads();
    if (live && sub == 0) {
      float t[20];
#pragma unroll
      for (int k = 0; k < 20; ++k) t[k] = 0.f;
#pragma unroll
      for (int w = 0; w < WPT; ++w)
#pragma unroll
        for (int k = 0; k < 20; ++k) t[k] += red[wave + w][k];
      float* dH = grad_H + tok * 16;
      float* dp = grad_hp + tok * 4;
#pragma unroll
      for (int k = 0; k < 16; ++k) dH[k] = t[k];
#pragma unroll
      for (int i = 0; i < 4; ++i) dp[i] = t[16 + i];
    }
  } else if (sub == 0) {
    float* dH = grad_H + tok * 16;
    float* dp = grad_hp + tok * 4;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      dp[i] = shp[i];
#pragma unroll
      for (int j = 0; j < 4; ++j) dH[i * 4 + j] = sH[i][j];
    }
  }
}

int launch_k4_fwd(const uint16_t* x, const uint16_t* lo, const float* H, const float* hp,
                  uint16_t* out, int64_t T, int C, hipStream_t s) {
  with_row_walk(C, aligned16(x) && aligned16(lo) && aligned16(out), [&](auto w) {
    constexpr int L = decltype(w)::LPT;
    // Tokens narrower than a wave are faster in the loop's schedule (T = 65536,
    // C = 176 42.7 -> 36.5 us, 256 50.5 -> 48.6); wider ones equal or slower.
    using Walk = RowWalk<L, decltype(w)::LOOP || L < kWave, decltype(w)::WHOLE>;
    // Residency cap (fmhc_common.h).
    static const unsigned own = own_lds(reinterpret_cast<const void*>(&k4_fwd_kernel<Walk>));
    for_launches(T, block_of<L>(), tokens_per_block(L), [&](int64_t t, int64_t n) {
      const dim3 grid(blocks_for(n, tokens_per_block(L)));
      unsigned lds = 0;
      if (decltype(w)::LOOP)
        lds = grid.x >= kCapMinBlocks ? kLdsCapFive : 0u;
      else
        lds = cap_lds(own, grid.x, block_of<L>(), L, C / 8, Walk::CAP);
      k4_fwd_kernel<Walk><<<grid, block_of<L>(), FMHC_LDS_CAP ? lds : 0u, s>>>(
          x + t * 4 * C, lo + t * C, H + t * 16, hp + t * 4, out + t * 4 * C, n, C);
    });
  });
  return launch_status();
}

constexpr int64_t kK4EarlyLanes = int64_t{16384} * 64;

int launch_k4_bwd(const uint16_t* x, const uint16_t* lo, const float* H, const float* hp,
                  const uint16_t* go, uint16_t* gx, uint16_t* glo, float* gH, float* ghp,
                  int64_t T, int C, hipStream_t s) {
  const bool aligned = aligned16(x) && aligned16(lo) && aligned16(go) && aligned16(gx) && aligned16(glo);
  with_row_walk(C, aligned, [&](auto w) {
    using Walk = decltype(w);
    constexpr int L = Walk::LPT;
    auto launch = [&](auto walk, auto early) {
      using W = decltype(walk);
      constexpr bool E = decltype(early)::value;
      // Residency cap (fmhc_common.h) with one group per lane, up to 256 lanes
      // (T = 30000, C = 3000 440 us with and without).
      static const unsigned own = own_lds(reinterpret_cast<const void*>(&k4_bwd_kernel<W, E>));
      for_launches(T, block_of<L>(), tokens_per_block(L), [&](int64_t t, int64_t n) {
        const dim3 grid(blocks_for(n, tokens_per_block(L)));
        unsigned lds = 0;
        if (FMHC_LDS_CAP && C / 8 <= L && L <= 256) lds = cap_lds(own, grid.x, block_of<L>(), L, C / 8, Walk::CAP);
        k4_bwd_kernel<W, E><<<grid, block_of<L>(), lds, s>>>(
            x + t * 4 * C, lo + t * C, H + t * 16, hp + t * 4, go + t * 4 * C, gx + t * 4 * C, glo + t * C,
            gH + t * 16, ghp + t * 4, n, C);
      });
    };
    // EARLY: all of a lane's loads go out before its first store, so a wave
    // waits for one round trip instead of five, but holds more registers and
    // leaves its stores to the end.  Few waves (up to 64 per CU) and unaligned
    // rows take it (T = 1000, C = 2560 15.6 us, in the plain order 16.4; T = 1024,
    // C = 1024 8.1 / 8.3; T = 30011, C = 1001 151 / 157); many waves are faster
    // in the plain order, as the loop over groups schedules it even for one
    // group per lane (T = 65536, C = 1000 322 -> 307 us, 1024 304 -> 299, 2048
    // 618 -> 599; T = 65537, C = 2560 765 -> 756).  Tokens narrower than a wave
    // keep the coefficients in vector registers and the plain order.
    if constexpr (L < kWave)
      launch(w, std::false_type{});
    else if (!Walk::WHOLE || T * L <= kK4EarlyLanes)
      launch(w, std::true_type{});
    else
      launch(RowWalk<L, true, Walk::WHOLE>{}, std::false_type{});
  });
  return launch_status();
}

bool bad_sizes(int64_t T, int64_t C, int64_t n) {
  return T < 0 || C <= 0 || C > (int64_t{1} << 30) || n != 4;
}

}  // namespace
}  // namespace fmhc

extern "C" int fmhc_k4_fwd(const uint16_t* x, const uint16_t* lo, const float* H,
                           const float* h_post, uint16_t* out, int64_t T, int64_t C, int64_t n,
                           void* stream) {
  using namespace fmhc;
  if (bad_sizes(T, C, n)) return FMHC_ERR_INVALID_ARGUMENT;
  if (T == 0) return FMHC_OK;
  if (!x || !lo || !H || !h_post || !out) return FMHC_ERR_INVALID_ARGUMENT;
  hipStream_t s = static_cast<hipStream_t>(stream);
  return launch_k4_fwd(x, lo, H, h_post, out, T, static_cast<int>(C), s);
}

extern "C" int fmhc_k4_bwd(const uint16_t* x, const uint16_t* lo, const float* H,
                           const float* h_post, const uint16_t* grad_out, uint16_t* grad_x,
                           uint16_t* grad_lo, float* grad_H, float* grad_h_post, int64_t T,
                           int64_t C, int64_t n, void* stream) {
  using namespace fmhc;
  if (bad_sizes(T, C, n)) return FMHC_ERR_INVALID_ARGUMENT;
  if (T == 0) return FMHC_OK;
  if (!x || !lo || !H || !h_post || !grad_out || !grad_x || !grad_lo || !grad_H || !grad_h_post)
    return FMHC_ERR_INVALID_ARGUMENT;
  hipStream_t s = static_cast<hipStream_t>(stream);
  return launch_k4_bwd(x, lo, H, h_post, grad_out, grad_x, grad_lo, grad_H, grad_h_post, T, static_cast<int>(C),
                       s);
}
