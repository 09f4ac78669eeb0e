// Correctly rounded square root, reciprocal and quotient for operands in a
// moderate range, and the pair geometry built on them (gfx950).
//
// The compiler's IEEE forms take 15 to 20 instructions each because they
// scale and fix up every float32 operand.  Between pairs of a neighbor list
// the operands are moderate (squared distances, densities, lengths of the
// order of the support), and there one Newton step in fused arithmetic on
// the hardware approximation gives the correctly rounded result: the
// quotient by Markstein's theorem (P. W. Markstein, "Computation of
// elementary functions on the IBM RISC System/6000 processor", IBM J. Res.
// Dev. 34(1), 1990: q + y fma(-b, q, a) with y the rounded 1/b), the
// reciprocal and the square root by comparison with the IEEE forms over
// every float32 in range on this hardware (dsph_near_check: 1.0e9 and 1.6e9
// values, no difference; 4e9 drawn quotients likewise).  So results are the
// same bits, quotients below 2^-100 aside; the kernels that use them test the
// range per group of entries and evaluate the IEEE forms where it does not
// hold.
#pragma once

#include "common.h"

namespace dsph {

// sqrt(x) for x = 0 or 2^-96 <= x <= 2^96 (NaN gives NaN).
__device__ __forceinline__ float sqrt_near(float x) {
  const float y = __builtin_amdgcn_rsqf(fmaxf(x, 0x1p-96f));
  const float g = x * y, h = 0.5f * y;
  return __builtin_fmaf(__builtin_fmaf(-g, g, x), h, g);
}

// 1 / x for 2^-60 <= |x| <= 2^60 from the hardware's approximation y.
__device__ __forceinline__ float rcp_near(float x, float y) {
  return __builtin_fmaf(__builtin_fmaf(-x, y, 1.0f), y, y);
}
__device__ __forceinline__ float rcp_near(float x) { return rcp_near(x, __builtin_amdgcn_rcpf(x)); }

// a / b with y = rcp_near(b), |a| < 2^60.  A quotient below 2^-100 may be one
// ulp off: it shows only in a row whose terms are all that small.  A zero one
// is positive: no sum of terms shows that.
__device__ __forceinline__ float div_near(float a, float b, float y) {
  const float q = a * y;
  return __builtin_fmaf(__builtin_fmaf(-b, q, a), y, q);
}

// Range checks of a group of entries, folded into one maximum and one
// minimum: each takes about two instructions per three operands.
struct NearRange {
  float top = 0.0f;           // largest |operand| (NaN is not counted: it stays NaN)
  uint32_t low = 0xffffffffu;  // smallest nonzero squared distance, as bits - 1
  __device__ __forceinline__ void d2(float v) {
    top = fmaxf(top, v);
    const uint32_t b = __float_as_uint(v) - 1u;
    low = b < low ? b : low;
  }
  __device__ __forceinline__ void operand(float v) { top = fmaxf(top, fabsf(v)); }
  // rcp_near of a divisor that may be out of range (the hardware's
  // reciprocal of zero is infinite)
  __device__ __forceinline__ float divisor(float v) {
    const float y = __builtin_amdgcn_rcpf(v);
    top = fmaxf(fmaxf(top, fabsf(v)), fabsf(y));
    return rcp_near(v, y);
  }
  __device__ __forceinline__ bool odd() const { return !(top < 0x1p58f) || low < 0x0f800000u - 1u; }  // 2^-96
};

// Whether a list's kernels may take the forms above: one uniform, moderate
// support, and the viscosity's denominator term eps h^2 (when used) away from
// zero.
inline bool near_support(const PairsDev& P) {
  return !P.qh && !P.rh && P.h0 >= 0x1p-40f && P.h0 <= 0x1p40f;
}

// pair_geom for a min-image offset already formed, without W.
__device__ __forceinline__ Geom pair_geom_near(float dx, float dy, float h, const KConst& k, NearRange& range) {
  Geom g;
  g.dx = dx;
  g.dy = dy;
  const float d2 = dist2_exact(dx, dy);
  range.d2(d2);
  g.r = sqrt_near(d2);
  g.h = h;
  g.q = g.r * k.ih;
  g.ri = rcp_near(g.r + 1e-7f);
  g.ex = dx * g.ri;
  g.ey = dy * g.ri;
  g.dw = wendland_dw(g.q, k);
  g.gx = g.ex * g.dw;
  g.gy = g.ey * g.dw;
  return g;
}

// Min-image offsets of a group of U pairs: mod_offset only when a lane of
// the wave has an offset beyond half the period (it returns the others
// unchanged).
template <int U>
__device__ __forceinline__ void wrap_offsets(float (&dx)[U], float (&dy)[U], const Dom& d) {
  float mx = 0.0f, my = 0.0f;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    mx = fmaxf(mx, fabsf(dx[u]));
    my = fmaxf(my, fabsf(dy[u]));
  }
  const bool far = (d.periodic[0] && mx > d.half[0]) || (d.periodic[1] && my > d.half[1]);
  if (__builtin_amdgcn_ballot_w64(far) == 0) return;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    dx[u] = mod_offset(dx[u], d, 0);
    dy[u] = mod_offset(dy[u], d, 1);
  }
}

// v of lane S of the group of L consecutive lanes.
template <int L, int S>
__device__ __forceinline__ float group_lane(float v) {
  static_assert(L == 1 || L == 4 || L == 16, "quad or row");
  if (L == 1) return v;
  const int b = __float_as_int(v);
  if (L == 4) return __int_as_float(__builtin_amdgcn_update_dpp(0, b, S * 0x55, 0xf, 0xf, true));  // quad_perm
  return __int_as_float(__builtin_amdgcn_update_dpp(0, b, 0x150 + S, 0xf, 0xf, true));             // row_newbcast
}

template <int L, int K, int S = 0>
__device__ __forceinline__ void add_lanes(float (&acc)[K], const float (&t)[K]) {
  if constexpr (S < L) {
#pragma unroll
    for (int k = 0; k < K; ++k) acc[k] += group_lane<L, S>(t[k]);
    add_lanes<L, K, S + 1>(acc, t);
  }
}

// acc[k] += the K terms of every entry of a neighbor row, in row order, by L
// consecutive lanes of a wave: lane g evaluates the entries n0 + g, then all
// lanes add the L terms one after the other (a DPP operand of the add), so
// the sum is that of one thread.  terms(d, t) fills t[u] for U entries with
// data d[u] = load(neighbor, list position); entries past the row's end load `self`
// (position -1) and count as zero (no sum is -0, so adding +0 keeps its bits).  All lanes of the
// wave call it.
template <int L, int U, int K, class Load, class Terms>
__device__ __forceinline__ void sum_row(const int32_t* __restrict__ nbr, const RowRef& rr, int self, float (&acc)[K],
                                        const Load& load, const Terms& terms) {
  const int g = L == 1 ? 0 : (int)(threadIdx.x & (L - 1));
  // the next group's entries are read ahead of the current group's work: the
  // list streams from HBM and a group's data loads wait for its entries
  int j[U], at[U];
  auto entries = [&](int n0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int n = n0 + u * L + g;
      at[u] = n < rr.cnt ? rr.base + n * rr.step : -1;
      j[u] = n < rr.cnt ? __builtin_nontemporal_load(nbr + at[u]) : self;
    }
  };
  entries(0);
  for (int n0 = 0; __builtin_amdgcn_ballot_w64(n0 < rr.cnt); n0 += U * L) {
    decltype(load(0, 0)) d[U];
#pragma unroll
    for (int u = 0; u < U; ++u) d[u] = load(j[u], at[u]);
    entries(n0 + U * L);
    float t[U][K];
    terms(d, t);
    if (__builtin_amdgcn_ballot_w64(n0 + U * L > rr.cnt)) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
#pragma unroll
        for (int k = 0; k < K; ++k) t[u][k] = n0 + u * L + g < rr.cnt ? t[u][k] : 0.0f;
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) add_lanes<L, K>(acc, t[u]);
  }
}

// Lanes per row of the DFSPH passes (16, 4, else tiles): few rows are a matter
// of latency, many fill the chip by themselves, and the lines lie where the
// times cross.  Density / prepare / source / sweep A in us: 8.1k rows with 16
// lanes 8 / 9 / 5 / 6, with 4 12 / 13 / 7 / 8; 12k 7 / 11 / 6 / 7 and 9 / 13 / 7 /
// 7; 16k 7 / 13 / 7 / 8 and 9 / 13 / 7 / 7; 160k with 4 lanes 22 / 41 / 20 / 19,
// tiles 27 / 46 / 23 / 22; 202k 25 / 51 / 23 / 22 and 29 / 51 / 24 / 23; 262k 28 /
// 61 / 27 / 26 and 28 / 53 / 25 / 24.
constexpr int kLanes16Rows = 3 << 12, kLanes4Rows = 3 << 16;

}  // namespace dsph
