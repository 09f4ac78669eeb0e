// Vector-Jacobian product of the delta-SPH right-hand side (fluid only,
// uniform support), the building block of the hand-written adjoint of the
// RK4 rollout.
//
// Forward (deltasph.hip): with d = x_i - x_j (min-image), r = |d|,
// xhat = d/(r+1e-7), q = r/h, rr = q h, w1 = dW/dr, gradW = xhat w1,
// V_j = m_j / rho_j:
//   a_i    = -(1/rho_i) sum_j V_j (p_i + p_j) gradW             p = c (rho - rho0)
//   visc_i = (cV_i/rho_i) sum_j V_j pi_ij gradW,  pi = (u_i-u_j).xhat / (rr + eps h^2)
//   cont_i = -sum_j m_j ((u_j-u_i).gradW) rho_i/rho_j
//   D_i    = cD_i sum_j V_j psi_ij.gradW,  psi = -2(rho_j-rho_i)/(rr+1e-6 h) xhat + g_i + g_j
//   g_i    = L_i s_i,  s_i = sum_j V_j (rho_i-rho_j) gradW,  L_i = pinv(M_i),
//   M_i    = sum_j V_j (-rr xhat) (x) gradW   (M_i = I, L_i constant, for rows < 4)
//   dudt = a + visc + g0, drho/dt = cont + D.
// Given cotangents (la = dl/d dudt, lc = dl/d drhodt) the VJP returns
// dl/dx, dl/du, dl/drho.  dL = -L dM L (the regularisation of the reference's
// closed-form pseudo-inverse changes it by ~1e-7 relative and is not
// differentiated), dt and the neighbor sets are constants.
//
// Uniform h makes the neighbor sets symmetric and the pair geometry exactly
// antisymmetric (fl(x_j - x_i) = -fl(x_i - x_j)), so every kernel gathers:
// particle k sums, over its own row, the pair terms where it is the row
// owner and those where it is the neighbor, using the neighbor's
// cotangents.  No atomics; results do not depend on scheduling.
#include "common.h"
#include "near_math.h"
#include "pmath.h"

namespace dsph {

struct VjpConst {
  float h;
  float rho0, eos_c, cs;
  float cV;        // viscid: 2(d+2) nu rho0; inviscid: alpha h cs rho0
  float eps;       // viscosity eps
  float cD;        // delta h cs / kernel_scale
  int visc;        // -1 none, 0 inviscid, 1 viscid
  int pi_switch;
  int diffusion;
};

__device__ __forceinline__ float dot2(float2 a, float2 b) { return __builtin_fmaf(a.y, b.y, a.x * b.x); }
__device__ __forceinline__ float2 axpy(float c, float2 x, float2 y) {
  return make_float2(__builtin_fmaf(c, x.x, y.x), __builtin_fmaf(c, x.y, y.y));
}

// lambda_s_i = L_i^T lambda_g_i with lambda_g_k = sum_j (cD lc_k V_j -
// cD lc_j V_k) gradW_kj, and g_i once more where L_i is not constant:
// lambda_M_i = -L_i^T (lambda_g_i s_i^T) L_i^T = -lambda_s_i (L_i s_i)^T =
// -lambda_s_i g_i^T (zero when the row has < 4 entries: M_i = I).  lsg[i] =
// (lambda_s_i, g_i or 0).  One pass forms both sums (lambda_g and M): they
// share the pair geometry, and neither is used elsewhere.  kLanes lanes per
// row; the pseudo-inverse on one thread per row (see k_dsph_normalization_near).
struct NbrGrad {
  float2 x;
  float m, r, lc;
};
template <int kLanes>
__global__ void __launch_bounds__(kBlock) k_vjp_grad(PairsDev P, VjpConst K, const float* __restrict__ mass,
                                                     const float* __restrict__ rho, const float* __restrict__ lc,
                                                     const float2* __restrict__ grad_rho, float4* __restrict__ lsg) {
  const int row = (int)((blockIdx.x * (unsigned)blockDim.x + threadIdx.x) / kLanes);
  const bool valid = row < P.nq;
  const int k = valid ? row : P.nq - 1;
  const float2 xk = P.qpos[k];
  const float cVk = K.cD * (mass[k] / rho[k]), cLk = K.cD * lc[k];
  const KConst kc = kconst(K.h);
  RowRef rr = row_ref(P, k);
  if (!valid) rr.cnt = 0;
  constexpr int U = 4;
  float acc[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  sum_row<kLanes, U>(
      P.nbr, rr, k, acc, [&](int j, int) { return NbrGrad{P.rpos[j], mass[j], rho[j], lc[j]}; },
      [&](const NbrGrad(&d)[U], float(&t)[U][6]) {
        float dx[U], dy[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          dx[u] = xk.x - d[u].x.x;
          dy[u] = xk.y - d[u].x.y;
        }
        wrap_offsets(dx, dy, P.dom);
        auto put = [&](const Geom& g, float Vj, float lcj, float(&o)[6]) {
          const float f = cLk * Vj - cVk * lcj;
          o[0] = f * g.gx;
          o[1] = f * g.gy;
          const float s = -(g.q * g.h);
          const float qx = s * g.ex, qy = s * g.ey;
          const float kx = Vj * g.gx, ky = Vj * g.gy;
          o[2] = qx * kx;
          o[3] = qx * ky;
          o[4] = qy * kx;
          o[5] = qy * ky;
        };
        NearRange range;
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const float ir = range.divisor(d[u].r);
          range.operand(d[u].m);
          put(pair_geom_near(dx[u], dy[u], K.h, kc, range), div_near(d[u].m, d[u].r, ir), d[u].lc, t[u]);
        }
        if (range.odd()) {
#pragma unroll
          for (int u = 0; u < U; ++u)
            put(pair_geom(xk, d[u].x, K.h, kc, P.dom), d[u].m / d[u].r, d[u].lc, t[u]);
        }
      });
  __shared__ float sums[7][kBlock / kLanes];
  const int r = threadIdx.x / kLanes;
  if ((threadIdx.x & (kLanes - 1)) == 0) {
    for (int q = 0; q < 6; ++q) sums[q][r] = acc[q];
    sums[6][r] = rr.cnt < 4 ? 1.f : 0.f;
  }
  __syncthreads();
  constexpr int rows = kBlock / kLanes;
  const int t = threadIdx.x, i = blockIdx.x * rows + t;
  if (t >= rows || i >= P.nq) return;
  const float2 l = make_float2(sums[0][t], sums[1][t]);
  if (sums[6][t] != 0.f) {
    lsg[i] = make_float4(l.x, l.y, 0.f, 0.f);  // L = I
    return;
  }
  const dsph_pm::Pinv2 L = dsph_pm::pinv2x2(sums[2][t], sums[3][t], sums[4][t], sums[5][t]);
  const float2 g = grad_rho[i];
  lsg[i] = make_float4(L.l00 * l.x + L.l10 * l.y, L.l01 * l.x + L.l11 * l.y, g.x, g.y);
}

struct VjpArgs {
  const float2* vel;
  const float* mass;
  const float* rho;
  const float2* grad_rho;
  const float2* la;
  const float* lc;
  const float4* lsg;
  const float2* lx_in;  // cotangent of dx/dt (= u), added to lambda_u; may be NULL
  float2* out_x;
  float2* out_u;
  float* out_rho;
};

// The cotangents and state of one particle as the pair terms take them.
struct Cot {
  float2 x, u, g, la;
  float4 lsg;
  float r, m, lc;
  int self;  // its index
};

// The geometry of a pair for d = x_k - x_j (d != 0).
struct PGeo {
  float2 d, e, G;              // offset, xhat, gradW
  float rr, w1, w1p, ri, Ei;   // q h, dW/dr, its derivative, 1/r, 1/(r + 1e-7)
};

// Everything particle k gets from its pair with j: as the owner of row k and
// as the neighbor in row j.  The mirrored pair has -d, -xhat, -gradW, -du and
// the same r, W', pi, so with J = d xhat / d d (symmetric, even in d) and
//   Y = V_j/rho_k la_k - V_k/rho_j la_j,        S = cV Y.gradW
//   F = lc_k V_j rho_k + lc_j V_k rho_j,        A = cD (lc_k V_j - lc_j V_k)
//   W = (pi cV - P) Y + F (u_k - u_j) + A (g_k + g_j)
//       + (rho_k - rho_j)(V_j ls_k + V_k ls_j)
//   T = V_j (ls_k (g_k.e) + g_k (ls_k.e)) + V_k (ls_j (g_j.e) + g_j (ls_j.e))
// both rows' terms are one J product, J (w1 W + S/den (u_k - u_j) + rr w1 T),
// and a multiple of d (J xhat = 1e-7 d / (r + 1e-7)^3).  The terms evaluated
// one by one for both rows, each with its own quotients, took ten times the
// instructions (262k particles: 493 us, now 82; with two passes for lambda_g
// and M 626 us, now 130; 16k particles 223 us, now 31).
__device__ __forceinline__ void pair_cotangent(const PGeo& g, const VjpConst& K, const Cot& k, float ik, float Vk,
                                               const Cot& j, float ij, float (&t)[5]) {
  const float Vj = j.m * ij;
  const float2 v = make_float2(k.u.x - j.u.x, k.u.y - j.u.y);
  const float2 lsk = make_float2(k.lsg.x, k.lsg.y), gmk = make_float2(k.lsg.z, k.lsg.w);
  const float2 lsj = make_float2(j.lsg.x, j.lsg.y), gmj = make_float2(j.lsg.z, j.lsg.w);
  const float ak = Vj * ik, aj = Vk * ij;
  const float2 Y = make_float2(ak * k.la.x - aj * j.la.x, ak * k.la.y - aj * j.la.y);
  const float YG = dot2(Y, g.G);
  const float P = K.eos_c * (k.r - K.rho0) + K.eos_c * (j.r - K.rho0);
  float pi = 0.f, S = 0.f, Sd = 0.f, Spi = 0.f;
  if (K.visc >= 0) {
    const float iden = rcp_near(g.rr + K.eps * (K.h * K.h));
    const float vr = dot2(v, g.e);
    const bool on = !K.pi_switch || vr < 0.0f;
    pi = on ? vr * iden : 0.f;
    S = on ? K.cV * YG : 0.f;
    Sd = S * iden;
    Spi = Sd * pi;
  }
  const float Fk = k.lc * Vj * k.r, Fj = j.lc * Vk * j.r, F = Fk + Fj;
  const float a1 = K.cD * k.lc * Vj, a2 = K.cD * j.lc * Vk, A = a1 - a2;
  const float i2 = rcp_near(g.rr + 1e-6f * K.h);
  const float dr = k.r - j.r;
  const float rt = -2.0f * dr * i2;
  const float xx = dot2(g.e, g.e), xw = xx * g.w1;
  const float2 Gs = make_float2(k.g.x + j.g.x, k.g.y + j.g.y);
  const float psiw = __builtin_fmaf(-rt, xw, dot2(Gs, g.G));
  const float eLk = dot2(g.e, lsk), eGk = dot2(g.e, gmk), eLj = dot2(g.e, lsj), eGj = dot2(g.e, gmj);
  const float pk = Vj * eGk, qk = Vj * eLk, pj = Vk * eGj, qj = Vk * eLj;
  const float rw = g.rr * g.w1;
  const float aN = __builtin_fmaf(qk, eGk, qj * eGj);  // minus e.(V_j M_k + V_k M_j) e
  float2 W = axpy(K.cV * pi - P, Y, make_float2(F * v.x, F * v.y));
  W = axpy(A, Gs, W);
  W = axpy(dr * Vj, lsk, W);
  W = axpy(dr * Vk, lsj, W);
  float2 T = axpy(pk, lsk, make_float2(qk * gmk.x, qk * gmk.y));
  T = axpy(pj, lsj, T);
  T = axpy(qj, gmj, T);
  float2 X = axpy(g.w1, W, make_float2(Sd * v.x, Sd * v.y));
  X = axpy(rw, T, X);
  float D = __builtin_fmaf(g.w1p, dot2(g.e, W), -Spi);
  const float Art = A * rt;
  D = __builtin_fmaf(Art, __builtin_fmaf(i2, xw, -xx * g.w1p), D);
  D = __builtin_fmaf(aN, __builtin_fmaf(g.rr, g.w1p, g.w1), D);
  const float E2 = g.Ei * g.Ei;
  const float c = g.ri * __builtin_fmaf(-E2, dot2(g.d, X), D) - 2e-7f * (Art * g.w1) * (E2 * g.Ei);
  t[0] = __builtin_fmaf(c, g.d.x, X.x * g.Ei);
  t[1] = __builtin_fmaf(c, g.d.y, X.y * g.Ei);
  t[2] = __builtin_fmaf(F, g.G.x, Sd * g.e.x);
  t[3] = __builtin_fmaf(F, g.G.y, Sd * g.e.y);
  // the terms with a factor 1 / rho_k first
  float q = __builtin_fmaf(P, YG, -pi * S);
  q = __builtin_fmaf(Fk - Fj, dot2(v, g.G), q);
  q = __builtin_fmaf(a2, psiw, q);
  q = __builtin_fmaf(Vk * j.r, dot2(lsj, g.G), q);
  q = __builtin_fmaf(-rw, qj * eGj, q);
  float l = __builtin_fmaf(q, ik, -K.eos_c * YG);
  l = __builtin_fmaf(2.0f * A * i2, xw, l);
  t[4] = __builtin_fmaf(Vj, dot2(lsk, g.G), l);
}

template <int kLanes>
__global__ void __launch_bounds__(kBlock) k_vjp_main(PairsDev P, VjpConst K, VjpArgs A) {
  const int row = (int)((blockIdx.x * (unsigned)blockDim.x + threadIdx.x) / kLanes);
  const bool valid = row < P.nq;
  const int k = valid ? row : P.nq - 1;
  auto load = [&](int j, int) {
    Cot c;
    c.x = P.rpos[j];
    c.u = A.vel[j];
    c.g = K.diffusion ? A.grad_rho[j] : make_float2(0.f, 0.f);
    c.la = A.la[j];
    c.lsg = A.lsg[j];
    c.r = A.rho[j];
    c.m = A.mass[j];
    c.lc = A.lc[j];
    c.self = j;
    return c;
  };
  Cot ck = load(k, -1);
  ck.x = P.qpos[k];
  const float ik = 1.0f / ck.r, Vk = ck.m / ck.r;
  const KConst kc = kconst(K.h);
  const float cp = kC2 / (((K.h * K.h) * K.h) * K.h);
  RowRef rr = row_ref(P, k);
  if (!valid) rr.cnt = 0;
  constexpr int U = 2;
  float acc[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
  sum_row<kLanes, U>(P.nbr, rr, k, acc, load, [&](const Cot(&d)[U], float(&t)[U][5]) {
    float dx[U], dy[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      dx[u] = ck.x.x - d[u].x.x;
      dy[u] = ck.x.y - d[u].x.y;
    }
    wrap_offsets(dx, dy, P.dom);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      NearRange range;
      PGeo g;
      g.d = make_float2(dx[u], dy[u]);
      const float d2 = dist2_exact(dx[u], dy[u]);
      range.d2(d2);
      float r = sqrt_near(d2), ij = range.divisor(d[u].r);
      if (range.odd()) {
        r = sqrt_rn(d2);
        ij = 1.0f / d[u].r;
      }
      g.Ei = rcp_near(r + 1e-7f);
      g.ri = rcp_near(r);
      g.e = make_float2(dx[u] * g.Ei, dy[u] * g.Ei);
      const float q = r * kc.ih;
      g.rr = q * K.h;
      const float s = clamp01(1.0f - q);
      g.w1 = wendland_dw(q, kc);
      // d w1 / dr = C/h^4 (-20) (1-q)^2 (1-4q)
      g.w1p = q < 1.0f ? ((-20.0f * (s * s)) * (1.0f - 4.0f * q)) * cp : 0.0f;
      g.G = make_float2(g.e.x * g.w1, g.e.y * g.w1);
      pair_cotangent(g, K, ck, ik, Vk, d[u], ij, t[u]);
      // the particle itself (and the padding of its row) has no pair; r = 0
      // between distinct particles stays NaN, as the gradient is
      const bool self = d[u].self == k;
      if (self) {
#pragma unroll
        for (int c = 0; c < 5; ++c) t[u][c] = 0.f;
      }
    }
  });
  if (!valid || (threadIdx.x & (kLanes - 1)) != 0) return;
  if (A.lx_in) {
    const float2 t = A.lx_in[k];
    acc[2] += t.x;
    acc[3] += t.y;
  }
  A.out_x[k] = make_float2(acc[0], acc[1]);
  A.out_u[k] = make_float2(acc[2], acc[3]);
  A.out_rho[k] = acc[4];
}

}  // namespace dsph

using namespace dsph;

// Lanes per row, where the times cross.  k_vjp_grad / k_vjp_main in us with 16
// and 4 lanes: 4k rows 9 / 7, 12 / 14; 8.1k 12 / 9, 13 / 15; 12k 13 / 11, 11 / 13;
// 16k 15 / 13, 11 / 13; 26k 18 / 20, 13 / 17; with 4 and 1: 132k 31 / 51, 36 / 63;
// 202k 42 / 71, 46 / 85; 262k 53 / 87, 49 / 84; 640k 110 / 203, 101 / 202.
constexpr int64_t kGrad16 = 1 << 13, kMain16 = 1 << 14, kVjp4 = 7 << 15;

extern "C" size_t dsph_deltasph_vjp_workspace(int64_t n) {
  return ((size_t)n * 4 * sizeof(float) + 255) / 256 * 256 + 256;
}

extern "C" int dsph_deltasph_rhs_vjp(const dsph_pairs* pairs, const dsph_deltasph_params* prm, const float* vel,
                                     const float* mass, const float* rho, const float* grad_rho,
                                     const float* cot_dxdt, const float* cot_dudt, const float* cot_drhodt,
                                     float* grad_pos, float* grad_vel, float* grad_rho_out, void* ws,
                                     size_t ws_bytes, void* stream) {
  int s = check_pairs(pairs);
  if (s != DSPH_OK) return s;
  if (!prm || pairs->nq != pairs->nr) return DSPH_ERR_ARG;
  // symmetric lists: one uniform support, scatter mode
  if (pairs->qh || pairs->rh || !(pairs->h_uniform > 0.0f) || pairs->mode != DSPH_MODE_SCATTER) return DSPH_ERR_ARG;
  if (prm->viscosity < -1 || prm->viscosity > 1 || prm->eos < 0 || prm->eos > 1) return DSPH_ERR_ARG;
  const int64_t n = pairs->nq;
  if (n == 0) return DSPH_OK;
  if (!vel || !mass || !rho || !cot_dudt || !cot_drhodt || !grad_pos || !grad_vel || !grad_rho_out)
    return DSPH_ERR_ARG;
  if (prm->diffusion && (!grad_rho || !(prm->kernel_scale > 0.0f))) return DSPH_ERR_ARG;
  if (!ws || ws_bytes < dsph_deltasph_vjp_workspace(n)) return DSPH_ERR_CAPACITY;
  hipStream_t st = as_stream(stream);
  PairsDev P = make_pairs(*pairs);
  VjpConst K;
  K.h = pairs->h_uniform;
  K.rho0 = prm->rho0;
  K.eos_c = prm->eos == 0 ? prm->cs * prm->cs : prm->eos_kappa;
  K.cs = prm->cs;
  K.cV = prm->viscosity == 1 ? (float)(2.0 * 4.0 * (double)prm->visc_coeff * (double)prm->rho0)
                             : (((prm->visc_coeff * K.h) * prm->cs) * prm->rho0);
  K.eps = prm->visc_eps;
  K.cD = prm->diffusion ? ((prm->delta * K.h) / prm->kernel_scale) * prm->cs : 0.0f;
  K.visc = prm->viscosity;
  K.pi_switch = prm->pi_switch;
  K.diffusion = prm->diffusion;
  char* w = static_cast<char*>(ws);
  float4* lsg = reinterpret_cast<float4*>(w);
  const int lanes = n <= kMain16 ? 16 : (n <= kVjp4 ? 4 : 1);
  const int grad_lanes = n <= kGrad16 ? 16 : (n <= kVjp4 ? 4 : 1);
  if (prm->diffusion) {
    auto go = [&](auto kernel) {
      kernel<<<grid_for(n, kBlock / grad_lanes), kBlock, 0, st>>>(P, K, mass, rho, cot_drhodt,
                                                                  reinterpret_cast<const float2*>(grad_rho), lsg);
    };
    grad_lanes == 16 ? go(k_vjp_grad<16>) : (grad_lanes == 4 ? go(k_vjp_grad<4>) : go(k_vjp_grad<1>));
  } else {
    DSPH_CHECK_HIP(hipMemsetAsync(lsg, 0, sizeof(float4) * n, st));
  }
  VjpArgs A;
  A.vel = reinterpret_cast<const float2*>(vel);
  A.mass = mass;
  A.rho = rho;
  A.grad_rho = reinterpret_cast<const float2*>(grad_rho);
  A.la = reinterpret_cast<const float2*>(cot_dudt);
  A.lc = cot_drhodt;
  A.lsg = lsg;
  A.lx_in = reinterpret_cast<const float2*>(cot_dxdt);
  A.out_x = reinterpret_cast<float2*>(grad_pos);
  A.out_u = reinterpret_cast<float2*>(grad_vel);
  A.out_rho = grad_rho_out;
  auto go = [&](auto kernel) { kernel<<<grid_for(n, kBlock / lanes), kBlock, 0, st>>>(P, K, A); };
  lanes == 16 ? go(k_vjp_main<16>) : (lanes == 4 ? go(k_vjp_main<4>) : go(k_vjp_main<1>));
  return launch_status();
}
