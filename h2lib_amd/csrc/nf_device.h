// Device code of the near-field quadrature (included by the per-family
// translation units nf_laplace.hip and nf_helmholtz_*.hip).
//
// Two kernels per operator, run in this order on one stream:
//
//  nf_regular_kernel  one workgroup (four wave64s) per tile of at most
//      64 x 64 DOFs.  Every pair (row support triangle, column support
//      triangle) without common vertices is evaluated by one lane with the
//      tensor-product Gauss rule from quadrature points precomputed per
//      triangle (16 kernel evaluations at q = 2, all from registers).  The
//      element matrix (1x1, 1x3, 3x1 or 3x3) is added into an LDS tile that
//      is stored once, coalesced; the constant-basis case stores entries
//      directly.  Pairs with common vertices are skipped (cc: stored as 0).
//
//  nf_singular_kernel one row of 16 lanes per pair with common vertices,
//      one launch per rule class (identical, edge, vertex) over the pair
//      list built at planning time.  The 2 q2^4 or 6 q2^4 Sauter-Schwab
//      points are formed on the fly from the q2 Gauss nodes (no rule tables
//      are read), the sums are reduced across the row and up to nine lanes
//      add the element matrix into the output with FP64 atomics.  x - y is
//      formed from differences of the permuted vertices, so the shared
//      vertices cancel exactly.
#pragma once

#include <algorithm>
#include <type_traits>

#include "dmath.h"
#include "h2hip_internal.h"

namespace h2hip {
namespace nf {

constexpr int NTHREADS = 256;
constexpr int NWAVES = NTHREADS / 64;
// pairs with common vertices up to which their three classes share a launch
constexpr uint32_t SING_ALL = 32768;

// K_HELM_*_SP: the Helmholtz kernels for surfaces on which the phase varies
// by less than pi/4 within a pair of triangles with common vertices and
// around a reference distance within any other pair (real k, 2 |k| h <= pi/4
// with the longest edge h): no argument reduction per evaluation, and no
// damping, whose exponential breaks up the evaluations of a pair.
// K_HELM_*_TP: the same for 2 |k| h <= 1/4 with shorter polynomials.
enum {
  K_LAP_SLP = 0,
  K_LAP_DLP = 1,
  K_HELM_SLP = 2,
  K_HELM_DLP = 3,
  K_HELM_SLP_SP = 4,
  K_HELM_DLP_SP = 5,
  K_HELM_SLP_TP = 6,
  K_HELM_DLP_TP = 7
};
constexpr bool is_dlp(int ker) { return ker & 1; }
constexpr bool small_phase(int ker) { return ker >= K_HELM_SLP_SP; }
constexpr bool tiny_phase(int ker) { return ker >= K_HELM_SLP_TP; }

// 1/sqrt(x): hardware estimate and one third-order correction
// y (1 + e/2 + 3 e^2/8), e = 1 - x y^2.  Positive finite x only (x = 0
// gives NaN where 1/sqrt gives inf; both are non-finite).
__device__ __forceinline__ double rsqrt_fast(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-x * y, y, 1.0);
  return fma(y * e, fma(e, 0.375, 0.5), y);
}

// x^(-3/2): y^3 (1 + 3e/2 + 15e^2/8) with y and e as above (two roundings
// and one operation less than the cube of rsqrt_fast).
__device__ __forceinline__ double rsqrt3_fast(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double y2 = y * y;
  const double e = fma(-x, y2, 1.0);
  const double t = y * y2;
  return fma(t * e, fma(e, 1.875, 1.5), t);
}

// Kernel function values without the 1/(4 pi) factor.
// Laplace SLP 1/r, DLP <d, n_y>/r^3 (Library/laplacebem3d.c:35-108);
// Helmholtz SLP e^{ikr}/r, DLP e^{ikr} (1 - ikr) <d, n_y>/r^3
// (Library/helmholtzbem3d.c:26-170), d = x - y, r = |d|,
// k = kr + i ki' with ki = -ki' (damping e^{ki r}).
//
// kcore: the part that does not depend on the normal, g (fr + i fi) with
// real g; the double layers multiply g by <d, n>.  The phase is k r - ph0
// (ph0 = 0: the kernel itself); the small-phase kernels take it without
// argument reduction.
template <int KER>
__device__ __forceinline__ void kcore(double r2, double kr, double ki,
                                      double ph0, double &g, double &fr,
                                      double &fi) {
  if constexpr (KER == K_LAP_SLP) {
    g = rsqrt_fast(r2);
    fr = 1.0;
    fi = 0.0;
  } else if constexpr (KER == K_LAP_DLP) {
    g = rsqrt3_fast(r2);
    fr = 1.0;
    fi = 0.0;
  } else {
    const double rs = rsqrt_fast(r2);
    const double r = r2 * rs;
    g = is_dlp(KER) ? rs * rs * rs : rs;
    double s, c;
    if constexpr (tiny_phase(KER)) {
      h2hip::sincos_poly_tiny(fma(kr, r, -ph0), s, c);
    } else if constexpr (small_phase(KER)) {
      h2hip::sincos_poly(fma(kr, r, -ph0), s, c);
    } else {
      if (ki != 0.0) g *= exp(ki * r);
      h2hip::sincos_cw(kr * r, s, c);
    }
    if constexpr (is_dlp(KER)) {
      const double kr_r = kr * r;
      fr = fma(kr_r, s, c);
      fi = fma(-c, kr_r, s);
    } else {
      fr = c;
      fi = s;
    }
  }
}

template <int KER>
__device__ __forceinline__ void kval(double dx, double dy, double dz,
                                     double nx, double ny, double nz,
                                     double kr, double ki, double &re,
                                     double &im) {
  const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
  double g, fr, fi;
  kcore<KER>(r2, kr, ki, 0.0, g, fr, fi);
  if constexpr (is_dlp(KER)) g *= fma(dx, nx, fma(dy, ny, dz * nz));
  re = KER >= K_HELM_SLP ? fr * g : g;
  im = KER >= K_HELM_SLP ? fi * g : 0.0;
}

// The same kernel values in FP32 (mixed precision), from a difference
// vector d that the caller formed in FP64 (singular pairs) or from an FP64
// difference of anchor points plus FP32 offsets (regular pairs).  1/r is
// the hardware reciprocal square root (1 ulp); the phase k r is reduced to
// [-1/2, 1/2] revolutions before the hardware sine and cosine, so their
// argument is always small; the damping e^{ki r} is the hardware 2^x of
// ki log2(e) r.
// kcore32, kval32: as kcore and kval.
template <int KER>
__device__ __forceinline__ void kcore32(float r2, float krf, float krev,
                                        float kil2, float &g, float &fr,
                                        float &fi) {
  const float rs = __builtin_amdgcn_rsqf(r2);
  g = is_dlp(KER) ? rs * rs * rs : rs;
  fr = 1.0f;
  fi = 0.0f;
  if constexpr (KER >= K_HELM_SLP) {
    const float r = r2 * rs;
    float rev = r * krev;
    rev -= __builtin_rintf(rev);
    const float s = __builtin_amdgcn_sinf(rev);
    const float c = __builtin_amdgcn_cosf(rev);
    if (kil2 != 0.0f) g *= __builtin_amdgcn_exp2f(kil2 * r);
    if constexpr (is_dlp(KER)) {
      const float kr_r = krf * r;
      fr = fmaf(kr_r, s, c);
      fi = fmaf(-c, kr_r, s);
    } else {
      fr = c;
      fi = s;
    }
  }
}

template <int KER>
__device__ __forceinline__ void kval32(float dx, float dy, float dz, float nx,
                                       float ny, float nz, float krf,
                                       float krev, float kil2, float &re,
                                       float &im) {
  float g, fr, fi;
  kcore32<KER>(fmaf(dx, dx, fmaf(dy, dy, dz * dz)), krf, krev, kil2, g, fr,
               fi);
  if constexpr (is_dlp(KER)) g *= fmaf(dx, nx, fmaf(dy, ny, dz * nz));
  re = KER >= K_HELM_SLP ? fr * g : g;
  im = KER >= K_HELM_SLP ? fi * g : 0.0f;
}

// Normal vector of the double layer kernels for the pair (row triangle
// rt, column triangle ct): n_y of the column triangle (double layer), or
// -n_x of the row triangle (adjoint double layer, <y - x, n_x> =
// <x - y, -n_x>; the reference's integrators pass the row triangle's
// normal as n_x also where its lc far rule swaps the point roles,
// Library/bem3d.c:2637-2649).
__device__ __forceinline__ void layer_normal(const KArgs &a, uint32_t rt,
                                             uint32_t ct, double (&nv)[3]) {
  const uint32_t t = a.adj ? rt : ct;
  const double sg = a.adj ? -1.0 : 1.0;
#pragma unroll
  for (int d = 0; d < 3; d++) nv[d] = sg * a.n[3 * t + d];
}

// kernel constant and Gram determinants of a pair of triangles (constant
// basis: in the order of the triangle numbers, as entry_sums)
template <bool CC>
__device__ __forceinline__ double pair_factor(const KArgs &a, uint32_t rt,
                                              uint32_t ct) {
  const uint32_t lo = CC && rt > ct ? ct : rt, hi = CC && rt > ct ? rt : ct;
  return a.kc * a.g[lo] * a.g[hi];
}

// a summed entry: stored, or added where a tile's pairs are split over
// several workgroups
__device__ __forceinline__ void put(const KArgs &a, size_t pos, double v,
                                    uint32_t nslice) {
  if (nslice > 1)
    atomicAdd(&a.out[pos], v);
  else
    a.out[pos] = v;
}

static __global__ __launch_bounds__(NTHREADS) void zero_out(double *out,
                                                            uint64_t n) {
  for (uint64_t i = blockIdx.x * (uint64_t)NTHREADS + threadIdx.x; i < n;
       i += gridDim.x * (uint64_t)NTHREADS)
    out[i] = 0.0;
}

static __global__ void zero_counter(uint32_t *c) { *c = 0u; }

__device__ __forceinline__ uint32_t loc_of(uint32_t packed, int l) {
  return (packed >> (8 * l)) & 0xffu;
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// Kahan's compensated sum s += x in FP32 (c carries the rounding error of
// the previous additions; the compiler must not reassociate, and does not
// without fast-math)
__device__ __forceinline__ void kahan_add(float &s, float &c, float x) {
  const float y = x - c;
  const float t = s + y;
  c = (t - s) - y;
  s = t;
}

// Element matrices of a pair of triangles without common vertices by the
// tensor-product rule with points x_i on triangle tt and y_b on triangle ts,
// d = x_i - y_b, over the local functions l of tt and k of ts (1 or 3 each).
// nt, ns: the triangles' normals and the means of their points' <p_i - p_0,
// n> (KArgs::regn).
//
// The double layers' <d, n> of one order of the pair takes the normal of ts,
// of the other that of tt: A = <d, ns> and B = <d, -nt> (the differences
// change sign).  S1[l][k] sums the kernel of one order: single layers the
// kernel, double layers sg A or, wantB, sg B.  TWO: both orders at once, S1
// with A and S2 with B, which share the difference, its length and the
// phase.  FP64 and a.plane (normals perpendicular to the triangles): A does
// not depend on b nor B on i, so A is a factor of the row point and B of the
// column point and no value takes a product of vectors (double layer, linear
// basis, 32768 triangles: 1011 -> 945 us).  Both are taken from the mean of
// the other triangle's points, not from one of them, whose rounding would be
// in every value: entries of touching clusters are then off by 0.97 to 1.01
// times what a product per value gives, from one point by 1.6 times (sphere
// of 8192 triangles, constant basis, against long double).
// MP: 0 FP64; 1 mixed (FP32 kernel values and inner sums, FP64 outer sums);
// 2 mixed with FP32 accumulation throughout, the outer sums compensated
// (Kahan); TWO is for MP 0 and single layers with MP 1 (S2 is not set: the
// single layers are symmetric).
// PL_: a.plane where the launch knows it (0, 1), -1 where it is looked up (a
// kernel with both ways takes the registers of the larger, up to 220).
template <int KER, int BR, int BC, int Q, int MP, bool TWO, int PL_>
__device__ __forceinline__ void pair_sums(
    const KArgs &a, uint32_t tt, uint32_t ts, const double (&nt)[4],
    const double (&ns)[4], bool wantB, double sg,
    double (&S1re)[BR ? 3 : 1][BC ? 3 : 1],
    double (&S1im)[BR ? 3 : 1][BC ? 3 : 1],
    double (&S2re)[BR ? 3 : 1][BC ? 3 : 1],
    double (&S2im)[BR ? 3 : 1][BC ? 3 : 1]) {
  constexpr bool CPLX = KER >= K_HELM_SLP;
  constexpr bool DLP = is_dlp(KER);
  constexpr int NR = BR ? 3 : 1;
  constexpr int NC = BC ? 3 : 1;
  constexpr int QQ = Q * Q;
  const double *__restrict__ W = a.regw;  // w | phi0 w | phi1 w | phi2 w
  const double *__restrict__ Pt = a.regpts + (size_t)tt * (3 * QQ);
  const double *__restrict__ Ps = a.regpts + (size_t)ts * (3 * QQ);
#pragma unroll
  for (int l = 0; l < NR; l++)
#pragma unroll
    for (int k = 0; k < NC; k++)
      S1re[l][k] = S1im[l][k] = S2re[l][k] = S2im[l][k] = 0.0;
  if constexpr (MP != 0) {
    static_assert(!TWO, "both orders of a double layer: FP64");
    double n1[3];
#pragma unroll
    for (int d = 0; d < 3; d++) n1[d] = sg * (wantB ? -nt[d] : ns[d]);
    // x_i - y_b = (P_t,i - P_s,0) - (P_s,b - P_s,0), the first difference in
    // FP64 (then rounded), the offsets of the column points in FP32
    const float *__restrict__ Os = a.regoff + (size_t)ts * (3 * QQ);
    const float *__restrict__ WF = a.regwf;
    const double sx0 = Ps[0], sy0 = Ps[1], sz0 = Ps[2];
    float ptx[QQ], pty[QQ], ptz[QQ];
#pragma unroll
    for (int i = 0; i < QQ; i++) {
      ptx[i] = (float)(Pt[3 * i] - sx0);
      pty[i] = (float)(Pt[3 * i + 1] - sy0);
      ptz[i] = (float)(Pt[3 * i + 2] - sz0);
    }
    const float n1x = (float)n1[0], n1y = (float)n1[1], n1z = (float)n1[2];
    // MP 2: the outer sums in FP32 with their compensations
    float Fre[NR][NC], Fim[NR][NC], Cre[NR][NC], Cim[NR][NC];
#pragma unroll
    for (int l = 0; l < NR; l++)
#pragma unroll
      for (int k = 0; k < NC; k++)
        Fre[l][k] = Fim[l][k] = Cre[l][k] = Cim[l][k] = 0.0f;
#pragma unroll
    for (int b = 0; b < QQ; b++) {
      const float qx = Os[3 * b], qy = Os[3 * b + 1], qz = Os[3 * b + 2];
      float Ure[NR], Uim[NR];
#pragma unroll
      for (int l = 0; l < NR; l++) Ure[l] = Uim[l] = 0.0f;
#pragma unroll
      for (int i = 0; i < QQ; i++) {
        const float dx = ptx[i] - qx, dy = pty[i] - qy, dz = ptz[i] - qz;
        float g, fr, fi;
        kcore32<KER>(fmaf(dx, dx, fmaf(dy, dy, dz * dz)), a.krf, a.krev,
                     a.kil2, g, fr, fi);
        float g1 = g;
        if constexpr (DLP) g1 = fmaf(dx, n1x, fmaf(dy, n1y, dz * n1z)) * g;
#pragma unroll
        for (int l = 0; l < NR; l++) {
          const float wr = BR ? WF[QQ * (1 + l) + i] : WF[i];
          Ure[l] = fmaf(wr, CPLX ? g1 * fr : g1, Ure[l]);
          if constexpr (CPLX) Uim[l] = fmaf(wr, g1 * fi, Uim[l]);
        }
      }
#pragma unroll
      for (int k = 0; k < NC; k++) {
        if constexpr (MP == 2) {
          const float wc = BC ? WF[QQ * (1 + k) + b] : WF[b];
#pragma unroll
          for (int l = 0; l < NR; l++) {
            kahan_add(Fre[l][k], Cre[l][k], wc * Ure[l]);
            if constexpr (CPLX) kahan_add(Fim[l][k], Cim[l][k], wc * Uim[l]);
          }
        } else {
          const double wc = BC ? W[QQ * (1 + k) + b] : W[b];
#pragma unroll
          for (int l = 0; l < NR; l++) {
            S1re[l][k] = fma(wc, (double)Ure[l], S1re[l][k]);
            if constexpr (CPLX)
              S1im[l][k] = fma(wc, (double)Uim[l], S1im[l][k]);
          }
        }
      }
    }
    if constexpr (MP == 2) {
#pragma unroll
      for (int l = 0; l < NR; l++)
#pragma unroll
        for (int k = 0; k < NC; k++) {
          S1re[l][k] = (double)Fre[l][k] - (double)Cre[l][k];
          S1im[l][k] = (double)Fim[l][k] - (double)Cim[l][k];
        }
    }
  } else {
    double ptx[QQ], pty[QQ], ptz[QQ];
#pragma unroll
    for (int i = 0; i < QQ; i++) {
      ptx[i] = Pt[3 * i];
      pty[i] = Pt[3 * i + 1];
      ptz[i] = Pt[3 * i + 2];
    }
    // small phase: k r is taken relative to that of the first points, the
    // sums are turned by it at the end
    double ph0 = 0.0;
    if constexpr (small_phase(KER)) {
      const double dx = ptx[0] - Ps[0], dy = pty[0] - Ps[1],
                   dz = ptz[0] - Ps[2];
      const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
      ph0 = a.kr * (r2 * rsqrt_fast(r2));
    }
    auto sums = [&](auto plane) {
      constexpr bool PL = DLP && decltype(plane)::value;
      // (the Helmholtz double layer with argument reduction and a product per
      // value: 127 VGPRs instead of 220; folded cylinder of 46240 triangles,
      // constant basis, 2.33 -> 2.11 ms)
      constexpr int UB = KER == K_HELM_DLP && !PL ? 1 : QQ;
      // the factors of the points and, without them, the normal of <d, n>
      double fi_[QQ], fb_[QQ], n1[3];
#pragma unroll
      for (int i = 0; i < QQ; i++) fi_[i] = fb_[i] = 1.0;
      if constexpr (PL) {
#pragma unroll
        for (int i = 0; i < QQ; i++) {
          const double A =
              fma(ptx[i] - Ps[0], ns[0],
                  fma(pty[i] - Ps[1], ns[1],
                      fma(ptz[i] - Ps[2], ns[2], -ns[3])));
          const double B = -fma(ptx[0] - Ps[3 * i], nt[0],
                                fma(pty[0] - Ps[3 * i + 1], nt[1],
                                    fma(ptz[0] - Ps[3 * i + 2], nt[2],
                                        nt[3])));
          fi_[i] = TWO ? A : wantB ? 1.0 : sg * A;
          fb_[i] = TWO ? B : wantB ? sg * B : 1.0;
        }
      } else if constexpr (DLP) {
#pragma unroll
        for (int d = 0; d < 3; d++) n1[d] = sg * (wantB ? -nt[d] : ns[d]);
      }
#pragma unroll UB
      for (int b = 0; b < QQ; b++) {
        const double qx = Ps[3 * b], qy = Ps[3 * b + 1], qz = Ps[3 * b + 2];
        double Ure[NR], Uim[NR], Vre[NR], Vim[NR];
#pragma unroll
        for (int l = 0; l < NR; l++) Ure[l] = Uim[l] = Vre[l] = Vim[l] = 0.0;
#pragma unroll
        for (int i = 0; i < QQ; i++) {
          const double dx = ptx[i] - qx, dy = pty[i] - qy, dz = ptz[i] - qz;
          double g, fr, fi;
          kcore<KER>(fma(dx, dx, fma(dy, dy, dz * dz)), a.kr, a.ki, ph0, g,
                     fr, fi);
          if constexpr (!BR && !BC) {
            // one weight for both parts of a complex value, the point's
            // factor in it
            double w1 = W[i];
            if constexpr (PL) w1 *= fi_[i];
            double v1 = w1 * g;
            if constexpr (DLP && !PL)
              v1 *= fma(dx, n1[0], fma(dy, n1[1], dz * n1[2]));
            if constexpr (CPLX) {
              Ure[0] = fma(v1, fr, Ure[0]);
              Uim[0] = fma(v1, fi, Uim[0]);
              if constexpr (TWO) {
                const double v2 = W[i] * g;
                Vre[0] = fma(v2, fr, Vre[0]);
                Vim[0] = fma(v2, fi, Vim[0]);
              }
            } else if constexpr (PL || !DLP) {
              Ure[0] = fma(w1, g, Ure[0]);
              if constexpr (TWO) Vre[0] = fma(W[i], g, Vre[0]);
            } else {
              Ure[0] += v1;
            }
          } else {
            double g1 = g;
            if constexpr (PL)
              g1 = g * fi_[i];
            else if constexpr (DLP)
              g1 = g * fma(dx, n1[0], fma(dy, n1[1], dz * n1[2]));
#pragma unroll
            for (int l = 0; l < NR; l++) {
              const double wr = BR ? W[QQ * (1 + l) + i] : W[i];
              Ure[l] = fma(wr, CPLX ? g1 * fr : g1, Ure[l]);
              if constexpr (CPLX) Uim[l] = fma(wr, g1 * fi, Uim[l]);
              if constexpr (TWO) {
                Vre[l] = fma(wr, CPLX ? g * fr : g, Vre[l]);
                if constexpr (CPLX) Vim[l] = fma(wr, g * fi, Vim[l]);
              }
            }
          }
        }
#pragma unroll
        for (int k = 0; k < NC; k++) {
          const double w0 = BC ? W[QQ * (1 + k) + b] : W[b];
          const double wB = PL ? w0 * fb_[b] : w0, wA = TWO ? w0 : wB;
#pragma unroll
          for (int l = 0; l < NR; l++) {
            S1re[l][k] = fma(wA, Ure[l], S1re[l][k]);
            if constexpr (CPLX) S1im[l][k] = fma(wA, Uim[l], S1im[l][k]);
            if constexpr (TWO) {
              S2re[l][k] = fma(wB, Vre[l], S2re[l][k]);
              if constexpr (CPLX) S2im[l][k] = fma(wB, Vim[l], S2im[l][k]);
            }
          }
        }
      }
    };
    // (TWO only with plane normals)
    if constexpr (!DLP || TWO || PL_ == 1)
      sums(std::true_type{});
    else if constexpr (PL_ == 0)
      sums(std::false_type{});
    else if (a.plane)  // uniform
      sums(std::true_type{});
    else
      sums(std::false_type{});
    if constexpr (small_phase(KER)) {
      double s0, c0;
      h2hip::sincos_cw(ph0, s0, c0);
#pragma unroll
      for (int l = 0; l < NR; l++)
#pragma unroll
        for (int k = 0; k < NC; k++) {
          const double x = S1re[l][k], y = S1im[l][k];
          S1re[l][k] = fma(x, c0, -(y * s0));
          S1im[l][k] = fma(x, s0, y * c0);
          if constexpr (TWO) {
            const double u = S2re[l][k], v = S2im[l][k];
            S2re[l][k] = fma(u, c0, -(v * s0));
            S2im[l][k] = fma(u, s0, v * c0);
          }
        }
    }
  }
}

// Whether a launch over mirrored tiles evaluates the regular pairs once for
// both entries (nf_pair_kernel): equal bases; FP64, or the single layers in
// mixed precision with FP64 outer sums.  Not the double layers in mixed
// precision: their <d, n> of nearly coplanar triangles is the rounding of
// d, which depends on the triangle whose point is the anchor.  Not the
// linear-basis Helmholtz double layers, whose four accumulators (128 KB of
// LDS) and 36 sums per lane leave one workgroup per CU.
constexpr int pair_arrays(int ker, int basis) {
  return basis == 0 ? 0 : (ker >= K_HELM_SLP ? 2 : 1) * (is_dlp(ker) ? 2 : 1);
}
constexpr bool paired(int ker, int rb, int cb, int mp) {
  return rb == cb && (mp == 0 || (mp == 1 && !is_dlp(ker))) &&
         pair_arrays(ker, rb) <= 2;
}

// The same sums for the entry (row triangle rt, column triangle ct).  The
// constant basis evaluates a pair of triangles in one order, the smaller
// number first, whichever of the two entries asks: both entries then have
// the same bits in every schedule.  Not the FP64 double layers without
// a.plane, whose tiles have no mirrors, in any schedule: there a wave's lanes
// read the same column triangle, not each its own.
template <int KER, int BR, int BC, int Q, int MP, int PL>
__device__ __forceinline__ void entry_sums(
    const KArgs &a, uint32_t rt, uint32_t ct,
    double (&Sre)[BR ? 3 : 1][BC ? 3 : 1],
    double (&Sim)[BR ? 3 : 1][BC ? 3 : 1]) {
  constexpr bool CC = (BR == 0) && (BC == 0);
  // The reference's lc far integrator maps the first rule coordinates onto
  // the column triangle (Library/bem3d.c:2637-2649); kept as is.
  const bool plane =
      PL == 1 || (PL == -1 && (!is_dlp(KER) || a.plane));  // uniform
  const bool sw = CC ? plane && paired(KER, 0, 0, MP) && rt > ct
                     : (BR && !BC) && a.far;
  const uint32_t tt = sw ? ct : rt, ts = sw ? rt : ct;
  // n_y belongs to the column triangle, the adjoint's -n_x to the row
  // triangle; d changes sign with the order except in the lc far rule
  const bool wantB = (a.adj != 0) != sw;
  double nv[4] = {0.0, 0.0, 0.0, 0.0};
  if constexpr (is_dlp(KER)) {
    const uint32_t t = a.adj ? rt : ct;
#pragma unroll
    for (int d = 0; d < 4; d++) nv[d] = a.regn[4 * (size_t)t + d];
  }
  double dre[BR ? 3 : 1][BC ? 3 : 1], dim[BR ? 3 : 1][BC ? 3 : 1];
  // (only the normal of the one order is read)
  pair_sums<KER, BR, BC, Q, MP, false, PL>(a, tt, ts, nv, nv, wantB,
                                       !CC && sw ? -1.0 : 1.0, Sre, Sim, dre,
                                       dim);
}

template <int KER, int BR, int BC, int CLS, int Q2, bool MP>
__device__ __forceinline__ void tile_singular(const KArgs &a, const Tile &T,
                                              const SPair *list, uint32_t n,
                                              double *acc_re, double *acc_im);

// One tile of the regular kernel, run by all NTHREADS threads of a
// workgroup (MP: pair_sums), or the slice-th of nslice parts of its pairs.
// FUSED: the tile's workgroup also evaluates the tile's pairs with common
// vertices (tlist + T.sbeg, T.ns[c] per class) before the tile is stored,
// so they add into the LDS accumulator instead of the output (constant
// basis: the regular pass leaves their entries to the singular pass).
template <int KER, int BR, int BC, int Q, int MP, bool FUSED = false,
          int PL = -1>
__device__ __forceinline__ void regular_tile(const KArgs &a, uint32_t tile,
                                             const SPair *tlist = nullptr,
                                             uint32_t slice = 0,
                                             uint32_t nslice = 1) {
  constexpr bool CPLX = KER >= K_HELM_SLP;
  constexpr bool CC = (BR == 0) && (BC == 0);
  constexpr int NR = BR ? 3 : 1;
  constexpr int NC = BC ? 3 : 1;

  __shared__ double acc_re[CC ? 1 : TILE * TILE];
  __shared__ double acc_im[(CC || !CPLX) ? 1 : TILE * TILE];

  const int tid = threadIdx.x;
  const Tile T = a.tiles[tile];
  const uint32_t nR = T.nrsup, nC = T.ncsup;
  const Supp *RS = a.supp + T.rsup;
  const Supp *CS = a.supp + T.csup;
  const bool conj = T.ntrans && (BR == BC);

  if constexpr (!CC) {
    for (int i = tid; i < TILE * TILE; i += NTHREADS) {
      acc_re[i] = 0.0;
      if constexpr (CPLX) acc_im[i] = 0.0;
    }
    __syncthreads();
  }

  const uint32_t npairs = nR * nC;
  // pair p = r + nR c, advanced without a division per pair
  const uint32_t p0 = tid + NTHREADS * slice, step = NTHREADS * nslice;
  const uint32_t dc = nR ? step / nR : 0, dr = step - dc * nR;
  uint32_t rr = nR ? p0 % nR : 0, cc = nR ? p0 / nR : 0;
  for (uint32_t p = p0; p < npairs; p += step) {
    const uint32_t r = rr, c = cc;
    rr += dr;
    cc += dc;
    if (rr >= nR) {
      rr -= nR;
      cc++;
    }
    const Supp sr = RS[r], sc = CS[c];
    int shared = 0;
    if (!a.far) {
#pragma unroll
      for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) shared += (sr.v[i] == sc.v[j]);
    }
    double Sre[NR][NC], Sim[NR][NC];
#pragma unroll
    for (int l = 0; l < NR; l++)
#pragma unroll
      for (int k = 0; k < NC; k++) Sre[l][k] = Sim[l][k] = 0.0;
    double f2 = 0.0;
    if (!shared) {
      f2 = pair_factor<CC>(a, sr.tri, sc.tri);
      entry_sums<KER, BR, BC, Q, MP, PL>(a, sr.tri, sc.tri, Sre, Sim);
    }
    if constexpr (CC) {
      // entry (r, c) of the tile; pairs with common vertices are stored as
      // zero and completed by the singular kernel (fused: stored by the
      // singular pass below)
      if (FUSED && shared) continue;
      const size_t pos = T.out_off + (T.ntrans ? (size_t)c + (size_t)r * T.ld
                                               : (size_t)r + (size_t)c * T.ld);
      if constexpr (CPLX) {
        a.out[2 * pos] = f2 * Sre[0][0];
        a.out[2 * pos + 1] = conj ? -(f2 * Sim[0][0]) : f2 * Sim[0][0];
      } else {
        a.out[pos] = f2 * Sre[0][0];
      }
    } else if (!shared) {
#pragma unroll
      for (int l = 0; l < NR; l++) {
        const uint32_t lr = loc_of(sr.loc, l);
        if (lr == 0xffu) continue;
#pragma unroll
        for (int k = 0; k < NC; k++) {
          const uint32_t lc = loc_of(sc.loc, k);
          if (lc == 0xffu) continue;
          const int e = lr + TILE * lc;
          atomicAdd(&acc_re[e], f2 * Sre[l][k]);
          if constexpr (CPLX) atomicAdd(&acc_im[e], f2 * Sim[l][k]);
        }
      }
    }
  }

  if constexpr (FUSED) {
    if (!a.far) {
      constexpr int Q2 = 4;
      constexpr bool SMP = MP != 0;
      const SPair *L = tlist + T.sbeg;
      tile_singular<KER, BR, BC, CLS_IDENTICAL, Q2, SMP>(a, T, L, T.ns[0],
                                                         acc_re, acc_im);
      L += T.ns[0];
      tile_singular<KER, BR, BC, CLS_EDGE, Q2, SMP>(a, T, L, T.ns[1], acc_re,
                                                    acc_im);
      L += T.ns[1];
      tile_singular<KER, BR, BC, CLS_VERTEX, Q2, SMP>(a, T, L, T.ns[2],
                                                      acc_re, acc_im);
    }
  }
  if constexpr (!CC) {
    __syncthreads();
    const int nr = T.nr, nc = T.nc;
    for (int e = tid; e < nr * nc; e += NTHREADS) {
      const int i = e % nr, j = e / nr;
      const size_t pos =
          T.out_off + (T.ntrans ? (size_t)j + (size_t)i * T.ld
                                : (size_t)i + (size_t)j * T.ld);
      const int s = i + TILE * j;
      if constexpr (CPLX) {
        put(a, 2 * pos, acc_re[s], nslice);
        put(a, 2 * pos + 1, conj ? -acc_im[s] : acc_im[s], nslice);
      } else {
        put(a, pos, acc_re[s], nslice);
      }
    }
  }
}

// (The Helmholtz double layer with argument reduction takes 220 VGPRs, two
// waves per SIMD, where it is free to.)
template <int KER, int BR, int BC, int Q, int MP, int PL>
__global__ __launch_bounds__(NTHREADS,
                             KER == K_HELM_DLP && Q == 2 && MP == 0 ? 3 : 1)
void nf_regular_kernel(KArgs a) {
  regular_tile<KER, BR, BC, Q, MP, false, PL>(a, blockIdx.x / a.split, nullptr,
                                              blockIdx.x % a.split, a.split);
}

// Two mirrored tiles per workgroup: tile T = (rows R, columns C) and its
// mirror (C, R) of a plan whose blocks come in mirrored pairs over one index
// array, as the near field of a mesh does.  Every pair of triangles is
// evaluated once for both entries (pair_sums TWO): the single layers' entry
// is symmetric, the double layers share the distance, its root and the
// phase.  A diagonal tile is its own mirror: its n (n - 1) / 2 unordered
// pairs are taken by distance j = 1 .. n/2 around the list (r, r + j mod n),
// so no lane idles.  Constant basis: both entries are stored at once.
// Linear basis: the pairs' contributions are summed in LDS as in
// regular_tile, the double layers with a second accumulator for the mirror
// tile, and both tiles stored at the end.
//
// Bound by FP64 VALU issue (MP: VALU and the transcendental unit).  Threads
// per workgroup follow the LDS accumulators so that 4 to 5 waves per SIMD
// are resident: 256 for 32 KB, 512 for 64 KB.  Against one workgroup per
// tile (nf_regular_kernel): Laplace double layer, linear basis, 32768
// triangles 1431 -> 1011 us by this kernel alone and 822 with the points'
// factors; Helmholtz single layer, constant basis, 131072 triangles, all
// launches, 5230 -> 2490 us with it and the small phase (2050 to 2190 with
// the tiny one).  Constant basis: 4 waves where 5 spill (Laplace double
// layer, 12800 triangles 230 -> 177 us), 3 for the tiny-phase double layer
// (260 -> 244 us).
constexpr int pair_threads(int ker, int basis) {
  return pair_arrays(ker, basis) > 1 ? 512 : NTHREADS;
}
constexpr int pair_waves(int ker, int basis) {
  return ker == K_HELM_DLP_TP && !basis ? 3
         : (basis ? pair_arrays(ker, basis) > 1 : ker != K_LAP_SLP) ? 4
                                                                    : 5;
}

template <int KER, int B, int Q, int MP>
__global__ __launch_bounds__(pair_threads(KER, B),
                             pair_waves(KER, B)) void nf_pair_kernel(
    KArgs a, const uint32_t *__restrict__ list) {
  constexpr bool CPLX = KER >= K_HELM_SLP;
  constexpr bool DLP = is_dlp(KER);
  constexpr int NL = B ? 3 : 1;
  constexpr int NTH = pair_threads(KER, B);
  constexpr int NA = pair_arrays(KER, B);
  // re, (im), (re of the mirror), (im of the mirror)
  __shared__ double acc[NA ? NA * TILE * TILE : 1];
  // (adjoint double layers: S1 is the mirror's entry)
  const int mo = DLP ? (CPLX ? 2 : 1) * TILE * TILE : 0;
  double *const acc_re = acc + (a.adj ? mo : 0);
  double *const acc_im = acc_re + (CPLX ? TILE * TILE : 0);
  double *const mir_re = acc + (a.adj ? 0 : mo);
  double *const mir_im = mir_re + (CPLX ? TILE * TILE : 0);
  double *const s1_re = acc, *const s1_im = acc + (CPLX ? TILE * TILE : 0);
  double *const s2_re = acc + mo;
  double *const s2_im = s2_re + (CPLX ? TILE * TILE : 0);

  const int tid = threadIdx.x;
  const uint32_t slice = blockIdx.x % a.split, nslice = a.split;
  const uint32_t tile = list[blockIdx.x / nslice];
  const Tile T = a.tiles[tile];
  const bool diag = T.mirror == tile;
  const Tile M = a.tiles[T.mirror];
  const uint32_t nR = T.nrsup, nC = T.ncsup;
  const Supp *RS = a.supp + T.rsup;
  const Supp *CS = a.supp + T.csup;

  if constexpr (B) {
    for (int i = tid; i < NA * TILE * TILE; i += NTH) acc[i] = 0.0;
    __syncthreads();
  } else if (diag && slice == 0) {
    // identical triangles: completed by the singular kernel
    for (uint32_t r = tid; r < nR; r += NTH) {
      const size_t pos = T.out_off + r + (size_t)r * T.ld;
      if constexpr (CPLX)
        a.out[2 * pos] = a.out[2 * pos + 1] = 0.0;
      else
        a.out[pos] = 0.0;
    }
  }

  const uint32_t npairs = diag ? nR * (nR - 1) / 2 : nR * nC;
  const uint32_t p0 = tid + NTH * slice, step = NTH * nslice;
  const uint32_t dc = nR ? step / nR : 0, dr = step - dc * nR;
  uint32_t rr = nR ? p0 % nR : 0, cc = nR ? p0 / nR : 0;
  for (uint32_t p = p0; p < npairs; p += step) {
    const uint32_t r = rr;
    uint32_t c = cc;
    rr += dr;
    cc += dc;
    if (rr >= nR) {
      rr -= nR;
      cc++;
    }
    if (diag) {
      c += r + 1;
      c -= c >= nR ? nR : 0;
    }
    const Supp sr = RS[r], sc = CS[c];
    int shared = 0;
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
      for (int j = 0; j < 3; j++) shared += (sr.v[i] == sc.v[j]);
    double S1re[NL][NL], S1im[NL][NL], S2re[NL][NL], S2im[NL][NL];
    double f2 = 0.0;
    // constant basis: in the order of the triangle numbers, as entry_sums
    const bool sw = !B && sr.tri > sc.tri;
    if (!shared) {
      f2 = pair_factor<!B>(a, sr.tri, sc.tri);
      const uint32_t tt = sw ? sc.tri : sr.tri, ts = sw ? sr.tri : sc.tri;
      double nt[4] = {0.0, 0.0, 0.0, 0.0}, ns[4] = {0.0, 0.0, 0.0, 0.0};
      if constexpr (DLP) {
#pragma unroll
        for (int d = 0; d < 4; d++) {
          nt[d] = a.regn[4 * (size_t)tt + d];
          ns[d] = a.regn[4 * (size_t)ts + d];
        }
      }
      pair_sums<KER, B, B, Q, MP, DLP, 1>(a, tt, ts, nt, ns, false, 1.0, S1re,
                                       S1im, S2re, S2im);
    } else {
#pragma unroll
      for (int l = 0; l < NL; l++)
#pragma unroll
        for (int k = 0; k < NL; k++)
          S1re[l][k] = S1im[l][k] = S2re[l][k] = S2im[l][k] = 0.0;
    }
    if constexpr (!B) {
      // pairs with common vertices are stored as zero and completed by the
      // singular kernel
      const size_t pos = T.out_off + r + (size_t)c * T.ld;
      const size_t mpos = M.out_off + c + (size_t)r * M.ld;
      // S1 belongs to the order (tt, ts) (adjoint double layers: (ts, tt))
      const bool ex = DLP && (a.adj != 0) != sw;
      const double vre = f2 * (ex ? S2re[0][0] : S1re[0][0]);
      const double wre = DLP ? f2 * (ex ? S1re[0][0] : S2re[0][0]) : vre;
      if constexpr (CPLX) {
        const double vim = f2 * (ex ? S2im[0][0] : S1im[0][0]);
        const double wim = DLP ? f2 * (ex ? S1im[0][0] : S2im[0][0]) : vim;
        a.out[2 * pos] = vre;
        a.out[2 * pos + 1] = vim;
        a.out[2 * mpos] = wre;
        a.out[2 * mpos + 1] = wim;
      } else {
        a.out[pos] = vre;
        a.out[mpos] = wre;
      }
    } else if (!shared) {
#pragma unroll
      for (int l = 0; l < NL; l++) {
        const uint32_t lr = loc_of(sr.loc, l);
        if (lr == 0xffu) continue;
#pragma unroll
        for (int k = 0; k < NL; k++) {
          const uint32_t lc = loc_of(sc.loc, k);
          if (lc == 0xffu) continue;
          const int e = lr + TILE * lc;
          atomicAdd(&s1_re[e], f2 * S1re[l][k]);
          if constexpr (CPLX) atomicAdd(&s1_im[e], f2 * S1im[l][k]);
          if constexpr (DLP) {
            atomicAdd(&s2_re[e], f2 * S2re[l][k]);
            if constexpr (CPLX) atomicAdd(&s2_im[e], f2 * S2im[l][k]);
          }
        }
      }
    }
  }

  if constexpr (B) {
    // without a second accumulator mir_re is acc_re
    __syncthreads();
    const int nr = T.nr, nc = T.nc;
    for (int e = tid; e < nr * nc; e += NTH) {
      const int i = e % nr, j = e / nr;
      const int s = i + TILE * j, t = j + TILE * i;
      const size_t pos = T.out_off + (size_t)i + (size_t)j * T.ld;
      if constexpr (CPLX) {
        put(a, 2 * pos, acc_re[s] + (diag ? mir_re[t] : 0.0), nslice);
        put(a, 2 * pos + 1, acc_im[s] + (diag ? mir_im[t] : 0.0), nslice);
      } else {
        put(a, pos, acc_re[s] + (diag ? mir_re[t] : 0.0), nslice);
      }
    }
    if (!diag)
      for (int e = tid; e < nr * nc; e += NTH) {
        const int j = e % nc, i = e / nc;
        const int s = i + TILE * j;
        const size_t pos = M.out_off + (size_t)j + (size_t)i * M.ld;
        if constexpr (CPLX) {
          put(a, 2 * pos, mir_re[s], nslice);
          put(a, 2 * pos + 1, mir_im[s], nslice);
        } else {
          put(a, pos, mir_re[s], nslice);
        }
      }
  }
}

// Persistent form: a grid sized to the resident workgroups takes tiles from
// a counter (zeroed before the launch) until all ntiles are taken; every
// workgroup leaves the loop once the counter has passed ntiles.
template <int KER, int BR, int BC, int Q, int MP>
__global__ __launch_bounds__(NTHREADS) void nf_regular_persistent(
    KArgs a, uint32_t ntiles, uint32_t *counter) {
  __shared__ uint32_t cur;
  for (;;) {
    if (threadIdx.x == 0) cur = atomicAdd(counter, 1u);
    __syncthreads();
    const uint32_t t = cur;
    // every thread has read cur (and finished the previous tile's LDS
    // stores) before thread 0 takes the next one
    __syncthreads();
    if (t >= ntiles) break;
    regular_tile<KER, BR, BC, Q, MP>(a, t);
  }
}

// Regular and singular pairs of each tile in one workgroup (singular rule
// order 4): one workgroup per tile, or, persistent, a resident grid taking
// tiles from a counter as nf_regular_persistent does.  tlist: the singular
// pairs grouped by tile.
template <int KER, int BR, int BC, int Q, int MP>
__global__ __launch_bounds__(NTHREADS) void nf_fused_kernel(
    KArgs a, const SPair *__restrict__ tlist) {
  regular_tile<KER, BR, BC, Q, MP, true, 1>(a, blockIdx.x, tlist);
}

template <int KER, int BR, int BC, int Q, int MP>
__global__ __launch_bounds__(NTHREADS) void nf_fused_persistent(
    KArgs a, const SPair *__restrict__ tlist, uint32_t ntiles,
    uint32_t *counter) {
  __shared__ uint32_t cur;
  for (;;) {
    if (threadIdx.x == 0) cur = atomicAdd(counter, 1u);
    __syncthreads();
    const uint32_t t = cur;
    __syncthreads();
    if (t >= ntiles) break;
    regular_tile<KER, BR, BC, Q, MP, true, 1>(a, t, tlist);
  }
}

// Sauter-Schwab points of one tensor tuple (g_i, g_j, g_k, g_l) with
// weights (w_i, w_j, w_k, w_l): the 2 (vertex) or 6 (edge, identical)
// subregion points (tx, sx; ty, sy) and their common weight, exactly as the
// tables of the reference are built (Library/singquad2d.c:80-281).
template <int CLS>
struct SSTuple;

template <>
struct SSTuple<CLS_VERTEX> {
  static constexpr int N = 2;
  template <class F>
  __device__ __forceinline__ static void run(double gi, double gj, double gk,
                                             double gl, double wi, double wj,
                                             double wk, double wl, F &&f) {
    const double e1 = gi, e2 = gj, e3 = gk, xi = gl;
    const double w = wi * wj * wk * wl * xi * xi * xi * e1;
    const double a = e2 * xi, b = e1 * xi, c = e1 * e3 * xi;
    f(w, xi, a, b, c);
    f(w, b, c, xi, a);
  }
};

template <>
struct SSTuple<CLS_EDGE> {
  static constexpr int N = 6;
  template <class F>
  __device__ __forceinline__ static void run(double gi, double gj, double gk,
                                             double gl, double wi, double wj,
                                             double wk, double wl, F &&f) {
    const double e1 = gi, e2 = gj, x1 = gk;
    const double x2 = gl * (1.0 - x1);
    const double w = wi * wj * wk * (wl * (1.0 - x1)) * x1 * x1 * e1;
    const double s = x1 + x2;
    const double p = x1 * e1, pq = x1 * e1 * e2;
    f(w, s, pq, x1 * (1.0 - e1) + x2, x1 * (1.0 - e1));
    f(w, s, p, x1 * (1.0 - e1 * e2) + x2, x1 * (1.0 - e1 * e2));
    f(w, s, x1, p + x2, pq);
    f(w, x1 * (1.0 - e1 + e1 * e2) + x2, pq, s, x1);
    f(w, pq + x2, pq, s, p);
    f(w, p + x2, p, s, pq);
  }
};

template <>
struct SSTuple<CLS_IDENTICAL> {
  static constexpr int N = 6;
  template <class F>
  __device__ __forceinline__ static void run(double gi, double gj, double gk,
                                             double gl, double wi, double wj,
                                             double wk, double wl, F &&f) {
    const double eta = gi, x1 = gj;
    const double x2 = gk * (1.0 - x1);
    const double x3 = gl * (1.0 - x1 - x2);
    const double w = wi * wj * (wk * (1.0 - x1)) * (wl * (1.0 - x1 - x2)) * x1;
    const double a = x1 + x2 + x3;
    const double b = x1 * (1.0 - eta);
    f(w, a, x1 + x2, b + x2 + x3, x2);
    f(w, b + x2 + x3, b + x2, a, x2);
    f(w, a, x1 * eta + x2, x2 + x3, x2);
    f(w, b + x2 + x3, x2, a, x1 + x2);
    f(w, a, x2, b + x2 + x3, b + x2);
    f(w, x2 + x3, x2, a, x1 * eta + x2);
  }
};

// sum over the 16 lanes of a row
__device__ __forceinline__ double row_sum(double v) {
#pragma unroll
  for (int off = 8; off > 0; off >>= 1) v += __shfl_xor(v, off, 16);
  return v;
}

// element i (0..2) of a three-vector by selects (a dynamic index would put
// the vector in private memory)
template <class V>
__device__ __forceinline__ V sel3(const V (&v)[3], int i) {
  return i == 0 ? v[0] : (i == 1 ? v[1] : v[2]);
}

// One pair with common vertices per row of 16 lanes.  Lane s of the row
// takes the tensor index pairs (k, l) = (s / q2, s % q2), (s + 16) / q2, ...
// and loops over (i, j); the quadrature points are formed on the fly from
// the Gauss nodes (a.gauss = [g | w], q2 each), so no rule tables are read.
// The row's lanes sum their moments; lanes e < NR NC then hand the entry
// (lr, lc) of the tile (tile-local row and column) to sink(lr, lc, re, im):
// global atomics for the launches per rule class, the tile's LDS
// accumulator (or a plain store, constant basis) when the tile's own
// workgroup evaluates its singular pairs.  The value is not conjugated.
//
// MIR: the entry of the exchanged pair (the column triangle as the row, in
// the mirror tile) as well; sink(lr, lc, re, im, re2, im2).  The vertex
// rule's two points of a tuple and the identical rule's six map onto each
// other when the triangles are exchanged, so the exchanged pair has the
// same points and the same moments, of the kernel with the other normal
// (single layer: the same values).  The edge rule has no such symmetry.
//
// PL: the normals are perpendicular to the triangles and no triangles fold
// back on each other (a.plane), so <d, n> may be formed from them.
template <int KER, int BR, int BC, int CLS, int Q2, bool MP, bool MIR,
          bool PL, class Sink>
__device__ __forceinline__ void singular_pair(const KArgs &a, const Tile &T,
                                              const SPair &P, int sub,
                                              Sink &&sink) {
  constexpr bool CPLX = KER >= K_HELM_SLP;
  constexpr bool DLP = is_dlp(KER);
  constexpr bool CC = (BR == 0) && (BC == 0);
  constexpr int NR = BR ? 3 : 1;
  constexpr int NC = BC ? 3 : 1;
  static_assert(!MIR || CLS != CLS_EDGE, "the edge rule is not symmetric");
  // directions summed: both only where the values differ beyond the sign
  constexpr bool TWO = MIR && DLP && CLS == CLS_VERTEX;
  constexpr int ND = TWO ? 2 : 1;

  const Supp sr = a.supp[T.rsup + P.r], sc = a.supp[T.csup + P.c];
  int tp[3], sp[3];
#pragma unroll
  for (int i = 0; i < 3; i++) {
    tp[i] = (P.perm >> (2 * i)) & 3;
    sp[i] = (P.perm >> (6 + 2 * i)) & 3;
  }
  // constant basis: in the order of the triangle numbers, as entry_sums
  const bool sw = CC && CLS == CLS_VERTEX && sr.tri > sc.tri;
  uint32_t tv[3], sv[3];
#pragma unroll
  for (int i = 0; i < 3; i++) {
    const uint32_t tvi = sel3(sr.v, tp[i]), svi = sel3(sc.v, sp[i]);
    tv[i] = sw ? svi : tvi;
    sv[i] = sw ? tvi : svi;
  }
  double D0[3], E1[3], E2[3], F1[3], F2[3];
#pragma unroll
  for (int d = 0; d < 3; d++) {
    const double At = a.x[3 * tv[0] + d], Bt = a.x[3 * tv[1] + d],
                 Ct = a.x[3 * tv[2] + d];
    const double As = a.x[3 * sv[0] + d], Bs = a.x[3 * sv[1] + d],
                 Cs = a.x[3 * sv[2] + d];
    D0[d] = At - As;
    E1[d] = Bt - At;
    E2[d] = Ct - Bt;
    F1[d] = Bs - As;
    F2[d] = Cs - Bs;
  }
  // normals of the entry and of the exchanged pair, for d = x - y
  double n1[3] = {0.0, 0.0, 0.0}, n2[3] = {0.0, 0.0, 0.0};
  if constexpr (DLP) {
    layer_normal(a, sr.tri, sc.tri, n1);
    if constexpr (TWO) layer_normal(a, sc.tri, sr.tri, n2);
#pragma unroll
    for (int d = 0; d < 3; d++) {
      n1[d] = sw ? -n1[d] : n1[d];
      n2[d] = sw ? n2[d] : -n2[d];
    }
  }
  double Sre[ND][NR][NC], Sim[ND][NR][NC];
#pragma unroll
  for (int z = 0; z < ND; z++)
#pragma unroll
    for (int l = 0; l < NR; l++)
#pragma unroll
      for (int k = 0; k < NC; k++) Sre[z][l][k] = Sim[z][l][k] = 0.0;

  // Moments M[a][b] = sum w v m_a(x) m_b(y) with m = (1, tx, sx) resp.
  // (1, ty, sy); the linear basis functions are phi = (1 - tx, tx - sx, sx)
  // = A m, so the element matrix A M A^T is formed once after the sum.
  // kernel values at the difference d (FP64; mixed precision: d in FP64,
  // the value in FP32)
  // w: the weight, one product with both parts of a complex value; m: the
  // products <d, n> per direction where the caller has them (double layers,
  // FP64, PLANE)
  auto value = [&](const double *d, double w, const double *m,
                   double (&vre)[ND], double (&vim)[ND]) {
    if constexpr (MP) {
      const float dx = (float)d[0], dy = (float)d[1], dz = (float)d[2];
      float g, fr, fi;
      kcore32<KER>(fmaf(dx, dx, fmaf(dy, dy, dz * dz)), a.krf, a.krev,
                   a.kil2, g, fr, fi);
#pragma unroll
      for (int z = 0; z < ND; z++) {
        const double *n = z ? n2 : n1;
        float v = g;
        if constexpr (DLP)
          v *= fmaf(dx, (float)n[0], fmaf(dy, (float)n[1], dz * (float)n[2]));
        vre[z] = w * (CPLX ? fr * v : v);
        vim[z] = CPLX ? w * (fi * v) : 0.0;
      }
    } else {
      double g, fr, fi;
      kcore<KER>(fma(d[0], d[0], fma(d[1], d[1], d[2] * d[2])), a.kr, a.ki,
                 0.0, g, fr, fi);
#pragma unroll
      for (int z = 0; z < ND; z++) {
        const double *n = z ? n2 : n1;
        double v = w * g;
        if constexpr (DLP)
          v *= m ? m[z] : fma(d[0], n[0], fma(d[1], n[1], d[2] * n[2]));
        vre[z] = CPLX ? fr * v : v;
        vim[z] = CPLX ? fi * v : 0.0;
      }
    }
  };
  auto point = [&](double wq, double tx, double sx, double ty, double sy) {
    double d[3];
#pragma unroll
    for (int k = 0; k < 3; k++)
      d[k] = fma(-F2[k], sy,
                 fma(-F1[k], ty, fma(E2[k], sx, fma(E1[k], tx, D0[k]))));
    double vre[ND], vim[ND];
    value(d, wq, nullptr, vre, vim);
    double ure[NR], uim[NR];
    ure[0] = vre[0];
    uim[0] = vim[0];
    if constexpr (BR) {
      ure[1] = ure[0] * tx;
      ure[2] = ure[0] * sx;
      uim[1] = uim[0] * tx;
      uim[2] = uim[0] * sx;
    }
#pragma unroll
    for (int l = 0; l < NR; l++) {
      Sre[0][l][0] += ure[l];
      if constexpr (CPLX) Sim[0][l][0] += uim[l];
      if constexpr (BC) {
        Sre[0][l][1] = fma(ure[l], ty, Sre[0][l][1]);
        Sre[0][l][2] = fma(ure[l], sy, Sre[0][l][2]);
        if constexpr (CPLX) {
          Sim[0][l][1] = fma(uim[l], ty, Sim[0][l][1]);
          Sim[0][l][2] = fma(uim[l], sy, Sim[0][l][2]);
        }
      }
    }
  };

  // PL, the rules of order 4: the double layers vanish on identical
  // triangles, whose differences lie in their plane, and on a common edge
  // <d, n> is one coordinate of the other triangle's point times a constant.
  // (Vertex pairs keep the products: the same there takes more registers,
  // 222 -> 254 us for the double layer at 32768 triangles.)
  constexpr bool PLANE = DLP && !MP && Q2 > 0 && PL;
  auto dot = [](const double (&u)[3], const double (&v)[3]) {
    return fma(u[0], v[0], fma(u[1], v[1], u[2] * v[2]));
  };
  if constexpr (PLANE && CLS == CLS_IDENTICAL) {
  } else if constexpr (Q2 > 0) {
    // order known at compile time (Q2^2 <= 16): one (k, l) per lane, the
    // nodes in registers, the (i, j) loops unrolled.  Not the Helmholtz
    // double layer with argument reduction in FP64: its evaluations are long
    // enough that 24 of them interleaved take up to 360 registers, one wave
    // per SIMD, so its loops (two, six or three evaluations a turn) stay
    // loops: 134 to 232 registers (constant basis), two to three waves.
    // Cylinder of 46240 triangles (no mirrored tiles), constant / linear
    // basis 2.54 -> 2.06 / 11.16 -> 10.19 ms (2.34 / 11.04 before the
    // branch-free sine and cosine let the compiler interleave them), sphere of
    // 3872, linear basis, k = 5, mirrored tiles 679 -> 617 us.
    static_assert(Q2 * Q2 <= 16, "one tensor index pair per lane");
    constexpr bool LONG = KER == K_HELM_DLP && !MP;
    constexpr int UN = LONG ? 1 : Q2;
    double gn[Q2], gw[Q2];
#pragma unroll
    for (int i = 0; i < Q2; i++) {
      gn[i] = a.gauss[i];
      gw[i] = a.gauss[Q2 + i];
    }
    // node and weight i, read again where the loop is not unrolled
    auto node = [&](int i) { return LONG ? a.gauss[i] : gn[i]; };
    auto weight = [&](int i) { return LONG ? a.gauss[Q2 + i] : gw[i]; };
    if (sub < Q2 * Q2) {
      const int k = sub / Q2, l = sub % Q2;
      const double gk = a.gauss[k], gl = a.gauss[l];
      const double wk = a.gauss[Q2 + k], wl = a.gauss[Q2 + l];
      if constexpr (CLS == CLS_VERTEX) {
        // The two points of a tuple (SSTuple<CLS_VERTEX>) with e1 = g_i,
        // e2 = g_j, e3 = g_k, xi = g_l:
        //   P1 (tx, sx, ty, sy) = (xi, e2 xi, e1 xi, e1 e3 xi)
        //   P2 (tx, sx, ty, sy) = (e1 xi, e1 e3 xi, xi, e2 xi)
        // so d = D0 + xi (E1 + E2 e2 - (F1 + F2 e3) e1) for P1 and
        // d = D0 + xi ((E1 + E2 e3) e1 - F1 - F2 e2) for P2: affine in e2
        // for fixed i.  In P1 the column moments (1, ty, sy) do not depend
        // on j and the row moments (1, tx, sx) are affine in e2 (P2 the
        // other way round), so the sums over j need only sum u and sum u e2
        // per point, and the moment matrix is updated once per i.
        const double e3 = gk, xi = gl;
        const double wkl = wk * wl * xi * xi * xi;
        double a1[3], b1[3], c1[3], a2[3], b2[3], c2[3];
#pragma unroll
        for (int d = 0; d < 3; d++) {
          a1[d] = fma(xi, E1[d], D0[d]);
          b1[d] = xi * E2[d];
          c1[d] = xi * fma(F2[d], e3, F1[d]);
          a2[d] = fma(-xi, F1[d], D0[d]);
          b2[d] = xi * fma(E2[d], e3, E1[d]);
          c2[d] = -xi * F2[d];
        }
#pragma unroll UN
        for (int i = 0; i < Q2; i++) {
          const double e1 = node(i);
          const double wi1 = wkl * weight(i) * e1;
          double t1[3], t2[3];
#pragma unroll
          for (int d = 0; d < 3; d++) {
            t1[d] = fma(-c1[d], e1, a1[d]);
            t2[d] = fma(b2[d], e1, a2[d]);
          }
          double U0r[ND], U0i[ND], U2r[ND], U2i[ND];
          double V0r[ND], V0i[ND], V2r[ND], V2i[ND];
#pragma unroll
          for (int z = 0; z < ND; z++)
            U0r[z] = U0i[z] = U2r[z] = U2i[z] = V0r[z] = V0i[z] = V2r[z] =
                V2i[z] = 0.0;
#pragma unroll UN
          for (int j = 0; j < Q2; j++) {
            const double e2 = node(j), w = wi1 * weight(j);
            double d1[3], d2[3];
#pragma unroll
            for (int d = 0; d < 3; d++) {
              d1[d] = fma(b1[d], e2, t1[d]);
              d2[d] = fma(c2[d], e2, t2[d]);
            }
            double v1r[ND], v1i[ND], v2r[ND], v2i[ND];
            value(d1, w, nullptr, v1r, v1i);
            value(d2, w, nullptr, v2r, v2i);
#pragma unroll
            for (int z = 0; z < ND; z++) {
              const double u1r = v1r[z], u2r = v2r[z];
              U0r[z] += u1r;
              U2r[z] = fma(u1r, e2, U2r[z]);
              V0r[z] += u2r;
              V2r[z] = fma(u2r, e2, V2r[z]);
              if constexpr (CPLX) {
                const double u1i = v1i[z], u2i = v2i[z];
                U0i[z] += u1i;
                U2i[z] = fma(u1i, e2, U2i[z]);
                V0i[z] += u2i;
                V2i[z] = fma(u2i, e2, V2i[z]);
              }
            }
          }
          // P1: row moments (U0, xi U0, xi U2), column moments
          // (1, e1 xi, e1 e3 xi); P2: row moments (1, e1 xi, e1 e3 xi),
          // column moments (V0, xi V0, xi V2)
          const double f1 = e1 * xi, f2 = e1 * e3 * xi;
          const double ms[3] = {1.0, f1, f2};
#pragma unroll
          for (int z = 0; z < ND; z++) {
            const double p1r[3] = {U0r[z], xi * U0r[z], xi * U2r[z]};
            const double p1i[3] = {U0i[z], xi * U0i[z], xi * U2i[z]};
            const double p2r[3] = {V0r[z], xi * V0r[z], xi * V2r[z]};
            const double p2i[3] = {V0i[z], xi * V0i[z], xi * V2i[z]};
#pragma unroll
            for (int l = 0; l < NR; l++)
#pragma unroll
              for (int kk = 0; kk < NC; kk++) {
                Sre[z][l][kk] = fma(p1r[l], ms[kk], Sre[z][l][kk]);
                Sre[z][l][kk] = fma(ms[l], p2r[kk], Sre[z][l][kk]);
                if constexpr (CPLX) {
                  Sim[z][l][kk] = fma(p1i[l], ms[kk], Sim[z][l][kk]);
                  Sim[z][l][kk] = fma(ms[l], p2i[kk], Sim[z][l][kk]);
                }
              }
          }
        }
      } else if constexpr (CLS == CLS_EDGE) {
        // The six points of SSTuple<CLS_EDGE> with e1 = g_i, e2 = g_j,
        // x1 = g_k, x2 = g_l (1 - x1), s = x1 + x2, p = x1 e1, pq = p e2:
        //   (tx, sx, ty, sy) = (s, pq, s - p, x1 - p), (s, p, s - pq, x1 - pq),
        //   (s, x1, p + x2, pq), (s - p + pq, pq, s, x1), (pq + x2, pq, s, p),
        //   (p + x2, p, s, pq).
        // The pair's first two (permuted) vertices are the shared ones, so
        // D0 = 0 and E1 = F1: d = E1 (tx - ty) + E2 sx - F2 sy is affine in
        // pq for fixed i.  In every point one side's moments are fixed for
        // fixed i and the other side's affine in pq, so the sums over j need
        // sum u and sum u pq per point and the moment matrix is updated once
        // per i.
        const double x1 = gk, x2 = gl * (1.0 - x1), s_ = x1 + x2;
        const double wkl = wk * (wl * (1.0 - x1)) * x1 * x1;
        // PLANE: <d, n of the column triangle> = <E2, n> sx, <d, -n of the
        // row triangle> = <F2, n> sy (the shared edge E1 = F1 lies in both)
        double ka = 0.0;
        if constexpr (PLANE) {
          const uint32_t t = a.adj ? sr.tri : sc.tri;
          const double nv[3] = {a.n[3 * t], a.n[3 * t + 1], a.n[3 * t + 2]};
          ka = a.adj ? dot(F2, nv) : dot(E2, nv);
        }
        // d = base + cp p + cq pq per point m
        double cA[3], cB[3], cC[3], Gv[3], Hv[3];
#pragma unroll
        for (int d = 0; d < 3; d++) {
          cA[d] = -F2[d] * x1;
          cB[d] = (E1[d] + E2[d]) * x1;
          cC[d] = -E1[d] * x1;
          Gv[d] = E1[d] + F2[d];
          Hv[d] = E1[d] + E2[d];
        }
#pragma unroll 1
        for (int i = 0; i < Q2; i++) {
          const double e1 = gn[i];
          const double wi1 = wkl * gw[i] * e1;
          const double p = x1 * e1;
          double bs[6][3];
#pragma unroll
          for (int d = 0; d < 3; d++) {
            bs[0][d] = fma(Gv[d], p, cA[d]);
            bs[1][d] = fma(E2[d], p, cA[d]);
            bs[2][d] = fma(-E1[d], p, cB[d]);
            bs[3][d] = fma(-E1[d], p, cA[d]);
            bs[4][d] = fma(-F2[d], p, cC[d]);
            bs[5][d] = fma(Hv[d], p, cC[d]);
          }
          double W0r[6], W1r[6], W0i[6], W1i[6];
#pragma unroll
          for (int m = 0; m < 6; m++) W0r[m] = W1r[m] = W0i[m] = W1i[m] = 0.0;
#pragma unroll UN
          for (int j = 0; j < Q2; j++) {
            const double pq = p * node(j), w = wi1 * weight(j);
#pragma unroll
            for (int m = 0; m < 6; m++) {
              double dd[3];
#pragma unroll
              for (int d = 0; d < 3; d++) {
                const double cq = m == 0 ? E2[d]
                                : m == 1 ? Gv[d]
                                : m == 2 ? -F2[d]
                                : m == 5 ? -F2[d]
                                         : Hv[d];
                dd[d] = fma(cq, pq, bs[m][d]);
              }
              double vr[ND], vi[ND];
              if constexpr (PLANE) {
                // the point's product: c0 + c1 pq, one of both zero in all
                // but one point of the adjoint; constants and kappa are
                // applied after the sums
                const double mm = a.adj ? (m == 1   ? x1 - pq
                                           : m == 2 ? pq
                                           : m == 5 ? pq
                                                    : 1.0)
                                        : (m == 0 || m == 3 || m == 4 ? pq
                                                                      : 1.0);
                value(dd, w, &mm, vr, vi);
              } else {
                value(dd, w, nullptr, vr, vi);
              }
              const double ur = vr[0];
              W0r[m] += ur;
              W1r[m] = fma(ur, pq, W1r[m]);
              if constexpr (CPLX) {
                const double ui = vi[0];
                W0i[m] += ui;
                W1i[m] = fma(ui, pq, W1i[m]);
              }
            }
          }
          if constexpr (PLANE) {
            const double fA[6] = {ka, p * ka, x1 * ka, ka, ka, p * ka};
            const double fB[6] = {(x1 - p) * ka, ka, ka, x1 * ka, p * ka, ka};
#pragma unroll
            for (int m = 0; m < 6; m++) {
              const double f = a.adj ? fB[m] : fA[m];
              W0r[m] *= f;
              W1r[m] *= f;
              if constexpr (CPLX) {
                W0i[m] *= f;
                W1i[m] *= f;
              }
            }
          }
          // row-affine points (1, 4, 5): M += T (x) ms; column-affine
          // points (2, 3, 6): M += mt (x) S
          const double ms1[3] = {1.0, s_ - p, x1 - p};
          const double ms4[3] = {1.0, s_, x1};
          const double ms5[3] = {1.0, s_, p};
          const double mt2[3] = {1.0, s_, p};
          const double mt3[3] = {1.0, s_, x1};
          const double mt6[3] = {1.0, p + x2, p};
          auto accum = [&](const double *W0, const double *W1, double (&Sx)[NR][NC]) {
            const double T1[3] = {W0[0], s_ * W0[0], W1[0]};
            const double S2[3] = {W0[1], s_ * W0[1] - W1[1],
                                  x1 * W0[1] - W1[1]};
            const double S3[3] = {W0[2], (p + x2) * W0[2], W1[2]};
            const double T4[3] = {W0[3], (s_ - p) * W0[3] + W1[3], W1[3]};
            const double T5[3] = {W0[4], x2 * W0[4] + W1[4], W1[4]};
            const double S6[3] = {W0[5], s_ * W0[5], W1[5]};
#pragma unroll
            for (int l = 0; l < NR; l++)
#pragma unroll
              for (int kk = 0; kk < NC; kk++) {
                double t = Sx[l][kk];
                t = fma(T1[l], ms1[kk], t);
                t = fma(mt2[l], S2[kk], t);
                t = fma(mt3[l], S3[kk], t);
                t = fma(T4[l], ms4[kk], t);
                t = fma(T5[l], ms5[kk], t);
                t = fma(mt6[l], S6[kk], t);
                Sx[l][kk] = t;
              }
          };
          accum(W0r, W1r, Sre[0]);
          if constexpr (CPLX) accum(W0i, W1i, Sim[0]);
        }
      } else {
        // The six points of SSTuple<CLS_IDENTICAL> with eta = g_i,
        // x1 = g_j, x2 = g_k (1 - x1), x3 = g_l (1 - x1 - x2),
        // a = x1 + x2 + x3, b = x1 (1 - eta):
        //   (tx, sx, ty, sy) = (a, x1 + x2, b + x2 + x3, x2),
        //   (b + x2 + x3, b + x2, a, x2), (a, x1 eta + x2, x2 + x3, x2),
        //   (b + x2 + x3, x2, a, x1 + x2), (a, x2, b + x2 + x3, b + x2),
        //   (x2 + x3, x2, a, x1 eta + x2).
        // Both triangles are the same (D0 = 0, E1 = F1, E2 = F2), so
        // d = E1 (tx - ty) + E2 (sx - sy) = x1 u with
        // u = eta E1 + E2, -eta E1 + (1 - eta) E2, E1 + eta E2 and their
        // negatives: the difference is formed without cancellation.  For
        // fixed j one side's moments are fixed and the other's affine in b,
        // so the sums over i need sum u and sum u b per point.
#pragma unroll 1
        for (int j = 0; j < Q2; j++) {
          const double x1 = gn[j];
          const double x2 = gk * (1.0 - x1);
          const double x3 = gl * (1.0 - x1 - x2);
          const double aa = x1 + x2 + x3;
          const double wj1 = gw[j] * (wk * (1.0 - x1)) *
                             (wl * (1.0 - x1 - x2)) * x1;
          double W0r[6], W1r[6], W0i[6], W1i[6];
#pragma unroll
          for (int m = 0; m < 6; m++) W0r[m] = W1r[m] = W0i[m] = W1i[m] = 0.0;
#pragma unroll UN
          for (int i = 0; i < Q2; i++) {
            const double eta = node(i), w = weight(i) * wj1;
            const double bb = x1 * (1.0 - eta);
            double dv[3][3], pr[3], pi[3];
#pragma unroll
            for (int d = 0; d < 3; d++) {
              dv[0][d] = x1 * fma(eta, E1[d], E2[d]);
              dv[1][d] = x1 * fma(1.0 - eta, E2[d], -eta * E1[d]);
              dv[2][d] = x1 * fma(eta, E2[d], E1[d]);
            }
#pragma unroll
            for (int m = 0; m < 6; m++) {
              // point order: P1 = +u1, P2 = +u2, P3 = +u3, P4 = -u1,
              // P5 = -u2, P6 = -u3; the kernels take -u to the same value
              // (single layer) or to its negative (double layer)
              double vr[ND], vi[ND];
              if (m < 3) {
                value(dv[m], w, nullptr, vr, vi);
                pr[m] = vr[0];
                pi[m] = vi[0];
              } else {
                vr[0] = DLP ? -pr[m - 3] : pr[m - 3];
                vi[0] = DLP ? -pi[m - 3] : pi[m - 3];
              }
              const double ur = vr[0];
              W0r[m] += ur;
              W1r[m] = fma(ur, bb, W1r[m]);
              if constexpr (CPLX) {
                const double ui = vi[0];
                W0i[m] += ui;
                W1i[m] = fma(ui, bb, W1i[m]);
              }
            }
          }
          // m = 0: P1, 1: P2, 2: P3, 3: P4, 4: P5, 5: P6
          const double x23 = x2 + x3, x12 = x1 + x2;
          const double mt1[3] = {1.0, aa, x12};
          const double ms2[3] = {1.0, aa, x2};
          const double ms3[3] = {1.0, x23, x2};
          const double ms4[3] = {1.0, aa, x12};
          const double mt5[3] = {1.0, aa, x2};
          const double mt6[3] = {1.0, x23, x2};
          auto accum = [&](const double *W0, const double *W1,
                           double (&Sx)[NR][NC]) {
            const double S1[3] = {W0[0], fma(x23, W0[0], W1[0]), x2 * W0[0]};
            const double T2[3] = {W0[1], fma(x23, W0[1], W1[1]),
                                  fma(x2, W0[1], W1[1])};
            const double T3[3] = {W0[2], aa * W0[2], fma(x12, W0[2], -W1[2])};
            const double T4[3] = {W0[3], fma(x23, W0[3], W1[3]), x2 * W0[3]};
            const double S5[3] = {W0[4], fma(x23, W0[4], W1[4]),
                                  fma(x2, W0[4], W1[4])};
            const double S6[3] = {W0[5], aa * W0[5], fma(x12, W0[5], -W1[5])};
#pragma unroll
            for (int l = 0; l < NR; l++)
#pragma unroll
              for (int kk = 0; kk < NC; kk++) {
                double t = Sx[l][kk];
                t = fma(mt1[l], S1[kk], t);
                t = fma(T2[l], ms2[kk], t);
                t = fma(T3[l], ms3[kk], t);
                t = fma(T4[l], ms4[kk], t);
                t = fma(mt5[l], S5[kk], t);
                t = fma(mt6[l], S6[kk], t);
                Sx[l][kk] = t;
              }
          };
          accum(W0r, W1r, Sre[0]);
          if constexpr (CPLX) accum(W0i, W1i, Sim[0]);
        }
      }
    }
  } else {
    const uint32_t q2 = a.q2;
    const double *__restrict__ gn = a.gauss;
    const double *__restrict__ gw = a.gauss + q2;
    for (uint32_t kl = sub; kl < q2 * q2; kl += 16) {
      const uint32_t k = kl / q2, l = kl - k * q2;
      const double gk = gn[k], gl = gn[l], wk = gw[k], wl = gw[l];
      for (uint32_t i = 0; i < q2; i++) {
        const double gi = gn[i], wi = gw[i];
        for (uint32_t j = 0; j < q2; j++)
          SSTuple<CLS>::run(gi, gn[j], gk, gl, wi, gw[j], wk, wl, point);
      }
    }
  }
#pragma unroll
  for (int z = 0; z < ND; z++) {
#pragma unroll
    for (int l = 0; l < NR; l++)
#pragma unroll
      for (int k = 0; k < NC; k++) {
        Sre[z][l][k] = row_sum(Sre[z][l][k]);
        if constexpr (CPLX) Sim[z][l][k] = row_sum(Sim[z][l][k]);
      }
    // moments -> element matrix: (1, t, s) -> (1 - t, t - s, s) on each side
    if constexpr (BR) {
#pragma unroll
      for (int k = 0; k < NC; k++) {
        Sre[z][0][k] -= Sre[z][1][k];
        Sre[z][1][k] -= Sre[z][2][k];
        if constexpr (CPLX) {
          Sim[z][0][k] -= Sim[z][1][k];
          Sim[z][1][k] -= Sim[z][2][k];
        }
      }
    }
    if constexpr (BC) {
#pragma unroll
      for (int l = 0; l < NR; l++) {
        Sre[z][l][0] -= Sre[z][l][1];
        Sre[z][l][1] -= Sre[z][l][2];
        if constexpr (CPLX) {
          Sim[z][l][0] -= Sim[z][l][1];
          Sim[z][l][1] -= Sim[z][l][2];
        }
      }
    }
  }
  if (sub >= NR * NC) return;
  // lane e hands over the entry of permuted local functions (l, k) =
  // (e % NR, e / NR)
  const int l = sub % NR, k = sub / NR;
  double vre[2] = {0.0, 0.0}, vim[2] = {0.0, 0.0};
#pragma unroll
  for (int z = 0; z < ND; z++)
#pragma unroll
    for (int ll = 0; ll < NR; ll++)
#pragma unroll
      for (int kk = 0; kk < NC; kk++)
        if (ll == l && kk == k) {
          vre[z] = Sre[z][ll][kk];
          vim[z] = Sim[z][ll][kk];
        }
  if constexpr (MIR && !TWO) {
    // single layer: the same sums; identical triangles, double layer: the
    // differences change sign and the normal does not
    vre[1] = DLP ? -vre[0] : vre[0];
    vim[1] = DLP ? -vim[0] : vim[0];
  }
  const uint32_t lr = loc_of(sr.loc, BR ? sel3(tp, l) : 0);
  const uint32_t lc = loc_of(sc.loc, BC ? sel3(sp, k) : 0);
  if (lr == 0xffu || lc == 0xffu) return;
  const double gt = a.g[sr.tri];
  const double f2 = pair_factor<CC>(a, sr.tri, sc.tri);
#pragma unroll
  for (int z = 0; z < 2; z++) {
    vre[z] *= f2;
    vim[z] *= f2;
  }
  if constexpr (CLS == CLS_IDENTICAL) {
    // identity term of the double layer on identical triangles (tp, sp are
    // the identity here): cc at (t, t) of the block
    // (Library/bem3d.c:1234-1241), otherwise Re(alpha) g mass[l, k]
    // (Library/bem3d.c:3205-3242, 1934-1966, 2530-2562)
    if constexpr (CC) {
      if (T.row0 + lr == T.col0 + lc) {
        vre[0] += 0.5 * a.are * gt;
        vim[0] += 0.5 * a.aim * gt;
      }
    } else {
      // the linear-basis integrators hold alpha g in a real variable
      // (Library/bem3d.c:1822-1823, 2418-2419, 3061-3062): only Re(alpha)
      // reaches the mass term
      const bool allowed = (BR && !BC) ? (T.flags & 1) : true;
      if (allowed) {
        const double m = (BR && BC) ? a.mass[l + 3 * k] : a.mass[BR ? l : k];
        vre[0] += m * a.are * gt;
        vre[1] += m * a.are * gt;  // the mass matrix is symmetric
      }
    }
  }
  sink(lr, lc, vre[0], vim[0], vre[1], vim[1]);
}

// The pairs with common vertices of one rule class, one pair per row of 16
// lanes (16 pairs per workgroup), added into the output with FP64 atomics
// (the regular kernel has stored the tiles before).
// MIR: the list holds one of each two exchanged pairs; the other's entry is
// added into the mirror tile.
template <int KER, int BR, int BC, int CLS, int Q2, bool MP, bool MIR,
          bool PL>
__device__ __forceinline__ void singular_list(const KArgs &a,
                                              const SPair *__restrict__ list,
                                              uint32_t npairs,
                                              uint32_t block) {
  constexpr bool CPLX = KER >= K_HELM_SLP;
  const uint32_t w = block * (NTHREADS / 16) + (threadIdx.x >> 4);
  const int sub = threadIdx.x & 15;
  if (w >= npairs) return;  // uniform per row of 16 lanes
  const SPair P = list[w];
  const Tile T = a.tiles[P.tile];
  const bool conj = T.ntrans && (BR == BC);
  // identical triangles of a diagonal tile have no exchanged pair
  const bool mir =
      MIR && !(CLS == CLS_IDENTICAL && T.mirror == P.tile);
  singular_pair<KER, BR, BC, CLS, Q2, MP, MIR, PL>(
      a, T, P, sub,
      [&](uint32_t lr, uint32_t lc, double vre, double vim, double vre2,
          double vim2) {
        const size_t pos =
            T.out_off + (T.ntrans ? (size_t)lc + (size_t)lr * T.ld
                                  : (size_t)lr + (size_t)lc * T.ld);
        if constexpr (CPLX) {
          atomicAdd(&a.out[2 * pos], vre);
          atomicAdd(&a.out[2 * pos + 1], conj ? -vim : vim);
        } else {
          atomicAdd(&a.out[pos], vre);
        }
        if (mir) {
          const Tile &M = a.tiles[T.mirror];
          const size_t mpos = M.out_off + (size_t)lc + (size_t)lr * M.ld;
          if constexpr (CPLX) {
            atomicAdd(&a.out[2 * mpos], vre2);
            atomicAdd(&a.out[2 * mpos + 1], vim2);
          } else {
            atomicAdd(&a.out[mpos], vre2);
          }
        }
      });
}

template <int KER, int BR, int BC, int CLS, int Q2, bool MP, bool MIR,
          bool PL>
__global__ __launch_bounds__(NTHREADS) void nf_singular_kernel(
    KArgs a, const SPair *__restrict__ list, uint32_t npairs) {
  singular_list<KER, BR, BC, CLS, Q2, MP, MIR, PL>(a, list, npairs,
                                                   blockIdx.x);
}

// The three classes (order 4) in one launch: identical pairs in the first
// b3 workgroups, edge pairs in the next b2, vertex pairs in the rest.  For
// lists that fit on the chip at once, where the launches one after the other
// cost each class its own latency (a 49 x 61 block, linear basis: 24 -> 9.5
// us, its launches 33 -> 20; 2048 triangles, constant basis: 25 -> 16 us;
// 2028 triangles, linear, 30000 pairs: 40 -> 35 us); the registers are
// those of the largest class, so long lists keep a launch per class.
template <int KER, int BR, int BC, bool MP, bool MIR, bool PL>
__global__ __launch_bounds__(NTHREADS) void nf_singular_all(
    KArgs a, const SPair *__restrict__ l3, uint32_t n3,
    const SPair *__restrict__ l2, uint32_t n2, const SPair *__restrict__ l1,
    uint32_t n1, uint32_t b3, uint32_t b2) {
  const uint32_t b = blockIdx.x;
  if (b < b3)
    singular_list<KER, BR, BC, CLS_IDENTICAL, 4, MP, MIR && BR != 0, PL>(
        a, l3, n3, b);
  else if (b < b3 + b2)
    singular_list<KER, BR, BC, CLS_EDGE, 4, MP, false, PL>(a, l2, n2, b - b3);
  else
    singular_list<KER, BR, BC, CLS_VERTEX, 4, MP, MIR, PL>(a, l1, n1,
                                                           b - b3 - b2);
}

// The pairs with common vertices of one tile and one rule class, by the
// tile's workgroup: 16 pairs per pass, the entries added into the tile's
// LDS accumulator (constant basis: stored, each entry belongs to one pair).
template <int KER, int BR, int BC, int CLS, int Q2, bool MP>
__device__ __forceinline__ void tile_singular(const KArgs &a, const Tile &T,
                                              const SPair *list, uint32_t n,
                                              double *acc_re,
                                              double *acc_im) {
  constexpr bool CPLX = KER >= K_HELM_SLP;
  constexpr bool CC = (BR == 0) && (BC == 0);
  const uint32_t row = threadIdx.x >> 4;
  const int sub = threadIdx.x & 15;
  const bool conj = T.ntrans && (BR == BC);
  for (uint32_t p0 = 0; p0 < n; p0 += NTHREADS / 16) {
    const uint32_t w = p0 + row;
    if (w >= n) continue;  // uniform per row of 16 lanes
    singular_pair<KER, BR, BC, CLS, Q2, MP, false, true>(
        a, T, list[w], sub,
        [&](uint32_t lr, uint32_t lc, double vre, double vim, double,
            double) {
          if constexpr (CC) {
            const size_t pos =
                T.out_off + (T.ntrans ? (size_t)lc + (size_t)lr * T.ld
                                      : (size_t)lr + (size_t)lc * T.ld);
            if constexpr (CPLX) {
              a.out[2 * pos] = vre;
              a.out[2 * pos + 1] = conj ? -vim : vim;
            } else {
              a.out[pos] = vre;
            }
          } else {
            const uint32_t e = lr + TILE * lc;
            atomicAdd(&acc_re[e], vre);
            if constexpr (CPLX) atomicAdd(&acc_im[e], vim);
          }
        });
  }
}

// The launches of one precision (MP: 0 FP64, 1 mixed, 2 mixed with
// compensated FP32 outer sums; the singular kernels are the same for 1 and
// 2).
template <int KER, int BR, int BC, int MP>
int launch_bases_p(uint32_t q, const KArgs &a, uint32_t ntiles,
                   const SPair *sp, const uint32_t *ncls, hipStream_t stream) {
  if (a.tlist && !a.far && q == 2 && a.q2 == 4) {
    // fused tiles: one launch for the regular and the singular pairs
    if (!ntiles) return H2HIP_OK;
    if (a.counter) {
      auto fk = nf_fused_persistent<KER, BR, BC, 2, MP>;
      int per_cu = 0, dev = 0, ncu = 0;
      if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fk, NTHREADS,
                                                       0) != hipSuccess ||
          hipGetDevice(&dev) != hipSuccess ||
          hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount,
                                dev) != hipSuccess)
        return H2HIP_EDEVICE;
      const uint32_t resident = (uint32_t)std::max(1, per_cu) * (uint32_t)ncu;
      const uint32_t grid = std::min(ntiles, std::max(1u, resident));
      hipLaunchKernelGGL(zero_counter, dim3(1), dim3(1), 0, stream, a.counter);
      hipLaunchKernelGGL(fk, dim3(grid), dim3(NTHREADS), 0, stream, a,
                         a.tlist, ntiles, a.counter);
    } else {
      hipLaunchKernelGGL((nf_fused_kernel<KER, BR, BC, 2, MP>), dim3(ntiles),
                         dim3(NTHREADS), 0, stream, a, a.tlist);
    }
    return H2HIP_OK;
  }
  constexpr bool SMP = MP != 0;
  constexpr uint32_t PPB = NTHREADS / 16;  // pairs per workgroup
  auto singular = [&](void (*k)(KArgs, const SPair *, uint32_t),
                      const SPair *list, uint32_t n) {
    if (n)
      hipLaunchKernelGGL(k, dim3((n + PPB - 1) / PPB), dim3(NTHREADS), 0,
                         stream, a, list, n);
  };
  const uint32_t n3 = ncls[CLS_IDENTICAL], n2 = ncls[CLS_EDGE],
                 n1 = ncls[CLS_VERTEX];
  // order 4, all classes: one launch while every pair has its lanes at once
  // (SING_ALL), else one per class
  auto singular4 = [&](auto mir, auto plane, uint32_t c3, uint32_t c1) {
    constexpr bool MIR = decltype(mir)::value;
    constexpr bool PL = decltype(plane)::value;
    if (c3 + n2 + c1 <= SING_ALL) {
      auto nb = [](uint32_t n) { return (n + PPB - 1) / PPB; };
      if (c3 + n2 + c1)
        hipLaunchKernelGGL((nf_singular_all<KER, BR, BC, SMP, MIR, PL>),
                           dim3(nb(c3) + nb(n2) + nb(c1)), dim3(NTHREADS), 0,
                           stream, a, sp, c3, sp + n3, n2, sp + n3 + n2, c1,
                           nb(c3), nb(n2));
      return;
    }
    singular(nf_singular_kernel<KER, BR, BC, CLS_IDENTICAL, 4, SMP,
                                MIR && BR != 0, PL>,
             sp, c3);
    singular(nf_singular_kernel<KER, BR, BC, CLS_EDGE, 4, SMP, false, PL>,
             sp + n3, n2);
    singular(nf_singular_kernel<KER, BR, BC, CLS_VERTEX, 4, SMP, MIR, PL>,
             sp + n3 + n2, c1);
  };
  if ((BR || BC) && a.split > 1) {
    const uint64_t n = a.entries * (KER >= K_HELM_SLP ? 2 : 1);
    const uint64_t blocks = (n + NTHREADS - 1) / NTHREADS;
    hipLaunchKernelGGL(zero_out, dim3((uint32_t)std::min<uint64_t>(blocks,
                                                                   2048)),
                       dim3(NTHREADS), 0, stream, a.out, n);
  }
  if constexpr (BR == BC) {
    // mirrored tiles: half the regular, vertex and (linear basis) identical
    // pairs; the lists hold the pairs to evaluate first
    if (a.nmir && !a.far && q == 2 && a.q2 == 4) {
      if constexpr (paired(KER, BR, BC, MP))
        hipLaunchKernelGGL((nf_pair_kernel<KER, BR, 2, MP>),
                           dim3(a.nmir * a.split),
                           dim3(pair_threads(KER, BR)), 0, stream, a,
                           a.mirlist);
      else
        hipLaunchKernelGGL((nf_regular_kernel<KER, BR, BC, 2, MP, 1>),
                           dim3(ntiles * a.split), dim3(NTHREADS), 0, stream,
                           a);
      singular4(std::true_type{}, std::true_type{}, BR ? a.nmain3 : n3,
                a.nmain1);
      return H2HIP_OK;
    }
  }
  // Laplace adjoint double layer at other orders than 2: a product <d, n> per
  // value, in a kernel without the points' factors, whose registers it would
  // pay for (order 3, 12800 triangles, linear basis 3190 -> 2983 us, constant
  // rows and linear columns 1684 -> 1502).  The double layer takes the
  // factors in the kernel with both (2884 us; 3022 by products, 3625 with the
  // factors alone, whose loads the compiler then holds in registers).
  constexpr bool LDLP = KER == K_LAP_DLP && MP == 0;
  KArgs ar = a;
  if (LDLP && q != 2 && a.adj) ar.plane = 0;
  if (ntiles && a.counter) {
    void (*reg)(KArgs, uint32_t, uint32_t *) = nullptr;
    switch (q) {
      case 1: reg = nf_regular_persistent<KER, BR, BC, 1, MP>; break;
      case 2: reg = nf_regular_persistent<KER, BR, BC, 2, MP>; break;
      case 3: reg = nf_regular_persistent<KER, BR, BC, 3, MP>; break;
      case 4: reg = nf_regular_persistent<KER, BR, BC, 4, MP>; break;
      default: return H2HIP_EINVAL;
    }
    int per_cu = 0, dev = 0, ncu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reg, NTHREADS,
                                                     0) != hipSuccess ||
        hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount,
                              dev) != hipSuccess)
      return H2HIP_EDEVICE;
    const uint32_t resident = (uint32_t)std::max(1, per_cu) * (uint32_t)ncu;
    const uint32_t grid = std::min(ntiles, std::max(1u, resident));
    hipLaunchKernelGGL(zero_counter, dim3(1), dim3(1), 0, stream, a.counter);
    hipLaunchKernelGGL(reg, dim3(grid), dim3(NTHREADS), 0, stream, ar, ntiles,
                       a.counter);
  } else if (ntiles) {
    void (*reg)(KArgs) = nullptr;
    switch (q) {
      case 1: reg = nf_regular_kernel<KER, BR, BC, 1, MP, -1>; break;
      case 2: reg = nf_regular_kernel<KER, BR, BC, 2, MP, 1>; break;
      case 3: reg = nf_regular_kernel<KER, BR, BC, 3, MP, -1>; break;
      case 4: reg = nf_regular_kernel<KER, BR, BC, 4, MP, -1>; break;
      default: return H2HIP_EINVAL;
    }
    if constexpr (MP == 0 && is_dlp(KER))
      if (q == 2 && !a.plane) reg = nf_regular_kernel<KER, BR, BC, 2, MP, 0>;
    if constexpr (LDLP)
      if (!ar.plane) switch (q) {
          case 1: reg = nf_regular_kernel<KER, BR, BC, 1, MP, 0>; break;
          case 3: reg = nf_regular_kernel<KER, BR, BC, 3, MP, 0>; break;
          case 4: reg = nf_regular_kernel<KER, BR, BC, 4, MP, 0>; break;
        }
    hipLaunchKernelGGL(reg, dim3(ntiles * a.split), dim3(NTHREADS), 0, stream,
                       a);
  }
  if (a.far) return H2HIP_OK;
  if (a.q2 == 4) {
    if constexpr (MP == 0 && is_dlp(KER)) {
      if (!a.plane) {
        singular4(std::false_type{}, std::false_type{}, n3, n1);
        return H2HIP_OK;
      }
    }
    singular4(std::false_type{}, std::true_type{}, n3, n1);
    return H2HIP_OK;
  }
  singular(nf_singular_kernel<KER, BR, BC, CLS_IDENTICAL, 0, SMP, false, true>, sp,
           n3);
  singular(nf_singular_kernel<KER, BR, BC, CLS_EDGE, 0, SMP, false, true>, sp + n3,
           n2);
  singular(nf_singular_kernel<KER, BR, BC, CLS_VERTEX, 0, SMP, false, true>,
           sp + n3 + n2, n1);
  return H2HIP_OK;
}

// Launches the regular tile kernel over `ntiles` tiles and then (unless
// far) one singular launch per rule class; sp holds the pairs sorted
// identical, edge, vertex with ncls[c] pairs of class c.  a.mp selects the
// mixed-precision kernels.
template <int KER, int BR, int BC>
int launch_bases(uint32_t q, const KArgs &a, uint32_t ntiles,
                 const SPair *sp, const uint32_t *ncls, hipStream_t stream) {
  if constexpr (!small_phase(KER)) {
    // (the FP32 kernels reduce every phase: their sine and cosine take
    // revolutions)
    if (a.mp == 2)
      return launch_bases_p<KER, BR, BC, 2>(q, a, ntiles, sp, ncls, stream);
    if (a.mp == 1)
      return launch_bases_p<KER, BR, BC, 1>(q, a, ntiles, sp, ncls, stream);
  }
  return launch_bases_p<KER, BR, BC, 0>(q, a, ntiles, sp, ncls, stream);
}

template <int KER>
int launch_family(int rb, int cb, uint32_t q, const KArgs &a,
                  uint32_t ntiles, const SPair *sp, const uint32_t *ncls,
                  hipStream_t stream) {
  if (!rb && !cb) return launch_bases<KER, 0, 0>(q, a, ntiles, sp, ncls, stream);
  if (rb && cb) return launch_bases<KER, 1, 1>(q, a, ntiles, sp, ncls, stream);
  if (cb) return launch_bases<KER, 0, 1>(q, a, ntiles, sp, ncls, stream);
  return launch_bases<KER, 1, 0>(q, a, ntiles, sp, ncls, stream);
}

}  // namespace nf
}  // namespace h2hip
