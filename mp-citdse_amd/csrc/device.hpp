// Device functions shared by the kernel files: the Fehlberg tableau, the
// laser field, cross-lane sums, the stage derivative and the step control.
#pragma once

#include "kernels.hpp"

namespace mpci {

// Fehlberg 7(8) tableau (NASA TR R-287, 1968), the coefficients of
// boost::odeint runge_kutta_fehlberg78.
static __constant__ double cA[kStages][kStages] = {
    {0},
    {2.0 / 27.0},
    {1.0 / 36.0, 1.0 / 12.0},
    {1.0 / 24.0, 0.0, 1.0 / 8.0},
    {5.0 / 12.0, 0.0, -25.0 / 16.0, 25.0 / 16.0},
    {1.0 / 20.0, 0.0, 0.0, 1.0 / 4.0, 1.0 / 5.0},
    {-25.0 / 108.0, 0.0, 0.0, 125.0 / 108.0, -65.0 / 27.0, 125.0 / 54.0},
    {31.0 / 300.0, 0.0, 0.0, 0.0, 61.0 / 225.0, -2.0 / 9.0, 13.0 / 900.0},
    {2.0, 0.0, 0.0, -53.0 / 6.0, 704.0 / 45.0, -107.0 / 9.0, 67.0 / 90.0, 3.0},
    {-91.0 / 108.0, 0.0, 0.0, 23.0 / 108.0, -976.0 / 135.0, 311.0 / 54.0,
     -19.0 / 60.0, 17.0 / 6.0, -1.0 / 12.0},
    {2383.0 / 4100.0, 0.0, 0.0, -341.0 / 164.0, 4496.0 / 1025.0,
     -301.0 / 82.0, 2133.0 / 4100.0, 45.0 / 82.0, 45.0 / 164.0, 18.0 / 41.0},
    {3.0 / 205.0, 0.0, 0.0, 0.0, 0.0, -6.0 / 41.0, -3.0 / 205.0, -3.0 / 41.0,
     3.0 / 41.0, 6.0 / 41.0, 0.0},
    {-1777.0 / 4100.0, 0.0, 0.0, -341.0 / 164.0, 4496.0 / 1025.0,
     -289.0 / 82.0, 2193.0 / 4100.0, 51.0 / 82.0, 33.0 / 164.0, 12.0 / 41.0,
     0.0, 1.0},
};
static __constant__ double cB[kStages] = {0, 0, 0, 0, 0, 34.0 / 105.0, 9.0 / 35.0,
                                   9.0 / 35.0, 9.0 / 280.0, 9.0 / 280.0, 0,
                                   41.0 / 840.0, 41.0 / 840.0};
// b - bhat: the embedded error weights.
static __constant__ double cDB[kStages] = {-41.0 / 840.0, 0, 0, 0, 0, 0, 0, 0, 0, 0,
                                    -41.0 / 840.0, 41.0 / 840.0,
                                    41.0 / 840.0};
static __constant__ double cC[kStages] = {0, 2.0 / 27.0, 1.0 / 9.0, 1.0 / 6.0,
                                   5.0 / 12.0, 0.5, 5.0 / 6.0, 1.0 / 6.0,
                                   2.0 / 3.0, 1.0 / 3.0, 1.0, 0, 1.0};

// ---------------------------------------------------------------------
// Laser field, src/tdse/pulse.cpp:34-39 (gauss), 52-56 (sineAA), 93-97
// (sineEE), plus the piecewise-linear envelope extension.
// Always inlined: hipcc (ROCm 7.2) emitted this as a call from inside a
// divergent branch and copied the saved thread id under the branch's exec
// mask, so lanes outside the branch lost threadIdx.x across the call.
// ---------------------------------------------------------------------
__device__ __forceinline__ double field_at(const PulseDev &p,
                                           const double *env, double t) {
  if (p.kind == kSine2) {
    double sinWt = sin(p.a * t);
    return (double)(t >= 0.0 && t <= M_PI / p.a) * p.Eo * sinWt * sinWt *
           sin(p.w * t + p.cepd);
  }
  if (p.kind == kGauss) {
    double t_diff = t - 0.5 * p.b;
    return (double)(t >= 0.0 && t <= p.b) * p.Eo *
           exp(-t_diff * t_diff / (p.a * p.a)) * sin(p.w * t + p.cepd);
  }
  if (!(t >= 0.0 && t <= p.t_end) || p.n_env < 2) return 0.0;
  const double *e = env + p.env_off;
  double dx = p.t_end / (p.n_env - 1);
  double u = t / dx;
  int k = (int)floor(u);
  if (k > p.n_env - 2) k = p.n_env - 2;
  if (k < 0) k = 0;
  double f = u - k;
  double en = (1.0 - f) * e[k] + f * e[k + 1];
  return p.scale * en * sin(p.w * t + p.cepd);
}

// ---------------------------------------------------------------------
// Cross-lane sums on the VALU (DPP and the gfx950 lane swaps), no LDS.
// ---------------------------------------------------------------------
template <int CTRL>
__device__ __forceinline__ double dpp_d(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xF,
                                             0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xF,
                                             0xF, false);
  return __hiloint2double(hi, lo);
}

// Sum over the 16 lanes of a row: quad_perm [1,0,3,2], quad_perm [2,3,0,1],
// row_half_mirror, row_mirror.  Each step adds two operands, which commute
// exactly, so every lane of the row ends with the same bits.
__device__ __forceinline__ double sum16(double v) {
  v += dpp_d<0xB1>(v);
  v += dpp_d<0x4E>(v);
  v += dpp_d<0x141>(v);
  v += dpp_d<0x140>(v);
  return v;
}

// v[l] + v[l ^ 16]: v_permlane16_swap of v with itself leaves the even rows
// in the first result and the odd rows in the second, so lane l holds both
// operands; l and l ^ 16 add them in the same order.
__device__ __forceinline__ double add_xor16(double v) {
  const unsigned lo = __double2loint(v), hi = __double2hiint(v);
  const auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
  const auto h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
  return __hiloint2double((int)h[0], (int)l[0]) +
         __hiloint2double((int)h[1], (int)l[1]);
}

// v[l] + v[l ^ 32], likewise with v_permlane32_swap (wave halves).
__device__ __forceinline__ double add_xor32(double v) {
  const unsigned lo = __double2loint(v), hi = __double2hiint(v);
  const auto l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
  const auto h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
  return __hiloint2double((int)h[0], (int)l[0]) +
         __hiloint2double((int)h[1], (int)l[1]);
}

// k_s of one (row, pulse) from the coupling sums cs = D^T x_{L-1} and
// rs = D x_{L+1}, the stage input xs, the energy e and the stage field F
// (MatVecV / MatVecL, src/tdse/tdse.cpp:14-143).  The fma is written out:
// left to the compiler, which of the two products it fuses may differ from
// one kernel to another, and with it the last bit.
__device__ __forceinline__ double2 stage_deriv(int gauge, double e, double2 xs,
                                               double F, double2 cs,
                                               double2 rs) {
  double2 k;
  if (gauge == 0) {  // velocity: -iE x + F (D^T x_{L-1} - D x_{L+1})
    k.x = fma(F, cs.x - rs.x, e * xs.y);
    k.y = fma(F, cs.y - rs.y, -e * xs.x);
  } else {           // length: -i (E x + F (D^T x_{L-1} + D x_{L+1}))
    k.x = fma(F, cs.y + rs.y, e * xs.y);
    k.y = fma(-F, cs.x + rs.x, -e * xs.x);
  }
  return k;
}

// |v|^2, likewise.
__device__ __forceinline__ double abs2(double x, double y) {
  return fma(x, x, y * y);
}

// ---------------------------------------------------------------------
// Row form (one pulse): a wave forms the coupling sums of four rows (a quad)
// from the row store (RowDesc), its lanes taking the columns of each
// 64-column chunk of [D_{L-1}^T | D_L] in turn.  The stage input enters the
// second part with the sign of the gauge's formula, so one sum per component
// holds D^T x_{L-1} - D x_{L+1} (velocity) or the plus form (length).
// ---------------------------------------------------------------------
__device__ __forceinline__ void quad_fma(double2 (&acc)[4], double2 d01,
                                         double2 d23, double2 x) {
  acc[0].x = fma(d01.x, x.x, acc[0].x);
  acc[0].y = fma(d01.x, x.y, acc[0].y);
  acc[1].x = fma(d01.y, x.x, acc[1].x);
  acc[1].y = fma(d01.y, x.y, acc[1].y);
  acc[2].x = fma(d23.x, x.x, acc[2].x);
  acc[2].y = fma(d23.x, x.y, acc[2].y);
  acc[3].x = fma(d23.y, x.x, acc[3].x);
  acc[3].y = fma(d23.y, x.y, acc[3].y);
}

// Lane-swap sum of two values: the lower wave half (HALF) or the even rows
// of 16 lanes keep the sum of a, the others that of b.
template <bool HALF>
__device__ __forceinline__ double pair_sum(double a, double b) {
  const unsigned al = __double2loint(a), ah = __double2hiint(a);
  const unsigned bl = __double2loint(b), bh = __double2hiint(b);
  if constexpr (HALF) {
    const auto l = __builtin_amdgcn_permlane32_swap(al, bl, false, false);
    const auto h = __builtin_amdgcn_permlane32_swap(ah, bh, false, false);
    return __hiloint2double((int)h[0], (int)l[0]) +
           __hiloint2double((int)h[1], (int)l[1]);
  } else {
    const auto l = __builtin_amdgcn_permlane16_swap(al, bl, false, false);
    const auto h = __builtin_amdgcn_permlane16_swap(ah, bh, false, false);
    return __hiloint2double((int)h[0], (int)l[0]) +
           __hiloint2double((int)h[1], (int)l[1]);
  }
}

// dpp_d for controls under which every lane reads a lane of its row.
template <int CTRL>
__device__ __forceinline__ double dpp_perm(double v) {
  const int lo =
      __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xF, 0xF, true);
  const int hi =
      __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xF, 0xF, true);
  return __hiloint2double(hi, lo);
}

// The eight sums of a wave over its 64 lanes in ten additions (a wave64
// instruction takes four cycles, so their number counts): every lane l
// returns both parts of row l >> 4.
__device__ __forceinline__ double2 quad_reduce(const double2 (&acc)[4],
                                               int lane) {
  // halves: rows 0, 1 | 2, 3; then rows of 16 lanes: 0 | 1 | 2 | 3
  const double re = pair_sum<false>(pair_sum<true>(acc[0].x, acc[2].x),
                                    pair_sum<true>(acc[1].x, acc[3].x));
  const double im = pair_sum<false>(pair_sum<true>(acc[0].y, acc[2].y),
                                    pair_sum<true>(acc[1].y, acc[3].y));
  // the lower eight lanes of a row go on with the real part
  const bool up = (lane & 8) != 0;
  double v = up ? im : re;
  v += dpp_perm<0x128>(up ? re : im);  // row_ror:8, the other half's share
  v += dpp_perm<0xB1>(v);
  v += dpp_perm<0x4E>(v);
  v += dpp_perm<0x141>(v);
  const double o = dpp_perm<0x128>(v);
  return up ? make_double2(o, v) : make_double2(v, o);
}

// (error max, |y|^2) of a quad's rows in order, from lanes 0, 16, 32, 48.
__device__ __forceinline__ double lane_value(double v, int lane) {
  return __hiloint2double(
      __builtin_amdgcn_readlane(__double2hiint(v), lane),
      __builtin_amdgcn_readlane(__double2loint(v), lane));
}
__device__ __forceinline__ double2 quad_norms(double errv, double nrm2) {
  double em = 0.0, ns = 0.0;
#pragma unroll
  for (int r = 0; r < kRwQuad; ++r) {
    const double e = lane_value(errv, 16 * r), m = lane_value(nrm2, 16 * r);
    em = e > em ? e : em;
    ns += m;
  }
  return make_double2(em, ns);
}

// The field at stage time s of pulse p's current attempt: the frozen
// per-step value of the fixed mode (src/tdse/tdse.cpp:187), the pulse at
// t + c_s h (adaptive and schedule modes) or a constant.
__device__ __forceinline__ double stage_field(const Ctl &c, int s, int p,
                                              const double *__restrict__ Ftab,
                                              const PulseDev *__restrict__ pulses,
                                              const double *__restrict__ env) {
  if (c.fmode == kFieldTable) return Ftab[(long long)p * c.hstride + c.step];
  if (c.fmode == kFieldPulse)
    return field_at(pulses[p], env, c.t + cC[s] * c.hc);
  return c.Fc;
}

// The step control of one attempt from its error ratio E and |y|^2:
// accept / reject, the next step size (adaptive), or the next step of a
// fixed or schedule run.
__device__ __forceinline__ Ctl control_step(Ctl c, double E, double n2, int p,
                                            const double *__restrict__ hs) {
  c.nrm = sqrt(n2);
  c.err = E;
  c.attempts++;
  if (c.mode == kModeAdaptive) {
    const double hh = c.hc;
    if (E > 1.0) {
      // reject: h *= max(0.9 E^(-1/(q-1)), 1/5), error order q = 7
      const double f = 0.9 / cbrt(sqrt(E));
      c.h = hh * (f > 0.2 ? f : 0.2);
      c.rejected++;
      c.accept = 0;
    } else {
      c.accept = 1;
      c.accepted++;
      c.hacc = hh;
      c.nlog++;
      if (c.last) {
        c.t = c.t_end;
        c.done = 1;
      } else {
        c.t += hh;
        if (E < 0.5) {
          // increase: h *= 0.9 max(E, 5^-8)^(-1/8), stepper order 8
          const double Em = E > 1.0 / 390625.0 ? E : 1.0 / 390625.0;
          c.h = hh * (0.9 / sqrt(sqrt(sqrt(Em))));
        } else {
          c.h = hh;
        }
      }
    }
    if (!c.done && c.attempts >= c.max_attempts) {
      c.done = 1;
      c.status = -1;
    }
    if (!c.done) {
      c.last = (c.t + c.h >= c.t_end);
      c.hc = c.last ? (c.t_end - c.t) : c.h;
    }
  } else {
    c.accept = 1;
    c.accepted++;
    c.hacc = c.hc;
    c.nlog++;
    c.t += c.hc;
    c.step++;
    if (c.step >= c.nsteps)
      c.done = 1;
    else if (c.mode == kModeSchedule)
      c.hc = hs[(long long)p * c.hstride + c.step];
  }
  return c;
}

}  // namespace mpci
