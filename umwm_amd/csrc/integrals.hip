// Spectral integrals taken once per dtg: stokes_drift (src/umwm_stokes.F90:
// 13-132), diag (src/umwm_physics.F90:89-205) and the significant wave height
// s_ice reads (src/umwm_source_functions.F90:108-153).
//
// One workgroup of kWaves waves owns LP sea points.  Waves take frequencies in
// rounds, one each, and the 64 / LP lane groups of a wave share its
// directions, so every spectrum access is a coalesced run of LP points and the
// spectrum is read once for both operators.  All sums are FP64; each wave adds
// up its own frequencies and the waves are added in order.
//
// Stokes drift needs util(o, l) at every frequency, level and point: an
// exponential each, the bulk of the work.  In a round the waves leave their
// directional sums and the frequency's factors in LDS, then each takes its
// share of the levels through the round's frequencies, keeping its levels'
// sums in registers.  With u = e^{-2kd} and E = e^{2kz} the finite-depth
// profile is
//   cosh 2k(z + d) / sinh^2 kd = 2 (E + u^2 / E) / (1 - u)^2,
// whose second term and denominator vanish to rounding where the reference
// switches to the deep-water form 2 E (src/umwm_stokes.F90:73-88), except
// near the bed at kd > 50, where it is dropped as there.  One exponential
// (the table-driven one of fmath64.hpp) replaces an exponential, a hyperbolic
// cosine and a hyperbolic sine.
//
// One thread per point, serial over its bins, had taken 572 us (Stokes) and
// 274 us (diag) at 155 points x 37x36 bins in FP64 (now 34 and 27 with the
// host's wait), 2.45 and 0.81 ms at 161,762 points (now 0.70 and 0.46), 7.9
// and 2.3 ms at 359,427 points x 49x72 in FP32 (now 2.1 and 1.5).  16 points a
// workgroup put four times the waves to work below kSmallTasks point blocks
// (72,057 points FP64: 64 points a workgroup 358 and 231 us, 16 points 423
// and 316).  Both operators in one pass save a launch and a read of the
// spectrum but halve the waves a SIMD holds: 43 against 60 us at 171 points,
// 7.0 against 3.6 ms at 359,427, so only below kFusedTasks point blocks.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "bufio.hpp"
#include "domain.hpp"
#include "fmath64.hpp"
#include "physics.hpp"

namespace umwm {
namespace {

constexpr int kWaves = 8;
constexpr int kSmallTasks = 512, kFusedTasks = 128;
constexpr int kRec = 6;   // per-frequency Stokes record in LDS
constexpr int kSums = 11;  // diag partial sums of a wave, and the dominant bin

__device__ const double kExpTab[fm64::kExpTabLen] = {UMWM_FM64_EXP_TABLE};

// 1 / x for positive normal x: the hardware estimate and two Newton steps.
__device__ __forceinline__ double rcp_pos(double x) {
  double r = __builtin_amdgcn_rcp(x);
  r = fma(r, fma(-x, r, 1.0), r);
  return fma(r, fma(-x, r, 1.0), r);
}

// A sum over the directions is four sums of every fourth direction, (0 + 1) +
// (2 + 3): over lane groups where a wave has four, else in one lane, so that
// the result does not depend on LP.
template <int LP>
__device__ __forceinline__ double dir_sum(const double* a) {
  if constexpr (LP == 64) return (a[0] + a[1]) + (a[2] + a[3]);
  static_assert(LP == 64 || LP == 16, "one or four lane groups");
  double v = a[0];
  v += __shfl_xor(v, 16, 64);
  v += __shfl_xor(v, 32, 64);
  return v;
}

template <typename T, int LP, int NL, bool STOKES, bool DIAG, bool ICE>
__global__ __launch_bounds__(64 * kWaves) void k_integrals(const DomainDev<T>* __restrict__ doms,
                                                           const BlockTask* __restrict__ tasks,
                                                           const EndDev* __restrict__ ends) {
  extern __shared__ double lds[];
  __shared__ double etab[STOKES ? fm64::kExpTabLen : 1];
  constexpr int SUBS = 64 / LP;
  const BlockTask tk = tasks[blockIdx.x];
  const DomainDev<T>& d = doms[tk.dom];
  const EndDev& out = ends[tk.dom];
  const int lane = (int)threadIdx.x & 63, w = wave_id();
  const int pl = lane & (LP - 1), sub = lane / LP;
  const int j = tk.i0 + (int)blockIdx.y * LP + pl;
  const bool valid = j < d.im;
  const int om = d.om, pm = d.pm, lm = d.lm;
  const size_t ldi = d.ldi;
  const int jc = valid ? j : d.im - 1;  // lanes past the end repeat the last point
  const uint32_t vj = (uint32_t)jc * (uint32_t)sizeof(T);
  const uint32_t rb = (uint32_t)ldi * (uint32_t)sizeof(T);
  if constexpr (STOKES) {
    for (int k = (int)threadIdx.x; k < fm64::kExpTabLen; k += 64 * kWaves) etab[k] = kExpTab[k];
  }
  const double dj = d.depth[jc];
  const int oc = d.oc[jc];
  // diag partial sums of this wave's frequencies
  double m0 = 0, m2 = 0, mk = 0, xc = 0, yc = 0, mx = 0, my = 0, gxx = 0, gxy = 0, gyy = 0;
  double best = -INFINITY;
  int opk = 0, ppk = 0;
  // Stokes sums of this lane group's levels g, g + kWaves SUBS, ...
  const int g = w * SUBS + sub;
  double us[NL], vs[NL], dep[NL], zmin = 0;
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    us[i] = vs[i] = 0;
    const int l = g + i * kWaves * SUBS;
    // a level below the sea bed drifts not at all: zeroed at the end
    const double z = STOKES && l < lm ? out.stokes.depth[l] : 0;
    dep[i] = fabs(z) > dj ? 0 : z;
    zmin = fmin(zmin, dep[i]);
  }
  for (int ob = 0, round = 0; ob < om; ob += kWaves, ++round) {
    const int o = ob + w;
    double* rec = lds + (size_t)(round & 1) * kWaves * kRec * LP;
    if (o < om) {  // wave-uniform
      const size_t t = (size_t)o * ldi + jc;
      const double kdk = d.kdk[t];
      const rsrc_t pe = row_rsrc(d.e, (size_t)o, (size_t)pm * ldi);
      constexpr int NP = 4 / SUBS;
      double a0[NP], ax[NP], ay[NP], axx[NP], axy[NP], ayy[NP], top = -INFINITY;
      int tp = 0;
#pragma unroll
      for (int i = 0; i < NP; ++i) a0[i] = ax[i] = ay[i] = axx[i] = axy[i] = ayy[i] = 0;
#pragma unroll 2
      for (int pb = sub; pb < pm; pb += 4) {
#pragma unroll
        for (int i = 0; i < NP; ++i) {
          const int p = pb + i;
          const double e = (double)bld<T>(pe, vj + (uint32_t)p * rb);
          const double c = d.cth[p], s = d.sth[p];
          a0[i] += e;
          if constexpr (STOKES || DIAG) {
            ax[i] = fma(e, c, ax[i]);
            ay[i] = fma(e, s, ay[i]);
          }
          if constexpr (DIAG) {
            const double ec = e * c, es = e * s;
            axx[i] = fma(ec, c, axx[i]);
            axy[i] = fma(ec, s, axy[i]);
            ayy[i] = fma(es, s, ayy[i]);
            const double ek = e * kdk;
            if (ek > top) {
              top = ek;
              tp = p;
            }
          }
        }
      }
      const double s0 = dir_sum<LP>(a0);
      [[maybe_unused]] double sx = 0, sy = 0;
      if constexpr (STOKES || DIAG) {
        sx = dir_sum<LP>(ax);
        sy = dir_sum<LP>(ay);
      }
      if constexpr (STOKES) {
        const double k = d.k[t], kd = k * dj;
        // 1 - u without cancellation in shallow water
        const double u = kd > 50 ? 0.0 : exp(-2 * kd), v = kd > 50 ? 1.0 : -expm1(-2 * kd);
        if (sub == 0) {
          double* r = rec + (size_t)w * kRec * LP + pl;
          r[0 * LP] = sx;
          r[1 * LP] = sy;
          r[2 * LP] = 2 * k;
          r[3 * LP] = kTwoPiD * (double)d.f[o] * 2 * (k * k) * (double)d.dwn[t] * d.dth / (v * v);
          r[4 * LP] = u * u;
          // the reflected term counts above e^-38 of the other
          r[5 * LP] = kd > 50 ? -INFINITY : 19.0 / (2 * k) - dj;
        }
      }
      if constexpr (ICE) m0 = fma(kdk, s0, m0);
      if constexpr (DIAG) {
        const double sxx = dir_sum<LP>(axx), sxy = dir_sum<LP>(axy), syy = dir_sum<LP>(ayy);
        const double f = d.f[o], icp = d.invcp0[t], cg = d.cg0[t];
        const double e0 = kdk * s0;
        m0 += e0;
        m2 = fma(f * f, e0, m2);
        mk = fma((double)d.k3dk[t], s0, mk);
        xc = fma(kdk, sx, xc);
        yc = fma(kdk, sy, yc);
        if (o <= oc) {
          const double ki = kdk * icp;
          mx = fma(ki, sx, mx);
          my = fma(ki, sy, my);
          gxx = fma(cg * ki, sxx, gxx);
          gxy = fma(cg * ki, sxy, gxy);
          gyy = fma(cg * ki, syy, gyy);
        }
        // dominant bin: the reference's maxloc over e kdk, o fastest
        // (src/umwm_physics.F90:157-160): of equal maxima the first in
        // (p, o) order
#pragma unroll
        for (int m = LP; m < 64; m <<= 1) {
          const double ot = __shfl_xor(top, m, 64);
          const int op = __shfl_xor(tp, m, 64);
          if (ot > top || (ot == top && op < tp)) {
            top = ot;
            tp = op;
          }
        }
        if (top > best || (top == best && (tp < ppk || (tp == ppk && o < opk)))) {
          best = top;
          opk = o;
          ppk = tp;
        }
      }
    }
    if constexpr (STOKES) {
      // double-buffered records: a wave writes the next round's while others
      // still read this one's, never the buffer of two rounds back
      __syncthreads();
      const int nf = min(kWaves, om - ob);
      for (int q = 0; q < nf; ++q) {
        const double* r = rec + (size_t)q * kRec * LP + pl;
        const double C = r[3 * LP], A = C * r[0 * LP], B = C * r[1 * LP], k2 = r[2 * LP];
        // the reflected term is rare below the first few frequencies: one
        // test per frequency leaves the levels' loop free of branches
        if (!__any(zmin < r[5 * LP])) {
#pragma unroll
          for (int i = 0; i < NL; ++i) {
            const double E = fm64::exp_t<false>(k2 * dep[i], etab);
            us[i] = fma(E, A, us[i]);
            vs[i] = fma(E, B, vs[i]);
          }
        } else {
          const double u2 = r[4 * LP];
#pragma unroll
          for (int i = 0; i < NL; ++i) {
            // negligible where it does not count; u2 = 0 where E may be 0
            double E = fm64::exp_t<false>(k2 * dep[i], etab);
            E = fma(u2, rcp_pos(fmax(E, 1e-300)), E);
            us[i] = fma(E, A, us[i]);
            vs[i] = fma(E, B, vs[i]);
          }
        }
      }
    }
  }
  if constexpr (STOKES) {
    __syncthreads();  // the records are read
    double* mag = lds;
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int l = g + i * kWaves * SUBS;
      if (l >= lm) continue;
      if (fabs(out.stokes.depth[l]) > dj) us[i] = vs[i] = 0;
      mag[(size_t)l * LP + pl] = sqrt(us[i] * us[i] + vs[i] * vs[i]);
      if (!valid) continue;
      out.stokes.us[(size_t)l * ldi + j] = us[i];
      out.stokes.vs[(size_t)l * ldi + j] = vs[i];
      if (l == 0) {
        d.us1[j] = us[i];
        d.vs1[j] = vs[i];
      }
    }
    __syncthreads();
    if (w == 0 && sub == 0 && valid) {
      // e-folding depth (src/umwm_stokes.F90:107-129)
      double ds = 0;
      const double m1 = mag[pl];
      if (m1 != 0) {
        const double ef = m1 * (1 / exp(1.0));
        for (int l = 1; l < lm; ++l) {
          const double ma = mag[(size_t)(l - 1) * LP + pl], mb = mag[(size_t)l * LP + pl];
          if (mb < ef) {
            ds = (fabs(ma - ef) * out.stokes.depth[l] + fabs(mb - ef) * out.stokes.depth[l - 1]) /
                 (ma - mb);
            break;
          }
        }
      }
      out.stokes.ds[j] = -ds;
    }
  }
  if constexpr (DIAG || ICE) {
    if constexpr (STOKES) __syncthreads();
    constexpr int N = DIAG ? kSums + 1 : 1;
    double* r = lds + (size_t)w * N * LP + pl;
    if (sub == 0) {
      r[0] = m0;
      if constexpr (DIAG) {
        const double v[kSums] = {m0, m2, mk, xc, yc, mx, my, gxx, gxy, gyy, best};
#pragma unroll
        for (int i = 1; i < kSums; ++i) r[(size_t)i * LP] = v[i];
        r[(size_t)kSums * LP] = __hiloint2double(opk, ppk);
      }
    }
    __syncthreads();
    if (w != 0 || sub != 0 || !valid) return;
    double v[N];
    for (int i = 0; i < N; ++i) v[i] = lds[(size_t)i * LP + pl];
    for (int q = 1; q < kWaves; ++q) {
      const double* a = lds + (size_t)q * N * LP + pl;
      if constexpr (DIAG) {
        for (int i = 0; i < kSums - 1; ++i) v[i] += a[(size_t)i * LP];
        const double bo = a[(size_t)(kSums - 1) * LP], id = a[(size_t)kSums * LP];
        const int o2 = __double2hiint(id), p2 = __double2loint(id);
        const int o1 = __double2hiint(v[N - 1]), p1 = __double2loint(v[N - 1]);
        if (bo > v[kSums - 1] || (bo == v[kSums - 1] && (p2 < p1 || (p2 == p1 && o2 < o1)))) {
          v[kSums - 1] = bo;
          v[N - 1] = id;
        }
      } else {
        v[0] += a[0];
      }
    }
    if constexpr (ICE) d.hs_ice[j] = 4 * sqrt(v[0] * d.dth);
    if constexpr (DIAG) {
      const DiagDev& G = out.diag;
      const double tiny = 2.2250738585072014e-308, rw = d.rhow[j];
      G.mwp[j] = sqrt(v[0] / (v[1] + tiny));
      G.momx[j] = v[5] * rw * d.dthg;
      G.momy[j] = v[6] * rw * d.dthg;
      G.cgmxx[j] = v[7] * rw * d.dthg;
      G.cgmxy[j] = v[8] * rw * d.dthg;
      G.cgmyy[j] = v[9] * rw * d.dthg;
      G.ht[j] = 4 * sqrt(v[0] * d.dth);
      G.mwd[j] = atan2(v[4], v[3]);
      G.mss[j] = v[2] * d.dth;
      G.mwl[j] = kTwoPiD * sqrt(v[0] / (v[2] + tiny));
      const int o = __double2hiint(v[N - 1]), p = __double2loint(v[N - 1]);
      const size_t t = (size_t)o * ldi + j;
      G.dwd[j] = d.th[p];
      G.dwl[j] = kTwoPiD / (double)d.k[t];
      G.dwp[j] = 1. / (double)d.f[o];
      G.dcp0[j] = d.cp0[t];
      G.dcg0[j] = d.cg0[t];
      const double cur = (double)d.uc[j] * d.cth[p] + (double)d.vc[j] * d.sth[p];
      G.dcp[j] = G.dcp0[j] + cur;
      G.dcg[j] = G.dcg0[j] + cur;
    }
  }
}

template <typename T, int LP, bool STOKES, bool DIAG, bool ICE>
void launch_lp(const DomainDev<T>* doms, const BlockTask* tasks, int ntasks, const EndDev* ends,
               int lm, hipStream_t s) {
  const dim3 grid(ntasks, 64 / LP), block(64 * kWaves);
  size_t n = 0;
  if (STOKES) n = std::max<size_t>((size_t)2 * kWaves * kRec * LP, (size_t)lm * LP);
  if (DIAG || ICE) n = std::max<size_t>(n, (size_t)kWaves * (DIAG ? kSums + 1 : 1) * LP);
  const size_t sh = n * sizeof(double);
  constexpr int groups = kWaves * (64 / LP);
  // levels per lane group: 48 and 104 levels cover the 100 of the namelist
  constexpr int few = (48 + groups - 1) / groups, most = (104 + groups - 1) / groups;
  if (STOKES && lm > few * groups)
    hipLaunchKernelGGL((k_integrals<T, LP, most, STOKES, DIAG, ICE>), grid, block, sh, s, doms,
                       tasks, ends);
  else
    hipLaunchKernelGGL((k_integrals<T, LP, STOKES ? few : 1, STOKES, DIAG, ICE>), grid, block, sh,
                       s, doms, tasks, ends);
}

int launched() {
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0
                         : fail(UMWM_ERR_HIP, std::string("k_integrals: ") + hipGetErrorString(e));
}

template <typename T, bool STOKES, bool DIAG, bool ICE>
int launch_any(const DomainDev<T>* doms, const BlockTask* tasks, int ntasks, const EndDev* ends,
               int lm, hipStream_t s) {
  if (ntasks < kSmallTasks)
    launch_lp<T, 16, STOKES, DIAG, ICE>(doms, tasks, ntasks, ends, lm, s);
  else
    launch_lp<T, 64, STOKES, DIAG, ICE>(doms, tasks, ntasks, ends, lm, s);
  return launched();
}

}  // namespace

template <typename T>
int launch_integrals(const DomainDev<T>* doms, const BlockTask* tasks, int ntasks,
                     const EndDev* ends, int lm, bool stokes, bool diag, hipStream_t s) {
  if (ntasks <= 0) return 0;
  stokes = stokes && lm > 0;
  if (stokes && diag && ntasks < kFusedTasks) {
    launch_lp<T, 16, true, true, false>(doms, tasks, ntasks, ends, lm, s);
    return launched();
  }
  if (stokes)
    if (int rc = launch_any<T, true, false, false>(doms, tasks, ntasks, ends, lm, s)) return rc;
  if (diag) return launch_any<T, false, true, false>(doms, tasks, ntasks, ends, lm, s);
  return 0;
}

template <typename T>
int launch_hs_ice(DomainImpl<T>& D) {
  return launch_any<T, false, false, true>(D.d, D.tasks, D.ntasks, D.end_d, 0, D.stream);
}

#define INST(T)                                                                              \
  template int launch_integrals<T>(const DomainDev<T>*, const BlockTask*, int, const EndDev*, \
                                   int, bool, bool, hipStream_t);                            \
  template int launch_hs_ice<T>(DomainImpl<T>&);
INST(float)
INST(double)

}  // namespace umwm
