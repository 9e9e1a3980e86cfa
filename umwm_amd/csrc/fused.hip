// Fused substep kernels for gfx950.
//
// One substep of the reference (src/umwm_top.F90:95-115) is four kernels:
//   k_rates      sin + sds + rate + per-point max|rate| -> physics_time_step,
//                then a grid-wide min (atomic max on order-preserving keys,
//                finished by the last block) -> dts, dta, sumt, dtr
//                (src/umwm_physics.F90:22-58, src/umwm_advection.F90:329-365).
//                Reads E^n up to each point block's last prognostic bin,
//                and its directional moments, whose running sum over
//                frequency is the sds prefix.
//   k_integrate  sin + sds + snl + exponential integration + diagnostic
//                tail (src/umwm_physics.F90:60-84); writes only
//                E* = (E^n + E_s)/2 (es).
//   k_advect     upwind propagation on E* (src/umwm_advection.F90:18-99),
//                refraction (:102-180) and e = ef, one wave per
//                (frequency, 64 sea points), with E_s recovered in place as
//                2 E* - E^n from the e it overwrites (one spectrum stream
//                fewer than storing E_s; the round-off is |E^n + E_s| ulp);
//                also the directional moments of the new spectrum and the
//                per-frequency partial sums of stress_vector_integral
//                (src/umwm_stress.F90:313-331).
//   k_stress     per point: frequency sums, tail and the FP64 form/skin
//                drag chain of stress('atm') (src/umwm_stress.F90:216-264).
//
// k_rates and k_integrate sweep frequencies in order inside the kernel: a
// wave owns 64 consecutive sea points (one per lane, so every spectrum and
// table access is a coalesced 64-wide stream of the i-contiguous layout), D
// directions and a chunk of consecutive frequencies (all of them on large
// grids).  The prefix over frequency of sum_pp e(o,pp) cos^2(th_pp - th_p)
// (src/umwm_source_functions.F90:92-97) uses cos^2(a-b) = (1 + cos2a cos2b +
// sin2a sin2b)/2: three directional moments per frequency, which turns the
// O(pm^2) convolution into O(pm).  k_advect leaves the moments of the
// spectrum it writes, so the waves of a point need no exchange.  Each sweep
// prefetches the next frequency's spectrum (and, in FP32, its tables) while
// computing the current one.  Launches whose waves all hold exactly DMAX
// directions take a variant without per-slot masks, and k_rates one that
// pairs each direction with its opposite (given tiles, the surrogate and spectra
// wider than 72 directions).
//
// snl(o) = bf1r(o) X(o+1) + bf2r(o) X(o+2) - snl_fac X(o), X = sds e
// (src/umwm_source_functions.F90:165-171) is folded into the integration
// as each X becomes known: k_integrate keeps per direction only the
// partial E* = (E^n + partial E_s)/2 of the two previous frequencies.
//
// Wind input per bin (src/umwm_source_functions.F90:38-80) is evaluated
// as y = |x| x times one of three per-frequency factors (sheltering for
// y > 0, sin_diss1 against the wind, sin_diss1 fieldscale2 for swell
// overrunning it), with x = A cos th + B sin th - cp0 from the angle-sum
// identity (A, B per frequency) - the reference's expression regrouped,
// equal to it up to rounding.
//
// All per-point streams go through raw buffer loads and stores (bufio.hpp):
// one descriptor per frequency in scalar registers, 32-bit lane offsets
// computed once per thread, directions reached with a scalar offset.  The
// FP32 sweeps derive their (frequency, point) tables from k and the depth
// (TabGen); FP64 reads an 8-value record per lane (four 16-byte loads).
// The directional moments and the stress partials are planes.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "bufio.hpp"
#include "domain.hpp"
#include "fmath64.hpp"
#include "physics.hpp"
#include "surrogate.hpp"

namespace umwm {
namespace {

template <typename U>
__device__ __forceinline__ U pload(const U* a, size_t n, int j) {
  return bld<U>(make_rsrc(a, (uint32_t)(n * sizeof(U))), (uint32_t)j * (uint32_t)sizeof(U));
}
template <typename U>
__device__ __forceinline__ void pstore(U* a, size_t n, int j, U v) {
  bst(make_rsrc(a, (uint32_t)(n * sizeof(U))), (uint32_t)j * (uint32_t)sizeof(U), v);
}

// Per-point inputs of the source terms (src/umwm_source_functions.F90:21-52,
// :174-177).
template <typename T>
struct PointState {
  T wspd, a;   // floored wind speed, 2.5 ustar
  T pre;       // (1 - fice) 2 pi rhorat
  T shelt;     // sheltering coefficient
  T uc, vc;
  T cw, sw;    // cos, sin of wdir
  T csdt;      // sdt_fac sqrt(rhorat) ustar
  T ice;       // Kohout attenuation coefficient (0 below fice_lth)
  int oc;      // 0-based last prognostic bin
};

// Fresh evaluation (k_rates): wind floor, cut-off bin, sheltering; wave 0
// stores them for the later kernels of the substep.
template <typename T>
__device__ inline PointState<T> point_fresh(const DomainDev<T>& d, int j, bool write) {
  const size_t ldi = d.ldi, ldq = d.ldq;
  PointState<T> s;
  T w = pload(d.wspd, ldq, j);
  w = w > T(1e-2) ? w : T(1e-2);
  T fc = T(0.53) * T(d.g) / w;
  if (fc > T(d.fprog)) fc = T(d.fprog);
  int oc = 0;
  for (int o = d.om - 3; o >= 0; --o) {  // src/umwm_source_functions.F90:30-36
    oc = o;
    if (fc > cld(d.f, o)) break;
  }
  const T wdir = pload(d.wdir, ldq, j);
  const T rr = pload(d.rhorat, ldq, j);
  const T fice = pload(d.fice, ldq, j);
  const T ust = T(pload(d.ustar, ldi, j));
  s.wspd = w;
  s.a = T(2.5) * ust;
  s.pre = (T(1) - fice) * T(kTwoPiD) * rr;
  s.shelt = sheltering_coare35(w);
  s.uc = pload(d.uc, ldq, j);
  s.vc = pload(d.vc, ldq, j);
  s.cw = cos(wdir);
  s.sw = sin(wdir);
  s.csdt = T(d.sdt_fac) * sqrt(rr) * ust;
  s.ice = fice > T(d.fice_lth) ? T(sice_coef(pload(d.hs_ice, ldi, j))) : T(0);
  s.oc = oc;
  if (write) {
    pstore(d.wspd, ldq, j, w);
    pstore(d.fcutoff, ldi, j, fc);
    pstore(d.oc, ldi, j, (int32_t)oc);
    pstore(d.shelt, ldi, j, s.shelt);
    pstore(d.cwdir, ldi, j, s.cw);
    pstore(d.swdir, ldi, j, s.sw);
  }
  return s;
}

// Later kernels of the substep read back what k_rates stored.
template <typename T>
__device__ inline PointState<T> point_stored(const DomainDev<T>& d, int j) {
  const size_t ldi = d.ldi, ldq = d.ldq;
  PointState<T> s;
  const T rr = pload(d.rhorat, ldq, j);
  const T fice = pload(d.fice, ldq, j);
  const T ust = T(pload(d.ustar, ldi, j));
  s.wspd = pload(d.wspd, ldq, j);
  s.a = T(2.5) * ust;
  s.pre = (T(1) - fice) * T(kTwoPiD) * rr;
  s.shelt = pload(d.shelt, ldi, j);
  s.uc = pload(d.uc, ldq, j);
  s.vc = pload(d.vc, ldq, j);
  s.cw = pload(d.cwdir, ldi, j);
  s.sw = pload(d.swdir, ldi, j);
  s.csdt = T(d.sdt_fac) * sqrt(rr) * ust;
  s.ice = fice > T(d.fice_lth) ? T(sice_coef(pload(d.hs_ice, ldi, j))) : T(0);
  s.oc = pload(d.oc, ldi, j);
  return s;
}

// Per-frequency factors of the wind input: ssin = y * (y > 0 ? pos :
// (overrun ? neg2 : neg1)), y = |x| x, x = A cth + B sth - cp0.
template <typename T>
struct SinFreq {
  T A, B, cp0, pos, neg1, neg2;
};

template <typename T>
__device__ __forceinline__ SinFreq<T> sin_freq(const PointState<T>& s, T logl2, T cp0, T fkovg,
                                               T sin_diss1, T fs2) {
  SinFreq<T> r;
  const T ba = s.wspd + s.a * logl2;
  r.A = ba * s.cw - s.uc;
  r.B = ba * s.sw - s.vc;
  r.cp0 = cp0;
  const T g = s.pre * fkovg;
  r.pos = g * s.shelt;
  r.neg1 = g * sin_diss1;
  r.neg2 = r.neg1 * fs2;
  return r;
}

template <typename T>
__device__ __forceinline__ T sin_bin(const SinFreq<T>& q, const PointState<T>& s, T ct, T st,
                                     bool tail) {
  const T x = q.A * ct + q.B * st - q.cp0;
  const T y = fabs(x) * x;
  const T cwt = s.cw * ct + s.sw * st;  // cos(wdir - th)
  // select between values (a select between members would become an
  // address select and spill the struct to scratch)
  const T pos = q.pos, neg1 = q.neg1, neg2 = q.neg2;
  const T neg = cwt > T(0) ? neg2 : neg1;
  T r = y * (y > T(0) ? pos : neg);
  if (tail) r = r < T(0) ? T(0) : r;  // src/umwm_source_functions.F90:73-80
  return r;
}

// Rotation tendency of src/umwm_advection.F90:335-338 for one direction:
// 0.5 ((dcx sth + dvc) odx - (dcy cth + duc) ody).
template <typename T>
__device__ __forceinline__ T rot_dir(T dcx, T dcy, T sth, T cth, T dvc, T duc, T odx, T ody) {
  return T(0.5) * ((dcx * sth + dvc) * odx - (dcy * cth + duc) * ody);
}

// Per-frequency, per-point tables of the source terms: one record of
// DomainDev::ftab.
template <typename T>
struct FreqTab {
  T v[FT_N + 2];  // the record, FT_KDK and FT_CG0
  __device__ __forceinline__ T operator[](int i) const { return v[i]; }
};

// Quotient of wave-uniform integers in a scalar register: the division runs
// on the vector unit, and what is derived from its result (descriptors, loop
// bounds) would stay there.
__device__ __forceinline__ int uniform_div(int a, int b) {
  return __builtin_amdgcn_readfirstlane(a / b);
}

// Descriptor of frequency o's slice of a [om][rows][ldi] spectrum (rows =
// pm; a direction is then the scalar offset p * ldi * sizeof(T)) or of a
// [om][ldi][rec] record block (rec values per point).
template <typename T>
__device__ __forceinline__ rsrc_t freq_rsrc(const T* base, int o, int rows, size_t ldi) {
  return row_rsrc(base, (size_t)o, (size_t)rows * ldi);
}

// Frequency o's slice of the surrogate's bf16 rate rows, [om][pm][ldi].
__device__ __forceinline__ rsrc_t sur_rsrc(const uint16_t* base, int o, int pm, size_t ldi) {
  return row_rsrc(base, (size_t)o, (size_t)pm * ldi);
}

// First N slots of the record of (o, j); vr = j * FT_N * sizeof(T).
template <int N, typename T>
__device__ __forceinline__ void load_tab(const T* ftab, size_t ldi, int o, uint32_t vr,
                                         FreqTab<T>& r) {
  T tmp[N];
  bldn<T, N>(freq_rsrc(ftab, o, FT_N, ldi), vr, tmp);
#pragma unroll
  for (int i = 0; i < N; ++i) r.v[i] = tmp[i];
  r.v[FT_KDK] = r.v[FT_CG0] = T(0);
}

// FP32 sweeps derive the (frequency, point) tables from k and the depth
// (src/umwm_init.F90:1480-1533) rather than load them: the sweeps are
// bound by memory traffic, and one k per (frequency, point) replaces a
// 9-value record.  With u = e^{-2 kd}, kd = min(k d, 20):
//   sinh(2 kd) = (1/u - u)/2,  cosh(kd) = (1/sqrt(u) + sqrt(u))/2,
//   coth(0.2 kd) = (1 + w)/(1 - w) with w = e^{-0.4 kd},
//   cp0 = 2 pi f / k, cg0 = cp0 (1/2 + k d / sinh(2 kd) + s k^2/(rho g + s k^2)),
//   kdk = k dom / |cg0|, bf1r(o) = snl_fac bf1 kdk(o+1)/kdk(o) (o <= om-3),
//   log(l2/z) with l2 = cp0/(2 f) capped at 20 m.
// It keeps k of the next three frequencies and kdk of the next two, so
// bf1r and bf2r need no look-back.  FP64 keeps the record tables: its
// library exp would cost more than the traffic saved.
struct TabGen {
  const float* kb;
  const float *fr, *domr;
  size_t ldi;
  uint32_t vj;
  int om;
  float dep, sgr, sbf, sbp, s1, s2, l2z, lz;
  float k0, k1, k2, kn;   // k(o), k(o+1), k(o+2), k(o+3) (loaded ahead)
  float kdk0, kdk1, kdk2;

  __device__ float load_k(int o) const {
    return bld<float>(row_rsrc(kb, (size_t)min(o, om - 1), ldi), vj);
  }
  __device__ float kdk_of(float k, int o) const {
    o = min(o, om - 1);
    const float kd = fminf(k * dep, 20.f);
    const float u = __builtin_amdgcn_exp2f(-2.f * 1.4426950408889634f * kd);
    const float sinh2 = 0.5f * (__builtin_amdgcn_rcpf(u) - u);
    const float cp = 6.283185307179586f * cld(fr, o) * __builtin_amdgcn_rcpf(k);
    const float sk2 = sgr * k * k;
    const float cg = cp * (0.5f + k * dep * __builtin_amdgcn_rcpf(sinh2) +
                           sk2 * __builtin_amdgcn_rcpf(1.f + sk2));
    return k * cld(domr, o) * __builtin_amdgcn_rcpf(fabsf(cg));
  }
  template <typename D>
  __device__ void init(const D& d, int j, uint32_t vj_, int o0) {
    kb = d.k;
    fr = d.f;
    domr = d.dom;
    ldi = d.ldi;
    vj = vj_;
    om = d.om;
    // lanes past im read a depth of 0; they take 1 m so that their tables
    // stay finite (the reference requires only dmin > 0 of sea points)
    dep = j < d.im ? pload(d.depth, ldi, j) : 1.f;
    sgr = float(d.sfct / (d.rhow0 * d.g));
    sbf = float(d.sbf_fac);
    sbp = float(d.sbp_fac);
    s1 = float(d.snl_fac * d.bf1);
    s2 = float(d.snl_fac * d.bf2);
    lz = float(log(d.z));
    l2z = float(log(20.0 / d.z));
    k0 = load_k(o0);
    k1 = load_k(o0 + 1);
    k2 = load_k(o0 + 2);
    kn = load_k(o0 + 3);
    kdk0 = kdk_of(k0, o0);
    kdk1 = kdk_of(k1, o0 + 1);
    kdk2 = kdk_of(k2, o0 + 2);
  }
  // slots of frequency o (the FreqTab layout of the record tables)
  __device__ void table(int o, FreqTab<float>& r) const {
    const float k = k0, fo = cld(fr, o);
    const float kd = fminf(k * dep, 20.f);
    const float u = __builtin_amdgcn_exp2f(-2.f * 1.4426950408889634f * kd);
    const float iu = __builtin_amdgcn_rcpf(u);
    const float isinh2 = __builtin_amdgcn_rcpf(0.5f * (iu - u));
    const float v = __builtin_amdgcn_sqrtf(u);
    const float ch = 0.5f * (__builtin_amdgcn_rcpf(v) + v);
    const float w = __builtin_amdgcn_exp2f(-0.4f * 1.4426950408889634f * kd);
    const float cp = 6.283185307179586f * fo * __builtin_amdgcn_rcpf(k);
    const float sk2 = sgr * k * k;
    const float l2 = 0.5f * cp * __builtin_amdgcn_rcpf(fo);
    r.v[FT_CP0] = cp;
    r.v[FT_LOGL2] = l2 > 20.f ? l2z : 0.6931471805599453f * __builtin_amdgcn_logf(l2) - lz;
    const float coth = (1.f + w) * __builtin_amdgcn_rcpf(1.f - w);
    r.v[FT_COTH] = coth;
    r.v[FT_L] = 0.f;  // FP64 only
    r.v[FT_SBF] = sbf * k * isinh2 + sbp * k * __builtin_amdgcn_rcpf(ch * ch);
    r.v[FT_K] = k;
    r.v[FT_CG0] = cp * (0.5f + k * dep * isinh2 + sk2 * __builtin_amdgcn_rcpf(1.f + sk2));
    const bool bo = o <= om - 3;
    const float ik = __builtin_amdgcn_rcpf(kdk0);
    r.v[FT_B1] = bo ? s1 * kdk1 * ik : 0.f;
    r.v[FT_B2] = bo ? s2 * kdk2 * ik : 0.f;
    r.v[FT_KDK] = kdk0;
  }
  // moves to frequency o+1; `next` is k(o+4), loaded during iteration o
  __device__ void advance(int o, float next) {
    k0 = k1;
    k1 = k2;
    k2 = kn;
    kn = next;
    kdk0 = kdk1;
    kdk1 = kdk2;
    kdk2 = kdk_of(k2, o + 3);
  }
};

// Transcendentals of the sweeps.  FP32 works in base 2 on the hardware
// log2/exp2 (exponents pre-scaled by log2 e where a natural exponential is
// meant).  FP64 uses the table-driven natural log and exp of fmath64.hpp
// (within 1 ulp, about 0.65x the instructions of the device library's) and
// a reciprocal from the hardware estimate refined by two Newton steps (its
// arguments are positive and normal: the spreading factor >= 1 and
// cf coth).  The tables (4.2 KB) are staged into LDS by every block of the
// FP64 sweeps: read from global memory they were 3.5 KB of divergent
// vector loads per wave and bin, more than the spectrum stream itself.
constexpr int kFm64Len = fm64::kExpTabLen + fm64::kLogTabLen + fm64::kInvTabLen;
__device__ const double kFm64Tab[kFm64Len] = {UMWM_FM64_EXP_TABLE, UMWM_FM64_LOG_TABLE,
                                              UMWM_FM64_INV_TABLE};
__shared__ __attribute__((aligned(16))) double sFm64[kFm64Len];

// Fills the LDS tables; every thread of the block must call it.
template <typename T>
__device__ __forceinline__ void stage_fm64() {
  if constexpr (std::is_same_v<T, double>) {
    for (int k = threadIdx.x; k < kFm64Len; k += blockDim.x) sFm64[k] = kFm64Tab[k];
    __syncthreads();
  }
}

template <typename T>
struct Tr;
template <>
struct Tr<float> {
  static constexpr float kExpScale = 1.4426950408889634f;  // log2(e)
  __device__ static __forceinline__ float lg(float x) { return __builtin_amdgcn_logf(x); }
  __device__ static __forceinline__ float ex(float x) { return __builtin_amdgcn_exp2f(x); }
  __device__ static __forceinline__ float lg_nn(float x) { return __builtin_amdgcn_logf(x); }
  __device__ static __forceinline__ float ex_nn(float x) { return __builtin_amdgcn_exp2f(x); }
  __device__ static __forceinline__ float rcp(float x) { return __builtin_amdgcn_rcpf(x); }
};
template <>
struct Tr<double> {
  static constexpr double kExpScale = 1.0;
  __device__ static __forceinline__ double lg(double x) {
    return fm64::log_t(x, sFm64 + fm64::kExpTabLen, sFm64 + fm64::kExpTabLen + fm64::kLogTabLen);
  }
  __device__ static __forceinline__ double ex(double x) { return fm64::exp_t(x, sFm64); }
  // The forms of the dissipation: its logarithms are of |e|, k and cf (finite,
  // >= 0) and a NaN spectral value reaches its rate or its X through e itself,
  // so the special cases reduce to log 0 = -inf (k_rates 0.9 ms less per
  // hurricane member-substep).  The integration's exponential and the
  // diagnostic tail keep them
  __device__ static __forceinline__ double lg_nn(double x) {
    return fm64::log_t<false>(x, sFm64 + fm64::kExpTabLen,
                              sFm64 + fm64::kExpTabLen + fm64::kLogTabLen);
  }
  __device__ static __forceinline__ double ex_nn(double x) { return fm64::exp_t<false>(x, sFm64); }
  __device__ static __forceinline__ double rcp(double x) {
    double r = __builtin_amdgcn_rcp(x);
    r = fma(r, fma(-x, r, 1.0), r);
    return fma(r, fma(-x, r, 1.0), r);
  }
};

// Per-frequency wind-input factors in the form the sweeps use: ssin =
// y * (y > 0 ? pos : neg1 * m), y = |x| x, x = A cth + B sth - cp0, with
// m = fieldscale2 where the wind overruns the direction (cos(wdir - th) >
// 0), else 1 (a per-lane, per-direction constant).
template <typename T>
__device__ __forceinline__ T sin_y(const SinFreq<T>& q, T ct, T st) {
  const T x = fma(q.A, ct, fma(q.B, st, -q.cp0));
  return fabs(x) * x;
}
template <typename T>
__device__ __forceinline__ T sin_m(const SinFreq<T>& q, T y, T m) {
  const T pos = q.pos, neg = q.neg1 * m;
  return y * (y > T(0) ? pos : neg);
}

// ---------------------------------------------------------------------
// Directional moments of E^n, the raw material of the sds prefix: per
// (frequency, point) the sums over the directions of e, e cos 2th and
// e sin 2th in FP64, planes [om][3][ldi].  k_advect forms them from the spectrum it writes, so the sweeps
// need no exchange between the waves of a point and may be split over
// directions and frequencies freely; k_moments forms them after anything else
// wrote the spectrum.  The order of the sums does not depend on the launch:
// the directions of a group in the working precision, the groups in FP64.
// ---------------------------------------------------------------------
// Direction groups of the sums: the fewest of up to 9 (18, 36 for wide
// spectra) directions, as evenly as they divide.
__host__ __device__ inline int dir_groups(int pm) {
  return pm <= 72 ? (pm + 8) / 9 : pm <= 144 ? (pm + 17) / 18 : (pm + 35) / 36;
}

template <typename T>
struct Mom {
  T m0, mc, ms;
};

// Three planes of frequency o at point j: the moments, or dth/2 times their
// prefix (DomainDev::pfx).
template <typename T>
__device__ __forceinline__ Mom<T> load_mom(const T* mom, size_t ldi, int o, int j) {
  const rsrc_t pf = row_rsrc(mom, (size_t)o, 3 * ldi);
  const uint32_t v = (uint32_t)j * (uint32_t)sizeof(T), pl = (uint32_t)ldi * (uint32_t)sizeof(T);
  return Mom<T>{bld<T>(pf, v), bld<T>(pf, v, pl), bld<T>(pf, v, 2 * pl)};
}

// Running prefix of the moments over frequency, sum_{o' < o} k^3 dk m(o'),
// in FP64 (src/umwm_source_functions.F90:92-97).
struct Prefix {
  double a0 = 0, ac = 0, as = 0;
  __device__ __forceinline__ void add(double k3, const Mom<double>& m) {
    a0 += k3 * m.m0;
    ac += k3 * m.mc;
    as += k3 * m.ms;
  }
};

// Whether k_rates leaves the prefix for k_integrate or k_integrate, with D
// directions a wave, sums it again: in FP64 that spilled (155 -> 350 us at 2,852
// points), in the surrogate's variant it cost a tenth (865 -> 959 us at 127,587
// points x 49x72, k_rates 593 -> 574), and FP32 waves of twelve lost a wave per
// SIMD to it (426 -> 519 us at 179,813 points x 37x36, 636 -> 786 at 93,870 x
// 49x72, k_rates 219 -> 189 and 270 -> 242).  In plain FP32 with other widths
// the store costs k_rates more than k_integrate saves (nine: 256 + 427 against
// 301 + 415 us at 179,776 points; eighteen: 206 + 601 against 243 + 576 at
// 93,870 x 49x72).
template <typename T, bool SUR>
constexpr bool stored_prefix(int D) {
  return sizeof(T) == 8 || SUR || D == 12;
}

// k^3 dk of (o, j): FP64 reads the table, FP32 forms it from k as the sweeps
// do (TabGen).
template <typename T>
__device__ __forceinline__ double k3dk_at(const DomainDev<T>& d, const TabGen& tg, int o,
                                          uint32_t vj) {
  if constexpr (sizeof(T) == 4) {
    const float k = tg.load_k(o);
    return k * k * tg.kdk_of(k, o);
  } else {
    return bld<T>(row_rsrc(d.k3dk, o, (size_t)d.ldi), vj);
  }
}

// The prefix at frequency o0 of a sweep that starts there.
template <typename T>
__device__ __forceinline__ Prefix prefix_at(const DomainDev<T>& d, const TabGen& tg, int o0, int j,
                                            uint32_t vj) {
  Prefix P;
#pragma unroll 4
  for (int o = 0; o < o0; ++o)
    P.add(k3dk_at(d, tg, o, vj), load_mom(d.mom, d.ldi, o, j));
  return P;
}

// A substep's sources are integrated ahead of its rates after one whose time
// scales were this much longer than the advective limit (see k_integrate); the
// length stands where they turn out longer than it by kSpecSlack.
constexpr double kSpecMargin = 1.05, kSpecSlack = 1.01;

// ---------------------------------------------------------------------
// k_rates
// ---------------------------------------------------------------------
// Wave `slot` of a point block (blockIdx.y W + w) takes directions p0 ..
// p0 + DMAX - 1 of direction group slot % ng and the frequencies of chunk
// slot / ng; slots past ng * chunks are idle.  SUR launches keep all of a
// point's waves in one workgroup (one chunk, gridDim.y = 1).
// The moments of a frequency enter the prefix at the end of its iteration.
// Carried from the one before, they and the next ones' cost six registers more
// than loaded at its start, which the narrow FP32 sweeps have (9 directions:
// 289 against 303 us at 179,813 points x 37x36); the others then keep a wave a
// SIMD, some with the bound of kWaves: 36 directions in pairs 222 -> 190 us
// there, 280 -> 206 at 93,870 x 49x72, the surrogate's 9 876 -> 862 at 127,587.
template <typename T, int DMAX, bool PAIR, bool SUR>
constexpr int kWaves = sizeof(T) == 4 && ((SUR && DMAX == 9) || (!SUR && PAIR && DMAX == 36)) ? 3 : 2;

template <typename T, int DMAX, bool FULL, bool PAIR, bool SUR, bool STORE>
__global__ __launch_bounds__(512, (kWaves<T, DMAX, PAIR, SUR>)) void k_rates(const DomainDev<T>* __restrict__ doms,
                                               const BlockTask* __restrict__ tasks, int first,
                                               int rot_all, int ng, int chunks) {
  extern __shared__ double smem[];
  const BlockTask tk = tasks[blockIdx.x];
  const DomainDev<T>& d = doms[tk.dom];
  Scalars* sc = d.sc;
  if (sc->done) return;  // uniform over a domain's workgroups: k_integrate has run ahead
  stage_fm64<T>();
  // rotation tendency on the first substep of the launch (rot_all) and on
  // every substep of a domain with currents (src/umwm_advection.F90:117,
  // currents .or. first): the choice is per domain, so that batch members
  // with and without currents each follow the reference
  const bool rotation = rot_all || d.currents;
  const int W = blockDim.x >> 6, lane = threadIdx.x & 63, w = wave_id();
  const int j = tk.i0 + lane;
  const bool active = sc->sumt < d.dtg;
  const bool valid = active && j < d.im;
  // substeps taken so far: the rotating audit group (read before the last
  // block counts this substep)
  [[maybe_unused]] const int nsub0 = sc->nsub;
  const int pm = d.pm, om = d.om;
  const size_t ldi = d.ldi, ldq = d.ldq;
  const int slot = (int)blockIdx.y * W + w, chunk = uniform_div(slot, ng), grp = slot - chunk * ng;
  const int D = FULL ? DMAX : uniform_div(pm + ng - 1, ng), p0 = grp * D;
  // directions of this wave (uniform); FULL launches have ng * DMAX = pm
  const int nd = FULL ? DMAX : max(0, min(D, pm - p0));
  const int oper = uniform_div(om + chunks - 1, chunks);
  const int o0 = chunk * oper, o1 = min(om, o0 + oper);  // empty for an idle slot
  const uint32_t vj = (uint32_t)j * (uint32_t)sizeof(T);
  const uint32_t vr = (uint32_t)j * (uint32_t)(FT_N * sizeof(T));
  const uint32_t rb = (uint32_t)ldi * (uint32_t)sizeof(T);  // bytes of one direction row
  // the surrogate's bf16 rate rows
  [[maybe_unused]] const uint32_t vj2 = (uint32_t)j * 2u, rb2 = (uint32_t)ldi * 2u;
  // Arrays the frequency loop uses, held in registers: buffer stores are
  // opaque to the compiler, which would otherwise reload these pointers
  // from the domain record after every store.
  const T* const eb = d.e;
  const double* const momb = d.mom;
  [[maybe_unused]] T* const pfxb = d.pfx;
  const T* const ftab = d.ftab;
  const T* const fr = d.f;
  const T* const dir4 = d.dir4;
  double pts = INFINITY, rotmax = -INFINITY;

  if (active) {
    const PointState<T> s = point_fresh(d, j, valid && slot == 0);
    const int oc = s.oc;
    const int ocmax = wave_max_i32(valid ? oc : -1);
    // cg0 is not in the FP64 record: only ice attenuation needs it
    [[maybe_unused]] const bool anyice = __any(valid && s.ice != T(0));
    if (rotation && valid && slot == 0) pstore(d.oc_rot, ldi, j, (int32_t)oc);
    uint32_t vie = 0, viw = 0, vin = 0, vis = 0;
    T dvc = 0, duc = 0, odx = 0, ody = 0;
    if (rotation) {
      vie = (uint32_t)pload(d.ie, ldi, j) * (uint32_t)sizeof(T);
      viw = (uint32_t)pload(d.iw, ldi, j) * (uint32_t)sizeof(T);
      vin = (uint32_t)pload(d.in_, ldi, j) * (uint32_t)sizeof(T);
      vis = (uint32_t)pload(d.is_, ldi, j) * (uint32_t)sizeof(T);
      dvc = pload(d.vc, ldq, pload(d.iie, ldi, j)) - pload(d.vc, ldq, pload(d.iiw, ldi, j));
      duc = pload(d.uc, ldq, pload(d.iin, ldi, j)) - pload(d.uc, ldq, pload(d.iis, ldi, j));
      odx = pload(d.oneovdx, ldi, j);
      ody = pload(d.oneovdy, ldi, j);
    }
    const T sin_diss1 = T(d.sin_fac * d.fieldscale1), fs2 = T(d.fieldscale2);
    [[maybe_unused]] const T tpsf = T(d.twopisds_fac);
    const T spow = T(d.sds_power), mssf = T(d.mss_fac);
    const T nu4 = T(4 * d.nu_water), ig = T(1 / d.g);
    const double hdth = 0.5 * d.dth;
    // Slots q >= nd are computed but never used: their spectrum loads go
    // through a zero-range descriptor and read 0, their direction records
    // are dir4's zero padding, and they are masked out of the rate
    // maximum.  With no per-slot branch the compiler can interleave the
    // directions.
    const rsrc_t rz = make_rsrc(eb, 0u);
    // PAIR launches (FULL with an even DMAX) pair each direction p with p + pm/2
    // (theta + pi): cos and sin change sign while cos 2theta and sin 2theta
    // do not, so a pair shares its direction record and the mss factor.  Wave
    // w then holds pairs w DMAX/2 + h in slots h and h + DMAX/2, which also
    // halves the direction records the loop keeps in scalar registers.
    static_assert(!PAIR || (FULL && DMAX % 2 == 0), "paired sweeps are mask-free and even");
    constexpr int H = DMAX / 2;
    const int ph = grp * H, half = pm / 2;
    auto dirp = [&](int q) { return PAIR ? (q < H ? ph + q : ph + q - H + half) : p0 + q; };
    // overrun factor of slot q: fieldscale2 where the wind overruns the
    // direction, else 1; the paired loop reads it as bit q of mb (one
    // register instead of DMAX)
    using MB = std::conditional_t<(DMAX > 32), uint64_t, uint32_t>;
    MB mb = 0;
    T mq[DMAX];
#pragma unroll
    for (int q = 0; q < DMAX; ++q) {
      T ct, st, c2, s2;
      cld4(dir4, dirp(q), ct, st, c2, s2);
      const bool over = s.cw * ct + s.sw * st > T(0);
      mq[q] = over ? fs2 : T(1);
      if (over) mb |= MB(1) << q;
    }
    // Surrogate (FP32): lanes whose inputs passed the range check take the
    // network's spreading factor dm^2 in place of the one the moment
    // prefix gives, so that sds = dm^2 s with s = cf coth (e k^4)^p the
    // closed form of the bin.  The residual check holds the network's dm^2
    // against the bounds the prefix sets, [1, (1 + 2 mss_fac m0)^2] (m0 the
    // frequency prefix of the zeroth moment, which bounds the cos^2-weighted
    // ones), and the value used is clamped to them; a lane whose
    // energy-weighted share of bins outside the bounds (widened by
    // kSurBoundTol) exceeds the residual tolerance, or whose audited
    // dissipation error exceeds the audit tolerance, falls back to the plain
    // rates, which these waves always evaluate.  All waves of a workgroup
    // hold the same 64 points, so these choices agree across waves.
    // The domain-wide gate: when the previous substep's audited workgroups
    // together found the network's dissipation error above the audit
    // tolerance, every point takes the plain rates this substep; the
    // audited workgroups still evaluate the network, so that the audit can
    // open the gate again.
    [[maybe_unused]] int sok = 0;
    [[maybe_unused]] bool aud = false, gate = false;
    bool do_sur = false;
    [[maybe_unused]] const uint16_t* const rsur = d.sur_r;
    if constexpr (SUR) {
      if (rsur) {
        sok = valid ? pload(d.sur_ok, ldi, j) : 0;
        aud = d.sur_audit_stride > 0 && ((tk.local + nsub0) % d.sur_audit_stride) == 0;
        gate = sc->sur_closed == 0;
        // in a scalar register: the sweep's range follows from it, and with it
        // in a vector one every buffer access became a loop over the lanes'
        // descriptors (1,179 -> 877 us at 127,587 points x 49x72)
        do_sur = __builtin_amdgcn_readfirstlane(__any(sok != 0) && (gate || aud)) != 0;
      }
    }
    T rmax = 0;
    [[maybe_unused]] T rmax_s = 0, neg = 0, tot = 0, anum = 0, aden = 0;
    // One sweep over this wave's frequencies: `ds` also evaluates the
    // network's dissipation.
    auto sweep = [&](bool ds) {
    // the rates count up to the cut-off: past the last prognostic bin of the
    // wave's points there is nothing to evaluate (16 of 37 frequencies at
    // 15 m/s) unless the network's share of the energy is being measured
    const int omain = ds ? o1 : min(o1, ocmax + 1);
    // FP32 derives the tables from k (TabGen); FP64 loads the record
    constexpr bool kDerive = sizeof(T) == 4;
    TabGen tg;
    if constexpr (kDerive) tg.init(d, j, vj, o0);
    Prefix P = prefix_at(d, tg, o0, j, vj);
    T ec[DMAX];
    // the network's dm^2 - 1 of this and the next frequency as raw bf16
    // bits; the direction's row offset joins the lane offset (a vector add)
    // rather than holding DMAX more scalar registers
    [[maybe_unused]] uint32_t rc[DMAX];
    FreqTab<T> tc;
    constexpr bool kAhead = sizeof(T) == 4 && !SUR && DMAX <= 9;  // see kWaves
    Mom<double> mo;
    if constexpr (kAhead) mo = load_mom(momb, ldi, o0, j);
    {
      const rsrc_t ep = freq_rsrc(eb, o0, pm, ldi);
#pragma unroll
      for (int q = 0; q < DMAX; ++q) ec[q] = bld<T>(FULL || q < nd ? ep : rz, vj, dirp(q) * rb);
      if constexpr (SUR) {
        if (ds) {
          const rsrc_t rp = sur_rsrc(rsur, o0, pm, ldi);
#pragma unroll
          for (int q = 0; q < DMAX; ++q) rc[q] = bld_u16(FULL || q < nd ? rp : rz, vj2 + dirp(q) * rb2);
        }
      }
    }
    // (stores of lanes past the end are dropped rather than branched around:
    // a divergent branch here moves what it shares with the loads of the
    // moments, their descriptors, to vector registers)
    auto store_prefix = [&](int o, T pa0, T pac, T pas) {
      if constexpr (STORE) {
        if (grp == 0) {
          const rsrc_t pf = freq_rsrc(pfxb, o, 3, ldi);
          const uint32_t v = valid ? vj : kDropOffset;
          bst(pf, v, pa0);
          bst(pf, v, pac, rb);
          bst(pf, v, pas, 2 * rb);
        }
      }
    };
    for (int o = o0; o < omain; ++o) {
      // issue the next frequency's loads before computing this one
      const int on = o + 1 < omain ? o + 1 : o;
      T en[DMAX];
      const rsrc_t epn = freq_rsrc(eb, on, pm, ldi);
#pragma unroll
      for (int q = 0; q < DMAX; ++q) en[q] = bld<T>(FULL || q < nd ? epn : rz, vj, dirp(q) * rb);
      [[maybe_unused]] uint32_t rn[DMAX];
      if constexpr (SUR) {
        if (ds) {
          const rsrc_t rp = sur_rsrc(rsur, on, pm, ldi);
#pragma unroll
          for (int q = 0; q < DMAX; ++q) rn[q] = bld_u16(FULL || q < nd ? rp : rz, vj2 + dirp(q) * rb2);
        }
      }
      const Mom<double> mn = load_mom(momb, ldi, kAhead ? on : o, j);
      T k3 = 0;
      if constexpr (!kDerive) k3 = bld<T>(row_rsrc(d.k3dk, o, ldi), vj);
      float knext = 0.f;
      if constexpr (kDerive) {
        knext = tg.load_k(o + 4);
        tg.table(o, tc);
      } else {
        load_tab<kSweepSlots>(ftab, ldi, o, vr, tc);
      }

      const T k = tc[FT_K], k2 = k * k, fo = cld(fr, o);
      const T sdt = s.csdt * k;
      T crest;  // sbf + sdt + sdv - sice
      if constexpr (kDerive) {
        const T sice = T(2) * tc[FT_CG0] * s.ice;
        crest = tc[FT_SBF] + sdt + nu4 * k2 - sice;
        k3 = k2 * tc[FT_KDK];
      } else {
        crest = tc[FT_SBF] + sdt + nu4 * k2;
        if (anyice) crest -= T(2) * s.ice * bld<T>(row_rsrc(d.cg0, o, ldi), vj);
      }
      const SinFreq<T> sf = sin_freq(s, tc[FT_LOGL2], tc[FT_CP0], fo * k * ig, sin_diss1, fs2);
      const T pa0 = T(hdth * P.a0), pac = T(hdth * P.ac), pas = T(hdth * P.as);
      store_prefix(o, pa0, pac, pas);
      // sds (after cothkd) = cf coth dm^2 (e k4)^p = dm^2 ex(p lg e + Lk)
      T Lk;  // lg(cf coth k^(4 p)), in the FP64 record
      if constexpr (kDerive) {
        const T cfo = tpsf * fo * tc[FT_COTH];
        Lk = T(4) * spow * Tr<T>::lg_nn(k) + Tr<T>::lg_nn(cfo);  // lg(k^4) = 4 lg k
      } else {
        Lk = tc[FT_L];
      }
      const T cs = T(1) - (tc[FT_B1] + tc[FT_B2]);                // snl_arg
      const T q0 = T(1) + mssf * pa0, qc = mssf * pac, qs = mssf * pas;
      [[maybe_unused]] const T kdkv = tc[FT_KDK];
      T rq = 0;
      [[maybe_unused]] T rqs = 0;
      // sds = dm^2 sat with sat = ex(p lg |e| + Lk) = cf coth (e k4)^p: of
      // |e|, so that a bin emptied by round-off to about -1e-30 gives a
      // vanishing sds, as the 0 the reference's power of a non-positive
      // base is taken to be here, without a clamp instruction
      // the network's dm^2 of one bin: its rate, the residual of the
      // spreading-factor bounds and the audit sums (sat = cf coth (e k^4)^p,
      // sdp = the plain sds = dm^2 sat)
      [[maybe_unused]] const T qhi = (T(1) + T(2) * mssf * pa0) * (T(1) + T(2) * mssf * pa0);
      auto sur_bin = [&](T ss, T qn, T e, T sat, T sdp, bool use_slot) {
        const T dmn = T(1) + qn;  // the network stores dm^2 - 1
        const T sdn = fmin(fmax(dmn, T(1)), qhi) * sat;
        const T r2 = ss - fma(sdn, cs, crest);
        rqs = fmax(rqs, use_slot ? fabs(r2) : T(0));
        const T wv = e * kdkv;
        const bool inb = dmn >= T(1 - kSurBoundTol) && dmn <= qhi * T(1 + kSurBoundTol);
        neg += inb ? T(0) : wv;  // NaN or Inf fail the bounds too
        tot += wv;
        if (aud) {
          anum = fma(fabs(sdn - sdp), wv, anum);
          aden = fma(sdp, wv, aden);
        }
      };
      // an opaque copy per frequency (an empty asm statement): without it the
      // compiler hoists the DMAX bit tests out of the frequency loop into
      // DMAX registers, which costs a wave per SIMD at DMAX = 36
      MB mbl = mb;
      asm volatile("" : "+v"(mbl));
      if constexpr (PAIR) {
#pragma unroll
        for (int h = 0; h < H; ++h) {
          T ct, st, c2, s2;
          cld4(dir4, ph + h, ct, st, c2, s2);
          const T ea = ec[h], eb2 = ec[h + H];
          const T u = fma(sf.A, ct, sf.B * st);  // x of theta + pi is -u - cp0
          const T xa = u - sf.cp0, xb = -u - sf.cp0;
          const T ya = fabs(xa) * xa, yb = fabs(xb) * xb;
          const T na = ((mbl >> h) & 1) ? sf.neg2 : sf.neg1;
          const T nb = ((mbl >> (h + H)) & 1) ? sf.neg2 : sf.neg1;
          const T ssa = ya * (ya > T(0) ? sf.pos : na), ssb = yb * (yb > T(0) ? sf.pos : nb);
          T dm = fma(qc, c2, fma(qs, s2, q0));
          dm = dm * dm;
          const T sata = Tr<T>::ex_nn(fma(spow, Tr<T>::lg_nn(fabs(ea)), Lk));
          const T satb = Tr<T>::ex_nn(fma(spow, Tr<T>::lg_nn(fabs(eb2)), Lk));
          const T spa = dm * sata, spb = dm * satb;
          const T ra = ssa - fma(spa, cs, crest);
          const T rbb = ssb - fma(spb, cs, crest);
          rq = fmax(rq, fmax(fabs(ra), fabs(rbb)));
          if constexpr (SUR) {
            if (ds) {
              sur_bin(ssa, bf16_bits_to_f(rc[h]), ea, sata, spa, true);
              sur_bin(ssb, bf16_bits_to_f(rc[h + H]), eb2, satb, spb, true);
            }
          }
        }
      } else {
#pragma unroll
        for (int q = 0; q < DMAX; ++q) {
          T ct, st, c2, s2;
          cld4(dir4, p0 + q, ct, st, c2, s2);
          const T e = ec[q];
          const T ss = sin_m(sf, sin_y(sf, ct, st), mq[q]);
          T dm = fma(qc, c2, fma(qs, s2, q0));
          dm = dm * dm;
          const T sat = Tr<T>::ex_nn(fma(spow, Tr<T>::lg_nn(fabs(e)), Lk));
          const T sp = dm * sat;
          const T r = ss - fma(sp, cs, crest);
          rq = fmax(rq, FULL || q < nd ? fabs(r) : T(0));
          if constexpr (SUR) {
            if (ds) sur_bin(ss, bf16_bits_to_f(rc[q]), e, sat, sp, FULL || q < nd);
          }
        }
      }
      if (o <= oc) {  // rates of prognostic bins only
        rmax = fmax(rmax, rq);
        if constexpr (SUR) rmax_s = fmax(rmax_s, rqs);
      }
      if (rotation) {
        // rotation tendency of the first substep (src/umwm_advection.F90:329-349)
        const rsrc_t cpr = row_rsrc(d.cp0, o, ldi);
        const T dcx = bld<T>(cpr, vie) - bld<T>(cpr, viw);
        const T dcy = bld<T>(cpr, vin) - bld<T>(cpr, vis);
        if (o <= oc) {
          for (int q = 0; q < nd; ++q) {
            const int p = dirp(q);
            rotmax = fmax(rotmax, (double)rot_dir(dcx, dcy, cld(d.sth, p), cld(d.cth, p), dvc, duc,
                                                  odx, ody));
          }
        }
      }
      P.add(k3, kAhead ? mo : mn);
      mo = mn;
#pragma unroll
      for (int q = 0; q < DMAX; ++q) ec[q] = en[q];
      if constexpr (SUR) {
        if (ds) {
#pragma unroll
          for (int q = 0; q < DMAX; ++q) rc[q] = rn[q];
        }
      }
      if constexpr (kDerive) tg.advance(o, knext);
    }
    if constexpr (STORE) {
      // the prefix of the diagnostic tail's bins, for k_integrate
      if (grp == 0) {
#pragma unroll 4
        for (int t = max(o0, omain); t < o1; ++t) {
          const int o = __builtin_amdgcn_readfirstlane(t);  // see uniform_div
          store_prefix(o, T(hdth * P.a0), T(hdth * P.ac), T(hdth * P.as));
          P.add(k3dk_at(d, tg, o, vj), load_mom(momb, ldi, o, j));
        }
      }
    }
    };
    if (o0 < o1) sweep(do_sur);
    // bins above the cut-off hold a rotation of 0 and join the signed max
    if (rotation && nd > 0) rotmax = fmax(rotmax, 0.0);
    // the surrogate's verdict per lane (the same in every wave)
    [[maybe_unused]] bool use = false;
    if constexpr (SUR) {
      if (rsur) {
        double sneg = neg, stot = tot, snum = anum, sden = aden;
        if (W > 1) {
          __syncthreads();
          smem[(0 * W + w) * 64 + lane] = sneg;
          smem[(1 * W + w) * 64 + lane] = stot;
          smem[(2 * W + w) * 64 + lane] = snum;
          smem[(3 * W + w) * 64 + lane] = sden;
          __syncthreads();
          sneg = stot = snum = sden = 0;
          for (int q = 0; q < W; ++q) {
            sneg += smem[(0 * W + q) * 64 + lane];
            stot += smem[(1 * W + q) * 64 + lane];
            snum += smem[(2 * W + q) * 64 + lane];
            sden += smem[(3 * W + q) * 64 + lane];
          }
        }
        // written as negated <= so that NaN sums count as failures
        const bool rfail = !(sneg <= (double)d.sur_resid_tol * stot);
        const bool afail = aud && !(snum <= (double)d.sur_audit_tol * sden);
        use = valid && sok && !rfail && !afail && gate;
        if (w == 0) {
          if (valid) pstore(d.sur_use, ldi, j, (int32_t)(use ? 1 : 0));
          // counts as 64-bit integer atomics (ballot counts), the audit sums
          // as FP64 atomics from audited workgroups only: FP64 atomic adds
          // from every workgroup to the same eight words serialised and cost
          // several times the sweep itself
          const bool cnt[SS_AUDIT_NUM] = {valid,
                                          use,
                                          valid && !sok,
                                          valid && sok && rfail,
                                          valid && sok && !rfail && (afail || !gate),
                                          valid && aud};
          auto* ctr = reinterpret_cast<unsigned long long*>(d.sur_stats);
#pragma unroll
          for (int q = 0; q < SS_AUDIT_NUM; ++q) {
            const unsigned long long c = __popcll(__ballot(cnt[q]));
            if (lane == 0 && c) atomicAdd(ctr + q, c);
          }
          if (aud) {
            const double a = wave_sum(valid ? snum : 0.0), b = wave_sum(valid ? sden : 0.0);
            if (lane == 0) {
              atomicAdd(d.sur_stats + SS_AUDIT_NUM, a);
              atomicAdd(d.sur_stats + SS_AUDIT_DEN, b);
              // this substep's sums for the gate (thread 0 of the block,
              // which waits for its atomics before the arrival count)
              atomicAdd(&sc->sur_anum, a);
              atomicAdd(&sc->sur_aden, b);
            }
          }
        }
      }
    }
    // max |rate| of the point over all waves
    __syncthreads();
    T rsel = rmax;
    if constexpr (SUR) rsel = use ? rmax_s : rmax;
    smem[w * 64 + lane] = (double)rsel;
    __syncthreads();
    if (w == 0) {
      double mx = 0;
      for (int q = 0; q < W; ++q) mx = fmax(mx, smem[q * 64 + lane]);
      pts = d.explim / mx;
      if (valid) {
        // a point whose waves span several workgroups collects its maximum
        // (rates are >= 0, so their bits order as they do); k_stress divides
        if (gridDim.y > 1)
          atomicMax(d.rkey + j, (unsigned long long)__double_as_longlong(mx));
        else
          pstore(d.pts, ldi, j, pts);
      }
      if (!valid) pts = INFINITY;
    }
    if (!valid) rotmax = -INFINITY;
  }
  // Block reductions, then the grid-wide ones through two agent-scope
  // atomics per block on order-preserving integer keys (okey) kept in the
  // domain's Scalars: an atomic max of ~okey(min pts) and of okey(max
  // rotation rate).  The last block to arrive reads and clears them.  There
  // are no per-block partials in memory, hence no release fence: on this
  // multi-XCD GPU an agent-scope release writes back and invalidates the
  // L2 and cost about a fifth of the kernel.  Device atomics are performed
  // at the device's coherence point; the wait for their completion before
  // the arrival count orders them ahead of it.
  __shared__ double bred[2][16];
  __shared__ int is_last;
  __syncthreads();
  const double wmin = wave_min(pts), wmax = wave_max(rotmax);
  if (lane == 0) {
    bred[0][w] = wmin;
    bred[1][w] = wmax;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double mn = INFINITY, mx = -INFINITY;
    for (int q = 0; q < W; ++q) {
      mn = fmin(mn, bred[0][q]);
      mx = fmax(mx, bred[1][q]);
    }
    atomicMax(&sc->pts_key, ~okey(mn));
    atomicMax(&sc->rot_key, okey(mx));
    // both atomics complete (s_waitcnt 0) before the arrival count
    __builtin_amdgcn_s_waitcnt(0);
    const unsigned tkt = atomicAdd(&sc->counter, 1u);
    is_last = (tkt == (unsigned)d.nblocks * gridDim.y - 1);
  }
  __syncthreads();
  if (!is_last) return;
  if (threadIdx.x == 0) {
    const unsigned long long kmin = atomicExch(&sc->pts_key, 0ull);
    const unsigned long long kmax = atomicExch(&sc->rot_key, 0ull);
    const double mn = kmin ? okey_inv(~kmin) : INFINITY;
    const double mx = kmax ? okey_inv(kmax) : -INFINITY;
    if (active) {
      // src/umwm_physics.F90:44-58
      double dts = fmin(fmin(mn, d.dtamin), d.dtg - sc->sumt);
      if (!d.restart && first) dts = 0;
      sc->dts = dts;
      sc->dta = dts;
      sc->sumt = sc->sumt + dts;
      // src/umwm_advection.F90:352-365 (signed maxval)
      if (rotation) {
        sc->maxrot = mx;
        sc->dtr_temp = (mx <= d.tiny) ? dts : d.dth / mx;
      }
      sc->dtr = fmin(sc->dtr_temp, dts);
      sc->nsub = sc->nsub + 1;
      sc->last = sc->sumt >= d.dtg ? 1 : 0;
      sc->spec = !d.currents && mn >= kSpecMargin * d.dtamin ? 1 : 0;
      if constexpr (SUR) {
        if (d.sur_r) {
          // the gate for the next substep: closed while the sampled error
          // exceeds the tolerance; a substep with no audited point keeps it
          const double an = __longlong_as_double(
              (long long)atomicExch(reinterpret_cast<unsigned long long*>(&sc->sur_anum), 0ull));
          const double ad = __longlong_as_double(
              (long long)atomicExch(reinterpret_cast<unsigned long long*>(&sc->sur_aden), 0ull));
          if (ad > 0) sc->sur_closed = an <= (double)d.sur_audit_tol * ad ? 0 : 1;
        }
      }
    }
    sc->active = active ? 1 : 0;
    sc->counter = 0;
  }
}

// ---------------------------------------------------------------------
// k_integrate
// ---------------------------------------------------------------------
// SPEC launches run before k_rates, over the substep length that is expected
// (Scalars::spec: the advective limit, or what is left of the dtg), and keep
// the largest |rate| of each point beside the integration.  If the point with
// the shortest time scale allows that length, it is the substep's length
// whatever the exact time scales are: the last workgroup then does k_rates'
// bookkeeping and the substep's k_rates and plain k_integrate return at once.
// Else they run as always and overwrite E*.  The rates share the
// integration's wind input and dissipation, which k_rates groups otherwise: in
// FP32 its dissipation differs by up to 6e-6 (the rounding of an exponent of
// several tens; 1e-5 at sds_power = 4), and a rate is a difference in which
// both may cancel.  So a length within kSpecSlack of the time scales is left to
// k_rates: the two would have to cancel a thousandfold in a point's largest
// rate before a length differed.  Lengths are the same bits then, the points'
// time scales agree to that rounding.  k_rates + k_integrate, and this kernel
// (with FP64's k_prefix) in their place, in us: 180,000 points x 37x36 FP32
// 258 + 454 -> 479; 399,424 x 49x72 FP32 914 + 2,603 -> 2,916; 129,000 x 49x72
// FP64 1,404 + 3,536 -> 60 + 3,504; 42,000 x 37x36 FP64 199 + 466 -> 29 + 455.
// The price of a wrong guess is this kernel's time, so one is made only after a
// substep whose time scales were a twentieth above the limit (kSpecMargin).
// All waves of a point are in one workgroup here (one chunk, gridDim.y = 1).
template <typename T, int DMAX, bool FULL, bool SUR, bool SPEC>
__global__ __launch_bounds__(512) void k_integrate(const DomainDev<T>* __restrict__ doms,
                                                   const BlockTask* __restrict__ tasks, int ng,
                                                   int chunks) {
  const BlockTask tk = tasks[blockIdx.x];
  const DomainDev<T>& d = doms[tk.dom];
  Scalars* const sc = d.sc;
  // uniform over a domain's workgroups
  if constexpr (SPEC) {
    if (!sc->spec || d.currents || !(sc->sumt < d.dtg)) return;
  } else {
    if (!sc->active || sc->done) return;
  }
  stage_fm64<T>();
  const int j = tk.i0 + (threadIdx.x & 63);
  const bool valid = j < d.im;
  const int pm = d.pm, om = d.om;
  const size_t ldi = d.ldi;
  const int slot = (int)blockIdx.y * (int)(blockDim.x >> 6) + wave_id();
  const int chunk = uniform_div(slot, ng), grp = slot - chunk * ng;
  const int D = FULL ? DMAX : uniform_div(pm + ng - 1, ng), p0 = grp * D;
  const int nd = FULL ? DMAX : max(0, min(D, pm - p0));
  // This wave completes bins o0 .. o1 - 1.  It sweeps two frequencies past
  // them for the snl gains their energy feeds down, of which it takes only
  // X; the wave of the next chunk integrates those bins.
  const int oper = uniform_div(om + chunks - 1, chunks);
  const int o0 = chunk * oper, o1 = min(om, o0 + oper);
  if constexpr (!SPEC) {
    if (o0 >= o1) return;  // an idle slot; no barrier follows
  }
  double dtd = sc->dts;
  if constexpr (SPEC) dtd = fmin(d.dtamin, d.dtg - sc->sumt);
  const T dts = T(dtd);
  const T dtx = dts * Tr<T>::kExpScale;  // dts in the exponential's base
  const uint32_t vj = (uint32_t)j * (uint32_t)sizeof(T);
  const uint32_t vr = (uint32_t)j * (uint32_t)(FT_N * sizeof(T));
  const uint32_t rb = (uint32_t)ldi * (uint32_t)sizeof(T);
  // Arrays the frequency loop uses, held in registers (see k_rates).
  const T* const eb = d.e;
  T* const esb = d.es;
  const T* const ftab = d.ftab;
  constexpr bool kStored = stored_prefix<T, SUR>(DMAX), kRegDirs = sizeof(T) == 4;
  [[maybe_unused]] const double* const momb = d.mom;
  [[maybe_unused]] const T* const pfxb = d.pfx;
  const T* const fr = d.f;

  PointState<T> s;
  if constexpr (SPEC)
    s = point_fresh(d, j, valid && slot == 0);
  else
    s = point_stored(d, j);
  const int oc = s.oc;
  [[maybe_unused]] T rmax = 0;  // SPEC: the largest |rate| of this wave's bins
  [[maybe_unused]] const bool anyice = __any(valid && s.ice != T(0));
  const T sin_diss1 = T(d.sin_fac * d.fieldscale1), fs2 = T(d.fieldscale2);
  [[maybe_unused]] const T tpsf = T(d.twopisds_fac);
  const T spow = T(d.sds_power), ipow = T(d.inv_sds_power);
  const T mssf = T(d.mss_fac), dsnl = dts * T(d.snl_fac);
  const T nu4 = T(4 * d.nu_water), ig = T(1 / d.g);
  // direction constants of this wave, loaded once.  Slots q >= nd are
  // computed but never used: their loads and stores go through a
  // zero-range descriptor (loads read 0, stores are dropped), so the
  // direction loop has no per-slot branch and the compiler can interleave
  // the directions.
  const rsrc_t rz = make_rsrc(eb, 0u);
  // direction constants of this wave.  FP32 keeps them in registers; in FP64
  // that cost a wave per SIMD, so it keeps the overrun factors (fieldscale2,
  // see sin_m) as bits of mb and re-reads the direction records per frequency
  [[maybe_unused]] uint32_t mb = 0;
  [[maybe_unused]] T mq[DMAX], ctq[DMAX], stq[DMAX];
#pragma unroll
  for (int q = 0; q < DMAX; ++q) {
    T ct, st, c2, s2;
    cld4(d.dir4, p0 + q, ct, st, c2, s2);
    const bool over = s.cw * ct + s.sw * st > T(0);
    if constexpr (kRegDirs) {
      mq[q] = over ? fs2 : T(1);
      ctq[q] = ct;
      stq[q] = st;
    } else {
      if (over) mb |= 1u << q;
    }
  }
  const T* const dir4 = d.dir4;
  // per direction, the partial E* = (E^n + partial E_s) / 2 of the two
  // previous frequencies, still waiting for their snl gains
  T H1[DMAX], H2[DMAX];
#pragma unroll
  for (int q = 0; q < DMAX; ++q) H1[q] = H2[q] = 0;
  T b1m1 = 0, b2m2 = 0, b2m1 = 0;  // bf1r(o-1), bf2r(o-2), bf2r(o-1)
  // Surrogate (FP32): the lanes k_rates let take the network's rates use
  // its spreading factor dm^2, clamped to [1, (1 + 2 mss_fac m0)^2] as
  // there, wherever the moment prefix's dm^2 would enter: the dissipation
  // in the integration, in snl and in the diagnostic tail.
  [[maybe_unused]] int use = 0;
  [[maybe_unused]] bool do_sur = false;
  [[maybe_unused]] const uint16_t* const rsur = d.sur_r;
  [[maybe_unused]] const uint32_t vj2 = (uint32_t)j * 2u, rb2 = (uint32_t)ldi * 2u;
  if constexpr (SUR) {
    if (rsur) {
      use = valid ? pload(d.sur_use, ldi, j) : 0;
      do_sur = __any(use != 0);
    }
  }
  T ec[DMAX];
  [[maybe_unused]] uint32_t rc[DMAX];  // raw bf16 bits of dm^2 - 1 (see k_rates)
  {
    const rsrc_t ep = freq_rsrc(eb, o0, pm, ldi);
#pragma unroll
    for (int q = 0; q < DMAX; ++q) ec[q] = bld<T>(FULL || q < nd ? ep : rz, vj, (p0 + q) * rb);
    if constexpr (SUR) {
      if (do_sur) {
        const rsrc_t rp = sur_rsrc(rsur, o0, pm, ldi);
#pragma unroll
        for (int q = 0; q < DMAX; ++q) rc[q] = bld_u16(FULL || q < nd ? rp : rz, vj2 + (p0 + q) * rb2);
      }
    }
  }
  FreqTab<T> tc;
  // FP32 derives the tables from k (TabGen); FP64 loads them when needed
  // (as in k_rates)
  constexpr bool kDerive = sizeof(T) == 4;
  TabGen tg;
  if constexpr (kDerive) tg.init(d, j, vj, o0);
  // the stored prefix (prefetched in FP32, loaded when needed in FP64) or
  // the moments it is summed from
  [[maybe_unused]] Mom<T> pc{};
  [[maybe_unused]] Prefix P;
  [[maybe_unused]] Mom<double> mo{};
  if constexpr (!kStored) {
    P = prefix_at(d, tg, o0, j, vj);
    mo = load_mom(momb, ldi, o0, j);
  } else if constexpr (kDerive) {
    pc = load_mom(pfxb, ldi, o0, j);
  }
  const int oend = min(om, o1 + 2);
  for (int o = o0; o < oend; ++o) {
    const int on = o + 1 < om ? o + 1 : o;
    T en[DMAX];
    const rsrc_t epn = freq_rsrc(eb, on, pm, ldi);
#pragma unroll
    for (int q = 0; q < DMAX; ++q) en[q] = bld<T>(FULL || q < nd ? epn : rz, vj, (p0 + q) * rb);
    [[maybe_unused]] uint32_t rn[DMAX];
    if constexpr (SUR) {
      if (do_sur) {
        const rsrc_t rp = sur_rsrc(rsur, on, pm, ldi);
#pragma unroll
        for (int q = 0; q < DMAX; ++q) rn[q] = bld_u16(FULL || q < nd ? rp : rz, vj2 + (p0 + q) * rb2);
      }
    }
    [[maybe_unused]] Mom<T> pn{};
    [[maybe_unused]] Mom<double> mn{};
    float knext = 0.f;
    if constexpr (kDerive) {
      knext = tg.load_k(o + 4);
      if constexpr (kStored)
        pn = load_mom(pfxb, ldi, on, j);
      else
        mn = load_mom(momb, ldi, on, j);
      tg.table(o, tc);
    } else {
      load_tab<kSweepSlots>(ftab, ldi, o, vr, tc);
      pc = load_mom(pfxb, ldi, o, j);
    }
    if constexpr (!kStored) {
      const double hdth = 0.5 * d.dth;
      pc = Mom<T>{T(hdth * P.a0), T(hdth * P.ac), T(hdth * P.as)};
    }
    const T pa0 = pc.m0, pac = pc.mc, pas = pc.ms;

    const T k = tc[FT_K], fo = cld(fr, o);
    const T sdt = s.csdt * k;
    T ctail;  // sdt + sdv - sice
    if constexpr (kDerive) {
      const T sice = T(2) * tc[FT_CG0] * s.ice;
      ctail = sdt + nu4 * (k * k) - sice;
    } else {
      ctail = sdt + nu4 * (k * k);
      if (anyice) ctail -= T(2) * s.ice * bld<T>(row_rsrc(d.cg0, o, ldi), vj);
    }
    const T crest = tc[FT_SBF] + ctail;
    const SinFreq<T> sf = sin_freq(s, tc[FT_LOGL2], tc[FT_CP0], fo * k * ig, sin_diss1, fs2);
    // FP32 forms sds before cothkd; FP64 takes lg(cf coth k^(4 p)) from its
    // record, so its sds and X are after cothkd and the snl weights carry
    // icx = 1 / cothkd instead
    T Lk, dtc, icx = T(1);
    [[maybe_unused]] T icfc = 0, lk4 = 0;
    if constexpr (kDerive) {
      const T cf = tpsf * fo;
      const T coth = tc[FT_COTH];
      lk4 = T(4) * Tr<T>::lg(k);          // lg(k^4)
      Lk = spow * lk4 + Tr<T>::lg(cf);
      dtc = dtx * coth;
      icfc = Tr<T>::rcp(cf * coth);
    } else {
      Lk = tc[FT_L];
      dtc = dtx;
      icx = Tr<T>::rcp(tc[FT_COTH]);
    }
    const T c0 = -dtx * crest;
    // snl_arg, for sds as this kernel forms it
    [[maybe_unused]] T csr = T(1) - (tc[FT_B1] + tc[FT_B2]), rq = 0;
    if constexpr (SPEC && kDerive) csr *= tc[FT_COTH];
    // the spreading factor's upper bound, from the zeroth-moment prefix
    [[maybe_unused]] const T qhi = (T(1) + T(2) * mssf * pa0) * (T(1) + T(2) * mssf * pa0);
    // dm = q0 + qc cos 2th + qs sin 2th = (q0 - qc) + ct (2 qc ct + 2 qs st),
    // with cos 2th = 2 ct^2 - 1 and sin 2th = 2 ct st: the sweep keeps
    // only ct and st per direction
    const T qc = mssf * pac;
    const T q0m = T(1) + mssf * pa0 - qc, qc2 = T(2) * qc, qs2 = T(2) * mssf * pas;
    const bool own = o < o1;  // false in the two frequencies past the chunk
    const bool prog = o <= oc;
    const bool in1 = (o >= 1) && (o - 1 <= oc);  // bin o-1 is prognostic
    const bool fin = valid && (o >= o0 + 2) && (o - 2 <= oc);  // bin o-2 completes now
    T hdb1 = in1 ? T(0.5) * dts * b1m1 : T(0), hdb2 = T(0.5) * dts * b2m2, dsc = dsnl;
    if constexpr (!kDerive) {
      hdb1 *= icx;
      hdb2 *= icx;
      dsc *= icx;
    }
    const uint32_t vtail = (valid && !prog && own) ? vj : kDropOffset;
    const uint32_t vfin = fin ? vj : kDropOffset;
    const bool anyfin = __any(fin), anytail = own && __any(valid && !prog);
    const rsrc_t rs0 = freq_rsrc(esb, o, pm, ldi);
    // max(o, 2) - 2 rather than a conditional: the latter becomes a vector
    // saturating subtract, which moves the descriptor to vector registers
    const rsrc_t rs2 = freq_rsrc(esb, max(o, 2) - 2, pm, ldi);
    // One pass over this wave's directions; PROG / TAIL / FIN say whether
    // any lane of the wave integrates a prognostic bin, fills a tail bin
    // or completes bin o-2 at this frequency (wave-uniform, so each
    // combination is a straight-line loop).
    // NEEDX: some bin of the wave takes snl gains or losses from this
    // frequency; past the cut-off's two followers none does and the
    // dissipation (an exponential and a logarithm per bin) is not formed.
    uint32_t mbl = mb;  // opaque copies: see k_rates
    int dz = 0;
    asm volatile("" : "+v"(mbl), "+s"(dz));
    auto sweep = [&](auto PROG, auto TAIL, auto FIN, auto NEEDX) {
#pragma unroll
      for (int q = 0; q < DMAX; ++q) {
        const uint32_t so = (uint32_t)(p0 + q) * rb;
        const T e = ec[q];
        T ct, st, ss;
        if constexpr (kRegDirs) {
          ct = ctq[q];
          st = stq[q];
          ss = sin_m(sf, sin_y(sf, ct, st), mq[q]);
        } else {
          T c2, s2;
          cld4(dir4, p0 + q + dz, ct, st, c2, s2);
          const T y = sin_y(sf, ct, st);
          const T pos = sf.pos, neg1 = sf.neg1, neg2 = sf.neg2;  // see sin_bin
          const T neg = ((mbl >> q) & 1) ? neg2 : neg1;
          ss = y * (y > T(0) ? pos : neg);
        }
        T dm = fma(ct, fma(qc2, ct, qs2 * st), q0m);
        dm = dm * dm;
        if constexpr (SUR) {
          if (do_sur && use) dm = fmin(fmax(T(1) + bf16_bits_to_f(rc[q]), T(1)), qhi);  // dm^2 - 1
        }
        T X = 0, G = 0;  // X: sds e
        if constexpr (decltype(NEEDX)::value) {
          // |e|: see k_rates; a NaN of e stays in X through e
          const T sds = dm * Tr<T>::ex_nn(fma(spow, Tr<T>::lg_nn(fabs(e)), Lk));
          X = sds * e;
          if constexpr (decltype(PROG)::value) {
            if constexpr (SPEC) {
              // FP64 has no registers left for a frequency's own maximum (31
              // spilled, 541 against 455 us at 42,000 points); FP32 has, and
              // saves the select per bin (2,916 against 3,039 us)
              if constexpr (kDerive)
                rq = fmax(rq, FULL || q < nd ? fabs(ss - fma(sds, csr, crest)) : T(0));
              else
                rmax = fmax(rmax, prog && (FULL || q < nd) ? fabs(ss - fma(sds, csr, crest)) : T(0));
            }
            // E_s = e exp(dts (ssin - sds - sbf - sdt - sdv + sice)) + dts snl
            const T a = fma(-dtc, sds, fma(dtx, ss, c0));
            G = prog ? fma(-dsc, X, e * Tr<T>::ex(a)) : T(0);
          }
        }
        if constexpr (decltype(TAIL)::value) {
          // diagnostic tail, src/umwm_physics.F90:70-80: k^-4 t^(1/p), t =
          // num / (cf coth dm^2); in FP64 ex((lg(num / dm^2) - Lk) / p)
          const T num = fmax(ss, T(0)) - ctail;
          T es_;
          if constexpr (kDerive) {
            const T t = fmax(num, T(0)) * (icfc * Tr<T>::rcp(dm));
            es_ = Tr<T>::ex(fma(ipow, Tr<T>::lg(t), -lk4));
          } else {
            es_ = Tr<T>::ex(ipow * (Tr<T>::lg(fmax(num, T(0)) * Tr<T>::rcp(dm)) - Lk));
          }
          bst(FULL || q < nd ? rs0 : rz, vtail, T(0.5) * (e + es_), so);
        }
        T h1 = H1[q];
        if constexpr (decltype(NEEDX)::value) h1 = fma(hdb1, X, h1);  // bf1r(o-1) X(o) into bin o-1
        if constexpr (decltype(FIN)::value)  // bf2r(o-2) X(o) completes bin o-2
          bst(FULL || q < nd ? rs2 : rz, vfin, fma(hdb2, X, H2[q]), so);
        H2[q] = h1;
        H1[q] = T(0.5) * (e + G);
      }
    };
    using Y = std::true_type;
    using N = std::false_type;
    const bool anyprog = own && __any(valid && prog);
    if (anyprog) {
      if (anytail) {
        if (anyfin) sweep(Y{}, Y{}, Y{}, Y{}); else sweep(Y{}, Y{}, N{}, Y{});
      } else {
        if (anyfin) sweep(Y{}, N{}, Y{}, Y{}); else sweep(Y{}, N{}, N{}, Y{});
      }
    } else if (anyfin || __any(valid && in1)) {
      if (anytail) sweep(N{}, Y{}, Y{}, Y{}); else sweep(N{}, N{}, Y{}, Y{});
    } else if (anytail) {
      sweep(N{}, Y{}, N{}, N{});
    }
    if constexpr (SPEC && kDerive) {
      if (prog) rmax = fmax(rmax, rq);
    }
    b2m2 = b2m1;
    b2m1 = tc[FT_B2];
    b1m1 = tc[FT_B1];
#pragma unroll
    for (int q = 0; q < DMAX; ++q) ec[q] = en[q];
    if constexpr (SUR) {
      if (do_sur) {
#pragma unroll
        for (int q = 0; q < DMAX; ++q) rc[q] = rn[q];
      }
    }
    if constexpr (!kStored) {
      const double k3 = k * k * tc[FT_KDK];  // k^3 dk
      P.add(k3, mo);
      mo = mn;
    }
    if constexpr (kDerive) {
      tg.advance(o, knext);
      if constexpr (kStored) pc = pn;
    }
  }
  if constexpr (SPEC) {
    // the point's time scale, and the grid's as in k_rates
    __shared__ double red[8][64];
    const int W = blockDim.x >> 6, w = wave_id(), lane = threadIdx.x & 63;
    red[w][lane] = (double)rmax;
    __syncthreads();
    if (w > 0) return;
    double mx = 0;
    for (int q = 0; q < W; ++q) mx = fmax(mx, red[q][lane]);
    const double pts = d.explim / mx;
    if (valid) pstore(d.pts, ldi, j, pts);
    const double mn = wave_min(valid ? pts : (double)INFINITY);
    if (lane > 0) return;
    atomicMax(&sc->pts_key, ~okey(mn));
    __builtin_amdgcn_s_waitcnt(0);  // complete before the arrival count
    if (atomicAdd(&sc->counter, 1u) != (unsigned)d.nblocks - 1) return;
    const double lim = okey_inv(~atomicExch(&sc->pts_key, 0ull));
    const bool fits = lim >= kSpecSlack * dtd;
    if (fits) {
      sc->dts = dtd;
      sc->dta = dtd;
      sc->sumt = sc->sumt + dtd;
      sc->dtr = fmin(sc->dtr_temp, dtd);
      sc->nsub = sc->nsub + 1;
      sc->last = sc->sumt >= d.dtg ? 1 : 0;
      sc->active = 1;
    }
    sc->spec = fits ? 1 : 0;
    sc->done = fits ? 1 : 0;
    if (fits) sc->ahead += 1; else sc->missed += 1;
    sc->counter = 0;
  }
}

// The prefix a SPEC launch reads where it is stored: k_rates, which leaves it
// otherwise, has not run.  A thread a point; bound by the six FP64 planes a
// frequency that it reads and writes.
template <typename T>
__global__ __launch_bounds__(64) void k_prefix(const DomainDev<T>* __restrict__ doms,
                                               const BlockTask* __restrict__ tasks) {
  const BlockTask tk = tasks[blockIdx.x];
  const DomainDev<T>& d = doms[tk.dom];
  const Scalars* sc = d.sc;
  if (!sc->spec || d.currents || !(sc->sumt < d.dtg)) return;
  const int j = tk.i0 + (int)threadIdx.x;
  if (j >= d.im) return;
  const size_t ldi = d.ldi;
  const uint32_t vj = (uint32_t)j * (uint32_t)sizeof(T);
  const uint32_t rb = (uint32_t)ldi * (uint32_t)sizeof(T);
  const double hdth = 0.5 * d.dth;
  const int om = d.om;
  TabGen tg;
  Prefix P;
#pragma unroll 4
  for (int o = 0; o < om; ++o) {
    const rsrc_t pf = freq_rsrc(d.pfx, o, 3, ldi);
    bst(pf, vj, T(hdth * P.a0));
    bst(pf, vj, T(hdth * P.ac), rb);
    bst(pf, vj, T(hdth * P.as), 2 * rb);
    P.add(k3dk_at(d, tg, o, vj), load_mom(d.mom, ldi, o, j));
  }
}

// ---------------------------------------------------------------------
// k_advect: propagation + refraction + e = ef, one wave per (frequency o,
// 64 sea points); workgroups of FW waves take FW consecutive frequencies.
// Directions are processed in blocks of NB (pm is a multiple of 4) with
// the next block's loads in flight while the current block is computed.
//
// The upwind flux of src/umwm_advection.F90:28-44 is evaluated by sign:
// both x-edge speeds cg(i)+cg(nbr) times cos(th + curv) share the sign of
// cos(th + curv), so the x flux is c (Ae E*(upwind east) - Aw E*(upwind
// west)), Ae = 2 (cg(i) + cg(ie)) dye, and likewise in y; refraction's
// upwind flux (:166-172) is r (E* upwind) per edge.  Regrouped, equal to
// the reference up to rounding.
// ---------------------------------------------------------------------
template <typename T>
struct AdvLoads {
  T eo, ee, ew, en, es;  // E* at the point and its four neighbours
  T en0;                 // E^n at the point
};

// Sums over the directions in the order of the moments (see Mom): `add`
// takes directions in sequence, `group` ends a group.  t: e, e cos 2th,
// e sin 2th and in FP64 the stress partials; FP32 keeps the stress partials
// and the wave height as one running sum over all directions each.
template <typename T>
struct DirSums {
  static constexpr bool kSeq = sizeof(T) == 4;
  static constexpr int kGrouped = kSeq ? 3 : 5;
  T q[5], hs;
  double t[5];
  __device__ __forceinline__ void clear() {
    hs = 0;
#pragma unroll
    for (int i = 0; i < 5; ++i) {
      q[i] = 0;
      t[i] = 0;
    }
  }
  // e, and its wind input in the stress partials
  __device__ __forceinline__ void add(T v, T wv, T ct, T st, T c2, T s2) {
    q[0] += v;
    q[1] = fma(v, c2, q[1]);
    q[2] = fma(v, s2, q[2]);
    q[3] = fma(wv, ct, q[3]);
    q[4] = fma(wv, st, q[4]);
    if constexpr (kSeq) hs += v;
  }
  __device__ __forceinline__ void group() {
#pragma unroll
    for (int i = 0; i < kGrouped; ++i) {
      t[i] += (double)q[i];
      q[i] = 0;
    }
  }
};

// Stores the moments of (o, j).
template <typename T>
__device__ __forceinline__ void store_mom(const DomainDev<T>& d, int o, int j, double m0, double mc,
                                          double ms) {
  const rsrc_t r = row_rsrc(d.mom, (size_t)o, 3 * (size_t)d.ldi);
  const uint32_t v = (uint32_t)j * 8u, pl = (uint32_t)d.ldi * 8u;
  bst(r, v, m0);
  bst(r, v, mc, pl);
  bst(r, v, ms, 2 * pl);
}

// The moments of the current spectrum, after anything but k_advect wrote it;
// one wave per (frequency, 64 sea points).
template <typename T>
__global__ __launch_bounds__(64) void k_moments(const DomainDev<T>* __restrict__ doms,
                                                const BlockTask* __restrict__ tasks) {
  const BlockTask tk = tasks[blockIdx.x];
  const DomainDev<T>& d = doms[tk.dom];
  const int o = (int)blockIdx.y, pm = d.pm;
  if (o >= d.om) return;
  const int j = tk.i0 + (int)threadIdx.x;
  const size_t ldi = d.ldi;
  const uint32_t vj = (uint32_t)j * (uint32_t)sizeof(T), rb = (uint32_t)ldi * (uint32_t)sizeof(T);
  const rsrc_t pe = freq_rsrc(d.e, o, pm, ldi);
  const int ng = dir_groups(pm), glen = uniform_div(pm + ng - 1, ng);
  DirSums<T> S;
  S.clear();
  int gend = glen;
  for (int p = 0; p < pm; p += 4) {
    T v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = bld<T>(pe, vj, (p + q) * rb);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      T ct, st, c2, s2;
      cld4(d.dir4, p + q, ct, st, c2, s2);
      S.add(v[q], T(0), ct, st, c2, s2);
      if (p + q + 1 == gend) {
        S.group();
        gend += glen;
      }
    }
  }
  S.group();
  if (j < d.im) store_mom(d, o, j, S.t[0], S.t[1], S.t[2]);
}

// SPLIT: one workgroup per (frequency, 64 sea points), a wave per direction
// group, for launches that would otherwise leave most of the GPU idle.
// Else fw = blockDim / 64 frequencies per workgroup, a wave taking all
// directions of one.  Both add in the same order, so that a domain's results
// do not depend on what else is in the launch: the waves' groups are joined in
// turn, and the running sums of FP32 are taken by one wave from the directions'
// terms, which the others leave in LDS.
template <typename T, int NB, bool SPLIT>
__global__ __launch_bounds__(SPLIT ? 512 : 256) void k_advect(
    const DomainDev<T>* __restrict__ doms, const BlockTask* __restrict__ tasks, int ng) {
  const BlockTask tk = tasks[blockIdx.x];
  const DomainDev<T>& d = doms[tk.dom];
  const int wid = wave_id();
  const int o = SPLIT ? (int)blockIdx.y : (int)blockIdx.y * (int)(blockDim.x >> 6) + wid;
  const Scalars* sc = d.sc;
  if (o >= d.om || !sc->active) return;  // uniform over the workgroup when SPLIT
  const int j = tk.i0 + (threadIdx.x & 63);
  const bool valid = j < d.im;
  const int pm = d.pm;
  const size_t ldi = d.ldi, ldq = d.ldq;
  const uint32_t vj = (uint32_t)j * (uint32_t)sizeof(T);
  const uint32_t vst = valid ? vj : kDropOffset;
  const uint32_t rb = (uint32_t)ldi * (uint32_t)sizeof(T);
  constexpr uint32_t E = sizeof(T);
  const T kdta = T(0.25) * T(sc->dta), dtr = T(sc->dtr);
  // wave-uniform in a scalar register, so that the current terms below are
  // a scalar branch rather than an exec-masked block issued for every bin
  const bool anycur = __builtin_amdgcn_readfirstlane(sc->anycur) != 0;

  const PointState<T> s = point_stored(d, j);
  const bool prog = o <= s.oc, rot = o <= pload(d.oc_rot, ldi, j);
  const T sin_diss1 = T(d.sin_fac * d.fieldscale1), fs2 = T(d.fieldscale2);
  // neighbour gathers read the frequency-major tables (one plane per
  // table), where 64 neighbours share a few cache lines
  const rsrc_t cpr = row_rsrc(d.cp0, o, ldi), cgr = row_rsrc(d.cg0, o, ldi);
  const T cp0 = bld<T>(cpr, vj);
  T logl2, fkovg;
  if constexpr (sizeof(T) == 4) {
    // FP32 forms both from cp0 = 2 pi f / k: f k / g = 2 pi f^2 / (g cp0),
    // log(l2/z) with l2 = cp0 / (2 f) capped at 20 m
    // (src/umwm_init.F90:1502,1507,1529-1533)
    const float fo = cld(d.f, o), icp = __builtin_amdgcn_rcpf(cp0);
    fkovg = float(kTwoPiD / d.g) * fo * fo * icp;
    const float l2 = 0.5f * cp0 * __builtin_amdgcn_rcpf(fo);
    logl2 = l2 > 20.f ? float(log(20.0 / d.z))
                      : 0.6931471805599453f * __builtin_amdgcn_logf(l2) - float(log(d.z));
  } else {
    logl2 = bld<T>(row_rsrc(d.logl2overz, o, ldi), vj);
    fkovg = bld<T>(row_rsrc(d.fkovg, o, ldi), vj);
  }
  const SinFreq<T> sf = sin_freq(s, logl2, cp0, fkovg, sin_diss1, fs2);
  const rsrc_t pe = freq_rsrc(d.e, o, pm, ldi);    // E^n in, E^{n+1} out
  const rsrc_t ps = freq_rsrc(d.es, o, pm, ldi);   // E*
  // the stress partials' cp0(o, i-1) (src/umwm_stress.F90:219,316), loaded
  // here so that its latency hides behind the direction loop
  const T cp_prev = bld<T>(cpr, (uint32_t)((j == 0) ? d.im : j - 1) * E);
  // direction tables in registers (see k_rates)
  const T* const cthb = d.cth;
  const T* const sthb = d.sth;
  const T* const dir4 = d.dir4;
  const int glen = uniform_div(pm + ng - 1, ng);
  const int plo = SPLIT ? wid * glen : 0, phi = SPLIT ? min(pm, plo + glen) : pm;
  // the moments of the new spectrum and the stress_vector_integral sums
  // over the directions of this frequency
  constexpr bool kSeq = DirSums<T>::kSeq;
  constexpr int NG = DirSums<T>::kGrouped;
  DirSums<T> S;
  S.clear();
  // SPLIT: the groups' sums, [ng][NG][64], and in FP32 the terms of the running
  // sums, [pm][2][64] (advect_lds)
  extern __shared__ double smem[];
  [[maybe_unused]] const int lane = (int)threadIdx.x & 63;
  [[maybe_unused]] T* const terms = reinterpret_cast<T*>(smem + ng * NG * 64);
  int gend = plo + glen;
  auto stress_acc = [&](int p, T v) {
    T ct, st, c2, s2;
    cld4(dir4, p, ct, st, c2, s2);
    const T m = s.cw * ct + s.sw * st > T(0) ? fs2 : T(1);
    T ss = sin_m(sf, sin_y(sf, ct, st), m);
    if (!prog) ss = fmax(ss, T(0));
    S.add(v, v * ss, ct, st, c2, s2);
    if constexpr (SPLIT && kSeq) {
      terms[2 * p * 64 + lane] = v;
      terms[(2 * p + 1) * 64 + lane] = v * ss;
    }
    if (p + 1 == gend) {  // wave-uniform
      S.group();
      gend += glen;
    }
  };
  if (__all(!prog || !valid)) {
    // above the cut-off only the diagnostic tail: e = ef = E_s
    for (int pb = plo; pb < phi; pb += NB) {
      T v[NB];
#pragma unroll
      for (int q = 0; q < NB; ++q) {
        const int p = SPLIT && pb + q >= pm ? 0 : pb + q;
        v[q] = fma(T(2), bld<T>(ps, vj, p * rb), -bld_nt<T>(pe, vj, p * rb));
      }
#pragma unroll
      for (int q = 0; q < NB; ++q) {
        if (SPLIT && pb + q >= phi) break;  // a group of odd length
        bst_stream(pe, vst, v[q], (pb + q) * rb);
        stress_acc(pb + q, v[q]);
      }
    }
  } else {
    const int ie = pload(d.ie, ldi, j), iw = pload(d.iw, ldi, j);
    const int in = pload(d.in_, ldi, j), is = pload(d.is_, ldi, j);
    const uint32_t vie = (uint32_t)ie * E, viw = (uint32_t)iw * E;
    const uint32_t vin = (uint32_t)in * E, vis = (uint32_t)is * E;
    const T dye = pload(d.dye, ldi, j), dyw = pload(d.dyw, ldi, j);
    const T dxn = pload(d.dxn, ldi, j), dxs = pload(d.dxs, ldi, j);
    const T kk = kdta * pload(d.oneovar, ldi, j);
    // ice above fice_uth zeroes the update (src/umwm_advection.F90:93-96)
    const T keep = pload(d.fice, ldq, j) > T(d.fice_uth) ? T(0) : T(1);
    T feup = 0, fedn = 0, fwup = 0, fwdn = 0, fnup = 0, fndn = 0, fsup = 0, fsdn = 0;
    if (anycur) {
      const int iie = pload(d.iie, ldi, j), iiw = pload(d.iiw, ldi, j);
      const int iin = pload(d.iin, ldi, j), iis = pload(d.iis, ldi, j);
      const T ue = s.uc + pload(d.uc, ldq, iie), uw = s.uc + pload(d.uc, ldq, iiw);
      const T vn = s.vc + pload(d.vc, ldq, iin), vs = s.vc + pload(d.vc, ldq, iis);
      feup = (ue + fabs(ue)) * dye;
      fedn = (ue - fabs(ue)) * dye;
      fwup = (uw + fabs(uw)) * dyw;
      fwdn = (uw - fabs(uw)) * dyw;
      fnup = (vn + fabs(vn)) * dxn;
      fndn = (vn - fabs(vn)) * dxn;
      fsup = (vs + fabs(vs)) * dxs;
      fsdn = (vs - fabs(vs)) * dxs;
    }
    // rotation: r(p)/2 = rx sth + ry cth + r0 (zero above the first
    // substep's cut-off), src/umwm_advection.F90:119-156
    T rx = 0, ry = 0, r0 = 0;
    if (rot) {
      const T dcx = bld<T>(cpr, vie) - bld<T>(cpr, viw);
      const T dcy = bld<T>(cpr, vin) - bld<T>(cpr, vis);
      const T dvc = pload(d.vc, ldq, pload(d.iie, ldi, j)) - pload(d.vc, ldq, pload(d.iiw, ldi, j));
      const T duc = pload(d.uc, ldq, pload(d.iin, ldi, j)) - pload(d.uc, ldq, pload(d.iis, ldi, j));
      const T odx = pload(d.oneovdx, ldi, j), ody = pload(d.oneovdy, ldi, j);
      rx = T(0.25) * dcx * odx;
      ry = T(-0.25) * dcy * ody;
      r0 = T(0.25) * (dvc * odx - duc * ody);
    }
    const T cgi = bld<T>(cgr, vj);
    const T Ae = T(2) * (cgi + bld<T>(cgr, vie)) * dye, Aw = T(2) * (cgi + bld<T>(cgr, viw)) * dyw;
    const T As = T(2) * (cgi + bld<T>(cgr, vis)) * dxs, An = T(2) * (cgi + bld<T>(cgr, vin)) * dxn;
    const T ccu = pload(d.ccurv, ldi, j), scu = pload(d.scurv, ldi, j);
    const T kr = dtr * T(d.oneovdth);
    auto rotp = [&](int p) { return fma(rx, cld(sthb, p), fma(ry, cld(cthb, p), r0)); };
    auto load_block = [&](int pb, AdvLoads<T>* L) {
#pragma unroll
      for (int q = 0; q < NB; ++q) {
        // past the last direction (a group of odd length) the first one, the
        // periodic neighbour
        const int p = SPLIT && pb + q >= pm ? 0 : pb + q;
        const uint32_t so = p * rb;
        L[q].eo = bld<T>(ps, vj, so);
        L[q].ee = bld<T>(ps, vie, so);
        L[q].ew = bld<T>(ps, viw, so);
        L[q].en = bld<T>(ps, vin, so);
        L[q].es = bld<T>(ps, vis, so);
        L[q].en0 = bld_nt<T>(pe, vj, so);
      }
    };
    AdvLoads<T> A[NB], B[NB];
    // E* of the directions before and after this wave's (periodic in pm)
    const int pbef = plo > 0 ? plo - 1 : pm - 1, paft = phi < pm ? phi : 0;
    const T efirst = bld<T>(ps, vj, paft * rb);
    T eprev = bld<T>(ps, vj, pbef * rb);
    load_block(plo, A);
    T rprev = rotp(pbef), rcur = rotp(plo);
    for (int pb = plo; pb < phi; pb += NB) {
      const bool more = pb + NB < phi;
      if (more) load_block(pb + NB, B);
#pragma unroll
      for (int q = 0; q < NB; ++q) {
        const int p = pb + q;
        if (SPLIT && p >= phi) break;  // a group of odd length
        const T enext = q + 1 < NB ? A[(q + 1) < NB ? q + 1 : 0].eo : (more ? B[0].eo : efirst);
        const int pn = p + 1 < pm ? p + 1 : 0;
        const T rnext = rotp(pn);
        const T ct = cld(cthb, p), st = cld(sthb, p);
        const T cc = fma(ct, ccu, -st * scu);  // cos(th + curv)
        const T sn = fma(st, ccu, ct * scu);   // sin(th + curv)
        const T e0 = A[q].eo, ee = A[q].ee, ew = A[q].ew, en = A[q].en, es = A[q].es;
        const bool px = cc > T(0), py = sn > T(0);
        T flux = cc * fma(Ae, px ? e0 : ee, -Aw * (px ? ew : e0)) +
                 sn * fma(An, py ? e0 : en, -As * (py ? es : e0));
        if (anycur)
          flux = flux + (feup * e0 + fedn * ee - fwup * ew - fwdn * e0 + fnup * e0 + fndn * en -
                         fsup * es - fsdn * e0);
        const T Es = fma(T(2), e0, -A[q].en0);  // E_s = 2 E* - E^n
        const T rl = rcur + rnext, rr = rcur + rprev;  // edge rotation rates
        const T fr = fma(rl, rl > T(0) ? e0 : enext, -rr * (rr > T(0) ? eprev : e0));
        T v = fma(-kr, fr, fma(-kk, flux, Es));
        v = prog ? v * keep : Es;
        bst_stream(pe, vst, v, p * rb);
        stress_acc(p, v);
        eprev = e0;
        rprev = rcur;
        rcur = rnext;
      }
#pragma unroll
      for (int q = 0; q < NB; ++q) A[q] = B[q];
    }
  }
  S.group();  // the last group, where it is short
  if constexpr (SPLIT) {
    double* const red = smem + lane;
#pragma unroll
    for (int i = 0; i < NG; ++i) red[(wid * NG + i) * 64] = S.t[i];
    __syncthreads();
    if (wid != 0) return;
    for (int q = 1; q < ng; ++q)
#pragma unroll
      for (int i = 0; i < NG; ++i) S.t[i] += red[(q * NG + i) * 64];
    if constexpr (kSeq) {
      S.q[3] = S.q[4] = S.hs = 0;
#pragma unroll 4
      for (int p = 0; p < pm; ++p) {
        T ct, st, c2, s2;
        cld4(dir4, p, ct, st, c2, s2);
        const T wv = terms[(2 * p + 1) * 64 + lane];
        S.q[3] = fma(wv, ct, S.q[3]);
        S.q[4] = fma(wv, st, S.q[4]);
        S.hs += terms[2 * p * 64 + lane];
      }
    }
  }
  if (valid) {
    const T icp = T(1) / cp_prev;
    T tx, ty, hs = 0;
    if constexpr (kSeq) {
      tx = S.q[3];
      ty = S.q[4];
      hs = S.hs * bld<T>(row_rsrc(d.kdk, o, ldi), vj);
    } else {
      tx = T(S.t[3]);
      ty = T(S.t[4]);
    }
    store_mom(d, o, j, S.t[0], S.t[1], S.t[2]);
    const rsrc_t sp = freq_rsrc(d.sp, o, kPartials<T>, ldi);
    bst(sp, vj, tx * icp);
    bst(sp, vj, ty * icp, rb);
    if constexpr (kPartials<T> == 3) bst(sp, vj, hs, 2 * rb);
  }
}

// ---------------------------------------------------------------------
// k_keep: on the substep that reaches dtg (and only when the domain keeps
// them), saves E^n and the incoming ustar, from which stress('ocn')
// rebuilds that substep's ssin, sds and snl at output time.  Launched
// between k_integrate (which reads E^n) and k_advect (which overwrites it).
// ---------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(64) void k_keep(const DomainDev<T>* __restrict__ doms,
                                             const BlockTask* __restrict__ tasks) {
  const BlockTask tk = tasks[blockIdx.x];
  const DomainDev<T>& d = doms[tk.dom];
  if (!d.sc->active || !d.sc->last || !d.e_keep) return;
  const int j = tk.i0 + (int)threadIdx.x;
  if (j >= d.im) return;
  const size_t ldi = d.ldi, rows = (size_t)d.om * d.pm;
  for (size_t r = 0; r < rows; ++r) d.e_keep[r * ldi + j] = d.e[r * ldi + j];
  d.ustar_keep[j] = d.ustar[j];
}

// ---------------------------------------------------------------------
// k_stress: frequency sums + stress('atm') chain per point
// ---------------------------------------------------------------------
// The frequency sums run in one wave while another forms the relative wind and
// the skin friction velocity of the same 64 points, two chains of about the
// same length; the sums' loads go out eight frequencies at a time.  One wave
// after the other had taken 20 us at 169 points, where nothing hides the
// latency, and 24 at 2,809; now 8.3 and 10.5.
template <typename T>
__global__ __launch_bounds__(128) void k_stress(const DomainDev<T>* __restrict__ doms,
                                                const BlockTask* __restrict__ tasks,
                                                int rates_split) {
  const BlockTask tk = tasks[blockIdx.x];
  const DomainDev<T>& d = doms[tk.dom];
  if (!d.sc->active) return;
  const int lane = (int)threadIdx.x & 63;
  const int j0 = tk.i0 + lane, j = min(j0, d.im - 1);  // lanes past the end repeat the last point
  if (tk.local == 0 && threadIdx.x == 0) d.sc->done = 0;
  const size_t ldi = d.ldi, ldq = d.ldq;
  const int om = d.om;
  constexpr uint32_t E = sizeof(T);
  __shared__ SkinWind skin[64];
  T w = pload(d.wspd, ldq, j);
  w = w > T(1e-2) ? w : T(1e-2);
  if (wave_id() == 1)
    skin[lane] = skin_wind(w, pload(d.wdir, ldq, j), pload(d.uc, ldq, j), pload(d.vc, ldq, j),
                           pload(d.us1, ldi, j), pload(d.vs1, ldi, j), d.z, d.nu_air, d.kappa);
  StressIn si;
  double hs = 0;
  if (wave_id() == 0) {
    const int oc = pload(d.oc, ldi, j);
    si.sx = si.sy = si.dx = si.dy = 0;
#pragma unroll 8
    for (int o = 0; o < om; ++o) {
      const double kdk = bld<T>(row_rsrc(d.kdk, o, ldi), (uint32_t)j * E);
      const rsrc_t sp = freq_rsrc(d.sp, o, kPartials<T>, ldi);
      const uint32_t vj = (uint32_t)j * E, rb = (uint32_t)ldi * E;
      const double tx = bld<T>(sp, vj), ty = bld<T>(sp, vj, rb);
      double hso;
      if constexpr (kPartials<T> == 3)
        hso = bld<T>(sp, vj, 2 * rb);
      else
        hso = bld<double>(row_rsrc(d.mom, (size_t)o, 3 * ldi), vj) * kdk;
      si.sx += tx * kdk;
      si.sy += ty * kdk;
      if (o >= oc) {
        si.dx += tx * kdk;
        si.dy += ty * kdk;
      }
      if (o == om - 1) {
        si.tomx = tx;
        si.tomy = ty;
      }
      hs += hso;
    }
    si.wspd = w;
    si.rhoa = pload(d.rhoa, ldq, j);
    si.rhow = pload(d.rhow, ldq, j);
    si.kom = bld<T>(row_rsrc(d.k, om - 1, ldi), (uint32_t)j * E);
  }
  __syncthreads();
  if (wave_id() == 1 || j0 >= d.im) return;
  store_stress(d, j, stress_atm_point(si, skin[lane], d.dthg));
  pstore(d.hs_ice, ldi, j, 4 * sqrt(hs * d.dth));
  if (rates_split) {  // k_rates' maximum over a point's workgroups
    d.pts[j] = d.explim / __longlong_as_double((long long)d.rkey[j]);
    d.rkey[j] = 0;
  }
}

// Launch shape of the fused kernels: direction groups and frequency chunks of
// the two sweeps, waves per workgroup, and whether k_advect is split.
struct Shape {
  int D1, ng1, c1, w1;
  int D2, ng2, c2, w2;
  bool paired;  // k_rates pairs opposite directions where it can
  bool split;
  bool spec;    // k_integrate runs ahead of k_rates where the domains expect it
};

template <typename T, int D, bool SUR, bool STORE>
void launch_rates(const DomainDev<T>* doms, const BlockTask* tasks, int ntasks, int pm, int first,
                  int rotation, const Shape& h, hipStream_t s) {
  // choose_shape's waves of 2 and 4 have a k_integrate as narrow
  if constexpr (sizeof(T) == 8 || D > 4 || !STORE) {
    const int slots = h.ng1 * h.c1;
    const dim3 grid(ntasks, (slots + h.w1 - 1) / h.w1), block(64 * h.w1);
    // the cross-wave maximum, and the surrogate's four cross-wave sums
    const size_t sh = (size_t)(SUR ? 4 : 1) * h.w1 * 64 * sizeof(double);
    // a launch whose waves all hold D directions takes a variant with no
    // per-slot masks
    if (h.ng1 * D == pm) {
      if constexpr (D % 2 == 0 && D > 4) {  // 2 and 4 are unpaired
        if (h.paired) {
          hipLaunchKernelGGL((k_rates<T, D, true, true, SUR, STORE>), grid, block, sh, s, doms, tasks,
                             first, rotation, h.ng1, h.c1);
          return;
        }
      }
      if constexpr (!(SUR && D % 2 == 0))
        hipLaunchKernelGGL((k_rates<T, D, true, false, SUR, STORE>), grid, block, sh, s, doms, tasks,
                           first, rotation, h.ng1, h.c1);
    } else if constexpr (D > 4) {
      hipLaunchKernelGGL((k_rates<T, D, false, false, SUR, STORE>), grid, block, sh, s, doms, tasks,
                         first, rotation, h.ng1, h.c1);
    }
  }
}

template <typename T, int D, bool SUR>
void launch_integrate(const DomainDev<T>* doms, const BlockTask* tasks, int ntasks, int pm,
                      const Shape& h, hipStream_t s) {
  const int slots = h.ng2 * h.c2;
  const dim3 grid(ntasks, (slots + h.w2 - 1) / h.w2), block(64 * h.w2);
  if (h.ng2 * D == pm)
    hipLaunchKernelGGL((k_integrate<T, D, true, SUR, false>), grid, block, 0, s, doms, tasks, h.ng2, h.c2);
  else if constexpr (D != 2 && D != 4)
    hipLaunchKernelGGL((k_integrate<T, D, false, SUR, false>), grid, block, 0, s, doms, tasks, h.ng2, h.c2);
}

template <typename T>
void launch_spec(const DomainDev<T>* doms, const BlockTask* tasks, int ntasks, int pm,
                 const Shape& h, hipStream_t s) {
  const dim3 grid(ntasks), block(64 * h.w2);
  if constexpr (stored_prefix<T, false>(9))
    hipLaunchKernelGGL((k_prefix<T>), grid, dim3(64), 0, s, doms, tasks);
  if (h.ng2 * h.D2 != pm) {  // FP32 waves of nine, see choose_shape
    if constexpr (sizeof(T) == 4)
      hipLaunchKernelGGL((k_integrate<T, 9, false, false, true>), grid, block, 0, s, doms, tasks, h.ng2, 1);
  } else if (h.D2 == 9)
    hipLaunchKernelGGL((k_integrate<T, 9, true, false, true>), grid, block, 0, s, doms, tasks, h.ng2, 1);
  else if (h.D2 == 6)
    hipLaunchKernelGGL((k_integrate<T, 6, true, false, true>), grid, block, 0, s, doms, tasks, h.ng2, 1);
  else
    hipLaunchKernelGGL((k_integrate<T, 4, true, false, true>), grid, block, 0, s, doms, tasks, h.ng2, 1);
}

// LDS of k_advect's split: at most 48 KB (FP32, 72 directions)
template <typename T>
size_t advect_lds(int ng, int pm) {
  size_t n = (size_t)ng * DirSums<T>::kGrouped * 64 * sizeof(double);
  if (DirSums<T>::kSeq) n += (size_t)pm * 2 * 64 * sizeof(T);
  return n;
}

template <typename T, bool SUR>
int launch_kernels(const DomainDev<T>* doms, const BlockTask* tasks, int ntasks, int omax, int pm,
                   int first, int rotation, const Shape& h, int nb, bool keep, hipStream_t s,
                   hipEvent_t* ev) {
  if (ev) (void)hipEventRecord(ev[0], s);
  if constexpr (!SUR) {
    // a timed substep keeps the kernels apart
    if (h.spec && !first && !rotation && !ev) launch_spec<T>(doms, tasks, ntasks, pm, h, s);
  }
#define UMWM_RATES(D_)                                                                       \
  case D_:                                                                                   \
    if (stored_prefix<T, SUR>(h.D2))                                                         \
      launch_rates<T, D_, SUR, true>(doms, tasks, ntasks, pm, first, rotation, h, s);        \
    else if constexpr (!stored_prefix<T, SUR>(0))                                            \
      launch_rates<T, D_, SUR, false>(doms, tasks, ntasks, pm, first, rotation, h, s);       \
    break;
  switch (h.D1) {
    UMWM_RATES(6)
    UMWM_RATES(9)
    UMWM_RATES(18)
    UMWM_RATES(36)
    default:
      if constexpr (!SUR) {
        switch (h.D1) {
          UMWM_RATES(2)
          UMWM_RATES(4)
          default: return fail(UMWM_ERR_ARGUMENT, "unsupported rates tile D");
        }
        break;
      }
      return fail(UMWM_ERR_ARGUMENT, "unsupported rates tile D");
  }
#undef UMWM_RATES
  if (ev) (void)hipEventRecord(ev[1], s);
#define UMWM_INTEGRATE(D_)                                                           \
  case D_: launch_integrate<T, D_, SUR>(doms, tasks, ntasks, pm, h, s); break;
  switch (h.D2) {
    UMWM_INTEGRATE(3)
    UMWM_INTEGRATE(6)
    UMWM_INTEGRATE(9)
    UMWM_INTEGRATE(12)
    UMWM_INTEGRATE(18)
    default:
      if constexpr (!SUR) {
        switch (h.D2) {
          UMWM_INTEGRATE(2)
          UMWM_INTEGRATE(4)
          default: return fail(UMWM_ERR_ARGUMENT, "unsupported integrate tile D");
        }
        break;
      }
      return fail(UMWM_ERR_ARGUMENT, "unsupported integrate tile D");
  }
#undef UMWM_INTEGRATE
  if (keep) hipLaunchKernelGGL((k_keep<T>), dim3(ntasks), dim3(64), 0, s, doms, tasks);
  if (ev) (void)hipEventRecord(ev[2], s);
  const int ng = dir_groups(pm);
  if (h.split && ng <= 8) {
    const dim3 ga(ntasks, omax), block(64 * ng);
    const size_t sh = advect_lds<T>(ng, pm);
    if (nb == 4)
      hipLaunchKernelGGL((k_advect<T, 4, true>), ga, block, sh, s, doms, tasks, ng);
    else
      hipLaunchKernelGGL((k_advect<T, 2, true>), ga, block, sh, s, doms, tasks, ng);
  } else {
    // one wave per (64 points, frequency), FW frequencies per workgroup (2
    // measured 1-2 % faster than 4 or 8 on 720x360)
    const int fw = 2;
    const dim3 ga(ntasks, (omax + fw - 1) / fw);
    if (nb == 4)
      hipLaunchKernelGGL((k_advect<T, 4, false>), ga, dim3(64 * fw), 0, s, doms, tasks, ng);
    else
      hipLaunchKernelGGL((k_advect<T, 2, false>), ga, dim3(64 * fw), 0, s, doms, tasks, ng);
  }
  if (ev) (void)hipEventRecord(ev[3], s);
  hipLaunchKernelGGL((k_stress<T>), dim3(ntasks), dim3(128), 0, s, doms, tasks,
                     h.ng1 * h.c1 > h.w1 ? 1 : 0);
  if (ev) (void)hipEventRecord(ev[4], s);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(UMWM_ERR_HIP, std::string("fused launch: ") + hipGetErrorString(e));
  return 0;
}

}  // namespace

bool tile_supported(int D) { return D == 3 || D == 6 || D == 9 || D == 12 || D == 18 || D == 36; }

namespace {

// Waves per workgroup for `slots` waves of a point block: the largest divisor
// up to 8, or 8 (the last workgroup then holds idle waves).
int waves_for(int slots) {
  for (int w = 8; w >= 4; --w)
    if (slots % w == 0) return w;
  return std::min(slots, 8);
}

// Launch shape of default tiles.  The sweeps need about kSweepWaves waves to
// fill the GPU; a point block offers pm / D of them, and a frequency chunk
// costs a prefix sum over the frequencies below it (both sweeps) and the
// dissipation of two more (k_integrate), so small grids are split over
// frequency as far as it takes, down to four frequencies a chunk, and then
// over pairs of directions.  37 x 36 bins, k_rates + k_integrate in us, before
// (one chunk of nine directions) and as chosen here:
//   169 points    FP64 267 -> 38   FP32 102 -> 33
//   2,809 points  FP64 284 -> 75   FP32 104 -> 41
//   11,449 points FP64 303 -> 188  FP32 108 -> 78
// D divides pm: masked slots cost as much as full ones (pm = 48 at 13,924
// points, D = 6 against 9: FP64 633 -> 310 us, FP32 125 -> 98).  Where only
// four would, an FP32 grid whose waves of nine fill the GPU at the four a SIMD
// holds takes nine, the last wave with idle slots: a frequency's tables weigh
// more on a narrow wave than those slots do.  Substeps of 79,921 points in us,
// D = 4 -> 9: 37x28 590 -> 558, 37x40 916 -> 879, 37x44 900 -> 911, 37x56
// 1,110 -> 1,050, 37x68 1,317 -> 1,160; 179,813 points x 37x28 1,308 -> 1,231.
// At 38,936 points the count of waves decides (37x28 339 and 312, 37x44 472 and
// 513, 37x64 601 and 626, 37x68 680 and 643).  FP64, whose directions weigh
// more, keeps four: 867 us against 914 at 38,936 points x 37x28, 1,557 against
// 1,549 at 79,921.  On FP32 grids as large k_rates alone takes eighteen where
// they divide pm: substeps whose sources limit them 1,433 -> 1,399 us at
// 179,813 points x 37x36 (k_rates 283 -> 250), 1,751 -> 1,746 at 93,870 x 49x72;
// no gain at 38,844 (55 -> 58 of 333).
// k_advect's split pays while its waves (one per frequency and point block)
// leave the GPU short of work: 2,809 points FP64 29.7 -> 25.7, FP32 25.6 ->
// 19.2 us; 11,449 points 84.9 -> 92.9 and 39.4 -> 49.1 us.
constexpr int kSweepWaves = 1536;
constexpr int kAdvectWaves = 4096;
constexpr int kFullWaves = 4096;

Shape choose_shape(const Tile& t, int ntasks, int omax, bool sur, bool fp32) {
  Shape h{t.D1, t.W1, 1, t.W1, t.D2, t.W2, 1, t.W2, true, false, false};
  const int pm = t.pmax;
  // the network's checks need all of a point's waves in one workgroup; wide
  // spectra keep the tile's own shape.  A given tile runs its sources ahead on
  // the grids that default tiles do (one chunk): 178,369 points x 37x36 with
  // (18, 2, 9, 4), FP32 1.27 -> 1.07 and FP64 3.26 -> 2.62 ms a substep.
  if (t.chosen || sur || pm > 72) {
    h.spec = !sur && (t.D2 == 6 || t.D2 == 9) && t.W2 * t.D2 == pm &&
             3 * ntasks * t.W2 > 2 * kSweepWaves;
    return h;
  }
  auto chunks = [&](int D) {
    const int waves = ntasks * (pm / D);
    return std::max(1, std::min((kSweepWaves + waves / 2) / waves, omax / 4));
  };
  int D = pm % 9 == 0 ? 9 : pm % 6 == 0 ? 6 : 4;
  if (ntasks * (pm / D) * chunks(D) < kSweepWaves / 2) D = 2;
  if (D == 4 && fp32 && ntasks * ((pm + 8) / 9) >= kFullWaves) D = 9;
  h.D1 = h.D2 = D;
  h.ng1 = h.ng2 = (pm + D - 1) / D;
  h.c1 = h.c2 = chunks(D);
  h.w1 = h.w2 = waves_for(h.ng1 * h.c1);
  h.paired = false;  // one order of operations whatever D
  if (fp32 && pm % 18 == 0 && h.c1 == 1 && ntasks * (pm / 9) >= kFullWaves) {
    h.D1 = 18;
    h.ng1 = h.w1 = pm / 18;
  }
  h.split = ntasks * omax < kAdvectWaves;
  h.spec = h.D2 >= 4 && h.c2 == 1 && h.w2 == h.ng2;  // launch_spec has D = 4, 6 and 9
  return h;
}

}  // namespace

template <typename T>
int launch_moments(const DomainDev<T>* doms, const BlockTask* tasks, int ntasks, int omax,
                   hipStream_t s) {
  if (ntasks <= 0) return 0;
  hipLaunchKernelGGL((k_moments<T>), dim3(ntasks, omax), dim3(64), 0, s, doms, tasks);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(UMWM_ERR_HIP, std::string("k_moments: ") + hipGetErrorString(e));
  return 0;
}
template int launch_moments<float>(const DomainDev<float>*, const BlockTask*, int, int, hipStream_t);
template int launch_moments<double>(const DomainDev<double>*, const BlockTask*, int, int,
                                    hipStream_t);

template <typename T>
int launch_fused(const DomainDev<T>* doms, const BlockTask* tasks, int ntasks, int omax,
                 int first, int rotation, Tile tile, bool keep, hipStream_t s, hipEvent_t* ev,
                 bool sur) {
  if (ntasks <= 0) return 0;
  if (tile.W1 < 1 || tile.W1 > 8 || tile.W2 < 1 || tile.W2 > 8)
    return fail(UMWM_ERR_ARGUMENT, "tile W must be 1..8");
  if (sur) {
    // the surrogate variants hold the network's dm^2 of this and the next
    // frequency beside the spectrum: more waves of fewer directions each,
    // the same W D, keep them off scratch (k_rates above 18 directions and
    // k_integrate above 9 spill)
    while (tile.D1 > 18 && tile.D1 % 2 == 0 && tile.W1 * 2 <= 8 && tile_supported(tile.D1 / 2)) {
      tile.D1 /= 2;
      tile.W1 *= 2;
    }
    while (tile.D2 > 9 && tile.D2 % 2 == 0 && tile.W2 * 2 <= 8 && tile_supported(tile.D2 / 2)) {
      tile.D2 /= 2;
      tile.W2 *= 2;
    }
  }
  const Shape h = choose_shape(tile, ntasks, omax, sur, sizeof(T) == 4);
  if constexpr (std::is_same_v<T, float>) {
    if (sur)
      return launch_kernels<T, true>(doms, tasks, ntasks, omax, tile.pmax, first, rotation, h,
                                     tile.NB, keep, s, ev);
  } else if (sur) {
    return fail(UMWM_ERR_ARGUMENT, "the surrogate serves the FP32 path only");
  }
  return launch_kernels<T, false>(doms, tasks, ntasks, omax, tile.pmax, first, rotation, h, tile.NB,
                                  keep, s, ev);
}

template int launch_fused<float>(const DomainDev<float>*, const BlockTask*, int, int, int, int,
                                 Tile, bool, hipStream_t, hipEvent_t*, bool);
template int launch_fused<double>(const DomainDev<double>*, const BlockTask*, int, int, int, int,
                                  Tile, bool, hipStream_t, hipEvent_t*, bool);

}  // namespace umwm
