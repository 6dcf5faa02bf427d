// Kirchhoff depth migration operators on MI355X: the image- and angle-domain
// kernels of src/migration/migration.cu:398-756 and the wavelet
// convolutions of :173-261.
//
// The reference launches one kernel per trace (source, receiver pair), one
// thread per padded node, each evaluating the node's weight from 9-point
// finite differences of both traveltime tables and adding into the image
// (adjoint) or the trace (forward) with atomicAdd.  Here:
//   - the per-table part of the weight is evaluated once per table
//     (k_kdm_prep): the reference's first and second derivatives, Hessian
//     determinant, gradient norm, incidence angle and cosine, folded into
//     one amplitude per node (the Hessian, obliquity and spreading factors of
//     the weight are products of a source and a receiver factor) and the
//     cosine and sine of the half angle (the reflection-angle factor's
//     cosine of the mean angle by the addition formula); a trace's weight is
//     then four products, the angle factor and the aperture taper (4 words
//     per node and table: T, amplitude, half-angle cosine and sine; 3 more,
//     the gradient, for the angle domain's bin);
//   - the same pass keeps each table's minimum traveltime over every 64
//     consecutive image points; rounded addition and division being
//     monotone, a wave whose chunk minima give a time index >= nt holds no
//     node that reaches the trace and passes over it with two scalar loads
//     (with the reference's recording lengths most node-trace pairs end
//     there); the other quantities are loaded only for nodes that reach it;
//   - adjoint: one thread per image point walks the traces grouped in source
//     blocks (four sources' quantities in registers, each receiver's loaded
//     once for up to four traces), the blocks spread over up to 16 waves per
//     64 points; image domain: each wave's sum stays in a register and the
//     partial images are added in a fixed order, deterministic, no atomics;
//     angle domain: adds into the (depth, angle, CMP) bins with atomics, as
//     the reference (their order varies);
//   - forward: short records: one workgroup (sixteen waves) per trace
//     accumulates the trace in an LDS histogram of its nt samples (FP64 LDS
//     atomics) and adds it to the trace once; the tables' minima over 64 chunks
//     let it pass over 4096 image points with one test.  Others: one workgroup
//     per image tile and source block, each trace's samples in an LDS window;
//   - convolution: the FFT product of the reference is a linear
//     (cross-)correlation with the wavelet, summed directly in double, eight
//     samples per thread from a trace staged in LDS.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <limits>
#include <string>
#include <vector>

#include "../../include/seisfat2d_kdm.h"
#include "eik_handle.h"
#include "kdm_window.h"

namespace seisfat {

constexpr float KDM_EPS = 1e-6f;  // EPS of src/migration/migration.cuh:7
// per-table quantities: T, amplitude, cos and sin of half the angle; the angle
// domain's bin also needs dT/dx, dT/dz, |grad T| + EPS
constexpr int kq_words(bool angle) { return angle ? 7 : 4; }

struct KdmK {
  int nz, nx, nzz, npts, nt, nang;
  int nchunk;     // 64-node chunks of the image points (one wave each)
  int nsup;       // super-chunks of 64 chunks (4096 image points)
  float thr;      // least x with RN(x / dt) >= nt: a traveltime sum x >= thr has time index >= nt
  float zh_dt, zl_dt;  // two-word reciprocal of dt (fdiv)
  int fastdiv_dt;      // fdiv(x, zh_dt, zl_dt) == RN(x / dt) for every 2^-100 <= x < 2^100 (checked exhaustively)
  int taper_rdiv;      // (x - cmp) / sig_e needs no operand rescaling at any node and trace (kdm_weight)
  float dx, dz, dt;
  // k_kdm_prep's constant divisors and their reciprocals RN(1 / b)
  float dz2, dx2, dxz4, r_dz, r_dx, r_dz2, r_dx2, r_dxz4;
  int prep_rdiv;        // dz and dx lie in [2^-20, 2^20]
  float da_m, r_da;     // da = da_m 2^da_e, da_m in [1, 2), and RN(1 / da_m)
  int da_e;
  unsigned nz_recip;    // floor(2^32 / nz) (nz > 1)
  float tan_ap;  // tanf(aperture in radians), the reference's sigma / z
  float scale;   // 1 / (2 pi) as the reference rounds it
};

// float -> int rounding down, as the GPU's conversion does it (NaN -> 0,
// saturating): the reference's __float2int_rd.
__device__ __forceinline__ int f2i_rd(float v) {
  if (v != v) return 0;
  if (v >= 2147483648.0f) return 2147483647;
  if (v < -2147483648.0f) return (-2147483647 - 1);
  return (int)floorf(v);
}

// Refined reciprocal of b (the r of rdiv).
__device__ __forceinline__ float recip_refined(float b) {
  const float r0 = __builtin_amdgcn_rcpf(b);
  return __builtin_fmaf(__builtin_fmaf(-b, r0, 1.0f), r0, r0);
}

// The per-table quantities of padded table T at interior node (i, j) (padded
// coordinates).  The reference's per-table expressions (float, its order):
// the derivatives, norm = |grad T| + EPS, det = |det H| + EPS, the angle
// theta = acos(clamp(-uz)) and cos = |-uz|, rs = max(T / S, EPS).  Its
// weight's Hessian, obliquity and spreading factors,
//   sqrt(det_s det_r) S / (norm_s norm_r) * sqrt(max(0, cos_s) max(0, cos_r))
//   / sqrt(rs_s rs_r),
// are S times the product of one amplitude per table,
//   amp = sqrt(det max(0, cos)) / (norm sqrt(rs))   (in double, rounded once),
// and its angle factor's cos((theta_s + theta_r) / 2) is
// ch_s ch_r - sh_s sh_r with ch, sh = cos, sin(theta / 2).  The weight a
// trace forms from them differs from the reference's order of roundings by a
// few ulp.
//
// One wave per chunk of 64 consecutive image points (p = i + j*nz) of a table,
// which also keeps the chunk's minimum traveltime (tmin).  For every node of a
// chunk, RN(RN(Ts + Tr) / dt) >= RN(RN(min_s + min_r) / dt) (rounded addition
// and division are monotone), so a chunk whose minima give a time index >= nt
// holds no node that reaches the trace.  The minimum propagates NaN: a chunk
// holding a NaN traveltime is never passed over (its node's time index would
// be 0).
//
// The kernel is bound by instruction issue, so the usual node (prep_rdiv, the
// nine traveltimes of magnitude in [2^-30, 2^40)) takes a short path: every
// difference of such floats is 0 or in [2^-54, 2^43), so the divisions by the
// grid's constants and by the gradient's norm are IEEE division by rdiv and
// the roots need no rescaling; the amplitude is one reciprocal square root,
//   amp = num rsqrt(num den), num = det |cos| s', den = norm^2 c'
// (c' / s' = max(c / S, EPS)), v_rsq_f64 with one Newton step (relative error
// near 2^-46), rounded once to float.  A wave with any other node (zero, tiny, huge,
// infinite or NaN traveltimes) takes the general path.  The row of a lane
// comes from its wave's first point (one scalar division by multiplication).
// 1001 x 1001, 252 tables, image domain: 1.85 ms; 3.15 ms with IEEE division,
// two FP64 roots and a division per node and seven words written in either
// domain.
__device__ __forceinline__ float min_nan(float a, float b) { return (a != a || b != b) ? __builtin_nanf("") : fminf(a, b); }
__device__ __forceinline__ float min3f(float a, float b, float c) { return fminf(fminf(a, b), c); }

template <bool ANGLE>
__global__ __launch_bounds__(256) void k_kdm_prep(const float* __restrict__ tables, int ntab,
                                                  const float* __restrict__ S, KdmK K, float* __restrict__ q,
                                                  float* __restrict__ tmin) {
  constexpr int KQ = kq_words(ANGLE);
  const int lane = threadIdx.x & 63;
  const size_t tsize = (size_t)K.nzz * (K.nx + 6);
  const int c = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)));
  if (c >= K.nchunk) return;  // whole wave past the end
  // row and column of the chunk's first point: umulhi(p, floor(2^32 / nz)) is
  // p / nz or at most two less (p < 2^30)
  const int pc = c * 64;
  int jc = K.nz > 1 ? (int)__umulhi((unsigned)pc, K.nz_recip) : pc, ic = pc - jc * K.nz;
  while (ic >= K.nz) ic -= K.nz, ++jc;
  const int p = pc + lane;
  int i = ic + lane, j = jc;
  while (i >= K.nz) i -= K.nz, ++j;
  const bool live = p < K.npts;
  if (!live) i = K.nz - 1, j = K.nx - 1;  // lanes past the end load in bounds and store nothing
  i += 3;
  j += 3;
  const int nzz = K.nzz, o0 = i + j * nzz;
  const float s = S[o0];
  for (int tab = blockIdx.y; tab < ntab; tab += gridDim.y) {
    const float* __restrict__ T = tables + tab * tsize + o0;
    const float t0 = T[0];
    const float up = T[-1], dn = T[1], lf = T[-nzz], rt = T[nzz];
    const float dr = T[1 + nzz], ur = T[-1 + nzz], dl = T[1 - nzz], ul = T[-1 - nzz];
    const float nzd = 0.5f * (dn - up), nxd = 0.5f * (rt - lf);
    const float nzzd = dn - 2.0f * t0 + up, nxxd = rt - 2.0f * t0 + lf, nxzd = dr - ur - dl + ul;
    // the nine magnitudes' least (their greatest is bounded through norm and det; a NaN fails those)
    const float least = min3f(min3f(fabsf(t0), fabsf(up), fabsf(dn)), min3f(fabsf(lf), fabsf(rt), fabsf(dr)),
                              min3f(fabsf(ur), fabsf(dl), fabsf(ul)));
    float d_z = rdiv(nzd, K.dz, K.r_dz), d_x = rdiv(nxd, K.dx, K.r_dx);
    float norm = rsqrt_rn(d_x * d_x + d_z * d_z) + KDM_EPS;
    float det = fabsf(rdiv(nxxd, K.dx2, K.r_dx2) * rdiv(nzzd, K.dz2, K.r_dz2) -
                      [](float a) { return a * a; }(rdiv(nxzd, K.dxz4, K.r_dxz4))) + KDM_EPS;
    float dot, amp, ch, sh;
    // (huge, infinite and NaN values show in norm or det)
    const bool usual = K.prep_rdiv && least >= 0x1p-30f && fabsf(t0) < 0x1p40f && norm < 0x1p40f && det < 0x1p80f;
    if (__all(usual)) {
      dot = -rdiv(d_z, norm, recip_refined(norm));  // unit gradient . (0, -1), the surface normal
      const float cth = fminf(1.0f, fmaxf(-1.0f, dot));
      const bool far = t0 >= KDM_EPS * s;
      const double num = (double)det * (double)fabsf(dot) * (double)(far ? s : 1.0f);
      const double den = (double)norm * (double)norm * (double)(far ? t0 : KDM_EPS);
      const double x = num * den;
      const double y = __builtin_amdgcn_rsq(x);
      const double y1 = __builtin_fma(0.5 * y, __builtin_fma(-x * y, y, 1.0), y);
      amp = num > 0.0 ? (float)(num * y1) : 0.0f;
      ch = rsqrt_rn(0.5f * (1.0f + cth));
      sh = rsqrt_rn(0.5f * (1.0f - cth));
    } else {
      d_z = nzd / K.dz;
      d_x = nxd / K.dx;
      const float d2z = nzzd / K.dz2, d2x = nxxd / K.dx2, dxz = nxzd / K.dxz4;
      norm = sqrtf(d_x * d_x + d_z * d_z) + KDM_EPS;
      det = fabsf(d2x * d2z - dxz * dxz) + KDM_EPS;
      const float ux = d_x / norm, uz = d_z / norm;
      dot = ux * 0.0f + uz * -1.0f;
      const float cth = fminf(1.0f, fmaxf(-1.0f, dot));  // cos(theta), theta = acos(cth) in the reference
      const float rs = fmaxf(t0 / s, KDM_EPS);
      amp = (float)(sqrt((double)det * (double)fmaxf(0.0f, fabsf(dot))) / ((double)norm * sqrt((double)rs)));
      ch = sqrtf(0.5f * (1.0f + cth));
      sh = sqrtf(0.5f * (1.0f - cth));
    }
    if (live) {
      float* __restrict__ o = q + (size_t)tab * KQ * K.npts + p;
      o[0] = t0;
      o[(size_t)1 * K.npts] = amp;
      // cos and sin of theta / 2 by the half-angle identities (1 +- cth exact
      // where it matters, by Sterbenz): within 5e-8 of those of acos(cth), closer
      // than the cosine and sine of the float acosf(cth)
      o[(size_t)2 * K.npts] = ch;
      o[(size_t)3 * K.npts] = sh;
      if (ANGLE) {
        o[(size_t)4 * K.npts] = d_x;
        o[(size_t)5 * K.npts] = d_z;
        o[(size_t)6 * K.npts] = norm;
      }
    }
    float tv = live ? t0 : __builtin_inff();
    for (int off = 32; off >= 1; off >>= 1) tv = min_nan(tv, __shfl_xor(tv, off, 64));
    if (lane == 0) tmin[(size_t)tab * K.nchunk + c] = tv;
  }
}

// Per table, the minimum of the chunk minima over each super-chunk of 64
// chunks (NaN-propagating): one wave per super-chunk.  The super-chunk minima
// bound every chunk's from below, so a super-chunk whose minima give a time
// index >= nt holds no chunk that reaches the trace.
__global__ __launch_bounds__(256) void k_kdm_tmin2(const float* __restrict__ tmin, int ntab, KdmK K,
                                                   float* __restrict__ tmin2) {
  const int lane = threadIdx.x & 63;
  const size_t nw = (size_t)ntab * K.nsup;
  const size_t wstride = (size_t)gridDim.x * (blockDim.x >> 6);
  for (size_t w = (size_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6); w < nw; w += wstride) {
    const int tab = (int)(w / K.nsup);
    const int c = (int)(w - (size_t)tab * K.nsup) * 64 + lane;
    float v = c < K.nchunk ? tmin[(size_t)tab * K.nchunk + c] : __builtin_inff();
    for (int off = 32; off >= 1; off >>= 1) v = min_nan(v, __shfl_xor(v, off, 64));
    if (lane == 0) tmin2[w] = v;
  }
}

// Whether a receiver table holds a negative value or a NaN at an image point
// (its least super-chunk minimum, NaN-propagating): one wave per table writes
// neg[r] and keeps *nneg the number of such tables.  While it is 0 a source may
// be passed over on its own minimum.  Counted as tables are set, so that it
// holds for whatever runs after them, on any stream and in a replayed graph
// (reading the chunk minima back took 1 ms on 201 tables of 1001 x 1001).
__global__ __launch_bounds__(64) void k_kdm_rec_neg(const float* __restrict__ tmin2, KdmK K, int* __restrict__ neg,
                                                    int* __restrict__ nneg) {
  const int lane = threadIdx.x, r = blockIdx.x;
  bool ok = true;
  for (int k = lane; k < K.nsup; k += 64) ok &= tmin2[(size_t)r * K.nsup + k] >= 0.0f;
  const int now = __all(ok) ? 0 : 1, before = neg[r];
  if (lane == 0 && now != before) {
    neg[r] = now;
    atomicAdd(nneg, now - before);
  }
}

struct Q7 {
  float t, amp, ch, sh, dx, dz, norm;
};
// The weight's quantities after T (loaded once the node is known to reach the
// trace).
template <int KQ>
__device__ __forceinline__ void q_amp(const float* __restrict__ q, int tab, int p, int npts, Q7& o) {
  const float* __restrict__ b = q + (size_t)tab * KQ * npts + p;
  o.amp = b[(size_t)npts];
  o.ch = b[(size_t)2 * npts];
  o.sh = b[(size_t)3 * npts];
}
// The gradient, for the angle domain's bin.
template <int KQ>
__device__ __forceinline__ void q_dir(const float* __restrict__ q, int tab, int p, int npts, Q7& o) {
  const float* __restrict__ b = q + (size_t)tab * KQ * npts + p;
  o.dx = b[(size_t)4 * npts];
  o.dz = b[(size_t)5 * npts];
  o.norm = b[(size_t)6 * npts];
}

// The index where every sum lies in [2^-100, 2^100) and the two-instruction
// division by dt is proven.
__device__ __forceinline__ int t_index_mid(float xs, const KdmK& K) { return (int)fdiv(xs, K.zh_dt, K.zl_dt); }

// Time index of a node for a trace with traveltime sum xs, as far as the
// kernels use it: the reference's tId = f2i_rd(RN(xs / dt)) where that lies in
// [0, nt) or xs is NaN (0), -1 or any value from nt to INT_MAX otherwise (so
// nothing may be added to an index that is not known to be below nt).  When
// every lane's sum lies in [2^-100, 2^100) (traveltimes are positive), RN(xs /
// dt) comes from the two-instruction known-divisor division the exhaustive
// check proved exact there, and the conversion truncates and saturates: the
// index is then >= nt exactly when xs >= thr.  Otherwise, for the whole wave,
// IEEE division where that division is not proven, and thr, NaN and the sign
// decided explicitly.
__device__ __forceinline__ int t_index(float xs, const KdmK& K) {
  const bool mid = __float_as_uint(xs) - 0x0d800000u < 0x64000000u;  // 2^-100 <= xs < 2^100
  const uint64_t all_mid = __builtin_amdgcn_ballot_w64(mid);
  // a positive finite quotient: truncation is the floor
  if (K.fastdiv_dt && all_mid == __builtin_amdgcn_read_exec()) return t_index_mid(xs, K);
  const float v = (K.fastdiv_dt && mid) ? fdiv(xs, K.zh_dt, K.zl_dt) : xs / K.dt;
  const int it = v != v ? 0 : (int)fminf(fmaxf(floorf(v), -1.0f), (float)K.nt);
  return xs >= K.thr ? K.nt : it;
}

// True when every node whose traveltime sum is at least RN(a + b) has a time
// index >= nt: RN(a + b) >= thr.  Exactly f2i_rd(RN(RN(a + b) / dt)) >= nt
// (NaN gives index 0 and fails the compare; +inf passes both).
__device__ __forceinline__ bool beyond(float a, float b, const KdmK& K) { return a + b >= K.thr; }

// Kirchhoff weight of one node for one trace (the product the reference
// kernels form): Hessian amplitude, obliquity and spreading (S times the two
// tables' amplitudes), the reflection-angle factor 1 + 0.2 cos of the mean
// angle (by the half angles' cosines and sines), and the aperture taper about
// the trace's CMP.  sS = S / (2 pi) and sig_e = sigma + EPS (with its refined
// reciprocal r_sig) come in evaluated per node.  The taper is the reference's
// expression: a = (x - cmp) / sig_e, by the reciprocal and one correction when the
// host found that no operand needs rescaling (RDIV, the operator's taper_rdiv:
// every divisor in [EPS, 2^40), every dividend 0 or of magnitude in [2^-59,
// 2^41)), then exp(-0.5 a a).

// e^(-y / 2) for a finite y >= 0: 2^(-y log2(e) / 2), the exponent split into
// its rounded product hi and the residual fma(y, L, -hi) + y Llo (L + Llo =
// -log2(e) / 2), the nearest integer n of hi applied by ldexp to the hardware
// 2^f of the remaining f in [-0.5, 0.5].  (The factor -1/2 only scales: the
// roundings are those of the exponential of x = -y / 2.)  y is clamped to 208,
// where the result is 0 or the least subnormals.
__device__ __forceinline__ float exp_mhalf(float y) {
#pragma clang fp contract(off)  // hi - n must use the rounded hi: lo holds its residual
  y = fminf(y, 208.0f);
  const float hi = y * -0x1.715476p-1f;
  const float lo = __builtin_fmaf(y, -0x1.4ae0bep-27f, __builtin_fmaf(y, -0x1.715476p-1f, -hi));
  const float n = __builtin_rintf(hi);
  return __builtin_ldexpf(__builtin_amdgcn_exp2f((hi - n) + lo), (int)n);
}

// The aperture taper of x about cmp: r_sig = RN(1 / sig_e) or its refined
// reciprocal.
template <bool RDIV>
__device__ __forceinline__ float kdm_taper(float x, float cmp, float sig_e, float r_sig) {
  const float n = x - cmp;
  if (!RDIV) {
    const float a = n / sig_e;
    return expf(-0.5f * a * a);
  }
  // |a| < 2^61, so a a is finite and >= 0.  One correction of q0 (off by at most
  // a few ulp, the residual exact) leaves the quotient within 0.5 + 2^-20 ulp
  const float q0 = n * r_sig;
  const float a = __builtin_fmaf(__builtin_fmaf(-sig_e, q0, n), r_sig, q0);
  return exp_mhalf(a * a);
}

template <bool RDIV>
__device__ __forceinline__ float kdm_weight(const Q7& s, const Q7& r, float sS, float x, float sig_e, float r_sig,
                                            float cmp) {
  const float rf = __builtin_fmaf(0.2f, __builtin_fmaf(s.ch, r.ch, -(s.sh * r.sh)), 1.0f);
  return sS * (s.amp * r.amp) * rf * kdm_taper<RDIV>(x, cmp, sig_e, r_sig);
}

// The same with the factors of a node that do not depend on the receiver
// already in the source's quantities (q_prefold): amp S / (2 pi), 0.2 ch and
// -0.2 sh.
__device__ __forceinline__ void q_prefold(Q7& s, float sS) {
  s.amp *= sS;
  s.ch *= 0.2f;
  s.sh *= -0.2f;
}
template <bool RDIV>
__device__ __forceinline__ float kdm_weight_pre(const Q7& s, const Q7& r, float x, float sig_e, float r_sig, float cmp) {
  const float rf = __builtin_fmaf(s.ch, r.ch, __builtin_fmaf(s.sh, r.sh, 1.0f));
  return (s.amp * r.amp) * rf * kdm_taper<RDIV>(x, cmp, sig_e, r_sig);
}

// Reflection-angle bin of the node for the trace (the reference's aId): the
// bits of float division, float acosf, division by pi in double, float division
// by da and rounding down (NaN -> 0), without the divisions' rescaling and
// without branches.  The norms are at least EPS; v_div_fixup gives the quotient
// of infinite and NaN operands.  The product with 1 / pi and one fma correction
// is the double quotient (the FMA division theorem).  da = da_m 2^da_e, da_m in
// [1, 2).
__device__ __forceinline__ int kdm_angle_bin(const Q7& s, const Q7& r, const KdmK& K) {
  const float num = s.dx * r.dx + s.dz * r.dz, den = s.norm * r.norm;
  const float c = __builtin_amdgcn_div_fixupf(rdiv(num, den, recip_refined(den)), den, num);
  const double a = 180.0f * (0.5f * acosf(c)), q = a * (1.0 / M_PI);
  const float ang = (float)__builtin_fma(__builtin_fma(-M_PI, q, a), 1.0 / M_PI, q);
  const float v = __builtin_ldexpf(rdiv(ang, K.da_m, K.r_da), -K.da_e);
  return (int)__builtin_amdgcn_fmed3f(v, 0.0f, 1e9f);  // (a NaN's median is the least of the others)
}

// Adjoint: thread per image point (a wave holds 64 consecutive points, one
// chunk).  The traces come grouped in source blocks: up to SB runs of equal
// sources (a run: consecutive traces with one source) per block, and per
// block a list of entries sorted by receiver, each one receiver table and,
// per source slot k, the trace pairing it with the block's k-th source (or
// -1): E = {receiver, t_0, ..., t_(SB-1)}.  A wave keeps the block's source
// quantities in registers and loads a receiver's quantities once per entry,
// for up to SB node-trace pairs.  It passes over a pair when the chunk minima
// keep every node beyond the last sample, over a source slot when the source
// minimum alone does (receiver tables non-negative), and loads nothing for
// either.  The blocks are split into gridDim.y consecutive parts, one wave per
// chunk and part, so that a chunk's work spreads over several waves.  Image
// domain: a part's sum stays in a register (no atomics), taking the
// contributions block by block, by receiver, by slot; with one part it is
// added to the model, with several it is written to part[h] and
// k_kdm_sum_parts adds the parts in order.  Angle domain: adds into the
// (depth, angle, CMP) bins with atomics, as the reference.
#ifndef SEISFAT_KDM_SB
#define SEISFAT_KDM_SB 4
#endif
constexpr int KDM_SB = SEISFAT_KDM_SB;
// Parts per chunk, at most (measured on a 1001 x 1001 image with 13 blocks:
// more waves per chunk, up to one block each, keep shortening both the
// 1 s and the 8 s record's adjoint).
#ifndef SEISFAT_KDM_PARTS
#define SEISFAT_KDM_PARTS 16
#endif
constexpr int KDM_PARTS = SEISFAT_KDM_PARTS;

// The angle domain asks the register allocator for 6 waves per SIMD (80
// vector registers instead of 87, no spills): 0.54 against 0.56 ms on the
// 1001 x 1001 survey.  The image domain's scalar registers allow 7; asking for
// 8 spills them into vector lanes (measured slower on long records).
template <bool ANGLE, int SB, bool RDIV>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(ANGLE ? 6 : 1))) void k_kdm_adjoint(const float* __restrict__ q, const float* __restrict__ tmin,
                                                     const float* __restrict__ S, const int* __restrict__ bsrc,
                                                     const int* __restrict__ bent, const int* __restrict__ ent,
                                                     const float* __restrict__ tcmp, const int* __restrict__ tcid,
                                                     int nb, int nsrc, const float* __restrict__ data,
                                                     float* __restrict__ model, float* __restrict__ part,
                                                     const int* __restrict__ nneg, KdmK K) {
  constexpr int KQ = kq_words(ANGLE);
  const bool rec_nonneg = *nneg == 0;
  const int p0 = blockIdx.x * blockDim.x + threadIdx.x;
  const int nparts = gridDim.y, h = blockIdx.y;
  const int b_begin = (int)((long long)nb * h / nparts), b_end = (int)((long long)nb * (h + 1) / nparts);
  const bool live = p0 < K.npts;
  const int p = live ? p0 : K.npts - 1;  // lanes past the end load in bounds and store nothing
  const int c = __builtin_amdgcn_readfirstlane(p0 >> 6);
  if (c >= K.nchunk) return;  // whole wave past the end
  const int lane = threadIdx.x & 63;
  const int i = p % K.nz, j = p / K.nz;
  const float z = (float)i * K.dz, x = (float)j * K.dx;
  const float sS = K.scale * S[(i + 3) + (size_t)(j + 3) * K.nzz];
  const float sig_e = K.tan_ap * z + KDM_EPS;
  const float r_sig = 1.0f / sig_e;
  float acc = (!ANGLE && live && nparts == 1) ? model[p] : 0.0f;
  for (int b = b_begin; b < b_end; ++b) {
    // slot k in use: bit k (one scalar register for the block)
    float ms[SB];
    unsigned use = 0;
#pragma unroll
    for (int k = 0; k < SB; ++k) {
      const int sk = bsrc[b * SB + k];
      ms[k] = sk >= 0 ? tmin[(size_t)sk * K.nchunk + c] : 0.0f;
      const bool u = sk >= 0 && !(rec_nonneg && beyond(ms[k], 0.0f, K));
      use |= (unsigned)__builtin_amdgcn_readfirstlane((int)u) << k;
    }
    if (!use) continue;
    // the first group of 64 entries holding a pair that passes the chunk
    // test: the sources' quantities are loaded only when there is one
    const int e1 = bent[b + 1];
    int e_first = bent[b];
    for (; e_first < e1; e_first += 64) {
      bool need = false;
      if (e_first + lane < e1) {
        const int* __restrict__ El = ent + (size_t)(e_first + lane) * (1 + SB);
        const float mr = tmin[(size_t)(nsrc + El[0]) * K.nchunk + c];
#pragma unroll
        for (int k = 0; k < SB; ++k) need |= El[1 + k] >= 0 && (use >> k & 1) && !beyond(ms[k], mr, K);
      }
      if (__ballot(need)) break;
    }
    if (e_first >= e1) continue;
    Q7 qs[SB];
#pragma unroll
    for (int k = 0; k < SB; ++k) {
      if (use >> k & 1) {
        const int sk = bsrc[b * SB + k];
        qs[k].t = q[(size_t)sk * KQ * K.npts + p];
        q_amp<KQ>(q, sk, p, K.npts, qs[k]);
        q_prefold(qs[k], sS);
        if (ANGLE) q_dir<KQ>(q, sk, p, K.npts, qs[k]);
      }
    }
    for (int e0 = e_first; e0 < e1; e0 += 64) {
      // lane l holds entry e0 + l (receiver, traces, receiver minimum) and
      // tests it: does any of its pairs pass the chunk test?  The entries that
      // pass are then taken one at a time, their words read from that lane.
      // bit k: slot k holds a trace that passes the chunk test; bit 8 + k: with
      // every sum of the chunk at least 2^-100 and no NaN
      int el_pass = 0;
      int el_r = 0, el_t[SB], el_a[SB];
      float mr_l = 0.0f, el_c[SB];
#pragma unroll
      for (int k = 0; k < SB; ++k) {
        el_t[k] = -1;
        el_a[k] = 0;
        el_c[k] = 0.0f;
      }
      if (e0 + lane < e1) {
        const int* __restrict__ El = ent + (size_t)(e0 + lane) * (1 + SB);
        el_r = nsrc + El[0];
#pragma unroll
        for (int k = 0; k < SB; ++k) el_t[k] = El[1 + k];
        mr_l = tmin[(size_t)el_r * K.nchunk + c];
#pragma unroll
        for (int k = 0; k < SB; ++k)
          if (el_t[k] >= 0 && (use >> k & 1) && !beyond(ms[k], mr_l, K))
            el_pass |= ((K.fastdiv_dt && ms[k] + mr_l >= 0x1p-100f) ? 257 : 1) << k;
        // the traces' CMP (and bin), read from this lane when the entry is taken
        if (el_pass) {
#pragma unroll
          for (int k = 0; k < SB; ++k) {
            if (el_t[k] >= 0) {
              el_c[k] = tcmp[el_t[k]];
              if (ANGLE) el_a[k] = tcid[el_t[k]];
            }
          }
        }
      }
      uint64_t m = __ballot(el_pass != 0);
      // the next entry's receiver traveltime is loaded while this one computes
      int r_next = 0;
      float rt_next = 0.0f;
      if (m) {
        r_next = __builtin_amdgcn_readlane(el_r, (int)__builtin_ctzll(m));
        rt_next = q[(size_t)r_next * KQ * K.npts + p];
      }
      while (m) {
        const int li = (int)__builtin_ctzll(m);
        m &= m - 1;
        const int r = r_next;
        const float rt = rt_next;
        const int pass = __builtin_amdgcn_readlane(el_pass, li);
        if (m) {
          r_next = __builtin_amdgcn_readlane(el_r, (int)__builtin_ctzll(m));
          rt_next = q[(size_t)r_next * KQ * K.npts + p];
        }
        // first the time indices and the data samples of every pair, then the
        // weights: the gathers of one entry are in flight together
        // (slots whose chunk test passes: bit k, uniform)
        int tk[SB];
        float dv[SB];
        bool ok[SB];
        bool anyok = false;
        unsigned slots = 0;
#pragma unroll
        for (int k = 0; k < SB; ++k) {
          ok[k] = false;
          dv[k] = 0.0f;
          tk[k] = -1;
          if (!(pass >> k & 1)) continue;
          tk[k] = __builtin_amdgcn_readlane(el_t[k], li);
          slots |= 1u << k;
          const float xs = qs[k].t + rt;
          // (the clamp keeps the quotient finite; no sample lies beyond it, dt
          // being at most 2^20 where the bit is used)
          const int it = (pass >> k & 256) ? t_index_mid(fminf(xs, 0x1p99f), K) : t_index(xs, K);
          ok[k] = live && (unsigned)it < (unsigned)K.nt;
          // the trace's base (uniform) plus a 32-bit byte offset (it < nt <= 16384)
          const char* __restrict__ dk = (const char*)(data + (size_t)tk[k] * K.nt);
          if (ok[k]) dv[k] = *(const float*)(dk + (unsigned)it * 4u);
          anyok |= ok[k];
        }
        if (!__any(anyok)) continue;  // (the while condition reads the updated m)
        Q7 qr;
        qr.t = rt;
        q_amp<KQ>(q, r, p, K.npts, qr);
        if (ANGLE) q_dir<KQ>(q, r, p, K.npts, qr);
        // every lane of a slot computes its weight; lanes that do not reach
        // the trace add nothing (a select, not a product: their weight may be
        // any value)
#pragma unroll
        for (int k = 0; k < SB; ++k) {
          if (!(slots >> k & 1)) continue;
          const float cmp = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(el_c[k]), li));
          const float w = kdm_weight_pre<RDIV>(qs[k], qr, x, sig_e, r_sig, cmp);
          if (ANGLE) {
            const int a = kdm_angle_bin(qs[k], qr, K);
            const int cb = __builtin_amdgcn_readlane(el_a[k], li);
            if (ok[k] && a >= 0 && a < K.nang)
              atomicAdd(model + i + (size_t)a * K.nz + (size_t)cb * K.nang * K.nz, w * dv[k]);
          } else {
            acc = __builtin_fmaf(ok[k] ? w : 0.0f, dv[k], acc);  // (dv is 0 where not ok)
          }
        }
      }
    }
  }
  if (!ANGLE && live) {
    if (nparts == 1)
      model[p] = acc;
    else
      part[(size_t)h * K.npts + p] = acc;
  }
}

// model[p] += part[0][p] + part[1][p] + ... in that order (the image adjoint's
// partial sums).
__global__ __launch_bounds__(256) void k_kdm_sum_parts(float* __restrict__ model, const float* __restrict__ part,
                                                       int nparts, int npts) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= npts) return;
  float v = model[p];
  for (int h = 0; h < nparts; ++h) v += part[(size_t)h * npts + p];
  model[p] = v;
}

// Forward (image or angle domain) for records that little of the image reaches:
// one workgroup per trace, the trace's nt samples in LDS (FP64, see
// k_kdm_forward_tile); a wave passes over 4096 image points whose super-chunk
// minima keep them beyond the last sample with one test, then over 64 when
// the chunk minima do.
// Threads per trace (one workgroup, sixteen waves sharing the trace's LDS
// histogram).  A call on the 1001 x 1001 survey's 1 s record with 256, 512 and
// 1024 threads: 268, 235 and 199 us (image), 500, 435 and 359 us (angle).
#ifndef SEISFAT_KDM_FWD_THREADS
#define SEISFAT_KDM_FWD_THREADS 1024
#endif
constexpr int KDM_FWD_THREADS = SEISFAT_KDM_FWD_THREADS;

template <bool ANGLE, bool RDIV>
__global__ __launch_bounds__(KDM_FWD_THREADS) void k_kdm_forward(const float* __restrict__ q, const float* __restrict__ tmin,
                                                     const float* __restrict__ S, const int* __restrict__ tsrc,
                                                     const int* __restrict__ trec, const float* __restrict__ tcmp,
                                                     const int* __restrict__ tcid, const float* __restrict__ tmin2,
                                                     int nsrc,
                                                     const float* __restrict__ model, float* __restrict__ data,
                                                     KdmK K) {
  constexpr int KQ = kq_words(ANGLE);
  extern __shared__ double hist[];
  const int t = blockIdx.x;
  for (int k = threadIdx.x; k < K.nt; k += blockDim.x) hist[k] = 0.0;
  __syncthreads();
  const int s = tsrc[t], r = nsrc + trec[t];
  const float cmp = tcmp[t];
  const size_t moff = ANGLE ? (size_t)tcid[t] * K.nang * K.nz : 0;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nwaves = blockDim.x >> 6;
  // each wave takes super-chunks wave, wave + nwaves, ..., tests them 64 at a
  // time (one per lane), and in each that passes tests its 64 chunks (one per
  // lane) and works through the chunks that pass
  for (int k0 = 0; wave + k0 * nwaves < K.nsup; k0 += 64) {
    const int sl = wave + (k0 + lane) * nwaves;
    const bool need2 = sl < K.nsup && !beyond(tmin2[(size_t)s * K.nsup + sl], tmin2[(size_t)r * K.nsup + sl], K);
    for (uint64_t m2 = __ballot(need2); m2; m2 &= m2 - 1) {
      const int c0 = (wave + (k0 + (int)__builtin_ctzll(m2)) * nwaves) * 64;
      const int cl = c0 + lane;
      const bool need = cl < K.nchunk && !beyond(tmin[(size_t)s * K.nchunk + cl], tmin[(size_t)r * K.nchunk + cl], K);
      for (uint64_t m = __ballot(need); m; m &= m - 1) {
        const int p = (c0 + __builtin_ctzll(m)) * 64 + lane;
        if (p >= K.npts) continue;
        Q7 qs, qr;
        qs.t = q[(size_t)s * KQ * K.npts + p];
        qr.t = q[(size_t)r * KQ * K.npts + p];
        const float xs = qs.t + qr.t;
        const int it = t_index(xs, K);
        if ((unsigned)it >= (unsigned)K.nt) continue;
        q_amp<KQ>(q, s, p, K.npts, qs);
        q_amp<KQ>(q, r, p, K.npts, qr);
        if (ANGLE) {
          q_dir<KQ>(q, s, p, K.npts, qs);
          q_dir<KQ>(q, r, p, K.npts, qr);
        }
        const int i = p % K.nz, j = p / K.nz;
        const float z = (float)i * K.dz, x = (float)j * K.dx;
        float sS = K.scale * S[(i + 3) + (size_t)(j + 3) * K.nzz];
        const float sig_e = K.tan_ap * z + KDM_EPS;
        // the weight's words in flight with the bin's: left alone the compiler
        // loads them behind the bin's range test, a memory latency later
        // (sample record 476 against 357 us)
        if (ANGLE)
          asm volatile("" : "+v"(sS), "+v"(qs.amp), "+v"(qs.ch), "+v"(qs.sh), "+v"(qr.amp), "+v"(qr.ch), "+v"(qr.sh),
                       "+v"(qs.dx), "+v"(qs.dz), "+v"(qs.norm), "+v"(qr.dx), "+v"(qr.dz), "+v"(qr.norm));
        const float w = kdm_weight<RDIV>(qs, qr, sS, x, sig_e, recip_refined(sig_e), cmp);
        if (ANGLE) {
          const int a = kdm_angle_bin(qs, qr, K);
          if (a >= 0 && a < K.nang) atomicAdd(hist + it, (double)(w * model[moff + i + (size_t)a * K.nz]));
        } else {
          atomicAdd(hist + it, (double)(w * model[p]));
        }
      }
    }
  }
  __syncthreads();
  float* __restrict__ d = data + (size_t)t * K.nt;
  for (int k = threadIdx.x; k < K.nt; k += blockDim.x) d[k] += (float)hist[k];
}

// Forward for records that much of the image reaches: one workgroup per image
// tile (64 rows x FT_WAVES * NPT columns; lane = row, wave = NPT columns) and
// slice of a source block's entries (the adjoint's blocks).  A node's source
// quantities stay in registers for the whole slice and a receiver's are loaded
// once for up to four traces, where the trace kernel above loads both for every
// pair (32 B a pair: that, beyond L2, bounds it).  Each trace's contributions
// gather in an LDS window of the samples the tile can reach: the index of the
// tile's least and greatest traveltime sums bounds every node's (rounded
// addition and division are monotone), windows longer than FT_WIN take several
// rounds.  The windows are flushed to the traces with global atomics, contiguous
// and several hundred nodes to a sample, and double-buffered, so an entry needs
// one barrier.  LDS sums are FP64: ds_add_f32 takes 169 cycles per wave
// instruction on this chip whatever its addresses, ds_add_f64 8 to 20 (39 with
// pairs of lanes on one address), and the sum is the more exact one.
// 1001 x 1001, 3609 traces of 8001 samples: 5.7 ms (6.1 before the next entry's
// receiver quantities were loaded one entry ahead), against 19.7 ms by trace
// with an FP32 histogram and 16.8 with an FP64 one.
constexpr int FT_WAVES = 8, FT_WIN = 1024, FT_LIST = 128;
constexpr int ft_npt(bool angle) { return angle ? 1 : 2; }

// The least (NaN-propagating) and greatest traveltime of every table over
// every tile of 64 rows and `cols` columns: one wave per table and tile.
__global__ __launch_bounds__(256) void k_kdm_tile_bounds(const float* __restrict__ q, int kq, int ntab, int ntz,
                                                         int ntile, int cols, KdmK K, float* __restrict__ lo,
                                                         float* __restrict__ hi) {
  const int lane = threadIdx.x & 63;
  const int tile = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (tile >= ntile) return;
  const int i = tile % ntz * 64 + lane, j0 = tile / ntz * cols;
  for (int tab = blockIdx.y; tab < ntab; tab += gridDim.y) {
    float a = __builtin_inff(), b = -__builtin_inff();
    if (i < K.nz) {
      const float* __restrict__ t0 = q + (size_t)tab * kq * K.npts + i;
#pragma unroll 8
      for (int j = j0; j < min(j0 + cols, K.nx); ++j) {
        const float t = t0[(size_t)j * K.nz];
        a = min_nan(a, t);
        b = fmaxf(b, t);
      }
    }
    for (int off = 32; off >= 1; off >>= 1) {
      a = min_nan(a, __shfl_xor(a, off, 64));
      b = fmaxf(b, __shfl_xor(b, off, 64));
    }
    if (lane == 0) {
      lo[(size_t)tab * ntile + tile] = a;
      hi[(size_t)tab * ntile + tile] = b;
    }
  }
}

// For launch_forward's choice, over the entries of the adjoint's list and the
// tiles that one of their traces reaches: cnt[0] += the traces that reach the
// tile, cnt[1] += the rounds of windows the entry takes.  One wave per entry.
template <int SB>
__global__ __launch_bounds__(64) void k_kdm_tile_count(const float* __restrict__ tlo, const float* __restrict__ thi,
                                                       int ntile, const int* __restrict__ bsrc,
                                                       const int* __restrict__ bent, int nb,
                                                       const int* __restrict__ ent, int nsrc, KdmK K,
                                                       unsigned long long* __restrict__ cnt) {
  const int e = blockIdx.x;
  int b = 0, b1 = nb;  // the entry's block: bent[b] <= e < bent[b + 1]
  while (b1 - b > 1) {
    const int m = (b + b1) / 2;
    (bent[m] <= e ? b : b1) = m;
  }
  const int* __restrict__ El = ent + (size_t)e * (1 + SB);
  const size_t r = (size_t)(nsrc + El[0]) * ntile;
  unsigned n[2] = {0, 0};
  for (int t = threadIdx.x; t < ntile; t += 64) {
    unsigned most = 0;
#pragma unroll
    for (int k = 0; k < SB; ++k) {
      if (El[1 + k] < 0) continue;
      const size_t s = (size_t)bsrc[b * SB + k] * ntile;
      if (beyond(tlo[s + t], tlo[r + t], K)) continue;
      const float w = (fminf(thi[s + t] + thi[r + t], K.thr) - fmaxf(tlo[s + t] + tlo[r + t], 0.0f)) / K.dt;
      ++n[0];
      most = max(most, 1 + (unsigned)(fminf(fmaxf(w, 0.0f), 16384.0f) / FT_WIN));
    }
    n[1] += most;
  }
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    for (int off = 32; off >= 1; off >>= 1) n[c] += __shfl_xor(n[c], off, 64);
    if (threadIdx.x == 0 && n[c]) atomicAdd(cnt + c, (unsigned long long)n[c]);
  }
}

__global__ void k_kdm_clear(unsigned long long* __restrict__ cnt) { cnt[threadIdx.x] = 0; }

// An entry of the adjoint's list that reaches the tile.
template <int SB>
struct FtEntry {
  int r, pass;                 // receiver table; bit k: slot k reaches, bit 8 + k: by the short index
  int t[SB], lo[SB], len[SB];  // trace, first sample the tile can reach, samples from there
  float cmp[SB];
  int bin[SB];
};

template <bool ANGLE, int SB, int NPT, bool RDIV>
__global__ __launch_bounds__(64 * FT_WAVES) void k_kdm_forward_tile(
    const float* __restrict__ q, const float* __restrict__ tlo, const float* __restrict__ thi, int ntz, int ntile,
    const float* __restrict__ S, const int* __restrict__ bsrc, const int* __restrict__ bent,
    const int* __restrict__ ent, const float* __restrict__ tcmp, const int* __restrict__ tcid, int nsplit, int nsrc,
    const float* __restrict__ model, float* __restrict__ data, KdmK K) {
  constexpr int KQ = kq_words(ANGLE), THREADS = 64 * FT_WAVES;
  constexpr float FAR = 0x1p90f;  // traveltime of a lane outside the image: no sample
  __shared__ double win[2][SB][FT_WIN];
  __shared__ FtEntry<SB> list[FT_LIST];
  __shared__ int count[FT_LIST / 64];
  // workgroups go round robin over the XCDs: the blocks of one tile follow each
  // other on one XCD, and tiles of one depth spread over all of them, the
  // shallowest (which a short record reaches) first.  (With a column's tiles in
  // turn, 8 or 16 of them put all shallow ones on one or two XCDs: 1001 x 1001,
  // 3691 traces, angle domain, nt 1401 2.23 ms against 0.65; the same where every
  // tile reaches the record.)
  const int order = blockIdx.y * 8 + (blockIdx.x & 7), b = (blockIdx.x >> 3) / nsplit, h = (blockIdx.x >> 3) % nsplit;
  if (order >= ntile) return;
  const int ntx = ntile / ntz, tile = order % ntx * ntz + order / ntx;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int i = tile % ntz * 64 + lane, ic = min(i, K.nz - 1);
  const int j0 = tile / ntz * (FT_WAVES * NPT) + wave * NPT;
  const float sig_e = K.tan_ap * ((float)ic * K.dz) + KDM_EPS;
  const float r_sig = 1.0f / sig_e;
  int p[NPT];
  float x[NPT], sS[NPT];
#pragma unroll
  for (int n = 0; n < NPT; ++n) {
    const int jc = min(j0 + n, K.nx - 1);
    p[n] = ic + jc * K.nz;
    x[n] = (float)jc * K.dx;
    sS[n] = 0.0f;
  }
  int par = 0;
  float ms[SB], mh[SB];
#pragma unroll
  for (int k = 0; k < SB; ++k) {
    const int sk = bsrc[b * SB + k];
    ms[k] = sk >= 0 ? tlo[(size_t)sk * ntile + tile] : 0.0f;
    mh[k] = sk >= 0 ? thi[(size_t)sk * ntile + tile] : 0.0f;
  }
  const int ne = bent[b + 1] - bent[b];
  const int e1 = bent[b] + (int)((long long)ne * (h + 1) / nsplit);
  bool started = false;
  Q7 qs[NPT][SB];
  for (int e0 = bent[b] + (int)((long long)ne * h / nsplit); e0 < e1; e0 += FT_LIST) {
    // the first waves list the entries that reach the tile
    if (wave < FT_LIST / 64) {
      const int el = e0 + 64 * wave + lane;
      FtEntry<SB> E;
      E.pass = 0;
      if (el < e1) {
        const int* __restrict__ El = ent + (size_t)el * (1 + SB);
        E.r = nsrc + El[0];
        const float rl = tlo[(size_t)E.r * ntile + tile], rh = thi[(size_t)E.r * ntile + tile];
#pragma unroll
        for (int k = 0; k < SB; ++k) {
          E.t[k] = El[1 + k];
          if (E.t[k] < 0) continue;
          const float lo = ms[k] + rl, hi = mh[k] + rh;
          if (beyond(ms[k], rl, K)) continue;
          E.cmp[k] = tcmp[E.t[k]];
          if (ANGLE) E.bin[k] = tcid[E.t[k]];
          // a NaN node's index is 0 and the lower bound NaN
          const SampleWindow win_k = lo != lo ? SampleWindow{0, K.nt} : sample_window(t_index(lo, K), t_index(hi, K), K.nt);
          E.lo[k] = win_k.first;
          E.len[k] = win_k.len;
          if (win_k.len <= 0) continue;  // every index negative
          E.pass |= 1 << k;
          // every sum in [2^-100, 2^100)
          if (K.fastdiv_dt && lo >= 0x1p-100f && hi < 0x1p80f) E.pass |= 256 << k;
        }
      }
      const uint64_t m = __ballot(E.pass != 0);
      if (E.pass) list[64 * wave + (int)__popcll(m & ((1ull << lane) - 1))] = E;
      if (lane == 0) count[wave] = (int)__popcll(m);
    }
    __syncthreads();
    const int n0 = __builtin_amdgcn_readfirstlane(count[0]), n1 = __builtin_amdgcn_readfirstlane(count[1]);
    if (!started && n0 + n1) {  // the first entry that reaches the tile
      started = true;
      for (int e = threadIdx.x; e < 2 * SB * FT_WIN; e += THREADS) (&win[0][0][0])[e] = 0.0;
#pragma unroll
      for (int n = 0; n < NPT; ++n) {
        sS[n] = K.scale * S[(ic + 3) + (size_t)(min(j0 + n, K.nx - 1) + 3) * K.nzz];
        if (!ANGLE) sS[n] *= model[p[n]];
      }
#pragma unroll
      for (int k = 0; k < SB; ++k) {
        const int sk = bsrc[b * SB + k];
        if (sk < 0) continue;
#pragma unroll
        for (int n = 0; n < NPT; ++n) {
          const bool live = i < K.nz && j0 + n < K.nx;
          qs[n][k].t = live ? q[(size_t)sk * KQ * K.npts + p[n]] : FAR;
          q_amp<KQ>(q, sk, p[n], K.npts, qs[n][k]);
          q_prefold(qs[n][k], sS[n]);
          if (ANGLE) q_dir<KQ>(q, sk, p[n], K.npts, qs[n][k]);
        }
      }
      __syncthreads();
    }
    // an entry's receiver quantities are loaded one entry ahead
    const auto entry = [&](int l) { return l < n0 ? l : 64 + l - n0; };
    Q7 qn[NPT];
    const auto load = [&](int l) {
      const int r = __builtin_amdgcn_readfirstlane(list[entry(min(l, n0 + n1 - 1))].r);
#pragma unroll
      for (int n = 0; n < NPT; ++n) {
        qn[n].t = q[(size_t)r * KQ * K.npts + p[n]];
        q_amp<KQ>(q, r, p[n], K.npts, qn[n]);
        if (ANGLE) q_dir<KQ>(q, r, p[n], K.npts, qn[n]);
      }
    };
    if (n0 + n1) load(0);
    for (int l = 0; l < n0 + n1; ++l) {
      const FtEntry<SB>& E = list[entry(l)];
      const int pass = __builtin_amdgcn_readfirstlane(E.pass);
      Q7 qr[NPT];
#pragma unroll
      for (int n = 0; n < NPT; ++n) qr[n] = qn[n];
      load(l + 1);
      bool more;
      int done = 0;  // samples of the windows already flushed
      do {
        more = false;
        // nothing of a pair is worth keeping in registers for another round
#pragma unroll
        for (int n = 0; n < NPT; ++n) asm volatile("" : "+v"(qr[n].t), "+v"(qr[n].amp), "+v"(qr[n].ch), "+v"(qr[n].sh));
#pragma unroll
        for (int k = 0; k < SB; ++k) {
          if (!(pass >> k & 1)) continue;
          const float cmp = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(E.cmp[k])));
          const int lo = __builtin_amdgcn_readfirstlane(E.lo[k]) + done;
          const int len = __builtin_amdgcn_readfirstlane(E.len[k]) - done;
          more |= len > FT_WIN;
          const unsigned lim = (unsigned)max(min(len, FT_WIN), 0);
          const int cb = ANGLE ? __builtin_amdgcn_readfirstlane(E.bin[k]) : 0;
#pragma unroll
          for (int n = 0; n < NPT; ++n) {
            const float xs = qs[n][k].t + qr[n].t;
            const int it = (pass >> k & 256) ? t_index_mid(xs, K) : t_index(xs, K);
            const unsigned rel = (unsigned)(it - lo);
            if (rel >= lim) continue;
            float w = kdm_weight_pre<RDIV>(qs[n][k], qr[n], x[n], sig_e, r_sig, cmp);
            if (ANGLE) {
              const int a = kdm_angle_bin(qs[n][k], qr[n], K);
              if ((unsigned)a >= (unsigned)K.nang) continue;
              w *= model[ic + (size_t)a * K.nz + (size_t)cb * K.nang * K.nz];
            }
            atomicAdd(&win[par][k][rel], (double)w);
          }
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < SB; ++k) {
          if (!(pass >> k & 1)) continue;
          float* __restrict__ d = data + (size_t)E.t[k] * K.nt + E.lo[k] + done;
          const int n = min(E.len[k] - done, FT_WIN);
          for (int e = threadIdx.x; e < n; e += THREADS) {
            const float v = (float)win[par][k][e];
            if (v != 0.0f) {
              atomicAdd(d + e, v);
              win[par][k][e] = 0.0;
            }
          }
        }
        par ^= 1;
        done += FT_WIN;
      } while (more);
    }
    __syncthreads();  // the list is about to change
  }
}

// Trace convolution: one thread per output sample.  Adjoint: out[k] =
// nfft * sum_m w[m] in[k - shift + m] for k >= shift (0 before); forward:
// out[k] = nfft * sum_m in[m] w[k + shift - m].  Sums in double, in the
// order of m.  For wavelets too long for LDS or not finite.
template <bool ADJ>
__global__ __launch_bounds__(256) void k_trace_conv(const float* __restrict__ in, float* __restrict__ out, int ntr,
                                                    int nt, const float* __restrict__ w, int nw, int shift,
                                                    double nfft) {
  const size_t g = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (g >= (size_t)ntr * nt) return;
  const int t = (int)(g / nt), k = (int)(g - (size_t)t * nt);
  const float* __restrict__ d = in + (size_t)t * nt;
  double acc = 0.0;
  if (ADJ) {
    if (k < shift) {
      out[g] = 0.0f;
      return;
    }
    const int k0 = k - shift;
    const int mmax = min(nw - 1, nt - 1 - k0);
    for (int m = 0; m <= mmax; ++m) acc += (double)w[m] * (double)d[k0 + m];
  } else {
    const int kk = k + shift;
    for (int m = max(0, kk - nw + 1); m <= min(kk, nt - 1); ++m) acc += (double)d[m] * (double)w[kk - m];
  }
  out[g] = (float)(acc * nfft);
}

// The same sums, eight consecutive samples per thread.  Both directions are
//   out[k] = nfft * sum_i h[i] x[k + off + i],  x = 0 outside the trace,
// with h = w, off = -shift (adjoint) or h = w reversed, off = shift - nw + 1
// (forward): a thread's eight sums share their samples, so a tap costs one LDS
// read, one conversion and eight FP64 fmas with h from scalar registers (a
// thread per sample reads and converts two operands per tap).  A product of
// two floats is exact in double, so the fma is the plain sum's rounding, and a
// sample outside the trace adds h * 0 (the host checks that h is finite): the
// same bits.  A wave passes over the taps that meet no sample of the trace from
// any of its sums, most of them where the wavelet is longer than the record
// (1000 traces of 1000 samples, 13000 taps, forward and adjoint: 109 and 32 us;
// 1318 when every tap was walked, 464 and 82 with a sample per thread).  A
// workgroup's threads (at most 256) take `tpw` traces of `groups` groups each, or
// one segment of CONV_SEG samples of a longer one; the samples lie in LDS with one
// word of padding per eight, so the threads' reads (stride 9) meet no bank
// conflict.  Bound by FP64 issue: 3609 traces of 8001 samples, 234 taps: 0.282 ms
// (24 T fma/s), 1.77 ms with a sample per thread; 1001 samples: 0.053 against
// 0.132-0.144 ms.
constexpr int CONV_R = 8, CONV_SEG = 256 * CONV_R;
constexpr int CONV_TAPS = 896;  // wavelet samples per k_put_taps launch (its argument's size)
struct Taps {
  float w[CONV_TAPS];
};

// The wavelet from the kernel's argument to device memory, as doubles: no
// host buffer has to outlive the launch.
__global__ __launch_bounds__(256) void k_put_taps(Taps a, int n, double* __restrict__ h) {
  for (int k = threadIdx.x; k < n; k += 256) h[k] = a.w[k];
}

__global__ __launch_bounds__(256) void k_trace_conv_reg(const float* __restrict__ in, float* __restrict__ out, int ntr,
                                                        int nt, const double* __restrict__ h, int nw, int off,
                                                        int first, double nfft, int tpw, int groups, int span) {
  extern __shared__ float sm[];
  const int tl = threadIdx.x / groups;  // the thread's trace in the workgroup
  const int t0 = blockIdx.x * tpw, k0 = blockIdx.y * CONV_SEG;
  const int pitch = span + span / CONV_R + 1;
  // the taps that meet the trace from the groups a .. b of the workgroup (the
  // first one a multiple of CONV_R)
  const auto tap0 = [&](int b) { return max(-(k0 + b * CONV_R + CONV_R - 1 + off), 0) / CONV_R * CONV_R; };
  const auto tap1 = [&](int a) { return min(nw, nt - (max(k0 + a * CONV_R, first) + off)); };
  const int base = tap0(groups - 1), need = groups * CONV_R + max(tap1(0) - base, 0) + 2 * CONV_R;
  for (int tr = 0; tr < tpw; ++tr)
    for (int q = threadIdx.x; q < need; q += blockDim.x) {
      const int x = k0 + off + base + q;
      sm[tr * pitch + q + q / CONV_R] = (t0 + tr < ntr && x >= 0 && x < nt) ? in[(size_t)(t0 + tr) * nt + x] : 0.0f;
    }
  __syncthreads();
  const int g = threadIdx.x - tl * groups, k = k0 + g * CONV_R;
  // (a wave's lanes of one trace: its first and last group; of several: any)
  const int ga = __builtin_amdgcn_readfirstlane(g), gb = __builtin_amdgcn_readlane(g, 63);
  const bool one = __builtin_amdgcn_readfirstlane(tl) == __builtin_amdgcn_readlane(tl, 63);
  const int i0 = tap0(one ? gb : groups - 1);
  const int i1 = k0 + (one ? gb : groups - 1) * CONV_R + CONV_R - 1 < first ? i0 : tap1(one ? ga : 0);
  if (tl >= tpw || t0 + tl >= ntr || k >= nt) return;
  const float* __restrict__ x = sm + tl * pitch + (g + (i0 - base) / CONV_R) * (CONV_R + 1);
  double acc[CONV_R], X[2 * CONV_R];
#pragma unroll
  for (int o = 0; o < CONV_R; ++o) {
    acc[o] = 0.0;
    X[o] = x[o];
  }
  int i = i0;
  for (; i + CONV_R <= i1; i += CONV_R) {
    x += CONV_R + 1;
#pragma unroll
    for (int o = 0; o < CONV_R; ++o) X[CONV_R + o] = x[o];
#pragma unroll
    for (int u = 0; u < CONV_R; ++u)
#pragma unroll
      for (int o = 0; o < CONV_R; ++o) acc[o] = __builtin_fma(h[i + u], X[u + o], acc[o]);
#pragma unroll
    for (int o = 0; o < CONV_R; ++o) X[o] = X[CONV_R + o];
  }
  x += CONV_R + 1;
#pragma unroll
  for (int o = 0; o < CONV_R - 1; ++o) X[CONV_R + o] = x[o];
#pragma unroll
  for (int u = 0; u < CONV_R - 1; ++u) {
    if (i + u >= i1) break;
#pragma unroll
    for (int o = 0; o < CONV_R; ++o) acc[o] = __builtin_fma(h[i + u], X[u + o], acc[o]);
  }
  float* __restrict__ d = out + (size_t)(t0 + tl) * nt;
#pragma unroll
  for (int o = 0; o < CONV_R; ++o)
    if (k + o < nt) d[k + o] = k + o < first ? 0.0f : (float)(acc[o] * nfft);
}

}  // namespace seisfat

using namespace seisfat;

struct seisfat_kdm_s {
  seisfat_eik_s* h = nullptr;
  seisfat_kdm_params p{};
  int nsrc = 0, nrec = 0, ntr = 0;
  KdmK K{};
  float* d_q = nullptr;    // per-table quantities, (nsrc + nrec) x kq x npts
  int kq = 0;              // words per node and table (kq_words)
  float* d_tmin = nullptr; // per-table chunk minima of T, (nsrc + nrec) x nchunk
  float* d_tmin2 = nullptr; // per-table minima over 64 chunks, (nsrc + nrec) x nsup
  float* d_tlo = nullptr;   // tile bounds of the forward operator, (nsrc + nrec) x ntile each
  float* d_thi = nullptr;
  unsigned long long* d_cnt = nullptr;  // k_kdm_tile_count's sums
  int ntz = 0, ntile = 0, tile_cols = 0;
  bool bounds_dirty = true;  // tables or traces changed since the bounds and the choice below
  bool tables_in_graph = false;  // tables were set under capture: a replay may change them at any time
  bool by_tiles = false;     // the forward operator's kernel
  int nsplit = 1;            // its workgroups per tile and source block (slices of the entries)
  int* d_neg = nullptr;     // behind d_cnt: per receiver table, a negative or NaN value; then their number (k_kdm_rec_neg)
  int* d_src = nullptr;    // trace tables
  int* d_rec = nullptr;
  int nb = 0;              // source blocks of the adjoint
  int nent = 0;            // entries of its list
  int* d_bsrc = nullptr;   // per block and slot: source table (-1: none)
  int* d_bent = nullptr;   // per block: first entry (nb + 1)
  int* d_ent = nullptr;    // entries {receiver, trace per slot}
  float* d_cmp = nullptr;
  int* d_cid = nullptr;
  int nparts = 1;            // adjoint waves per chunk (block ranges)
  float* d_part = nullptr;   // image adjoint partial sums, nparts x npts (nparts > 1)
  std::vector<char> tab_set;  // per table (sources, then receivers): quantities evaluated
  int tabs_missing = 0;
  unsigned s_version = 0;      // the handle's slowness the set tables were evaluated with
  bool taper_geom = false;     // the divisors and x positions allow rdiv for the taper (taper_geometry_ok)
};

namespace {

int kfail(int code, const std::string& m) { return seisfat::set_error(code, m.c_str()); }

// The least float x with RN(x / dt) >= nt (+inf when none): RN(x / dt) is
// monotone in x, so a bisection over the bit patterns of x >= 0 finds it.
float index_threshold(float dt, int nt) {
  auto ge = [&](float x) {
    volatile float v = x / dt;
    return v >= (float)nt;
  };
  const float big = std::numeric_limits<float>::max();
  if (!ge(big)) return std::numeric_limits<float>::infinity();
  if (ge(0.0f)) return 0.0f;
  uint32_t lo = 0, hi;
  std::memcpy(&hi, &big, 4);
  while (hi - lo > 1) {
    const uint32_t mid = lo + (hi - lo) / 2;
    float x;
    std::memcpy(&x, &mid, 4);
    (ge(x) ? hi : lo) = mid;
  }
  float x;
  std::memcpy(&x, &hi, 4);
  return x;
}

#define KHIP(expr)                                                                                  \
  do {                                                                                              \
    hipError_t e_ = (expr);                                                                         \
    if (e_ != hipSuccess)                                                                           \
      return kfail(e_ == hipErrorOutOfMemory ? SEISFAT_ENOMEM : SEISFAT_EHIP,                       \
                   std::string(#expr) + ": " + hipGetErrorString(e_));                              \
  } while (0)

template <class T>
void kfree(T*& p) {
  if (p) (void)hipFree((void*)p);
  p = nullptr;
}

// The aperture quotient (x - cmp) / sig_e needs no operand rescaling (rdiv is
// then IEEE division) when every divisor sig_e = tan_ap z + EPS lies in
// [EPS, 2^40) (tan_ap >= 0: it grows with z, largest at the last row) and
// every x = j dx and every CMP is 0 or of magnitude in [2^-36, 2^40): the
// difference of two such floats is 0 or of magnitude in [2^-59, 2^41) (both
// are multiples of 2^-59), and the quotient normal.  Here the divisors and the
// x positions; set_traces checks the CMPs.
bool taper_geometry_ok(const KdmK& K) {
  if (!(K.tan_ap >= 0.0f) || !std::isfinite(K.tan_ap)) return false;
  const double zmax = (double)(K.nz - 1) * K.dz, xmax = (double)(K.nx - 1) * K.dx;
  if (!((double)K.tan_ap * zmax + KDM_EPS <= 0x1p39)) return false;
  return (K.nx == 1 || K.dx >= 0x1p-36f) && xmax <= 0x1p39;
}

// The quantities and chunk minima of ntab consecutive tables (padded grids at
// d_tables) into table slots tab0, tab0 + 1, ...: one wave per chunk.
void launch_prep(seisfat_kdm_s* k, const float* d_tables, int tab0, int ntab, hipStream_t st) {
  // a wave keeps its chunk and walks up to 8 tables (their slowness and
  // position loaded once), fewer where that leaves the chip short of waves
  const unsigned bx = (k->K.nchunk + 3) / 4;
  const unsigned by = (unsigned)std::min<long long>(std::max<long long>((ntab + 7) / 8, 8192 / bx + 1),
                                                    std::min(ntab, 65535));
  float* q = k->d_q + (size_t)tab0 * k->kq * k->K.npts;
  float* tmin = k->d_tmin + (size_t)tab0 * k->K.nchunk;
  if (k->p.domain == SEISFAT_KDM_ANGLE)
    hipLaunchKernelGGL(k_kdm_prep<true>, dim3(bx, by), dim3(256), 0, st, d_tables, ntab, k->h->d_spad, k->K, q, tmin);
  else
    hipLaunchKernelGGL(k_kdm_prep<false>, dim3(bx, by), dim3(256), 0, st, d_tables, ntab, k->h->d_spad, k->K, q, tmin);
  const size_t ns = (size_t)ntab * k->K.nsup;
  const int blocks2 = (int)std::min<size_t>((ns + 3) / 4, 16384);
  hipLaunchKernelGGL(k_kdm_tmin2, dim3(blocks2), dim3(256), 0, st, tmin, ntab, k->K,
                     k->d_tmin2 + (size_t)tab0 * k->K.nsup);
  if (tab0 >= k->nsrc)
    hipLaunchKernelGGL(k_kdm_rec_neg, dim3(ntab), dim3(64), 0, st, k->d_tmin2 + (size_t)tab0 * k->K.nsup, k->K,
                       k->d_neg + (tab0 - k->nsrc), k->d_neg + k->nrec);
}

// The operators' launches, one instantiation per domain and taper division.
template <bool ANGLE, bool RDIV>
void launch_adjoint(seisfat_kdm_s* k, const float* d_data, float* d_model, hipStream_t st) {
  const dim3 grid((k->K.npts + 255) / 256, k->nparts);
  hipLaunchKernelGGL((k_kdm_adjoint<ANGLE, KDM_SB, RDIV>), grid, dim3(256), 0, st, k->d_q, k->d_tmin, k->h->d_spad,
                     k->d_bsrc, k->d_bent, k->d_ent, k->d_cmp, k->d_cid, k->nb, k->nsrc, d_data, d_model,
                     ANGLE ? nullptr : k->d_part, k->d_neg + k->nrec, k->K);
}

template <bool ANGLE, bool RDIV>
void launch_forward(seisfat_kdm_s* k, const float* d_model, float* d_data, hipStream_t st) {
  if (k->by_tiles) {
    hipLaunchKernelGGL((k_kdm_forward_tile<ANGLE, KDM_SB, ft_npt(ANGLE), RDIV>),
                       dim3(8 * k->nb * k->nsplit, (k->ntile + 7) / 8), dim3(64 * FT_WAVES), 0, st, k->d_q, k->d_tlo,
                       k->d_thi, k->ntz, k->ntile, k->h->d_spad, k->d_bsrc, k->d_bent, k->d_ent, k->d_cmp, k->d_cid,
                       k->nsplit, k->nsrc, d_model, d_data, k->K);
    return;
  }
  const size_t lds = (size_t)k->K.nt * sizeof(double);
  if (lds > 65536)  // at most 16384 samples: 128 of the 160 KB
    (void)hipFuncSetAttribute((const void*)k_kdm_forward<ANGLE, RDIV>, hipFuncAttributeMaxDynamicSharedMemorySize,
                              131072);
  hipLaunchKernelGGL((k_kdm_forward<ANGLE, RDIV>), dim3(k->ntr), dim3(KDM_FWD_THREADS), lds, st, k->d_q, k->d_tmin,
                     k->h->d_spad, k->d_src, k->d_rec, k->d_cmp, k->d_cid, k->d_tmin2, k->nsrc, d_model, d_data,
                     k->K);
}

// After tables were set on a stream: the forward's bounds are stale.
int tables_changed(seisfat_kdm_s* k, hipStream_t st) {
  k->bounds_dirty = true;
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  KHIP(hipStreamIsCapturing(st, &cap));
  if (cap != hipStreamCaptureStatusNone) k->tables_in_graph = true;
  return SEISFAT_OK;
}

bool cmp_ok(float c) { return c == 0.0f || (std::fabs(c) >= 0x1p-36f && std::fabs(c) < 0x1p40f); }

// The table quantities hold the slowness they were evaluated with (the
// amplitudes): a slowness upload to the handle makes every table set before it
// stale, to be set again.
void track_slowness(seisfat_kdm_s* k) {
  if (k->s_version == k->h->version) return;
  std::fill(k->tab_set.begin(), k->tab_set.end(), 0);
  k->tabs_missing = k->nsrc + k->nrec;
  k->s_version = k->h->version;
}

void free_traces(seisfat_kdm_s* k) {
  kfree(k->d_src);
  kfree(k->d_rec);
  kfree(k->d_cmp);
  kfree(k->d_cid);
  kfree(k->d_bsrc);
  kfree(k->d_bent);
  kfree(k->d_ent);
  kfree(k->d_part);
  k->ntr = k->nb = 0;
  k->nparts = 1;
}

}  // namespace

extern "C" {

int seisfat_kdm_create(seisfat_eik_t h, const seisfat_kdm_params* p, int nsrc, int nrec, seisfat_kdm_t* out) {
  if (!out) return kfail(SEISFAT_EINVAL, "null output pointer");
  *out = nullptr;
  if (!h || !p) return kfail(SEISFAT_EINVAL, "null handle or parameters");
  if (!h->has_s) return kfail(SEISFAT_ESTATE, "slowness not set (seisfat_eik_set_slowness)");
  if (p->domain != SEISFAT_KDM_IMAGE && p->domain != SEISFAT_KDM_ANGLE)
    return kfail(SEISFAT_EINVAL, "domain must be SEISFAT_KDM_IMAGE (0) or SEISFAT_KDM_ANGLE (1)");
  if (p->nt <= 0 || p->nt > 16384) return kfail(SEISFAT_EINVAL, "nt must lie in [1, 16384]");
  if (!(p->dt > 0.0f) || !std::isfinite(p->dt)) return kfail(SEISFAT_EINVAL, "dt must be positive");
  if (!std::isfinite(p->aperture)) return kfail(SEISFAT_EINVAL, "aperture must be finite");
  if (p->domain == SEISFAT_KDM_ANGLE && (p->nang <= 0 || p->ncmp <= 0 || !(p->da > 0.0f)))
    return kfail(SEISFAT_EINVAL, "angle domain: nang and ncmp must be positive, da positive");
  if (nsrc <= 0 || nrec <= 0) return kfail(SEISFAT_EINVAL, "nsrc and nrec must be positive");
  const size_t npts = (size_t)h->nz * h->nx;
  if (npts > (size_t)1 << 30) return kfail(SEISFAT_EINVAL, "model too large");
  auto* k = new (std::nothrow) seisfat_kdm_s();
  if (!k) return kfail(SEISFAT_ENOMEM, "host allocation");
  k->h = h;
  k->p = *p;
  k->nsrc = nsrc;
  k->nrec = nrec;
  KdmK& K = k->K;
  K.nz = h->nz;
  K.nx = h->nx;
  K.nzz = h->nzz;
  K.npts = (int)npts;
  K.nchunk = (int)((npts + 63) / 64);
  K.nsup = (K.nchunk + 63) / 64;
  K.nt = p->nt;
  K.nang = p->domain == SEISFAT_KDM_ANGLE ? p->nang : 0;
  K.dx = h->dx;
  K.dz = h->dz;
  K.dz2 = K.dz * K.dz;
  K.dx2 = K.dx * K.dx;
  K.dxz4 = 4.0f * K.dx * K.dz;
  K.r_dz = 1.0f / K.dz;
  K.r_dx = 1.0f / K.dx;
  K.r_dz2 = 1.0f / K.dz2;
  K.r_dx2 = 1.0f / K.dx2;
  K.r_dxz4 = 1.0f / K.dxz4;
  const auto mid = [](float v) { return v >= 0x1p-20f && v <= 0x1p20f; };
  K.prep_rdiv = mid(K.dz) && mid(K.dx);
  K.nz_recip = K.nz > 1 ? (unsigned)(((uint64_t)1 << 32) / (unsigned)K.nz) : 0;
  K.dt = p->dt;
  K.thr = index_threshold(p->dt, p->nt);
  // two-word reciprocal of dt: zh = RN(1/dt); 1 - dt*zh is exact (one fma)
  K.zh_dt = 1.0f / p->dt;
  K.zl_dt = std::fma(-p->dt, K.zh_dt, 1.0f) / p->dt;
  K.fastdiv_dt = 0;
  K.da_m = 2.0f * std::frexp(p->domain == SEISFAT_KDM_ANGLE ? p->da : 1.0f, &K.da_e);
  K.da_e -= 1;
  K.r_da = 1.0f / K.da_m;
  // sigma = tanf(aperture * pi / 180) * z, the angle rounded to float as the
  // reference's float argument takes it; 1 / (2 pi) rounded from double
  K.tan_ap = std::tan((float)((double)p->aperture * M_PI / 180.0));
  K.scale = (float)(1.0 / (2.0 * M_PI));
  k->kq = kq_words(p->domain == SEISFAT_KDM_ANGLE);
  hipError_t e = hipMalloc((void**)&k->d_q, (size_t)(nsrc + nrec) * k->kq * npts * sizeof(float));
  if (e == hipSuccess) e = hipMalloc((void**)&k->d_tmin, (size_t)(nsrc + nrec) * K.nchunk * sizeof(float));
  if (e == hipSuccess) e = hipMalloc((void**)&k->d_tmin2, (size_t)(nsrc + nrec) * K.nsup * sizeof(float));
  k->ntz = (K.nz + 63) / 64;
  k->tile_cols = FT_WAVES * ft_npt(p->domain == SEISFAT_KDM_ANGLE);
  k->ntile = k->ntz * ((K.nx + k->tile_cols - 1) / k->tile_cols);
  if (e == hipSuccess) e = hipMalloc((void**)&k->d_tlo, (size_t)(nsrc + nrec) * k->ntile * sizeof(float));
  if (e == hipSuccess) e = hipMalloc((void**)&k->d_thi, (size_t)(nsrc + nrec) * k->ntile * sizeof(float));
  const size_t words = 4 + ((size_t)nrec + 1);  // the two counts, then the receivers' flags and their number
  if (e == hipSuccess) e = hipMalloc((void**)&k->d_cnt, words * sizeof(int));
  if (e == hipSuccess) {
    k->d_neg = (int*)(k->d_cnt + 2);
    launch_fill((float*)k->d_cnt, words, 0.0f, nullptr);
    // exhaustive check of the known-divisor division by dt (every dividend of
    // magnitude in [2^-100, 2^100)) against IEEE division
    float* d = nullptr;
    const float w[3] = {K.dt, K.zh_dt, K.zl_dt};
    int bad = 1;
    e = hipMalloc((void**)&d, 4 * sizeof(float));
    if (e == hipSuccess) e = hipMemcpy(d, w, sizeof(w), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemset(d + 3, 0, sizeof(int));
    if (e == hipSuccess) {
      launch_fastdiv_check(d, d + 1, d + 2, 1, (int*)(d + 3), nullptr);
      e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpy(&bad, d + 3, sizeof(int), hipMemcpyDeviceToHost);
    if (d) (void)hipFree(d);
    K.fastdiv_dt = (e == hipSuccess && bad == 0 && mid(K.dt)) ? 1 : 0;  // (and no quotient overflows)
  }
  if (e != hipSuccess) {
    kfree(k->d_q);
    kfree(k->d_tmin);
    kfree(k->d_tmin2);
    kfree(k->d_tlo);
    kfree(k->d_thi);
    kfree(k->d_cnt);
    delete k;
    return kfail(SEISFAT_ENOMEM, std::string("hipMalloc of the table quantities: ") + hipGetErrorString(e));
  }
  k->tab_set.assign(nsrc + nrec, 0);
  k->tabs_missing = nsrc + nrec;
  k->s_version = h->version;
  k->taper_geom = taper_geometry_ok(K);
  K.taper_rdiv = 0;
  *out = k;
  return SEISFAT_OK;
}

int seisfat_kdm_set_tables(seisfat_kdm_t k, const float* d_src, const float* d_rec, void* stream) {
  if (!k || !d_src || !d_rec) return kfail(SEISFAT_EINVAL, "null operator or table pointer");
  hipStream_t st = (hipStream_t)stream;
  track_slowness(k);
  launch_prep(k, d_src, 0, k->nsrc, st);
  launch_prep(k, d_rec, k->nsrc, k->nrec, st);
  KHIP(hipGetLastError());
  std::fill(k->tab_set.begin(), k->tab_set.end(), 1);
  k->tabs_missing = 0;
  return tables_changed(k, st);
}

int seisfat_kdm_set_table(seisfat_kdm_t k, int which, int index, const float* d_table, void* stream) {
  if (!k || !d_table) return kfail(SEISFAT_EINVAL, "null operator or table pointer");
  if (which != 0 && which != 1) return kfail(SEISFAT_EINVAL, "which must be 0 (source) or 1 (receiver)");
  const int n = which ? k->nrec : k->nsrc;
  if (index < 0 || index >= n) return kfail(SEISFAT_EINVAL, "table index out of range");
  const int tab = (which ? k->nsrc : 0) + index;
  hipStream_t st = (hipStream_t)stream;
  track_slowness(k);
  launch_prep(k, d_table, tab, 1, st);
  KHIP(hipGetLastError());
  if (!k->tab_set[tab]) {
    k->tab_set[tab] = 1;
    --k->tabs_missing;
  }
  return tables_changed(k, st);
}

namespace {

// Before a launch: every table set with the current slowness.
int ready(seisfat_kdm_s* k) {
  if (k->s_version != k->h->version)
    return kfail(SEISFAT_ESTATE, "the slowness changed since the tables were set (set them again)");
  if (k->tabs_missing) return kfail(SEISFAT_ESTATE, "tables not set (seisfat_kdm_set_tables / _set_table)");
  return SEISFAT_OK;
}

// The forward operator's tile bounds and its choice between its two kernels,
// once per tables and traces: it waits for two counts.  A stream under capture
// cannot: there the choice stands as the last call made it (the kernel that
// needs no bounds if tables or traces changed since), and the bounds' launch is
// recorded with the tile kernel's, so that a replay follows tables set after the
// capture.  The same launch precedes every tile kernel once tables were set
// under capture.
//
// The two kernels' times in ns, fitted over 350 surveys (120 to 1001 rows, 200 to
// 1001 columns, 400 to 8001 samples, both domains).  Tiles: `round` for an entry's
// round in a tile it reaches, `entry` for each entry of a workgroup's slice (they
// are taken one after another), `group` for a workgroup.  By traces: for each tile
// a trace reaches, `near` (more where the image has fewer super-chunks than half
// of a workgroup's waves: 48000 traces on 65 x 98 take 5.6 ms, by tiles 1.4), up
// to `far` more as a table outgrows the caches, and `few` more as the traces are
// too few to fill the chip; its workgroups are larger, 8 us more a launch.
// The chosen kernel is 1.4 % (image) and 3 % (angle) slower in the mean than the
// faster one; of 261 surveys in the angle domain 12 run more than 5 % slower than
// by traces (at most 1.23 times).  Trace / tile kernel, ms: 1001x1001, 3691 traces
// at 1 ms, image: nt 701 0.102 / 0.128, 1001 0.203 / 0.192, 1501 0.444 / 0.305,
// 2501 1.18 / 0.65, 5001 4.5 / 2.3; angle: nt 600 0.124 / 0.248, 1001 0.363 /
// 0.405, 1401 0.79 / 0.65, 2001 1.65 / 1.11, 8001 21.6 / 10.8; 499x209, 1120 traces
// at 4 ms, angle: nt 425 0.267 / 0.219, 900 0.58 / 0.40.
struct FtCosts {
  double round, entry, group, near, far, few;
};
constexpr FtCosts ft_costs(bool angle) {
  return angle ? FtCosts{8.0, 1400.0, 3.0, 1.8, 2.0, 0.6} : FtCosts{6.0, 1300.0, 2.0, 2.1, 1.0, 1.1};
}
constexpr double FT_LAUNCH = 8000.0, FT_CACHED = 3e5;  // (image points of a table that the caches hold)
int derive_bounds(seisfat_kdm_s* k, hipStream_t st) {
  if (k->bounds_dirty) k->by_tiles = false;
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  KHIP(hipStreamIsCapturing(st, &cap));
  const bool captured = cap != hipStreamCaptureStatusNone;
  const bool choose = !captured && k->bounds_dirty;
  if (!choose && !(k->by_tiles && (captured || k->tables_in_graph))) return SEISFAT_OK;
  hipLaunchKernelGGL(k_kdm_tile_bounds, dim3((k->ntile + 3) / 4, std::min(k->nsrc + k->nrec, 65535)), dim3(256), 0, st,
                     k->d_q, k->kq, k->nsrc + k->nrec, k->ntz, k->ntile, k->tile_cols, k->K, k->d_tlo, k->d_thi);
  if (!choose) return SEISFAT_OK;
  hipLaunchKernelGGL(k_kdm_clear, dim3(1), dim3(2), 0, st, k->d_cnt);
  hipLaunchKernelGGL(k_kdm_tile_count<KDM_SB>, dim3(k->nent), dim3(64), 0, st, k->d_tlo, k->d_thi, k->ntile, k->d_bsrc,
                     k->d_bent, k->nb, k->d_ent, k->nsrc, k->K, k->d_cnt);
  KHIP(hipGetLastError());
  unsigned long long n[2] = {0, 0};
  KHIP(hipMemcpyAsync(n, k->d_cnt, sizeof(n), hipMemcpyDeviceToHost, st));
  KHIP(hipStreamSynchronize(st));
  const FtCosts f = ft_costs(k->p.domain == SEISFAT_KDM_ANGLE);
  const double by_tile = f.round * n[1] + f.entry * k->nent / ((double)k->nb * k->nsplit) +
                         f.group * k->ntile * k->nb * k->nsplit;
  const double by_trace =
      FT_LAUNCH + n[0] * (f.near / std::min(1.0, k->K.nsup / (KDM_FWD_THREADS / 128.0)) +
                          f.far * std::min(1.0, k->K.npts / FT_CACHED) + f.few / std::min(1.0, k->ntr / 512.0));
  k->by_tiles = by_tile < by_trace && k->ntile <= 8 * 65535 && 4096.0 * k->nb * k->nsplit < 0x1p32 && k->K.dt < 0x1p60f;
  k->bounds_dirty = false;
  return SEISFAT_OK;
}

}  // namespace

int seisfat_kdm_set_traces(seisfat_kdm_t k, int ntr, const int* src, const int* rec, const float* cmp,
                           const int* cmp_id) {
  if (!k) return kfail(SEISFAT_EINVAL, "null operator");
  if (ntr < 0 || (ntr > 0 && (!src || !rec || !cmp))) return kfail(SEISFAT_EINVAL, "bad trace arrays");
  if (k->p.domain == SEISFAT_KDM_ANGLE && ntr > 0 && !cmp_id)
    return kfail(SEISFAT_EINVAL, "the angle domain needs CMP bins");
  for (int t = 0; t < ntr; ++t) {
    if (src[t] < 0 || src[t] >= k->nsrc || rec[t] < 0 || rec[t] >= k->nrec)
      return kfail(SEISFAT_EINVAL, "trace " + std::to_string(t) + ": table index out of range");
    if (!std::isfinite(cmp[t])) return kfail(SEISFAT_EINVAL, "trace " + std::to_string(t) + ": CMP not finite");
    if (k->p.domain == SEISFAT_KDM_ANGLE && (cmp_id[t] < 0 || cmp_id[t] >= k->p.ncmp))
      return kfail(SEISFAT_EINVAL, "trace " + std::to_string(t) + ": CMP bin out of range");
  }
  KHIP(hipDeviceSynchronize());  // runs in flight may read the previous trace tables
  free_traces(k);
  k->bounds_dirty = true;
  k->K.taper_rdiv = (k->taper_geom && std::all_of(cmp, cmp + ntr, cmp_ok)) ? 1 : 0;
  if (ntr == 0) return SEISFAT_OK;
  KHIP(hipMalloc((void**)&k->d_src, ntr * sizeof(int)));
  KHIP(hipMalloc((void**)&k->d_rec, ntr * sizeof(int)));
  KHIP(hipMalloc((void**)&k->d_cmp, ntr * sizeof(float)));
  KHIP(hipMalloc((void**)&k->d_cid, ntr * sizeof(int)));
  // source blocks for the adjoint: SB runs of equal sources per block, each
  // block's pairs sorted by (receiver, slot), traces in order within equal keys
  std::vector<int> run0;
  for (int t = 0; t < ntr; ++t)
    if (t == 0 || src[t] != src[t - 1]) run0.push_back(t);
  run0.push_back(ntr);
  const int nruns = (int)run0.size() - 1;
  const int nb = (nruns + KDM_SB - 1) / KDM_SB;
  std::vector<int> bsrc((size_t)nb * KDM_SB, -1), bent(nb + 1, 0), ent;
  struct Pair {
    int r, k, t;
  };
  std::vector<Pair> pairs;
  for (int b = 0; b < nb; ++b) {
    pairs.clear();
    for (int k = 0; k < KDM_SB && b * KDM_SB + k < nruns; ++k) {
      const int r0 = run0[b * KDM_SB + k], r1 = run0[b * KDM_SB + k + 1];
      bsrc[(size_t)b * KDM_SB + k] = src[r0];
      for (int t = r0; t < r1; ++t) pairs.push_back({rec[t], k, t});
    }
    std::stable_sort(pairs.begin(), pairs.end(),
                     [](const Pair& a, const Pair& c) { return a.r != c.r ? a.r < c.r : a.k < c.k; });
    size_t cur = (size_t)-1;
    for (const Pair& pr : pairs) {
      if (cur == (size_t)-1 || ent[cur] != pr.r || ent[cur + 1 + pr.k] != -1) {
        cur = ent.size();
        ent.push_back(pr.r);
        ent.insert(ent.end(), KDM_SB, -1);
      }
      ent[cur + 1 + pr.k] = pr.t;
    }
    bent[b + 1] = (int)(ent.size() / (1 + KDM_SB));
  }
  KHIP(hipMalloc((void**)&k->d_bsrc, bsrc.size() * sizeof(int)));
  KHIP(hipMalloc((void**)&k->d_bent, bent.size() * sizeof(int)));
  KHIP(hipMalloc((void**)&k->d_ent, ent.size() * sizeof(int)));
  KHIP(hipMemcpy(k->d_bsrc, bsrc.data(), bsrc.size() * sizeof(int), hipMemcpyHostToDevice));
  KHIP(hipMemcpy(k->d_bent, bent.data(), bent.size() * sizeof(int), hipMemcpyHostToDevice));
  KHIP(hipMemcpy(k->d_ent, ent.data(), ent.size() * sizeof(int), hipMemcpyHostToDevice));
  k->nb = nb;
  k->nent = (int)(ent.size() / (1 + KDM_SB));
  // the forward's tiles: enough workgroups for the chip, at least 8 entries each
  const long long wgs = (long long)k->ntile * nb, per_block = (long long)(ent.size() / (1 + KDM_SB)) / nb;
  k->nsplit = (int)std::max<long long>(1, std::min((1024 + wgs - 1) / wgs, per_block / 8));
  // adjoint parts: up to KDM_PARTS, no more than the blocks; the image
  // domain's partial sums within 1 GiB
  int np = std::max(1, std::min(KDM_PARTS, nb));
  if (k->p.domain == SEISFAT_KDM_IMAGE) {
    while (np > 1 && (size_t)np * k->K.npts * sizeof(float) > ((size_t)1 << 30)) --np;
    if (np > 1) KHIP(hipMalloc((void**)&k->d_part, (size_t)np * k->K.npts * sizeof(float)));
  }
  k->nparts = np;
  std::vector<int> cid(ntr, 0);
  if (k->p.domain == SEISFAT_KDM_ANGLE) cid.assign(cmp_id, cmp_id + ntr);
  KHIP(hipMemcpy(k->d_src, src, ntr * sizeof(int), hipMemcpyHostToDevice));
  KHIP(hipMemcpy(k->d_rec, rec, ntr * sizeof(int), hipMemcpyHostToDevice));
  KHIP(hipMemcpy(k->d_cmp, cmp, ntr * sizeof(float), hipMemcpyHostToDevice));
  KHIP(hipMemcpy(k->d_cid, cid.data(), ntr * sizeof(int), hipMemcpyHostToDevice));
  k->ntr = ntr;
  return SEISFAT_OK;
}

int seisfat_kdm_adjoint(seisfat_kdm_t k, const float* d_data, float* d_model, void* stream) {
  if (!k) return kfail(SEISFAT_EINVAL, "null operator");
  hipStream_t st = (hipStream_t)stream;
  if (const int rc = ready(k)) return rc;
  if (k->ntr == 0) return SEISFAT_OK;  // no traces: the model is unchanged
  if (!d_data || !d_model) return kfail(SEISFAT_EINVAL, "null buffer");
  const bool rd = k->K.taper_rdiv != 0;
  if (k->p.domain == SEISFAT_KDM_IMAGE) {
    if (rd)
      launch_adjoint<false, true>(k, d_data, d_model, st);
    else
      launch_adjoint<false, false>(k, d_data, d_model, st);
    if (k->nparts > 1)
      hipLaunchKernelGGL(k_kdm_sum_parts, dim3((k->K.npts + 255) / 256), dim3(256), 0, st, d_model, k->d_part,
                         k->nparts, k->K.npts);
  } else if (rd) {
    launch_adjoint<true, true>(k, d_data, d_model, st);
  } else {
    launch_adjoint<true, false>(k, d_data, d_model, st);
  }
  KHIP(hipGetLastError());
  return SEISFAT_OK;
}

int seisfat_kdm_forward(seisfat_kdm_t k, const float* d_model, float* d_data, void* stream) {
  if (!k) return kfail(SEISFAT_EINVAL, "null operator");
  hipStream_t st = (hipStream_t)stream;
  if (const int rc = ready(k)) return rc;
  if (k->ntr == 0) return SEISFAT_OK;  // no traces to add into
  if (!d_data || !d_model) return kfail(SEISFAT_EINVAL, "null buffer");
  if (const int rc = derive_bounds(k, st)) return rc;
  const bool rd = k->K.taper_rdiv != 0;
  if (k->p.domain == SEISFAT_KDM_IMAGE) {
    if (rd)
      launch_forward<false, true>(k, d_model, d_data, st);
    else
      launch_forward<false, false>(k, d_model, d_data, st);
  } else if (rd) {
    launch_forward<true, true>(k, d_model, d_data, st);
  } else {
    launch_forward<true, false>(k, d_model, d_data, st);
  }
  KHIP(hipGetLastError());
  return SEISFAT_OK;
}

int seisfat_kdm_destroy(seisfat_kdm_t k) {
  if (!k) return SEISFAT_OK;
  (void)hipDeviceSynchronize();
  free_traces(k);
  kfree(k->d_q);
  kfree(k->d_tmin);
  kfree(k->d_tmin2);
  kfree(k->d_tlo);
  kfree(k->d_thi);
  kfree(k->d_cnt);
  delete k;
  return SEISFAT_OK;
}

int seisfat_trace_convolve(int adjoint, int ntr, int nt, const float* wavelet, int nw, const float* d_in,
                           float* d_out, void* stream) {
  if (ntr < 0 || nt <= 0 || nw <= 0 || !wavelet || (ntr > 0 && (!d_in || !d_out || d_in == d_out)))
    return kfail(SEISFAT_EINVAL, "bad convolution arguments (distinct device buffers, positive sizes)");
  if (ntr == 0) return SEISFAT_OK;
  // nfft = the power of two >= nt + nw - 1 (the reference's nextpow2)
  long long nfft = 1;
  while (nfft < (long long)nt + nw - 1) nfft <<= 1;
  const int shift = nw / 2 + nw / 10;
  hipStream_t st = (hipStream_t)stream;
  const size_t n = (size_t)ntr * nt;
  // out[k] = nfft sum_i h[i] in[k + off + i] for k >= first, and the taps that
  // meet a sample of the trace from any of these outputs
  const int first = adjoint ? shift : 0;
  long long off = adjoint ? -(long long)shift : (long long)shift - nw + 1;
  const int tap0 = (int)std::max<long long>(0, -(nt - 1 + off));
  const int ntap = first >= nt ? 0 : (int)std::max<long long>(0, std::min<long long>(nw, nt - (first + off)) - tap0);
  off += tap0;
  // samples a workgroup stages per trace: its outputs, its taps, and up to the next whole group
  const int groups = std::min((nt + CONV_R - 1) / CONV_R, 256);
  const long long taps = std::min<long long>(ntap, (long long)nt + (groups + 1) * CONV_R);
  const long long span = (long long)groups * CONV_R + (taps + CONV_R - 1) / CONV_R * CONV_R + 2 * CONV_R;
  const size_t lds1 = (size_t)(span + span / CONV_R + 1) * sizeof(float);
  if (lds1 <= 65536 && std::all_of(wavelet, wavelet + nw, [](float v) { return std::isfinite(v); })) {
    // several short traces per workgroup, within 40 KB (four workgroups per CU)
    const int tpw = (int)std::max<size_t>(1, std::min<size_t>(256 / groups, 40960 / lds1));
    double* d_h = nullptr;
    KHIP(hipMallocAsync((void**)&d_h, std::max(ntap, 1) * sizeof(double), st));
    for (int i0 = 0; i0 < ntap; i0 += CONV_TAPS) {
      Taps a;
      const int m = std::min(CONV_TAPS, ntap - i0), t = tap0 + i0;
      for (int i = 0; i < m; ++i) a.w[i] = adjoint ? wavelet[t + i] : wavelet[nw - 1 - (t + i)];
      hipLaunchKernelGGL(k_put_taps, dim3(1), dim3(256), 0, st, a, m, d_h + i0);
    }
    const dim3 grid((ntr + tpw - 1) / tpw, (nt + CONV_SEG - 1) / CONV_SEG);
    hipLaunchKernelGGL(k_trace_conv_reg, grid, dim3((tpw * groups + 63) / 64 * 64), tpw * lds1, st, d_in, d_out, ntr,
                       nt, d_h, ntap, (int)off, first, (double)nfft, tpw, groups, (int)span);
    const hipError_t e = hipGetLastError();
    KHIP(hipFreeAsync(d_h, st));
    KHIP(e);
    return SEISFAT_OK;
  }
  float* d_w = nullptr;
  KHIP(hipMallocAsync((void**)&d_w, nw * sizeof(float), st));
  KHIP(hipMemcpyAsync(d_w, wavelet, nw * sizeof(float), hipMemcpyHostToDevice, st));
  const int blocks = (int)((n + 255) / 256);
  if (adjoint)
    hipLaunchKernelGGL(k_trace_conv<true>, dim3(blocks), dim3(256), 0, st, d_in, d_out, ntr, nt, d_w, nw, shift,
                       (double)nfft);
  else
    hipLaunchKernelGGL(k_trace_conv<false>, dim3(blocks), dim3(256), 0, st, d_in, d_out, ntr, nt, d_w, nw, shift,
                       (double)nfft);
  KHIP(hipGetLastError());
  KHIP(hipFreeAsync(d_w, st));
  KHIP(hipStreamSynchronize(st));  // the host wavelet is the caller's
  return SEISFAT_OK;
}

int seisfat_ricker(float dt, float fmax, float* out, int cap) {
  if (!(dt > 0.0f) || !(fmax > 0.0f) || !std::isfinite(dt) || !std::isfinite(fmax) || cap < 0 || (cap > 0 && !out))
    return kfail(SEISFAT_EINVAL, "ricker: dt and fmax must be positive, out non-null when cap > 0");
  const float t0 = 2.0f * std::sqrt((float)M_PI) / fmax;
  const float fc = fmax / (3.0f * std::sqrt((float)M_PI));
  const float len = (t0 - 0.5f * dt) / dt;
  if (!(len < 1e9f)) return kfail(SEISFAT_EINVAL, "ricker: wavelet too long (dt too small for fmax)");
  const int nw = std::max(2 * (int)len, 0);
  for (int k = 0; k < std::min(nw, cap); ++k) {
    const float td = k * dt - t0;
    const float arg = (float)(M_PI * M_PI * M_PI * fc * fc * td * td);  // double product, as the reference's
    out[k] = (1.0f - 2.0f * arg) * std::exp(-arg);
  }
  return nw;
}

}  // extern "C"
