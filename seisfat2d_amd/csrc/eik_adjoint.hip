// Adjoint-state (reverse-mode) gradient kernels of the single-pass eikonal
// solve.  The forward is SeisFAT2D's time_init + one pass of four sweeps
// (src/modeling/modeling.cu:110-159, local solver :308-357); the gradient is
// the exact derivative of that discrete map, so it is what a finite
// difference of the forward converges to.  The reference's tomography uses a
// ray-traced sensitivity instead (src/inversion/inversion.cpp:95-177), which
// this gradient replaces.
//
// Branch decisions and local derivatives come from an fp64 trajectory of the
// solve recorded on the device; the adjoint recurrence runs in fp32 and the
// cross-shot accumulation in fp64.  Every reduction runs in a fixed order, so
// the gradient is deterministic.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "eik_adjoint.h"

namespace seisfat {

// ---------------------------------------------------------------------------
__global__ void k_fill_d(double* __restrict__ p, size_t n, double v) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    p[i] = v;
}

__global__ void k_adj_seed(const size_t* __restrict__ node, const int* __restrict__ ptr,
                           const int* __restrict__ rec, const float* __restrict__ wt, int nseed,
                           const float* __restrict__ w, float* __restrict__ lam) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= nseed) return;
  float acc = 0.0f;
  for (int e = ptr[n]; e < ptr[n + 1]; ++e) acc += w[rec[e]] * wt[e];
  lam[node[n]] = acc;
}

// ---------------------------------------------------------------------------
// The recorded trajectory is an fp64 solve of the same single-pass scheme:
// fp32 rounding decides near-tied branch choices (two sweeps' candidates
// agreeing to a few ulps, common where the wave travels along a grid axis),
// and the derivative of the fp32 map then differs locally from the derivative
// the fp64 map (and finite differences of it) has.  Decisions and partials
// are taken from the fp64 trajectory; the adjoint recurrence runs in fp32.
struct ConstsD {
  double dx, dz, dx2i, dz2i, sum, sum4, prod, hyp;
  double r_dx, r_dz, r_sum, r_hyp;  // RN(1/divisor), for cdiv
};

// RN(a / b) for a model-constant divisor b, from y = RN(1/b) (computed on the
// host by IEEE division): q = RN(a y) is within one ulp of a/b, the residual
// a - b q is exact (one fma), and RN(q + (a - b q) y) is the correctly
// rounded quotient (Markstein, IBM J. Res. Dev. 34(1), 1990; Muller et al.,
// Handbook of Floating-Point Arithmetic, the FMA-based division theorems),
// for every a whose quotient neither underflows nor overflows.  Three
// instructions instead of the general division's scale / reciprocal /
// iteration / fix-up sequence; the dividends here are traveltime differences
// and slowness products of a validated model, far from both limits.
__device__ __forceinline__ double cdiv(double a, double b, double y) {
  const double q = a * y;
  const double r = __builtin_fma(-b, q, a);
  return __builtin_fma(r, y, q);
}

__device__ __forceinline__ double dpp_shr1_d(double old, double src) {
  const long long o = __double_as_longlong(old), s = __double_as_longlong(src);
  const int lo = __builtin_amdgcn_update_dpp((int)o, (int)s, 0x138, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp((int)(o >> 32), (int)(s >> 32), 0x138, 0xf, 0xf, false);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// wave_shl:1: lane k receives lane k+1's `src`; lane 63 keeps `old`.
__device__ __forceinline__ float dpp_shl1f(float old, float src) {
  return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(old), __float_as_int(src), 0x130, 0xf, 0xf,
                                                    false));
}

// time_set + time_init in fp64 (T0 holds 1e6 elsewhere for good).
__global__ void k_fwd64_init(const AdjShot* __restrict__ shots, int nshots, int nzz, double dx, double dz,
                             double* __restrict__ T0) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nshots * 9) return;
  const AdjShot sh = shots[t / 9];
  const int ii = (t % 9) % 3, jj = (t % 9) / 3;
  const double sx = sh.sd.sx, sz = sh.sd.sz;
  const int sIdx = (int)((sx + 0.5 * dx) / dx) + NB;
  const int sIdz = (int)((sz + 0.5 * dz) / dz) + NB;
  const int zi = sIdz + (ii - 1), xi = sIdx + (jj - 1);
  const double ddx = (double)(xi - NB) * dx - sx;
  const double ddz = (double)(zi - NB) * dz - sz;
  T0[sh.toff + zi + (size_t)xi * nzz] = (double)s_at(sh.sd, nzz, zi, xi) * sqrt(ddx * ddx + ddz * ddz);
}

// Minimum of two doubles, neither a NaN (no quieting of loaded operands).
__device__ __forceinline__ double vmin_d(double a, double b) {
  double r;
  asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

// sqrt(x) for a normal x whose root needs no rescaling: the hardware estimate
// of 1 / sqrt(x) and the coupled iteration for the root and half its
// reciprocal (Markstein), with two residual corrections: IEEE's root.
__device__ __forceinline__ double sqrt_rn_d(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  const double r = __builtin_fma(-h, g, 0.5);
  g = __builtin_fma(g, r, g);
  h = __builtin_fma(h, r, h);
  g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
  return __builtin_fma(__builtin_fma(-g, g, x), h, g);
}

// What the local solver derives from the reference cell, evaluated when the
// cell is first read (as the previous step's z-other cell).
struct CellD {
  double dzs, dxs, s2, s4, thrB, thrC;
};

__device__ __forceinline__ double thr_b(double s, const ConstsD& k) { return cdiv(k.dz * s * k.dz, k.hyp, k.r_hyp); }

template <bool EQH>
__device__ __forceinline__ CellD cell_d(double s, double thrB, const ConstsD& k) {
  CellD c;
  c.dzs = k.dz * s;
  c.dxs = EQH ? c.dzs : k.dx * s;
  c.s2 = s * s;
  c.s4 = c.s2 * k.sum4;  // (4s s) sum: the factors of 4 only scale
  c.thrB = thrB;
  c.thrC = EQH ? thrB : cdiv(c.dxs * k.dx, k.hyp, k.r_hyp);
  return c;
}

// The local solver (src/modeling/modeling.cu:308-357) in fp64, operation for
// operation as the fp64 oracle evaluates it, and its minimum with told, without
// branches: every lane evaluates all candidates and the values of branches not
// taken are selected away; branches A, B and C share one square root.  Its radicand is positive wherever it is used (A: the
// difference of the upwind times is at most a cell's edge time; B, C: the
// threshold keeps q below s) and, with the validated slowness, far from the
// range that needs rescaling.  h min(a, b) = min(h a, h b) for h > 0.
template <bool EQH>
__device__ __forceinline__ double local_sel_d(double tv, double te, double tev, const CellD& r, double dz_zo,
                                              double dx_xo, double told, const ConstsD& k) {
  const double t1d = vmin_d(tv + vmin_d(r.dzs, dz_zo), te + vmin_d(r.dxs, dx_xo));
  const double de = te - tev, dv = tv - tev;
  // Every condition is one compare whose mask goes straight to the selects (a
  // mask combined on the scalar unit costs the step two crossings).  Branch A's
  // four: a difference of doubles rounds to zero only when it is zero, so
  // RN(a - b) >= 0 exactly when a >= b, and the minimum is >= 0 when all are.
  const bool cA = vmin_d(vmin_d((te + r.dxs) - tv, (tv + r.dzs) - te), vmin_d(de, dv)) >= 0.0;
  // 0 < d <= thr (thr > 0): positive doubles order as their bits, and zeros and
  // negatives less one are at least as large as any positive double's
  const bool cB = (unsigned long long)__double_as_longlong(de) - 1 < (unsigned long long)__double_as_longlong(r.thrB);
  const bool cC = (unsigned long long)__double_as_longlong(dv) - 1 < (unsigned long long)__double_as_longlong(r.thrC);
  const double ta = tev + te - tv, tb = tev - te + tv, dab = ta - tb;
  const double dd = cB ? de : dv;
  const double q = EQH ? cdiv(dd, k.dz, k.r_dz) : cdiv(dd, cB ? k.dz : k.dx, cB ? k.r_dz : k.r_dx);
  double radA = r.s4 - k.prod * dab * dab, radBC = r.s2 - q * q;
  asm("" : "+v"(radA), "+v"(radBC));  // both evaluated: no branch around either
  const double root = sqrt_rn_d(cA ? radA : radBC);
  double vA = cdiv((tb * k.dz2i + ta * k.dx2i) + root, k.sum, k.r_sum);
  double vBC = (cB ? te : tv) + (EQH ? k.dz : cB ? k.dx : k.dz) * root;
  asm("" : "+v"(vA), "+v"(vBC));
  double two = cC ? vBC : 1e6;
  two = cB ? vBC : two;
  two = cA ? vA : two;
  return vmin_d(vmin_d(t1d, told), two);  // (told <= 1e6 already)
}

// One fp64 sweep, Tnew = sweep(Told), out of place (ring nodes of Tnew hold
// 1e6 for good).  A workgroup walks one strip of 64 sweep-local rows of one
// shot.  Its first wave computes: lane k holds row 64r + k and visits column
// t - k at step t; its z-upwind and diagonal neighbours are lane k-1's results
// one and two steps back (DPP shift), its x-upwind neighbour its own previous
// result.  Traveltimes pass through an LDS ring of WK_R columns, which the
// second and third wave fill and empty by whole columns (contiguous rows, as
// global memory holds them): every step's 64 nodes lie in 64 different columns,
// and a wave that loads and stores them itself touches 64 cache lines three
// times a step (that version took 1.1 ms for 640 independent strips of 1207
// columns against 0.47 ms for one alone, and 1.35 ms for 128 shots of 5
// dependent strips).  In the ring the nodes of one step are 64 words of
// different banks; results replace the old values in place.  Blocks of WK_B
// steps end with one barrier; the column waves load two blocks ahead.
// The first wave's step is bound by its instruction count (about 83, one in
// four cycles) and the traveltime chain; a sweep of 128 shots of 307 x 1207
// nodes takes 0.38 ms (1.20-1.36 before), one shot alone 0.29 (0.65), one strip
// 0.23 (0.47).
//
// The strips of a shot run concurrently, each trailing the one above: lane 0's
// upwind inputs are the upper strip's lane-63 results (its last row), which the
// upper strip's column waves publish as they empty the ring, each double as two
// 64-bit words (one 32-bit half + the launch's tag in the high half), written
// and read as single agent-scope atomics: a reader that sees the tag in both
// words has the value, with no fence on either side.  The fourth wave polls the
// next block's words (bounded: past the limit it sets the flag and stops
// waiting for the rest of the strip, so a broken dependency cannot stall the
// device) and hands them to the first through LDS, with the slowness cells
// below the strip's last row.  Strips are claimed from a ticket counter
// strip-major (every shot's strip r before any strip r+1), so a strip's upper
// neighbour always holds a smaller ticket and is running: the walk drains for
// any number of resident workgroups.
constexpr int WALK_SPIN = 1 << 16;
constexpr int WK_B = 8;             // steps per block
constexpr int WK_R = 64 + 2 * WK_B;  // ring columns: a step's 64, a block arriving, a block leaving
constexpr int WK_C = WK_B / 2;       // columns per block and column wave

__global__ void k_walk_begin(int* __restrict__ ctl) {
  if (threadIdx.x == 0) ctl[0] = 0;
}

__device__ __forceinline__ unsigned long long walk_word(unsigned half, unsigned tag) {
  return ((unsigned long long)tag << 32) | half;
}

// Workgroup barrier after this wave's LDS operations (its global ones may stay
// in flight).
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// The slowness cell that lane k of strip r (k = 64: the row below it) reads as
// its z-other cell at local column c: s_at's row, and its column clamped to the
// cells and to the shot's view in one median.  Byte offsets (below 2^32: at most
// 2^30 padded nodes) from the uniform base.
template <int SA, int SB>
struct ZoCell {
  typedef __attribute__((address_space(1))) const char gchar;
  gchar* base;
  unsigned row, pitch;
  int first, hi;
  __device__ ZoCell(const ShotDev& sd, int nzz, int fi) {
    const int f = min(max(fi, 1), nzz - 1);
    base = (gchar*)sd.sbase;
    row = 4u * (unsigned)((SA > 0 ? f : nzz - 1 - f) - (SA + 1) / 2);
    pitch = 4u * (unsigned)nzz;
    first = (SB > 0 ? 0 : sd.nxx - 2) - sd.sofs;
    hi = min(max(sd.nxx - 2 - sd.sofs, 0), sd.smax);
  }
  __device__ unsigned offset(int c) const {
    return row + (unsigned)min(max(SB > 0 ? first + c : first - c, 0), hi) * pitch;
  }
  __device__ float at_offset(unsigned o) const { return *(__attribute__((address_space(1))) const float*)(base + o); }
  __device__ float at(int c) const { return at_offset(offset(c)); }
  // no column from c0 to c1 is clamped
  __device__ bool plain(int c0, int c1) const {
    return SB > 0 ? first + c0 >= 0 && first + c1 <= hi : first - c1 >= 0 && first - c0 <= hi;
  }
};

template <int SA, int SB, bool EQH>
__global__ __launch_bounds__(256) void k_fwd64_sweep(const AdjShot* __restrict__ shots, int nshots, int nzz,
                                                    int nstr, ConstsD K, SkewView sk,
                                                    const double* __restrict__ Told, double* __restrict__ Tnew,
                                                    int* __restrict__ ctl, unsigned long long* __restrict__ xw,
                                                    int ldx, unsigned tag) {
  typedef __attribute__((address_space(1))) unsigned long long gword;
  // column c, row k lies at ring[((c + k) mod WK_R) * 64 + k]: the nodes of step
  // c + k are 64 consecutive words
  __shared__ double ring[WK_R * 64];
  __shared__ double thr_l[2][WK_B][64];  // a block's z-other cells: branch B's threshold
  __shared__ float s_l[2][WK_B][66];     // and slowness (lane 64: the row below the strip)
  __shared__ double xup_l[2][WK_B];      // upper strip's last row, columns of a block's steps
  __shared__ int ticket;
  const int lane = threadIdx.x & 63;
  // (the hardware starts each workgroup of a CU on another SIMD, so the compute
  // waves of up to four share none)
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  for (;;) {
    if (threadIdx.x == 0) ticket = atomicAdd(ctl, 1);
    __syncthreads();
    const int tk = __builtin_amdgcn_readfirstlane(ticket);
    if (tk >= nshots * nstr) break;
    const int r = tk / nshots, ks = tk - r * nshots;
    const AdjShot sh = shots[ks];
    const int nxx = sh.sd.nxx;
    const int NBLK = (nxx + 63 + WK_B - 1) / WK_B;
    // this strip's published last row, and the upper strip's
    gword* xme = (gword*)(xw + ((size_t)ks * nstr + r) * ldx);
    const gword* xup = (const gword*)(xw + ((size_t)ks * nstr + max(r - 1, 0)) * ldx);
    const int fi = 64 * r + lane;
    const bool row_int = fi >= 1 && fi <= nzz - 2;
    // block n: the compute wave takes steps 8n .. 8n + 7; the others bring what
    // block n + 1 reads.  (Blocks -1 and NBLK, NBLK + 1 only move data.)
    if (wave == 0) {
      double prev = 1e6, tev = 1e6;
      CellD ref = cell_d<EQH>(1.0, 1.0, K);  // the previous step's z-other cell (unused at step 0)
      const auto block = [&](int t0, int buf, auto edge) {
        double* __restrict__ rg = ring + (t0 % WK_R) * 64 + lane;
        unsigned zero = 0;
        asm volatile("" : "+v"(zero));  // (one address register for the block's broadcasts)
        // a step's operands are read one step ahead
        double told = rg[0], gv = xup_l[buf][zero], thr = thr_l[buf][0][lane];
        float szo = s_l[buf][0][lane], sxo = s_l[buf][0][lane + 1];
#pragma unroll
        for (int u = 0; u < WK_B; ++u) {
          const double told_u = told, thr_u = thr;
          const float szo_u = szo, sxo_u = sxo;
          // z-upwind: lane k-1's last result (lane 0: the upper strip's); the
          // diagonal one was it a step ago
          const double tv = dpp_shr1_d(gv, prev);
          if (u + 1 < WK_B) {
            told = rg[64 * (u + 1)];
            gv = xup_l[buf][zero + u + 1];
            thr = thr_l[buf][u + 1][lane];
            szo = s_l[buf][u + 1][lane];
            sxo = s_l[buf][u + 1][lane + 1];
          }
          const CellD next = cell_d<EQH>((double)szo_u, thr_u, K);
          double out = local_sel_d<EQH>(tv, prev, tev, ref, next.dzs, K.dx * (double)sxo_u, told_u, K);
          ref = next;
          const int fj = t0 + u - lane;
          if (!(row_int && (!edge.value || (fj >= 1 && fj <= nxx - 2)))) out = 1e6;
          rg[64 * u] = out;
          tev = tv;
          prev = out;
        }
      };
      lds_barrier();  // block -1
      for (int n = 0; n < NBLK; ++n) {
        const int t0 = n * WK_B;
        if (t0 >= 64 && t0 + WK_B - 1 <= nxx - 2)
          block(t0, n & 1, std::false_type());
        else
          block(t0, n & 1, std::true_type());
        lds_barrier();
      }
      lds_barrier();
      lds_barrier();
    } else if (wave < 3) {
      const double* __restrict__ To = Told + sh.toff;
      double* __restrict__ Tn = Tnew + sh.toff;
      const int fic = min(max(fi, 1), nzz - 2);
      const int i = SA > 0 ? fic : nzz - 1 - fic;
      const int c_off = (wave - 1) * WK_C;  // this wave's columns of a block
      const auto col = [&](int fj) { return (size_t)(SB > 0 ? fj : nxx - 1 - fj) * nzz; };
      const auto load = [&](int c, double& v) { v = (To + col(min(max(c, 1), nxx - 2)))[(unsigned)i]; };
      double qa[WK_C], qb[WK_C];
#pragma unroll
      for (int u = 0; u < WK_C; ++u) load(c_off + u, qa[u]);
#pragma unroll
      for (int u = 0; u < WK_C; ++u) load(WK_B + c_off + u, qb[u]);
      const bool pub = lane == 63 && r + 1 < nstr;
      // during block n: columns 8n + 8 .. 8n + 15 arrive in the words of columns
      // 8n - 72 .. 8n - 65, whose last node block n - 1 computed
      const auto move = [&](int n, double (&q)[WK_C]) {
        const int c_in = (n + 1) * WK_B + c_off, c_out = c_in - WK_R;
        double done[WK_C];
        unsigned o[WK_C];
#pragma unroll
        for (int u = 0; u < WK_C; ++u) {
          o[u] = (unsigned)(c_in % WK_R + u + lane);  // (WK_C divides WK_R: below 2 WK_R)
          o[u] = min(o[u], o[u] - WK_R) * 64 + lane;
          done[u] = ring[o[u]];
        }
#pragma unroll
        for (int u = 0; u < WK_C; ++u) ring[o[u]] = q[u];
#pragma unroll
        for (int u = 0; u < WK_C; ++u) {
          const int fj = c_out + u;
          if (pub && fj >= 1 && fj <= nxx - 2) {
            __hip_atomic_store(xme + 2 * fj, walk_word((unsigned)__double2hiint(done[u]), tag), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(xme + 2 * fj + 1, walk_word((unsigned)__double2loint(done[u]), tag), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
          }
        }
#pragma unroll
        for (int u = 0; u < WK_C; ++u) {
          const int fj = c_out + u;
          if (row_int && fj >= 1 && fj <= nxx - 2) (Tn + col(fj))[(unsigned)i] = done[u];
        }
#pragma unroll
        for (int u = 0; u < WK_C; ++u) load(c_in + 2 * WK_B + u, q[u]);
      };
      // NBLK + 3 blocks, in pairs (a block past the last moves nothing of the grid)
      for (int n = -1; n < NBLK + 2; n += 2) {
        move(n, qa);
        lds_barrier();
        if (n + 1 < NBLK + 2) {
          move(n + 1, qb);
          lds_barrier();
        }
      }
    } else {
      const ZoCell<SA, SB> zo(sh.sd, nzz, fi), zo64(sh.sd, nzz, 64 * r + 64);
      bool gave_up = false;
      // the cells of steps 8(n + 1) .., one block ahead (lane u: the row below
      // the strip at step u)
      float q[WK_B], q64;
      // Away from the clamped columns they come from the model's skewed copy
      // (see SkewView): cell row kap = f - 1 of lane k >= 1 has kap mod 64 =
      // k - 1, so the cells of one step share a skewed column; lane 0's (row
      // 64r - 1) lie 64 columns further along the sweep (1 in strip 0, whose row
      // 0 reads cell row 0).  64 lines a step without it: the strips of a shot
      // then wait for one another (1.5 times the time of one strip alone with
      // three workgroups on a CU).
      const int kap = min(max(fi, 1), nzz - 1) - 1;
      const int lead = lane > 0 ? 0 : r > 0 ? 64 : 1;
      const unsigned lane_off = 4u * (unsigned)(kap + (SB > 0 ? lead : 64 - lead) * sk.KP);
      const auto load = [&](int t0) {
        if (sk.base && zo.plain(t0 - 64, t0 + WK_B - 1)) {
          const int sig = sh.sd.x0 + sh.sd.sofs + (SB > 0 ? zo.first + t0 - 1 : zo.first - t0);
          typedef __attribute__((address_space(1))) const char gchar;
          gchar* b = (gchar*)(sk.base + (size_t)(sig + SK_OFF) * sk.KP);
#pragma unroll
          for (int u = 0; u < WK_B; ++u)
            q[u] = *(__attribute__((address_space(1))) const float*)(b + (long long)(SB * u) * sk.KP * 4 + lane_off);
        } else {
#pragma unroll
          for (int u = 0; u < WK_B; ++u) q[u] = zo.at(t0 + u - lane);
        }
        q64 = zo64.at(t0 + (lane & (WK_B - 1)) - 64);
      };
      load(0);
      for (int n = -1; n < NBLK + 2; ++n) {
        const int t = (n + 1) * WK_B + (lane & (WK_B - 1)), buf = (n + 1) & 1;
        // the upper strip's value of column clamp(t, 1, nxx-2) (strip 0 has no
        // upper strip: its first row is the ring)
        const int fjc = min(max(t, 1), nxx - 2);
        double v = 1e6;
        if (r > 0 && n + 1 < NBLK) {
          for (int it = 0;; ++it) {
            const unsigned long long hw = __hip_atomic_load(xup + 2 * fjc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const unsigned long long lw =
                __hip_atomic_load(xup + 2 * fjc + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            v = __hiloint2double((int)(unsigned)hw, (int)(unsigned)lw);
            if (gave_up || __all((unsigned)(hw >> 32) == tag && (unsigned)(lw >> 32) == tag)) break;
            if (it > WALK_SPIN) {
              if (lane == 0) atomicOr(ctl + 1, 1);
              gave_up = true;
              break;
            }
            __builtin_amdgcn_s_sleep(1);
          }
        }
        // step 0's value is only step 1's diagonal one: the ring's
        if (lane < WK_B) xup_l[buf][lane] = t == 0 ? 1e6 : v;
        // (the cells after the words: the poll does not queue behind the next
        // block's loads, which touch 64 lines each)
#pragma unroll
        for (int u = 0; u < WK_B; ++u) {
          s_l[buf][u][lane] = q[u];
          thr_l[buf][u][lane] = thr_b((double)q[u], K);
        }
        if (lane < WK_B) s_l[buf][lane][64] = q64;
        load((n + 2) * WK_B);
        lds_barrier();
      }
    }
  }
}

// Catmull-Rom picks of the fp64 trajectory's final traveltimes (the residuals
// of the misfit gradient), as the fp64 oracle evaluates them.
__device__ __forceinline__ double cubic1d_d(const double P[4], double d) {
  return P[1] + 0.5 * d * (P[2] - P[0] + d * (2.0 * P[0] - 5.0 * P[1] + 4.0 * P[2] - P[3] +
                                             d * (3.0 * (P[1] - P[2]) + P[3] - P[0])));
}

__global__ void k_picks64(const AdjShot* __restrict__ shots, const int* __restrict__ rec_shot,
                          const float* __restrict__ rx, const float* __restrict__ rz, int nrec, int nzz, double dx,
                          double dz, const double* __restrict__ T4, double* __restrict__ out) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= nrec) return;
  const double* __restrict__ T = T4 + shots[rec_shot[r]].toff;
  const double x = rx[r], z = rz[r];
  const double x0 = floor((x + 0.5 * dx) / dx) * dx;
  const double z0 = floor((z + 0.5 * dz) / dz) * dz;
  const double x1 = floor((x + 0.5 * dx) / dx) * dx + dx;
  const double z1 = floor((z + 0.5 * dz) / dz) * dz + dz;
  const double xd = (x - x0) / (x1 - x0);
  const double zd = (z - z0) / (z1 - z0);
  const int i = (int)((z + 0.5 * dz) / dz) + NB;
  const int j = (int)((x + 0.5 * dx) / dx) + NB;
  double p[4];
  for (int pIdx = 0; pIdx < 4; ++pIdx) {
    double P[4];
    for (int pIdz = 0; pIdz < 4; ++pIdz) P[pIdz] = T[(i + pIdz - 1) + (size_t)(j + pIdx - 1) * nzz];
    p[pIdx] = cubic1d_d(P, zd);
  }
  out[r] = cubic1d_d(p, xd);
}

// ---------------------------------------------------------------------------
// Local partials of one node.  ds < 0 marks a node the sweep left unchanged
// (T_old kept: the adjoint passes through); bit (di | dj << 1) of code marks
// slowness cell (i - di, j - dj) as receiving ds, split evenly when two bits
// are set.
struct AdjCoef {
  float dtv, dte, dtev, ds;
  int code;
};

// The branch the fp64 forward took at a node (same expressions and
// comparisons as local_sel_d) and its partial derivatives.  Ties follow the
// oracle: T_old wins when T_old <= candidate; 1-D before 2-D when equal;
// z-edge before x-edge when equal; min(S, S') of two equal cells splits dS
// half and half (what central differences measure).
template <int SA, int SB>
__device__ __forceinline__ AdjCoef adj_local(double tv, double te, double tev, double sref, double szo,
                                             double sxo, double told, const ConstsD& k) {
  constexpr int di_ref = (SA + 1) / 2, dj_ref = (SB + 1) / 2;
  constexpr int c_ref = di_ref | (dj_ref << 1);
  constexpr int c_zo = di_ref | (((1 - SB) / 2) << 1);
  constexpr int c_xo = ((1 - SA) / 2) | (dj_ref << 1);
  const double t1d1 = tv + k.dz * fmin(sref, szo);
  const double t1d2 = te + k.dx * fmin(sref, sxo);
  const double t1D = fmin(t1d1, t1d2);
  double tbr = 1e6;
  bool taken = false;
  double p_tv = 0.0, p_te = 0.0, p_tev = 0.0, p_s = 0.0;
  if ((tv <= te + k.dx * sref) && (te <= tv + k.dz * sref) && (te - tev >= 0.0) && (tv - tev >= 0.0)) {
    const double ta = tev + te - tv;
    const double tb = tev - te + tv;
    const double sq = sqrt(4.0 * sref * sref * k.sum - k.prod * (ta - tb) * (ta - tb));
    tbr = cdiv((tb * k.dz2i + ta * k.dx2i) + sq, k.sum, k.r_sum);
    taken = true;
    // t = ((tb dz2i + ta dx2i) + sqrt(4 S^2 D - dz2i dx2i (ta - tb)^2)) / D
    const double kk = 2.0 * k.prod * (ta - tb) / sq;
    p_te = cdiv(k.dx2i - k.dz2i - kk, k.sum, k.r_sum);
    p_tv = cdiv(k.dz2i - k.dx2i + kk, k.sum, k.r_sum);
    p_tev = 1.0;
    p_s = 4.0 * sref / sq;
  } else if ((te - tev <= cdiv(sref * k.dz * k.dz, k.hyp, k.r_hyp)) && (te - tev > 0.0)) {
    // t = te + dx sqrt(S^2 - q^2), q = (te - tev) / dz
    const double q = cdiv(te - tev, k.dz, k.r_dz);
    const double Q = sqrt(sref * sref - q * q);
    tbr = te + k.dx * Q;
    taken = true;
    const double r = k.dx * q / (k.dz * Q);
    p_te = 1.0 - r;
    p_tev = r;
    p_s = k.dx * sref / Q;
  } else if ((tv - tev <= cdiv(sref * k.dx * k.dx, k.hyp, k.r_hyp)) && (tv - tev > 0.0)) {
    const double p = cdiv(tv - tev, k.dx, k.r_dx);
    const double P = sqrt(sref * sref - p * p);
    tbr = tv + k.dz * P;
    taken = true;
    const double r = k.dz * p / (k.dx * P);
    p_tv = 1.0 - r;
    p_tev = r;
    p_s = k.dz * sref / P;
  }
  const double t2D = fmin(tbr, 1e6);
  const double cand = fmin(t1D, t2D);
  AdjCoef c{0.0f, 0.0f, 0.0f, -1.0f, 0};
  if (!(cand < told)) return c;
  if (t1D <= t2D) {
    if (t1d1 <= t1d2) {
      c.dtv = 1.0f;
      c.ds = (float)k.dz;
      c.code = sref == szo ? (1 << c_ref) | (1 << c_zo) : sref < szo ? 1 << c_ref : 1 << c_zo;
    } else {
      c.dte = 1.0f;
      c.ds = (float)k.dx;
      c.code = sref == sxo ? (1 << c_ref) | (1 << c_xo) : sref < sxo ? 1 << c_ref : 1 << c_xo;
    }
    return c;
  }
  if (!taken || !(tbr < 1e6)) {  // the 1e6 constant won: no dependence
    c.ds = 0.0f;
    return c;
  }
  c.dtv = (float)p_tv;
  c.dte = (float)p_te;
  c.dtev = (float)p_tev;
  c.ds = (float)p_s;
  c.code = 1 << c_ref;
  return c;
}

// One workgroup per (strip rs, block of ADJ_CB reverse-local columns, shot):
// first each wave takes whole columns of the block in natural order, lane =
// row, so its loads of T and S are contiguous runs (a wave reading one step
// of the strip-skewed layout reads a diagonal instead: 64 cache lines per
// load, which bounded this kernel); the partials go to LDS by column, and
// then the workgroup writes the skewed entries (lane k, step t) whose node
// (64rs + k, t - k) lies in the block, each step a contiguous run of lanes.
// Entries outside the grid are left untouched.
constexpr int ADJ_CB = 32;

template <int SA, int SB>
__global__ __launch_bounds__(256) void k_adj_coef(const AdjShot* __restrict__ shots, int nzz, int nstr, ConstsD k,
                                                  const double* __restrict__ Tnew, const double* __restrict__ Told,
                                                  int pa, int pb, const float* __restrict__ lam_src,
                                                  float* __restrict__ lam_dst, float4* __restrict__ coef,
                                                  uint8_t* __restrict__ code) {
  __shared__ float P[4][ADJ_CB][64];
  __shared__ uint8_t Pc[ADJ_CB][64];
  const AdjShot sh = shots[blockIdx.y];
  const int nxx = sh.sd.nxx, NTP = sh.NTP;
  const int rs = (int)(blockIdx.x % (unsigned)nstr), jp0 = (int)(blockIdx.x / (unsigned)nstr) * ADJ_CB;
  if (jp0 >= nxx) return;  // whole workgroup: blocks past this shot's width
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int ip = 64 * rs + lane;
  const double* __restrict__ Tn = Tnew + sh.toff;
  for (int col = w; col < ADJ_CB; col += 4) {
    const int jp = jp0 + col;
    AdjCoef c{0.0f, 0.0f, 0.0f, -1.0f, 0};
    if (ip < nzz && jp < nxx) {
      const int i = adj_ip(ip, SA, nzz), j = adj_jp(jp, SB, nxx);  // (both maps are involutions)
      if (i >= 1 && i <= nzz - 2 && j >= 1 && j <= nxx - 2) {
        const double tv = Tn[(i - SA) + (size_t)j * nzz];
        const double te = Tn[i + (size_t)(j - SB) * nzz];
        const double tev = Tn[(i - SA) + (size_t)(j - SB) * nzz];
        const double told = Told[sh.toff + i + (size_t)j * nzz];
        const int i1 = i - (SA + 1) / 2, j1 = j - (SB + 1) / 2;
        const double sref = s_at(sh.sd, nzz, i1, j1);
        const double szo = s_at(sh.sd, nzz, i1, j1 + SB);
        const double sxo = s_at(sh.sd, nzz, i1 + SA, j1);
        c = adj_local<SA, SB>(tv, te, tev, sref, szo, sxo, told, k);
      }
    }
    P[0][col][lane] = c.dtv;
    P[1][col][lane] = c.dte;
    P[2][col][lane] = c.dtev;
    P[3][col][lane] = c.ds;
    Pc[col][lane] = (uint8_t)c.code;
  }
  __syncthreads();
  // step t = jp0 + e/64 of the skewed strip, lane e%64 (= this thread's lane)
  const size_t sbase = sh.koff + (size_t)rs * NTP * 64;
  for (int e = threadIdx.x; e < (ADJ_CB + 63) * 64; e += 256) {
    const int t = jp0 + (e >> 6), jp = t - lane, col = jp - jp0;
    if (col < 0 || col >= ADJ_CB || jp >= nxx || ip >= nzz) continue;
    const size_t ko = sbase + (size_t)t * 64 + lane;
    if (lam_src) {
      const int i = adj_ip(ip, SA, nzz), j = adj_jp(jp, SB, nxx);
      lam_dst[ko] = lam_src[sh.koff + adj_kidx(adj_ip(i, pa, nzz), adj_jp(j, pb, nxx), NTP)];
    }
    coef[ko] = make_float4(P[0][col][lane], P[1][col][lane], P[2][col][lane], P[3][col][lane]);
    code[ko] = Pc[col][lane];
  }
}

// ---------------------------------------------------------------------------
// Reverse sweep: one wave per strip of 64 reverse-local rows; lane k holds
// row 64r + k and visits column t - k at step t.  The z-upwind and diagonal
// messages come from lane k-1 (DPP shift), the x message from the lane's own
// previous step.  Lane 0's messages are the upper strip's lane-63 ones, which
// that strip publishes column by column as tagged words (word 2jp = the launch's
// tag and mv of column jp, word 2jp+1 the same for mev), written at its step
// jp+63 and read with the forward walker's protocol: one block load per
// ADJ_PF steps (lane u holds step u's words), one block ahead, and a bounded
// poll of the column while a tag is stale.  Strip 0 and the columns no strip
// publishes read zero messages.  Strips are claimed strip-major from the
// ticket counter ctl[0], so every upper neighbour is already running.  Inputs
// of ADJ_PF steps ahead are kept in flight; nodes outside the grid hold zero
// inputs and produce zero outputs.
__global__ __launch_bounds__(64) void k_adj_sweep(const AdjShot* __restrict__ shots, int nshots, int nstr,
                                                  const float* __restrict__ lam_in,
                                                  const float4* __restrict__ coef, float* __restrict__ lam_out,
                                                  float* __restrict__ gc, int* __restrict__ ctl,
                                                  unsigned long long* __restrict__ xw, int ldx, unsigned tag) {
  typedef __attribute__((address_space(1))) unsigned long long gword;
  const int lane = threadIdx.x;
  for (;;) {
    int tk = 0;
    if (lane == 0) tk = atomicAdd(ctl, 1);
    tk = __builtin_amdgcn_readfirstlane(tk);
    if (tk >= nshots * nstr) break;
    const int r = tk / nshots, ks = tk - r * nshots;
    const AdjShot sh = shots[ks];
    const int NTP = sh.NTP, nxx = sh.sd.nxx;
    const size_t base = sh.koff + (size_t)r * NTP * 64 + lane;
    gword* xme = (gword*)(xw + ((size_t)ks * nstr + r) * ldx);
    const gword* xup = (const gword*)(xw + ((size_t)ks * nstr + max(r - 1, 0)) * ldx);
    const bool up = r > 0;
    const bool pub = lane == 63 && r + 1 < nstr;
    float ql[ADJ_PF];
    float4 qc[ADJ_PF];
#pragma unroll
    for (int u = 0; u < ADJ_PF; ++u) {
      ql[u] = lam_in[base + (size_t)u * 64];
      qc[u] = coef[base + (size_t)u * 64];
    }
    // step t's words: mv of column t (word 2t) and mev of column t-1 (word
    // 2t-1), at clamped addresses (the step ignores the columns out of range)
    auto wv = [&](int t) { return xup + 2 * min(t, nxx - 1); };
    auto we = [&](int t) { return xup + max(2 * min(t, nxx) - 1, 0); };
    // unconditional (strip 0 reads its own words and ignores them)
    auto xload = [&](int tb, unsigned long long& v, unsigned long long& e) {
      const int t = tb + (lane & (ADJ_PF - 1));
      v = __hip_atomic_load(wv(t), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      e = __hip_atomic_load(we(t), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    float mv = 0.0f, me = 0.0f, mev = 0.0f, mevp = 0.0f;
    bool gave_up = false;
    auto block = [&](int t0, unsigned long long bv, unsigned long long be) {
#pragma unroll
      for (int u = 0; u < ADJ_PF; ++u) {
        const int t = t0 + u;
        float xv = 0.0f, xe = 0.0f;
        if (up) {
          const bool nv = t < nxx, ne = t >= 1 && t <= nxx;
          unsigned vw = __builtin_amdgcn_readlane((unsigned)bv, u);
          unsigned vt = __builtin_amdgcn_readlane((unsigned)(bv >> 32), u);
          unsigned ew = __builtin_amdgcn_readlane((unsigned)be, u);
          unsigned et = __builtin_amdgcn_readlane((unsigned)(be >> 32), u);
          for (int it = 0; !gave_up && ((nv && vt != tag) || (ne && et != tag)); ++it) {
            if (it > WALK_SPIN) {
              if (lane == 0) atomicOr(ctl + 1, 1);
              gave_up = true;
              break;
            }
            __builtin_amdgcn_s_sleep(1);
            const unsigned long long v = __hip_atomic_load(wv(t), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const unsigned long long e = __hip_atomic_load(we(t), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            vw = __builtin_amdgcn_readfirstlane((unsigned)v);
            vt = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
            ew = __builtin_amdgcn_readfirstlane((unsigned)e);
            et = __builtin_amdgcn_readfirstlane((unsigned)(e >> 32));
          }
          xv = nv ? __uint_as_float(vw) : 0.0f;
          xe = ne ? __uint_as_float(ew) : 0.0f;
        }
        // messages into (ip, jp): from (ip-1, jp) [lane k-1, step t-1],
        // (ip, jp-1) [own lane, step t-1], (ip-1, jp-1) [lane k-1, step t-2]
        const float in_v = dpp_shr1(xv, mv);
        const float in_ev = dpp_shr1(xe, mevp);
        const float mu = ((ql[u] + in_v) + me) + in_ev;
        mevp = mev;
        const float4 cf = qc[u];
        const bool upd = cf.w >= 0.0f;
        mv = upd ? mu * cf.x : 0.0f;
        me = upd ? mu * cf.y : 0.0f;
        mev = upd ? mu * cf.z : 0.0f;
        lam_out[base + (size_t)t * 64] = upd ? 0.0f : mu;
        gc[base + (size_t)t * 64] = upd ? mu * cf.w : 0.0f;
        const int jp = t - 63;
        if (pub && jp >= 0 && jp < nxx) {
          __hip_atomic_store(xme + 2 * jp, walk_word(__float_as_uint(mv), tag), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
          __hip_atomic_store(xme + 2 * jp + 1, walk_word(__float_as_uint(mev), tag), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
        }
        // reload the slot after its last use (it keeps its register)
        const int tn = min(t + ADJ_PF, NTP - 1);
        ql[u] = lam_in[base + (size_t)tn * 64];
        qc[u] = coef[base + (size_t)tn * 64];
      }
    };
    unsigned long long av, ae, bv, be;
    xload(0, av, ae);
    __builtin_amdgcn_s_waitcnt(0);  // once per strip (see k_fwd64_sweep)
    for (int t0 = 0; t0 < NTP; t0 += 2 * ADJ_PF) {
      xload(t0 + ADJ_PF, bv, be);
      block(t0, av, ae);
      if (t0 + ADJ_PF >= NTP) break;  // NTP is a multiple of ADJ_PF only
      xload(t0 + 2 * ADJ_PF, av, ae);
      block(t0 + ADJ_PF, bv, be);
    }
  }
}

// ---------------------------------------------------------------------------
// Slowness contributions of sweep s onto padded cell (i, j): the nodes
// (i + di, j + dj) whose code marks offset (di, dj), in a fixed order.  One
// workgroup per (strip rs, block of ADJ_CB reverse-local columns, shot) owns
// the cells whose nodes lie in the block: it first copies the block's
// entries, with one row and one column of halo on each side, from the
// strip-skewed layout into LDS by column (each step a contiguous run of
// lanes), then sums each cell's contributions from LDS, a wave per column
// with lane = row, so the cell updates are contiguous.
template <int SA, int SB>
__global__ __launch_bounds__(256) void k_adj_fold(const AdjShot* __restrict__ shots, int nzz, int nstr,
                                                  const float* __restrict__ gc, const uint8_t* __restrict__ code,
                                                  float* __restrict__ gshot) {
  constexpr int W = ADJ_CB + 2, H = 66;  // columns jp0-1 .. jp0+ADJ_CB, rows 64rs-1 .. 64rs+64
  __shared__ float G[W][H];
  __shared__ uint8_t C[W][H];
  const AdjShot sh = shots[blockIdx.y];
  const int nxx = sh.sd.nxx, NTP = sh.NTP;
  const int rs = (int)(blockIdx.x % (unsigned)nstr), jp0 = (int)(blockIdx.x / (unsigned)nstr) * ADJ_CB;
  if (jp0 >= nxx) return;  // whole workgroup: blocks past this shot's width
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int ip = 64 * rs + lane;
  // the strip's own rows: step t = jp0 - 1 + e/64, lane e%64
  const size_t sbase = sh.koff + (size_t)rs * NTP * 64;
  for (int e = threadIdx.x; e < (W + 63) * 64; e += 256) {
    const int t = jp0 - 1 + (e >> 6), jp = t - lane;
    if (jp < max(jp0 - 1, 0) || jp > jp0 + ADJ_CB || jp >= nxx || ip >= nzz) continue;
    const size_t ko = sbase + (size_t)t * 64 + lane;
    G[jp - jp0 + 1][lane + 1] = gc[ko];
    C[jp - jp0 + 1][lane + 1] = code[ko];
  }
  // halo rows: the last row of strip rs-1 and the first of strip rs+1
  if (threadIdx.x < 2 * W) {
    const int h = threadIdx.x / W, jp = jp0 - 1 + threadIdx.x % W;
    const int iph = h == 0 ? 64 * rs - 1 : 64 * rs + 64;
    if (iph >= 0 && iph < nzz && jp >= 0 && jp < nxx) {
      const size_t ko = sh.koff + adj_kidx(iph, jp, NTP);
      G[jp - jp0 + 1][h == 0 ? 0 : H - 1] = gc[ko];
      C[jp - jp0 + 1][h == 0 ? 0 : H - 1] = code[ko];
    }
  }
  __syncthreads();
  for (int col = w; col < ADJ_CB; col += 4) {
    const int jp = jp0 + col;
    if (ip >= nzz || jp >= nxx) continue;
    const int i = adj_ip(ip, SA, nzz), j = adj_jp(jp, SB, nxx);
    float acc = 0.0f;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int di = c & 1, dj = c >> 1;
      const int ni = i + di, nj = j + dj;
      if (ni >= 1 && ni <= nzz - 2 && nj >= 1 && nj <= nxx - 2) {
        // node (ni, nj) in reverse-local coordinates, within the LDS window
        const int r = adj_ip(ni, SA, nzz) - 64 * rs + 1, q = adj_jp(nj, SB, nxx) - jp0 + 1;
        const int m = C[q][r];
        if (m & (1 << c)) acc += (m & (m - 1)) ? 0.5f * G[q][r] : G[q][r];
      }
    }
    gshot[sh.toff + i + (size_t)j * nzz] += acc;
  }
}

// T0 = S(node) * distance on the source stencil: dT0/dS(node) = distance.
__global__ void k_adj_source(const AdjShot* __restrict__ shots, int nshots, int nzz, double dx, double dz,
                             const float* __restrict__ lam0, float* __restrict__ gshot) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nshots * 9) return;
  const AdjShot sh = shots[t / 9];
  const int ii = (t % 9) % 3, jj = (t % 9) / 3;
  const int sIdx = (int)(((double)sh.sd.sx + 0.5 * dx) / dx) + NB;
  const int sIdz = (int)(((double)sh.sd.sz + 0.5 * dz) / dz) + NB;
  const int zi = sIdz + (ii - 1), xi = sIdx + (jj - 1);
  const double ddx = (double)(xi - NB) * dx - (double)sh.sd.sx;
  const double ddz = (double)(zi - NB) * dz - (double)sh.sd.sz;
  const float lam = lam0[sh.koff + adj_kidx(adj_ip(zi, 1, nzz), adj_jp(xi, 1, sh.sd.nxx), sh.NTP)];
  gshot[sh.toff + zi + (size_t)xi * nzz] += lam * (float)sqrt(ddx * ddx + ddz * ddz);
}

// d/ds of the unpadded model: every padded node of every shot maps to the
// model cell it replicates (rows clamped to the model, columns clamped to the
// shot's window); sums in fp64, shots in order.  fixed_border: the model's
// border was uploaded as given (not the replication of its edges), so its
// rows, and the border columns of shots on the whole model, are constants
// with no derivative; a window's own replicated columns still fold.
__global__ __launch_bounds__(256) void k_adj_reduce(const AdjShot* __restrict__ shots, int nshots, int nz,
                                                    int nx, int nzz, const float* __restrict__ gshot,
                                                    double* __restrict__ grad, int fixed_border) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= nz * nx) return;
  const int iz = idx % nz, ix = idx / nz;
  const int plo = (iz == 0 && !fixed_border) ? 0 : iz + NB;
  const int phi = (iz == nz - 1 && !fixed_border) ? nz - 1 + 2 * NB : iz + NB;
  double acc = 0.0;
  for (int s = 0; s < nshots; ++s) {
    const int x0 = shots[s].sd.x0, w = shots[s].sd.w;
    if (ix < x0 || ix >= x0 + w) continue;
    const int lq = ix - x0;
    const bool cfix = fixed_border && shots[s].sd.sofs == 0;  // a whole-model shot reads the border as given
    const int qlo = (lq == 0 && !cfix) ? 0 : lq + NB;
    const int qhi = (lq == w - 1 && !cfix) ? w - 1 + 2 * NB : lq + NB;
    const float* __restrict__ g = gshot + shots[s].toff;
    for (int q = qlo; q <= qhi; ++q)
      for (int p = plo; p <= phi; ++p) acc += (double)g[p + (size_t)q * nzz];
  }
  grad[idx] = acc;
}

// ---------------------------------------------------------------------------
void launch_fill_d(double* p, size_t n, double v, hipStream_t st) {
  const int blocks = (int)std::min<size_t>((n + 255) / 256, 16384);
  hipLaunchKernelGGL(k_fill_d, dim3(blocks), dim3(256), 0, st, p, n, v);
}

void launch_adj_seed(const size_t* node, const int* ptr, const int* rec, const float* wt, int nseed,
                     const float* w, float* lam, hipStream_t st) {
  if (nseed <= 0) return;
  hipLaunchKernelGGL(k_adj_seed, dim3((nseed + 255) / 256), dim3(256), 0, st, node, ptr, rec, wt, nseed, w, lam);
}

static ConstsD consts_d(double dx, double dz) {
  ConstsD k;
  k.dx = dx;
  k.dz = dz;
  k.dz2i = 1.0 / (dz * dz);
  k.dx2i = 1.0 / (dx * dx);
  k.sum = k.dz2i + k.dx2i;
  k.sum4 = 4.0 * k.sum;
  k.prod = k.dz2i * k.dx2i;
  k.hyp = std::sqrt(dx * dx + dz * dz);
  k.r_dx = 1.0 / k.dx;
  k.r_dz = 1.0 / k.dz;
  k.r_sum = 1.0 / k.sum;
  k.r_hyp = 1.0 / k.hyp;
  return k;
}

void launch_fwd64_init(const AdjShot* shots, int nshots, int nzz, double dx, double dz, double* T0, hipStream_t st) {
  const int n = nshots * 9;
  hipLaunchKernelGGL(k_fwd64_init, dim3((n + 255) / 256), dim3(256), 0, st, shots, nshots, nzz, dx, dz, T0);
}

void launch_fwd64_sweep(int sweep, const AdjShot* shots, int nshots, int nzz, int nstr, double dx, double dz,
                        const SkewView& skew, const double* Told, double* Tnew, int* walk_ctl,
                        unsigned long long* walk_x, int ldx, unsigned tag, hipStream_t st) {
  const ConstsD k = consts_d(dx, dz);
  hipLaunchKernelGGL(k_walk_begin, dim3(1), dim3(64), 0, st, walk_ctl);
  // a workgroup per strip, at most what is resident at once (three per CU;
  // the tickets keep any count correct)
  const int grid = std::min(nshots * nstr, 768);
  auto* f = dx == dz ? (sweep == 0 ? k_fwd64_sweep<1, 1, true> : sweep == 1 ? k_fwd64_sweep<-1, 1, true>
                        : sweep == 2 ? k_fwd64_sweep<1, -1, true> : k_fwd64_sweep<-1, -1, true>)
                     : (sweep == 0 ? k_fwd64_sweep<1, 1, false> : sweep == 1 ? k_fwd64_sweep<-1, 1, false>
                        : sweep == 2 ? k_fwd64_sweep<1, -1, false> : k_fwd64_sweep<-1, -1, false>);
  hipLaunchKernelGGL(f, dim3(grid), dim3(256), 0, st, shots, nshots, nzz, nstr, k,
                     skew.KP <= 1 << 20 ? skew : SkewView{nullptr, 0},  // (a lane's byte offset in 32 bits)
                     Told, Tnew, walk_ctl, walk_x, ldx, tag);
}

void launch_picks64(const AdjShot* shots, const int* rec_shot, const float* rx, const float* rz, int nrec, int nzz,
                    double dx, double dz, const double* T4, double* out, hipStream_t st) {
  if (nrec <= 0) return;
  hipLaunchKernelGGL(k_picks64, dim3((nrec + 255) / 256), dim3(256), 0, st, shots, rec_shot, rx, rz, nrec, nzz, dx,
                     dz, T4, out);
}

void launch_adj_coef(int sweep, const AdjShot* shots, int nshots, int nstr, int max_nxx, int nzz, double dx,
                     double dz, const double* Tnew, const double* Told, const float* lam_src, float* lam_dst,
                     float4* coef, uint8_t* code, hipStream_t st) {
  const dim3 grid(nstr * ((max_nxx + ADJ_CB - 1) / ADJ_CB), nshots);
  const int pa = adj_a(sweep + 1), pb = adj_b(sweep + 1);
  const ConstsD k = consts_d(dx, dz);
  switch (sweep) {
    case 0: hipLaunchKernelGGL((k_adj_coef<1, 1>), grid, dim3(256), 0, st, shots, nzz, nstr, k, Tnew, Told, pa, pb, lam_src, lam_dst, coef, code); break;
    case 1: hipLaunchKernelGGL((k_adj_coef<-1, 1>), grid, dim3(256), 0, st, shots, nzz, nstr, k, Tnew, Told, pa, pb, lam_src, lam_dst, coef, code); break;
    case 2: hipLaunchKernelGGL((k_adj_coef<1, -1>), grid, dim3(256), 0, st, shots, nzz, nstr, k, Tnew, Told, pa, pb, lam_src, lam_dst, coef, code); break;
    default: hipLaunchKernelGGL((k_adj_coef<-1, -1>), grid, dim3(256), 0, st, shots, nzz, nstr, k, Tnew, Told, pa, pb, lam_src, lam_dst, coef, code); break;
  }
}

void launch_adj_sweep(const AdjShot* shots, int nshots, int nstr, const float* lam_in, const float4* coef,
                      float* lam_out, float* gc, int* walk_ctl, unsigned long long* walk_x, int ldx, unsigned tag,
                      hipStream_t st) {
  hipLaunchKernelGGL(k_walk_begin, dim3(1), dim3(64), 0, st, walk_ctl);
  const int grid = std::min(nshots * nstr, 4096);
  hipLaunchKernelGGL(k_adj_sweep, dim3(grid), dim3(64), 0, st, shots, nshots, nstr, lam_in, coef, lam_out, gc,
                     walk_ctl, walk_x, ldx, tag);
}

void launch_adj_fold(int sweep, const AdjShot* shots, int nshots, int nstr, int max_nxx, int nzz, const float* gc,
                     const uint8_t* code, float* gshot, hipStream_t st) {
  const dim3 grid(nstr * ((max_nxx + ADJ_CB - 1) / ADJ_CB), nshots);
  switch (sweep) {
    case 0: hipLaunchKernelGGL((k_adj_fold<1, 1>), grid, dim3(256), 0, st, shots, nzz, nstr, gc, code, gshot); break;
    case 1: hipLaunchKernelGGL((k_adj_fold<-1, 1>), grid, dim3(256), 0, st, shots, nzz, nstr, gc, code, gshot); break;
    case 2: hipLaunchKernelGGL((k_adj_fold<1, -1>), grid, dim3(256), 0, st, shots, nzz, nstr, gc, code, gshot); break;
    default: hipLaunchKernelGGL((k_adj_fold<-1, -1>), grid, dim3(256), 0, st, shots, nzz, nstr, gc, code, gshot); break;
  }
}

void launch_adj_source(const AdjShot* shots, int nshots, int nzz, double dx, double dz, const float* lam0,
                       float* gshot, hipStream_t st) {
  const int n = nshots * 9;
  hipLaunchKernelGGL(k_adj_source, dim3((n + 255) / 256), dim3(256), 0, st, shots, nshots, nzz, dx, dz, lam0,
                     gshot);
}

void launch_adj_reduce(const AdjShot* shots, int nshots, int nz, int nx, int nzz, const float* gshot,
                       double* grad, bool fixed_border, hipStream_t st) {
  const int n = nz * nx;
  hipLaunchKernelGGL(k_adj_reduce, dim3((n + 255) / 256), dim3(256), 0, st, shots, nshots, nz, nx, nzz, gshot,
                     grad, fixed_border ? 1 : 0);
}

}  // namespace seisfat
