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
// 1 / b for a normal b whose reciprocal is normal (the refined reciprocal of
// IEEE division) and, with it, RN(a / b).
__device__ __forceinline__ double recip_d(double b) {
  double y = __builtin_amdgcn_rcp(b);
  y = __builtin_fma(y, __builtin_fma(-b, y, 1.0), y);
  return __builtin_fma(y, __builtin_fma(-b, y, 1.0), y);
}

// Local partials of one node: (dT/dtv, dT/dte, dT/dtev, dT/dS), dT/dS < 0 at a
// node the sweep left unchanged (T_old kept: the adjoint passes through).  Bit
// (di | dj << 1) of code marks slowness cell (i - di, j - dj) as receiving
// dT/dS, split evenly when two bits are set.
struct AdjCoef {
  float4 c;
  unsigned code;
};

// The partials of the branch the fp64 forward took at an updated node with
// value tn (same expressions and comparisons as local_sel_d): a 1-D candidate
// when one equals tn, else the 2-D branch whose conditions hold.  Ties follow
// the oracle: 1-D before 2-D when equal; z-edge before x-edge when equal;
// min(S, S') of two equal cells splits dS half and half (what central
// differences measure).
template <int SA, int SB>
__device__ __forceinline__ AdjCoef adj_local(double tn, double tv, double te, double tev, double sref, double szo,
                                             double sxo, bool upd, const ConstsD& k) {
  constexpr int di_ref = (SA + 1) / 2, dj_ref = (SB + 1) / 2;
  constexpr unsigned c_ref = 1u << (di_ref | (dj_ref << 1));
  constexpr unsigned c_zo = 1u << (di_ref | (((1 - SB) / 2) << 1));
  constexpr unsigned c_xo = 1u << (((1 - SA) / 2) | (dj_ref << 1));
  const double t1d1 = tv + k.dz * vmin_d(sref, szo);
  const double t1d2 = te + k.dx * vmin_d(sref, sxo);
  const bool one = vmin_d(t1d1, t1d2) == tn, z = t1d1 <= t1d2;
  const double de = te - tev, dv = tv - tev;
  const bool cA = (tv <= te + k.dx * sref) & (te <= tv + k.dz * sref) & (de >= 0.0) & (dv >= 0.0);
  AdjCoef r{};
  if (__any(upd & !one & cA)) {
    // t = ((tb dz2i + ta dx2i) + sqrt(4 S^2 D - dz2i dx2i (ta - tb)^2)) / D
    const double dab = (tev + te - tv) - (tev - te + tv);
    const double sq = sqrt_rn_d(4.0 * sref * sref * k.sum - k.prod * dab * dab), y = recip_d(sq);
    const double ak = 2.0 * k.prod * dab, as = 4.0 * sref, qk = ak * y, qs = as * y;
    const double kk = __builtin_fma(__builtin_fma(-sq, qk, ak), y, qk);
    const double te_d = cdiv(k.dx2i - k.dz2i - kk, k.sum, k.r_sum);  // (dT/dtv is its opposite)
    r.c = make_float4((float)-te_d, (float)te_d, 1.0f, (float)__builtin_fma(__builtin_fma(-sq, qs, as), y, qs));
  }
  if (__any(upd & !one & !cA)) {
    const bool cB = (de <= cdiv(sref * k.dz * k.dz, k.hyp, k.r_hyp)) & (de > 0.0);
    // B: t = te + dx sqrt(S^2 - q^2), q = (te - tev) / dz; C: the same with the axes exchanged
    const double h1 = cB ? k.dz : k.dx, h2 = cB ? k.dx : k.dz;
    const double q = cdiv(cB ? de : dv, h1, cB ? k.r_dz : k.r_dx);
    const double Q = sqrt_rn_d(sref * sref - q * q);
    const double rr = h2 * q / (h1 * Q);
    const float p = (float)(1.0 - rr);
    if (!cA) r.c = make_float4(cB ? 0.0f : p, cB ? p : 0.0f, (float)rr, (float)(h2 * sref / Q));
  }
  r.code = c_ref;
  if (one) {
    const double other = z ? szo : sxo;
    const unsigned c_o = z ? c_zo : c_xo;
    r.code = sref == other ? c_ref | c_o : sref < other ? c_ref : c_o;
    r.c = make_float4(z ? 1.0f : 0.0f, z ? 0.0f : 1.0f, 0.0f, (float)(z ? k.dz : k.dx));
  }
  if (!upd) {
    r.c = make_float4(0.0f, 0.0f, 0.0f, -1.0f);
    r.code = 0;
  }
  return r;
}

// One reverse sweep: mu(n) = lam(n) + sum over the three nodes m that read n of
// mu(m) d(new_m)/d(n), in reverse dependency order; a node the sweep updated
// passes mu on through its partials and leaves 0 in lam, another keeps mu
// there; g and code get mu dT/dS and the cells it goes to.  A workgroup walks
// one strip of 64 reverse-local rows of one shot; step t holds row 64r + k at
// column t - k, as the forward walk's.  Wave 0 runs the recurrence from LDS
// (messages from lane k-1 by DPP, from its own previous step, and lane 0's from
// the upper strip); wave 1 brings whole columns of lam, wave 2 those of the
// traveltimes before and after the sweep, whose difference marks the nodes it
// updated (the sign of the word); waves 4 and 5 store the finished columns of
// lam, g and code; waves 6 to 13 evaluate the partials of a step of a block
// each, one block ahead, and skip the steps no node of which was updated; wave 3
// exchanges the last row's messages with the neighbouring strips (tagged words as
// in the forward walk, bounded polls) and brings the row of traveltimes below
// the strip.  The columns pass through skewed LDS rings ([step][lane], see k_fwd64_sweep), so
// nothing skewed is stored: 16 B of traveltimes read, 8 B of lam, 5 B of g and
// code per node.  The chain of a strip's steps is the bound while the strips are
// fewer than the CUs, the partials' FP64 instructions beyond: one strip of
// 58 x 1201 123 us a sweep, 301 x 1201 163 with 1 shot, 230 with 50 and 525 with
// 128 (640 strips); as three kernels (partials, recurrence, contributions to the
// cells, through skewed arrays of 37 B per node) it was 1.5 ms with 128.  Loads
// and stores are kept in separate waves: with both in one, its loads wait for the
// acknowledgement of its stores (730 us with 128 shots against 614).  8 waves for
// the partials against 4: 123 / 163 / 230 / 525 against 155 / 201 / 258 / 557;
// blocks of 16 steps with 4 waves 150 / 195 / 242 / 514; two workgroups a CU
// (blocks of 4 steps) 621 with 128.
constexpr int AB = 8;               // steps per block
constexpr int AT = 64 + 3 * AB;     // ring steps.  Traveltimes: a step's columns, two blocks' lead (and one to
                                    // round up); lam (the node's result replaces it): a block arriving, one leaving
constexpr int ADJ_OUT = 2, ADJ_COEF = 8;    // waves that store and that evaluate partials
constexpr int ADJ_THREADS = 64 * (4 + ADJ_OUT + ADJ_COEF);
constexpr unsigned ADJ_UPD = 0x80;  // in the ring of codes: the node was updated

// x mod n for 0 <= x < 2n
__device__ __forceinline__ unsigned wrap(unsigned x, unsigned n) { return min(x, x - n); }

template <int SA, int SB>
__global__ __launch_bounds__(ADJ_THREADS) void k_adj_sweep(const AdjShot* __restrict__ shots, int nshots, int nzz, int nstr,
                                                  ConstsD K, SkewView sk, const double* __restrict__ Tnew,
                                                  const double* __restrict__ Told, float* __restrict__ lam,
                                                  float* __restrict__ g, uint8_t* __restrict__ code,
                                                  int* __restrict__ ctl, unsigned long long* __restrict__ xw, int ldx,
                                                  unsigned tag) {
  typedef __attribute__((address_space(1))) unsigned long long gword;
  __shared__ double ringT[AT * 65];
  __shared__ float ringV[AT * 64];
  __shared__ uint8_t ringC[AT * 64];
  __shared__ float4 cf[2][AB][64];
  __shared__ float2 xin[2][AB];            // upper strip's messages (to the row below, to the diagonal)
  __shared__ float2 pub[2][AB][2];         // this strip's last row's (second word: the other lanes' dummy)
  __shared__ int ticket;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  for (;;) {
    if (threadIdx.x == 0) ticket = atomicAdd(ctl, 1);
    __syncthreads();
    const int tk = __builtin_amdgcn_readfirstlane(ticket);
    if (tk >= nshots * nstr) break;
    const int r = tk / nshots, ks = tk - r * nshots;
    const AdjShot sh = shots[ks];
    const int nxx = sh.sd.nxx;
    const int NBLK = (nxx + 63 + AB - 1) / AB;
    const int ip = 64 * r + lane;
    const int ipc = min(ip, nzz - 1);
    const int i = adj_ip(ipc, SA, nzz);
    // column jp, clamped to the grid (its first and last columns are ring nodes,
    // which no sweep updates), and the step from it to the next
    const auto col = [&](int jp) { return (size_t)adj_jp(min(max(jp, 0), nxx - 1), SB, nxx) * nzz; };
    const auto next = [&](int jp) { return jp >= 0 && jp + 1 < nxx ? (SB > 0 ? -nzz : nzz) : 0; };
    // block n: wave 0 takes steps 8n .. 8n + 7 (for 0 <= n < NBLK)
    const int n_first = -3, n_last = NBLK + 1;
    if (wave == 0) {
      float mv = 0.0f, me = 0.0f, mev = 0.0f, mevp = 0.0f;
      for (int n = n_first; n <= n_last; ++n) {
        if (n >= 0 && n < NBLK) {
          const int buf = n & 1;
          float* __restrict__ rv = ringV + (n * AB % AT) * 64 + lane;
          float2* __restrict__ pb = &pub[buf][0][lane == 63 ? 0 : 1];
          unsigned zero = 0;
          asm volatile("" : "+v"(zero));  // (one address register for the block's broadcasts)
          float ql = rv[0];
          float4 c = cf[buf][0][lane];
          float2 x = xin[buf][zero];
#pragma unroll
          for (int u = 0; u < AB; ++u) {
            const float qu = ql;
            const float4 cu = c;
            const float2 xu = x;
            if (u + 1 < AB) {  // a step's operands are read one step ahead
              ql = rv[64 * (u + 1)];
              c = cf[buf][u + 1][lane];
              x = xin[buf][zero + u + 1];
            }
            // messages into (ip, jp): from (ip-1, jp) [lane k-1, step t-1],
            // (ip, jp-1) [own lane, step t-1], (ip-1, jp-1) [lane k-1, step t-2]
            const float mu = ((qu + dpp_shr1(xu.x, mv)) + me) + dpp_shr1(xu.y, mevp);
            mevp = mev;
            const bool upd = cu.w >= 0.0f;
            mv = upd ? mu * cu.x : 0.0f;
            me = upd ? mu * cu.y : 0.0f;
            mev = upd ? mu * cu.z : 0.0f;
            rv[64 * u] = upd ? mu * cu.w : mu;
            pb[2 * u] = make_float2(mv, mev);
          }
        }
        lds_barrier();
      }
    } else if (wave == 1) {
      // lam of columns 8n + 8 .. 8n + 15
      const float* __restrict__ L = lam + sh.toff + col(0);  // the next column to load
      int jl = 0;
      const auto load = [&](float (&q)[AB]) {
#pragma unroll
        for (int u = 0; u < AB; ++u) {
          q[u] = L[(unsigned)i];
          L += next(jl++);
        }
      };
      float qa[AB], qb[AB];
      load(qa);
      load(qb);
      const auto move = [&](int n, float (&q)[AB]) {
        const int c_in = (n + 1) * AB;
        if (c_in < 0) return;
        const unsigned c = (unsigned)(c_in % AT) + lane;
#pragma unroll
        for (int u = 0; u < AB; ++u) ringV[wrap(c + u, AT) * 64 + lane] = q[u];
        load(q);
      };
      for (int n = n_first; n <= n_last; n += 2) {
        move(n, qa);
        lds_barrier();
        if (n + 1 <= n_last) {
          move(n + 1, qb);
          lds_barrier();
        }
      }
    } else if (wave == 2) {
      // traveltimes of columns 8n + 17 .. 8n + 24
      const double* __restrict__ Tn = Tnew + sh.toff;
      const double* __restrict__ To = Told + sh.toff;
      int jl = (n_first + 2) * AB + 1;
      const double* __restrict__ pn = Tn + col(jl);  // the next column to load
      const double* __restrict__ po = To + col(jl);
      const auto load = [&](double (&a)[AB], double (&b)[AB]) {
#pragma unroll
        for (int u = 0; u < AB; ++u) {
          a[u] = pn[(unsigned)i];
          b[u] = po[(unsigned)i];
          const int d = next(jl++);
          pn += d;
          po += d;
        }
      };
      double qa[2][AB], qb[2][AB];
      load(qa[0], qa[1]);
      load(qb[0], qb[1]);
      const auto move = [&](int n, double (&q)[2][AB]) {
        const int c_in = (n + 2) * AB + 1;
        const unsigned c = (unsigned)((c_in + AT) % AT) + lane;
#pragma unroll
        for (int u = 0; u < AB; ++u)
          ringT[wrap(c + u, AT) * 65 + lane] = __longlong_as_double(
              __double_as_longlong(q[0][u]) | (q[0][u] < q[1][u] ? (long long)0x8000000000000000ull : 0));
        load(q[0], q[1]);
      };
      for (int n = n_first; n <= n_last; n += 2) {
        move(n, qa);
        lds_barrier();
        if (n + 1 <= n_last) {
          move(n + 1, qb);
          lds_barrier();
        }
      }
    } else if (wave == 3) {
      gword* xme = (gword*)(xw + ((size_t)ks * nstr + r) * ldx);
      const gword* xup = (const gword*)(xw + ((size_t)ks * nstr + max(r - 1, 0)) * ldx);
      const double* __restrict__ Tb = Tnew + sh.toff + adj_ip(min(64 * r + 64, nzz - 1), SA, nzz);
      const int u = lane & (AB - 1);
      bool gave_up = false;
      double below = Tb[col((n_first + 2) * AB + 1 + u)];
      for (int n = n_first; n <= n_last; ++n) {
        // publish block n - 1's last row: column 8(n - 1) + u - 63
        if (n >= 1 && n <= NBLK && r + 1 < nstr) {
          const int jp = (n - 1) * AB + u - 63;
          const float2 m = pub[(n - 1) & 1][u][0];
          if (lane < AB && jp >= 0 && jp < nxx) {
            __hip_atomic_store(xme + 2 * jp, walk_word(__float_as_uint(m.x), tag), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(xme + 2 * jp + 1, walk_word(__float_as_uint(m.y), tag), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
          }
        }
        // the upper strip's messages of step t = 8(n + 1) + u: to the row below
        // of column t (word 2t), to the diagonal of column t - 1 (word 2t - 1);
        // strip 0 and the columns no strip publishes read zero
        const int t = (n + 1) * AB + u;
        float2 x = make_float2(0.0f, 0.0f);
        if (r > 0 && n >= -1 && n + 1 < NBLK) {
          const bool nv = t < nxx, ne = t >= 1 && t <= nxx;
          const gword* pv = xup + 2 * min(t, nxx - 1);
          const gword* pe = xup + max(2 * min(t, nxx) - 1, 0);
          for (int it = 0;; ++it) {
            const unsigned long long v = __hip_atomic_load(pv, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const unsigned long long e = __hip_atomic_load(pe, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            x = make_float2(nv ? __uint_as_float((unsigned)v) : 0.0f, ne ? __uint_as_float((unsigned)e) : 0.0f);
            if (gave_up ||
                __all((!nv || (unsigned)(v >> 32) == tag) && (!ne || (unsigned)(e >> 32) == tag)))
              break;
            if (it > WALK_SPIN) {
              if (lane == 0) atomicOr(ctl + 1, 1);
              gave_up = true;
              break;
            }
            __builtin_amdgcn_s_sleep(1);
          }
        }
        if (lane < AB) {
          xin[(n + 1) & 1][u] = x;
          const int jp = (n + 2) * AB + 1 + u;
          if (jp >= 0) ringT[wrap((unsigned)(jp % AT + 64), AT) * 65 + 64] = below;
        }
        below = Tb[col((n + 3) * AB + 1 + u)];
        lds_barrier();
      }
    } else if (wave < 4 + ADJ_OUT) {
      // the block of columns whose last node block n - 1 took (8n - 72 .. 8n - 65) leaves (these
      // waves load nothing from memory, so they never wait for a store)
      constexpr int C = AB / ADJ_OUT;
      const int u0 = (wave - 4) * C;
      const bool row = ip < nzz;
      for (int n = n_first; n <= n_last; ++n) {
        const int c_out = (n - 1) * AB - 64 + u0;
        if (c_out + C > 0 && c_out < nxx) {
          float v[C];
          unsigned cd[C];
          const unsigned c = (unsigned)((c_out + AT) % AT) + lane;
#pragma unroll
          for (int u = 0; u < C; ++u) {
            const unsigned o = wrap(c + u, AT) * 64 + lane;
            v[u] = ringV[o];
            cd[u] = ringC[o];
          }
          const size_t o = sh.toff + col(c_out);
          float* __restrict__ L = lam + o;
          float* __restrict__ G = g + o;
          uint8_t* __restrict__ Cd = code + o;
          if (row) {
#pragma unroll
            for (int u = 0; u < C; ++u) {
              if (c_out + u >= 0 && c_out + u < nxx) {
                const bool upd = (cd[u] & ADJ_UPD) != 0;
                L[(unsigned)i] = upd ? 0.0f : v[u];
                G[(unsigned)i] = upd ? v[u] : 0.0f;
                Cd[(unsigned)i] = (uint8_t)(cd[u] & 15u);
              }
              const int d = next(c_out + u);
              L += d;
              G += d;
              Cd += d;
            }
          }
        }
        lds_barrier();
      }
    } else {
      // slowness of step t: the reference cell of (ip, jp) is cell row ip of the
      // opposite orientation, so step t's are consecutive in its skewed copy
      // (column sig); the z-other cell is the previous step's; the x-other cell
      // lane k-1's previous step's (lane 0: the upper strip's last row, 63 steps on).
      // Where a column is clamped, by s_at.
      constexpr int C = AB / ADJ_COEF;
      const int u0 = (wave - 4 - ADJ_OUT) * C;
      const int pitch = (SB > 0 ? -1 : 1) * sk.KP;  // words from one step's column to the next's
      const unsigned rowk = (unsigned)min(64 * r + lane, sk.KP - 1);
      // the x-other cell relative to the lowest of the lanes' columns
      const int lead = lane == 0 && r > 0 ? 64 : 0;
      const unsigned up_off = rowk - (lane == 0 && r == 0 ? 0u : 1u) + (unsigned)((SB > 0 ? 64 - lead : lead) * sk.KP);
      const int i1 = i - (SA + 1) / 2;
      typedef __attribute__((address_space(1))) const float cfloat;
      // step u0's column (the pointers advance a block at a time)
      cfloat* bp = (cfloat*)sk.base + (long long)(sh.sd.x0 + (SB > 0 ? nxx - 2 + 63 : 0) + SK_OFF) * sk.KP + (long long)u0 * pitch;
      const int jbase = (SB > 0 ? nxx - 2 : 0) - sh.sd.sofs;
      float sr[C], sz[C], sx[C];
      const auto load = [&](int v, int t) {
        // columns t - 64 .. t unclamped
        if (sk.base && (SB > 0 ? jbase - t >= 0 && jbase - t + 64 <= sh.sd.smax
                               : jbase + t - 64 >= 0 && jbase + t <= sh.sd.smax)) {
          cfloat* b = bp + (long long)v * pitch;
          cfloat* z = b - pitch;
          sr[v] = b[rowk];
          sz[v] = z[rowk];
          sx[v] = (SB > 0 ? z + 64 * (long long)pitch : z)[up_off];
        } else {
          const int jp = min(max(t - lane, 1), nxx - 2);
          const int j1 = adj_jp(jp, SB, nxx) - (SB + 1) / 2;
          const int i1c = min(max(i1, 0), nzz - 1), i2c = min(max(i1 + SA, 0), nzz - 1);
          sr[v] = s_at(sh.sd, nzz, i1c, j1);
          sz[v] = s_at(sh.sd, nzz, i1c, j1 + SB);
          sx[v] = s_at(sh.sd, nzz, i2c, j1);
        }
      };
#pragma unroll
      for (int v = 0; v < C; ++v) load(v, u0 + v);
      for (int n = n_first; n <= n_last; ++n) {
        if (n >= -1 && n + 1 < NBLK) {
          bp += AB * (long long)pitch;
#pragma unroll
          for (int v = 0; v < C; ++v) {
            const int t = (n + 1) * AB + u0 + v;
            const double sref = (double)sr[v], szo = (double)sz[v], sxo = (double)sx[v];
            const unsigned o0 = (unsigned)(t % AT), o1 = wrap(o0 + 1, AT), o2 = wrap(o0 + 2, AT);
            const double tn = ringT[o0 * 65 + lane], te = ringT[o1 * 65 + lane], tv = ringT[o1 * 65 + lane + 1],
                         tev = ringT[o2 * 65 + lane + 1];
            // (a column before the grid holds another step's or nothing)
            const bool upd = t >= lane && __double2hiint(tn) < 0;
            AdjCoef a{make_float4(0.0f, 0.0f, 0.0f, -1.0f), 0};
            if (__any(upd)) {
              a = adj_local<SA, SB>(fabs(tn), fabs(tv), fabs(te), fabs(tev), sref, szo, sxo, upd, K);
              if (upd) a.code |= ADJ_UPD;
            }
            load(v, t + AB);
            cf[(n + 1) & 1][u0 + v][lane] = a.c;
            ringC[o0 * 64 + lane] = (uint8_t)a.code;
          }
        }
        lds_barrier();
      }
    }
  }
}

// Per-shot slowness gradient on padded cells: cell (i, j) receives, sweep 3
// first, the contributions g of the nodes (i + di, j + dj) whose code marks
// offset (di, dj), in a fixed order, then the source initialisation's (T0 =
// S(node) * distance on the source stencil).  A wave takes 64 rows of ADJ_FC
// consecutive columns, so a node column is read once for the two cell columns
// it contributes to, and adds all four sweeps in one pass: 0.29 ms for 128 shots
// of 301 x 1201 (28 B per node), against 4 x 0.30 with a pass per sweep.
constexpr int ADJ_FC = 8;

__global__ __launch_bounds__(256) void k_adj_fold(const AdjShot* __restrict__ shots, int nzz, size_t tsize, double dx,
                                                  double dz, const float* __restrict__ g,
                                                  const uint8_t* __restrict__ code, const float* __restrict__ lam,
                                                  float* __restrict__ gshot) {
  const AdjShot sh = shots[blockIdx.z];
  const int nxx = sh.sd.nxx;
  const int i = blockIdx.x * 64 + (threadIdx.x & 63);
  const int j0 = (blockIdx.y * 4 + (threadIdx.x >> 6)) * ADJ_FC;
  if (j0 >= nxx || i >= nzz) return;
  const bool r0 = i >= 1 && i <= nzz - 2, r1 = i + 1 <= nzz - 2;  // rows i, i + 1 interior
  const size_t row1 = i + 1 < nzz ? 1 : 0;
  // the previous node column's contributions to this cell column: nodes (i, j)
  // and (i + 1, j), per sweep
  float pa[4], pb[4];
  const int sIdx = (int)(((double)sh.sd.sx + 0.5 * dx) / dx) + NB;
  const int sIdz = (int)(((double)sh.sd.sz + 0.5 * dz) / dz) + NB;
#pragma unroll
  for (int q = 0; q <= ADJ_FC; ++q) {
    const int nj = j0 + q;
    const bool in = nj >= 1 && nj <= nxx - 2;
    float ga[4], gb[4];
    unsigned ma[4], mb[4];
    const size_t o = sh.toff + i + (size_t)min(nj, nxx - 1) * nzz;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      ga[s] = g[s * tsize + o];
      gb[s] = g[s * tsize + o + row1];
      ma[s] = code[s * tsize + o];
      mb[s] = code[s * tsize + o + row1];
    }
    float sum = 0.0f;
#pragma unroll
    for (int s = 3; s >= 0; --s) {
      const unsigned a = in && r0 ? ma[s] : 0u, b = in && r1 ? mb[s] : 0u;
      const float fa = (a & (a - 1)) ? 0.5f * ga[s] : ga[s], fb = (b & (b - 1)) ? 0.5f * gb[s] : gb[s];
      if (q > 0) {
        float acc = pa[s] + pb[s];
        acc += (a & 4u) ? fa : 0.0f;
        acc += (b & 8u) ? fb : 0.0f;
        sum += acc;
      }
      pa[s] = (a & 1u) ? fa : 0.0f;
      pb[s] = (b & 2u) ? fb : 0.0f;
    }
    const int j = nj - 1;  // the cell column that is complete
    if (q > 0 && j < nxx) {
      const size_t c = sh.toff + i + (size_t)j * nzz;
      if (abs(i - sIdz) <= 1 && abs(j - sIdx) <= 1) {
        const double ddx = (double)(j - NB) * dx - (double)sh.sd.sx;
        const double ddz = (double)(i - NB) * dz - (double)sh.sd.sz;
        sum += lam[c] * (float)sqrt(ddx * ddx + ddz * ddz);
      }
      gshot[c] = sum;
    }
  }
}

// d/ds of the unpadded model: every padded cell of every shot maps to the
// model cell it replicates (rows clamped to the model, columns clamped to the
// shot's window); sums in fp64, shots in order.  fixed_border: the model's
// border was uploaded as given (not the replication of its edges), so its
// rows, and the border columns of shots on the whole model, are constants
// with no derivative; a window's own replicated columns still fold.
//
// A cell on an edge takes 4 padded cells of each shot and a corner 16, one
// away from the edges a single one; with a loop over them in the cell's own thread,
// no two shots' loads are in flight together.  So k_adj_border first sums each
// shot's edge cells, and k_adj_reduce adds one value a shot and cell, those of
// ADJ_RS shots loaded together (128 shots of 301 x 1201: 0.42 ms in one kernel, 0.027 + 0.095 now).
// edge: [shot][row 0: w][row nz-1: w][column 0: nz][column w-1: nz]; where the
// rows have a border, their corners are read from the rows' part.
constexpr int ADJ_RS = 16;

struct EdgeRange {
  int lo, hi;  // padded indices of the cells that map to cell c of n
};
__device__ __forceinline__ EdgeRange edge_range(int c, int n, bool fixed) {
  return {c == 0 && !fixed ? 0 : c + NB, c == n - 1 && !fixed ? n - 1 + 2 * NB : c + NB};
}

__global__ __launch_bounds__(256) void k_adj_border(const AdjShot* __restrict__ shots, int nz, int nzz,
                                                    const float* __restrict__ gshot, double* __restrict__ edge,
                                                    int pitch, int fixed_border) {
  const AdjShot& sh = shots[blockIdx.y];
  const int w = sh.sd.w, e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= 2 * (w + nz)) return;
  const bool cfix = fixed_border && sh.sd.sofs == 0;  // a whole-model shot reads the border as given
  const int c = e < 2 * w ? e : e - 2 * w;
  const int iz = e < 2 * w ? (c < w ? 0 : nz - 1) : c < nz ? c : c - nz;
  const int lq = e < 2 * w ? (c < w ? c : c - w) : c < nz ? 0 : w - 1;
  const EdgeRange p = edge_range(iz, nz, fixed_border), q = edge_range(lq, w, cfix);
  const float* __restrict__ gs = gshot + sh.toff;
  double acc = 0.0;
  for (int j = q.lo; j <= q.hi; ++j)
    for (int i = p.lo; i <= p.hi; ++i) acc += (double)gs[i + (size_t)j * nzz];
  edge[(size_t)blockIdx.y * pitch + e] = acc;
}

__global__ __launch_bounds__(256) void k_adj_reduce(const AdjShot* __restrict__ shots, int nshots, int nz,
                                                    int nx, int nzz, const float* __restrict__ gshot,
                                                    const double* __restrict__ edge, int pitch,
                                                    double* __restrict__ grad, int fixed_border) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= nz * nx) return;
  const int iz = idx % nz, ix = idx / nz;
  const bool redge = !fixed_border && (iz == 0 || iz == nz - 1);
  double acc = 0.0;
  for (int s0 = 0; s0 < nshots; s0 += ADJ_RS) {
    double v[ADJ_RS];
#pragma unroll
    for (int u = 0; u < ADJ_RS; ++u) {
      const int s = min(s0 + u, nshots - 1);
      const AdjShot& sh = shots[s];
      const int lq = ix - sh.sd.x0, w = sh.sd.w;
      const bool in = s0 + u < nshots && lq >= 0 && lq < w;
      const bool cedge = (lq == 0 || lq == w - 1) && !(fixed_border && sh.sd.sofs == 0);
      v[u] = (gshot + sh.toff)[(unsigned)(iz + NB) + (unsigned)(min(max(lq, 0), w - 1) + NB) * (unsigned)nzz];
      if (in && (redge || cedge))
        v[u] = edge[(size_t)s * pitch + (redge ? (iz == 0 ? 0 : w) + lq : 2 * w + (lq == 0 ? 0 : nz) + iz)];
      if (!in) v[u] = 0.0;
    }
#pragma unroll
    for (int u = 0; u < ADJ_RS; ++u) acc += v[u];
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

void launch_adj_sweep(int sweep, const AdjShot* shots, int nshots, int nzz, int nstr, double dx, double dz,
                      const SkewView& skew_opposite, const double* Tnew, const double* Told, float* lam, float* g,
                      uint8_t* code, int* walk_ctl, unsigned long long* walk_x, int ldx, unsigned tag,
                      hipStream_t st) {
  const ConstsD k = consts_d(dx, dz);
  hipLaunchKernelGGL(k_walk_begin, dim3(1), dim3(64), 0, st, walk_ctl);
  const int grid = std::min(nshots * nstr, 256);  // one workgroup per CU (LDS)
  auto* f = sweep == 0 ? k_adj_sweep<1, 1> : sweep == 1 ? k_adj_sweep<-1, 1> : sweep == 2 ? k_adj_sweep<1, -1>
                                                                                        : k_adj_sweep<-1, -1>;
  hipLaunchKernelGGL(f, dim3(grid), dim3(ADJ_THREADS), 0, st, shots, nshots, nzz, nstr, k, skew_opposite, Tnew, Told, lam, g,
                     code, walk_ctl, walk_x, ldx, tag);
}

void launch_adj_fold(const AdjShot* shots, int nshots, int max_nxx, int nzz, size_t tsize, double dx, double dz,
                     const float* g, const uint8_t* code, const float* lam, float* gshot, hipStream_t st) {
  const dim3 grid((nzz + 63) / 64, (max_nxx + 4 * ADJ_FC - 1) / (4 * ADJ_FC), nshots);
  hipLaunchKernelGGL(k_adj_fold, grid, dim3(256), 0, st, shots, nzz, tsize, dx, dz, g, code, lam, gshot);
}

void launch_adj_reduce(const AdjShot* shots, int nshots, int nz, int nx, int nzz, int max_w, const float* gshot,
                       double* edge, double* grad, bool fixed_border, hipStream_t st) {
  const int n = nz * nx, pitch = 2 * (max_w + nz);
  const dim3 grid((pitch + 255) / 256, nshots);
  hipLaunchKernelGGL(k_adj_border, grid, dim3(256), 0, st, shots, nz, nzz, gshot, edge, pitch, fixed_border ? 1 : 0);
  hipLaunchKernelGGL(k_adj_reduce, dim3((n + 255) / 256), dim3(256), 0, st, shots, nshots, nz, nx, nzz, gshot,
                     edge, pitch, grad, fixed_border ? 1 : 0);
}

}  // namespace seisfat
