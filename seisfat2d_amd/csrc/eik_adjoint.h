// Adjoint-state gradient of the single-pass eikonal solve: device layout and
// launchers (host side of eik_adjoint.hip).
//
// The forward solve is init + four directional sweeps; node (i, j) of sweep s
// becomes min(T_old, cand(tv, te, tev, S)) with tv, te, tev its upwind
// neighbours after sweep s.  The adjoint walks the sweeps backwards
// (k_adj_sweep): it re-derives the branch the forward took at every node and
// its local partials d(new)/d(tv, te, tev, S) from a recorded fp64 trajectory of
// the solve (k_fwd64_sweep), and runs the linear recurrence
//   mu(n) = lam_in(n) + sum over the three nodes m that read n of
//           mu(m) * d(new_m)/d(n)
// in reverse dependency order, one workgroup per 64-row strip.  k_adj_fold
// folds mu(n) * d(new_n)/dS onto the cells and adds the source initialisation's
// T0 = S(node) * distance; k_adj_reduce sums the shots in FP64 onto the unpadded
// model.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "eik_device.h"

namespace seisfat {

// A shot as the adjoint kernels see it.
struct AdjShot {
  ShotDev sd;   // final traveltimes (sd.T), slowness view, width, source, window
  size_t toff;  // offset of the shot's grid in every array below
};

// Forward sweep s runs rows in direction a and columns in direction b
// (s0 (+,+), s1 (-,+), s2 (+,-), s3 (-,-)).  Its adjoint processes
// "reverse-local" coordinates (ip, jp) in increasing order; a node reads the
// messages of (ip-1, jp), (ip, jp-1), (ip-1, jp-1).
__host__ __device__ inline int adj_a(int s) { return (s & 1) ? -1 : 1; }
__host__ __device__ inline int adj_b(int s) { return (s & 2) ? -1 : 1; }
__host__ __device__ inline int adj_ip(int i, int a, int nzz) { return a > 0 ? nzz - 1 - i : i; }
__host__ __device__ inline int adj_jp(int j, int b, int nxx) { return b > 0 ? nxx - 1 - j : j; }

// Pick seeds: lam[node[n]] = sum_{e in ptr[n]..ptr[n+1]} w[rec[e]] * wt[e].
void launch_adj_seed(const size_t* node, const int* ptr, const int* rec, const float* wt, int nseed,
                     const float* w, float* lam, hipStream_t st);
// fp64 trajectory: T0 stencil (T0 otherwise 1e6), and sweep s: Tnew = sweep(Told).
void launch_fill_d(double* p, size_t n, double v, hipStream_t st);
void launch_fwd64_init(const AdjShot* shots, int nshots, int nzz, double dx, double dz, double* T0, hipStream_t st);
// walk_ctl: 2 ints (ticket counter, reset by the launch; wait-limit flag);
// walk_x: nshots * nstr * ldx exchange words (ldx >= 2 * nxx); tag: a value
// no earlier launch on the same walk_x used
void launch_fwd64_sweep(int sweep, const AdjShot* shots, int nshots, int nzz, int nstr, double dx, double dz,
                        const SkewView& skew, const double* Told, double* Tnew, int* walk_ctl,
                        unsigned long long* walk_x, int ldx, unsigned tag, hipStream_t st);
// Picks of the fp64 trajectory's final traveltimes (rx, rz relative to each
// receiver's shot grid).
void launch_picks64(const AdjShot* shots, const int* rec_shot, const float* rx, const float* rz, int nrec, int nzz,
                    double dx, double dz, const double* T4, double* out, hipStream_t st);
// Reverse sweep s from the fp64 trajectory (Tnew = T after sweep s, Told =
// before): lam in place; g and code: every node's slowness contribution and the
// cells it goes to.  skew_opposite: the skewed slowness copy of the opposite
// orientation (sweep 3 - s).  walk_ctl, walk_x, tag as for the forward walk.
void launch_adj_sweep(int sweep, const AdjShot* shots, int nshots, int nzz, int nstr, double dx, double dz,
                      const SkewView& skew_opposite, const double* Tnew, const double* Told, float* lam, float* g,
                      uint8_t* code, int* walk_ctl, unsigned long long* walk_x, int ldx, unsigned tag,
                      hipStream_t st);
// Per-shot slowness gradient on padded cells from the four sweeps' g and code
// (sweep s at [s * tsize]) and lam after sweep 0.
void launch_adj_fold(const AdjShot* shots, int nshots, int max_nxx, int nzz, size_t tsize, double dx, double dz,
                     const float* g, const uint8_t* code, const float* lam, float* gshot, hipStream_t st);
// fixed_border: the model's border is not the replication of its edges (a
// padded upload), so only interior cells (and windows' replicated columns) fold
// edge: scratch, nshots x 2 (max_w + nz), each shot's sums over the cells its model edges replicate to
void launch_adj_reduce(const AdjShot* shots, int nshots, int nz, int nx, int nzz, int max_w, const float* gshot,
                       double* edge, double* grad, bool fixed_border, hipStream_t st);

}  // namespace seisfat
