// Ionosphere (MI) coupling on the device: field-aligned current on the sample
// shell, its samples on the two polar grids, the potential solve, and the
// view of the potential that the step kernels read
// (cubedsphere/cubedsphere_mi_dipole.c:157-436, NO/nonorthogonal_mi.c).
//
// Geometry-only parts (donor faces and bilinear weights of the shell fringe
// and of every polar sample point, the sample-shell radius) are computed once
// on the host with the C library, exactly as the reference computes them on
// every update. The per-update work is five kernels plus the solve.
//
// Solvers. The Pedersen-only potential uses the reference's algorithm:
// Jacobi-preconditioned CG on the reduced sin(theta)-weighted system with
// true-residual checks (NO/nonorthogonal_mi.c:412-609). With a Hall
// conductance the operator is the reference's five-point tensor stencil
// solved by right-preconditioned BiCGStab (:959-1151); the reference's
// preconditioner is a symmetric Gauss-Seidel sweep, which is sequential over
// all unknowns, so here each colatitude ring is solved exactly instead (a
// periodic tridiagonal solve of the ring's longitude coupling). Dot products
// are reductions in a fixed order; the iterates therefore differ from the
// reference's by rounding, and the converged potential agrees with it to the
// solve's tolerance. Both hemispheres run in the same launches. The solves
// keep their vectors in registers, one wavefront per ring (k_ring_cg,
// k_ring_bicgstab). Where their workgroups cannot all be resident, a fixed
// number of workgroups solves the tensor system (k_mi_bicgstab_pair) and one
// workgroup per hemisphere the Pedersen one (k_mi_cg); without cooperative
// launches one workgroup per hemisphere solves either (k_mi_bicgstab).
#include <hip/hip_cooperative_groups.h>
#include <hip/hip_runtime.h>

#include <cfloat>
#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <random>
#include <vector>

#include "gcs_device.hpp"
#include "gcs_math.hpp"
#include "gcs_unet.hpp"

namespace gcs {

namespace {

constexpr int kT = 256;

// value = (1-wx) [(1-wy) v[b] + wy v[b+1]] + wx [(1-wy) v[b+s] + wy v[b+s+1]]
// (cubedsphere_mi_dipole.c:326-331, :361-366)
struct Bilinear {
  int target, base, step, zero;
  double wx, wy;
};

enum Slot {  // what a solve leaves per hemisphere
  SL_ITER, SL_OK, SL_NORM, SL_FIRST,
  SL_GAVE_UP,  // a workgroup of k_ring_cg or k_ring_bicgstab gave up a wait
  SL_COUNT
};

}  // namespace

struct MiState {
  gamera_cs_mi_dipole_config cfg;
  double hall = 0.0;
  int np = 0, nt = 0, n = 0, S = 0, si = 0;
  double sample_radius = 0.0, sample_max_colat = 0.0, max_colat = 0.0;
  double b_norm = 0.0, current_norm = 0.0, potential_norm = 0.0;
  double next_update = 0.0, epoch = 0.0;
  bool ready = false;
  int updates = 0;
  int iterations[2] = {0, 0};
  double initial_residual[2] = {0.0, 0.0};
  double final_residual[2] = {0.0, 0.0};
  int converged[2] = {0, 0};
  double solve_ms = 0.0;
  // device arrays
  double *shell_fac = nullptr;  // [6][S][S]
  // J.b0/|b0| (A/m^2, before the dipole mapping), magnetic latitude and
  // longitude (degrees) of the active sample-shell cells at the last update,
  // [3][6][n][n]
  double *shell_current = nullptr;
  double *fac = nullptr;        // [2][nt][np]
  double *potential = nullptr;  // [2][nt][np]
  // E x B drift of the inner ghost cells for the current potential
  // (MiView::drift), refreshed by every writer of `potential`
  double *drift = nullptr;
  double *work = nullptr;       // [2][kVectors][n] + ring scratch
  double *scal = nullptr;       // [2][SL_COUNT]
  double *host_scal = nullptr;  // pinned mirror of scal
  Bilinear *bfringe = nullptr, *ffringe = nullptr, *samples = nullptr;
  int n_bfringe = 0, n_ffringe = 0, n_samples = 0;
  int *active = nullptr;  // per-hemisphere "still iterating" flags
  // learned warm start (not owned): the initial guess becomes the previous
  // potential plus the network's answer for the current residual
  unet::Net *net = nullptr;
  double *warm_scale = nullptr;  // [2] residual-current RMS, [2] step lengths
  // exchange buffers of the register-resident solve (null: its workgroups do
  // not fit) and its workgroups per hemisphere
  unsigned long long *ring_words = nullptr;
  int ring_groups = 0;
  int ring_spins = 0;  // polls after which its waits are given up
  // of the tensor solve by grid-wide barriers (null: not used): partial sums
  // and the per-hemisphere liveness exchange
  double *coop_slots = nullptr;
  int *coop_flags = nullptr;
};

namespace {

constexpr int kVectors = 20;   // solver vectors per hemisphere

struct MiK {
  Layout L;
  double *pl;
  uint8_t *by;
  StepScalars *sc;
  int cur;
  int np, nt, n, S, si;
  double ri, max_colat, current_norm, pedersen, r2;
  double *shell_fac, *fac, *potential, *work, *scal;
  __device__ double *p(int q) const { return pl + (long)q * L.total; }
  __device__ const uint8_t *b(int q) const { return by + (long)q * L.total; }
  __device__ double *vec(int h, int v) const { return work + ((long)h * kVectors + v) * n; }
  __device__ double *sl(int h) const { return scal + h * SL_COUNT; }
  __device__ void fail(unsigned stage, long index) const {
    if (atomicOr(&sc->failed, 1u) == 0u) {
      sc->fail_stage = stage;
      sc->fail_index = (int)index;
    }
  }
};

// vectors of one hemisphere's solve
// V_SCR, V_SCR2, V_IB, V_RDEN: the ring preconditioner's factors (forward
// factors g, Sherman-Morrison vector z, 1 / pivots, per-ring denominator).
enum Vec { V_RHS, V_DIAG, V_X, V_R, V_Z, V_P, V_AP, V_SH, V_PP, V_S, V_PS, V_AS,
           V_LO, V_HI, V_LLO, V_LHI, V_SCR, V_SCR2, V_IB, V_RDEN };

GCS_DEV long gtid() { return blockIdx.x * (long)blockDim.x + threadIdx.x; }

// ---- shell FAC (cubedsphere_mi_dipole.c:223-342) ---------------------------------

// Current-level B of shells si-1..si+1 into the scratch planes.
__global__ void k_mi_copy_shell(MiK c) {
  const Layout &L = c.L;
  const long per = 3L * L.NJ * L.NK;
  const long t = gtid();
  if (t >= 6 * per) return;
  const int f = (int)(t / per);
  long r = t - f * per;
  const int di = (int)(r / ((long)L.NJ * L.NK));
  r -= (long)di * L.NJ * L.NK;
  const int j = (int)(r / L.NK), k = (int)(r - (long)j * L.NK);
  const long at = L.at(f, c.si - 1 + di, j, k);
  for (int d = 0; d < 3; ++d) c.p(P_FVEL + d)[at] = c.p(plane_b(c.cur, d))[at];
}

// One-cell B fringe from the owning face (:236-276).
__global__ void k_mi_fringe_b(MiK c, const Bilinear *e, int n) {
  const long t = gtid();
  if (t >= n) return;
  const Bilinear h = e[t];
  const double w[4] = {(1.0 - h.wx) * (1.0 - h.wy), (1.0 - h.wx) * h.wy,
                       h.wx * (1.0 - h.wy), h.wx * h.wy};
  const long src[4] = {h.base, h.base + 1, h.base + h.step, h.base + h.step + 1};
  for (int d = 0; d < 3; ++d) {
    double v = 0.0;
    for (int q = 0; q < 4; ++q) v += w[q] * c.p(plane_b(c.cur, d))[src[q]];
    c.p(P_FVEL + d)[h.target] = v;
  }
}

// NO/nonorthogonal_mi.c:43-95: 4-cell average of B along one edge.
GCS_DEV bool edge_line(const MiK &c, int dir, long at, double &out) {
  const Layout &L = c.L;
  if (!c.b(Q_VALID + dir)[at]) return false;
  const long step[3] = {L.di(), (long)L.SK, 1};
  const int t1 = dir == 0 ? 1 : 0, t2 = dir == 2 ? 1 : 2;
  const long cell[4] = {at, at - step[t1], at - step[t2], at - step[t1] - step[t2]};
  double avg[3] = {0.0, 0.0, 0.0};
  for (int q = 0; q < 4; ++q)
    for (int m = 0; m < 3; ++m) avg[m] += 0.25 * c.p(P_FVEL + m)[cell[q]];
  const int eb = P_EDGE + EDGE_PLANES * dir;
  double dot = 0.0;
  for (int m = 0; m < 3; ++m) dot += avg[m] * c.p(eb + EO_N + m)[at];
  out = dot * c.p(eb + EO_LEN)[at];
  return isfinite(out);
}

// :97-136: circulation of B around the face of direction dir at `at`.
GCS_DEV bool face_circulation(const MiK &c, int dir, long at, double &out) {
  const Layout &L = c.L;
  const long si = L.di(), sj = L.SK;
  double e1, e2, e3, e4;
  bool ok;
  if (dir == 0)
    ok = edge_line(c, 1, at, e1) && edge_line(c, 2, at + sj, e2) &&
         edge_line(c, 1, at + 1, e3) && edge_line(c, 2, at, e4);
  else if (dir == 1)
    ok = edge_line(c, 2, at, e1) && edge_line(c, 0, at + 1, e2) &&
         edge_line(c, 2, at + si, e3) && edge_line(c, 0, at, e4);
  else
    ok = edge_line(c, 0, at, e1) && edge_line(c, 1, at + si, e2) &&
         edge_line(c, 0, at + sj, e3) && edge_line(c, 1, at, e4);
  if (!ok) return false;
  out = e1 + e2 - e3 - e4;
  return isfinite(out);
}

// FAC of the active shell cells (:277-307).
__global__ void k_mi_shell_fac(MiK c, double *shell_current) {
  const Layout &L = c.L;
  const int n = L.n;
  const long t = gtid();
  if (t >= 6L * n * n) return;
  const int f = (int)(t / ((long)n * n));
  const int r = (int)(t - (long)f * n * n);
  const int lj = 1 + r / n, lk = 1 + r % n;
  const int j = L.ghost - 1 + lj, k = L.ghost - 1 + lk;
  const long at = L.at(f, c.si, j, k);
  const long step[3] = {L.di(), (long)L.SK, 1};
  double flux[6];
  for (int d = 0; d < 3; ++d)
    if (!face_circulation(c, d, at, flux[2 * d]) ||
        !face_circulation(c, d, at + step[d], flux[2 * d + 1])) {
      c.fail(91, at);
      return;
    }
  double fc[6][3], cen[3], rec[9], cur[3];
  for (int d = 0; d < 3; ++d)
    for (int s = 0; s < 2; ++s)
      for (int m = 0; m < 3; ++m)
        fc[2 * d + s][m] = c.p(P_FACE + FACE_PLANES * d + FO_CEN + m)[at + s * step[d]];
  for (int m = 0; m < 3; ++m) cen[m] = c.p(P_CEN + m)[at];
  for (int q = 0; q < 9; ++q) rec[q] = c.p(P_REC + q)[at];
  const int piv = c.b(Q_PIV)[at];
  if (piv == 0xff || !recover_cell(flux, fc, cen, c.p(P_VOL)[at], rec, piv, cur)) {
    c.fail(92, at);
    return;
  }
  double b0[3], x[3];
  for (int m = 0; m < 3; ++m) {
    b0[m] = c.p(P_B0C + m)[at];
    x[m] = cen[m];
  }
  const double rad = sqrt(x[0] * x[0] + x[1] * x[1] + x[2] * x[2]);
  const double bm = sqrt(b0[0] * b0[0] + b0[1] * b0[1] + b0[2] * b0[2]);
  if (!(rad > 0.0) || !(bm > 0.0)) {
    c.fail(93, at);
    return;
  }
  const double colat = acos(fmin(1.0, fabs(x[2]) / rad));
  // NO/nonorthogonal_mi.c:183-196
  double s = sin(colat) * sqrt(c.ri / rad);
  s = fmax(-1.0, fmin(1.0, s));
  const double ti = asin(s);
  const double q = rad / c.ri;
  const double ratio = q * q * q * sqrt(1.0 + 3.0 * pow(cos(ti), 2.0)) /
                       sqrt(1.0 + 3.0 * pow(cos(colat), 2.0));
  const double jb = cur[0] * b0[0] + cur[1] * b0[1] + cur[2] * b0[2];
  const double fac = jb / bm * ratio * c.current_norm;
  if (!isfinite(fac)) {
    c.fail(94, at);
    return;
  }
  c.shell_fac[(long)f * c.S * c.S + lj * c.S + lk] = fac;
  // the shell's own J-parallel, magnetic latitude and longitude
  // (cubedsphere_mi_dipole.c:590-618)
  if (shell_current != nullptr) {
    const long q = ((long)f * n + (lj - 1)) * n + (lk - 1), per = 6L * n * n;
    double phi = atan2(x[1], x[0]) * 180.0 / kPi;
    if (phi < 0.0) phi += 360.0;
    shell_current[q] = jb / bm * c.current_norm;
    shell_current[per + q] = asin(x[2] / rad) * 180.0 / kPi;
    shell_current[2 * per + q] = phi;
  }
}

// FAC fringe (:308-342) and polar samples (:344-370, :391-406).
__global__ void k_mi_bilinear(const Bilinear *e, int n, const double *src, double *dst) {
  const long t = gtid();
  if (t >= n) return;
  const Bilinear h = e[t];
  if (h.zero) {
    dst[h.target] = 0.0;
    return;
  }
  const double *v = src + h.base;
  const double lo = (1.0 - h.wy) * v[0] + h.wy * v[1];
  const double hi = (1.0 - h.wy) * v[h.step] + h.wy * v[h.step + 1];
  dst[h.target] = (1.0 - h.wx) * lo + h.wx * hi;
}

// ---- polar solver (NO/nonorthogonal_mi.c) -----------------------------------

GCS_DEV int red_at(int np, int i, int j) { return 1 + (i - 1) * np + j; }

GCS_DEV double incl2(double th) {
  const double cs = cos(th);
  return 4.0 * cs * cs / (1.0 + 3.0 * cs * cs);
}
GCS_DEV double cos_incl(double th, int hemisphere) {
  const double cs = cos(th);
  return (double)hemisphere * 2.0 * cs / sqrt(1.0 + 3.0 * cs * cs);
}
GCS_DEV int hemi_sign(int h) { return h == 0 ? GAMERA_MI_NORTH : GAMERA_MI_SOUTH; }

// :234-241
GCS_DEV double theta_coeff(double sigma, double half, double center, double dt) {
  return sin(half) * sigma / (incl2(half) * sin(center) * dt * dt);
}

// One interior row (colatitude index i) of the five-point tensor stencil
// (:777-833) for uniform conductances: the averages of neighbouring Pedersen
// values are the value itself; the Hall term enters through
// d(-SigmaH / cos I)/dtheta. y = diag x + lo x(i-1) + hi x(i+1)
// + llo x(j-1) + lhi x(j+1).
struct TensorRow {
  double diag, lo, hi, llo, lhi;
};
GCS_DEV TensorRow tensor_row(double sp, double hall, int i, double dt, double dp, int hemi) {
  const double th = (double)i * dt;
  const double w = sin(th);
  const double inc = cos_incl(th, hemi);
  const double lt = th - 0.5 * dt, ut = th + 0.5 * dt;
  const double lo = sin(lt) * 0.5 * (sp + sp) / (incl2(lt) * dt * dt);
  const double hi = sin(ut) * 0.5 * (sp + sp) / (incl2(ut) * dt * dt);
  const double llo = 0.5 * (sp + sp) / (w * dp * dp);
  const double lhi = 0.5 * (sp + sp) / (w * dp * dp);
  const double f_up = -hall / cos_incl((double)(i + 1) * dt, hemi);
  const double f_dn = -hall / cos_incl((double)(i - 1) * dt, hemi);
  const double dft = (f_up - f_dn) / (2.0 * dt);
  const double dfp = (-hall / inc - -hall / inc) / (2.0 * dp);
  TensorRow t;
  t.diag = lo + hi + llo + lhi;
  t.lo = -lo - dfp / (2.0 * dt);
  t.hi = -hi + dfp / (2.0 * dt);
  t.llo = -llo + dft / (2.0 * dp);
  t.lhi = -lhi - dft / (2.0 * dp);
  return t;
}

// Right-hand side (:428-448, weighted by sin theta), initial guess from the
// previous potential (:449-464), and the diagonal (Pedersen, :322-344) or the
// five-point tensor stencil (:777-833).
// The exchange words of the register-resident solve and its report of waits
// given up are cleared here too.
__global__ void k_mi_setup(MiK c, int tensor, double hall, unsigned long long *words,
                           long n_words) {
  const int h = blockIdx.y;
  const long q = gtid();
  for (long t = q + h * (long)gridDim.x * blockDim.x; t < n_words;
       t += 2L * gridDim.x * blockDim.x)
    words[t] = 0ull;
  if (q >= c.n) return;
  const int np = c.np;
  const double dt = c.max_colat / (double)(c.nt - 1);
  const double dp = 2.0 * kPi / (double)np;
  double *rhs = c.vec(h, V_RHS), *x = c.vec(h, V_X), *diag = c.vec(h, V_DIAG);
  const double *pot = c.potential + (long)h * c.nt * np;
  const double *fac = c.fac + (long)h * c.nt * np;
  if (q == 0) {
    c.sl(h)[SL_GAVE_UP] = 0.0;
    rhs[0] = 0.0;
    double pole = 0.0;
    for (int j = 0; j < np; ++j) {
      const double v = pot[j];
      if (isfinite(v)) pole += v / (double)np;
    }
    x[0] = pole;
    const double half = 0.5 * dt;
    if (!tensor) {
      diag[0] = (double)np * (sin(half) * c.pedersen / (incl2(half) * dt * dt));
    } else {
      // uniform Pedersen: every pole edge has the same coefficient
      double d0 = 0.0;
      for (int j = 0; j < np; ++j) d0 += sin(half) * c.pedersen / (incl2(half) * dt * dt);
      diag[0] = d0;
    }
    return;
  }
  const int i = 1 + (int)((q - 1) / np), j = (int)((q - 1) % np);
  const double th = (double)i * dt;
  const double w = sin(th);
  const double inc = cos_incl(th, hemi_sign(h));
  const double u = -c.r2 * fac[i * np + j] * inc;
  rhs[q] = w * u;
  const double v = pot[i * np + j];
  x[q] = isfinite(v) ? v : 0.0;
  if (!tensor) {
    const double lo = theta_coeff(c.pedersen, th - 0.5 * dt, th, dt);
    const double hi = theta_coeff(c.pedersen, th + 0.5 * dt, th, dt);
    const double lon = c.pedersen / (sin(th) * sin(th) * dp * dp);
    diag[q] = w * (lo + hi + 2.0 * lon);
    return;
  }
  const TensorRow t = tensor_row(c.pedersen, hall, i, dt, dp, hemi_sign(h));
  diag[q] = t.diag;
  c.vec(h, V_LO)[q] = t.lo;
  c.vec(h, V_HI)[q] = t.hi;
  c.vec(h, V_LLO)[q] = t.llo;
  c.vec(h, V_LHI)[q] = t.lhi;
}

// y = A x on the reduced unknowns: the sin(theta)-weighted Pedersen operator
// (:355-392) or the tensor stencil (:871-900).
__global__ void k_mi_apply(MiK c, int tensor, int xin, int yout, const int *active) {
  const int h = blockIdx.y;
  if (!active[h]) return;
  const long q = gtid();
  if (q >= c.n) return;
  const int np = c.np, nt = c.nt;
  const double *x = c.vec(h, xin);
  double *y = c.vec(h, yout);
  const double *diag = c.vec(h, V_DIAG);
  const double dt = c.max_colat / (double)(nt - 1);
  if (q == 0) {
    if (!tensor) {
      const double half = 0.5 * dt;
      const double pe = sin(half) * c.pedersen / (incl2(half) * dt * dt);
      double ring = 0.0;
      for (int j = 0; j < np; ++j) ring += x[red_at(np, 1, j)];
      y[0] = pe * ((double)np * x[0] - ring);
    } else {
      const double half = 0.5 * dt;
      const double pe = sin(half) * c.pedersen / (incl2(half) * dt * dt);
      double v = diag[0] * x[0];
      for (int j = 0; j < np; ++j) v -= pe * x[red_at(np, 1, j)];
      y[0] = v;
    }
    return;
  }
  const int i = 1 + (int)((q - 1) / np), j = (int)((q - 1) % np);
  const int jm = j == 0 ? np - 1 : j - 1, jp = j + 1 == np ? 0 : j + 1;
  const double below = i == 1 ? x[0] : x[red_at(np, i - 1, j)];
  const double above = i + 2 < nt ? x[red_at(np, i + 1, j)] : 0.0;
  if (!tensor) {
    const double dp = 2.0 * kPi / (double)np;
    const double th = (double)i * dt;
    const double w = sin(th);
    const double lo = theta_coeff(c.pedersen, th - 0.5 * dt, th, dt);
    const double hi = theta_coeff(c.pedersen, th + 0.5 * dt, th, dt);
    const double lon = c.pedersen / (sin(th) * sin(th) * dp * dp);
    y[q] = w * (lo * (x[q] - below) + hi * (x[q] - above) +
                lon * (2.0 * x[q] - x[red_at(np, i, jm)] - x[red_at(np, i, jp)]));
  } else {
    y[q] = diag[q] * x[q] + c.vec(h, V_LO)[q] * below + c.vec(h, V_HI)[q] * above +
           c.vec(h, V_LLO)[q] * x[red_at(np, i, jm)] +
           c.vec(h, V_LHI)[q] * x[red_at(np, i, jp)];
  }
}

// Elementwise steps outside the fused solves.
enum Op {
  OP_RESIDUAL,  // r = rhs - ap; shadow = r
  OP_EXPAND     // potential from x (outer ring = extra)
};

__global__ void k_mi_vec(MiK c, int op, double extra, const int *active) {
  const int h = blockIdx.y;
  if (!active[h]) return;
  const long q = gtid();
  if (op == OP_EXPAND) {
    const long np = c.np, nt = c.nt;
    if (q >= np * nt) return;
    const int i = (int)(q / np), j = (int)(q % np);
    const double *x = c.vec(h, V_X);
    double *pot = c.potential + (long)h * nt * np;
    pot[q] = i == 0 ? x[0] : i == nt - 1 ? extra : x[red_at((int)np, i, j)];
    return;
  }
  if (q >= c.n) return;
  double *r = c.vec(h, V_R);
  r[q] = c.vec(h, V_RHS)[q] - c.vec(h, V_AP)[q];
  c.vec(h, V_SH)[q] = r[q];
}

template <typename T>
int upload_vec(const std::vector<T> &v, T **out) {
  *out = nullptr;
  if (v.empty()) return 0;
  GCS_HIP(hipMalloc(out, v.size() * sizeof(T)));
  GCS_HIP(hipMemcpy(*out, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
  return 0;
}

unsigned blocks_of(long n, int t = kT) { return (unsigned)((n + t - 1) / t); }

MiK make_mik(Problem &P) {
  MiState &m = *P.mi;
  MiK c;
  c.L = P.L;
  c.pl = P.planes;
  c.by = P.bytes;
  c.sc = P.scalars;
  c.cur = P.level;
  c.np = m.np;
  c.nt = m.nt;
  c.n = m.n;
  c.S = m.S;
  c.si = m.si;
  c.ri = m.cfg.ionosphere_radius_re;
  c.max_colat = m.max_colat;
  c.current_norm = m.current_norm;
  c.pedersen = m.cfg.pedersen_siemens;
  const double rm = m.cfg.ionosphere_radius_re * m.cfg.length_norm_m;
  c.r2 = rm * rm;
  c.shell_fac = m.shell_fac;
  c.fac = m.fac;
  c.potential = m.potential;
  c.work = m.work;
  c.scal = m.scal;
  return c;
}

// ---- fused solves: one workgroup per hemisphere runs the whole Krylov loop -------
//
// The solves of devices without cooperative launches or with
// GCS_MI_COOPERATIVE=0, and the Pedersen solve of grids whose rings the
// register-resident kernel's workgroups cannot hold at once.
//
// The same iterations as the reference's solvers (CG: :516-600, BiCGStab:
// :1029-1131, with the ring preconditioner above), but every scalar stays on
// the device: the workgroup's threads stride over the unknowns, dot products
// are workgroup reductions in a fixed order, and the loop, its breakdown and
// convergence tests and the periodic true-residual checks run in the kernel.
// The host launches once and reads the iteration count and final residual.
// Every branch depends only on values all threads share, so the whole
// workgroup leaves the loop together, at the latest after maximum_iterations.

constexpr int kSolveThreads = 1024;

// Sum over the workgroup, returned to every thread (fixed order).
GCS_DEV double block_sum(double v, double *red) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  __syncthreads();  // red[] may still be read from the previous call
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0.0;
  for (int w = 0; w < kSolveThreads / 64; ++w) s += red[w];
  return s;
}

// One term of the residual norm of the unweighted equations (:394-410).
GCS_DEV double orig_term(const MiK &c, double a, long q, double ps, double dt) {
  if (q == 0) {
    const double pr = a / ps;
    return (double)c.np * pr * pr;
  }
  const int i = 1 + (int)((q - 1) / c.np);
  const double v = a / sin((double)i * dt);
  return v * v;
}

// Rows of the Pedersen operator (w, lo, hi, lon per colatitude index),
// computed with k_mi_apply's expressions.
GCS_DEV void pedersen_rows(const MiK &c, double *rows) {
  const double dt = c.max_colat / (double)(c.nt - 1);
  const double dp = 2.0 * kPi / (double)c.np;
  for (int i = 1 + threadIdx.x; i + 1 < c.nt; i += blockDim.x) {
    const double th = (double)i * dt;
    rows[4 * i + 0] = sin(th);
    rows[4 * i + 1] = theta_coeff(c.pedersen, th - 0.5 * dt, th, dt);
    rows[4 * i + 2] = theta_coeff(c.pedersen, th + 0.5 * dt, th, dt);
    rows[4 * i + 3] = c.pedersen / (sin(th) * sin(th) * dp * dp);
  }
}

// (A x)[q], q >= 1, with k_mi_apply's arithmetic (Pedersen rows from `rows`).
GCS_DEV double apply_at(const MiK &c, int h, bool tensor, const double *x, long q,
                        const double *rows, double pe) {
  const int np = c.np, nt = c.nt;
  const int i = 1 + (int)((q - 1) / np), j = (int)((q - 1) % np);
  const int jm = j == 0 ? np - 1 : j - 1, jp = j + 1 == np ? 0 : j + 1;
  const double below = i == 1 ? x[0] : x[red_at(np, i - 1, j)];
  const double above = i + 2 < nt ? x[red_at(np, i + 1, j)] : 0.0;
  if (!tensor) {
    const double w = rows[4 * i], lo = rows[4 * i + 1], hi = rows[4 * i + 2],
                 lon = rows[4 * i + 3];
    return w * (lo * (x[q] - below) + hi * (x[q] - above) +
                lon * (2.0 * x[q] - x[red_at(np, i, jm)] - x[red_at(np, i, jp)]));
  }
  return c.vec(h, V_DIAG)[q] * x[q] + c.vec(h, V_LO)[q] * below +
         c.vec(h, V_HI)[q] * above + c.vec(h, V_LLO)[q] * x[red_at(np, i, jm)] +
         c.vec(h, V_LHI)[q] * x[red_at(np, i, jp)];
}

// Longitude-line preconditioner of the tensor system: out = M^-1 in with M
// the pole diagonal plus, on each colatitude ring, the ring's own periodic
// tridiagonal coupling, solved by the Thomas algorithm with a
// Sherman-Morrison correction for the periodic corners.
//
// The factors depend on the matrix only, so each solve computes them once
// (one thread per ring): g (forward factors), 1 / pivots, the correction
// vector z and the correction's denominator. Each application is then two
// first-order linear recurrences per ring, which one wavefront evaluates as
// a parallel prefix of affine maps (x -> A + B x) across its 64 lanes.
GCS_DEV void ring_factor(const MiK &c, int h, int ring) {
  const int np = c.np;
  const int base = 1 + ring * np;
  const double *__restrict__ a = c.vec(h, V_LLO) + base;  // coefficient of x[j-1]
  const double *__restrict__ b = c.vec(h, V_DIAG) + base;
  const double *__restrict__ cc = c.vec(h, V_LHI) + base; // coefficient of x[j+1]
  double *__restrict__ g = c.vec(h, V_SCR) + base;
  double *__restrict__ z = c.vec(h, V_SCR2) + base;
  double *__restrict__ ib = c.vec(h, V_IB) + base;
  const double gam = -b[0];
  const double alpha = cc[np - 1];  // row np-1's coupling to x[0]
  const double beta = a[0];         // row 0's coupling to x[np-1]
  double inv = 1.0 / (b[0] - gam);
  double zp = gam * inv;
  ib[0] = inv;
  g[0] = 0.0;
  z[0] = zp;
  for (int j = 1; j < np; ++j) {
    const double gj = cc[j - 1] * inv;
    g[j] = gj;
    const double bj = j == np - 1 ? b[j] - alpha * beta / gam : b[j];
    inv = 1.0 / (bj - a[j] * gj);
    ib[j] = inv;
    zp = ((j == np - 1 ? alpha : 0.0) - a[j] * zp) * inv;
    z[j] = zp;
  }
  const double zl = zp;
  for (int j = np - 2; j >= 0; --j) {
    zp = z[j] - g[j + 1] * zp;
    z[j] = zp;
  }
  c.vec(h, V_RDEN)[base] = 1.0 + zp + beta * zl / gam;
}

GCS_DEV void factor_rings(const MiK &c, int h) {
  for (int ring = threadIdx.x; ring < c.nt - 2; ring += blockDim.x) ring_factor(c, h, ring);
}

// One ring's solve by one wavefront (lane = threadIdx.x & 63): each lane
// holds kRingChunk consecutive points of the ring in registers, so a ring
// costs one load phase and one store phase.
constexpr int kRingChunk = 8;  // rings up to 64 * 8 = 512 points

GCS_DEV void ring_apply(const MiK &c, int h, const double *in, double *out, int ring,
                        int lane) {
  const int np = c.np;
  const int base = 1 + ring * np;
  const double *a = c.vec(h, V_LLO) + base;
  const double *g = c.vec(h, V_SCR) + base;
  const double *z = c.vec(h, V_SCR2) + base;
  const double *ib = c.vec(h, V_IB) + base;
  const double *rhs = in + base;
  double *x = out + base;
  const int k = (np + 63) / 64;
  const int j0 = min(np, lane * k);
  const int cnt = min(np, j0 + k) - j0;
  double fa[kRingChunk], fb[kRingChunk], gd[kRingChunk], zz[kRingChunk], v[kRingChunk];
#pragma unroll
  for (int t = 0; t < kRingChunk; ++t) {
    const int j = j0 + t;
    const bool in_range = t < cnt;
    const double ibj = in_range ? ib[j] : 0.0;
    fa[t] = in_range ? ibj * rhs[j] : 0.0;
    fb[t] = in_range && j > 0 ? -a[j] * ibj : 0.0;
    gd[t] = in_range && j < np - 1 ? -g[j + 1] : 0.0;
    zz[t] = in_range ? z[j] : 0.0;
  }
  // forward: x_j = fa_j + fb_j x_{j-1}, as a prefix of affine maps
  double A = 0.0, B = 1.0;
#pragma unroll
  for (int t = 0; t < kRingChunk; ++t)
    if (t < cnt) {
      A = fa[t] + fb[t] * A;
      B = fb[t] * B;
    }
  for (int off = 1; off < 64; off <<= 1) {
    const double ao = __shfl_up(A, off, 64), bo = __shfl_up(B, off, 64);
    if (lane >= off) {
      A = A + B * ao;
      B = B * bo;
    }
  }
  double w = __shfl_up(A, 1, 64);
#pragma unroll
  for (int t = 0; t < kRingChunk; ++t)
    if (t < cnt) {
      w = fa[t] + fb[t] * w;
      v[t] = w;
    }
  // backward: y_j = x_j + gd_j y_{j+1} (gd_j = -g_{j+1}; 0 for the last point)
  double C = 0.0, D = 1.0;
#pragma unroll
  for (int t = kRingChunk - 1; t >= 0; --t)
    if (t < cnt) {
      C = v[t] + gd[t] * C;
      D = gd[t] * D;
    }
  for (int off = 1; off < 64; off <<= 1) {
    const double co = __shfl_down(C, off, 64), dd = __shfl_down(D, off, 64);
    if (lane + off < 64) {
      C = C + D * co;
      D = D * dd;
    }
  }
  w = __shfl_down(C, 1, 64);
#pragma unroll
  for (int t = kRingChunk - 1; t >= 0; --t)
    if (t < cnt) {
      w = v[t] + gd[t] * w;
      v[t] = w;
    }
  // Sherman-Morrison correction with y_0 and y_{np-1}
  const double y0 = __shfl(v[0], 0, 64);
  const int owner = (np - 1) / k;
  double mine_last = v[0];
#pragma unroll
  for (int t = 0; t < kRingChunk; ++t)
    if (t == (np - 1) - owner * k) mine_last = v[t];
  const double yl = __shfl(mine_last, owner, 64);
  const double gam = -c.vec(h, V_DIAG)[base];
  const double fact = (y0 + a[0] * yl / gam) / c.vec(h, V_RDEN)[base];
#pragma unroll
  for (int t = 0; t < kRingChunk; ++t)
    if (t < cnt) x[j0 + t] = v[t] - fact * zz[t];
}

GCS_DEV void precondition_all(const MiK &c, int h, const double *in, double *out) {
  __syncthreads();  // `in` complete
  if (threadIdx.x == 0) out[0] = in[0] / c.vec(h, V_DIAG)[0];
  const int lane = threadIdx.x & 63, waves = blockDim.x >> 6;
  for (int ring = threadIdx.x >> 6; ring < c.nt - 2; ring += waves)
    ring_apply(c, h, in, out, ring, lane);
  __syncthreads();  // `out` complete
}

// (A x)[0], the pole row, by wavefront 0 (every lane returns it).
GCS_DEV double pole_row(const MiK &c, int h, bool tensor, const double *x, double pe) {
  const int np = c.np;
  double ring = 0.0;
  for (int j = threadIdx.x & 63; j < np; j += 64) ring += x[red_at(np, 1, j)];
  for (int off = 32; off > 0; off >>= 1) ring += __shfl_xor(ring, off, 64);
  if (!tensor) return pe * ((double)np * x[0] - ring);
  return c.vec(h, V_DIAG)[0] * x[0] - pe * ring;
}

struct SolveResult {
  int iters;
  bool ok;
  double last;
};

GCS_DEV void store_result(const MiK &c, int h, const SolveResult &r, double first) {
  if (threadIdx.x != 0) return;
  double *sl = c.sl(h);
  sl[SL_ITER] = (double)r.iters;
  sl[SL_OK] = r.ok ? 1.0 : 0.0;
  sl[SL_NORM] = r.last;
  sl[SL_FIRST] = first;
}

// Jacobi-preconditioned CG on the reduced Pedersen system (:516-600).
__global__ void __launch_bounds__(kSolveThreads) k_mi_cg(MiK c, double rel_tol, int maxit) {
  __shared__ double red[kSolveThreads / 64];
  extern __shared__ double rows[];
  const int h = blockIdx.x;
  const long n = c.n;
  const long t0 = threadIdx.x, st = blockDim.x;
  const double dt = c.max_colat / (double)(c.nt - 1);
  const double half = 0.5 * dt;
  const double pe = sin(half) * c.pedersen / (incl2(half) * dt * dt);
  const double ps = (double)c.np * pe;
  pedersen_rows(c, rows);
  __syncthreads();
  double *x = c.vec(h, V_X), *r = c.vec(h, V_R), *z = c.vec(h, V_Z), *p = c.vec(h, V_P),
         *ap = c.vec(h, V_AP);
  const double *rhs = c.vec(h, V_RHS), *diag = c.vec(h, V_DIAG);
  double a = 0.0, b = 0.0;
  const double pole = threadIdx.x < 64 ? pole_row(c, h, false, x, pe) : 0.0;
  for (long q = t0; q < n; q += st) {
    r[q] = rhs[q] - (q == 0 ? pole : apply_at(c, h, false, x, q, rows, pe));
    a += orig_term(c, r[q], q, ps, dt);
    b += q == 0 ? 0.0 : orig_term(c, rhs[q], q, ps, dt);
  }
  double norm = sqrt(fmax(0.0, block_sum(a, red)));
  const double first = norm;
  const double target = rel_tol * fmax(sqrt(fmax(0.0, block_sum(b, red))), 1.0);
  SolveResult res{0, norm <= target, norm};
  if (!res.ok) {
    a = 0.0;
    for (long q = t0; q < n; q += st) {
      z[q] = r[q] / diag[q];
      p[q] = z[q];
      a += r[q] * z[q];
    }
    double rz = block_sum(a, red);
    for (int it = 1; it <= maxit; ++it) {
      a = 0.0;
      const double pole = threadIdx.x < 64 ? pole_row(c, h, false, p, pe) : 0.0;
      for (long q = t0; q < n; q += st) {
        ap[q] = (q == 0 ? pole : apply_at(c, h, false, p, q, rows, pe));
        a += p[q] * ap[q];
      }
      const double pap = block_sum(a, red);
      if (!isfinite(rz) || rz <= DBL_MIN || !isfinite(pap) || pap <= DBL_MIN) break;
      const double alpha = rz / pap;
      a = 0.0;
      for (long q = t0; q < n; q += st) {
        x[q] += alpha * p[q];
        r[q] -= alpha * ap[q];
        a += orig_term(c, r[q], q, ps, dt);
      }
      norm = sqrt(fmax(0.0, block_sum(a, red)));
      res.iters = it;
      res.last = norm;
      if (norm <= target || it % 1024 == 0) {
        __syncthreads();  // x complete
        a = 0.0;
        const double pole = threadIdx.x < 64 ? pole_row(c, h, false, x, pe) : 0.0;
        for (long q = t0; q < n; q += st) {
          r[q] = rhs[q] - (q == 0 ? pole : apply_at(c, h, false, x, q, rows, pe));
          a += orig_term(c, r[q], q, ps, dt);
        }
        norm = sqrt(fmax(0.0, block_sum(a, red)));
        res.last = norm;
        if (norm <= target) {
          res.ok = true;
          break;
        }
        a = 0.0;
        for (long q = t0; q < n; q += st) {
          z[q] = r[q] / diag[q];
          p[q] = z[q];
          a += r[q] * z[q];
        }
        rz = block_sum(a, red);
        continue;
      }
      a = 0.0;
      for (long q = t0; q < n; q += st) {
        z[q] = r[q] / diag[q];
        a += r[q] * z[q];
      }
      const double rzn = block_sum(a, red);
      for (long q = t0; q < n; q += st) p[q] = z[q] + (rzn / rz) * p[q];
      rz = rzn;
      __syncthreads();  // p complete before the next product
    }
  }
  store_result(c, h, res, first);
}

// Right-preconditioned BiCGStab on the tensor system (:1029-1131).
__global__ void __launch_bounds__(kSolveThreads) k_mi_bicgstab(MiK c, double rel_tol,
                                                               int maxit) {
  __shared__ double red[kSolveThreads / 64];
  const int h = blockIdx.x;
  const long n = c.n;
  const long t0 = threadIdx.x, st = blockDim.x;
  const double dt = c.max_colat / (double)(c.nt - 1);
  const double half = 0.5 * dt;
  const double pe = sin(half) * c.pedersen / (incl2(half) * dt * dt);
  const double ps = (double)c.np * pe;
  double *x = c.vec(h, V_X), *r = c.vec(h, V_R), *p = c.vec(h, V_P), *ap = c.vec(h, V_AP),
         *sh = c.vec(h, V_SH), *pp = c.vec(h, V_PP), *s = c.vec(h, V_S), *psv = c.vec(h, V_PS),
         *as = c.vec(h, V_AS);
  const double *rhs = c.vec(h, V_RHS);
  factor_rings(c, h);
  __syncthreads();  // ring factors complete
  double a = 0.0, b = 0.0;
  const double pole = threadIdx.x < 64 ? pole_row(c, h, true, x, pe) : 0.0;
  for (long q = t0; q < n; q += st) {
    r[q] = rhs[q] - (q == 0 ? pole : apply_at(c, h, true, x, q, nullptr, pe));
    sh[q] = r[q];
    p[q] = 0.0;
    ap[q] = 0.0;
    a += orig_term(c, r[q], q, ps, dt);
    b += q == 0 ? 0.0 : orig_term(c, rhs[q], q, ps, dt);
  }
  double norm = sqrt(fmax(0.0, block_sum(a, red)));
  const double first = norm;
  const double target = rel_tol * fmax(sqrt(fmax(0.0, block_sum(b, red))), 1.0);
  SolveResult res{0, norm <= target, norm};
  double rho_prev = 1.0, alpha = 1.0, omega = 1.0;
  for (int it = 1; it <= maxit && !res.ok; ++it) {
    a = 0.0;
    for (long q = t0; q < n; q += st) a += sh[q] * r[q];
    const double rho = block_sum(a, red);
    if (!isfinite(rho) || fabs(rho) <= DBL_MIN || !isfinite(omega) || fabs(omega) <= DBL_MIN)
      break;
    const double beta = (rho / rho_prev) * (alpha / omega);
    for (long q = t0; q < n; q += st) p[q] = r[q] + beta * (p[q] - omega * ap[q]);
    precondition_all(c, h, p, pp);
    a = 0.0;
    const double pole = threadIdx.x < 64 ? pole_row(c, h, true, pp, pe) : 0.0;
    for (long q = t0; q < n; q += st) {
      ap[q] = (q == 0 ? pole : apply_at(c, h, true, pp, q, nullptr, pe));
      a += sh[q] * ap[q];
    }
    const double den = block_sum(a, red);
    alpha = rho / den;
    a = 0.0;
    for (long q = t0; q < n; q += st) {
      s[q] = r[q] - alpha * ap[q];
      a += orig_term(c, s[q], q, ps, dt);
    }
    const double snorm = sqrt(fmax(0.0, block_sum(a, red)));
    if (!isfinite(den) || fabs(den) <= DBL_MIN) break;
    if (snorm <= target) {
      res.last = snorm;
      res.iters = it;
      res.ok = true;
      for (long q = t0; q < n; q += st) x[q] += alpha * pp[q];
      break;
    }
    precondition_all(c, h, s, psv);
    a = 0.0;
    b = 0.0;
    const double pole_s = threadIdx.x < 64 ? pole_row(c, h, true, psv, pe) : 0.0;
    for (long q = t0; q < n; q += st) {
      as[q] = (q == 0 ? pole_s : apply_at(c, h, true, psv, q, nullptr, pe));
      a += as[q] * as[q];
      b += as[q] * s[q];
    }
    const double wden = block_sum(a, red);
    const double wnum = block_sum(b, red);
    omega = wnum / wden;
    if (!isfinite(wden) || wden <= DBL_MIN || !isfinite(omega) || fabs(omega) <= DBL_MIN)
      break;
    a = 0.0;
    for (long q = t0; q < n; q += st) {
      x[q] += alpha * pp[q] + omega * psv[q];
      r[q] = s[q] - omega * as[q];
      a += orig_term(c, r[q], q, ps, dt);
    }
    norm = sqrt(fmax(0.0, block_sum(a, red)));
    res.iters = it;
    res.last = norm;
    if (norm <= target || it % 256 == 0) {
      __syncthreads();  // x complete
      a = 0.0;
      const double pole = threadIdx.x < 64 ? pole_row(c, h, true, x, pe) : 0.0;
      for (long q = t0; q < n; q += st) {
        r[q] = rhs[q] - (q == 0 ? pole : apply_at(c, h, true, x, q, nullptr, pe));
        sh[q] = r[q];
        a += orig_term(c, r[q], q, ps, dt);
      }
      norm = sqrt(fmax(0.0, block_sum(a, red)));
      res.last = norm;
      if (norm <= target) {
        res.ok = true;
        break;
      }
      for (long q = t0; q < n; q += st) {
        p[q] = 0.0;
        ap[q] = 0.0;
      }
      rho_prev = alpha = omega = 1.0;
      continue;
    }
    rho_prev = rho;
  }
  store_result(c, h, res, first);
}

// The Hall-tensor solve of grids with more rings than k_ring_bicgstab's
// workgroups can hold at once (768 on 256 compute units): each hemisphere's
// solve spread over kCoopBlocks workgroups (the same iterations as
// k_mi_bicgstab, with grid-wide barriers where one workgroup's barrier
// sufficed there). What bounds it is its ten barriers an iteration and, on
// large grids, the vectors' traffic through L2. 2 x 800 x 256 points, 3,400 -
// 3,900 iterations: 900 ms (k_mi_bicgstab: 9,221); 2 x 771 x 64: 400 ms
// (3,219). Below that limit k_ring_bicgstab is the faster one: 2 x 770 x 64,
// 43 against 384 ms; 2 x 128 x 256, 4.0 against 45. Dot products sum the
// workgroups' partial sums in workgroup order from two alternating slot
// banks (a bank is rewritten only after every workgroup passed the barrier
// that follows its last read), so every workgroup of a hemisphere computes
// the same sums and takes the same branches.
constexpr int kCoopBlocks = 16;

// Both hemispheres in one cooperative launch: workgroups [0, kCoopBlocks)
// solve the north, [kCoopBlocks, 2 kCoopBlocks) the south, concurrently. The
// grid barriers are shared, so every workgroup must pass the same sequence
// of barriers whatever its hemisphere does: each iteration runs a fixed
// schedule of ten barrier-carrying steps, and a hemisphere that has
// converged, broken down or needs no true-residual check this iteration
// skips the work of a step but not its barrier. No branch contains a
// barrier, the loop bound and its exit test are grid-uniform (the exit reads
// both hemispheres' flags after a barrier), so every workgroup leaves after
// the same number of barriers, at the latest after maximum_iterations.
// Per hemisphere the arithmetic is k_mi_bicgstab's.
__global__ void __launch_bounds__(kSolveThreads) k_mi_bicgstab_pair(MiK c, double rel_tol,
                                                                    int maxit, double *slots,
                                                                    int *flags) {
  namespace cg = cooperative_groups;
  cg::grid_group grid = cg::this_grid();
  __shared__ double red[kSolveThreads / 64];
  const int h = blockIdx.x / kCoopBlocks, lb = blockIdx.x % kCoopBlocks;
  const long n = c.n;
  const long t0 = lb * (long)blockDim.x + threadIdx.x;
  const long st = (long)kCoopBlocks * blockDim.x;
  const bool pole_wave = lb == 0 && threadIdx.x < 64;
  int bank = 0;
  // sums of up to two values over this hemisphere's workgroups
  auto gsum2 = [&](double v, double w, double &sv, double &sw) {
    const double bv = block_sum(v, red);
    const double bw = block_sum(w, red);
    double *sl = slots + bank * (4 * kCoopBlocks) + h * (2 * kCoopBlocks);
    if (threadIdx.x == 0) {
      sl[lb] = bv;
      sl[kCoopBlocks + lb] = bw;
    }
    bank ^= 1;
    grid.sync();
    sv = 0.0;
    sw = 0.0;
    for (int i = 0; i < kCoopBlocks; ++i) {
      sv += sl[i];
      sw += sl[kCoopBlocks + i];
    }
  };
  auto gsum = [&](double v) {
    double sv, sw;
    gsum2(v, 0.0, sv, sw);
    return sv;
  };
  const double dt = c.max_colat / (double)(c.nt - 1);
  const double half = 0.5 * dt;
  const double pe = sin(half) * c.pedersen / (incl2(half) * dt * dt);
  const double ps = (double)c.np * pe;
  double *x = c.vec(h, V_X), *r = c.vec(h, V_R), *p = c.vec(h, V_P), *ap = c.vec(h, V_AP),
         *sh = c.vec(h, V_SH), *pp = c.vec(h, V_PP), *s = c.vec(h, V_S), *psv = c.vec(h, V_PS),
         *as = c.vec(h, V_AS);
  const double *rhs = c.vec(h, V_RHS);
  const int lane = threadIdx.x & 63;
  auto precondition = [&](bool work, const double *in, double *out) {
    grid.sync();  // `in` complete
    if (work) {
      if (t0 == 0) out[0] = in[0] / c.vec(h, V_DIAG)[0];
      for (long ring = t0 >> 6; ring < c.nt - 2; ring += st >> 6)
        ring_apply(c, h, in, out, (int)ring, lane);
    }
    grid.sync();  // `out` complete
  };
  for (long ring = t0; ring < c.nt - 2; ring += st) ring_factor(c, h, (int)ring);
  double a = 0.0, b = 0.0;
  {
    const double pole = pole_wave ? pole_row(c, h, true, x, pe) : 0.0;
    for (long q = t0; q < n; q += st) {
      r[q] = rhs[q] - (q == 0 ? pole : apply_at(c, h, true, x, q, nullptr, pe));
      sh[q] = r[q];
      p[q] = 0.0;
      ap[q] = 0.0;
      a += orig_term(c, r[q], q, ps, dt);
      b += q == 0 ? 0.0 : orig_term(c, rhs[q], q, ps, dt);
    }
  }
  double n0, b0;
  gsum2(a, b, n0, b0);  // also orders the ring factors before their first use
  double norm = sqrt(fmax(0.0, n0));
  const double first = norm;
  const double target = rel_tol * fmax(sqrt(fmax(0.0, b0)), 1.0);
  SolveResult res{0, norm <= target, norm};
  bool live = !res.ok;  // this hemisphere still iterates
  double rho_prev = 1.0, alpha = 1.0, omega = 1.0;
  bool other_live = true;
  for (int it = 1; it <= maxit && (live || other_live); ++it) {
    // 1: rho
    a = 0.0;
    if (live)
      for (long q = t0; q < n; q += st) a += sh[q] * r[q];
    const double rho = gsum(a);
    if (live && (!isfinite(rho) || fabs(rho) <= DBL_MIN || !isfinite(omega) ||
                 fabs(omega) <= DBL_MIN))
      live = false;
    // 2, 3: p and its preconditioned image
    if (live) {
      const double beta = (rho / rho_prev) * (alpha / omega);
      for (long q = t0; q < n; q += st) p[q] = r[q] + beta * (p[q] - omega * ap[q]);
    }
    precondition(live, p, pp);
    // 4: A pp and den
    a = 0.0;
    {
      const double pole = (live && pole_wave) ? pole_row(c, h, true, pp, pe) : 0.0;
      if (live)
        for (long q = t0; q < n; q += st) {
          ap[q] = q == 0 ? pole : apply_at(c, h, true, pp, q, nullptr, pe);
          a += sh[q] * ap[q];
        }
    }
    const double den = gsum(a);
    // 5: s and its norm
    a = 0.0;
    if (live) {
      alpha = rho / den;
      for (long q = t0; q < n; q += st) {
        s[q] = r[q] - alpha * ap[q];
        a += orig_term(c, s[q], q, ps, dt);
      }
    }
    const double snorm = sqrt(fmax(0.0, gsum(a)));
    if (live && (!isfinite(den) || fabs(den) <= DBL_MIN)) live = false;
    if (live && snorm <= target) {
      res.last = snorm;
      res.iters = it;
      res.ok = true;
      live = false;
      for (long q = t0; q < n; q += st) x[q] += alpha * pp[q];
    }
    // 6, 7: preconditioned s
    precondition(live, s, psv);
    // 8: A ps and omega
    a = 0.0;
    b = 0.0;
    {
      const double pole = (live && pole_wave) ? pole_row(c, h, true, psv, pe) : 0.0;
      if (live)
        for (long q = t0; q < n; q += st) {
          as[q] = q == 0 ? pole : apply_at(c, h, true, psv, q, nullptr, pe);
          a += as[q] * as[q];
          b += as[q] * s[q];
        }
    }
    double wden, wnum;
    gsum2(a, b, wden, wnum);
    if (live) {
      omega = wnum / wden;
      if (!isfinite(wden) || wden <= DBL_MIN || !isfinite(omega) || fabs(omega) <= DBL_MIN)
        live = false;
    }
    // 9: x, r and the recursive residual norm
    a = 0.0;
    if (live)
      for (long q = t0; q < n; q += st) {
        x[q] += alpha * pp[q] + omega * psv[q];
        r[q] = s[q] - omega * as[q];
        a += orig_term(c, r[q], q, ps, dt);
      }
    const double rn = gsum(a);
    bool verify = false;
    if (live) {
      norm = sqrt(fmax(0.0, rn));
      res.iters = it;
      res.last = norm;
      verify = norm <= target || it % 256 == 0;
    }
    // 10: true residual when checked; the exit flags of both hemispheres
    a = 0.0;
    if (verify) {
      const double pole = pole_wave ? pole_row(c, h, true, x, pe) : 0.0;
      for (long q = t0; q < n; q += st) {
        r[q] = rhs[q] - (q == 0 ? pole : apply_at(c, h, true, x, q, nullptr, pe));
        sh[q] = r[q];
        a += orig_term(c, r[q], q, ps, dt);
      }
    }
    const double tn = gsum(a);
    if (verify) {
      norm = sqrt(fmax(0.0, tn));
      res.last = norm;
      if (norm <= target) {
        res.ok = true;
        live = false;
      } else {
        for (long q = t0; q < n; q += st) {
          p[q] = 0.0;
          ap[q] = 0.0;
        }
        rho_prev = alpha = omega = 1.0;
      }
    } else if (live) {
      rho_prev = rho;
    }
    // exchange liveness: written now, read after the next iteration's first
    // barrier; one more round trip than needed only delays the exit
    if (lb == 0 && threadIdx.x == 0) flags[(it & 1) * 2 + h] = live ? 1 : 0;
    grid.sync();
    other_live = flags[(it & 1) * 2 + (1 - h)] != 0;
  }
  if (lb == 0) store_result(c, h, res, first);
}

// ---- register-resident solves: one wavefront per colatitude ring ------------------
//
// The iterations of k_mi_cg and k_mi_bicgstab with the solver vectors held in
// registers: a wavefront owns one ring, a lane kRingPoints = ceil(np / 64)
// consecutive points of it, and a workgroup kRingOwn rings plus a ghost copy
// of the ring on each side. Neighbour rings inside a workgroup meet in LDS.
// A ghost wavefront runs the same vector updates as the ring's owner (so its
// values are the owner's, bit for bit) and receives from it only the product
// A p that it cannot form itself. Workgroups exchange two things, both as
// words of the LL protocol of the collective libraries (32 bits of a double
// and a 32-bit sequence number in one 64-bit store, so that a word that has
// arrived says so itself): the partial sums of the dot products, and those
// boundary rings, which are sent before a reduction and read after it, so
// that their way is hidden behind the reduction's. A reduction is therefore
// the only wait: one per CG iteration, two per BiCGStab iteration, where a
// grid barrier per dot product and per vector took ten. What bounds an
// iteration is the latency of these reductions and of the ring solve's two
// wavefront-wide prefixes, as long as the vectors fit: a lane has 256
// registers (512 threads a workgroup). CG's fit up to 512 points a ring
// (255), BiCGStab's nine vectors and factors up to 256 (235); at 5, 6, 7 and
// 8 points a lane 32, 86, 127 and 231 registers are spilled to scratch memory.
// Measured, solves from zero on 2 x 128 rings (ms; in brackets BiCGStab with
// grid-wide barriers, CG on one workgroup per hemisphere, vectors in memory):
//   points a ring      256          320          384          448         512
//   BiCGStab      4.0 (45)     4.7 (46)     5.8 (50)     8.4 (53)   12.6 (56)
//   CG            3.6 (81)    4.6 (117)    6.1 (169)   10.0 (308)  14.9 (494)
// that is 9.5 us a BiCGStab iteration at 256 points (100) and 28 at 512 (135),
// 3.9 us (87) and 5.2 (171) of CG; on 2 x 33 x 57, 7.7 us and 0.85 ms, 3.3 us
// and 0.63 ms. Putting a hemisphere's workgroups on one XCD changed nothing
// (3 %).
//
// The hemispheres are independent groups of workgroups. Every workgroup of a
// hemisphere sums the same words in the same order and so takes the same
// branches. All workgroups must be resident (a cooperative launch); a wait
// ends after RingComm::spins polls at the latest, one at least (a loop that
// may run none keeps what it loads live around it: 24 registers more, 3.95 ->
// 4.58 ms on 2 x 128 x 256). A workgroup that gave one up says so in its
// hemisphere's results (SL_GAVE_UP) and leaves, after which its neighbours'
// waits end the same way; the host then has the system, which these kernels
// leave as it was, solved without waits between workgroups.

typedef unsigned long long ll_word;

constexpr int kRingWaves = 8;
constexpr int kRingOwn = kRingWaves - 2;
constexpr int kRingThreads = 64 * kRingWaves;
constexpr int kRingSums = 7;         // most values of one reduction
constexpr int kSpinLimit = 1 << 20;  // polls of a wait by default, about a second

// Device buffers of the exchange, zeroed before each solve (the sequence
// numbers of a solve start at 1): red [2 banks][2 hemispheres][groups]
// [kRingSums][2 words], halo [2 banks][2 hemispheres][groups][2 sides]
// [points][2 halves][64 lanes]. A bank is used again two messages later; by
// then a reduction has passed, which its reader entered after reading it.
struct RingComm {
  ll_word *red, *halo;
  int groups, points;
  int spins;  // polls of a wait (one at least)
  static size_t red_words(int groups) { return 2UL * 2 * groups * kRingSums * 2; }
  static size_t halo_words(int groups, int points) {
    return 2UL * 2 * groups * 2 * points * 2 * 64;
  }
};

GCS_DEV void ll_put(ll_word *hi, ll_word *lo, double v, unsigned seq) {
  const ll_word b = (ll_word)__double_as_longlong(v);
  __hip_atomic_store(hi, (b & 0xffffffff00000000ull) | seq, __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(lo, (b << 32) | seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
GCS_DEV ll_word ll_load(const ll_word *w) {
  return __hip_atomic_load(const_cast<ll_word *>(w), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
GCS_DEV double ll_value(ll_word hi, ll_word lo) {
  return __longlong_as_double((long long)((hi & 0xffffffff00000000ull) | (lo >> 32)));
}

// Lane moves by DPP (a few cycles; a shuffle through LDS takes over a hundred):
// v of the lane the control names, `old` where there is none.
enum Dpp {
  DPP_ROW_SHL = 0x100, DPP_ROW_SHR = 0x110,  // + n: within rows of 16 lanes
  DPP_WAVE_SHL1 = 0x130, DPP_WAVE_SHR1 = 0x138, DPP_BCAST15 = 0x142, DPP_BCAST31 = 0x143
};
template <int Ctrl, int RowMask = 0xf>
GCS_DEV double dpp_move(double old, double v) {
  const int lo = __builtin_amdgcn_update_dpp(__double2loint(old), __double2loint(v), Ctrl,
                                             RowMask, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(__double2hiint(old), __double2hiint(v), Ctrl,
                                             RowMask, 0xf, false);
  return __hiloint2double(hi, lo);
}
GCS_DEV double read_lane(double v, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                          __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// Sum over the wavefront, in every lane.
GCS_DEV double wave_sum(double v) {
  v += dpp_move<DPP_ROW_SHR + 1>(0.0, v);
  v += dpp_move<DPP_ROW_SHR + 2>(0.0, v);
  v += dpp_move<DPP_ROW_SHR + 4>(0.0, v);
  v += dpp_move<DPP_ROW_SHR + 8>(0.0, v);
  v += dpp_move<DPP_BCAST15, 0xa>(0.0, v);
  v += dpp_move<DPP_BCAST31, 0xc>(0.0, v);
  return read_lane(v, 63);
}

// One step of a prefix (N lanes to the left) or suffix of affine maps
// x -> a + b x; a lane without such a neighbour composes with the identity.
template <int Ctrl>
GCS_DEV void affine_step(double &a, double &b) {
  const double ao = dpp_move<Ctrl>(0.0, a), bo = dpp_move<Ctrl>(1.0, b);
  a = a + b * ao;
  b = b * bo;
}

// What a wavefront knows of its place in the solve.
template <int KP>
struct RingWave {
  int h, g, groups;      // hemisphere, workgroup of it, workgroups of it
  int w, lane, nown;     // wavefront, lane, rings this workgroup owns
  int ring;              // colatitude index of the wavefront's ring
  bool own, ghost;       // owner or ghost copy of `ring` (neither: idle)
  int j0, cnt;           // this lane's points j0 .. j0 + cnt - 1
  int last_lane, last_t; // where the ring's last point is
  unsigned seq, hseq;    // sequence numbers of the last reduction and message
  bool dead;             // a wait was given up
  RingComm comm;
  double (*rows)[64 * KP];         // LDS [kRingWaves][points, t-major]
  double (*part)[kRingWaves];      // LDS [kRingSums][kRingWaves]
  double *total;                   // LDS [kRingSums + 1]
  int *gave_up;                    // LDS

  GCS_DEV void init(const MiK &c, const RingComm &cm, double (*r)[64 * KP],
                    double (*p)[kRingWaves], double *t, int *gu) {
    comm = cm;
    groups = cm.groups;
    h = blockIdx.x / groups;
    g = blockIdx.x % groups;
    w = threadIdx.x >> 6;
    lane = threadIdx.x & 63;
    nown = min(kRingOwn, c.nt - 2 - g * kRingOwn);
    ring = g * kRingOwn + w;
    own = w >= 1 && w <= nown;
    ghost = (w == 0 && g > 0) || (w == nown + 1 && ring <= c.nt - 2);
    j0 = min(c.np, lane * KP);
    cnt = min(c.np, j0 + KP) - j0;
    last_lane = (c.np - 1) / KP;
    last_t = (c.np - 1) - last_lane * KP;
    seq = hseq = 0;
    dead = false;
    rows = r;
    part = p;
    total = t;
    gave_up = gu;
    if (threadIdx.x == 0) *gave_up = 0;
    __syncthreads();
  }

  GCS_DEV ll_word *halo_slot(int group, int side) const {
    return comm.halo + ((((hseq & 1) * 2 + h) * (long)groups + group) * 2 + side) *
                           (KP * 2 * 64);
  }

  // Start sending the boundary rings of v to the neighbour workgroups.
  GCS_DEV void send(const double v[KP]) {
    ++hseq;
    for (int side = 0; side < 2; ++side) {
      // side 0: my first ring is the upper ghost of workgroup g - 1
      const bool mine = own && (side == 0 ? w == 1 && g > 0 : w == nown && g + 1 < groups);
      if (!mine) continue;
      ll_word *s = halo_slot(side == 0 ? g - 1 : g + 1, side == 0 ? 1 : 0);
#pragma unroll
      for (int t = 0; t < KP; ++t)
        if (t < cnt) ll_put(s + (2 * t) * 64 + lane, s + (2 * t + 1) * 64 + lane, v[t], hseq);
    }
  }

  // Ghost wavefronts: v of the ghost ring, sent by its owner.
  GCS_DEV void receive(double v[KP]) {
    if (!ghost) return;
    const ll_word *s = halo_slot(g, w == 0 ? 0 : 1);
    int spin = 0;
    do {
      ll_word a[KP], b[KP];
      bool ok = true;
#pragma unroll
      for (int t = 0; t < KP; ++t)
        if (t < cnt) {
          a[t] = ll_load(s + (2 * t) * 64 + lane);
          b[t] = ll_load(s + (2 * t + 1) * 64 + lane);
        }
#pragma unroll
      for (int t = 0; t < KP; ++t)
        if (t < cnt) ok = ok && (unsigned)a[t] == hseq && (unsigned)b[t] == hseq;
      if (__all(ok)) {
#pragma unroll
        for (int t = 0; t < KP; ++t)
          if (t < cnt) v[t] = ll_value(a[t], b[t]);
        return;
      }
    } while (++spin < comm.spins);
    *gave_up = 1;
  }

  // Sums of NV values over the hemisphere (ghosts and idle wavefronts give
  // zero), the same in every thread of it.
  template <int NV>
  GCS_DEV void sum(double (&v)[NV]) {
    ++seq;
#pragma unroll
    for (int n = 0; n < NV; ++n) {
      const double s = wave_sum(own ? v[n] : 0.0);
      if (lane == 0) part[n][w] = s;
    }
    __syncthreads();
    if (w == 0) {
      ll_word *bank = comm.red + (((seq & 1) * 2 + h) * (long)groups) * (kRingSums * 2);
      if (lane < NV) {
        double s = 0.0;
        for (int q = 0; q < kRingWaves; ++q) s += part[lane][q];
        ll_word *mine = bank + (g * kRingSums + lane) * 2;
        ll_put(mine, mine + 1, s, seq);
      }
      double acc[NV];
#pragma unroll
      for (int n = 0; n < NV; ++n) acc[n] = 0.0;
      bool got = true;
      for (int q = lane; q < (groups + 63) / 64 * 64; q += 64) {
        const ll_word *slot = bank + (long)min(q, groups - 1) * (kRingSums * 2);
        int spin = 0;
        bool here = false;
        do {
          ll_word a[NV], b[NV];
          bool ok = true;
#pragma unroll
          for (int n = 0; n < NV; ++n) {
            a[n] = ll_load(slot + 2 * n);
            b[n] = ll_load(slot + 2 * n + 1);
          }
#pragma unroll
          for (int n = 0; n < NV; ++n)
            ok = ok && (unsigned)a[n] == seq && (unsigned)b[n] == seq;
          here = __all(ok);
          if (here) {
#pragma unroll
            for (int n = 0; n < NV; ++n)
              if (q < groups) acc[n] += ll_value(a[n], b[n]);
          }
        } while (!here && ++spin < comm.spins);
        got = got && here;
      }
#pragma unroll
      for (int n = 0; n < NV; ++n) {
        const double s = wave_sum(acc[n]);
        if (lane == 0) total[n] = s;
      }
      if (lane == 0) {
        if (!got) *gave_up = 1;
        // one thread's reading, so that the workgroup leaves together
        total[kRingSums] = *(volatile int *)gave_up != 0 ? 1.0 : 0.0;
      }
    }
    __syncthreads();
#pragma unroll
    for (int n = 0; n < NV; ++n) v[n] = total[n];
    dead = dead || total[kRingSums] != 0.0;
  }

  // At the end: whether a wait was given up, in the hemisphere's results (the
  // same value from every workgroup that says so).
  GCS_DEV void report(const MiK &c) const {
    __syncthreads();
    if (threadIdx.x == 0 && *gave_up != 0) c.sl(h)[SL_GAVE_UP] = 1.0;
  }

  // Put v into this wavefront's LDS row, for the neighbour rings.
  GCS_DEV void publish(const double v[KP]) {
    if (own || ghost)
#pragma unroll
      for (int t = 0; t < KP; ++t) rows[w][t * 64 + lane] = v[t];
    __syncthreads();
  }

  // v at j - 1 of this lane's first point and at j + 1 of its last one.
  GCS_DEV void ends(const double v[KP], double &left, double &right) const {
    const double lv = v[KP - 1];
    double mine_last = v[0];
#pragma unroll
    for (int t = 0; t < KP; ++t)
      if (t == last_t) mine_last = v[t];
    // the lane reads stand outside the selections: under a branch, the value
    // read would be computed for the branch's own lanes only
    const double before = dpp_move<DPP_WAVE_SHR1>(0.0, lv), end = read_lane(mine_last, last_lane);
    const double after = dpp_move<DPP_WAVE_SHL1>(0.0, v[0]), start = read_lane(v[0], 0);
    left = lane == 0 ? end : before;
    right = lane == last_lane ? start : after;
  }
};

// The ring's row of the operator (uniform along the ring) and the pole's.
struct RingRow {
  double diag, lo, hi, llo, lhi;  // tensor: coefficients as k_mi_setup stores them
  double w, plo, phi, plon;       // Pedersen: k_mi_apply's factors
  double pe, pole_diag;
};

// out = A v on own rings (v published), and the pole row in the wavefront
// of ring 1; k_mi_apply's arithmetic.
template <int KP, bool Tensor>
GCS_DEV void ring_product(const MiK &c, const RingWave<KP> &s, const RingRow &row,
                          const double v[KP], double v_pole, double out[KP], double &out_pole) {
  if (!s.own) return;
  double left, right;
  s.ends(v, left, right);
  const bool first = s.ring == 1, last = s.ring == c.nt - 2;
  double below[KP], above[KP];
#pragma unroll
  for (int t = 0; t < KP; ++t) {
    below[t] = first ? v_pole : s.rows[s.w - 1][t * 64 + s.lane];
    above[t] = last ? 0.0 : s.rows[s.w + 1][t * 64 + s.lane];
  }
  double ring = 0.0;
#pragma unroll
  for (int t = 0; t < KP; ++t) {
    const double vm = t == 0 ? left : v[t - 1];
    const double vp = (t == KP - 1 || t == s.cnt - 1) ? right : v[t < KP - 1 ? t + 1 : t];
    if (Tensor)
      out[t] = row.diag * v[t] + row.lo * below[t] + row.hi * above[t] + row.llo * vm +
               row.lhi * vp;
    else
      out[t] = row.w * (row.plo * (v[t] - below[t]) + row.phi * (v[t] - above[t]) +
                        row.plon * (2.0 * v[t] - vm - vp));
    if (t < s.cnt) ring += v[t];
    if (t >= s.cnt) out[t] = 0.0;
  }
  if (first) {
    ring = wave_sum(ring);
    out_pole = Tensor ? row.pole_diag * v_pole - row.pe * ring
                      : row.pe * ((double)c.np * v_pole - ring);
  }
}

template <int KP>
GCS_DEV double ring_dot(const double a[KP], const double b[KP]) {
  double s = 0.0;
#pragma unroll
  for (int t = 0; t < KP; ++t) s += a[t] * b[t];
  return s;
}

// Constants of the wavefront's ring; rings of the tensor system also need
// the sums' weight of the unweighted residual (orig_term).
template <int KP, bool Tensor>
GCS_DEV RingRow ring_row(const MiK &c, const RingWave<KP> &s, double &inv_sin2, double &ps) {
  RingRow r = {};
  const double dt = c.max_colat / (double)(c.nt - 1);
  const double dp = 2.0 * kPi / (double)c.np;
  const double half = 0.5 * dt;
  r.pe = sin(half) * c.pedersen / (incl2(half) * dt * dt);
  ps = (double)c.np * r.pe;
  r.pole_diag = c.vec(s.h, V_DIAG)[0];
  inv_sin2 = 0.0;
  if (!s.own && !s.ghost) return r;
  const int base = red_at(c.np, s.ring, 0);
  const double th = (double)s.ring * dt;
  r.diag = c.vec(s.h, V_DIAG)[base];
  if (Tensor) {
    r.lo = c.vec(s.h, V_LO)[base];
    r.hi = c.vec(s.h, V_HI)[base];
    r.llo = c.vec(s.h, V_LLO)[base];
    r.lhi = c.vec(s.h, V_LHI)[base];
  } else {
    r.w = sin(th);
    r.plo = theta_coeff(c.pedersen, th - 0.5 * dt, th, dt);
    r.phi = theta_coeff(c.pedersen, th + 0.5 * dt, th, dt);
    r.plon = c.pedersen / (sin(th) * sin(th) * dp * dp);
  }
  inv_sin2 = 1.0 / (sin(th) * sin(th));
  return r;
}

template <int KP>
GCS_DEV void ring_load(const RingWave<KP> &s, const MiK &c, const double *vec, double out[KP]) {
  const int base = red_at(c.np, max(s.ring, 1), 0);
#pragma unroll
  for (int t = 0; t < KP; ++t)
    out[t] = (s.own || s.ghost) && t < s.cnt ? vec[base + s.j0 + t] : 0.0;
}

// The solved potential to the polar grid: pole row, rings, zero outer row.
template <int KP>
GCS_DEV void ring_store(const RingWave<KP> &s, const MiK &c, const double x[KP], double x_pole) {
  double *pot = c.potential + (long)s.h * c.nt * c.np;
  if (!s.own) return;
#pragma unroll
  for (int t = 0; t < KP; ++t)
    if (t < s.cnt) {
      const int j = s.j0 + t;
      pot[(long)s.ring * c.np + j] = x[t];
      if (s.ring == 1) pot[j] = x_pole;
      if (s.ring == c.nt - 2) pot[(long)(c.nt - 1) * c.np + j] = 0.0;
    }
}

// Jacobi-preconditioned CG on the reduced Pedersen system (:516-600), with
// its two dot products and the residual norm in one reduction: A p follows
// from A z by the recurrence of p, and p . A p from z . A z (Chronopoulos and
// Gear, J. Comput. Appl. Math. 25, 1989). The iterates are CG's up to
// rounding; convergence is decided on the true residual, as before.
template <int KP>
__global__ void __launch_bounds__(kRingThreads) k_ring_cg(MiK c, RingComm comm, double rel_tol,
                                                          int maxit) {
  __shared__ double rows[kRingWaves][64 * KP], part[kRingSums][kRingWaves], total[kRingSums + 1];
  __shared__ int gave_up;
  RingWave<KP> s;
  s.init(c, comm, rows, part, total, &gave_up);
  double is2, ps;
  const RingRow row = ring_row<KP, false>(c, s, is2, ps);
  const bool pole = s.own && s.ring == 1;     // carries the pole unknown
  const bool pole_lane = pole && s.lane == 0; // adds it to the sums
  const double inv_diag = (s.own || s.ghost) ? 1.0 / row.diag : 0.0;
  const double inv_pole = 1.0 / row.pole_diag;
  // u = z of the current residual, w = A u, p and s = A p
  double x[KP], r[KP], u[KP], w[KP], p[KP], sv[KP];
  double x0, r0, u0 = 0.0, w0 = 0.0, p0 = 0.0, s0 = 0.0;
  // r = rhs - A x, sent to the ghosts; b2 = this wavefront's part of |rhs|^2
  auto residual = [&](double &b2) {
    double rhs[KP];
    ring_load<KP>(s, c, c.vec(s.h, V_RHS), rhs);
    s.publish(x);
    ring_product<KP, false>(c, s, row, x, x0, w, w0);
    if (s.own)
#pragma unroll
      for (int t = 0; t < KP; ++t) r[t] = rhs[t] - w[t];
    r0 = c.vec(s.h, V_RHS)[0] - w0;
    b2 = ring_dot<KP>(rhs, rhs) * is2;
    s.send(r);
  };
  // |r|^2 of the unweighted equations
  auto norm_part = [&]() {
    return ring_dot<KP>(r, r) * is2 + (pole_lane ? (double)c.np * (r0 / ps) * (r0 / ps) : 0.0);
  };
#pragma unroll
  for (int t = 0; t < KP; ++t) r[t] = u[t] = w[t] = p[t] = sv[t] = 0.0;
  ring_load<KP>(s, c, c.vec(s.h, V_X), x);
  x0 = c.vec(s.h, V_X)[0];
  double v2[2];
  residual(v2[1]);
  v2[0] = norm_part();
  s.sum(v2);
  s.receive(r);
  double norm = sqrt(fmax(0.0, v2[0]));
  const double first = norm;
  const double target = rel_tol * fmax(sqrt(fmax(0.0, v2[1])), 1.0);
  SolveResult res{0, norm <= target, norm};
  bool restart = true;
  double alpha = 0.0, gamma_prev = 1.0;
  for (int it = 0; it <= maxit && !res.ok && !s.dead; ++it) {
    // r is the residual after `it` iterations
#pragma unroll
    for (int t = 0; t < KP; ++t) u[t] = r[t] * inv_diag;
    u0 = r0 * inv_pole;
    s.publish(u);
    ring_product<KP, false>(c, s, row, u, u0, w, w0);
    s.send(w);
    double v3[3] = {ring_dot<KP>(r, u) + (pole_lane ? r0 * u0 : 0.0),
                    ring_dot<KP>(w, u) + (pole_lane ? w0 * u0 : 0.0), norm_part()};
    s.sum(v3);
    s.receive(w);
    const double gamma = v3[0], delta = v3[1];
    norm = sqrt(fmax(0.0, v3[2]));
    res.iters = it;
    res.last = norm;
    if (!restart && (norm <= target || it % 1024 == 0)) {
      residual(v2[1]);
      v2[0] = norm_part();
      s.sum(v2);
      s.receive(r);
      norm = sqrt(fmax(0.0, v2[0]));
      res.last = norm;
      if (norm <= target) res.ok = true;
      restart = true;
      --it;  // the same iteration again, from the true residual
      continue;
    }
    if (it == maxit) break;
    const double beta = restart ? 0.0 : gamma / gamma_prev;
    // p . A p = u . A u - beta^2 p_prev . A p_prev, with the latter
    // gamma_prev / alpha
    const double pap = restart ? delta : delta - beta * gamma / alpha;
    if (!isfinite(gamma) || gamma <= DBL_MIN || !isfinite(pap) || pap <= DBL_MIN) break;
    alpha = gamma / pap;
    gamma_prev = gamma;
#pragma unroll
    for (int t = 0; t < KP; ++t) {
      p[t] = u[t] + (restart ? 0.0 : beta * p[t]);
      sv[t] = w[t] + (restart ? 0.0 : beta * sv[t]);
      x[t] += alpha * p[t];
      r[t] -= alpha * sv[t];
    }
    p0 = u0 + (restart ? 0.0 : beta * p0);
    s0 = w0 + (restart ? 0.0 : beta * s0);
    x0 += alpha * p0;
    r0 -= alpha * s0;
    restart = false;
  }
  ring_store<KP>(s, c, x, x0);
  if (s.g == 0) store_result(c, s.h, res, first);
  s.report(c);
}

// Factors of the ring preconditioner (ring_factor) that a lane applies.
template <int KP>
struct RingFactors {
  double ib[KP], gd[KP], zz[KP], a, corner, inv_den;
};

template <int KP>
GCS_DEV RingFactors<KP> ring_factors(const RingWave<KP> &s, const MiK &c, const RingRow &row) {
  RingFactors<KP> f = {};
  if (!s.own && !s.ghost) return f;
  const int base = red_at(c.np, s.ring, 0);
  const double *g = c.vec(s.h, V_SCR) + base, *z = c.vec(s.h, V_SCR2) + base,
               *ib = c.vec(s.h, V_IB) + base;
#pragma unroll
  for (int t = 0; t < KP; ++t) {
    const int j = s.j0 + t;
    const bool in = t < s.cnt;
    f.ib[t] = in ? ib[j] : 0.0;
    f.gd[t] = in && j < c.np - 1 ? -g[j + 1] : 0.0;
    f.zz[t] = in ? z[j] : 0.0;
  }
  f.a = row.llo;
  f.corner = row.llo / -row.diag;  // the periodic corner's weight, a / gamma
  f.inv_den = 1.0 / c.vec(s.h, V_RDEN)[base];
  return f;
}

// out = M^-1 in on the wavefront's ring: ring_apply with its operands in
// registers.
template <int KP>
GCS_DEV void ring_solve(const RingWave<KP> &s, const RingFactors<KP> &f, const double in[KP],
                        double out[KP]) {
  const int lane = s.lane;
  double fa[KP], fb[KP];
  double A = 0.0, B = 1.0;
#pragma unroll
  for (int t = 0; t < KP; ++t) {
    fa[t] = f.ib[t] * in[t];
    fb[t] = (t == 0 && lane == 0) ? 0.0 : -f.a * f.ib[t];
    if (t < s.cnt) {
      A = fa[t] + fb[t] * A;
      B = fb[t] * B;
    }
  }
  // rows of 16 lanes, then the value at the end of the rows before
  affine_step<DPP_ROW_SHR + 1>(A, B);
  affine_step<DPP_ROW_SHR + 2>(A, B);
  affine_step<DPP_ROW_SHR + 4>(A, B);
  affine_step<DPP_ROW_SHR + 8>(A, B);
  const double p1 = read_lane(A, 15);
  const double p2 = read_lane(A, 31) + read_lane(B, 31) * p1;
  const double p3 = read_lane(A, 47) + read_lane(B, 47) * p2;
  const int rowid = lane >> 4;
  A = A + B * (rowid == 0 ? 0.0 : rowid == 1 ? p1 : rowid == 2 ? p2 : p3);
  double w = dpp_move<DPP_WAVE_SHR1>(0.0, A);
  double v[KP];
#pragma unroll
  for (int t = 0; t < KP; ++t) {
    v[t] = 0.0;
    if (t < s.cnt) {
      w = fa[t] + fb[t] * w;
      v[t] = w;
    }
  }
  double C = 0.0, D = 1.0;
#pragma unroll
  for (int t = KP - 1; t >= 0; --t)
    if (t < s.cnt) {
      C = v[t] + f.gd[t] * C;
      D = f.gd[t] * D;
    }
  affine_step<DPP_ROW_SHL + 1>(C, D);
  affine_step<DPP_ROW_SHL + 2>(C, D);
  affine_step<DPP_ROW_SHL + 4>(C, D);
  affine_step<DPP_ROW_SHL + 8>(C, D);
  const double q2 = read_lane(C, 48);
  const double q1 = read_lane(C, 32) + read_lane(D, 32) * q2;
  const double q0 = read_lane(C, 16) + read_lane(D, 16) * q1;
  C = C + D * (rowid == 3 ? 0.0 : rowid == 2 ? q2 : rowid == 1 ? q1 : q0);
  w = dpp_move<DPP_WAVE_SHL1>(0.0, C);
#pragma unroll
  for (int t = KP - 1; t >= 0; --t)
    if (t < s.cnt) {
      w = v[t] + f.gd[t] * w;
      v[t] = w;
    }
  const double y0 = read_lane(v[0], 0);
  double mine_last = v[0];
#pragma unroll
  for (int t = 0; t < KP; ++t)
    if (t == s.last_t) mine_last = v[t];
  const double yl = read_lane(mine_last, s.last_lane);
  const double fact = (y0 + f.corner * yl) * f.inv_den;
#pragma unroll
  for (int t = 0; t < KP; ++t) out[t] = t < s.cnt ? v[t] - fact * f.zz[t] : 0.0;
}

// ring_factor with the ring's coefficients read once (they are uniform along
// it) and the serial recurrences in LDS: one workgroup per ring, spread over
// the chip, whose first lane factors and whose lanes store.
__global__ void __launch_bounds__(64) k_ring_factor(MiK c) {
  __shared__ double g[64 * kRingChunk], z[64 * kRingChunk], ib[64 * kRingChunk];
  const int h = blockIdx.y, np = c.np, base = red_at(np, 1 + blockIdx.x, 0);
  if (threadIdx.x == 0) {
    const double a = c.vec(h, V_LLO)[base], b = c.vec(h, V_DIAG)[base],
                 cc = c.vec(h, V_LHI)[base];
    const double gam = -b, tail = b - cc * a / gam;
    double inv = 1.0 / (b - gam), zp = gam * inv;
    ib[0] = inv;
    g[0] = 0.0;
    z[0] = zp;
    for (int j = 1; j < np; ++j) {
      const bool last = j == np - 1;
      const double gj = cc * inv;
      g[j] = gj;
      inv = 1.0 / ((last ? tail : b) - a * gj);
      ib[j] = inv;
      zp = ((last ? cc : 0.0) - a * zp) * inv;
      z[j] = zp;
    }
    const double zl = zp;
    for (int j = np - 2; j >= 0; --j) {
      zp = z[j] - g[j + 1] * zp;
      z[j] = zp;
    }
    c.vec(h, V_RDEN)[base] = 1.0 + zp + a * zl / gam;
  }
  __syncthreads();
  for (int j = threadIdx.x; j < np; j += 64) {
    c.vec(h, V_SCR)[base + j] = g[j];
    c.vec(h, V_SCR2)[base + j] = z[j];
    c.vec(h, V_IB)[base + j] = ib[j];
  }
}

// Right-preconditioned BiCGStab on the tensor system (:1029-1131). The norm
// of the new residual s - omega A s and its product with the shadow vector
// are formed from the sums that omega needs anyway, so that an iteration has
// two reductions; the norm decides only when the true residual is computed.
template <int KP>
__global__ void __launch_bounds__(kRingThreads) k_ring_bicgstab(MiK c, RingComm comm,
                                                                double rel_tol, int maxit) {
  __shared__ double rows[kRingWaves][64 * KP], part[kRingSums][kRingWaves], total[kRingSums + 1];
  __shared__ int gave_up;
  RingWave<KP> s;
  s.init(c, comm, rows, part, total, &gave_up);
  double is2, ps;
  const RingRow row = ring_row<KP, true>(c, s, is2, ps);
  const RingFactors<KP> fac = ring_factors<KP>(s, c, row);
  const bool pole = s.own && s.ring == 1;
  const bool pole_lane = pole && s.lane == 0;
  double x[KP], r[KP], p[KP], ap[KP], sh[KP], pp[KP], sv[KP], psv[KP], as[KP];
  double x0, r0, p0 = 0.0, ap0 = 0.0, sh0, pp0 = 0.0, s0 = 0.0, ps0 = 0.0, as0 = 0.0;
  // one vector's part of the squared norm of the unweighted equations
  auto norm_part = [&](const double v[KP], double v0) {
    double q = ring_dot<KP>(v, v) * is2;
    if (pole_lane) q += (double)c.np * (v0 / ps) * (v0 / ps);
    return q;
  };
  auto residual = [&](double &b2) {
    double rhs[KP];
    ring_load<KP>(s, c, c.vec(s.h, V_RHS), rhs);
    s.publish(x);
    double t0 = 0.0;
    ring_product<KP, true>(c, s, row, x, x0, as, t0);
    if (s.own)
#pragma unroll
      for (int t = 0; t < KP; ++t) r[t] = rhs[t] - as[t];
    r0 = c.vec(s.h, V_RHS)[0] - t0;
    b2 = ring_dot<KP>(rhs, rhs) * is2;
    s.send(r);
  };
#pragma unroll
  for (int t = 0; t < KP; ++t) r[t] = p[t] = ap[t] = pp[t] = sv[t] = psv[t] = as[t] = 0.0;
  ring_load<KP>(s, c, c.vec(s.h, V_X), x);
  x0 = c.vec(s.h, V_X)[0];
  double v3[3];
  residual(v3[2]);
  v3[0] = norm_part(r, r0);
  v3[1] = ring_dot<KP>(r, r) + (pole_lane ? r0 * r0 : 0.0);
  s.sum(v3);
  s.receive(r);
  double norm = sqrt(fmax(0.0, v3[0])), rho = v3[1];
  const double first = norm;
  const double target = rel_tol * fmax(sqrt(fmax(0.0, v3[2])), 1.0);
  SolveResult res{0, norm <= target, norm};
#pragma unroll
  for (int t = 0; t < KP; ++t) sh[t] = r[t];
  sh0 = r0;
  double rho_prev = 1.0, alpha = 1.0, omega = 1.0;
  for (int it = 1; it <= maxit && !res.ok && !s.dead; ++it) {
    if (!isfinite(rho) || fabs(rho) <= DBL_MIN || !isfinite(omega) || fabs(omega) <= DBL_MIN)
      break;
    const double beta = (rho / rho_prev) * (alpha / omega);
#pragma unroll
    for (int t = 0; t < KP; ++t) p[t] = r[t] + beta * (p[t] - omega * ap[t]);
    p0 = r0 + beta * (p0 - omega * ap0);
    ring_solve<KP>(s, fac, p, pp);
    pp0 = p0 / row.pole_diag;
    s.publish(pp);
    ring_product<KP, true>(c, s, row, pp, pp0, ap, ap0);
    s.send(ap);
    double v1[1] = {ring_dot<KP>(sh, ap) + (pole_lane ? sh0 * ap0 : 0.0)};
    s.sum(v1);
    s.receive(ap);
    const double den = v1[0];
    if (!isfinite(den) || fabs(den) <= DBL_MIN) break;
    alpha = rho / den;
#pragma unroll
    for (int t = 0; t < KP; ++t) sv[t] = r[t] - alpha * ap[t];
    s0 = r0 - alpha * ap0;
    ring_solve<KP>(s, fac, sv, psv);
    ps0 = s0 / row.pole_diag;
    s.publish(psv);
    ring_product<KP, true>(c, s, row, psv, ps0, as, as0);
    s.send(as);
    double v7[7] = {ring_dot<KP>(as, as), ring_dot<KP>(as, sv), ring_dot<KP>(sh, sv),
                    ring_dot<KP>(sh, as), 0.0, 0.0, norm_part(sv, s0)};
    v7[4] = v7[0] * is2;
    v7[5] = v7[1] * is2;
    if (pole_lane) {
      v7[0] += as0 * as0;
      v7[1] += as0 * s0;
      v7[2] += sh0 * s0;
      v7[3] += sh0 * as0;
      v7[4] += (double)c.np * (as0 / ps) * (as0 / ps);
      v7[5] += (double)c.np * (as0 / ps) * (s0 / ps);
    }
    s.sum(v7);
    s.receive(as);
    const double wden = v7[0], wnum = v7[1], snorm = sqrt(fmax(0.0, v7[6]));
    if (snorm <= target) {
      res.last = snorm;
      res.iters = it;
      res.ok = true;
#pragma unroll
      for (int t = 0; t < KP; ++t) x[t] += alpha * pp[t];
      x0 += alpha * pp0;
      break;
    }
    omega = wnum / wden;
    if (!isfinite(wden) || wden <= DBL_MIN || !isfinite(omega) || fabs(omega) <= DBL_MIN) break;
#pragma unroll
    for (int t = 0; t < KP; ++t) {
      x[t] += alpha * pp[t] + omega * psv[t];
      r[t] = sv[t] - omega * as[t];
    }
    x0 += alpha * pp0 + omega * ps0;
    r0 = s0 - omega * as0;
    // |r|^2 and shadow . r of r = s - omega A s, from the sums above
    double v2[2] = {v7[6] - omega * (2.0 * v7[5] - omega * v7[4]), v7[2] - omega * v7[3]};
    norm = sqrt(fmax(0.0, v2[0]));
    res.iters = it;
    res.last = norm;
    if (norm <= target || it % 256 == 0) {
      residual(v3[2]);
      v2[0] = norm_part(r, r0);
      v2[1] = ring_dot<KP>(r, r) + (pole_lane ? r0 * r0 : 0.0);
      s.sum(v2);
      s.receive(r);
      norm = sqrt(fmax(0.0, v2[0]));
      res.last = norm;
      if (norm <= target) res.ok = true;
#pragma unroll
      for (int t = 0; t < KP; ++t) {
        sh[t] = r[t];
        p[t] = ap[t] = 0.0;
      }
      sh0 = r0;
      p0 = ap0 = 0.0;
      rho = v2[1];
      rho_prev = alpha = omega = 1.0;
      continue;
    }
    rho_prev = rho;
    rho = v2[1];
  }
  ring_store<KP>(s, c, x, x0);
  if (s.g == 0) store_result(c, s.h, res, first);
  s.report(c);
}

// The kernels by points per lane, 1 .. kRingChunk.
typedef void (*RingKernel)(MiK, RingComm, double, int);
template <int KP>
RingKernel ring_kernel_of(bool tensor) {
  return tensor ? k_ring_bicgstab<KP> : k_ring_cg<KP>;
}
RingKernel ring_kernel(int points, bool tensor) {
  static_assert(kRingChunk == 8, "one case per points per lane");
  switch (points) {
    case 1: return ring_kernel_of<1>(tensor);
    case 2: return ring_kernel_of<2>(tensor);
    case 3: return ring_kernel_of<3>(tensor);
    case 4: return ring_kernel_of<4>(tensor);
    case 5: return ring_kernel_of<5>(tensor);
    case 6: return ring_kernel_of<6>(tensor);
    case 7: return ring_kernel_of<7>(tensor);
    default: return ring_kernel_of<8>(tensor);
  }
}

// ---- learned warm start ----------------------------------------------------------

// Current density equivalent to a residual row: the right-hand side of
// interior row (i, j) is -R^2 FAC cos(I) sin(theta) (:428-448), so a residual
// r there is what a current -r / (sin(theta) R^2 cos I) would add. The pole
// and outer rows carry none.
GCS_DEV double equivalent_current(double r, int i, int nt, double dt, double r2, int hemi) {
  if (i <= 0 || i >= nt - 1) return 0.0;
  const double th = (double)i * dt;
  return -(r / sin(th)) / (r2 * cos_incl(th, hemi));
}

// Network features of one point of its grid (kInChannels floats): the f x f
// fine currents of the point's block / scale in channels 0 .. f*f - 1 (row
// major; f <= 4), SigmaP / 10, SigmaH / 10, colatitude / maximum
// colatitude and hemisphere sign in channels 16 .. 19, zeros elsewhere.
constexpr int kFeatCurrent = 16, kFeatSp = 16, kFeatSh = 17, kFeatColat = 18, kFeatHemi = 19;

GCS_DEV void write_features(float *f, const double *current, int f2, double scale, double sp,
                            double sh, double colat_fraction, int hemi) {
  for (int k = 0; k < unet::kInChannels; ++k) f[k] = 0.f;
  for (int k = 0; k < f2; ++k) f[k] = scale > 0.0 ? (float)(current[k] / scale) : 0.f;
  f[kFeatSp] = (float)(sp / 10.0);
  f[kFeatSh] = (float)(sh / 10.0);
  f[kFeatColat] = (float)colat_fraction;
  f[kFeatHemi] = (float)hemi;
}

// The network runs on the polar grid pooled by f x f (f = nt / H): the
// Krylov iterations remove short-wavelength error quickly, the network
// supplies the long-wavelength part, and a coarse grid lets a 4-level
// U-Net's receptive field span the polar cap. Row of a coarse point, as a
// fraction of the fine grid's colatitude range:
GCS_DEV double coarse_row_fraction(int rc, int f, int nt) {
  return ((double)rc * f + 0.5 * (double)(f - 1)) / (double)(nt - 1);
}

// Bilinear sample of a coarse [Hc][Wc] field at fine point (i, j):
// rows clamped, columns periodic.
GCS_DEV double coarse_sample(const float *o, int Hc, int Wc, int f, int i, int j) {
  double y = ((double)i + 0.5) / f - 0.5, x = ((double)j + 0.5) / f - 0.5;
  y = fmin(fmax(y, 0.0), (double)(Hc - 1));
  const int y0 = min((int)floor(y), Hc - 2 < 0 ? 0 : Hc - 2);
  const double wy = Hc > 1 ? y - y0 : 0.0;
  const int y1 = min(y0 + 1, Hc - 1);
  const double xf = floor(x);
  const double wx = x - xf;
  int x0 = (int)xf % Wc;
  if (x0 < 0) x0 += Wc;
  const int x1 = (x0 + 1) % Wc;
  const double a = (1.0 - wx) * o[y0 * Wc + x0] + wx * o[y0 * Wc + x1];
  const double b = (1.0 - wx) * o[y1 * Wc + x0] + wx * o[y1 * Wc + x1];
  return (1.0 - wy) * a + wy * b;
}

// RMS of the residual's equivalent current over the interior rows, per
// hemisphere (one block each).
__global__ void k_warm_scale(MiK c, double *scale) {
  __shared__ double red[kT];
  const int h = blockIdx.y;
  const double dt = c.max_colat / (double)(c.nt - 1);
  const long count = (long)(c.nt - 2) * c.np;
  double sum = 0.0;
  for (long q = threadIdx.x; q < count; q += kT) {
    const int i = 1 + (int)(q / c.np), j = (int)(q % c.np);
    const double v = equivalent_current(c.vec(h, V_R)[red_at(c.np, i, j)], i, c.nt, dt, c.r2,
                                        hemi_sign(h));
    sum += v * v;
  }
  red[threadIdx.x] = sum;
  __syncthreads();
  for (int w = kT / 2; w > 0; w >>= 1) {
    if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) scale[h] = sqrt(red[0] / (double)count);
}

// Features on the coarse grid: the residual's equivalent current of each
// point of the f x f block, one channel each (space to depth).
__global__ void k_warm_features(MiK c, const double *scale, double hall, int f, float *feat) {
  const int h = blockIdx.y;
  const int Hc = c.nt / f, Wc = c.np / f;
  const long q = gtid();
  if (q >= (long)Hc * Wc) return;
  const int rc = (int)(q / Wc), cc = (int)(q % Wc);
  const double dt = c.max_colat / (double)(c.nt - 1);
  double cur[kFeatCurrent];
  for (int a = 0; a < f; ++a)
    for (int b = 0; b < f; ++b) {
      const int i = rc * f + a, j = cc * f + b;
      const double r = (i > 0 && i < c.nt - 1) ? c.vec(h, V_R)[red_at(c.np, i, j)] : 0.0;
      cur[a * f + b] = equivalent_current(r, i, c.nt, dt, c.r2, hemi_sign(h));
    }
  write_features(feat + ((long)h * Hc * Wc + q) * unet::kInChannels, cur, f * f, scale[h],
                 c.pedersen, hall, coarse_row_fraction(rc, f, c.nt), hemi_sign(h));
}

// The network's potential correction d in V_Z, interpolated from the coarse
// grid (out * out_scale * R^2 * scale / SigmaP; the pole unknown takes the
// mean over row 0); zero where the residual was zero.
__global__ void k_warm_correction(MiK c, const double *scale, const float *out,
                                  double out_scale, int f) {
  const int h = blockIdx.y;
  const long q = gtid();
  if (q >= c.n) return;
  double *d = c.vec(h, V_Z);
  const double s = scale[h];
  if (!(s > 0.0) || !isfinite(s)) {
    d[q] = 0.0;
    return;
  }
  const double k = out_scale * c.r2 * s / c.pedersen;
  const int Hc = c.nt / f, Wc = c.np / f;
  const float *o = out + (long)h * Hc * Wc;
  if (q == 0) {
    double mean = 0.0;
    for (int j = 0; j < c.np; ++j) mean += coarse_sample(o, Hc, Wc, f, 0, j);
    d[0] = k * (mean / (double)c.np);
    return;
  }
  const int i = 1 + (int)((q - 1) / c.np), j = (int)((q - 1) % c.np);
  d[q] = k * coarse_sample(o, Hc, Wc, f, i, j);
}

// Step length along the correction in the operator's energy norm:
// alpha = (d . r) / (d . A d) (r the residual of the previous potential, A d
// in V_AS) minimises the A-norm of the guess's error for the symmetric
// Pedersen operator, and weighs the long-wavelength error the Krylov
// iterations reduce slowest more than the residual norm does. One block per
// hemisphere; alpha = 0 when d . A d is not positive or not finite.
__global__ void k_warm_alpha(MiK c, double *alpha) {
  __shared__ double rn[kT], rd[kT];
  const int h = blockIdx.y;
  const double *r = c.vec(h, V_R), *d = c.vec(h, V_Z), *ad = c.vec(h, V_AS);
  double num = 0.0, den = 0.0;
  for (long q = threadIdx.x; q < c.n; q += kT) {
    num += d[q] * r[q];
    den += d[q] * ad[q];
  }
  rn[threadIdx.x] = num;
  rd[threadIdx.x] = den;
  __syncthreads();
  for (int w = kT / 2; w > 0; w >>= 1) {
    if (threadIdx.x < w) {
      rn[threadIdx.x] += rn[threadIdx.x + w];
      rd[threadIdx.x] += rd[threadIdx.x + w];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    const double a = rn[0] / rd[0];
    alpha[h] = (rd[0] > 0.0 && isfinite(a)) ? a : 0.0;
  }
}

__global__ void k_warm_update(MiK c, const double *alpha) {
  const int h = blockIdx.y;
  const long q = gtid();
  if (q >= c.n) return;
  c.vec(h, V_X)[q] += alpha[h] * c.vec(h, V_Z)[q];
}

// The guess in V_X (previous potential) becomes guess + alpha N(residual):
// the residual, the network's forward pass on both hemispheres, the
// correction d, and the energy-norm step alpha along it (which shrinks a
// correction that does not point along the error). The solve that follows
// recomputes the residual of the new guess.
int warm_start(Problem &P, const MiK &c, bool tensor) {
  MiState &m = *P.mi;
  unet::Net &n = *m.net;
  hipStream_t s = P.stream;
  const dim3 g2(blocks_of(m.n), 2);
  k_mi_apply<<<g2, kT, 0, s>>>(c, tensor ? 1 : 0, V_X, V_AP, m.active);
  k_mi_vec<<<g2, kT, 0, s>>>(c, OP_RESIDUAL, 0.0, m.active);
  k_warm_scale<<<dim3(1, 2), kT, 0, s>>>(c, m.warm_scale);
  const int f = m.nt / n.H;
  k_warm_features<<<dim3(blocks_of((long)n.H * n.W), 2), kT, 0, s>>>(c, m.warm_scale, m.hall, f,
                                                                    n.input);
  hipStream_t keep = n.stream;
  n.stream = s;
  const int rc = unet::forward_device(n, 2);
  n.stream = keep;
  if (rc != 0) return -1;
  k_warm_correction<<<g2, kT, 0, s>>>(c, m.warm_scale, n.out, n.out_scale, f);
  k_mi_apply<<<g2, kT, 0, s>>>(c, tensor ? 1 : 0, V_Z, V_AS, m.active);
  k_warm_alpha<<<dim3(1, 2), kT, 0, s>>>(c, m.warm_scale + 2);
  k_warm_update<<<g2, kT, 0, s>>>(c, m.warm_scale + 2);
  GCS_HIP(hipGetLastError());
  return 0;
}

// The polar solves of both hemispheres; 0 when both converge. Setup (right-
// hand side, guess, stencil), the optional learned correction of the guess,
// then one fused Krylov kernel per solve (both hemispheres in one launch).
int solve(Problem &P, bool tensor) {
  MiState &m = *P.mi;
  MiK c = make_mik(P);
  hipStream_t s = P.stream;
  const auto t0 = std::chrono::steady_clock::now();
  const dim3 g2(blocks_of(m.n), 2);
  const int points = (m.np + 63) / 64;
  RingComm comm{m.ring_words, nullptr, m.ring_groups, points, m.ring_spins};
  const long red = (long)RingComm::red_words(m.ring_groups);
  const long words =
      comm.red != nullptr ? red + (long)RingComm::halo_words(m.ring_groups, points) : 0;
  comm.halo = comm.red + red;
  k_mi_setup<<<g2, kT, 0, s>>>(c, tensor ? 1 : 0, m.hall, m.ring_words, words);
  if (m.net != nullptr && warm_start(P, c, tensor) != 0) return -1;
  double rel = m.cfg.relative_tolerance;
  int maxit = m.cfg.maximum_iterations;
  auto cooperative = [&](const void *kernel, int groups, int threads, void **args) {
    if (hipLaunchCooperativeKernel(kernel, dim3(groups), dim3(threads), args, 0, s) == hipSuccess)
      return true;
    (void)hipGetLastError();
    return false;
  };
  auto single_workgroups = [&]() {
    if (tensor)
      k_mi_bicgstab<<<2, kSolveThreads, 0, s>>>(c, rel, maxit);
    else
      k_mi_cg<<<2, kSolveThreads, 4 * (size_t)m.nt * sizeof(double), s>>>(c, rel, maxit);
  };
  auto expand = [&]() {
    k_mi_vec<<<dim3(blocks_of((long)m.np * m.nt), 2), kT, 0, s>>>(c, OP_EXPAND, 0.0, m.active);
  };
  auto results = [&]() -> int {
    GCS_HIP(hipGetLastError());
    GCS_HIP(hipMemcpyAsync(m.host_scal, m.scal, 2 * SL_COUNT * sizeof(double),
                           hipMemcpyDeviceToHost, s));
    GCS_HIP(hipStreamSynchronize(s));
    return 0;
  };
  bool resident = comm.red != nullptr;
  if (resident) {
    if (tensor) k_ring_factor<<<dim3(m.nt - 2, 2), 64, 0, s>>>(c);
    void *args[] = {&c, &comm, &rel, &maxit};
    resident = cooperative((const void *)ring_kernel(points, tensor), 2 * m.ring_groups,
                           kRingThreads, args);
  }
  if (!resident) {
    void *args[] = {&c, &rel, &maxit, &m.coop_slots, &m.coop_flags};
    const bool pair = tensor && m.coop_slots != nullptr &&
                      cooperative((const void *)k_mi_bicgstab_pair, 2 * kCoopBlocks,
                                  kSolveThreads, args);
    if (!pair) single_workgroups();
    expand();
  }
  if (results() != 0) return -1;
  if (resident && (m.host_scal[SL_GAVE_UP] != 0.0 || m.host_scal[SL_COUNT + SL_GAVE_UP] != 0.0)) {
    // a wait of the register-resident solve was given up (a workgroup did not
    // run for about a second): the same system with no such waits
    single_workgroups();
    expand();
    if (results() != 0) return -1;
  }
  m.solve_ms = std::chrono::duration<double, std::milli>(
                   std::chrono::steady_clock::now() - t0).count();
  bool ok = true;
  for (int h = 0; h < 2; ++h) {
    const double *sl = m.host_scal + h * SL_COUNT;
    m.iterations[h] = (int)sl[SL_ITER];
    m.final_residual[h] = sl[SL_NORM];
    m.initial_residual[h] = sl[SL_FIRST];
    m.converged[h] = sl[SL_OK] != 0.0 ? 1 : 0;
    ok = ok && sl[SL_OK] != 0.0;
  }
  if (!ok) {
    set_error("ionosphere potential solve did not converge");
    return -1;
  }
  return 0;
}

}  // namespace

int mi_create(Problem &P) {
  const gcs_problem_config &cfg = P.cfg;
  const gamera_cs_mi_dipole_config &mc = cfg.mi;
  const Layout &L = P.L;
  // cubedsphere_mi_dipole.c:45-57, :157-177
  if (mc.azimuth_points < 8 || mc.colatitude_points < 3 || mc.current_shell >= 64 ||
      !(mc.ionosphere_radius_re > 0.0) || !(mc.pedersen_siemens > 0.0) ||
      !(mc.coupling_interval_s > 0.0) || !(mc.length_norm_m > 0.0) ||
      !(mc.speed_norm_m_s > 0.0) || !(mc.mass_density_norm_kg_m3 > 0.0) ||
      mc.maximum_iterations <= 0 || !(mc.relative_tolerance > 0.0) ||
      L.nr < 3 || (int)mc.current_shell + 1 >= L.nr ||
      !(mc.ionosphere_radius_re < cfg.startup.inner_radius) ||
      !(cfg.hall_siemens >= 0.0) || mc.azimuth_points > 64 * kRingChunk) {
    set_error("invalid MI configuration (azimuth points must be 8..512)");
    return -1;
  }
  MiState *mp = new MiState();
  P.mi = mp;
  MiState &m = *mp;
  m.cfg = mc;
  m.hall = cfg.hall_siemens;
  m.np = (int)mc.azimuth_points;
  m.nt = (int)mc.colatitude_points;
  m.n = 1 + m.np * (m.nt - 2);
  m.S = L.n + 2;
  m.si = L.ghost + (int)mc.current_shell;
  m.max_colat = asin(sqrt(mc.ionosphere_radius_re / cfg.startup.inner_radius));
  const double mu0 = 4.0e-7 * acos(-1.0);
  m.b_norm = mc.speed_norm_m_s * sqrt(mu0 * mc.mass_density_norm_kg_m3);
  m.current_norm = m.b_norm / (mu0 * mc.length_norm_m);
  m.potential_norm = mc.speed_norm_m_s * m.b_norm * mc.length_norm_m;
  // centroids for the sample radius and the plans
  std::vector<double> cen(3 * L.total);
  for (int e = 0; e < 3; ++e)
    GCS_HIP(hipMemcpy(cen.data() + e * L.total, P.plane(P_CEN + e),
                      L.total * sizeof(double), hipMemcpyDeviceToHost));
  auto centroid = [&](long at, double x[3]) {
    for (int e = 0; e < 3; ++e) x[e] = cen[e * L.total + at];
  };
  double sum = 0.0;
  long count = 0;
  for (int f = 0; f < 6; ++f)
    for (int j = L.ghost; j < L.ghost + L.n; ++j)
      for (int k = L.ghost; k < L.ghost + L.n; ++k) {
        double x[3];
        centroid(L.at(f, m.si, j, k), x);
        sum += sqrt(x[0] * x[0] + x[1] * x[1] + x[2] * x[2]);
        ++count;
      }
  m.sample_radius = sum / (double)count;
  m.sample_max_colat = asin(sqrt(mc.ionosphere_radius_re / m.sample_radius));
  if (!std::isfinite(m.sample_radius) || !(m.sample_radius > cfg.startup.inner_radius)) {
    set_error("MI sample shell inside the inner radius");
    return -1;
  }
  const double qp = 0.25 * acos(-1.0);
  const int n = L.n, S = m.S, g = L.ghost;
  // B fringe on shells si-1..si+1 and the FAC fringe on si (:236-276, :308-342)
  std::vector<Bilinear> bf, ff;
  for (int f = 0; f < 6; ++f)
    for (int i = m.si - 1; i <= m.si + 1; ++i)
      for (int lj = 0; lj < S; ++lj)
        for (int lk = 0; lk < S; ++lk) {
          if (lj > 0 && lj <= n && lk > 0 && lk <= n) continue;
          const long at = L.at(f, i, g - 1 + lj, g - 1 + lk);
          double x[3], a, b;
          int df;
          centroid(at, x);
          if (!cube_inverse(x, df, a, b) || df == f) {
            set_error("MI fringe donor");
            return -1;
          }
          const double xx = (a + qp) * (double)n / (2.0 * qp) - 0.5;
          const double yy = (b + qp) * (double)n / (2.0 * qp) - 0.5;
          const int j0 = (int)fmax(0.0, fmin((double)n - 2.0, floor(xx)));
          const int k0 = (int)fmax(0.0, fmin((double)n - 2.0, floor(yy)));
          Bilinear e{};
          e.wx = xx - (double)j0;
          e.wy = yy - (double)k0;
          e.target = (int)at;
          e.base = (int)L.at(df, i, g + j0, g + k0);
          e.step = L.SK;
          bf.push_back(e);
          if (i == m.si) {
            Bilinear q = e;
            q.target = f * S * S + lj * S + lk;
            q.base = df * S * S + (j0 + 1) * S + k0 + 1;
            q.step = S;
            ff.push_back(q);
          }
        }
  // polar samples (:391-406, :344-370)
  std::vector<Bilinear> sm;
  const int np = m.np, nt = m.nt;
  const double dt = m.max_colat / (double)(nt - 1);
  const double dp = 2.0 * acos(-1.0) / (double)np;
  for (int h = 0; h < 2; ++h) {
    const double sign = h == 0 ? 1.0 : -1.0;
    for (int t = 0; t < nt; ++t) {
      const double ti = (double)t * dt;
      const bool zero = ti > m.sample_max_colat + 4e-14;
      const double arg = fmin(1.0, sin(ti) * sqrt(m.sample_radius / mc.ionosphere_radius_re));
      const double tm = asin(arg);
      for (int p = 0; p < np; ++p) {
        Bilinear e{};
        e.target = h * nt * np + t * np + p;
        if (zero) {
          e.zero = 1;
          sm.push_back(e);
          continue;
        }
        const double phi = (double)p * dp;
        const double x[3] = {m.sample_radius * sin(tm) * cos(phi),
                             m.sample_radius * sin(tm) * sin(phi),
                             sign * m.sample_radius * cos(tm)};
        int f;
        double a, b;
        if (!cube_inverse(x, f, a, b)) {
          set_error("MI sample point");
          return -1;
        }
        const double scale = (double)n / (2.0 * qp);
        const double xx = (a + qp) * scale - 0.5, yy = (b + qp) * scale - 0.5;
        const long jj = (long)floor(xx), kk = (long)floor(yy);
        if (jj < -1 || kk < -1 || jj >= n || kk >= n) {
          set_error("MI sample outside the shell");
          return -1;
        }
        e.wx = xx - (double)jj;
        e.wy = yy - (double)kk;
        e.base = f * S * S + (int)(jj + 1) * S + (int)(kk + 1);
        e.step = S;
        sm.push_back(e);
      }
    }
  }
  m.n_bfringe = (int)bf.size();
  m.n_ffringe = (int)ff.size();
  m.n_samples = (int)sm.size();
  if (upload_vec(bf, &m.bfringe) != 0 || upload_vec(ff, &m.ffringe) != 0 ||
      upload_vec(sm, &m.samples) != 0)
    return -1;
  const long polar = 2L * nt * np;
  GCS_HIP(hipMalloc(&m.shell_fac, 6L * S * S * sizeof(double)));
  GCS_HIP(hipMalloc(&m.shell_current, 18L * L.n * L.n * sizeof(double)));
  GCS_HIP(hipMemset(m.shell_current, 0, 18L * L.n * L.n * sizeof(double)));
  GCS_HIP(hipMalloc(&m.fac, polar * sizeof(double)));
  GCS_HIP(hipMalloc(&m.potential, polar * sizeof(double)));
  GCS_HIP(hipMalloc(&m.drift, 18L * L.ghost * L.NJ * L.NK * sizeof(double)));
  GCS_HIP(hipMalloc(&m.work, 2L * kVectors * m.n * sizeof(double)));
  {
    // the register-resident solves and the one by grid-wide barriers need all
    // their workgroups resident at once; GCS_MI_COOPERATIVE=0 selects the
    // single-workgroup solves instead (for tools that cannot follow a
    // cooperative launch, such as the kernel tracer of rocprofv3 7.2, which
    // faults at exit after one)
    const char *env = std::getenv("GCS_MI_COOPERATIVE");
    const bool allowed = env == nullptr || std::strcmp(env, "0") != 0;
    const int points = (m.np + 63) / 64, groups = (m.nt - 2 + kRingOwn - 1) / kRingOwn;
    int dev = 0, coop = 0, per_cu = 0, cus = 0;
    if (allowed && hipGetDevice(&dev) == hipSuccess &&
        hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, dev) == hipSuccess &&
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess &&
        hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &per_cu, (const void *)ring_kernel(points, m.hall > 0.0), kRingThreads, 0) ==
            hipSuccess &&
        coop != 0) {
      if ((long)per_cu * cus >= 2L * groups) {
        // GCS_MI_SPIN_LIMIT is for tests of the solve after a wait that was
        // given up
        const char *spins = std::getenv("GCS_MI_SPIN_LIMIT");
        m.ring_spins = spins != nullptr ? std::atoi(spins) : kSpinLimit;
        m.ring_groups = groups;
        GCS_HIP(hipMalloc(&m.ring_words, (RingComm::red_words(groups) +
                                          RingComm::halo_words(groups, points)) *
                                             sizeof(ll_word)));
      } else if (m.hall > 0.0 &&
                 hipOccupancyMaxActiveBlocksPerMultiprocessor(
                     &per_cu, k_mi_bicgstab_pair, kSolveThreads, 0) == hipSuccess &&
                 per_cu * cus >= 2 * kCoopBlocks) {
        GCS_HIP(hipMalloc(&m.coop_slots, 8 * kCoopBlocks * sizeof(double)));
        GCS_HIP(hipMalloc(&m.coop_flags, 4 * sizeof(int)));
      }
    }
    (void)hipGetLastError();
  }
  GCS_HIP(hipMalloc(&m.scal, 2 * SL_COUNT * sizeof(double)));
  GCS_HIP(hipHostMalloc(&m.host_scal, 2 * SL_COUNT * sizeof(double)));
  GCS_HIP(hipMalloc(&m.active, 2 * sizeof(int)));
  const int act[2] = {1, 1};
  GCS_HIP(hipMemcpy(m.active, act, sizeof(act), hipMemcpyHostToDevice));
  GCS_HIP(hipMemset(m.shell_fac, 0, 6L * S * S * sizeof(double)));
  GCS_HIP(hipMemset(m.fac, 0, polar * sizeof(double)));
  GCS_HIP(hipMemset(m.potential, 0, polar * sizeof(double)));
  GCS_HIP(hipMemset(m.work, 0, 2L * kVectors * m.n * sizeof(double)));
  GCS_HIP(hipMemset(m.scal, 0, 2 * SL_COUNT * sizeof(double)));
  // the view the step kernels read (potential set once ready)
  MiView &v = P.mi_view;
  v = MiView();
  v.np = np;
  v.nt = nt;
  v.ri = mc.ionosphere_radius_re;
  v.max_colat = m.max_colat;
  v.potential_norm = m.potential_norm;
  v.length_norm = mc.length_norm_m;
  v.speed_norm = mc.speed_norm_m_s;
  v.b_norm = m.b_norm;
  for (int e = 0; e < 3; ++e) v.moment[e] = cfg.startup.dipole.moment.value[e];
  v.cut_radius = cfg.startup.cut_radius;
  v.cut_length = cfg.startup.cut_length;
  return 0;
}

void mi_destroy(Problem &P) {
  MiState *m = P.mi;
  if (m == nullptr) return;
  (void)hipFree(m->shell_fac);
  (void)hipFree(m->shell_current);
  (void)hipFree(m->fac);
  (void)hipFree(m->potential);
  (void)hipFree(m->drift);
  (void)hipFree(m->work);
  (void)hipFree(m->scal);
  (void)hipFree(m->bfringe);
  (void)hipFree(m->ffringe);
  (void)hipFree(m->samples);
  (void)hipFree(m->active);
  if (m->host_scal) (void)hipHostFree(m->host_scal);
  (void)hipFree(m->warm_scale);
  (void)hipFree(m->ring_words);
  (void)hipFree(m->coop_slots);
  (void)hipFree(m->coop_flags);
  delete m;
  P.mi = nullptr;
}

// cubedsphere_mi_dipole.c:372-436
int mi_maybe_update(Problem &P, double time_code) {
  MiState *mp = P.mi;
  if (mp == nullptr) return 0;
  MiState &m = *mp;
  const double ts = time_code * m.cfg.length_norm_m / m.cfg.speed_norm_m_s;
  if (m.ready && !(ts + 1e-10 >= m.next_update)) return 0;
  mark_stage(P, S_MI);
  if (mi_sample_current(P) != 0) return -1;
  if (solve(P, m.hall > 0.0) != 0) return -1;
  m.ready = true;
  m.epoch = ts;
  ++m.updates;
  do {
    m.next_update += m.cfg.coupling_interval_s;
  } while (m.next_update <= ts + 1e-10);
  if (refresh_mi_drift(P, m.potential, m.drift) != 0) return -1;
  P.mi_view.potential = m.potential;
  return 1;
}

const double *mi_drift_cache(const Problem &P) {
  return P.mi != nullptr && P.mi->drift != nullptr && P.mi_view.potential != nullptr &&
                 P.mi_view.potential == P.mi->potential
             ? P.mi->drift
             : nullptr;
}

// The field-aligned current of the current state on the polar grids
// (:223-370): shell FAC, its fringe, bilinear samples.
int mi_sample_current(Problem &P) {
  MiState &m = *P.mi;
  MiK c = make_mik(P);
  hipStream_t s = P.stream;
  const Layout &L = P.L;
  k_mi_copy_shell<<<blocks_of(6L * 3 * L.NJ * L.NK), kT, 0, s>>>(c);
  k_mi_fringe_b<<<blocks_of(m.n_bfringe), kT, 0, s>>>(c, m.bfringe, m.n_bfringe);
  k_mi_shell_fac<<<blocks_of(6L * L.n * L.n), kT, 0, s>>>(c, m.shell_current);
  // the copy above used the face-velocity planes, where a fidelity step's
  // update leaves the stress rates
  P.rates_stored = false;
  k_mi_bilinear<<<blocks_of(m.n_ffringe), kT, 0, s>>>(m.ffringe, m.n_ffringe, m.shell_fac,
                                                     m.shell_fac);
  k_mi_bilinear<<<blocks_of(m.n_samples), kT, 0, s>>>(m.samples, m.n_samples, m.shell_fac,
                                                      m.fac);
  GCS_HIP(hipGetLastError());
  StepScalars sc;
  if (read_scalars(P, sc) != 0) return -1;
  if (sc.failed) {
    set_error("MI field-aligned current failed at stage " + std::to_string(sc.fail_stage));
    return -1;
  }
  return 0;
}

void mi_report(const Problem &P, MiReport &out) {
  std::memset(&out, 0, sizeof(out));
  if (P.mi == nullptr) return;
  const MiState &m = *P.mi;
  out.updates = m.updates;
  out.ready = m.ready;
  for (int h = 0; h < 2; ++h) {
    out.iterations[h] = m.iterations[h];
    out.final_residual[h] = m.final_residual[h];
  }
  out.epoch_s = m.epoch;
  out.solve_ms = m.solve_ms;
}

void mi_info(const Problem &P, MiInfo &out) {
  out = MiInfo();
  if (P.mi == nullptr) return;
  const MiState &m = *P.mi;
  out.ready = m.ready;
  out.updates = m.updates;
  out.epoch_s = m.epoch;
  out.next_update_s = m.next_update;
  out.sample_radius = m.sample_radius;
  out.max_colat = m.max_colat;
  out.potential_norm = m.potential_norm;
  out.potential = m.potential;
  for (int h = 0; h < 2; ++h) {
    out.iterations[h] = m.iterations[h];
    out.initial_residual[h] = m.initial_residual[h];
    out.final_residual[h] = m.final_residual[h];
    out.converged[h] = m.converged[h];
  }
}

void mi_view_enable(Problem &P, bool on) {
  P.mi_view.potential = on && P.mi != nullptr && P.mi->ready ? P.mi->potential : nullptr;
}

int mi_import_potential(Problem &P, const double *values, double epoch_s,
                        double next_update_s) {
  if (P.mi == nullptr) {
    set_error("MI is not enabled");
    return -1;
  }
  MiState &m = *P.mi;
  GCS_HIP(hipStreamSynchronize(P.stream));
  GCS_HIP(hipMemcpy(m.potential, values, 2L * m.nt * m.np * sizeof(double),
                    hipMemcpyHostToDevice));
  m.epoch = epoch_s;
  m.next_update = next_update_s;
  m.ready = true;
  if (refresh_mi_drift(P, m.potential, m.drift) != 0) return -1;
  P.mi_view.potential = m.potential;
  return 0;
}

int mi_shell_current(Problem &P, std::vector<double> &out) {
  if (P.mi == nullptr) {
    set_error("MI is not enabled");
    return -1;
  }
  out.resize(18L * P.L.n * P.L.n);
  GCS_HIP(hipStreamSynchronize(P.stream));
  GCS_HIP(hipMemcpy(out.data(), P.mi->shell_current, out.size() * sizeof(double),
                    hipMemcpyDeviceToHost));
  return 0;
}

int mi_download(Problem &P, int what, std::vector<double> &out) {
  if (P.mi == nullptr) {
    set_error("MI is not enabled");
    return -1;
  }
  const MiState &m = *P.mi;
  out.resize(2L * m.nt * m.np);
  GCS_HIP(hipStreamSynchronize(P.stream));
  GCS_HIP(hipMemcpy(out.data(), what == 0 ? m.potential : m.fac,
                    out.size() * sizeof(double), hipMemcpyDeviceToHost));
  return 0;
}


// ---- training pairs for the warm-start network ------------------------------------
//
// A pair is a potential and the field-aligned current for which it solves the
// polar system exactly: a random smooth potential (Gaussian bumps in
// colatitude times von Mises bumps in longitude, tapered to zero at the
// low-latitude edge, the pole row set to the mean of the first ring as the
// reduced system's pole equation requires) is multiplied by the tensor
// operator of a uniform (SigmaP, SigmaH), and the interior rows of the product
// are turned back into the current that produces them.

namespace {

constexpr int kBumps = 6;

struct GenSample {
  int hemi;
  double sp, sh;
  double amp[kBumps], th[kBumps], sth[kBumps], ph[kBumps], kap[kBumps];
};

__global__ void k_gen_potential(const GenSample *smp, int nt, int np, double max_colat,
                                double *phi) {
  const int b = blockIdx.y;
  const long q = gtid();
  if (q >= (long)nt * np) return;
  const int i = (int)(q / np), j = (int)(q % np);
  const double dt = max_colat / (double)(nt - 1), dp = 2.0 * kPi / (double)np;
  const double th = (double)i * dt, ph = (double)j * dp;
  const GenSample &g = smp[b];
  double v = 0.0;
  for (int k = 0; k < kBumps; ++k) {
    const double d = (th - g.th[k]) / g.sth[k];
    v += g.amp[k] * exp(-0.5 * d * d) * exp(g.kap[k] * (cos(ph - g.ph[k]) - 1.0));
  }
  const double taper = 1.0 - (th / max_colat) * (th / max_colat);
  phi[(long)b * nt * np + q] = i == nt - 1 ? 0.0 : taper * v;
}

// Pole row = mean of ring 1 (one block per sample).
__global__ void k_gen_pole(int nt, int np, double *phi) {
  __shared__ double red[kT];
  double *p = phi + (long)blockIdx.x * nt * np;
  double sum = 0.0;
  for (int j = threadIdx.x; j < np; j += kT) sum += p[np + j];
  red[threadIdx.x] = sum;
  __syncthreads();
  for (int w = kT / 2; w > 0; w >>= 1) {
    if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  const double mean = red[0] / (double)np;
  for (int j = threadIdx.x; j < np; j += kT) p[j] = mean;
}

__global__ void k_gen_current(const GenSample *smp, int nt, int np, double max_colat,
                              double r2, const double *phi, double *fac) {
  const int b = blockIdx.y;
  const long q = gtid();
  if (q >= (long)nt * np) return;
  const int i = (int)(q / np), j = (int)(q % np);
  const long base = (long)b * nt * np;
  if (i == 0 || i == nt - 1) {
    fac[base + q] = 0.0;
    return;
  }
  const GenSample &g = smp[b];
  const double dt = max_colat / (double)(nt - 1), dp = 2.0 * kPi / (double)np;
  const TensorRow t = tensor_row(g.sp, g.sh, i, dt, dp, g.hemi);
  const double *p = phi + base;
  const int jm = j == 0 ? np - 1 : j - 1, jp = j + 1 == np ? 0 : j + 1;
  const double below = p[(long)(i - 1) * np + (i == 1 ? 0 : j)];
  const double above = i + 2 < nt ? p[(long)(i + 1) * np + j] : 0.0;
  const double y = t.diag * p[q] + t.lo * below + t.hi * above + t.llo * p[(long)i * np + jm] +
                   t.lhi * p[(long)i * np + jp];
  fac[base + q] = equivalent_current(y, i, nt, dt, r2, g.hemi);
}

// RMS of the current over the interior rows (one block per sample).
__global__ void k_gen_scale(int nt, int np, const double *fac, double *scale) {
  __shared__ double red[kT];
  const double *f = fac + (long)blockIdx.x * nt * np;
  const long count = (long)(nt - 2) * np;
  double sum = 0.0;
  for (long q = threadIdx.x; q < count; q += kT) sum += f[np + q] * f[np + q];
  red[threadIdx.x] = sum;
  __syncthreads();
  for (int w = kT / 2; w > 0; w >>= 1) {
    if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) scale[blockIdx.x] = sqrt(red[0] / (double)count);
}

// Features and targets on the coarse grid: the fine currents of each f x f
// block as channels, the block mean of the potential as the target.
__global__ void k_gen_features(const GenSample *smp, int nt, int np, int f, double r2,
                               const double *fac, const double *phi, const double *scale,
                               double out_scale, float *feat, float *target) {
  const int b = blockIdx.y;
  const int Hc = nt / f, Wc = np / f;
  const long q = gtid();
  if (q >= (long)Hc * Wc) return;
  const int rc = (int)(q / Wc), cc = (int)(q % Wc);
  const GenSample &g = smp[b];
  const long base = (long)b * nt * np;
  double cur[kFeatCurrent], pot = 0.0;
  for (int a = 0; a < f; ++a)
    for (int e = 0; e < f; ++e) {
      const long at = base + (long)(rc * f + a) * np + cc * f + e;
      cur[a * f + e] = fac[at];
      pot += phi[at];
    }
  pot /= (double)(f * f);
  const long out = (long)b * Hc * Wc + q;
  write_features(feat + out * unet::kInChannels, cur, f * f, scale[b], g.sp, g.sh,
                 coarse_row_fraction(rc, f, nt), g.hemi);
  target[out] = (float)(pot * g.sp / (r2 * scale[b] * out_scale));
}

// A batch of random pair parameters (host side, seeded).
void draw_samples(std::mt19937_64 &rng, int count, double max_colat, double sp_lo,
                  double sp_hi, double sh_lo, double sh_hi, GenSample *out) {
  std::uniform_real_distribution<double> u(0.0, 1.0);
  std::normal_distribution<double> z(0.0, 1.0);
  for (int b = 0; b < count; ++b) {
    GenSample &g = out[b];
    g.hemi = u(rng) < 0.5 ? GAMERA_MI_NORTH : GAMERA_MI_SOUTH;
    g.sp = sp_lo + (sp_hi - sp_lo) * u(rng);
    g.sh = sh_lo + (sh_hi - sh_lo) * u(rng);
    for (int k = 0; k < kBumps; ++k) {
      g.amp[k] = z(rng);
      g.th[k] = max_colat * (0.05 + 0.85 * u(rng));
      g.sth[k] = max_colat * (0.03 + 0.22 * u(rng));
      g.ph[k] = 2.0 * kPi * u(rng);
      g.kap[k] = 0.3 + 8.0 * u(rng);
    }
  }
}

}  // namespace

// Device buffers of a pair generator for `batch` samples on an nt x np grid.
struct PairBatch {
  GenSample *host = nullptr, *dev = nullptr;
  double *phi = nullptr, *fac = nullptr, *scale = nullptr;
  int batch = 0;
  ~PairBatch() {
    if (host) (void)hipHostFree(host);
    (void)hipFree(dev);
    (void)hipFree(phi);
    (void)hipFree(fac);
    (void)hipFree(scale);
  }
  int allocate(int b, int nt, int np) {
    batch = b;
    GCS_HIP(hipHostMalloc(&host, b * sizeof(GenSample)));
    GCS_HIP(hipMalloc(&dev, b * sizeof(GenSample)));
    GCS_HIP(hipMalloc(&phi, (size_t)b * nt * np * sizeof(double)));
    GCS_HIP(hipMalloc(&fac, (size_t)b * nt * np * sizeof(double)));
    GCS_HIP(hipMalloc(&scale, (size_t)b * sizeof(double)));
    return 0;
  }
};

// Potentials and currents of host->dev samples on stream s.
static int make_pairs(PairBatch &pb, int nt, int np, double max_colat, double r2,
                      hipStream_t s) {
  GCS_HIP(hipMemcpyAsync(pb.dev, pb.host, pb.batch * sizeof(GenSample), hipMemcpyHostToDevice,
                         s));
  const dim3 g(blocks_of((long)nt * np), pb.batch);
  k_gen_potential<<<g, kT, 0, s>>>(pb.dev, nt, np, max_colat, pb.phi);
  k_gen_pole<<<pb.batch, kT, 0, s>>>(nt, np, pb.phi);
  k_gen_current<<<g, kT, 0, s>>>(pb.dev, nt, np, max_colat, r2, pb.phi, pb.fac);
  k_gen_scale<<<pb.batch, kT, 0, s>>>(nt, np, pb.fac, pb.scale);
  GCS_HIP(hipGetLastError());
  return 0;
}

// The pooling factor f of a network for this MI grid (nt = f H, np = f W),
// or 0 when the grids do not fit.
static int coarsening(const MiState &m, const unet::Net &n) {
  if (n.H <= 0 || n.W <= 0 || m.nt % n.H != 0 || m.np % n.W != 0) return 0;
  const int f = m.nt / n.H;
  return m.np / n.W == f && f * f <= kFeatCurrent ? f : 0;
}

int mi_attach_warm_start(Problem &P, unet::Net *net) {
  if (P.mi == nullptr) {
    set_error("MI is not enabled");
    return -1;
  }
  MiState &m = *P.mi;
  if (net != nullptr && (coarsening(m, *net) <= 0 || net->max_batch < 2)) {
    set_error("warm-start network grid must be the MI grid (colatitude x azimuth) pooled "
              "by one factor in both directions, and its batch at least 2");
    return -1;
  }
  if (m.warm_scale == nullptr) GCS_HIP(hipMalloc(&m.warm_scale, 4 * sizeof(double)));
  m.net = net;
  return 0;
}

int mi_make_pairs(Problem &P, uint64_t seed, int count, double sp, double sh, double *fac_out,
                  double *phi_out) {
  if (P.mi == nullptr || count <= 0) {
    set_error(P.mi == nullptr ? "MI is not enabled" : "count must be positive");
    return -1;
  }
  const MiState &m = *P.mi;
  const double rm = m.cfg.ionosphere_radius_re * m.cfg.length_norm_m;
  PairBatch pb;
  if (pb.allocate(count, m.nt, m.np) != 0) return -1;
  std::mt19937_64 rng(seed);
  draw_samples(rng, count, m.max_colat, sp, sp, sh, sh, pb.host);
  for (int b = 0; b < count; ++b) pb.host[b].hemi = b % 2 == 0 ? GAMERA_MI_NORTH : GAMERA_MI_SOUTH;
  if (make_pairs(pb, m.nt, m.np, m.max_colat, rm * rm, P.stream) != 0) return -1;
  GCS_HIP(hipStreamSynchronize(P.stream));
  const size_t bytes = (size_t)count * m.nt * m.np * sizeof(double);
  GCS_HIP(hipMemcpy(fac_out, pb.fac, bytes, hipMemcpyDeviceToHost));
  GCS_HIP(hipMemcpy(phi_out, pb.phi, bytes, hipMemcpyDeviceToHost));
  return 0;
}

int mi_train_warm_start(Problem &P, unet::Net &n, const gcs_warm_train_config &t,
                        float *loss_history) {
  if (P.mi == nullptr) {
    set_error("MI is not enabled");
    return -1;
  }
  const MiState &m = *P.mi;
  if (coarsening(m, n) <= 0 || unet::check_batch(n, t.batch) != 0 || t.steps <= 0 ||
      !(t.learning_rate > 0.0) || !(t.pedersen_min > 0.0) ||
      !(t.pedersen_max >= t.pedersen_min) || !(t.hall_min >= 0.0) ||
      !(t.hall_max >= t.hall_min)) {
    set_error("invalid warm-start training configuration");
    return -1;
  }
  const double rm = m.cfg.ionosphere_radius_re * m.cfg.length_norm_m;
  const double r2 = rm * rm;
  hipStream_t s = n.stream;
  PairBatch pb;
  if (pb.allocate(t.batch, m.nt, m.np) != 0) return -1;
  float *host_loss = nullptr;
  GCS_HIP(hipHostMalloc(&host_loss, sizeof(float)));
  std::mt19937_64 rng(t.seed);
  const int f = coarsening(m, n);
  const dim3 g(blocks_of((long)n.H * n.W), t.batch);
  int rc = 0;
  for (long step = 0; step < t.steps && rc == 0; ++step) {
    // the previous step's copy of the pinned samples must finish before
    // they are redrawn
    if (step > 0 && loss_history == nullptr && hipStreamSynchronize(s) != hipSuccess) {
      set_error("warm-start training: stream error");
      rc = -1;
      break;
    }
    draw_samples(rng, t.batch, m.max_colat, t.pedersen_min, t.pedersen_max, t.hall_min,
                 t.hall_max, pb.host);
    if (make_pairs(pb, m.nt, m.np, m.max_colat, r2, s) != 0) {
      rc = -1;
      break;
    }
    if (n.adam_t == 0 && step == 0) {
      // output scale: unit RMS of the first batch's targets
      k_gen_features<<<g, kT, 0, s>>>(pb.dev, m.nt, m.np, f, r2, pb.fac, pb.phi, pb.scale,
                                      1.0, n.input, n.target);
      std::vector<float> tg((size_t)t.batch * n.H * n.W);
      if (hipMemcpyAsync(tg.data(), n.target, tg.size() * sizeof(float),
                         hipMemcpyDeviceToHost, s) != hipSuccess ||
          hipStreamSynchronize(s) != hipSuccess) {
        set_error("warm-start training: target readback failed");
        rc = -1;
        break;
      }
      double ss = 0.0;
      for (float v : tg) ss += (double)v * v;
      n.out_scale = std::sqrt(ss / (double)tg.size());
      if (!(n.out_scale > 0.0) || !std::isfinite(n.out_scale)) n.out_scale = 1.0;
    }
    k_gen_features<<<g, kT, 0, s>>>(pb.dev, m.nt, m.np, f, r2, pb.fac, pb.phi, pb.scale,
                                    n.out_scale, n.input, n.target);
    // cosine decay to 5% of the rate after a short linear warmup
    const double warm = std::min(1.0, (double)(step + 1) / 50.0);
    const double frac = (double)step / (double)std::max(1L, t.steps - 1);
    const double lr = t.learning_rate * warm * (0.05 + 0.95 * 0.5 * (1.0 + std::cos(kPi * frac)));
    if (unet::forward_device(n, t.batch) != 0 || unet::loss_relative_device(n, t.batch) != 0 ||
        unet::backward_device(n, t.batch) != 0 || unet::adam_device(n, (float)lr) != 0) {
      rc = -1;
      break;
    }
    if (loss_history != nullptr) {
      if (hipMemcpyAsync(host_loss, n.loss, sizeof(float), hipMemcpyDeviceToHost, s) !=
              hipSuccess ||
          hipStreamSynchronize(s) != hipSuccess) {
        set_error("warm-start training: loss readback failed");
        rc = -1;
        break;
      }
      loss_history[step] = *host_loss;
    }
  }
  (void)hipHostFree(host_loss);
  if (rc == 0 && hipStreamSynchronize(s) != hipSuccess) {
    set_error("warm-start training: stream error");
    rc = -1;
  }
  return rc;
}

// Training on given pairs (for instance currents logged from MHD runs and
// the potentials the plain solve gives for them): the same loss, Adam
// steps and learning-rate schedule as mi_train_warm_start, each batch drawn
// uniformly (seeded) from the `count` pairs, which stay on the device. The
// conductances are the problem's (Pedersen of its MI configuration, its
// Hall conductance).
int mi_train_warm_start_on(Problem &P, unet::Net &n, const gcs_warm_train_config &t,
                           const double *fac, const double *phi, const int *hemi, int count,
                           float *loss_history) {
  if (P.mi == nullptr) {
    set_error("MI is not enabled");
    return -1;
  }
  const MiState &m = *P.mi;
  if (coarsening(m, n) <= 0 || unet::check_batch(n, t.batch) != 0 || t.steps <= 0 ||
      !(t.learning_rate > 0.0) || count <= 0 || fac == nullptr || phi == nullptr ||
      hemi == nullptr) {
    set_error("invalid warm-start training configuration or data");
    return -1;
  }
  for (int b = 0; b < count; ++b)
    if (hemi[b] != GAMERA_MI_NORTH && hemi[b] != GAMERA_MI_SOUTH) {
      set_error("hemisphere must be GAMERA_MI_NORTH or GAMERA_MI_SOUTH");
      return -1;
    }
  const double rm = m.cfg.ionosphere_radius_re * m.cfg.length_norm_m;
  const double r2 = rm * rm;
  const size_t per = (size_t)m.nt * m.np;
  hipStream_t s = n.stream;
  PairBatch pb;
  if (pb.allocate(t.batch, m.nt, m.np) != 0) return -1;
  double *data_fac = nullptr, *data_phi = nullptr;
  float *host_loss = nullptr;
  int rc = 0;
  if (hipMalloc(&data_fac, count * per * sizeof(double)) != hipSuccess ||
      hipMalloc(&data_phi, count * per * sizeof(double)) != hipSuccess ||
      hipHostMalloc(&host_loss, sizeof(float)) != hipSuccess ||
      hipMemcpy(data_fac, fac, count * per * sizeof(double), hipMemcpyHostToDevice) !=
          hipSuccess ||
      hipMemcpy(data_phi, phi, count * per * sizeof(double), hipMemcpyHostToDevice) !=
          hipSuccess) {
    set_error("warm-start training: device buffers for the pairs");
    rc = -1;
  }
  std::mt19937_64 rng(t.seed);
  std::uniform_int_distribution<int> pick(0, count - 1);
  const int f = coarsening(m, n);
  const dim3 g(blocks_of((long)n.H * n.W), t.batch);
  for (long step = 0; step < t.steps && rc == 0; ++step) {
    // the pinned samples of the previous step must be copied before reuse
    if (hipStreamSynchronize(s) != hipSuccess) {
      set_error("warm-start training: stream error");
      rc = -1;
      break;
    }
    for (int b = 0; b < t.batch && rc == 0; ++b) {
      const int idx = pick(rng);
      GenSample &gs = pb.host[b];
      gs.hemi = hemi[idx];
      gs.sp = m.cfg.pedersen_siemens;
      gs.sh = m.hall;
      if (hipMemcpyAsync(pb.fac + b * per, data_fac + idx * per, per * sizeof(double),
                         hipMemcpyDeviceToDevice, s) != hipSuccess ||
          hipMemcpyAsync(pb.phi + b * per, data_phi + idx * per, per * sizeof(double),
                         hipMemcpyDeviceToDevice, s) != hipSuccess) {
        set_error("warm-start training: batch gather");
        rc = -1;
      }
    }
    if (rc != 0) break;
    if (hipMemcpyAsync(pb.dev, pb.host, t.batch * sizeof(GenSample), hipMemcpyHostToDevice,
                       s) != hipSuccess) {
      set_error("warm-start training: sample upload");
      rc = -1;
      break;
    }
    k_gen_scale<<<t.batch, kT, 0, s>>>(m.nt, m.np, pb.fac, pb.scale);
    if (n.adam_t == 0 && step == 0) {
      // output scale: unit RMS of the first batch's targets
      k_gen_features<<<g, kT, 0, s>>>(pb.dev, m.nt, m.np, f, r2, pb.fac, pb.phi, pb.scale,
                                      1.0, n.input, n.target);
      std::vector<float> tg((size_t)t.batch * n.H * n.W);
      if (hipMemcpyAsync(tg.data(), n.target, tg.size() * sizeof(float),
                         hipMemcpyDeviceToHost, s) != hipSuccess ||
          hipStreamSynchronize(s) != hipSuccess) {
        set_error("warm-start training: target readback failed");
        rc = -1;
        break;
      }
      double ss = 0.0;
      for (float v : tg) ss += (double)v * v;
      n.out_scale = std::sqrt(ss / (double)tg.size());
      if (!(n.out_scale > 0.0) || !std::isfinite(n.out_scale)) n.out_scale = 1.0;
    }
    k_gen_features<<<g, kT, 0, s>>>(pb.dev, m.nt, m.np, f, r2, pb.fac, pb.phi, pb.scale,
                                    n.out_scale, n.input, n.target);
    const double warm = std::min(1.0, (double)(step + 1) / 50.0);
    const double frac = (double)step / (double)std::max(1L, t.steps - 1);
    const double lr = t.learning_rate * warm * (0.05 + 0.95 * 0.5 * (1.0 + std::cos(kPi * frac)));
    if (unet::forward_device(n, t.batch) != 0 || unet::loss_relative_device(n, t.batch) != 0 ||
        unet::backward_device(n, t.batch) != 0 || unet::adam_device(n, (float)lr) != 0) {
      rc = -1;
      break;
    }
    if (loss_history != nullptr) {
      if (hipMemcpyAsync(host_loss, n.loss, sizeof(float), hipMemcpyDeviceToHost, s) !=
              hipSuccess ||
          hipStreamSynchronize(s) != hipSuccess) {
        set_error("warm-start training: loss readback failed");
        rc = -1;
        break;
      }
      loss_history[step] = *host_loss;
    }
  }
  if (hipStreamSynchronize(s) != hipSuccess && rc == 0) {
    set_error("warm-start training: stream error");
    rc = -1;
  }
  if (host_loss) (void)hipHostFree(host_loss);
  (void)hipFree(data_fac);
  (void)hipFree(data_phi);
  return rc;
}

// One polar solve of both hemispheres from host arrays ([2][nt][np] current
// and guess; the solution replaces the guess), with or without the attached
// network. Leaves the problem's MI state at the solved potential.
int mi_solve_current(Problem &P, const double *fac, double *potential, int use_net,
                     int iterations[2], double *ms) {
  if (P.mi == nullptr) {
    set_error("MI is not enabled");
    return -1;
  }
  MiState &m = *P.mi;
  if (use_net && m.net == nullptr) {
    set_error("no warm-start network attached");
    return -1;
  }
  const size_t bytes = 2UL * m.nt * m.np * sizeof(double);
  GCS_HIP(hipStreamSynchronize(P.stream));
  GCS_HIP(hipMemcpy(m.fac, fac, bytes, hipMemcpyHostToDevice));
  GCS_HIP(hipMemcpy(m.potential, potential, bytes, hipMemcpyHostToDevice));
  unet::Net *keep = m.net;
  if (!use_net) m.net = nullptr;
  const int rc = solve(P, m.hall > 0.0);
  m.net = keep;
  // a later step reads this potential
  if (refresh_mi_drift(P, m.potential, m.drift) != 0) return -1;
  iterations[0] = m.iterations[0];
  iterations[1] = m.iterations[1];
  *ms = m.solve_ms;
  if (rc != 0) return -1;
  GCS_HIP(hipMemcpy(potential, m.potential, bytes, hipMemcpyDeviceToHost));
  return 0;
}

}  // namespace gcs
