// advect.hip -- level-set advection for gfx950 behind the C ABI of
// include/scihpc_hip.h: WENO5-Z derivatives (weno_solver.cpp:16-278),
// convection RHS s = -u.grad(phi) (source.cpp:8-40), TVD-RK3 in the
// reference's cumulative form (runge_kutta.cpp:13-49) and the bc_factory
// ghost fills (bc_factory.cpp:61-375 with neumann.cpp, dirichlet.cpp,
// periodic.cpp, no_slip.cpp, slip.cpp).
//
// Storage: the reference's padded scalar_data layout made contiguous
// (data[i][j][k], k fastest, 3 ghost cells on every axis < ndim).  One
// fused kernel per RK stage computes the WENO-Z face values on the upwind
// side only, the convection RHS, the stage update into a second buffer and
// that buffer's ghosts (the reference's order of axes matters only for
// Dirichlet sides, whose ghosts small kernels per axis fill: x, y, z; right
// side before left side).  Corner ghosts are never written, as in the
// reference.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <utility>
#include <vector>

#include "common.hpp"

namespace scihpc {

constexpr int kGhc = 3;
constexpr int kLsBlock = 256;

struct Grid {
  int ndim;
  int n[3], N[3], off[3];
  long s[3];
  long total;     // padded cells
  long interior;  // interior cells
  double h[3];
};

static Grid make_grid(int ndim, int nx, int ny, int nz, double dx, double dy, double dz) {
  Grid g{};
  g.ndim = ndim;
  const int n[3] = {nx, ny, nz};
  for (int a = 0; a < 3; ++a) {
    if (a < ndim) {
      g.n[a] = n[a];
      g.N[a] = n[a] + 2 * kGhc;
      g.off[a] = kGhc;
    } else {
      g.n[a] = 1;
      g.N[a] = 1;
      g.off[a] = 0;
    }
  }
  g.s[2] = 1;
  g.s[1] = g.N[2];
  g.s[0] = (long)g.N[1] * g.N[2];
  g.total = (long)g.N[0] * g.N[1] * g.N[2];
  g.interior = (long)g.n[0] * g.n[1] * g.n[2];
  g.h[0] = dx;
  g.h[1] = dy;
  g.h[2] = dz;
  return g;
}

// padded index of interior cell number t (last axis fastest)
__device__ __forceinline__ long interior_index(const Grid &g, long t) {
  const int k = (int)(t % g.n[2]);
  const long r = t / g.n[2];
  const int j = (int)(r % g.n[1]);
  const int i = (int)(r / g.n[1]);
  return (long)(i + g.off[0]) * g.s[0] + (long)(j + g.off[1]) * g.s[1] + (k + g.off[2]);
}

// ------------------------------------------------------------- WENO-Z
// Face value at I+1/2 from the five values a..e (left-biased, centred on c:
// interpolation_m/indicators_m) with the WENO-Z weights of
// weno_solver.cpp:50-66 (epsilon = 1e-8, global.h:14).
__device__ __forceinline__ double weno_face(double a, double b, double c, double d, double e,
                                            bool left_biased) {
  double q0, q1, q2, b0, b1, b2;
  if (left_biased) {
    q2 = (-e + 5.0 * d + 2.0 * c) / 6.0;
    q1 = (2.0 * d + 5.0 * c - b) / 6.0;
    q0 = (11.0 * c - 7.0 * b + 2.0 * a) / 6.0;
    b0 = 13.0 * (a - 2.0 * b + c) * (a - 2.0 * b + c) + 3.0 * (a - 4.0 * b + 3.0 * c) * (a - 4.0 * b + 3.0 * c);
    b1 = 13.0 * (b - 2.0 * c + d) * (b - 2.0 * c + d) + 3.0 * (b - d) * (b - d);
    b2 = 13.0 * (c - 2.0 * d + e) * (c - 2.0 * d + e) + 3.0 * (3.0 * c - 4.0 * d + e) * (3.0 * c - 4.0 * d + e);
  } else {
    // right-biased: a..e = f[I-1..I+3], centre c = f[I+1]
    q2 = (-a + 5.0 * b + 2.0 * c) / 6.0;
    q1 = (2.0 * b + 5.0 * c - d) / 6.0;
    q0 = (11.0 * c - 7.0 * d + 2.0 * e) / 6.0;
    b0 = 13.0 * (c - 2.0 * d + e) * (c - 2.0 * d + e) + 3.0 * (3.0 * c - 4.0 * d + e) * (3.0 * c - 4.0 * d + e);
    b1 = 13.0 * (b - 2.0 * c + d) * (b - 2.0 * c + d) + 3.0 * (b - d) * (b - d);
    b2 = 13.0 * (a - 2.0 * b + c) * (a - 2.0 * b + c) + 3.0 * (a - 4.0 * b + 3.0 * c) * (a - 4.0 * b + 3.0 * c);
  }
  const double eps = 1e-8;
  const double tau = fabs(b0 - b2);
  const double a0 = 1.0 * (1.0 + tau / (eps + b0));
  const double a1 = 6.0 * (1.0 + tau / (eps + b1));
  const double a2 = 3.0 * (1.0 + tau / (eps + b2));
  const double w0 = a0 / (a0 + a1 + a2), w1 = a1 / (a0 + a1 + a2), w2 = a2 / (a0 + a1 + a2);
  return w0 * q0 + w1 * q1 + w2 * q2;
}

// upwinded face flux fh at face P+1/2 along a stride: fm if v[P]+v[P+1] > 0
// else fp (weno_solver.cpp:185-199)
__device__ __forceinline__ double face_flux(const double *__restrict__ f, const double *__restrict__ v,
                                            long c, long st) {
  if (v[c] + v[c + st] > 0.0)
    return weno_face(f[c - 2 * st], f[c - st], f[c], f[c + st], f[c + 2 * st], true);
  return weno_face(f[c - st], f[c], f[c + st], f[c + 2 * st], f[c + 3 * st], false);
}

// derivative along axis a at padded cell c: (fh[P] - fh[P-1]) / h
__device__ __forceinline__ double weno_deriv(const double *__restrict__ f, const double *__restrict__ v, long c,
                                             long st, double h) {
  return (face_flux(f, v, c, st) - face_flux(f, v, c - st, st)) / h;
}

// weno5_find_derivatives on interior cells
template <int DIM>
__global__ void __launch_bounds__(kLsBlock) k_weno_derivs(Grid g, const double *__restrict__ f,
                                                          const double *__restrict__ u, const double *__restrict__ v,
                                                          const double *__restrict__ w, double *fx, double *fy,
                                                          double *fz) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= g.interior) return;
  const long c = interior_index(g, t);
  fx[c] = weno_deriv(f, u, c, g.s[0], g.h[0]);
  if constexpr (DIM > 1) fy[c] = weno_deriv(f, v, c, g.s[1], g.h[1]);
  if constexpr (DIM > 2) fz[c] = weno_deriv(f, w, c, g.s[2], g.h[2]);
}

// One TVD-RK3 stage of a 1-D field fused with the convection RHS
// (source.cpp:12-39): s = -u*fx on interior cells, then
//   stage 1: out = in + dt*s                 (s1 <- s)
//   stage 2: out = in + dt*(s - 3 s1)/4      (s2 <- s)
//   stage 3: out = in + dt*(-s1 - s2 + 8 s)/12
// (2-D and 3-D: k_rk3_fused)
template <int STAGE>
__global__ void __launch_bounds__(kLsBlock) k_rk3_stage(Grid g, const double *__restrict__ in, double *__restrict__ out,
                                                        const double *__restrict__ u, double *__restrict__ s1,
                                                        double *__restrict__ s2, double dt) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= g.interior) return;
  const long c = interior_index(g, t);
  const double s = -u[c] * weno_deriv(in, u, c, g.s[0], g.h[0]);
  const double x = in[c];
  if constexpr (STAGE == 1) {
    s1[c] = s;
    out[c] = x + dt * s;
  } else if constexpr (STAGE == 2) {
    s2[c] = s;
    out[c] = x + dt * (s - 3.0 * s1[c]) / 4.0;
  } else {
    out[c] = x + dt * (-s1[c] - s2[c] + 8.0 * s) / 12.0;
  }
}

// ------------------------------------------------------------- BCs
// One boundary line along an axis; p points to padded position 0 of the
// axis, st is the stride.  `face` selects the staggered variant.
__device__ void bc_line(double *p, long st, int n, int N, int type, bool right, bool face, double U, double h) {
  const int g = kGhc;
#define F(q) p[(long)(q) * st]
  if (right) {
    const int I = n - 1 + g;
    switch (type) {
      case SCIHPC_BC_NEUMANN:
        if (face) F(I) = F(I - 1) + U * h;
        for (int i = 1; i <= g; ++i) F(I + i) = F(I + i - 1) + U * h;
        break;
      case SCIHPC_BC_DIRICHLET:
        if (face) F(I) = U;
        else F(I) = F(I - 1) / 3.0 + 2.0 * U / 3.0;
        for (int i = 1; i <= g; ++i) F(I + i) = 2.0 * F(I + i - 1) - F(I + i - 2);
        break;
      case SCIHPC_BC_PERIODIC:
        for (int i = 1; i <= g; ++i) F(I + i) = F(g + (i - 1));
        break;
      case SCIHPC_BC_NO_SLIP:
        if (face) {
          for (int i = 1; i <= g; ++i) F(I + i) = -F(I - i);
          F(I) = 0.0;
        } else {
          for (int i = 1; i <= g; ++i) F(I + i) = -F(I + 1 - i);
        }
        break;
      case SCIHPC_BC_SLIP:
        if (face) {
          for (int i = 1; i <= g; ++i) F(I + i) = F(I - i);
          F(I) = 0.0;
        } else {
          for (int i = 1; i <= g; ++i) F(I + i) = F(I + 1 - i);
        }
        break;
    }
  } else {
    const int I = g;
    switch (type) {
      case SCIHPC_BC_NEUMANN:
        if (face) {
          F(I - 1) = F(I) - U * h;
          for (int i = 1; i <= g - 1; ++i) F(I - 1 - i) = F(I - i) - U * h;
        } else {
          for (int i = 1; i <= g; ++i) F(I - i) = F(I - i + 1) - U * h;
        }
        break;
      case SCIHPC_BC_DIRICHLET:
        if (face) {
          F(I - 1) = U;
          for (int i = 2; i <= g; ++i) F(I - i) = 2.0 * F(I - i + 1) - F(I - i + 2);
        } else {
          F(I) = F(I + 1) / 3.0 + 2.0 * U / 3.0;
          for (int i = 1; i <= g; ++i) F(I - i) = 2.0 * F(I - i + 1) - F(I - i + 2);
        }
        break;
      case SCIHPC_BC_PERIODIC:
        for (int i = 1; i <= g; ++i) F(I - i) = F(N - g - 1 - (i - 1));
        break;
      case SCIHPC_BC_NO_SLIP:
        if (face) {
          for (int i = 1; i <= g; ++i) F(I - i) = -F(I - 2 + i);
          F(I - 1) = 0.0;
        } else {
          for (int i = 1; i <= g; ++i) F(I - i) = -F(I - 1 + i);
        }
        break;
      case SCIHPC_BC_SLIP:
        if (face) {
          for (int i = 1; i <= g; ++i) F(I - i) = F(I - 2 + i);
          F(I - 1) = 0.0;
        } else {
          for (int i = 1; i <= g; ++i) F(I - i) = F(I - 1 + i);
        }
        break;
    }
  }
#undef F
}

struct BcSpec {
  int type[6];
  double value[6];
};

// ghost fill of both sides of axis a, one thread per boundary line
__global__ void __launch_bounds__(kLsBlock) k_bc_axis(Grid g, double *f, BcSpec bc, int a, int stag) {
  const int t1 = (a + 1) % 3, t2 = (a + 2) % 3;
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long lines = (long)g.n[t1] * g.n[t2];
  if (t >= lines) return;
  const int u = (int)(t / g.n[t2]), v = (int)(t % g.n[t2]);
  double *p = f + (long)(u + g.off[t1]) * g.s[t1] + (long)(v + g.off[t2]) * g.s[t2];
  const bool face = stag == a;
  bc_line(p, g.s[a], g.n[a], g.N[a], bc.type[2 * a + 1], true, face, bc.value[2 * a + 1], g.h[a]);
  bc_line(p, g.s[a], g.n[a], g.N[a], bc.type[2 * a], false, face, bc.value[2 * a], g.h[a]);
}

// k_bc_axis for up to three fields in one launch (thread t: field t /
// lines, line t % lines).  A field's BC on one axis touches only that
// field, so the fields of one axis are independent; the axes stay in
// separate launches, in the reference's order.
struct BcFields {
  double *f[3];
  BcSpec bc[3];
  int stag[3];
  int nf;
};
__global__ void __launch_bounds__(kLsBlock) k_bc_axis_fields(Grid g, BcFields m, int a) {
  const int t1 = (a + 1) % 3, t2 = (a + 2) % 3;
  const long lines = (long)g.n[t1] * g.n[t2];
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= lines * m.nf) return;
  const int q = (int)(t / lines);
  const long l = t - (long)q * lines;
  const int u = (int)(l / g.n[t2]), v = (int)(l % g.n[t2]);
  double *p = m.f[q] + (long)(u + g.off[t1]) * g.s[t1] + (long)(v + g.off[t2]) * g.s[t2];
  const bool face = m.stag[q] == a;
  const BcSpec &bc = m.bc[q];
  bc_line(p, g.s[a], g.n[a], g.N[a], bc.type[2 * a + 1], true, face, bc.value[2 * a + 1], g.h[a]);
  bc_line(p, g.s[a], g.n[a], g.N[a], bc.type[2 * a], false, face, bc.value[2 * a], g.h[a]);
}

// ---- fused TVD-RK3 stage, 2-D and 3-D
// k_rk3_stage<1>'s work with every face value formed once and the ghosts
// filled by the cells they copy.  The last axis is contiguous: a wavefront
// takes 64 faces and so 63 cells of a row, each lane handing its face to the
// next, or several short rows (SHORT: `lanes` lanes each).  Threads march `run`
// cells along the first axis and carry the face between them.  In 3-D a
// workgroup's eight wavefronts hold rows of the middle axis, the lowest of
// which only forms faces for the row above it.
// What bounds it: FP64 issue (the VALU is active in 59 % of the cycles in
// which a SIMD has work, at 1024 x 512).  A face took ten IEEE divisions (about 14
// instructions each) and was formed by both its cells; here it takes four
// reciprocals (v_rcp_f64 and two Newton steps).  The WENO-Z weights are
// ratios, so their common denominator is left out; the reciprocal of their sum
// is applied to them before the values are, as next to a flat stencil a weight
// is a squared difference over 1e-8 (from values of 1e100 on its product
// overflows; as many operations as one corrected quotient, and over 14 grids
// its error against 64 bits 1.011e-16, the divisions' 1.016e-16).
// Measured at 1024 x 512: a stage with its boundary conditions 20.3 + 2 x 4.7
// us in three launches before, 11.9 us here (a step 81 -> 36 us).
constexpr int kRkRows = 8;

__device__ __forceinline__ double weno_rcp(double d) {
  double r = __builtin_amdgcn_rcp(d);
  r = __builtin_fma(r, __builtin_fma(-d, r, 1.0), r);
  return __builtin_fma(r, __builtin_fma(-d, r, 1.0), r);
}

// weno_face(a, b, c, d, e, left-biased): the value right of c
__device__ __forceinline__ double weno_face_left(double a, double b, double c, double d, double e) {
  const double p0 = a - 2.0 * b + c, q0 = a - 4.0 * b + 3.0 * c;
  const double p1 = b - 2.0 * c + d, q1 = b - d;
  const double p2 = c - 2.0 * d + e, q2 = 3.0 * c - 4.0 * d + e;
  const double b0 = 13.0 * p0 * p0 + 3.0 * q0 * q0;
  const double b1 = 13.0 * p1 * p1 + 3.0 * q1 * q1;
  const double b2 = 13.0 * p2 * p2 + 3.0 * q2 * q2;
  const double eps = 1e-8;
  const double tau = fabs(b0 - b2);
  const double a0 = 1.0 + tau * weno_rcp(eps + b0);
  const double a1 = 6.0 + 6.0 * tau * weno_rcp(eps + b1);
  const double a2 = 3.0 + 3.0 * tau * weno_rcp(eps + b2);
  const double v0 = 2.0 * a - 7.0 * b + 11.0 * c, v1 = 5.0 * c - b + 2.0 * d, v2 = 2.0 * c + 5.0 * d - e;
  const double den = 6.0 * (a0 + a1 + a2);
  const double r = weno_rcp(den);
  return (a0 * r) * v0 + (a1 * r) * v1 + (a2 * r) * v2;
}

// upwinded value right of f[2] from f[0..5]; vel: the two cells' velocities
__device__ __forceinline__ double weno_upwind(const double (&f)[6], double vl, double vr) {
  const bool left = vl + vr > 0.0;
  return weno_face_left(left ? f[0] : f[5], left ? f[1] : f[4], left ? f[2] : f[3], left ? f[3] : f[2],
                        left ? f[4] : f[1]);
}

// The ghosts of axis a that a cell-centred BC (but Dirichlet, which changes
// the boundary cell itself) takes from interior cell i with value x; f: that
// cell.  bc_line's values, bit for bit.
__device__ __forceinline__ void ghosts_of(const BcSpec &bc, int a, int n, double h, long st, int i, double x,
                                          double *f) {
#pragma clang fp contract(off)
  if (i >= kGhc && i < n - kGhc) return;
  const int l = bc.type[2 * a], r = bc.type[2 * a + 1];
  if (r == SCIHPC_BC_NEUMANN) {
    if (i == n - 1) {
      double y = x;
      for (int q = 1; q <= kGhc; ++q) f[q * st] = y = y + bc.value[2 * a + 1] * h;
    }
  } else if (r == SCIHPC_BC_PERIODIC) {
    if (i < kGhc) f[(long)n * st] = x;
  } else if (n - 1 - i < kGhc) {  // no slip, slip
    f[(long)(2 * (n - 1 - i) + 1) * st] = r == SCIHPC_BC_NO_SLIP ? -x : x;
  }
  if (l == SCIHPC_BC_NEUMANN) {
    if (i == 0) {
      double y = x;
      for (int q = 1; q <= kGhc; ++q) f[-q * st] = y = y - bc.value[2 * a] * h;
    }
  } else if (l == SCIHPC_BC_PERIODIC) {
    if (i >= n - kGhc) f[-(long)n * st] = x;
  } else if (i < kGhc) {
    f[-(long)(2 * i + 1) * st] = l == SCIHPC_BC_NO_SLIP ? -x : x;
  }
}

template <int DIM, int STAGE, bool SHORT>
__global__ void __launch_bounds__(DIM == 3 ? kWave *kRkRows : kLsBlock)
    k_rk3_fused(Grid g, const double *__restrict__ in, double *__restrict__ out, const double *__restrict__ u,
                const double *__restrict__ v, const double *__restrict__ w, double *__restrict__ s1,
                double *__restrict__ s2, double dt, BcSpec bc, int ghosts, int tiles_c, int tiles_r,
                int run, int lanes) {
  constexpr int C = DIM - 1;  // the contiguous axis
  __shared__ double yf[DIM == 3 ? 2 : 1][DIM == 3 ? kRkRows * kWave : 1];
  const int width = SHORT ? lanes : kWave;
  const int sub = kWave / width, part = (int)threadIdx.x % kWave / width;  // rows a wavefront, this lane's
  const int lane = (int)threadIdx.x % kWave - part * width, row = (int)threadIdx.x / kWave * sub + part;
  const bool spare = part >= sub;  // a lane too many
  // 2-D: every row of a wavefront has a tile of its own
  int tile = DIM == 3 ? (int)blockIdx.x : (int)blockIdx.x * (kLsBlock / kWave) * sub + row;
  const int tc = tile % tiles_c;
  tile /= tiles_c;
  const int tr = DIM == 3 ? tile % tiles_r : 0;
  if (DIM == 3) tile /= tiles_r;
  const int i0 = tile * run, i1 = min(g.n[0], i0 + run);
  if (DIM == 2 && (spare || i0 >= g.n[0])) return;  // whole rows, no barrier in 2-D
  const int nc = g.n[C], nr = DIM == 3 ? g.n[1] : 1;
  const int c = tc * (width - 1) + lane - 1, r = DIM == 3 ? tr * (kRkRows * sub - 1) + row - 1 : 0;
  const bool own = !spare && lane > 0 && c < nc && (DIM == 2 || (row > 0 && r < nr));  // lane 0 and row 0 form faces only
  const int cc = min(c, nc - 1), rc = min(r, nr - 1);
  const long sx = g.s[0], sr = g.s[1];
  const double *vc = DIM == 3 ? w : v;
  long p = (long)(i0 + g.off[0]) * sx + (DIM == 3 ? (long)(rc + g.off[1]) * sr : 0) + cc + g.off[C];
  double f[6], uc = u[p];  // f[2]: the cell at hand, along the march
#pragma unroll
  for (int q = 0; q < 6; ++q) f[q] = in[p + (q - 3) * sx];
  double lower = weno_upwind(f, u[p - sx], uc);
#pragma unroll
  for (int q = 0; q < 5; ++q) f[q] = f[q + 1];
  for (int i = i0; i < i1; ++i, p += sx) {
    f[5] = in[p + 3 * sx];
    double a[6];
#pragma unroll
    for (int q = 0; q < 6; ++q) a[q] = q == 2 ? f[2] : in[p + q - 2];
    const double vl = vc[p], ur = u[p + sx];
    const double fc = weno_upwind(a, vl, vc[p + 1]);
    const double upper = weno_upwind(f, uc, ur);
    double fr = 0.0, vr = 0.0;
    if constexpr (DIM == 3) {
#pragma unroll
      for (int q = 0; q < 6; ++q) a[q] = q == 2 ? f[2] : in[p + (q - 2) * sr];
      vr = v[p];
      fr = weno_upwind(a, vr, v[p + sr]);
      if (!spare) yf[i & 1][row * width + lane] = fr;
      __syncthreads();
    }
    const double fl = __shfl_up(fc, 1, kWave);
    if (own) {
      double s = -uc * ((upper - lower) / g.h[0]);
      if constexpr (DIM == 3) s -= vr * ((fr - yf[i & 1][(row - 1) * width + lane]) / g.h[1]);
      s -= vl * ((fc - fl) / g.h[C]);
      const double x = f[2];
      double y;
      if constexpr (STAGE == 1) {
        s1[p] = s;
        y = x + dt * s;
      } else if constexpr (STAGE == 2) {
        s2[p] = s;
        y = x + dt * (s - 3.0 * s1[p]) / 4.0;
      } else {
        y = x + dt * (-s1[p] - s2[p] + 8.0 * s) / 12.0;
      }
      out[p] = y;
      if (ghosts) {
        ghosts_of(bc, 0, g.n[0], g.h[0], sx, i, y, out + p);
        if constexpr (DIM == 3) ghosts_of(bc, 1, nr, g.h[1], sr, r, y, out + p);
        ghosts_of(bc, C, nc, g.h[C], 1, c, y, out + p);
      }
    }
    lower = upper;
    uc = ur;
#pragma unroll
    for (int q = 0; q < 5; ++q) f[q] = f[q + 1];
  }
}

// find_density: rho = H + (1-H) ratio (or mirrored), lsm.cpp:8-18
__global__ void __launch_bounds__(kLsBlock) k_density(const double *__restrict__ phi, long n, double w, double ratio,
                                                      int positive_ref, double *__restrict__ rho) {
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n) return;
  const double x = phi[c];
  const double pi = 3.14159265358979323846;
  double h;
  if (x < -w) h = 0.0;
  else if (x > w) h = 1.0;
  else h = 0.5 * (1 + x / w + sin(pi * x / w) / pi);
  rho[c] = positive_ref ? h + (1.0 - h) * ratio : (1.0 - h) + h * ratio;
}

// ------------------------------------------------- projection step
// The projection kernels round like the reference (no fused multiply-add
// contraction), so their results are bit-identical for the same inputs.
// padded index of interior cell (I, J, K)
__device__ __forceinline__ long pidx(const Grid &g, int I, int J, int K) {
  return (long)(I + g.off[0]) * g.s[0] + (long)(J + g.off[1]) * g.s[1] + (K + g.off[2]);
}
__device__ __forceinline__ void interior_ijk(const Grid &g, long t, int &I, int &J, int &K) {
  // MG order: x fastest
  I = (int)(t % g.n[0]);
  J = (int)((t / g.n[0]) % g.n[1]);
  K = (int)(t / ((long)g.n[0] * g.n[1]));
}

// pressure_guess_solution (projection_method.cpp:803-815), every padded cell
__global__ void __launch_bounds__(kLsBlock) k_pressure_guess(const double *__restrict__ old,
                                                             const double *__restrict__ old2, double *__restrict__ phat,
                                                             long n, double dt_old, double dt_old2) {
#pragma clang fp contract(off)  // the reference rounds every product (no FMA)
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n) return;
  const double dpdt = (old[c] - old2[c]) / dt_old2;
  phat[c] = old[c] + dt_old * dpdt;
}

// MG right-hand side of the FPC step (projection_method.cpp:667-692) with
// RHS = sum C p_hat of init_ppe_fpc_coefficients (:467-541) formed in place;
// one thread per interior cell, written in the multigrid layout
template <int DIM>
__global__ void __launch_bounds__(kLsBlock) k_fpc_rhs(Grid g, const double *__restrict__ rho,
                                                      const double *__restrict__ f, const double *__restrict__ u,
                                                      const double *__restrict__ v, const double *__restrict__ w,
                                                      double dt, double rho12, double *__restrict__ mg_rhs) {
#pragma clang fp contract(off)  // the reference rounds every product (no FMA)
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= g.interior) return;
  int I, J, K;
  interior_ijk(g, t, I, J, K);
  const long c = pidx(g, I, J, K), sx = g.s[0], sy = g.s[1], sz = g.s[2];
  const double dx = g.h[0], dy = g.h[1], dz = g.h[2];
  const double R = 0.5 * (rho[c] + rho[c + sx]), L = 0.5 * (rho[c] + rho[c - sx]);
  const double U = 0.5 * (rho[c] + rho[c + sy]), D = 0.5 * (rho[c] + rho[c - sy]);
  double CR = (1.0 - rho12 / R) / dx / dx, CL = (1.0 - rho12 / L) / dx / dx;
  double CU = (1.0 - rho12 / U) / dy / dy, CD = (1.0 - rho12 / D) / dy / dy;
  if (I == 0) CL = 0.0;
  if (I == g.n[0] - 1) CR = 0.0;
  if (J == 0) CD = 0.0;
  if (J == g.n[1] - 1) CU = 0.0;
  double CF = 0.0, CB = 0.0;
  if constexpr (DIM > 2) {
    const double Fz = 0.5 * (rho[c] + rho[c + sz]), B = 0.5 * (rho[c] + rho[c - sz]);
    CF = (1.0 - rho12 / Fz) / dz / dz;
    CB = (1.0 - rho12 / B) / dz / dz;
    if (K == 0) CB = 0.0;
    if (K == g.n[2] - 1) CF = 0.0;
  }
  double CC = -(CR + CL + CU + CD);
  if constexpr (DIM > 2) CC -= (CF + CB);
  double RHS = CC * f[c] + CR * f[c + sx] + CL * f[c - sx] + CU * f[c + sy] + CD * f[c - sy];
  if constexpr (DIM > 2) RHS += CF * f[c + sz] + CB * f[c - sz];
  double r = (u[c] - u[c - sx]) / dx + (v[c] - v[c - sy]) / dy;
  if constexpr (DIM > 2) r += (w[c] - w[c - sz]) / dz;
  r *= rho12 / dt;
  r += RHS;
  mg_rhs[t] = r;
}

// MG right-hand side of the variable-density projection: div(u*) / dt
// (projection_method.cpp:546-568) in the multigrid layout; part[block] = sum
template <int DIM>
__global__ void __launch_bounds__(kLsBlock) k_div_rhs(Grid g, const double *__restrict__ u,
                                                      const double *__restrict__ v, const double *__restrict__ w,
                                                      double dt, double *__restrict__ mg_rhs,
                                                      double *__restrict__ part) {
#pragma clang fp contract(off)  // the reference rounds every product (no FMA)
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  double r = 0.0;
  if (t < g.interior) {
    int I, J, K;
    interior_ijk(g, t, I, J, K);
    const long c = pidx(g, I, J, K);
    r = (u[c] - u[c - g.s[0]]) / g.h[0] + (v[c] - v[c - g.s[1]]) / g.h[1];
    if constexpr (DIM > 2) r += (w[c] - w[c - g.s[2]]) / g.h[2];
    r /= dt;
    mg_rhs[t] = r;
  }
  r = block_sum(r);
  if (threadIdx.x == 0) part[blockIdx.x] = r;
}

__global__ void __launch_bounds__(kLsBlock) k_sub_const(double *__restrict__ x, long n, double m) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) x[t] -= m;
}

// p (padded interior) <- multigrid solution (projection_method.cpp:708-720)
__global__ void __launch_bounds__(kLsBlock) k_mg_to_padded(Grid g, const double *__restrict__ sol,
                                                           double *__restrict__ p) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= g.interior) return;
  int I, J, K;
  interior_ijk(g, t, I, J, K);
  p[pidx(g, I, J, K)] = sol[t];
}

// velocity corrections over the padded range i < Nx-1, j < Ny-1, k < Nz:
// FPC (projection_method.cpp:723-750) when phat != null, else the
// variable-density projection (projection_method.cpp:630-654)
template <int DIM>
__global__ void __launch_bounds__(kLsBlock) k_correct_velocity(Grid g, const double *__restrict__ rho,
                                                               const double *__restrict__ p,
                                                               const double *__restrict__ ph, double dt,
                                                               double rho12, double *__restrict__ u,
                                                               double *__restrict__ v, double *__restrict__ w) {
#pragma clang fp contract(off)  // the reference rounds every product (no FMA)
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int Ni = g.N[0] - 1, Nj = g.N[1] - 1, Nk = g.N[2];
  if (t >= (long)Ni * Nj * Nk) return;
  const int k = (int)(t % Nk), j = (int)((t / Nk) % Nj), i = (int)(t / ((long)Nk * Nj));
  const long c = (long)i * g.s[0] + (long)j * g.s[1] + k;
  const long sx = g.s[0], sy = g.s[1], sz = g.s[2];
  const double dx = g.h[0], dy = g.h[1], dz = g.h[2];
  if (ph) {
    const double px = (p[c + sx] - p[c]) / dx, px2 = (ph[c + sx] - ph[c]) / dx;
    double density = 0.5 * (rho[c] + rho[c + sx]);
    u[c] -= dt * ((px - px2) / rho12 + px2 / density);
    const double py = (p[c + sy] - p[c]) / dy, py2 = (ph[c + sy] - ph[c]) / dy;
    density = 0.5 * (rho[c] + rho[c + sy]);
    v[c] -= dt * ((py - py2) / rho12 + py2 / density);
    if (DIM > 2 && k < Nk - 1) {
      const double pz = (p[c + sz] - p[c]) / dz, pz2 = (ph[c + sz] - ph[c]) / dz;
      density = 0.5 * (rho[c] + rho[c + sz]);
      w[c] -= dt * ((pz - pz2) / rho12 + pz2 / density);
    }
  } else {
    double density = 0.5 * (rho[c] + rho[c + sx]);
    u[c] -= dt / dx / density * (p[c + sx] - p[c]);
    density = 0.5 * (rho[c] + rho[c + sy]);
    v[c] -= dt / dy / density * (p[c + sy] - p[c]);
    if (DIM > 2 && k < Nk - 1) {
      density = 0.5 * (rho[c] + rho[c + sz]);
      w[c] -= dt / dz / density * (p[c + sz] - p[c]);
    }
  }
}

// ------------------------------------------------- momentum predictor
// find_source_sec (projection_method.cpp:314-382) and
// find_intermediate_velocity (:384-402) on padded fields, fused per
// direction.  Ghost extrapolations (identity_with_extrapolation[_face_a],
// flux.cpp:98-375) are index clamps: copying the boundary value outward
// axis by axis over every index of the other axes leaves flux(i,j,k) =
// data(clamp(i), clamp(j), clamp(k)), the face variant clamping its face
// axis to [off-1, off+n-1] (the wall face is kept).  Derivative arrays the
// reference writes only on the interior of their axis are zero elsewhere
// (zero-initialised and never written there), so those terms are 0.  Every
// product is rounded (no FMA), as in the reference.

struct FlowParams {
  double dt, re, fr, we, w, ratio_rho, ratio_mu;
  int positive_ref;
};

__device__ __forceinline__ void padded_ijk(const Grid &g, long c, int q[3]) {
  if (g.total <= 0xffffffffL) {  // 64-bit divisions cost several times as much
    const unsigned u = (unsigned)c, w = u / (unsigned)g.s[1];
    q[0] = (int)(u / (unsigned)g.s[0]);
    q[1] = (int)(w % (unsigned)g.N[1]);
    q[2] = (int)(u % (unsigned)g.N[2]);
    return;
  }
  q[0] = (int)(c / g.s[0]);
  q[1] = (int)((c / g.s[1]) % g.N[1]);
  q[2] = (int)(c % g.N[2]);
}

__device__ __forceinline__ int clampi(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }

// flux index of padded position r: clamp every real axis to its interior;
// `fa` (or -1) is the face axis whose low clamp is the wall face off-1
template <int DIM>
__device__ __forceinline__ long ext_index(const Grid &g, const int r[3], int fa) {
  long c = 0;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    int v = r[a];
    if (a < DIM) v = clampi(v, g.off[a] - (a == fa ? 1 : 0), g.off[a] + g.n[a] - 1);
    c += (long)v * g.s[a];
  }
  return c;
}

// level-set derivatives on the whole padded range (second_order_solver.cpp:
// 13-88 and mixed_xy/yz/zx :173-230), one-sided at the array ends
template <int DIM>
__device__ __forceinline__ double ls_at(const Grid &g, const double *__restrict__ phi, const int q[3], int a, int d) {
  int r[3] = {q[0], q[1], q[2]};
  r[a] += d;
  return phi[ext_index<DIM>(g, r, -1)];
}

template <int DIM>
__device__ double ls_d1(const Grid &g, const double *__restrict__ phi, const int q[3], int a) {
#pragma clang fp contract(off)
  const double h = g.h[a];
  if (q[a] == 0) return (-1.5 * ls_at<DIM>(g, phi, q, a, 0) + 2 * ls_at<DIM>(g, phi, q, a, 1) -
                         0.5 * ls_at<DIM>(g, phi, q, a, 2)) / h;
  if (q[a] == g.N[a] - 1) return (1.5 * ls_at<DIM>(g, phi, q, a, 0) - 2 * ls_at<DIM>(g, phi, q, a, -1) +
                                  0.5 * ls_at<DIM>(g, phi, q, a, -2)) / h;
  return (ls_at<DIM>(g, phi, q, a, 1) - ls_at<DIM>(g, phi, q, a, -1)) / (2 * h);
}

template <int DIM>
__device__ double ls_d2(const Grid &g, const double *__restrict__ phi, const int q[3], int a) {
#pragma clang fp contract(off)
  const double h = g.h[a];
  if (q[a] == 0) return (2 * ls_at<DIM>(g, phi, q, a, 0) - 5 * ls_at<DIM>(g, phi, q, a, 1) +
                         4 * ls_at<DIM>(g, phi, q, a, 2) - ls_at<DIM>(g, phi, q, a, 3)) / (h * h);
  if (q[a] == g.N[a] - 1) return (2 * ls_at<DIM>(g, phi, q, a, 0) - 5 * ls_at<DIM>(g, phi, q, a, -1) +
                                  4 * ls_at<DIM>(g, phi, q, a, -2) - ls_at<DIM>(g, phi, q, a, -3)) / (h * h);
  return (ls_at<DIM>(g, phi, q, a, 1) - 2 * ls_at<DIM>(g, phi, q, a, 0) + ls_at<DIM>(g, phi, q, a, -1)) / (h * h);
}

// d/d(axis b) of the first derivative along a
template <int DIM>
__device__ double ls_mixed(const Grid &g, const double *__restrict__ phi, const int q[3], int a, int b) {
#pragma clang fp contract(off)
  const double h = g.h[b];
  auto G = [&](int d) {
    int r[3] = {q[0], q[1], q[2]};
    r[b] += d;
    return ls_d1<DIM>(g, phi, r, a);
  };
  if (q[b] == 0) return (-1.5 * G(0) + 2 * G(1) - 0.5 * G(2)) / h;
  if (q[b] == g.N[b] - 1) return (1.5 * G(0) - 2 * G(-1) + 0.5 * G(-2)) / h;
  return (G(1) - G(-1)) / (2 * h);
}

// find_delta, find_density, find_viscosity (wrapper_func.cpp:20-29,
// 387-416, lsm.cpp:8-30), the level-set gradient and, with surface tension,
// find_curvature (wrapper_func.cpp:115-172), on every padded cell
template <int DIM, bool ST>
__global__ void __launch_bounds__(kLsBlock)
    k_mom_props(Grid g, FlowParams fp, const double *__restrict__ phi, double *__restrict__ dl,
                double *__restrict__ rho, double *__restrict__ mu, double *__restrict__ lf0,
                double *__restrict__ lf1, double *__restrict__ lf2, double *__restrict__ curv) {
#pragma clang fp contract(off)
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= g.total) return;
  const double pi = 3.14159265358979323846;
  const double x = phi[c], w = fp.w;
  double d, H;
  if (x < -w) d = 0;
  else if (x > w) d = 0;
  else d = 0.5 * (1 + cos(pi * x / w)) / w;
  if (x < -w) H = 0;
  else if (x > w) H = 1;
  else H = 0.5 * (1 + x / w + sin(pi * x / w) / pi);
  dl[c] = d;
  rho[c] = fp.positive_ref ? H + (1.0 - H) * fp.ratio_rho : (1.0 - H) + H * fp.ratio_rho;
  mu[c] = fp.positive_ref ? H + (1.0 - H) * fp.ratio_mu : (1.0 - H) + H * fp.ratio_mu;
  int q[3];
  padded_ijk(g, c, q);
  const double fx = ls_d1<DIM>(g, phi, q, 0), fy = ls_d1<DIM>(g, phi, q, 1);
  lf0[c] = fx;
  lf1[c] = fy;
  double fz = 0.0;
  if constexpr (DIM == 3) {
    fz = ls_d1<DIM>(g, phi, q, 2);
    lf2[c] = fz;
  }
  if constexpr (ST) {
    const double fxx = ls_d2<DIM>(g, phi, q, 0), fyy = ls_d2<DIM>(g, phi, q, 1);
    const double fxy = ls_mixed<DIM>(g, phi, q, 0, 1);
    double k;
    if constexpr (DIM == 2) {
      k = (fxx * fy * fy + fyy * fx * fx - 2.0 * fxy * fx * fy) / pow(fx * fx + fy * fy, 1.5);
      if (k > 0.0) k = 1.0 / (1.0 / k + x);
      else k = -1.0 / (-1.0 / k + x);
    } else {
      const double fzz = ls_d2<DIM>(g, phi, q, 2);
      const double fyz = ls_mixed<DIM>(g, phi, q, 1, 2), fxz = ls_mixed<DIM>(g, phi, q, 2, 0);
      k = (fx * fx * (fyy + fzz) + fy * fy * (fxx + fzz) + fz * fz * (fxx + fyy) -
           2.0 * (fx * fy * fxy + fx * fz * fxz + fy * fz * fyz)) /
          pow(fx * fx + fy * fy + fz * fz, 1.5);
      if (k > 0.0) k = 1.0 / (2.0 / k + x);
      else k = -1.0 / (-2.0 / k + x);
    }
    curv[c] = k;
  }
}

// all_to_face_a (wrapper_func.cpp:177-262) over the padded range 1..N-2
// (every k in 2-D)
template <int DIM>
__global__ void __launch_bounds__(kLsBlock)
    k_to_face(Grid g, int A, const double *__restrict__ v0, const double *__restrict__ v1,
              const double *__restrict__ v2, double *__restrict__ n0, double *__restrict__ n1,
              double *__restrict__ n2) {
#pragma clang fp contract(off)
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= g.total) return;
  int q[3];
  padded_ijk(g, c, q);
  if (q[0] < 1 || q[0] > g.N[0] - 2 || q[1] < 1 || q[1] > g.N[1] - 2) return;
  if (DIM == 3 && (q[2] < 1 || q[2] > g.N[2] - 2)) return;
  const double *vel[3] = {v0, v1, v2};
  double *nv[3] = {n0, n1, n2};
  const long sa = g.s[A];
  nv[A][c] = vel[A][c];
#pragma unroll
  for (int b = 0; b < DIM; ++b) {
    if (b == A) continue;
    const long sb = g.s[b];
    const double *f = vel[b];
    nv[b][c] = 0.25 * (f[c] + f[c + sa] + f[c - sb] + f[c + sa - sb]);
  }
}

// upwind first and central second derivative along axis a of the
// face-extrapolated field f (second_order_solver.cpp:90-148)
template <int DIM>
__device__ __forceinline__ void upwind(const Grid &g, const double *__restrict__ f, int fa, const int q[3], int a,
                                       double vel, double &d1, double &d2) {
#pragma clang fp contract(off)
  auto F = [&](int d) {
    int r[3] = {q[0], q[1], q[2]};
    r[a] += d;
    return f[ext_index<DIM>(g, r, fa)];
  };
  const double h = g.h[a];
  const double f0 = F(0);
  if (vel > 0.0) d1 = (1.5 * f0 - 2 * F(-1) + 0.5 * F(-2)) / h;
  else d1 = (-1.5 * f0 + 2 * F(1) - 0.5 * F(2)) / h;
  d2 = (F(1) - 2 * f0 + F(-1)) / (h * h);
}

// the new source of velocity component A on every padded cell:
// convection_sec (source.cpp:42-73), add_stress_A (projection_method.cpp:
// 31-181, interior), add_body_force (:183-203), add_surface_force (:205-240)
template <int DIM, int A>
__global__ void __launch_bounds__(kLsBlock)
    k_mom_src(Grid g, FlowParams fp, const double *__restrict__ va, const double *__restrict__ n0,
              const double *__restrict__ n1, const double *__restrict__ n2, const double *__restrict__ dl,
              const double *__restrict__ rho, const double *__restrict__ mu, const double *__restrict__ lf0,
              const double *__restrict__ lf1, const double *__restrict__ lf2, const double *__restrict__ curv,
              double *__restrict__ src) {
#pragma clang fp contract(off)
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= g.total) return;
  int q[3];
  padded_ijk(g, c, q);
  const double *nv[3] = {n0, n1, n2};
  bool in[3], all = true;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    in[a] = a >= DIM || (q[a] >= g.off[a] && q[a] < g.off[a] + g.n[a]);
    all = all && in[a];
  }
  double d1[3] = {0, 0, 0}, d2[3] = {0, 0, 0};
#pragma unroll
  for (int a = 0; a < DIM; ++a)
    if (in[a]) upwind<DIM>(g, va, A, q, a, nv[a][c], d1[a], d2[a]);
  double s = -nv[0][c] * d1[0];
  s -= nv[1][c] * d1[1];
  if constexpr (DIM > 2) s -= nv[2][c] * d1[2];
  const long sa = g.s[A];
  if (all) {
    // derivatives along A of the other transferred components, upwinded by
    // the transferred A component
    double cr[3] = {0, 0, 0}, unused;
#pragma unroll
    for (int b = 0; b < DIM; ++b)
      if (b != A) upwind<DIM>(g, nv[b], A, q, A, nv[A][c], cr[b], unused);
    const double delta = 0.5 * (dl[c] + dl[c + sa]);
    const double m = 0.5 * (mu[c] + mu[c + sa]);
    const double r = 0.5 * (rho[c] + rho[c + sa]);
    const double ph0 = 0.5 * (lf0[c] + lf0[c + sa]), ph1 = 0.5 * (lf1[c] + lf1[c + sa]);
    const double ph2 = DIM > 2 ? 0.5 * (lf2[c] + lf2[c + sa]) : 0.0;
    double p1, p2;
    if constexpr (A == 0) {
      p1 = d2[0] + d2[1];
      p2 = 2.0 * ph0 * d1[0] + ph1 * (d1[1] + cr[1]);
      if constexpr (DIM > 2) {
        p1 += d2[2];
        p2 += ph2 * (d1[2] + cr[2]);
      }
    } else if constexpr (A == 1) {
      p1 = d2[0] + d2[1];
      p2 = 2.0 * ph1 * d1[1] + ph0 * (d1[0] + cr[0]);
      if constexpr (DIM > 2) {
        p1 += d2[2];
        p2 += ph2 * (d1[2] + cr[2]);
      }
    } else {  // add_stress_z carries no w_zz term (projection_method.cpp:171)
      p1 = d2[0] + d2[1];
      p2 = 2.0 * ph2 * d1[2] + ph0 * (d1[0] + cr[0]) + ph1 * (d1[1] + cr[1]);
    }
    const double ref = fp.positive_ref ? 1.0 : -1.0;
    p1 *= m;
    p2 *= ref * delta * (1.0 - fp.ratio_mu);
    s += (p1 + p2) / fp.re / r;
  }
  if (fp.fr > 0.0 && A == (DIM == 2 ? 1 : 2)) s += -1.0 / fp.fr;
  if (fp.we > 0.0 && q[0] < g.N[0] - 1 && q[1] < g.N[1] - 1 && (A != 2 || q[2] < g.N[2] - 1)) {
    const double cv = 0.5 * (curv[c] + curv[c + sa]);
    const double delta = 0.5 * (dl[c] + dl[c + sa]);
    const double *lf = A == 0 ? lf0 : (A == 1 ? lf1 : lf2);
    const double pa = 0.5 * (lf[c] + lf[c + sa]);
    const double r = 0.5 * (rho[c] + rho[c + sa]);
    s -= cv * delta * pa / (fp.we * r);
  }
  src[c] = s;
}

// find_intermediate_velocity: AB2 on every padded cell of u, v, w
__global__ void __launch_bounds__(kLsBlock)
    k_ab2(long n, double dt, double *__restrict__ u, double *__restrict__ v, double *__restrict__ w,
          const double *__restrict__ su, const double *__restrict__ sv, const double *__restrict__ sw,
          const double *__restrict__ ou, const double *__restrict__ ov, const double *__restrict__ ow) {
#pragma clang fp contract(off)
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n) return;
  u[c] += dt * (1.5 * su[c] - 0.5 * ou[c]);
  v[c] += dt * (1.5 * sv[c] - 0.5 * ov[c]);
  w[c] += dt * (1.5 * sw[c] - 0.5 * ow[c]);
}

// node_from_face (wrapper_func.cpp:264-293): i, j in 1..N-2; k every
// index in 2-D, 1..Nz-1 in 3-D
template <int DIM>
__global__ void __launch_bounds__(kLsBlock)
    k_node_from_face(Grid g, const double *__restrict__ u, const double *__restrict__ v,
                     const double *__restrict__ w, double *__restrict__ nu, double *__restrict__ nv,
                     double *__restrict__ nw) {
#pragma clang fp contract(off)
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= g.total) return;
  int q[3];
  padded_ijk(g, c, q);
  if (q[0] < 1 || q[0] > g.N[0] - 2 || q[1] < 1 || q[1] > g.N[1] - 2) return;
  if (DIM == 3 && q[2] < 1) return;
  nu[c] = 0.5 * (u[c] + u[c - g.s[0]]);
  nv[c] = 0.5 * (v[c] + v[c - g.s[1]]);
  if constexpr (DIM == 3) nw[c] = 0.5 * (w[c] + w[c - g.s[2]]);
}

// ------------------------------------------------- interface maintenance
// Compact line derivatives (ccd_solver.cpp:14-142, uccd_solver.cpp:14-206):
// along every padded line of axis a the right-hand sides of the scheme are
// formed and the 2x2-block tridiagonal system is solved by the reference's
// twin back substitution (matrix_solver.cpp:58-83) with the factorised
// coefficients of the axis (twin_dec, :21-56, done once on the host).  One
// thread per line; the forward sweep keeps the previous unknowns in
// registers and parks the line in scratch arrays for the backward sweep.
// Lines are enumerated with the contiguous k axis fastest where the line
// does not run along k.  Coefficient set: 12 arrays of n (a0 a1 a2 b0 b1 b2
// aa0 aa1 aa2 bb0 bb1 bb2).

__device__ __forceinline__ bool line_base(const Grid &g, int a, long t, long &base) {
  long lines;
  if (a == 0) {
    lines = (long)g.N[1] * g.N[2];
    if (t >= lines) return false;
    base = (t / g.N[2]) * g.s[1] + (t % g.N[2]);
  } else if (a == 1) {
    lines = (long)g.N[0] * g.N[2];
    if (t >= lines) return false;
    base = (t / g.N[2]) * g.s[0] + (t % g.N[2]);
  } else {
    lines = (long)g.N[0] * g.N[1];
    if (t >= lines) return false;
    base = (t / g.N[1]) * g.s[0] + (t % g.N[1]) * g.s[1];
  }
  return true;
}

// right-hand side at position i of one line; KIND 0 CCD, 1 UCCD upwind,
// 2 UCCD downwind (whose ends are the upwind ones)
template <int KIND>
__device__ __forceinline__ void compact_rhs(const double *__restrict__ f, long st, int n, double h, int i,
                                            double &s, double &ss) {
#pragma clang fp contract(off)
  const double bda1 = -3.5, bdb1 = 4.0, bdc1 = -0.5, bda2 = 9.0, bdb2 = -12.0, bdc2 = 3.0;
  const double c3 = -0.06096119008109, c2 = 1.99692238016218, c1 = -1.93596119008109;
#define F(q) f[(long)(q) * st]
  if (i == 0) {
    s = (bda1 * F(0) + bdb1 * F(1) + bdc1 * F(2)) / h;
    ss = (bda2 * F(0) + bdb2 * F(1) + bdc2 * F(2)) / h / h;
  } else if (i == n - 1) {
    s = -(bda1 * F(n - 1) + bdb1 * F(n - 2) + bdc1 * F(n - 3)) / h;
    ss = (bda2 * F(n - 1) + bdb2 * F(n - 2) + bdc2 * F(n - 3)) / h / h;
  } else {
    if (KIND == 0) s = 15.0 / 16.0 * (F(i + 1) - F(i - 1)) / h;
    else if (KIND == 1) s = (c1 * F(i - 1) + c2 * F(i) + c3 * F(i + 1)) / h;
    else s = -(c3 * F(i - 1) + c2 * F(i) + c1 * F(i + 1)) / h;
    ss = (3.0 * F(i - 1) - 6.0 * F(i) + 3.0 * F(i + 1)) / h / h;
  }
#undef F
}

// the twin sweeps load a chunk of kLineChunk positions (right-hand sides
// and coefficients) before running the recurrence on it, so the loads of a
// chunk overlap instead of serialising with the recurrence
constexpr int kLineChunk = 16;

// The line systems in three passes, each one launch for every axis: the
// right-hand sides of every padded cell (all divisions of the scheme's
// stencils, fully parallel), the twin back substitution in place, one thread
// per (axis, line, system) so the axes' lines and UCCD's upwind and downwind
// systems all run side by side (the sequential recurrences of one
// derivative cost the longest line, not the sum over axes), and the
// selection of the outputs (parallel again).  Same operations per value as
// the reference.  Each axis has its own scratch.
struct LineScratch {
  double *su[3], *ssu[3], *sd[3], *ssd[3];
};
// A kernel with a gate does nothing unless *flag is `call` (nullptr: no gate)
struct LineGate {
  const unsigned *flag;
  unsigned call;
  __device__ __forceinline__ bool closed() const { return flag && *flag != call; }
};
struct LineCoefs {
  const double *cu[3], *cd[3];
};

template <bool UP>
__global__ void __launch_bounds__(kLsBlock)
    k_compact_rhs(Grid g, const double *__restrict__ f, LineScratch sc, LineGate gate) {
#pragma clang fp contract(off)
  if (gate.closed()) return;
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= g.total) return;
  int q[3];
  padded_ijk(g, c, q);
  for (int a = 0; a < g.ndim; ++a) {
    const int i = q[a], n = g.N[a];
    const long st = g.s[a];
    const double *line = f + (c - (long)i * st);
    const double h = g.h[a];
    double s, ss;
    if (UP) {
      compact_rhs<1>(line, st, n, h, i, s, ss);
      sc.su[a][c] = s;
      sc.ssu[a][c] = ss;
      if (i > 0 && i < n - 1) compact_rhs<2>(line, st, n, h, i, s, ss);  // the ends are the upwind ones
      sc.sd[a][c] = s;
      sc.ssd[a][c] = ss;
    } else {
      compact_rhs<0>(line, st, n, h, i, s, ss);
      sc.su[a][c] = s;
      sc.ssu[a][c] = ss;
    }
  }
}

// twin_bks (matrix_solver.cpp:58-83) in place on S/SS holding the
// right-hand sides; thread t: axis a, then line t % lines, system t / lines
template <bool GATE>  // (looking at a gate costs a call of long lines 3 %)
__global__ void __launch_bounds__(64) k_twin_line(Grid g, int nsys, LineCoefs co, LineScratch sc, LineGate gate) {
#pragma clang fp contract(off)
  if (GATE && gate.closed()) return;
  constexpr int B = kLineChunk;
  long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  int a = 0;
  long lines = 0;
  for (; a < g.ndim; ++a) {
    lines = (long)g.N[(a + 1) % 3] * g.N[(a + 2) % 3];
    if (t < lines * nsys) break;
    t -= lines * nsys;
  }
  if (a >= g.ndim) return;
  const int sys = (int)(t / lines);
  long base;
  line_base(g, a, t % lines, base);
  const double *c = sys == 0 ? co.cu[a] : co.cd[a];
  double *S = (sys == 0 ? sc.su[a] : sc.sd[a]) + base, *SS = (sys == 0 ? sc.ssu[a] : sc.ssd[a]) + base;
  const int n = g.N[a];
  const long st = g.s[a];
  const double *a0 = c, *a1 = c + n, *a2 = c + 2 * n, *b0 = c + 3 * n, *b1 = c + 4 * n, *b2 = c + 5 * n;
  const double *aa0 = c + 6 * n, *aa1 = c + 7 * n, *aa2 = c + 8 * n, *bb0 = c + 9 * n, *bb1 = c + 10 * n,
               *bb2 = c + 11 * n;
  double sp = S[0], ssp = SS[0];
  for (int i0 = 1; i0 < n; i0 += B) {
    double r[B], rr[B], A0[B], B0[B], AA0[B], BB0[B];
#pragma unroll
    for (int q = 0; q < B; ++q) {
      const int i = i0 + q;
      if (i < n) {
        r[q] = S[(long)i * st];
        rr[q] = SS[(long)i * st];
        A0[q] = a0[i];
        B0[q] = b0[i];
        AA0[q] = aa0[i];
        BB0[q] = bb0[i];
      }
    }
#pragma unroll
    for (int q = 0; q < B; ++q) {
      const int i = i0 + q;
      if (i < n) {
        const double si = r[q] - (A0[q] * sp + B0[q] * ssp);
        const double ssi = rr[q] - (AA0[q] * sp + BB0[q] * ssp);
        S[(long)i * st] = si;
        SS[(long)i * st] = ssi;
        sp = si;
        ssp = ssi;
      }
    }
  }
  double den = a1[n - 1] * bb1[n - 1] - aa1[n - 1] * b1[n - 1];
  double sn = -(b1[n - 1] * ssp - bb1[n - 1] * sp) / den;
  double ssn = (a1[n - 1] * ssp - aa1[n - 1] * sp) / den;
  S[(long)(n - 1) * st] = sn;
  SS[(long)(n - 1) * st] = ssn;
  for (int i0 = n - 2; i0 >= 0; i0 -= B) {
    double Sv[B], SSv[B], A1[B], B1[B], AA1[B], BB1[B], A2[B], B2[B], AA2[B], BB2[B];
#pragma unroll
    for (int q = 0; q < B; ++q) {
      const int i = i0 - q;
      if (i >= 0) {
        Sv[q] = S[(long)i * st];
        SSv[q] = SS[(long)i * st];
        A1[q] = a1[i];
        B1[q] = b1[i];
        AA1[q] = aa1[i];
        BB1[q] = bb1[i];
        A2[q] = a2[i];
        B2[q] = b2[i];
        AA2[q] = aa2[i];
        BB2[q] = bb2[i];
      }
    }
#pragma unroll
    for (int q = 0; q < B; ++q) {
      const int i = i0 - q;
      if (i >= 0) {
        const double si = Sv[q] - (A2[q] * sn + B2[q] * ssn);
        const double ssi = SSv[q] - (AA2[q] * sn + BB2[q] * ssn);
        den = A1[q] * BB1[q] - AA1[q] * B1[q];
        const double sols = -(B1[q] * ssi - BB1[q] * si) / den;
        const double solss = (A1[q] * ssi - AA1[q] * si) / den;
        S[(long)i * st] = sols;
        SS[(long)i * st] = solss;
        sn = sols;
        ssn = solss;
      }
    }
  }
}

// ---- the sequential sweeps' values without their chain of 2 n steps.
// Both sweeps contract (|eig M_i| <= 0.25 and |eig D_i^-1 N_i| <= 0.65
// inside a line), and not only in exact arithmetic: two forward (backward)
// sweeps over the same right-hand sides that start from different states
// round to the same bits after some steps.  So every line is cut into
// segments, one thread each: a segment starts `warm` positions early from a
// zero state (or, if that reaches the line's end, from the exact one), sweeps
// up to its own first position, then sweeps its own positions in place.
// Whether the incoming state it arrived at equals the neighbour's final value
// is checked: if all do the result is the sequential sweep's, bit for bit.
// With the warm lengths below one of the workgroup's 500 states is not equal
// in 13 of 9.5 million workgroups (random, smooth and distance fields, 300 to
// 1400 points a line, UCCD; CCD none of 0.25 million), and always where the
// right-hand side is exactly 0 over a whole warm-up (fields of two values),
// which a zero state next to another one shows early.  Then, or if a value is
// not finite or nearly denormal, the workgroup forms its right-hand sides again
// and sweeps its lines end to end; where there are too many workgroups for that
// (scihpc_ls::twin_seg) the call is left to the three passes above, which
// return at once otherwise.
//
// A workgroup holds LINES whole lines in LDS, UCCD's two systems side by
// side, and does everything from the field to the derivatives: right-hand
// sides, sweeps, selection.  The factorised coefficients repeat along the
// line from about the 27th position on with a period of at most 3 (their
// elimination reaches a fixed point of the rounding), so a table of about 30
// rows serves any line; the host checks the period.  The backward sweep's
// quotients by the rows' determinants are formed from the stored reciprocal
// with two exact-remainder corrections, which rounds them correctly
// (Markstein: after the first correction the quotient is within an ulp, and
// the second, with the reciprocal correctly rounded, gives the nearest);
// only the sign of a zero may differ.  Segment lengths are odd, so the 64
// lanes of a wavefront (LINES lines x 64 / LINES segments) read different
// banks.
// What bounds it: the dependent FP64 operations of a lone wavefront for about
// 240 steps forward and 230 backward (instead of 2 x 1030; it issues in 30 %
// of its cycles), and LDS: whole lines leave one workgroup a CU, so 388
// workgroups run as two rounds.  Measured at 1024 x 512: 93 us, where right-hand sides, one thread a line and selection
// took 11.7 + 383 + 7.2 us in three launches; a UCCD TVD-RK3 step 1.24 ->
// 0.30 ms, of a field of two values 1.24 -> 0.77 (end to end with a thread a
// line and divisions it was 1.24).  Lines that do not fit LDS (over 4416
// points for UCCD, 6336 for CCD) keep the three passes.
struct TwinTable {
  const double *row[3][2];           // [axis][system]: rows of kTwinRow values
  int start[3][2], period[3][2], rows[3][2];
};
constexpr int kTwinRow = 14;         // a0 b0 aa0 bb0 | a2 b2 aa2 bb2 | a1 b1 aa1 bb1 | den 1/den
constexpr int kTwinRowsMax = 96;
struct TwinPlan {
  int waves;                         // wavefronts a system
  int len[3], segs[3];               // positions a segment (odd), segments
  int cap;                           // LDS doubles of one array
  int blocks[3];                     // workgroups of each axis
  unsigned *state;                   // [0]: the last call left to the three passes, [1]: workgroups that failed
  unsigned call;                     // number of this call
  int pass_on;                       // a failure leaves the whole call to the three passes
};
// warm-up positions [CCD, UCCD upwind, UCCD downwind]
__device__ constexpr int kTwinWarmF[3] = {102, 210, 48}, kTwinWarmB[3] = {102, 48, 192};

__device__ __forceinline__ double twin_quot(double a, double d, double r) {
#pragma clang fp contract(off)
  double q = a * r;
  q = __builtin_fma(__builtin_fma(-d, q, a), r, q);
  return __builtin_fma(__builtin_fma(-d, q, a), r, q);
}

// 0 < |x| < 2^-862 (but for |x| < 2^-1042): there twin_quot's remainders are
// no longer exact
constexpr unsigned kTwinTiny = ((1023u - 862u) << 21) - 1u;
__device__ __forceinline__ unsigned twin_size(double x) { return ((unsigned)__double2hiint(x) << 1) - 1u; }
__device__ __forceinline__ bool twin_tiny(double x) { return twin_size(x) < kTwinTiny; }

// the value of the other lane of a pair
__device__ __forceinline__ double twin_other(double x) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(x), 0xb1, 0xf, 0xf, true);
  return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(x), 0xb1, 0xf, 0xf, true), lo);
}

template <int LINES, bool UP>
__global__ void __launch_bounds__(512)  // two systems, at most four wavefronts each
    k_twin_seg(Grid g, const double *__restrict__ f, const double *__restrict__ u, const double *__restrict__ v,
               const double *__restrict__ w, TwinTable tb, TwinPlan pl, double *__restrict__ d1x,
               double *__restrict__ d1y, double *__restrict__ d1z, double *__restrict__ d2x,
               double *__restrict__ d2y, double *__restrict__ d2z) {
#pragma clang fp contract(off)
  constexpr int NS = UP ? 2 : 1;
  extern __shared__ __align__(16) double twin_lds[];
  // neighbouring line groups on one XCD, where their number allows: they share the field's cache lines
  int b = blockIdx.x;
  if (gridDim.x % 8 == 0) b = (b % 8) * (int)(gridDim.x / 8) + b / 8;
  int a = 0;
  while (a < 2 && b >= pl.blocks[a]) b -= pl.blocks[a++];
  const int n = g.N[a], len = pl.len[a], segs = pl.segs[a];
  const long st = g.s[a];
  const int tid = threadIdx.x, nt = blockDim.x;
  const int sys = UP ? tid / (64 * pl.waves) : 0;
  const int ts = tid - sys * 64 * pl.waves;
  __shared__ int whole;  // a thread found that the workgroup's lines have to be swept end to end
  if (tid == 0) whole = 0;
  if (pl.pass_on) {  // another workgroup has failed: its lines and these are the three passes' now
    __shared__ unsigned failed;
    if (tid == 0) failed = __hip_atomic_load(pl.state, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (failed == pl.call) return;
  }
  const int ln = ts % LINES, seg = ts / LINES;
  double *const S = twin_lds + (size_t)sys * 2 * pl.cap, *const SS = S + pl.cap;
  double *const tab = twin_lds + (size_t)(UP ? 4 : 3) * pl.cap;

  // The workgroup's cells, kTwinBatch a thread at a time so that their loads
  // are in flight together: get(address) of each, then put(value, LDS index,
  // address, line exists).  Neighbouring lanes take neighbouring cells in
  // memory: along the line where it is contiguous, else across the lines.
  constexpr int kTwinBatch = 16;
  const long line0 = (long)b * LINES, lines = (long)g.N[(a + 1) % 3] * g.N[(a + 2) % 3];
  const bool along = st == 1;
  long own_base = 0;
  const bool own_ok = line_base(g, a, line0 + tid % LINES, own_base);
  const int hop = along ? nt : nt / LINES;
  const long hop_c = hop * st;
  auto cells = [&](auto get, auto put) {
    for (int i0 = along ? tid : tid / LINES; i0 < n; i0 += (along ? kTwinBatch / LINES : kTwinBatch) * hop) {
      double v[kTwinBatch];
      const long c0 = (along ? line0 * n : own_base) + i0 * st;
#pragma unroll
      for (int q = 0; q < kTwinBatch; ++q) {
        const int i = i0 + (along ? q / LINES : q) * hop;
        const bool ok = i < n && (along ? line0 + q % LINES < lines : own_ok);
        const long c = c0 + (along ? (q % LINES) * n + (q / LINES) * hop : q * hop_c);
        v[q] = ok ? get(c) : 0.0;
      }
#pragma unroll
      for (int q = 0; q < kTwinBatch; ++q) {
        const int i = i0 + (along ? q / LINES : q) * hop, l = along ? q % LINES : tid % LINES;
        const bool ok = along ? line0 + q % LINES < lines : own_ok;
        const long c = c0 + (along ? (q % LINES) * n + (q / LINES) * hop : q * hop_c);
        if (i < n) put(v[q], i, l, c, ok);
      }
    }
  };
  // the right-hand sides, exactly: compact_rhs from the field in memory
  auto fill = [&]() {
    cells([](long) { return 0.0; }, [&](double, int i, int l, long c, bool ok) {
      double s0 = 0.0, ss0 = 0.0, s1 = 0.0, ss1 = 0.0;
      if (ok) {
        const double *line = f + (c - (long)i * st);
        if (UP) {
          compact_rhs<1>(line, st, n, g.h[a], i, s0, ss0);
          s1 = s0;
          ss1 = ss0;
          if (i > 0 && i < n - 1) compact_rhs<2>(line, st, n, g.h[a], i, s1, ss1);  // the ends are the upwind ones
        } else {
          compact_rhs<0>(line, st, n, g.h[a], i, s0, ss0);
        }
      }
      double *p = twin_lds + i * LINES + l;
      p[0] = s0;
      p[pl.cap] = ss0;
      if (UP) {
        p[2 * pl.cap] = s1;
        p[3 * pl.cap] = ss1;
      }
    });
  };
  for (int y = 0; y < NS; ++y)
    for (int t = tid; t < kTwinRow * tb.rows[a][y]; t += nt) tab[y * kTwinRow * kTwinRowsMax + t] = tb.row[a][y][t];
  {
    // The same values from LDS: the field goes to the last array (UCCD: the
    // downwind f'' array, which gets its values from the upwind one), then
    // every right-hand side to its own.  The
    // divisions by h are twin_quot's (a value that is not finite there ends in
    // the exact path below).
    double *const F = twin_lds + (size_t)(UP ? 3 : 2) * pl.cap;
    cells([&](long c) { return f[c]; }, [&](double z, int i, int l, long, bool) { F[i * LINES + l] = z; });
    __syncthreads();
    const double h = g.h[a], rh = 1.0 / h;
    auto rhs = [&](int l, int i, double &s0, double &ss0, double &s1) {
      const double *z = F + l;
      if (i == 0 || i == n - 1) {  // the one-sided ends
        const int o = i == 0 ? 0 : (n - 1) * LINES, d = i == 0 ? LINES : -LINES;
        const double x0 = z[o], x1 = z[o + d], x2 = z[o + 2 * d];
        const double e = -3.5 * x0 + 4.0 * x1 + -0.5 * x2, ee = 9.0 * x0 + -12.0 * x1 + 3.0 * x2;
        s0 = s1 = twin_quot(i == 0 ? e : -e, h, rh);
        ss0 = twin_quot(twin_quot(ee, h, rh), h, rh);
        return;
      }
      const double c3 = -0.06096119008109, c2 = 1.99692238016218, c1 = -1.93596119008109;
      const double m = z[(i - 1) * LINES], c = z[i * LINES], q = z[(i + 1) * LINES];
      if (UP) {
        s0 = twin_quot(c1 * m + c2 * c + c3 * q, h, rh);
        s1 = twin_quot(-(c3 * m + c2 * c + c1 * q), h, rh);
      } else {
        s0 = twin_quot(15.0 / 16.0 * (q - m), h, rh);
      }
      ss0 = twin_quot(twin_quot(3.0 * m - 6.0 * c + 3.0 * q, h, rh), h, rh);
    };
    const int m = n * LINES;  // cell t of these: position t / LINES, line t % LINES
#pragma unroll 4
    for (int t = tid; t < m; t += nt) {
      double s0, ss0, s1 = 0.0;
      rhs(t % LINES, t / LINES, s0, ss0, s1);
      twin_lds[t] = s0;
      twin_lds[pl.cap + t] = ss0;
      if (UP) twin_lds[2 * pl.cap + t] = s1;
    }
    if (UP) {
      __syncthreads();
#pragma unroll 4
      for (int t = tid; t < m; t += nt) twin_lds[3 * pl.cap + t] = twin_lds[pl.cap + t];
    }
  }
  __syncthreads();

  const double *const T = tab + sys * kTwinRow * kTwinRowsMax;
  const int start = tb.start[a][sys], period = tb.period[a][sys], rows = tb.rows[a][sys];
  const int kind = UP ? 1 + sys : 0;
  const int lo = seg * len, hi = min(n, lo + len);
  const bool on = seg < segs && lo < n;
  int bad = 0;  // a state that does not match, or a value that twin_quot may not round exactly
  auto at = [&](int i) { return i * LINES + ln; };

  // A step's cost is the instructions a lone wavefront issues for it, so
  // where the rows repeat (from `start` on; the period divides kTwinUnroll)
  // a thread keeps its kTwinUnroll rows in registers and runs blocks of that
  // many steps with nothing but the values to load; single steps with the
  // row looked up are left for the line's beginning and the remainders.
  constexpr int kTwinUnroll = 6;
  auto frow = [&](const double *c, double vs, double vss, double &p, double &q) {
    const double x = vs - (c[0] * p + c[1] * q);
    const double y = vss - (c[2] * p + c[3] * q);
    p = x;
    q = y;
  };
  auto fstep = [&](int i, int r, bool keep, double &p, double &q) {
    frow(T + r * kTwinRow, S[at(i)], SS[at(i)], p, q);
    if (keep) {
      S[at(i)] = p;
      SS[at(i)] = q;
    }
  };
  auto forward = [&](int i, int end, bool keep, double &p, double &q) {
#pragma unroll 2
    for (; i < min(end, start); ++i) fstep(i, i == n - 1 ? rows - 1 : i, keep, p, q);
    if (i >= end) return;
    const int stop = min(end, n - 1);
    int ph = (int)((unsigned)(i - start) % (unsigned)period);
    if (i + kTwinUnroll <= stop) {
      double c[kTwinUnroll][4];
      int w = ph;
#pragma unroll
      for (int k = 0; k < kTwinUnroll; ++k) {
#pragma unroll
        for (int e = 0; e < 4; ++e) c[k][e] = T[(start + w) * kTwinRow + e];
        w = w + 1 == period ? 0 : w + 1;
      }
      do {
        double vs[kTwinUnroll], vss[kTwinUnroll];
#pragma unroll
        for (int k = 0; k < kTwinUnroll; ++k) {
          vs[k] = S[at(i + k)];
          vss[k] = SS[at(i + k)];
        }
#pragma unroll
        for (int k = 0; k < kTwinUnroll; ++k) {
          frow(c[k], vs[k], vss[k], p, q);
          if (keep) {
            S[at(i + k)] = p;
            SS[at(i + k)] = q;
          }
        }
        i += kTwinUnroll;
      } while (i + kTwinUnroll <= stop);
    }
    for (; i < end; ++i) {
      fstep(i, i == n - 1 ? rows - 1 : start + ph, keep, p, q);
      ph = ph + 1 == period ? 0 : ph + 1;
    }
  };
  // backward, the same way; the closure at n - 1 is not one of these steps
  auto solve2 = [&](const double *c, double si, double ti, double &x, double &y) {
    x = twin_quot(-(c[5] * ti - c[7] * si), c[8], c[9]);
    y = twin_quot(c[4] * ti - c[6] * si, c[8], c[9]);
  };
  auto brow = [&](const double *c, double vs, double vss, double &x, double &y) {
    solve2(c, vs - (c[0] * x + c[1] * y), vss - (c[2] * x + c[3] * y), x, y);
  };
  auto bstep = [&](int i, int r, bool keep, double &x, double &y) {
    brow(T + r * kTwinRow + 4, S[at(i)], SS[at(i)], x, y);
    if (keep) {
      bad |= twin_tiny(x) || twin_tiny(y);
      S[at(i)] = x;
      SS[at(i)] = y;
    }
  };
  auto backward = [&](int i, int end, bool keep, double &x, double &y) {
    const int stop = max(end, start);
    if (i >= stop) {
      int ph = (int)((unsigned)(i - start) % (unsigned)period);
      if (i - kTwinUnroll + 1 >= stop) {
        double c[kTwinUnroll][10];
        int w = ph;
#pragma unroll
        for (int k = 0; k < kTwinUnroll; ++k) {
#pragma unroll
          for (int e = 0; e < 10; ++e) c[k][e] = T[(start + w) * kTwinRow + 4 + e];
          w = w == 0 ? period - 1 : w - 1;
        }
        do {
          double vs[kTwinUnroll], vss[kTwinUnroll];
#pragma unroll
          for (int k = 0; k < kTwinUnroll; ++k) {
            vs[k] = S[at(i - k)];
            vss[k] = SS[at(i - k)];
          }
#pragma unroll
          for (int k = 0; k < kTwinUnroll; ++k) {
            brow(c[k], vs[k], vss[k], x, y);
            if (keep) {
              bad |= twin_tiny(x) || twin_tiny(y);
              S[at(i - k)] = x;
              SS[at(i - k)] = y;
            }
          }
          i -= kTwinUnroll;
        } while (i - kTwinUnroll + 1 >= stop);
      }
      for (; i >= stop; --i) {
        bstep(i, start + ph, keep, x, y);
        ph = ph == 0 ? period - 1 : ph - 1;
      }
    }
#pragma unroll 2
    for (; i >= end; --i) bstep(i, i, keep, x, y);
  };
  // A zero state after a warm-up that did not reach the line's start, next to
  // a segment with another state: the right-hand side is 0 over the whole
  // warm-up but not before it, and the neighbour's final state is what is left
  // of that, not 0.  No need to sweep on before the lines are swept end to
  // end (a pair of segments in two wavefronts is left to the comparison).
  double p = 0.0, q = 0.0;
  bool flat = false;
  if (on) {
    const int i = max(lo - kTwinWarmF[kind], 1);
    if (i == 1 || seg == 0) {
      p = S[at(0)];
      q = SS[at(0)];
    }
    flat = i > 1;
    forward(i, lo, false, p, q);
  }
  {
    const int rest = p != 0.0 || q != 0.0, before = __shfl_up(rest, LINES, 64);
    flat = flat && !rest && before;  // lanes of the first segment keep their own: not flat
  }
  // `whole` is written between two barriers and read after the second: a
  // thread that is ahead can't write it again before all have read it
  if (flat) whole = 1;
  __syncthreads();
  double x = 0.0, y = 0.0;
  bool alone = whole;
  if (!alone) {
    const double pin = p, qin = q;
    if (on) forward(max(lo, 1), hi, true, p, q);
    __syncthreads();
    if (on && seg > 0)
      bad |= S[at(lo - 1)] != pin || SS[at(lo - 1)] != qin;
    flat = false;
    if (on) {
      int i = min(hi - 1 + kTwinWarmB[kind], n - 1);
      flat = i < n - 1;
      if (i == n - 1) {  // the closure
        solve2(T + (rows - 1) * kTwinRow + 4, S[at(i)], SS[at(i)], x, y);
        --i;
      }
      backward(i, hi, false, x, y);
    }
    const int rest = x != 0.0 || y != 0.0, after = __shfl_down(rest, LINES, 64);
    if (bad || (flat && !rest && after)) whole = 1;
    __syncthreads();
    alone = whole;
  }
  if (!alone) {
    const double xin = x, yin = y;
    if (on) {
      if (hi == n) {
        S[at(n - 1)] = x;
        SS[at(n - 1)] = y;
      }
      backward(min(hi - 1, n - 2), lo, true, x, y);
      bad |= !(fabs(x) < __builtin_inf()) || !(fabs(y) < __builtin_inf());
    }
    __syncthreads();
    if (on && hi < n)
      bad |= S[at(hi)] != xin || SS[at(hi)] != yin;
    if (bad) whole = 1;
    __syncthreads();
    alone = whole;
  }
  if (alone && tid == 0) {
    atomicAdd(pl.state + 1, 1u);
    if (pl.pass_on) __hip_atomic_store(pl.state, pl.call, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (alone && pl.pass_on) return;
  if (alone) {
    // From end to end, two lanes a line: one holds f', the other f'', and they
    // exchange them; a wavefront on its own is bound by the instructions of a
    // step, and this halves them (68 clocks a position forward and 150
    // backward, 110 and 270 with one lane and divisions).  Blocks of steps
    // whose quotients may not be IEEE ones are done again with divisions.
    fill();
    __syncthreads();
    if (ts < 2 * LINES) {
      const int half = ts & 1;
      double *const V = (half ? SS : S) + (ts >> 1);
      // where this lane's coefficients are in a row: of its own and of the
      // other's value, in the recurrences (backward: 4 further) and in the
      // numerators
      const int cm = half ? 3 : 0, co = half ? 2 : 1, nm = half ? 8 : 11, no = half ? 10 : 9;
      double m = V[0];
      auto next = [&](double v, double a, double b) { return v - (a * m + b * twin_other(m)); };
      auto fone = [&](int i, int r) {
        m = next(V[i * LINES], T[r * kTwinRow + cm], T[r * kTwinRow + co]);
        V[i * LINES] = m;
      };
      int i = 1;
      for (; i < min(start, n - 1); ++i) fone(i, i);
      if (i + kTwinUnroll <= n - 1) {
        double c[kTwinUnroll][2];
#pragma unroll
        for (int k = 0; k < kTwinUnroll; ++k) {
          const double *r = T + (start + (i - start + k) % period) * kTwinRow;
          c[k][0] = r[cm];
          c[k][1] = r[co];
        }
        for (; i + kTwinUnroll <= n - 1; i += kTwinUnroll) {
          double v[kTwinUnroll];
#pragma unroll
          for (int k = 0; k < kTwinUnroll; ++k) v[k] = V[(i + k) * LINES];
#pragma unroll
          for (int k = 0; k < kTwinUnroll; ++k) V[(i + k) * LINES] = m = next(v[k], c[k][0], c[k][1]);
        }
      }
      for (; i < n - 1; ++i) fone(i, start + (i - start) % period);
      fone(i, rows - 1);
      // backward from the closure
      auto num = [&](double w, double a, double b) { return a * w - b * twin_other(w); };
      const double *const R = T + (rows - 1) * kTwinRow;
      V[(n - 1) * LINES] = m = num(m, R[nm], R[no]) / R[12];
      auto bone = [&](int j, int r) {
        const double *c = T + r * kTwinRow;
        V[j * LINES] = m = num(next(V[j * LINES], c[4 + cm], c[4 + co]), c[nm], c[no]) / c[12];
      };
      for (i = n - 2; i >= start && (i - start + 1) % kTwinUnroll != 0; --i) bone(i, start + (i - start) % period);
      if (i >= start) {
        double c[kTwinUnroll][6];
#pragma unroll
        for (int k = 0; k < kTwinUnroll; ++k) {
          const double *r = T + (start + (kTwinUnroll - 1 - k) % period) * kTwinRow;
          c[k][0] = r[4 + cm];
          c[k][1] = r[4 + co];
          c[k][2] = r[nm];
          c[k][3] = r[no];
          c[k][4] = r[12];
          c[k][5] = r[13];
        }
        for (; i >= start; i -= kTwinUnroll) {
          double v[kTwinUnroll], z[kTwinUnroll];
#pragma unroll
          for (int k = 0; k < kTwinUnroll; ++k) v[k] = V[(i - k) * LINES];
          const double m0 = m;
          unsigned low = 0xffffffffu;
#pragma unroll
          for (int k = 0; k < kTwinUnroll; ++k) {
            z[k] = m = twin_quot(num(next(v[k], c[k][0], c[k][1]), c[k][2], c[k][3]), c[k][4], c[k][5]);
            low = min(low, twin_size(m));
          }
          int redo = low < kTwinTiny || !(fabs(m) < __builtin_inf());  // what isn't finite stays so
          redo |= __builtin_amdgcn_mov_dpp(redo, 0xb1, 0xf, 0xf, true);
          if (redo) {
            m = m0;
#pragma unroll
            for (int k = 0; k < kTwinUnroll; ++k)
              z[k] = m = num(next(v[k], c[k][0], c[k][1]), c[k][2], c[k][3]) / c[k][4];
          }
#pragma unroll
          for (int k = 0; k < kTwinUnroll; ++k) V[(i - k) * LINES] = z[k];
        }
      }
      for (; i >= 0; --i) bone(i, i);
    }
    __syncthreads();
  }

  // the derivatives, as k_compact_select forms them
  const double *vel = a == 0 ? u : a == 1 ? v : w;
  double *const d1 = a == 0 ? d1x : a == 1 ? d1y : d1z, *const d2 = a == 0 ? d2x : a == 1 ? d2y : d2z;
  cells([&](long c) { return UP ? vel[c] : 0.0; }, [&](double vc, int i, int l, long c, bool ok) {
    if (!ok) return;
    const double *z = twin_lds + i * LINES + l;
    if (UP) {
      d1[c] = vc > 0 ? z[0] : z[2 * pl.cap];
      if (d2) d2[c] = 0.5 * (z[pl.cap] + z[3 * pl.cap]);
    } else {
      d1[c] = z[0];
      if (d2) d2[c] = z[pl.cap];
    }
  });
}

// The twin sweeps partitioned along the line, for the latency of the
// recurrence: k_twin_line's chain of 2 n dependent steps per line (with two
// FP64 divisions per backward step) on a few thousand threads becomes about
// 4 L steps on ceil(n / L) threads per line, L = 9 (17 for lines of more
// than 1152 points) positions a segment.  Both sweeps are
// affine recurrences in the state (s, ss):
//   forward   y_i = r_i - M_i y_{i-1},               M_i = [a0 b0; aa0 bb0]
//   backward  u_i = D_i^-1 (y_i - N_i u_{i+1}),      D_i = [a1 b1; aa1 bb1],
//                                                    N_i = [a2 b2; aa2 bb2]
// so a segment's end state is its end state from a zero incoming state
// plus a fixed 2x2 propagator times the true incoming state (Phi: the
// product of -M_i over the segment; Psi: of -D_i^-1 N_i, from the top; both
// depend only on the coefficients and are formed on the host).  A
// workgroup holds LINES lines x SEGS segments: (1) every segment runs its
// recurrence from a zero incoming state (segment 0 from y_0, the top
// segment from the closure u_{n-1}: both exact), (2) one thread per line
// chains the segment ends through the propagators (staged in LDS), giving every
// segment its true incoming state, (3) every segment runs the recurrence
// again from that state, with k_twin_line's arithmetic, and keeps the
// result -- so a value differs from the sequential sweep's only through the
// carried incoming state, whose rounding the contracting recurrences damp
// (|eig M_i| <= 0.25 and |eig D_i^-1 N_i| <= 0.65 inside the line).  The
// segment's right-hand sides stay in registers between the passes: HBM
// sees one read and one write per value.  Thread t: line t % LINES of the
// group, segment t / LINES; block b: axis, then system, then line group.
struct LineCarry {
  const double *phi[3][2], *psi[3][2];  // [axis][system]: SEGS 2x2 propagators, row-major
};

template <int LINES, int L, bool CL>  // L: positions a segment (in registers); CL: coefficients in LDS
__global__ void __launch_bounds__(1024) k_twin_part(Grid g, int nsys, LineCoefs co, LineScratch sc, LineCarry cr) {
#pragma clang fp contract(off)
  constexpr int SEGS = 1024 / LINES;
  __shared__ double e0[SEGS][LINES], e1[SEGS][LINES];  // segment end states, then incoming states
  __shared__ double prop[2][4 * SEGS];                  // Phi and Psi of this axis and system
  int b = blockIdx.x, a = 0, sys = 0;
  long lines = 0;
  for (; a < g.ndim; ++a) {
    lines = (long)g.N[(a + 1) % 3] * g.N[(a + 2) % 3];
    const int nbl = (int)((lines + LINES - 1) / LINES);
    if (b < nbl * nsys) {
      sys = b / nbl;
      b -= sys * nbl;
      break;
    }
    b -= nbl * nsys;
  }
  if (a >= g.ndim) return;  // uniform over the block
  const int n = g.N[a];
  const int Lp = L, ns = (n + L - 1) / L, top = ns - 1;  // ns <= SEGS (host)
  const int ln = (int)threadIdx.x % LINES, seg = (int)threadIdx.x / LINES;
  long base = 0;
  const bool line_ok = line_base(g, a, (long)b * LINES + ln, base);
  const int lo = seg * Lp;
  const int len = line_ok && lo < n ? min(Lp, n - lo) : 0;
  for (int q = threadIdx.x; q < 4 * ns; q += blockDim.x) {
    prop[0][q] = cr.phi[a][sys][q];
    prop[1][q] = cr.psi[a][sys][q];
  }
  const double *cg = sys == 0 ? co.cu[a] : co.cd[a];
  // the coefficients in LDS (dynamic, 96 n bytes) when the launch gave it
  extern __shared__ double cl[];
  if (CL)
    for (int q = threadIdx.x; q < 12 * n; q += blockDim.x) cl[q] = cg[q];
  const double *c = CL ? cl : cg;
  const double *a0 = c, *a1 = c + n, *a2 = c + 2 * n, *b0 = c + 3 * n, *b1 = c + 4 * n, *b2 = c + 5 * n;
  const double *aa0 = c + 6 * n, *aa1 = c + 7 * n, *aa2 = c + 8 * n, *bb0 = c + 9 * n, *bb1 = c + 10 * n,
               *bb2 = c + 11 * n;
  double *S = (sys == 0 ? sc.su[a] : sc.sd[a]) + base, *SS = (sys == 0 ? sc.ssu[a] : sc.ssd[a]) + base;
  const long st = g.s[a];
  double v[L], vv[L];
#pragma unroll
  for (int q = 0; q < L; ++q) {
    if (q < len) {
      v[q] = S[(long)(lo + q) * st];
      vv[q] = SS[(long)(lo + q) * st];
    }
  }
  // forward sweep over the segment from (p, pp); keep = store the states
  auto forward = [&](double p, double pp, bool keep) {
#pragma unroll
    for (int q = 0; q < L; ++q) {
      const int i = lo + q;
      if (q < len && i > 0) {
        const double si = v[q] - (a0[i] * p + b0[i] * pp);
        const double ssi = vv[q] - (aa0[i] * p + bb0[i] * pp);
        if (keep) {
          v[q] = si;
          vv[q] = ssi;
        }
        p = si;
        pp = ssi;
      }
    }
    e0[seg][ln] = p;
    e1[seg][ln] = pp;
  };
  if (CL) __syncthreads();  // the coefficients are staged
  forward(seg == 0 && len > 0 ? v[0] : 0.0, seg == 0 && len > 0 ? vv[0] : 0.0, false);
  __syncthreads();
  if (seg == 0 && line_ok) {
    double y = e0[0][ln], yy = e1[0][ln];
#pragma unroll 4
    for (int k = 1; k < ns; ++k) {
      const double *F = &prop[0][4 * k];
      const double h0 = e0[k][ln], h1 = e1[k][ln];
      e0[k][ln] = y;
      e1[k][ln] = yy;
      const double y0 = h0 + (F[0] * y + F[1] * yy), y1 = h1 + (F[2] * y + F[3] * yy);
      y = y0;
      yy = y1;
    }
  }
  __syncthreads();
  forward(seg == 0 ? (len > 0 ? v[0] : 0.0) : e0[seg][ln], seg == 0 ? (len > 0 ? vv[0] : 0.0) : e1[seg][ln], true);
  // the closure at i = n - 1 (in the top segment's registers)
  if (seg == top && len > 0) {
    const int i = n - 1;
#pragma unroll
    for (int q = 0; q < L; ++q) {  // static register indices
      if (q == len - 1) {
        const double den = a1[i] * bb1[i] - aa1[i] * b1[i];
        const double sn = -(b1[i] * vv[q] - bb1[i] * v[q]) / den;
        const double ssn = (a1[i] * vv[q] - aa1[i] * v[q]) / den;
        v[q] = sn;
        vv[q] = ssn;
      }
    }
  }
  __syncthreads();  // the forward pass's stores to e0/e1 are read no more
  // backward sweep over the segment from the incoming (p, pp) at lo + len
  auto backward = [&](double p, double pp, bool keep) {
#pragma unroll
    for (int q = L - 1; q >= 0; --q) {
      const int i = lo + q;
      if (q < len && i < n - 1) {
        const double si = v[q] - (a2[i] * p + b2[i] * pp);
        const double ssi = vv[q] - (aa2[i] * p + bb2[i] * pp);
        const double den = a1[i] * bb1[i] - aa1[i] * b1[i];
        const double sols = -(b1[i] * ssi - bb1[i] * si) / den;
        const double solss = (a1[i] * ssi - aa1[i] * si) / den;
        if (keep) {
          v[q] = sols;
          vv[q] = solss;
        }
        p = sols;
        pp = solss;
      } else if (q < len) {  // i = n - 1: the closure value, already in place
        p = v[q];
        pp = vv[q];
      }
    }
    e0[seg][ln] = p;
    e1[seg][ln] = pp;
  };
  backward(0.0, 0.0, false);
  __syncthreads();
  if (seg == 0 && line_ok) {
    double u = e0[top][ln], uu = e1[top][ln];
#pragma unroll 4
    for (int k = top - 1; k >= 0; --k) {
      const double *G = &prop[1][4 * k];
      const double h0 = e0[k][ln], h1 = e1[k][ln];
      e0[k][ln] = u;
      e1[k][ln] = uu;
      const double u0 = h0 + (G[0] * u + G[1] * uu), u1 = h1 + (G[2] * u + G[3] * uu);
      u = u0;
      uu = u1;
    }
  }
  __syncthreads();
  backward(seg == top ? 0.0 : e0[seg][ln], seg == top ? 0.0 : e1[seg][ln], true);
#pragma unroll
  for (int q = 0; q < L; ++q) {
    if (q < len) {
      S[(long)(lo + q) * st] = v[q];
      SS[(long)(lo + q) * st] = vv[q];
    }
  }
}

template <bool UP>
__global__ void __launch_bounds__(kLsBlock)
    k_compact_select(long total, int ndim, const double *__restrict__ u, const double *__restrict__ v,
                     const double *__restrict__ w, LineScratch sc, double *d1x, double *d1y, double *d1z,
                     double *d2x, double *d2y, double *d2z, LineGate gate) {
#pragma clang fp contract(off)
  if (gate.closed()) return;
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= total) return;
  const double *vel[3] = {u, v, w};
  double *d1[3] = {d1x, d1y, d1z}, *d2[3] = {d2x, d2y, d2z};
  for (int a = 0; a < ndim; ++a) {
    if (UP) {
      d1[a][c] = vel[a][c] > 0 ? sc.su[a][c] : sc.sd[a][c];
      if (d2[a]) d2[a][c] = 0.5 * (sc.ssu[a][c] + sc.ssd[a][c]);
    } else {
      d1[a][c] = sc.su[a][c];
      if (d2[a]) d2[a][c] = sc.ssu[a][c];
    }
  }
}

// the TVD-RK3 stage update (runge_kutta.cpp:13-49) at padded cell c: from
// value x and rate s
template <int STAGE>
__device__ __forceinline__ double rk3_update(double x, double s, long c, double *__restrict__ s1,
                                                double *__restrict__ s2, double dt) {
#pragma clang fp contract(off)
  if (STAGE == 1) {
    s1[c] = s;
    return x + dt * s;
  }
  if (STAGE == 2) {
    s2[c] = s;
    return x + dt * (s - 3.0 * s1[c]) / 4.0;
  }
  return x + dt * (-s1[c] - s2[c] + 8.0 * s) / 12.0;
}

// convection (source.cpp:8-40), the TVD-RK3 stage update and the ghosts of
// any boundary condition but Dirichlet (`ghosts`), in place.  Ghosts outside
// on one axis are their boundary condition's; those outside on more are
// advanced like cells.  Bound by its 64 bytes a cell; with the ghosts in
// launches of their own a stage at 1024 x 512 took 7 + 2 x 4.7 us, here 8.
template <int DIM, int STAGE>
__global__ void __launch_bounds__(kLsBlock)
    k_uccd_stage(Grid g, double *__restrict__ phi, const double *__restrict__ u, const double *__restrict__ v,
                 const double *__restrict__ w, const double *__restrict__ fx, const double *__restrict__ fy,
                 const double *__restrict__ fz, double *__restrict__ s1, double *__restrict__ s2, double dt,
                 BcSpec bc, int ghosts) {
#pragma clang fp contract(off)
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= g.total) return;
  int q[3] = {0, 0, 0}, out = 0;
  if (ghosts) {  // (else every cell is advanced and apply_bc fills the ghosts)
    padded_ijk(g, c, q);
#pragma unroll
    for (int a = 0; a < DIM; ++a) out += q[a] < g.off[a] || q[a] >= g.off[a] + g.n[a];
    if (out == 1) return;
  }
  double s = -u[c] * fx[c];
  if (DIM > 1) s -= v[c] * fy[c];
  if (DIM > 2) s -= w[c] * fz[c];
  const double y = rk3_update<STAGE>(phi[c], s, c, s1, s2, dt);
  phi[c] = y;
  if (out == 0 && ghosts) {
#pragma unroll
    for (int a = 0; a < DIM; ++a) ghosts_of(bc, a, g.n[a], g.h[a], g.s[a], q[a] - g.off[a], y, phi + c);
  }
}

__device__ __forceinline__ double ls_heav(double x, double w) {
#pragma clang fp contract(off)
  const double pi = 3.14159265358979323846;
  if (x < -w) return 0;
  if (x > w) return 1;
  return 0.5 * (1 + x / w + sin(pi * x / w) / pi);
}

__device__ __forceinline__ double ls_delta(double x, double w) {
#pragma clang fp contract(off)
  const double pi = 3.14159265358979323846;
  if (x < -w) return 0;
  if (x > w) return 0;
  return 0.5 * (1 + cos(pi * x / w)) / w;
}

// identity_with_extrapolation: flux(c) = phi(clamped c) on every padded cell
template <int DIM>
__global__ void __launch_bounds__(kLsBlock) k_extrap(Grid g, const double *__restrict__ phi,
                                                     double *__restrict__ flux) {
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= g.total) return;
  int q[3];
  padded_ijk(g, c, q);
  flux[c] = phi[ext_index<DIM>(g, q, -1)];
}

__device__ __forceinline__ double grad_mag(int dim, double fx, double fy, double fz) {
#pragma clang fp contract(off)
  double gr = fx * fx;
  if (dim > 1) gr += fy * fy;
  if (dim > 2) gr += fz * fz;
  return sqrt(gr);
}

// per interior cell: the lsf_mass term (wrapper_func.cpp:450-511) and the
// mpls denominator term g delta |grad| (source.cpp:119-138); part[2b],
// part[2b+1] = block sums
template <int DIM>
__global__ void __launch_bounds__(kLsBlock)
    k_mpls_sums(Grid g, const double *__restrict__ phi, const double *__restrict__ fx,
                const double *__restrict__ fy, const double *__restrict__ fz, double w, double ratio,
                int positive_ref, double dv, double *__restrict__ part) {
#pragma clang fp contract(off)
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  double m = 0.0, e = 0.0;
  if (t < g.interior) {
    int I, J, K;
    interior_ijk(g, t, I, J, K);
    const long c = pidx(g, I, J, K);
    auto dens = [&](long q, double &H) {
      H = ls_heav(phi[q], w);
      return positive_ref ? H + (1.0 - H) * ratio : (1.0 - H) + H * ratio;
    };
    double Hc;
    const double dc = dens(c, Hc);
    const bool inner = I != 0 && I != g.n[0] - 1 && J != 0 && J != g.n[1] - 1 &&
                       (DIM == 2 || (K != 0 && K != g.n[2] - 1));
    if (DIM == 2) {
      if (inner) {
        double lm = 15.0 * dc * Hc;
        for (int ii = -1; ii < 2; ++ii)
          for (int jj = -1; jj < 2; ++jj) {
            double H;
            const long q = c + ii * g.s[0] + jj * g.s[1];
            const double d = dens(q, H);
            lm += d * H;
          }
        m = lm / 24.0;
      } else {
        m = dc * Hc;
      }
    } else {
      if (inner) {
        double lm = 50.0 * dc * Hc;
        for (int ii = -1; ii < 2; ++ii)
          for (int jj = -1; jj < 2; ++jj)
            for (int kk = -1; kk < 2; ++kk) {
              double H;
              const long q = c + ii * g.s[0] + jj * g.s[1] + kk * g.s[2];
              const double d = dens(q, H);
              lm += d * H;
            }
        m = lm * dv / 77.0;
      } else {
        m = dc * Hc * dv;
      }
    }
    const double dl = ls_delta(phi[c], w);
    const double gr = grad_mag(DIM, fx[c], fy[c], DIM > 2 ? fz[c] : 0.0);
    double gg = dl * (2.0 * (1.0 - ratio) * Hc + ratio);
    if (!positive_ref) gg = dl * (2.0 * (ratio - 1.0) * Hc + 1.0);
    e = gg * dl * gr;
  }
  m = block_sum(m);
  e = block_sum(e);
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = m;
    part[2 * blockIdx.x + 1] = e;
  }
}

// runge_kutta::euler with s = eta delta |grad| on every padded cell; the
// delta of the pre-update phi is kept (dummy->delta)
template <int DIM>
__global__ void __launch_bounds__(kLsBlock)
    k_mpls_update(long n, double *__restrict__ phi, const double *__restrict__ fx, const double *__restrict__ fy,
                  const double *__restrict__ fz, double w, const double *__restrict__ eta_p, double dt,
                  double *__restrict__ delta) {
#pragma clang fp contract(off)
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n) return;
  const double eta = *eta_p;
  const double dl = ls_delta(phi[c], w);
  const double gr = grad_mag(DIM, fx[c], fy[c], DIM > 2 ? fz[c] : 0.0);
  delta[c] = dl;
  phi[c] += dt * (eta * dl * gr);
}

// eta = (mass0 - mass) / (den dv dt) from the block sums of k_mpls_sums,
// on the device (one workgroup, fixed summation order): the Euler update
// then needs no host round trip
__global__ void __launch_bounds__(kLsBlock)
    k_mpls_eta(const double *__restrict__ part, int nb, double mass0, double dv, double dt,
               double *__restrict__ eta) {
#pragma clang fp contract(off)
  double m = 0.0, e = 0.0;
  for (int b = threadIdx.x; b < nb; b += blockDim.x) {
    m += part[2 * b];
    e += part[2 * b + 1];
  }
  m = block_sum(m);
  e = block_sum(e);
  if (threadIdx.x == 0) {
    const double mass = m * dv;
    eta[0] = (mass0 - mass) / (e * dv * dt);
  }
}

__global__ void __launch_bounds__(kLsBlock)
    k_sign_delta(long n, const double *__restrict__ phi, double w, double *__restrict__ sign,
                 double *__restrict__ delta) {
#pragma clang fp contract(off)
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n) return;
  const double x = phi[c];
  if (sign) {
    double sg;
    if (x < -w) sg = -1;
    else if (x > w) sg = 1;
    else sg = x / sqrt(x * x + w * w);
    sign[c] = sg;
  }
  if (delta) delta[c] = ls_delta(x, w);
}

// weno5_for_godunov (godunov_gradient.cpp:184-201): w0 / 3 (a - 2b + c) +
// (w2 - 1/2) / 6 (b - 2c + d) with weights w_k = alpha_k / (alpha_0 +
// alpha_1 + alpha_2), alpha = (1, 6, 3) / e_k^2.  Over their common
// denominator the weights are products of the e_k^2, and one reciprocal
// takes the place of seven IEEE divisions.  Those products leave the range
// of a double for e beyond 1e50: there the e_k are first divided by the
// smallest, and one that is still beyond 1e50 weighs less than 1e-100.
__device__ __forceinline__ double weno_godunov(double a, double b, double c, double d) {
  const double eps = 1e-8;
  const double t0 = a - b, t1 = a - 3.0 * b, t2 = b - c, t3 = b + c, t4 = c - d, t5 = 3.0 * c - d;
  double e0 = eps + (13.0 * (t0 * t0) + 3.0 * (t1 * t1));
  double e1 = eps + (13.0 * (t2 * t2) + 3.0 * (t3 * t3));
  double e2 = eps + (13.0 * (t4 * t4) + 3.0 * (t5 * t5));
  if (fmax(e0, fmax(e1, e2)) > 1e50) {
    const double lo = fmin(e0, fmin(e1, e2));
    e0 = fmin(e0 / lo, 1e50);
    e1 = fmin(e1 / lo, 1e50);
    e2 = fmin(e2 / lo, 1e50);
  }
  e0 *= e0;
  e1 *= e1;
  e2 *= e2;
  const double p = e1 * e2, q = 6.0 * (e0 * e2), r = 3.0 * (e0 * e1);
  const double v = weno_rcp(12.0 * (p + q + r));
  return 4.0 * p * v * (a - 2.0 * b + c) + (r - p - q) * v * (b - 2.0 * c + d);
}

struct GodunovH {
  double h12[3], h[3];  // 1 / (12 h) and 1 / h
};
static GodunovH godunov_h(const Grid &g) {
  GodunovH r;
  for (int a = 0; a < 3; ++a) {
    r.h12[a] = 1.0 / (12.0 * g.h[a]);
    r.h[a] = 1.0 / g.h[a];
  }
  return r;
}

// one axis' share of the squared Godunov gradient at phi[0] (stride st; cell
// size h: rh12 = 1 / (12 h), rh = 1 / h): the upwind one-sided slope, squared
__device__ __forceinline__ double godunov_axis(const double *__restrict__ phi, long st, double rh12, double rh,
                                               bool inside) {
#pragma clang fp contract(off)
#define P(k) phi[(k) * st]
  const double v =
      rh12 * (-(P(-1) - P(-2)) + 7.0 * (P(0) - P(-1)) + 7.0 * (P(1) - P(0)) - (P(2) - P(1)));
  const double up = v + rh *
                            weno_godunov(P(3) - 2.0 * P(2) + P(1), P(2) - 2.0 * P(1) + P(0),
                                         P(1) - 2.0 * P(0) + P(-1), P(0) - 2.0 * P(-1) + P(-2));
  const double um = v - rh *
                            weno_godunov(P(-3) - 2.0 * P(-2) + P(-1), P(-2) - 2.0 * P(-1) + P(0),
                                         P(-1) - 2.0 * P(0) + P(1), P(0) - 2.0 * P(1) + P(2));
#undef P
  double m;
  if (inside) m = fmax(-fmin(up, 0.0), fmax(um, 0.0));
  else m = fmax(fmax(up, 0.0), -fmin(um, 0.0));
  return m * m;
}

// godunov_gradient (godunov_gradient.cpp:7-152) on every padded cell (0 on
// the ghosts)
template <int DIM>
__global__ void __launch_bounds__(kLsBlock)
    k_godunov(Grid g, GodunovH r, const double *__restrict__ phi, const double *__restrict__ sign,
              double *__restrict__ grad) {
#pragma clang fp contract(off)
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= g.total) return;
  int q[3];
  padded_ijk(g, c, q);
  bool in = true;
#pragma unroll
  for (int a = 0; a < DIM; ++a) in = in && q[a] >= g.off[a] && q[a] < g.off[a] + g.n[a];
  double gsum = 0.0;
  if (in) {
#pragma unroll
    for (int a = 0; a < DIM; ++a) {
      const double m2 = godunov_axis(phi + c, g.s[a], r.h12[a], r.h[a], sign[c] > 0.0);
      gsum = a == 0 ? m2 : gsum + m2;
    }
  }
  grad[c] = sqrt(gsum);
}

// lsf_redistance_lambda (source.cpp:148-240), the RK3 stage update and the
// ghosts of any boundary condition but Dirichlet (`ghosts`) in place, 1-D and
// 3-D; a and b at the diagonal neighbours are read at clamped positions
// (zero_order_extrapolation, simple_bc.cpp:7-43).  Ghosts outside on one axis
// are their boundary condition's; those outside on more are advanced like
// cells of zero gradient.
template <int DIM, int STAGE>
__global__ void __launch_bounds__(kLsBlock)
    k_redist_stage(Grid g, double *__restrict__ phi, const double *__restrict__ sign,
                   const double *__restrict__ delta, const double *__restrict__ grad, double *__restrict__ s1,
                   double *__restrict__ s2, double dt, double rdt, BcSpec bc, int ghosts) {
#pragma clang fp contract(off)
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= g.total) return;
  int q[3];
  padded_ijk(g, c, q);
  int out = 0;
#pragma unroll
  for (int a = 0; a < DIM; ++a) out += q[a] < g.off[a] || q[a] >= g.off[a] + g.n[a];
  if (out == 1) return;
  double s = -sign[c] * (grad[c] - 1.0) * rdt / dt;
  if (out == 0 && DIM == 3) {
    auto AB = [&](int di, int dj, int dk, double &A, double &B) {
      int r[3] = {q[0] + di, q[1] + dj, q[2] + dk};
      const long p = ext_index<DIM>(g, r, -1);
      A = sign[p] * delta[p] * (grad[p] - 1.0);
      B = grad[p] * delta[p] * delta[p];
    };
    double A, B;
    AB(0, 0, 0, A, B);
    double a = 51.0 * A, b = 51.0 * B;
    for (int ii = -1; ii < 2; ii += 2)
      for (int jj = -1; jj < 2; jj += 2)
        for (int kk = -1; kk < 2; kk += 2) {
          AB(ii, jj, kk, A, B);
          a += A;
          b += B;
        }
    if (fabs(b) > 1e-8) s += a / b * delta[c] * grad[c] * rdt / dt;
  }
  const double y = rk3_update<STAGE>(phi[c], s, c, s1, s2, dt);
  phi[c] = y;
  if (out == 0 && ghosts) {
#pragma unroll
    for (int a = 0; a < DIM; ++a) ghosts_of(bc, a, g.n[a], g.h[a], g.s[a], q[a] - g.off[a], y, phi + c);
  }
}

// k_godunov and k_redist_stage in one launch for 2-D, from `in` to `outp`.
// A thread forms the gradient of one position of a 16 x 32 tile, clamped to
// the interior; a and b stay in LDS for the diagonal neighbours, and the
// inner 14 x 30 positions are advanced.  The rim's gradients are formed twice
// (512 for 420 cells), which costs less than the gradient's way through
// memory and a launch.  What bounds it: FP64 issue, some 480 instructions a
// position (the VALU is active in 72 % of the cycles in which a SIMD has work,
// at 1024 x 512), and on small grids the chain of one wavefront.
// Measured: a step's three stages at 501 x 333 65 us in twelve launches
// before, 24 here; 64 x 128 16 us, 1024^2 74, 3000 x 2000 368.  Tiles of 8 x
// 32 / 8 x 64 / 16 x 16: 25 / 24 / 26, 15 / 17 / 15, 79 / 78 / 77, 390 / 401
// / 378 us.
constexpr int kRdRows = 16, kRdCols = 32;
template <int STAGE>
__global__ void __launch_bounds__(kRdRows *kRdCols)
    k_redist2d(Grid g, GodunovH r, const double *__restrict__ in, double *__restrict__ outp, const double *__restrict__ sign,
               const double *__restrict__ delta, double *__restrict__ s1, double *__restrict__ s2, double dt,
               double rdt, BcSpec bc, int ghosts, int tiles_c) {
#pragma clang fp contract(off)
  __shared__ double As[kRdRows][kRdCols], Bs[kRdRows][kRdCols];
  const int ty = (int)threadIdx.x / kRdCols, tx = (int)threadIdx.x % kRdCols;
  const int tr = (int)blockIdx.x / tiles_c, tc = (int)blockIdx.x - tr * tiles_c;
  const int i = tr * (kRdRows - 2) + ty - 1, j = tc * (kRdCols - 2) + tx - 1;  // padded
  const int ci = clampi(i, g.off[0], g.off[0] + g.n[0] - 1), cj = clampi(j, g.off[1], g.off[1] + g.n[1] - 1);
  const long c = (long)ci * g.s[0] + (long)cj * g.s[1];
  const double sg = sign[c], dl = delta[c], x = in[c];
  double gr = godunov_axis(in + c, g.s[0], r.h12[0], r.h[0], sg > 0.0);
  gr = sqrt(gr + godunov_axis(in + c, g.s[1], r.h12[1], r.h[1], sg > 0.0));
  const double A = sg * dl * (gr - 1.0), B = gr * dl * dl;
  As[ty][tx] = A;
  Bs[ty][tx] = B;
  __syncthreads();
  const bool own = ty > 0 && ty < kRdRows - 1 && tx > 0 && tx < kRdCols - 1 && i < g.N[0] && j < g.N[1];
  if (!own || (i != ci) != (j != cj)) return;
  if (i != ci) {  // a corner's ghost: gradient 0
    const long p = (long)i * g.s[0] + (long)j * g.s[1];
    outp[p] = rk3_update<STAGE>(in[p], -sign[p] * (0.0 - 1.0) * rdt / dt, p, s1, s2, dt);
    return;
  }
  double s = -sg * (gr - 1.0) * rdt / dt;
  double a = 16.0 * A, b = 16.0 * B;
#pragma unroll
  for (int ii = -1; ii < 2; ii += 2)
#pragma unroll
    for (int jj = -1; jj < 2; jj += 2) {
      a += As[ty + ii][tx + jj];
      b += Bs[ty + ii][tx + jj];
    }
  if (fabs(b) > 1e-8) s += a / b * dl * gr * rdt / dt;
  const double y = rk3_update<STAGE>(x, s, c, s1, s2, dt);
  outp[c] = y;
  if (ghosts) {
    ghosts_of(bc, 0, g.n[0], g.h[0], g.s[0], i - g.off[0], y, outp + c);
    ghosts_of(bc, 1, g.n[1], g.h[1], g.s[1], j - g.off[1], y, outp + c);
  }
}

// Coefficients of the compact schemes' line systems, factorised.  Along a
// grid line of n cells CCD (kind 0; ccd_base.cpp:43-104) and UCCD (kind 1
// upwind, 2 downwind; uccd_base.cpp:16-117) solve a block-tridiagonal
// system for y_i = (f'_i, f''_i):
//   L_i y_{i-1} + D_i y_i + U_i y_{i+1} = rhs_i,
// every block 2 x 2, [[a, b], [aa, bb]]: the f' equation's coefficients of
// f' and f'' in the first row, the f'' equation's in the second.  Interior
// rows hold the schemes' stencils; rows 0 and n-1 their one-sided
// closures.  The factorisation is block LU without pivoting (the
// elimination of twin_dec, matrix_solver.cpp:21-56): for i = 1 .. n-1 the
// multiplier M_i = L_i D'_{i-1}^{-1} replaces L_i and D'_i = D_i - M_i
// U_{i-1}; the 2 x 2 inverse is the adjugate over the determinant.  The
// back substitution (k_twin_line) reads L_0 and U_{n-1} as [[0, 1], [0, 1]].
// Every product, sum and quotient is formed in the order the reference's
// elimination forms it, so the coefficients are bit-identical to its.
// Layout: 12 arrays of n, entry e (a, b, aa, bb) of band k (L, D, U) at
// [(3 e + k) n, (3 e + k + 1) n).
namespace {
struct Blk2 {
  double a, b, aa, bb;
};
struct BandRow {
  Blk2 L, D, U;
};

BandRow compact_interior_row(int kind, double h) {
  // the f'' equation is shared: -9/(8h) (f_{i+1} - f_{i-1}) stencil side
  const Blk2 none{0.0, 0.0, 0.0, 0.0};
  BandRow r{none, none, none};
  r.L.aa = -9.0 / 8.0 / h;
  r.D.aa = 0.0;
  r.U.aa = 9.0 / 8.0 / h;
  r.L.bb = -1.0 / 8.0;
  r.D.bb = 1.0;
  r.U.bb = -1.0 / 8.0;
  // the f' equation: centred (CCD) or upwind-biased (UCCD) weights
  const double w1 = 0.875, v1 = 0.1251282341599089, v2 = -0.2487176584009104, v3 = 0.0001282341599089;
  r.D.a = 1.0;
  if (kind == 0) {
    r.L.a = 7.0 / 16.0;
    r.U.a = 7.0 / 16.0;
    r.L.b = h / 16.0;
    r.D.b = 0.0;
    r.U.b = -h / 16.0;
  } else if (kind == 1) {
    r.L.a = w1;
    r.U.a = 0.0;
    r.L.b = v1 * h;
    r.D.b = v2 * h;
    r.U.b = v3 * h;
  } else {
    r.L.a = 0.0;
    r.U.a = w1;
    r.L.b = -v3 * h;
    r.D.b = -v2 * h;
    r.U.b = -v1 * h;
  }
  return r;
}
}  // namespace

static std::vector<double> compact_coefficients(int kind, int n, double h) {
#pragma clang fp contract(off)
  std::vector<BandRow> row(n);
  for (int i = 0; i < n; ++i) row[i] = compact_interior_row(kind, h);
  // one-sided closures of the first and last cells (shared by all kinds)
  const double c1 = 2.0, d1 = -1.0, c2 = 5.0, d2 = -6.0;
  const Blk2 unused{0.0, 1.0, 0.0, 1.0};  // what the back substitution reads outside the band
  row[0].L = unused;
  row[0].D = Blk2{1.0, 0.0, 0.0, 1.0};
  row[0].U = Blk2{c1, d1 * h, d2 / h, c2};
  row[n - 1].L = Blk2{c1, -d1 * h, -d2 / h, c2};
  row[n - 1].D = Blk2{1.0, 0.0, 0.0, 1.0};
  row[n - 1].U = unused;
  for (int i = 1; i < n; ++i) {
    const Blk2 P = row[i - 1].D, Q = row[i - 1].U, Lw = row[i].L;
    const double det = P.a * P.bb - P.aa * P.b;
    // M = Lw P^-1, P^-1 = [[bb, -b], [-aa, a]] / det
    const Blk2 M{(Lw.a * P.bb - P.aa * Lw.b) / det, (Lw.b * P.a - P.b * Lw.a) / det,
                 (Lw.aa * P.bb - P.aa * Lw.bb) / det, (Lw.bb * P.a - P.b * Lw.aa) / det};
    Blk2 &D = row[i].D;
    D.a = D.a - (M.a * Q.a + M.b * Q.aa);
    D.b = D.b - (M.a * Q.b + M.b * Q.bb);
    D.aa = D.aa - (M.aa * Q.a + M.bb * Q.aa);
    D.bb = D.bb - (M.aa * Q.b + M.bb * Q.bb);
    row[i].L = M;
  }
  std::vector<double> c(12 * (size_t)n);
  for (int i = 0; i < n; ++i) {
    const Blk2 *band[3] = {&row[i].L, &row[i].D, &row[i].U};
    for (int k = 0; k < 3; ++k) {
      c[(0 + k) * (size_t)n + i] = band[k]->a;
      c[(3 + k) * (size_t)n + i] = band[k]->b;
      c[(6 + k) * (size_t)n + i] = band[k]->aa;
      c[(9 + k) * (size_t)n + i] = band[k]->bb;
    }
  }
  return c;
}

// Segment propagators of the partitioned twin sweeps (k_twin_part) for the
// factorised coefficients cf (12 n) of one line system cut into segments of
// Lp positions (the last one shorter): phi[4 k..] = product over segment
// k of -M_i (first position innermost; segment 0 starts at 1),
// psi[4 k..] = product over segment k of -D_i^-1 N_i from its top position
// down (the top segment ends at n - 2), both 2x2 row-major.
static void twin_propagators(const std::vector<double> &cf, int n, int Lp, double *phi, double *psi) {
  const double *a0 = &cf[0], *a1 = &cf[n], *a2 = &cf[2 * n], *b0 = &cf[3 * n], *b1 = &cf[4 * n], *b2 = &cf[5 * n];
  const double *aa0 = &cf[6 * n], *aa1 = &cf[7 * n], *aa2 = &cf[8 * n], *bb0 = &cf[9 * n], *bb1 = &cf[10 * n],
               *bb2 = &cf[11 * n];
  const int ns = (n + Lp - 1) / Lp;
  auto mul = [](const double (&x)[4], const double (&y)[4], double (&z)[4]) {
    z[0] = x[0] * y[0] + x[1] * y[2];
    z[1] = x[0] * y[1] + x[1] * y[3];
    z[2] = x[2] * y[0] + x[3] * y[2];
    z[3] = x[2] * y[1] + x[3] * y[3];
  };
  for (int k = 0; k < ns; ++k) {
    const int lo = k * Lp, hi = std::min(lo + Lp, n);
    double F[4] = {1, 0, 0, 1}, T[4];
    for (int i = std::max(lo, 1); i < hi; ++i) {
      const double m[4] = {-a0[i], -b0[i], -aa0[i], -bb0[i]};
      mul(m, F, T);
      std::copy(T, T + 4, F);
    }
    std::copy(F, F + 4, phi + 4 * k);
    double G[4] = {1, 0, 0, 1};
    for (int i = std::min(hi, n - 1) - 1; i >= lo; --i) {
      const double den = a1[i] * bb1[i] - aa1[i] * b1[i];
      const double di[4] = {bb1[i] / den, -b1[i] / den, -aa1[i] / den, a1[i] / den};
      const double nm[4] = {a2[i], b2[i], aa2[i], bb2[i]};
      double P[4];
      mul(di, nm, P);
      for (double &x : P) x = -x;
      mul(P, G, T);
      std::copy(T, T + 4, G);
    }
    std::copy(G, G + 4, psi + 4 * k);
  }
}

}  // namespace scihpc

using namespace scihpc;

struct scihpc_ls {
  Grid g{};
  BcSpec bc{};
  double *phi[2] = {nullptr, nullptr};  // ping-pong stage buffers
  int cur = 0;
  double *u = nullptr, *v = nullptr, *w = nullptr;
  double *fx = nullptr, *fy = nullptr, *fz = nullptr;
  double *s1 = nullptr, *s2 = nullptr, *tmp = nullptr;
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;

  double *alloc() {
    void *p = nullptr;
    SCIHPC_HIP(hipMalloc(&p, sizeof(double) * g.total));
    SCIHPC_HIP(hipMemsetAsync(p, 0, sizeof(double) * g.total, stream));
    return static_cast<double *>(p);
  }

  unsigned grid_interior() const { return ceil_div(g.interior, kLsBlock); }

  void apply_bc(double *f, int stag) {
    for (int a = 0; a < g.ndim; ++a) {
      const int t1 = (a + 1) % 3, t2 = (a + 2) % 3;
      const long lines = (long)g.n[t1] * g.n[t2];
      k_bc_axis<<<ceil_div(lines, kLsBlock), kLsBlock, 0, stream>>>(g, f, bc, a, stag);
      SCIHPC_CHECK_LAUNCH();
    }
  }

  // interface maintenance state (allocated on first use): line-system
  // coefficients per axis (CCD; UCCD upwind and downwind), line scratch,
  // derivatives, sign, delta, gradient, reduction partials
  int scheme = 0;  // tvd_rk3 convection: 0 WENO5, 1 UCCD
  double *coef_ccd[3] = {nullptr, nullptr, nullptr}, *coef_up[3] = {nullptr, nullptr, nullptr};
  double *coef_dn[3] = {nullptr, nullptr, nullptr};
  double *ls_scr[3][4] = {};  // line scratch per axis: su, ssu, sd, ssd
  double *fxx = nullptr, *fyy = nullptr, *fzz = nullptr;
  double *sgn = nullptr, *dlt = nullptr, *grd = nullptr, *flux = nullptr;
  double *lpart = nullptr, *lhost = nullptr;
  // partitioned twin sweeps (chosen by scihpc_ls_set_line_solver): lines
  // per workgroup (16 or 8; 0 = lines too long to partition in registers,
  // which always sweep sequentially), the segment propagators
  // ([axis][CCD, UCCD up, UCCD down][Phi, Psi][segment] 2x2)
  int twin_lines = 0, twin_len = 0;
  double *carry = nullptr;
  bool twin_partitioned = false;
  // segmented sequential sweeps (k_twin_seg): coefficient rows [axis][CCD,
  // UCCD up, UCCD down], and the rows' repetition along a line; seg_ok when
  // every axis has one
  double *seg_rows[3][3] = {};
  int seg_start[3][3] = {}, seg_period[3][3] = {}, seg_count[3][3] = {};
  bool seg_ok = false;
  unsigned *seg_state = nullptr;  // TwinPlan::state
  unsigned seg_call = 0;          // segmented calls so far (never 0 in one)
  long long seg_groups = 0;       // their workgroups
  int lds_max = 65536;      // LDS bytes a workgroup may hold on this device
  int num_cu = 256;         // compute units

  void ensure_iface() {
    if (sgn) return;
    for (int a = 0; a < g.ndim; ++a) {
      const int n = g.N[a];
      const std::vector<double> cc = compact_coefficients(0, n, g.h[a]);
      const std::vector<double> cu = compact_coefficients(1, n, g.h[a]);
      const std::vector<double> cd = compact_coefficients(2, n, g.h[a]);
      seg_ok = (a == 0 || seg_ok) && seg_table(a, 0, cc) && seg_table(a, 1, cu) && seg_table(a, 2, cd);
      for (double **dst : {&coef_ccd[a], &coef_up[a], &coef_dn[a]})
        SCIHPC_HIP(hipMalloc(reinterpret_cast<void **>(dst), sizeof(double) * 12 * n));
      SCIHPC_HIP(hipMemcpyAsync(coef_ccd[a], cc.data(), sizeof(double) * 12 * n, hipMemcpyHostToDevice, stream));
      SCIHPC_HIP(hipMemcpyAsync(coef_up[a], cu.data(), sizeof(double) * 12 * n, hipMemcpyHostToDevice, stream));
      SCIHPC_HIP(hipMemcpyAsync(coef_dn[a], cd.data(), sizeof(double) * 12 * n, hipMemcpyHostToDevice, stream));
      SCIHPC_HIP(hipStreamSynchronize(stream));  // the host vectors go out of scope
    }
    SCIHPC_HIP(hipMalloc(reinterpret_cast<void **>(&seg_state), sizeof(unsigned) * 2));
    SCIHPC_HIP(hipMemsetAsync(seg_state, 0, sizeof(unsigned) * 2, stream));
    int nmax = 0;
    for (int a = 0; a < g.ndim; ++a) nmax = std::max(nmax, g.N[a]);
    // 16 lines x 64 segments or 8 x 128, segments of 9 (or 17) positions
    twin_lines = nmax <= 64 * 9 ? 16 : (nmax <= 128 * 17 ? 8 : 0);
    twin_len = nmax <= 128 * 9 ? 9 : 17;
    if (twin_lines) {
      const int segs = 1024 / twin_lines;
      SCIHPC_HIP(hipMalloc(reinterpret_cast<void **>(&carry), sizeof(double) * 3 * 3 * 2 * 4 * segs));
      std::vector<double> all((size_t)3 * 3 * 2 * 4 * segs, 0.0);
      for (int a = 0; a < g.ndim; ++a)
        for (int kind = 0; kind < 3; ++kind) {
          const std::vector<double> cf = compact_coefficients(kind, g.N[a], g.h[a]);
          double *phi = &all[(size_t)((a * 3 + kind) * 2 + 0) * 4 * segs];
          double *psi = &all[(size_t)((a * 3 + kind) * 2 + 1) * 4 * segs];
          twin_propagators(cf, g.N[a], twin_len, phi, psi);
        }
      SCIHPC_HIP(hipMemcpyAsync(carry, all.data(), sizeof(double) * all.size(), hipMemcpyHostToDevice, stream));
      SCIHPC_HIP(hipStreamSynchronize(stream));
    }
    for (int a = 0; a < g.ndim; ++a)
      for (auto &q : ls_scr[a]) q = alloc();
    fxx = alloc();
    fyy = alloc();
    fzz = alloc();
    sgn = alloc();
    dlt = alloc();
    grd = alloc();
    flux = alloc();
    const long nb = (long)ceil_div(g.interior, kLsBlock);
    SCIHPC_HIP(hipMalloc(reinterpret_cast<void **>(&lpart), sizeof(double) * (2 * nb + 1)));
    SCIHPC_HIP(hipHostMalloc(reinterpret_cast<void **>(&lhost), sizeof(double) * 2 * nb, hipHostMallocDefault));
  }

  // k_twin_seg's table of one line system: the rows of the factorised
  // coefficients cf (12 n) up to where they repeat, one period, and the last
  // row; false when they do not repeat soon enough
  bool seg_table(int a, int kind, const std::vector<double> &cf) {
#pragma clang fp contract(off)
    const int n = g.N[a];
    auto same = [&](int i, int j) {
      for (int e = 0; e < 12; ++e)
        if (std::memcmp(&cf[(size_t)e * n + i], &cf[(size_t)e * n + j], sizeof(double)) != 0) return false;
      return true;
    };
    // rows 0 .. n - 2 repeat with `period` from `start` on (short lines: all rows are kept)
    int start = n - 1, period = 1;
    if (n > kTwinRowsMax) {
      bool found = false;
      for (int p = 1; p <= 6 && !found; ++p) {  // divisors of k_twin_seg's block of six steps
        if (6 % p != 0) continue;
        int i = n - 2 - p;
        while (i >= 0 && same(i, i + p)) --i;
        if (i + 1 + p + 1 <= kTwinRowsMax) {
          start = i + 1;
          period = p;
          found = true;
        }
      }
      if (!found) return false;
    }
    const int rows = std::min(n - 1, start + (n - 1 > start ? period : 0)) + 1;
    std::vector<double> t((size_t)kTwinRow * rows);
    for (int r = 0; r < rows; ++r) {
      const int i = r == rows - 1 ? n - 1 : r;
      auto c = [&](int e, int band) { return cf[(size_t)(3 * e + band) * n + i]; };
      double *o = &t[(size_t)kTwinRow * r];
      for (int e = 0; e < 4; ++e) {
        o[e] = c(e, 0);
        o[4 + e] = c(e, 2);
        o[8 + e] = c(e, 1);
      }
      o[12] = o[8] * o[11] - o[10] * o[9];
      o[13] = 1.0 / o[12];
    }
    SCIHPC_HIP(hipMalloc(reinterpret_cast<void **>(&seg_rows[a][kind]), sizeof(double) * t.size()));
    SCIHPC_HIP(hipMemcpyAsync(seg_rows[a][kind], t.data(), sizeof(double) * t.size(), hipMemcpyHostToDevice, stream));
    SCIHPC_HIP(hipStreamSynchronize(stream));
    seg_start[a][kind] = start;
    seg_period[a][kind] = period;
    seg_count[a][kind] = rows;
    return true;
  }

  // the segmented sweeps, in the way that pays for these sizes
  enum SegWay { kSegNoRoom, kSegDone, kSegPassOn, kSegThreePasses };
  template <int LINES, bool UP>
  SegWay twin_seg(const double *f, double *d1[3], double *d2[3]) {
    constexpr int NS = UP ? 2 : 1;
    int nmax = 0;
    for (int a = 0; a < g.ndim; ++a) nmax = std::max(nmax, g.N[a]);
    TwinPlan pl{};
    pl.cap = (nmax * LINES + 1) / 2 * 2;
    const size_t lds = sizeof(double) * ((UP ? 4 : 3) * (size_t)pl.cap + NS * kTwinRow * kTwinRowsMax);
    if (lds + 1024 > (size_t)lds_max) return kSegNoRoom;
    // about 33 positions a segment on the longest lines
    pl.waves = std::max(1, std::min(4, (int)std::lround(nmax * LINES / (64.0 * 33.0))));
    TwinTable tb{};
    long total = 0;
    for (int a = 0; a < g.ndim; ++a) {
      const int n = g.N[a], most = 64 * pl.waves / LINES;
      pl.len[a] = std::max((n + most - 1) / most, std::min(n, 25)) | 1;
      pl.segs[a] = (n + pl.len[a] - 1) / pl.len[a];
      pl.blocks[a] = (int)ceil_div((long)g.N[(a + 1) % 3] * g.N[(a + 2) % 3], LINES);
      total += pl.blocks[a];
      for (int y = 0; y < NS; ++y) {
        const int kind = UP ? 1 + y : 0;
        tb.row[a][y] = seg_rows[a][kind];
        tb.start[a][y] = seg_start[a][kind];
        tb.period[a][y] = seg_period[a][kind];
        tb.rows[a][y] = seg_count[a][kind];
      }
    }
    if (total > 0x7fffffffL) return kSegThreePasses;
    // Segments, or the three passes?  In units of 91 ns a workgroup that has
    // to sweep its n positions end to end takes 440 + n, the three passes 80 +
    // 4.1 n of the longest line (latency; many cells take longer).  The line
    // lies where fields of two values, whose workgroups all fail, take as long
    // as with the three passes, or where all workgroups run at once.
    // us a UCCD step, segments (ordinary field / two values) against three
    // passes: 100^2 132 / 169 : 171, 512^2 305 / 579 : 689, 1024^2 489 / 1329 :
    // 1377, 1400 x 374 551 / 1259 : 1553, 24^3 79 / 79 : 90; 48^3 251 / 251 :
    // 172, 96 x 70 x 76 639 / 805 : 321, 900 x 64 x 64 10126 / 11323 : 3511.
    // Beyond it segments are still tried where ordinary fields gain, but a
    // failure leaves the call to the three passes: 1400 x 1000 842 / 1855 :
    // 1681, 2048^2 1575 / 3379 : 3159 (end to end 6668).
    double work = 0.0;
    for (int a = 0; a < g.ndim; ++a) work += double(pl.blocks[a]) * (440 + g.N[a]);
    // workgroups that run side by side: whole lines in LDS, 192 registers a thread
    const double slots = (double)num_cu * std::max(1, std::min((int)(lds_max / (lds + 1024)), 8 / (NS * pl.waves)));
    SegWay way = kSegDone;
    if (total > slots && work / slots > 3.6 * nmax) way = total / slots <= nmax / 220.0 ? kSegPassOn : kSegThreePasses;
    if (way == kSegThreePasses) return way;
    pl.state = seg_state;
    pl.call = ++seg_call;
    pl.pass_on = way == kSegPassOn;
    seg_groups += total;
    // the allowance is the function's, not the handle's: always the same, the most any handle needs
    if (lds > 65536)
      SCIHPC_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_twin_seg<LINES, UP>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, lds_max - 1024));
    double *none[3] = {nullptr, nullptr, nullptr};
    double **dd = d2 ? d2 : none;
    k_twin_seg<LINES, UP><<<(unsigned)total, 64 * NS * pl.waves, lds, stream>>>(g, f, u, v, w, tb, pl, d1[0], d1[1],
                                                                                d1[2], dd[0], dd[1], dd[2]);
    SCIHPC_CHECK_LAUNCH();
    return way;
  }

  // derivatives of f along every real axis: UCCD by (u, v, w) or CCD
  void compact(const double *f, bool upwind, double *d1[3], double *d2[3]) {
    LineGate gate{};
    if (seg_ok && !(twin_lines && twin_partitioned)) {
      SegWay way = upwind ? twin_seg<4, true>(f, d1, d2) : twin_seg<4, false>(f, d1, d2);
      if (way == kSegNoRoom) way = upwind ? twin_seg<2, true>(f, d1, d2) : twin_seg<2, false>(f, d1, d2);
      if (way == kSegNoRoom) way = upwind ? twin_seg<1, true>(f, d1, d2) : twin_seg<1, false>(f, d1, d2);
      if (way == kSegDone) return;
      if (way == kSegPassOn) gate = LineGate{seg_state, seg_call};
    }
    LineScratch sc{};
    LineCoefs co{};
    long work = 0;
    const int nsys = upwind ? 2 : 1;
    for (int a = 0; a < g.ndim; ++a) {
      sc.su[a] = ls_scr[a][0];
      sc.ssu[a] = ls_scr[a][1];
      sc.sd[a] = ls_scr[a][2];
      sc.ssd[a] = ls_scr[a][3];
      co.cu[a] = upwind ? coef_up[a] : coef_ccd[a];
      co.cd[a] = coef_dn[a];
      work += (long)g.N[(a + 1) % 3] * g.N[(a + 2) % 3] * nsys;
    }
    const unsigned nbc = ceil_div(g.total, kLsBlock);
    if (upwind) k_compact_rhs<true><<<nbc, kLsBlock, 0, stream>>>(g, f, sc, gate);
    else k_compact_rhs<false><<<nbc, kLsBlock, 0, stream>>>(g, f, sc, gate);
    SCIHPC_CHECK_LAUNCH();
    if (twin_lines && twin_partitioned) {
      const int segs = 1024 / twin_lines;
      LineCarry cr{};
      long blocks = 0;
      for (int a = 0; a < g.ndim; ++a) {
        for (int sy = 0; sy < 2; ++sy) {
          const int kind = upwind ? 1 + sy : 0;
          cr.phi[a][sy] = carry + (size_t)((a * 3 + kind) * 2 + 0) * 4 * segs;
          cr.psi[a][sy] = carry + (size_t)((a * 3 + kind) * 2 + 1) * 4 * segs;
        }
        blocks += (long)ceil_div((long)g.N[(a + 1) % 3] * g.N[(a + 2) % 3], twin_lines) * nsys;
      }
      int nmax = 0;
      for (int a = 0; a < g.ndim; ++a) nmax = std::max(nmax, g.N[a]);
      const size_t lds = sizeof(double) * 12 * (size_t)nmax;  // + at most 24 KiB static
      if (twin_len == 9 && lds + 24576 <= (size_t)lds_max) {
        SCIHPC_HIP(hipFuncSetAttribute(twin_lines == 16 ? reinterpret_cast<const void *>(&k_twin_part<16, 9, true>)
                                                        : reinterpret_cast<const void *>(&k_twin_part<8, 9, true>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, lds_max - 24576));
        if (twin_lines == 16) k_twin_part<16, 9, true><<<(unsigned)blocks, 1024, lds, stream>>>(g, nsys, co, sc, cr);
        else k_twin_part<8, 9, true><<<(unsigned)blocks, 1024, lds, stream>>>(g, nsys, co, sc, cr);
      } else if (twin_lines == 16) {
        k_twin_part<16, 9, false><<<(unsigned)blocks, 1024, 0, stream>>>(g, nsys, co, sc, cr);
      } else if (twin_len == 9) {
        k_twin_part<8, 9, false><<<(unsigned)blocks, 1024, 0, stream>>>(g, nsys, co, sc, cr);
      } else {
        k_twin_part<8, 17, false><<<(unsigned)blocks, 1024, 0, stream>>>(g, nsys, co, sc, cr);
      }
    } else {
      if (gate.flag) k_twin_line<true><<<ceil_div(work, 64), 64, 0, stream>>>(g, nsys, co, sc, gate);
      else k_twin_line<false><<<ceil_div(work, 64), 64, 0, stream>>>(g, nsys, co, sc, gate);
    }
    SCIHPC_CHECK_LAUNCH();
    double *e2[3] = {nullptr, nullptr, nullptr};
    double **dd = d2 ? d2 : e2;
    if (upwind)
      k_compact_select<true><<<nbc, kLsBlock, 0, stream>>>(g.total, g.ndim, u, v, w, sc, d1[0], d1[1], d1[2], dd[0],
                                                           dd[1], dd[2], gate);
    else
      k_compact_select<false><<<nbc, kLsBlock, 0, stream>>>(g.total, g.ndim, nullptr, nullptr, nullptr, sc, d1[0],
                                                            d1[1], d1[2], dd[0], dd[1], dd[2], gate);
    SCIHPC_CHECK_LAUNCH();
  }

  // boundary conditions of phi that change boundary cells, which other
  // axes read: they can't be filled by the cells they copy
  bool dirichlet() const {
    for (int q = 0; q < 2 * g.ndim; ++q)
      if (bc.type[q] == SCIHPC_BC_DIRICHLET) return true;
    return false;
  }

  // tvd_rk3 with the UCCD convection term, phi[cur] in place
  template <int DIM, int STAGE>
  void uccd_stage(double dt) {
    double *d1[3] = {fx, fy, fz};
    double *f = phi[cur];
    const bool d = dirichlet();
    compact(f, true, d1, nullptr);
    k_uccd_stage<DIM, STAGE><<<ceil_div(g.total, kLsBlock), kLsBlock, 0, stream>>>(g, f, u, v, w, fx, fy, fz, s1, s2,
                                                                                 dt, bc, !d);
    SCIHPC_CHECK_LAUNCH();
    if (d) apply_bc(f, -1);
  }

  template <int DIM>
  void uccd_step(double dt) {
    ensure_iface();
    uccd_stage<DIM, 1>(dt);
    uccd_stage<DIM, 2>(dt);
    uccd_stage<DIM, 3>(dt);
  }

  // lsf_mass and the mpls denominator of the current phi (needs fx, fy, fz
  // of its extrapolated CCD derivatives for the denominator)
  template <int DIM>
  void mpls_sums(double w_, double ratio, int positive_ref, double &mass, double &den) {
    const unsigned nb = ceil_div(g.interior, kLsBlock);
    const double dv = DIM == 2 ? g.h[0] * g.h[1] : g.h[0] * g.h[1] * g.h[2];
    k_mpls_sums<DIM><<<nb, kLsBlock, 0, stream>>>(g, phi[cur], fx, fy, fz, w_, ratio, positive_ref, dv, lpart);
    SCIHPC_CHECK_LAUNCH();
    SCIHPC_HIP(hipMemcpyAsync(lhost, lpart, sizeof(double) * 2 * nb, hipMemcpyDeviceToHost, stream));
    SCIHPC_HIP(hipStreamSynchronize(stream));
    double m = 0.0, e = 0.0;
    for (unsigned b = 0; b < nb; ++b) {
      m += lhost[2 * b];
      e += lhost[2 * b + 1];
    }
    mass = m * dv;
    den = e;
  }

  // runge_kutta::euler with mpls (source.cpp:109-146)
  template <int DIM>
  void mpls_step(double dt, double w_, double ratio, int positive_ref, double mass0) {
    ensure_iface();
    double *f = phi[cur];
    const unsigned nb = ceil_div(g.total, kLsBlock);
    k_extrap<DIM><<<nb, kLsBlock, 0, stream>>>(g, f, flux);
    SCIHPC_CHECK_LAUNCH();
    double *d1[3] = {fx, fy, fz};
    compact(flux, false, d1, nullptr);
    const unsigned nbi = ceil_div(g.interior, kLsBlock);
    const double dv = DIM == 2 ? g.h[0] * g.h[1] : g.h[0] * g.h[1] * g.h[2];
    k_mpls_sums<DIM><<<nbi, kLsBlock, 0, stream>>>(g, f, fx, fy, fz, w_, ratio, positive_ref, dv, lpart);
    SCIHPC_CHECK_LAUNCH();
    double *eta = lpart + 2 * (long)nbi;  // one slot past the block sums
    k_mpls_eta<<<1, kLsBlock, 0, stream>>>(lpart, (int)nbi, mass0, dv, dt, eta);
    SCIHPC_CHECK_LAUNCH();
    k_mpls_update<DIM><<<nb, kLsBlock, 0, stream>>>(g.total, f, fx, fy, fz, w_, eta, dt, dlt);
    SCIHPC_CHECK_LAUNCH();
    apply_bc(f, -1);
  }

  // one stage of redistancing with its boundary conditions
  template <int DIM, int STAGE>
  void redist_stage(const double *in, double *out, double dt, double rdt) {
    const bool d = dirichlet();
    if constexpr (DIM == 2) {
      const unsigned tc = ceil_div(g.N[1], kRdCols - 2), tr = ceil_div(g.N[0], kRdRows - 2);
      k_redist2d<STAGE><<<tc * tr, kRdRows * kRdCols, 0, stream>>>(g, godunov_h(g), in, out, sgn, dlt, s1, s2, dt, rdt, bc, !d,
                                                                   (int)tc);
    } else {
      const unsigned nb = ceil_div(g.total, kLsBlock);
      k_godunov<DIM><<<nb, kLsBlock, 0, stream>>>(g, godunov_h(g), out, sgn, grd);
      SCIHPC_CHECK_LAUNCH();
      k_redist_stage<DIM, STAGE><<<nb, kLsBlock, 0, stream>>>(g, out, sgn, dlt, grd, s1, s2, dt, rdt, bc, !d);
    }
    SCIHPC_CHECK_LAUNCH();
    if (d) apply_bc(out, -1);
  }

  // tvd_rk3 with lsf_redistance_lambda on the stored sign and delta; 2-D
  // stages go from buffer to buffer and end in phi[cur] again
  template <int DIM>
  void redistance_step(double dt, double rdt) {
    double *f = phi[cur], *a = DIM == 2 ? grd : f, *b = DIM == 2 ? flux : f;
    redist_stage<DIM, 1>(f, a, dt, rdt);
    redist_stage<DIM, 2>(a, b, dt, rdt);
    redist_stage<DIM, 3>(b, f, dt, rdt);
  }

  // k_rk3_fused's shape for this grid: rows a wavefront, tiles across the
  // last and the middle axis, cells a march
  struct RkPlan {
    int sub = 0, tc = 0, tr = 0, run = 0;
  } rk;
  template <int DIM>
  const RkPlan &rk_plan() {
    if (rk.sub) return rk;
    // Several short rows a wavefront where that takes under 0.8 of the
    // wavefronts (a last axis of few cells, or of few more than a multiple of
    // 63) and those are several for every SIMD: on smaller grids a launch's
    // latency counts, which it lengthens (32^3 18 -> 20 us a step).
    // Microseconds a step, one row / several / a thread a cell with the ghosts
    // apart: 600 x 16 x 16 90 / 39 / 82, with Dirichlet sides 136 / 87 /
    // 101; 256 x 16 x 64 72 / 54 / 92, Dirichlet 126 / 105 / 111; 80 x 70 x 90
    // 97 / 62 / 128, 128^3 (0.74) 236 / 211 / 351, 128 x 128 x 33 101 / 82 / 135.
    const int nc = g.n[DIM - 1];
    auto tiles_c = [&](int q) { return (int)ceil_div(nc, kWave / q - 1); };
    auto tiles_r = [&](int q) { return DIM == 3 ? (int)ceil_div(g.n[1], kRkRows * q - 1) : 1; };
    auto cost = [&](int q) { return (DIM == 3 ? 1.0 : 1.0 / q) * tiles_c(q) * tiles_r(q); };
    rk.sub = 1;
    for (int q = 2; q <= 8 && cost(1) * g.n[0] * (DIM == 3 ? kRkRows : 1) >= 16.0 * num_cu; ++q)
      if (cost(q) < 0.8 * cost(1) && cost(q) < cost(rk.sub)) rk.sub = q;
    rk.tc = tiles_c(rk.sub);
    rk.tr = tiles_r(rk.sub);
    // cells a march: a wavefront forms DIM faces a cell and one more, so
    // long marches form fewer, but the 1024 SIMDs want two or three
    // wavefronts each to hide their chains.  Microseconds a step measured with
    // 1 / 2 / 3 / 4 / 6 / 8 cells: 1024 x 512 42 / 39 / 36 / 39 / 40 / 48,
    // 333 x 501 21 / 22 / 22 / 24 / 29 / 35, 2048^2 264 / 188 / 163 / 157 /
    // 145 / 146, 128^3 (one row) 356 / 273 / 245 / 246 / 224 / 231.
    rk.run = 6;
    auto waves = [&](int q) {
      const long t = (long)rk.tc * rk.tr * ceil_div(g.n[0], q);
      return DIM == 3 ? t * kRkRows : t / rk.sub;
    };
    while (rk.run > 1 && waves(rk.run) < 4L * num_cu * (DIM == 3 ? 3 : 5) / 2) --rk.run;
    return rk;
  }

  // one WENO stage with its boundary conditions: in the stage's kernel but
  // for Dirichlet sides, which change boundary cells other axes read
  template <int DIM, int STAGE>
  void rk3_stage(const double *in, double *out, double dt) {
    if constexpr (DIM == 1) {
      k_rk3_stage<STAGE><<<grid_interior(), kLsBlock, 0, stream>>>(g, in, out, u, s1, s2, dt);
      SCIHPC_CHECK_LAUNCH();
      apply_bc(out, -1);
    } else {
      const bool dir = dirichlet();
      const RkPlan &pl = rk_plan<DIM>();
      const long tiles = (long)pl.tc * pl.tr * ceil_div(g.n[0], pl.run);
      const int per = DIM == 3 ? 1 : kLsBlock / kWave * pl.sub;
      const unsigned nb = ceil_div(tiles, per), nt = DIM == 3 ? kWave * kRkRows : kLsBlock;
      if (pl.sub > 1)
        k_rk3_fused<DIM, STAGE, true><<<nb, nt, 0, stream>>>(g, in, out, u, v, w, s1, s2, dt, bc, !dir, pl.tc, pl.tr,
                                                             pl.run, kWave / pl.sub);
      else
        k_rk3_fused<DIM, STAGE, false><<<nb, nt, 0, stream>>>(g, in, out, u, v, w, s1, s2, dt, bc, !dir, pl.tc, pl.tr,
                                                              pl.run, kWave);
      SCIHPC_CHECK_LAUNCH();
      if (dir) apply_bc(out, -1);
    }
  }

  template <int DIM>
  void rk3_step(double dt) {
    if (scheme == 1) {
      uccd_step<DIM>(dt);
      return;
    }
    double *a = phi[cur], *b = phi[cur ^ 1];
    rk3_stage<DIM, 1>(a, b, dt);
    rk3_stage<DIM, 2>(b, a, dt);
    rk3_stage<DIM, 3>(a, b, dt);
    cur ^= 1;
  }

  void step(double dt) {
    if (g.ndim == 1) rk3_step<1>(dt);
    else if (g.ndim == 2) rk3_step<2>(dt);
    else rk3_step<3>(dt);
  }
};

static void ls_check(const scihpc_ls *h) { SCIHPC_REQUIRE(h, "null handle"); }

extern "C" int scihpc_ls_create(int ndim, int nx, int ny, int nz, double dx, double dy, double dz,
                                const int *bc_types, const double *bc_values, scihpc_ls **out) {
  return guarded([&] {
    SCIHPC_REQUIRE(out, "out is null");
    *out = nullptr;
    SCIHPC_REQUIRE(ndim >= 1 && ndim <= 3, "ndim must be 1, 2 or 3");
    SCIHPC_REQUIRE(nx > 2 && (ndim < 2 || ny > 2) && (ndim < 3 || nz > 2), "each axis needs > 2 cells");
    SCIHPC_REQUIRE(dx > 0 && (ndim < 2 || dy > 0) && (ndim < 3 || dz > 0), "spacings must be positive");
    SCIHPC_REQUIRE(bc_types, "bc_types is null");
    auto *h = new scihpc_ls;
    try {
      h->g = make_grid(ndim, nx, ny, nz, dx, dy, dz);
      for (int q = 0; q < 6; ++q) {
        const int t = bc_types[q];
        SCIHPC_REQUIRE(q >= 2 * ndim || (t >= 0 && t <= 4), "unknown bc type");
        h->bc.type[q] = t;
        h->bc.value[q] = bc_values ? bc_values[q] : 0.0;
      }
      for (int a = 0; a < ndim; ++a)  // bc_factory::check_bc (bc_factory.cpp:16-19)
        SCIHPC_REQUIRE((h->bc.type[2 * a] == SCIHPC_BC_PERIODIC) == (h->bc.type[2 * a + 1] == SCIHPC_BC_PERIODIC),
                       "periodic must be set on both sides of an axis");
      SCIHPC_HIP(hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking));
      {
        int dev = 0, lds = 0;
        SCIHPC_HIP(hipGetDevice(&dev));
        if (hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) == hipSuccess && lds > 0)
          h->lds_max = lds;
        int cu = 0;
        if (hipDeviceGetAttribute(&cu, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && cu > 0)
          h->num_cu = cu;
      }
      SCIHPC_HIP(hipEventCreate(&h->ev0));
      SCIHPC_HIP(hipEventCreate(&h->ev1));
      h->phi[0] = h->alloc();
      h->phi[1] = h->alloc();
      h->u = h->alloc();
      h->v = h->alloc();
      h->w = h->alloc();
      h->fx = h->alloc();
      h->fy = h->alloc();
      h->fz = h->alloc();
      h->s1 = h->alloc();
      h->s2 = h->alloc();
      h->tmp = h->alloc();
      SCIHPC_HIP(hipStreamSynchronize(h->stream));
    } catch (...) {
      scihpc_ls_destroy(h);
      throw;
    }
    *out = h;
  });
}

extern "C" int scihpc_ls_destroy(scihpc_ls *h) {
  if (!h) return SCIHPC_OK;
  if (h->stream) (void)hipStreamSynchronize(h->stream);
  for (double *p : {h->phi[0], h->phi[1], h->u, h->v, h->w, h->fx, h->fy, h->fz, h->s1, h->s2, h->tmp, h->fxx,
                    h->fyy, h->fzz, h->sgn, h->dlt, h->grd, h->flux, h->lpart})
    if (p) (void)hipFree(p);
  for (int a = 0; a < 3; ++a)
    for (double *p : {h->coef_ccd[a], h->coef_up[a], h->coef_dn[a], h->seg_rows[a][0], h->seg_rows[a][1],
                      h->seg_rows[a][2]})
      if (p) (void)hipFree(p);
  if (h->carry) (void)hipFree(h->carry);
  if (h->seg_state) (void)hipFree(h->seg_state);
  for (auto &axis : h->ls_scr)
    for (double *p : axis)
      if (p) (void)hipFree(p);
  if (h->lhost) (void)hipHostFree(h->lhost);
  if (h->ev0) (void)hipEventDestroy(h->ev0);
  if (h->ev1) (void)hipEventDestroy(h->ev1);
  if (h->stream) (void)hipStreamDestroy(h->stream);
  delete h;
  return SCIHPC_OK;
}

static void h2d(scihpc_ls *h, double *dst, const double *src) {
  SCIHPC_HIP(hipMemcpyAsync(dst, src, sizeof(double) * h->g.total, hipMemcpyHostToDevice, h->stream));
}
static void d2h(scihpc_ls *h, double *dst, const double *src) {
  SCIHPC_HIP(hipMemcpyAsync(dst, src, sizeof(double) * h->g.total, hipMemcpyDeviceToHost, h->stream));
}

extern "C" int scihpc_ls_set_phi(scihpc_ls *h, const double *phi) {
  return guarded([&] {
    ls_check(h);
    SCIHPC_REQUIRE(phi, "phi is null");
    // both stage buffers start identical so ghost corners (never written)
    // keep the caller's values whichever buffer holds the result
    h2d(h, h->phi[0], phi);
    SCIHPC_HIP(hipMemcpyAsync(h->phi[1], h->phi[0], sizeof(double) * h->g.total, hipMemcpyDeviceToDevice,
                              h->stream));
    h->cur = 0;
    SCIHPC_HIP(hipStreamSynchronize(h->stream));
  });
}

extern "C" int scihpc_ls_get_phi(scihpc_ls *h, double *phi) {
  return guarded([&] {
    ls_check(h);
    SCIHPC_REQUIRE(phi, "phi is null");
    d2h(h, phi, h->phi[h->cur]);
    SCIHPC_HIP(hipStreamSynchronize(h->stream));
  });
}

extern "C" int scihpc_ls_set_velocity(scihpc_ls *h, const double *u, const double *v, const double *w) {
  return guarded([&] {
    ls_check(h);
    SCIHPC_REQUIRE(u && (h->g.ndim < 2 || v) && (h->g.ndim < 3 || w), "velocity component is null");
    h2d(h, h->u, u);
    if (v) h2d(h, h->v, v);
    if (w) h2d(h, h->w, w);
    SCIHPC_HIP(hipStreamSynchronize(h->stream));
  });
}

extern "C" int scihpc_ls_weno5_derivatives(scihpc_ls *h, const double *flux, double *fx, double *fy, double *fz) {
  return guarded([&] {
    ls_check(h);
    SCIHPC_REQUIRE(flux && fx, "null array");
    h2d(h, h->tmp, flux);
    const unsigned nb = h->grid_interior();
    SCIHPC_HIP(hipMemsetAsync(h->fx, 0, sizeof(double) * h->g.total, h->stream));
    SCIHPC_HIP(hipMemsetAsync(h->fy, 0, sizeof(double) * h->g.total, h->stream));
    SCIHPC_HIP(hipMemsetAsync(h->fz, 0, sizeof(double) * h->g.total, h->stream));
    if (h->g.ndim == 1)
      k_weno_derivs<1><<<nb, kLsBlock, 0, h->stream>>>(h->g, h->tmp, h->u, h->v, h->w, h->fx, h->fy, h->fz);
    else if (h->g.ndim == 2)
      k_weno_derivs<2><<<nb, kLsBlock, 0, h->stream>>>(h->g, h->tmp, h->u, h->v, h->w, h->fx, h->fy, h->fz);
    else
      k_weno_derivs<3><<<nb, kLsBlock, 0, h->stream>>>(h->g, h->tmp, h->u, h->v, h->w, h->fx, h->fy, h->fz);
    SCIHPC_CHECK_LAUNCH();
    d2h(h, fx, h->fx);
    if (fy) d2h(h, fy, h->fy);
    if (fz) d2h(h, fz, h->fz);
    SCIHPC_HIP(hipStreamSynchronize(h->stream));
  });
}

extern "C" int scihpc_ls_tvd_rk3(scihpc_ls *h, double dt, int nsteps) {
  return guarded([&] {
    ls_check(h);
    SCIHPC_REQUIRE(nsteps >= 0, "nsteps must be >= 0");
    for (int s = 0; s < nsteps; ++s) h->step(dt);
    SCIHPC_HIP(hipStreamSynchronize(h->stream));
  });
}

extern "C" int scihpc_ls_set_scheme(scihpc_ls *h, int scheme) {
  return guarded([&] {
    ls_check(h);
    SCIHPC_REQUIRE(scheme == SCIHPC_LS_WENO5 || scheme == SCIHPC_LS_UCCD, "unknown scheme");
    h->scheme = scheme;
  });
}

extern "C" int scihpc_ls_set_line_solver(scihpc_ls *h, int partitioned) {
  return guarded([&] {
    ls_check(h);
    SCIHPC_REQUIRE(partitioned == 0 || partitioned == 1, "partitioned must be 0 or 1");
    h->twin_partitioned = partitioned != 0;
  });
}

extern "C" int scihpc_ls_line_sweeps(scihpc_ls *h, long long *segmented, long long *end_to_end) {
  return guarded([&] {
    ls_check(h);
    SCIHPC_REQUIRE(segmented && end_to_end, "null argument");
    unsigned state[2] = {0, 0};
    if (h->seg_state) {
      SCIHPC_HIP(hipMemcpyAsync(state, h->seg_state, sizeof(state), hipMemcpyDeviceToHost, h->stream));
      SCIHPC_HIP(hipStreamSynchronize(h->stream));
    }
    *segmented = h->seg_groups;
    *end_to_end = state[1];
  });
}

extern "C" int scihpc_ls_compact_derivatives(scihpc_ls *h, const double *f, int upwind, double *fx, double *fy,
                                             double *fz, double *fxx, double *fyy, double *fzz) {
  return guarded([&] {
    ls_check(h);
    SCIHPC_REQUIRE(f && fx && fxx, "null argument");
    SCIHPC_REQUIRE(h->g.ndim < 2 || (fy && fyy), "fy/fyy required for ndim >= 2");
    SCIHPC_REQUIRE(h->g.ndim < 3 || (fz && fzz), "fz/fzz required for ndim 3");
    h->ensure_iface();
    h2d(h, h->tmp, f);
    double *d1[3] = {h->fx, h->fy, h->fz}, *d2[3] = {h->fxx, h->fyy, h->fzz};
    h->compact(h->tmp, upwind != 0, d1, d2);
    double *o1[3] = {fx, fy, fz}, *o2[3] = {fxx, fyy, fzz};
    for (int a = 0; a < h->g.ndim; ++a) {
      d2h(h, o1[a], d1[a]);
      d2h(h, o2[a], d2[a]);
    }
    SCIHPC_HIP(hipStreamSynchronize(h->stream));
  });
}

extern "C" int scihpc_ls_mass(scihpc_ls *h, double ls_width, double ratio, int positive_ref, double *mass) {
  return guarded([&] {
    ls_check(h);
    SCIHPC_REQUIRE(mass && ls_width > 0, "bad argument");
    SCIHPC_REQUIRE(h->g.ndim >= 2, "lsf_mass is defined for 2-D and 3-D");
    h->ensure_iface();
    double den;
    if (h->g.ndim == 2) h->mpls_sums<2>(ls_width, ratio, positive_ref, *mass, den);
    else h->mpls_sums<3>(ls_width, ratio, positive_ref, *mass, den);
  });
}

extern "C" int scihpc_ls_mpls(scihpc_ls *h, double dt, double ls_width, double ratio, int positive_ref,
                              double mass0, int count) {
  return guarded([&] {
    ls_check(h);
    SCIHPC_REQUIRE(dt > 0 && ls_width > 0 && count >= 0, "bad argument");
    SCIHPC_REQUIRE(h->g.ndim >= 2, "mpls is defined for 2-D and 3-D");
    for (int it = 0; it < count; ++it) {
      if (h->g.ndim == 2) h->mpls_step<2>(dt, ls_width, ratio, positive_ref, mass0);
      else h->mpls_step<3>(dt, ls_width, ratio, positive_ref, mass0);
    }
    SCIHPC_HIP(hipStreamSynchronize(h->stream));
  });
}

extern "C" int scihpc_ls_find_sign(scihpc_ls *h, double ls_width) {
  return guarded([&] {
    ls_check(h);
    SCIHPC_REQUIRE(ls_width > 0, "ls_width must be positive");
    h->ensure_iface();
    k_sign_delta<<<ceil_div(h->g.total, kLsBlock), kLsBlock, 0, h->stream>>>(h->g.total, h->phi[h->cur], ls_width,
                                                                             h->sgn, nullptr);
    SCIHPC_CHECK_LAUNCH();
    SCIHPC_HIP(hipStreamSynchronize(h->stream));
  });
}

extern "C" int scihpc_ls_find_delta(scihpc_ls *h, double ls_width) {
  return guarded([&] {
    ls_check(h);
    SCIHPC_REQUIRE(ls_width > 0, "ls_width must be positive");
    h->ensure_iface();
    k_sign_delta<<<ceil_div(h->g.total, kLsBlock), kLsBlock, 0, h->stream>>>(h->g.total, h->phi[h->cur], ls_width,
                                                                             nullptr, h->dlt);
    SCIHPC_CHECK_LAUNCH();
    SCIHPC_HIP(hipStreamSynchronize(h->stream));
  });
}

extern "C" int scihpc_ls_set_field(scihpc_ls *h, int which, const double *src) {
  return guarded([&] {
    ls_check(h);
    SCIHPC_REQUIRE(src && (which == SCIHPC_LS_SIGN || which == SCIHPC_LS_DELTA), "bad argument");
    h->ensure_iface();
    h2d(h, which == SCIHPC_LS_SIGN ? h->sgn : h->dlt, src);
    SCIHPC_HIP(hipStreamSynchronize(h->stream));
  });
}

extern "C" int scihpc_ls_get_field(scihpc_ls *h, int which, double *dst) {
  return guarded([&] {
    ls_check(h);
    SCIHPC_REQUIRE(dst && (which == SCIHPC_LS_SIGN || which == SCIHPC_LS_DELTA), "bad argument");
    h->ensure_iface();
    d2h(h, dst, which == SCIHPC_LS_SIGN ? h->sgn : h->dlt);
    SCIHPC_HIP(hipStreamSynchronize(h->stream));
  });
}

// per-block maxima of x (x >= 0; empty lanes count 0, as the reference's
// running maximum starts from 0.0)
__global__ void __launch_bounds__(kLsBlock) k_block_max(const double *__restrict__ x, long n,
                                                        double *__restrict__ out) {
  __shared__ double part[kLsBlock / kWave];
  double v = 0.0;
  for (long c = (long)blockIdx.x * blockDim.x + threadIdx.x; c < n; c += (long)gridDim.x * blockDim.x)
    v = fmax(v, x[c]);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off, kWave));
  if (threadIdx.x % kWave == 0) part[threadIdx.x / kWave] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    double m = 0.0;
    for (int w = 0; w < (int)(blockDim.x / kWave); ++w) m = fmax(m, part[w]);
    out[blockIdx.x] = m;
  }
}

// f /= *den on every padded cell
__global__ void __launch_bounds__(kLsBlock) k_div_by(double *__restrict__ f, long n, const double *__restrict__ den) {
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c < n) f[c] = f[c] / *den;
}

extern "C" int scihpc_ls_stabilize_gradient(scihpc_ls *h, double *grad, double *max_grad) {
  return guarded([&] {
    ls_check(h);
    h->ensure_iface();
    const long n = h->g.total;
    const unsigned nb = std::min<unsigned>(ceil_div(n, kLsBlock), 1024);
    double *f = h->phi[h->cur];
    const GodunovH r = godunov_h(h->g);
    if (h->g.ndim == 1) k_godunov<1><<<ceil_div(n, kLsBlock), kLsBlock, 0, h->stream>>>(h->g, r, f, h->sgn, h->grd);
    else if (h->g.ndim == 2) k_godunov<2><<<ceil_div(n, kLsBlock), kLsBlock, 0, h->stream>>>(h->g, r, f, h->sgn, h->grd);
    else k_godunov<3><<<ceil_div(n, kLsBlock), kLsBlock, 0, h->stream>>>(h->g, r, f, h->sgn, h->grd);
    SCIHPC_CHECK_LAUNCH();
    // maxima into the stage scratch s1: nb block maxima, then one
    k_block_max<<<nb, kLsBlock, 0, h->stream>>>(h->grd, n, h->s1);
    SCIHPC_CHECK_LAUNCH();
    k_block_max<<<1, kLsBlock, 0, h->stream>>>(h->s1, (long)nb, h->s1 + nb);
    SCIHPC_CHECK_LAUNCH();
    k_div_by<<<ceil_div(n, kLsBlock), kLsBlock, 0, h->stream>>>(f, n, h->s1 + nb);
    SCIHPC_CHECK_LAUNCH();
    if (grad) d2h(h, grad, h->grd);
    if (max_grad) SCIHPC_HIP(hipMemcpyAsync(max_grad, h->s1 + nb, sizeof(double), hipMemcpyDeviceToHost, h->stream));
    SCIHPC_HIP(hipStreamSynchronize(h->stream));
  });
}

extern "C" int scihpc_ls_redistance(scihpc_ls *h, double dt, double rdt, int nsteps) {
  return guarded([&] {
    ls_check(h);
    SCIHPC_REQUIRE(dt > 0 && rdt > 0 && nsteps >= 0, "bad argument");
    h->ensure_iface();
    for (int it = 0; it < nsteps; ++it) {
      if (h->g.ndim == 1) h->redistance_step<1>(dt, rdt);
      else if (h->g.ndim == 2) h->redistance_step<2>(dt, rdt);
      else h->redistance_step<3>(dt, rdt);
    }
    SCIHPC_HIP(hipStreamSynchronize(h->stream));
  });
}

extern "C" int scihpc_ls_apply_bc(scihpc_ls *h, double *f, int stag) {
  return guarded([&] {
    ls_check(h);
    SCIHPC_REQUIRE(f, "null array");
    SCIHPC_REQUIRE(stag >= -1 && stag < h->g.ndim, "stag must be -1 or an axis < ndim");
    h2d(h, h->tmp, f);
    h->apply_bc(h->tmp, stag);
    d2h(h, f, h->tmp);
    SCIHPC_HIP(hipStreamSynchronize(h->stream));
  });
}

extern "C" int scihpc_ls_density(scihpc_ls *h, double ls_width, double ratio, int positive_ref, double *rho) {
  return guarded([&] {
    ls_check(h);
    SCIHPC_REQUIRE(rho && ls_width > 0, "bad density arguments");
    k_density<<<ceil_div(h->g.total, kLsBlock), kLsBlock, 0, h->stream>>>(h->phi[h->cur], h->g.total, ls_width,
                                                                          ratio, positive_ref, h->tmp);
    SCIHPC_CHECK_LAUNCH();
    d2h(h, rho, h->tmp);
    SCIHPC_HIP(hipStreamSynchronize(h->stream));
  });
}

extern "C" int scihpc_ls_time_step(scihpc_ls *h, double dt, int iters, double *ms, double *bytes) {
  return guarded([&] {
    ls_check(h);
    SCIHPC_REQUIRE(iters > 0, "iters must be > 0");
    h->step(dt);  // warm-up
    SCIHPC_HIP(hipEventRecord(h->ev0, h->stream));
    for (int s = 0; s < iters; ++s) h->step(dt);
    SCIHPC_HIP(hipEventRecord(h->ev1, h->stream));
    SCIHPC_HIP(hipEventSynchronize(h->ev1));
    float t = 0.f;
    SCIHPC_HIP(hipEventElapsedTime(&t, h->ev0, h->ev1));
    if (ms) *ms = t / iters;
    // minimal Shu-Osher traffic per step: (7 + 3 d) * 8 B per interior cell
    if (bytes) *bytes = (7.0 + 3.0 * h->g.ndim) * 8.0 * (double)h->g.interior;
  });
}

// ================================================= projection step (C ABI)
// One projection step on the padded fields of one grid, around a multigrid
// handle of the same interior grid: the FPC step of SciHPC
// (pressure_guess_solution, init_ppe_fpc_coefficients,
// fast_pressure_correction; projection_method.cpp:467-541, 659-753,
// 803-815) with the reference-faithful full cycles, and the
// variable-density projection (projection_method.cpp:544-657) with the SOR
// replaced by the A(rho) multigrid solve.
struct scihpc_proj {
  Grid g{};
  BcSpec pbc{};     // pressure: Neumann (the pressure wrapper of the drivers)
  BcSpec vbc[3]{};  // velocity components: SLIP -> NO_SLIP wall-normal (wrapper.cpp:111-125)
  hipStream_t stream = nullptr;
  double *rho = nullptr, *pold = nullptr, *pold2 = nullptr, *phat = nullptr, *p = nullptr;
  double *u = nullptr, *v = nullptr, *w = nullptr;
  double *mg_rhs = nullptr, *sol = nullptr, *part = nullptr, *hpart = nullptr;

  double *alloc(long n) {
    void *q = nullptr;
    SCIHPC_HIP(hipMalloc(&q, sizeof(double) * n));
    SCIHPC_HIP(hipMemsetAsync(q, 0, sizeof(double) * n, stream));
    return static_cast<double *>(q);
  }
  void bc(double *f, const BcSpec &b, int stag) {
    for (int a = 0; a < g.ndim; ++a) {
      const int t1 = (a + 1) % 3, t2 = (a + 2) % 3;
      const long lines = (long)g.n[t1] * g.n[t2];
      k_bc_axis<<<ceil_div(lines, kLsBlock), kLsBlock, 0, stream>>>(g, f, b, a, stag);
      SCIHPC_CHECK_LAUNCH();
    }
  }
  // the BCs of three fields (u, v, w or their node values), one launch per
  // axis instead of one per field and axis; the same result as three bc()
  void bc3(double *f0, double *f1, double *f2, const BcSpec *b, int s0, int s1, int s2) {
    BcFields m{{f0, f1, f2}, {b[0], b[1], b[2]}, {s0, s1, s2}, 3};
    for (int a = 0; a < g.ndim; ++a) {
      const int t1 = (a + 1) % 3, t2 = (a + 2) % 3;
      const long lines = (long)g.n[t1] * g.n[t2];
      k_bc_axis_fields<<<ceil_div(3 * lines, kLsBlock), kLsBlock, 0, stream>>>(g, m, a);
      SCIHPC_CHECK_LAUNCH();
    }
  }
  void h2d(double *dst, const double *src) {
    SCIHPC_HIP(hipMemcpyAsync(dst, src, sizeof(double) * g.total, hipMemcpyHostToDevice, stream));
  }
  void d2h(double *dst, const double *src) {
    SCIHPC_HIP(hipMemcpyAsync(dst, src, sizeof(double) * g.total, hipMemcpyDeviceToHost, stream));
  }
  void check_mg(scihpc_mg *mg) {
    SCIHPC_REQUIRE(mg, "null multigrid handle");
    int a = 0, b = 0, c = 0, deg = 0;
    const int rc = scihpc_mg_level_shape(mg, 0, &a, &b, &c, &deg);
    SCIHPC_REQUIRE(rc == SCIHPC_OK, "bad multigrid handle");
    SCIHPC_REQUIRE(a == g.n[0] && b == g.n[1] && c == (g.ndim > 2 ? g.n[2] : 1), "multigrid grid differs");
  }
  // momentum predictor state and scratch (allocated on first use): phi, the
  // transferred velocities nvel, sources (current / other, ping-pong per
  // component), delta, viscosity, the level-set gradient and curvature
  double *phi = nullptr, *nvel[3] = {nullptr, nullptr, nullptr};
  double *src[3] = {nullptr, nullptr, nullptr}, *src_alt[3] = {nullptr, nullptr, nullptr};
  double *dl = nullptr, *mu = nullptr, *lf[3] = {nullptr, nullptr, nullptr}, *curv = nullptr;

  void ensure_momentum() {
    if (phi) return;
    const long T = g.total;
    phi = alloc(T);
    dl = alloc(T);
    mu = alloc(T);
    curv = alloc(T);
    for (int a = 0; a < 3; ++a) {
      nvel[a] = alloc(T);
      src[a] = alloc(T);
      src_alt[a] = alloc(T);
      lf[a] = alloc(T);
    }
  }

  // find_source_sec + find_intermediate_velocity on the device-resident
  // phi, u, v, w, nvel and sources; rho <- find_density
  // find_source_sec (projection_method.cpp:314-382): the new sources of
  // every component; the handle's sources rotate (src_alt <- old, src <-
  // new) and the velocity is not touched
  void sources(const FlowParams &fp) {
    const unsigned nb = ceil_div(g.total, kLsBlock);
    const bool st = fp.we > 0.0;
#define SCIHPC_PROPS(D, S) \
  k_mom_props<D, S><<<nb, kLsBlock, 0, stream>>>(g, fp, phi, dl, rho, mu, lf[0], lf[1], lf[2], curv)
    if (g.ndim == 2) { if (st) SCIHPC_PROPS(2, true); else SCIHPC_PROPS(2, false); }
    else { if (st) SCIHPC_PROPS(3, true); else SCIHPC_PROPS(3, false); }
#undef SCIHPC_PROPS
    SCIHPC_CHECK_LAUNCH();
    double *vel[3] = {u, v, w};
    for (int a = 0; a < g.ndim; ++a) {
      if (g.ndim == 2)
        k_to_face<2><<<nb, kLsBlock, 0, stream>>>(g, a, u, v, w, nvel[0], nvel[1], nvel[2]);
      else
        k_to_face<3><<<nb, kLsBlock, 0, stream>>>(g, a, u, v, w, nvel[0], nvel[1], nvel[2]);
      SCIHPC_CHECK_LAUNCH();
      // nvel->apply_vel_a_bc (wrapper.cpp:40-59)
      bc3(nvel[0], nvel[1], nvel[2], vbc, a, a, a);
#define SCIHPC_SRC(D, A)                                                                                 \
  k_mom_src<D, A><<<nb, kLsBlock, 0, stream>>>(g, fp, vel[A], nvel[0], nvel[1], nvel[2], dl, rho, mu, lf[0], \
                                               lf[1], lf[2], curv, src_alt[A])
      if (g.ndim == 2) {
        if (a == 0) SCIHPC_SRC(2, 0); else SCIHPC_SRC(2, 1);
      } else {
        if (a == 0) SCIHPC_SRC(3, 0); else if (a == 1) SCIHPC_SRC(3, 1); else SCIHPC_SRC(3, 2);
      }
#undef SCIHPC_SRC
      SCIHPC_CHECK_LAUNCH();
    }
    for (int a = 0; a < g.ndim; ++a) std::swap(src[a], src_alt[a]);
  }

  // find_intermediate_velocity (projection_method.cpp:384-402): AB2 with the
  // current and previous sources, then the velocity BCs; components beyond
  // ndim keep their source (2-D: w_src is never written), so both terms of
  // their update read it
  void ab2(const FlowParams &fp) {
    const unsigned nb = ceil_div(g.total, kLsBlock);
    const double *sn[3], *so[3];
    for (int a = 0; a < 3; ++a) {
      sn[a] = src[a];
      so[a] = a < g.ndim ? src_alt[a] : src[a];
    }
    k_ab2<<<nb, kLsBlock, 0, stream>>>(g.total, fp.dt, u, v, w, sn[0], sn[1], sn[2], so[0], so[1], so[2]);
    SCIHPC_CHECK_LAUNCH();
    bc3(u, v, w, vbc, 0, 1, 2);
  }

  void momentum(const FlowParams &fp) {
    sources(fp);
    ab2(fp);
  }

  // node_from_face + nvel->apply_nvel_bc (wrapper_func.cpp:264-293,
  // wrapper.cpp:28-33)
  void node_velocity() {
    const unsigned nb = ceil_div(g.total, kLsBlock);
    if (g.ndim == 2) k_node_from_face<2><<<nb, kLsBlock, 0, stream>>>(g, u, v, w, nvel[0], nvel[1], nvel[2]);
    else k_node_from_face<3><<<nb, kLsBlock, 0, stream>>>(g, u, v, w, nvel[0], nvel[1], nvel[2]);
    SCIHPC_CHECK_LAUNCH();
    bc3(nvel[0], nvel[1], nvel[2], vbc, -1, -1, -1);
  }

  void finish_pressure_and_velocity(scihpc_mg *mg, const double *ph, double dt, double rho12) {
    SCIHPC_REQUIRE(scihpc_mg_get_sol_device(mg, sol) == SCIHPC_OK, scihpc_last_error());
    k_mg_to_padded<<<ceil_div(g.interior, kLsBlock), kLsBlock, 0, stream>>>(g, sol, p);
    SCIHPC_CHECK_LAUNCH();
    bc(p, pbc, -1);
    const long nv = (long)(g.N[0] - 1) * (g.N[1] - 1) * g.N[2];
    if (g.ndim == 2)
      k_correct_velocity<2><<<ceil_div(nv, kLsBlock), kLsBlock, 0, stream>>>(g, rho, p, ph, dt, rho12, u, v, w);
    else
      k_correct_velocity<3><<<ceil_div(nv, kLsBlock), kLsBlock, 0, stream>>>(g, rho, p, ph, dt, rho12, u, v, w);
    SCIHPC_CHECK_LAUNCH();
    bc3(u, v, w, vbc, 0, 1, 2);
  }
};

extern "C" int scihpc_proj_create(int ndim, int nx, int ny, int nz, double dx, double dy, double dz,
                                  const int *vel_bc_types, scihpc_proj **out) {
  return guarded([&] {
    SCIHPC_REQUIRE(out, "out is null");
    *out = nullptr;
    SCIHPC_REQUIRE(ndim == 2 || ndim == 3, "ndim must be 2 or 3");
    SCIHPC_REQUIRE(nx > 2 && ny > 2 && (ndim < 3 || nz > 2), "each axis needs > 2 cells");
    SCIHPC_REQUIRE(dx > 0 && dy > 0 && (ndim < 3 || dz > 0), "spacings must be positive");
    SCIHPC_REQUIRE(vel_bc_types, "vel_bc_types is null");
    auto *h = new scihpc_proj;
    try {
      h->g = make_grid(ndim, nx, ny, nz, dx, dy, dz);
      for (int q = 0; q < 6; ++q) {
        const int t = vel_bc_types[q];
        SCIHPC_REQUIRE(q >= 2 * ndim || (t >= 0 && t <= 4 && t != SCIHPC_BC_PERIODIC), "unsupported bc type");
        h->pbc.type[q] = SCIHPC_BC_NEUMANN;
        for (int a = 0; a < 3; ++a) {
          const bool normal = q / 2 == a;
          h->vbc[a].type[q] = (normal && t == SCIHPC_BC_SLIP) ? SCIHPC_BC_NO_SLIP : t;
        }
      }
      SCIHPC_HIP(hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking));
      const long T = h->g.total;
      h->rho = h->alloc(T);
      h->pold = h->alloc(T);
      h->pold2 = h->alloc(T);
      h->phat = h->alloc(T);
      h->p = h->alloc(T);
      h->u = h->alloc(T);
      h->v = h->alloc(T);
      h->w = h->alloc(T);
      h->mg_rhs = h->alloc(h->g.interior);
      h->sol = h->alloc(h->g.interior);
      h->part = h->alloc(ceil_div(h->g.interior, kLsBlock));
      SCIHPC_HIP(hipHostMalloc(reinterpret_cast<void **>(&h->hpart),
                               sizeof(double) * ceil_div(h->g.interior, kLsBlock), hipHostMallocDefault));
      SCIHPC_HIP(hipStreamSynchronize(h->stream));
    } catch (...) {
      scihpc_proj_destroy(h);
      throw;
    }
    *out = h;
  });
}

extern "C" int scihpc_proj_destroy(scihpc_proj *h) {
  if (!h) return SCIHPC_OK;
  if (h->stream) (void)hipStreamSynchronize(h->stream);
  for (double *q : {h->rho, h->pold, h->pold2, h->phat, h->p, h->u, h->v, h->w, h->mg_rhs, h->sol, h->part,
                    h->phi, h->dl, h->mu, h->curv})
    if (q) (void)hipFree(q);
  for (int a = 0; a < 3; ++a)
    for (double *q : {h->nvel[a], h->src[a], h->src_alt[a], h->lf[a]})
      if (q) (void)hipFree(q);
  if (h->hpart) (void)hipHostFree(h->hpart);
  if (h->stream) (void)hipStreamDestroy(h->stream);
  delete h;
  return SCIHPC_OK;
}

extern "C" int scihpc_proj_fpc_step(scihpc_proj *h, scihpc_mg *mg, const scihpc_fpc_params *prm, const double *rho,
                                    const double *p_old, const double *p_old2, double *u, double *v, double *w,
                                    double *p, double *phat, int *cycles) {
  return guarded([&] {
    SCIHPC_REQUIRE(h && prm && rho && p_old && p_old2 && u && v && w && p && phat, "null argument");
    SCIHPC_REQUIRE(prm->dt > 0 && prm->dt_old2 != 0 && prm->rho12 > 0 && prm->max_cycles >= 0, "bad parameters");
    SCIHPC_REQUIRE(prm->cycle == 0 || prm->cycle == 1, "cycle must be 0 (reference full cycles) or 1 (red-black)");
    h->check_mg(mg);
    const Grid &g = h->g;
    h->h2d(h->rho, rho);
    h->h2d(h->pold, p_old);
    h->h2d(h->pold2, p_old2);
    h->h2d(h->u, u);
    h->h2d(h->v, v);
    h->h2d(h->w, w);
    k_pressure_guess<<<ceil_div(g.total, kLsBlock), kLsBlock, 0, h->stream>>>(h->pold, h->pold2, h->phat, g.total,
                                                                             prm->dt_old, prm->dt_old2);
    if (g.ndim == 2)
      k_fpc_rhs<2><<<ceil_div(g.interior, kLsBlock), kLsBlock, 0, h->stream>>>(g, h->rho, h->phat, h->u, h->v, h->w,
                                                                             prm->dt, prm->rho12, h->mg_rhs);
    else
      k_fpc_rhs<3><<<ceil_div(g.interior, kLsBlock), kLsBlock, 0, h->stream>>>(g, h->rho, h->phat, h->u, h->v, h->w,
                                                                             prm->dt, prm->rho12, h->mg_rhs);
    SCIHPC_CHECK_LAUNCH();
    SCIHPC_HIP(hipStreamSynchronize(h->stream));
    // the loop of fast_pressure_correction (projection_method.cpp:694-706):
    // full cycles (or, cycle = 1, red-black V(2,2) cycles) from the
    // handle's current solution until the absolute residual is <= ppe_tol
    SCIHPC_REQUIRE(scihpc_mg_set_rhs_device(mg, h->mg_rhs) == SCIHPC_OK, scihpc_last_error());
    double err = 0.0;
    SCIHPC_REQUIRE(scihpc_mg_residual(mg, 0, &err) == SCIHPC_OK, scihpc_last_error());
    int it = 0;
    while (err > prm->ppe_tol && it < prm->max_cycles) {
      ++it;
      if (prm->cycle == 1) SCIHPC_REQUIRE(scihpc_mg_vcycle(mg, 2, 2) == SCIHPC_OK, scihpc_last_error());
      else SCIHPC_REQUIRE(scihpc_mg_fullcycle_ref(mg) == SCIHPC_OK, scihpc_last_error());
      SCIHPC_REQUIRE(scihpc_mg_residual(mg, 0, &err) == SCIHPC_OK, scihpc_last_error());
    }
    // the reference's cycles leave the level-0 solution mean-free
    // (compatibility_condition after every relax); the red-black cycles do
    // not, so the constant is removed here
    if (prm->cycle == 1 && it > 0) SCIHPC_REQUIRE(scihpc_mg_compat(mg, 0, 1) == SCIHPC_OK, scihpc_last_error());
    h->finish_pressure_and_velocity(mg, h->phat, prm->dt, prm->rho12);
    h->d2h(u, h->u);
    h->d2h(v, h->v);
    h->d2h(w, h->w);
    h->d2h(p, h->p);
    h->d2h(phat, h->phat);
    SCIHPC_HIP(hipStreamSynchronize(h->stream));
    if (cycles) *cycles = it;
  });
}

extern "C" int scihpc_proj_step(scihpc_proj *h, scihpc_mg *mg, double dt, const scihpc_solve_opts *opts,
                                const double *rho, double *u, double *v, double *w, double *p,
                                scihpc_solve_stats *stats) {
  int rc = SCIHPC_OK;
  const int g_rc = guarded([&] {
    SCIHPC_REQUIRE(h && opts && rho && u && v && w && p && dt > 0, "null or bad argument");
    h->check_mg(mg);
    const Grid &g = h->g;
    SCIHPC_REQUIRE(scihpc_mg_set_density_padded(mg, rho) == SCIHPC_OK, scihpc_last_error());
    h->h2d(h->rho, rho);
    h->h2d(h->u, u);
    h->h2d(h->v, v);
    h->h2d(h->w, w);
    const unsigned nb = ceil_div(g.interior, kLsBlock);
    if (g.ndim == 2)
      k_div_rhs<2><<<nb, kLsBlock, 0, h->stream>>>(g, h->u, h->v, h->w, dt, h->mg_rhs, h->part);
    else
      k_div_rhs<3><<<nb, kLsBlock, 0, h->stream>>>(g, h->u, h->v, h->w, dt, h->mg_rhs, h->part);
    SCIHPC_CHECK_LAUNCH();
    // compatibility of the all-Neumann problem: remove the mean of div u / dt
    SCIHPC_HIP(hipMemcpyAsync(h->hpart, h->part, sizeof(double) * nb, hipMemcpyDeviceToHost, h->stream));
    SCIHPC_HIP(hipStreamSynchronize(h->stream));
    double sum = 0.0;
    for (unsigned b = 0; b < nb; ++b) sum += h->hpart[b];
    k_sub_const<<<nb, kLsBlock, 0, h->stream>>>(h->mg_rhs, g.interior, sum / (double)g.interior);
    SCIHPC_CHECK_LAUNCH();
    SCIHPC_HIP(hipStreamSynchronize(h->stream));
    SCIHPC_REQUIRE(scihpc_mg_set_rhs_device(mg, h->mg_rhs) == SCIHPC_OK, scihpc_last_error());
    scihpc_solve_stats st{};
    rc = scihpc_mg_solve(mg, opts, &st);
    SCIHPC_REQUIRE(rc == SCIHPC_OK || rc == SCIHPC_NOT_CONVERGED, scihpc_last_error());
    h->finish_pressure_and_velocity(mg, nullptr, dt, 1.0);
    h->d2h(u, h->u);
    h->d2h(v, h->v);
    h->d2h(w, h->w);
    h->d2h(p, h->p);
    SCIHPC_HIP(hipStreamSynchronize(h->stream));
    if (stats) *stats = st;
  });
  return g_rc != SCIHPC_OK ? g_rc : rc;
}

static FlowParams flow_params(const scihpc_flow_params *p) {
  SCIHPC_REQUIRE(p, "null parameters");
  SCIHPC_REQUIRE(p->dt > 0 && p->reynolds > 0 && p->ls_width > 0 && p->density_ratio > 0 &&
                     p->viscosity_ratio > 0,
                 "dt, reynolds, ls_width and the ratios must be positive");
  return FlowParams{p->dt, p->reynolds, p->froude, p->weber, p->ls_width, p->density_ratio, p->viscosity_ratio,
                    p->positive_ref != 0};
}

extern "C" int scihpc_proj_momentum_step(scihpc_proj *h, const scihpc_flow_params *prm, const double *phi,
                                         double *u, double *v, double *w, double *nu, double *nv, double *nw,
                                         double *rho) {
  return guarded([&] {
    SCIHPC_REQUIRE(h && phi && u && v && w && nu && nv && nw, "null argument");
    const FlowParams fp = flow_params(prm);
    h->ensure_momentum();
    h->h2d(h->phi, phi);
    h->h2d(h->u, u);
    h->h2d(h->v, v);
    h->h2d(h->w, w);
    h->h2d(h->nvel[0], nu);
    h->h2d(h->nvel[1], nv);
    h->h2d(h->nvel[2], nw);
    h->momentum(fp);
    h->d2h(u, h->u);
    h->d2h(v, h->v);
    h->d2h(w, h->w);
    h->d2h(nu, h->nvel[0]);
    h->d2h(nv, h->nvel[1]);
    h->d2h(nw, h->nvel[2]);
    if (rho) h->d2h(rho, h->rho);
    SCIHPC_HIP(hipStreamSynchronize(h->stream));
  });
}

extern "C" int scihpc_proj_find_sources(scihpc_proj *h, const scihpc_flow_params *prm, const double *phi,
                                        const double *u, const double *v, const double *w, double *nu, double *nv,
                                        double *nw, double *rho) {
  return guarded([&] {
    SCIHPC_REQUIRE(h && phi && u && v && w && nu && nv && nw, "null argument");
    const FlowParams fp = flow_params(prm);
    h->ensure_momentum();
    h->h2d(h->phi, phi);
    h->h2d(h->u, u);
    h->h2d(h->v, v);
    h->h2d(h->w, w);
    h->h2d(h->nvel[0], nu);
    h->h2d(h->nvel[1], nv);
    h->h2d(h->nvel[2], nw);
    h->sources(fp);
    h->d2h(nu, h->nvel[0]);
    h->d2h(nv, h->nvel[1]);
    h->d2h(nw, h->nvel[2]);
    if (rho) h->d2h(rho, h->rho);
    SCIHPC_HIP(hipStreamSynchronize(h->stream));
  });
}

extern "C" int scihpc_proj_intermediate_velocity(scihpc_proj *h, const scihpc_flow_params *prm, double *u,
                                                 double *v, double *w) {
  return guarded([&] {
    SCIHPC_REQUIRE(h && u && v && w, "null argument");
    const FlowParams fp = flow_params(prm);
    h->ensure_momentum();
    h->h2d(h->u, u);
    h->h2d(h->v, v);
    h->h2d(h->w, w);
    h->ab2(fp);
    h->d2h(u, h->u);
    h->d2h(v, h->v);
    h->d2h(w, h->w);
    SCIHPC_HIP(hipStreamSynchronize(h->stream));
  });
}

extern "C" int scihpc_proj_set_sources(scihpc_proj *h, const double *su, const double *sv, const double *sw) {
  return guarded([&] {
    SCIHPC_REQUIRE(h && su && sv && sw, "null argument");
    h->ensure_momentum();
    h->h2d(h->src[0], su);
    h->h2d(h->src[1], sv);
    h->h2d(h->src[2], sw);
    SCIHPC_HIP(hipStreamSynchronize(h->stream));
  });
}

extern "C" int scihpc_proj_get_sources(scihpc_proj *h, double *su, double *sv, double *sw) {
  return guarded([&] {
    SCIHPC_REQUIRE(h && su && sv && sw, "null argument");
    h->ensure_momentum();
    h->d2h(su, h->src[0]);
    h->d2h(sv, h->src[1]);
    h->d2h(sw, h->src[2]);
    SCIHPC_HIP(hipStreamSynchronize(h->stream));
  });
}

extern "C" int scihpc_proj_node_velocity(scihpc_proj *h, const double *u, const double *v, const double *w,
                                         double *nu, double *nv, double *nw) {
  return guarded([&] {
    SCIHPC_REQUIRE(h && u && v && w && nu && nv && nw, "null argument");
    h->ensure_momentum();
    h->h2d(h->u, u);
    h->h2d(h->v, v);
    h->h2d(h->w, w);
    h->h2d(h->nvel[0], nu);
    h->h2d(h->nvel[1], nv);
    h->h2d(h->nvel[2], nw);
    h->node_velocity();
    h->d2h(nu, h->nvel[0]);
    h->d2h(nv, h->nvel[1]);
    h->d2h(nw, h->nvel[2]);
    SCIHPC_HIP(hipStreamSynchronize(h->stream));
  });
}

extern "C" int scihpc_proj_time_momentum(scihpc_proj *h, const scihpc_flow_params *prm, int iters, double *ms) {
  return guarded([&] {
    SCIHPC_REQUIRE(h && ms && iters > 0, "bad argument");
    const FlowParams fp = flow_params(prm);
    h->ensure_momentum();
    hipEvent_t a, b;
    SCIHPC_HIP(hipEventCreate(&a));
    SCIHPC_HIP(hipEventCreate(&b));
    h->momentum(fp);
    SCIHPC_HIP(hipEventRecord(a, h->stream));
    for (int it = 0; it < iters; ++it) h->momentum(fp);
    SCIHPC_HIP(hipEventRecord(b, h->stream));
    SCIHPC_HIP(hipEventSynchronize(b));
    float t = 0;
    SCIHPC_HIP(hipEventElapsedTime(&t, a, b));
    *ms = t / iters;
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
  });
}
