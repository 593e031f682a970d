// mg_tile3d.hpp -- the middle levels of a 3-D V-cycle: a whole pre- or
// post-smoothing in one launch.  Included by mg.hip after mg_block.hpp, whose
// patches it uses.
//
// A workgroup owns an 8 x 8 x 8 tile and works on it grown by four cells, 16^3
// cells in 512 threads: two red-black sweeps are four colour passes, and each
// pass makes the outermost ring that was still right wrong (its neighbours
// outside are missing), so after four the tile itself is what the sweeps give
// and nothing is exchanged between workgroups.  A thread keeps four pairs of
// cells, one above the other in z, for the whole launch: faces, right-hand
// side, diagonal, iterate in registers; only the iterate is in LDS, red and
// black apart (BlockPatch, with z for the patch's axis and y for the third).
//   k_pre3d : from a zero iterate (no read of it): sweeps, residual, child
//             average to the coarse level, tile written.
//   k_post3d: coarse correction added, sweeps, tile written to a second buffer.
// What bounds it: the latency of one batch of loads and of four passes (8
// cells are computed for one that is kept), which on levels of up to 64^3
// cells costs less than the launches it replaces (scihpc_mg::tile3_level has
// both sides): a 128^3 FP64 solve with 64^3 and 32^3 levels in z-marching sweeps
// took 6.53 ms, in colour passes 5.17, here 4.96.
#pragma once

namespace scihpc {

constexpr int kT3 = 8, kT3Halo = 4, kT3Threads = 512;
constexpr int kT3Sx = 10, kT3Sz = 10 * 18, kT3Xc = 10 * 18 * 18;  // row, plane and size of a colour array

template <typename T>
struct Tile3 {
  BlockPatch<T, 3, 4> q;
  int i2, j, k;        // pair column, row, first plane in the grown tile
  int gx, gy, gz;      // cell of the even one, first plane
  bool row_in;         // gx, gy inside the level
};

// where the thread's pairs are, and everything but the iterate
template <typename T, bool VAR>
__device__ __forceinline__ void tile3_load(const DLevel<T> &F, int x0, int y0, int z0, Tile3<T> &t) {
  const int tid = threadIdx.x;
  t.i2 = tid & 7;
  t.j = (tid >> 3) & 15;
  t.k = (tid >> 7) * 4;
  t.gx = x0 - kT3Halo + 2 * t.i2;
  t.gy = y0 - kT3Halo + t.j;
  t.gz = z0 - kT3Halo + t.k;
  t.row_in = t.gx >= 0 && t.gx < F.nx && t.gy >= 0 && t.gy < F.ny;
  BlockPatch<T, 3, 4> &q = t.q;
  q.at = t.i2 + 1 + kT3Sx * (t.j + 1) + kT3Sz * (t.k + 1);
  q.side = ((t.gy + t.gz) & 1) ? 1 : -1;
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    BlockRec<T, 3> rec = {};
    T be = T(0), bo = T(0);
    const int gz = t.gz + m;
    if (t.row_in && gz >= 0 && gz < F.nz) {
      const int c = t.gx + F.nx * (t.gy + F.ny * gz);
      be = F.rhs[c];
      bo = F.rhs[c + 1];
      T below[2] = {T(0), T(0)}, above[2];
      if (VAR && t.gy > 0) {
        below[0] = F.cy[c - F.nx];
        below[1] = F.cy[c - F.nx + 1];
      }
      rec = block_record<T, 3>(F, VAR ? F.cx : nullptr, F.cy, F.cz, t.gx >> 1, t.gy, gz, below, above);
    }
    const bool swap = ((q.side > 0) ^ (m & 1)) != 0;  // the odd cell is the red one
    q.b[0][m] = swap ? bo : be;
    q.b[1][m] = swap ? be : bo;
    q.x[0][m] = q.x[1][m] = T(0);
    q.wp[m] = rec.wp;
#pragma unroll
    for (int col = 0; col < 2; ++col) {
      q.ws[col][m] = rec.ws[col];
      q.wv[col][m] = rec.wb[col];
      if (m == 3) q.wv[1 - col][4] = rec.wf[col];
      q.wb[col][m] = rec.wd[col];
      q.wf[col][m] = rec.wu[col];
      q.d[col][m] = rec.d[col];
      q.rd[col][m] = block_rcp(rec.d[col]);
    }
  }
}

// the thread's cells of the tile itself
template <typename T>
__device__ __forceinline__ bool tile3_own(const Tile3<T> &t) {
  return t.row_in && t.i2 >= 2 && t.i2 < 6 && t.j >= 4 && t.j < 12 && t.k >= 4 && t.k < 12;
}

template <typename T>
__device__ __forceinline__ void tile3_store(const DLevel<T> &F, const Tile3<T> &t, T *__restrict__ out) {
  if (!tile3_own(t)) return;
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    if (t.gz + m >= F.nz) break;
    const int c = t.gx + F.nx * (t.gy + F.ny * (t.gz + m));
    const bool swap = ((t.q.side > 0) ^ (m & 1)) != 0;
    out[c] = swap ? t.q.x[1][m] : t.q.x[0][m];
    out[c + 1] = swap ? t.q.x[0][m] : t.q.x[1][m];
  }
}

__device__ __forceinline__ bool tile3_origin(int nx, int ny, int nz, int &x0, int &y0, int &z0) {
  const int tx = (nx + kT3 - 1) / kT3, ty = (ny + kT3 - 1) / kT3, n = tx * ty * ((nz + kT3 - 1) / kT3);
  const int b = blockIdx.x;
  const int tile = n % 8 ? b : (b % 8) * (n / 8) + b / 8;  // neighbouring tiles on one XCD
  x0 = tile % tx * kT3;
  y0 = tile / tx % ty * kT3;
  z0 = tile / (tx * ty) * kT3;
  return tile < n;
}

template <typename T, bool VAR>
__global__ void __launch_bounds__(kT3Threads) k_pre3d(DLevel<T> F, DLevel<T> G, T *__restrict__ out, int nu1) {
  __shared__ T X[2 * kT3Xc];
  __shared__ T R[kT3][kT3][kT3 / 2];
  int x0, y0, z0;
  if (!tile3_origin(F.nx, F.ny, F.nz, x0, y0, z0)) return;  // the whole workgroup
  Tile3<T> t;
  tile3_load<T, VAR>(F, x0, y0, z0, t);
  for (int s = threadIdx.x; s < 2 * kT3Xc; s += kT3Threads) X[s] = T(0);
  __syncthreads();
  block_sweeps<T, 3, 4, 0>(t.q, true, X, kT3Sz, kT3Sx, kT3Xc, nu1, true);
  if (tile3_own(t)) {
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      T r[2];
#pragma unroll
      for (int col = 0; col < 2; ++col)
        r[col] = t.q.b[col][m] - (block_off<T, 3, 4>(t.q, col, m, X + (1 - col) * kT3Xc + t.q.at, kT3Sz, kT3Sx) +
                                  t.q.d[col][m] * t.q.x[col][m]);
      R[t.k + m - 4][t.j - 4][t.i2 - 2] = r[0] + r[1];
    }
  }
  tile3_store(F, t, out);
  __syncthreads();
  if (threadIdx.x < 64) {
    const int I = threadIdx.x & 3, J = threadIdx.x >> 2 & 3, K = threadIdx.x >> 4;
    const int gi = x0 / 2 + I, gj = y0 / 2 + J, gk = z0 / 2 + K;
    if (gi < G.nx && gj < G.ny && gk < G.nz) {
      T s = R[2 * K][2 * J][I] + R[2 * K][2 * J + 1][I];
      s += R[2 * K + 1][2 * J][I] + R[2 * K + 1][2 * J + 1][I];
      const int c = gi + G.nx * (gj + G.ny * gk);
      G.rhs[c] = s * T(0.125);
      G.sol[c] = T(0);
    }
  }
}

template <typename T, bool VAR>
__global__ void __launch_bounds__(kT3Threads) k_post3d(DLevel<T> G, DLevel<T> F, T *__restrict__ out, int nu2, int dir) {
  constexpr int N = kT3 / 2 + kT3Halo + 2;  // coarse cells under the grown tile and one more on each side
  __shared__ T X[2 * kT3Xc];
  __shared__ T C[N][N][N];
  int x0, y0, z0;
  if (!tile3_origin(F.nx, F.ny, F.nz, x0, y0, z0)) return;
  const int cx0 = (x0 - kT3Halo) / 2 - 1, cy0 = (y0 - kT3Halo) / 2 - 1, cz0 = (z0 - kT3Halo) / 2 - 1;
  T cv[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int s = threadIdx.x + h * kT3Threads;
    int I = cx0 + s % N, J = cy0 + s / N % N, K = cz0 + s / (N * N);
    const bool in = I >= 0 && I < G.nx && J >= 0 && J < G.ny && K >= 0 && K < G.nz;
    I = min(max(I, 0), G.nx - 1);
    J = min(max(J, 0), G.ny - 1);
    K = min(max(K, 0), G.nz - 1);
    // a Dirichlet ghost is 0, a Neumann one the nearest cell
    cv[h] = s < N * N * N && (in || !dir) ? G.sol[I + G.nx * (J + G.ny * K)] : T(0);
  }
  Tile3<T> t;
  tile3_load<T, VAR>(F, x0, y0, z0, t);
  T xe[4], xo[4];
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const bool in = t.row_in && t.gz + m >= 0 && t.gz + m < F.nz;
    const int c = t.gx + F.nx * (t.gy + F.ny * (t.gz + m));
    xe[m] = in ? F.sol[c] : T(0);
    xo[m] = in ? F.sol[c + 1] : T(0);
  }
  for (int s = threadIdx.x; s < 2 * kT3Xc; s += kT3Threads) X[s] = T(0);
#pragma unroll
  for (int h = 0; h < 2; ++h)
    if (threadIdx.x + h * kT3Threads < N * N * N) (&C[0][0][0])[threadIdx.x + h * kT3Threads] = cv[h];
  __syncthreads();
  const T ty = (t.j & 1) ? T(0.25) : T(0.75);
  const int Ja = (t.j + 1) >> 1;  // row floor((2 j - 1) / 4) of the coarse values, which start one before
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    if (!(t.row_in && t.gz + m >= 0 && t.gz + m < F.nz)) continue;
    const int Ka = (t.k + m + 1) >> 1;
    const T tz = (m & 1) ? T(0.25) : T(0.75);
    T v[2][2];  // [plane][even, odd]
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      T a[3], b[3];
#pragma unroll
      for (int ii = 0; ii < 3; ++ii) {
        a[ii] = C[Ka + kk][Ja][t.i2 + ii];
        b[ii] = C[Ka + kk][Ja + 1][t.i2 + ii];
      }
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const T tx = e ? T(0.25) : T(0.75);
        const T v00 = (T(1) - tx) * a[e] + tx * a[e + 1], v10 = (T(1) - tx) * b[e] + tx * b[e + 1];
        v[kk][e] = (T(1) - ty) * v00 + ty * v10;
      }
    }
    xe[m] += (T(1) - tz) * v[0][0] + tz * v[1][0];
    xo[m] += (T(1) - tz) * v[0][1] + tz * v[1][1];
    const bool swap = ((t.q.side > 0) ^ (m & 1)) != 0;
    t.q.x[0][m] = swap ? xo[m] : xe[m];
    t.q.x[1][m] = swap ? xe[m] : xo[m];
    X[t.q.at + m * kT3Sz] = t.q.x[0][m];
    X[t.q.at + kT3Xc + m * kT3Sz] = t.q.x[1][m];
  }
  __syncthreads();
  block_sweeps<T, 3, 4, 1>(t.q, true, X, kT3Sz, kT3Sx, kT3Xc, nu2, false);
  tile3_store(F, t, out);
}

}  // namespace scihpc
