// mg_block.hpp -- the coarse levels of a V-cycle in one workgroup.
//
// From the first level that fits (scihpc_mg::block_level) a single
// workgroup (512 or 1024 threads) runs the whole remaining V-cycle: sweeps, residual,
// child average, dense coarsest solve, prolongation, sweeps.  Included by
// mg.hip (DLevel, smooth_rcp, interp_axis come from there).
//
// What bounds it is not bytes (under 0.3 MB) but the chain of about ten
// barrier-separated phases a level and the one round trip to memory at its
// start, so every phase is made short:
//  * cells are owned in pairs (2 m, 2 m + 1) of a row, one red and one
//    black; a thread keeps the P pairs it owns on the top level (rows one
//    above the other) for the whole cycle in registers: face coefficients,
//    right-hand sides, diagonals, their reciprocals and the iterate.  A
//    neighbour inside the thread's own patch costs nothing; a colour update
//    reads P + 2 values from LDS instead of 4 P, and writes P;
//  * red and black values have an LDS array each, so the lanes of a
//    wavefront read consecutive words (interleaved they would hit every
//    second bank);
//  * iterates carry a halo of zeros and a coefficient toward a wall is 0, so
//    no update tests for walls; a cell that does not exist (odd sizes) has a
//    record of zeros and stays 0;
//  * the levels below the top need one pair a thread.  Their coefficients
//    are packed in thread order behind the level descriptions in one device
//    buffer (k_block_pack, after the operator changes), which is copied into
//    LDS as it is: one batch of loads, in flight with the top level's;
//  * the coarsest right-hand side is multiplied by the transposed inverse
//    (coalesced, two rows a thread, columns split over up to 16 threads a
//    row, loaded at the start when it is small), with the mean removal of
//    the all-Neumann problem folded into the matrix.
// Measured on MI355X, per cycle, against the phase loop over LDS-resident
// coefficients it replaces (2.4 GHz cycle counter): 64 x 128 bubble, FP32
// levels 32 x 64 .. 4 x 8, 22.1 -> 10.5 us; 512 x 1024 bubble, FP32, 23.5 us
// for 32 x 64 .. plus 13 us for the 64 x 128 level's two tiled launches and
// their gaps -> 19.2 us for 64 x 128 .. 4 x 8; 256^2 Dirichlet, FP64 levels
// 64^2 .. 4^2, 37.7 -> 15.2 us; 128^3, FP64, 16^3 .. 4^3 in 18.4 us (8^3 ..
// took 14.3 us and the 16^3 level's six launches 75 us).  What is left: about
// 2 us of memory latency at the start, 2 us a level of dependent LDS phases,
// and a large coarsest matrix (375 unknowns: 12 us, one CU's load rate).
#pragma once

namespace scihpc {

constexpr int kMaxBlockLevels = 12;
constexpr int kBlockSplit = 16;  // most threads that share a row pair of the coarsest product
constexpr int kBlockEarly = 2;  // columns a thread may load at the start

// one level as the kernel sees it; offsets are LDS elements of T.  Cell
// (i, j, k) lies in the array of its colour (i + j + k) & 1 at
// (i >> 1) + 1 + sx (j + 1) (+ sz (k + 1)).
template <typename T>
struct alignas(16) BlockGeo {
  int nx, ny, nz, hx;  // hx: pairs a row
  int pairs;           // hx * ny * nz
  int n, ratio;        // cells; coarsening ratio to the next level
  int sx, sz, xc;      // row and plane stride of a colour array, and its size
  int xo;              // iterate: red, black
  int co;              // records (block_fields each), field by field
  int bo;              // right-hand sides: red, black, `pairs` each
  float ihx, iny;      // 1 / hx, 1 / ny
  int spare;
};
static_assert(sizeof(BlockGeo<float>) == 64 && sizeof(BlockGeo<double>) == 64, "packed as int4");

// partner, then per colour: side, down, up(, back, front), diagonal
template <int DIM>
constexpr int block_fields() {
  return 1 + 2 * (DIM == 3 ? 6 : 4);
}

typedef int BlockWords __attribute__((ext_vector_type(4)));

template <typename T>
struct BlockArgs {
  BlockGeo<T> top;
  const T *cx, *cy, *cz;   // top level (nullptr: constant coefficients)
  const T *rhs, *sol_in;
  T *sol_out;
  const BlockWords *pack;  // level descriptions and records, as in LDS
  const double *Mt;
  int pack16, xo16, xn16;  // in 16 bytes: the pack; where the iterates start; their size
  int nlev, dir, nu1, nu2, zero_top;
  int ro;                  // residuals of the even and odd cells of pairs
  int dense;               // byte offset of the coarsest right-hand side and partial sums
  int nc, ld, split, per;  // coarsest unknowns, row stride of Mt, threads and columns a row pair
  // constant-coefficient operator of the top level
  T ax, ay, az, dconst, wx, wy, wz;
  int dirichlet, rbwall;
};

template <typename T, int DIM>
struct BlockRec {  // one pair, [colour: red, black]
  T wp;            // partner
  T ws[2], wd[2], wu[2], wb[DIM == 3 ? 2 : 1], wf[DIM == 3 ? 2 : 1], d[2];
};

// the record of pair (i2, j, k) of a level from its global face arrays (or
// constant coefficients), the diagonal summed in stencil<>'s order; `b`: the
// pair's right-hand sides by colour
template <typename T, int DIM, typename L>
__device__ __forceinline__ BlockRec<T, DIM> block_record(const L &g, const T *__restrict__ cx,
                                                         const T *__restrict__ cy, const T *__restrict__ cz, int i2,
                                                         int j, int k, const T (&below)[2], T (&above)[2]) {
  BlockRec<T, DIM> q;
  const int i = 2 * i2, c = i + g.nx * (j + g.ny * k);
  const bool odd = i + 1 < g.nx, hl = i > 0, hu = j < g.ny - 1;
  const bool hr = i + 2 < g.nx;
  T w[2][6], d[2];  // [even, odd][left, right, down, up, back, front]
  if (cx) {
    const T ce = cx[c], co = odd ? cx[c + 1] : T(0), cl = hl ? cx[c - 1] : T(0);
    above[0] = cy[c];
    above[1] = odd ? cy[c + 1] : T(0);
    w[0][0] = cl;
    w[0][1] = odd ? ce : T(0);
    w[1][0] = odd ? ce : T(0);
    w[1][1] = hr ? co : T(0);
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      w[e][2] = below[e];
      w[e][3] = hu ? above[e] : T(0);
      d[e] = -((e ? co : ce) + w[e][0] + above[e] + w[e][2]);
    }
    if constexpr (DIM == 3) {
      const int sz = g.nx * g.ny;
      const bool hb = k > 0, hf = k < g.nz - 1;
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const bool in = e == 0 || odd;
        const T cF = in ? cz[c + e] : T(0);
        w[e][4] = in && hb ? cz[c + e - sz] : T(0);
        w[e][5] = hf ? cF : T(0);
        d[e] -= (cF + w[e][4]);
      }
    }
  } else {
    const T wx = g.rbwall ? g.wx : T(0), wy = g.rbwall ? g.wy : T(0);
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const bool l = e ? true : hl, r = e ? hr : odd, dn = j > 0;
      w[e][0] = l ? g.ax : T(0);
      w[e][1] = r ? g.ax : T(0);
      w[e][2] = dn ? g.ay : T(0);
      w[e][3] = hu ? g.ay : T(0);
      T cc = T(0);
      cc += l ? g.ax : wx;
      cc += r ? g.ax : wx;
      cc += dn ? g.ay : wy;
      cc += hu ? g.ay : wy;
      if constexpr (DIM == 3) {
        const T wz = g.rbwall ? g.wz : T(0);
        const bool hb = k > 0, hf = k < g.nz - 1;
        w[e][4] = hb ? g.az : T(0);
        w[e][5] = hf ? g.az : T(0);
        cc += hb ? g.az : wz;
        cc += hf ? g.az : wz;
      }
      d[e] = (g.dirichlet && !g.rbwall) ? g.dconst : -cc;
    }
    above[0] = above[1] = hu ? g.ay : T(0);
  }
  if (!odd) {
#pragma unroll
    for (int f = 0; f < (DIM == 3 ? 6 : 4); ++f) w[1][f] = T(0);
    d[1] = T(0);
  }
  const int par = (j + k) & 1;  // 1: the odd cell is the red one
  q.wp = w[0][1];
#pragma unroll
  for (int col = 0; col < 2; ++col) {
    const bool o = (par ^ col) != 0;  // the odd cell
    q.ws[col] = o ? w[1][1] : w[0][0];
    q.wd[col] = o ? w[1][2] : w[0][2];
    q.wu[col] = o ? w[1][3] : w[0][3];
    if constexpr (DIM == 3) {
      q.wb[col] = o ? w[1][4] : w[0][4];
      q.wf[col] = o ? w[1][5] : w[0][5];
    }
    q.d[col] = o ? d[1] : d[0];
  }
  return q;
}

// records of a level below the top, field by field in pair order
template <typename T, int DIM>
__global__ void __launch_bounds__(kBlock) k_block_pack(DLevel<T> g, int hx, int pairs, T *__restrict__ out) {
  const int t = blockIdx.x * kBlock + threadIdx.x;
  if (t >= pairs) return;
  const int r = t / hx, i2 = t - r * hx, k = DIM == 3 ? r / g.ny : 0, j = r - k * g.ny;
  T below[2] = {T(0), T(0)}, above[2];
  if (g.cx && j > 0) {
    const int c = 2 * i2 + g.nx * (j - 1 + g.ny * k);
    below[0] = g.cy[c];
    below[1] = 2 * i2 + 1 < g.nx ? g.cy[c + 1] : T(0);
  }
  const BlockRec<T, DIM> q = block_record<T, DIM>(g, g.cx, g.cy, g.cz, i2, j, k, below, above);
  T *p = out + t;
  *p = q.wp;
#pragma unroll
  for (int col = 0; col < 2; ++col) {
    *(p += pairs) = q.ws[col];
    *(p += pairs) = q.wd[col];
    *(p += pairs) = q.wu[col];
    if constexpr (DIM == 3) {
      *(p += pairs) = q.wb[col];
      *(p += pairs) = q.wf[col];
    }
    *(p += pairs) = q.d[col];
  }
}

// the P pairs a thread owns on one level, rows j .. j + P - 1 of column i2
template <typename T, int DIM, int P>
struct BlockPatch {
  T wp[P], ws[2][P], wv[2][P + 1];  // wv[col][m]: face below cell (col, m); [col][P]: above cell (1 - col, P - 1)
  T wb[2][DIM == 3 ? P : 1], wf[2][DIM == 3 ? P : 1];
  T d[2][P], rd[2][P], b[2][P], x[2][P];
  int at;    // LDS index of row j in the red array of the iterate
  int side;  // where the red cell of row 0 has its side neighbour: -1 or +1
};

template <typename T>
__device__ __forceinline__ T block_rcp(T d) {
  return d != T(0) ? smooth_rcp<T>(d) : T(0);  // 0: no such cell
}

template <typename T, int DIM, int P>
__device__ __forceinline__ T block_off(const BlockPatch<T, DIM, P> &q, int col, int m, const T *__restrict__ X, int sx,
                                       int sz) {
  // X: the other colour's array at `at`
  const int s = ((m ^ col) & 1) ? -q.side : q.side;
  T o = q.ws[col][m] * X[m * sx + s];
  o += q.wp[m] * q.x[1 - col][m];
  o += q.wv[col][m] * (m == 0 ? X[-sx] : q.x[1 - col][m > 0 ? m - 1 : 0]);
  o += q.wv[1 - col][m + 1] * (m == P - 1 ? X[P * sx] : q.x[1 - col][m < P - 1 ? m + 1 : m]);
  if constexpr (DIM == 3) {
    o += q.wb[col][m] * X[m * sx - sz];
    o += q.wf[col][m] * X[m * sx + sz];
  }
  return o;
}

// one colour: x = (b - off) / d, the quotient as gs_div forms it
template <typename T, int DIM, int P, int COL>
__device__ __forceinline__ void block_pass(BlockPatch<T, DIM, P> &q, T *X, int sx, int sz, int xc, bool zero) {
  T *own = X + COL * xc + q.at;
  const T *other = X + (1 - COL) * xc + q.at;
#pragma unroll
  for (int m = 0; m < P; ++m) {
    T a = q.b[COL][m];
    if (!zero) a -= block_off<T, DIM, P>(q, COL, m, other, sx, sz);
    T v = a * q.rd[COL][m];
    if constexpr (sizeof(T) == 8) v = __builtin_fma(__builtin_fma(-q.d[COL][m], v, a), q.rd[COL][m], v);
    q.x[COL][m] = v;
  }
#pragma unroll
  for (int m = 0; m < P; ++m) own[m * sx] = q.x[COL][m];
}

// nu sweeps, colour FIRST first; zero: the iterate is zero before them.
// on: the thread owns cells here.
template <typename T, int DIM, int P, int FIRST>
__device__ __forceinline__ void block_sweeps(BlockPatch<T, DIM, P> &q, bool on, T *X, int sx, int sz, int xc, int nu,
                                             bool zero) {
  for (int s = 0; s < nu; ++s) {
    if (on) block_pass<T, DIM, P, FIRST>(q, X, sx, sz, xc, zero && s == 0);
    __syncthreads();
    if (on) block_pass<T, DIM, P, 1 - FIRST>(q, X, sx, sz, xc, false);
    __syncthreads();
  }
}

// residuals of the pairs: ratio 2 stores the sum of a pair (its cells are
// children of one coarse cell) in R, other ratios even and odd cells apart.
// t: pair index of row 0 (+ hx a row); rows past ny are not stored.
template <typename T, int DIM, int P>
__device__ __forceinline__ void block_residual(const BlockPatch<T, DIM, P> &q, const T *X, T *R, int sx, int sz, int xc,
                                               int t, int hx, int pairs, int rows, bool two) {
#pragma unroll
  for (int m = 0; m < P; ++m) {
    T r[2];
#pragma unroll
    for (int col = 0; col < 2; ++col)
      r[col] = q.b[col][m] -
               (block_off<T, DIM, P>(q, col, m, X + (1 - col) * xc + q.at, sx, sz) + q.d[col][m] * q.x[col][m]);
    if (m >= rows) break;
    if (two) {
      R[t + m * hx] = r[0] + r[1];
    } else {
      const bool swap = ((q.side > 0) ^ (m & 1)) != 0;  // the odd cell is the red one
      R[t + m * hx] = swap ? r[1] : r[0];
      R[t + m * hx + pairs] = swap ? r[0] : r[1];
    }
  }
}

// mean over the ratio^DIM children of coarse cell (I, J, K) of the finer
// level F's residuals
template <typename T, int DIM>
__device__ __forceinline__ T block_child_mean(const BlockGeo<T> &F, const T *R, int I, int J, int K) {
  T s = T(0);
  if (F.ratio == 2) {
    const T *p = R + I + F.hx * (2 * J + (DIM == 3 ? F.ny * 2 * K : 0));
    s = p[0] + p[F.hx];
    if constexpr (DIM == 3) {
      const int z = F.hx * F.ny;
      s += p[z] + p[z + F.hx];
    }
    return s * T(DIM == 3 ? 0.125 : 0.25);
  }
#pragma unroll
  for (int kk = 0; kk < (DIM == 3 ? 3 : 1); ++kk)
#pragma unroll
    for (int jj = 0; jj < 3; ++jj)
#pragma unroll
      for (int ii = 0; ii < 3; ++ii) {
        const int i = I * 3 + ii;
        s += R[(i & 1) * F.pairs + (i >> 1) + F.hx * (J * 3 + jj + (DIM == 3 ? F.ny * (K * 3 + kk) : 0))];
      }
  return s / T(DIM == 3 ? 27 : 9);
}

// The iterate X of level G at cell (I, J, K), halo included (both colours are 0 there).
template <typename T, int DIM>
__device__ __forceinline__ T block_at(const BlockGeo<T> &G, const T *X, int I, int J, int K) {
  return X[((I + J + K) & 1) * G.xc + (I >> 1) + 1 + G.sx * (J + 1) + (DIM == 3 ? G.sz * (K + 1) : 0)];
}

// prolong_cell's increments for factor-2 coarsening of pair (i2, j, k), even
// and odd cell, from the coarse iterate X of level G
template <typename T, int DIM>
__device__ __forceinline__ void block_interp2(const BlockGeo<T> &G, const T *X, int dir, int i2, int j, int k,
                                              T (&v)[2]) {
  // the ghost of a Dirichlet wall is the halo's 0, of a Neumann wall the nearest cell
  const int lo = dir ? -1 : 0, hi = dir ? 0 : -1;
  const int I[3] = {max(i2 - 1, lo), i2, min(i2 + 1, G.nx + hi)};
  const int J0 = (j - 1) >> 1, Ja = max(J0, lo), Jb = min(J0 + 1, G.ny + hi);
  const T ty = (j & 1) ? T(0.25) : T(0.75);
  const auto plane = [&](int K, T (&o)[2]) {
    T a[3], b[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      a[q] = block_at<T, DIM>(G, X, I[q], Ja, K);
      b[q] = block_at<T, DIM>(G, X, I[q], Jb, K);
    }
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const T tx = e ? T(0.25) : T(0.75);
      const T v00 = (T(1) - tx) * a[e] + tx * a[e + 1], v10 = (T(1) - tx) * b[e] + tx * b[e + 1];
      o[e] = (T(1) - ty) * v00 + ty * v10;
    }
  };
  if constexpr (DIM == 2) {
    plane(0, v);
  } else {
    const int K0 = (k - 1) >> 1;
    const T tz = (k & 1) ? T(0.25) : T(0.75);
    T a[2], b[2];
    plane(max(K0, lo), a);
    plane(min(K0 + 1, G.nz + hi), b);
#pragma unroll
    for (int e = 0; e < 2; ++e) v[e] = (T(1) - tz) * a[e] + tz * b[e];
  }
}

// interp_axis for ratio 3 without divisions: coarse index (2 i - 2) / 6
// rounded down, and the weight of the next one
template <typename T>
__device__ __forceinline__ void block_axis3(int i, int &I0, T &t) {
  const unsigned m = (unsigned)i + 2, q = m / 3;
  const unsigned rem = m - 3 * q;
  I0 = (int)q - 1;
  t = rem == 0 ? T(0) : rem == 1 ? T(2.0 / 6.0) : T(4.0 / 6.0);
}

// prolong_cell's increment of cell (i, j, k) for factor-3 coarsening
template <typename T, int DIM>
__device__ __forceinline__ T block_interp3(const BlockGeo<T> &G, const T *X, int dir, int i, int j, int k) {
  const int lo = dir ? -1 : 0, hi = dir ? 0 : -1;
  int I0, J0, K0 = 0;
  T tx, ty, tz = T(0);
  block_axis3<T>(i, I0, tx);
  block_axis3<T>(j, J0, ty);
  if (DIM == 3) block_axis3<T>(k, K0, tz);
  const int Ia = max(I0, lo), Ib = min(I0 + 1, G.nx + hi), Ja = max(J0, lo), Jb = min(J0 + 1, G.ny + hi);
  const auto plane = [&](int K) {
    const T v00 = (T(1) - tx) * block_at<T, DIM>(G, X, Ia, Ja, K) + tx * block_at<T, DIM>(G, X, Ib, Ja, K);
    const T v10 = (T(1) - tx) * block_at<T, DIM>(G, X, Ia, Jb, K) + tx * block_at<T, DIM>(G, X, Ib, Jb, K);
    return (T(1) - ty) * v00 + ty * v10;
  };
  if constexpr (DIM == 2) return plane(0);
  else return (T(1) - tz) * plane(max(K0, lo)) + tz * plane(min(K0 + 1, G.nz + hi));
}

// the coarse correction added to a patch (rows rows of P), in registers and LDS
template <typename T, int DIM, int P>
__device__ __forceinline__ void block_prolong(BlockPatch<T, DIM, P> &q, const BlockGeo<T> &g, const BlockGeo<T> &G,
                                              T *smem, int dir, int i2, int j, int k, int rows) {
  const T *X = smem + G.xo;
  if (g.ratio == 2) {
#pragma unroll
    for (int m = 0; m < P; ++m) {
      if (m >= rows) break;
      T v[2];
      block_interp2<T, DIM>(G, X, dir, i2, j + m, k, v);
      const bool swap = ((q.side > 0) ^ (m & 1)) != 0;  // the odd cell is the red one
      q.x[0][m] += swap ? v[1] : v[0];
      q.x[1][m] += swap ? v[0] : v[1];
      smem[q.at + m * g.sx] = q.x[0][m];
      smem[q.at + g.xc + m * g.sx] = q.x[1][m];
    }
    return;
  }
  // ratio 3: added in LDS by a rolled loop (short code, rarely taken)
#pragma unroll 1
  for (int c = 0; c < 2 * rows; ++c) {
    const int m = c >> 1, i = 2 * i2 + (c & 1);
    if (i < g.nx)
      smem[q.at + ((i + j + m + k) & 1) * g.xc + m * g.sx] +=
          block_interp3<T, DIM>(G, X, dir, i, j + m, k);
  }
#pragma unroll
  for (int m = 0; m < P; ++m) {
    q.x[0][m] = smem[q.at + m * g.sx];
    q.x[1][m] = smem[q.at + g.xc + m * g.sx];
  }
}

// wave-uniform copy of a level's description out of LDS
template <typename T>
__device__ __forceinline__ BlockGeo<T> block_geo(const BlockWords *s, int l) {
  union {
    BlockGeo<T> g;
    int w[16];
  } u;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const BlockWords v = s[4 * l + q];
    u.w[4 * q] = __builtin_amdgcn_readfirstlane(v.x);
    u.w[4 * q + 1] = __builtin_amdgcn_readfirstlane(v.y);
    u.w[4 * q + 2] = __builtin_amdgcn_readfirstlane(v.z);
    u.w[4 * q + 3] = __builtin_amdgcn_readfirstlane(v.w);
  }
  return u.g;
}

// row r of a level's pairs is t / hx by a float reciprocal: exact for
// t < 2^20 (the half-integer offset keeps the quotient away from integers)
__device__ __forceinline__ int block_div(int t, float inv) { return (int)((float(t) + 0.5f) * inv); }

// NT: workgroup size, a constant so that no loop reads it from the dispatch
// packet.  2-D: 512 threads while they hold the top level in patches of one
// row (a barrier is cheaper), else 1024 with patches of up to four rows
// (FP32 64 x 128) or two (FP64 64 x 64: 36.4 k cycles, 39.8 k with 512
// threads).  3-D: 512 threads and patches of up to four rows, as their 256
// registers hold the FP64 patch (16^3: 44 k cycles; at 1024 threads it
// spilled inside the sweeps, 104 k).
template <typename T, int DIM, int P, int NT>
__global__ void __launch_bounds__(NT) k_block_vcycle(const BlockArgs<T> B) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T *const smem = reinterpret_cast<T *>(smem_raw);
  BlockWords *const smem16 = reinterpret_cast<BlockWords *>(smem_raw);
  const int tid = threadIdx.x, L = B.nlev;
  const BlockGeo<T> &g0 = B.top;

  // ---- staging: every global load is issued before the first is needed.
  // The pack, 16 bytes a load, up to kPk a thread at once
  constexpr int kPk = 4096 / NT;
  BlockWords pk[kPk];
#pragma unroll
  for (int h = 0; h < kPk; ++h) {
    const int t = tid + h * NT;
    pk[h] = t < B.pack16 ? B.pack[t] : BlockWords{0, 0, 0, 0};
  }
  // the top level's patch
  BlockPatch<T, DIM, P> q;
  const int nyp = (g0.ny + P - 1) / P;
  int i2 = 0, j = 0, k = 0, rows = 0;
  {
    const int r = block_div(tid, g0.ihx);
    i2 = tid - r * g0.hx;
    k = DIM == 3 ? block_div(r, P == 1 ? g0.iny : 1.0f / float(nyp)) : 0;
    j = (r - k * nyp) * P;
    if (L > 1 && k < g0.nz) rows = max(0, min(P, g0.ny - j));
  }
  const bool on = rows > 0;
  const int t0 = i2 + g0.hx * (j + g0.ny * k);
  q.at = g0.xo + i2 + 1 + g0.sx * (j + 1) + (DIM == 3 ? g0.sz * (k + 1) : 0);
  q.side = ((j + k) & 1) ? 1 : -1;
  {
    T below[2] = {T(0), T(0)}, above[2] = {T(0), T(0)};
    if (on && B.cx && j > 0) {
      const int c = 2 * i2 + g0.nx * (j - 1 + g0.ny * k);
      below[0] = B.cy[c];
      below[1] = 2 * i2 + 1 < g0.nx ? B.cy[c + 1] : T(0);
    }
    struct {
      int nx, ny, nz, dirichlet, rbwall;
      T ax, ay, az, dconst, wx, wy, wz;
    } lv = {g0.nx, g0.ny, g0.nz, B.dirichlet, B.rbwall, B.ax, B.ay, B.az, B.dconst, B.wx, B.wy, B.wz};
#pragma unroll
    for (int m = 0; m < P; ++m) {
      BlockRec<T, DIM> rec = {};
      T be = T(0), bo = T(0), xe = T(0), xo = T(0);
      if (m < rows) {
        const int c = 2 * i2 + g0.nx * (j + m + g0.ny * k);
        const bool odd = 2 * i2 + 1 < g0.nx;
        be = B.rhs[c];
        bo = odd ? B.rhs[c + 1] : T(0);
        if (!B.zero_top) {
          xe = B.sol_in[c];
          xo = odd ? B.sol_in[c + 1] : T(0);
        }
        rec = block_record<T, DIM>(lv, B.cx, B.cy, B.cz, i2, j + m, k, below, above);
        if (!B.cx) above[0] = above[1] = T(0);
        below[0] = above[0];
        below[1] = above[1];
      }
      const bool swap = ((q.side > 0) ^ (m & 1)) != 0;  // the odd cell is the red one
      q.b[0][m] = swap ? bo : be;
      q.b[1][m] = swap ? be : bo;
      q.x[0][m] = swap ? xo : xe;
      q.x[1][m] = swap ? xe : xo;
      q.wp[m] = rec.wp;
#pragma unroll
      for (int col = 0; col < 2; ++col) {
        q.ws[col][m] = rec.ws[col];
        q.wv[col][m] = rec.wd[col];
        if (m == P - 1) q.wv[1 - col][P] = rec.wu[col];
        if constexpr (DIM == 3) {
          q.wb[col][m] = rec.wb[col];
          q.wf[col][m] = rec.wf[col];
        }
        q.d[col][m] = rec.d[col];
        q.rd[col][m] = block_rcp(rec.d[col]);
      }
    }
  }
  // a small coarsest matrix
  const int nrp = (B.nc + 1) >> 1;                      // row pairs
  const int ds = tid / nrp, dr = (tid - ds * nrp) * 2;  // this thread's columns and rows
  const bool early = B.per <= kBlockEarly && ds < B.split;
  double2 mt[kBlockEarly];
#pragma unroll
  for (int h = 0; h < kBlockEarly; ++h) {
    const int c = ds * B.per + h;
    mt[h] = early && h < B.per && c < B.nc ? *reinterpret_cast<const double2 *>(B.Mt + (long)c * B.ld + dr)
                                           : make_double2(0.0, 0.0);
  }
  // iterates: zero (halos included); then what was loaded
  for (int t = tid; t < B.xn16; t += NT) smem16[B.xo16 + t] = BlockWords{0, 0, 0, 0};
#pragma unroll
  for (int h = 0; h < kPk; ++h)
    if (tid + h * NT < B.pack16) smem16[tid + h * NT] = pk[h];
  for (int t = tid + kPk * NT; t < B.pack16; t += NT) smem16[t] = B.pack[t];
  T *const R = smem + B.ro;
  __syncthreads();

  // ---- down
  if (L > 1) {
    if (!B.zero_top) {
      if (on) {
#pragma unroll
        for (int m = 0; m < P; ++m) {
          smem[q.at + m * g0.sx] = q.x[0][m];
          smem[q.at + g0.xc + m * g0.sx] = q.x[1][m];
        }
      }
      __syncthreads();
    }
    block_sweeps<T, DIM, P, 0>(q, on, smem, g0.sx, g0.sz, g0.xc, B.nu1, B.zero_top != 0);
    if (on)
      block_residual<T, DIM, P>(q, smem, R, g0.sx, g0.sz, g0.xc, t0, g0.hx, g0.pairs, rows, g0.ratio == 2);
    __syncthreads();
  }
  // the pair `tid` of level g: its record and where it lies
  const auto load_pair = [&](const BlockGeo<T> &g, BlockPatch<T, DIM, 1> &p, int &pi, int &pj, int &pk_) {
    const int r = block_div(tid, g.ihx);
    pi = tid - r * g.hx;
    pk_ = DIM == 3 ? block_div(r, g.iny) : 0;
    pj = r - pk_ * g.ny;
    p.at = g.xo + pi + 1 + g.sx * (pj + 1) + (DIM == 3 ? g.sz * (pk_ + 1) : 0);
    p.side = ((pj + pk_) & 1) ? 1 : -1;
    const T *f = smem + g.co + tid;
    p.wp[0] = *f;
#pragma unroll
    for (int col = 0; col < 2; ++col) {
      p.ws[col][0] = *(f += g.pairs);
      p.wv[col][0] = *(f += g.pairs);
      p.wv[1 - col][1] = *(f += g.pairs);
      if constexpr (DIM == 3) {
        p.wb[col][0] = *(f += g.pairs);
        p.wf[col][0] = *(f += g.pairs);
      }
      p.d[col][0] = *(f += g.pairs);
    }
    p.rd[0][0] = block_rcp(p.d[0][0]);
    p.rd[1][0] = block_rcp(p.d[1][0]);
  };
  for (int l = 1; l < L - 1; ++l) {
    const BlockGeo<T> F = block_geo<T>(smem16, l - 1), g = block_geo<T>(smem16, l);
    BlockPatch<T, DIM, 1> p;
    const bool pon = tid < g.pairs;
    if (pon) {
      int pi, pj, pk_;
      load_pair(g, p, pi, pj, pk_);
      const T be = block_child_mean<T, DIM>(F, R, 2 * pi, pj, pk_);
      const T bo = 2 * pi + 1 < g.nx ? block_child_mean<T, DIM>(F, R, 2 * pi + 1, pj, pk_) : T(0);
      p.b[0][0] = p.side > 0 ? bo : be;
      p.b[1][0] = p.side > 0 ? be : bo;
      p.x[0][0] = p.x[1][0] = T(0);
      smem[g.bo + tid] = p.b[0][0];
      smem[g.bo + g.pairs + tid] = p.b[1][0];
    }
    if (B.nu1 == 0) __syncthreads();  // R is read above and written below
    block_sweeps<T, DIM, 1, 0>(p, pon, smem, g.sx, g.sz, g.xc, B.nu1, true);
    if (pon)
      block_residual<T, DIM, 1>(p, smem, R, g.sx, g.sz, g.xc, tid, g.hx, g.pairs, 1, g.ratio == 2);
    __syncthreads();
  }

  // ---- dense coarsest solve, FP64: x = Mt^T b, two rows a thread, the
  // columns of a row pair over `split` threads, their sums added in order
  {
    const BlockGeo<T> g = block_geo<T>(smem16, L - 1);
    const int n = B.nc;
    constexpr int kFly = NT == 1024 ? 6 : DIM == 3 && sizeof(T) == 8 ? 8 : 16;  // loads in flight a thread (registers: the top level's patch stays live)
    double *const bs = reinterpret_cast<double *>(smem_raw + B.dense);
    double *const part = bs + 2 * nrp;
    for (int c = tid; c < n; c += NT) {
      int I, J, K;
      cell_ijk(c, g.nx, g.ny, I, J, K);
      bs[c] = L > 1 ? double(block_child_mean<T, DIM>(block_geo<T>(smem16, L - 2), R, I, J, K)) : double(B.rhs[c]);
    }
    __syncthreads();
    if (B.per <= kBlockEarly) {
      if (ds < B.split) {
        double a0 = 0.0, a1 = 0.0;
#pragma unroll
        for (int h = 0; h < kBlockEarly; ++h) {
          const double b = bs[min(ds * B.per + h, n - 1)];
          a0 = __builtin_fma(mt[h].x, b, a0);
          a1 = __builtin_fma(mt[h].y, b, a1);
        }
        part[ds * 2 * nrp + dr] = a0;
        part[ds * 2 * nrp + dr + 1] = a1;
      }
    } else {
      for (int u = tid; u < nrp * B.split; u += NT) {
        const int us = u / nrp, ur = (u - us * nrp) * 2;
        const int c1 = min(n, (us + 1) * B.per);
        const double *m = B.Mt + ur;
        double a0 = 0.0, a1 = 0.0;
        for (int c = us * B.per; c < c1; c += kFly) {
          double2 v[kFly];
#pragma unroll
          for (int h = 0; h < kFly; ++h)
            v[h] = c + h < c1 ? *reinterpret_cast<const double2 *>(m + (long)(c + h) * B.ld) : make_double2(0.0, 0.0);
#pragma unroll
          for (int h = 0; h < kFly; ++h) {
            const double b = bs[min(c + h, n - 1)];
            a0 = __builtin_fma(v[h].x, b, a0);
            a1 = __builtin_fma(v[h].y, b, a1);
          }
        }
        part[us * 2 * nrp + ur] = a0;
        part[us * 2 * nrp + ur + 1] = a1;
      }
    }
    __syncthreads();
    for (int c = tid; c < n; c += NT) {
      int I, J, K;
      cell_ijk(c, g.nx, g.ny, I, J, K);
      double x = part[c];
      for (int s = 1; s < B.split; ++s) x += part[c + s * 2 * nrp];
      if (L > 1)
        smem[g.xo + ((I + J + K) & 1) * g.xc + (I >> 1) + 1 + g.sx * (J + 1) + (DIM == 3 ? g.sz * (K + 1) : 0)] = T(x);
      else
        B.sol_out[c] = T(x);
    }
    __syncthreads();
  }

  // ---- up
  for (int l = L - 2; l > 0; --l) {
    const BlockGeo<T> g = block_geo<T>(smem16, l), G = block_geo<T>(smem16, l + 1);
    BlockPatch<T, DIM, 1> p;
    const bool pon = tid < g.pairs;
    if (pon) {
      int pi, pj, pk_;
      load_pair(g, p, pi, pj, pk_);
      p.b[0][0] = smem[g.bo + tid];
      p.b[1][0] = smem[g.bo + g.pairs + tid];
      p.x[0][0] = smem[p.at];
      p.x[1][0] = smem[p.at + g.xc];
      block_prolong<T, DIM, 1>(p, g, G, smem, B.dir, pi, pj, pk_, 1);
    }
    __syncthreads();
    block_sweeps<T, DIM, 1, 1>(p, pon, smem, g.sx, g.sz, g.xc, B.nu2, false);
  }
  if (L > 1) {
    const BlockGeo<T> G = block_geo<T>(smem16, 1);
    if (on) block_prolong<T, DIM, P>(q, g0, G, smem, B.dir, i2, j, k, rows);
    __syncthreads();
    block_sweeps<T, DIM, P, 1>(q, on, smem, g0.sx, g0.sz, g0.xc, B.nu2, false);
#pragma unroll
    for (int m = 0; m < P; ++m) {
      if (m >= rows) break;
      const int c = 2 * i2 + g0.nx * (j + m + g0.ny * k);
      const bool swap = ((q.side > 0) ^ (m & 1)) != 0;
      B.sol_out[c] = swap ? q.x[1][m] : q.x[0][m];
      if (2 * i2 + 1 < g0.nx) B.sol_out[c + 1] = swap ? q.x[0][m] : q.x[1][m];
    }
  }
}

}  // namespace scihpc
