// Geometric multigrid of libdec_hip.so (src/Multigrid.jl): the binary-
// subdivision hierarchy in DirectMode with op = fast_laplace_beltrami, and the
// μ-cycles / full multigrid / tolerance solves on the GPU.
//
// Per level the operator is held in slot-major ELL with rows sorted by
// (colour, vertex): a multicolour Gauss-Seidel pass over one colour is then a
// contiguous range of rows.  The same slots with rows in vertex order serve
// residuals and the CG smoother.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <memory>

#include "dec_internal.h"
#include "ell_rows.h"
#include "kernels_common.h"
#include "learned.h"

using dec::DBuf;
using dec::fail;
using dec::wave_sum;

namespace {

constexpr int kBlock = 256;
constexpr int kDotBlocks = 256;
constexpr int kNormSlots = 4;  // residual norms of a solve in flight (at most 2 are)

// ---------------------------------------------------------------- kernels

template <class T>
__global__ void k_zero(int n, T *__restrict__ x) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] = static_cast<T>(0);
}

// r[v] = b[v] - (A u)[v], row sums in ascending column order (b - A*u); the
// rows at ELL positions p are rowid[p] (rows in vertex order: rowid null).
template <int W, class T>
__global__ void k_residual(int n, int width, const int *__restrict__ col, const T *__restrict__ val,
                           const int *__restrict__ rowid, const T *__restrict__ b, const T *__restrict__ u,
                           T *__restrict__ r) {
  int p = dec_ell::xcd_block() * blockDim.x + threadIdx.x;
  if (p >= n) return;
  T acc = dec_ell::row<W, T, T>(n, width, p, col, val, u);
  int v = rowid ? rowid[p] : p;
  r[v] = b[v] - acc;
}

// The residual r = b - A u of k_residual (in float64, in float32 where a float32
// cycle takes it, or both) and, per workgroup, the sum of its
// rows' r² (a fixed tree) into part[blockIdx.x]; k_sum_rows adds the
// partial sums.  (A ticket letting the last workgroup add them needs a
// device-scope fence in every workgroup, which writes back the XCD's L2:
// measured six times slower.)
template <int W>
__global__ void __launch_bounds__(256)
    k_residual_norm(int n, int width, const int *__restrict__ col, const double *__restrict__ val,
                    const int *__restrict__ rowid, const double *__restrict__ b, const double *__restrict__ u,
                    double *__restrict__ r, float *__restrict__ rf, double *__restrict__ part) {
  __shared__ double sh[256];
  int p = blockIdx.x * blockDim.x + threadIdx.x;
  double rr = 0.0;
  if (p < n) {
    double acc = dec_ell::row<W, double, double>(n, width, p, col, val, u);
    int v = rowid ? rowid[p] : p;
    double ri = b[v] - acc;
    if (r) r[v] = ri;
    if (rf) rf[v] = static_cast<float>(ri);
    rr = ri * ri;
  }
  sh[threadIdx.x] = rr;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) sh[threadIdx.x] = sh[threadIdx.x] + sh[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}

// *out = Σ part[0..nb) in a fixed order: 256 consecutive runs, then a tree.
__global__ void __launch_bounds__(256) k_sum_rows(int nb, const double *__restrict__ part, double *__restrict__ out) {
  __shared__ double sh[256];
  int per = (nb + 255) / 256;
  double acc = 0.0;
  for (int j = threadIdx.x * per; j < min(nb, (static_cast<int>(threadIdx.x) + 1) * per); j++) acc = acc + part[j];
  sh[threadIdx.x] = acc;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) sh[threadIdx.x] = sh[threadIdx.x] + sh[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = sh[0];
}

// One colour of Gauss-Seidel: u[v] = (b[v] - Σ_{w≠v} A[v,w] u[w]) / A[v,v].
template <int W, class T>
__global__ void k_gs_color(int p0, int p1, int n, int width, const int *__restrict__ col,
                           const T *__restrict__ val, const int *__restrict__ rowid, const T *__restrict__ b,
                           T *__restrict__ u) {
  int p = p0 + dec_ell::xcd_block() * blockDim.x + threadIdx.x;
  if (p >= p1) return;
  int v = rowid[p];
  T s, d;
  dec_ell::gs_row<W, T>(n, width, p, v, col, val, u, s, d);
  u[v] = (b[v] - s) / d;
}

// Damped Jacobi: un[v] = u[v] + ω (b[v] - (A u)[v]) / A[v,v].
template <int W, class T>
__global__ void k_jacobi(int n, int width, const int *__restrict__ col, const T *__restrict__ val,
                         const int *__restrict__ rowid, const T *__restrict__ b, const T *__restrict__ u,
                         T *__restrict__ un, T omega) {
  int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  int v = rowid[p];
  T s, d;
  dec_ell::gs_row<W, T>(n, width, p, v, col, val, u, s, d);
  // (A u)[v] in ascending column order: the diagonal term enters at its place
  T full = dec_ell::row<W, T, T>(n, width, p, col, val, u);
  (void)s;
  un[v] = u[v] + omega * ((b[v] - full) / d);
}

template <class T>
__global__ void k_copy(int n, const T *__restrict__ x, T *__restrict__ y) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = x[i];
}

// b_c = R r_f; rows are coarse vertices in natural order (CSC order of R:
// the identity column first, then the midpoint columns ascending).
// uc (when given) is the coarse iterate, zeroed here for the coarse cycle.
template <int W, class T>
__global__ void k_restrict(int nc, int width, const int *__restrict__ col, const T *__restrict__ val,
                           const T *__restrict__ rf, T *__restrict__ bc, T *__restrict__ uc) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nc) return;
  bc[i] = dec_ell::row<W, T, T>(nc, width, i, col, val, rf);
  if (uc) uc[i] = static_cast<T>(0);
}

// k_residual and k_restrict in one launch for levels where launches, not
// bytes, bound the cycle.  Eight lanes per coarse row i: lane s evaluates
// r_j = b_j - (A u)_j for the row's slot s (j = R's column; the fine rows in
// vertex order, summed as k_residual does) and multiplies it by R's
// entry; lane 0 then adds the eight products in slot order, so b_c is
// bit-identical to the two launches.  Fine rows shared by two coarse rows are
// evaluated twice.  R's width is at most 8.
template <int W, class T>
__global__ void __launch_bounds__(256)
    k_residual_restrict(int nc, int rwidth, const int *__restrict__ rcol, const T *__restrict__ rval, int n,
                        int width, const int *__restrict__ col, const T *__restrict__ val, const T *__restrict__ b,
                        const T *__restrict__ u, T *__restrict__ bc, T *__restrict__ uc) {
  __shared__ T prod[256];
  int t = blockIdx.x * blockDim.x + threadIdx.x;
  int i = t >> 3, sl = t & 7;
  T pr = static_cast<T>(0);
  bool has = false;
  if (i < nc && sl < rwidth) {
    size_t q = static_cast<size_t>(sl) * nc + i;
    int j = rcol[q];
    if (j >= 0) {
      T rj = b[j] - dec_ell::row<W, T, T>(n, width, j, col, val, u);
      pr = rval[q] * rj;
      has = true;
    }
  }
  prod[threadIdx.x] = pr;
  unsigned long long m = __ballot(has);
  __syncthreads();
  if (sl == 0 && i < nc) {
    T acc = static_cast<T>(0);
    int base = threadIdx.x;
    unsigned lanebits = static_cast<unsigned>((m >> (threadIdx.x & 63)) & 0xffu);
    for (int k = 0; k < 8; k++)
      if (lanebits & (1u << k)) acc = acc + prod[base + k];
    bc[i] = acc;
    if (uc) uc[i] = static_cast<T>(0);
  }
}

// u_f += P z_c, P in ELL rows (for a binary subdivision P = transpose(S):
// a coarse vertex copies its value with weight 1, a midpoint takes 0.5 of its
// edge's endpoints in the order (min, max) of S's column).
template <int W, class T>
__global__ void k_prolong_add(int nf, int width, const int *__restrict__ pcol, const T *__restrict__ pval,
                              const T *__restrict__ zc, T *__restrict__ uf) {
  int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= nf) return;
  uf[j] = uf[j] + dec_ell::row<W, T, T>(nf, width, j, pcol, pval, zc);
}

// u[j], or with zc given u[j] + (P zc)[j] (P an ELL of width 2: the sum of
// k_prolong_add), for sweeps that apply the prolongation themselves.
template <class T>
__device__ __forceinline__ T prolonged(int n, int j, const T *__restrict__ u, const int *__restrict__ pcol,
                                       const T *__restrict__ pval, const T *__restrict__ zc) {
  return zc ? u[j] + dec_ell::row<2, T, T>(n, 2, j, pcol, pval, zc) : u[j];
}

// One hybrid block Gauss-Seidel sweep.  The level's vertices are numbered so
// that every block is a contiguous range [bstart[k], bstart[k+1]); the ELL rows
// are sorted by (colour, vertex), so the rows of colour c in block k are the
// positions [seg[c*(nb+1)+k], seg[c*(nb+1)+k+1]).  One workgroup per block
// stages the block's iterate in LDS and runs the colours in order (reversed
// for the post-smoother) with a barrier between colours; a neighbour in
// another block enters with its value in uin (the iterate at the start of the
// sweep).  The result goes to uout, so no workgroup reads a value another one
// writes in the same launch.  Per row: the sum over the off-diagonal entries
// in slot (ascending column) order, then (b - sum) / diagonal.
// For levels that the panel sweep below does not take (rows wider than 8 slots,
// many colours, one block of a whole level, blocks with very many neighbours).
template <int W, class T>
__global__ void __launch_bounds__(256)
    k_block_gs(int n, int width, int ncolors, int nb, const int *__restrict__ col, const T *__restrict__ val,
               const int *__restrict__ rowid, const int *__restrict__ bstart, const int *__restrict__ seg,
               const T *__restrict__ b, const T *__restrict__ uin, T *__restrict__ uout, int reverse) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T *x = reinterpret_cast<T *>(smem_raw);
  int k = blockIdx.x;
  int r0 = bstart[k], nr = bstart[k + 1] - r0;
  for (int i = threadIdx.x; i < nr; i += blockDim.x) x[i] = uin[r0 + i];
  __syncthreads();
  for (int ci = 0; ci < ncolors; ci++) {
    int c = reverse ? ncolors - 1 - ci : ci;
    int p0 = seg[c * (nb + 1) + k], p1 = seg[c * (nb + 1) + k + 1];
    for (int p = p0 + static_cast<int>(threadIdx.x); p < p1; p += blockDim.x) {
      int v = rowid[p];
      T s = static_cast<T>(0), d = static_cast<T>(0);
      if constexpr (W > 0) {
        int cc[W];
        T vv[W], xv[W];
#pragma unroll
        for (int q = 0; q < W; q++) {
          size_t o = static_cast<size_t>(q) * n + p;
          cc[q] = col[o];
          vv[q] = val[o];
        }
#pragma unroll
        for (int q = 0; q < W; q++) {
          unsigned loc = static_cast<unsigned>(cc[q] - r0);
          xv[q] = (cc[q] < 0 || loc < static_cast<unsigned>(nr)) ? static_cast<T>(0)
                                                                 : uin[cc[q]];
        }
#pragma unroll
        for (int q = 0; q < W; q++) {
          if (cc[q] < 0) continue;
          unsigned loc = static_cast<unsigned>(cc[q] - r0);
          if (cc[q] == v) d = vv[q];
          else s = s + vv[q] * (loc < static_cast<unsigned>(nr) ? x[loc] : xv[q]);
        }
      } else {
        for (int q = 0; q < width; q++) {
          size_t o = static_cast<size_t>(q) * n + p;
          int cq = col[o];
          if (cq < 0) break;
          unsigned loc = static_cast<unsigned>(cq - r0);
          if (cq == v) d = val[o];
          else s = s + val[o] * (loc < static_cast<unsigned>(nr) ? x[loc] : uin[cq]);
        }
      }
      x[v - r0] = (b[v] - s) / d;
    }
    __syncthreads();
  }
  for (int i = threadIdx.x; i < nr; i += blockDim.x) uout[r0 + i] = x[i];
}

template <class T>
struct Vec2T;
template <>
struct Vec2T<double> {
  using type = double2;
};
template <>
struct Vec2T<float> {
  using type = float2;
};

// The sweep from the level's panels: every load is issued before the colour
// phases, which touch only registers and LDS.  A block's panel holds its rows
// sorted by colour, contiguously: per row one uint4 (the local indices of its up
// to 7 off-diagonal slots, 16 bits each, and the row's own number and colour), the
// off-diagonal values slot by slot and the diagonal; its halo (the rows of other
// blocks that its rows name) is a list of fixed stride, and local indices from B
// on name halo rows, the last one (a row's unused slots, of value 0) a zero: whatever
// a row's own value was, an infinity or NaN among them, it doesn't enter its sum.  So a row costs 72 bytes where a slot-major ELL with 32-bit
// columns and a row number costs 88, a halo value is loaded once per block, and
// a full block (the first `nfull`, exactly B rows each) needs no table before its
// loads: they take two round trips (rows, vectors and halo numbers; the halo's
// values).  ZERO: u is zero on entry and is not read.  zc: the sweep starts from
// u + P zc (P of width 2, also for the halo).  dot (when given): the block's Σ b u
// after the sweep.  add (float32, when given): the swept u is added to it
// and not stored.  Per-row arithmetic is k_block_gs's, bit for bit.
// Measured (µs a sweep, float64, levels 3->8): 655,362 rows 14.4 (11.6 from zero;
// bound by bytes: 3.9 TB/s), against 18.2 with the colours' rows streamed one
// after the other; below 200,000 rows 4.7 (4.1 from zero; bound by the two round
// trips, the colour phases and the launch), against 6.5 with rows and halo values
// gathered per row.  float32 at 25,000 to 102,000 rows: 3.8 (3.4), against 5.5.
template <class T>
struct Panels {
  int B, nfull, hs, ncolors;
  const int *bstart;
  const uint4 *idx;    // [row]
  const T *off, *diag; // [block][slot][row], [row]
  const int *halo;     // [block][hs], padded with a row of the block
  const int2 *own_p, *halo_p;  // P's columns of the rows and of the halo
  const typename Vec2T<T>::type *own_w, *halo_w;
};

template <int W, class T, int R, bool ZERO>
__global__ void __launch_bounds__(256)
    k_panel_sweep(Panels<T> P, const T *__restrict__ b, const T *__restrict__ uin, T *__restrict__ uout, int reverse,
                  const T *__restrict__ zc, double *__restrict__ dot, double *__restrict__ add) {
  constexpr int S = W - 1;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T *x = reinterpret_cast<T *>(smem_raw), *bl = x + P.B + P.hs + 1;
  const int k = blockIdx.x, t = threadIdx.x, nt = blockDim.x;
  int r0, nr;
  if (k < P.nfull) {
    r0 = k * P.B;
    nr = P.B;
  } else {
    r0 = P.bstart[k];
    nr = P.bstart[k + 1] - r0;
  }
  uint4 id[R];
  T off[R][S > 0 ? S : 1], dg[R], bv[R], xv[R];
  int hid[2];
  T hv[2];
  int2 hp[2], op[R];
  typename Vec2T<T>::type hw[2], ow[R];
#pragma unroll
  for (int m = 0; m < R; m++) {
    int i = min(t + m * nt, nr - 1);
    id[m] = P.idx[r0 + i];
#pragma unroll
    for (int q = 0; q < S; q++) off[m][q] = P.off[static_cast<size_t>(r0) * S + static_cast<size_t>(q) * nr + i];
    dg[m] = P.diag[r0 + i];
    bv[m] = b[r0 + i];
  }
  if constexpr (!ZERO) {
#pragma unroll
    for (int m = 0; m < R; m++) xv[m] = uin[r0 + min(t + m * nt, nr - 1)];
#pragma unroll
    for (int m = 0; m < 2; m++) hid[m] = P.halo[k * P.hs + min(t + m * nt, P.hs - 1)];
    if (zc) {
#pragma unroll
      for (int m = 0; m < R; m++) {
        int i = r0 + min(t + m * nt, nr - 1);
        op[m] = P.own_p[i];
        ow[m] = P.own_w[i];
      }
#pragma unroll
      for (int m = 0; m < 2; m++) {
        int i = k * P.hs + min(t + m * nt, P.hs - 1);
        hp[m] = P.halo_p[i];
        hw[m] = P.halo_w[i];
      }
    }
#pragma unroll
    for (int m = 0; m < 2; m++) hv[m] = uin[hid[m]];
    if (zc) {
      // u + P zc with the sums of k_prolong_add (a column < 0 pads)
      T oz[R][2], hz[2][2];
#pragma unroll
      for (int m = 0; m < R; m++) {
        oz[m][0] = zc[op[m].x < 0 ? 0 : op[m].x];
        oz[m][1] = zc[op[m].y < 0 ? 0 : op[m].y];
      }
#pragma unroll
      for (int m = 0; m < 2; m++) {
        hz[m][0] = zc[hp[m].x < 0 ? 0 : hp[m].x];
        hz[m][1] = zc[hp[m].y < 0 ? 0 : hp[m].y];
      }
      auto sum = [](int2 c, typename Vec2T<T>::type w, T z0, T z1) {
        T a = static_cast<T>(0);
        if (c.x >= 0) a = a + w.x * z0;
        if (c.y >= 0) a = a + w.y * z1;
        return a;
      };
#pragma unroll
      for (int m = 0; m < R; m++) xv[m] = xv[m] + sum(op[m], ow[m], oz[m][0], oz[m][1]);
#pragma unroll
      for (int m = 0; m < 2; m++) hv[m] = hv[m] + sum(hp[m], hw[m], hz[m][0], hz[m][1]);
    }
  }
#pragma unroll
  for (int m = 0; m < R; m++) {
    int i = t + m * nt;
    if (i < nr) {
      x[i] = ZERO ? static_cast<T>(0) : xv[m];
      bl[i] = bv[m];
    }
  }
#pragma unroll
  for (int m = 0; m < 2; m++) {
    int i = t + m * nt;
    if (i <= P.hs) x[P.B + i] = ZERO || i == P.hs ? static_cast<T>(0) : hv[m];  // the halo, then the zero
  }
  __syncthreads();
  int color[R], row[R];
#pragma unroll
  for (int m = 0; m < R; m++) {
    unsigned int w = id[m].w >> 16;
    color[m] = t + m * nt < nr ? static_cast<int>(w >> 12) : -1;
    row[m] = static_cast<int>(w & 0xfffu);
    bv[m] = bl[row[m]];
  }
  double added[R];  // what the sweep's result is added to, on its way during the colours
#pragma unroll
  for (int m = 0; m < R; m++) {
    int i = t + m * nt;
    added[m] = sizeof(T) == 4 && add && i < nr ? add[r0 + i] : 0.0;
  }
  for (int ci = 0; ci < P.ncolors; ci++) {
    int c = reverse ? P.ncolors - 1 - ci : ci;
#pragma unroll
    for (int m = 0; m < R; m++) {
      if (color[m] != c) continue;
      const unsigned int w[4] = {id[m].x, id[m].y, id[m].z, id[m].w};
      T xs[S > 0 ? S : 1], s = static_cast<T>(0);
#pragma unroll
      for (int q = 0; q < S; q++) xs[q] = x[(w[q >> 1] >> (16 * (q & 1))) & 0xffffu];
      // (a pad is 0 times the zero: it leaves the sum as it is)
#pragma unroll
      for (int q = 0; q < S; q++) s = s + off[m][q] * xs[q];
      x[row[m]] = (bv[m] - s) / dg[m];
    }
    __syncthreads();
  }
  double acc = 0.0;
#pragma unroll
  for (int m = 0; m < R; m++) {
    int i = t + m * nt;
    if (i < nr) {
      T v = x[i];
      if (sizeof(T) == 4 && add) add[r0 + i] = added[m] + static_cast<double>(v);
      else uout[r0 + i] = v;
      acc = acc + static_cast<double>(bl[i]) * static_cast<double>(v);
    }
  }
  if (!dot) return;
  __shared__ double red[4];
  acc = wave_sum(acc);
  if ((t & 63) == 0) red[t >> 6] = acc;
  __syncthreads();
  if (t == 0) {
    double d = red[0];
    for (int w = 1; w < nt / 64; w++) d = d + red[w];
    dot[k] = d;
  }
}

// ---- set-up: what a level keeps besides its vertex-ordered ELL --------------

// the rows of an ELL in another order: row p is row order[p]
__global__ void k_order_rows(int n, int width, const int *__restrict__ order, const int *__restrict__ vcol,
                             const double *__restrict__ vval, int *__restrict__ col, double *__restrict__ val) {
  int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  for (int q = 0; q < width; q++) {
    size_t o = static_cast<size_t>(q) * n;
    col[o + p] = vcol[o + order[p]];
    val[o + p] = vval[o + order[p]];
  }
}

__global__ void k_to_float(size_t n, const double *__restrict__ x, float *__restrict__ y) {
  size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) y[i] = static_cast<float>(x[i]);
}

// The panels (see Panels), one workgroup per block: row i of block k is the
// level's row order[r0 + i]; halo: its sorted halo rows, hcount of them.
__global__ void k_build_panels(int n, int width, int B, int hs, const int *__restrict__ vcol,
                               const double *__restrict__ vval, const int *__restrict__ order,
                               const signed char *__restrict__ color, const int *__restrict__ bstart,
                               const int *__restrict__ halo, const int *__restrict__ hcount, uint4 *__restrict__ idx,
                               double *__restrict__ off, double *__restrict__ diag) {
  const int k = blockIdx.x, S = width - 1;
  const int r0 = bstart[k], nr = bstart[k + 1] - r0, nh = hcount[k];
  const int *h = halo + static_cast<size_t>(k) * hs;
  for (int i = threadIdx.x; i < nr; i += blockDim.x) {
    int r = order[r0 + i], q = 0;
    unsigned int w[8];
    for (int j = 0; j < 8; j++) w[j] = static_cast<unsigned int>(B + hs);
    double d = 0.0;
    double *o = off + static_cast<size_t>(r0) * S + i;
    for (int sl = 0; sl < width; sl++) {
      int c = vcol[static_cast<size_t>(sl) * n + r];
      double v = vval[static_cast<size_t>(sl) * n + r];
      if (c < 0) continue;
      if (c == r) {
        d = v;
        continue;
      }
      if (q >= S) break;  // (the host has checked that no row has more)
      unsigned int l;
      if (c >= r0 && c < r0 + nr) {
        l = static_cast<unsigned int>(c - r0);
      } else {
        int a = 0, e = nh - 1;
        while (a < e) {
          int m = (a + e) >> 1;
          if (h[m] < c) a = m + 1;
          else e = m;
        }
        l = static_cast<unsigned int>(B + a);
      }
      w[q] = l;
      o[static_cast<size_t>(q) * nr] = v;
      q++;
    }
    for (; q < S; q++) o[static_cast<size_t>(q) * nr] = 0.0;
    diag[r0 + i] = d;
    w[7] = (static_cast<unsigned int>(color[r]) << 12) | static_cast<unsigned int>(r - r0);
    idx[r0 + i] = make_uint4(w[0] | (w[1] << 16), w[2] | (w[3] << 16), w[4] | (w[5] << 16), w[6] | (w[7] << 16));
  }
}

// P's two slots of rows ids[i] (null: of row i), side by side
template <class T>
__global__ void k_panel_p(int m, int n, const int *__restrict__ ids, const int *__restrict__ pcol,
                          const T *__restrict__ pval, int2 *__restrict__ c, typename Vec2T<T>::type *__restrict__ w) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= m) return;
  int r = ids ? ids[i] : i;
  c[i] = make_int2(pcol[r], pcol[n + r]);
  typename Vec2T<T>::type v;
  v.x = pval[r];
  v.y = pval[n + r];
  w[i] = v;
}

// Renumbering between the caller's vertex order and the hierarchy's own:
// perm[i] is the caller's index of internal vertex i.
template <class T>
__global__ void k_perm_gather(int n, const int *__restrict__ perm, const T *__restrict__ src, T *__restrict__ dst) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = src[perm[i]];
}

template <class T>
__global__ void k_perm_scatter(int n, const int *__restrict__ perm, const T *__restrict__ src, T *__restrict__ dst) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[perm[i]] = src[i];
}

// u += Z r with Z stored column-major (ZT[j * n + i] = Z[i, j]), in two
// launches so that the whole chip streams Z: the columns are cut into chunks of
// coarse_chunk(n), one workgroup of 64 rows per (row tile, chunk) writes
// part[c * n + i] = Σ_{j in chunk c, ascending} Z[i, j] r[j], and the second
// pass adds Σ_c part[c * n + i] (c ascending) to u.  The fused coarse tail
// uses the same two sums in the same order.
// (16 columns where the coarse tail, whose threads hold a chunk's part of a row in
// registers, can be the one that multiplies; 64 above, for fewer partial sums.  1,792 is
// a choice: a dense level has a quarter of the rows above it in a refined mesh, so at most
// 768 beside the tail's 3,072; 1,792 leaves room for hierarchies that coarsen less, and the
// tail's LDS would hold 2,047.)
__host__ __device__ inline int coarse_chunk(int n) { return n <= 1792 ? 16 : 64; }

template <class T>
__global__ void __launch_bounds__(64)
    k_coarse_partial(int n, const T *__restrict__ ZT, const T *__restrict__ r, T *__restrict__ part) {
  int i = blockIdx.x * 64 + threadIdx.x;
  int j0 = blockIdx.y * coarse_chunk(n);
  int j1 = min(n, j0 + coarse_chunk(n));
  if (i >= n) return;
  T acc = static_cast<T>(0);
#pragma unroll 16
  for (int j = j0; j < j1; j++) acc = acc + ZT[static_cast<size_t>(j) * n + i] * r[j];
  part[static_cast<size_t>(blockIdx.y) * n + i] = acc;
}

template <class T>
__device__ __forceinline__ T coarse_sum(int n, int nchunks, int i, const T *__restrict__ part) {
  T acc = static_cast<T>(0);
#pragma unroll 8
  for (int c = 0; c < nchunks; c++) acc = acc + part[static_cast<size_t>(c) * n + i];
  return acc;
}

template <class T>
__global__ void k_coarse_finish(int n, int nchunks, const T *__restrict__ part, T *__restrict__ u) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) u[i] = u[i] + coarse_sum(n, nchunks, i, part);
}

__host__ __device__ inline int coarse_chunks(int n) { return (n + coarse_chunk(n) - 1) / coarse_chunk(n); }

template <class T>
__device__ double block_sum(double v) {
  __shared__ double sh[kBlock];
  sh[threadIdx.x] = v;
  __syncthreads();
  for (int s = kBlock / 2; s > 0; s >>= 1) {
    if (threadIdx.x < s) sh[threadIdx.x] = sh[threadIdx.x] + sh[threadIdx.x + s];
    __syncthreads();
  }
  return sh[0];
}

// Deterministic dot product: fixed grid of partial sums, then one block.
template <class T>
__global__ void k_dot_partial(int n, const T *__restrict__ x, const T *__restrict__ y, double *__restrict__ part,
                              const int *__restrict__ done) {
  if (done && *done) return;
  double acc = 0.0;
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += kDotBlocks * kBlock)
    acc = acc + static_cast<double>(x[i]) * static_cast<double>(y[i]);
  double s = block_sum<T>(acc);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

__global__ void k_sum_partials(const double *__restrict__ part, double *__restrict__ out,
                               const int *__restrict__ done) {
  if (done && *done) return;
  double s = block_sum<double>(threadIdx.x < kDotBlocks ? part[threadIdx.x] : 0.0);
  if (threadIdx.x == 0) *out = s;
}

// Krylov.jl cg recurrence (warm start, atol = rtol = sqrt(eps), zero-curvature
// exit), the multigrid's default smoother.  One reduction per step: with
// p·Ap, Ap·Ap, r·Ap and r·r known, α = r·r / p·Ap and the next r·r is
// r·r - 2 α r·Ap + α² Ap·Ap, from which β follows, so a step needs no second
// reduction for β (the recurrence's own r·r enters α one step later).  Against
// the usual two reductions the iterates agree to rounding: over 40 hierarchies
// of V-, W- and full cycles within 4.5e-13 of the result's norm, apart from a constant.
// (The constants are the Laplacian's null space, where either form accumulates its own
// rounding, up to 5e-11 on hierarchies that end in a few dozen rows.)  Summing in
// pairs of doubles came no closer to 64-bit numpy and took 10 % longer.
//
// State of a smoothing on a level of several workgroups.  `stop` is the launch
// (step + 1) whose scalars ended it (0: none); rbuf: which residual buffer
// holds the last residual, xok: whether a step was added to x.  ‖p‖² is kept in
// two slots: step `it` reads one and writes the other.
struct CgState {
  double pnorm2[2], eps_stop;
  int stop, rbuf, xok;
};

constexpr int kCgBlocksMax = 1024;  // partial sums per reduction

// r·r - 2 α r·Ap + α² Ap·Ap is good to about 1e-16 r·r.  Where it is less than
// this share of r·r, few digits of the next r·r are left, or none: it is then
// summed from r - α Ap (both forms of the smoother).
constexpr double kCgCancelled = 1e-6;

inline int cg_blocks(int n) { return std::min(kCgBlocksMax, dec::nblocks(n, kBlock)); }

// Σ part[0..np) in a fixed order, the same in every workgroup: thread t adds
// a run of ceil(np / kBlock) consecutive partials, then block_sum's tree
// (every thread has read the result before a later block_sum of the kernel
// writes the same LDS array)
__device__ double sum_partials(const double *__restrict__ part, int np) {
  constexpr int kRun = 16;  // runs up to this long load all their partials at once
  int per = (np + kBlock - 1) / kBlock;
  int j0 = min(np, static_cast<int>(threadIdx.x) * per), j1 = min(np, j0 + per);
  double acc = 0.0;
  if (per <= kRun) {
    double v[kRun];
#pragma unroll
    for (int k = 0; k < kRun; k++) v[k] = part[min(j0 + k, np - 1)];
#pragma unroll
    for (int k = 0; k < kRun; k++)
      if (j0 + k < j1) acc = acc + v[k];
  } else {
    for (int j = j0; j < j1; j++) acc = acc + part[j];
  }
  double s = block_sum<double>(acc);
  __syncthreads();
  return s;
}

// The workgroup's sums of K values in every thread: the wavefronts' sums, then
// those in order.  Successive calls (of any K ≤ KMAX) alternate between the
// halves of red: a thread writes a half again only two calls later, after the
// barrier of the call between, so one barrier per call suffices.
template <int K, int WAVES, int KMAX>
__device__ __forceinline__ void group_sums(double (&v)[K], double (*red)[WAVES * KMAX], int &half) {
  static_assert(K <= KMAX, "a half holds WAVES * KMAX sums");
#pragma unroll
  for (int k = 0; k < K; k++) v[k] = wave_sum(v[k]);
  double *h = red[half];
  half ^= 1;
  if ((threadIdx.x & 63) == 0) {
#pragma unroll
    for (int k = 0; k < K; k++) h[(threadIdx.x >> 6) * K + k] = v[k];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < K; k++) {
    double t = h[k];
#pragma unroll
    for (int w = 1; w < WAVES; w++) t = t + h[w * K + k];
    v[k] = t;
  }
}

// ---- levels of several workgroups: one launch per step ---------------------
// k_cg_start (r = b - A u and r·r), k_cg_step per step, k_cg_finish (the last
// α, u += x, and before a coarse correction its right-hand side R r).  Every
// workgroup adds the previous launch's partial sums itself, in one fixed order,
// so all hold the same scalars; workgroup 0 alone writes the state.  A step
// forms r and p of its own rows from the previous step's r, Ap and p, and the
// same values at every column of its rows, the expressions the column's own row
// stores, so A p needs no launch in between; r, p and Ap are double-buffered.
// Levels of up to some 100,000 rows are bound by the launch and its chain of
// dependent loads (4 to 6 µs each), not by bytes: a smoothing of three steps
// with its restriction is 5 launches, where a direction and a step launch per
// step, the residual and the restriction were 8 or 9.  dec_Δ⁻¹ on levels 3->7
// (with the one-workgroup kernels below): 3.80 against 6.78 ms; five V-cycles
// on 12,513 rows: 0.46 against 0.92 ms; as close to 64 bits as before (1e-12).
constexpr int kCgWaves = kBlock / 64;

// sums[k] = Σ part[k * kCgBlocksMax + j], j < nb
template <int K>
__device__ __forceinline__ void partial_sums(const double *__restrict__ part, int nb, double (&sums)[K],
                                             double (*red)[kCgWaves * 4], int &half) {
  double v[K];
  const int t = static_cast<int>(threadIdx.x);
#pragma unroll
  for (int k = 0; k < K; k++) {
    double q = part[k * kCgBlocksMax + min(t, nb - 1)];
    v[k] = t < nb ? q : 0.0;
  }
  if (nb > kBlock) {  // all further loads at once
    constexpr int kRun = kCgBlocksMax / kBlock - 1;
    double q[K][kRun];
#pragma unroll
    for (int m = 0; m < kRun; m++)
#pragma unroll
      for (int k = 0; k < K; k++) q[k][m] = part[k * kCgBlocksMax + min(t + (m + 1) * kBlock, nb - 1)];
#pragma unroll
    for (int m = 0; m < kRun; m++)
#pragma unroll
      for (int k = 0; k < K; k++) v[k] = t + (m + 1) * kBlock < nb ? v[k] + q[k][m] : v[k];
  }
  group_sums<K, kCgWaves, 4>(v, red, half);
#pragma unroll
  for (int k = 0; k < K; k++) sums[k] = v[k];
}

template <int K>
__device__ __forceinline__ void put_partials(double (&v)[K], int slot0, double *__restrict__ part,
                                             double (*red)[kCgWaves * 4], int &half) {
  group_sums<K, kCgWaves, 4>(v, red, half);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int k = 0; k < K; k++) part[(slot0 + k) * kCgBlocksMax + blockIdx.x] = v[k];
  }
}

// r = b - A u, with zc given (P an ELL of width 2) for u2 = u + P zc, which is
// stored; the partial sums of r·r (slot 3); clears the state's stop.
template <int W, bool FOLD>
__global__ void __launch_bounds__(kBlock)
    k_cg_start(CgState *st, int n, int width, const int *__restrict__ vcol, const double *__restrict__ vval,
               const double *__restrict__ b, const double *__restrict__ u, const int *__restrict__ pcol,
               const double *__restrict__ pval, const double *__restrict__ zc, double *__restrict__ u2,
               double *__restrict__ r, double *__restrict__ part) {
  __shared__ double red[2][kCgWaves * 4];
  int half = 0;
  if (blockIdx.x == 0 && threadIdx.x == 0) st->stop = 0;
  double rr[1] = {0.0};
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
    double s;
    if constexpr (FOLD && W > 0) {
      int c[W];
      double v[W], uv[W];
#pragma unroll
      for (int k = 0; k < W; k++) {
        size_t o = static_cast<size_t>(k) * n + i;
        c[k] = vcol[o];
        v[k] = vval[o];
      }
#pragma unroll
      for (int k = 0; k < W; k++) uv[k] = prolonged(n, c[k] < 0 ? i : c[k], u, pcol, pval, zc);
      u2[i] = prolonged(n, i, u, pcol, pval, zc);
      s = 0.0;
#pragma unroll
      for (int k = 0; k < W; k++)
        if (c[k] >= 0) s = s + v[k] * uv[k];
    } else {
      s = dec_ell::row<W, double, double>(n, width, i, vcol, vval, u);
    }
    double ri = b[i] - s;
    r[i] = ri;
    rr[0] = rr[0] + ri * ri;
  }
  put_partials<1>(rr, 3, part, red, half);
}

// r_i - α Ap_i
__device__ __forceinline__ double next_r(double r, double a, double q) { return r - a * q; }

// Step `it`.  IT0 (it = 0): p = r; Ap and the partial sums.  Else: the
// scalars of step it - 1 from its partial sums (part_in), r = r_old - α Ap_old,
// x += α p_old, p = r + β p_old (FIRST, it = 1: p_old = r_old and x = 0), then
// Ap and the partial sums p·Ap, Ap·Ap, r·Ap, r·r.
template <int W, bool IT0, bool FIRST>
__global__ void __launch_bounds__(kBlock)
    k_cg_step(CgState *st, int it, int n, int width, const int *__restrict__ vcol, const double *__restrict__ vval,
              const double *__restrict__ r0, const double *__restrict__ p0, const double *__restrict__ q0,
              double *__restrict__ r, double *__restrict__ p, double *__restrict__ q, double *__restrict__ x,
              const double *__restrict__ part_in, int nb, double *__restrict__ part) {
  __shared__ double red[2][kCgWaves * 4];
  int half = 0;
  const double eps = 2.220446049250313e-16;
  const int stride = gridDim.x * kBlock, i0 = blockIdx.x * kBlock + threadIdx.x;
  const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
  int stop = 0;
  if constexpr (!IT0) stop = st->stop;
  // The thread's first row is loaded before the scalars, which it does not
  // need, so its loads are in flight while the partial sums are added.
  constexpr int WP = W > 0 ? W : 1;
  int c0[WP];
  double v0[WP], rc[WP], qc[WP], pc[WP];
  const int ia = min(i0, n - 1);
  if constexpr (W > 0) {
#pragma unroll
    for (int k = 0; k < W; k++) {
      size_t o = static_cast<size_t>(k) * n + ia;
      c0[k] = vcol[o];
      v0[k] = vval[o];
    }
#pragma unroll
    for (int k = 0; k < W; k++) {
      int cc = c0[k] < 0 ? 0 : c0[k];
      rc[k] = r0[cc];
      if constexpr (!IT0) qc[k] = q0[cc];
      if constexpr (!IT0 && !FIRST) pc[k] = p0[cc];
    }
  }
  double ri0 = r0[ia], qi0 = 0.0, pi0 = 0.0, xi0 = 0.0;
  if constexpr (!IT0) qi0 = q0[ia];
  if constexpr (!IT0 && !FIRST) {
    pi0 = p0[ia];
    xi0 = x[ia];
  }
  double a = 0.0, beta = 0.0;
  if constexpr (IT0) {
    double g[1];
    partial_sums<1>(part_in + 3 * kCgBlocksMax, nb, g, red, half);
    const double sq = 1.4901161193847656e-08;
    double rn = sqrt(g[0]), es = sq + sq * rn;
    bool done = g[0] == 0.0 || rn <= es;
    if (lead) {
      st->eps_stop = es;
      st->pnorm2[0] = g[0];
      if (done) {
        st->rbuf = 0;
        st->xok = 0;
        st->stop = 1;
      }
    }
    if (done) return;
  } else {
    // block 0 may set `stop` to it + 1 in this launch: only an earlier one ends it
    if (stop != 0 && stop <= it) return;
    double t[4];
    partial_sums<4>(part_in, nb, t, red, half);
    double pn2 = st->pnorm2[(it - 1) & 1], es = st->eps_stop;
    if (t[0] <= eps * pn2 && fabs(t[0]) <= eps * pn2) {  // zero curvature: x and r stay
      if (lead) {
        st->rbuf = (it - 1) & 1;
        st->xok = it > 1;
        st->stop = it + 1;
      }
      return;
    }
    a = t[3] / t[0];
    double gn = t[3] - 2.0 * a * t[2] + a * a * t[1];
    if (!(gn > kCgCancelled * t[3])) {
      // too much cancelled: the sum itself, by every workgroup in the same order (a
      // pass over r and Ap by each, on the rare step that cuts ‖r‖ a thousandfold)
      double g[1] = {0.0};
#pragma unroll 1
      for (int i = threadIdx.x; i < n; i += kBlock) {
        double v = next_r(r0[i], a, q0[i]);
        g[0] = g[0] + v * v;
      }
      group_sums<1, kCgWaves, 4>(g, red, half);
      gn = g[0];
    }
    double rn = sqrt(gn);
    if (rn <= es || rn + 1.0 <= 1.0) {  // solved: the step still counts
      for (int i = i0; i < n; i += stride) {
        x[i] = (FIRST ? 0.0 : x[i]) + a * (FIRST ? r0[i] : p0[i]);
        r[i] = next_r(r0[i], a, q0[i]);
      }
      if (lead) {
        st->rbuf = it & 1;
        st->xok = 1;
        st->stop = it + 1;
      }
      return;
    }
    beta = gn / t[3];
    if (lead) st->pnorm2[it & 1] = gn + beta * beta * pn2;
  }
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  auto own = [&](int i, double ro, double qo, double po, double xo, double s) {
    double ri = IT0 ? ro : next_r(ro, a, qo), po_ = FIRST ? ro : po;
    double pi = IT0 ? ri : ri + beta * po_;
    if constexpr (!IT0) {
      r[i] = ri;
      p[i] = pi;
      x[i] = xo + a * po_;
    }
    q[i] = s;
    acc[0] = acc[0] + pi * s;
    acc[1] = acc[1] + s * s;
    acc[2] = acc[2] + ri * s;
    acc[3] = acc[3] + ri * ri;
  };
  auto at = [&](double ro, double qo, double po) {
    if constexpr (IT0) return ro;
    double ri = next_r(ro, a, qo);
    return ri + beta * (FIRST ? ro : po);
  };
  int i = i0;
  if constexpr (W > 0) {
    if (i0 < n) {
      double s = 0.0;
#pragma unroll
      for (int k = 0; k < W; k++)
        if (c0[k] >= 0) s = s + v0[k] * at(rc[k], IT0 ? 0.0 : qc[k], IT0 || FIRST ? 0.0 : pc[k]);
      own(i0, ri0, qi0, pi0, xi0, s);
    }
    i += stride;
  }
  for (; i < n; i += stride) {
    double s = 0.0;
    if constexpr (W > 0) {
      int c[W];
      double v[W], rv[W], qv[W], pv[W];
#pragma unroll
      for (int k = 0; k < W; k++) {
        size_t o = static_cast<size_t>(k) * n + i;
        c[k] = vcol[o];
        v[k] = vval[o];
      }
#pragma unroll
      for (int k = 0; k < W; k++) {
        int cc = c[k] < 0 ? 0 : c[k];
        rv[k] = r0[cc];
        qv[k] = IT0 ? 0.0 : q0[cc];
        pv[k] = IT0 || FIRST ? 0.0 : p0[cc];
      }
#pragma unroll
      for (int k = 0; k < W; k++)
        if (c[k] >= 0) s = s + v[k] * at(rv[k], qv[k], pv[k]);
    } else {
      for (int k = 0; k < width; k++) {
        size_t o = static_cast<size_t>(k) * n + i;
        int cc = vcol[o];
        if (cc < 0) break;
        s = s + vval[o] * at(r0[cc], IT0 ? 0.0 : q0[cc], IT0 || FIRST ? 0.0 : p0[cc]);
      }
    }
    own(i, r0[i], IT0 ? 0.0 : q0[i], IT0 || FIRST ? 0.0 : p0[i], IT0 || FIRST ? 0.0 : x[i], s);
  }
  put_partials<4>(acc, 0, part, red, half);
}

// After the last step (steps of them): its α, u = u2 + x + α p, and with bc
// given bc = R (r - α Ap) and a zero coarse iterate uc.  After an early exit u =
// u2 + x and the residual is the one the exit left (ra / rb: the two buffers).
template <int RW>
__global__ void __launch_bounds__(kBlock)
    k_cg_finish(const CgState *__restrict__ st, int steps, int n, const double *u2,
                const double *__restrict__ x, const double *__restrict__ p, const double *__restrict__ ra,
                const double *__restrict__ rb, const double *__restrict__ q, const double *__restrict__ part, int nb,
                double *u, int nc, int rwidth, const int *__restrict__ rcol,
                const double *__restrict__ rval, double *__restrict__ bc, double *__restrict__ uc) {
  __shared__ double red[2][kCgWaves * 4];
  int half = 0;
  const double eps = 2.220446049250313e-16;
  const int stride = gridDim.x * kBlock, i0 = blockIdx.x * kBlock + threadIdx.x, ia = min(i0, n - 1);
  const int stop = st->stop, rbuf = st->rbuf, xok = st->xok;
  const double pn2 = st->pnorm2[(steps - 1) & 1];
  double u0 = u2[ia], x0 = steps > 1 ? x[ia] : 0.0, p0 = p[ia];
  const double *r = ((steps - 1) & 1) ? rb : ra;
  // the thread's first coarse row, in flight while the partial sums are added
  constexpr int RP = RW > 0 ? RW : 1;
  int c0[RP];
  double v0[RP], rv0[RP], qv0[RP];
  if constexpr (RW > 0) {
    int ca = min(i0, nc - 1);
#pragma unroll
    for (int k = 0; k < RW; k++) {
      size_t o = static_cast<size_t>(k) * nc + ca;
      c0[k] = rcol[o];
      v0[k] = rval[o];
    }
#pragma unroll
    for (int k = 0; k < RW; k++) {
      int cc = c0[k] < 0 ? 0 : c0[k];
      rv0[k] = r[cc];
      qv0[k] = q[cc];
    }
  }
  double t[4];
  partial_sums<4>(part, nb, t, red, half);
  double a = 0.0;
  bool with_x = steps > 1;
  if (stop != 0) {
    with_x = xok != 0;
    r = rbuf ? rb : ra;
  } else if (!(t[0] <= eps * pn2 && fabs(t[0]) <= eps * pn2)) {
    a = t[3] / t[0];
  }
  // (a = 0 adds nothing: p and Ap then hold values of an earlier smoothing,
  // finite ones, or this one's)
  auto step = [&](double ui, double xi, double pi) {
    double xs = with_x ? xi : 0.0;
    return (a != 0.0 ? xs + a * pi : xs) + ui;
  };
  if (i0 < n) u[i0] = step(u0, x0, p0);
  for (int i = i0 + stride; i < n; i += stride) u[i] = step(u2[i], steps > 1 ? x[i] : 0.0, p[i]);
  if (!bc) return;
  int i = i0;
  if constexpr (RW > 0) {
    if (stop == 0) {
      if (i0 < nc) {
        double s = 0.0;
#pragma unroll
        for (int k = 0; k < RW; k++)
          if (c0[k] >= 0) s = s + v0[k] * (a != 0.0 ? next_r(rv0[k], a, qv0[k]) : rv0[k]);
        bc[i0] = s;
        uc[i0] = 0.0;
      }
      i += stride;
    }
  }
  for (; i < nc; i += stride) {
    double s = 0.0;
    if constexpr (RW > 0) {
      int c[RW];
      double v[RW], rv[RW], qv[RW];
#pragma unroll
      for (int k = 0; k < RW; k++) {
        size_t o = static_cast<size_t>(k) * nc + i;
        c[k] = rcol[o];
        v[k] = rval[o];
      }
#pragma unroll
      for (int k = 0; k < RW; k++) {
        int cc = c[k] < 0 ? 0 : c[k];
        rv[k] = r[cc];
        qv[k] = q[cc];
      }
#pragma unroll
      for (int k = 0; k < RW; k++)
        if (c[k] >= 0) s = s + v[k] * (a != 0.0 ? next_r(rv[k], a, qv[k]) : rv[k]);
    } else {
      for (int k = 0; k < rwidth; k++) {
        size_t o = static_cast<size_t>(k) * nc + i;
        int cc = rcol[o];
        if (cc < 0) break;
        s = s + rval[o] * (a != 0.0 ? next_r(r[cc], a, q[cc]) : r[cc]);
      }
    }
    bc[i] = s;
    uc[i] = 0.0;
  }
}

// ---- small levels: one workgroup, in registers and LDS ---------------------
// A level of at most kCgSmallRows rows of at most kCgWidth slots: thread t of
// kCgThreads owns rows t + kCgThreads k (k < R) and holds their columns (16
// bits each) and values in registers; p lives in LDS, so a product is LDS
// gathers only.  512 threads of up to 256 registers hold 7 rows each, where 1024
// threads of 128 held 3 (with 32-bit columns).  A smoothing of three steps takes
// 7.0 µs at 642 rows, 12.9 at 2,562 and 14.6 at 3,185 (1.2 to 2.3 µs a step: the
// product's LDS gathers, one reduction, two barriers), against 11 and 15.1 µs at
// 642 and 2,562 rows with two reductions by LDS shuffles per step; a level of
// 10,242 rows on several workgroups takes 20.
constexpr int kCgThreads = 512;
constexpr int kCgWidth = 7;
constexpr int kCgRowsMax = 7;
constexpr int kCgSmallRows = kCgThreads * kCgRowsMax;
constexpr int kCgCoarseRows = 2;  // rows per thread of the coarsest level in the tail
constexpr int kCgGroupWaves = kCgThreads / 64;

struct CgLevel {
  int n, width;
  const int *col;
  const double *val;
};

// *(p + off bytes): a uniform base and a 32-bit offset per lane
template <class T>
__device__ __forceinline__ T at_byte(const T *__restrict__ p, unsigned int off) {
  return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(p) + off);
}

template <int R>
struct CgRows {
  unsigned int c[R][4];  // columns' byte offsets (8 c) in pairs; a pad is the row itself with value 0
  double v[R][kCgWidth];
};

template <int R>
__device__ __forceinline__ void load_cg_rows(CgRows<R> &o, const CgLevel &L) {
#pragma unroll
  for (int k = 0; k < R; k++) {
    int i = static_cast<int>(threadIdx.x) + k * kCgThreads, ia = min(i, L.n - 1);
    unsigned int c[kCgWidth + 1];
    c[kCgWidth] = 0;
#pragma unroll
    for (int s = 0; s < kCgWidth; s++) {
      unsigned int q = static_cast<unsigned int>(min(s, L.width - 1) * L.n + ia);
      int cc = at_byte(L.col, 4u * q);
      double vv = at_byte(L.val, 8u * q);
      bool has = s < L.width && cc >= 0 && i < L.n;
      c[s] = 8u * static_cast<unsigned int>(has ? cc : ia);
      o.v[k][s] = has ? vv : 0.0;
    }
#pragma unroll
    for (int s = 0; s < 4; s++) o.c[k][s] = c[2 * s] | (c[2 * s + 1] << 16);
  }
}

// v, as a value the compiler knows nothing about: what is computed from it
// inside a loop is not kept in registers across the loop
__device__ __forceinline__ unsigned int opaque(unsigned int v) {
  asm volatile("" : "+v"(v));
  return v;
}

// Σ_s v[s] x[c[s]] in slot order, by fused multiply-adds
template <int R>
__device__ __forceinline__ double cg_row(const CgRows<R> &o, int k, const double *x) {
  double xv[kCgWidth];
#pragma unroll
  for (int j = 0; j < 4; j++) {
    unsigned int c = opaque(o.c[k][j]);
    xv[2 * j] = at_byte(x, c & 0xffffu);
    if (2 * j + 1 < kCgWidth) xv[2 * j + 1] = at_byte(x, c >> 16);
  }
  double acc = 0.0;
#pragma unroll
  for (int s = 0; s < kCgWidth; s++) acc = __builtin_fma(o.v[k][s], xv[s], acc);
  return acc;
}

typedef double CgRed[2][kCgGroupWaves * 3];

// Up to `steps` CG steps from the residual r (each thread's rows), added to
// u; r is the residual after them.  p: n values of LDS, free on entry (a barrier
// has passed since their last use).
template <int R>
__device__ __forceinline__ void cg_run(const CgRows<R> &o, int n, int steps, double (&u)[R], double (&r)[R], double *p,
                                       CgRed &red, int &half) {
  const double sq = 1.4901161193847656e-08, eps = 2.220446049250313e-16;
  double g[1] = {0.0};
#pragma unroll
  for (int k = 0; k < R; k++) {
    int i = static_cast<int>(threadIdx.x) + k * kCgThreads;
    if (i < n) p[i] = r[k];
    g[0] = g[0] + r[k] * r[k];
  }
  group_sums<1, kCgGroupWaves, 3>(g, red, half);
  double gamma = g[0], pnorm2 = gamma;
  const double rn = sqrt(gamma), es = sq + sq * rn;
  if (gamma == 0.0 || rn <= es) return;
  // ‖r‖ ≤ es or ‖r‖ + 1 ≤ 1, as tests of r·r: no square root in the steps
  const double solved = fmax(es * es, 1.23e-32);
  // (the sums' barrier has made p complete)
  for (int it = 0; it < steps; it++) {
    const double over = 1.0 / gamma;  // ready before β needs it
    double q[R], t[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < R; k++) {
      int i = static_cast<int>(threadIdx.x) + k * kCgThreads;
      q[k] = 0.0;
      if (i < n) {
        q[k] = cg_row<R>(o, k, p);
        t[0] = t[0] + p[i] * q[k];
        t[1] = t[1] + q[k] * q[k];
        t[2] = t[2] + r[k] * q[k];
      }
      __builtin_amdgcn_sched_barrier(0);  // rows one after the other: registers
    }
    group_sums<3, kCgGroupWaves, 3>(t, red, half);
    if (t[0] <= eps * pnorm2 && fabs(t[0]) <= eps * pnorm2) return;
    double a = gamma / t[0];
    double gn = gamma - 2.0 * a * t[2] + a * a * t[1];
#pragma unroll
    for (int k = 0; k < R; k++) {
      int i = static_cast<int>(threadIdx.x) + k * kCgThreads;
      if (i < n) {
        u[k] = u[k] + a * p[i];
        r[k] = r[k] - a * q[k];
      }
    }
    if (it + 1 == steps) return;
    if (!(gn > kCgCancelled * gamma)) {
      // too much cancelled: the sum itself (the same branch in every thread)
      g[0] = 0.0;
#pragma unroll
      for (int k = 0; k < R; k++) g[0] = g[0] + r[k] * r[k];
      group_sums<1, kCgGroupWaves, 3>(g, red, half);
      gn = g[0];
    }
    if (gn <= solved) return;
    double beta = gn * over;
    pnorm2 = gn + beta * beta * pnorm2;
    gamma = gn;
#pragma unroll
    for (int k = 0; k < R; k++) {
      int i = static_cast<int>(threadIdx.x) + k * kCgThreads;
      if (i < n) p[i] = r[k] + beta * p[i];
    }
    __syncthreads();
  }
}

// r = b - A u of the thread's rows, u in LDS (complete)
template <int R>
__device__ __forceinline__ void cg_residual(const CgRows<R> &o, int n, const double *__restrict__ b, const double *u,
                                            double (&r)[R]) {
  double bv[R];
  const int t = static_cast<int>(opaque(threadIdx.x));
#pragma unroll
  for (int k = 0; k < R; k++) bv[k] = at_byte(b, 8u * static_cast<unsigned int>(min(t + k * kCgThreads, n - 1)));
#pragma unroll
  for (int k = 0; k < R; k++) {
    int i = static_cast<int>(threadIdx.x) + k * kCgThreads;
    r[k] = i < n ? bv[k] - cg_row<R>(o, k, u) : 0.0;
    __builtin_amdgcn_sched_barrier(0);
  }
}

// The transfer to the next coarser level: R's rows (nc) and P's.
struct CgTransfer {
  int nc, rwidth, pwidth;
  const int *rcol, *pcol;
  const double *rval, *pval;
};

// u += P z of the thread's rows, z in LDS or memory
template <int R>
__device__ __forceinline__ void cg_prolong(const CgTransfer &T, int n, const double *z, double (&u)[R]) {
#pragma unroll
  for (int k = 0; k < R; k++) {
    int ia = min(static_cast<int>(opaque(threadIdx.x)) + k * kCgThreads, n - 1);
    u[k] = u[k] + (T.pwidth == 2 ? dec_ell::row<2, double, double>(n, T.pwidth, ia, T.pcol, T.pval, z)
                                 : dec_ell::row<0, double, double>(n, T.pwidth, ia, T.pcol, T.pval, z));
  }
}

// row i of R r, r in LDS
__device__ __forceinline__ double cg_restrict(const CgTransfer &T, int i, const double *r) {
  return T.rwidth == 7 ? dec_ell::row<7, double, double>(T.nc, T.rwidth, i, T.rcol, T.rval, r)
                       : dec_ell::row<0, double, double>(T.nc, T.rwidth, i, T.rcol, T.rval, r);
}

// `reps` smoothings of one small level, one after the other: u += x.  With zc
// given they start from u + P zc; with bc given the residual is restricted
// (bc = R r, and a zero coarse iterate uc).
template <int R>
__global__ void __launch_bounds__(kCgThreads)
    k_cg_small(CgLevel L, const double *__restrict__ b, double *__restrict__ u, int steps, int reps, CgTransfer T,
               const double *__restrict__ zc, double *__restrict__ bc, double *__restrict__ uc) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  double *p = reinterpret_cast<double *>(smem_raw);
  __shared__ CgRed red;
  int half = 0;
  CgRows<R> o;
  load_cg_rows<R>(o, L);
  double uv[R], r[R];
#pragma unroll
  for (int k = 0; k < R; k++) uv[k] = u[min(static_cast<int>(threadIdx.x) + k * kCgThreads, L.n - 1)];
  if (zc) cg_prolong<R>(T, L.n, zc, uv);
  for (int q = 0; q < reps; q++) {
#pragma unroll
    for (int k = 0; k < R; k++) {
      int i = static_cast<int>(threadIdx.x) + k * kCgThreads;
      if (i < L.n) p[i] = uv[k];
    }
    __syncthreads();
    cg_residual<R>(o, L.n, b, p, r);
    __syncthreads();
    cg_run<R>(o, L.n, steps, uv, r, p, red, half);
    __syncthreads();
  }
#pragma unroll
  for (int k = 0; k < R; k++) {
    int i = static_cast<int>(threadIdx.x) + k * kCgThreads;
    if (i < L.n) {
      u[i] = uv[k];
      if (bc) p[i] = r[k];
    }
  }
  if (!bc) return;
  __syncthreads();
  for (int i = threadIdx.x; i < T.nc; i += kCgThreads) {
    bc[i] = cg_restrict(T, i, p);
    uc[i] = 0.0;
  }
}

// `cycles` μ-cycles of the two coarsest levels A and C (C of at most 1024 rows)
// in one launch: each smooths A, restricts, smooths C once or twice (twice, the
// W-cycle's, in the first `wcycles` of them), prolongs and smooths A again.
// Both levels' rows stay in registers throughout; vectors pass through LDS.  In
// place of six or seven launches a cycle that each loaded a level again: 44 µs
// for a W-cycle's two visits of 2,562 and 642 rows, against about 110.
template <int R, int RC>
__global__ void __launch_bounds__(kCgThreads)
    k_cg_tail(CgLevel A, CgLevel C, const double *__restrict__ b, double *__restrict__ u, int steps, int cycles,
              int wcycles, CgTransfer T) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  double *pa = reinterpret_cast<double *>(smem_raw), *pc = pa + A.n;
  __shared__ CgRed red;
  int half = 0;
  CgRows<R> oa;
  CgRows<RC> oc;
  load_cg_rows<R>(oa, A);
  double ua[R];
#pragma unroll
  for (int k = 0; k < R; k++) ua[k] = u[min(static_cast<int>(threadIdx.x) + k * kCgThreads, A.n - 1)];
  load_cg_rows<RC>(oc, C);
  for (int cyc = 0; cyc < cycles; cyc++) {
    double r[R], rc[RC], uc[RC];
    auto smooth_a = [&]() {
#pragma unroll
      for (int k = 0; k < R; k++) {
        int i = static_cast<int>(threadIdx.x) + k * kCgThreads;
        if (i < A.n) pa[i] = ua[k];
      }
      __syncthreads();
      cg_residual<R>(oa, A.n, b, pa, r);
      __syncthreads();
      cg_run<R>(oa, A.n, steps, ua, r, pa, red, half);
      __syncthreads();
    };
    smooth_a();
#pragma unroll
    for (int k = 0; k < R; k++) {
      int i = static_cast<int>(threadIdx.x) + k * kCgThreads;
      if (i < A.n) pa[i] = r[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < RC; k++) {
      int i = static_cast<int>(opaque(threadIdx.x)) + k * kCgThreads;
      rc[k] = cg_restrict(T, min(i, C.n - 1), pa);
      if (i >= C.n) rc[k] = 0.0;
      uc[k] = 0.0;
    }
    // C starts at zero: its residual is b_c, then what the steps leave
    for (int v = 0; v < (cyc < wcycles ? 2 : 1); v++) {
      cg_run<RC>(oc, C.n, steps, uc, rc, pc, red, half);
      __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < RC; k++) {
      int i = static_cast<int>(threadIdx.x) + k * kCgThreads;
      if (i < C.n) pc[i] = uc[k];
    }
    __syncthreads();
    cg_prolong<R>(T, A.n, pc, ua);
    smooth_a();
  }
#pragma unroll
  for (int k = 0; k < R; k++) {
    int i = static_cast<int>(threadIdx.x) + k * kCgThreads;
    if (i < A.n) u[i] = ua[k];
  }
}

__global__ void k_add_f2d(int n, const float *__restrict__ c, double *__restrict__ u) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) u[i] = u[i] + static_cast<double>(c[i]);
}

// ---------------------------------------------- V-cycle-preconditioned CG
// Conjugate gradients on the finest level with one V-cycle (from a zero
// start) as the preconditioner z = M r:
//   β = (r·z) / (r·z)_prev,  p = z + β p,  q = A p,  α = (r·z) / (p·q),
//   x += α p,  r -= α q.
// Three launches per iteration after the V-cycle, one element per thread,
// with the scalars on the device: every workgroup adds the previous launch's
// per-workgroup partial sums itself, in one fixed order (sum_partials), so all
// hold the same β or α.  Vectors are indexed by the hierarchy's vertex
// numbers; the product runs over the level's rows in vertex order.
// sc[0] = (r·z)_prev (1 before the first iteration, when p = 0),
// sc[1] = r·z, sc[2] = α: the direction launch reads sc[0] and its block 0
// writes sc[1]; a one-workgroup launch forms α and copies sc[1] to sc[0];
// the update launch reads α.  No launch with several workgroups reads a slot
// it writes.  The update launch also prepares the next V-cycle's input: z = 0
// (float64 preconditioner), or the float32 r and a zero float32 iterate
// (float32 preconditioner); the zeros only where the cycle reads them.


// kPcgDotBlocks partial sums of r·z over a grid-stride loop (z32 non-null:
// z = the float32 preconditioner's result, stored in float64 first)
constexpr int kPcgDotBlocks = kBlock;

__global__ void __launch_bounds__(kBlock) k_pcg_dot(int n, const double *__restrict__ r, const float *__restrict__ z32,
                                                    double *__restrict__ z, double *__restrict__ part) {
  double acc = 0.0;
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += kPcgDotBlocks * kBlock) {
    double zi;
    if (z32) {
      zi = static_cast<double>(z32[i]);
      z[i] = zi;
    } else {
      zi = z[i];
    }
    acc = acc + r[i] * zi;
  }
  double s = block_sum<double>(acc);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// α = (r·z) / (p·q) into sc[2] (zero when p·q is not positive), from the
// direction launch's per-workgroup partial sums of p·q; sc[0] = sc[1] for
// the next iteration's β
__global__ void __launch_bounds__(kBlock) k_pcg_alpha(const double *__restrict__ part_pq, int np,
                                                      double *__restrict__ sc) {
  double pq = sum_partials(part_pq, np);
  if (threadIdx.x != 0) return;
  double rz = sc[1];
  double alpha = pq > 0.0 ? rz / pq : 0.0;
  if (!(alpha == alpha) || fabs(alpha) > 1e300) alpha = 0.0;
  sc[2] = alpha;
  sc[0] = rz;
}

// β, then per row p = z + β p and q = A z + β q (= A p, the product of the
// previous direction carried over, so one vector is gathered; slots in
// ascending column order), in place, and the partial sums of p·q
template <int W>
__global__ void __launch_bounds__(kBlock)
    k_pcg_dir(int n, int width, const int *__restrict__ col, const double *__restrict__ val,
              const int *__restrict__ rowid, const double *__restrict__ z, double *__restrict__ p,
              double *__restrict__ q, const double *__restrict__ part_rz, int np, double *__restrict__ sc,
              double *__restrict__ part_pq) {
  double rz = sum_partials(part_rz, np);
  double beta = rz / sc[0];
  if (blockIdx.x == 0 && threadIdx.x == 0) sc[1] = rz;
  int pos = dec_ell::xcd_block() * kBlock + threadIdx.x;
  double acc = 0.0;
  if (pos < n) {
    double s = dec_ell::row<W, double, double>(n, width, pos, col, val, z);
    int v = rowid ? rowid[pos] : pos;
    double pv = z[v] + beta * p[v];
    double qv = s + beta * q[v];
    p[v] = pv;
    q[v] = qv;
    acc = pv * qv;
  }
  double t = block_sum<double>(acc);
  if (threadIdx.x == 0) part_pq[blockIdx.x] = t;
}

// x += α p, r -= α q, the partial sums of r·r, and the next V-cycle's input
__global__ void __launch_bounds__(kBlock)
    k_pcg_update(int n, double *__restrict__ x, double *__restrict__ r, const double *__restrict__ p,
                 const double *__restrict__ q, const double *__restrict__ sc, double *__restrict__ part_rr,
                 double *__restrict__ z, float *__restrict__ b32, float *__restrict__ u32) {
  const double alpha = sc[2];
  int i = blockIdx.x * kBlock + threadIdx.x;
  double acc = 0.0;
  if (i < n) {
    x[i] = x[i] + alpha * p[i];
    double ri = r[i] - alpha * q[i];
    r[i] = ri;
    acc = ri * ri;
    if (z) z[i] = 0.0;
    if (b32) b32[i] = static_cast<float>(ri);
    if (u32) u32[i] = 0.0f;
  }
  double t = block_sum<double>(acc);
  if (threadIdx.x == 0) part_rr[blockIdx.x] = t;
}

// (re)start: r = src, p = q = 0, sc[0] = 1 (the first direction is z), and
// the first V-cycle's input as k_pcg_update prepares it
__global__ void k_pcg_start(int n, const double *__restrict__ src, double *__restrict__ r, double *__restrict__ p,
                            double *__restrict__ q, double *__restrict__ sc, double *__restrict__ z,
                            float *__restrict__ b32, float *__restrict__ u32) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    double ri = src[i];
    r[i] = ri;
    p[i] = 0.0;
    q[i] = 0.0;
    if (z) z[i] = 0.0;
    if (b32) b32[i] = static_cast<float>(ri);
    if (u32) u32[i] = 0.0f;
  }
  if (i == 0) {
    sc[0] = 1.0;
    sc[1] = 0.0;
    sc[2] = 0.0;
  }
}


// ------------------------------------------------------------- fused coarse tail
// The levels whose size is at most fuse_rows (DEC_MG_FUSE_ROWS, default
// kFuseRowsDefault, at most kFuseRowsMax) run as one workgroup of 1024
// threads: every phase of the V-cycle below that level (colour sweeps,
// residual, restriction, prolongation) is a strided loop over the level's
// rows followed by a workgroup barrier, in place of one kernel launch per
// phase.  Per-row arithmetic is the same as the multi-kernel path (same
// expressions, same order).  One workgroup streams at a small fraction of
// the chip's bandwidth, so this pays only for levels of a few thousand rows.
constexpr int kFuseRowsDefault = 3000;
constexpr int kFuseRowsMax = 4096;  // levels up to this size are one block (LDS)
constexpr int kFuseThreads = 1024;
constexpr int kMaxColors = 16;

template <class T>
struct LevelDesc {
  int n, width, ncolors, nc, rwidth, pwidth;
  int cstart[kMaxColors + 1];
  const int *col, *rowid, *rcol, *pcol;
  const T *val, *rval, *pval;
  T *u, *b, *r;
};

template <class T>
__device__ __forceinline__ T fused_row(const LevelDesc<T> &L, int p, const T *x) {
  return L.width == 7 ? dec_ell::row<7, T, T>(L.n, L.width, p, L.col, L.val, x)
                      : dec_ell::row<0, T, T>(L.n, L.width, p, L.col, L.val, x);
}

template <class T>
__device__ void fused_smooth(const LevelDesc<T> &L, const T *b, T *u, int steps, int alg, T omega, bool post) {
  for (int it = 0; it < steps; it++) {
    if (alg == DEC_SMOOTH_GS || alg == DEC_SMOOTH_BLOCK_GS) {
      // a level in the fused tail is one block: the hybrid sweep is the
      // multicolour sweep
      for (int ci = 0; ci < L.ncolors; ci++) {
        int c = post ? L.ncolors - 1 - ci : ci;
        for (int p = L.cstart[c] + threadIdx.x; p < L.cstart[c + 1]; p += blockDim.x) {
          int v = L.rowid[p];
          T sum, d;
          if (L.width == 7) dec_ell::gs_row<7, T>(L.n, L.width, p, v, L.col, L.val, u, sum, d);
          else dec_ell::gs_row<0, T>(L.n, L.width, p, v, L.col, L.val, u, sum, d);
          u[v] = (b[v] - sum) / d;
        }
        __syncthreads();
      }
    } else {
      for (int p = threadIdx.x; p < L.n; p += blockDim.x) {
        int v = L.rowid[p];
        T sum, d;
        if (L.width == 7) dec_ell::gs_row<7, T>(L.n, L.width, p, v, L.col, L.val, u, sum, d);
        else dec_ell::gs_row<0, T>(L.n, L.width, p, v, L.col, L.val, u, sum, d);
        T full = fused_row(L, p, u);
        L.r[v] = u[v] + omega * ((b[v] - full) / d);
      }
      __syncthreads();
      for (int i = threadIdx.x; i < L.n; i += blockDim.x) u[i] = L.r[i];
      __syncthreads();
    }
  }
}

// phase 0: the whole V-cycle below l0, the coarsest level smoothed.
// phase 1: the down sweep; at the coarsest level only its residual is formed
//          (into Ls[nl-1].r) for the dense direct solve, which runs as
//          k_coarse_partial on the whole chip.
// phase 2: the coarsest correction u += Σ_c part[c] (k_coarse_finish's sum),
//          then the up sweep.
template <class T>
__global__ void __launch_bounds__(kFuseThreads)
    k_fused_vcycle(const LevelDesc<T> *__restrict__ Ls, int l0, int nl, T *u0, const T *b0, int steps, int alg,
                   T omega, int phase, const T *__restrict__ part) {
  if (phase != 2) {
    for (int l = l0; l < nl; l++) {
      const LevelDesc<T> &L = Ls[l];
      T *u = l == l0 ? u0 : L.u;
      const T *b = l == l0 ? b0 : L.b;
      if (l > l0) {
        for (int i = threadIdx.x; i < L.n; i += blockDim.x) u[i] = static_cast<T>(0);
        __syncthreads();
      }
      if (l == nl - 1 && phase == 1) {
        for (int p = threadIdx.x; p < L.n; p += blockDim.x) {
          int v = L.rowid[p];
          L.r[v] = b[v] - fused_row(L, p, u);
        }
        return;
      }
      fused_smooth(L, b, u, steps, alg, omega, false);
      if (l == nl - 1) break;
      for (int p = threadIdx.x; p < L.n; p += blockDim.x) {
        int v = L.rowid[p];
        L.r[v] = b[v] - fused_row(L, p, u);
      }
      __syncthreads();
      const LevelDesc<T> &C = Ls[l + 1];
      for (int i = threadIdx.x; i < L.nc; i += blockDim.x) {
        T acc = L.rwidth == 7 ? dec_ell::row<7, T, T>(L.nc, L.rwidth, i, L.rcol, L.rval, L.r)
                              : dec_ell::row<0, T, T>(L.nc, L.rwidth, i, L.rcol, L.rval, L.r);
        C.b[i] = acc;
      }
      __syncthreads();
    }
  } else {
    const LevelDesc<T> &C = Ls[nl - 1];
    T *uc = nl - 1 == l0 ? u0 : C.u;
    int nch = coarse_chunks(C.n);
    for (int i = threadIdx.x; i < C.n; i += blockDim.x) uc[i] = uc[i] + coarse_sum(C.n, nch, i, part);
    __syncthreads();
  }
  for (int l = nl - 2; l >= l0; l--) {
    const LevelDesc<T> &L = Ls[l];
    const LevelDesc<T> &C = Ls[l + 1];
    T *u = l == l0 ? u0 : L.u;
    const T *b = l == l0 ? b0 : L.b;
    for (int j = threadIdx.x; j < L.n; j += blockDim.x)
      u[j] = u[j] + (L.pwidth == 2 ? dec_ell::row<2, T, T>(L.n, L.pwidth, j, L.pcol, L.pval, C.u)
                                   : dec_ell::row<0, T, T>(L.n, L.pwidth, j, L.pcol, L.pval, C.u));
    __syncthreads();
    fused_smooth(L, b, u, steps, alg, omega, true);
  }
}

// The coarse tail in Gauss-Seidel V-cycles above a dense coarsest level: for each
// smoothed level A of at most 3 x 1024 rows of 1-8 slots a launch on the way down
// and one on the way up, with A's rows in registers (thread t owns positions
// t + 1024 i of the rows sorted by colour) and its vectors in LDS, so that the
// colour phases wait on no memory access.  A row is one uint4 (the 12-bit numbers
// of its up to 7 off-diagonal slots; beside the first the diagonal's place among
// them, in the last 16 bits the row's own number and colour), the off-diagonal values
// slot by slot and the diagonal; nothing that is loaded names another load.
//   k_tail_down: A's pre-smoothing, residual and restriction.  Above the dense
//     coarsest level C also its direct solve Z r (C's iterate starts at zero):
//     Z is too much for one workgroup, so one for every 16 of C's rows does the whole
//     of A's part by itself and then its rows of Z r, and a launch is saved.
//   k_tail_up: the prolongation of C's correction to A and A's post-smoothing.
// Every sum is k_fused_vcycle's and k_coarse_partial's, bit for bit.
// Bound by the colour phases (a barrier each) and one round trip for the loads.
// Measured with 2,562 rows above 642, three sweeps either way, float64: 14.3 + 10.2
// µs, where rows that were read by number, their colours searched in a table and
// the product in a launch of its own took 16.8 + 4.7 + 16.8; 1,700 rows above
// 437, two sweeps, float32: 9.3 + 5.7, against 11 + 4.7 + 11.
template <class T>
struct Tail {
  int n, nc, ncolors, rwidth, pwidth;
  const uint4 *idx;
  const T *off, *diag;
  const int *rcol, *pcol;
  const T *rval, *pval;
  const T *ZT;  // null: C is not the dense coarsest level
};

constexpr int kTailRows = 3 * kFuseThreads;  // 12-bit numbers, three rows a thread
constexpr int kTailZ = 16;                   // rows of C in a workgroup

// x and a zero, which a row's unused slots name (later the chunks' parts of 16 rows
// of Z r), w, and C's right-hand side
__host__ __device__ inline int tail_x(int n, int nc) {
  int parts = coarse_chunks(nc) * kTailZ;
  return n + 1 > parts ? n + 1 : parts;
}
inline size_t tail_lds(int n, int nc, size_t bytes) {
  return (static_cast<size_t>(tail_x(n, nc)) + n + nc) * bytes;
}

__global__ void k_build_tail(const LevelDesc<double> A, int S, uint4 *__restrict__ idx, double *__restrict__ off,
                             double *__restrict__ diag) {
  int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= A.n) return;
  unsigned int v = static_cast<unsigned int>(A.rowid[q]), w[8], at = 0, k = 0, c = 0;
  while (static_cast<int>(c) + 1 < A.ncolors && q >= A.cstart[c + 1]) c++;
  for (int j = 0; j < 7; j++) w[j] = static_cast<unsigned int>(A.n);
  w[7] = v;
  for (int sl = 0; sl < A.width; sl++) {
    size_t o = static_cast<size_t>(sl) * A.n + q;
    int cc = A.col[o];
    if (cc < 0) continue;
    if (static_cast<unsigned int>(cc) == v) {
      at = k;
      diag[q] = A.val[o];
    } else if (k < static_cast<unsigned int>(S)) {  // (the host has checked that no row has more)
      w[k] = static_cast<unsigned int>(cc);
      off[static_cast<size_t>(k) * A.n + q] = A.val[o];
      k++;
    }
  }
  for (; k < static_cast<unsigned int>(S); k++) off[static_cast<size_t>(k) * A.n + q] = 0.0;
  w[0] |= at << 12;
  w[7] |= c << 12;
  idx[q] = make_uint4(w[0] | (w[1] << 16), w[2] | (w[3] << 16), w[4] | (w[5] << 16), w[6] | (w[7] << 16));
}

template <int S, class T, int R>
struct TailRows {
  uint4 ix[R];
  T off[R][S], d[R], b[R];

  __device__ __forceinline__ void load(const Tail<T> &A) {
#pragma unroll
    for (int i = 0; i < R; i++) {
      int q = static_cast<int>(threadIdx.x) + i * kFuseThreads, qc = min(q, A.n - 1);
      ix[i] = A.idx[qc];
      if (q >= A.n) ix[i].w = 0xf0000000u;  // no colour
      d[i] = A.diag[qc];
#pragma unroll
      for (int k = 0; k < S; k++) off[i][k] = A.off[static_cast<size_t>(k) * A.n + qc];
    }
  }
  __device__ __forceinline__ int row(int i) const { return (ix[i].w >> 16) & 0xfff; }
  __device__ __forceinline__ int color(int i) const { return ix[i].w >> 28; }
  __device__ __forceinline__ int slot(int i, int k) const {
    unsigned int w = k < 2 ? ix[i].x : k < 4 ? ix[i].y : k < 6 ? ix[i].z : ix[i].w;
    w = opaque(w);
    return (k & 1 ? w >> 16 : w) & 0xfff;
  }
  // b in w, a barrier behind it
  __device__ __forceinline__ void rhs(const T *w) {
#pragma unroll
    for (int i = 0; i < R; i++) b[i] = w[row(i)];
  }
  __device__ __forceinline__ void sweep(T *x, int ncolors, bool reverse) {
    for (int ci = 0; ci < ncolors; ci++) {
      int c = reverse ? ncolors - 1 - ci : ci;
#pragma unroll
      for (int i = 0; i < R; i++) {
        if (color(i) != c) continue;
        T xs[S], sum = static_cast<T>(0);
#pragma unroll
        for (int k = 0; k < S; k++) xs[k] = x[slot(i, k)];
#pragma unroll
        for (int k = 0; k < S; k++) sum = sum + off[i][k] * xs[k];
        x[row(i)] = (b[i] - sum) / d[i];
      }
      __syncthreads();
    }
  }
};

template <int S, class T, int R>
__global__ void __launch_bounds__(kFuseThreads)
    k_tail_down(const Tail<T> A, const T *__restrict__ u, const T *__restrict__ b, T *__restrict__ us,
                T *__restrict__ z, int steps) {
  constexpr int kGroups = kFuseThreads / kTailZ, kZ = 16;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int n = A.n, nc = A.nc, tid = threadIdx.x;
  T *x = reinterpret_cast<T *>(smem_raw), *w = x + tail_x(n, nc), *rl = w + n;
  TailRows<S, T, R> o;
  o.load(A);
#pragma unroll
  for (int i = 0; i < R; i++) {
    int r = tid + i * kFuseThreads;
    if (r < n) {
      x[r] = u ? u[r] : static_cast<T>(0);
      w[r] = b[r];
    }
  }
  if (tid == 0) x[n] = static_cast<T>(0);
  __syncthreads();
  o.rhs(w);
  __syncthreads();
  for (int it = 0; it < steps; it++) o.sweep(x, A.ncolors, false);
  // the thread's first half chunk of a row of Z and its row of the restriction,
  // on their way while the residual is formed
  const int zi = blockIdx.x * kTailZ + tid % kTailZ, g = tid / kTailZ, j0 = g * kZ;
  const bool direct = A.ZT != nullptr, zrow = direct && zi < nc;
  T zt[kZ];
  auto zload = [&](int k0, int k1) {
#pragma unroll
    for (int k = 0; k < kZ; k++)
      if (k >= k0 && k < k1)
        zt[k] = zrow && j0 + k < nc ? A.ZT[static_cast<size_t>(j0 + k) * nc + zi] : static_cast<T>(0);
  };
  zload(0, kZ / 2);
  const bool pre = A.rwidth <= 8 && tid < nc;
  int rc[8];
  T rv[8];
#pragma unroll
  for (int k = 0; k < 8; k++) {
    rc[k] = -1;
    rv[k] = static_cast<T>(0);
    if (pre && k < A.rwidth) {
      rc[k] = A.rcol[static_cast<size_t>(k) * nc + tid];
      rv[k] = A.rval[static_cast<size_t>(k) * nc + tid];
    }
  }
#pragma unroll
  for (int i = 0; i < R; i++) {
    if (o.color(i) == 15) continue;
    int at = (o.ix[i].x >> 12) & 0xf;
    T acc = static_cast<T>(0), dx = o.d[i] * x[o.row(i)];
#pragma unroll
    for (int k = 0; k < S; k++) {
      if (k == at) acc = acc + dx;
      acc = acc + o.off[i][k] * x[o.slot(i, k)];
    }
    if (at >= S) acc = acc + dx;
    w[o.row(i)] = o.b[i] - acc;
  }
  zload(kZ / 2, kZ);
  for (int r = blockIdx.x * kFuseThreads + tid; r < n; r += static_cast<int>(gridDim.x) * kFuseThreads) us[r] = x[r];
  __syncthreads();
  for (int i = tid; i < nc; i += kFuseThreads) {
    T acc = static_cast<T>(0);
    if (i == tid && pre) {
#pragma unroll
      for (int k = 0; k < 8; k++)
        if (rc[k] >= 0) acc = acc + rv[k] * w[rc[k]];
    } else {
      acc = dec_ell::row<0, T, T>(nc, A.rwidth, i, A.rcol, A.rval, w);
    }
    if (direct) rl[i] = acc;
    else z[i] = acc;
  }
  if (!direct) return;
  __syncthreads();
  const int nch = coarse_chunks(nc);
  if (zrow && g < nch) {
    T acc = static_cast<T>(0);
#pragma unroll
    for (int k = 0; k < kZ; k++)
      if (j0 + k < nc) acc = acc + zt[k] * rl[j0 + k];
    x[g * kTailZ + tid % kTailZ] = acc;
    for (int c = g + kGroups; c < nch; c += kGroups) {
      acc = static_cast<T>(0);
#pragma unroll 8
      for (int j = c * kZ; j < min(nc, (c + 1) * kZ); j++) acc = acc + A.ZT[static_cast<size_t>(j) * nc + zi] * rl[j];
      x[c * kTailZ + tid % kTailZ] = acc;
    }
  }
  __syncthreads();
  if (tid < kTailZ && zrow) {
    T t = static_cast<T>(0);
#pragma unroll 8
    for (int c = 0; c < nch; c++) t = t + x[c * kTailZ + tid];
    z[zi] = t;
  }
}

template <int S, class T, int R>
__global__ void __launch_bounds__(kFuseThreads)
    k_tail_up(const Tail<T> A, const T *__restrict__ us, const T *__restrict__ z, const T *__restrict__ b,
              T *__restrict__ u, int steps) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int n = A.n, nc = A.nc, tid = threadIdx.x;
  T *x = reinterpret_cast<T *>(smem_raw), *w = x + tail_x(n, nc), *rl = w + n;
  TailRows<S, T, R> o;
  int pc[R][2];
  T pv[R][2], ur[R];
#pragma unroll
  for (int i = 0; i < R; i++) {
    int r = tid + i * kFuseThreads, rc = min(r, n - 1);
    ur[i] = us[rc];
#pragma unroll
    for (int k = 0; k < 2; k++) {
      pc[i][k] = A.pwidth == 2 ? A.pcol[static_cast<size_t>(k) * n + rc] : -1;
      pv[i][k] = A.pwidth == 2 ? A.pval[static_cast<size_t>(k) * n + rc] : static_cast<T>(0);
    }
    if (r < n) w[r] = b[r];
  }
  for (int i = tid; i < nc; i += kFuseThreads) rl[i] = z[i];
  if (tid == 0) x[n] = static_cast<T>(0);
  o.load(A);
  __syncthreads();
  o.rhs(w);
#pragma unroll
  for (int i = 0; i < R; i++) {
    int r = tid + i * kFuseThreads;
    if (r >= n) continue;
    T acc = static_cast<T>(0);
    if (A.pwidth == 2) {
#pragma unroll
      for (int k = 0; k < 2; k++)
        if (pc[i][k] >= 0) acc = acc + pv[i][k] * rl[pc[i][k]];
    } else {
      acc = dec_ell::row<0, T, T>(n, A.pwidth, r, A.pcol, A.pval, rl);
    }
    x[r] = ur[i] + acc;
  }
  __syncthreads();
  for (int it = 0; it < steps; it++) o.sweep(x, A.ncolors, true);
#pragma unroll
  for (int i = 0; i < R; i++) {
    int r = tid + i * kFuseThreads;
    if (r < n) u[r] = x[r];
  }
}

// ---------------------------------------------------------------- storage

template <class T>
struct LevelVals {
  DBuf<T> val;   // ELL values of A (colour-sorted rows)
  DBuf<T> vval;  // the same rows in vertex order (residuals and the CG product)
  DBuf<T> rval;  // ELL values of R (this level -> next coarser)
  DBuf<T> pval;  // ELL values of P (next coarser -> this level)
  DBuf<T> poff, pdiag;  // values of the Gauss-Seidel panels (k_panel_sweep)
  DBuf<T> pown_w, phalo_w;  // and P's values, two per row and per halo row
  DBuf<T> toff, tdiag;  // values of the coarse tail's rows (Tail)
  DBuf<T> Z;     // dense coarse operator, column-major (coarsest level, direct solve)
  DBuf<T> zpart; // chunk partial products of the direct solve (coarsest level)
  DBuf<T> u, b, r, t;  // work vectors
};

// Every level keeps its own vertex numbering (internal numbers): vertices are
// grouped into blocks grown breadth-first over the operator's graph, each
// block a contiguous range, so that a block is a compact patch of the mesh
// (few neighbours outside it) and its vectors are contiguous.  The caller's
// order is restored at the boundary (solve, cycles, full multigrid); host
// copies and exports stay in the caller's order.  A level of at most
// fuse_rows rows is one block and keeps the caller's order.
struct Level {
  int n = 0, width = 0;
  DBuf<int32_t> col, rowid;  // ELL of A over internal numbers, rows sorted by (colour, vertex)
  DBuf<int32_t> vcol;        // the same ELL with rows in vertex order (same slots)
  std::vector<int> cstart;  // colour ranges of positions
  int ncolors = 0;
  // restriction to the next coarser level (rows: coarse internal numbers)
  int nc = 0, rwidth = 0;
  DBuf<int32_t> rcol;
  // prolongation from the next coarser level (rows: this level's internal numbers)
  int pwidth = 0;
  DBuf<int32_t> pcol;
  LevelVals<double> d;
  LevelVals<float> f;
  dec::HostCsr A, R, P;  // host copies for export (caller's numbering)
  std::vector<int32_t> color;  // Gauss-Seidel colour of each vertex (caller's numbering)
  std::vector<double> Zh;
  // numbering: perm[i] = caller's index of internal vertex i, iperm its inverse
  std::vector<int32_t> perm, iperm;
  bool identity = true;
  DBuf<int32_t> dperm;
  // hybrid block Gauss-Seidel: block ranges and (colour, block) ELL segments
  int nblk = 0, bmax = 0, seg_threads = 64;
  DBuf<int32_t> bstart, seg;
  std::vector<int32_t> hbstart;
  // panels of the sweep (panel_hs < 0: none), see Panels
  int panel_b = 0, panel_full = 0, panel_hs = -1;
  DBuf<uint32_t> pidx;
  DBuf<int32_t> phalo, pown_p, phalo_p;
  DBuf<uint32_t> tidx;  // the coarse tail's rows (empty: not one), see Tail
};

}  // namespace

struct dec_mg_s {
  std::vector<std::unique_ptr<dec_mesh_s>> meshes;  // finest first
  std::vector<std::unique_ptr<Level>> lv;            // finest first
  int alg = DEC_SMOOTH_CG, steps = 3, coarse_direct = 0;
  double omega = 2.0 / 3.0;
  DBuf<double> part, part2, scal;  // reduction partials, scalar outputs
  DBuf<CgState> cg;
  DBuf<double> cgx, cgr, cgp, cgp2, cgAp, cgAp2;  // CG vectors (finest size; r, p and Ap double-buffered)
  int fuse_from = -1;           // first level handled by the fused coarse kernel
  DBuf<LevelDesc<double>> desc64;
  DBuf<LevelDesc<float>> desc32;
  bool use_fused = true;
  int fuse_rows = kFuseRowsDefault;
  // graph of one solve cycle or preconditioned-CG iteration (per variant)
  // for fixed u, b
  static constexpr int kGraphs = 4;
  hipGraphExec_t gexec[kGraphs] = {};
  hipGraph_t graph[kGraphs] = {};
  const void *gu[kGraphs] = {}, *gb[kGraphs] = {};
  int gkey[kGraphs] = {-1, -1, -1, -1};
  // preconditioned CG on the finest level: residual, preconditioned residual,
  // direction, A times the direction, the partial sums
  // of r·z, p·q and r·r (at most one per workgroup of the finest level's
  // element launches) and the scalars (r·z)_prev, r·z, α
  DBuf<double> pcg_r, pcg_z, pcg_p, pcg_q, pcg_part, pcg_sc;
  hipStream_t cap = nullptr;
  bool use_graph = true;
  // where the finest level's last post-sweep puts its blocks' sums of b u
  // (set while a preconditioned-CG iteration is queued, else null)
  double *sweep_dot = nullptr;
  double *sweep_add = nullptr;  // the float64 iterate that takes the finest level's last float32 sweep
  // residual norms of a solve on their way to the host (pinned ring + events)
  DBuf<double> rpart;  // per-workgroup partial sums of the finest residual's r²
  // (slot kNormSlots: ||b||^2 of the solve)
  double *hnorm = nullptr;
  hipEvent_t nev[kNormSlots + 1] = {};
  // learned smoother (float32 cycles, levels of learned_min_rows to
  // learned_max_rows rows; learned_max_rows <= 0: no upper bound)
  dec_nn_s *nn = nullptr;
  int learned = 0, learned_min_rows = 16385, learned_max_rows = 0, learned_apps = 1;
  bool learned_active = false;
  int fallbacks = 0, learned_cycles = 0;
  ~dec_mg_s() {
    for (int i = 0; i < kGraphs; i++) {
      if (gexec[i]) (void)hipGraphExecDestroy(gexec[i]);
      if (graph[i]) (void)hipGraphDestroy(graph[i]);
    }
    if (cap) (void)hipStreamDestroy(cap);
    for (auto &e : nev)
      if (e) (void)hipEventDestroy(e);
    if (hnorm) (void)hipHostFree(hnorm);
  }
};

namespace {

inline dim3 G(long long n) { return dim3(dec::nblocks(n, kBlock)); }

template <class T>
LevelVals<T> &vals(Level &L);
template <>
LevelVals<double> &vals<double>(Level &L) { return L.d; }
template <>
LevelVals<float> &vals<float>(Level &L) { return L.f; }

// Symmetric adjacency (CSR, no diagonal) of the sparsity pattern of A.
void adjacency(const dec::HostCsr &A, std::vector<int32_t> &deg, std::vector<int32_t> &adj) {
  int n = A.m;
  deg.assign(n + 1, 0);
  for (int r = 0; r < n; r++)
    for (int k = A.ptr[r]; k < A.ptr[r + 1]; k++)
      if (A.col[k] != r) {
        deg[r + 1]++;
        deg[A.col[k] + 1]++;
      }
  for (int r = 0; r < n; r++) deg[r + 1] += deg[r];
  adj.assign(deg[n], 0);
  std::vector<int32_t> w(deg.begin(), deg.end() - 1);
  for (int r = 0; r < n; r++)
    for (int k = A.ptr[r]; k < A.ptr[r + 1]; k++)
      if (A.col[k] != r) {
        adj[w[r]++] = A.col[k];
        adj[w[A.col[k]]++] = r;
      }
}

// Blocks of about B vertices grown breadth-first over the symmetric graph
// (deg, adj) of a level's operator: a block grows from its seed until it
// holds B vertices, and the next block is seeded next to it (from the
// unassigned neighbours of the last block's BFS frontier, else the lowest
// unassigned vertex), so consecutive blocks are neighbours.  perm lists the
// vertices block by block in BFS order; bstart holds the block ranges.  Blocks
// of exactly B vertices come first (about seven of eight; the others are what
// growing left between them), each kind in the order it grew, so that a full
// block's range follows from its number; returns how many are full.
int grow_blocks(int n, const std::vector<int32_t> &deg, const std::vector<int32_t> &adj, int B,
                std::vector<int32_t> &perm, std::vector<int32_t> &bstart) {
  std::vector<int32_t> blk(n, -1);
  perm.clear();
  perm.reserve(n);
  bstart.assign(1, 0);
  std::vector<int32_t> seeds, queue;
  size_t sh = 0;
  int next = 0, nb = 0;
  while (static_cast<int>(perm.size()) < n) {
    int seed = -1;
    while (sh < seeds.size() && seed < 0) {
      int c = seeds[sh++];
      if (blk[c] < 0) seed = c;
    }
    if (seed < 0) {
      while (next < n && blk[next] >= 0) next++;
      seed = next;
    }
    queue.clear();
    queue.push_back(seed);
    blk[seed] = nb;
    size_t qh = 0;
    int cnt = 1;
    while (qh < queue.size() && cnt < B) {
      int v = queue[qh++];
      for (int k = deg[v]; k < deg[v + 1] && cnt < B; k++) {
        int w = adj[k];
        if (blk[w] < 0) {
          blk[w] = nb;
          cnt++;
          queue.push_back(w);
        }
      }
    }
    seeds.clear();
    sh = 0;
    for (size_t q = qh; q < queue.size(); q++)
      for (int k = deg[queue[q]]; k < deg[queue[q] + 1]; k++)
        if (blk[adj[k]] < 0) seeds.push_back(adj[k]);
    perm.insert(perm.end(), queue.begin(), queue.end());
    bstart.push_back(static_cast<int32_t>(perm.size()));
    nb++;
  }
  std::vector<int32_t> grown;
  grown.swap(perm);
  std::vector<int32_t> at;
  at.swap(bstart);
  bstart.assign(1, 0);
  int nfull = 0;
  for (int full = 1; full >= 0; full--)
    for (int k = 0; k < nb; k++)
      if ((at[k + 1] - at[k] == B) == (full == 1)) {
        perm.insert(perm.end(), grown.begin() + at[k], grown.begin() + at[k + 1]);
        bstart.push_back(static_cast<int32_t>(perm.size()));
        nfull += full;
      }
  return nfull;
}

// Block size of the hybrid Gauss-Seidel: the largest power of two from 64 to
// 512 rows that still gives at least 640 blocks (2.5 per CU).  The
// icosphere levels hold 10 * 4^k + 2 rows, just above a power of two: at
// 163,842 rows the rule picks 256-row blocks (640 blocks), where a threshold
// of "b * 640 < n" picked 512 (320 blocks), and the 3->8 solve takes 2.01
// against 2.14 ms.
int block_rows(int n) {
  int b = 64;
  while (b < 512 && n / (2 * b) >= 640) b *= 2;
  return b;
}
// threads of a block's workgroup in k_panel_sweep: one row each up to 256
int panel_threads(int b) { return std::min(kBlock, b); }

void to_float(const DBuf<double> &x, DBuf<float> &y) {
  if (y.n != x.n) y.alloc(x.n);
  if (x.n) hipLaunchKernelGGL(k_to_float, dim3(dec::nblocks(static_cast<long long>(x.n))), dim3(256), 0, 0, x.n, x.p, y.p);
}

// The panels of k_panel_sweep, or none: rows of 2 to 8 slots with a diagonal entry, at
// most 16 colours (4 bits), and halos that two loads per thread cover.
void build_panels(Level &L, const std::vector<int32_t> &color) {
  const dec::HostCsr &A = L.A;
  const int n = L.n, B = L.panel_b, nb = L.nblk, S = L.width - 1;
  if (L.width < 2 || L.width > 8 || L.ncolors > 16) return;
  const int most = 2 * panel_threads(B) - 1;  // (and the zero behind the halo)
  std::vector<int32_t> order(n), stamp(n, -1), halo, count(nb), first(nb + 1, 0);
  int hs = 1;
  for (int k = 0; k < nb; k++) {
    int r0 = L.hbstart[k], r1 = L.hbstart[k + 1];
    // rows by colour, then by number
    int at[17] = {0};
    for (int i = r0; i < r1; i++) at[color[L.perm[i]] + 1]++;
    for (int c = 0; c < 16; c++) at[c + 1] += at[c];
    for (int i = r0; i < r1; i++) order[r0 + at[color[L.perm[i]]]++] = i;
    size_t h0 = halo.size();
    for (int i = r0; i < r1; i++) {
      int v = L.perm[i], off = 0;
      for (int q = A.ptr[v]; q < A.ptr[v + 1]; q++) {
        if (A.col[q] == v) continue;
        off++;
        int c = L.iperm[A.col[q]];
        if ((c < r0 || c >= r1) && stamp[c] != k) {
          stamp[c] = k;
          halo.push_back(c);
        }
      }
      if (off > S) return;
    }
    std::sort(halo.begin() + h0, halo.end());
    count[k] = static_cast<int>(halo.size() - h0);
    first[k + 1] = static_cast<int>(halo.size());
    hs = std::max(hs, count[k]);
    if (hs > most) return;
  }
  std::vector<int32_t> list(static_cast<size_t>(nb) * hs);
  for (int k = 0; k < nb; k++)
    for (int j = 0; j < hs; j++)
      list[static_cast<size_t>(k) * hs + j] = j < count[k] ? halo[first[k] + j] : L.hbstart[k];
  std::vector<signed char> vcl(n);
  for (int i = 0; i < n; i++) vcl[i] = static_cast<signed char>(color[L.perm[i]]);
  DBuf<int32_t> dorder, dcount;
  DBuf<signed char> dcolor;
  dorder.upload(order);
  dcount.upload(count);
  dcolor.upload(vcl);
  L.panel_hs = hs;
  L.phalo.upload(list);
  L.pidx.alloc(4 * static_cast<size_t>(n));
  L.d.poff.alloc(static_cast<size_t>(n) * S);
  L.d.pdiag.alloc(n);
  hipLaunchKernelGGL(k_build_panels, dim3(nb), dim3(256), 0, 0, n, L.width, B, hs, L.vcol.p, L.d.vval.p, dorder.p,
                     dcolor.p, L.bstart.p, L.phalo.p, dcount.p, reinterpret_cast<uint4 *>(L.pidx.p), L.d.poff.p,
                     L.d.pdiag.p);
  to_float(L.d.poff, L.f.poff);
  to_float(L.d.pdiag, L.f.pdiag);
  dec::check_launch("multigrid panels");
}

// The rows of the coarse tail (see Tail) of a level that can be one: every row
// with a diagonal, at most 7 other entries, vectors that fit in 64 KiB of LDS, and
// above the dense coarsest level its product in chunks of 16.
void build_tail(Level &L, const LevelDesc<double> &D, bool above_dense) {
  const int n = L.n, S = std::max(L.width - 1, 1);
  if (n < 1 || n > kTailRows || L.width < 1 || L.width > 8 || L.ncolors > 15 || L.nc < 1 ||
      (above_dense && coarse_chunk(L.nc) != 16) || tail_lds(n, L.nc, sizeof(double)) > 64 * 1024)
    return;
  for (int r = 0; r < n; r++) {
    int diag = 0;
    for (int q = L.A.ptr[r]; q < L.A.ptr[r + 1]; q++) diag += L.A.col[q] == r;
    if (diag != 1 || L.A.ptr[r + 1] - L.A.ptr[r] - 1 > S) return;
  }
  L.tidx.alloc(4 * static_cast<size_t>(n));
  L.d.toff.alloc(static_cast<size_t>(S) * n);
  L.d.tdiag.alloc(n);
  hipLaunchKernelGGL(k_build_tail, dim3(dec::nblocks(n)), dim3(256), 0, 0, D, S, reinterpret_cast<uint4 *>(L.tidx.p),
                     L.d.toff.p, L.d.tdiag.p);
  auto to_float = [](const DBuf<double> &x, DBuf<float> &y) {
    y.alloc(x.n);
    hipLaunchKernelGGL(k_to_float, dim3(dec::nblocks(static_cast<long long>(x.n))), dim3(256), 0, 0, x.n, x.p, y.p);
  };
  to_float(L.d.toff, L.f.toff);
  to_float(L.d.tdiag, L.f.tdiag);
  dec::check_launch("multigrid tail");
}

// P's rows (width 2) of a level's own rows and of its panels' halos, for the
// sweep that adds the coarse correction itself.
template <class T>
void panel_transfer(Level &L) {
  LevelVals<T> &V = vals<T>(L);
  using V2 = typename Vec2T<T>::type;
  auto rows = [&](size_t m, const int *ids, DBuf<int32_t> &c, DBuf<T> &w) {
    if (c.n != 2 * m) c.alloc(2 * m);
    w.alloc(2 * m);
    hipLaunchKernelGGL(k_panel_p<T>, dim3(dec::nblocks(static_cast<long long>(m))), dim3(256), 0, 0,
                       static_cast<int>(m), L.n, ids, L.pcol.p, V.pval.p, reinterpret_cast<int2 *>(c.p),
                       reinterpret_cast<V2 *>(w.p));
  };
  rows(L.n, nullptr, L.pown_p, V.pown_w);
  rows(L.phalo.n, L.phalo.p, L.phalo_p, V.phalo_w);
}

// Colour-sorted ELL of a host CSR (caller's numbering) over the level's
// internal numbers.  `color` is the proposed Gauss-Seidel colouring (empty:
// none); a proposal that is not a proper colouring of A's pattern is replaced
// by greedy colours.  On return `color` holds the colouring used.  A level of
// more than `block_min` rows is renumbered into BFS-grown blocks; slots keep
// the caller's ascending column order, so row sums are those of A.
void build_level_matrix(Level &L, const dec::HostCsr &A, std::vector<int32_t> &color, int block_min) {
  int n = A.m;
  L.n = n;
  std::vector<int32_t> deg, adj;
  adjacency(A, deg, adj);
  int nc = 0;
  for (int c : color) nc = std::max(nc, c + 1);
  if (color.empty() || !dec::proper_coloring(n, deg, adj, color, nc)) nc = dec::greedy_colors(n, deg, adj, color);
  L.ncolors = nc;
  L.color = color;
  std::vector<int32_t> bstart;
  if (n > block_min) {
    L.panel_b = block_rows(n);
    L.panel_full = grow_blocks(n, deg, adj, L.panel_b, L.perm, bstart);
  } else {
    L.perm.resize(n);
    for (int v = 0; v < n; v++) L.perm[v] = v;
    bstart = {0, n};
  }
  L.iperm.assign(n, 0);
  L.identity = true;
  for (int i = 0; i < n; i++) {
    L.iperm[L.perm[i]] = i;
    L.identity = L.identity && L.perm[i] == i;
  }
  L.dperm.upload(L.perm);
  // positions: rows sorted by (colour, internal number)
  std::vector<int32_t> order(n);
  L.cstart.assign(L.ncolors + 1, 0);
  for (int v = 0; v < n; v++) L.cstart[color[v] + 1]++;
  for (int c = 0; c < L.ncolors; c++) L.cstart[c + 1] += L.cstart[c];
  std::vector<int32_t> pos(L.cstart.begin(), L.cstart.end() - 1);
  for (int i = 0; i < n; i++) order[pos[color[L.perm[i]]]++] = i;
  // (colour, block) segments of the positions
  int nb = static_cast<int>(bstart.size()) - 1;
  L.nblk = nb;
  L.bmax = 0;
  for (int k = 0; k < nb; k++) L.bmax = std::max(L.bmax, bstart[k + 1] - bstart[k]);
  std::vector<int32_t> seg(static_cast<size_t>(L.ncolors) * (nb + 1));
  {
    std::vector<int32_t> blk_of(n);
    for (int k = 0; k < nb; k++)
      for (int i = bstart[k]; i < bstart[k + 1]; i++) blk_of[i] = k;
    std::vector<int32_t> cnt(static_cast<size_t>(L.ncolors) * nb, 0);
    for (int i = 0; i < n; i++) cnt[static_cast<size_t>(color[L.perm[i]]) * nb + blk_of[i]]++;
    for (int c = 0; c < L.ncolors; c++) {
      int p = L.cstart[c];
      for (int k = 0; k < nb; k++) {
        seg[static_cast<size_t>(c) * (nb + 1) + k] = p;
        p += cnt[static_cast<size_t>(c) * nb + k];
      }
      seg[static_cast<size_t>(c) * (nb + 1) + nb] = p;
    }
    // threads per block of the sweep kernel: one per row of the largest
    // (colour, block) segment, in whole wavefronts, at most 256
    int smax = 0;
    for (int c : cnt) smax = std::max(smax, c);
    L.seg_threads = std::min(256, std::max(64, (smax + 63) / 64 * 64));
  }
  L.bstart.upload(bstart);
  L.seg.upload(seg);
  L.hbstart = bstart;
  int width = 0;
  for (int r = 0; r < n; r++) width = std::max(width, A.ptr[r + 1] - A.ptr[r]);
  L.width = width;
  // rows in vertex order, for the kernels that sweep no colours: their vector
  // accesses are then contiguous, where colour-sorted rows touch every cache
  // line of a vector once per colour
  size_t sz = static_cast<size_t>(n) * std::max(width, 1);
  std::vector<int32_t> col(sz, -1);
  std::vector<double> vd(sz, 0.0);
  for (int i = 0; i < n; i++) {
    int r = L.perm[i];
    for (int k = A.ptr[r]; k < A.ptr[r + 1]; k++) {
      size_t q = static_cast<size_t>(k - A.ptr[r]) * n + i;
      col[q] = L.iperm[A.col[k]];
      vd[q] = A.val[k];
    }
  }
  L.vcol.upload(col);
  L.d.vval.upload(vd);
  L.rowid.upload(order);
  // the colour-sorted rows and the float values follow on the device
  L.col.alloc(sz);
  L.d.val.alloc(sz);
  L.f.val.alloc(sz);
  L.f.vval.alloc(sz);
  if (n > 0) {
    hipLaunchKernelGGL(k_order_rows, dim3(dec::nblocks(n)), dim3(256), 0, 0, n, std::max(width, 1), L.rowid.p,
                       L.vcol.p, L.d.vval.p, L.col.p, L.d.val.p);
    to_float(L.d.val, L.f.val);
    to_float(L.d.vval, L.f.vval);
  }
  L.A = A;
  if (n > block_min) build_panels(L, color);
}

// make_restriction(transpose(S)) (Multigrid.jl:595-612) as rows of R, and the
// endpoints of P = transpose(S) = subdivision_matrix(BinarySubdivision) (:191-219).
// R = row-normalised S and P = Sᵀ of one binary refinement of `coarse`
// (Multigrid.jl:191-219, 595-612); pa, pb are the endpoints of each midpoint.
void transfer_csr(const dec::Topo &coarse, dec::HostCsr &R, dec::HostCsr &P, std::vector<int32_t> &pa,
                  std::vector<int32_t> &pb) {
  int nc = coarse.nv, ne = coarse.ne, nf = nc + ne;
  std::vector<std::vector<int32_t>> mids(nc);
  pa.assign(ne, 0);
  pb.assign(ne, 0);
  for (int e = 0; e < ne; e++) {
    int a = std::min(coarse.v0[e], coarse.v1[e]), b = std::max(coarse.v0[e], coarse.v1[e]);
    pa[e] = a;
    pb[e] = b;
    mids[a].push_back(nc + e);
    if (b != a) mids[b].push_back(nc + e);
  }
  R = dec::HostCsr();
  R.m = nc;
  R.n = nf;
  R.ptr.assign(nc + 1, 0);
  for (int i = 0; i < nc; i++) {
    double rs = 1.0;  // row sum in storage order: 1.0, then 0.5 per midpoint
    for (size_t k = 0; k < mids[i].size(); k++) rs += 0.5;
    R.col.push_back(i);
    R.val.push_back(1.0 / rs);
    for (int c : mids[i]) {
      R.col.push_back(c);
      R.val.push_back(0.5 / rs);
    }
    R.ptr[i + 1] = static_cast<int32_t>(R.col.size());
  }
  P = dec::HostCsr();
  P.m = nf;
  P.n = nc;
  P.ptr.assign(nf + 1, 0);
  for (int j = 0; j < nf; j++) {
    if (j < nc) {
      P.col.push_back(j);
      P.val.push_back(1.0);
    } else {
      P.col.push_back(pa[j - nc]);
      P.val.push_back(0.5);
      P.col.push_back(pb[j - nc]);
      P.val.push_back(0.5);
    }
    P.ptr[j + 1] = static_cast<int32_t>(P.col.size());
  }
}

// Slot-major ELL of a host CSR with rows and columns renumbered: row i is
// CSR row rperm[i], columns map through cimap; slots keep the CSR order.
void ell_renumbered(const dec::HostCsr &M, const std::vector<int32_t> &rperm, const std::vector<int32_t> &cimap,
                    int &width, std::vector<int32_t> &col, std::vector<double> &val) {
  int m = M.m;
  width = 0;
  for (int r = 0; r < m; r++) width = std::max(width, M.ptr[r + 1] - M.ptr[r]);
  size_t sz = static_cast<size_t>(m) * std::max(width, 1);
  col.assign(sz, -1);
  val.assign(sz, 0.0);
  for (int i = 0; i < m; i++) {
    int r = rperm[i];
    for (int k = M.ptr[r]; k < M.ptr[r + 1]; k++) {
      size_t q = static_cast<size_t>(k - M.ptr[r]) * m + i;
      col[q] = cimap[M.col[k]];
      val[q] = M.val[k];
    }
  }
}

// R (fine -> coarse) and P (coarse -> fine) of one level pair as ELL over
// the two levels' internal numbers; R and P are host CSRs in the caller's
// numbering, kept for export.
void set_transfer(Level &fine, const Level &coarse, dec::HostCsr R, dec::HostCsr P) {
  if (R.m != coarse.n || R.n != fine.n || P.m != fine.n || P.n != coarse.n)
    fail(DEC_ERR_ARG, "multigrid: transfer operator shapes do not match the levels");
  fine.nc = coarse.n;
  std::vector<int32_t> col;
  std::vector<double> vd;
  ell_renumbered(R, coarse.perm, fine.iperm, fine.rwidth, col, vd);
  fine.rcol.upload(col);
  fine.d.rval.upload(vd);
  to_float(fine.d.rval, fine.f.rval);
  ell_renumbered(P, fine.perm, coarse.iperm, fine.pwidth, col, vd);
  fine.pcol.upload(col);
  fine.d.pval.upload(vd);
  to_float(fine.d.pval, fine.f.pval);
  if (fine.panel_hs >= 0 && fine.pwidth == 2) {
    panel_transfer<double>(fine);
    panel_transfer<float>(fine);
  }
  fine.R = std::move(R);
  fine.P = std::move(P);
}

void build_transfer(Level &fine, const Level &coarse, const dec::Topo &coarse_topo) {
  dec::HostCsr R, P;
  std::vector<int32_t> pa, pb;
  transfer_csr(coarse_topo, R, P, pa, pb);
  set_transfer(fine, coarse, std::move(R), std::move(P));
}

void alloc_work(Level &L) {
  for (auto *v : {&L.d.u, &L.d.b, &L.d.r, &L.d.t}) v->alloc(L.n);
  for (auto *v : {&L.f.u, &L.f.b, &L.f.r, &L.f.t}) v->alloc(L.n);
}

dec_mesh_s *copy_mesh(const dec_mesh_s &m) {
  auto *c = new dec_mesh_s();
  c->h = m.h;
  c->hp = m.hp;
  c->to_dfs = m.to_dfs;
  c->v0.upload(c->h.v0);
  c->v1.upload(c->h.v1);
  c->e0.upload(c->h.e0);
  c->e1.upload(c->h.e1);
  c->e2.upload(c->h.e2);
  c->p.upload(c->hp);
  return c;
}

// Gauss-Seidel colours of every level (finest first), four per level where
// possible.  The base level is 4-coloured by search.  A proper colouring c of
// a level with values in {0,1,2,3} colours the next finer level properly:
// coarse vertices take 0 and the midpoint of coarse edge (a, b) takes
// c(a) ^ c(b), which is nonzero because a and b are adjacent; two midpoints
// are adjacent only when their edges (a, b), (b, z) bound a common coarse
// triangle, and c(a) ^ c(b) = c(b) ^ c(z) would force c(a) = c(z) for the
// adjacent a, z; coarse vertices are never adjacent on the finer level.
// A level without a proposal (or whose proposal fails the check in
// build_level_matrix) is coloured greedily.
std::vector<std::vector<int32_t>> level_colors(const dec_mg_s &mg, const std::vector<dec::HostCsr> &As) {
  int nl = static_cast<int>(As.size());
  std::vector<std::vector<int32_t>> colors(nl);
  const dec::HostCsr &Ab = As[nl - 1];
  if (Ab.m <= 65536) {
    std::vector<int32_t> deg, adj;
    adjacency(Ab, deg, adj);
    if (!dec::four_colors(Ab.m, deg, adj, colors[nl - 1], 64L * Ab.m + 4096)) colors[nl - 1].clear();
  }
  for (int l = nl - 2; l >= 0; l--) {
    const std::vector<int32_t> &cc = colors[l + 1];
    if (cc.empty()) break;
    const dec::Topo &coarse = mg.meshes[l + 1]->h;
    int nc = coarse.nv;
    std::vector<int32_t> &cf = colors[l];
    cf.assign(static_cast<size_t>(nc) + coarse.ne, 0);
    for (int e = 0; e < coarse.ne; e++) cf[nc + e] = cc[coarse.v0[e]] ^ cc[coarse.v1[e]];
  }
  return colors;
}

// Levels, transfers, the dense coarse operator and the fused-tail
// descriptors of a hierarchy, from its operators (caller's numbering, finest
// first), R_l / P_l between levels l and l+1, and proposed colourings.
void finish_hierarchy(dec_mg_s &mg, const std::vector<dec::HostCsr> &As, std::vector<dec::HostCsr> &Rs,
                      std::vector<dec::HostCsr> &Ps, std::vector<std::vector<int32_t>> &colors) {
  int nl = static_cast<int>(As.size());
  for (int l = 0; l < nl; l++) {
    auto L = std::make_unique<Level>();
    build_level_matrix(*L, As[l], colors[l], mg.fuse_rows);
    alloc_work(*L);
    mg.lv.push_back(std::move(L));
  }
  for (int l = 0; l + 1 < nl; l++) set_transfer(*mg.lv[l], *mg.lv[l + 1], std::move(Rs[l]), std::move(Ps[l]));
  // dense coarse operator for the direct solve (over the level's internal numbers)
  Level &C = *mg.lv.back();
  int n = C.n;
  if (static_cast<long long>(n) * n <= 64LL * 1024 * 1024) {
    std::vector<double> Ad(static_cast<size_t>(n) * n, 0.0);
    for (int r = 0; r < n; r++)
      for (int k = C.A.ptr[r]; k < C.A.ptr[r + 1]; k++) Ad[static_cast<size_t>(r) * n + C.A.col[k]] += C.A.val[k];
    dec::coarse_inverse(n, Ad, C.Zh);
    std::vector<double> zt(C.Zh.size());
    for (int i = 0; i < n; i++)
      for (int j = 0; j < n; j++)
        zt[static_cast<size_t>(j) * n + i] = C.Zh[static_cast<size_t>(C.perm[i]) * n + C.perm[j]];
    C.d.Z.upload(zt);
    std::vector<float> zf(zt.begin(), zt.end());
    C.f.Z.upload(zf);
    C.d.zpart.alloc(static_cast<size_t>(coarse_chunks(n)) * n);
    C.f.zpart.alloc(static_cast<size_t>(coarse_chunks(n)) * n);
  }
  // descriptors of the coarse tail for the fused kernel
  for (int l = 0; l < nl; l++)
    if (mg.lv[l]->n <= mg.fuse_rows && mg.lv[l]->ncolors <= kMaxColors) {
      bool ok = true;
      for (int q = l; q < nl; q++) ok = ok && mg.lv[q]->n <= mg.fuse_rows && mg.lv[q]->ncolors <= kMaxColors;
      if (ok) {
        mg.fuse_from = l;
        break;
      }
    }
  {
    std::vector<LevelDesc<double>> d64(nl);
    std::vector<LevelDesc<float>> d32(nl);
    for (int l = 0; l < nl; l++) {
      Level &L = *mg.lv[l];
      auto fill = [&](auto &D, auto &V) {
        D.n = L.n;
        D.width = L.width;
        D.ncolors = L.ncolors;
        D.nc = L.nc;
        D.rwidth = L.rwidth;
        D.pwidth = L.pwidth;
        for (int c = 0; c <= kMaxColors; c++) D.cstart[c] = c < static_cast<int>(L.cstart.size()) ? L.cstart[c] : L.n;
        D.col = L.col.p;
        D.rowid = L.rowid.p;
        D.rcol = L.rcol.p;
        D.pcol = L.pcol.p;
        D.val = V.val.p;
        D.rval = V.rval.p;
        D.pval = V.pval.p;
        D.u = V.u.p;
        D.b = V.b.p;
        D.r = V.r.p;
      };
      fill(d64[l], L.d);
      fill(d32[l], L.f);
    }
    mg.desc64.upload(d64);
    mg.desc32.upload(d32);
    for (int l = 0; l + 1 < nl; l++) build_tail(*mg.lv[l], d64[l], l + 2 == nl);
  }
  mg.part.alloc(4 * kCgBlocksMax);  // also the dot partials (kDotBlocks of them)
  mg.part2.alloc(4 * kCgBlocksMax);
  mg.scal.alloc(8);
  mg.rpart.alloc(static_cast<size_t>(dec::nblocks(mg.lv[0]->n, kBlock)));
  if (hipHostMalloc(reinterpret_cast<void **>(&mg.hnorm), sizeof(double) * (kNormSlots + 1), hipHostMallocDefault) !=
      hipSuccess)
    fail(DEC_ERR_OOM, "multigrid: pinned host buffer");
  for (auto &e : mg.nev)
    if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) fail(DEC_ERR_HIP, "hipEventCreate failed");
  mg.cg.alloc(1);
  int nf = mg.lv[0]->n;
  for (auto *v : {&mg.cgx, &mg.cgr, &mg.cgp, &mg.cgp2, &mg.cgAp, &mg.cgAp2}) v->alloc(nf);
}

void env_switches(dec_mg_s &mg) {
  // debugging switches: run every phase as its own launch / launch cycles eagerly
  mg.use_fused = std::getenv("DEC_MG_NO_FUSE") == nullptr;
  if (const char *e = std::getenv("DEC_MG_FUSE_ROWS")) mg.fuse_rows = std::min(std::max(std::atoi(e), 0), kFuseRowsMax);
  mg.use_graph = std::getenv("DEC_MG_NO_GRAPH") == nullptr;
}

// A caller's m x n CSR (index_base 0 or 1) checked and copied 0-based.
dec::HostCsr csr_in(int m, int n, const int32_t *ptr, const int32_t *col, const double *val, int base,
                    const char *what) {
  if (!ptr || (!col && ptr[m] > ptr[0]) || (!val && ptr[m] > ptr[0]))
    fail(DEC_ERR_ARG, std::string("dec_mg_create_from_csr: NULL array for ") + what);
  dec::HostCsr A;
  A.m = m;
  A.n = n;
  A.ptr.resize(m + 1);
  for (int r = 0; r <= m; r++) {
    A.ptr[r] = ptr[r] - ptr[0];
    if (r > 0 && A.ptr[r] < A.ptr[r - 1])
      fail(DEC_ERR_ARG, std::string("dec_mg_create_from_csr: row pointers of ") + what + " decrease");
  }
  int nnz = A.ptr[m];
  A.col.resize(nnz);
  A.val.assign(val ? val : static_cast<const double *>(nullptr), val ? val + nnz : nullptr);
  for (int k = 0; k < nnz; k++) {
    int c = col[k] - base;
    if (c < 0 || c >= n) fail(DEC_ERR_ARG, std::string("dec_mg_create_from_csr: column out of range in ") + what);
    A.col[k] = c;
  }
  for (int r = 0; r < m; r++)
    for (int k = A.ptr[r] + 1; k < A.ptr[r + 1]; k++)
      if (A.col[k] == A.col[k - 1])
        fail(DEC_ERR_ARG, std::string("dec_mg_create_from_csr: repeated column in a row of ") + what);
  return A;
}

// MultigridData(ops, restrictions, prolongations, steps) (Multigrid.jl:545-546):
// a hierarchy from the caller's matrices, finest first.
dec_mg_s *mg_from_csr(int nl, const int32_t *sizes, const int32_t *const *ap, const int32_t *const *ac,
                      const double *const *av, const int32_t *const *rp, const int32_t *const *rc,
                      const double *const *rv, const int32_t *const *pp, const int32_t *const *pc,
                      const double *const *pv, int base, int steps) {
  if (nl < 1 || nl > 16) fail(DEC_ERR_ARG, "dec_mg_create_from_csr: 1 to 16 levels");
  if (!sizes || !ap || !ac || !av || (nl > 1 && (!rp || !rc || !rv || !pp || !pc || !pv)))
    fail(DEC_ERR_ARG, "dec_mg_create_from_csr: NULL argument");
  if (base != 0 && base != 1) fail(DEC_ERR_ARG, "dec_mg_create_from_csr: index_base must be 0 or 1");
  if (steps < 0) fail(DEC_ERR_ARG, "dec_mg_create_from_csr: steps must be >= 0");
  for (int l = 0; l < nl; l++)
    if (sizes[l] < 1) fail(DEC_ERR_ARG, "dec_mg_create_from_csr: empty level");
  auto mg = std::make_unique<dec_mg_s>();
  mg->steps = steps;
  env_switches(*mg);
  std::vector<dec::HostCsr> As(nl), Rs(nl - 1), Ps(nl - 1);
  for (int l = 0; l < nl; l++) {
    As[l] = csr_in(sizes[l], sizes[l], ap[l], ac[l], av[l], base, "an operator");
    bool diag = true;
    for (int r = 0; r < sizes[l] && diag; r++) {
      bool has = false;
      for (int k = As[l].ptr[r]; k < As[l].ptr[r + 1]; k++) has = has || (As[l].col[k] == r && As[l].val[k] != 0.0);
      diag = has;
    }
    if (!diag) fail(DEC_ERR_ARG, "dec_mg_create_from_csr: an operator has a zero diagonal entry");
  }
  for (int l = 0; l + 1 < nl; l++) {
    Rs[l] = csr_in(sizes[l + 1], sizes[l], rp[l], rc[l], rv[l], base, "a restriction");
    Ps[l] = csr_in(sizes[l], sizes[l + 1], pp[l], pc[l], pv[l], base, "a prolongation");
  }
  std::vector<std::vector<int32_t>> colors(nl);  // greedy colours per level
  finish_hierarchy(*mg, As, Rs, Ps, colors);
  return mg.release();
}

dec_mg_s *mg_create(const dec_mesh_s &base, int levels, bool project, int hodge, int center, int steps,
                    bool galerkin) {
  if (base.dim != 2) fail(DEC_ERR_UNSUPPORTED, "dec_mg_create: the multigrid hierarchy refines 2-D complexes");
  if (levels < 0 || levels > 11) fail(DEC_ERR_ARG, "dec_mg_create: levels must be in 0..11");
  if (steps < 0) fail(DEC_ERR_ARG, "dec_mg_create: steps must be >= 0");
  auto mg = std::make_unique<dec_mg_s>();
  mg->steps = steps;
  env_switches(*mg);
  // coarse -> fine walk (Multigrid.jl:752-797), stored finest first
  std::vector<std::unique_ptr<dec_mesh_s>> walk;
  walk.emplace_back(copy_mesh(base));
  for (int i = 0; i < levels; i++) walk.emplace_back(dec::subdivide(*walk.back(), project));
  for (int i = levels; i >= 0; i--) mg->meshes.push_back(std::move(walk[i]));
  int nl = levels + 1;
  std::vector<dec::HostCsr> As(nl);
  for (int l = 0; l < nl; l++) {
    dec_mesh_s &m = *mg->meshes[l];
    m.owned_by_mg = true;
    if (galerkin && l > 0) {
      // GalerkinMode: only the finest mesh is dualized; Aₖ₊₁ = (Rₖ Aₖ) Pₖ (Multigrid.jl:740-748)
      dec::HostCsr R, P, RA;
      std::vector<int32_t> pa, pb;
      transfer_csr(m.h, R, P, pa, pb);
      dec::spgemm(R, As[l - 1], RA);
      dec::spgemm(RA, P, As[l]);
      continue;
    }
    dec::dualize(m, center);
    std::vector<double> h0 = m.h0.download(), h1 = m.h1.download(), ih0(m.h.nv);
    for (int v = 0; v < m.h.nv; v++) ih0[v] = 1 / h0[v];
    if (hodge == DEC_GEOMETRIC_HODGE) {
      dec::HostCsr H;
      dec::geo_hodge1(m, H);
      dec::assemble_laplacian0(m.h, ih0, h1, &H, As[l]);
    } else {
      dec::assemble_laplacian0(m.h, ih0, h1, nullptr, As[l]);
    }
  }
  std::vector<std::vector<int32_t>> colors = level_colors(*mg, As);
  std::vector<dec::HostCsr> Rs(nl > 0 ? nl - 1 : 0), Ps(nl > 0 ? nl - 1 : 0);
  for (int l = 0; l + 1 < nl; l++) {
    std::vector<int32_t> pa, pb;
    transfer_csr(mg->meshes[l + 1]->h, Rs[l], Ps[l], pa, pb);
  }
  finish_hierarchy(*mg, As, Rs, Ps, colors);
  dec::check_launch("dec_mg_create");
  dec::dsync();
  return mg.release();
}



// ---------------------------------------------------------------- cycles

template <class T>
void residual(Level &L, const T *b, const T *u, T *r, hipStream_t s) {
  LevelVals<T> &V = vals<T>(L);
  DEC_ELL_WIDTH_SWITCH(L.width, hipLaunchKernelGGL((k_residual<W, T>), dim3(dec::xcd_grid(L.n)), dim3(kBlock), 0, s,
                                                   L.n, L.width, L.vcol.p, V.vval.p, static_cast<const int *>(nullptr),
                                                   b, u, r));
}

void dot(dec_mg_s &mg, int n, const double *x, const double *y, double *out, const int *done, hipStream_t s) {
  hipLaunchKernelGGL(k_dot_partial<double>, dim3(kDotBlocks), dim3(kBlock), 0, s, n, x, y, mg.part.p, done);
  hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(kBlock), 0, s, mg.part.p, out, done);
}

// cg(A, b, u; itmax = steps) as in Multigrid.jl:860 (float64 only) on a level of
// several workgroups: 2 + steps launches.  zc: the coarse correction, u + P zc
// the iterate it starts from (P's ELL of width 2); coarse: the next coarser
// level, whose b and zero iterate the last launch writes (R of the residual).
void cg_smooth(dec_mg_s &mg, Level &L, const double *b, double *u, int steps, const double *zc, Level *coarse,
               hipStream_t s) {
  int n = L.n, nb = cg_blocks(n);
  CgState *st = mg.cg.p;
  double *x = mg.cgx.p, *rb[2] = {L.d.t.p, mg.cgr.p}, *pb[2] = {mg.cgp.p, mg.cgp2.p}, *qb[2] = {mg.cgAp.p, mg.cgAp2.p};
  double *part[2] = {mg.part.p, mg.part2.p};
  double *u2 = zc ? L.d.r.p : u;
  DEC_ELL_WIDTH_SWITCH(L.width, {
    if (zc)
      hipLaunchKernelGGL((k_cg_start<W, true>), dim3(nb), dim3(kBlock), 0, s, st, n, L.width, L.vcol.p, L.d.vval.p, b,
                         u, L.pcol.p, L.d.pval.p, zc, u2, rb[0], part[1]);
    else
      hipLaunchKernelGGL((k_cg_start<W, false>), dim3(nb), dim3(kBlock), 0, s, st, n, L.width, L.vcol.p, L.d.vval.p,
                         b, u, static_cast<const int *>(nullptr), static_cast<const double *>(nullptr),
                         static_cast<const double *>(nullptr), static_cast<double *>(nullptr), rb[0], part[1]);
  });
  for (int it = 0; it < steps; it++) {
    int w = it & 1, o = w ^ 1;
    const double *r0 = it == 0 ? rb[0] : rb[o], *p0 = it <= 1 ? rb[0] : pb[o];
#define DEC_CG_STEP(A, B)                                                                                              \
  DEC_ELL_WIDTH_SWITCH(L.width, hipLaunchKernelGGL((k_cg_step<W, A, B>), dim3(nb), dim3(kBlock), 0, s, st, it, n,  \
                                                   L.width, L.vcol.p, L.d.vval.p, r0, p0, qb[o], rb[w], pb[w], qb[w], \
                                                   x, part[o], nb, part[w]))
    if (it == 0) {
      DEC_CG_STEP(true, false);
    } else if (it == 1) {
      DEC_CG_STEP(false, true);
    } else {
      DEC_CG_STEP(false, false);
    }
#undef DEC_CG_STEP
  }
  int w = (steps - 1) & 1;
  const double *p = steps == 1 ? rb[0] : pb[w];
  int nc = coarse ? L.nc : 0, rw = coarse ? L.rwidth : 0;
  DEC_ELL_WIDTH_SWITCH(rw, hipLaunchKernelGGL((k_cg_finish<W>), dim3(nb), dim3(kBlock), 0, s, st, steps, n, u2, x, p,
                                              rb[0], rb[1], qb[w], part[w], nb, u, nc, rw, L.rcol.p, L.d.rval.p,
                                              coarse ? coarse->d.b.p : nullptr, coarse ? coarse->d.u.p : nullptr));
}

// Levels that one workgroup smooths (k_cg_small, k_cg_tail).
inline bool cg_small(const Level &L) { return L.n <= kCgSmallRows && L.width >= 1 && L.width <= kCgWidth; }

inline CgLevel cg_level(Level &L) { return CgLevel{L.n, L.width, L.vcol.p, L.d.vval.p}; }

// LAUNCH with R = the least of 1, 2, 4, 6 and 7 rows per thread that hold n rows
#define DEC_CG_ROWS_SWITCH(n, LAUNCH)                                   \
  do {                                                                  \
    if ((n) <= kCgThreads) { constexpr int R = 1; LAUNCH; }             \
    else if ((n) <= 2 * kCgThreads) { constexpr int R = 2; LAUNCH; }    \
    else if ((n) <= 4 * kCgThreads) { constexpr int R = 4; LAUNCH; }    \
    else if ((n) <= 6 * kCgThreads) { constexpr int R = 6; LAUNCH; }    \
    else { constexpr int R = kCgRowsMax; LAUNCH; }                      \
  } while (0)

inline CgTransfer cg_transfer(Level &L) {
  return CgTransfer{L.nc, L.rwidth, L.pwidth, L.rcol.p, L.pcol.p, L.d.rval.p, L.d.pval.p};
}

// zc, coarse: as for cg_smooth (P's ELL of any width)
void cg_small_smooth(Level &L, const double *b, double *u, int steps, int reps, const double *zc, Level *coarse,
                     hipStream_t s) {
  size_t lds = static_cast<size_t>(L.n) * sizeof(double);
  DEC_CG_ROWS_SWITCH(L.n, hipLaunchKernelGGL((k_cg_small<R>), dim3(1), dim3(kCgThreads), lds, s, cg_level(L), b, u,
                                             steps, reps, cg_transfer(L), zc, coarse ? coarse->d.b.p : nullptr,
                                             coarse ? coarse->d.u.p : nullptr));
}

// Whether the cycles of level lvl run as k_cg_tail.
bool cg_tail_at(const dec_mg_s &mg, int lvl) {
  int nl = static_cast<int>(mg.lv.size());
  if (!mg.use_fused || mg.alg != DEC_SMOOTH_CG || mg.steps == 0 || mg.coarse_direct || lvl != nl - 2) return false;
  const Level &A = *mg.lv[lvl], &C = *mg.lv[nl - 1];
  return cg_small(A) && cg_small(C) && C.n <= kCgCoarseRows * kCgThreads;
}

// `cycles` μ-cycles of level lvl, the first `wcycles` of them with two visits of
// the coarsest level.
void cg_tail(dec_mg_s &mg, int lvl, double *u, const double *b, int cycles, int wcycles, hipStream_t s) {
  Level &A = *mg.lv[lvl], &C = *mg.lv[lvl + 1];
  size_t lds = static_cast<size_t>(A.n + C.n) * sizeof(double);
#define DEC_CG_TAIL(RC)                                                                                              \
  DEC_CG_ROWS_SWITCH(A.n, hipLaunchKernelGGL((k_cg_tail<R, RC>), dim3(1), dim3(kCgThreads), lds, s, cg_level(A),    \
                                             cg_level(C), b, u, mg.steps, cycles, wcycles, cg_transfer(A)))
  if (C.n <= kCgThreads) {
    DEC_CG_TAIL(1);
  } else {
    DEC_CG_TAIL(kCgCoarseRows);
  }
#undef DEC_CG_TAIL
}

inline bool learned_rows(const dec_mg_s &mg, int n) {
  return n >= mg.learned_min_rows && (mg.learned_max_rows <= 0 || n <= mg.learned_max_rows);
}

// Whether a cycle on this level that starts from zero does not read its iterate
// (the first pre-sweep takes it as zero), so that nobody need clear it.
template <class T>
bool zero_unread(const dec_mg_s &mg, const Level &L) {
  bool learned = sizeof(T) == 4 && mg.nn && mg.learned && mg.learned_active && learned_rows(mg, L.n);
  return mg.alg == DEC_SMOOTH_BLOCK_GS && mg.steps > 0 && L.panel_hs >= 0 && !learned && mg.lv.size() > 1;
}

inline bool learned_on(const dec_mg_s &mg) { return mg.nn && mg.learned && mg.learned_active; }

// Residual and restriction run as one launch on levels up to this many rows
// (measured: 6.8 against 9.0 µs at 40,962 rows, 18.5 against 10.6 µs at
// 163,842, where evaluating shared fine rows twice costs more than a launch).
constexpr int kFusedRestrictMaxRows = 50000;
// The CG smoother's first launch after the coarse correction adds it itself on
// levels up to this many rows.
constexpr int kCgFoldMaxRows = 100000;

// One panel sweep (k_panel_sweep) from src (zero: src is zero and not read) to dst.
template <class T>
void panel_sweep(Level &L, const T *b, const T *src, T *dst, bool post, bool zero, const T *zc, double *dot,
                 double *add, hipStream_t s) {
  LevelVals<T> &V = vals<T>(L);
  using V2 = typename Vec2T<T>::type;
  Panels<T> P{L.panel_b,
              L.panel_full,
              L.panel_hs,
              L.ncolors,
              L.bstart.p,
              reinterpret_cast<const uint4 *>(L.pidx.p),
              V.poff.p,
              V.pdiag.p,
              L.phalo.p,
              reinterpret_cast<const int2 *>(L.pown_p.p),
              reinterpret_cast<const int2 *>(L.phalo_p.p),
              reinterpret_cast<const V2 *>(V.pown_w.p),
              reinterpret_cast<const V2 *>(V.phalo_w.p)};
  int nt = panel_threads(P.B);
  size_t lds = static_cast<size_t>(2 * P.B + P.hs + 1) * sizeof(T);
  int rev = post ? 1 : 0;
#define DEC_PANEL(WW, RR, ZZ) \
  hipLaunchKernelGGL((k_panel_sweep<WW, T, RR, ZZ>), dim3(L.nblk), dim3(nt), lds, s, P, b, src, dst, rev, zc, dot, add)
#define DEC_PANEL_W(WW)                      \
  case WW:                                   \
    if (P.B <= kBlock) {                     \
      if (zero) DEC_PANEL(WW, 1, true);      \
      else DEC_PANEL(WW, 1, false);          \
    } else {                                 \
      if (zero) DEC_PANEL(WW, 2, true);      \
      else DEC_PANEL(WW, 2, false);          \
    }                                        \
    break;
  switch (L.width) {
    DEC_PANEL_W(2) DEC_PANEL_W(3) DEC_PANEL_W(4) DEC_PANEL_W(5) DEC_PANEL_W(6) DEC_PANEL_W(7) DEC_PANEL_W(8)
    default: fail(DEC_ERR_ARG, "multigrid: panel width");
  }
#undef DEC_PANEL_W
#undef DEC_PANEL
}

template <class T>
void smooth(dec_mg_s &mg, int lvl, Level &L, const T *b, T *u, bool post, bool u_zero, hipStream_t s,
            const T *zc = nullptr, Level *coarse = nullptr) {
  int steps = mg.steps;
  if (steps == 0) return;
  LevelVals<T> &V = vals<T>(L);
  if constexpr (sizeof(T) == 4) {
    if (learned_on(mg) && learned_rows(mg, L.n)) {
      for (int a = 0; a < mg.learned_apps; a++) {
        if (a == 0 && u_zero) {
          dec::nn_smooth(*mg.nn, lvl, b, u, s);
          continue;
        }
        residual<float>(L, b, u, V.r.p, s);
        dec::nn_smooth(*mg.nn, lvl, V.r.p, u, s);
      }
      return;
    }
  }
  if (mg.alg == DEC_SMOOTH_CG) {
    if constexpr (sizeof(T) == 8) {
      if (cg_small(L)) cg_small_smooth(L, b, u, steps, 1, zc, coarse, s);
      else cg_smooth(mg, L, b, u, steps, zc, coarse, s);
    } else {
      fail(DEC_ERR_UNSUPPORTED, "the CG smoother runs in float64 only");
    }
    return;
  }
  if (mg.alg == DEC_SMOOTH_BLOCK_GS) {
    // one launch per sweep, ping-ponging between u and the level's t
    // (an odd step count ends with a copy back into u); zc (post-smoothing
    // only) folds the prolongation u += P zc into the first sweep
    T *bufs[2] = {u, V.t.p};
    size_t lds = static_cast<size_t>(L.bmax) * sizeof(T);
    for (int it = 0; it < steps; it++) {
      const T *src = bufs[it & 1];
      T *dst = bufs[(it + 1) & 1];
      if (L.panel_hs >= 0)
        panel_sweep<T>(L, b, src, dst, post, u_zero && it == 0, it == 0 ? zc : nullptr,
                       post && lvl == 0 && it + 1 == steps ? mg.sweep_dot : nullptr,
                       post && lvl == 0 && it + 1 == steps ? mg.sweep_add : nullptr, s);
      else
        DEC_ELL_WIDTH_SWITCH(L.width, hipLaunchKernelGGL((k_block_gs<W, T>), dim3(L.nblk), dim3(L.seg_threads), lds,
                                                         s, L.n, L.width, L.ncolors, L.nblk, L.col.p, V.val.p,
                                                         L.rowid.p, L.bstart.p, L.seg.p, b, src, dst, post ? 1 : 0));
    }
    if (steps & 1 && !(post && lvl == 0 && mg.sweep_add))
      hipLaunchKernelGGL(k_copy<T>, G(L.n), dim3(kBlock), 0, s, L.n, V.t.p, u);
    return;
  }
  for (int it = 0; it < steps; it++) {
    if (mg.alg == DEC_SMOOTH_GS) {
      for (int ci = 0; ci < L.ncolors; ci++) {
        int c = post ? L.ncolors - 1 - ci : ci;
        int p0 = L.cstart[c], p1 = L.cstart[c + 1];
        if (p1 > p0)
          DEC_ELL_WIDTH_SWITCH(L.width, hipLaunchKernelGGL((k_gs_color<W, T>), dim3(dec::xcd_grid(p1 - p0)), dim3(kBlock),
                                                           0, s, p0, p1,
                                                           L.n, L.width, L.col.p, V.val.p, L.rowid.p, b, u));
      }
    } else {
      DEC_ELL_WIDTH_SWITCH(L.width, hipLaunchKernelGGL((k_jacobi<W, T>), G(L.n), dim3(kBlock), 0, s, L.n, L.width,
                                                     L.col.p, V.val.p, L.rowid.p, b, u, V.t.p,
                                                     static_cast<T>(mg.omega)));
      hipLaunchKernelGGL(k_copy<T>, G(L.n), dim3(kBlock), 0, s, L.n, V.t.p, u);
    }
  }
}

// u += Z r (r = the level's residual vector) by the chunked two-pass product.
template <class T>
void coarse_partials(Level &L, hipStream_t s) {
  LevelVals<T> &V = vals<T>(L);
  dim3 grid(static_cast<unsigned>((L.n + 63) / 64), static_cast<unsigned>(coarse_chunks(L.n)));
  hipLaunchKernelGGL(k_coarse_partial<T>, grid, dim3(64), 0, s, L.n, V.Z.p, V.r.p, V.zpart.p);
}

template <class T>
void coarse_gemv(Level &L, T *u, hipStream_t s) {
  coarse_partials<T>(L, s);
  hipLaunchKernelGGL(k_coarse_finish<T>, G(L.n), dim3(kBlock), 0, s, L.n, coarse_chunks(L.n), vals<T>(L).zpart.p, u);
}

template <class T>
void coarse_solve(dec_mg_s &mg, Level &L, const T *b, T *u, hipStream_t s) {
  LevelVals<T> &V = vals<T>(L);
  if (!V.Z.p) fail(DEC_ERR_UNSUPPORTED, "coarsest level too large for the dense direct solve");
  residual<T>(L, b, u, V.r.p, s);
  coarse_gemv<T>(L, u, s);
  (void)mg;
}

// The coarse tail's launch at level l, on the way down (C's solution, or above
// the level before the last C's right-hand side, from b and u; the smoothed u goes to
// the level's r) or up.
template <class T>
void tail_launch(dec_mg_s &mg, int l, const T *b, T *u, bool u_zero, bool up, hipStream_t s) {
  Level &L = *mg.lv[l], &C = *mg.lv[l + 1];
  LevelVals<T> &V = vals<T>(L), &CV = vals<T>(C);
  const bool last = l + 2 == static_cast<int>(mg.lv.size());
  Tail<T> A{L.n,      L.nc,      L.ncolors, L.rwidth, L.pwidth, reinterpret_cast<const uint4 *>(L.tidx.p),
            V.toff.p, V.tdiag.p, L.rcol.p,  L.pcol.p, V.rval.p, V.pval.p,
            last ? CV.Z.p : nullptr};
  const size_t lds = tail_lds(L.n, L.nc, sizeof(T));
  const dim3 grid(up || !last ? 1 : (L.nc + kTailZ - 1) / kTailZ), blk(kFuseThreads);
  auto run = [&](auto S, auto R) {
    if (up)
      hipLaunchKernelGGL((k_tail_up<S.value, T, R.value>), grid, blk, lds, s, A, V.r.p, last ? CV.zpart.p : CV.u.p, b,
                         u, mg.steps);
    else
      hipLaunchKernelGGL((k_tail_down<S.value, T, R.value>), grid, blk, lds, s, A,
                         u_zero ? static_cast<const T *>(nullptr) : u, b, V.r.p, last ? CV.zpart.p : CV.b.p, mg.steps);
  };
  auto rows = [&](auto S) {
    switch ((L.n + kFuseThreads - 1) / kFuseThreads) {
      case 1: run(S, std::integral_constant<int, 1>{}); break;
      case 2: run(S, std::integral_constant<int, 2>{}); break;
      default: run(S, std::integral_constant<int, 3>{}); break;
    }
  };
  switch (std::max(L.width - 1, 1)) {
    case 1: rows(std::integral_constant<int, 1>{}); break;
    case 2: rows(std::integral_constant<int, 2>{}); break;
    case 3: rows(std::integral_constant<int, 3>{}); break;
    case 4: rows(std::integral_constant<int, 4>{}); break;
    case 5: rows(std::integral_constant<int, 5>{}); break;
    case 6: rows(std::integral_constant<int, 6>{}); break;
    default: rows(std::integral_constant<int, 7>{}); break;
  }
}

// _multigrid_μ_cycle (Multigrid.jl:857-872).
template <class T>
void mu_cycle(dec_mg_s &mg, int lvl, T *u, const T *b, int mu, bool u_zero, hipStream_t s) {
  int nl = static_cast<int>(mg.lv.size());
  Level &L = *mg.lv[lvl];
  // the fused tail has no learned smoother: a level that uses it runs unfused
  bool learned_here = sizeof(T) == 4 && learned_on(mg) && learned_rows(mg, L.n);
  if (mg.use_fused && mu == 1 && mg.alg != DEC_SMOOTH_CG && mg.fuse_from >= 0 && lvl >= mg.fuse_from &&
      !learned_here && (mg.coarse_direct == 0 || vals<T>(*mg.lv.back()).Z.p)) {
    const LevelDesc<T> *D;
    if constexpr (sizeof(T) == 8) D = mg.desc64.p;
    else D = mg.desc32.p;
    T om = static_cast<T>(mg.omega);
    if (!mg.coarse_direct) {
      hipLaunchKernelGGL(k_fused_vcycle<T>, dim3(1), dim3(kFuseThreads), 0, s, D, lvl, nl, u, b, mg.steps, mg.alg, om,
                         0, static_cast<const T *>(nullptr));
      return;
    }
    Level &C = *mg.lv.back();
    // Gauss-Seidel levels above the dense coarsest level: the register/LDS tail
    bool tail = lvl < nl - 1 && mg.alg != DEC_SMOOTH_JACOBI;
    for (int l = lvl; l < nl - 1; l++) tail = tail && mg.lv[l]->tidx.p;
    if (tail) {
      for (int l = lvl; l < nl - 1; l++)
        tail_launch<T>(mg, l, l > lvl ? vals<T>(*mg.lv[l]).b.p : b, l > lvl ? vals<T>(*mg.lv[l]).u.p : u,
                       l > lvl || u_zero, false, s);
      for (int l = nl - 2; l >= lvl; l--)
        tail_launch<T>(mg, l, l > lvl ? vals<T>(*mg.lv[l]).b.p : b, l > lvl ? vals<T>(*mg.lv[l]).u.p : u, false, true,
                       s);
      return;
    }
    hipLaunchKernelGGL(k_fused_vcycle<T>, dim3(1), dim3(kFuseThreads), 0, s, D, lvl, nl, u, b, mg.steps, mg.alg, om,
                       1, static_cast<const T *>(nullptr));
    coarse_partials<T>(C, s);
    hipLaunchKernelGGL(k_fused_vcycle<T>, dim3(1), dim3(kFuseThreads), 0, s, D, lvl, nl, u, b, mg.steps, mg.alg, om,
                       2, static_cast<const T *>(vals<T>(C).zpart.p));
    return;
  }
  if (lvl == nl - 1 && mg.coarse_direct) {
    coarse_solve<T>(mg, L, b, u, s);
    return;
  }
  // the CG smoother restricts its residual itself
  bool cg_on = sizeof(T) == 8 && mg.alg == DEC_SMOOTH_CG && mg.steps > 0;
  if constexpr (sizeof(T) == 8)
    if (cg_tail_at(mg, lvl)) {
      cg_tail(mg, lvl, u, b, 1, mu > 1 ? 1 : 0, s);
      return;
    }
  smooth<T>(mg, lvl, L, b, u, false, u_zero, s, nullptr, cg_on && lvl < nl - 1 ? mg.lv[lvl + 1].get() : nullptr);
  if (lvl >= nl - 1) return;
  Level &C = *mg.lv[lvl + 1];
  LevelVals<T> &V = vals<T>(L);
  LevelVals<T> &CV = vals<T>(C);
  if (cg_on) {
    // b and u of the coarser level are in place
  } else if (L.n <= kFusedRestrictMaxRows && L.rwidth <= 8) {
    DEC_ELL_WIDTH_SWITCH(L.width, hipLaunchKernelGGL((k_residual_restrict<W, T>), G(8LL * L.nc), dim3(kBlock), 0, s,
                                                     L.nc, L.rwidth, L.rcol.p, V.rval.p, L.n, L.width, L.vcol.p,
                                                     V.vval.p, b, u, CV.b.p, CV.u.p));
  } else {
    residual<T>(L, b, u, V.r.p, s);
    DEC_ELL_WIDTH_SWITCH(L.rwidth, hipLaunchKernelGGL((k_restrict<W, T>), G(L.nc), dim3(kBlock), 0, s, L.nc,
                                                      L.rwidth, L.rcol.p, V.rval.p, V.r.p, CV.b.p, CV.u.p));
  }
  bool tail = false;
  if constexpr (sizeof(T) == 8) {
    tail = cg_tail_at(mg, lvl + 1);
    // (both visits of the two coarsest levels in one launch)
    if (tail) cg_tail(mg, lvl + 1, CV.u.p, CV.b.p, mu > 1 ? 2 : 1, mu > 2 ? 2 : (mu > 1 ? 1 : 0), s);
  }
  if (!tail) {
    mu_cycle<T>(mg, lvl + 1, CV.u.p, CV.b.p, mu, true, s);
    if (mu > 1) mu_cycle<T>(mg, lvl + 1, CV.u.p, CV.b.p, mu - 1, false, s);
  }
  // the hybrid smoother's first post-sweep, or the CG smoother's first launch,
  // applies the prolongation itself
  bool fold = mg.alg == DEC_SMOOTH_BLOCK_GS && mg.steps > 0 && L.pwidth == 2 && L.panel_hs >= 0 &&
              !(sizeof(T) == 4 && learned_on(mg) && learned_rows(mg, L.n));
  fold = fold || (cg_on && (cg_small(L) || (L.pwidth == 2 && L.width >= 1 && L.width <= 8 && L.n <= kCgFoldMaxRows)));
  if (!fold)
    DEC_ELL_WIDTH_SWITCH(L.pwidth, hipLaunchKernelGGL((k_prolong_add<W, T>), G(L.n), dim3(kBlock), 0, s, L.n,
                                                      L.pwidth, L.pcol.p, V.pval.p, CV.u.p, u));
  smooth<T>(mg, lvl, L, b, u, true, false, s, fold ? static_cast<const T *>(CV.u.p) : nullptr);
}

// _full_multigrid (Multigrid.jl:839-855).
void fmg_rec(dec_mg_s &mg, int lvl, const double *b, double *z, int mu, int cycles, hipStream_t s) {
  int nl = static_cast<int>(mg.lv.size());
  Level &L = *mg.lv[lvl];
  hipLaunchKernelGGL(k_zero<double>, G(L.n), dim3(kBlock), 0, s, L.n, z);
  if (lvl < nl - 1) {
    Level &C = *mg.lv[lvl + 1];
    DEC_ELL_WIDTH_SWITCH(L.rwidth, hipLaunchKernelGGL((k_restrict<W, double>), G(L.nc), dim3(kBlock), 0, s, L.nc,
                                                      L.rwidth, L.rcol.p, L.d.rval.p, b, C.d.b.p,
                                                      static_cast<double *>(nullptr)));
    fmg_rec(mg, lvl + 1, C.d.b.p, C.d.u.p, mu, cycles, s);
    DEC_ELL_WIDTH_SWITCH(L.pwidth, hipLaunchKernelGGL((k_prolong_add<W, double>), G(L.n), dim3(kBlock), 0, s, L.n,
                                                      L.pwidth, L.pcol.p, L.d.pval.p, C.d.u.p, z));
  }
  if (lvl == 0) return;
  if (cg_tail_at(mg, lvl)) {
    if (cycles > 0) cg_tail(mg, lvl, z, b, cycles, mu > 1 ? cycles : 0, s);
  } else if (lvl == nl - 1 && mg.alg == DEC_SMOOTH_CG && mg.steps > 0 && !mg.coarse_direct && cg_small(L)) {
    if (cycles > 0) cg_small_smooth(L, b, z, mg.steps, cycles, nullptr, nullptr, s);
  } else {
    for (int c = 0; c < cycles; c++) mu_cycle<double>(mg, lvl, z, b, mu, false, s);
  }
}

// The caller's finest-level vectors in the hierarchy's numbering: b into
// the finest level's b, u (when load_u) into its u; the caller's own pointers
// when the finest level keeps the caller's order.
struct FineIO {
  double *u;
  const double *b;
};

FineIO fine_in(dec_mg_s &mg, double *u, const double *b, bool load_u, hipStream_t s) {
  Level &F = *mg.lv[0];
  if (F.identity) return FineIO{u, b};
  hipLaunchKernelGGL(k_perm_gather<double>, G(F.n), dim3(kBlock), 0, s, F.n, F.dperm.p, b, F.d.b.p);
  if (load_u) hipLaunchKernelGGL(k_perm_gather<double>, G(F.n), dim3(kBlock), 0, s, F.n, F.dperm.p, u, F.d.u.p);
  return FineIO{F.d.u.p, F.d.b.p};
}

void fine_out(dec_mg_s &mg, double *u, hipStream_t s) {
  Level &F = *mg.lv[0];
  if (F.identity) return;
  hipLaunchKernelGGL(k_perm_scatter<double>, G(F.n), dim3(kBlock), 0, s, F.n, F.dperm.p, F.d.u.p, u);
}

double norm2(dec_mg_s &mg, int n, const double *x, hipStream_t s) {
  dot(mg, n, x, x, mg.scal.p, nullptr, s);
  double v = 0.0;
  if (hipMemcpyAsync(&v, mg.scal.p, sizeof(double), hipMemcpyDeviceToHost, s) != hipSuccess ||
      hipStreamSynchronize(s) != hipSuccess)
    fail(DEC_ERR_HIP, "norm: copy failed");
  return std::sqrt(v);
}

// What the finest level's last sweep also does, for one cycle (also where that
// cycle ends with an exception).
struct Hook {
  double *&slot;
  Hook(double *&s, double *p) : slot(s) { slot = p; }
  ~Hook() { slot = nullptr; }
  Hook(const Hook &) = delete;
  Hook &operator=(const Hook &) = delete;
};

// r = b - A u on the finest level with the per-workgroup sums of r² (rpart),
// before a cycle of the variant: the mixed variant's cycle takes the residual
// rounded to float32 in F.f.b and forms none itself, so it is written here.
// r: where the float64 residual is wanted too, or null.
void finest_residual(dec_mg_s &mg, int variant, const double *b, const double *u, double *r, hipStream_t s) {
  Level &F = *mg.lv[0];
  int nb = dec::nblocks(F.n, kBlock);
  if (mg.rpart.n < static_cast<size_t>(nb)) fail(DEC_ERR_ARG, "multigrid: residual partials");
  float *rounded = variant == DEC_SOLVE_MIXED_IR ? F.f.b.p : nullptr;
  DEC_ELL_WIDTH_SWITCH(F.width, hipLaunchKernelGGL((k_residual_norm<W>), dim3(nb), dim3(kBlock), 0, s, F.n, F.width,
                                                   F.vcol.p, F.d.vval.p, static_cast<const int *>(nullptr), b, u, r,
                                                   rounded, mg.rpart.p));
}

// One cycle; for the mixed variant finest_residual has formed the residual of u.
void cycle_body(dec_mg_s &mg, int variant, double *u, const double *b, hipStream_t s) {
  Level &F = *mg.lv[0];
  int n = F.n;
  if (variant == DEC_SOLVE_PLAIN_F64) {
    mu_cycle<double>(mg, 0, u, b, 1, false, s);
  } else {
    // float32 V-cycle on the rounded residual (F.f.b), correction added in
    // float64: by the cycle's last sweep where it is a panel sweep, which saves a launch (2.3 µs at 100,000 rows)
    bool swept = zero_unread<float>(mg, F);
    if (!swept) hipLaunchKernelGGL(k_zero<float>, G(n), dim3(kBlock), 0, s, n, F.f.u.p);
    {
      Hook hook(mg.sweep_add, swept ? u : nullptr);
      mu_cycle<float>(mg, 0, F.f.u.p, F.f.b.p, 1, true, s);
    }
    if (!swept) hipLaunchKernelGGL(k_add_f2d, G(n), dim3(kBlock), 0, s, n, F.f.u.p, u);
  }
}

void gcheck(hipError_t e, const char *what) {
  if (e != hipSuccess) fail(DEC_ERR_HIP, std::string(what) + ": " + hipGetErrorString(e));
}

// ||b||^2 on its way to the host (pinned slot kNormSlots with its event), and
// its square root once it has arrived
void send_bnorm(dec_mg_s &mg, int n, const double *b, hipStream_t s) {
  dot(mg, n, b, b, mg.scal.p + kNormSlots, nullptr, s);
  gcheck(hipMemcpyAsync(mg.hnorm + kNormSlots, mg.scal.p + kNormSlots, sizeof(double), hipMemcpyDeviceToHost, s),
         "hipMemcpyAsync");
  gcheck(hipEventRecord(mg.nev[kNormSlots], s), "hipEventRecord");
}
double read_bnorm(dec_mg_s &mg) {
  gcheck(hipEventSynchronize(mg.nev[kNormSlots]), "hipEventSynchronize");
  return std::sqrt(mg.hnorm[kNormSlots]);
}

// body(stream) replayed from the hipGraph in slot i, captured for (u, b) and
// the current smoother settings (key); captured again when any of them changes.
template <class Body>
void replay(dec_mg_s &mg, int i, const void *u, const void *b, Body body, hipStream_t s) {
  int key = mg.alg * 1000003 + mg.steps * 1009 + mg.coarse_direct * 7 + static_cast<int>(mg.omega * 1e6) +
            (mg.learned && mg.learned_active ? 1 << 29 : 0) + mg.learned_apps * 31 + mg.learned_min_rows +
            mg.learned_max_rows * 7919;
  if (!mg.gexec[i] || mg.gu[i] != u || mg.gb[i] != b || mg.gkey[i] != key) {
    if (mg.gexec[i]) (void)hipGraphExecDestroy(mg.gexec[i]);
    if (mg.graph[i]) (void)hipGraphDestroy(mg.graph[i]);
    mg.gexec[i] = nullptr;
    mg.graph[i] = nullptr;
    if (!mg.cap) gcheck(hipStreamCreateWithFlags(&mg.cap, hipStreamNonBlocking), "hipStreamCreate");
    gcheck(hipStreamBeginCapture(mg.cap, hipStreamCaptureModeThreadLocal), "hipStreamBeginCapture");
    try {
      body(mg.cap);
    } catch (...) {
      // close the capture, or every later allocation on this thread fails
      hipGraph_t partial = nullptr;
      (void)hipStreamEndCapture(mg.cap, &partial);
      if (partial) (void)hipGraphDestroy(partial);
      throw;
    }
    gcheck(hipStreamEndCapture(mg.cap, &mg.graph[i]), "hipStreamEndCapture");
    gcheck(hipGraphInstantiate(&mg.gexec[i], mg.graph[i], nullptr, nullptr, 0), "hipGraphInstantiate");
    mg.gu[i] = u;
    mg.gb[i] = b;
    mg.gkey[i] = key;
  }
  gcheck(hipGraphLaunch(mg.gexec[i], s), "hipGraphLaunch");
}

// One cycle of the solve, replayed from a hipGraph captured for (u, b) and
// the current smoother settings.
void run_cycle(dec_mg_s &mg, int variant, double *u, const double *b, hipStream_t s) {
  if (!mg.use_graph) {
    cycle_body(mg, variant, u, b, s);
    return;
  }
  replay(mg, variant == DEC_SOLVE_PLAIN_F64 ? 0 : 1, u, b,
         [&](hipStream_t cs) { cycle_body(mg, variant, u, b, cs); }, s);
}

void solve(dec_mg_s &mg, int variant, double tol, int max_cycles, double *u_caller, const double *b_caller,
           int *done_cycles, double *relres, hipStream_t s) {
  Level &F = *mg.lv[0];
  int n = F.n;
  // With the iterate in the hierarchy's own numbering, the caller's u stays
  // untouched until the end, so the first cycles are queued before the host
  // has read ||b|| and the starting residual (one wait instead of two, with
  // the GPU busy during it); a b of zero or a start that already meets the
  // tolerance then returns without them.
  const bool ahead = !F.identity;
  double bn = 0.0;
  if (ahead) {
    send_bnorm(mg, n, b_caller, s);
  } else {
    bn = norm2(mg, n, b_caller, s);
    if (bn == 0.0) {
      hipLaunchKernelGGL(k_zero<double>, G(n), dim3(kBlock), 0, s, n, u_caller);
      *done_cycles = 0;
      *relres = 0.0;
      return;
    }
  }
  FineIO io = fine_in(mg, u_caller, b_caller, true, s);
  double *u = io.u;
  const double *b = io.b;
  // the network smooths the float32 cycles on the levels of at least
  // learned_min_rows .. learned_max_rows rows; with no such level the solve
  // is a plain mixed one
  bool any = false;
  for (auto &Lv : mg.lv) any = any || learned_rows(mg, Lv->n);
  mg.learned_active = mg.learned && mg.nn && variant == DEC_SOLVE_MIXED_IR && any;
  mg.fallbacks = 0;
  mg.learned_cycles = 0;
  // A residual norm is copied to pinned host memory with an event per slot,
  // and the host reads it when it must decide whether to stop.
  bool plain = variant == DEC_SOLVE_PLAIN_F64;
  // after cycle k: the float64 residual (which the mixed variant's next cycle
  // refines) and, when `check`, its norm on its way to the host
  auto post = [&](int k, bool check) {
    if (plain && !check) return;
    finest_residual(mg, variant, b, u, nullptr, s);
    if (!check) return;
    double *slot = mg.scal.p + (k % kNormSlots);
    hipLaunchKernelGGL(k_sum_rows, dim3(1), dim3(kBlock), 0, s, dec::nblocks(n, kBlock), mg.rpart.p, slot);
    gcheck(hipMemcpyAsync(mg.hnorm + (k % kNormSlots), slot, sizeof(double), hipMemcpyDeviceToHost, s),
           "hipMemcpyAsync");
    gcheck(hipEventRecord(mg.nev[k % kNormSlots], s), "hipEventRecord");
  };
  auto read_norm = [&](int k) {
    gcheck(hipEventSynchronize(mg.nev[k % kNormSlots]), "hipEventSynchronize");
    return std::sqrt(mg.hnorm[k % kNormSlots]) / bn;
  };
  int enq = 0;               // cycles queued
  bool enq_checked = true;   // whether the norm after cycle `enq` was queued
  auto enqueue_cycle = [&](bool check) {
    enq++;
    if (mg.learned_active) mg.learned_cycles++;
    run_cycle(mg, variant, u, b, s);
    post(enq, check);
    enq_checked = check;
  };
  // The norm is read only where the decision needs it: after cycle 1 (the
  // convergence rate), then at the first cycle that could meet the
  // tolerance, then after every cycle (every cycle while the learned
  // smoother is on: its fallback test needs each drop).  Cycles before a
  // check run without waiting for the host; while the last known residual
  // stays above 1000 tol after the queued cycles, the cycle after the check
  // is queued too (no V-cycle cuts the residual 1000x).
  post(0, true);
  if (ahead) {
    // what the loop below queues first for a start far from the solution
    if (max_cycles >= 1) enqueue_cycle(true);
    if (max_cycles >= 2) enqueue_cycle(false);
    bn = read_bnorm(mg);
    if (bn == 0.0) {
      hipLaunchKernelGGL(k_zero<double>, G(n), dim3(kBlock), 0, s, n, u_caller);
      mg.learned_cycles = 0;
      *done_cycles = 0;
      *relres = 0.0;
      return;
    }
  }
  double rr = read_norm(0), prev = rr, rho = -1.0;
  int c = 0;
  if (ahead && rr <= tol) {
    mg.learned_cycles = 0;
    *done_cycles = 0;
    *relres = rr;
    return;
  }
  while (rr > tol && c < max_cycles) {
    int kc = c + 1;
    // (the prediction takes each cycle to cut twice as much as the last ones
    // did, so the check comes no later than the first cycle that can meet
    // the tolerance)
    if (rho > 0.0 && !mg.learned_active)
      while (kc < max_cycles && rr * std::pow(0.5 * rho, kc - c) > tol) kc++;
    while (enq < kc) enqueue_cycle(enq + 1 == kc);
    if (enq == kc && !enq_checked) {
      // the check cycle was queued ahead without its norm; nothing after it
      // is queued, so the iterate is still the one after cycle kc
      post(kc, true);
      enq_checked = true;
    }
    if (enq < kc + 1 && kc + 1 <= max_cycles && rr * std::pow(1e-3, kc + 1 - c) > tol) enqueue_cycle(false);
    double rk = read_norm(kc);
    rho = std::min(0.95, std::max(1e-4, std::pow(rk / rr, 1.0 / (kc - c))));
    // a learned cycle that cut the residual by less than 0.5x hands the rest
    // of the solve to Gauss-Seidel (from the next cycle not yet queued)
    if (mg.learned_active && rk > 0.5 * prev) {
      mg.learned_active = false;
      mg.fallbacks++;
    }
    prev = rr = rk;
    c = kc;
  }
  if (enq > c) {  // a queued cycle ran past the stop (a drop above 1000x): report it
    if (!enq_checked) post(enq, true);
    c = enq;
    rr = read_norm(c);
  }
  fine_out(mg, u_caller, s);
  *done_cycles = c;
  *relres = rr;
  if (rr > tol) fail(DEC_ERR_NOCONV, "dec_mg_solve: relative residual " + std::to_string(rr) + " above tolerance after " +
                                         std::to_string(c) + " cycles");
}

// partial sums of r·z that an iteration may leave
inline int pcg_dots(const Level &F) { return std::max(kPcgDotBlocks, F.nblk); }

// One iteration of the preconditioned CG: z = one V-cycle on r from a zero
// start (float32 cycles on the rounded residual for the mixed variant, z
// their float64 value), then the three CG launches.  The V-cycle's input (a
// zero z, or the float32 r and iterate) was prepared by the previous
// iteration's update launch or by the start.
void pcg_iteration(dec_mg_s &mg, bool mixed, double *x, hipStream_t s) {
  Level &F = *mg.lv[0];
  int n = F.n, nb = dec::nblocks(n, kBlock), ng = dec::xcd_grid(n);
  // partial sums: r·z in [0, pcg_dots), then p·q (one per workgroup of
  // the direction launch, ng) and r·r (one per workgroup of the update, nb)
  double *r = mg.pcg_r.p, *z = mg.pcg_z.p, *part = mg.pcg_part.p;
  double *part_pq = part + pcg_dots(F), *part_rr = part_pq + ng;
  // the float64 cycle's last post-sweep leaves the partial sums of r·z itself
  // (its b is r, its iterate z): one launch less (5.2 µs at 655,362 rows)
  bool swept = !mixed && zero_unread<double>(mg, F);
  int np = swept ? F.nblk : kPcgDotBlocks;
  if (!mixed) {
    Hook hook(mg.sweep_dot, swept ? part : nullptr);
    mu_cycle<double>(mg, 0, z, r, 1, true, s);
  } else {
    mu_cycle<float>(mg, 0, F.f.u.p, F.f.b.p, 1, true, s);
  }
  if (!swept)
    hipLaunchKernelGGL(k_pcg_dot, dim3(kPcgDotBlocks), dim3(kBlock), 0, s, n, r, mixed ? F.f.u.p : nullptr, z, part);
  DEC_ELL_WIDTH_SWITCH(F.width, hipLaunchKernelGGL((k_pcg_dir<W>), dim3(ng), dim3(kBlock), 0, s, n,
                                                   F.width, F.vcol.p, F.d.vval.p, static_cast<const int *>(nullptr),
                                                   z, mg.pcg_p.p,
                                                   mg.pcg_q.p, part, np, mg.pcg_sc.p, part_pq));
  hipLaunchKernelGGL(k_pcg_alpha, dim3(1), dim3(kBlock), 0, s, part_pq, ng, mg.pcg_sc.p);
  hipLaunchKernelGGL(k_pcg_update, dim3(nb), dim3(kBlock), 0, s, n, x, r, mg.pcg_p.p, mg.pcg_q.p, mg.pcg_sc.p,
                     part_rr, mixed || swept ? nullptr : z, mixed ? F.f.b.p : nullptr,
                     mixed && !zero_unread<float>(mg, F) ? F.f.u.p : nullptr);
}

// Solve with the preconditioned CG (variants DEC_SOLVE_PCG_F64 / _MIXED).
// The stop test reads the recursively updated residual's norm where the
// decision needs it, as solve() does; once it meets the tolerance the true
// residual b - A x is formed and must meet it too (otherwise CG restarts
// from the true residual).  An iteration rate of 0.9 or worse hands the rest
// of the solve to plain V-cycles from the current iterate.  The learned
// smoother is not used in these variants.
void pcg_solve(dec_mg_s &mg, bool mixed, double tol, int max_iters, double *u_caller, const double *b_caller,
               int *done_iters, double *relres, hipStream_t s) {
  Level &F = *mg.lv[0];
  int n = F.n;
  // the first iterations are queued before the host reads ||b|| and the
  // starting residual, as in solve()
  const bool ahead = !F.identity;
  double bn = 0.0;
  if (ahead) {
    send_bnorm(mg, n, b_caller, s);
  } else {
    bn = norm2(mg, n, b_caller, s);
    if (bn == 0.0) {
      hipLaunchKernelGGL(k_zero<double>, G(n), dim3(kBlock), 0, s, n, u_caller);
      *done_iters = 0;
      *relres = 0.0;
      return;
    }
  }
  int nb = dec::nblocks(n, kBlock);
  if (mg.pcg_r.n < static_cast<size_t>(n)) {
    for (auto *v : {&mg.pcg_r, &mg.pcg_z, &mg.pcg_p, &mg.pcg_q}) v->alloc(n);
    mg.pcg_part.alloc(pcg_dots(F) + static_cast<size_t>(dec::xcd_grid(n)) + nb);
    mg.pcg_sc.alloc(3);
  }
  FineIO io = fine_in(mg, u_caller, b_caller, true, s);
  double *x = io.u;
  const double *b = io.b;
  mg.learned_active = false;
  // a norm on its way to the host: the partial sums part[0..np) added into
  // ring slot k with an event
  auto send = [&](int k, const double *part, int np) {
    double *slot = mg.scal.p + (k % kNormSlots);
    hipLaunchKernelGGL(k_sum_rows, dim3(1), dim3(kBlock), 0, s, np, part, slot);
    gcheck(hipMemcpyAsync(mg.hnorm + (k % kNormSlots), slot, sizeof(double), hipMemcpyDeviceToHost, s),
           "hipMemcpyAsync");
    gcheck(hipEventRecord(mg.nev[k % kNormSlots], s), "hipEventRecord");
  };
  auto read_norm = [&](int k) {
    gcheck(hipEventSynchronize(mg.nev[k % kNormSlots]), "hipEventSynchronize");
    return std::sqrt(mg.hnorm[k % kNormSlots]) / bn;
  };
  // the true residual b - A x into F.d.r and where the fallback's cycle reads it, its norm to slot k
  const int fallback = mixed ? DEC_SOLVE_MIXED_IR : DEC_SOLVE_PLAIN_F64;
  auto true_residual = [&](int k) {
    finest_residual(mg, fallback, b, x, F.d.r.p, s);
    send(k, mg.rpart.p, nb);
  };
  // CG from the true residual in F.d.r
  auto restart = [&]() {
    hipLaunchKernelGGL(k_pcg_start, G(n), dim3(kBlock), 0, s, n, F.d.r.p, mg.pcg_r.p, mg.pcg_p.p, mg.pcg_q.p,
                       mg.pcg_sc.p, mixed ? nullptr : mg.pcg_z.p, mixed ? F.f.b.p : nullptr,
                       mixed ? F.f.u.p : nullptr);
  };
  int enq = 0;
  bool enq_checked = true;
  auto enqueue = [&](bool check) {
    enq++;
    if (mg.use_graph)
      replay(mg, mixed ? 3 : 2, x, b, [&](hipStream_t cs) { pcg_iteration(mg, mixed, x, cs); }, s);
    else
      pcg_iteration(mg, mixed, x, s);
    if (check) send(enq, mg.pcg_part.p + pcg_dots(F) + dec::xcd_grid(n), nb);
    enq_checked = check;
  };
  true_residual(0);
  restart();
  if (ahead) {
    if (max_iters >= 1) enqueue(true);
    if (max_iters >= 2) enqueue(false);
    bn = read_bnorm(mg);
    if (bn == 0.0) {
      hipLaunchKernelGGL(k_zero<double>, G(n), dim3(kBlock), 0, s, n, u_caller);
      *done_iters = 0;
      *relres = 0.0;
      return;
    }
  }
  double rr = read_norm(0), rho = -1.0;
  int c = 0;
  bool stalled = false, verified = rr <= tol;
  if (ahead && verified) {
    *done_iters = 0;
    *relres = rr;
    return;
  }
  while (c < max_iters && !verified) {
    if (rr <= tol) {
      // the recursive residual meets the tolerance: confirm it on the
      // iterate after every queued iteration
      c = enq;
      true_residual(c);
      rr = read_norm(c);
      verified = rr <= tol;
      if (!verified) {
        restart();
        rho = -1.0;
      }
      continue;
    }
    // the check comes no later than the first iteration that can meet the
    // tolerance (each predicted to cut twice as much as the last ones did)
    int kc = c + 1;
    if (rho > 0.0)
      while (kc < max_iters && rr * std::pow(0.5 * rho, kc - c) > tol) kc++;
    while (enq < kc) enqueue(enq + 1 == kc);
    if (enq == kc && !enq_checked) {
      // queued ahead without its norm; nothing after it is queued, so its
      // partial sums are still in place
      send(kc, mg.pcg_part.p + pcg_dots(F) + dec::xcd_grid(n), nb);
      enq_checked = true;
    }
    if (enq < kc + 1 && kc + 1 <= max_iters && rr * std::pow(1e-3, kc + 1 - c) > tol) enqueue(false);
    double rk = read_norm(kc);
    double rate = std::pow(rk / rr, 1.0 / (kc - c));
    rr = rk;
    c = kc;
    if (!(rate < 0.9)) {
      stalled = true;
      break;
    }
    rho = std::min(0.95, std::max(1e-4, rate));
  }
  if (!verified) {
    // the true residual after every queued iteration; when CG stalled,
    // plain V-cycles from there
    c = enq;
    true_residual(c);
    rr = read_norm(c);
    while (stalled && rr > tol && c < max_iters) {
      run_cycle(mg, fallback, x, b, s);
      c++;
      true_residual(c);
      rr = read_norm(c);
    }
  }
  fine_out(mg, u_caller, s);
  *done_iters = c;
  *relres = rr;
  if (rr > tol) fail(DEC_ERR_NOCONV, "dec_mg_solve: relative residual " + std::to_string(rr) + " above tolerance after " +
                                         std::to_string(c) + " iterations");
}

}  // namespace

extern "C" {

int dec_mg_create(dec_mesh base, int32_t levels, int32_t project, int32_t hodge, int32_t center, int32_t steps,
                  dec_mg *out) {
  DEC_TRY
  if (!base || !out) fail(DEC_ERR_ARG, "dec_mg_create: NULL handle");
  *out = nullptr;
  *out = mg_create(*base, levels, project != 0, hodge, center, steps, false);
  DEC_CATCH
}

int dec_mg_create_mode(dec_mesh base, int32_t levels, int32_t project, int32_t hodge, int32_t center,
                       int32_t steps, int32_t mode, dec_mg *out) {
  DEC_TRY
  if (!base || !out) fail(DEC_ERR_ARG, "dec_mg_create_mode: NULL handle");
  if (mode != DEC_MG_DIRECT && mode != DEC_MG_GALERKIN) fail(DEC_ERR_ARG, "dec_mg_create_mode: unknown mode");
  *out = nullptr;
  *out = mg_create(*base, levels, project != 0, hodge, center, steps, mode == DEC_MG_GALERKIN);
  DEC_CATCH
}

int dec_mg_create_from_csr(int32_t nlevels, const int32_t *sizes, const int32_t *const *a_rowptr,
                           const int32_t *const *a_col, const double *const *a_val,
                           const int32_t *const *r_rowptr, const int32_t *const *r_col,
                           const double *const *r_val, const int32_t *const *p_rowptr,
                           const int32_t *const *p_col, const double *const *p_val, int32_t index_base,
                           int32_t steps, dec_mg *out) {
  DEC_TRY
  if (!out) fail(DEC_ERR_ARG, "dec_mg_create_from_csr: out is NULL");
  *out = nullptr;
  dec_mg_s *mg = mg_from_csr(nlevels, sizes, a_rowptr, a_col, a_val, r_rowptr, r_col, r_val, p_rowptr, p_col,
                             p_val, index_base, steps);
  dec::check_launch("dec_mg_create_from_csr");
  dec::dsync();
  *out = mg;
  DEC_CATCH
}

int dec_mg_nlevels(dec_mg mg, int32_t *nlevels) {
  DEC_TRY
  if (!mg || !nlevels) fail(DEC_ERR_ARG, "dec_mg_nlevels: NULL argument");
  *nlevels = static_cast<int32_t>(mg->lv.size());
  DEC_CATCH
}

int dec_mg_level_size(dec_mg mg, int32_t level, int32_t *n) {
  DEC_TRY
  if (!mg || !n) fail(DEC_ERR_ARG, "dec_mg_level_size: NULL argument");
  if (level < 0 || level >= static_cast<int>(mg->lv.size())) fail(DEC_ERR_ARG, "dec_mg_level_size: bad level");
  *n = mg->lv[level]->n;
  DEC_CATCH
}

int dec_mg_finest_mesh(dec_mg mg, dec_mesh *m) {
  DEC_TRY
  if (!mg || !m) fail(DEC_ERR_ARG, "dec_mg_finest_mesh: NULL argument");
  if (mg->meshes.empty()) fail(DEC_ERR_UNSUPPORTED, "dec_mg_finest_mesh: the hierarchy was built from matrices");
  *m = mg->meshes[0].get();
  DEC_CATCH
}

int dec_mg_export_level(dec_mg mg, int32_t level, int32_t which, int64_t *nnz, int32_t *rowptr, int32_t *col,
                        double *val) {
  DEC_TRY
  if (!mg) fail(DEC_ERR_ARG, "dec_mg_export_level: NULL handle");
  int nl = static_cast<int>(mg->lv.size());
  if (level < 0 || level >= nl) fail(DEC_ERR_ARG, "dec_mg_export_level: bad level");
  if (which != 0 && level == nl - 1) fail(DEC_ERR_ARG, "dec_mg_export_level: coarsest level has no transfer");
  const dec::HostCsr &A = which == 0 ? mg->lv[level]->A : (which == 1 ? mg->lv[level]->R : mg->lv[level]->P);
  if (which < 0 || which > 2) fail(DEC_ERR_ARG, "dec_mg_export_level: which must be 0 (A), 1 (R) or 2 (P)");
  if (nnz) *nnz = static_cast<int64_t>(A.col.size());
  if (rowptr) std::copy(A.ptr.begin(), A.ptr.end(), rowptr);
  if (col) std::copy(A.col.begin(), A.col.end(), col);
  if (val) std::copy(A.val.begin(), A.val.end(), val);
  DEC_CATCH
}

int dec_mg_export_colors(dec_mg mg, int32_t level, int32_t *color, int32_t *ncolors) {
  DEC_TRY
  if (!mg) fail(DEC_ERR_ARG, "dec_mg_export_colors: NULL handle");
  if (level < 0 || level >= static_cast<int>(mg->lv.size())) fail(DEC_ERR_ARG, "dec_mg_export_colors: bad level");
  const Level &L = *mg->lv[level];
  if (color) std::copy(L.color.begin(), L.color.end(), color);
  if (ncolors) *ncolors = L.ncolors;
  DEC_CATCH
}

int dec_mg_export_blocks(dec_mg mg, int32_t level, int32_t *block, int32_t *nblocks) {
  DEC_TRY
  if (!mg) fail(DEC_ERR_ARG, "dec_mg_export_blocks: NULL handle");
  if (level < 0 || level >= static_cast<int>(mg->lv.size())) fail(DEC_ERR_ARG, "dec_mg_export_blocks: bad level");
  const Level &L = *mg->lv[level];
  if (block)
    for (int k = 0; k < L.nblk; k++)
      for (int i = L.hbstart[k]; i < L.hbstart[k + 1]; i++) block[L.perm[i]] = k;
  if (nblocks) *nblocks = L.nblk;
  DEC_CATCH
}

int dec_mg_set_smoother(dec_mg mg, int32_t alg, int32_t steps, double omega, int32_t coarse_direct) {
  DEC_TRY
  if (!mg) fail(DEC_ERR_ARG, "dec_mg_set_smoother: NULL handle");
  if (alg < DEC_SMOOTH_CG || alg > DEC_SMOOTH_BLOCK_GS) fail(DEC_ERR_ARG, "dec_mg_set_smoother: unknown smoother");
  if (steps < 0) fail(DEC_ERR_ARG, "dec_mg_set_smoother: steps must be >= 0");
  if (coarse_direct && !mg->lv.back()->d.Z.p)
    fail(DEC_ERR_UNSUPPORTED, "dec_mg_set_smoother: coarsest level too large for the dense direct solve");
  mg->alg = alg;
  mg->steps = steps;
  mg->omega = omega;
  mg->coarse_direct = coarse_direct != 0;
  DEC_CATCH
}

int dec_mg_cycles(dec_mg mg, int32_t mu, int32_t cycles, void *u, const void *b, void *stream) {
  DEC_TRY
  if (!mg || !u || !b) fail(DEC_ERR_ARG, "dec_mg_cycles: NULL argument");
  if (mu < 1 || cycles < 0) fail(DEC_ERR_ARG, "dec_mg_cycles: mu >= 1 and cycles >= 0 required");
  hipStream_t s = static_cast<hipStream_t>(stream);
  FineIO io = fine_in(*mg, static_cast<double *>(u), static_cast<const double *>(b), true, s);
  for (int c = 0; c < cycles; c++) mu_cycle<double>(*mg, 0, io.u, io.b, mu, false, s);
  fine_out(*mg, static_cast<double *>(u), s);
  dec::check_launch("dec_mg_cycles");
  DEC_CATCH
}

int dec_mg_full_multigrid(dec_mg mg, int32_t mu, int32_t cycles, const void *b, void *u, void *stream) {
  DEC_TRY
  if (!mg || !u || !b) fail(DEC_ERR_ARG, "dec_mg_full_multigrid: NULL argument");
  if (mu < 1 || cycles < 0) fail(DEC_ERR_ARG, "dec_mg_full_multigrid: mu >= 1 and cycles >= 0 required");
  hipStream_t s = static_cast<hipStream_t>(stream);
  FineIO io = fine_in(*mg, static_cast<double *>(u), static_cast<const double *>(b), false, s);
  fmg_rec(*mg, 0, io.b, io.u, mu, cycles, s);
  for (int c = 0; c < cycles; c++) mu_cycle<double>(*mg, 0, io.u, io.b, mu, false, s);
  fine_out(*mg, static_cast<double *>(u), s);
  dec::check_launch("dec_mg_full_multigrid");
  DEC_CATCH
}

int dec_mg_solve(dec_mg mg, int32_t variant, double tol, int32_t max_cycles, void *u, const void *b,
                 int32_t *cycles_done, double *relres, void *stream) {
  DEC_TRY
  if (!mg || !u || !b) fail(DEC_ERR_ARG, "dec_mg_solve: NULL argument");
  if (variant < DEC_SOLVE_PLAIN_F64 || variant > DEC_SOLVE_PCG_MIXED) fail(DEC_ERR_ARG, "dec_mg_solve: bad variant");
  if ((variant == DEC_SOLVE_MIXED_IR || variant == DEC_SOLVE_PCG_MIXED) && mg->alg == DEC_SMOOTH_CG)
    fail(DEC_ERR_UNSUPPORTED, "dec_mg_solve: the mixed variants need a Gauss-Seidel or Jacobi smoother");
  if ((variant == DEC_SOLVE_PCG_F64 || variant == DEC_SOLVE_PCG_MIXED) && mg->alg == DEC_SMOOTH_CG)
    fail(DEC_ERR_UNSUPPORTED, "dec_mg_solve: the CG variants take the V-cycle of a Gauss-Seidel or Jacobi smoother");
  int c = 0;
  double rr = 0.0;
  try {
    if (variant == DEC_SOLVE_PCG_F64 || variant == DEC_SOLVE_PCG_MIXED)
      pcg_solve(*mg, variant == DEC_SOLVE_PCG_MIXED, tol, max_cycles, static_cast<double *>(u),
                static_cast<const double *>(b), &c, &rr, static_cast<hipStream_t>(stream));
    else
      solve(*mg, variant, tol, max_cycles, static_cast<double *>(u), static_cast<const double *>(b), &c, &rr,
            static_cast<hipStream_t>(stream));
  } catch (...) {
    if (cycles_done) *cycles_done = c;
    if (relres) *relres = rr;
    throw;
  }
  if (cycles_done) *cycles_done = c;
  if (relres) *relres = rr;
  DEC_CATCH
}

int dec_nn_create(dec_mg mg, uint64_t seed, dec_nn *out) {
  DEC_TRY
  if (!mg || !out) fail(DEC_ERR_ARG, "dec_nn_create: NULL argument");
  std::vector<dec::NnOps> ops;
  int nl = static_cast<int>(mg->lv.size());
  for (int l = 0; l < nl; l++) {
    Level &L = *mg->lv[l];
    bool has = l + 1 < nl;
    ops.push_back({&L.A, has ? &L.R : nullptr, has ? &L.P : nullptr, &L.perm});
  }
  *out = dec::nn_create(ops, seed);
  DEC_CATCH
}

int dec_mg_set_learned(dec_mg mg, dec_nn nn, int32_t enable, int32_t min_rows, int32_t max_rows,
                       int32_t applications) {
  DEC_TRY
  if (!mg) fail(DEC_ERR_ARG, "dec_mg_set_learned: NULL handle");
  if (enable && !nn) fail(DEC_ERR_ARG, "dec_mg_set_learned: no network");
  if (applications < 1) fail(DEC_ERR_ARG, "dec_mg_set_learned: applications must be >= 1");
  if (nn) {
    std::vector<int> sizes;
    for (auto &L : mg->lv) sizes.push_back(L->n);
    // the network must carry this hierarchy's operators; its work buffers
    // are sized here, outside any graph capture of the cycles
    dec::nn_bind(*nn, sizes);
  }
  mg->nn = nn;
  mg->learned = enable != 0;
  mg->learned_min_rows = min_rows;
  mg->learned_max_rows = max_rows;
  mg->learned_apps = applications;
  DEC_CATCH
}

int dec_mg_learned_stats(dec_mg mg, int32_t *fallbacks, int32_t *learned_cycles) {
  DEC_TRY
  if (!mg) fail(DEC_ERR_ARG, "dec_mg_learned_stats: NULL handle");
  if (fallbacks) *fallbacks = mg->fallbacks;
  if (learned_cycles) *learned_cycles = mg->learned_cycles;
  DEC_CATCH
}

int dec_mg_destroy(dec_mg mg) {
  DEC_TRY
  if (mg)
    for (auto &m : mg->meshes) m->owned_by_mg = false;
  delete mg;
  DEC_CATCH
}

}  // extern "C"
