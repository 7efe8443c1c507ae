// tdhf_gs.h -- device kernels of the ground-state (Krylov / Rayleigh-Ritz)
// iteration: GS_calculation, KS_ubk2_SVD and Subspace_diag
// (src/GS_calculation.f90:26-57,124-237).
//
// The H applications reuse the context's path (gs_product).  The small per-k
// dense steps run one workgroup per k-point, on columns held in LDS:
//   orth_kernel : dvcell-weighted modified Gram-Schmidt, right-looking: once a
//                 column is normalised, its projection leaves all later ones,
//                 each on its own wave, so the chain is one column and not one
//                 pair of columns long.  Two passes make the Krylov basis (it
//                 replaces the left singular vectors of ZGESVD('O') rescaled by
//                 1/sqrt(dvcell), :161-166; both are a dvcell-orthonormal basis
//                 of the same span, and the Rayleigh-Ritz step depends on the
//                 span only), one pass is Gram_Schmidt (src/mATTOHF.f90:134-157).
//   rr_kernel   : subspace matrix <w_r|H|w_c> dvcell (:173-181 / :217-224),
//                 cyclic complex Jacobi eigensolver standing in for ZHEEV
//                 (ascending eigenvalues), and the rotation into the lowest
//                 NB Ritz vectors (:184-190 / :227-233).
#pragma once
#include "tdhf_kspace.h"

struct tdhf_ctx;

namespace tdhf {

struct GsWork {
  zd* W = nullptr;   // Krylov columns (NG, NB*ncg, NK)
  zd* HW = nullptr;  // their H images
  zd *KW = nullptr, *KH = nullptr;  // the same, padded, on the density-matrix path
  double* eps = nullptr;
  int* nonconv = nullptr;  // set by rr_kernel when its eigensolver does not converge
  int ncg = 0;
};

__device__ __forceinline__ double bsum(double v, double* red) {
  const int t = threadIdx.x;
  red[t] = v;
  __syncthreads();
  for (int h = blockDim.x >> 1; h > 0; h >>= 1) {
    if (t < h) red[t] += red[t + h];
    __syncthreads();
  }
  const double r = red[0];
  __syncthreads();
  return r;
}

// ---------------------------------------------------------------------------
// Modified Gram-Schmidt of the m columns W[k][c][x] at every k-point (one
// workgroup each, NG x fastest), npass passes, in place and, with copy, also to
// copy (m columns per k of ldc).  Columns in LDS (pitch NG + 1); wave w updates
// columns w, w + W, ...  Step b: every wave removes column b from its later
// columns; the wave of column b + 1 then normalises that one, and one barrier
// ends the step.  The projections reach a column in the order of the plain
// algorithm.  Bound by the chain of m steps (dot product, wave sum, update, norm,
// barrier), ~0.8 us each: 16 columns of NG=64, two passes, on 64 k-points 27 us
// against 323 us with one pair of columns at a time and a barrier per level of
// the sums.
// ---------------------------------------------------------------------------
__host__ __device__ constexpr size_t orth_lds(int ng, int m) {
  return (size_t)m * (ng + 1) * sizeof(zd);
}
__global__ void __launch_bounds__(1024) orth_kernel(zd* Wk, int ng, int m, double dv, int npass,
                                                   zd* copy, int ldc) {
  extern __shared__ zd sh[];
  const int ik = blockIdx.x, tid = threadIdx.x, lane = tid & 63, nth = blockDim.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), W = nth >> 6;
  zd* wk = Wk + (size_t)ik * m * ng;
  const int ld = ng + 1;
  for (int e = tid; e < m * ng; e += nth) {
    const int c = e / ng, x = e - c * ng;
    sh[c * ld + x] = gload(wk + e);
  }
  // the (up to two) points of a column that a lane holds
  const bool h0 = lane < ng, h1 = lane + 64 < ng;
  const zd zero = mk(0.0, 0.0);
  auto normalise = [&](zd* col, zd v0, zd v1) {
    const double r = rsqrt(wave_sum(zabs2(v0) + zabs2(v1)) * dv);
    if (h0) col[lane] = zscal(v0, r);
    if (h1) col[lane + 64] = zscal(v1, r);
  };
  for (int pass = 0; pass < npass; ++pass) {
    lds_barrier();
    if (wave == 0) normalise(sh, h0 ? sh[lane] : zero, h1 ? sh[lane + 64] : zero);
    lds_barrier();
    for (int b = 0; b + 1 < m; ++b) {
      const zd* yb = sh + b * ld;
      const zd y0 = h0 ? yb[lane] : zero, y1 = h1 ? yb[lane + 64] : zero;
      // the wave of column b + 1 takes it first
      int c = wave;
      while (c <= b) c += W;
      for (; c < m; c += W) {
        zd* xc = sh + c * ld;
        zd v0 = h0 ? xc[lane] : zero, v1 = h1 ? xc[lane + 64] : zero;
        const double re =
            dv * wave_sum(y0.x * v0.x + y0.y * v0.y + (y1.x * v1.x + y1.y * v1.y));
        const double im =
            dv * wave_sum(y0.x * v0.y - y0.y * v0.x + (y1.x * v1.y - y1.y * v1.x));
        v0 = mk(v0.x - (re * y0.x - im * y0.y), v0.y - (re * y0.y + im * y0.x));
        v1 = mk(v1.x - (re * y1.x - im * y1.y), v1.y - (re * y1.y + im * y1.x));
        if (c == b + 1) {
          normalise(xc, v0, v1);
        } else {
          if (h0) xc[lane] = v0;
          if (h1) xc[lane + 64] = v1;
        }
      }
      lds_barrier();
    }
  }
  for (int e = tid; e < m * ng; e += nth) {
    const int c = e / ng, x = e - c * ng;
    const zd v = sh[c * ld + x];
    gstore(wk + e, v);
    if (copy) gstore(copy + (size_t)ik * ldc * ng + e, v);
  }
}

// ---------------------------------------------------------------------------
// Rayleigh-Ritz at one k-point per workgroup: m basis columns W[k][c][x], their
// H images HW alike; writes the lowest nb Ritz vectors to uout[k][b][x].  If the
// cyclic Jacobi iteration has not converged after 100 sweeps, *nonconv is set to
// 1 + ik (the caller reports it).
//
// The rotations of a row-cyclic sweep, (0,1), (0,2), ..., (1,2), ..., that share
// no index commute, and those that share one lie on different antidiagonals
// p + q in that same order, so all rotations of an antidiagonal run at once: 2m - 3
// steps a sweep instead of m(m-1)/2, with the same rotations.  In a step the
// matrix splits into the 2 x 2 blocks of the pairs (and the rows and columns
// of the indices without a partner), one thread each applies the rotations of
// its rows and columns together, and two barriers suffice (angles, blocks).
// Bound by the latency of a step, 0.95 us (0.3 the angles, 0.65 the blocks):
// m = 16 on 64 k-points, six sweeps, 200 us against 845 us with one rotation at
// a time.
// Dynamic LDS: A and V (m^2 complex each), the columns if they fit (WL, pitch
// NG + 1), the rotations (2 m complex) and the order (m ints).
// ---------------------------------------------------------------------------
__host__ __device__ constexpr size_t rr_lds(int ng, int m, bool wl) {
  return ((size_t)2 * m * m + 2 * m + (wl ? (size_t)m * (ng + 1) : 0)) * sizeof(zd) +
         8 * sizeof(double) + (size_t)m * sizeof(int) + 16;
}

template <bool WL>
__global__ void __launch_bounds__(256) rr_kernel(const zd* Wk, const zd* HWk, int ng, int nb, int m,
                                                 double dv, zd* uout, int* nonconv) {
  extern __shared__ zd sh[];
  zd* A = sh;
  zd* V = sh + (size_t)m * m;
  zd* Ws = V + (size_t)m * m;
  zd* rot = Ws + (WL ? (size_t)m * (ng + 1) : 0);
  double* red = reinterpret_cast<double*>(rot + 2 * m);
  int* idx = reinterpret_cast<int*>(red + 8);
  const int ik = blockIdx.x, t = threadIdx.x, nt = blockDim.x;
  const zd* wk = Wk + (size_t)ik * m * ng;
  const zd* hk = HWk + (size_t)ik * m * ng;
  const int ld = WL ? ng + 1 : ng;
  if constexpr (WL) {
    for (int e = t; e < m * ng; e += nt) {
      const int c = e / ng, x = e - c * ng;
      Ws[c * ld + x] = gload(wk + e);
    }
    lds_barrier();
  }
  auto wval = [&](int c, int x) { return WL ? Ws[c * ld + x] : gload(wk + c * ld + x); };
  // subspace matrix: lower triangle and diagonal, mirrored
  for (int e = t; e < m * m; e += nt) {
    const int r = e % m, cc = e / m;
    V[e] = mk(r == cc ? 1.0 : 0.0, 0.0);
    if (cc > r) continue;
    double re = 0.0, im = 0.0;
    for (int x = 0; x < ng; ++x) {
      const zd a = wval(r, x), b = gload(hk + cc * ng + x);
      re += a.x * b.x + a.y * b.y;
      im += a.x * b.y - a.y * b.x;
    }
    A[r + m * cc] = mk(re * dv, cc == r ? 0.0 : im * dv);
    if (cc < r) A[cc + m * r] = mk(re * dv, -im * dv);
  }
  lds_barrier();
  const int r0 = t % m, c0 = t / m, dr = nt % m, dc = nt / m;  // of the thread's elements
  bool converged = false;
  for (int sweep = 0; sweep <= 100; ++sweep) {
    double off = 0.0, tot = 0.0;
    for (int e = t; e < m * m; e += nt) {
      const double v = zabs2(A[e]);
      tot += v;
      if ((e % m) != (e / m)) off += v;
    }
    off = wave_sum(off);
    tot = wave_sum(tot);
    if ((t & 63) == 0) {
      red[2 * (t >> 6)] = off;
      red[2 * (t >> 6) + 1] = tot;
    }
    lds_barrier();
    off = tot = 0.0;
    for (int w = 0; w < nt >> 6; ++w) {
      off += red[2 * w];
      tot += red[2 * w + 1];
    }
    if (off <= 1e-32 * tot) {
      converged = true;
      break;
    }
    if (sweep == 100 || off != off) break;
    for (int s = 1; s <= 2 * m - 3; ++s) {
      // index i rotates with s - i; J's columns p < q are
      // (cs, sn) and (-sn conj(e), cs conj(e)), e = a_pq/|a_pq|: new column i
      // is al_i (column i) + be_i (column s - i)
      if (t < m) {
        const int o = s - t;
        zd al = mk(1.0, 0.0), be = mk(0.0, 0.0);
        if (o >= 0 && o < m && o != t) {
          const int p = t < o ? t : o, q = t < o ? o : t;
          const zd apq = A[p + m * q];
          const double r2 = zabs2(apq);
          if (r2 > 1e-290) {  // (below, the rotation is none in any finite matrix)
            // with d = a_qq - a_pp and h = sqrt(d^2 + 4 |a_pq|^2): cs^2 = (1 + |d|/h)/2,
            // sn = sign(d) |a_pq| / (h cs); two reciprocal roots deep
            const double d = A[q + m * q].x - A[p + m * p].x;
            const double ri = rsqrt(r2), hi = rsqrt(fma(d, d, 4.0 * r2));
            const double w = fma(0.5 * fabs(d), hi, 0.5), ics = rsqrt(w);
            const double cs = w * ics, sn = copysign(r2 * ri * hi * ics, d);
            const zd ec = mk(apq.x * ri, -apq.y * ri);
            al = t == p ? mk(cs, 0.0) : zscal(ec, cs);
            be = t == p ? zscal(ec, -sn) : mk(sn, 0.0);
          }
        }
        rot[2 * t] = al;
        rot[2 * t + 1] = be;
      }
      lds_barrier();
      // thread (r, c), the lower of its pair of rows and of columns, makes the
      // 2 x 2 block A' = J^H A J in place; the higher of the columns V' = V J
      // (an index without a partner is its own, with the identity's factors)
      int r = r0, c = c0;
      for (int e = t; e < m * m; e += nt) {
        int cp = s - c, rp = s - r;
        if (cp < 0 || cp >= m) cp = c;
        if (rp < 0 || rp >= m) rp = r;
        const bool low = c <= cp && r <= rp && (c < cp || r < rp), vec = cp < c;
        if (low || vec) {
          const zd al = rot[2 * c], be = rot[2 * c + 1], al2 = rot[2 * cp], be2 = rot[2 * cp + 1];
          if (vec) {
            const zd v = V[r + m * c], v2 = V[r + m * cp];
            V[r + m * c] = zadd(zmul(al, v), zmul(be, v2));
            V[r + m * cp] = zadd(zmul(al2, v2), zmul(be2, v));
          } else {
            const zd ga = rot[2 * r], gb = rot[2 * r + 1], ga2 = rot[2 * rp], gb2 = rot[2 * rp + 1];
            const zd a0 = A[r + m * c], b0 = A[r + m * cp], d0 = A[rp + m * c], f0 = A[rp + m * cp];
            const zd a1 = zadd(zmul(al, a0), zmul(be, b0)), b1 = zadd(zmul(al2, b0), zmul(be2, a0));
            const zd d1 = zadd(zmul(al, d0), zmul(be, f0)), f1 = zadd(zmul(al2, f0), zmul(be2, d0));
            zd a = zadd(zmulc(a1, ga), zmulc(d1, gb)), b = zadd(zmulc(b1, ga), zmulc(f1, gb));
            zd d = zadd(zmulc(d1, ga2), zmulc(a1, gb2)), f = zadd(zmulc(f1, ga2), zmulc(b1, gb2));
            if (r == c) {  // the rotated pair itself
              a.y = 0.0;
              f.y = 0.0;
              b = d = mk(0.0, 0.0);
            }
            A[r + m * c] = a;
            if (cp != c) A[r + m * cp] = b;
            if (rp != r) A[rp + m * c] = d;
            if (cp != c && rp != r) A[rp + m * cp] = f;
          }
        }
        r += dr;
        c += dc;
        if (r >= m) {
          r -= m;
          ++c;
        }
      }
      lds_barrier();
    }
  }
  if (t == 0 && !converged && nonconv) *nonconv = 1 + ik;
  lds_barrier();
  // ascending order by rank (an order is set for values that are not numbers too)
  for (int i = t; i < m; i += nt) idx[i] = i;
  lds_barrier();
  for (int i = t; i < m; i += nt) {
    const double a = A[i + m * i].x;
    int rank = 0;
    for (int j = 0; j < m; ++j) {
      const double b = A[j + m * j].x;
      rank += b < a || (b == a && j < i) ? 1 : 0;
    }
    if (a == a) idx[rank] = i;
  }
  lds_barrier();
  // rotation: u(:,ib,ik) = sum_c w_c V(c, idx(ib))
  for (int e = t; e < ng * nb; e += nt) {
    const int x = e % ng, ib = e / ng;
    const int col = idx[ib];
    zd s = mk(0.0, 0.0);
    for (int cc = 0; cc < m; ++cc) s = zadd(s, zmul(wval(cc, x), V[cc + m * col]));
    gstore(uout + (size_t)ik * nb * ng + e, s);
  }
}

// ubk_epsbk / ubk_epserrorbk (src/Functions.f90:321-358) from u and H u:
// one workgroup of ng threads per orbital (ib,ik).
__global__ void epsbk_kernel(const zd* u, const zd* hu, int ng, double dv, double* eps,
                             double* err) {
  __shared__ double red[128];
  const int row = blockIdx.x, x = threadIdx.x;
  const zd a = u[(size_t)ng * row + x], h = hu[(size_t)ng * row + x];
  const double e = bsum(a.x * h.x + a.y * h.y, red) * dv;
  const zd r = mk(h.x - e * a.x, h.y - e * a.y);
  const double s = bsum(sqrt(r.x * r.x + r.y * r.y), red);
  if (x == 0) {
    if (eps) eps[row] = e;
    if (err) err[row] = sqrt(s * dv);
  }
}

int ctx_fail(tdhf_ctx* c, int code, const char* msg);
void gs_free(GsWork& g);

}  // namespace tdhf
