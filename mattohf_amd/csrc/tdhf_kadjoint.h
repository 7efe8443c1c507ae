// tdhf_kadjoint.h -- reverse (adjoint) RK4 stages through the density matrices
// of the k-points (gfx950, FP64).  No counterpart in the reference: like
// adjoint_kernel (tdhf_adjoint.h) they differentiate ubkwbk_hwbk,
// src/Functions.f90:187-209, with the matrices of tdhf_kspace.h.
//
// For the cotangent gbar of H y, with K_k of y as in tdhf_kspace.h,
//     J^T gbar = T_a gbar + (vion + vH) gbar + 2 occ (K_H s) y
//                + sum_x' K_k(x,x') gbar_ki(x') + Q_k(x,x') y_ki(x'),
//     Q_k(x,x') = sum_q conj(T_{q-k}(x-x')) P_q(x,x'),
//     P_q(x,x') = sum_j gbar_qj(x) conj(y_qj(x')) + y_qj(x) conj(gbar_qj(x')),
// (the variation of K is the Toeplitz product of the variation of rho, and its
// transpose the one with the conjugate spectra).  Both matrices are Hermitian.
// So a reverse stage is two Toeplitz products per pair of grid points and two
// matrix products, instead of two convolutions per pair of orbitals.  The
// density, s = Re sum conj(gbar) y and the field derivative follow from rho and
// P: n(x) = sum_k rho_k(x,x), s(x) = sum_k P_k(x,x)/2, and
//     Re sum conj(gbar) (K_1 * y) = sum_{x > x'} Re K_1(x-x') conj(P(x,x')) + ...
// with the diagonal counted half.
#pragma once
#include "tdhf_adjoint.h"
#include "tdhf_kspace.h"

namespace tdhf {

struct KAdjArgs {
  AdjArgs a;            // mode, fields, buffers, tape and batch strides (states padded)
  int ng, n, nchunk;
  const zd* ktab;
  const zd* tw;
  const zd* om;
  zd* hm;               // H matrices, then the Q matrices qoff later; per trajectory hstride
  size_t qoff, hstride;
  double* nx;           // n(x), s(x), then the tasks' field derivatives; per trajectory nstride
  size_t nstride;
  const double* J;      // per-step J (current-squared objective), or nullptr
  double vcell;
};

__host__ __device__ constexpr size_t kadj_extra(int ng, int gpw) {
  return (size_t)2 * ng + kmat_tasks(ng, gpw);
}

// Operands of trajectory blockIdx.y and the field of the stage.
struct KAdjView {
  const zd *y, *g;
  int step;
  double fa;
};
__device__ __forceinline__ KAdjView kadj_view(const KAdjArgs& ka) {
  const AdjArgs& a = ka.a;
  const int tr = blockIdx.y;
  KAdjView v;
  v.step = a.step;
  v.y = a.y;
  if (a.step_base) {
    v.step = *a.step_base - a.jstep;
    v.y = a.tape + ((size_t)(v.step % a.tape_seg) * 4 + (a.mode - 1)) * a.blk;
  }
  v.y += (size_t)tr * a.tstride;
  v.g = a.mode == A_EGRAD ? v.y : a.gb + (size_t)tr * a.tstride;
  const double At = a.Aarr[(size_t)tr * a.fstride + v.step];
  const double Av = a.Aavearr[(size_t)tr * a.fstride + v.step];
  v.fa = a.mode == A_S1 ? 2.0 * Av - At : (a.mode == A_S2 || a.mode == A_S3) ? Av : At;
  return v;
}

// One of the two matrices (QM: Q, else H) of one (x, block of x'), one wave per
// task as kmat_kernel; grid z chooses the matrix (both in one wave do not fit
// the registers).  A_EGRAD: y in the place of gbar; Q is then half of itself
// plus the kinetic elements, so that the two sum to dE/du's.
template <int N, bool QM>
__device__ __forceinline__ void kadj_mat_task(const KAdjArgs& ka, zd* smem) {
  using K = KGeo<N>;
  using F = GroupFFT<N>;
  constexpr int R = K::R, L = K::L, KK = K::KK, XR = K::XR, GPW = K::GPW;
  constexpr int DEPTH = QM ? 1 : 4;  // bands in flight
  const AdjArgs& a = ka.a;
  const int NG = ka.ng, nb = a.nb, tr = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63, nth = blockDim.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int W = nth >> 6;
  const int l = lane % L, gw = lane / L;
  const int kl = lane % K::KL, xs = lane / K::KL;
  zd* tile = smem + (size_t)wave * K::TILE;
  zd* T = tile + gw * K::P;
  zd* sOm = smem + (size_t)W * K::TILE;
  zd* sTw = sOm + N;
  zd* sK1 = sTw + F::TWN;
  double* sK2 = reinterpret_cast<double*>(sK1 + NG);
  const int task = blockIdx.x * W + wave;
  const bool live = task < kmat_tasks(NG, GPW);
  const int q0 = (live ? task : 0) / GPW;
  int X = (int)((__fsqrt_rn(8.0f * (float)q0 + 1.0f) - 1.0f) * 0.5f);
  while (X * (X + 1) / 2 > q0) --X;
  while ((X + 1) * (X + 2) / 2 <= q0) ++X;
  const int b = __builtin_amdgcn_readfirstlane(q0 - X * (X + 1) / 2);
  const int x = __builtin_amdgcn_readfirstlane(X * GPW + (live ? task : 0) % GPW);
  const int x0 = b * GPW;
  const KAdjView v0 = kadj_view(ka);
  const unsigned xstride = (unsigned)(nb * N);
  const unsigned uoff = (unsigned)((xs * XR * xstride + kl) * sizeof(zd));
  const unsigned coff = (unsigned)(kl * sizeof(zd));
  const size_t po = (size_t)x0 * xstride, co = (size_t)x * xstride;
  zd by[DEPTH][R], bg[DEPTH][R], oy[DEPTH][KK], og[DEPTH][KK];
  auto fetch = [&](auto dc, int j) {
    constexpr int d = decltype(dc)::value;
    static_for<0, R>([&](auto rc) {
      constexpr int r = decltype(rc)::value, kk = r / XR, xr = r % XR;
      by[d][r] = gload_at(v0.y + po + xr * xstride + j * N + 64 * kk, uoff);
      if constexpr (QM) bg[d][r] = gload_at(v0.g + po + xr * xstride + j * N + 64 * kk, uoff);
    });
    static_for<0, KK>([&](auto kc) {
      constexpr int kk = decltype(kc)::value;
      oy[d][kk] = gload_at(v0.y + co + j * N + 64 * kk, coff);
      if constexpr (QM) og[d][kk] = gload_at(v0.g + co + j * N + 64 * kk, coff);
    });
  };
  static_for<0, DEPTH>([&](auto dc) {
    constexpr int d = decltype(dc)::value;
    fetch(dc, d < nb ? d : nb - 1);
  });
  for (int i = tid; i < N; i += nth) sOm[i] = gload(ka.om + i);
  for (int i = tid; i < F::TWN; i += nth) sTw[kspace_tw_slot<N>(i)] = gload(ka.tw + i);
  for (int i = tid; i < NG; i += nth) {
    sK1[i] = gload(reinterpret_cast<const zd*>(a.kc + 2 * NG) + i);
    sK2[i] = gload(a.kc + NG + i);
  }
  auto tw1 = [&](int g) { return sTw[g * L + l]; };
  auto tw2 = [&](int i) { return N == 128 ? sTw[N + 4 * i + (l & 3)] : sTw[N + i * L + l]; };
  F fft;
  auto fwd = [&](zd(&v)[R]) {
    if constexpr (N == 128) fft.fwd_t(v, T, l, tw1, tw2);
    else fft.fwd_t(v, T, l, tw1);
  };
  auto inv = [&](zd(&v)[R]) { fft.inv_t(v, T, l, tw1, tw2); };
  double kA[KK];
  static_for<0, KK>([&](auto kc) {
    constexpr int kk = decltype(kc)::value;
    kA[kk] = gload(a.kx + kl + 64 * kk) + v0.fa;
  });
  lds_barrier();  // tables in LDS; no further barrier
  if (!live) return;

  // ---- rho_k or P_k at (x,x'), lanes over k ----
  zd src[R];
  static_for<0, R>([&](auto rc) { src[decltype(rc)::value] = mk(0.0, 0.0); });
  for (int j0 = 0; j0 < nb; j0 += DEPTH)
    static_for<0, DEPTH>([&](auto dc) {
      constexpr int d = decltype(dc)::value;
      if (j0 + d < nb) {
        static_for<0, R>([&](auto rc) {
          constexpr int r = decltype(rc)::value, kk = r / XR;
          if constexpr (QM) {
            zfmac(src[r], og[d][kk], by[d][r]);
            zfmac(src[r], oy[d][kk], bg[d][r]);
          } else {
            zfmac(src[r], oy[d][kk], by[d][r]);
          }
        });
        if (j0 + d + DEPTH < nb) fetch(dc, j0 + d + DEPTH);
      }
    });
  // ---- density or s on the diagonal; field derivative ----
  double* nx = ka.nx + (size_t)tr * ka.nstride;
  double fd = 0.0;
  if (b == X) {
    double n = 0.0;
    static_for<0, R>([&](auto rc) {
      constexpr int r = decltype(rc)::value, kk = r / XR, xr = r % XR;
      if (x0 + xs * XR + xr == x) {
        n += src[r].x;
        fd = fma(kA[kk], src[r].x, fd);
      }
    });
    n = wave_sum(n);
    if (lane == 0) gstore(nx + (QM ? NG : 0) + x, QM ? 0.5 * n : n);
  }
  if constexpr (QM) {
    static_for<0, XR>([&](auto rc) {
      constexpr int xr = decltype(rc)::value;
      const int yy = (x - (x0 + xs * XR + xr)) & (NG - 1);
      const zd k1 = sK1[yy];
      static_for<0, KK>([&](auto kc) {
        const zd p = src[decltype(kc)::value * XR + xr];
        fd = fma(k1.x, p.x, fd);
        fd = fma(k1.y, p.y, fd);
      });
    });
    fd = wave_sum(fd) * (b == X ? 0.5 : 1.0);
    if (lane == 0) gstore(nx + 2 * NG + task, fd);
  }

  // ---- the Toeplitz product: spectra as they are for rho, conjugate for P ----
  to_groups<N>(src, tile, kl, xs, gw, l);
  const unsigned toff = (unsigned)((((x - x0 - gw) & (NG - 1)) * 2 * N + l) * sizeof(zd));
  zd kv[R];
  static_for<0, 2>([&](auto ec) {
    constexpr int eo = decltype(ec)::value;
    zd tb[R];
    static_for<0, R>([&](auto jc_) {
      constexpr int j = decltype(jc_)::value;
      tb[j] = gload_at(ka.ktab + (eo * R + j) * L, toff);
    });
    zd v[R];
    static_for<0, R>([&](auto mc) {
      constexpr int m = decltype(mc)::value;
      v[m] = eo == 0 ? src[m] : zmul(src[m], sOm[L * m + l]);
    });
    fwd(v);
    static_for<0, R>([&](auto jc_) {
      constexpr int j = decltype(jc_)::value;
      v[j] = QM ? zmulc(v[j], tb[j]) : zmul(v[j], tb[j]);
    });
    inv(v);
    static_for<0, R>([&](auto mc) {
      constexpr int m = decltype(mc)::value;
      kv[m] = eo == 0 ? v[m] : zadd(kv[m], zmulc(v[m], sOm[L * m + l]));
    });
    __builtin_amdgcn_sched_barrier(0);
  });
  to_lanes<N>(kv, tile, kl, xs, gw, l);
  const bool eg = a.mode == A_EGRAD;
  const double ht = !QM || eg ? 1.0 : 0.0, hs = QM && eg ? 0.5 : 1.0;
  zd* out = ka.hm + (size_t)tr * ka.hstride + (QM ? ka.qoff : 0);
  static_for<0, XR>([&](auto rc) {
    constexpr int xr = decltype(rc)::value;
    const int xp = x0 + xs * XR + xr, yy = (x - xp) & (NG - 1);
    const double k2 = ht * sK2[yy];
    const zd k1 = zscal(sK1[yy], ht);
    static_for<0, KK>([&](auto kc) {
      constexpr int kk = decltype(kc)::value;
      const zd q = kv[kk * XR + xr];
      gstore(out + ((size_t)x * (NG + 1) + xp) * N + kl + 64 * kk,
             mk(fma(hs, q.x, fma(kA[kk], k1.x, k2)), fma(hs, q.y, kA[kk] * k1.y)));
    });
  });
}

template <int N>
__global__ void __launch_bounds__(256, 2) kadj_mat_kernel(KAdjArgs ka) {
  extern __shared__ zd smem[];
  if (blockIdx.z == 0) kadj_mat_task<N, false>(ka, smem);
  else kadj_mat_task<N, true>(ka, smem);
}

// J^T gbar from the matrices and the reverse RK4 combination (as adjoint_kernel)
// for XT grid points x, NBT bands and up to 64 k-points per workgroup; split as
// kapply_kernel.  In stage 1 of the current-squared objective the cotangent of
// J after the step before, jf P_A y with jf = 2 dt J (-2 occ dv/vcell) and
// P_A y = K_1 * y + (k + A) y, joins the matrix that multiplies y.
__host__ __device__ constexpr size_t kadj_apply_lds(int nw, int nbt, int xt, int ng) {
  return (size_t)nw * xt * kapply_round(nbt) * 64 * sizeof(zd) + ng * sizeof(zd) +
         16 * sizeof(double);
}

template <int NBT, int XT>
__global__ void __launch_bounds__(512, 2) kadj_apply_kernel(KAdjArgs ka) {
  constexpr int BR = kapply_round(NBT);
  extern __shared__ zd smem[];
  const AdjArgs& a = ka.a;
  const int NG = ka.ng, N = ka.n, nb = a.nb, mode = a.mode, tr = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63, nth = blockDim.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int W = nth >> 6;
  const int KL = N < 64 ? N : 64, XS = 64 / KL;
  const int kb = N > 64 ? N / 64 : 1, item = blockIdx.x;
  const int kc = item % kb, ch = (item / kb) % ka.nchunk, x0 = item / (kb * ka.nchunk) * XT;
  const int i0 = ch * NBT, ni = nb - i0 < NBT ? nb - i0 : NBT;
  const int k = 64 * kc + (lane & (KL - 1)), xs = lane / KL;
  zd* sK1 = smem + (size_t)W * XT * BR * 64;
  double* sVh = reinterpret_cast<double*>(sK1 + NG);  // vH, K_H s at the XT points
  const KAdjView v0 = kadj_view(ka);
  const zd* hm = ka.hm + (size_t)tr * ka.hstride;
  const zd* qm = hm + ka.qoff;
  const double* nx = ka.nx + (size_t)tr * ka.nstride;
  const size_t wstride = (size_t)nb * N;
  const bool js = ka.J && mode == A_S1 && v0.step > 0;
  double jf = 0.0, Ap = 0.0;
  if (js) {
    jf = 2.0 * a.dt * gload(ka.J + (size_t)tr * a.fstride + v0.step - 1) *
         (-2.0 * a.occ * a.dv / ka.vcell);
    Ap = a.Aarr[(size_t)tr * a.fstride + v0.step - 1];
    for (int i = tid; i < NG; i += nth)
      sK1[i] = gload(reinterpret_cast<const zd*>(a.kc + 2 * NG) + i);
    lds_barrier();
  }
  zd acc[XT][NBT];
  static_for<0, XT>([&](auto xc) {
    static_for<0, NBT>(
        [&](auto ic) { acc[decltype(xc)::value][decltype(ic)::value] = mk(0.0, 0.0); });
  });
  const int bshift = N == 128 ? 2 : N == 64 ? 3 : 4;
  const int per = NG / (W * XS);  // x' per lane
  for (int it = 0; it < per; ++it) {
    const int xp = (it * W + wave) * XS + xs;
    zd h[XT], q[XT];
    static_for<0, XT>([&](auto xc) {
      constexpr int i = decltype(xc)::value;
      const int x = x0 + i;
      const bool low = (xp >> bshift) <= (x >> bshift);
      const size_t e = ((size_t)(low ? x : xp) * (NG + 1) + (low ? xp : x)) * N + k;
      const zd hv = gload(hm + e), qv = gload(qm + e);
      h[i] = mk(hv.x, low ? hv.y : -hv.y);
      q[i] = mk(qv.x, low ? qv.y : -qv.y);
    });
    if (js)
      static_for<0, XT>([&](auto xc) {
        constexpr int i = decltype(xc)::value;
        const zd k1 = sK1[(x0 + i - xp) & (NG - 1)];
        q[i].x = fma(jf, k1.x, q[i].x);
        q[i].y = fma(jf, k1.y, q[i].y);
      });
    const size_t wo = (size_t)xp * wstride + (size_t)i0 * N + k;
    zd gv[NBT], yv[NBT];
    static_for<0, NBT>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      const size_t e = wo + (i < ni ? i : ni - 1) * N;
      gv[i] = gload(v0.g + e);
      yv[i] = gload(v0.y + e);
    });
    static_for<0, XT>([&](auto xc) {
      constexpr int i = decltype(xc)::value;
      static_for<0, NBT>([&](auto ic) {
        constexpr int j = decltype(ic)::value;
        zfma(acc[i][j], h[i], gv[j]);
        zfma(acc[i][j], q[i], yv[j]);
      });
    });
  }
  // ---- Hartree potential and response at the XT points ----
  for (int i = wave; i < XT; i += W) {
    double s = 0.0, r = 0.0;
    for (int xp = lane; xp < NG; xp += 64) {
      const double kh = gload(a.kc + ((x0 + i - xp) & (NG - 1)));
      s = fma(kh, gload(nx + xp), s);
      r = fma(kh, gload(nx + NG + xp), r);
    }
    s = wave_sum(s);
    r = wave_sum(r);
    if (lane == 0) {
      sVh[i] = a.occ * s;
      sVh[XT + i] = r;
    }
  }
  const bool eg = mode == A_EGRAD;
  const size_t so = (size_t)tr * a.tstride;
  static_for<0, (NBT + BR - 1) / BR>([&](auto rc) {
    constexpr int r0 = decltype(rc)::value * BR;
    if (r0 < ni) {
      if constexpr (r0 > 0) lds_barrier();
      static_for<0, XT>([&](auto xc) {
        static_for<0, BR>([&](auto ic) {
          constexpr int i = decltype(xc)::value, j = decltype(ic)::value;
          if constexpr (r0 + j < NBT) smem[((wave * XT + i) * BR + j) * 64 + lane] = acc[i][r0 + j];
        });
      });
      lds_barrier();
      for (int q = tid; q < XT * BR * KL; q += nth) {
        const int kq = q & (KL - 1), j = (q / KL) % BR, i = q / (KL * BR);
        if (r0 + j >= ni) continue;
        const int x = x0 + i;
        const size_t o = (size_t)x * wstride + (size_t)(i0 + r0 + j) * N + 64 * kc + kq;
        const zd gv = gload(v0.g + o), yv = gload(v0.y + o);
        const double kx = gload(a.kx + 64 * kc + kq), vi = gload(a.vion + x);
        zd ubv = mk(0.0, 0.0), uav = ubv;
        if (!eg) {
          ubv = gload(a.ub + so + o);
          if (mode != A_S4) uav = gload(a.ua + so + o);
        }
        zd h = mk(0.0, 0.0);
        for (int w2 = 0; w2 < W; ++w2)
          for (int s2 = 0; s2 < XS; ++s2)
            h = zadd(h, smem[((w2 * XT + i) * BR + j) * 64 + s2 * KL + kq]);
        const double kA = kx + v0.fa;
        const double d = fma(0.5 * kA, kA, sVh[i] + vi);
        if (eg) {
          // dE/du = occ dv (2 (T y + (vion + vH) y) + (V_F + V'_F) y)
          h = zadd(h, zscal(yv, 2.0 * d));
          const zd c = zscal(h, a.occ * a.dv);
          const double w = a.dt / 6.0;  // gbar_4 = i (dt/6) c
          gstore(a.cout + so + o, c);
          gstore(a.gout + so + o, mk(-w * c.y, w * c.x));
          continue;
        }
        h = zadd(h, zadd(zscal(gv, d), zscal(yv, 2.0 * a.occ * sVh[XT + i])));
        if (js) h = zadd(h, zscal(yv, jf * (kx + Ap)));
        zd kb;
        if (mode == A_S4) {
          uav = zadd(ubv, h);
          kb = zadd(zscal(ubv, a.dt / 3.0), zscal(h, a.dt));
        } else {
          uav = zadd(uav, h);
          if (mode == A_S3) kb = zadd(zscal(ubv, a.dt / 3.0), zscal(h, 0.5 * a.dt));
          else if (mode == A_S2) kb = zadd(zscal(ubv, a.dt / 6.0), zscal(h, 0.5 * a.dt));
          else kb = zscal(uav, a.dt / 6.0);  // A_S1: the next step's gbar_4
        }
        gstore(a.ua + so + o, uav);
        gstore(a.gout + so + o, mk(-kb.y, kb.x));  // i kbar
      }
    }
  });
  // field derivative of the stage at x: the sums of its tasks
  if (!eg && a.abar && ch == 0 && kc == 0 && tid < XT) {
    const int x = x0 + tid, gpw = 1 << bshift, X = x >> bshift;
    const double* p = nx + 2 * NG + (gpw * (X * (X + 1) / 2) + x - X * gpw);
    double s = 0.0;
    for (int b = 0; b <= X; ++b, p += gpw) s += gload(p);
    const size_t slot = a.step_base ? (size_t)(v0.step % a.tape_seg) * 4 + (mode - 1) : 0;
    gstore(a.abar + (size_t)tr * a.abar_tstride + slot * NG + x, s);
  }
}

// Start of the reverse sweep of the current-squared objective, at the final
// state y: ua = c, gb = i (dt/6) c with c = 2 dt J (-2 occ dv/vcell) P_A y,
// P_A y = K_1 * y + (k + A) y; one thread per (band, k) at x (once per call),
// blocks of them in grid z.  Bound by the latency of the reads of y, sixteen in
// flight: three states of NG=128, NK=128, NB=8 128 -> 36 us against one block
// of threads per x and one read at a time.
__global__ void __launch_bounds__(256) kadj_jinit_kernel(JgradArgs j, int ng, int n) {
  __shared__ zd sK1[128];
  const int x = blockIdx.x, tr = blockIdx.y, q = blockIdx.z * 256 + threadIdx.x;
  const size_t so = (size_t)tr * j.tstride;
  const int m = j.nb * n;
  for (int i = threadIdx.x; i < ng; i += 256)
    sK1[i] = gload(reinterpret_cast<const zd*>(j.kc + 2 * ng) + i);
  const double A = j.Aarr[(size_t)tr * j.fstride + j.step];
  const double J = j.J[(size_t)tr * j.fstride + j.step];
  const double f = 2.0 * j.dt * J * (-2.0 * j.occ * j.dv / j.vcell);
  lds_barrier();
  if (q >= m) return;
  const size_t o = so + (size_t)x * m + q;
  zd p = zscal(gload(j.y + o), gload(j.kx + q % n) + A);
#pragma unroll 16
  for (int xp = 0; xp < ng; ++xp)
    zfma(p, sK1[(x - xp) & (ng - 1)], gload(j.y + so + (size_t)xp * m + q));
  const zd c = zscal(p, f);
  const double w = j.dt / 6.0;
  gstore(j.ua + o, c);
  gstore(j.gb + o, mk(-w * c.y, w * c.x));
}

}  // namespace tdhf
