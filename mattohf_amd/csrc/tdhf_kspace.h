// tdhf_kspace.h -- H application and RK4 stages through the density matrices
// of the k-points (gfx950, FP64).
//
// The Fock exchange of ubkwbk_vFwbk (src/Functions.f90:237-261) is a sum over
// pairs of orbitals of one convolution over the grid each.  Written out in
// real space it is one matrix per k-point,
//     V_F w_ki(x) = sum_x' K_k(x,x') w_ki(x'),
//     K_k(x,x')   = sum_q T_{k-q}(x-x') rho_q(x,x'),
//     rho_q(x,x') = sum_j u_qj(x) conj(u_qj(x')),
//     T_d(y)      = sum_G t_d(G) exp(2 pi i G y/NG),  t_d(G) = -v(G+d)/(NG NK),
// and for fixed (x,x') the sum over q is a Toeplitz product over the k-mesh.
// It is evaluated as the sum of a circulant and a skew-circulant one of
// length N >= NK (N = 16, 32, 64 or 128), i.e. one transform pair of length N
// over the k-points each:
//     c_d = (T_d + T_{d-N})/2,  s_d = (T_d - T_{d-N})/2,  w = exp(-i pi/N),
//     K = IFFT[c^/N FFT[rho]] + w^-k IFFT[s^/N FFT[w^q rho]],
//     c^ = FFT[c],  s^ = FFT[w^d s]            (tables, kspace_spectrum_kernel).
// So a stage costs 2 NG^2 transform pairs of length N instead of NK^2 NB NBocc
// of length NG (NG=64, NK=64, NB=4: 8192 instead of 65536; NG=128, NK=128,
// NB=8: 32768 instead of 1048576), and the whole of H is in K once the kinetic
// elements K_2(x-x') + (k+A) K_1(x-x') are added to it (the circulant kernels
// of tdhf_kernels.h).  Nothing is approximated: every T_d is used as given,
// so a caller's own table works as well, and no symmetry of v is assumed.
//
// Layout: states are U[x][b][k], k fastest and padded with zeros to N.  A
// wave's loads over k are then contiguous, and the padded entries stay zero
// by themselves (rho_q = 0 and w = 0 there).
//
// A stage is two launches.  kmat_kernel makes H_k(x,x') = K_k(x,x') + the
// kinetic elements, one wave per x and block of x' (as many as a wave has
// transform groups), the blocks up to the one that holds x only: H is
// Hermitian.  Per task:
//   1. lanes over k: rho_k(x,x') from u, the density from the diagonal, and for
//      the observables the traces sum T_k(x-x') conj(rho_k(x,x'));
//   2. through LDS to the transform groups (one group per x', lanes over k
//      as in GroupFFT), the two convolutions, and back;
//   3. lanes over k: the kinetic elements, and out.
// kapply_kernel multiplies the matrices into the columns, adds the local
// potential and applies the RK4 stage update.
//
// Measured per stage (MI355X; row-wise exchange or pair tiles before): one
// trajectory NG=128, NK=128, NB=8 418 -> 42 us; NG=64, NK=100, NB=8 with 4
// occupied 75 -> 25 us; 64 trajectories NG=64, NK=64, NB=4 361 -> 146 us (of
// which kmat 83 us, kapply 60 us); 48 of NK=16, 32, 64 147 -> 75 us.
// kmat_kernel is bound by latency at its three waves per SIMD (35 % of the FP64
// issue slots), kapply_kernel by reading the matrices (245 MB in 58 us for the
// 64 trajectories, 4.2 TB/s).
#pragma once
#include "tdhf_kernels.h"

namespace tdhf {

// Length of the k transforms that hold nk points (0: none does).
__host__ __device__ constexpr int kspace_len(int nk) {
  return nk <= 16 ? 16 : nk <= 32 ? 32 : nk <= 64 ? 64 : nk <= 128 ? 128 : 0;
}

// Geometry of a wave for transforms of length N: R points per lane, groups of
// L lanes, GPW groups (x' values) per wave.  In the lane domain the wave's
// R x 64 values are held as k = lane % KL + 64 kk and x' = (lane / KL) XR + xr,
// register r = kk XR + xr.
template <int N>
struct KGeo {
  using F = GroupFFT<N>;
  static constexpr int R = F::R, L = F::L, GPW = 64 / L;
  static constexpr int KL = N < 64 ? N : 64, XS = 64 / KL, KK = N / KL, XR = R / KK;
  // LDS pitch of a group: the transpose tile of its transforms, and one x'
  // row of N values on the way between the two domains; 8 mod 16 elements
  // where L < 16, so that the groups served together start in different banks
  static constexpr int need = F::TSZ > N ? F::TSZ : N;
  static constexpr int P = L < 16 ? need + ((8 - need % 16) + 16) % 16 : need;
  static constexpr int TILE = GPW * P;  // complex elements per wave
  static_assert(GPW == XS * XR, "lane domain and groups hold the same x'");
};

// Operands of one trajectory (the launch's own, or from the batch table).
struct KTraj {
  int nk;
  double occ;
  const double* kx;    // padded to at least N entries
  const double* vion;
  const double* kc;    // circulant kernels K_H, K_2, K_1 (4 NG)
  const zd* ktab;      // spectra: [(y 2 + eo) R + j] L + l, y = x - x' mod NG
  const double* Aarr;
  const double* Aavearr;
  const zd* u;         // state that defines rho
  const zd* w;         // columns H acts on
  zd* out;
  zd* u0;
  zd* ksum;
  zd* unext;
  zd* tape0;
  double* obs;
  zd* hm;              // matrices of the stage (kmat_kernel)
  double* nx;          // density n(x), then the tasks' observables sums
};

// Per-step slot of the observables: 6 sums per grid point (Ekin, J, Ex, N,
// Eion, EH), reduced by kspace_obs_reduce_kernel.
__host__ __device__ constexpr int kspace_obs_stride(int ng) { return 6 * ng; }

struct KArgs {
  ApplyArgs a;          // mode, field, step, tape and batch strides; u, w, ... of a plain launch
  int ng;
  int n;                // transform length (plain launch)
  int nchunk;           // blocks of bands per grid point
  const zd* ktab;       // plain launch
  const zd* tw[4];      // twiddle tables of GroupFFT<16 << i>
  const zd* om[4];      // exp(-i pi q/N), q < N = 16 << i
  zd* hm;               // plain launch; trajectory t of a uniform batch at + t hstride, t nstride
  double* nx;
  size_t hstride, nstride;
  const int2* amap;     // batch: (trajectory, entry) of kmat_kernel's and kapply_kernel's workgroups
  const int2* bmap;
};

// Lane twiddles from an LDS copy of the table instead of registers.  Its
// entries (lane-major in the table: 8 consecutive ones per lane, which as LDS
// reads would meet in two banks) are transposed to lanes fastest.
template <int N>
__host__ __device__ constexpr bool kspace_lds_twiddles() {
  return N >= 32;
}
template <int N>
__device__ __forceinline__ int kspace_tw_slot(int i) {
  using F = GroupFFT<N>;
  if (i < N) return (i % F::R) * F::L + i / F::R;
  const int r = i - N;
  if constexpr (N == 128) return N + (r % 4) * 4 + r / 4;
  else return N + (r % F::R) * F::L + r / F::R;
}

__device__ __forceinline__ void zfma(zd& s, zd a, zd b) {  // s += a b
  s.x = fma(a.x, b.x, s.x);
  s.x = fma(-a.y, b.y, s.x);
  s.y = fma(a.x, b.y, s.y);
  s.y = fma(a.y, b.x, s.y);
}
__device__ __forceinline__ void zfmac(zd& s, zd a, zd b) {  // s += a conj(b)
  s.x = fma(a.x, b.x, s.x);
  s.x = fma(a.y, b.y, s.x);
  s.y = fma(a.y, b.x, s.y);
  s.y = fma(-a.x, b.y, s.y);
}

// Between the lane domain and the transform groups, through the wave's tile.
template <int N>
__device__ __forceinline__ void to_groups(zd (&v)[KGeo<N>::R], zd* tile, int kl, int xs, int gw,
                                          int l) {
  using K = KGeo<N>;
  static_for<0, K::R>([&](auto rc) {
    constexpr int r = decltype(rc)::value, kk = r / K::XR, xr = r % K::XR;
    tile[(xs * K::XR + xr) * K::P + kl + 64 * kk] = v[r];
  });
  wave_sync();
  static_for<0, K::R>([&](auto mc) {
    constexpr int m = decltype(mc)::value;
    v[m] = tile[gw * K::P + K::L * m + l];
  });
  wave_sync();
}
template <int N>
__device__ __forceinline__ void to_lanes(zd (&v)[KGeo<N>::R], zd* tile, int kl, int xs, int gw,
                                         int l) {
  using K = KGeo<N>;
  static_for<0, K::R>([&](auto mc) {
    constexpr int m = decltype(mc)::value;
    tile[gw * K::P + K::L * m + l] = v[m];
  });
  wave_sync();
  static_for<0, K::R>([&](auto rc) {
    constexpr int r = decltype(rc)::value, kk = r / K::XR, xr = r % K::XR;
    v[r] = tile[(xs * K::XR + xr) * K::P + kl + 64 * kk];
  });
  wave_sync();
}

// ---------------------------------------------------------------------------
// the matrices, then their product with the columns
// ---------------------------------------------------------------------------
// H_k(x,x') without its diagonal potential is Hermitian, so kmat_kernel makes
// the blocks of x' up to the one that holds x only, one wave per (x, block),
// and kapply_kernel reads an element above them as the conjugate of its
// mirror.  Elements: hm[(x NG1 + x') N + k], NG1 = NG + 1 (the odd pitch
// spreads a column's reads over the memory channels).
__host__ __device__ constexpr size_t kmat_elems(int ng, int n) { return (size_t)ng * (ng + 1) * n; }

// Waves' tasks of one trajectory: block row X (GPW rows) has X + 1 blocks.
__host__ __device__ constexpr int kmat_tasks(int ng, int gpw) {
  return gpw * ((ng / gpw) * (ng / gpw + 1) / 2);
}

// Doubles after the matrices: density n(x), then Ekin, J, Ex of each task.
__host__ __device__ constexpr size_t kmat_extra(int ng, int gpw) {
  return (size_t)ng + 3 * kmat_tasks(ng, gpw);
}

template <int N>
__host__ __device__ constexpr size_t kmat_lds(int nw, int ng) {
  return ((size_t)nw * KGeo<N>::TILE + N + GroupFFT<N>::TWN + ng) * sizeof(zd) +
         (size_t)ng * sizeof(double);
}

// Fields of a launch from the step counter (or its arguments).
__device__ __forceinline__ void kspace_fields(const ApplyArgs& a, const KTraj& t, double& Akin,
                                              double& Aobs, int& slot) {
  slot = a.obs_slot;
  Akin = a.A;
  Aobs = a.Aobs;
  if (a.step_base) {
    const int step = *a.step_base + a.jstep;
    const double At = gload(t.Aarr + step), Aav = gload(t.Aavearr + step);
    if (a.mode == M_S1) {
      Akin = 2.0 * Aav - At;  // A(it-1) as in RT_RK4_ubk
      Aobs = step > 0 ? gload(t.Aarr + step - 1) : 0.0;
      slot = step;
    } else if (a.mode == M_S2 || a.mode == M_S3) {
      Akin = Aav;
    } else if (a.mode == M_S4) {
      Akin = At;
    } else {  // M_OBS after step 'step'
      Akin = At;
      Aobs = At;
      slot = step + 1;
    }
  }
}

// DEPTH: bands whose loads are in flight together.
template <int N, bool OBS, int DEPTH>
__device__ __forceinline__ void kmat_task(const KArgs& ka, const KTraj& t, int task, int ntask,
                                          const zd* twt, const zd* omt, zd* smem) {
  using K = KGeo<N>;
  using F = GroupFFT<N>;
  constexpr int R = K::R, L = K::L, KK = K::KK, XR = K::XR, GPW = K::GPW;
  const ApplyArgs& a = ka.a;
  const int NG = ka.ng, nb = a.nb, nbocc = a.nbocc;
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
  const bool live = task < ntask;  // a wave past the last task only fills the tables

  // (x, block b): block row X from its triangular number
  const int q0 = (live ? task : 0) / GPW;
  int X = (int)((__fsqrt_rn(8.0f * (float)q0 + 1.0f) - 1.0f) * 0.5f);
  while (X * (X + 1) / 2 > q0) --X;
  while ((X + 1) * (X + 2) / 2 <= q0) ++X;
  const int b = __builtin_amdgcn_readfirstlane(q0 - X * (X + 1) / 2);
  const int x = __builtin_amdgcn_readfirstlane(X * GPW + (live ? task : 0) % GPW);
  const int x0 = b * GPW;

  const unsigned xstride = (unsigned)(nb * N);
  const unsigned uoff = (unsigned)((xs * XR * xstride + kl) * sizeof(zd));
  const unsigned coff = (unsigned)(kl * sizeof(zd));
  const zd* up = t.u + (size_t)x0 * xstride;
  const zd* uc = t.u + (size_t)x * xstride;
  zd buf[DEPTH][R], own[DEPTH][KK];
  auto fetch = [&](auto dc, int j) {
    constexpr int d = decltype(dc)::value;
    static_for<0, R>([&](auto rc) {
      constexpr int r = decltype(rc)::value, kk = r / XR, xr = r % XR;
      buf[d][r] = gload_at(up + xr * xstride + j * N + 64 * kk, uoff);
    });
    static_for<0, KK>([&](auto kc) {
      constexpr int kk = decltype(kc)::value;
      own[d][kk] = gload_at(uc + j * N + 64 * kk, coff);
    });
  };
  // (past the last band that one again: a guard would keep the buffers' old
  // values alive)
  static_for<0, DEPTH>([&](auto dc) {
    constexpr int d = decltype(dc)::value;
    fetch(dc, d < nbocc ? d : nbocc - 1);
  });
  for (int i = tid; i < N; i += nth) sOm[i] = gload(omt + i);
  for (int i = tid; i < F::TWN; i += nth) sTw[kspace_tw_slot<N>(i)] = gload(twt + i);
  for (int i = tid; i < NG; i += nth) {
    sK1[i] = gload(reinterpret_cast<const zd*>(t.kc + 2 * NG) + i);
    sK2[i] = gload(t.kc + NG + i);
  }
  auto tw1 = [&](int g) { return sTw[g * L + l]; };
  auto tw2 = [&](int i) { return N == 128 ? sTw[N + 4 * i + (l & 3)] : sTw[N + i * L + l]; };
  F fft;
  auto fwd = [&](zd(&v)[R]) {
    if constexpr (N == 128) fft.fwd_t(v, T, l, tw1, tw2);
    else fft.fwd_t(v, T, l, tw1);
  };
  auto inv = [&](zd(&v)[R]) { fft.inv_t(v, T, l, tw1, tw2); };
  double Akin, Aobs;
  int slot;
  kspace_fields(a, t, Akin, Aobs, slot);
  double kxv[KK];
  static_for<0, KK>([&](auto kc) {
    constexpr int kk = decltype(kc)::value;
    kxv[kk] = gload(t.kx + kl + 64 * kk);
  });
  lds_barrier();  // tables in LDS; no further barrier
  if (!live) return;

  // ---- density matrix rho_k(x,x'), lanes over k ----
  zd rho[R];
  static_for<0, R>([&](auto rc) { rho[decltype(rc)::value] = mk(0.0, 0.0); });
  for (int j0 = 0; j0 < nbocc; j0 += DEPTH)
    static_for<0, DEPTH>([&](auto dc) {
      constexpr int d = decltype(dc)::value;
      if (j0 + d < nbocc) {
        static_for<0, R>([&](auto rc) {
          constexpr int r = decltype(rc)::value;
          zfmac(rho[r], own[d][r / XR], buf[d][r]);
        });
        if (j0 + d + DEPTH < nbocc) fetch(dc, j0 + d + DEPTH);
      }
    });
  double ek = 0.0, jc = 0.0, ex = 0.0;
  double* nx = t.nx;
  if (b == X) {
    // the element (x,x): density at x and the diagonal terms of Ekin and J
    double n = 0.0;
    static_for<0, R>([&](auto rc) {
      constexpr int r = decltype(rc)::value, kk = r / XR, xr = r % XR;
      if (x0 + xs * XR + xr == x) {
        const double kA = kxv[kk] + Aobs, p = rho[r].x;
        n += p;
        if (OBS) {
          ek = fma(0.5 * kA * kA, p, ek);
          jc = fma(kA, p, jc);
        }
      }
    });
    n = wave_sum(n);
    if (lane == 0) gstore(nx + x, n);
  }
  if (OBS) {
    // sum_x' T_k(x-x') conj(rho_k(x,x')): kinetic energy and current; blocks
    // below the diagonal one stand for their mirrors too
    const double wt = b == X ? 1.0 : 2.0;
    static_for<0, XR>([&](auto rc) {
      constexpr int xr = decltype(rc)::value;
      const int y = (x - (x0 + xs * XR + xr)) & (NG - 1);
      const double k2 = wt * sK2[y];
      const zd k1 = zscal(sK1[y], wt);
      static_for<0, KK>([&](auto kc) {
        constexpr int kk = decltype(kc)::value;
        const zd p = rho[kk * XR + xr];
        const double e1 = k1.x * p.x + k1.y * p.y;
        jc += e1;
        ek = fma(kxv[kk] + Aobs, e1, ek);
        ek = fma(k2, p.x, ek);
      });
    });
  }

  // ---- Toeplitz product over the k-mesh: circulant + skew-circulant ----
  to_groups<N>(rho, tile, kl, xs, gw, l);
  const unsigned toff = (unsigned)((((x - x0 - gw) & (NG - 1)) * 2 * N + l) * sizeof(zd));
  zd kv[R];
  static_for<0, 2>([&](auto ec) {
    constexpr int eo = decltype(ec)::value;
    zd tb[R];
    static_for<0, R>([&](auto jc_) {
      constexpr int j = decltype(jc_)::value;
      tb[j] = gload_at(t.ktab + (eo * R + j) * L, toff);
    });
    zd v[R];
    static_for<0, R>([&](auto mc) {
      constexpr int m = decltype(mc)::value;
      v[m] = eo == 0 ? rho[m] : zmul(rho[m], sOm[L * m + l]);
    });
    fwd(v);
    if (OBS) {
      // sum_k K_k conj(rho_k) by Parseval
      static_for<0, R>([&](auto jc_) {
        constexpr int j = decltype(jc_)::value;
        ex = fma(tb[j].x, zabs2(v[j]), ex);
      });
    }
    static_for<0, R>([&](auto jc_) {
      constexpr int j = decltype(jc_)::value;
      v[j] = zmul(v[j], tb[j]);
    });
    inv(v);
    static_for<0, R>([&](auto mc) {
      constexpr int m = decltype(mc)::value;
      kv[m] = eo == 0 ? v[m] : zadd(kv[m], zmulc(v[m], sOm[L * m + l]));
    });
    // the two products one after the other: overlapped by the scheduler they
    // do not fit the registers
    __builtin_amdgcn_sched_barrier(0);
  });
  to_lanes<N>(kv, tile, kl, xs, gw, l);
  // ---- kinetic elements; out ----
  static_for<0, XR>([&](auto rc) {
    constexpr int xr = decltype(rc)::value;
    const int xp = x0 + xs * XR + xr, y = (x - xp) & (NG - 1);
    const double k2 = sK2[y];
    const zd k1 = sK1[y];
    static_for<0, KK>([&](auto kc) {
      constexpr int kk = decltype(kc)::value;
      const double kA = kxv[kk] + Akin;
      const zd q = kv[kk * XR + xr];
      gstore(t.hm + ((size_t)x * (NG + 1) + xp) * N + kl + 64 * kk,
             mk(q.x + fma(kA, k1.x, k2), fma(kA, k1.y, q.y)));
    });
  });
  if (OBS) {
    ek = wave_sum(ek);
    jc = wave_sum(jc);
    ex = wave_sum(ex) * (b == X ? 1.0 : 2.0);
    if (lane == 0) {
      double* p = nx + NG + 3 * task;
      gstore(p, ek);
      gstore(p + 1, jc);
      gstore(p + 2, ex);
    }
  }
}

// Operands of the workgroup's trajectory; false: padding entry of a batch's
// list.  item: entry of the trajectory's work.
__device__ __forceinline__ bool kspace_traj(const KArgs& ka, const int2* map, KTraj& t, int& item,
                                            int& n) {
  const ApplyArgs& a = ka.a;
  item = blockIdx.x;
  n = ka.n;
  t.occ = a.occ;
  t.kx = a.kx;
  t.vion = a.vion;
  t.kc = a.kc;
  t.ktab = ka.ktab;
  t.Aarr = a.Aarr;
  t.Aavearr = a.Aavearr;
  t.u = a.u;
  t.w = a.w;
  t.out = a.out;
  t.u0 = a.u0;
  t.ksum = a.ksum;
  t.unext = a.unext;
  t.tape0 = nullptr;
  t.obs = a.obs;
  t.hm = ka.hm;
  t.nx = ka.nx;
  if (a.td) {
    const int2 rm = map[blockIdx.x];
    if (rm.x < 0) return false;
    const TrajDesc& d = a.td[rm.x];
    item = rm.y;
    n = d.n;
    t.occ = d.occ;
    t.kx = d.kx;
    t.vion = d.vion;
    t.kc = d.kc;
    t.ktab = d.ktab;
    t.Aarr = d.A;
    t.Aavearr = d.Aave;
    t.u0 = d.u0;
    t.ksum = d.ksum;
    t.obs = d.obs;
    t.hm = d.hm;
    t.nx = d.nx;
    switch (a.mode) {
      case M_S1: t.u = d.u0; t.unext = d.sa; break;
      case M_S2: t.u = d.sa; t.unext = d.sb; break;
      case M_S3: t.u = d.sb; t.unext = d.sa; break;
      case M_S4: t.u = d.sa; t.unext = nullptr; break;
      default: t.u = d.u0; t.unext = nullptr; break;
    }
    t.w = t.u;
  }
  // taped forward: the stage states live in the tape slots of this step
  if (a.tape && a.step_base) {
    const int tstep = *a.step_base + a.jstep;
    zd* tp = a.tape + (size_t)(tstep % a.tape_seg) * 4 * a.nstate;
    switch (a.mode) {
      case M_S1: t.tape0 = tp; t.unext = tp + a.nstate; break;
      case M_S2: t.u = t.w = tp + a.nstate; t.unext = tp + 2 * a.nstate; break;
      case M_S3: t.u = t.w = tp + 2 * a.nstate; t.unext = tp + 3 * a.nstate; break;
      case M_S4: t.u = t.w = tp + 3 * a.nstate; break;
      default: break;
    }
  }
  const int tr = blockIdx.y;  // trajectory of a uniform batch (0 otherwise)
  if (tr > 0) {
    const size_t so = (size_t)tr * a.tstride;
    t.Aarr += (size_t)tr * a.fstride;
    t.Aavearr += (size_t)tr * a.fstride;
    t.u += so;
    t.w += so;
    if (t.u0) t.u0 += so;
    if (t.ksum) t.ksum += so;
    if (t.unext) t.unext += so;
    if (t.out) t.out += so;
    if (t.tape0) t.tape0 += so;
    if (t.obs) t.obs += (size_t)tr * a.ostride;
    t.hm += (size_t)tr * ka.hstride;
    t.nx += (size_t)tr * ka.nstride;
  }
  return true;
}

// N = 0: the transform length of each workgroup follows its trajectory.
// DEEP: four bands in flight and two waves per SIMD, for grids that do not
// fill the chip with more; else two bands and three waves.
template <int N, bool OBS, bool DEEP>
__global__ void __launch_bounds__(256, DEEP ? 2 : 3) kmat_kernel(KArgs ka) {
  extern __shared__ zd smem[];
  KTraj t;
  int item, n;
  if (!kspace_traj(ka, ka.amap, t, item, n)) return;
  const int task = item * (int)(blockDim.x >> 6) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  auto go = [&](auto nc) {
    constexpr int M = decltype(nc)::value, c = M == 16 ? 0 : M == 32 ? 1 : M == 64 ? 2 : 3;
    kmat_task<M, OBS, DEEP ? 4 : 2>(ka, t, task, kmat_tasks(ka.ng, KGeo<M>::GPW), ka.tw[c], ka.om[c], smem);
  };
  if constexpr (N != 0) {
    go(std::integral_constant<int, N>{});
  } else {
    switch (n) {
      case 16: go(std::integral_constant<int, 16>{}); break;
      case 32: go(std::integral_constant<int, 32>{}); break;
      case 64: go(std::integral_constant<int, 64>{}); break;
      default: go(std::integral_constant<int, 128>{}); break;
    }
  }
}

// out = H w and the stage update for XT grid points x, NBT bands and up to 64
// k-points per workgroup: its waves share out the x', lanes over k (for N < 64
// the lanes' upper bits over x' too), each element of the matrices is read
// once per workgroup and multiplied into every band.

__host__ __device__ constexpr int kapply_round(int nbt) { return nbt < 4 ? nbt : 4; }
__host__ __device__ constexpr size_t kapply_lds(int nw, int nbt, int xt) {
  return (size_t)nw * xt * kapply_round(nbt) * 64 * sizeof(zd) + 16 * sizeof(double);
}

template <int NBT, int XT>
__global__ void __launch_bounds__(512, 2) kapply_kernel(KArgs ka) {
  constexpr int BR = kapply_round(NBT);
  // x' in flight: as many as the registers hold where few workgroups run
  constexpr int DEPTH = XT > 1 ? 2 : NBT <= 4 ? 8 : 4;
  extern __shared__ zd smem[];
  const ApplyArgs& a = ka.a;
  KTraj t;
  int item, N;
  if (!kspace_traj(ka, ka.bmap, t, item, N)) return;
  const int NG = ka.ng, nbw = a.nbw, mode = a.mode;
  const int tid = threadIdx.x, lane = tid & 63, nth = blockDim.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int W = nth >> 6;
  const int KL = N < 64 ? N : 64, XS = 64 / KL;
  // item: k block fastest, then bands, then the x tile
  const int kb = N > 64 ? N / 64 : 1;
  const int kc = item % kb, ch = (item / kb) % ka.nchunk, x0 = item / (kb * ka.nchunk) * XT;
  const int i0 = ch * NBT, ni = nbw - i0 < NBT ? nbw - i0 : NBT;
  const int k = 64 * kc + (lane & (KL - 1)), xs = lane / KL;
  double* sVh = reinterpret_cast<double*>(smem + (size_t)W * XT * BR * 64);
  const unsigned wstride = (unsigned)(nbw * N);
  const int bshift = N == 128 ? 2 : N == 64 ? 3 : 4;  // x' per block of kmat_kernel: 1 << bshift

  // ---- first loads in flight: the matrices and columns of DEPTH x' ----
  zd hb[DEPTH][XT], wb[DEPTH][NBT];
  auto load = [&](auto dc, int xp) {
    constexpr int d = decltype(dc)::value;
    static_for<0, XT>([&](auto xc) {
      constexpr int i = decltype(xc)::value;
      const int x = x0 + i;
      const bool low = (xp >> bshift) <= (x >> bshift);
      const unsigned e = (unsigned)((low ? x : xp) * (NG + 1) + (low ? xp : x)) * N + k;
      hb[d][i] = gload_at(t.hm, e * (unsigned)sizeof(zd));
    });
    const unsigned wo = ((unsigned)xp * wstride + k) * (unsigned)sizeof(zd);
    static_for<0, NBT>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      wb[d][i] = gload_at(t.w + (i0 + (i < ni ? i : ni - 1)) * N, wo);
    });
  };
  const int per = mode == M_OBS ? 0 : NG / (W * XS);  // x' per lane
  auto xpof = [&](int it) { return ((it < per ? it : per - 1) * W + wave) * XS + xs; };
  if (per > 0) static_for<0, DEPTH>([&](auto dc) { load(dc, xpof(decltype(dc)::value)); });
  // operands of the thread's first (x, band, k), used at the end
  const int q0 = tid & (KL - 1), j0 = (tid / KL) % BR, xi0 = tid / (KL * BR);
  const bool first = per > 0 && xi0 < XT && j0 < ni;
  const size_t o0 = (size_t)(x0 + xi0) * wstride + (size_t)(i0 + j0) * N + 64 * kc + q0;
  const bool rk = mode >= M_S2 && mode <= M_S4;
  zd wv0 = mk(0.0, 0.0), u00 = wv0, ks0 = wv0;
  double kx0 = 0.0, vi0 = 0.0;
  if (first) {
    wv0 = gload(t.w + o0);
    kx0 = gload(t.kx + 64 * kc + q0);
    vi0 = gload(t.vion + x0 + xi0);
    if (rk) {
      u00 = gload(t.u0 + o0);
      ks0 = gload(t.ksum + o0);
    }
  }
  // Hartree potential at the XT points: wave i sums for x0 + i
  for (int i = wave; i < XT; i += W) {
    double s = 0.0;
    for (int xp = lane; xp < NG; xp += 64)
      s = fma(gload(t.kc + ((x0 + i - xp) & (NG - 1))), gload(t.nx + xp), s);
    s = wave_sum(s);
    if (lane == 0) sVh[i] = t.occ * s;
  }
  double Akin, Aobs;
  int slot;
  kspace_fields(a, t, Akin, Aobs, slot);

  // ---- sum_x' H_k(x,x') w_ki(x') ----
  zd acc[XT][NBT];
  static_for<0, XT>([&](auto xc) {
    static_for<0, NBT>(
        [&](auto ic) { acc[decltype(xc)::value][decltype(ic)::value] = mk(0.0, 0.0); });
  });
  for (int it = 0; it < per; it += DEPTH)
    static_for<0, DEPTH>([&](auto dc) {
      constexpr int d = decltype(dc)::value;
      if (it + d < per) {
        const int xp = xpof(it + d);
        static_for<0, XT>([&](auto xc) {
          constexpr int i = decltype(xc)::value;
          const bool low = (xp >> bshift) <= ((x0 + i) >> bshift);
          const zd h = mk(hb[d][i].x, low ? hb[d][i].y : -hb[d][i].y);
          static_for<0, NBT>([&](auto ic) {
            constexpr int j = decltype(ic)::value;
            zfma(acc[i][j], h, wb[d][j]);
          });
        });
        if (it + d + DEPTH < per) load(dc, xpof(it + d + DEPTH));
      }
    });

  const bool want_obs = (mode == M_S1 || mode == M_OBS) && t.obs != nullptr && ch == 0 && kc == 0;
  if (mode == M_OBS) lds_barrier();
  else
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
        // thread: (x, band, k) of the round
        for (int q = tid; q < XT * BR * KL; q += nth) {
          const int kq = q & (KL - 1), j = (q / KL) % BR, i = q / (KL * BR);
          if (r0 + j >= ni) continue;
          const int x = x0 + i;
          const size_t o = (size_t)x * wstride + (size_t)(i0 + r0 + j) * N + 64 * kc + kq;
          zd wv = wv0, u0v = u00, ksv = ks0;
          double kA = kx0, vi = vi0;
          if (r0 > 0 || q != tid) {
            wv = gload(t.w + o);
            kA = gload(t.kx + 64 * kc + kq);
            vi = gload(t.vion + x);
            if (rk) {
              u0v = gload(t.u0 + o);
              ksv = gload(t.ksum + o);
            }
          }
          kA += Akin;
          zd h = mk(0.0, 0.0);
          for (int w2 = 0; w2 < W; ++w2)
            for (int s2 = 0; s2 < XS; ++s2)
              h = zadd(h, smem[((w2 * XT + i) * BR + j) * 64 + s2 * KL + kq]);
          const double d = fma(0.5 * kA, kA, sVh[i] + vi);
          h.x = fma(d, wv.x, h.x);
          h.y = fma(d, wv.y, h.y);
          const zd kk = mk(h.y, -h.x);  // -i H w
          const double hdt = 0.5 * a.dt;
          if (mode == M_HPSI) {
            gstore(t.out + o, h);
          } else if (mode == M_S1) {
            if (t.tape0) gstore(t.tape0 + o, wv);
            gstore(t.ksum + o, kk);
            gstore(t.unext + o, mk(wv.x + hdt * kk.x, wv.y + hdt * kk.y));
          } else if (mode == M_S4) {
            gstore(t.u0 + o, mk(u0v.x + (ksv.x + kk.x) * a.dt / 6.0,
                                u0v.y + (ksv.y + kk.y) * a.dt / 6.0));
          } else {
            gstore(t.ksum + o, mk(ksv.x + 2.0 * kk.x, ksv.y + 2.0 * kk.y));
            const double c = mode == M_S2 ? hdt : a.dt;
            gstore(t.unext + o, mk(u0v.x + c * kk.x, u0v.y + c * kk.y));
          }
        }
      }
    });
  // ---- observables of the points: their tasks' sums and the density terms ----
  if (want_obs && tid < XT) {
    const int x = x0 + tid, gpw = 1 << bshift, X = x >> bshift;
    const double* p = t.nx + NG + 3 * (size_t)(gpw * (X * (X + 1) / 2) + x - X * gpw);
    double s1 = 0.0, s2 = 0.0, s3 = 0.0;
    for (int b = 0; b <= X; ++b, p += 3 * gpw) {
      s1 += gload(p);
      s2 += gload(p + 1);
      s3 += gload(p + 2);
    }
    const double rho = t.occ * gload(t.nx + x), vi = gload(t.vion + x);
    double* o = t.obs + (size_t)slot * kspace_obs_stride(NG) + 6 * x;
    gstore(o + 0, t.occ * s1 * a.dv);
    gstore(o + 1, t.occ * s2);
    gstore(o + 2, t.occ * s3 * a.dv);
    gstore(o + 3, rho * a.dv);
    gstore(o + 4, vi * rho * a.dv);
    gstore(o + 5, 0.5 * sVh[tid] * rho * a.dv);
  }
}

// ---------------------------------------------------------------------------
// tables
// ---------------------------------------------------------------------------
struct CompZ {
  CompSum re, im;
  __device__ __forceinline__ void add(double x, double y) {
    re.add(x);
    im.add(y);
  }
  __device__ __forceinline__ zd value() const { return mk(re.value(), im.value()); }
};

// tsp[d NG + y] = T_{d-NK+1}(y) = scale sum_G vq[d NG + G] exp(2 pi i G y/NG),
// one thread per value, compensated sums (once per context).
__global__ void kspace_space_kernel(const double* vq, int nd, int ng, double scale, zd* tsp) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nd * ng) return;
  const int d = i / ng, y = i - d * ng;
  CompZ s;
  for (int g = 0; g < ng; ++g) {
    double sn, cs;
    sincospi(2.0 * (double)((g * y) & (ng - 1)) / (double)ng, &sn, &cs);
    const double v = vq[(size_t)d * ng + g];
    s.add(v * cs, v * sn);
  }
  tsp[i] = zscal(s.value(), scale);
}

// Spectra of the circulant (eo = 0) and skew-circulant (eo = 1) parts, over N,
// in the G layout of GroupFFT<N>: one thread per (y, eo, theta),
//   1/N sum_{d<N} (T_d +- T_{d-N})/2 exp(-i pi d (2 theta + eo)/N).
template <int N>
__global__ void kspace_spectrum_kernel(const zd* tsp, int nk, int ng, zd* ktab) {
  using F = GroupFFT<N>;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= ng * 2 * N) return;
  const int l = i % F::L, j = (i / F::L) % F::R, eo = (i / N) & 1, y = i / (2 * N);
  const int th = F::gindex(l, j);
  CompZ s;
  for (int d = 0; d < N; ++d) {
    zd c = mk(0.0, 0.0);
    if (d < nk) c = tsp[(size_t)(d + nk - 1) * ng + y];
    if (N - d < nk) {  // T_{d-N}
      const zd m = tsp[(size_t)(d - N + nk - 1) * ng + y];
      c = eo ? zsub(c, m) : zadd(c, m);
    }
    double sn, cs;
    sincospi((double)((d * (2 * th + eo)) % (2 * N)) / (double)N, &sn, &cs);
    s.add(c.x * cs + c.y * sn, c.y * cs - c.x * sn);
  }
  ktab[i] = zscal(s.value(), 0.5 / (double)N);
}

// exp(-i pi q/N), q < N
__global__ void kspace_om_kernel(zd* om, int n) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n) return;
  double sn, cs;
  sincospi((double)q / (double)n, &sn, &cs);
  om[q] = mk(cs, -sn);
}

// ---------------------------------------------------------------------------
// layout: (NG,NB,NK) with x fastest <-> U[x][b][k] with k padded to n
// ---------------------------------------------------------------------------
struct KLayoutArgs {
  const zd* src;
  zd* dst;
  int ng, nb, nk, n;
  int ld;                   // columns per k-point of the (NG,.,NK) side (0: nb)
  size_t sstride, dstride;  // per trajectory
  // batch: offsets and k-meshes of the trajectories instead
  const TrajDesc* td;
  const size_t* roff;       // of the (NG,NB,NK) states
  const size_t* koff;       // of the padded ones
  int to_k;
};

// 16 x 16 tiles through LDS, so that both sides move 256-byte runs.  The grid's x is
// trajectory * nb + band, the only count without a small bound (a grid's y and z
// end at 65535, x at 2^32 threads), y the k and z the x tile.
__global__ void __launch_bounds__(256) kspace_layout_kernel(KLayoutArgs a) {
  __shared__ zd s[16][17];
  const int tr = blockIdx.x / a.nb, b = blockIdx.x - tr * a.nb, ld = a.ld ? a.ld : a.nb;
  int nk = a.nk, n = a.n;
  size_t ro = a.to_k ? tr * a.sstride : tr * a.dstride;
  size_t ko = a.to_k ? tr * a.dstride : tr * a.sstride;
  if (a.td) {
    nk = a.td[tr].nk;
    n = a.td[tr].n;
    ro = a.roff[tr];
    ko = a.koff[tr];
  }
  const int x0 = blockIdx.z * 16, k0 = blockIdx.y * 16;
  if (k0 >= n) return;
  const int p = threadIdx.x & 15, q = threadIdx.x >> 4;
  if (a.to_k) {
    const int k = k0 + q;
    s[q][p] = k < nk ? a.src[ro + (size_t)(x0 + p) + (size_t)a.ng * (b + (size_t)ld * k)]
                     : mk(0.0, 0.0);
    __syncthreads();
    a.dst[ko + ((size_t)(x0 + q) * a.nb + b) * n + k0 + p] = s[p][q];
  } else {
    s[q][p] = a.src[ko + ((size_t)(x0 + q) * a.nb + b) * n + k0 + p];
    __syncthreads();
    const int k = k0 + q;
    if (k < nk) a.dst[ro + (size_t)(x0 + p) + (size_t)a.ng * (b + (size_t)ld * k)] = s[p][q];
  }
}

// ---------------------------------------------------------------------------
// observables
// ---------------------------------------------------------------------------
// (Etot, N, J, Ekin, Eion, EH, Ex) of each slot (src/Functions.f90:74-91,
// :289-318) from its 6 NG sums: one wave per slot, a compensated sum per lane
// over x = lane, lane + 64, ..., then the lanes' sums added with compensation
// in a fixed order.  td: batch, slot s of trajectory t = wave / nslots.
__global__ void __launch_bounds__(256) kspace_obs_reduce_kernel(const double* obs,
                                                                const TrajDesc* td, int ng,
                                                                int nslots, int nw, double dv,
                                                                double vcell, size_t tstride,
                                                                double* out) {
  const int i = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (i >= nw) return;
  const int t = i / nslots, s = i - t * nslots;
  const double* p = (td ? td[t].obs : obs + (size_t)t * tstride) + (size_t)s * kspace_obs_stride(ng);
  CompSum c[6];
  for (int x = lane; x < ng; x += 64)
    for (int m = 0; m < 6; ++m) c[m].add(p[6 * x + m]);
  comp_wave_sum(c, 64);
  if (lane == 0) {
    CompSum et;
    et.add(c[0].s);
    et.add(c[4].s);
    et.add(c[5].s);
    et.add(0.5 * c[2].s);
    et.add(c[0].c + c[4].c + c[5].c);
    et.add(0.5 * c[2].c);
    double* o = out + (size_t)7 * i;
    o[0] = et.value();
    o[1] = c[3].value();
    o[2] = -(c[1].value() * dv / vcell);
    o[3] = c[0].value();
    o[4] = c[4].value();
    o[5] = c[5].value();
    o[6] = 0.5 * c[2].value();
  }
}

}  // namespace tdhf
