// tdhf_gs_impl.h -- host side of the ground-state iteration (included by
// tdhf.hip after the context helpers).  Mirrors GS_calculation
// (src/GS_calculation.f90:26-57): per iteration Gram_Schmidt, KS_ubk2_SVD,
// Gram_Schmidt, Subspace_diag, then the total energy at A=0.
#pragma once

namespace tdhf {

void gs_free(GsWork& g) {
  if (g.W) (void)hipFree(g.W);
  if (g.HW) (void)hipFree(g.HW);
  if (g.KW) (void)hipFree(g.KW);
  if (g.KH) (void)hipFree(g.KH);
  if (g.eps) (void)hipFree(g.eps);
  if (g.nonconv) (void)hipFree(g.nonconv);
  g.W = g.HW = g.KW = g.KH = nullptr;
  g.eps = nullptr;
  g.nonconv = nullptr;
  g.ncg = 0;
}

}  // namespace tdhf

namespace {

int gs_alloc(tdhf_ctx* c, int ncg) {
  if (c->gs.ncg >= ncg) return 0;
  tdhf::gs_free(c->gs);
  const size_t n = nstate(c) * (size_t)ncg;
  CHKRET(dalloc(c, &c->gs.W, n));
  CHKRET(dalloc(c, &c->gs.HW, n));
  if (c->kpath) {
    CHKRET(dalloc(c, &c->gs.KW, kcount(c) * (size_t)ncg));
    CHKRET(dalloc(c, &c->gs.KH, kcount(c) * (size_t)ncg));
  }
  CHKRET(dalloc(c, &c->gs.eps, (size_t)c->nb * c->nk * 2));
  CHKRET(dalloc(c, &c->gs.nonconv, 1));
  c->gs.ncg = ncg;
  return 0;
}

// Clears the eigensolver's non-convergence flag (before a GS run).
int gs_flag_clear(tdhf_ctx* c) {
  HIPCHK(c, hipMemsetAsync(c->gs.nonconv, 0, sizeof(int), c->stream));
  return 0;
}

// Fails if a Rayleigh-Ritz eigensolve since the last clear did not converge.
int gs_flag_check(tdhf_ctx* c) {
  int f = 0;
  HIPCHK(c, hipMemcpyAsync(&f, c->gs.nonconv, sizeof f, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  if (f)
    return fail(c, TDHF_ENUMERIC,
                "subspace eigensolver (cyclic Jacobi) did not converge in 100 sweeps at k-point %d",
                f - 1);
  return 0;
}

// Gram-Schmidt of m columns per k-point, npass passes, in place and to copy
// (ldc columns per k-point).  One wave per column, up to sixteen.
int launch_orth(tdhf_ctx* c, zd* w, int m, int npass, zd* copy, int ldc) {
  const size_t lds = tdhf::orth_lds(c->ng, m);
  if (lds > 160 * 1024) {  // more bands than LDS holds (one pass only)
    if (npass != 1 || copy) return fail(c, TDHF_EINVAL, "%d columns do not fit LDS", m);
    hipLaunchKernelGGL(tdhf::gram_schmidt_kernel, dim3(c->nk), dim3(c->ng), 0, c->stream, w, c->ng,
                       m, c->vcell);
    HIPCHK(c, hipGetLastError());
    return 0;
  }
  if (lds > 64 * 1024)
    HIPCHK(c, hipFuncSetAttribute((const void*)tdhf::orth_kernel,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
  hipLaunchKernelGGL(tdhf::orth_kernel, dim3(c->nk), dim3(64 * std::min(m, 16)), lds, c->stream, w,
                     c->ng, m, c->dv, npass, copy, ldc);
  HIPCHK(c, hipGetLastError());
  return 0;
}

int launch_rr(tdhf_ctx* c, const zd* W, const zd* HW, int m, zd* uout) {
  const bool wl = tdhf::rr_lds(c->ng, m, true) <= 160 * 1024;
  const size_t lds = tdhf::rr_lds(c->ng, m, wl);
  const void* fn =
      wl ? (const void*)tdhf::rr_kernel<true> : (const void*)tdhf::rr_kernel<false>;
  if (lds > 64 * 1024)
    HIPCHK(c, hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
  if (wl)
    hipLaunchKernelGGL(tdhf::rr_kernel<true>, dim3(c->nk), dim3(256), lds, c->stream, W, HW, c->ng,
                       c->nb, m, c->dv, uout, c->gs.nonconv);
  else
    hipLaunchKernelGGL(tdhf::rr_kernel<false>, dim3(c->nk), dim3(256), lds, c->stream, W, HW,
                       c->ng, c->nb, m, c->dv, uout, c->gs.nonconv);
  HIPCHK(c, hipGetLastError());
  return 0;
}

// H of the orbitals u (NG,NB,NK) at A = 0, for the gs_product calls after it:
// on the density-matrix path its matrices are made once.
int gs_hamiltonian(tdhf_ctx* c, const zd* u) {
  if (!c->kpath) return 0;
  CHKRET(kspace_layout(c, u, c->d_sa, true));
  tdhf::ApplyArgs a = base_args(c);
  a.mode = tdhf::M_HPSI;
  a.u = a.w = c->d_sa;
  tdhf::KArgs k = kspace_args(c, a);
  return timed(c, c->timing, [&] { return launch_kmat(c, k, 1, c->stream); });
}

// out = H[u] w for nbw columns per k-point, w and out held in ld columns per
// k-point; u is that of the gs_hamiltonian call before.
int gs_product(tdhf_ctx* c, const zd* u, const zd* w, int nbw, int ld, zd* out) {
  tdhf::ApplyArgs a = base_args(c);
  a.mode = tdhf::M_HPSI;
  a.nbw = nbw;
  if (!c->kpath) {
    a.wld = ld;
    a.u = u;
    a.w = w;
    a.out = out;
    return launch_apply(c, a, nbw * c->nk);
  }
  CHKRET(kspace_layout(c, w, c->gs.KW, true, 1, nullptr, nbw, ld));
  a.u = c->d_sa;
  a.w = c->gs.KW;
  a.out = c->gs.KH;
  tdhf::KArgs k = kspace_args(c, a);
  CHKRET(timed(c, c->timing, [&] { return launch_kapply(c, k, 1, c->stream); }));
  return kspace_layout(c, c->gs.KH, out, false, 1, nullptr, nbw, ld);
}

// KS_ubk2_SVD (src/GS_calculation.f90:124-194) on the state in d_u0, which is
// orthonormalised first (Gram_Schmidt).
int gs_krylov(tdhf_ctx* c, int ncg) {
  const int m = c->nb * ncg;
  const size_t blk = (size_t)c->ng * c->nb;  // columns of a Krylov block start here at each k
  zd* W = c->gs.W;
  CHKRET(launch_orth(c, c->d_u0, c->nb, 1, W, m));
  CHKRET(gs_hamiltonian(c, c->d_u0));
  for (int icg = 1; icg < ncg; ++icg)
    CHKRET(gs_product(c, c->d_u0, W + (icg - 1) * blk, c->nb, m, W + icg * blk));
  CHKRET(launch_orth(c, W, m, 2, nullptr, 0));
  CHKRET(gs_product(c, c->d_u0, W, m, m, c->gs.HW));
  return launch_rr(c, W, c->gs.HW, m, c->d_u0);
}

// Gram_Schmidt and Subspace_diag (src/GS_calculation.f90:197-237) on the state
// in d_u0.
int gs_subspace(tdhf_ctx* c) {
  CHKRET(launch_orth(c, c->d_u0, c->nb, 1, c->gs.W, c->nb));
  CHKRET(gs_hamiltonian(c, c->d_u0));
  CHKRET(gs_product(c, c->d_u0, c->d_u0, c->nb, c->nb, c->gs.HW));
  return launch_rr(c, c->gs.W, c->gs.HW, c->nb, c->d_u0);
}

// Observables at A = 0 of the state in d_u0 (host layout) into slot 'slot'.
int gs_observe(tdhf_ctx* c, long slot) {
  tdhf::ApplyArgs a = base_args(c);
  a.mode = tdhf::M_OBS;
  a.u = a.w = c->d_u0;
  a.obs = c->d_obs;
  a.obs_slot = (int)slot;
  if (!c->kpath) return launch_apply(c, a, c->nb * c->nk);
  CHKRET(kspace_layout(c, c->d_u0, c->d_sa, true));
  a.u = a.w = c->d_sa;
  return launch_kspace(c, a);
}

// Energies of slots s0 .. s0 + n - 1.
int gs_energies(tdhf_ctx* c, long s0, long n, double* e) {
  const size_t stride = c->kpath ? tdhf::kspace_obs_stride(c->ng) : c->obs_stride;
  if (c->kpath) {
    CHKRET(launch_obs_reduce(c, c->d_obs + stride * s0, n, 1, 0, c->d_res));
  } else {
    hipLaunchKernelGGL(tdhf::obs_reduce_kernel, dim3((unsigned)((n + 3) / 4)), dim3(256), 0,
                       c->stream, c->d_obs + stride * s0, c->obs_stride, c->nb * c->nk, (int)n,
                       c->dv, c->vcell, c->d_res);
    HIPCHK(c, hipGetLastError());
  }
  std::vector<double> r((size_t)7 * n);
  HIPCHK(c, hipMemcpyAsync(r.data(), c->d_res, r.size() * sizeof(double), hipMemcpyDeviceToHost,
                           c->stream));
  CHKRET(sync(c));
  for (long i = 0; i < n; ++i) e[i] = r[(size_t)7 * i];
  return 0;
}

}  // namespace

extern "C" int tdhf_gs_run(tdhf_ctx* c, double* u, int nscf, int ncg, double tol,
                           double* etot_hist, double* epsbk, double* epserr, int* niter) {
  if (!c) return fail(nullptr, TDHF_EINVAL, "ctx is NULL");
  if (!u || nscf < 0 || ncg < 1) return fail(c, TDHF_EINVAL, "invalid GS arguments");
  const int m = c->nb * ncg;
  if (m > 64) return fail(c, TDHF_EINVAL, "NB*NCG=%d exceeds 64", m);
  if (m > c->ng) return fail(c, TDHF_EINVAL, "NB*NCG=%d exceeds NG=%d", m, c->ng);
  CHKRET(gs_alloc(c, ncg));
  CHKRET(gs_flag_clear(c));
  CHKRET(upload(c, c->d_u0, u));
  c->u0_padded = false;
  // the energies are read one by one where the loop may end on them, else sixteen
  // at a time (a read waits for the iteration: 20 us of an idle device), so that
  // a run whose energy is no longer a number ends within fifteen iterations of it
  const bool each = tol > 0.0;
  constexpr int kRead = 16;
  const int cap = each ? 1 : std::min(nscf, kRead - 1) + 1;
  double e[kRead], eprev = 0.0;
  CHKRET(ensure_obs(c, cap));
  int it = 0;
  for (int n = 0;; ++it) {
    CHKRET(gs_observe(c, n++));
    bool conv = false;
    if (n == cap || it == nscf) {
      CHKRET(gs_energies(c, 0, n, e));
      for (int i = 0; i < n; ++i) {
        const int at = it + 1 - n + i;
        if (etot_hist) etot_hist[at] = e[i];
        if (at > 0 && !std::isfinite(e[i]))
          return fail(c, TDHF_ENUMERIC, "GS energy is not finite at iteration %d", at);
      }
      conv = each && it > 0 && std::fabs(e[0] - eprev) < tol;
      eprev = e[0];
      n = 0;
    }
    if (conv || it == nscf) break;
    CHKRET(gs_krylov(c, ncg));
    CHKRET(gs_subspace(c));
  }
  CHKRET(gs_flag_check(c));
  if (niter) *niter = it;
  if (epsbk || epserr) {
    CHKRET(gs_hamiltonian(c, c->d_u0));
    CHKRET(gs_product(c, c->d_u0, c->d_u0, c->nb, c->nb, c->gs.HW));
    const int rows = c->nb * c->nk;
    hipLaunchKernelGGL(tdhf::epsbk_kernel, dim3(rows), dim3(c->ng), 0, c->stream, c->d_u0,
                       c->gs.HW, c->ng, c->dv, c->gs.eps, c->gs.eps + rows);
    HIPCHK(c, hipGetLastError());
    std::vector<double> h((size_t)2 * rows);
    HIPCHK(c, hipMemcpyAsync(h.data(), c->gs.eps, h.size() * sizeof(double),
                             hipMemcpyDeviceToHost, c->stream));
    CHKRET(sync(c));
    if (epsbk) std::memcpy(epsbk, h.data(), rows * sizeof(double));
    if (epserr) std::memcpy(epserr, h.data() + rows, rows * sizeof(double));
  }
  return download(c, u, c->d_u0);
}
