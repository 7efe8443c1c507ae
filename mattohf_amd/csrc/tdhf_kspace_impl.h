// tdhf_kspace_impl.h -- host side of the density-matrix path (included by
// tdhf.hip after the row-wise launch helpers): when it is used, its tables,
// launches, layout conversions and observables.
#pragma once

namespace {

// Whether the density-matrix path pays for nk k-points of ntraj trajectories:
// its cost against that of the row-wise exchange, in microseconds per stage as
// measured over NG = 16..128, NK = 4..128, NB = 1..8 and 1..64 trajectories.
// Row-wise: 5.5 + 0.42 per 10^6 grid points in the pair transforms, weighted by
// log2 NG.  Density matrices: 13 (two launches, each with its own memory round
// trips) + 12 per 10^6 matrix elements.  Both are averages: the row-wise time goes
// up in rounds of 256 workgroups (NG=64, NB=4: 256 rows of NK=64 13.4, 260 of NK=65
// 25.6), the other with the bands too.  Near the line, measured, row-wise against
// matrices: NG=128, NK=64, NB=4 31.0 and 27.3, NK=16, NB=11 23.2 and 20.5; NG=64,
// NK=33, NB=8 25.7 and 20.7; NG=32, NK=65, NB=6 22.8 and 18.0 take the matrices,
// NG=128, NK=48, NB=4 24.8 and 27.3; NG=64, NK=32, NB=6 11.1 and 16.4; NG=32, NK=24,
// NB=11 17.8 and 17.9; NG=16, NK=128, NB=4 11.9 and 14.7 do not.
struct KspaceCost {
  double rows = 0.0, mat = 0.0;
  bool fits = true;  // kapply_kernel's byte offsets into a padded state are 32 bits wide
  void add(int ng, int nk, int nb, int nbocc, int ntraj = 1) {
    int lg = 0;
    while ((1 << lg) < ng) ++lg;
    rows += 1e-6 * ntraj * nk * nk * nb * nbocc * (double)ng * lg;
    mat += 1e-6 * ntraj * (double)ng * ng * tdhf::kspace_len(nk);
    fits = fits && (size_t)ng * nb * tdhf::kspace_len(nk) * sizeof(zd) <= UINT32_MAX;
  }
  double matrices() const { return 13.0 + 12.0 * mat; }
  double gain() const { return fits ? 5.5 + 0.42 * rows - matrices() : 0.0; }
  bool pays() const { return gain() > 0.0; }
};

bool kspace_pays(int ng, int nk, int nb, int nbocc, int ntraj) {
  if (!tdhf::kspace_len(nk)) return false;
  KspaceCost c;
  c.add(ng, nk, nb, nbocc, ntraj);
  return c.pays();
}

// The same for a context's own runs.  Where all rows have a CU each (one round of
// the row-wise kernel) the averages above mislead, most at NG = 64: the row-wise
// stage is then 5.5 us + 0.030 per pair of a row, at NG = 128 7.0 + 0.093, and the
// matrices' with more than four bands a quarter above their price.  Row-wise
// against matrices: NG=64, NK=32, NB=8 13.5 and 17.5, NK=16, NB=16 13.5 and 18.6;
// NG=128, NK=40, NB=6 30.0 and 32.5, NK=16, NB=16 with 8 occupied 18.7 and 20.1 are
// row-wise, NK=24, NB=8 24.8 and 23.7, NK=64, NB=4 31.0 and 27.3 are not.
// (Gradients, whose reverse stage gains more, are faster through the matrices
// there too.)
bool kspace_run_pays(const tdhf_ctx* c) {
  if (!kspace_pays(c->ng, c->nk, c->nb, c->nbocc, 1)) return false;
  if (c->ng < 64 || (long)c->nk * c->nb > device_cus()) return true;
  const double pairs = (double)c->nk * c->nbocc;
  const double rows = c->ng == 64 ? 5.5 + 0.030 * pairs : 7.0 + 0.093 * pairs;
  KspaceCost k;
  k.add(c->ng, c->nk, c->nb, c->nbocc);
  return rows > k.matrices() * (c->nb > 4 ? 1.25 : 1.0);
}

// Whether one H application of host arrays pays on the path.  Its two states and
// its result change layout: with pinned memory the staging kernels do that on
// their way, else it is three launches between the copies, 20 to 30 us.  Measured
// per call, row-wise against matrices, with KspaceCost's gain: NG=64, NK=32, NB=9
// 92 and 114 us (3), NK=64, NB=8 131 and 140 (32), NK=64, NB=11 184 and 160 (69);
// NG=128, NK=16, NB=16 119 and 141 (14), NK=32, NB=9 158 and 151 (17); NG=32,
// NK=128, NB=6 with 4 occupied 117 and 120 (17), NB=8 174 and 136 (61).
bool kspace_hpsi_pays(const tdhf_ctx* c) {
  KspaceCost k;
  k.add(c->ng, c->nk, c->nb, c->nbocc);
  return c->kpath && (c->h_stage || k.gain() > (c->ng == 64 ? 40.0 : 15.0));
}

// x' values per wave (transform groups).
int kspace_gpw(int n) { return n == 128 ? 4 : n == 64 ? 8 : 16; }

// Bands per workgroup: 2, 4 or 8 accumulators per lane and k (a variant of
// the kernel each); more bands go to further workgroups.
int kspace_nbt(int nbw) { return nbw <= 2 ? 2 : nbw <= 4 ? 4 : 8; }
int kspace_chunks(int nbw) { return (nbw + kspace_nbt(nbw) - 1) / kspace_nbt(nbw); }

template <int N>
const void* kmat_fn(bool obs, bool deep) {
  if (deep)
    return obs ? (const void*)tdhf::kmat_kernel<N, true, true>
               : (const void*)tdhf::kmat_kernel<N, false, true>;
  return obs ? (const void*)tdhf::kmat_kernel<N, true, false>
             : (const void*)tdhf::kmat_kernel<N, false, false>;
}
const void* kmat_fn_for(int n, bool obs, bool deep) {
  switch (n) {
    case 16: return kmat_fn<16>(obs, deep);
    case 32: return kmat_fn<32>(obs, deep);
    case 64: return kmat_fn<64>(obs, deep);
    case 128: return kmat_fn<128>(obs, deep);
  }
  return kmat_fn<0>(obs, deep);
}
template <int XT>
const void* kapply_fn(int nbt) {
  return nbt == 2   ? (const void*)tdhf::kapply_kernel<2, XT>
         : nbt == 4 ? (const void*)tdhf::kapply_kernel<4, XT>
                    : (const void*)tdhf::kapply_kernel<8, XT>;
}
const void* kapply_fn(int nbt, int xt) { return xt == 1 ? kapply_fn<1>(nbt) : kapply_fn<2>(nbt); }
const void* kadj_mat_fn(int n) {
  switch (n) {
    case 16: return (const void*)tdhf::kadj_mat_kernel<16>;
    case 32: return (const void*)tdhf::kadj_mat_kernel<32>;
    case 64: return (const void*)tdhf::kadj_mat_kernel<64>;
  }
  return (const void*)tdhf::kadj_mat_kernel<128>;
}
template <int XT>
const void* kadj_apply_fn(int nbt) {
  return nbt == 2   ? (const void*)tdhf::kadj_apply_kernel<2, XT>
         : nbt == 4 ? (const void*)tdhf::kadj_apply_kernel<4, XT>
                    : (const void*)tdhf::kadj_apply_kernel<8, XT>;
}
const void* kadj_apply_fn(int nbt, int xt) {
  return xt == 1 ? kadj_apply_fn<1>(nbt) : kadj_apply_fn<2>(nbt);
}
size_t kmat_lds_for(int n, int nw, int ng) {
  switch (n) {
    case 16: return tdhf::kmat_lds<16>(nw, ng);
    case 32: return tdhf::kmat_lds<32>(nw, ng);
    case 64: return tdhf::kmat_lds<64>(nw, ng);
    case 128: return tdhf::kmat_lds<128>(nw, ng);
  }
  return std::max(tdhf::kmat_lds<64>(nw, ng), tdhf::kmat_lds<128>(nw, ng));
}
// Two waves per SIMD hold all tasks at once: the deep variant.
bool kmat_deep(long tasks) { return tasks <= 8L * device_cus(); }
hipError_t kmat_lds_limits(int n, int nbw) {
  hipError_t e = hipSuccess;
  for (int v = 0; v < 4 && e == hipSuccess; ++v)
    e = hipFuncSetAttribute(kmat_fn_for(n, v & 1, v & 2),
                            hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
  // (the product kernel in every variant: the ground state multiplies NB NCG columns)
  const int nbt = kspace_nbt(nbw);
  const void* more[] = {kapply_fn(2, 1), kapply_fn(2, 2), kapply_fn(4, 1), kapply_fn(4, 2),
                        kapply_fn(8, 1), kapply_fn(8, 2), kadj_mat_fn(n), kadj_apply_fn(nbt, 1),
                        kadj_apply_fn(nbt, 2)};
  for (auto f : more)
    if (e == hipSuccess)
      e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
  return e;
}
// Workgroups of the two launches for one trajectory (nw waves each).
int kmat_groups(int n, int ng, int nw) {
  return (tdhf::kmat_tasks(ng, kspace_gpw(n)) + nw - 1) / nw;
}
int kapply_groups(int n, int ng, int nbw, int xt) {
  return ng / xt * kspace_chunks(nbw) * (n > 64 ? n / 64 : 1);
}
int kmat_waves(long tasks) { return tasks >= 4096 ? 4 : tasks >= 1024 ? 2 : 1; }
// Grid points per workgroup of the product launch: two share the columns they
// read where one each would already fill the CUs.
int kapply_points(long groups1) { return groups1 >= 512 ? 2 : 1; }
int kapply_waves(int n, int ng) {
  const int xs = n < 64 ? 64 / n : 1;
  int nw = 8;
  while (nw > 1 && nw * xs > ng) nw /= 2;
  return nw;
}

size_t kcount(const tdhf_ctx* c) { return (size_t)c->ng * c->nb * c->kn; }

// complex elements of a state in the path's layout
size_t path_count(const tdhf_ctx* c) { return c->kpath ? kcount(c) : nstate(c); }

// The orbital buffers of a context in its path's layout and, on the
// density-matrix path, the matrices of a stage.
int alloc_states(tdhf_ctx* c) {
  const size_t n = path_count(c);
  for (zd** p : {&c->d_u0, &c->d_ksum, &c->d_sa, &c->d_sb, &c->d_w, &c->d_out})
    CHKRET(dalloc(c, p, n));
  if (!c->kpath) return 0;
  CHKRET(dalloc(c, &c->d_hm, tdhf::kmat_elems(c->ng, c->kn)));
  return dalloc(c, &c->d_nx, tdhf::kmat_extra(c->ng, kspace_gpw(c->kn)));
}

// Spectra, twiddles of the k transforms and the twist factors of a context, made
// when the first run on the path needs them (a context that stays row-wise does
// without: NG=16, NK=40, NB=8 created in 309 us, 377 with them).
int kspace_tables(tdhf_ctx* c) {
  if (c->d_ktab) return 0;
  const int NG = c->ng, NK = c->nk, ND = 2 * NK - 1, N = c->kn;
  zd* tsp = nullptr;
  int rc = dalloc(c, &c->d_ktab, (size_t)NG * 2 * N);
  if (!rc) rc = dalloc(c, &c->d_ktw, 2 * N);
  if (!rc) rc = dalloc(c, &c->d_om, N);
  if (!rc) rc = dalloc(c, &tsp, (size_t)ND * NG);
  auto undo = [&] {
    dfree(c->d_ktab);
    dfree(c->d_ktw);
    dfree(c->d_om);
  };
  if (rc) {
    undo();
    return rc;
  }
  hipStream_t s = c->stream;
  hipLaunchKernelGGL(tdhf::kspace_space_kernel, dim3((ND * NG + 255) / 256), dim3(256), 0, s,
                     c->d_vq, ND, NG, -1.0 / ((double)NG * (double)NK), tsp);
  const dim3 g((NG * 2 * N + 255) / 256), b(256), g1(1);
  switch (N) {
    case 16:
      hipLaunchKernelGGL(tdhf::kspace_spectrum_kernel<16>, g, b, 0, s, tsp, NK, NG, c->d_ktab);
      hipLaunchKernelGGL(tdhf::twiddle_kernel<16>, g1, b, 0, s, c->d_ktw);
      break;
    case 32:
      hipLaunchKernelGGL(tdhf::kspace_spectrum_kernel<32>, g, b, 0, s, tsp, NK, NG, c->d_ktab);
      hipLaunchKernelGGL(tdhf::twiddle_kernel<32>, g1, b, 0, s, c->d_ktw);
      break;
    case 64:
      hipLaunchKernelGGL(tdhf::kspace_spectrum_kernel<64>, g, b, 0, s, tsp, NK, NG, c->d_ktab);
      hipLaunchKernelGGL(tdhf::twiddle_kernel<64>, g1, b, 0, s, c->d_ktw);
      break;
    default:
      hipLaunchKernelGGL(tdhf::kspace_spectrum_kernel<128>, g, b, 0, s, tsp, NK, NG, c->d_ktab);
      hipLaunchKernelGGL(tdhf::twiddle_kernel<128>, g1, b, 0, s, c->d_ktw);
      break;
  }
  hipLaunchKernelGGL(tdhf::kspace_om_kernel, g1, dim3(128), 0, s, c->d_om, N);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  dfree(tsp);
  if (e == hipSuccess) e = kmat_lds_limits(N, c->nb);
  if (e != hipSuccess) {
    undo();
    return fail(c, TDHF_EDEVICE, "k-space tables: %s", hipGetErrorString(e));
  }
  return 0;
}

int kspace_class(int n) { return n == 16 ? 0 : n == 32 ? 1 : n == 64 ? 2 : 3; }

// Arguments of a launch on the context's own tables (states in the padded
// k-fastest layout); a as for launch_apply.
tdhf::KArgs kspace_args(const tdhf_ctx* c, const tdhf::ApplyArgs& a) {
  tdhf::KArgs k{};
  k.a = a;
  k.ng = c->ng;
  k.n = c->kn;
  k.nchunk = kspace_chunks(a.nbw);
  k.ktab = c->d_ktab;
  k.hm = c->d_hm;
  k.nx = c->d_nx;
  k.tw[kspace_class(c->kn)] = c->d_ktw;
  k.om[kspace_class(c->kn)] = c->d_om;
  return k;
}

// Matrices and density scratch of ntraj trajectories.
struct KScratch {
  zd* hm;
  double* nx;
  size_t hstride, nstride;
};

// The matrices of the states a.u.
int launch_kmat(tdhf_ctx* c, tdhf::KArgs& k, int ntraj, hipStream_t s) {
  void* args[] = {&k};
  const bool obs = k.a.mode == tdhf::M_S1 || k.a.mode == tdhf::M_OBS;
  const long tasks = (long)tdhf::kmat_tasks(c->ng, kspace_gpw(c->kn)) * ntraj;
  const int wa = kmat_waves(tasks);
  HIPCHK(c, hipLaunchKernel(kmat_fn_for(c->kn, obs, kmat_deep(tasks)),
                            dim3(kmat_groups(c->kn, c->ng, wa), ntraj), dim3(64 * wa), args,
                            kmat_lds_for(c->kn, wa, c->ng), s));
  return 0;
}
// Their product with the columns a.w and the stage update.
int launch_kapply(tdhf_ctx* c, tdhf::KArgs& k, int ntraj, hipStream_t s) {
  void* args[] = {&k};
  const int wb = kapply_waves(c->kn, c->ng), nbt = kspace_nbt(k.a.nbw);
  const int xt = kapply_points((long)kapply_groups(c->kn, c->ng, k.a.nbw, 1) * ntraj);
  HIPCHK(c, hipLaunchKernel(kapply_fn(nbt, xt),
                            dim3(kapply_groups(c->kn, c->ng, k.a.nbw, xt), ntraj), dim3(64 * wb),
                            args, tdhf::kapply_lds(wb, nbt, xt), s));
  return 0;
}

// launch() on the context's stream, between two events where on.
template <typename F>
int timed(tdhf_ctx* c, bool on, F launch) {
  hipEvent_t e0 = nullptr, e1 = nullptr;
  if (on) {
    CHKRET(take_events(c, &e0, &e1));
    HIPCHK(c, hipEventRecord(e0, c->stream));
  }
  CHKRET(launch());
  if (on) HIPCHK(c, hipEventRecord(e1, c->stream));
  return 0;
}

int launch_kspace(tdhf_ctx* c, const tdhf::ApplyArgs& a, int ntraj = 1,
                  hipStream_t st = nullptr, const KScratch* sc = nullptr) {
  tdhf::KArgs k = kspace_args(c, a);
  if (sc) {
    k.hm = sc->hm;
    k.nx = sc->nx;
    k.hstride = sc->hstride;
    k.nstride = sc->nstride;
  }
  hipStream_t s = st ? st : c->stream;
  return timed(c, c->timing && !st, [&] {
    CHKRET(launch_kmat(c, k, ntraj, s));
    return launch_kapply(c, k, ntraj, s);
  });
}

// One stage launch of the context's path, states in that path's layout.
int launch_stage(tdhf_ctx* c, const tdhf::ApplyArgs& a) {
  return c->kpath ? launch_kspace(c, a) : launch_apply(c, a, c->nb * c->nk);
}

// dst = src in the other layout, for ntraj states back to back (or nb columns
// per k-point, held in ld on the host layout's side).
int kspace_layout(tdhf_ctx* c, const zd* src, zd* dst, bool to_k, int ntraj = 1,
                  hipStream_t st = nullptr, int nb = 0, int ld = 0) {
  if (nb == 0) nb = c->nb;
  tdhf::KLayoutArgs l{};
  l.src = src;
  l.dst = dst;
  l.ng = c->ng;
  l.nb = nb;
  l.ld = ld;
  l.nk = c->nk;
  l.n = c->kn;
  l.sstride = to_k ? nstate(c) : kcount(c);
  l.dstride = to_k ? kcount(c) : nstate(c);
  l.to_k = to_k;
  hipLaunchKernelGGL(tdhf::kspace_layout_kernel, dim3(nb * ntraj, c->kn / 16, c->ng / 16),
                     dim3(256), 0, st ? st : c->stream, l);
  HIPCHK(c, hipGetLastError());
  return 0;
}

// Host state to dst in the path's layout (through d_ksum, which holds nothing
// between steps), and back.
int upload_state(tdhf_ctx* c, zd* dst, const double* src) {
  if (!c->kpath) return upload(c, dst, src);
  CHKRET(upload(c, c->d_ksum, src));
  return kspace_layout(c, c->d_ksum, dst, true);
}

int download_state(tdhf_ctx* c, double* dst, const zd* src) {
  if (!c->kpath) return download(c, dst, src);
  CHKRET(kspace_layout(c, src, c->d_ksum, false));
  return download(c, dst, c->d_ksum);
}

// A call on one small state is mostly copies: each from or to pageable memory
// takes 10 us, an H application of 16 KB 6.  States of up to 256 KB go through
// the context's pinned memory instead, which a kernel reads and another writes
// (H of 32 x 2 x 4: 36 -> 24 us; a step of 64 x 3 x 21: 87 -> 51 us).  Beyond
// that the copy engines are as fast as a kernel over the bus.
constexpr size_t kStageState = 256 * 1024 / sizeof(zd);

// The caller's state (and a second one) to dst (dst2), padded with kp.
int stage_in(tdhf_ctx* c, bool kp, zd* dst, const double* src, zd* dst2 = nullptr,
             const double* src2 = nullptr) {
  if (!c->h_stage) {
    if (!kp) {
      CHKRET(upload(c, dst, src));
      return src2 ? upload(c, dst2, src2) : 0;
    }
    if (!src2) return upload_state(c, dst, src);
    // both copies, then both kernels: a copy after a kernel waits for it on
    // another engine (d_out holds nothing before the product)
    CHKRET(upload(c, c->d_ksum, src));
    CHKRET(upload(c, c->d_out, src2));
    CHKRET(kspace_layout(c, c->d_ksum, dst, true));
    return kspace_layout(c, c->d_out, dst2, true);
  }
  const size_t n = nstate(c);
  std::memcpy(c->h_stage, src, n * sizeof(zd));
  if (src2) std::memcpy(c->h_stage + n, src2, n * sizeof(zd));
  if (kp) {
    CHKRET(kspace_layout(c, c->h_stage, dst, true));
    return src2 ? kspace_layout(c, c->h_stage + n, dst2, true) : 0;
  }
  const long m = (long)(src2 ? 2 * n : n);
  hipLaunchKernelGGL(tdhf::stage_kernel, dim3((unsigned)((m + 255) / 256)), dim3(256), 0,
                     c->stream, c->h_stage, dst, dst2, (long)n, m);
  HIPCHK(c, hipGetLastError());
  return 0;
}

// src, padded with kp, to the caller's state, after all that is queued.
int stage_out(tdhf_ctx* c, bool kp, double* dst, const zd* src) {
  if (!c->h_stage) {
    CHKRET(kp ? download_state(c, dst, src) : download(c, dst, src));
    return harvest_timing(c);
  }
  const size_t n = nstate(c);
  zd* h = c->h_stage + 2 * n;
  if (kp) {
    CHKRET(kspace_layout(c, src, h, false));
  } else if (src != h) {
    hipLaunchKernelGGL(tdhf::stage_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                       c->stream, src, h, (zd*)nullptr, (long)n, (long)n);
    HIPCHK(c, hipGetLastError());
  }
  CHKRET(sync(c));
  std::memcpy(dst, h, n * sizeof(zd));
  return 0;
}

// The resident state in the path's layout (the ground state leaves it in the
// host's).
int resident_to_path(tdhf_ctx* c) {
  if (!c->kpath || c->u0_padded) return 0;
  CHKRET(kspace_layout(c, c->d_u0, c->d_ksum, true));
  HIPCHK(c, hipMemcpyAsync(c->d_u0, c->d_ksum, kcount(c) * sizeof(zd), hipMemcpyDeviceToDevice,
                           c->stream));
  c->u0_padded = true;
  return 0;
}

// Observables of nslots slots reduced into out (7 values each), ntraj
// trajectories ostride doubles apart.
int launch_obs_reduce(tdhf_ctx* c, const double* obs, long nslots, int ntraj, size_t ostride,
                      double* out) {
  const long nw = nslots * ntraj;
  hipLaunchKernelGGL(tdhf::kspace_obs_reduce_kernel, dim3((unsigned)((nw + 3) / 4)), dim3(256), 0,
                     c->stream, obs, (const tdhf::TrajDesc*)nullptr, c->ng, (int)nslots, (int)nw,
                     c->dv, c->vcell, ostride, out);
  HIPCHK(c, hipGetLastError());
  return 0;
}

// Observables of the state u (in the path's layout) at field A.
int path_observables_of(tdhf_ctx* c, const zd* u, double A, double* res7) {
  if (!c->kpath) return observables_of(c, u, A, res7);
  CHKRET(ensure_obs(c, 1));
  tdhf::ApplyArgs a = base_args(c);
  a.mode = tdhf::M_OBS;
  a.u = a.w = u;
  a.A = A;
  a.Aobs = A;
  a.obs = c->d_obs;
  a.obs_slot = 0;
  CHKRET(launch_kspace(c, a));
  CHKRET(launch_obs_reduce(c, c->d_obs, 1, 1, 0, c->d_res));
  HIPCHK(c, hipMemcpyAsync(res7, c->d_res, 7 * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  return sync(c);
}

// out = H[u] w, padded states with kp.
int path_hpsi(tdhf_ctx* c, bool kp, const zd* u, const zd* w, double A, zd* out) {
  tdhf::ApplyArgs a = base_args(c);
  a.mode = tdhf::M_HPSI;
  a.u = u;
  a.w = w;
  a.A = A;
  a.Aobs = A;
  a.out = out;
  return kp ? launch_kspace(c, a) : launch_apply(c, a, c->nb * c->nk);
}

}  // namespace
