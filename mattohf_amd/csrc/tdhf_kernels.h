// tdhf_kernels.h -- device kernels of the TDHF path (gfx950, FP64).
//
// The dominant kernel is apply_kernel<NG>: one workgroup per output orbital
// (k,i) ("row").  Its groups of L lanes stream the occupied orbitals u(q,j)
// of every k-point q and, for each, do the exchange pair round trip of
// ubkwbk_vFwbk (src/Functions.f90:247-257):
//     rho = w(k,i) * conj(u(q,j))  ->  FFT  ->  * -v(G+k-q)/(NG*NK)  ->  IFFT
//     acc += result * u(q,j)
// entirely in registers plus one LDS transpose per transform.  The same pass
// accumulates the density sum_{q,j} |u(q,j)|^2 (ubk_dns, src/Functions.f90
// :55-71), so no separate density kernel is needed.  After a workgroup-wide
// reduction, the Hartree round trip (dns_vH, :147-162) and the kinetic round
// trip of w (ubk_tubk, :212-234) are evaluated either as the circulant
// products they are, vH = K_H * rho and T w = K_2 * w + (k+A) K_1 * w +
// (k+A)^2/2 w, with
//     K_H(d) = 1/NG sum_G vCG(G) cos(2 pi g d/NG),
//     K_2(d) = 1/NG sum_G G^2/2 cos(2 pi g d/NG),
//     K_1(d) = 1/NG sum_G G exp(2 pi i g d/NG)
// (G in FFT order, Nyquist at -NG/2 b), by all threads of the workgroup, or,
// at NG = 128 with fewer than four waves, as one transform round trip each,
//     vH = occ IFFT[vCG/NG . FFT[rho]],   T w = IFFT[(G+k+A)^2/(2 NG) . FFT[w]],
// on two groups of the first wave.  The epilogue forms
// H w = T w + (vH + vion) w + V_F w (ubkwbk_hwbk, :187-209) and applies the
// mode-specific update (plain H|w>, one RK4 stage of RT_RK4_ubk,
// src/RT_calculation.f90:154-173, or observables only).  Per-row partial sums
// of Ekin and J (src/Functions.f90:94-119,289-318) follow by Parseval, from
// the circulant products, sum_x conj(w) (K_f * w) = sum_G f(G)|w_G|^2/NG, or
// from FFT[w]; Ex (:165-183) from V_F w.
#pragma once
#include "tdhf_fft.h"

namespace tdhf {

enum ApplyMode : int {
  M_HPSI = 0,  // out = H[u] w
  M_S1 = 1,    // RK4 stage 1 (+ observables of the stage input)
  M_S2 = 2,
  M_S3 = 3,
  M_S4 = 4,
  M_OBS = 5    // observables only
};

// One trajectory of a batch: its k-mesh, tables, RK4 buffers, field and
// observables slots.  The batched launch covers the rows of all trajectories.
struct TrajDesc {
  int nk;
  int obs_stride;           // 3*NB*nk + 3
  double occ;               // 2/nk
  const double* kx;
  const double* vion;
  const double* vtl;
  const double* kc;
  zd* u0;
  zd* ksum;
  zd* sa;
  zd* sb;
  const double* A;
  const double* Aave;
  double* obs;
  // exchange from the pair tiles (tdhf_pairtile.h, read by
  // pair_epilogue_kernel): nblk partial sums per row (row r, block c at
  // (r * nblk + c) * NG) and nblk density partials (block b at b * NG)
  zd* xpart;
  double* dpart;
  int nblk;
  const double* vhg;  // vCG(G)/NG in the G layout of GroupFFT<NG> (pair-tile epilogue)
  // density-matrix path (tdhf_kspace.h): length of the k transforms (the
  // padded number of k-points) and the Coulomb spectra
  int n;
  const zd* ktab;
  zd* hm;
  double* nx;
};

// Offsets inside one observables slot: rows*3 partials then (N, Eion, EH).
struct ApplyArgs {
  int nk, nb, nbocc, nbw;  // nbw = columns of w / out per k-point
  int wld;                  // columns per k-point w and out are held in (0: nbw)
  double bx, dv, occ, dt;
  double A, Aobs;           // used when Aarr == nullptr
  const double* Aarr;       // per-step A(it), or nullptr
  const double* Aavearr;    // per-step Aave(it)
  const int* step_base;     // device step counter (graph replay), or nullptr
  int jstep;                // step = *step_base + jstep
  int obs_slot;             // slot when step_base == nullptr
  int obs_stride;           // doubles per observables slot
  const double* kx;         // NK
  const double* vion;       // NG
  const double* vtl;        // (2NK-1)*NG, G layout, -v(G+k-q)/(NG*NK)
  const double* kc;         // 4*NG: circulant kernels K_H, K_2, K_1 (complex)
  const double* vhg;        // NG: vCG(G)/NG in the G layout of GroupFFT<NG>
  const zd* tw;             // twiddle table of GroupFFT<NG> (2*NG)
  const zd* u;              // (NG,NB,NK) orbitals defining rho and V_F
  const zd* w;              // (NG,nbw,NK) orbitals H acts on
  zd* out;                  // M_HPSI output (NG,nbw,NK)
  zd* u0;                   // RK4: state at the start of the step
  zd* ksum;                 // RK4: k1 + 2 k2 + 2 k3
  zd* unext;                // RK4: next stage input
  double* obs;              // observables slots, or nullptr
  int mode;
  const TrajDesc* td;       // batched launch: trajectory table, or nullptr
  const int2* rowmap;       // batched launch: (trajectory, row) per workgroup
  zd* tape;                 // RK4 stage states y1..y4 per step (adjoint), or nullptr
  int tape_seg;             // steps held by the tape: step it in slot it % tape_seg
  size_t nstate;            // tape stride of one stage block (all trajectories)
  // uniform batch (grid y = trajectory, same NK and tables): offsets of
  // trajectory t are t*tstride (states, zd), t*fstride (A, Aave), t*ostride
  // (observables)
  size_t tstride;
  int fstride;
  size_t ostride;
  int balance;  // 1: balance the waves of a SIMD by issue priority (set by the launcher)
};

__device__ __forceinline__ double gvalue(int g, int NG, double bx) {
  // Gx in FFT order, src/Initialization.f90:97-102
  return g < NG / 2 ? (double)g * bx : (double)(g - NG) * bx;
}

// Exchange-and-add steps of wave_reduce_scatter for a pair of values (x, y)
// over one lane bit: lanes with the bit clear return x summed over the lane
// pair, lanes with the bit set return y summed over the pair.
// Bit 5: v_permlane32_swap exchanges the upper half of x with the lower half
// of y, so x' + y' is (x_lo + x_hi | y_lo + y_hi).
__device__ __forceinline__ double pair_sum_bit5(double x, double y) {
  const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)__double2loint(x),
                                                   (unsigned)__double2loint(y), false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)__double2hiint(x),
                                                   (unsigned)__double2hiint(y), false, false);
  return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}
// Bit 4: v_permlane16_swap exchanges the odd 16-lane rows of x with the even
// rows of y.
__device__ __forceinline__ double pair_sum_bit4(double x, double y) {
  const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)__double2loint(x),
                                                   (unsigned)__double2loint(y), false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)__double2hiint(x),
                                                   (unsigned)__double2hiint(y), false, false);
  return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}
// Bit 3: DPP row_ror:8 reads lane (i ^ 8) within each 16-lane row.
__device__ __forceinline__ double pair_sum_bit3(double x, double y, bool bit) {
  const double send = bit ? x : y, keep = bit ? y : x;
  const int rl = __builtin_amdgcn_update_dpp(0, __double2loint(send), 0x128, 0xf, 0xf, false);
  const int rh = __builtin_amdgcn_update_dpp(0, __double2hiint(send), 0x128, 0xf, 0xf, false);
  return keep + __hiloint2double(rh, rl);
}

// Bit 2: ds_bpermute (__shfl_xor) from lane i ^ 4.
__device__ __forceinline__ double pair_sum_bit2(double x, double y, bool bit) {
  const double send = bit ? x : y, keep = bit ? y : x;
  return keep + __shfl_xor(send, 4);
}

// Sum of v over the 64 lanes of a wave, the same in every lane, without LDS:
// DPP within 16 lanes (lane ^ 1, ^ 2, then mirrors, which act as ^ 4 and ^ 8
// once the quads and half rows are equal), permlane swaps across them.
__device__ __forceinline__ double wave_sum(double v) {
  auto dpp = [](double x, auto ctrl) {
    constexpr int c = decltype(ctrl)::value;
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), c, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), c, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
  };
  v += dpp(v, std::integral_constant<int, 0xB1>{});   // quad_perm [1,0,3,2]
  v += dpp(v, std::integral_constant<int, 0x4E>{});   // quad_perm [2,3,0,1]
  v += dpp(v, std::integral_constant<int, 0x141>{});  // row_half_mirror
  v += dpp(v, std::integral_constant<int, 0x140>{});  // row_mirror
  v = pair_sum_bit4(v, v);
  return pair_sum_bit5(v, v);
}

// Sums the NV values v[] of every lane over the groups of L lanes of a wave
// (lane bits log2(L)..5) without LDS, as a reduce-scatter: each step hands
// half of the values to the partner lane of one lane bit and keeps the other
// half, summed.  Afterwards v[k], k < NV L / 64, holds the sum over the
// wave's groups of value k + (NV L / 64) gw, where gw = lane / L.
template <int L, int NV>
__device__ __forceinline__ void wave_reduce_scatter(double* v) {
  static_assert(L == 4 || L == 8 || L == 16 || L == 32, "lane groups of 4 to 32");
  static_assert((NV * L) % 64 == 0, "values must split evenly over the groups");
  const int lane = threadIdx.x & 63;
  static_for<0, NV / 2>([&](auto kc) {
    constexpr int k = decltype(kc)::value;
    v[k] = pair_sum_bit5(v[k], v[k + NV / 2]);
  });
  if constexpr (L <= 16) {
    static_for<0, NV / 4>([&](auto kc) {
      constexpr int k = decltype(kc)::value;
      v[k] = pair_sum_bit4(v[k], v[k + NV / 4]);
    });
  }
  if constexpr (L <= 8) {
    const bool b3 = (lane & 8) != 0;
    static_for<0, NV / 8>([&](auto kc) {
      constexpr int k = decltype(kc)::value;
      v[k] = pair_sum_bit3(v[k], v[k + NV / 8], b3);
    });
  }
  if constexpr (L <= 4) {
    const bool b2 = (lane & 4) != 0;
    static_for<0, NV / 16>([&](auto kc) {
      constexpr int k = decltype(kc)::value;
      v[k] = pair_sum_bit2(v[k], v[k + NV / 16], b2);
    });
  }
}

// p[0] + p[stride] + ... (n terms in order), the reads of up to four ahead of
// the sums.
__device__ __forceinline__ double ordered_sum(const double* p, int stride, int n) {
  double s = 0.0;
  int i = 0;
  for (; i + 4 <= n; i += 4, p += 4 * stride) {
    const double a = p[0], b = p[stride], c = p[2 * stride], d = p[3 * stride];
    s = (((s + a) + b) + c) + d;
  }
  for (; i < n; ++i, p += stride) s += p[0];
  return s;
}

// Sets the issue priority (0..3) of the executing wave; p must be the same in
// every lane of the wave.
__device__ __forceinline__ void set_wave_priority(int p) {
  switch (__builtin_amdgcn_readfirstlane(p)) {
    case 3: __builtin_amdgcn_s_setprio(3); break;
    case 2: __builtin_amdgcn_s_setprio(2); break;
    case 1: __builtin_amdgcn_s_setprio(1); break;
    default: __builtin_amdgcn_s_setprio(0); break;
  }
}

// Per-group LDS slot of apply_kernel (complex elements): the transpose tile
// during the pair loop; afterwards the slot area holds the wave partials of
// the reduction (3 NG doubles per wave), the circulant-product partials or the
// tiles of the Hartree and kinetic transforms, and the observables staging.  At least 3 NG / 2 elements, rounded up to 8 mod 16
// elements, so that consecutive groups start half a bank cycle (32 of the 64
// four-byte banks) apart and the transposes of two groups served in one LDS
// pass do not collide.
template <int NG>
__host__ __device__ constexpr int apply_slot() {
  constexpr int need = GroupFFT<NG>::TSZ >= (3 * NG + 1) / 2 ? GroupFFT<NG>::TSZ : (3 * NG + 1) / 2;
  return need + ((8 - need % 16) + 16) % 16;
}

// LDS footprint of apply_kernel<NG> with nw waves (bytes): the groups' slots
// (also the circulant-product partials and observables staging after the
// pair loop), then w, V_F w (followed by rho), K_1 or T w (complex NG each),
// rho, K_H or vH, K_2 or vCG/NG in the G layout (NG doubles each), a small
// scratch and the twiddle table.
template <int NG>
__host__ __device__ constexpr size_t apply_lds_bytes(int nw) {
  return (size_t)nw * (64 / GroupFFT<NG>::L) * apply_slot<NG>() * sizeof(zd) +
         3 * NG * sizeof(zd) + 3 * NG * sizeof(double) + 16 * sizeof(double) +
         GroupFFT<NG>::TWL * sizeof(zd);
}

// A launch of a small system is a chain of latencies, of which an empty kernel in
// a graph takes 1.6 us: the arguments, one round trip to memory, the transforms
// of one pair, two reductions, the stores.  So each link has one wait: scalar
// loads in one batch, field values and twiddles off the way of the operands,
// sums whose reads go ahead.  Per RK4 stage, against one batch per use and one
// read per product:
//   NG 16, 40 k-points, 8 bands, 1 occupied   5.55 -> 4.93 us
//   NG 32, 32 k-points, 2 bands               7.51 -> 5.80 us
//   NG 64, 21 k-points, 3 bands               8.55 -> 7.14 us
//   NG 64, 64 k-points, 4 bands               15.9 -> 14.4 us (four passes per wave)
//   NG 128, 16 k-points, 4 bands              13.75 -> 12.8 us
//
// TE: the Hartree and kinetic round trips as transforms (else circulant
// products); the launcher chooses: transforms where the 1024 blocks of the
// products at NG = 128 meet few waves.  Per stage, transforms against products: NG = 128
// with two waves 7.3 against 8.2 us, four 8.0 against 8.05, eight 12.8 against
// 12.7; NG = 64 with one wave 6.3 against 6.2, two 6.45 against 5.8.
template <int NG>
__host__ __device__ constexpr bool apply_by_transforms(int nw) {
  return NG == 128 && nw < 4;
}

// ONE: at NG = 32, rows of one wave with many passes: twiddles in registers,
// multipliers read at the start of their pass, not ahead of it, and no last pass of
// its own.  12 trajectories of 140 k-points, 4 bands 319 us per stage against 329
// (8 bands 1.21 against 1.25 ms); the same form costs 120 pairs a row 24.6 against
// 23.8 and eight waves (16 k-points, 16 bands) 10.5 against 9.3.
constexpr int kOnePairs = 192;  // pairs a row from which it pays
template <int NG, bool TE, bool ONE = false>
__global__ void __launch_bounds__(512, NG == 16 ? 4 : 2) apply_kernel(ApplyArgs a) {
  using F = GroupFFT<NG>;
  constexpr int R = F::R, L = F::L, GPW = 64 / L;
  constexpr int SSZ = apply_slot<NG>();
  // circulant products: points of a block, and waves that work on them
  constexpr int CB = NG >= 64 ? 4 : 2, CW = (NG / CB) * (NG / CB) / 64;
  // after the reduction the slot area holds 5 NG partials per wave and the
  // observables staging (6 NG doubles); checked at the smallest launch (one
  // wave, or NG/64 waves)
  constexpr int NW1 = NG > 64 ? NG / 64 : 1;
  static_assert(5 * NG * NW1 + 6 * NG <= 2 * SSZ * GPW * NW1,
                "slot area too small for the epilogue scratch");
  extern __shared__ zd smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l = lane % L, gw = lane / L;
  const int lane0 = lane_zero();
  // per-workgroup operands: from the arguments, or from the trajectory table
  int row = blockIdx.x;
  int nk = a.nk, obs_stride = a.obs_stride;
  double occ = a.occ;
  const double *kx = a.kx, *vion = a.vion, *vtl = a.vtl, *kc = a.kc, *vhg = a.vhg;
  const double *Aarr = a.Aarr, *Aavearr = a.Aavearr;
  const zd *u = a.u, *w = a.w;
  zd *u0 = a.u0, *ksum = a.ksum, *unext = a.unext, *out = a.out;
  double* obs = a.obs;
  // read in one batch of scalar loads (where each is first used, they are a
  // chain of five batches, 0.5 us)
  int mode = a.mode, jstep = a.jstep, nbw = a.nbw;
  const int* step_base = a.step_base;
  asm("" : "+s"(nk), "+s"(nbw), "+s"(mode), "+s"(jstep), "+s"(step_base), "+s"(kx), "+s"(vtl),
           "+s"(kc), "+s"(u), "+s"(w), "+s"(u0), "+s"(ksum), "+s"(unext), "+s"(obs));
  int wld = a.wld, balance = a.balance, nthr = blockDim.x;
  zd* tape = a.tape;
  asm("" : "+s"(row), "+s"(wld), "+s"(balance), "+s"(nthr), "+s"(tape), "+s"(vion), "+s"(vhg));
  const int tr = blockIdx.y;  // trajectory of a uniform batch (0 otherwise)
  if (tr > 0) {
    Aarr += (size_t)tr * a.fstride;
    Aavearr += (size_t)tr * a.fstride;
  }
  if (a.td) {
    const int2 rm = a.rowmap[blockIdx.x];
    if (rm.x < 0) return;  // padding entry of the schedule (whole workgroup)
    const TrajDesc& t = a.td[rm.x];
    row = rm.y;
    nk = t.nk;
    obs_stride = t.obs_stride;
    occ = t.occ;
    kx = t.kx;
    vion = t.vion;
    vtl = t.vtl;
    kc = t.kc;
    vhg = t.vhg;
    Aarr = t.A;
    Aavearr = t.Aave;
    u0 = t.u0;
    ksum = t.ksum;
    obs = t.obs;
    switch (mode) {
      case M_S1: u = t.u0; unext = t.sa; break;
      case M_S2: u = t.sa; unext = t.sb; break;
      case M_S3: u = t.sb; unext = t.sa; break;
      case M_S4: u = t.sa; unext = nullptr; break;
      default: u = t.u0; unext = nullptr; break;
    }
    w = u;
  }
  const int ik = row / nbw, ib = row - ik * nbw;

  const int nw = nthr >> 6;
  const int grp = wave * GPW + gw, ngrp = nw * GPW;
  zd* T = smem + grp * SSZ;
  zd* sW = smem + ngrp * SSZ;
  zd* sVF = sW + NG;
  double* sRho = reinterpret_cast<double*>(sVF + NG);  // follows V_F w (one reduction)
  zd* sK1 = reinterpret_cast<zd*>(sRho + NG);          // K_1, or T w
  double* sKH = reinterpret_cast<double*>(sK1 + NG);   // K_H, or vH
  double* sK2 = sKH + NG;                              // K_2, or vCG/NG (G layout)
  double* sRed = sK2 + NG;
  zd* sTw = reinterpret_cast<zd*>(sRed + 16);  // twiddle table (GroupFFT<NG>::TWL)

  // taped forward: the stage states live in the tape slots of this step
  const bool fields = step_base != nullptr;  // field arrays at the device step counter
  const int step0 = gload_lanes(fields ? step_base : reinterpret_cast<const int*>(a.tw), lane0);
  zd* tape0 = nullptr;
  if (tape && step_base) {
    zd* tp = tape + (size_t)((__builtin_amdgcn_readfirstlane(step0) + jstep) % a.tape_seg) * 4 * a.nstate;
    switch (mode) {
      case M_S1: tape0 = tp; unext = tp + a.nstate; break;
      case M_S2: u = w = tp + a.nstate; unext = tp + 2 * a.nstate; break;
      case M_S3: u = w = tp + 2 * a.nstate; unext = tp + 3 * a.nstate; break;
      case M_S4: u = w = tp + 3 * a.nstate; break;
      default: break;
    }
  }
  if (tr > 0) {
    const size_t so = (size_t)tr * a.tstride;
    u += so;
    w += so;
    if (u0) u0 += so;
    if (ksum) ksum += so;
    if (unext) unext += so;
    if (out) out += so;
    if (tape0) tape0 += so;
    if (obs) obs += (size_t)tr * a.ostride;
  }

  // ---- prologue: every operand load of the first pass is issued before the
  // first wait, so the loop starts after one memory round trip: w of this row,
  // the kinetic kernels and the twiddle table, which go to LDS (each wave
  // loading its lanes' twiddles itself kept the L1 of the CU busy for 1 us),
  // then the first u(q,j) and multipliers ----
  const size_t o = (size_t)NG * (wld ? ib + wld * ik : row) + (tid < NG ? tid : 0);
  zd w_o = mk(0.0, 0.0), k1_o = mk(0.0, 0.0), tw_o[2];
  double k2_o = 0.0;
  const double kxv = gload(kx + (ik + lane0));
  if (tid < NG) {
    w_o = gload(w + o);
    if constexpr (TE) {
      k2_o = gload(vhg + tid);
    } else {
      k2_o = gload(kc + NG + tid);
      k1_o = gload(reinterpret_cast<const zd*>(kc + 2 * NG) + tid);
    }
  }
  static_for<0, 2>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
    const int t = tid + i * nthr;
    if ((i == 0 || NG == 128) && t < F::TWL) tw_o[i] = gload(a.tw + t);
  });

  zd acc[R], un[R];
  double den[R], vtr[R];

  // ---- exchange pair loop (ubkwbk_vFwbk, src/Functions.f90:247-257) ----
  // u(q,j) and the multipliers of the next pair are fetched while the current
  // pair is transformed; the last pass, the only one of a small system, fetches
  // nothing.
  const int nitem = nk * a.nbocc;
  // item = jb + nbocc iq; a group's items are ngrp apart
  const int dq = ngrp / a.nbocc, dj = ngrp - dq * a.nbocc;
  // item of the current pass (a group without one loads the last: the waits
  // for w and the twiddles then count exactly the loads issued after them)
  const int item0 = grp < nitem ? grp : nitem - 1;
  int cq = item0 / a.nbocc, cj = item0 - cq * a.nbocc;
  auto fetch_u = [&](int iq, int jb) {
    const zd* urow = u + (size_t)NG * (jb + a.nb * iq);
    static_for<0, R>([&](auto mc) {
      constexpr int m = decltype(mc)::value;
      un[m] = gload(urow + L * m + l);
    });
  };
  auto fetch_v = [&](int iq) {
    const double* vt = vtl + (size_t)(ik - iq + nk - 1) * NG + l * R;
    static_for<0, R>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      vtr[j] = gload(vt + j);
    });
  };
  fetch_u(cq, cj);
  fetch_v(cq);
  static_for<0, R>([&](auto mc) {
    constexpr int m = decltype(mc)::value;
    acc[m] = mk(0.0, 0.0);
    den[m] = 0.0;
  });
  if (tid < NG) {
    sW[tid] = w_o;
    sK2[tid] = k2_o;
    sK1[tid] = k1_o;
  }
  static_for<0, 2>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
    const int t = tid + i * nthr;
    if ((i == 0 || NG == 128) && t < F::TWL) sTw[t] = tw_o[i];
  });
  // When the whole grid is one workgroup per CU, the two waves sharing a SIMD
  // belong to this workgroup and would otherwise finish far apart (the older
  // one is issued first whenever both are ready, and the other then runs the
  // rest of its items alone), while the workgroup waits for the later one.
  // With balance each wave lowers its issue priority as it passes quarters
  // of its items, so a wave that falls behind is issued first until it
  // catches up.  With more workgroups than CUs the partner wave belongs to
  // another workgroup and the default (oldest first) order is faster.
  const int wave_items =  // of its first group
      __builtin_amdgcn_readfirstlane((nitem - wave * GPW + ngrp - 1) / ngrp);
  lds_barrier();  // sW and sTw visible
  // NG = 32 reads one of its two sets of twiddles where they are used (both fill the
  // registers: 9.3 against 10.0 us at 16 k-points, 16 bands); read there at NG = 16,
  // whose 122 registers hold both, they cost many passes 3 to 12 % (NG = 16, 140
  // k-points, 8 bands: 46.1 against 43.1 us)
  F fft;
  fft.init_lds(sTw, l);
  auto fwd = [&](zd (&v)[R]) { fft.fwd(v, T, l); };
  auto inv = [&](zd (&v)[R]) {
    if constexpr (NG == 32 && !ONE)
      fft.inv_t(v, T, l, [&](int g0) { return fft.fw[g0]; },
                [&](int i) { return sTw[NG + l * R + i]; });
    else
      fft.inv(v, T, l);
  };

  int it = 0;
  auto pass = [&](auto lastc) {
    constexpr bool last = decltype(lastc)::value;
    if constexpr (ONE) {
      if (it > 0) fetch_v(cq);
    }
    if (balance) set_wave_priority(3 - (4 * it) / wave_items);
    zd uq[R], v[R];
    static_for<0, R>([&](auto mc) {
      constexpr int m = decltype(mc)::value;
      uq[m] = un[m];
    });
    if constexpr (!last) {
      // (a group without a next item re-reads its own)
      if (grp + (it + 1) * ngrp < nitem) {
        cq += dq;
        cj += dj;
        if (cj >= a.nbocc) {
          cj -= a.nbocc;
          ++cq;
        }
      }
      fetch_u(cq, cj);
    }
    static_for<0, R>([&](auto mc) {
      constexpr int m = decltype(mc)::value;
      v[m] = zmulc(sW[L * m + l], uq[m]);
      den[m] += zabs2(uq[m]);
    });
    fwd(v);
    static_for<0, R>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      v[j] = zscal(v[j], vtr[j]);
    });
    if constexpr (!last && !ONE) fetch_v(cq);
    inv(v);
    static_for<0, R>([&](auto mc) {
      constexpr int m = decltype(mc)::value;
      acc[m].x = fma(v[m].x, uq[m].x, acc[m].x);
      acc[m].x = fma(-v[m].y, uq[m].y, acc[m].x);
      acc[m].y = fma(v[m].x, uq[m].y, acc[m].y);
      acc[m].y = fma(v[m].y, uq[m].x, acc[m].y);
    });
  };
  if constexpr (ONE) {
    for (; grp + it * ngrp < nitem; ++it) pass(std::false_type{});
  } else {
    for (; it + 1 < wave_items; ++it) pass(std::false_type{});
    if (grp + it * ngrp < nitem) pass(std::true_type{});
  }
  if (balance) set_wave_priority(0);

  // field values of this launch: read only now, so that they do not hold back
  // the operand loads of the pair loop, and looked at only when they are used
  const int step = step0 + jstep;
  const double* none = reinterpret_cast<const double*>(a.tw);
  const int fi = fields ? step : 0;
  const double At = gload((fields ? Aarr : none) + fi), Aav = gload((fields ? Aavearr : none) + fi),
               Ap = gload((fields ? Aarr : none) + (fi > 0 ? fi - 1 : 0));
  auto akin = [&] {  // stage 1: A(it-1) as in RT_RK4_ubk
    return !fields ? a.A
           : mode == M_S1 ? 2.0 * Aav - At
           : mode == M_S2 || mode == M_S3 ? Aav : At;
  };
  auto aobs = [&] {  // of the stage input, or (M_OBS) after the step
    return !fields ? a.Aobs : mode != M_S1 ? At : step > 0 ? Ap : 0.0;
  };

  // epilogue operands: loaded now, used after the reduction (whose barriers
  // order LDS only, so these loads stay in flight meanwhile)
  zd u0v = mk(0.0, 0.0), ksv = mk(0.0, 0.0);
  double vionv = 0.0, khv = 0.0, v0 = 0.0;
  if (tid < NG) {
    if constexpr (!TE) khv = gload(kc + tid);
    if constexpr (!TE && NG >= 64) v0 = gload(vhg + lane0);  // vCG(0)/NG
    vionv = gload(vion + tid);
    if (mode >= M_S1 && mode <= M_S4) {
      u0v = gload(u0 + o);
      if (mode != M_S1) ksv = gload(ksum + o);
    }
  }

  // ---- one reduction over all groups (fixed order) of V_F w and the density
  // sum; the sums land in sVF and, right after it, sRho (sum |u|^2, without
  // occ) ----
  {
    // the groups of a wave are summed in registers (values padded with zeros
    // to a multiple of the group count), then the nw wave partials through
    // LDS, each parked in its own wave's slots as [re | im | rho][x]
    constexpr int NV = (3 * R + GPW - 1) / GPW * GPW, VF = NV / GPW;
    double v3[NV];
    static_for<0, R>([&](auto mc) {
      constexpr int m = decltype(mc)::value;
      v3[3 * m] = acc[m].x;
      v3[3 * m + 1] = acc[m].y;
      v3[3 * m + 2] = den[m];
    });
    static_for<3 * R, NV>([&](auto kc) { v3[decltype(kc)::value] = 0.0; });
    wave_reduce_scatter<L, NV>(v3);
    double* wp = reinterpret_cast<double*>(smem + (size_t)wave * GPW * SSZ);
    static_for<0, VF>([&](auto kc) {
      constexpr int k = decltype(kc)::value;
      const int vi = k + VF * gw;  // value 3 m + c of the groups, m = point
      if (vi < 3 * R) wp[(vi % 3) * NG + L * (vi / 3) + l] = v3[k];
    });
    lds_barrier();
    for (int t = tid; t < 3 * NG; t += nthr) {
      const int c = t / NG, x = t - c * NG;
      const double sum = ordered_sum(reinterpret_cast<const double*>(smem) + t, 2 * GPW * SSZ, nw);
      if (c < 2)
        reinterpret_cast<double*>(sVF)[2 * x + c] = sum;
      else
        sRho[x] = sum;
    }
  }
  if (!TE && tid < NG) sKH[tid] = khv;
  lds_barrier();  // V_F w and rho complete; the slot area is free

  const bool want_obs = (mode == M_S1 || mode == M_OBS) && obs != nullptr;
  if constexpr (TE) {
    // ---- one transform round trip each: group 0 of the first wave on rho,
    // group 1 on w (the wave's other groups repeat group 1's work and store
    // nothing); group 1 also sums Ekin and J of the row by Parseval ----
    if (wave == 0) {
      const double kA = kxv + akin(), kAo = kxv + aobs();
      zd v[R];
      static_for<0, R>([&](auto mc) {
        constexpr int m = decltype(mc)::value;
        const int x = L * m + l;
        v[m] = gw == 0 ? mk(sRho[x], 0.0) : sW[x];
      });
      fwd(v);
      double ek = 0.0, jc = 0.0;
      static_for<0, R>([&](auto jc_) {
        constexpr int j = decltype(jc_)::value;
        const double G = gvalue(F::gindex(l, j), NG, a.bx);
        if (want_obs) {
          const double p2 = zabs2(v[j]), q = G + kAo;
          ek = fma(0.5 * q * q, p2, ek);
          jc = fma(q, p2, jc);
        }
        const double q = G + kA;
        v[j] = zscal(v[j], gw == 0 ? sK2[l * R + j] : (0.5 / NG) * q * q);
      });
      inv(v);
      static_for<0, R>([&](auto mc) {
        constexpr int m = decltype(mc)::value;
        const int x = L * m + l;
        if (gw == 0) sKH[x] = occ * v[m].x;  // the density sum holds sum |u|^2
        else if (gw == 1) sK1[x] = v[m];
      });
      if (want_obs) {
#pragma unroll
        for (int off = 1; off < L; off <<= 1) {
          ek += __shfl_xor(ek, off);
          jc += __shfl_xor(jc, off);
        }
        if (gw == 1 && l == 0) {
          sRed[0] = ek / NG;
          sRed[1] = jc / NG;
        }
      }
    }
  } else {
    // ---- circulant products K_H * rho, K_2 * w, K_1 * w: thread (x, y) takes
    // the B x B points x, x + XN, ... and y, y + XN, ... (XN = NG/B), between
    // which only B differences mod NG occur, so B reads of each operand serve
    // B^2 products (one read each per product: the LDS bandwidth, 0.85 us at
    // NG = 64, now 0.4).  The threads of a wave with the same x add theirs in
    // registers; the sums are parked in the slot area (free after the
    // reduction) as [wave][value][x], and thread x adds those in order.  From
    // NG = 64 the products are of the differences to the value at x (the kernels
    // sum to their terms at G = 0: none in K_2 and K_1; K_H's, zero unless a
    // caller's table has one, is added in the epilogue): K_2 is hundreds near
    // d = 0 and alternates, and what cancels in its sum costs digits that the
    // transforms keep (kinetic energy at NG = 128: 4e-15 of it, 2e-16 with the
    // differences or by Parseval; H w 3e-14 and 4e-15).  They cost 0.1 us with
    // four waves, 0.3 with one ----
    static_assert(F::gindex(0, 0) == 0, "vhg[0] is the term at G = 0");
    constexpr bool DIFF = NG >= 64;
    constexpr int B = CB, XN = NG / B, NV = (5 * B * XN + 63) / 64 * 64 / XN, VF = NV * XN / 64;
    const int xr = tid % XN;
    if (wave < CW) {
      double s5[NV];
      static_for<0, NV>([&](auto kc) { s5[decltype(kc)::value] = 0.0; });
      zd wx[B];
      double rx[B];
      if constexpr (DIFF) {
        static_for<0, B>([&](auto ic) {
          constexpr int i = decltype(ic)::value;
          wx[i] = sW[xr + i * XN];
          rx[i] = sRho[xr + i * XN];
        });
      }
      for (int yr = tid / XN; yr < XN; yr += nthr / XN) {
        double kh[B], k2[B];
        zd k1[B];
        static_for<0, B>([&](auto ic) {
          constexpr int i = decltype(ic)::value;
          const int d = (xr - yr + i * XN) & (NG - 1);
          kh[i] = sKH[d];
          k2[i] = sK2[d];
          k1[i] = sK1[d];
        });
        static_for<0, B>([&](auto jc) {
          constexpr int jj = decltype(jc)::value;
          const zd wy = sW[yr + jj * XN];
          const double ry = sRho[yr + jj * XN];
          static_for<0, B>([&](auto ic) {
            constexpr int i = decltype(ic)::value, m = (i - jj + B) % B;
            zd d = wy;
            double r = ry;
            if constexpr (DIFF) {
              d = zsub(wy, wx[i]);
              r = ry - rx[i];
            }
            s5[i] = fma(kh[m], r, s5[i]);
            s5[B + i] = fma(k2[m], d.x, s5[B + i]);
            s5[2 * B + i] = fma(k2[m], d.y, s5[2 * B + i]);
            s5[3 * B + i] = fma(k1[m].x, d.x, s5[3 * B + i]);
            s5[3 * B + i] = fma(-k1[m].y, d.y, s5[3 * B + i]);
            s5[4 * B + i] = fma(k1[m].x, d.y, s5[4 * B + i]);
            s5[4 * B + i] = fma(k1[m].y, d.x, s5[4 * B + i]);
          });
        });
      }
      wave_reduce_scatter<XN, NV>(s5);
      double* q = reinterpret_cast<double*>(smem) + 5 * NG * (size_t)wave + xr;
      static_for<0, VF>([&](auto kc) {
        constexpr int k = decltype(kc)::value;
        const int vi = k + VF * (lane / XN);
        if (vi < 5 * B) q[vi * XN] = s5[k];
      });
    }
  }
  lds_barrier();

  // ---- epilogue: H w and the mode-specific update ----
  const int np = nw < CW ? nw : CW;  // circulant partials
  if (tid < NG) {
    const zd wv = sW[tid];
    const zd vf = sVF[tid];
    double vh, ekt = 0.0, jt = 0.0;  // per-point Ekin and J terms (circulant form)
    zd tw;
    if constexpr (TE) {
      vh = sKH[tid];
      tw = sK1[tid];
    } else {
      const double* cp = reinterpret_cast<const double*>(smem);
      zd c2 = mk(0.0, 0.0), c1 = mk(0.0, 0.0);
      vh = 0.0;
#pragma unroll 4
      for (int p = 0; p < np; ++p) {
        const double* q = cp + 5 * NG * (size_t)p + tid;
        vh += q[0];
        c2.x += q[NG];
        c2.y += q[2 * NG];
        c1.x += q[3 * NG];
        c1.y += q[4 * NG];
      }
      if constexpr (NG >= 64) vh = fma(NG * v0, sRho[tid], vh);
      vh *= occ;  // the density sum holds sum |u|^2
      const double kA = kxv + akin();
      // T w = K_2 * w + (k+A) K_1 * w + (k+A)^2/2 w
      tw = mk(c2.x + kA * c1.x + 0.5 * kA * kA * wv.x, c2.y + kA * c1.y + 0.5 * kA * kA * wv.y);
      if (want_obs) {
        const double kAo = kxv + aobs();
        const double w2 = zabs2(wv);
        const double wc1 = wv.x * c1.x + wv.y * c1.y;  // Re conj(w) (K_1 * w)
        const double wc2 = wv.x * c2.x + wv.y * c2.y;
        ekt = wc2 + kAo * wc1 + 0.5 * kAo * kAo * w2;
        jt = wc1 + kAo * w2;
      }
    }
    zd h = zadd(tw, zscal(wv, vh + vionv));
    h = zadd(h, vf);
    if (mode == M_HPSI) {
      gstore(out + o, h);
    } else if (mode >= M_S1 && mode <= M_S4) {
      const zd kk = mk(h.y, -h.x);  // -i * H w
      const double hdt = 0.5 * a.dt;
      if (mode == M_S1) {
        if (tape0) gstore(tape0 + o, u0v);
        gstore(ksum + o, kk);
        gstore(unext + o, mk(u0v.x + hdt * kk.x, u0v.y + hdt * kk.y));
      } else if (mode == M_S2 || mode == M_S3) {
        gstore(ksum + o, mk(ksv.x + 2.0 * kk.x, ksv.y + 2.0 * kk.y));
        const double c = (mode == M_S2) ? hdt : a.dt;
        gstore(unext + o, mk(u0v.x + c * kk.x, u0v.y + c * kk.y));
      } else {
        gstore(u0 + o,
               mk(u0v.x + (ksv.x + kk.x) * a.dt / 6.0, u0v.y + (ksv.y + kk.y) * a.dt / 6.0));
      }
    }
    if (want_obs) {
      // per-point terms of Ekin, J (circulant form), Ex (this row) and N,
      // Eion, EH (row 0)
      const double rho = occ * sRho[tid];
      double* st = reinterpret_cast<double*>(smem) + 5 * NG * np;
      st[0 * NG + tid] = ekt;
      st[1 * NG + tid] = jt;
      st[2 * NG + tid] = wv.x * vf.x + wv.y * vf.y;
      st[3 * NG + tid] = rho;
      st[4 * NG + tid] = vionv * rho;
      st[5 * NG + tid] = vh * rho;
    }
  }
  if (want_obs) {
    // six fixed-order sums over x, one wave each in turn
    const int nv = row == 0 ? 6 : 3;
    lds_barrier();
    const double* st = reinterpret_cast<const double*>(smem) + 5 * NG * np;
    const int slot = !fields ? a.obs_slot : mode == M_S1 ? step : step + 1;
    double* p = obs + (size_t)slot * obs_stride;
    const double occr = ib < a.nbocc ? occ : 0.0;
    for (int v = wave; v < nv; v += nw) {
      double s = 0.0;
      static_for<0, (NG + 63) / 64>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        if (lane + 64 * i < NG) s += st[v * NG + 64 * i + lane];
      });
      s = wave_sum(s);
      if constexpr (TE) {  // Ekin and J from the transform of w
        if (v < 2) s = sRed[v];
      }
      s *= v < 3 ? occr : v == 5 ? 0.5 : 1.0;
      if (v != 1) s *= a.dv;
      if (lane == 0) gstore(p + (v < 3 ? 3 * row : 3 * nbw * nk - 3) + v, s);
    }
  }
}

// d0 = the first n elements of src, d1 = the next m - n.
__global__ void __launch_bounds__(256) stage_kernel(const zd* src, zd* d0, zd* d1, long n,
                                                    long m) {
  const long i = blockIdx.x * 256L + threadIdx.x;
  if (i < m) gstore(i < n ? d0 + i : d1 + (i - n), gload(src + i));
}

// Twiddle tables of GroupFFT<NG> (2*NG complex).
template <int NG>
__global__ void twiddle_kernel(zd* tw) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < 2 * NG) tw[i] = GroupFFT<NG>::table_value(i);
}

// Compensated (Neumaier) sum: the rounding error of every addition is kept in
// c, so the result carries about one rounding of the total instead of one per
// term.  The energy objective of the adjoint is a difference of two such
// totals, and its finite-difference check divides that difference by h.
struct CompSum {
  double s = 0.0, c = 0.0;
  __device__ __forceinline__ void add(double x) {
    const double t = s + x;
    c += fabs(s) >= fabs(x) ? (s - t) + x : (x - t) + s;
    s = t;
  }
  __device__ __forceinline__ double value() const { return s + c; }
};

// Adds the sums of the first n lanes of a wave (the others' are zero), compensated
// and in a fixed order; M sums at a time, whose exchanges overlap; in lane 0.
template <int M>
__device__ __forceinline__ void comp_wave_sum(CompSum (&c)[M], int n) {
  const int lane = threadIdx.x & 63;
  for (int off = 1; off < 64 && off < n; off <<= 1) {
    static_for<0, M>([&](auto mc) {
      constexpr int m = decltype(mc)::value;
      const double os = __shfl_xor(c[m].s, off), oc = __shfl_xor(c[m].c, off);
      // the same pair of operands in both lanes of the exchange
      const double lo = (lane & off) ? os : c[m].s, hi = (lane & off) ? c[m].s : os;
      CompSum r;
      r.add(lo);
      r.add(hi);
      r.c += c[m].c + oc;
      c[m] = r;
    });
  }
}

// Sums the per-row partials of one observables slot p (rows rows) into
// (Etot, N, J, Ekin, Eion, EH, Ex), src/Functions.f90:74-91 and :289-318; one
// wave per slot, rows lane, lane + 64, ... of a lane first (one thread per slot
// took 78 us for 256 rows, one wave 5 us; four rows need two of the six exchanges
// of the lanes' sums: tdhf_observables 31.8 us, 33.0 with all six one by one, 32.3
// with one thread).
__device__ __forceinline__ void obs_reduce_slot(const double* p, int rows, double dv, double vcell,
                                                double* o) {
  const int lane = threadIdx.x & 63;
  CompSum c[3];
  for (int r = lane; r < rows; r += 64) {
    c[0].add(p[3 * r + 0]);
    c[1].add(p[3 * r + 1]);
    c[2].add(p[3 * r + 2]);
  }
  comp_wave_sum(c, rows);
  const CompSum &ek = c[0], &jj = c[1], &ex = c[2];
  if (lane != 0) return;
  const double n = p[3 * rows + 0], ei = p[3 * rows + 1], eh = p[3 * rows + 2];
  CompSum et;
  et.add(ek.s);
  et.add(ei);
  et.add(eh);
  et.add(0.5 * ex.s);
  et.add(ek.c);
  et.add(0.5 * ex.c);
  o[0] = et.value();
  o[1] = n;
  o[2] = -(jj.value() * dv / vcell);
  o[3] = ek.value();
  o[4] = ei;
  o[5] = eh;
  o[6] = 0.5 * ex.value();
}

// Four waves (slots) per workgroup.
__global__ void __launch_bounds__(256) obs_reduce_kernel(const double* obs, int stride, int rows,
                                                         int nslots, double dv, double vcell,
                                                         double* out) {
  const int s = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (s >= nslots) return;
  obs_reduce_slot(obs + (size_t)s * stride, rows, dv, vcell, out + (size_t)7 * s);
}

// Batched variant: one wave per (trajectory, slot); out[(t*nslots + s)*7].
__global__ void __launch_bounds__(256) obs_reduce_batch_kernel(const TrajDesc* td, int ntraj,
                                                               int nb, int nslots, double dv,
                                                               double vcell, double* out) {
  const int i = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (i >= ntraj * nslots) return;
  const int t = i / nslots, s = i - t * nslots;
  obs_reduce_slot(td[t].obs + (size_t)s * td[t].obs_stride, nb * td[t].nk, dv, vcell,
                  out + (size_t)7 * i);
}

__global__ void step_advance_kernel(int* step_base, int by) {
  if (threadIdx.x == 0 && blockIdx.x == 0) *step_base += by;
}

__global__ void step_set_kernel(int* step_base, int value) {
  if (threadIdx.x == 0 && blockIdx.x == 0) *step_base = value;
}

// k_vCk (src/Functions.f90:33-52) for a list of n arguments: four per workgroup,
// the nsteps trapezoid terms split over the threads and summed by a fixed-shape
// tree (deterministic).  Bound by FP64 operations (the cosine of every term), so
// each end of the steps is evaluated once and its 1/sqrt serves four arguments:
// a context of NG=128, NK=128 is made in 24 ms (59 with both ends of every step
// for one argument at a time).
constexpr int kVckArgs = 4;
__global__ void __launch_bounds__(256) kvck_kernel(const double* q, int n, double dx, long nsteps,
                                                   double* out) {
  __shared__ double red[kVckArgs][256];
  const int a0 = blockIdx.x * kVckArgs, t = threadIdx.x;
  double k[kVckArgs], s[kVckArgs];
  static_for<0, kVckArgs>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
    k[i] = q[a0 + i < n ? a0 + i : n - 1];
    s[i] = 0.0;
  });
  for (long ix = t; ix <= nsteps; ix += 256) {
    const double x = (double)ix * dx;
    const double r = (ix == 0 || ix == nsteps ? 0.5 : 1.0) / sqrt(x * x + 1.0);
    static_for<0, kVckArgs>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      s[i] += cos(k[i] * x) * r;
    });
  }
  static_for<0, kVckArgs>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
    red[i][t] = s[i];
  });
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if (t < h)
      static_for<0, kVckArgs>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        red[i][t] += red[i][t + h];
      });
    __syncthreads();
  }
  if (t < kVckArgs && a0 + t < n) out[a0 + t] = nsteps > 0 ? 2.0 * red[t][0] * dx : 0.0;
}

// Rearranges a raw table t[d*NG + g] into the G layout of GroupFFT<NG>,
// scaled: out[d*NG + l*R + j] = scale * t[d*NG + gindex(l,j)].
template <int NG>
__global__ void relayout_kernel(const double* t, int nrows, double scale, double* out) {
  using F = GroupFFT<NG>;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nrows * NG) return;
  const int d = i / NG, r = i - d * NG;
  const int l = r / F::R, j = r - l * F::R;
  out[i] = scale * t[(size_t)d * NG + F::gindex(l, j)];
}

// Prep_periodic_ion_potential (src/Prep_periodic_ion_potential.f90:10-20);
// one workgroup of NG threads.
__global__ void ion_kernel(int ng, int nk, double ax, int nion, const double* z,
                           const double* alpha, const double* rion, double* vion) {
  __shared__ double red[128];
  const int x = threadIdx.x;
  double v = 0.0;
  if (x < ng) {
    const double rx = (double)x / (double)ng * ax;
    for (int ii = 0; ii < nion; ++ii)
      for (int icell = -4 * nk; icell <= 4 * nk; ++icell) {
        const double dist = fabs(rx - ax * rion[ii] - ax * (double)icell);
        v = v - z[ii] / sqrt(dist * dist + alpha[ii] * alpha[ii]);
      }
    red[x] = v;
  }
  __syncthreads();
  if (x == 0) {
    double top = red[0];
    for (int i = 1; i < ng; ++i) top = red[i] > top ? red[i] : top;
    red[127] = top;
  }
  __syncthreads();
  const double top = red[127];
  __syncthreads();
  if (x < ng) vion[x] = v - top;
}

// Gram_Schmidt for more bands than orth_kernel holds in LDS.
// Block-wide deterministic sum over blockDim.x (power of two, <= 128).
__device__ __forceinline__ double block_sum(double v, double* red) {
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

// Gram_Schmidt (src/mATTOHF.f90:134-157): one workgroup (NG threads) per
// k-point, modified Gram-Schmidt with the vcell/NG weight.
__global__ void gram_schmidt_kernel(zd* u, int ng, int nb, double vcell) {
  __shared__ double red[2][128];
  const int ik = blockIdx.x, x = threadIdx.x;
  zd* uk = u + (size_t)ng * nb * ik;
  for (int ib = 0; ib < nb; ++ib) {
    zd ui = uk[(size_t)ng * ib + x];
    for (int ibt = 0; ibt < ib; ++ibt) {
      const zd ut = uk[(size_t)ng * ibt + x];
      double re = block_sum(ut.x * ui.x + ut.y * ui.y, red[0]);
      double im = block_sum(ut.x * ui.y - ut.y * ui.x, red[1]);
      re = re * vcell / (double)ng;
      im = im * vcell / (double)ng;
      ui = mk(ui.x - (ut.x * re - ut.y * im), ui.y - (ut.x * im + ut.y * re));
    }
    double s = block_sum(ui.x * ui.x + ui.y * ui.y, red[0]);
    s = s * vcell / (double)ng;
    const double r = sqrt(s);
    ui = mk(ui.x / r, ui.y / r);
    uk[(size_t)ng * ib + x] = ui;
    __syncthreads();
  }
}

}  // namespace tdhf
