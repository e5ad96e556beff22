// Chirp z-transform (Bluestein) propagation: CZT / VCZT / high-NA VCZT and
// their adjoints, plain FP32 form.
//
// Reference: Bluestein_method / compute_fft (xlumina/wave_optics.py:385-460),
// CZT_jit (:333-357), CZT_for_high_NA_jit (:359-371), VCZT_jit
// (vectorized_optics.py:375-384), VCZT_objective_lens
// (optical_elements.py:600-638).  Per axis the reference computes
//   out_k = post_k * sum_j g[m + k - j] * pre_j * x_j,   k < M, j < m,
// by a length-np2 circular convolution, with
//   pre_j  = A^{-j} W^{j^2/2},  g_s = W^{-(s-m+1)^2/2} (s < m+M; the reference's
//   table lacks s = m+M-1 when M >= m), post_k = W^{k^2/2} e^{-i2pi l_k(1/2-m/2)/Dm}.
// That is a Toeplitz product out_k = post_k sum_j gamma(k - j) pre_j x_j with the
// lag kernel gamma(d) = g[m + d]; the adjoint axis has pre' = conj(post),
// post' = conj(pre), gamma'(d) = conj(g[m - d]).  Here the kernel is laid out
// on the circle of length Q >= m + M - 1 by lag (lag d at index d mod Q), so
// the outputs are the first M samples of the inverse transform whatever the
// direction.  When the input and the output each fit in half the (power-of-
// two) length, the first forward pass skips the zero upper half of its
// inputs and the last inverse pass forms only the lower half of its outputs.
// The tables are generated on the device with float64 phases
// (czt_setup_kernel); the FFT of the kernel is stored pre-divided by Q.
//
// The 2-D transform is separable (K_y E K_x^T), so the row pass runs along x on
// the row-major input (contiguous loads) and writes a 4x4-tiled intermediate
// ordered [x-output group][row group]; the column pass reads it back column-
// contiguously, runs the y axis and applies the output-plane factor.
#pragma once
#include "fft.h"
#include "fftio.h"
#include "masks.h"
#include "rs.h"
#include "pre.h"

namespace xl {

enum { PRE_NONE = 0, PRE_RS = 1, PRE_HNA = 2, PRE_CONJ_RS = 3, PRE_CONST = 4 };
enum { POST_NONE = 0, POST_RS = 1, POST_CONST = 2, POST_CONJ_RS = 3 };

struct CztAxis {
  int lin, lout, zl, q;   // zl: zero-half first / last passes (lin, lout <= q/2, q a power of two)
  const float2* pre;   // lin
  const float2* gf;    // q, FFT of the kernel divided by q
  const float2* post;  // lout
};

struct CztArgs {
  const float2* in;
  int64_t in_cs;
  int nin;
  float2* out;
  int64_t out_cs;
  float2* t;           // intermediate, per component rin4 x lout4 in 4x4 tiles (czt_tidx)
  int rin, ncomp;      // input rows (cols = ax.lin)
  int pre_mode, post_mode, ez_mode;
  const double* px;    // grid of the input plane (pre-op)
  const double* py;
  const double* qx;    // grid of the output plane (post-op)
  const double* qy;
  double z, k;
  float2 cte;          // constant factor (forward) or its conjugate (adjoint)
  double hna_radius, hna_f, hna_stm2;
  MaskArgs mask;
  CztAxis ax, ay;
  int64_t in_bs, out_bs, t_bs, mask_bs;   // batch strides (blockIdx.y / .z selects the member)
  int rin4;            // rin rounded up to a multiple of 4
  int64_t t_cs;        // component stride of the intermediate (rin4 * lout4)
  // Optional tables of the input-plane factor (rin x ax.lin) and the
  // output-plane factor (ay.lout x ax.lout), shared by a batch: built once by
  // czt_ftab_kernel instead of per member in float64.
  const float2* ftab;
  const float2* f0tab;
};

// Offset of (row, k) in the tiled intermediate: 4 rows x 4 outputs per 128-byte
// tile, tiles ordered [k / 4][row / 4], so the column pass reads whole lines.
__device__ __forceinline__ int64_t czt_tidx(int rin4, int row, int k) {
  return ((int64_t)(k >> 2) * (rin4 >> 2) + (row >> 2)) * 16 + (row & 3) * 4 + (k & 3);
}

// The arguments of batch member b: inputs, outputs, intermediate and
// per-pixel mask parameters offset by their batch strides.
__device__ __forceinline__ CztArgs czt_member(const CztArgs& a0, int b) {
  CztArgs a = a0;
  a.in += b * a0.in_bs;
  a.out += b * a0.out_bs;
  a.t += b * a0.t_bs;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    if (a.mask.st[i].m0) a.mask.st[i].m0 += b * a0.mask_bs;
    if (a.mask.st[i].m1) a.mask.st[i].m1 += b * a0.mask_bs;
  }
  return a;
}

struct CztSetupArgs {
  float2* pre;
  float2* gf;
  float2* post;
  int m, M, q, adjoint;
  double d1_dm;        // D1 / Dm
  double dl_dm;        // Delta / Dm,  Delta = (D2 - D1) / M
  double th_turns;     // angle(W) / (2 pi), principal branch
};

// One workgroup of q/16 threads builds one axis' tables (block b takes args b).
struct CztSetupPair {
  CztSetupArgs ax[2];
};

// Tables of one axis on a block of NT threads: the chirps and the kernel
// (float64 phases, the bulk of the work) on all NT threads, the kernel's FFT
// on the first Q/16 (the others only join its barriers).
template <int Q, int NT>
__device__ __forceinline__ void czt_setup_body(const CztSetupArgs& a, float2* s, int t) {
  constexpr int TPF = Q / 16;
  static_assert(NT >= TPF, "the FFT needs Q/16 threads");
  const double th = a.th_turns;
  const double shift = 0.5 - 0.5 * a.m;
  // forward tables
  auto pre_f = [&](int j) {   // A^{-j} W^{j^2/2}
    const double jj = (double)j;
    return expi_turns(-jj * a.d1_dm + th * 0.5 * jj * jj);
  };
  auto post_f = [&](int k) {  // W^{k^2/2} e^{-i 2pi l_k (1/2 - m/2)/Dm}
    const double kk = (double)k;
    return expi_turns(th * 0.5 * kk * kk - (a.d1_dm + kk * a.dl_dm) * shift);
  };
  auto g_f = [&](int sidx) -> float2 {   // W^{-(s-m+1)^2/2}, s < m+M, last tap dropped if M >= m
    if (sidx < 0 || sidx >= a.m + a.M) return make_float2(0.f, 0.f);
    if (a.M >= a.m && sidx == a.m + a.M - 1) return make_float2(0.f, 0.f);
    const double u = (double)(sidx - a.m + 1);
    return expi_turns(-th * 0.5 * u * u);
  };
  if (!a.adjoint) {
    for (int j = t; j < a.m; j += NT) a.pre[j] = pre_f(j);
    for (int k = t; k < a.M; k += NT) a.post[k] = post_f(k);
  } else {
    for (int k = t; k < a.M; k += NT) a.pre[k] = conjf2(post_f(k));
    for (int j = t; j < a.m; j += NT) a.post[j] = conjf2(pre_f(j));
  }
  // lag d = k - j in [-(lin-1), lout-1] at index d mod Q (Q >= lin + lout - 1)
  const int lin = a.adjoint ? a.M : a.m, lout = a.adjoint ? a.m : a.M;
  for (int i = t; i < Q; i += NT) {
    const int d = i < lout ? i : (i > Q - lin ? i - Q : INT_MIN);
    float2 v = make_float2(0.f, 0.f);
    if (d != INT_MIN) v = a.adjoint ? conjf2(g_f(a.m - d)) : g_f(a.m + d);
    s[lpad(i)] = v;
  }
  __syncthreads();
  fft_lds<Q, TPF, false, 0, (NT > TPF)>(s, t);
  const float iq = 1.0f / (float)Q;
  for (int i = t; i < Q; i += NT) a.gf[i] = s[lpad(i)] * iq;
}

// Threads per set-up block: the float64 table work spreads over 1024 threads
// (the block runs alone on its CU; one or two such blocks make up the launch).
constexpr int CZT_SETUP_THREADS = 1024;

template <int Q>
__global__ __launch_bounds__(CZT_SETUP_THREADS) void czt_setup_kernel(CztSetupPair pair) {
  __shared__ float2 s[LdsLen<Q>::value];
  czt_setup_body<Q, CZT_SETUP_THREADS>(pair.ax[blockIdx.x], s, threadIdx.x);
}

// Both axes in one launch when their lengths differ (block 0: QA, block 1: QB).
template <int QA, int QB>
__global__ __launch_bounds__(CZT_SETUP_THREADS) void czt_setup2_kernel(CztSetupPair pair) {
  constexpr int QM = QA > QB ? QA : QB;
  __shared__ float2 s[LdsLen<QM>::value];
  if (blockIdx.x == 0) czt_setup_body<QA, CZT_SETUP_THREADS>(pair.ax[0], s, threadIdx.x);
  else czt_setup_body<QB, CZT_SETUP_THREADS>(pair.ax[1], s, threadIdx.x);
}

// Pre-op families the row kernel is specialised for.
enum { PREK_SIMPLE = 0, PREK_F = 1, PREK_HNA = 2 };

// All pre-op components of a pixel's masked field (e0, e1, e2) at input-plane
// coordinates (X, Y): Ez or the lens map, and the plane factor (fpix for
// PREK_F, cte for PRE_CONST).
template <int K>
__device__ __forceinline__ void czt_pre_compute(const CztArgs& a, float2 e0, float2 e1, float2 e2, double X, double Y,
                                                float2 fpix, float2 (&v)[3]) {
  if constexpr (K == PREK_HNA) {
    // optical_elements.py:528-594: theta = rho/f, phi = atan2(Y, X), Richards-Wolf map
    float A[3][2];
    hna_map(X, Y, a.hna_radius, a.hna_f, a.hna_stm2, A);
#pragma unroll
    for (int c = 0; c < 3; ++c) v[c] = c_add(c_scale(e0, A[c][0]), c_scale(e1, A[c][1]));
  } else {
    if (a.ez_mode != EZ_NONE) e2 = build_ez(a.ez_mode, e0, e1, X, Y, a.z);
    v[0] = e0;
    v[1] = e1;
    v[2] = e2;
    float2 m = make_float2(1.f, 0.f);
    if constexpr (K == PREK_F) m = fpix;
    else if (a.pre_mode == PRE_CONST) m = a.cte;
#pragma unroll
    for (int c = 0; c < 3; ++c) v[c] = c_mul(v[c], m);
  }
}

// Transfer function of the input plane at (X, Y) (or its conjugate times cte
// for the adjoint).
__device__ __forceinline__ float2 czt_f_at(const CztArgs& a, double X, double Y) {
  float2 h = rs_kernel_value(X, Y, a.z, a.k);
  if (a.pre_mode == PRE_CONJ_RS) h = c_mul(conjf2(h), a.cte);
  return h;
}
__device__ __forceinline__ float2 czt_f_compute(const CztArgs& a, int row, int col) {
  return czt_f_at(a, a.px[col], a.py[row]);
}

// Output-plane factor of element (ky, kx): F0 cte (forward), conj(F0)
// (adjoint), cte, or 1.
__device__ __forceinline__ float2 czt_post_factor(const CztArgs& a, int ky, int kx) {
  if (a.post_mode == POST_RS) return c_mul(rs_kernel_value(a.qx[kx], a.qy[ky], a.z, a.k), a.cte);
  if (a.post_mode == POST_CONJ_RS) return conjf2(rs_kernel_value(a.qx[kx], a.qy[ky], a.z, a.k));
  if (a.post_mode == POST_CONST) return a.cte;
  return make_float2(1.f, 0.f);
}

// Both factor tables of a batched RS-mode CZT: elements first, first + stride, ..
// (planes of up to 4096^2 samples: 32-bit indices, whose division by the row
// length costs a tenth of the 64-bit one).
__device__ __forceinline__ void czt_ftab_body(const CztArgs& a, float2* ftab, float2* f0tab, uint32_t first,
                                              uint32_t stride) {
  const uint32_t lin = a.ax.lin, lout = a.ax.lout, n1 = (uint32_t)a.rin * lin, n2 = (uint32_t)a.ay.lout * lout;
  for (uint32_t e = first; e < n1 + n2; e += stride) {
    if (e < n1) {
      const uint32_t r = e / lin;
      ftab[e] = czt_f_compute(a, (int)r, (int)(e - r * lin));
    } else {
      const uint32_t f = e - n1, r = f / lout;
      f0tab[f] = czt_post_factor(a, (int)r, (int)(f - r * lout));
    }
  }
}
__global__ __launch_bounds__(256) void czt_ftab_kernel(CztArgs a, float2* ftab, float2* f0tab) {
  czt_ftab_body(a, ftab, f0tab, blockIdx.x * 256 + threadIdx.x, gridDim.x * 256);
}

// The axis tables (blocks 0 and 1, both axes at one length) and the factor
// tables (the other blocks) of a batched RS-mode CZT in one launch: the two
// set-up blocks, 6.5 us of latency alone, run beside the others (8 x 1024^2:
// 6.5 + 12 us in two launches, 12.9 in one).
template <int Q>
__global__ __launch_bounds__(CZT_SETUP_THREADS) void czt_setup_ftab_kernel(CztSetupPair pair, CztArgs a, float2* ftab,
                                                                           float2* f0tab) {
  __shared__ float2 s[LdsLen<Q>::value];
  if (blockIdx.x < 2) czt_setup_body<Q, CZT_SETUP_THREADS>(pair.ax[blockIdx.x], s, threadIdx.x);
  else
    czt_ftab_body(a, ftab, f0tab, (blockIdx.x - 2) * CZT_SETUP_THREADS + threadIdx.x,
                  (gridDim.x - 2) * CZT_SETUP_THREADS);
}

// One block per input row: component c runs its FFT on threads
// [c*TPF, (c+1)*TPF) and LDS buffer c; the pre-op of each pixel (masks, Ez,
// transfer function in float64 phase, lens map) is computed once by one
// thread for all components.  The chirp spectrum is applied in registers
// between the forward and inverse chains and only the output window is
// stored, into the tiled intermediate (consecutive rows run on one XCD, so
// the four rows of a tile meet in one L2).  ZL: the input and the output fit
// in half the length (zero-half first pass, lower-half last pass).
template <int Q, bool ZL> struct CztRowsShape {
  // At 1024 and 2048 the three buffers (26 / 52 KB) leave room for 6 / 3
  // blocks of 3 / 6 waves per CU, which a SIMD holds at 5 waves (<= 96 VGPRs);
  // the zero-half forms fit that without spilling.
  static constexpr int WAVES = (ZL && (Q == 1024 || Q == 2048)) ? 5 : 1;
  // Pixels staged per thread at a time, their loads grouped ahead of the
  // pre-ops (measured: 1 -> 3 took the 4f rows from 3.04 to 2.44 ms per step
  // and the VCZT rows from 122 to 111 us; 2 is close behind).
  static constexpr int U = 3;
};

template <int Q, int K, bool ZL>
__global__ __launch_bounds__(3 * Q / 16)
__attribute__((amdgpu_waves_per_eu(CztRowsShape<Q, ZL>::WAVES))) void czt_rows_kernel(CztArgs a0) {
  const CztArgs a = czt_member(a0, blockIdx.y);
  constexpr int TPF = Q / 16, LS = LdsLen<Q>::value;
  using HO = HandOff<Q, TPF>;
  extern __shared__ float2 lds[];
  const int tid = threadIdx.x, nthr = blockDim.x;
  const int f = tid / TPF, t = tid % TPF;
  const int row = xcd_remap(blockIdx.x, gridDim.x);
  const int lin = a.ax.lin, lout = a.ax.lout;
  const int nc = a.ncomp;
  // Staging: the pre-op of each pixel once for all components, U pixels per
  // thread at a time with their loads issued ahead of the pre-ops; columns
  // lin..LIM-1 are the zero padding.
  constexpr int LIM = ZL ? Q / 2 : Q, U = CztRowsShape<Q, ZL>::U;
  // the input-plane grid is read only by the forms that use it
  const bool grid = K == PREK_HNA || (K == PREK_F && !a.ftab) || a.ez_mode != EZ_NONE;
  const bool ftab = K == PREK_F && a.ftab;
  const double Y = grid ? a.py[row] : 0.0;
  for (int c0 = tid; c0 < LIM; c0 += U * nthr) {
    PixRaw raw[U];
    int64_t pix[U];
    double X[U];
    float2 fr[U], pr[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int col = c0 + u * nthr;
      const int cc = col < lin ? col : 0;
      pix[u] = (int64_t)row * lin + cc;
      pr[u] = a.ax.pre[cc];
      X[u] = 0.0;
      fr[u] = make_float2(1.f, 0.f);
    }
    pix_load_n<U>(a.in, a.in_cs, a.nin, a.mask, pix, raw);
    if (grid) {
#pragma unroll
      for (int u = 0; u < U; ++u) X[u] = a.px[pix[u] - (int64_t)row * lin];
    }
    if (ftab) {
#pragma unroll
      for (int u = 0; u < U; ++u) fr[u] = a.ftab[pix[u]];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int col = c0 + u * nthr;
      if (col < LIM) {
        float2 v[3] = {make_float2(0.f, 0.f), make_float2(0.f, 0.f), make_float2(0.f, 0.f)};
        if (col < lin) {
          float2 e0, e1, e2;
          pix_masked(a.mask, raw[u], e0, e1, e2);
          float2 fv = make_float2(1.f, 0.f);
          if constexpr (K == PREK_F) fv = ftab ? fr[u] : czt_f_at(a, X[u], Y);
          czt_pre_compute<K>(a, e0, e1, e2, X[u], Y, fv, v);
#pragma unroll
          for (int c = 0; c < 3; ++c) v[c] = c_mul(v[c], pr[u]);
        }
#pragma unroll
        for (int c = 0; c < 3; ++c)
          if (c < nc) lds[c * LS + lpad(col)] = v[c];
      }
    }
  }
  __syncthreads();
  float2* s = lds + f * LS;
  typename HO::Type u;
  NoIO none;
  fft_forward_to_regs<Q, TPF, SRC_LDS, ZL>(s, t, none, u);
#pragma unroll
  for (int b = 0; b < HO::BPT; ++b)
#pragma unroll
    for (int q = 0; q < HO::R; ++q) u.v[b][q] = cmul(u.v[b][q], a.ax.gf[HO::index(t, b, q)]);
  float2* dst = a.t + (int64_t)f * a.t_cs;
  auto store = [&](int k0, float2 v) {
    const int k = t + k0;
    if (k < lout) dst[czt_tidx(a.rin4, row, k)] = cmul(v, a.ax.post[k]);
  };
  fft_inverse_from_regs<Q, TPF, DST_FN, ZL>(s, t, u, store);
}

// The same pass with one buffer per transform: a row per block of Q/16
// threads, the components transformed one after the other.  Thread t's
// first-pass inputs are the columns t + r Q/16, so it forms the pre-ops of
// exactly its own pixels (8 where the upper half is zero, ZL) and keeps all
// components of them in registers: no staging pass, and a CU holds three or
// four independent blocks where the three-buffer block of a 4096-point row
// runs alone.  MULTI: more than one component.  Used for one component (8 x
// 1024^2 of the 4f systems 95 -> 86 us, 777 -> 301 samples 14.1 -> 12.7 us)
// and for the 4096-point zero-half rows (2048 -> 512, three components, 121 ->
// 104 us: accesses and exchanges alone take 65, transforms and pre-ops 82; it
// needs 168 VGPRs).  At 2048 and below with several components the
// three-buffer block already shares its CU and stays faster (1024^2, HNA rows:
// 33 us against 38 us, whose registers spill).
template <int Q> using CztRows1 = Units<Q, rs_g(Q, 1, 1, 1)>;

template <int Q, int K, bool ZL, bool MULTI>
__global__ __launch_bounds__(CztRows1<Q>::NT, MULTI ? 3 : 4) void czt_rows1_kernel(CztArgs a0) {
  const CztArgs a = czt_member(a0, blockIdx.y);
  using U = CztRows1<Q>;
  constexpr int TPF = U::TPF, H = ZL ? 8 : 16, NC = MULTI ? 3 : 1;
  using HO = HandOff<Q, TPF>;
  static_assert(FftPlan<Q, TPF>::radix(true, 0) == 16, "first pass: one radix-16 butterfly per thread");
  __shared__ float2 lds[U::G * U::LS];
  const int g = U::row_g(threadIdx.x), t = U::row_t(threadIdx.x);
  float2* s = lds + g * U::LS;
  const int row0 = xcd_remap(blockIdx.x, gridDim.x) * U::G, row = row0 + g;
  const int lin = a.ax.lin, lout = a.ax.lout, nc = a.ncomp;
  const bool rowok = row < a.rin;
  // the input-plane grid is read only by the forms that use it
  const bool ftab = K == PREK_F && a.ftab;
  const bool grid = K == PREK_HNA || (K == PREK_F && !ftab) || a.ez_mode != EZ_NONE;
  const uint32_t r0 = rowok ? row : 0, row_at = r0 * lin;
  const double Y = grid ? a.py[r0] : 0.0;
  float2 e[NC][H];
  // PXG pixels at a time: their loads, then their pre-ops (columns beyond lin
  // read the row's last pixel and are zeroed)
  constexpr int PXG = 4;
#pragma unroll
  for (int r1 = 0; r1 < H; r1 += PXG) {
    PixRaw raw[PXG];
    uint32_t pix[PXG], cc[PXG];
    float2 fr[PXG], pr[PXG];
    double X[PXG];
#pragma unroll
    for (int u = 0; u < PXG; ++u) {
      cc[u] = min(t + (r1 + u) * TPF, lin - 1);
      pix[u] = row_at + cc[u];
      fr[u] = make_float2(1.f, 0.f);
      X[u] = 0.0;
    }
    pix_load_n<PXG>(a.in, a.in_cs, MULTI ? a.nin : 1, a.mask, pix, raw);
    if (grid) {
#pragma unroll
      for (int u = 0; u < PXG; ++u) X[u] = at32(a.px, cc[u]);
    }
    if (ftab) {
#pragma unroll
      for (int u = 0; u < PXG; ++u) fr[u] = at32(a.ftab, pix[u]);
    }
#pragma unroll
    for (int u = 0; u < PXG; ++u) pr[u] = at32(a.ax.pre, cc[u]);
#pragma unroll
    for (int u = 0; u < PXG; ++u) {
      const int r = r1 + u, col = t + r * TPF;
      float2 v[3] = {make_float2(0.f, 0.f), make_float2(0.f, 0.f), make_float2(0.f, 0.f)};
      if (rowok && col < lin) {
        float2 e0, e1, e2;
        pix_masked(a.mask, raw[u], e0, e1, e2);
        float2 fv = make_float2(1.f, 0.f);
        if constexpr (K == PREK_F) fv = ftab ? fr[u] : czt_f_at(a, X[u], Y);
        czt_pre_compute<K>(a, e0, e1, e2, X[u], Y, fv, v);
#pragma unroll
        for (int c = 0; c < 3; ++c) v[c] = c_mul(v[c], pr[u]);
      }
#pragma unroll
      for (int c = 0; c < NC; ++c) e[c][r] = v[c];
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  // roundings end here (the first pass's sums take the products as they are)
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int r = 0; r < H; ++r) asm volatile("" : "+v"(e[c][r].x), "+v"(e[c][r].y));
  const uint32_t lane = (uint32_t)((t >> 2) * (a.rin4 >> 2) + (g >> 2)) * 16 + (g & 3) * 4 + (t & 3);
  NoIO none;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    if (c >= nc) break;
    Regs<1, 16> in;
    typename HO::Type u;
#pragma unroll
    for (int r = 0; r < 16; ++r) in.v[0][r] = r < H ? e[c][r < H ? r : 0] : make_float2(0.f, 0.f);
    chain_io<Q, TPF, false, true, 0, SRC_REG, DST_REG, ZL, false>(s, t, none, none, in, u);
#pragma unroll
    for (int b = 0; b < HO::BPT; ++b)
#pragma unroll
      for (int q = 0; q < HO::R; ++q) u.v[b][q] = cmul(u.v[b][q], ld_at(a.ax.gf + HO::koff(b, q), t));
    float2* dst = a.t + (int64_t)c * a.t_cs + (row0 >> 2) * 16 + (row0 & 3) * 4;
    auto store = [&](int k, float2 v) {
      if (rowok && t + k < lout) st_at(dst + (int64_t)(k >> 2) * (a.rin4 >> 2) * 16, lane, cmul(v, ld_at(a.ax.post + k, t)));
    };
    fft_inverse_from_regs<Q, TPF, DST_FN, ZL>(s, t, u, store);
  }
}

// Column pass of the 3 * 2^k lengths.  Per block CPB output columns of the x
// axis (one per thread group) of one component: the columns of the tiled
// intermediate feed the first pass, the chirp spectrum is applied in
// registers, and only the output window is stored with the output-plane
// factor.  A 128 B tile line holds four columns: the CPB groups of a block
// (and at CPB = 2 the neighbouring block, kept on the same XCD) share it.
template <int Q> struct CztColsShape {
  static constexpr int CPB = Q >= 3072 ? 2 : 4;   // columns per block (more blocks at 3072)
  // At 3072 three blocks (52 KB of LDS, 6 waves each) fit a CU when a SIMD
  // holds 5 waves, i.e. at most 96 VGPRs; unbounded, the compiler takes 112.
  static constexpr int WAVES = Q == 3072 ? 5 : 1;
};

template <int Q>
__global__ __launch_bounds__(CztColsShape<Q>::CPB * Q / 16)
__attribute__((amdgpu_waves_per_eu(CztColsShape<Q>::WAVES))) void czt_cols_kernel(CztArgs a0) {
  const CztArgs a = czt_member(a0, blockIdx.z);
  constexpr int TPF = Q / 16, LS = LdsLen<Q>::value;
  constexpr int CPB = CztColsShape<Q>::CPB;
  using HO = HandOff<Q, TPF>;
  __shared__ float2 lds[CPB * LS];
  const int tid = threadIdx.x, f = tid / TPF, t = tid % TPF;
  float2* s = lds + f * LS;
  const int og = xcd_remap(blockIdx.x, gridDim.x);
  const int c = blockIdx.y;
  const int lout_x = a.ax.lout;
  const int kx = og * CPB + f;
  const bool colok = kx < lout_x;
  const int lin = a.ay.lin, lout = a.ay.lout;
  const float2* src = a.t + (int64_t)c * a.t_cs;
  typename HO::Type u;
  auto load = [&](int k0) -> float2 {
    const int r = t + k0;
    return (colok && r < lin) ? cmul(src[czt_tidx(a.rin4, r, kx)], a.ay.pre[r]) : make_float2(0.f, 0.f);
  };
  // (twiddle bases loaded at each pass: prefetched, they cost the 5-wave bound)
  fft_forward_to_regs<Q, TPF, SRC_FN, false, false>(s, t, load, u);
#pragma unroll
  for (int b = 0; b < HO::BPT; ++b)
#pragma unroll
    for (int q = 0; q < HO::R; ++q) u.v[b][q] = cmul(u.v[b][q], a.ay.gf[HO::index(t, b, q)]);
  float2* oc = a.out + (int64_t)c * a.out_cs;
  auto store = [&](int k0, float2 v) {
    const int ky = t + k0;
    if (colok && ky < lout) {
      v = cmul(v, a.ay.post[ky]);
      if (a.f0tab) v = c_mul(v, a.f0tab[(int64_t)ky * lout_x + kx]);
      else if (a.post_mode != POST_NONE) v = c_mul(v, czt_post_factor(a, ky, kx));
      oc[(int64_t)ky * lout_x + kx] = v;
    }
  };
  fft_inverse_from_regs<Q, TPF, DST_FN, false, false>(s, t, u, store);
}

// Column pass of the power-of-two lengths: G columns of one component per
// block, Q/16 threads each, neighbouring lanes on the G columns: a wave reads
// G/4 of each tile line it touches and stores G-column row segments, straight
// from and to its registers.  (Staged through LDS by blocks of half the
// threads per transform, 232 VGPRs at 4096: the adjoint 256^2 -> 2048^2, three
// components, 109 us, now 76 us of which the accesses alone take 59; zoom
// 2048 -> 512 columns 31 -> 24 us; against the staged form at the other lengths
// see czt_cols_staged.  G = 1, 2, 4 at 4096: 83, 78, 88 us; at 2048, 1024^2 ->
// 400^2: 13.5, 13.3, 16.8 us.)
template <int Q> using CztCols1 = Units<Q, rs_g(Q, 2, 2, 2)>;

template <int Q, bool ZL>
__global__ __launch_bounds__(CztCols1<Q>::NT, 4) void czt_cols1_kernel(CztArgs a0) {
  const CztArgs a = czt_member(a0, blockIdx.z);
  using U = CztCols1<Q>;
  constexpr int TPF = U::TPF;
  using HO = HandOff<Q, TPF>;
  using LP = LastPass<Q, TPF, false>;
  __shared__ float2 lds[U::G * U::LS];
  const int g = U::col_g(threadIdx.x), t = U::col_t(threadIdx.x);
  float2* s = lds + g * U::LS;
  const int kx0 = xcd_remap(blockIdx.x, gridDim.x) * U::G, kx = kx0 + g, c = blockIdx.y;
  const int lout_x = a.ax.lout, lin = a.ay.lin, lout = a.ay.lout;
  const bool colok = kx < lout_x;
  const float2* src = a.t + (int64_t)c * a.t_cs + (int64_t)(kx0 >> 2) * (a.rin4 >> 2) * 16 + (kx0 & 3);
  const uint32_t lane = (g >> 2) * (a.rin4 >> 2) * 16 + (g & 3) + 4 * t;
  auto load = [&](int k) -> float2 {
    return (colok && t + k < lin) ? cmul(ld_at(src + 4 * k, lane), ld_at(a.ay.pre + k, t)) : make_float2(0.f, 0.f);
  };
  Regs<1, 16> in;
  typename HO::Type u;
  NoIO none;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    in.v[0][r] = (ZL && r >= 8) ? make_float2(0.f, 0.f) : load(r * TPF);
    if (!ZL || r < 8) asm volatile("" : "+v"(in.v[0][r].x), "+v"(in.v[0][r].y));
  }
  chain_io<Q, TPF, false, true, 0, SRC_REG, DST_REG, ZL, false>(s, t, none, none, in, u);
#pragma unroll
  for (int b = 0; b < HO::BPT; ++b)
#pragma unroll
    for (int q = 0; q < HO::R; ++q) u.v[b][q] = cmul(u.v[b][q], ld_at(a.ay.gf + HO::koff(b, q), t));
  typename LP::Type o;
  chain_io<Q, TPF, true, false, 0, SRC_REG, DST_REG, false, ZL>(s, t, none, none, u, o);
  float2* oc = a.out + (int64_t)c * a.out_cs + kx0;
  const uint32_t olane = (uint32_t)t * lout_x + g;
#pragma unroll
  for (int b = 0; b < LP::BPT; ++b)
#pragma unroll
    for (int q = 0; q < (ZL ? LP::R / 2 : LP::R); ++q) {
      const int k = LP::index(0, b, q), ky = t + k;
      if (!colok || ky >= lout) continue;
      float2 v = cmul(o.v[b][q], ld_at(a.ay.post + k, t));
      asm volatile("" : "+v"(v.x), "+v"(v.y));
      if (a.f0tab) v = c_mul(v, ld_at(a.f0tab + (int64_t)k * lout_x + kx0, olane));
      else if (a.post_mode != POST_NONE) v = c_mul(v, czt_post_factor(a, ky, kx));
      st_at(oc + (int64_t)k * lout_x, olane, v);
    }
}

// The same pass staged through LDS: the block's four columns, one tile group,
// are loaded with lane-contiguous accesses and the outputs are transposed to
// rows, so that a row segment of 32 B is stored at once.  The first pass reads
// LDS, the last one leaves its outputs in registers.
template <int Q, bool ZL>
__global__ __launch_bounds__(4 * Q / 16) void czt_cols_staged_kernel(CztArgs a0) {
  const CztArgs a = czt_member(a0, blockIdx.z);
  constexpr int TPF = Q / 16, LS = LdsLen<Q>::value, CPB = 4, NT = CPB * TPF;
  using HO = HandOff<Q, TPF>;
  using LP = LastPass<Q, TPF, false>;
  __shared__ float2 lds[CPB * LS];
  const int f = threadIdx.x / TPF, t = threadIdx.x % TPF;
  float2* s = lds + f * LS;
  const int kx0 = xcd_remap(blockIdx.x, gridDim.x) * CPB, c = blockIdx.y;
  const int lout_x = a.ax.lout, lin = a.ay.lin, lout = a.ay.lout;
  const float2* src = a.t + (int64_t)c * a.t_cs;
  typename HO::Type u;
  NoIO none;
  // IT elements per thread, loaded U at a time before their products
  constexpr int IT = (ZL ? Q / 2 : Q) / TPF, U = IT < 8 ? IT : 8;
#pragma unroll
  for (int i0 = 0; i0 < IT; i0 += U) {
    float2 tv[U], pv[U];
#pragma unroll
    for (int u1 = 0; u1 < U; ++u1) {
      const int e = threadIdx.x + (i0 + u1) * NT, r = e / CPB, g = e % CPB;
      const bool ok = r < lin && kx0 + g < lout_x;
      tv[u1] = src[czt_tidx(a.rin4, ok ? r : 0, ok ? kx0 + g : kx0)];
      pv[u1] = a.ay.pre[ok ? r : 0];
    }
#pragma unroll
    for (int u1 = 0; u1 < U; ++u1) {
      const int e = threadIdx.x + (i0 + u1) * NT, r = e / CPB, g = e % CPB;
      const bool ok = r < lin && kx0 + g < lout_x;
      lds[g * LS + lpad(r)] = ok ? cmul(tv[u1], pv[u1]) : make_float2(0.f, 0.f);
    }
  }
  __syncthreads();
  fft_forward_to_regs<Q, TPF, SRC_LDS, ZL>(s, t, none, u);
#pragma unroll
  for (int b = 0; b < HO::BPT; ++b)
#pragma unroll
    for (int q = 0; q < HO::R; ++q) u.v[b][q] = cmul(u.v[b][q], a.ay.gf[HO::index(t, b, q)]);
  typename LP::Type o;
  chain_io<Q, TPF, true, false, 0, SRC_REG, DST_REG, false, ZL>(s, t, none, none, u, o);
  __syncthreads();   // the last pass of other waves may still read LDS
#pragma unroll
  for (int b = 0; b < LP::BPT; ++b)
#pragma unroll
    for (int q = 0; q < (ZL ? LP::R / 2 : LP::R); ++q) {
      const int ky = LP::index(t, b, q);
      if (ky < lout) lds[ky * CPB + f] = cmul(o.v[b][q], a.ay.post[ky]);
    }
  __syncthreads();
  float2* oc = a.out + (int64_t)c * a.out_cs;
  for (int e = threadIdx.x; e < lout * CPB; e += NT) {
    const int ky = e / CPB, kx = kx0 + e % CPB;
    if (kx >= lout_x) continue;
    float2 v = lds[e];
    if (a.f0tab) v = c_mul(v, a.f0tab[(int64_t)ky * lout_x + kx]);
    else if (a.post_mode != POST_NONE) v = c_mul(v, czt_post_factor(a, ky, kx));
    oc[(int64_t)ky * lout_x + kx] = v;
  }
}

// Power-of-two lengths (the 3 * 2^k ones serve the column pass only).
template <int Q> struct CztPow2 { static constexpr bool value = (Q & (Q - 1)) == 0; };

// Three-buffer blocks of a 4096-point row that run at once (104 KB of LDS: one
// per CU).
constexpr int CZT_ROWS_RESIDENT = 256;

// The one-buffer form for one component and for the 4096-point zero-half rows
// from the second round of three-buffer blocks on, the three-buffer form
// otherwise (see czt_rows1_kernel).  The 4096-point rows of three components,
// three buffers against one: 64 rows 16.7 / 26.6 us, 192 20.7 / 28.6, 256 23.3 /
// 30.0, 320 34.1 / 31.7, 768 44.7 / 37.6.  One component keeps three buffers'
// staging where a batch takes its plane factors from a table (nothing but loads
// to wait for) and most of a full-length row is input: 4 members of 1500 -> 500
// 59.5 / 67.6 us, of 700 -> 300 19.7 / 23.4, 16 members of 1200 -> 800 187.6 /
// 180.0; elsewhere the one buffer is 4 to 50 % faster.
template <int Q, int K, bool ZL>
inline void czt_rows_launch_k(const CztArgs& a, int batch, hipStream_t st) {
  using U1 = CztRows1<Q>;
  const dim3 g1((a.rin + U1::G - 1) / U1::G, batch), b1(U1::NT);
  const bool tabled = !ZL && Q >= 1024 && a.ftab && 8 * a.ax.lin > 5 * Q;
  if constexpr (K != PREK_HNA)
    if (a.ncomp == 1 && !tabled) {
      hipLaunchKernelGGL((czt_rows1_kernel<Q, K, ZL, false>), g1, b1, 0, st, a);
      return;
    }
  if constexpr (ZL && Q >= 4096)
    if (a.ncomp > 1 && (int64_t)a.rin * batch > CZT_ROWS_RESIDENT) {
      hipLaunchKernelGGL((czt_rows1_kernel<Q, K, ZL, true>), g1, b1, 0, st, a);
      return;
    }
  const dim3 g(a.rin, batch), b(a.ncomp * Q / 16);
  const size_t lds = (size_t)a.ncomp * LdsLen<Q>::value * sizeof(float2);
  hipLaunchKernelGGL((czt_rows_kernel<Q, K, ZL>), g, b, lds, st, a);
}
template <int Q, bool ZL>
inline void czt_rows_launch_zl(const CztArgs& a, int batch, hipStream_t st) {
  if (a.pre_mode == PRE_RS || a.pre_mode == PRE_CONJ_RS) czt_rows_launch_k<Q, PREK_F, ZL>(a, batch, st);
  else if (a.pre_mode == PRE_HNA) czt_rows_launch_k<Q, PREK_HNA, ZL>(a, batch, st);
  else czt_rows_launch_k<Q, PREK_SIMPLE, ZL>(a, batch, st);
}
template <int Q>
inline void czt_rows_launch(const CztArgs& a, int batch, hipStream_t st) {
  KTimer t(K_CZT_ROWS, st);   // (the x axis has a power-of-two length)
  if (a.ax.zl) czt_rows_launch_zl<Q, true>(a, batch, st);
  else czt_rows_launch_zl<Q, false>(a, batch, st);
}
// Dynamic-LDS limit of the three-buffer row kernel, set once per device by
// the library's initialisation for every length it runs at.
template <int Q, bool ZL> inline hipError_t czt_set_attribute_zl() {
  hipError_t e = hipSuccess;
  const int mx = 3 * LdsLen<Q>::value * (int)sizeof(float2);
  for (const void* f : {(const void*)czt_rows_kernel<Q, PREK_F, ZL>, (const void*)czt_rows_kernel<Q, PREK_HNA, ZL>,
                        (const void*)czt_rows_kernel<Q, PREK_SIMPLE, ZL>}) {
    const hipError_t r = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, mx);
    if (r != hipSuccess) e = r;
  }
  return e;
}
template <int Q> inline hipError_t czt_set_attribute() {
  const hipError_t e = czt_set_attribute_zl<Q, false>(), r = czt_set_attribute_zl<Q, true>();
  return e != hipSuccess ? e : r;
}
inline hipError_t czt_set_attributes() {
  hipError_t e = hipSuccess;
  for (hipError_t r : {czt_set_attribute<64>(), czt_set_attribute<128>(), czt_set_attribute<256>(),
                       czt_set_attribute<512>(), czt_set_attribute<1024>(), czt_set_attribute<2048>(),
                       czt_set_attribute<4096>()})
    if (r != hipSuccess) e = r;
  return e;
}

// Whether the power-of-two column pass of a.ay stages its columns through LDS
// (us, staged / direct, MI355X).  Up to 1024 points it does, unless the outputs
// outnumber the inputs (twice where both fit half the length), when the staging
// of the zero padding costs more than the stores gain: 250 -> 99 samples 8.3 /
// 9.3, 400 -> 61 8.4 / 10.8, 61 -> 400 15.6 / 13.4, 512 -> 512 (three
// components) 14.0 / 15.1, 700 -> 300 (4 members) 12.3 / 15.4, 300 -> 700 20.6 /
// 19.8, 100 -> 500 12.6 / 11.0.  At 2048 its blocks of four columns are fewer
// and wait longer (1024 -> 400, three components, 17.0 / 14.0), but read a tile
// line once where the direct blocks of two columns read it twice, which shows
// when the tiles no longer stay in the caches: 1024 -> 1024, 4 members 36.0 /
// 36.5, 8 members 62.6 / 65, 16 members 130 / 152, 64 members 503 / 640, and
// 900 -> 900, 32 members 255 / 287 (1200 -> 800, 16 members 115 / 110).  At 4096
// direct blocks always win.
constexpr int64_t CZT_STAGED_TILE_BYTES = 64 << 20;
template <int Q> inline bool czt_cols_staged(const CztArgs& a, int batch) {
  if (Q > 2048) return false;
  if (Q == 2048) return a.ay.zl && batch * a.ncomp * a.t_cs * (int64_t)sizeof(float2) >= CZT_STAGED_TILE_BYTES;
  return a.ay.zl ? a.ay.lout < 2 * a.ay.lin : a.ay.lout <= a.ay.lin;
}

template <int Q>
inline void czt_cols_launch(const CztArgs& a, int batch, hipStream_t st) {
  KTimer t(K_CZT_COLS, st);
  if constexpr (CztPow2<Q>::value) {
    if constexpr (Q <= 2048)
      if (czt_cols_staged<Q>(a, batch)) {
        const dim3 g((a.ax.lout + 3) / 4, a.ncomp, batch), b(Q / 4);
        if (a.ay.zl) hipLaunchKernelGGL((czt_cols_staged_kernel<Q, true>), g, b, 0, st, a);
        else hipLaunchKernelGGL((czt_cols_staged_kernel<Q, false>), g, b, 0, st, a);
        return;
      }
    using U = CztCols1<Q>;
    const dim3 g((a.ax.lout + U::G - 1) / U::G, a.ncomp, batch);
    if (a.ay.zl) hipLaunchKernelGGL((czt_cols1_kernel<Q, true>), g, dim3(U::NT), 0, st, a);
    else hipLaunchKernelGGL((czt_cols1_kernel<Q, false>), g, dim3(U::NT), 0, st, a);
  } else {
    constexpr int CPB = CztColsShape<Q>::CPB;
    const dim3 g((a.ax.lout + CPB - 1) / CPB, a.ncomp, batch), b(CPB * Q / 16);
    hipLaunchKernelGGL(czt_cols_kernel<Q>, g, b, 0, st, a);
  }
}
template <int Q>
inline void czt_setup_launch(const CztSetupPair& p, int nblocks, hipStream_t st) {
  KTimer t(K_CZT_SETUP, st);
  hipLaunchKernelGGL(czt_setup_kernel<Q>, dim3(nblocks), dim3(CZT_SETUP_THREADS), 0, st, p);
}
template <int Q>
inline void czt_setup_ftab_launch(const CztSetupPair& p, const CztArgs& a, float2* ftab, float2* f0tab, int64_t elems,
                                  hipStream_t st) {
  KTimer t(K_CZT_SETUP, st);
  const int64_t b = (elems + CZT_SETUP_THREADS - 1) / CZT_SETUP_THREADS;
  hipLaunchKernelGGL(czt_setup_ftab_kernel<Q>, dim3(2 + (unsigned)(b < 4096 ? b : 4096)), dim3(CZT_SETUP_THREADS), 0, st,
                     p, a, ftab, f0tab);
}
template <int QA, int QB>
inline void czt_setup2_launch(const CztSetupPair& p, hipStream_t st) {
  KTimer t(K_CZT_SETUP, st);
  hipLaunchKernelGGL((czt_setup2_kernel<QA, QB>), dim3(2), dim3(CZT_SETUP_THREADS), 0, st, p);
}

}  // namespace xl
