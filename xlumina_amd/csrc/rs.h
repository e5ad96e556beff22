// Rayleigh-Sommerfeld convolution (scalar RS / vectorial VRS) on a P x P grid,
// P >= 2N-1 (the next power of two; a plain call from N = 513 on the shortest of
// 2^k, 3 * 2^k and 5 * 2^k),
// with the pre-propagation Jones masks and the Ez construction fused into the
// first row pass.
//
// Reference operator (xlumina/wave_optics.py:281-289): zero-pad the N x N field
// into a (2N-1)^2 grid, multiply fft2(U) by fft2(H) of the sampled RS impulse
// response on the lag grid (wave_optics.py:265-279, :291-297), ifft2, scale by
// dx*dy, keep [N-1:, N-1:].  That is the linear convolution
//     out[q,p] = sum_ij U[j,i] h(x_p - x_i, y_q - y_j) dx dy.
// Here lag +t sits at index t and lag -t at index P-t (slots N..P-N are zero),
// which gives the same linear convolution on any P >= 2N-1.  The kernel array
// is even in both axes, so only rows 0..N-1 of its row transform are built
// and the column pass mirrors them.
//
// Passes (intermediates of N x P samples in 4x4 tiles of 128 B, ordered [column
// group][row group]: a row pass touches 32 B of each line per row, a column
// pass every line of its columns):
//   rs_hrow   : H rows 0..N-1 generated in float64 phase -> row FFT -> Hr (tiles)
//   rs_hcol   : per column kx <= P/2: FFT(Hr col, mirrored) -> Hhat, one contiguous
//               column of ky <= P/2 (quarter spectrum: the kernel array is even)
//   rs_urow   : masks + Ez on the input rows -> zero-padded row FFT -> T (tiles)
//   rs_col    : per (column, component): FFT(T col) * Hhat -> IFFT, keep rows
//               0..N-1 -> T
//   rs_final  : row IFFT of T, keep columns 0..N-1 -> output (+ |E|^2)
// Hr lies beside Hhat in the spectrum's part of the workspace, with its last
// columns in T where both do not fit (RsArgs::hr, hr2).
#pragma once
#include "fft.h"
#include "fftio.h"
#include "masks.h"
#include "timing.h"

namespace xl {

struct RsArgs {
  const float2* in;       // nin components of N x N, row-major [y][x]
  int64_t in_cs;          // component stride (elements)
  float2* out;            // ncomp components of N x N
  int64_t out_cs;
  float* intensity;       // optional N x N, sum_c |out_c|^2
  float2* t;              // tiles, ncomp x NR4*4 x P
  float2* hr;             // Hr: N rows x (P/2 + 1) columns in tiles (rs_hr_elems): columns < rs_hr_split(P),
  float2* hr2;            // and the others, at the same offsets from hr2 (hr itself, or T)
  float2* hh;             // Hhat: columns kx <= P/2 of stride rs_hh_stride, ky <= P/2 (even in kx and ky)
  const double* x;
  const double* y;
  double z, k;
  const double* z_dev;    // if set, z is read from device memory
  float scale;            // dx*dy/P^2
  int n, nin, ncomp, ez_mode, adjoint;
  int kernel_dz;          // 1: convolve with dH/dz instead of H, 2: with dH/dk
  int hstored;            // the spectrum lives in a caller buffer, unconjugated (adjoints conjugate on read)
  int hreuse;             // the spectrum is already there: skip rs_hrow / rs_hcol
  MaskArgs mask;
  // Batch of independent problems of one geometry (blockIdx.y = member): element strides
  // between the members' inputs, outputs, intensities, mask parameters, tiles and kernel
  // spectra; with z_dev set, member b reads z_dev[b].
  int batch;
  int64_t in_bs, out_bs, inten_bs, mask_bs, t_bs, hh_bs;
  // Gradients by Parseval (one problem).  spec_mode 1: rs_col keeps the input
  // column spectra in `spec`, in the hand-off register order of its blocks
  // (block b, slot j, thread tid at (b SLOTS + j) NT + tid).  spec_mode 2: rs_col adds
  // Re(conj(G) dg[i] U) over its column into gpart[i][comp P + column] for each
  // derivative spectrum dg[i] (Hhat layout) that is set.
  int spec_mode;
  int dg_built;           // spec_mode 2: the derivative spectra were built by the forward call
  int partials_only;      // spec_mode 2: leave the partial sums in gpart (no grad_out reduction)
  float2* spec;
  float2* dg[2];          // spec_mode 1: derivative spectra to build with the kernel spectrum
  float2* dgr[2];         // their row transforms (Hr layout), while they are built with it
  double* gpart[2];
  double* grad_out;       // spec_mode 2: out[i] = sum of gpart[i]
  double* qf_out;         // optional: quality factor of member b at qf_out[b]
  double qf_rmax, qf_dr, qf_wl;
};

// Quality factor of a propagation to z (wave_optics.py:187-191).
__device__ __forceinline__ double rs_quality_factor(double z, double rmax, double dr_real, double wl) {
  return (sqrt(wl * wl + rmax * rmax + 2.0 * wl * sqrt(rmax * rmax + z * z)) - rmax) / dr_real;
}

// The arguments of batch member b (pointers offset by the batch strides).
__device__ __forceinline__ RsArgs rs_member(const RsArgs& a0, int b) {
  if (a0.batch <= 1) return a0;
  RsArgs a = a0;
  a.in += b * a0.in_bs;
  a.out += b * a0.out_bs;
  if (a.intensity) a.intensity += b * a0.inten_bs;
  a.t += b * a0.t_bs;
  a.hr += b * a0.t_bs;
  a.hr2 += b * a0.t_bs;
  a.hh += b * a0.hh_bs;
  if (a.z_dev) a.z_dev += b;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    if (a.mask.st[i].m0) a.mask.st[i].m0 += b * a0.mask_bs;
    if (a.mask.st[i].m1) a.mask.st[i].m1 += b * a0.mask_bs;
  }
  return a;
}

// 1/sqrt(x) in float64 for x > 0: the hardware estimate (v_rsq_f64) refined by
// two Newton steps y <- y (3/2 - x y^2 / 2), which take any estimate within
// 2^-20 to the last bits of float64; the kernel values need r = x / sqrt(x) to
// ~1e-14 relative, for phases k r of up to ~1e6 rad.  One estimate and six
// fused multiply-adds replace a correctly rounded square root and a division.
__device__ __forceinline__ double rsqrt_f64(double x) {
  double y = __builtin_amdgcn_rsq(x);
  const double hx = 0.5 * x;
  y = y * fma(-hx * y, y, 1.5);
  y = y * fma(-hx * y, y, 1.5);
  return y;
}

// h(x, y; z) of wave_optics.py:291-297 with the phase k r reduced in float64.
__device__ __forceinline__ float2 rs_kernel_value(double X, double Y, double z, double k) {
  const double r2 = X * X + Y * Y + z * z;
  const double ir = rsqrt_f64(r2);
  const double r = r2 * ir;
  const double turns = k * r * 0.15915494309189535;   // k r / (2 pi)
  const float2 e = expi_turns(z > 0 ? turns : -turns);
  const double f = 0.15915494309189535 * z * ir * ir;   // (1/2pi) z / r^2
  const float fr = (float)(f * ir), fi = (float)(-f * k);   // f * (1/r - i k)
  return make_float2(fr * e.x - fi * e.y, fr * e.y + fi * e.x);
}

// dH/dz of rs_kernel_value (product rule, dr/dz = z/r, s = sign of the phase):
//   (1/2pi) e^{i s k r} [ (r^2 - 3z^2)/r^5 + s k^2 z^2/r^3 + i k (s z^2 - (r^2 - 2 z^2))/r^4 ].
__device__ __forceinline__ float2 rs_kernel_dz_value(double X, double Y, double z, double k) {
  const double r2 = X * X + Y * Y + z * z;
  const double ir = rsqrt_f64(r2), ir2 = ir * ir;
  const double r = r2 * ir;
  const double s = z > 0 ? 1.0 : -1.0;
  const double turns = k * r * 0.15915494309189535;
  const float2 e = expi_turns(s * turns);
  const double z2 = z * z;
  const double cr = (r2 - 3.0 * z2) * ir2 * ir2 * ir + s * k * k * z2 * ir2 * ir;
  const double ci = k * (s * z2 - (r2 - 2.0 * z2)) * ir2 * ir2;
  const float fr = (float)(0.15915494309189535 * cr), fi = (float)(0.15915494309189535 * ci);
  return make_float2(fr * e.x - fi * e.y, fr * e.y + fi * e.x);
}

// dH/dk of rs_kernel_value (k = 2 pi / lambda; r and z do not depend on k):
//   (1/2pi)(z/r^2) e^{i s k r} [ s k r + i (s - 1) ].
__device__ __forceinline__ float2 rs_kernel_dk_value(double X, double Y, double z, double k) {
  const double r2 = X * X + Y * Y + z * z;
  const double ir = rsqrt_f64(r2);
  const double r = r2 * ir;
  const double s = z > 0 ? 1.0 : -1.0;
  const double turns = k * r * 0.15915494309189535;
  const float2 e = expi_turns(s * turns);
  const double f = 0.15915494309189535 * z * ir * ir;
  const float fr = (float)(f * s * k * r), fi = (float)(f * (s - 1.0));
  return make_float2(fr * e.x - fi * e.y, fr * e.y + fi * e.x);
}

// h with its derivatives in z (DM bit 0) and k (DM bit 1) at one lag, the
// geometry (r, 1/r, the phase factor) formed once for all three; each value
// is the expression of rs_kernel_value / rs_kernel_dz_value /
// rs_kernel_dk_value.
template <int DM>
__device__ __forceinline__ void rs_kernel_with_derivatives(double X, double Y, double z, double k, float2& h,
                                                           float2& hz, float2& hk) {
  const double r2 = X * X + Y * Y + z * z;
  const double ir = rsqrt_f64(r2), ir2 = ir * ir;
  const double r = r2 * ir;
  const double s = z > 0 ? 1.0 : -1.0;
  const double turns = k * r * 0.15915494309189535;
  const float2 e = expi_turns(s * turns);
  auto rot = [&](float fr, float fi) { return make_float2(fr * e.x - fi * e.y, fr * e.y + fi * e.x); };
  const double f = 0.15915494309189535 * z * ir * ir;
  h = rot((float)(f * ir), (float)(-f * k));
  if constexpr ((DM & 1) != 0) {
    const double z2 = z * z;
    const double cr = (r2 - 3.0 * z2) * ir2 * ir2 * ir + s * k * k * z2 * ir2 * ir;
    const double ci = k * (s * z2 - (r2 - 2.0 * z2)) * ir2 * ir2;
    hz = rot((float)(0.15915494309189535 * cr), (float)(0.15915494309189535 * ci));
  }
  if constexpr ((DM & 2) != 0) hk = rot((float)(f * s * k * r), (float)(f * (s - 1.0)));
}

// The kept input spectra are written once and read once, by another launch:
// non-temporal accesses, so that they do not displace the tile lines the
// column pass shares through the caches.
__device__ __forceinline__ void stream_store(float2* p, float2 v) {
  __builtin_nontemporal_store(v.x, &p->x);
  __builtin_nontemporal_store(v.y, &p->y);
}
__device__ __forceinline__ float2 stream_load(const float2* p) {
  return make_float2(__builtin_nontemporal_load(&p->x), __builtin_nontemporal_load(&p->y));
}

// Elements of Hr (n rows, columns kx <= P/2 or below `cols`): at most half the
// n x P tiles of one component of T.
__host__ __device__ constexpr int64_t rs_hr_elems(int n, int P, int cols = 0) {
  return (int64_t)(cols ? cols / 4 : P / 8 + 1) * ((n + 3) / 4) * 16;
}
// First column of Hr's second part, a multiple of every pass's last stride.
// T's lines are still in the caches of the XCDs that ran the last passes of
// the call before, and writes to them cost more.  With all of Hr in T, RS
// 1000^2 takes 16.4 us for the kernel's rows, 16.9 for the field's rows after
// them and 64.5 in all, with Hr beside Hhat 13.2, 15.3 and 59.3; 1024^2, where
// seven eighths fit, 17.7, 17.2 and 66 against 13.4, 16.7 and 61.4.
constexpr int RS_HR_SPLIT_MIN = 256;   // shorter lengths have Hr in one place
__host__ __device__ constexpr int rs_hr_split(int P) { return P / 16 * 7; }
// Column stride of Hhat: ky = 0..P/2 and a pad to whole 128 B lines.
__host__ __device__ constexpr int rs_hh_stride(int P) { return P / 2 + 16; }

// A transform of P points runs on TPF threads (one butterfly each per pass,
// P/16 for the powers of two) in one LDS buffer.  A block takes G rows (or columns) of one
// 4x4 tile group, lanes spread over the G transforms, so that an access of a
// wave covers G/4 of each 128 B line it touches instead of a quarter; more
// than one 35 KB buffer behind common barriers hides less of the transforms'
// latency, and small grids need all their blocks.  Chosen per kernel (us within
// repeated calls of P/2 squared samples, MI355X):
//                      P = 4096          2048                1024
//                      G = 1     2       1     2     4       1     2     4
//   hrow               25.3  25.7    13.1  12.9  13.5     8.7   8.8   9.3
//   hcol               17.3  20.1     7.3   7.6  10.4     5.3   5.8   6.6
//   urow, SLM          36.8  42.5    17.5  16.4  16.8    10.0  10.1  10.4
//   urow, LCD and Ez   86.4   105    28.0  25.6  29.2    19.6  20.0  21.8
//   urow, 3 plain      80.3  66.5    16.4  16.0  18.4    12.2  11.5  12.0
//   col (1 comp.)      48.5  53.5    15.8  16.3  19.6     9.2   8.9  10.6
//   col (3 comp.)       142   158    35.1  37.5  53.0    16.6  17.4  19.9
//   col, dots (3)                    65.8  61.6
//   final (1 comp.)    19.5  20.4     7.8   7.5   8.0     4.3   4.5   4.8
//   final (3 comp.)    56.3  53.6    16.2  15.0  16.7     6.6   6.4   6.9
// The column pass of kept spectra (their layout follows its blocks) has a line
// of its own.  1280 and 1536 take the 1024 column, 2560 and 3072 that of 4096
// (VRS 1200^2 at 2560, G = 1 / 2: col 67 / 82, urow 35 / 41, hrow 13.4 / 15.5).
// Below P = 1024 a block holds at least one wave.
constexpr int rs_g(int P, int g4096, int g2048, int g1024) {
  return P > 2048 ? g4096 : P == 2048 ? g2048 : P >= 1024 ? g1024 : 1024 / P;
}
// Threads per transform: P over the first radix of its passes.
constexpr int rs_tpf(int P) { return P % 3 == 0 ? P / 12 : P % 5 == 0 ? P / 10 : P / 16; }
template <int P, int G_> struct Units {
  static constexpr int TPF = rs_tpf(P);
  static constexpr int G = G_;
  static constexpr int NT = G * TPF;   // threads per block
  static_assert(NT >= 64, "whole waves");
  // buffer stride: the G buffers start 32 / G bank pairs apart
  static constexpr int RAW = LdsLen<P>::value;
  static constexpr int WANT = G == 1 ? 0 : (G >= 8 ? 4 : 32 / G);
  static constexpr int LS = G == 1 ? RAW : RAW + (WANT - RAW % 32 + 32) % 32;
  // Up to four rows per block divide a tile's four: the blocks' rows are all
  // among the tiled ones, and the accesses carry no predicate for them.
  static constexpr bool WHOLE = G <= 4;
  // column pass: neighbouring lanes on the G columns of a row
  __device__ static int col_g(int tid) { return G == 1 ? 0 : tid % G; }
  __device__ static int col_t(int tid) { return G == 1 ? tid : tid / G; }
  // row passes: four neighbouring lanes on four columns, then the G rows
  __device__ static int row_g(int tid) { return G == 1 ? 0 : (tid / 4) % G; }
  __device__ static int row_t(int tid) { return G == 1 ? tid : tid / (4 * G) * 4 + tid % 4; }
};
template <int P> using UHrow = Units<P, rs_g(P, 1, 1, 1)>;
template <int P> using UHcol = Units<P, rs_g(P, 1, 1, 1)>;
template <int P, bool ONE> using UUrow = Units<P, rs_g(P, ONE ? 2 : 1, 2, 2)>;
template <int P, bool KEPT> using UCol = Units<P, rs_g(P, 1, KEPT ? 2 : 1, 1)>;
template <int P> using UFinal = Units<P, rs_g(P, 2, 2, 2)>;

// Element `off` (a per-lane 32-bit offset) from a block-uniform base: one
// offset register serves all accesses of a thread.
__device__ __forceinline__ float2 ld_at(const float2* base, uint32_t off) {
  return *reinterpret_cast<const float2*>(reinterpret_cast<const char*>(base) + off * (uint32_t)sizeof(float2));
}
__device__ __forceinline__ void st_at(float2* base, uint32_t off, float2 v) {
  *reinterpret_cast<float2*>(reinterpret_cast<char*>(base) + off * (uint32_t)sizeof(float2)) = v;
}

// The tiles of G rows row0..row0+G-1 seen by a row pass's thread (transform g,
// sample t + k): uniform base of row0, lane offset, and step(k) from k (a
// multiple of 4).
struct RowTiles {
  int nrg;
  uint32_t lane;
  __device__ RowTiles(int n, int g, int t) : nrg((n + 3) >> 2) {
    lane = (uint32_t)((t >> 2) * nrg + (g >> 2)) * 16 + (g & 3) * 4 + (t & 3);
  }
  __device__ static int64_t base(int row0) { return (row0 >> 2) * 16 + (row0 & 3) * 4; }
  __device__ int64_t step(int k) const { return (int64_t)(k >> 2) * nrg * 16; }
};

// G kernel rows per block: H of rows 0..N-1 generated in float64 phase
// (the array is even in x: columns above P/2 mirror), row FFT, stored as Hr
// for kx <= P/2 (the transform of an even row is even).  DM != 0: the rows
// of the derivative kernels in the bit set DM (bit 0 dH/dz, bit 1 dH/dk) are
// formed from the same geometry, held in registers while H is transformed,
// then transformed in turn into dgr[i] (a forward call that will be
// differentiated in z / lambda builds its derivative spectra this way).
template <int P, int DM = 0>
__global__ __launch_bounds__(UHrow<P>::NT, 4) void rs_hrow_kernel(RsArgs a0) {
  const RsArgs a = rs_member(a0, blockIdx.y);
  using U = UHrow<P>;
  constexpr int TPF = U::TPF;
  constexpr int NCOL = (P / 2 + 1 + TPF - 1) / TPF;   // columns kx <= P/2 per thread
  __shared__ float2 lds[U::G * U::LS];
  const int g = U::row_g(threadIdx.x), t = U::row_t(threadIdx.x);
  float2* s = lds + g * U::LS;
  const int row0 = xcd_remap(blockIdx.x, gridDim.x) * U::G, r = row0 + g;
  const RowTiles rt(a.n, g, t);
  const bool store_ok = U::WHOLE || r < rt.nrg * 4;
  const double z = a.z_dev ? *a.z_dev : a.z;
  // columns c < N of a row r < N (N <= P/2: the lags above are mirrors)
  const int ncol = r < a.n ? a.n : 0;
  const double dy = a.y[r < a.n ? r : 0] - a.y[0];
  float2 dv[2][NCOL];
#pragma unroll
  for (int i = 0; i < NCOL; ++i) {
    const int c = t + i * TPF;
    if (c > P / 2) break;
    float2 v = make_float2(0.f, 0.f), vz = v, vk = v;
    if (c < ncol) {
      const double dx = a.x[c] - a.x[0];
      if constexpr (DM == 0)
        v = a.kernel_dz == 1   ? rs_kernel_dz_value(dx, dy, z, a.k)
            : a.kernel_dz == 2 ? rs_kernel_dk_value(dx, dy, z, a.k)
                               : rs_kernel_value(dx, dy, z, a.k);
      else
        rs_kernel_with_derivatives<DM>(dx, dy, z, a.k, v, vz, vk);
    }
    s[lpad(c)] = v;
    if (c > 0 && c < P / 2) s[lpad(P - c)] = v;
    dv[0][i] = vz;
    dv[1][i] = vk;
  }
  __syncthreads();
  NoIO none;
  typename LastPass<P, TPF, true>::Type unused;
  {
    float2 *dst = a.hr + RowTiles::base(row0), *dst2 = a.hr2 + RowTiles::base(row0);
    auto store = [&](int k, float2 v) {
      if (store_ok && (k < P / 2 || (k == P / 2 && t == 0)))
        st_at((k < rs_hr_split(P) ? dst : dst2) + rt.step(k), rt.lane, v);
    };
    fft_io<P, TPF, false, SRC_LDS, DST_FN>(s, t, none, store, unused);
  }
#pragma unroll
  for (int d = 0; d < 2; ++d) {
    if constexpr (DM == 0) break;
    if (!(DM >> d & 1)) continue;
    __syncthreads();   // the last pass of other waves may still read LDS
#pragma unroll
    for (int i = 0; i < NCOL; ++i) {
      const int c = t + i * TPF;
      if (c > P / 2) break;
      s[lpad(c)] = dv[d][i];
      if (c > 0 && c < P / 2) s[lpad(P - c)] = dv[d][i];
    }
    __syncthreads();
    float2* dst = a.dgr[d] + RowTiles::base(row0);
    auto store = [&](int k, float2 v) {
      if (store_ok && (k < P / 2 || (k == P / 2 && t == 0))) st_at(dst + rt.step(k), rt.lane, v);
    };
    fft_io<P, TPF, false, SRC_LDS, DST_FN>(s, t, none, store, unused);
  }
}

// G input rows per block.  Thread t's first-pass inputs are the columns
// t + r TPF; the nonzero ones (columns < N <= P/2) are the lower half of the
// first radix (8 at the powers of two), so each thread computes the masks and
// Ez of exactly those pixels once, keeps all components in registers, and the
// components are transformed one after the other from there (no LDS staging
// pass).
// ONE (inputs without masks or Ez construction: the adjoint's cotangent): one
// component (blockIdx.z) per block, for grids whose row blocks alone leave
// resident slots empty.
template <int P, bool ONE = false>
__global__ __launch_bounds__((UUrow<P, ONE>::NT), P == 1536 ? 3 : 1) void rs_urow_kernel(RsArgs a0) {
  const RsArgs a = rs_member(a0, blockIdx.y);
  using U = UUrow<P, ONE>;
  constexpr int TPF = U::TPF;
  constexpr int R0 = FftPlan<P, TPF>::radix(true, 0);
  static_assert(P / R0 == TPF, "first pass: one butterfly per thread");
  constexpr int H = R0 / 2;   // inputs r < H hold the N <= P/2 pixels
  __shared__ float2 lds[U::G * U::LS];
  const int g = U::row_g(threadIdx.x), t = U::row_t(threadIdx.x);
  float2* s = lds + g * U::LS;
  const int row0 = xcd_remap(blockIdx.x, gridDim.x) * U::G, row = row0 + g;
  const RowTiles rt(a.n, g, t);
  const bool store_ok = U::WHOLE || row < rt.nrg * 4, rowok = row < a.n;
  NoIO none;
  typename LastPass<P, TPF, true>::Type unused;
  if constexpr (ONE) {
    const int c = blockIdx.z;
    const float2* src = a.in + (int64_t)c * a.in_cs + (int64_t)row0 * a.n;
    Regs<1, R0> rin;
#pragma unroll
    for (int r = 0; r < R0; ++r) {
      const int col = t + r * TPF;
      rin.v[0][r] = (r < H && rowok && col < a.n) ? ld_at(src + r * TPF, g * a.n + t) : make_float2(0.f, 0.f);
    }
    float2* dst = a.t + (int64_t)c * rt.nrg * 4 * P + RowTiles::base(row0);
    auto store = [&](int k, float2 v) {
      if (store_ok) st_at(dst + rt.step(k), rt.lane, v);
    };
    chain_io<P, TPF, false, true, 0, SRC_REG, DST_FN, true, false>(s, t, none, store, rin, unused);
    return;
  }
  const int nc = a.ncomp;
  const double z = a.z_dev ? *a.z_dev : a.z;
  // all loads of a thread's pixels first (in flight together), then the masks and Ez
  const bool ez = a.ez_mode != EZ_NONE;
  // (columns beyond N read the row's last pixel and are zeroed below)
  PixRaw raw[H];
  uint32_t pix[H];
  const uint32_t row_at = (uint32_t)(rowok ? row : 0) * a.n;
#pragma unroll
  for (int r = 0; r < H; ++r) pix[r] = row_at + min(t + r * TPF, a.n - 1);
  pix_load_n<H>(a.in, a.in_cs, a.nin, a.mask, pix, raw);
  const double yr = ez ? a.y[rowok ? row : 0] : 0.0;
  float2 e[3][H];
#pragma unroll
  for (int r = 0; r < H; ++r) {
    const int col = t + r * TPF;
    float2 e0 = make_float2(0.f, 0.f), e1 = e0, e2 = e0;
    if (rowok && col < a.n) {
      pix_masked(a.mask, raw[r], e0, e1, e2);
      if (ez) e2 = build_ez(a.ez_mode, e0, e1, at32(a.x, col), yr, z);
    }
    e[0][r] = e0;
    e[1][r] = e1;
    e[2][r] = e2;
  }
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    if (c >= nc) break;
    Regs<1, R0> rin;
#pragma unroll
    for (int r = 0; r < R0; ++r) rin.v[0][r] = r < H ? e[c][r] : make_float2(0.f, 0.f);
    float2* dst = a.t + (int64_t)c * rt.nrg * 4 * P + RowTiles::base(row0);
    auto store = [&](int k, float2 v) {
      if (store_ok) st_at(dst + rt.step(k), rt.lane, v);
    };
    chain_io<P, TPF, false, true, 0, SRC_REG, DST_FN, true, false>(s, t, none, store, rin, unused);
  }
}

// The masked row pass of several components at the short lengths: a row per
// block, component c on threads [c TPF, (c + 1) TPF) and LDS buffer c, the
// pre-ops of each pixel formed once.  A small grid waits for one row's chain
// of transforms, which here run side by side (VRS 64^2: 6.6 us against 10.4
// one after the other, 256^2: 8.0 against 13.3).  A batch fills the chip: at
// P = 512 components one after the other win from about 2500 rows on (4000
// rows of 250: 28.7 against 23.4 us; 2000: 15.9 against 23.5), at 256 not yet
// at 4096 (13.0 against 18.3 us).
template <int P>
__global__ __launch_bounds__(3 * rs_tpf(P)) void rs_urow_comps_kernel(RsArgs a0) {
  const RsArgs a = rs_member(a0, blockIdx.y);
  constexpr int TPF = rs_tpf(P), LS = LdsLen<P>::value;
  __shared__ float2 lds[3 * LS];
  const int c = threadIdx.x / TPF, t = threadIdx.x % TPF;
  const int row = xcd_remap(blockIdx.x, gridDim.x), nc = a.ncomp;
  const RowTiles rt(a.n, 0, t);
  const double z = a.z_dev ? *a.z_dev : a.z;
  const float2 zero = make_float2(0.f, 0.f);
  for (int col = threadIdx.x; col < P / 2; col += blockDim.x) {
    float2 e0 = zero, e1 = zero, e2 = zero;
    if (row < a.n && col < a.n) {
      const int64_t pix = (int64_t)row * a.n + col;
      e0 = a.in[pix];
      if (a.nin > 1) e1 = a.in[a.in_cs + pix];
      if (a.nin > 2) e2 = a.in[2 * a.in_cs + pix];
      apply_mask(a.mask, pix, e0, e1, e2);
      if (a.ez_mode != EZ_NONE) e2 = build_ez(a.ez_mode, e0, e1, a.x[col], a.y[row], z);
    }
    lds[lpad(col)] = e0;
    lds[lpad(col + P / 2)] = zero;
    lds[LS + lpad(col)] = e1;
    lds[LS + lpad(col + P / 2)] = zero;
    if (nc > 2) {
      lds[2 * LS + lpad(col)] = e2;
      lds[2 * LS + lpad(col + P / 2)] = zero;
    }
  }
  __syncthreads();
  float2* dst = a.t + (int64_t)c * rt.nrg * 4 * P + RowTiles::base(row);
  NoIO none;
  auto store = [&](int k, float2 v) { st_at(dst + rt.step(k), rt.lane, v); };
  typename LastPass<P, TPF, true>::Type unused;
  fft_io<P, TPF, false, SRC_LDS, DST_FN>(lds + c * LS, t, none, store, unused);
}

// Kernel spectrum.  Per column kx <= P/2: the Hr column (rows mirrored, rows
// N..P-N zero) is transformed along y and the spectrum, times dx dy / P^2
// (conjugated for the adjoint), stored contiguously for ky <= P/2.  The array
// is even in y and in x, so ky > P/2 and kx > P/2 are not formed
// (Hhat(P - ky, kx) = Hhat(ky, P - kx) = Hhat(ky, kx)).
template <int P>
__global__ __launch_bounds__(UHcol<P>::NT, 4) void rs_hcol_kernel(RsArgs a0) {
  const RsArgs a = rs_member(a0, blockIdx.y);
  using U = UHcol<P>;
  constexpr int TPF = U::TPF;
  static_assert(P < RS_HR_SPLIT_MIN || rs_hr_split(P) % U::G == 0, "a block's columns lie in one part of Hr");
  using HO = HandOff<P, TPF>;
  __shared__ float2 lds[U::G * U::LS];
  const int g = U::col_g(threadIdx.x), t = U::col_t(threadIdx.x);
  float2* s = lds + g * U::LS;
  const int col0 = xcd_remap(blockIdx.x, gridDim.x) * U::G, col = col0 + g;
  const bool act = U::G == 1 || col <= P / 2;
  const int nrg = (a.n + 3) >> 2;
  const float2* hc = (col0 < rs_hr_split(P) ? a.hr : a.hr2) + (int64_t)(col0 >> 2) * nrg * 16 + (col0 & 3);
  const uint32_t lane = (g >> 2) * nrg * 16 + (g & 3);
  auto load = [&](int k) -> float2 {
    // (rows beyond N read row N - 1 and are zeroed: a select, where a predicate
    // would put a branch around each load)
    const int r = t + k, rr = r <= P / 2 ? r : P - r;
    const float2 v = ld_at(hc, lane + 4 * min(rr, a.n - 1));
    return act && rr < a.n ? v : make_float2(0.f, 0.f);
  };
  typename HO::Type u;
  fft_forward_to_regs<P, TPF, SRC_FN>(s, t, load, u);
  constexpr int HS = rs_hh_stride(P);
  float2* dst = a.hh + (int64_t)col0 * HS;
#pragma unroll
  for (int b = 0; b < HO::BPT; ++b)
#pragma unroll
    for (int q = 0; q < HO::R; ++q) {
      const int k = HO::koff(b, q);
      if (k > P / 2 || !HO::valid(t, b)) continue;
      float2 h = u.v[b][q] * a.scale;
      if (a.adjoint && !a.hstored) h = conjf2(h);
      if (act && (k < P / 2 || t == 0)) st_at(dst + k, g * HS + t, h);
    }
}

// Sum of v over the threads of each of the block's G columns (column g on the
// lanes tid % G), fixed order; every thread of the block calls it and thread
// t = 0 of the column holds the sum.  `red` holds G * (waves per block) values.
template <int P> __device__ __forceinline__ double column_sum_f64(double v, double* red) {
  using U = UCol<P, true>;
  constexpr int NW = U::NT / 64;
#pragma unroll
  for (int o = 32; o >= U::G; o >>= 1) v += __shfl_xor(v, o, 64);
  if constexpr (NW > 1) {
    const int g = U::col_g(threadIdx.x), lane = threadIdx.x & 63;
    if (lane < U::G) red[g * NW + (threadIdx.x >> 6)] = v;
    __syncthreads();
    v = 0.0;
#pragma unroll
    for (int w = 0; w < NW; ++w) v += red[g * NW + w];
  }
  return v;
}

// Column pass.  G columns of one component (blockIdx.z) per block: each T
// column (rows 0..N-1, zero padded) is transformed along y straight from the
// tiles, multiplied in registers by the kernel spectrum of its column (a
// contiguous column, mirrored for ky > P/2), inverse-transformed, and rows
// 0..N-1 stored back in place.  Tile neighbours run back to back on one XCD,
// so the 128 B tile lines are fetched once into its L2.
// What bounds it (2048^2, three components): the accesses alone take 112 us
// (448 MB, 4.0 TB/s), the transforms alone 99 us, together 133 us (141 us with
// the spectrum in 4x4 tiles and 64-bit addresses per access); more waves, wave
// priorities or keeping Hhat in registers across the components gain nothing.
// SPEC 1 also keeps the column's spectrum; SPEC = 2 + GB, GB in 1..3, adds
// its gradient dots for the derivative spectra in the bit set GB (spec_mode 2
// of RsArgs): acc[i] = sum over the column's ky of Re(conj(G) dg[i] U), G the
// spectrum in registers (the cotangent's), U the kept input spectrum.
template <int P, int SPEC>
__global__ __launch_bounds__((UCol<P, SPEC != 0>::NT), 4) void rs_col_kernel(RsArgs a0) {
  const RsArgs a = rs_member(a0, blockIdx.y);
  if (a.qf_out && blockIdx.x == 0 && blockIdx.z == 0 && threadIdx.x == 0)
    a.qf_out[blockIdx.y] = rs_quality_factor(a.z_dev ? *a.z_dev : a.z, a.qf_rmax, a.qf_dr, a.qf_wl);
  using U = UCol<P, SPEC != 0>;
  constexpr int TPF = U::TPF, NT = U::NT, HS = rs_hh_stride(P);
  using HO = HandOff<P, TPF>;
  constexpr int SLOTS = HO::BPT * HO::R;
  __shared__ float2 lds[U::G * U::LS];
  const int g = U::col_g(threadIdx.x), t = U::col_t(threadIdx.x);
  float2* s = lds + g * U::LS;
  const int ub = xcd_remap(blockIdx.x, gridDim.x), comp = blockIdx.z;
  const int col0 = ub * U::G, col = col0 + g;
  const int nrg = (a.n + 3) >> 2, nr = nrg * 4;
  // column element r of a tile group is 4 r elements in
  float2* tc = a.t + (int64_t)comp * nrg * 4 * P + (int64_t)(col0 >> 2) * nrg * 16 + (col0 & 3);
  const uint32_t lane = (g >> 2) * nrg * 16 + (g & 3) + 4 * t;
  auto load = [&](int k) -> float2 { return t + k < nr ? ld_at(tc + 4 * k, lane) : make_float2(0.f, 0.f); };
  // Hhat is even in kx and ky: ky = t + k at lo + k for k < P/2 (and ky = P/2),
  // at hi + (P - k) above
  const uint32_t hcol = (uint32_t)(col <= P / 2 ? col : P - col) * HS;
  auto hat = [&](const float2* base, int k) -> float2 {
    return k < P / 2 ? ld_at(base + k, hcol + t) : ld_at(base, hcol + (P - k) - t);
  };
  typename HO::Type u, h;
  constexpr int GB = SPEC >= 3 ? SPEC - 2 : 0;
  float2* sp = nullptr;
  if constexpr (SPEC != 0) sp = a.spec + ((int64_t)comp * gridDim.x + ub) * SLOTS * NT;
  // the gradient dots (SPEC >= 3) read the kept input spectrum U: up to
  // P = 2048 its loads issue before the forward transform and complete behind
  // it (at 4096, or with both derivatives, they would not fit beside the
  // transform's registers)
  constexpr bool UPRE = (GB == 1 || GB == 2) && P <= 2048;
  typename HO::Type uk;
  if constexpr (UPRE) {
#pragma unroll
    for (int b = 0; b < HO::BPT; ++b)
#pragma unroll
      for (int q = 0; q < HO::R; ++q) uk.v[b][q] = stream_load(sp + (b * HO::R + q) * NT + threadIdx.x);
  }
  // rows >= N <= P/2 are zero padding, and the rows kept are < N: the first
  // forward pass skips the upper half of its inputs, the last inverse pass
  // the upper half of its outputs
  constexpr bool HPRE = GB == 0;
  auto hook = [&]() {
    if constexpr (HPRE) {
#pragma unroll
      for (int b = 0; b < HO::BPT; ++b)
#pragma unroll
        for (int q = 0; q < HO::R; ++q)
          if (HO::valid(t, b)) h.v[b][q] = hat(a.hh, HO::koff(b, q));
    }
  };
  fft_forward_to_regs<P, TPF, SRC_FN, true>(s, t, load, u, hook);
  if constexpr (SPEC == 1) {
#pragma unroll
    for (int b = 0; b < HO::BPT; ++b)
#pragma unroll
      for (int q = 0; q < HO::R; ++q) stream_store(sp + (b * HO::R + q) * NT + threadIdx.x, u.v[b][q]);
  }
  const float hs = (a.adjoint && a.hstored) ? -1.f : 1.f;   // stored spectrum: conjugate for the adjoint
  double acc[2] = {0.0, 0.0};
  static_assert(SPEC == 0 || HO::NB % TPF == 0, "spectra are kept at the power-of-two lengths");
#pragma unroll
  for (int b = 0; b < HO::BPT; ++b)
#pragma unroll
    for (int q = 0; q < HO::R; ++q) {
      const int k = HO::koff(b, q);
      if (!HO::valid(t, b)) continue;
      float2 hv = HPRE ? h.v[b][q] : hat(a.hh, k);
      hv.y *= hs;
      if constexpr (GB != 0) {
        const float2 uv = UPRE ? uk.v[b][q] : stream_load(sp + (b * HO::R + q) * NT + threadIdx.x);
        const float2 gv = u.v[b][q];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          if (!(GB >> i & 1)) continue;
          // roundings written out: the float64 gradient shows them
          const float2 d = hat(a.dg[i], k);
          const float wx = fmaf(d.x, uv.x, -__fmul_rn(d.y, uv.y)), wy = fmaf(d.x, uv.y, __fmul_rn(d.y, uv.x));
          acc[i] += (double)fmaf(gv.x, wx, __fmul_rn(gv.y, wy));
        }
        // the sums are formed here: sunk behind the inverse transform, their
        // operands would spill
#pragma unroll
        for (int i = 0; i < 2; ++i)
          if (GB >> i & 1) asm volatile("" : "+v"(acc[i]));
      }
      u.v[b][q] = cmul(u.v[b][q], hv);
    }
  auto store = [&](int k, float2 v) {
    if (t + k < nr) st_at(tc + 4 * k, lane, v);
  };
  fft_inverse_from_regs<P, TPF, DST_FN, true>(s, t, u, store);
  if constexpr (GB != 0) {
    __shared__ double red[2][U::G * (NT / 64)];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if (!(GB >> i & 1)) continue;
      const double v = column_sum_f64<P>(acc[i], red[i]);
      if (t == 0) a.gpart[i][comp * P + col] = v;
    }
  }
}

// G output rows per block: the components are inverse-transformed one after
// the other, each read straight from its tiles into the first pass (the
// blocks of a tile's other rows run next on the same XCD), each last pass left
// in registers, where the first N samples are stored and |E|^2 is accumulated
// over the components.
// ONE: one component (blockIdx.z) per block (no |E|^2 to accumulate across
// components): ncomp N / G blocks instead of N / G, and the last round of them
// over the chip is fuller (at P = 4096 1024 blocks of two rows make 1.33
// rounds, 3072 make 4).
// Below P = 1024 the passes run in the forward order and form every output
// (roundings are those of the whole transform).
template <int P, bool ONE = false>
__global__ __launch_bounds__(UFinal<P>::NT) void rs_final_kernel(RsArgs a0) {
  const RsArgs a = rs_member(a0, blockIdx.y);
  using U = UFinal<P>;
  constexpr int TPF = U::TPF;
  constexpr bool SMALL = P < 1024;
  using LP = LastPass<P, TPF, SMALL>;
  __shared__ float2 lds[U::G * U::LS];
  const int g = U::row_g(threadIdx.x), t = U::row_t(threadIdx.x);
  float2* s = lds + g * U::LS;
  const int row0 = xcd_remap(blockIdx.x, gridDim.x) * U::G, row = row0 + g;
  const RowTiles rt(a.n, g, t);
  const bool load_ok = U::WHOLE || row < rt.nrg * 4;
  // output columns < N <= P/2 are slots q < R/2 of the last pass
  constexpr int QH = LP::R / 2;
  float inten[LP::BPT][QH];
#pragma unroll
  for (int b = 0; b < LP::BPT; ++b)
#pragma unroll
    for (int q = 0; q < QH; ++q) inten[b][q] = 0.f;
  NoIO none;
  for (int c = ONE ? blockIdx.z : 0; c < (ONE ? blockIdx.z + 1 : a.ncomp); ++c) {
    const float2* tc = a.t + (int64_t)c * rt.nrg * 4 * P + RowTiles::base(row0);
    auto load = [&](int k) -> float2 { return load_ok ? ld_at(tc + rt.step(k), rt.lane) : make_float2(0.f, 0.f); };
    typename LP::Type o, unused;
    // the kept columns are < N <= P/2: the last pass forms the lower half only
    chain_io<P, TPF, true, SMALL, 0, SRC_FN, DST_REG, false, !SMALL>(s, t, load, none, unused, o);
    if constexpr (SMALL) {
#pragma unroll
      for (int b = 0; b < LP::BPT; ++b)
#pragma unroll
        for (int q = QH; q < LP::R; ++q) asm volatile("" ::"v"(o.v[b][q].x), "v"(o.v[b][q].y));
    }
    float2* oc = a.out + (int64_t)c * a.out_cs + (int64_t)row0 * a.n;
#pragma unroll
    for (int b = 0; b < LP::BPT; ++b) {
      if (!LP::valid(t, b)) continue;
#pragma unroll
      for (int q = 0; q < QH; ++q) {
        const int k = LP::index(0, b, q);
        if (t + k < a.n && row < a.n) {
          const float2 v = o.v[b][q];
          st_at(oc + k, g * a.n + t, v);
          if constexpr (!ONE) inten[b][q] += v.x * v.x + v.y * v.y;
        }
      }
    }
  }
  if (!ONE && a.intensity) {
#pragma unroll
    for (int b = 0; b < LP::BPT; ++b) {
      if (!LP::valid(t, b)) continue;
#pragma unroll
      for (int q = 0; q < QH; ++q) {
        const int k = LP::index(0, b, q);
        if (t + k < a.n && row < a.n) a.intensity[(int64_t)row * a.n + t + k] = inten[b][q];
      }
    }
  }
}

// out[i] = sum of the n per-unit partials of gradient i (block i of 1024
// threads; a null partial array skips its block), fixed order.
__global__ __launch_bounds__(1024) void rs_grad_reduce_kernel(const double* p0, const double* p1, int n,
                                                              double* out) {
  const double* p = blockIdx.x == 0 ? p0 : p1;
  if (!p) return;   // whole block
  __shared__ double red[16];
  double s = 0.0;
  for (int i = threadIdx.x; i < n; i += 1024) s += p[i];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    double v = 0.0;
    for (int w = 0; w < 16; ++w) v += red[w];
    out[blockIdx.x] = v;
  }
}

inline int rs_rows4(int n) { return ((n + 3) >> 2) * 4; }
// Grid of `units` rows or columns of nb members and nz components.
template <class U> inline dim3 rs_grid(int units, int nb, int nz = 1) { return dim3((units + U::G - 1) / U::G, nb, nz); }

// Launches the kernel-spectrum passes of `a` (H, or the derivative that
// kernel_dz names) through Hr into a.hh.
template <int P> inline void rs_spectrum_launch(const RsArgs& a, int nb, hipStream_t st) {
  hipLaunchKernelGGL((rs_hrow_kernel<P, 0>), rs_grid<UHrow<P>>(rs_rows4(a.n), nb), dim3(UHrow<P>::NT), 0, st, a);
  hipLaunchKernelGGL(rs_hcol_kernel<P>, rs_grid<UHcol<P>>(P / 2 + 1, nb), dim3(UHcol<P>::NT), 0, st, a);
}

// The kernel-spectrum passes of a call that keeps or reuses spectra: the
// derivative spectra it asks for, and (unless an earlier call built it) Hhat
// with the derivatives of a forward call that will be differentiated.
template <int P>
inline void rs_kept_spectra_launch(const RsArgs& a, int nb, hipStream_t st) {
  const dim3 ghr = rs_grid<UHrow<P>>(rs_rows4(a.n), nb), bhr(UHrow<P>::NT), ghc = rs_grid<UHcol<P>>(P / 2 + 1, nb),
             bhc(UHcol<P>::NT);
  // a forward call that keeps its spectra for a gradient builds the derivative
  // spectra with its own kernel rows (one float64 geometry for all of them)
  const int dm = (a.dg[0] ? 1 : 0) | (a.dg[1] ? 2 : 0);
  const bool with_h = a.spec_mode == 1 && dm && !a.hreuse;
  if ((a.spec_mode == 2 && !a.dg_built) || (a.spec_mode == 1 && dm && !with_h)) {
    // derivative spectra (dH/dz, dH/dk) with the spectrum passes, unconjugated
    for (int i = 0; i < 2; ++i) {
      if (!a.dg[i]) continue;
      RsArgs d = a;
      d.hh = a.dg[i];
      d.kernel_dz = i + 1;
      d.adjoint = 0;
      d.hstored = 1;
      KTimer t(K_RS_HROW, st);
      rs_spectrum_launch<P>(d, nb, st);
    }
  }
  if (a.hreuse) return;
  {
    KTimer t(K_RS_HROW, st);
    if (with_h && dm == 1)
      hipLaunchKernelGGL((rs_hrow_kernel<P, 1>), ghr, bhr, 0, st, a);
    else if (with_h && dm == 2)
      hipLaunchKernelGGL((rs_hrow_kernel<P, 2>), ghr, bhr, 0, st, a);
    else if (with_h)
      hipLaunchKernelGGL((rs_hrow_kernel<P, 3>), ghr, bhr, 0, st, a);
    else
      hipLaunchKernelGGL((rs_hrow_kernel<P, 0>), ghr, bhr, 0, st, a);
  }
  KTimer t(K_RS_HCOL, st);
  hipLaunchKernelGGL(rs_hcol_kernel<P>, ghc, bhc, 0, st, a);
  for (int i = 0; with_h && i < 2; ++i) {
    if (!a.dg[i]) continue;
    RsArgs d = a;   // the derivative row transforms, unconjugated
    d.hr = d.hr2 = a.dgr[i];
    d.hh = a.dg[i];
    d.adjoint = 0;
    d.hstored = 1;
    hipLaunchKernelGGL(rs_hcol_kernel<P>, ghc, bhc, 0, st, d);
  }
}

// All passes up to the column pass.  KEEP: calls that keep or reuse spectra
// (hhat, spec) run at this length.
template <int P, bool KEEP>
inline void rs_launch(const RsArgs& a, hipStream_t st) {
  const int rows = rs_rows4(a.n);
  const int nb = a.batch > 1 ? a.batch : 1;
  // Hr may lie in the tiles that rs_urow fills later, so the spectra come first
  if (KEEP && (a.hstored || a.spec_mode)) {
    if constexpr (KEEP) rs_kept_spectra_launch<P>(a, nb, st);
  } else {
    {
      KTimer t(K_RS_HROW, st);
      hipLaunchKernelGGL((rs_hrow_kernel<P, 0>), rs_grid<UHrow<P>>(rows, nb), dim3(UHrow<P>::NT), 0, st, a);
    }
    KTimer t(K_RS_HCOL, st);
    hipLaunchKernelGGL(rs_hcol_kernel<P>, rs_grid<UHcol<P>>(P / 2 + 1, nb), dim3(UHcol<P>::NT), 0, st, a);
  }
  {
    KTimer t(K_RS_UROW, st);
    // plain inputs (no masks, no Ez): one block per (row, component), where
    // the row blocks alone leave resident slots empty, and at P = 4096 (two
    // rows per block: 69 us against 84 us at 2048^2, three components)
    const bool one = a.ncomp > 1 && a.nin == a.ncomp && a.ez_mode == EZ_NONE && !a.mask.st[0].kind &&
                     !a.mask.st[1].kind && (P >= 4096 || rows * nb < 2048);
    using U1 = UUrow<P, true>;
    using U3 = UUrow<P, false>;
    const bool comps = P <= 512 && a.ncomp > 1 && !one && (P <= 256 || rows * nb <= 2048);
    if (one) hipLaunchKernelGGL((rs_urow_kernel<P, true>), rs_grid<U1>(rows, nb, a.ncomp), dim3(U1::NT), 0, st, a);
    else if (!comps) hipLaunchKernelGGL((rs_urow_kernel<P, false>), rs_grid<U3>(rows, nb), dim3(U3::NT), 0, st, a);
    if constexpr (P <= 512)
      if (comps) hipLaunchKernelGGL(rs_urow_comps_kernel<P>, dim3(rows, nb), dim3(a.ncomp * rs_tpf(P)), 0, st, a);
  }
  {
    KTimer t(K_RS_COL, st);
    bool done = false;
    if constexpr (KEEP) {
      using UK = UCol<P, true>;
      const dim3 grid = rs_grid<UK>(P, nb, a.ncomp), blk(UK::NT);
      const int gb = a.spec_mode == 2 ? (a.dg[0] ? 1 : 0) | (a.dg[1] ? 2 : 0) : 0;
      done = a.spec_mode == 1 || gb != 0;
      if (a.spec_mode == 1) hipLaunchKernelGGL((rs_col_kernel<P, 1>), grid, blk, 0, st, a);
      else if (gb == 1) hipLaunchKernelGGL((rs_col_kernel<P, 3>), grid, blk, 0, st, a);
      else if (gb == 2) hipLaunchKernelGGL((rs_col_kernel<P, 4>), grid, blk, 0, st, a);
      else if (gb == 3) hipLaunchKernelGGL((rs_col_kernel<P, 5>), grid, blk, 0, st, a);
    }
    using U0 = UCol<P, false>;
    if (!done) hipLaunchKernelGGL((rs_col_kernel<P, 0>), rs_grid<U0>(P, nb, a.ncomp), dim3(U0::NT), 0, st, a);
  }
  if (KEEP && a.spec_mode == 2 && !a.partials_only) {
    KTimer t(K_LOSS, st);
    hipLaunchKernelGGL(rs_grad_reduce_kernel, dim3(2), dim3(1024), 0, st, a.gpart[0], a.gpart[1], P * a.ncomp,
                       a.grad_out);
  }
}

// The last pass of a call that returns the field.
template <int P>
inline void rs_final_launch(const RsArgs& a, hipStream_t st) {
  const int nb = a.batch > 1 ? a.batch : 1;
  KTimer t(K_RS_FINAL, st);
  const dim3 blk(UFinal<P>::NT);
  if (a.intensity)
    hipLaunchKernelGGL((rs_final_kernel<P, false>), rs_grid<UFinal<P>>(a.n, nb), blk, 0, st, a);
  else
    hipLaunchKernelGGL((rs_final_kernel<P, true>), rs_grid<UFinal<P>>(a.n, nb, a.ncomp), blk, 0, st, a);
}

}  // namespace xl
