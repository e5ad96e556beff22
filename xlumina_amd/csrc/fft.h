// LDS-staged Stockham FFT building blocks for gfx950 (64-wide waves).
//
// A workgroup runs one or more independent complex64 FFTs of length L = 2^k
// (64..4096), 3 * 2^k or 5 * 2^k, each on TPF threads, one butterfly per thread
// and pass: radix 16 at the powers of two with a final radix 2/4/8 when log2(L)
// is not a multiple of 4, the mixed radices of FftPlan at the others.  Data
// lives in LDS between passes (natural order in, natural order out); each
// thread keeps its R points of a butterfly in registers.  LDS indices are
// padded by one slot per 16 complex values so the stride-16 writes of the
// first pass spread over the banks.
//
// Inter-pass twiddles come from tables e^{-2 pi i k/N} (N = 4096, 3072, 2560)
// generated once per device in float64 (xl_fft_init_kernel).  A butterfly
// loads w (mixed radices: w and w^4) and forms the other powers by complex
// products.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace xl {

constexpr int TWN = 4096;                 // twiddle table length == max FFT length
constexpr int TWN3 = 3072;                // table for the lengths 3 * 2^k
constexpr int TWN5 = 2560;                // table for the lengths 5 * 2^k
constexpr int MAX_FFT = 4096;

__device__ float2 g_tw[TWN];              // e^{-2 pi i k / TWN}, float64-generated
__device__ float2 g_tw3[TWN3];            // e^{-2 pi i k / TWN3}, float64-generated
__device__ float2 g_tw5[TWN5];            // e^{-2 pi i k / TWN5}, float64-generated

__global__ void xl_fft_init_kernel() {
  int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < TWN) {
    double s, c;
    sincospi(-2.0 * (double)k / (double)TWN, &s, &c);
    g_tw[k] = make_float2((float)c, (float)s);
  }
  if (k < TWN3) {
    double s, c;
    sincospi(-2.0 * (double)k / (double)TWN3, &s, &c);
    g_tw3[k] = make_float2((float)c, (float)s);
  }
  if (k < TWN5) {
    double s, c;
    sincospi(-2.0 * (double)k / (double)TWN5, &s, &c);
    g_tw5[k] = make_float2((float)c, (float)s);
  }
}

// Lengths are 2^k (64..4096), 3 * 2^k (768..3072) and 5 * 2^k (1280, 2560);
// the latter two take their twiddles from tables of their own.
template <int L> struct Tw {
  static constexpr bool TRI = L % 3 == 0, PENT = L % 5 == 0;
  static constexpr int N = TRI ? TWN3 : PENT ? TWN5 : TWN;
  __device__ static float2 at(int i) { return TRI ? g_tw3[i] : PENT ? g_tw5[i] : g_tw[i]; }
};

constexpr int ilog2c(int x) { return x <= 1 ? 0 : 1 + ilog2c(x / 2); }

// Pass sequence of an L-point FFT on TPF threads; the inverse runs the same
// radices in reverse order, so the last forward pass and the first inverse
// pass share one register layout.
//   2^k                               16, ..., 16, REM
//   3072, 1536 with TPF = L/12        12, 16 or 8, 16
//   2560, 1280 (TPF = L/10)           10, 16 or 8, 16
//   3 * 2^k otherwise (TPF = L/16)    3, 16, ..., 16, REM
// All but the last kind split a zero upper half of the inputs, or a cropped
// upper half of the outputs, evenly in their first and last passes.  (The odd
// radix last at 2560 and 3072, on L/16 threads: rs_final of VRS 1200^2 21 -> 35
// us, the rest equal.)
template <int L, int TPF> struct FftPlan {
  static constexpr bool TRI = L % 3 == 0, PENT = L % 5 == 0;
  static constexpr bool MIXED = PENT || (TRI && TPF * 12 == L);
  static constexpr bool EVEN = !TRI || MIXED;
  static constexpr int ODD = TRI ? 12 : 10;
  static constexpr int L2 = TRI ? L / 3 : L;
  static constexpr int LG = ilog2c(L2);
  static constexpr int N16 = LG / 4;
  static constexpr int REM = 1 << (LG % 4);
  static constexpr int NP = MIXED ? 3 : (TRI ? 1 : 0) + N16 + (REM > 1 ? 1 : 0);
  static constexpr int fwd_radix(int i) {
    if (MIXED) return i == 0 ? ODD : i == 2 ? 16 : L / (ODD * 16);
    if (TRI) {
      if (i == 0) return 3;
      i -= 1;
    }
    return i < N16 ? 16 : REM;
  }
  static constexpr int radix(bool fwd, int i) { return fwd ? fwd_radix(i) : fwd_radix(NP - 1 - i); }
  static constexpr int ns(bool fwd, int i) {
    int p = 1;
    for (int k = 0; k < i; ++k) p *= radix(fwd, k);
    return p;
  }
  // register layout at the forward/inverse hand-off
  static constexpr int RH = radix(true, NP - 1);
  static constexpr int NBH = L / RH;
};

__device__ __forceinline__ int lpad(int i) { return i + (i >> 4); }
template <int L> struct LdsLen { static constexpr int value = L + L / 16; };
// lpad(i + k) - lpad(i) for a constant k, where no carry from the low four
// bits depends on i: a pass adds it to one address per thread (left to the
// compiler, some passes formed every second address by itself and wrote
// unpaired: czt_rows<2048>, 400 rows, one in ten us).
__host__ __device__ constexpr int lstep(int k) { return k + (k >> 4); }
// Whether that holds for the outputs idxD + r NS of a radix-R pass of stride
// NS (idxD = (j / NS) NS R + j % NS).
constexpr bool lpad_flat(int NS, int R) { return NS % 16 == 0 || ((NS & (NS - 1)) == 0 && NS * R % 16 == 0); }

__device__ __forceinline__ float2 operator+(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 operator-(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ float2 operator*(float2 a, float s) { return make_float2(a.x * s, a.y * s); }
__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
  return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
// a * conj(b)
__device__ __forceinline__ float2 cmulc(float2 a, float2 b) {
  return make_float2(a.x * b.x + a.y * b.y, a.y * b.x - a.x * b.y);
}
__device__ __forceinline__ float2 conjf2(float2 a) { return make_float2(a.x, -a.y); }
template <bool INV> __device__ __forceinline__ float2 twmul(float2 v, float2 w) {
  return INV ? cmulc(v, w) : cmul(v, w);
}

// cos / sin of 2 pi q / 16, q = 0..7
__device__ constexpr float kC16[8] = {1.0f, 0.92387953251128674f, 0.70710678118654752f, 0.38268343236508978f,
                                      0.0f, -0.38268343236508978f, -0.70710678118654752f, -0.92387953251128674f};
__device__ constexpr float kS16[8] = {0.0f, 0.38268343236508978f, 0.70710678118654752f, 0.92387953251128674f,
                                      1.0f, 0.92387953251128674f, 0.70710678118654752f, 0.38268343236508978f};

// v * e^{-+ 2 pi i q / 16} with q a compile-time constant after unrolling.
template <bool INV> __device__ __forceinline__ float2 rot16(float2 v, int q) {
  if (q == 0) return v;
  if (q == 4) return INV ? make_float2(-v.y, v.x) : make_float2(v.y, -v.x);
  const float c = kC16[q], s = INV ? kS16[q] : -kS16[q];
  return make_float2(v.x * c - v.y * s, v.x * s + v.y * c);
}

// In-register DFT of R points (R = 1, 2, 4, 8, 16), natural order in and out.
template <int R, bool INV> struct DFT {
  __device__ __forceinline__ static void run(float2* v) {
    float2 e[R / 2], o[R / 2];
#pragma unroll
    for (int i = 0; i < R / 2; ++i) { e[i] = v[2 * i]; o[i] = v[2 * i + 1]; }
    DFT<R / 2, INV>::run(e);
    DFT<R / 2, INV>::run(o);
#pragma unroll
    for (int k = 0; k < R / 2; ++k) {
      const float2 t = rot16<INV>(o[k], k * (16 / R));
      v[k] = e[k] + t;
      v[k + R / 2] = e[k] - t;
    }
  }
};
template <bool INV> struct DFT<1, INV> {
  __device__ __forceinline__ static void run(float2*) {}
};
// DFT of R points whose upper half v[R/2..R-1] is zero (a zero-padded
// input): the bottom radix-2 stage of the recursion is a copy.
template <int R, bool INV> struct DFTHalf {
  __device__ __forceinline__ static void run(float2* v) {
    float2 e[R / 2], o[R / 2];
#pragma unroll
    for (int i = 0; i < R / 2; ++i) { e[i] = v[2 * i]; o[i] = v[2 * i + 1]; }
    DFTHalf<R / 2, INV>::run(e);
    DFTHalf<R / 2, INV>::run(o);
#pragma unroll
    for (int k = 0; k < R / 2; ++k) {
      const float2 t = rot16<INV>(o[k], k * (16 / R));
      v[k] = e[k] + t;
      v[k + R / 2] = e[k] - t;
    }
  }
};
template <bool INV> struct DFTHalf<2, INV> {
  __device__ __forceinline__ static void run(float2* v) { v[1] = v[0]; }
};
// DFT of R points of which only the lower half of the outputs is kept
// (a cropped output): the top radix-2 stage forms v[0..R/2-1] only.
template <int R, bool INV> struct DFTLow {
  __device__ __forceinline__ static void run(float2* v) {
    float2 e[R / 2], o[R / 2];
#pragma unroll
    for (int i = 0; i < R / 2; ++i) { e[i] = v[2 * i]; o[i] = v[2 * i + 1]; }
    DFT<R / 2, INV>::run(e);
    DFT<R / 2, INV>::run(o);
#pragma unroll
    for (int k = 0; k < R / 2; ++k) v[k] = e[k] + rot16<INV>(o[k], k * (16 / R));
  }
};

// X1,2 = a - (b + c)/2 -+ i (sqrt(3)/2)(b - c) (signs swapped for the inverse).
template <bool INV> struct DFT<3, INV> {
  __device__ __forceinline__ static void run(float2* v) {
    const float2 a = v[0], t1 = v[1] + v[2], d = v[1] - v[2];
    const float2 t2 = a - t1 * 0.5f;
    const float h = 0.86602540378443865f;
    const float2 m = make_float2(-d.y * h, d.x * h);   // i h d
    v[0] = a + t1;
    v[1] = INV ? t2 + m : t2 - m;
    v[2] = INV ? t2 - m : t2 + m;
  }
};

// Radix 5 (Winograd's sums, cos / sin of 72 and 144 degrees).
template <bool INV> struct DFT<5, INV> {
  __device__ __forceinline__ static void run(float2* v) {
    const float c1 = 0.30901699437494742f, c2 = -0.80901699437494742f;
    const float s1 = 0.95105651629515357f, s2 = 0.58778525229247313f;
    const float2 a = v[0], t1 = v[1] + v[4], t2 = v[2] + v[3], t3 = v[1] - v[4], t4 = v[2] - v[3];
    const float2 m1 = a + t1 * c1 + t2 * c2, m2 = a + t1 * c2 + t2 * c1;
    const float2 n1 = t3 * s1 + t4 * s2, n2 = t3 * s2 - t4 * s1;
    const float2 j1 = make_float2(-n1.y, n1.x), j2 = make_float2(-n2.y, n2.x);   // i n
    v[0] = a + t1 + t2;
    v[1] = INV ? m1 + j1 : m1 - j1;
    v[4] = INV ? m1 - j1 : m1 + j1;
    v[2] = INV ? m2 + j2 : m2 - j2;
    v[3] = INV ? m2 - j2 : m2 + j2;
  }
};

// cos / sin of 2 pi q / R for the even radices 6, 10 and 12, q < R / 2.
template <int R> struct Rot;
template <> struct Rot<6> {
  __device__ static constexpr float c(int q) { constexpr float t[3] = {1.f, 0.5f, -0.5f}; return t[q]; }
  __device__ static constexpr float s(int q) {
    constexpr float t[3] = {0.f, 0.86602540378443865f, 0.86602540378443865f};
    return t[q];
  }
};
template <> struct Rot<10> {
  __device__ static constexpr float c(int q) {
    constexpr float t[5] = {1.f, 0.80901699437494742f, 0.30901699437494742f, -0.30901699437494742f, -0.80901699437494742f};
    return t[q];
  }
  __device__ static constexpr float s(int q) {
    constexpr float t[5] = {0.f, 0.58778525229247313f, 0.95105651629515357f, 0.95105651629515357f, 0.58778525229247313f};
    return t[q];
  }
};
template <> struct Rot<12> {
  __device__ static constexpr float c(int q) {
    constexpr float t[6] = {1.f, 0.86602540378443865f, 0.5f, 0.f, -0.5f, -0.86602540378443865f};
    return t[q];
  }
  __device__ static constexpr float s(int q) {
    constexpr float t[6] = {0.f, 0.5f, 0.86602540378443865f, 1.f, 0.86602540378443865f, 0.5f};
    return t[q];
  }
};
// v e^{-+ 2 pi i q / R}, q a constant after unrolling
template <int R, bool INV> __device__ __forceinline__ float2 rot_r(float2 v, int q) {
  if (q == 0) return v;
  if (4 * q == R) return INV ? make_float2(-v.y, v.x) : make_float2(v.y, -v.x);
  const float c = Rot<R>::c(q), s = INV ? Rot<R>::s(q) : -Rot<R>::s(q);
  return make_float2(v.x * c - v.y * s, v.x * s + v.y * c);
}

// DFT of R = 2 M points (R = 6, 10, 12) from two of M, even and odd inputs.
template <int R, bool INV, bool LOW> __device__ __forceinline__ void dft_even(float2* v) {
  constexpr int M = R / 2;
  float2 e[M], o[M];
#pragma unroll
  for (int i = 0; i < M; ++i) { e[i] = v[2 * i]; o[i] = v[2 * i + 1]; }
  DFT<M, INV>::run(e);
  DFT<M, INV>::run(o);
#pragma unroll
  for (int k = 0; k < M; ++k) {
    const float2 t = rot_r<R, INV>(o[k], k);
    v[k] = e[k] + t;
    if (!LOW) v[k + M] = e[k] - t;
  }
}
template <bool INV> struct DFT<6, INV> { __device__ __forceinline__ static void run(float2* v) { dft_even<6, INV, false>(v); } };
template <bool INV> struct DFT<10, INV> { __device__ __forceinline__ static void run(float2* v) { dft_even<10, INV, false>(v); } };
template <bool INV> struct DFT<12, INV> { __device__ __forceinline__ static void run(float2* v) { dft_even<12, INV, false>(v); } };
template <bool INV> struct DFTLow<10, INV> { __device__ __forceinline__ static void run(float2* v) { dft_even<10, INV, true>(v); } };
template <bool INV> struct DFTLow<12, INV> { __device__ __forceinline__ static void run(float2* v) { dft_even<12, INV, true>(v); } };
// Upper half zero: even outputs are the DFT of the M inputs, odd outputs that
// of the inputs turned by w^r.
template <int R, bool INV> __device__ __forceinline__ void dft_half_even(float2* v) {
  constexpr int M = R / 2;
  float2 e[M], o[M];
#pragma unroll
  for (int i = 0; i < M; ++i) { e[i] = v[i]; o[i] = rot_r<R, INV>(v[i], i); }
  DFT<M, INV>::run(e);
  DFT<M, INV>::run(o);
#pragma unroll
  for (int i = 0; i < M; ++i) { v[2 * i] = e[i]; v[2 * i + 1] = o[i]; }
}
template <bool INV> struct DFTHalf<10, INV> { __device__ __forceinline__ static void run(float2* v) { dft_half_even<10, INV>(v); } };
template <bool INV> struct DFTHalf<12, INV> { __device__ __forceinline__ static void run(float2* v) { dft_half_even<12, INV>(v); } };

// v[r] *= w^r for r < R (w1 = w, e^{-+2 pi i base / TWN}, one table entry);
// w^2, w^4, w^8 by squaring and the other powers as products formed next to
// their use, so that only the four bases stay live.  Loads cost more than the
// products here (each is a scattered L1 access per lane); the squarings add
// at most a few float32 ulps to w^8.  T4 (the mixed-radix plans): w^4 is a table
// entry too (wt4), which halves the error of the upper powers.
template <int R, bool INV, bool T4 = false>
__device__ __forceinline__ void apply_twiddles_w(float2* v, const float2 w1, const float2 wt4 = float2()) {
  if constexpr (R == 3) {
    v[1] = twmul<INV>(v[1], w1);
    v[2] = twmul<INV>(v[2], cmul(w1, w1));
  } else if constexpr (R == 10 || R == 12) {
    const float2 w2 = cmul(w1, w1), w3 = cmul(w1, w2), w8 = cmul(wt4, wt4);
    v[1] = twmul<INV>(v[1], w1);
    v[2] = twmul<INV>(v[2], w2);
    v[3] = twmul<INV>(v[3], w3);
    v[4] = twmul<INV>(v[4], wt4);
    v[5] = twmul<INV>(v[5], cmul(w1, wt4));
    v[6] = twmul<INV>(v[6], cmul(w2, wt4));
    v[7] = twmul<INV>(v[7], cmul(w3, wt4));
    v[8] = twmul<INV>(v[8], w8);
    v[9] = twmul<INV>(v[9], cmul(w1, w8));
    if constexpr (R == 12) {
      v[10] = twmul<INV>(v[10], cmul(w2, w8));
      v[11] = twmul<INV>(v[11], cmul(w3, w8));
    }
  } else if constexpr (R >= 2) {
    v[1] = twmul<INV>(v[1], w1);
    if constexpr (R >= 4) {
      const float2 w2 = cmul(w1, w1);
      v[2] = twmul<INV>(v[2], w2);
      const float2 w3 = cmul(w1, w2);
      v[3] = twmul<INV>(v[3], w3);
      if constexpr (R >= 8) {
        const float2 w4 = T4 ? wt4 : cmul(w2, w2);
        v[4] = twmul<INV>(v[4], w4);
        v[5] = twmul<INV>(v[5], cmul(w1, w4));
        v[6] = twmul<INV>(v[6], cmul(w2, w4));
        const float2 w7 = cmul(w3, w4);
        v[7] = twmul<INV>(v[7], w7);
        if constexpr (R >= 16) {
          const float2 w8 = cmul(w4, w4);
          v[8] = twmul<INV>(v[8], w8);
          v[9] = twmul<INV>(v[9], cmul(w1, w8));
          v[10] = twmul<INV>(v[10], cmul(w2, w8));
          v[11] = twmul<INV>(v[11], cmul(w3, w8));
          v[12] = twmul<INV>(v[12], cmul(w4, w8));
          v[13] = twmul<INV>(v[13], cmul(cmul(w1, w4), w8));
          v[14] = twmul<INV>(v[14], cmul(cmul(w2, w4), w8));
          v[15] = twmul<INV>(v[15], cmul(w7, w8));
        }
      }
    }
  }
}

template <int R, bool INV, int L> __device__ __forceinline__ void apply_twiddles(float2* v, int base) {
  static_assert(R != 10 && R != 12, "the mixed-radix plans load their bases ahead (TwSet)");
  apply_twiddles_w<R, INV>(v, Tw<L>::at(base));
}

// One Stockham radix-R pass of an L-point FFT over TPF threads (thread t).
// GUARD: the block has more than TPF threads; the others only join the
// barriers.
template <int L, int R, int NS, int TPF, bool INV, bool GUARD = false>
__device__ __forceinline__ void stockham_pass(float2* s, int t) {
  constexpr int NB = L / R;
  constexpr int BPT = (NB + TPF - 1) / TPF;
  float2 v[BPT][R];
  const bool act = !GUARD || t < TPF;
#pragma unroll
  for (int b = 0; b < BPT; ++b) {
    const int j = t + b * TPF;
    if (act && (NB % TPF == 0 || j < NB)) {
#pragma unroll
      for (int r = 0; r < R; ++r) v[b][r] = NB % 16 ? s[lpad(j + r * NB)] : s[lpad(j) + lstep(r * NB)];
      if constexpr (NS > 1) apply_twiddles<R, INV, L>(v[b], (j % NS) * (Tw<L>::N / (NS * R)));
      DFT<R, INV>::run(v[b]);
    }
  }
  __syncthreads();
#pragma unroll
  for (int b = 0; b < BPT; ++b) {
    const int j = t + b * TPF;
    if (act && (NB % TPF == 0 || j < NB)) {
      const int idxD = (j / NS) * NS * R + (j % NS);
#pragma unroll
      for (int r = 0; r < R; ++r) s[lpad_flat(NS, R) ? lpad(idxD) + lstep(r * NS) : lpad(idxD + r * NS)] = v[b][r];
    }
  }
  __syncthreads();
}

template <int L, int TPF, bool INV, int I = 0, bool GUARD = false>
__device__ __forceinline__ void fft_lds(float2* s, int t) {
  using PL = FftPlan<L, TPF>;
  if constexpr (I < PL::NP) {
    stockham_pass<L, PL::radix(true, I), PL::ns(true, I), TPF, INV, GUARD>(s, t);
    fft_lds<L, TPF, INV, I + 1, GUARD>(s, t);
  }
}

// Block-index remap so that consecutive logical blocks (which share 128-byte
// lines of the tiled intermediates) land on the same XCD: hardware dispatches
// block b to XCD b % 8, whose blocks take one contiguous logical range (the
// first nblocks % 8 ranges are one block longer).
__device__ __forceinline__ int xcd_remap(int b, int nblocks) {
  constexpr int NX = 8;
  const int x = b % NX, rem = nblocks % NX;
  return x * (nblocks / NX) + (x < rem ? x : rem) + b / NX;
}

// --- float64 phase helpers ---------------------------------------------------
// e^{i 2 pi t} for a float64 number of turns t: the integer part is removed in
// float64, the remainder in [-1/2, 1/2] goes to float32 sincospi.
__device__ __forceinline__ float2 expi_turns(double t) {
  const double f = t - rint(t);
  float s, c;
  sincospif((float)(2.0 * f), &s, &c);
  return make_float2(c, s);
}

}  // namespace xl
