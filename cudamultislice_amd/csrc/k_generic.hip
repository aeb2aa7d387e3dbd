// k_generic.hip -- 2D FFT and pointwise hooks for grids whose sides are not
// both powers of two (the reference's cuFFT plan takes any resX x resY,
// U.cu:1961; its GUI offers 4008x2672, 2004x1336 and 1002x668, MW.cs:147-149).
//
// A line of any length n is transformed as a chirp convolution (Bluestein,
// 1970): with c_k = exp(-i pi k^2 / n),
//   X_j = c_j sum_k (x_k c_k) conj(c_{j-k}),
// a cyclic convolution of length M, the power of two from 2 n - 1 up: two
// transforms of length M in registers and LDS and a product with the
// precomputed transform of the chirp.  It costs the same for every n, primes
// included, and a whole line stays in one workgroup, so one launch does what
// the passes of the power-of-two grids do: rows with the transmission
// multiply, columns with the k-space factor between the forward and the
// inverse transform.  A side that is a power of two from 64 up is
// transformed directly (M = n).
//
// The transforms run in FP64, whose multiply-adds issue at the rate of
// unpacked FP32 here.  In FP32 (same times) the chirp form is as close per
// transform as a direct one (1.5e-7), but a plane wave meets the same
// rounding errors at every slice and they add up: 1.7e-5 after 37 slices of
// 2004 x 1336, against 2.7e-6 for what this replaced (one launch per prime
// factor over global memory with direct sums over the factor); in FP64 the
// exit wave of 1002 x 668 is within 1e-7 of the 64-bit one, before 4.6e-6.
// One wave of 1002 x 668 (M = 2048): rows 18.3 us, columns forward and back
// 33.7 us, 70 us per slice where ten launches of 63 us stood before.  Bound
// by LDS exchanges and their barriers at two waves per SIMD (170-242 VGPRs).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <complex>
#include <type_traits>
#include <utility>
#include <vector>

#include "msl_fft.hpp"
#include "msl_internal.hpp"

namespace msl {

namespace {

inline long long gnblk(long long n, int b) { return (n + b - 1) / b; }

// transforms of length M: T threads of E = M / T values, up to four radix
// stages (msl_fft.hpp's canonical order: thread t holds elements t + c T)
template <int M> struct GPlan;
template <> struct GPlan<64> { static constexpr int T = 8, R1 = 8, R2 = 8, R3 = 1, R4 = 1; };
template <> struct GPlan<128> { static constexpr int T = 8, R1 = 16, R2 = 8, R3 = 1, R4 = 1; };
template <> struct GPlan<256> { static constexpr int T = 16, R1 = 16, R2 = 16, R3 = 1, R4 = 1; };
template <> struct GPlan<512> { static constexpr int T = 64, R1 = 8, R2 = 8, R3 = 8, R4 = 1; };
template <> struct GPlan<1024> { static constexpr int T = 64, R1 = 16, R2 = 8, R3 = 8, R4 = 1; };
template <> struct GPlan<2048> { static constexpr int T = 128, R1 = 16, R2 = 16, R3 = 8, R4 = 1; };
template <> struct GPlan<4096> { static constexpr int T = 256, R1 = 16, R2 = 16, R3 = 16, R4 = 1; };
template <> struct GPlan<8192> { static constexpr int T = 512, R1 = 16, R2 = 16, R3 = 16, R4 = 2; };
template <> struct GPlan<16384> { static constexpr int T = 1024, R1 = 16, R2 = 16, R3 = 16, R4 = 4; };

__device__ __forceinline__ double2 operator+(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 operator-(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ double2 mul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 wide(float2 a) { return make_double2(a.x, a.y); }
// a exp(DIR i pi / 2)
template <int DIR> __device__ __forceinline__ double2 quarter(double2 a) {
  return DIR < 0 ? make_double2(a.y, -a.x) : make_double2(-a.y, a.x);
}

// HALF: the upper half of the inputs is zero (a line padded to M >= 2 n - 1)
template <int DIR, bool HALF = false>
__device__ __forceinline__ void gdft4(double2& a0, double2& a1, double2& a2, double2& a3) {
  const double2 t0 = HALF ? a0 : a0 + a2, t1 = HALF ? a0 : a0 - a2;
  const double2 t2 = HALF ? a1 : a1 + a3, t3 = quarter<DIR>(HALF ? a1 : a1 - a3);
  a0 = t0 + t2;
  a2 = t0 - t2;
  a1 = t1 + t3;
  a3 = t1 - t3;
}
template <int R, int DIR, bool HALF> __device__ __forceinline__ void gdft(double2 (&a)[R]) {
  constexpr double h = 0.70710678118654752440;
  if constexpr (R == 2) {
    const double2 t = a[0];
    a[0] = t + a[1];
    a[1] = t - a[1];
  } else if constexpr (R == 4) {
    gdft4<DIR, HALF>(a[0], a[1], a[2], a[3]);
  } else if constexpr (R == 8) {
    double2 e[4] = {a[0], a[2], a[4], a[6]}, o[4] = {a[1], a[3], a[5], a[7]};
    gdft4<DIR, HALF>(e[0], e[1], e[2], e[3]);
    gdft4<DIR, HALF>(o[0], o[1], o[2], o[3]);
    o[1] = mul(o[1], make_double2(h, DIR * h));
    o[2] = quarter<DIR>(o[2]);
    o[3] = mul(o[3], make_double2(-h, DIR * h));
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      a[k] = e[k] + o[k];
      a[k + 4] = e[k] - o[k];
    }
  } else {
    constexpr double c1 = 0.92387953251128675613, s1 = 0.38268343236508977173;
#pragma unroll
    for (int n = 0; n < 4; ++n) gdft4<DIR, HALF>(a[n], a[n + 4], a[n + 8], a[n + 12]);
    const double2 w1 = make_double2(c1, DIR * s1), w2 = make_double2(h, DIR * h), w3 = make_double2(s1, DIR * c1);
    const double2 w6 = make_double2(-h, DIR * h), w9 = make_double2(-c1, -DIR * s1);
    a[5] = mul(a[5], w1);
    a[9] = mul(a[9], w2);
    a[13] = mul(a[13], w3);
    a[6] = mul(a[6], w2);
    a[10] = quarter<DIR>(a[10]);
    a[14] = mul(a[14], w6);
    a[7] = mul(a[7], w3);
    a[11] = mul(a[11], w6);
    a[15] = mul(a[15], w9);
#pragma unroll
    for (int k = 0; k < 4; ++k) gdft4<DIR>(a[4 * k], a[4 * k + 1], a[4 * k + 2], a[4 * k + 3]);
    double2 o[16];
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int q = 0; q < 4; ++q) o[k + 4 * q] = a[4 * k + q];
#pragma unroll
    for (int i = 0; i < 16; ++i) a[i] = o[i];
  }
}

// element p of a line in LDS: one element of padding per 16 spreads the
// stages' strides over the banks; columns interleave with stride C
__device__ __forceinline__ int gpad(int p) { return p + (p >> 4); }
template <int M> struct GLds {
  // 16384 elements of 16 bytes exceed the LDS: real and imaginary parts are
  // exchanged one after the other there
  static constexpr bool PARTS = M > 8192;
  static constexpr int N = M + M / 16;  // elements (parts) of a line
  using E = typename std::conditional<PARTS, double, double2>::type;
};

// the values v[b + m NB] of this thread's butterflies go to their output
// positions and come back in canonical order
template <int M, int R, int L, class S>
__device__ __forceinline__ void gexchange(double2 (&v)[M / GPlan<M>::T], int t, typename GLds<M>::E* lds, int stride) {
  constexpr int T = GPlan<M>::T, E = M / T, NB = E / R;
  auto pos = [&](int b, int m) {
    const int j = t + b * T, k = j & (L - 1);
    return gpad((j / L) * L * R + k + m * L) * stride;
  };
  if constexpr (GLds<M>::PARTS) {
#pragma unroll
    for (int part = 0; part < 2; ++part) {
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int m = 0; m < R; ++m) lds[pos(b, m)] = part ? v[b + m * NB].y : v[b + m * NB].x;
      S::sync();
#pragma unroll
      for (int c = 0; c < E; ++c) (part ? v[c].y : v[c].x) = lds[gpad(t + c * T) * stride];
      S::sync();
    }
  } else {
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int m = 0; m < R; ++m) lds[pos(b, m)] = v[b + m * NB];
    S::sync();
#pragma unroll
    for (int c = 0; c < E; ++c) v[c] = lds[gpad(t + c * T) * stride];
    S::sync();
  }
}

// one Stockham stage of radix R after L points; the powers of its twiddle
// are formed from one table entry per butterfly
template <int M, int R, int L, int DIR, bool HALF>
__device__ __forceinline__ void gstage(double2 (&v)[M / GPlan<M>::T], int t, const double2* __restrict__ tw) {
  constexpr int T = GPlan<M>::T, E = M / T, NB = E / R;
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    double2 a[R];
#pragma unroll
    for (int m = 0; m < R; ++m) a[m] = v[b + m * NB];
    if constexpr (L > 1) {
      double2 w = tw[((t + b * T) & (L - 1)) * (M / (L * R))];
      if (DIR > 0) w.y = -w.y;
      double2 p = w;
#pragma unroll
      for (int m = 1; m < R; ++m) {
        a[m] = mul(a[m], p);
        if (m + 1 < R) p = mul(p, w);
      }
    }
    gdft<R, DIR, HALF>(a);
#pragma unroll
    for (int m = 0; m < R; ++m) v[b + m * NB] = a[m];
  }
}

template <int M, int DIR, bool HALF, class S>
__device__ __forceinline__ void gen_fft(double2 (&v)[M / GPlan<M>::T], int t, const double2* __restrict__ tw,
                                        typename GLds<M>::E* lds, int stride) {
  using P = GPlan<M>;
  constexpr int R1 = P::R1, R2 = P::R2, R3 = P::R3, R4 = P::R4;
  gstage<M, R1, 1, DIR, HALF>(v, t, tw);
  gexchange<M, R1, 1, S>(v, t, lds, stride);
  gstage<M, R2, R1, DIR, false>(v, t, tw);
  if constexpr (R3 > 1) {
    gexchange<M, R2, R1, S>(v, t, lds, stride);
    gstage<M, R3, R1 * R2, DIR, false>(v, t, tw);
  }
  if constexpr (R4 > 1) {
    gexchange<M, R3, R1 * R2, S>(v, t, lds, stride);
    gstage<M, R4, R1 * R2 * R3, DIR, false>(v, t, tw);
  }
}

// unnormalised transform of length g.n of the line in v (element t + c T;
// elements from n on are ignored and left undefined); inverse: the conjugate
// of the transform of the conjugate.  A padded line has n <= M / 2: its
// upper half is neither read nor needed.
template <int M, bool BLUE, class S>
__device__ __forceinline__ void gen_line(double2 (&v)[M / GPlan<M>::T], int t, typename GLds<M>::E* lds, int stride,
                                         const GenLen& g, bool inverse) {
  constexpr int T = GPlan<M>::T, E = M / T, H = BLUE ? E / 2 : E;
  const double s = inverse ? -1.0 : 1.0;
#pragma unroll
  for (int c = 0; c < H; ++c) {
    v[c].y *= s;
    if constexpr (BLUE) {
      const int i = t + c * T;
      v[c] = i < g.n ? mul(v[c], g.chirp[i]) : make_double2(0.0, 0.0);
    }
  }
  gen_fft<M, -1, BLUE, S>(v, t, g.tw, lds, stride);
  if constexpr (BLUE) {
#pragma unroll
    for (int c = 0; c < E; ++c) v[c] = mul(v[c], g.filt[t + c * T]);
    gen_fft<M, +1, false, S>(v, t, g.tw, lds, stride);
  }
#pragma unroll
  for (int c = 0; c < H; ++c) {
    if constexpr (BLUE) {
      const int i = t + c * T;
      if (i < g.n) v[c] = mul(v[c], g.chirp[i]);
    }
    v[c].y *= s;
  }
}

template <int M> struct GenRow {
  static constexpr int T = GPlan<M>::T, E = M / T;
  static constexpr bool WAVE = T <= 64;
  static constexpr int LINES = 256 / T > 0 ? 256 / T : 1, THREADS = LINES * T;
};

template <int M, bool BLUE> __global__ void __launch_bounds__(GenRow<M>::THREADS) k_gen_row(GenRowArgs a) {
  using Cfg = GenRow<M>;
  using S = typename std::conditional<Cfg::WAVE, WaveSync, BlockSync>::type;
  constexpr int T = Cfg::T, E = Cfg::E, H = BLUE ? E / 2 : E;
  __shared__ typename GLds<M>::E lds[Cfg::LINES * GLds<M>::N];
  const int t = threadIdx.x % T, ln = threadIdx.x / T;
  const long long line = (long long)blockIdx.x * Cfg::LINES + ln;
  const bool ok = line < (long long)a.ny * a.nbatch;
  const long long o = ok ? line * a.nx : 0;
  const int n = a.len.n;
  double2 v[E];
#pragma unroll
  for (int c = 0; c < H; ++c) {
    const int i = t + c * T;
    v[c] = (ok && i < n) ? wide(a.src[o + i]) : make_double2(0.0, 0.0);
  }
  if (a.t) {
    const float2* tr = a.t + (ok ? line % a.ny : 0) * a.nx;
#pragma unroll
    for (int c = 0; c < H; ++c) {
      const int i = t + c * T;
      if (i < n) v[c] = mul(v[c], wide(tr[i]));
    }
  }
  gen_line<M, BLUE, S>(v, t, lds + ln * GLds<M>::N, 1, a.len, a.inverse != 0);
  if (!ok) return;
#pragma unroll
  for (int c = 0; c < H; ++c) {
    const int i = t + c * T;
    if (i >= n) continue;
    const float2 r = make_float2((float)v[c].x, (float)v[c].y);
    if (a.inten) a.inten[o + i] = r.x * r.x + r.y * r.y;
    if (a.dst) a.dst[o + i] = r;
    if (a.dst2) a.dst2[o + i] = r;
  }
}

// k-space factor of column x, row y (ColMul, scale included): CM_PROP the
// Fresnel propagator px[x] py[y] inside |k| < kmax (CreatePropsKernel,
// U.cu:419), CM_BAND the band limit |k| <= kmax (BandLimitKernel,
// U.cu:1037-1040), CM_GRAD -4 pi^2 k^2 (gradKernel, U.cu:959-960, pi =
// 3.14159f), CM_SCALE the scale only
__device__ __forceinline__ double2 gen_factor(const GenColArgs& a, int x, int y) {
  if (a.mul == CM_SCALE) return make_double2(a.scale, 0.0);
  const float kxv = a.kx[x], kyv = a.ky[y];
  const float k = sqrtf(kxv * kxv + kyv * kyv);
  if (a.mul == CM_PROP) {
    const double2 p = mul(wide(a.px[x]), wide(a.py[y]));
    const double m = k < a.kmax ? a.scale : 0.0;
    return make_double2(p.x * m, p.y * m);
  }
  if (a.mul == CM_GRAD) return make_double2(a.scale * (-4.f * 3.14159f * 3.14159f * (kxv * kxv + kyv * kyv)), 0.0);
  return make_double2(k <= a.kmax ? a.scale : 0.0, 0.0);
}

template <int M> struct GenCol {
  static constexpr int T = GPlan<M>::T, E = M / T;
  // 512 threads (1024 at 16384): the registers of two waves per SIMD, and at
  // most 139 KB of LDS
  static constexpr int C = M >= 8192 ? 1 : 512 / T < 16 ? 512 / T : 16, THREADS = C * T;
};

// columns: forward, inverse, or forward, factor, inverse (mode COL_FWD,
// COL_INV, COL_FWD_MUL_INV); C neighbouring columns per workgroup
template <int M, bool BLUE> __global__ void __launch_bounds__(GenCol<M>::THREADS) k_gen_col(GenColArgs a) {
  using Cfg = GenCol<M>;
  constexpr int T = Cfg::T, E = Cfg::E, C = Cfg::C, H = BLUE ? E / 2 : E;
  __shared__ typename GLds<M>::E lds[GLds<M>::N * C];
  const int col = threadIdx.x % C, t = threadIdx.x / C;
  const int x = blockIdx.x * C + col, n = a.len.n;
  const bool ok = x < a.nx;
  const long long o = (long long)blockIdx.y * a.nx * a.ny + (ok ? x : 0);
  double2 v[E];
#pragma unroll
  for (int c = 0; c < H; ++c) {
    const int y = t + c * T;
    v[c] = (ok && y < n) ? wide(a.src[o + (long long)y * a.nx]) : make_double2(0.0, 0.0);
  }
  // one copy of the transform serves both directions
  const int passes = a.mode == COL_FWD_MUL_INV ? 2 : 1;
#pragma unroll 1
  for (int p = 0; p < passes; ++p) {
    gen_line<M, BLUE, BlockSync>(v, t, lds + col, C, a.len, a.mode == COL_INV || p == 1);
    if (p == 0) {
#pragma unroll
      for (int c = 0; c < H; ++c) {
        const int y = t + c * T;
        if (y < n) v[c] = mul(v[c], gen_factor(a, ok ? x : 0, y));
      }
    }
  }
  if (!ok) return;
#pragma unroll
  for (int c = 0; c < H; ++c) {
    const int y = t + c * T;
    if (y < n) a.dst[o + (long long)y * a.nx] = make_float2((float)v[c].x, (float)v[c].y);
  }
}

template <int M> hipError_t gen_row_m(const GenRowArgs& a, hipStream_t s) {
  const dim3 grid((unsigned)gnblk((long long)a.ny * a.nbatch, GenRow<M>::LINES)), block(GenRow<M>::THREADS);
  if (a.len.chirp) hipLaunchKernelGGL((k_gen_row<M, true>), grid, block, 0, s, a);
  else if constexpr (M <= 8192) hipLaunchKernelGGL((k_gen_row<M, false>), grid, block, 0, s, a);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}
template <int M> hipError_t gen_col_m(const GenColArgs& a, hipStream_t s) {
  const dim3 grid((unsigned)gnblk(a.nx, GenCol<M>::C), a.nbatch), block(GenCol<M>::THREADS);
  if (a.len.chirp) hipLaunchKernelGGL((k_gen_col<M, true>), grid, block, 0, s, a);
  else if constexpr (M <= 8192) hipLaunchKernelGGL((k_gen_col<M, false>), grid, block, 0, s, a);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

bool len_ok(const GenLen& g, int n) {
  return g.n == n && n >= 1 && g.tw && (g.chirp ? g.filt && g.M >= 2 * n - 1 : g.M == n);
}

// in-place FFT of a power-of-two length in 64 bits (the tables)
void fft64(std::complex<double>* a, int n, const std::vector<double2>& tw) {
  for (int i = 1, j = 0; i < n; ++i) {
    int bit = n >> 1;
    for (; j & bit; bit >>= 1) j ^= bit;
    j ^= bit;
    if (i < j) std::swap(a[i], a[j]);
  }
  for (int len = 2; len <= n; len <<= 1)
    for (int i = 0; i < n; i += len)
      for (int k = 0; k < len / 2; ++k) {
        const std::complex<double> u = a[i + k], z = a[i + k + len / 2];
        const double2 q = tw[(size_t)k * (n / len)];
        const std::complex<double> v(z.real() * q.x - z.imag() * q.y,
                                     z.real() * q.y + z.imag() * q.x);
        a[i + k] = u + v;
        a[i + k + len / 2] = u - v;
      }
}

}  // namespace

int gen_fft_length(int n) {
  int M = 64;
  while (M < n) M <<= 1;
  if (M == n) return n;
  while (M < 2 * n - 1) M <<= 1;
  return M;
}

void gen_tables(int n, std::vector<double2>& tw, std::vector<double2>& chirp, std::vector<double2>& filt) {
  chirp.clear();
  filt.clear();
  const int M = gen_fft_length(n);
  tw.resize(M);
  for (int k = 0; k < M / 4; ++k) {  // M >= 64; the other quarters by rotation
    const double c = std::cos(2.0 * M_PI * k / M), s = std::sin(2.0 * M_PI * k / M);
    tw[k] = make_double2(c, -s);
    tw[k + M / 4] = make_double2(-s, -c);
    tw[k + M / 2] = make_double2(-c, s);
    tw[k + 3 * M / 4] = make_double2(s, c);
  }
  if (M == n) return;
  std::vector<std::complex<double>> b(M, 0.0);
  chirp.resize(n);
  filt.resize(M);
  for (int k = 0; k < n; ++k) {
    const long long q = (long long)k * k % (2LL * n);
    const std::complex<double> c = std::polar(1.0, -M_PI * (double)q / (double)n);
    chirp[k] = make_double2(c.real(), c.imag());
    b[k] = std::conj(c);
    if (k) b[M - k] = std::conj(c);
  }
  fft64(b.data(), M, tw);
  for (int k = 0; k < M; ++k) filt[k] = make_double2(b[k].real() / M, b[k].imag() / M);
}

#define MSL_GEN_LEN(F, A, S)                       \
  switch ((A).len.M) {                             \
    case 64: return F<64>(A, S);                   \
    case 128: return F<128>(A, S);                 \
    case 256: return F<256>(A, S);                 \
    case 512: return F<512>(A, S);                 \
    case 1024: return F<1024>(A, S);               \
    case 2048: return F<2048>(A, S);               \
    case 4096: return F<4096>(A, S);               \
    case 8192: return F<8192>(A, S);               \
    case 16384: return F<16384>(A, S);             \
  }                                                \
  return hipErrorInvalidValue

hipError_t launch_gen_row(const GenRowArgs& a, hipStream_t s) {
  if (!a.src || !(a.dst || a.inten) || a.ny < 1 || a.nbatch < 0 || !len_ok(a.len, a.nx)) return hipErrorInvalidValue;
  if (a.nbatch == 0) return hipSuccess;
  MSL_GEN_LEN(gen_row_m, a, s);
}

hipError_t launch_gen_col(const GenColArgs& a, hipStream_t s) {
  if (!a.src || !a.dst || a.nx < 1 || a.nbatch < 0 || !len_ok(a.len, a.ny)) return hipErrorInvalidValue;
  if (a.mode != COL_FWD && a.mode != COL_INV && a.mode != COL_FWD_MUL_INV) return hipErrorInvalidValue;
  if (a.mul != CM_SCALE && a.mul != CM_PROP && a.mul != CM_BAND && a.mul != CM_GRAD) return hipErrorInvalidValue;
  if (a.mul != CM_SCALE && (!a.kx || !a.ky)) return hipErrorInvalidValue;
  if (a.mul == CM_PROP && (!a.px || !a.py)) return hipErrorInvalidValue;
  const long long np = (long long)a.nx * a.ny;
  for (int b0 = 0; b0 < a.nbatch; b0 += 65535) {  // waves on grid.y
    GenColArgs c = a;
    c.nbatch = std::min(65535, a.nbatch - b0);
    c.src = a.src + b0 * np;
    c.dst = a.dst + b0 * np;
    const hipError_t e = [&]() -> hipError_t { MSL_GEN_LEN(gen_col_m, c, s); }();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}
#undef MSL_GEN_LEN

// per-block sums of scale |F|^2 over kin <= |k| < kout (one wave), then one
// block adds the partial sums in a fixed order into out[0]
__global__ void k_gen_annulus(const float2* F, int nx, long long np, const float* kx, const float* ky, float kin,
                              float kout, float scale, float* partial) {
  __shared__ float sh[256];
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  float v = 0.f;
  if (i < np) {
    const int y = (int)(i / nx), x = (int)(i - (long long)y * nx);
    const float k = sqrtf(kx[x] * kx[x] + ky[y] * ky[y]);
    if (k >= kin && k < kout) v = scale * (F[i].x * F[i].x + F[i].y * F[i].y);
  }
  sh[threadIdx.x] = v;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) sh[threadIdx.x] += sh[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = sh[0];
}

__global__ void k_gen_sum(const float* partial, int n, float* out) {
  __shared__ float sh[256];
  float v = 0.f;
  for (int i = threadIdx.x; i < n; i += 256) v += partial[i];
  sh[threadIdx.x] = v;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) sh[threadIdx.x] += sh[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[0] = sh[0];
}

int gen_annulus_blocks(long long np) { return (int)gnblk(np, 256); }

hipError_t launch_gen_annulus(const float2* F, int nx, int ny, const float* kx, const float* ky, float kin,
                              float kout, float scale, float* partial, float* out, hipStream_t s) {
  const long long np = (long long)nx * ny;
  const int nb = gen_annulus_blocks(np);
  hipLaunchKernelGGL(k_gen_annulus, dim3(nb), dim3(256), 0, s, F, nx, np, kx, ky, kin, kout, scale, partial);
  hipLaunchKernelGGL(k_gen_sum, dim3(1), dim3(256), 0, s, partial, nb, out);
  return hipGetLastError();
}

}  // namespace msl
