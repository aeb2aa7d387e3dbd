// k_physics.hip -- atom binning, potential synthesis, probe, CTF, detector
// and finite-difference kernels.  Citations are to the reference's
// "GUI Simulation/UnmanagedGUISimulation.cu" (U.cu).
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "msl_fft.hpp"
#include "msl_internal.hpp"

namespace msl {

static inline __host__ __device__ unsigned nblk(long long n, int b) { return (unsigned)((n + b - 1) / b); }

// ============================================================== binning
// atombin2 (U.cu:277-303): bin ids from FP32 sub, div, mul(50), floor --
// evaluated with IEEE division and no contraction so ids are bit-exact.
__global__ void k_bin_keys(BinArgs a) {
#pragma clang fp contract(off)
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.n) return;
  const float t1 = a.x[i] - a.MinX, t2 = a.MaxX - a.MinX;
  const float t3 = t1 / t2;
  const float t4 = t3 * 50.0f;
  const int bidx = (int)floorf(t4);
  const float u1 = a.y[i] - a.MinY, u2 = a.MaxY - a.MinY;
  const float u3 = u1 / u2;
  const float u4 = u3 * 50.0f;
  const int bidy = (int)floorf(u4);
  const float w1 = a.MaxZ - a.z[i];
  const float w2 = w1 / 1.0f;
  const int zid = (int)floorf(w2);
  if (bidx < 0 || bidx >= 50 || bidy < 0 || bidy >= 50 || zid < 0 || zid >= a.nslab) {
    a.key[i] = -1;
    atomicOr(a.bad, 1);
    return;
  }
  const int key = zid * 2500 + bidy * 50 + bidx;
  a.key[i] = key;
  atomicAdd(&a.count[key], 1);
}

// exclusive scan of count[0..nb] into start[0..nb], three phases
constexpr int SCAN_B = 256, SCAN_PER = 4, SCAN_CHUNK = SCAN_B * SCAN_PER;

__device__ int block_excl_scan(int v, int* sh, int& total) {
  // Hillis-Steele over 256 threads
  const int tid = threadIdx.x;
  sh[tid] = v;
  __syncthreads();
  for (int off = 1; off < SCAN_B; off <<= 1) {
    int x = tid >= off ? sh[tid - off] : 0;
    __syncthreads();
    sh[tid] += x;
    __syncthreads();
  }
  total = sh[SCAN_B - 1];
  const int incl = sh[tid];
  __syncthreads();
  return incl - v;
}

__global__ void __launch_bounds__(SCAN_B) k_scan_local(const int* in, int* out, int n, int* sums) {
  __shared__ int sh[SCAN_B];
  const long long base = (long long)blockIdx.x * SCAN_CHUNK + threadIdx.x * SCAN_PER;
  int v[SCAN_PER], s = 0;
  for (int k = 0; k < SCAN_PER; ++k) {
    v[k] = (base + k < n) ? in[base + k] : 0;
    s += v[k];
  }
  int total;
  int ex = block_excl_scan(s, sh, total);
  for (int k = 0; k < SCAN_PER; ++k) {
    if (base + k < n) out[base + k] = ex;
    ex += v[k];
  }
  if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

__global__ void __launch_bounds__(SCAN_B) k_scan_sums(int* sums, int nsums) {
  __shared__ int sh[SCAN_B];
  int carry = 0;
  for (int b0 = 0; b0 < nsums; b0 += SCAN_B) {
    const int i = b0 + threadIdx.x;
    const int v = i < nsums ? sums[i] : 0;
    int total;
    const int ex = block_excl_scan(v, sh, total);
    if (i < nsums) sums[i] = ex + carry;
    carry += total;
  }
}

__global__ void k_scan_add(int* out, int n, const int* sums) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] += sums[i / SCAN_CHUNK];
}

__global__ void k_bin_scatter(BinArgs a) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.n) return;
  const int key = a.key[i];
  if (key < 0) return;
  a.perm[a.start[key] + atomicAdd(&a.fill[key], 1)] = i;
}

// restore input order inside each bin (the reference's push_back order,
// U.cu:1479-1482), so the CSR is identical on every run
__global__ void k_bin_sort(BinArgs a, int nb) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= nb) return;
  const int s = a.start[b], e = a.start[b + 1];
  for (int i = s + 1; i < e; ++i) {
    const int v = a.perm[i];
    int j = i - 1;
    while (j >= s && a.perm[j] > v) {
      a.perm[j + 1] = a.perm[j];
      --j;
    }
    a.perm[j + 1] = v;
  }
}

// positions relative to Minimum*, U.cu:1479-1481
__global__ void k_bin_gather(BinArgs a, int nb) {
#pragma clang fp contract(off)
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= a.start[nb]) return;  // only slots filled by k_bin_scatter
  const int i = a.perm[s];
  if (i < 0 || i >= a.n) return;
  a.bx[s] = a.x[i] - a.MinX;
  a.by[s] = a.y[i] - a.MinY;
  a.bz[s] = a.z[i] - a.MinZ;
  a.bZ[s] = a.Z[i];
}

hipError_t launch_bin(const BinArgs& a, hipStream_t s) {
  const int nb = a.nslab * 2500;
  hipLaunchKernelGGL(k_bin_keys, dim3(nblk(a.n, 256)), dim3(256), 0, s, a);
  const int nscan = nb + 1;  // count[nb] == 0, so start[nb] = total
  const int nchunks = (int)nblk(nscan, SCAN_CHUNK);
  hipLaunchKernelGGL(k_scan_local, dim3(nchunks), dim3(SCAN_B), 0, s, a.count, a.start, nscan, a.scan_tmp);
  hipLaunchKernelGGL(k_scan_sums, dim3(1), dim3(SCAN_B), 0, s, a.scan_tmp, nchunks);
  hipLaunchKernelGGL(k_scan_add, dim3(nblk(nscan, 256)), dim3(256), 0, s, a.start, nscan, a.scan_tmp);
  hipLaunchKernelGGL(k_bin_scatter, dim3(nblk(a.n, 256)), dim3(256), 0, s, a);
  hipLaunchKernelGGL(k_bin_sort, dim3(nblk(nb, 256)), dim3(256), 0, s, a, nb);
  hipLaunchKernelGGL(k_bin_gather, dim3(nblk(a.n, 256)), dim3(256), 0, s, a, nb);
  return hipGetLastError();
}

// ============================================================== potential
// Radial tables.  The potential of an atom depends on the squared distance
// alone: vatom (U.cu:160-193)
//   V(r) = sum_i A_i exp(-B_i r) / r + sum_i C_i exp(-D_i r^2)
//   A = 150.4121417 a, B = 2 pi sqrt(b), C = 266.5157269 c d^-1.5, D = pi^2 / d
// and vzatom2 (U.cu:119-152)
//   Vz(r) = sum_i A'_i K0(B_i r) + sum_i C'_i exp(-D_i r^2)
//   A' = 300.8242834 a, C' = 150.4121417 c / d,
// both constant for r <= 0.25 A and cut off at r^2 = 5 A^2.  Evaluated
// directly a sample costs six exponentials, a square root and a reciprocal
// at a quarter of the FP32 rate each (57 issue slots; the potential kernels
// were bound by them).  Each species gets instead a piecewise cubic in
// x = r^2, fitted in FP64: 32 intervals per octave of [1/16, 5), so the
// interval is the top bits of x and the local coordinate the rest, and one
// interval of zeros from 5 on, which is where the cutoff lands (5 is an
// interval's edge, so r^2 < 5 is decided exactly).  Over all 103 species the
// cubic is within 5.2e-7 relative of the FP64 value (1.0e-7 rms), the direct
// FP32 form within 1.3e-6; 16 intervals per octave would leave 7e-6.
constexpr int VT_OCT = 32, VT_SHIFT = 18;            // intervals per octave; 23 - log2(32) mantissa bits left
constexpr int VT_N = 6 * VT_OCT + VT_OCT / 4 + 1;    // [1/16, 4), [4, 5), zeros
constexpr int VT_FIRST = 0x3D800000 >> VT_SHIFT;     // 1/16
constexpr float VT_LO = 0.0625f, VT_HI = 5.0f;

// Abramowitz & Stegun 9.8.1-9.8.6 (the forms of U.cu:41-111, with their value
// at 0: a term that a parameter file leaves out, a = b = 0, adds nothing)
__device__ double bessk0_f64(double x) {
  if (!(x > 0.0)) return 1.0e20;
  if (x <= 2.0) {
    double t = x / 3.75, u = x * 0.5;
    t = t * t;
    u = u * u;
    const double i0 = 1.0 + t * (3.5156229 + t * (3.0899424 + t * (1.2067492 + t * (0.2659732 + t * (0.0360768 +
                      t * 0.0045813)))));
    return -log(x * 0.5) * i0 - 0.57721566 + u * (0.42278420 + u * (0.23069756 + u * (0.03488590 + u * (0.00262698 +
           u * (0.00010750 + u * 0.00000740)))));
  }
  const double u = 2.0 / x;
  return exp(-x) / sqrt(x) * (1.25331414 + u * (-0.07832358 + u * (0.02189568 + u * (-0.01062446 + u * (0.00587872 +
         u * (-0.00251540 + u * 0.00053208))))));
}

// one thread per interval; blockIdx.y: species, blockIdx.z: 0 vatom, 1 vzatom
__global__ void k_vatom_table(const float* fp, float4* tab) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= VT_N) return;
  const int zi = blockIdx.y, proj = blockIdx.z;
  float4* o = tab + ((long long)proj * gridDim.y + zi) * VT_N + k;
  if (k == VT_N - 1) {
    *o = make_float4(0.f, 0.f, 0.f, 0.f);
    return;
  }
  const float* p = fp + zi * 12;
  const double pi = 3.141592654;
  double A[3], B[3], C[3], D[3];
  for (int i = 0; i < 3; ++i) {
    const double a = p[2 * i], b = p[2 * i + 1], c = p[6 + 2 * i], d = p[6 + 2 * i + 1];
    A[i] = (proj ? 300.8242834 : 150.4121417) * a;
    B[i] = 2.0 * pi * sqrt(b);
    C[i] = proj ? 150.4121417 * c / d : 266.5157269 * c / (d * sqrt(d));
    D[i] = pi * pi / d;
  }
  const double x0 = ldexp(1.0 + (double)(k % VT_OCT) / VT_OCT, k / VT_OCT - 4);
  const double w = ldexp(1.0 / VT_OCT, k / VT_OCT - 4);
  // cubic through the four Chebyshev nodes (Newton's divided differences)
  const double n[4] = {0.038060233744356624, 0.30865828381745514, 0.69134171618254486, 0.96193976625564338};
  double f[4];
  for (int j = 0; j < 4; ++j) {
    const double x = x0 + w * n[j], r = sqrt(x);
    double v = 0.0;
    for (int i = 0; i < 3; ++i)
      v += (proj ? A[i] * bessk0_f64(B[i] * r) : A[i] * exp(-B[i] * r) / r) + C[i] * exp(-D[i] * x);
    f[j] = v;
  }
  for (int l = 1; l < 4; ++l)
    for (int j = 3; j >= l; --j) f[j] = (f[j] - f[j - 1]) / (n[j] - n[j - l]);
  // Newton form to powers of the node coordinate, then of t = x - x0
  double c0 = f[3], c1 = 0.0, c2 = 0.0, c3 = 0.0;
  for (int j = 2; j >= 0; --j) {
    c3 = c2 - n[j] * c3;
    c2 = c1 - n[j] * c2;
    c1 = c0 - n[j] * c1;
    c0 = f[j] - n[j] * c0;
  }
  *o = make_float4((float)c0, (float)(c1 / w), (float)(c2 / (w * w)), (float)(c3 / (w * w * w)));
}

size_t vatom_table_size() { return (size_t)2 * 103 * VT_N; }

hipError_t launch_vatom_table(const float* fparams, float4* tab, hipStream_t s) {
  hipLaunchKernelGGL(k_vatom_table, dim3(nblk(VT_N, 64), 103, 2), dim3(64), 0, s, fparams, tab);
  return hipGetLastError();
}

// the table's value at r2; base: byte offset of the species' first entry, less
// that of the interval of 0
constexpr int VT_ZERO = VT_FIRST * (int)sizeof(float4);
template <class T> __device__ __forceinline__ float vt_at(T tab, int base, float r2) {
  const float x = __builtin_amdgcn_fmed3f(r2, VT_LO, VT_HI);
  // the interval's lower end; its number times 16 are the same bits further down
  const unsigned k = __float_as_uint(x) & ~((1u << VT_SHIFT) - 1u);
  const float4 c = *(T)((const char*)tab + (int)((k >> (VT_SHIFT - 4)) + (unsigned)base));
  const float t = x - __uint_as_float(k);
  return fmaf(t, fmaf(t, fmaf(t, c.w, c.z), c.y), c.x);
}

// FP32 distance decisions of the reference kernels (U.cu:637-640, 784, 931):
// pixel position fma(x, ps, offset), squared distance as fma(dy, dy, dx*dx)
// and fma(dz, dz, rxy).  Written out explicitly, with contraction off, so
// the r^2 < 5 cutoff is decided the same way on every build.
__device__ __forceinline__ float pix_pos(int i, float ps, float off) {
#pragma clang fp contract(off)
  return fmaf((float)i, ps, off);
}
__device__ __forceinline__ float dist2_xy(float px, float py, float ax, float ay) {
#pragma clang fp contract(off)
  const float dx = px - ax, dy = py - ay;
  return fmaf(dy, dy, dx * dx);
}
__device__ __forceinline__ float dist2_z(float rxy, float z, float az) {
#pragma clang fp contract(off)
  const float dd = z - az;
  return fmaf(dd, dd, rxy);
}
__device__ __forceinline__ float sample_z(float zf, int m, float dz) {
#pragma clang fp contract(off)
  return zf - ((float)m * dz) / 20.0f;
}
// binnedAtomPKernelRS samples z - m dz / 10 with an integer dz of 1 (U.cu:700)
__device__ __forceinline__ float sample_z_rs(float zf, int m) {
#pragma clang fp contract(off)
  return zf - (float)m / 10.0f;
}

constexpr int PT = 16;      // pixel tile edge of the grouped launches (serving)
// pixel tiles of 256 threads selectable per handle (PotArgs::tile, chosen by
// msl_autotune_potential): 16x16, 32x8, 64x4, 8x32.  Every shape sums each
// pixel's atoms in the same (slab, bin row, bin, CSR) order, so all give the
// same bits; they differ in the bin window each workgroup stages.
template <int V> struct PotTile;
template <> struct PotTile<0> { static constexpr int X = 16, Y = 16; };
template <> struct PotTile<1> { static constexpr int X = 32, Y = 8; };
template <> struct PotTile<2> { static constexpr int X = 64, Y = 4; };
template <> struct PotTile<3> { static constexpr int X = 8, Y = 32; };
constexpr int kPotTiles = 4;
constexpr int ACAP = 512;   // atoms staged in LDS per chunk
constexpr int kTabLds = 4;  // species whose tables fit the LDS stage

// what a launch sums per atom: the samples of a slice (modes 0 and 3), the
// projected potential (mode 1) or one plane (mode 2)
enum PotKind { POT_SAMPLES = 0, POT_PROJECTED = 1, POT_PLANE = 2 };
static inline __host__ __device__ constexpr int pot_kind(int mode) {
  return mode == 1 ? POT_PROJECTED : mode == 2 ? POT_PLANE : POT_SAMPLES;
}

// the potential arguments as device code reads them from a table in memory
// (pointers in the global address space, same layout)
struct PotArgsG {
  MSL_POT_ARGS(MSL_GLOBAL)
};
static_assert(sizeof(PotArgsG) == sizeof(PotArgs), "layouts differ");

__device__ __forceinline__ float readlane_f(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// binnedAtomPKernel3 (U.cu:582-653), binnedAtomPKernelConventional3
// (U.cu:730-795), binnedAtomPKernelFD (U.cu:883-946) and binnedAtomPKernelRS
// (U.cu:656-727): pixel tile (tx, ty) of TX x TY pixels of slice `slice`
// (relative to first_slice), one thread per pixel and, with SPLIT 4, four
// waves per 8 x 8 pixels that share the atoms between them.
//
// The bin rows of every slab of the window are gathered in one go (one scan
// over all of them, one round of atom loads): a workgroup waits for three
// dependent loads in all, not for three per slab.  Then each wave works on
// an 8 x 8 pixel patch of its own: its lanes test 64 atoms at a time against
// the patch and find the samples each can reach, and only those atoms and
// samples are summed, with the atom in scalar registers.  Lanes out of an
// atom's reach read the table's zero interval, so there is no divergence.
// Bound by VALU issue at large grids (11 instructions and a 16-byte LDS read
// per sample), by those three loads and the launch at small ones.  Per slice,
// before (slab after slab, transcendentals, a divergent loop per pixel) and
// now: Si 1024^2 of 0.074 A 114.6 -> 34.5 us, SrTiO3 512^2 of 0.078 A 51.0 ->
// 17.2, Si 256^2 of 0.085 A 27.9 -> 7.9, 64^2 of 0.2 A 27.2 -> 5.8; one plane
// of Si at 256^2 16.0 -> 4.6.
template <int TX, int TY, int SPLIT, int KIND, class A>
__device__ __forceinline__ void potential_tile(const A& a, int tx, int ty, int slice, float4* tabs) {
  static_assert(TX * TY * SPLIT == 256, "256-thread workgroups");
  __shared__ float4 sa[ACAP];      // x, y, z, table base (as int)
  __shared__ int si[ACAP];
  __shared__ int wsum[4];
  __shared__ float red[SPLIT > 1 ? 256 : 1];
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  // the wave's patch: 8 x 8 pixels, 16 x 4 in the 64 x 4 tile
  constexpr int PW = TY % 8 == 0 ? 8 : 16, PH = 64 / PW;
  const int pt = SPLIT > 1 ? 0 : wv;
  const int wx = tx * TX + (pt % (TX / PW)) * PW, wy = ty * TY + (pt / (TX / PW)) * PH;
  const int ix = wx + lane % PW, iy = wy + lane / PW;
  constexpr int kPart = KIND == POT_PROJECTED ? 103 * VT_N : 0;
  const bool in_lds = KIND != POT_PLANE && a.nspec > 0;
  if (in_lds)
    for (int q = tid; q < a.nspec * VT_N; q += 256) {
      const int sp = q / VT_N;
      tabs[q] = a.vtab[kPart + (a.spec[sp] - 1) * VT_N + (q - sp * VT_N)];
    }
  float zf, h;
  {
#pragma clang fp contract(off)
    h = a.MaxZ - a.MinZ;
    // compat=physical: slice i starts at the top of the specimen (i - 1 slices down)
    const int phys = (a.mode < 2 && a.physical) ? 1 : 0;
    zf = (a.mode >= 2) ? a.zplane : h - a.dz * (float)(a.first_slice + slice - phys);
  }
  int k0, k1;
  if constexpr (KIND == POT_PROJECTED) {
    k0 = (int)floorf(h - zf);
    k1 = (int)floorf(h - zf + a.dz) - 1;
  } else {
    const int kc = (int)floorf((h - zf) / 1.0f);
    k0 = kc - a.loadslicesz;
    k1 = kc + a.loadslicesz;
    if (a.mode == 0 && a.physical) {
      // down to the slab of the lowest sample, +-3 (every atom within sqrt(5))
#pragma clang fp contract(off)
      const float zb = zf - a.dz;
      k1 = (int)floorf((h - zb) / 1.0f) + a.loadslicesz;
    }
  }
  k0 = max(k0, 0);
  k1 = min(k1, a.nslab - 1);
  const float offx = a.mode == 2 ? 0.f : a.offx, offy = a.mode == 2 ? 0.f : a.offy;
  const float px = pix_pos(ix, a.ps, offx), py = pix_pos(iy, a.ps, offy);
  const float bx0 = pix_pos(wx, a.ps, offx), bx1 = pix_pos(wx + PW - 1, a.ps, offx);
  const float by0 = pix_pos(wy, a.ps, offy), by1 = pix_pos(wy + PH - 1, a.ps, offy);
  // bin window of the tile: every bin that may hold an atom within sqrt(5)
  const float bwx = (a.MaxX - a.MinX) / 50.f, bwy = (a.MaxY - a.MinY) / 50.f, reach = 2.2360680f;
  const float tx0 = offx + (float)(tx * TX) * a.ps, tx1 = offx + (float)(tx * TX + TX - 1) * a.ps;
  const float ty0 = offy + (float)(ty * TY) * a.ps, ty1 = offy + (float)(ty * TY + TY - 1) * a.ps;
  const int i0 = max(0, (int)floorf((tx0 - reach) / bwx) - 1), i1 = min(49, (int)floorf((tx1 + reach) / bwx) + 1);
  const int j0 = max(0, (int)floorf((ty0 - reach) / bwy) - 1), j1 = min(49, (int)floorf((ty1 + reach) / bwy) + 1);
  const int nj = j1 - j0 + 1;
  const int runs = (i0 <= i1 && nj > 0 && k0 <= k1) ? nj * (k1 - k0 + 1) : 0;
  // lane m holds sample position m; the lanes past the last sample are out
  // of every atom's reach
  const int nsamp = a.mode == 3 ? 10 : 20;
  const float hs = a.mode == 3 ? 0.1f : a.dz / 20.0f, us = 1.0f / hs;
  float zl = 3.0e18f;
  if constexpr (KIND == POT_SAMPLES)
    if (lane >= 1 && lane <= nsamp) zl = a.mode == 3 ? sample_z_rs(zf, lane) : sample_z(zf, lane, a.dz);
  // the patch test may err on the side of keeping an atom: FP32 rounding of
  // positions a thousand angstroms away is 1e-3 A^2 in r^2
  constexpr float kReach2 = 5.05f;
  float sum = 0.f;
  int seen = 0;  // atoms of the patch so far (SPLIT: atom n goes to wave n % SPLIT)
  // the atoms of a chunk, in sa[0 .. cn - 1]
  auto stage = [&](int q, int src) {
    const int Z = a.bZ[src];
    int base = (Z - 1) * VT_N + kPart;
    if (in_lds) {
      base = 0;
      for (int sp = 1; sp < a.nspec; ++sp) base = Z == a.spec[sp] ? sp * VT_N : base;
    }
    const float x = a.bx[src], y = a.by[src], z = a.bz[src];
    // a position that is no number is put out of every patch's reach: it is at
    // no distance below the cutoff (the patch test and the table's clamp would
    // take it for one at the centre)
    const bool num = x == x && y == y && (KIND == POT_PROJECTED || z == z);
    sa[q] = make_float4(num ? x : 1e18f, y, z, __int_as_float(base * (int)sizeof(float4) - VT_ZERO));
  };
  auto sum_chunk = [&](int cn) {
    auto atoms = [&](auto tab) {
      for (int b0 = 0; b0 < cn; b0 += 64) {
        float4 at = make_float4(0.f, 0.f, 0.f, 0.f);
        bool hit = false;
        int mlo = 1, mhi = 0;
        if (b0 + lane < cn) {
          at = sa[b0 + lane];
          const float ex = fmaxf(fmaxf(bx0 - at.x, at.x - bx1), 0.f);
          const float ey = fmaxf(fmaxf(by0 - at.y, at.y - by1), 0.f);
          float room = kReach2 - (ex * ex + ey * ey);
          hit = room > 0.f;
          if constexpr (KIND == POT_SAMPLES) {
            // samples with |zf - m hs - z| within the patch's reach (0.011 A
            // more than any pixel's, which covers the rounding of positions)
            const float hz = __builtin_amdgcn_sqrtf(fmaxf(room, 0.f)), zc = zf - at.z;
            mlo = max(1, (int)fmaxf(ceilf((zc - hz) * us), 0.f));
            mhi = min(nsamp, (int)fminf(floorf((zc + hz) * us), 64.f));
            hit = hit && mlo <= mhi;
          } else if constexpr (KIND == POT_PLANE) {
            room -= (zf - at.z) * (zf - at.z);
            hit = room > 0.f;
          }
        }
        unsigned long long mask = __ballot(hit);
        while (mask) {
          const int l = __builtin_ctzll(mask);
          mask &= mask - 1;
          if (SPLIT > 1 && (seen++ % SPLIT) != wv) continue;
          const float ax = readlane_f(at.x, l), ay = readlane_f(at.y, l), az = readlane_f(at.z, l);
          const int base = __builtin_amdgcn_readlane(__float_as_int(at.w), l);
          const float rxy = dist2_xy(px, py, ax, ay);
          if constexpr (KIND == POT_PROJECTED) {
            sum += vt_at(tab, base, rxy);
          } else if constexpr (KIND == POT_PLANE) {
            sum += vt_at(tab, base, dist2_z(rxy, zf, az));
          } else {
            const int m0 = __builtin_amdgcn_readlane(mlo, l), m1 = __builtin_amdgcn_readlane(mhi, l);
            const float dl = zl - az;
            float s = 0.f;
            // four samples at a time, their table reads in flight together
            auto samples = [&](int m, auto count) {
              constexpr int C = decltype(count)::value;
              float v[C];
#pragma unroll
              for (int u = 0; u < C; ++u) {
                const float dd = readlane_f(dl, m + u);
                v[u] = vt_at(tab, base, fmaf(dd, dd, rxy));
              }
#pragma unroll
              for (int u = 0; u < C; ++u) s += v[u];
            };
            int m = m0;
            for (; m + 3 <= m1; m += 4) samples(m, std::integral_constant<int, 4>{});
            if (m + 1 <= m1) {
              samples(m, std::integral_constant<int, 2>{});
              m += 2;
            }
            if (m <= m1) samples(m, std::integral_constant<int, 1>{});
            sum = fmaf(hs, s, sum);
          }
        }
      }
    };
    if (in_lds) atoms((const float4*)tabs);
    else atoms(a.vtab);
  };
  // Small launches: where the window's slabs hold no more than a chunk of atoms
  // (one run of the CSR), they are taken as they come and the patch test culls
  // them, 64 at a time, without the bin rows' scan and their expansion (256^2:
  // 8.5 -> 7.9 us, 64^2 6.7 -> 5.8, a plane 5.5 -> 4.9).  Full launches, whose
  // windows seldom qualify, lose 2 to 5 % to the registers it takes.
  bool all = false;
  if constexpr (SPLIT > 1) {
    if (runs > 0) {
      const int s0 = a.start[k0 * 2500], n = a.start[(k1 + 1) * 2500] - s0;
      all = n <= ACAP;
      if (all) {
        for (int q = tid; q < n; q += 256) stage(q, s0 + q);
        __syncthreads();
        sum_chunk(n);
      }
    }
  }
  for (int rb = all ? runs : 0; rb < runs; rb += 256) {
    int len = 0, r0 = 0;
    if (rb + tid < runs) {
      const int k = (rb + tid) / nj, j = (rb + tid) - k * nj;
      const int bb = (k0 + k) * 2500 + (j0 + j) * 50;
      r0 = a.start[bb + i0];
      len = a.start[bb + i1 + 1] - r0;
    }
    int incl = len;
    for (int d = 1; d < 64; d <<= 1) {
      const int v = __shfl_up(incl, d, 64);
      if (lane >= d) incl += v;
    }
    if (lane == 63) wsum[wv] = incl;
    __syncthreads();
    int off = incl - len, tot = 0;
    for (int w = 0; w < 4; ++w) {
      const int v = wsum[w];
      off += w < wv ? v : 0;
      tot += v;
    }
    for (int c0 = 0; c0 < tot; c0 += ACAP) {
      const int cn = min(ACAP, tot - c0);
      for (int j = max(0, c0 - off); j < len && off + j < c0 + cn; ++j) si[off + j - c0] = r0 + j;
      __syncthreads();
      for (int q = tid; q < cn; q += 256) stage(q, si[q]);
      __syncthreads();
      sum_chunk(cn);
      __syncthreads();  // si / sa are rewritten by the next chunk
    }
    __syncthreads();  // wsum is rewritten by the next runs
  }
  if constexpr (SPLIT > 1) {
    red[tid] = sum;
    __syncthreads();
    if (wv != 0) return;
    sum = ((red[lane] + red[64 + lane]) + red[128 + lane]) + red[192 + lane];
  }
  if (ix >= a.nx || iy >= a.ny) return;
  const long long o = (long long)slice * a.out_sstride + (long long)iy * a.nx + ix;
  if (a.out_kind == 0) {
    float sn, cs;
    sincosf(a.sigma * sum, &sn, &cs);
    ((float2*)a.out)[o] = make_float2(cs, sn);
  } else if (a.out_kind == 1) {
    ((float2*)a.out)[o] = make_float2(sum, 0.f);
  } else {
    ((float*)a.out)[o] = sum;
  }
}

template <int V, int KIND>
__global__ void __launch_bounds__(256) k_potential(PotArgs a) {
  extern __shared__ float4 pot_tabs[];
  potential_tile<PotTile<V>::X, PotTile<V>::Y, 1, KIND>(a, blockIdx.x, blockIdx.y, blockIdx.z, pot_tabs);
}

// small launches: 64 pixels per workgroup, its four waves sharing the atoms
template <int KIND>
__global__ void __launch_bounds__(256) k_potential_split(PotArgs a) {
  extern __shared__ float4 pot_tabs[];
  potential_tile<8, 8, 4, KIND>(a, blockIdx.x, blockIdx.y, blockIdx.z, pot_tabs);
}

// slice `first` of njobs jobs in one launch: workgroup id -> (job, tile)
// through the block offsets blk0[0..njobs] (ascending)
template <int KIND>
__global__ void __launch_bounds__(256) k_potential_group(const PotArgs* tab, const long long* blk0, int njobs,
                                                         int first) {
  extern __shared__ float4 pot_tabs[];
  const long long id = blockIdx.x;
  int lo = 0, hi = njobs - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) / 2;
    if (blk0[mid] <= id) lo = mid;
    else hi = mid - 1;
  }
  PotArgsG a = reinterpret_cast<const PotArgsG*>(tab)[lo];
  a.first_slice = first;
  const int tx = nblk(a.nx, PT);
  const long long local = id - blk0[lo];
  potential_tile<PT, PT, 1, KIND>(a, (int)(local % tx), (int)(local / tx), 0, pot_tabs);
}

// dynamic LDS of a launch: the tables of its species (the one read per atom
// of a plane comes from the caches)
template <int KIND> static size_t pot_lds(const PotArgs& a) {
  return KIND == POT_PLANE ? 0 : a.nspec * VT_N * sizeof(float4);
}

template <int V, int KIND> static hipError_t potential_v(const PotArgs& a, hipStream_t s) {
  dim3 grid(nblk(a.nx, PotTile<V>::X), nblk(a.ny, PotTile<V>::Y), a.nslices);
  hipLaunchKernelGGL((k_potential<V, KIND>), grid, dim3(256), pot_lds<KIND>(a), s, a);
  return hipGetLastError();
}

// one wave per 8 x 8 pixels leaves SIMDs (1024 on the chip) with fewer than
// four waves each below 4096 patches: four waves then share a patch, and the
// pixel tiles have no part in it
bool potential_tiled(int nx, int ny, int nslices) {
  return (long long)nblk(nx, 8) * nblk(ny, 8) * nslices >= 4096;
}

template <int KIND> static hipError_t potential_k(const PotArgs& a, hipStream_t s) {
  if (!potential_tiled(a.nx, a.ny, a.nslices)) {
    hipLaunchKernelGGL(k_potential_split<KIND>, dim3(nblk(a.nx, 8), nblk(a.ny, 8), a.nslices), dim3(256),
                       pot_lds<KIND>(a), s, a);
    return hipGetLastError();
  }
  switch (a.tile) {
    case 1: return potential_v<1, KIND>(a, s);
    case 2: return potential_v<2, KIND>(a, s);
    case 3: return potential_v<3, KIND>(a, s);
    default: return potential_v<0, KIND>(a, s);
  }
}

hipError_t launch_potential(const PotArgs& a, hipStream_t s) {
  if (a.nslices <= 0) return hipSuccess;
  if (!a.vtab || a.nspec < 0 || a.nspec > kTabLds) return hipErrorInvalidValue;
  switch (pot_kind(a.mode)) {
    case POT_PROJECTED: return potential_k<POT_PROJECTED>(a, s);
    case POT_PLANE: return potential_k<POT_PLANE>(a, s);
    default: return potential_k<POT_SAMPLES>(a, s);
  }
}

int potential_tile_variants() { return kPotTiles; }

int potential_tiles(int nx, int ny) { return nblk(nx, PT) * nblk(ny, PT); }

hipError_t launch_potential_group(const PotArgs* tab, const long long* blk0, int njobs, long long nblocks, int first,
                                  int mode, hipStream_t s) {
  if (njobs <= 0 || nblocks <= 0) return hipSuccess;
  if (nblocks > 0x7fffffffLL || mode < 0 || mode > 1) return hipErrorInvalidValue;
  const size_t lds = kTabLds * VT_N * sizeof(float4);
  const dim3 grid((unsigned)nblocks), block(256);
  if (mode == 1) hipLaunchKernelGGL(k_potential_group<POT_PROJECTED>, grid, block, lds, s, tab, blk0, njobs, first);
  else hipLaunchKernelGGL(k_potential_group<POT_SAMPLES>, grid, block, lds, s, tab, blk0, njobs, first);
  return hipGetLastError();
}

// ============================================================== probe
// STEMinitializingKernel (U.cu:354-383): exp(i(theta - chi)) inside
// k < apert.  theta = 2 pi (kx posx + ky posy) ps is reduced in FP64 so the
// ramp stays accurate for positions far from the origin.
__global__ void k_probe_kspace(ProbeArgs a) {
  int x = blockIdx.x * blockDim.x + threadIdx.x;
  const int y = blockIdx.y, b = blockIdx.z;
  if (a.band_cols > 0) {
    if (x >= 2 * a.band_cols) return;
    if (x >= a.band_cols) x += a.nx - 2 * a.band_cols;
  } else if (x >= a.nx) {
    return;
  }
  const float k0x = a.kx[x], k0y = a.ky[y];
  const float k = sqrtf(k0x * k0x + k0y * k0y);
  float2 v = make_float2(0.f, 0.f);
  if (k < a.apert) {
    const int px = a.posx ? a.posx[b] : a.px0, py = a.posy ? a.posy[b] : a.py0;
    const double k2 = (double)k0x * k0x + (double)k0y * k0y, wl = a.wavel, pi = 3.14159265;
    const double chi = pi * wl * k2 * ((double)a.Cs * wl * wl * k2 * 0.5 + (double)a.df);
    const double th = 2.0 * pi * ((double)k0x * px * (double)a.ps + (double)k0y * py * (double)a.ps);
    double ph = th - chi;
    ph -= 6.283185307179586 * floor(ph / 6.283185307179586);
    float sn, cs;
    sincosf((float)ph, &sn, &cs);
    v = make_float2(cs, sn);
  }
  a.out[(long long)b * a.bstride + (long long)y * a.nx + x] = v;
}

hipError_t launch_probe_kspace(const ProbeArgs& a, hipStream_t s) {
  if (a.band_cols < 0 || 2 * a.band_cols > a.nx) return hipErrorInvalidValue;
  // probes on grid.z, at most 65535 per launch
  constexpr int kMaxGridZ = 65535;
  for (int b0 = 0; b0 < a.nprobe; b0 += kMaxGridZ) {
    ProbeArgs c = a;
    c.nprobe = a.nprobe - b0 < kMaxGridZ ? a.nprobe - b0 : kMaxGridZ;
    c.out = a.out + (long long)b0 * a.bstride;
    if (a.posx) {
      c.posx = a.posx + b0;
      c.posy = a.posy + b0;
    }
    const int cols = a.band_cols > 0 ? 2 * a.band_cols : a.nx;
    hipLaunchKernelGGL(k_probe_kspace, dim3(nblk(cols, 256), a.ny, c.nprobe), dim3(256), 0, s, c);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

// ============================================================== tables
// k-grids (PreCalculateFrequencies, U.cu:1877-1964; the FP32 division the host
// takes too) and twiddles of both axes, and the separable
// Fresnel factors exp(-i pi dz lambda k^2) of CreatePropsKernel
// (U.cu:399-428), evaluated in FP64.  Made where they are used: uploads from
// host memory cost a run of 64^2 five waits and 70 us of 440.
__global__ void k_ktables(float* kx, float* ky, float2* twx, float2* twy, int nx, int ny, float ksx, float ksy) {
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= nx + ny) return;
  const bool isx = g < nx;
  const int i = isx ? g : g - nx, n = isx ? nx : ny;
  const float ks = isx ? ksx : ksy;
  (isx ? kx : ky)[i] = i > n / 2 ? (float)(i - n) / ks : (float)i / ks;
  float2* tw = isx ? twx : twy;
  if (tw) {
    double sn, cs;
    sincospi(-2.0 * (double)i / (double)n, &sn, &cs);
    tw[i] = twiddle(cs, sn, i, n);
  }
}
hipError_t launch_ktables(float* kx, float* ky, float2* twx, float2* twy, int nx, int ny, float ksx, float ksy,
                          hipStream_t s) {
  hipLaunchKernelGGL(k_ktables, dim3(nblk(nx + ny, 64)), dim3(64), 0, s, kx, ky, twx, twy, nx, ny, ksx, ksy);
  return hipGetLastError();
}
__global__ void k_prop_factors(const float* kx, const float* ky, float2* px, float2* py, int nx, int ny, float dz,
                               float wavel) {
#pragma clang fp contract(off)
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= nx + ny) return;
  const double k = g < nx ? kx[g] : ky[g - nx];
  const double a = 3.14159265 * (double)dz * (double)wavel * k * k;
  (g < nx ? px : py)[g < nx ? g : g - nx] = make_float2((float)cos(a), (float)-sin(a));
}
hipError_t launch_prop_factors(const float* kx, const float* ky, float2* px, float2* py, int nx, int ny, float dz,
                               float wavel, hipStream_t s) {
  hipLaunchKernelGGL(k_prop_factors, dim3(nblk(nx + ny, 64)), dim3(64), 0, s, kx, ky, px, py, nx, ny, dz, wavel);
  return hipGetLastError();
}

// ============================================================== reductions
constexpr int RB = 256;

__device__ float block_sum(float v, float* sh) {
  sh[threadIdx.x] = v;
  __syncthreads();
  for (int s = RB / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) sh[threadIdx.x] += sh[threadIdx.x + s];
    __syncthreads();
  }
  const float r = sh[0];
  __syncthreads();
  return r;
}

// per wave: partial[b][blk] = sum |w| over a fixed 4096-element chunk
constexpr int L1_CHUNK = 4096;
__global__ void __launch_bounds__(RB) k_abs_partial(const float2* w, long long n, long long bstride, float* partial,
                                                    int nchunk, int l2) {
  __shared__ float sh[RB];
  const int b = blockIdx.y, blk = blockIdx.x;
  const float2* p = w + (long long)b * bstride;
  float acc = 0.f;
  const long long s0 = (long long)blk * L1_CHUNK;
  for (int i = threadIdx.x; i < L1_CHUNK; i += RB) {
    const long long j = s0 + i;
    if (j < n) {
      const float i2 = p[j].x * p[j].x + p[j].y * p[j].y;
      acc += l2 ? i2 : sqrtf(i2);
    }
  }
  const float r = block_sum(acc, sh);
  if (threadIdx.x == 0) partial[(long long)b * nchunk + blk] = r;
}

__global__ void __launch_bounds__(RB) k_abs_final(float* partial, int nchunk, float* norm, int l2) {
  __shared__ float sh[RB];
  const int b = blockIdx.x;
  float acc = 0.f;
  for (int i = threadIdx.x; i < nchunk; i += RB) acc += partial[(long long)b * nchunk + i];
  const float r = block_sum(acc, sh);
  if (threadIdx.x == 0) norm[b] = l2 ? sqrtf(r) : r;
}

__global__ void k_div_by(float2* w, long long n, long long bstride, const float* norm) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const int b = blockIdx.y;
  if (i >= n) return;
  const float inv = 1.0f / norm[b];
  float2* p = w + (long long)b * bstride;
  p[i] = cscale(p[i], inv);
}

hipError_t launch_l1_normalise(float2* w, long long n, int nbatch, long long bstride, float* scratch, hipStream_t s) {
  return launch_probe_normalise(w, n, nbatch, bstride, scratch, 0, s);
}

hipError_t launch_probe_normalise(float2* w, long long n, int nbatch, long long bstride, float* scratch, int l2,
                                  hipStream_t s) {
  const int nchunk = (int)nblk(n, L1_CHUNK);
  float* partial = scratch;
  float* norm = scratch + (long long)nbatch * nchunk;
  hipLaunchKernelGGL(k_abs_partial, dim3(nchunk, nbatch), dim3(RB), 0, s, w, n, bstride, partial, nchunk, l2);
  hipLaunchKernelGGL(k_abs_final, dim3(nbatch), dim3(RB), 0, s, partial, nchunk, norm, l2);
  hipLaunchKernelGGL(k_div_by, dim3(nblk(n, 256), nbatch), dim3(256), 0, s, w, n, bstride, norm);
  return hipGetLastError();
}

__global__ void k_fill(float2* w, long long n, float2 v) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) w[i] = v;
}
hipError_t launch_fill(float2* w, long long n, float2 v, hipStream_t s) {
  hipLaunchKernelGGL(k_fill, dim3(nblk(n, 256)), dim3(256), 0, s, w, n, v);
  return hipGetLastError();
}

__global__ void k_hash_fill(float2* w, long long n, unsigned seed, int unit) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  unsigned h = (unsigned)i * 2654435761u ^ seed;
  h ^= h >> 16; h *= 0x7feb352du; h ^= h >> 15; h *= 0x846ca68bu; h ^= h >> 16;
  const float u = (float)(h & 0xffffff) * (1.0f / 16777216.0f), v = (float)(h >> 8) * (1.0f / 16777216.0f);
  if (unit) {
    float sn, cs;
    sincosf(6.2831853f * u, &sn, &cs);
    w[i] = make_float2(cs, sn);
  } else {
    w[i] = make_float2(2.f * u - 1.f, 2.f * v - 1.f);
  }
}
hipError_t launch_hash_fill(float2* w, long long n, unsigned seed, int unit, hipStream_t s) {
  hipLaunchKernelGGL(k_hash_fill, dim3(nblk(n, 256)), dim3(256), 0, s, w, n, seed, unit);
  return hipGetLastError();
}

// plain streaming copy (16-byte vectors), used to calibrate traffic counters
__global__ void k_copy16(const float4* __restrict__ src, float4* __restrict__ dst, long long n) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    dst[i] = src[i];
}
hipError_t launch_copy16(const void* src, void* dst, long long bytes, hipStream_t s) {
  const long long n = bytes / 16;
  hipLaunchKernelGGL(k_copy16, dim3((unsigned)std::min<long long>(nblk(n, 256), 65536)), dim3(256), 0, s,
                     (const float4*)src, (float4*)dst, n);
  return hipGetLastError();
}

__global__ void k_scale(float2* w, long long n, float f) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) w[i] = cscale(w[i], f);
}
hipError_t launch_scale(float2* w, long long n, float f, hipStream_t s) {
  hipLaunchKernelGGL(k_scale, dim3(nblk(n, 256)), dim3(256), 0, s, w, n, f);
  return hipGetLastError();
}

__global__ void k_cmul(const float2* a, const float2* b, float2* o, long long n, float f) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) o[i] = cscale(cmul(a[i], b[i]), f);
}
hipError_t launch_cmul(const float2* a, const float2* b, float2* o, long long n, float f, hipStream_t s) {
  hipLaunchKernelGGL(k_cmul, dim3(nblk(n, 256)), dim3(256), 0, s, a, b, o, n, f);
  return hipGetLastError();
}

__global__ void k_reduce_rows(const float* partial, int nbatch, int ntiles, float* out, int acc) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= nbatch) return;
  float s = 0.f;
  for (int i = 0; i < ntiles; ++i) s += partial[(long long)b * ntiles + i];
  out[b] = acc ? out[b] + s : s;
}
hipError_t launch_reduce_rows(const float* partial, int nbatch, int ntiles, float* out, int acc, hipStream_t s) {
  hipLaunchKernelGGL(k_reduce_rows, dim3(nblk(nbatch, 256)), dim3(256), 0, s, partial, nbatch, ntiles, out, acc);
  return hipGetLastError();
}

__global__ void k_abs(const float2* w, float* o, long long n) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) o[i] = sqrtf(w[i].x * w[i].x + w[i].y * w[i].y);
}
hipError_t launch_abs(const float2* w, float* o, long long n, hipStream_t s) {
  hipLaunchKernelGGL(k_abs, dim3(nblk(n, 256)), dim3(256), 0, s, w, o, n);
  return hipGetLastError();
}

// ============================================================== real-space multislice
// One term of MultisliceStepRS's series (RSMS with DifferentialXKernel /
// DifferentialYKernel, U.cu:798-877): out = w + i pre (Lx w + Ly w + V w)
// with L (4/3 d1 - d2/12) / ps^2 per axis, d1 = f[+1] + f[-1] - f[0],
// d2 = f[+2] + f[-2] - f[0], and neighbours outside the grid reading element
// 0 of the row / column; the first term (w == null) is 1 + i pre V.
__global__ void k_rs_term(const float2* w, float2* out, const float2* V, int nx, int ny, float ps, float pre) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y;
  if (x >= nx) return;
  const long long row = (long long)y * nx, id = row + x;
  const float v = V[id].x;
  if (!w) {
    out[id] = make_float2(1.0f, pre * v);
    return;
  }
  const int xp1 = x > 0 ? x - 1 : 0, xp2 = x > 1 ? x - 2 : 0, xn1 = x < nx - 1 ? x + 1 : 0, xn2 = x < nx - 2 ? x + 2 : 0;
  const int yp1 = y > 0 ? y - 1 : 0, yp2 = y > 1 ? y - 2 : 0, yn1 = y < ny - 1 ? y + 1 : 0, yn2 = y < ny - 2 ? y + 2 : 0;
  const float2 f = w[id];
  const float2 a1 = w[row + xn1], b1 = w[row + xp1], a2 = w[row + xn2], b2 = w[row + xp2];
  const float2 c1 = w[(long long)yn1 * nx + x], e1 = w[(long long)yp1 * nx + x];
  const float2 c2 = w[(long long)yn2 * nx + x], e2 = w[(long long)yp2 * nx + x];
  const float s = 1.0f / (ps * ps);
  const float dxx = s * (4.0f * ((a1.x + b1.x) - f.x) / 3.0f - ((a2.x + b2.x) - f.x) / 12.0f);
  const float dxy = s * (4.0f * ((a1.y + b1.y) - f.y) / 3.0f - ((a2.y + b2.y) - f.y) / 12.0f);
  const float dyx = s * (4.0f * ((c1.x + e1.x) - f.x) / 3.0f - ((c2.x + e2.x) - f.x) / 12.0f);
  const float dyy = s * (4.0f * ((c1.y + e1.y) - f.y) / 3.0f - ((c2.y + e2.y) - f.y) / 12.0f);
  const float r1x = -1.0f * pre * (dxy + dyy + v * f.y);
  const float r1y = pre * (dxx + dyx + v * f.x);
  out[id] = make_float2(f.x + r1x, f.y + r1y);
}
hipError_t launch_rs_term(const float2* w, float2* out, const float2* V, int nx, int ny, float ps, float pre,
                          hipStream_t s) {
  hipLaunchKernelGGL(k_rs_term, dim3((nx + 255) / 256, ny), dim3(256), 0, s, w, out, V, nx, ny, ps, pre);
  return hipGetLastError();
}

// ============================================================== detector model
// Radial curve of DQEFunc (U.cu:1120-1132): signed frequency indices, radius
// sqrtf(x'^2 + y'^2) / binning in FP32, entry floor(radius) up to 724, else
// 0.0001.  F *= scale * (root ? sqrtf(curve) : curve)  (DQEKernel takes the
// square root, NTFKernel the curve itself, U.cu:1134-1186).
__global__ void k_detector_filter(float2* F, int nx, int ny, const float* tab, int binning, int root, float scale) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y;
  if (x >= nx) return;
  const int xd = x < nx / 2 ? x : x - nx, yd = y < ny / 2 ? y : y - ny;
  const float r = sqrtf((float)(xd * xd + yd * yd)) / (float)binning;
  const int i = (int)floorf(r);
  const float v = i <= 724 ? tab[i] : 0.0001f;
  const float f = (root ? sqrtf(v) : v) * scale;
  float2& e = F[(long long)y * nx + x];
  e = make_float2(e.x * f, e.y * f);
}
hipError_t launch_detector_filter(float2* F, int nx, int ny, const float* tab, int binning, int root, float scale,
                                  hipStream_t s) {
  hipLaunchKernelGGL(k_detector_filter, dim3((nx + 255) / 256, ny), dim3(256), 0, s, F, nx, ny, tab, binning, root,
                     scale);
  return hipGetLastError();
}

// Philox4x64-10 (Salmon et al., SC'11) on the device; the same generator as
// the host's frozen-phonon displacements.
__device__ void philox4x64_dev(unsigned long long c[4], unsigned long long k0, unsigned long long k1) {
  const unsigned long long M0 = 0xD2E7470EE14C6C93ULL, M1 = 0xCA5A826395121157ULL;
  const unsigned long long W0 = 0x9E3779B97F4A7C15ULL, W1 = 0xBB67AE8584CAA73BULL;
  for (int r = 0; r < 10; ++r) {
    const unsigned long long hi0 = __umul64hi(M0, c[0]), lo0 = M0 * c[0];
    const unsigned long long hi1 = __umul64hi(M1, c[2]), lo1 = M1 * c[2];
    const unsigned long long n0 = hi1 ^ c[1] ^ k0, n2 = hi0 ^ c[3] ^ k1;
    c[0] = n0; c[1] = lo1; c[2] = n2; c[3] = lo0;
    k0 += W0; k1 += W1;
  }
}

// Shot noise of the detector (U.cu:2375-2396), seeded: a = |z| zscale,
// m = dose a, counts = round(m + sqrt(|m|) g) with g the Box-Muller normal of
// Philox block (i, 0xDE7EC7, 3, 0) under key (seed, 0x4D534C), clamped to
// +-3; out = (counts, 0).
__global__ void k_shot_noise(const float2* z, float2* out, long long n, float zscale, float dose,
                             unsigned long long seed) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  unsigned long long c[4] = {(unsigned long long)i, 0xDE7EC7ULL, 3ULL, 0ULL};
  philox4x64_dev(c, seed, 0x4D534CULL);
  const double u1 = ((double)(c[0] >> 11) + 1.0) * (1.0 / 9007199254740992.0);
  const double u2 = (double)(c[1] >> 11) * (1.0 / 9007199254740992.0);
  double g = sqrt(-2.0 * log(u1)) * cos(2.0 * 3.141592653589793 * u2);
  g = g < -3.0 ? -3.0 : (g > 3.0 ? 3.0 : g);
  const float2 v = z[i];
  const double a = (double)(sqrtf(v.x * v.x + v.y * v.y) * zscale);
  const double m = (double)dose * a;
  out[i] = make_float2((float)round(m + sqrt(fabs(m)) * g), 0.f);
}
hipError_t launch_shot_noise(const float2* z, float2* out, long long n, float zscale, float dose,
                             unsigned long long seed, hipStream_t s) {
  hipLaunchKernelGGL(k_shot_noise, dim3(nblk(n, 256)), dim3(256), 0, s, z, out, n, zscale, dose, seed);
  return hipGetLastError();
}

__global__ void k_real_to_complex(const float* in, float2* out, long long n) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = make_float2(in[i], 0.f);
}
hipError_t launch_real_to_complex(const float* in, float2* out, long long n, hipStream_t s) {
  hipLaunchKernelGGL(k_real_to_complex, dim3(nblk(n, 256)), dim3(256), 0, s, in, out, n);
  return hipGetLastError();
}

// ============================================================== CTF
// imagingKernel2, U.cu:1044-1080.  chi and the envelope arguments are
// evaluated in FP64 (they reach ~1e2 rad at large Cs).
__global__ void k_ctf(CtfArgs a) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y, d = blockIdx.z;
  if (x >= a.nx) return;
  const long long id = (long long)y * a.nx + x;
  const float k0x = a.kx[x], k0y = a.ky[y];
  const float k2f = k0x * k0x + k0y * k0y;
  const float objap2 = ((a.obj * 0.001f) / a.wavel) * ((a.obj * 0.001f) / a.wavel);
  float2 out = make_float2(0.f, 0.f);
  if (k2f < objap2) {
    const double lam = a.wavel, k2 = (double)k0x * k0x + (double)k0y * k0y, k = sqrt(k2);
    const double df = a.dfs[d], cs = a.css ? a.css[d] : a.Cs, b = a.beta, dl = a.delta, p1 = 3.141593;
    const double factor = b * b / (4.0 * lam * lam);
    const double esa = p1 * k * lam * 2.0 * df + 2.0 * p1 * lam * lam * lam * cs * k2 * k;
    const double es = exp(-factor * esa * esa);
    const double ed = exp(-0.25 * dl * dl * p1 * p1 * k2 * k2 * lam * lam);
    const double phi = atan2((double)k0y, (double)k0x);
    const double chi = 3.1415926 * lam * k2 *
                       (0.5 * cs * lam * lam * k2 + df + (double)a.A1 * sin(2.0 * (phi - (double)a.A1phi)) +
                        2.0 * (double)a.A2 * lam * k * sin(3.0 * (phi - (double)a.A2phi)) / 3.0);
    double c = chi - 6.283185307179586 * floor(chi / 6.283185307179586);
    float sn, cs_;
    sincosf((float)c, &sn, &cs_);
    const float e = (float)(es * ed) * a.scale;
    const float2 v = a.in[id];
    out = make_float2(e * (v.x * cs_ + v.y * sn), e * (-v.x * sn + v.y * cs_));
  }
  a.out[(long long)d * a.nx * a.ny + id] = out;
}
hipError_t launch_ctf(const CtfArgs& a, hipStream_t s) {
  hipLaunchKernelGGL(k_ctf, dim3(nblk(a.nx, 256), a.ny, a.ndf), dim3(256), 0, s, a);
  return hipGetLastError();
}

// ============================================================== detectors
// CentreKernel + conjugationKernel + host sum of AddTDSWaves (U.cu:2734-2755)
__global__ void k_tds_accum(const float2* F, float* tds, int nx, int ny, int intensity, float scale) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y;
  if (x >= nx) return;
  const int x2 = x >= nx / 2 ? x - nx / 2 : x + nx / 2;
  const int y2 = y >= ny / 2 ? y - ny / 2 : y + ny / 2;
  const float2 v = F[(long long)y2 * nx + x2];
  const float i2 = v.x * v.x + v.y * v.y;
  tds[(long long)y * nx + x] += intensity ? scale * i2 : sqrtf(i2);
}
hipError_t launch_tds_accum(const float2* F, float* tds, int nx, int ny, hipStream_t s) {
  return launch_tds_accum_mode(F, tds, nx, ny, 0, 1.0f, s);
}
hipError_t launch_tds_accum_mode(const float2* F, float* tds, int nx, int ny, int intensity, float scale,
                                 hipStream_t s) {
  hipLaunchKernelGGL(k_tds_accum, dim3(nblk(nx, 256), ny), dim3(256), 0, s, F, tds, nx, ny, intensity, scale);
  return hipGetLastError();
}

__global__ void k_sum_maps(const float* in, int nb, long long n, float* out, int acc) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float s = 0.f;
  for (int b = 0; b < nb; ++b) s += in[(long long)b * n + i];
  out[i] = acc ? out[i] + s : s;
}
hipError_t launch_sum_maps(const float* in, int nb, long long n, float* out, int acc, hipStream_t s) {
  hipLaunchKernelGGL(k_sum_maps, dim3(nblk(n, 256)), dim3(256), 0, s, in, nb, n, out, acc);
  return hipGetLastError();
}

// ============================================================== readback statistics
// Extrema (and for images mean and variance) of a result that is about to be
// read back, so that the host needs neither a copy of its own nor a pass over
// it: 1.4-2.2 ms per megapixel there, 10 us here (two launches, four with the
// variance; bound by their latency).  Partial results per block in a fixed
// order, combined by one block.
// kind 0: modulus of complex values, 1: absolute value of real ones.
constexpr int ST_B = 256;

__device__ __forceinline__ float stat_value(const void* src, long long i, int kind) {
#pragma clang fp contract(off)
  if (kind == 1) return fabsf(((const float*)src)[i]);
  const float2 v = ((const float2*)src)[i];
  return sqrtf(v.x * v.x + v.y * v.y);
}

// sum over the workgroup in a fixed order (every thread gets it)
__device__ __forceinline__ double stat_sum(double v, double* sh) {
  sh[threadIdx.x] = v;
  __syncthreads();
  for (int d = ST_B / 2; d > 0; d >>= 1) {
    if ((int)threadIdx.x < d) sh[threadIdx.x] += sh[threadIdx.x + d];
    __syncthreads();
  }
  const double r = sh[0];
  __syncthreads();
  return r;
}

// largest and smallest value that is a number (-1 and infinity if there is
// none)
__device__ __forceinline__ void stat_range(float& mx, float& mn, float* sh) {
  sh[threadIdx.x] = mx;
  sh[ST_B + threadIdx.x] = mn;
  __syncthreads();
  for (int d = ST_B / 2; d > 0; d >>= 1) {
    if ((int)threadIdx.x < d) {
      sh[threadIdx.x] = fmaxf(sh[threadIdx.x], sh[threadIdx.x + d]);
      sh[ST_B + threadIdx.x] = fminf(sh[ST_B + threadIdx.x], sh[ST_B + threadIdx.x + d]);
    }
    __syncthreads();
  }
  mx = sh[0];
  mn = sh[ST_B];
  __syncthreads();
}

// sum over the w x h corner of |value| (mean == null) or of its squared
// difference from *mean; with mean == null also the extrema of all n values
__global__ void __launch_bounds__(ST_B) k_stat_partial(const void* src, long long n, int kind, int nx, int w, int h,
                                                       const double* mean, double* part, float* range) {
  __shared__ double shd[ST_B];
  __shared__ float shf[2 * ST_B];
  const long long step = (long long)gridDim.x * ST_B, i0 = (long long)blockIdx.x * ST_B + threadIdx.x;
  if (!mean) {
    float mx = -1.f, mn = __builtin_inff();
    for (long long i = i0; i < n; i += step) {
      const float a = stat_value(src, i, kind);  // fmaxf and fminf pass over NaN
      mx = fmaxf(mx, a);
      mn = fminf(mn, a);
    }
    stat_range(mx, mn, shf);
    if (threadIdx.x == 0) {
      range[2 * blockIdx.x] = mx;
      range[2 * blockIdx.x + 1] = mn;
    }
  }
  const double m = mean ? *mean : 0.0;
  double s = 0.0;
  for (long long i = i0; i < (long long)w * h; i += step) {
    const double d = (double)stat_value(src, (i / w) * nx + i % w, kind) - m;
    s += mean ? d * d : d;
  }
  s = stat_sum(s, shd);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// out[0] max, out[1] min, out[2] value of element 0, out[3] mean (mean ==
// null), or out[4] the variance
__global__ void __launch_bounds__(ST_B) k_stat_final(const void* src, int kind, int nblocks, long long count, int var,
                                                     const double* part, const float* range, double* out) {
  __shared__ double shd[ST_B];
  __shared__ float shf[2 * ST_B];
  double s = 0.0;
  for (int i = threadIdx.x; i < nblocks; i += ST_B) s += part[i];
  s = stat_sum(s, shd);
  if (var) {
    if (threadIdx.x == 0) out[4] = s / (double)count;
    return;
  }
  float mx = -1.f, mn = __builtin_inff();
  for (int i = threadIdx.x; i < nblocks; i += ST_B) {
    mx = fmaxf(mx, range[2 * i]);
    mn = fminf(mn, range[2 * i + 1]);
  }
  stat_range(mx, mn, shf);
  if (threadIdx.x == 0) {
    out[0] = mx;
    out[1] = mn;
    out[2] = stat_value(src, 0, kind);
    out[3] = count > 0 ? s / (double)count : 0.0;
  }
}

size_t stat_scratch_doubles() { return 8 + 2 * 1024; }

// statistics of n values (rows of nx) into out5 = scratch[0..4]; w x h is the
// corner of the mean and the variance (0: extrema only).  scratch holds
// stat_scratch_doubles().
hipError_t launch_stats(const void* src, long long n, int kind, int nx, int w, int h, double* scratch, hipStream_t s) {
  if (n < 1 || !src || !scratch) return hipErrorInvalidValue;
  const int nb = (int)std::min<long long>(1024, nblk(n, ST_B * 4));
  double* part = scratch + 8;
  float* range = (float*)(scratch + 8 + 1024);
  const long long cnt = (long long)w * h;
  hipLaunchKernelGGL(k_stat_partial, dim3(nb), dim3(ST_B), 0, s, src, n, kind, nx, w, h, (const double*)nullptr, part,
                     range);
  hipLaunchKernelGGL(k_stat_final, dim3(1), dim3(ST_B), 0, s, src, kind, nb, cnt, 0, part, range, scratch);
  if (cnt > 0) {
    hipLaunchKernelGGL(k_stat_partial, dim3(nb), dim3(ST_B), 0, s, src, n, kind, nx, w, h,
                       (const double*)(scratch + 3), part, range);
    hipLaunchKernelGGL(k_stat_final, dim3(1), dim3(ST_B), 0, s, src, kind, nb, cnt, 1, part, range, scratch);
  }
  return hipGetLastError();
}

// CentreKernel's half-grid shift (U.cu:2734-2755) of one wave
__global__ void k_centre(const float2* in, float2* out, int nx, int ny) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y;
  if (x >= nx) return;
  const int x2 = x >= nx / 2 ? x - nx / 2 : x + nx / 2, y2 = y >= ny / 2 ? y - ny / 2 : y + ny / 2;
  out[(long long)y * nx + x] = in[(long long)y2 * nx + x2];
}
hipError_t launch_centre(const float2* in, float2* out, int nx, int ny, hipStream_t s) {
  hipLaunchKernelGGL(k_centre, dim3(nblk(nx, 256), ny), dim3(256), 0, s, in, out, nx, ny);
  return hipGetLastError();
}

// ============================================================== FD
// finiteDifferenceKernel, U.cu:995-1023 (pi written 3.14159f there)
__global__ void k_fd_update(const float2* grad, const float2* psim, float2* psip, const float2* psi, const float2* V,
                            long long n, long long vper, float sigma, float wavel, float dz) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float a = 2.f * 3.14159f * dz / wavel;
  const float den = 1.f + a * a;
  const float2 rcp = make_float2(1.f / den, -a / den);                     // 1 / (1 + i a)
  const float2 ratio = make_float2((1.f - a * a) / den, -2.f * a / den);   // (1 - i a) / (1 + i a)
  const float2 p = psi[i], g = grad[i], m = psim[i];
  const float vv = dz * dz * 4.f * 3.14159f * sigma * V[i % vper].x / wavel;
  const float2 A = make_float2(2.f * p.x - dz * dz * g.x - vv * p.x, 2.f * p.y - dz * dz * g.y - vv * p.y);
  psip[i] = csub(cmul(rcp, A), cmul(ratio, m));
}
hipError_t launch_fd_update(const float2* grad, const float2* psim, float2* psip, const float2* psi, const float2* V,
                            long long n, long long vper, float sigma, float wavel, float dz, hipStream_t s) {
  if (vper <= 0) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_fd_update, dim3(nblk(n, 256)), dim3(256), 0, s, grad, psim, psip, psi, V, n, vper, sigma, wavel,
                     dz);
  return hipGetLastError();
}

// ============================================================== transmission
// t = exp(i sigma V) of every slice, computed once and read by the row pass
// for every probe of the differentiable path.  Four values per thread (16-byte
// loads, two 16-byte stores) where the arrays allow, one otherwise.  A launch
// per slice cost 4.9 us each at 512^2, latency mostly: 60 slices 293 us, 45
// us in one launch; bound by the stores.
__device__ __forceinline__ float2 phase_of(float v, float sigma) {
  float sn, cs;
  sincosf(sigma * v, &sn, &cs);
  return make_float2(cs, sn);
}
__global__ void __launch_bounds__(256) k_transmission4(const float4* V, float4* t, long long n4, float sigma) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n4) return;
  const float4 v = V[i];
  const float2 a = phase_of(v.x, sigma), b = phase_of(v.y, sigma), c = phase_of(v.z, sigma), d = phase_of(v.w, sigma);
  t[2 * i] = make_float4(a.x, a.y, b.x, b.y);
  t[2 * i + 1] = make_float4(c.x, c.y, d.x, d.y);
}
__global__ void k_transmission(const float* V, float2* t, long long n, float sigma) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) t[i] = phase_of(V[i], sigma);
}
hipError_t launch_transmission(const float* V, float2* t, long long n, float sigma, hipStream_t s) {
  // a launch holds fewer than 2^32 threads: 2^31 values each, a multiple of
  // four (16 GiB of transmissions)
  constexpr long long kPiece = 1LL << 31;
  for (long long o = 0; o < n; o += kPiece) {
    const long long m = std::min(kPiece, n - o);
    const float* v = V + o;
    float2* w = t + o;
    if (m % 4 == 0 && (uintptr_t)v % 16 == 0 && (uintptr_t)w % 16 == 0)
      hipLaunchKernelGGL(k_transmission4, dim3(nblk(m / 4, 256)), dim3(256), 0, s, (const float4*)v, (float4*)w, m / 4,
                         sigma);
    else
      hipLaunchKernelGGL(k_transmission, dim3(nblk(m, 256)), dim3(256), 0, s, v, w, m, sigma);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace msl
