// Smooth particle-mesh Ewald (Essmann et al., J. Chem. Phys. 103, 8577 (1995)), gfx950.
// mdpy has no PME (mdpy/constraint/__init__.py:22 names it; nothing implements it), so this
// is new physics, checked against the float64 oracle in oracle/ewald.py.
//
//   spread   order-4 cardinal B-splines, q_i * sqrt(ke) added to an int64 fixed-point grid
//            (deterministic), one lane per atom
//   FFT      hand-written mixed-radix (2 ... 16) Stockham passes in LDS. The charge grid is real, so
//            two rows along z share one complex transform and Kz/2 + 1 columns go on along y and
//            x; the x-axis kernel also applies the influence function B*C, sums the reciprocal
//            energy and runs the inverse x transform on the same LDS tile
//   gather   one lane per atom, 64 grid values, force = -q grad(theta) . conv
//   corrections  float64 excluded-pair erf correction, self energy and neutralising background,
//                launched with the bonded terms (mdx_bonded.hip)
#include "mdx_internal.h"
#include "mdx_bonded_terms.h"
#include "mdx_nonbonded_body.h"
#include <cmath>

#define PME_BLOCK 256
#define FFT_THREADS 256
#define MAX_RADICES 8

// radix of pass p in bits [8p, 8p+8) of `code` (a register-friendly stand-in for an array that
// a dynamically indexed kernel argument would otherwise put in scratch memory)
struct FftPlan {
  int K;
  int nrad;
  unsigned long long code;
};

struct FftLines {
  int nlines;   // number of lines
  int B;        // lines per block
  int inner, inner_stride, outer_stride, estride;
};

__device__ __forceinline__ float2 cmul(float2 a, float2 b) { return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x); }
__device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ float2 cscale(float2 a, float s) { return make_float2(a.x * s, a.y * s); }
__device__ __forceinline__ float2 mul_i(float2 a, float s) { return make_float2(-s * a.y, s * a.x); }  // (i s) a

// small DFTs, sign s = -1 forward, +1 inverse: U_m = sum_r u_r exp(s 2 pi i r m / R)
__device__ __forceinline__ void dft2(float2* u) {
  float2 a = u[0], b = u[1];
  u[0] = cadd(a, b);
  u[1] = csub(a, b);
}
__device__ __forceinline__ void dft3(float2* u, float s) {
  const float h = 0.86602540378443865f;  // sin(2 pi / 3)
  float2 t1 = cadd(u[1], u[2]);
  float2 t2 = csub(u[0], cscale(t1, 0.5f));
  float2 t3 = mul_i(csub(u[1], u[2]), s * h);
  u[0] = cadd(u[0], t1);
  u[1] = cadd(t2, t3);
  u[2] = csub(t2, t3);
}
__device__ __forceinline__ void dft4(float2* u, float s) {
  float2 a = cadd(u[0], u[2]), b = csub(u[0], u[2]);
  float2 c = cadd(u[1], u[3]), d = mul_i(csub(u[1], u[3]), s);
  u[0] = cadd(a, c);
  u[2] = csub(a, c);
  u[1] = cadd(b, d);
  u[3] = csub(b, d);
}
__device__ __forceinline__ void dft5(float2* u, float s) {
  const float c1 = 0.30901699437494742f, c2 = -0.80901699437494742f;
  const float s1 = 0.95105651629515357f, s2 = 0.58778525229247313f;
  float2 a1 = cadd(u[1], u[4]), b1 = csub(u[1], u[4]);
  float2 a2 = cadd(u[2], u[3]), b2 = csub(u[2], u[3]);
  float2 u0 = u[0];
  float2 p1 = cadd(u0, cadd(cscale(a1, c1), cscale(a2, c2)));
  float2 p2 = cadd(u0, cadd(cscale(a1, c2), cscale(a2, c1)));
  float2 q1 = mul_i(cadd(cscale(b1, s1), cscale(b2, s2)), s);
  float2 q2 = mul_i(csub(cscale(b1, s2), cscale(b2, s1)), s);
  u[0] = cadd(u0, cadd(a1, a2));
  u[1] = cadd(p1, q1);
  u[4] = csub(p1, q1);
  u[2] = cadd(p2, q2);
  u[3] = csub(p2, q2);
}

// W_R^j = cos(2 pi j / R) + i sin(2 pi j / R) of the composite radices
template <int R> struct Roots;
template <> struct Roots<6> { static constexpr float w[6][2] = {{1.0f, 0.0f}, {0.5f, 0.866025404f}, {-0.5f, 0.866025404f}, {-1.0f, 1.2246468e-16f}, {-0.5f, -0.866025404f}, {0.5f, -0.866025404f}}; };
template <> struct Roots<8> { static constexpr float w[8][2] = {{1.0f, 0.0f}, {0.707106781f, 0.707106781f}, {6.123234e-17f, 1.0f}, {-0.707106781f, 0.707106781f}, {-1.0f, 1.2246468e-16f}, {-0.707106781f, -0.707106781f}, {-1.8369702e-16f, -1.0f}, {0.707106781f, -0.707106781f}}; };
template <> struct Roots<9> { static constexpr float w[9][2] = {{1.0f, 0.0f}, {0.766044443f, 0.64278761f}, {0.173648178f, 0.984807753f}, {-0.5f, 0.866025404f}, {-0.939692621f, 0.342020143f}, {-0.939692621f, -0.342020143f}, {-0.5f, -0.866025404f}, {0.173648178f, -0.984807753f}, {0.766044443f, -0.64278761f}}; };
template <> struct Roots<10> { static constexpr float w[10][2] = {{1.0f, 0.0f}, {0.809016994f, 0.587785252f}, {0.309016994f, 0.951056516f}, {-0.309016994f, 0.951056516f}, {-0.809016994f, 0.587785252f}, {-1.0f, 1.2246468e-16f}, {-0.809016994f, -0.587785252f}, {-0.309016994f, -0.951056516f}, {0.309016994f, -0.951056516f}, {0.809016994f, -0.587785252f}}; };
template <> struct Roots<12> { static constexpr float w[12][2] = {{1.0f, 0.0f}, {0.866025404f, 0.5f}, {0.5f, 0.866025404f}, {6.123234e-17f, 1.0f}, {-0.5f, 0.866025404f}, {-0.866025404f, 0.5f}, {-1.0f, 1.2246468e-16f}, {-0.866025404f, -0.5f}, {-0.5f, -0.866025404f}, {-1.8369702e-16f, -1.0f}, {0.5f, -0.866025404f}, {0.866025404f, -0.5f}}; };
template <> struct Roots<16> { static constexpr float w[16][2] = {{1.0f, 0.0f}, {0.923879533f, 0.382683432f}, {0.707106781f, 0.707106781f}, {0.382683432f, 0.923879533f}, {6.123234e-17f, 1.0f}, {-0.382683432f, 0.923879533f}, {-0.707106781f, 0.707106781f}, {-0.923879533f, 0.382683432f}, {-1.0f, 1.2246468e-16f}, {-0.923879533f, -0.382683432f}, {-0.707106781f, -0.707106781f}, {-0.382683432f, -0.923879533f}, {-1.8369702e-16f, -1.0f}, {0.382683432f, -0.923879533f}, {0.707106781f, -0.707106781f}, {0.923879533f, -0.382683432f}}; };

template <int R>
__device__ __forceinline__ void dft(float2* u, float s);
// R = R1 R2: R2 transforms of R1 points (stride R2), the roots between, R1 transforms of R2 points
template <int R1, int R2>
__device__ __forceinline__ void dft_split(float2* u, float s) {
  constexpr int R = R1 * R2;
  float2 v[R];
#pragma unroll
  for (int b = 0; b < R2; ++b) {
    float2 x[R1];
#pragma unroll
    for (int a = 0; a < R1; ++a) x[a] = u[a * R2 + b];
    dft<R1>(x, s);
#pragma unroll
    for (int k = 0; k < R1; ++k) {
      const int j = b * k % R;
      v[k * R2 + b] = j == 0 ? x[k] : cmul(x[k], make_float2(Roots<R>::w[j][0], s * Roots<R>::w[j][1]));
    }
  }
#pragma unroll
  for (int k = 0; k < R1; ++k) {
    dft<R2>(v + k * R2, s);
#pragma unroll
    for (int m = 0; m < R2; ++m) u[k + R1 * m] = v[k * R2 + m];
  }
}
template <int R>
__device__ __forceinline__ void dft(float2* u, float s) {
  if constexpr (R == 2) dft2(u);
  else if constexpr (R == 3) dft3(u, s);
  else if constexpr (R == 4) dft4(u, s);
  else if constexpr (R == 5) dft5(u, s);
  else if constexpr (R == 6) dft_split<2, 3>(u, s);
  else if constexpr (R == 8) dft_split<2, 4>(u, s);
  else if constexpr (R == 9) dft_split<3, 3>(u, s);
  else if constexpr (R == 10) dft_split<2, 5>(u, s);
  else if constexpr (R == 12) dft_split<3, 4>(u, s);
  else dft_split<4, 4>(u, s);
}

// one Stockham pass of radix R over B lines (element e of line l at l*ls + e*es); p is the
// product of the radices of the passes already done, rest = K/p, iB and ip the reciprocals of B and
// p. Consecutive lanes take consecutive lines:
// with ls odd or 1 (in 8-byte elements) every LDS access falls on distinct banks. The quotients by
// B and p are exact in float32 (operands below 2^20).
template <int R>
__device__ __forceinline__ void stockham_pass(const float2* src, float2* dst, int K, int p, int rest, int B, float iB,
                                              float ip, const float2* __restrict__ tw, int ls, int es, float s) {
  const int T = K / R;         // uniform: scalar multiplications
  const int tstep = rest / R;  // K / (p R)
  for (int b = threadIdx.x; b < B * T; b += blockDim.x) {
    const int i = (int)(((float)b + 0.5f) * iB), l = b - i * B;
    const int k = i - (int)(((float)i + 0.5f) * ip) * p;  // i mod p
    const float2* X = src + l * ls;
    float2* Y = dst + l * ls;
    float2 u[R];
#pragma unroll
    for (int r = 0; r < R; ++r) u[r] = X[(i + r * T) * es];
    if (p > 1) {
#pragma unroll
      for (int r = 1; r < R; ++r) {
        float2 w = tw[r * k * tstep];  // r k T/p < K; exp(-2 pi i j/K), conjugated for the inverse
        w.y *= -s;
        u[r] = cmul(u[r], w);
      }
    }
    dft<R>(u, s);
    const int j = (i - k) * R + k;
#pragma unroll
    for (int r = 0; r < R; ++r) Y[(j + r * p) * es] = u[r];
  }
}

// B lines of length K held in LDS (src); element e of line l sits at l*ls + e*es; s = -1 forward,
// +1 inverse. Stockham passes ping-pong with dst; returns the buffer holding the result. The
// kernels run every transform of a workgroup through one call in a loop: a pass is a few hundred
// instructions that a latency-bound workgroup executes once, so a second copy of the code
// (another direction or axis) costs its instruction fetches again.
__device__ __forceinline__ float2* lds_fft(float2* src, float2* dst, const FftPlan& pl, int B,
                                           const float2* __restrict__ tw, int ls, int es, float s) {
  const int K = pl.K;
  const float iB = __builtin_amdgcn_rcpf((float)B);
  float ip = 1.f;
  int p = 1, rest = K;
#pragma unroll 1
  for (int pass = 0; pass < pl.nrad; ++pass) {
    const int R = (int)((pl.code >> (8 * pass)) & 255ull);
    switch (R) {
      case 2: stockham_pass<2>(src, dst, K, p, rest, B, iB, ip, tw, ls, es, s); break;
      case 3: stockham_pass<3>(src, dst, K, p, rest, B, iB, ip, tw, ls, es, s); break;
      case 4: stockham_pass<4>(src, dst, K, p, rest, B, iB, ip, tw, ls, es, s); break;
      case 5: stockham_pass<5>(src, dst, K, p, rest, B, iB, ip, tw, ls, es, s); break;
      case 6: stockham_pass<6>(src, dst, K, p, rest, B, iB, ip, tw, ls, es, s); break;
      case 8: stockham_pass<8>(src, dst, K, p, rest, B, iB, ip, tw, ls, es, s); break;
      case 9: stockham_pass<9>(src, dst, K, p, rest, B, iB, ip, tw, ls, es, s); break;
      case 10: stockham_pass<10>(src, dst, K, p, rest, B, iB, ip, tw, ls, es, s); break;
      case 12: stockham_pass<12>(src, dst, K, p, rest, B, iB, ip, tw, ls, es, s); break;
      default: stockham_pass<16>(src, dst, K, p, rest, B, iB, ip, tw, ls, es, s); break;
    }
    __syncthreads();
    float2* t = src;
    src = dst;
    dst = t;
    p *= R;
    rest = K / p;
    ip = __builtin_amdgcn_rcpf((float)p);
  }
  return src;
}

__device__ __forceinline__ void load_twiddles(float2* dst, const float2* __restrict__ src, int K) {
  for (int i = threadIdx.x; i < K; i += blockDim.x) dst[i] = src[i];
}

__device__ __forceinline__ long long line_base(const FftLines& ln, int l) {
  return (long long)(l / ln.inner) * ln.outer_stride + (long long)(l % ln.inner) * ln.inner_stride;
}

// The axis passes of the path without plane kernels (a full complex grid).
// MODE 0: complex in/out.  MODE 1: load int64 fixed grid (real), clear it.  MODE 2: store real
// part to a float grid.  MODE 3: forward, multiply by B*C (+ energy), inverse, in place.
// lines [l0, l0 + B) of one axis pass, by one workgroup, in the LDS region lds
template <int DIR, int MODE>
__device__ __forceinline__ void fft_axis_body(const FftPlan& pl, const FftLines& ln, const float2* __restrict__ tw,
                              float2* __restrict__ cg, long long* __restrict__ qfix, float* __restrict__ rout,
                              const float* __restrict__ bc, long long* __restrict__ eslot, int l0, float2* lds) {
  const int K = pl.K;
  const int B = ln.B;
  const int nb = min(B, ln.nlines - l0);
  const bool contiguous = ln.estride == 1;
  const int ls = K | 1;  // odd: lanes on consecutive lines use distinct banks
  float2* A = lds;
  float2* Bf = lds + B * ls;
  float2* stw = Bf + B * ls;
  load_twiddles(stw, tw, K);
  // load
  for (int idx = threadIdx.x; idx < nb * K; idx += blockDim.x) {
    int l, e;
    if (contiguous) { l = idx / K; e = idx - l * K; }
    else { e = idx / nb; l = idx - e * nb; }
    long long g = line_base(ln, l0 + l) + (long long)e * ln.estride;
    float2 v;
    if (MODE == 1) {
      long long q = qfix[g];
      qfix[g] = 0;
      v = make_float2((float)((double)q * kFixInv), 0.f);
    } else {
      v = cg[g];
    }
    A[l * ls + e] = v;
  }
  __syncthreads();
  float2* res = A;
  float2* other = Bf;
  double en = 0.0;
#pragma unroll 1
  for (int q = 0; q < (MODE == 3 ? 2 : 1); ++q) {
    float2* r = lds_fft(res, other, pl, nb, stw, ls, 1, MODE == 3 && q == 1 ? (float)-DIR : (float)DIR);
    other = r == res ? other : res;
    res = r;
    if (MODE == 3 && q == 0) {
      for (int idx = threadIdx.x; idx < nb * K; idx += blockDim.x) {
        int l = idx / K, e = idx - l * K;
        long long g = line_base(ln, l0 + l) + (long long)e * ln.estride;
        float f = bc[g];
        float2 v = res[l * ls + e];
        en += 0.5 * (double)f * ((double)v.x * v.x + (double)v.y * v.y);
        res[l * ls + e] = cscale(v, f);
      }
      __syncthreads();
    }
  }
  if (MODE == 3) {  // block energy
    __shared__ double sm[16];
    for (int off = 32; off > 0; off >>= 1) en += __shfl_xor(en, off, 64);
    if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = en;
    __syncthreads();
    if (threadIdx.x == 0) {
      double sacc = 0;
      for (int w = 0; w < (int)(blockDim.x >> 6); ++w) sacc += sm[w];
      atomicAdd((unsigned long long*)eslot, (unsigned long long)to_fix(sacc));
    }
  }
  // store
  for (int idx = threadIdx.x; idx < nb * K; idx += blockDim.x) {
    int l, e;
    if (contiguous) { l = idx / K; e = idx - l * K; }
    else { e = idx / nb; l = idx - e * nb; }
    long long g = line_base(ln, l0 + l) + (long long)e * ln.estride;
    float2 v = res[l * ls + e];
    if (MODE == 2) rout[g] = v.x;
    else cg[g] = v;
  }
}

template <int DIR, int MODE>
__global__ __launch_bounds__(FFT_THREADS) void k_fft_axis(FftPlan pl, FftLines ln, const float2* __restrict__ tw,
                                                        float2* __restrict__ cg, long long* __restrict__ qfix,
                                                        float* __restrict__ rout, const float* __restrict__ bc,
                                                        long long* __restrict__ eslot) {
  extern __shared__ float2 lds[];
  fft_axis_body<DIR, MODE>(pl, ln, tw, cg, qfix, rout, bc, eslot, blockIdx.x * ln.B, lds);
}

// The x-axis pass of the plane path: lines [l0, l0 + B) of the nl = Ky nz columns (y, kz) of the
// half spectrum, element x of line l at x nl + l. Forward transform, multiply by B C (`bc`, same
// layout), reciprocal energy (a column stands for its mirror image too, except kz = 0 and, for
// even Kz, kz = Kz/2), inverse transform, in place.
#define XBC 6  // elements per lane whose influence function is loaded ahead
struct XPass {
  FftPlan pl;
  int nl, nz, kz_even, B;
};
__device__ __forceinline__ void fft_x_body(const XPass& xp, const float2* __restrict__ tw, float2* __restrict__ cg,
                           const float* __restrict__ bc, long long* __restrict__ eslot, int l0, float2* lds) {
  __shared__ double sm[16];
  const int K = xp.pl.K, nb = min(xp.B, xp.nl - l0);
  const int es = xp.B | 1;  // odd: the lanes' strided stores of a pass spread over the banks
  float2* A = lds;
  float2* Bf = lds + es * K;
  float2* stw = Bf + es * K;
  load_twiddles(stw, tw, K);
  const float inb = 1.f / (float)nb;
  float fc[XBC];  // influence function of this lane's first elements, loaded with the grid
#pragma unroll
  for (int q = 0; q < XBC; ++q) {
    const int idx = threadIdx.x + q * blockDim.x;
    fc[q] = 0.f;
    if (idx < nb * K) {
      const int e = (int)(((float)idx + 0.5f) * inb), l = idx - e * nb;
      const long long g = (long long)e * xp.nl + l0 + l;
      fc[q] = bc[g];
      A[e * es + l] = cg[g];
    }
  }
  for (int idx = threadIdx.x + XBC * blockDim.x; idx < nb * K; idx += blockDim.x) {
    const int e = (int)(((float)idx + 0.5f) * inb), l = idx - e * nb;
    A[e * es + l] = cg[(long long)e * xp.nl + l0 + l];
  }
  __syncthreads();
  float2* res = A;
  float2* other = Bf;
  double en = 0.0;
#pragma unroll 1
  for (int q = 0; q < 2; ++q) {
    float2* r = lds_fft(res, other, xp.pl, nb, stw, 1, es, q == 0 ? -1.f : 1.f);
    other = r == res ? other : res;
    res = r;
    if (q == 1) break;
    auto times = [&](int idx, bool held, float fh) {
      const int e = (int)(((float)idx + 0.5f) * inb), l = idx - e * nb;
      const float f = held ? fh : bc[(long long)e * xp.nl + l0 + l];
      const float2 v = res[e * es + l];
      const int kz = (l0 + l) % xp.nz;
      const double w = kz == 0 || (xp.kz_even && kz == xp.nz - 1) ? 0.5 : 1.0;
      en += w * (double)f * ((double)v.x * v.x + (double)v.y * v.y);
      res[e * es + l] = cscale(v, f);
    };
#pragma unroll
    for (int k = 0; k < XBC; ++k)
      if ((int)(threadIdx.x + k * blockDim.x) < nb * K) times(threadIdx.x + k * blockDim.x, true, fc[k]);
    for (int idx = threadIdx.x + XBC * blockDim.x; idx < nb * K; idx += blockDim.x) times(idx, false, 0.f);
    __syncthreads();
  }
  for (int idx = threadIdx.x; idx < nb * K; idx += blockDim.x) {
    const int e = (int)(((float)idx + 0.5f) * inb), l = idx - e * nb;
    cg[(long long)e * xp.nl + l0 + l] = res[e * es + l];
  }
  for (int off = 32; off > 0; off >>= 1) en += __shfl_xor(en, off, 64);
  if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = en;
  __syncthreads();
  if (threadIdx.x == 0) {
    double sacc = 0;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) sacc += sm[w];
    atomicAdd((unsigned long long*)eslot, (unsigned long long)to_fix(sacc));
  }
}

// Latency bound: one 128-byte segment per x and workgroup, two register-level passes each way.
#define FFTX_THREADS 128
#define FFTX_B 8
__global__ __launch_bounds__(FFTX_THREADS) __attribute__((amdgpu_waves_per_eu(4))) void k_fft_x(XPass xp, const float2* __restrict__ tw,
                                                        float2* __restrict__ cg, const float* __restrict__ bc,
                                                        long long* __restrict__ eslot) {
  extern __shared__ float2 lds[];
  fft_x_body(xp, tw, cg, bc, eslot, blockIdx.x * xp.B, lds);
}

// ---------------------------------------------------------------- spread / gather
// weights of the order-4 cardinal B-spline at offset w (grid point base - k) and their derivatives. One
// is the complement of the others, so the weights' sum is 1 and the derivatives' 0 to the last rounding: a
// charge spread with an error in its sum is a long wave, to which the reciprocal energy is most
// sensitive (104 water boxes: energies' error 1.5 to 7 times smaller, forces' 0.95)
__device__ __forceinline__ void bspline4(float w, float* th, float* dth) {
  const float w2 = w * w, w3 = w2 * w, om = 1.f - w;
  th[0] = w3 * (1.f / 6.f);
  th[1] = (-3.f * w3 + 3.f * w2 + 3.f * w + 1.f) * (1.f / 6.f);
  th[3] = om * om * om * (1.f / 6.f);
  th[2] = (1.f - th[1]) - (th[0] + th[3]);
  if (dth) {
    dth[0] = 0.5f * w2;
    dth[1] = 0.5f * (-3.f * w2 + 2.f * w + 1.f);
    dth[3] = -0.5f * om * om;
    dth[2] = -(dth[1] + (dth[0] + dth[3]));
  }
}

struct PmeArgs {
  int n;
  int Kx, Ky, Kz;
  double Lx, Ly, Lz;
  double iLx, iLy, iLz;
};

// fractional grid coordinate of x along an axis with inverse edge iL and K points
__device__ __forceinline__ void frac_coord(double x, double iL, int K, int* base, float* w) {
  double s = x * iL;
  s -= floor(s);
  double u = s * K;
  double f = floor(u);
  // NaN or infinite x: base 0 (range decided before the conversion); u == K after rounding wraps
  int b = f >= 0.0 && f <= (double)K ? (int)f : 0;
  *w = (float)(u - f);
  if (b >= K) b -= K;
  *base = b;
}

// 16 lanes per atom, one per (kx, ky) pencil of the 4x4x4 stencil, each adding the 4 z points
// of its pencil: 16x the parallelism of one lane per atom for the same atomics.
__global__ __launch_bounds__(PME_BLOCK) void k_spread(PmeArgs a, const double* __restrict__ pos,
                                                    const float* __restrict__ qs, long long* __restrict__ qfix) {
  const long long gt = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const int i = (int)(gt >> 4);
  const int kx = (int)(gt >> 2) & 3, ky = (int)gt & 3;
  if (i >= a.n) return;
  const float q = qs[i];
  if (q == 0.f) return;
  int bx, by, bz;
  float wx, wy, wz;
  frac_coord(pos[3 * i], a.iLx, a.Kx, &bx, &wx);
  frac_coord(pos[3 * i + 1], a.iLy, a.Ky, &by, &wy);
  frac_coord(pos[3 * i + 2], a.iLz, a.Kz, &bz, &wz);
  float tx[4], ty[4], tz[4];
  bspline4(wx, tx, nullptr);
  bspline4(wy, ty, nullptr);
  bspline4(wz, tz, nullptr);
  int gx = bx - kx;
  gx += gx < 0 ? a.Kx : 0;
  int gy = by - ky;
  gy += gy < 0 ? a.Ky : 0;
  const float qxy = q * tx[kx] * ty[ky];
  const long long row = ((long long)gx * a.Ky + gy) * a.Kz;
#pragma unroll
  for (int kz = 0; kz < 4; ++kz) {
    int gz = bz - kz;
    gz += gz < 0 ? a.Kz : 0;
    atomicAdd((unsigned long long*)&qfix[row + gz], (unsigned long long)to_fix_f(qxy * tz[kz]));
  }
}

__global__ __launch_bounds__(PME_BLOCK) void k_gather(PmeArgs a, const double* __restrict__ pos,
                                                    const float* __restrict__ qs, const float* __restrict__ conv,
                                                    long long* __restrict__ ffix) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.n) return;
  float q = qs[i];
  if (q == 0.f) return;
  int bx, by, bz;
  float wx, wy, wz;
  frac_coord(pos[3 * i], a.iLx, a.Kx, &bx, &wx);
  frac_coord(pos[3 * i + 1], a.iLy, a.Ky, &by, &wy);
  frac_coord(pos[3 * i + 2], a.iLz, a.Kz, &bz, &wz);
  float tx[4], ty[4], tz[4], dx[4], dy[4], dz[4];
  bspline4(wx, tx, dx);
  bspline4(wy, ty, dy);
  bspline4(wz, tz, dz);
  float gx = 0.f, gy = 0.f, gz = 0.f;
  for (int kx = 0; kx < 4; ++kx) {
    int ix = bx - kx;
    ix += ix < 0 ? a.Kx : 0;
    for (int ky = 0; ky < 4; ++ky) {
      int iy = by - ky;
      iy += iy < 0 ? a.Ky : 0;
      const float* row = conv + ((long long)ix * a.Ky + iy) * a.Kz;
      for (int kz = 0; kz < 4; ++kz) {
        int iz = bz - kz;
        iz += iz < 0 ? a.Kz : 0;
        float cv = row[iz];
        gx += dx[kx] * ty[ky] * tz[kz] * cv;
        gy += tx[kx] * dy[ky] * tz[kz] * cv;
        gz += tx[kx] * ty[ky] * dz[kz] * cv;
      }
    }
  }
  double fx = -(double)q * gx * (a.Kx / a.Lx);
  double fy = -(double)q * gy * (a.Ky / a.Ly);
  double fz = -(double)q * gz * (a.Kz / a.Lz);
  atomicAdd((unsigned long long*)&ffix[i], (unsigned long long)to_fix(fx));
  atomicAdd((unsigned long long*)&ffix[a.n + i], (unsigned long long)to_fix(fy));
  atomicAdd((unsigned long long*)&ffix[2 * a.n + i], (unsigned long long)to_fix(fz));
}

// ---------------------------------------------------------------- plane kernels
// One workgroup per x-plane x0 of the grid. The atoms that touch the plane (floor(u_x) - kx ==
// x0 for some kx in 0..3) are found in the cell-sorted atom order of the neighbour-list grid:
// cells are x-major, so the x-slices of cells that can hold such atoms form at most two
// contiguous ranges of sorted slots, and no atom is more than skin/2 away from its slice.
// Phase 1 (one lane per candidate) lists the touching atoms' slots in LDS; phase 2 (one lane per
// touching atom) computes its splines, adds its 4x4 points and writes the record that the gather
// reads. A plane occupies one compute unit and its VALU and LDS atomics bound it, so both kernels
// are written for few instructions: the second phase runs on touching atoms only (a quarter of the
// candidates), the gather uses one lane per record (the splines once, not once per ky), and the
// set-up of a transform pass runs on scalars (16 waves repeat it). Forward / x pass / gather alone:
// 23,328 atoms, 64^3 20.7 / 8.8 / 16.2 -> 17.1 / 11.1 / 10.3 us; 30,021 atoms, 72^3 28.9 / 16.3 / 27.0
// -> 17.7 / 12.7 / 11.4; 98,304 atoms, 100^3 31.5 / 19.1 / 18.2, against 292 on the global grid, which
// complex planes in LDS left to grids beyond 81 x 81 (half spectra reach 128 x 128).
#define PLANE_THREADS 1024
#define PLANE_REG 8  // row pairs' values held per lane between the two layouts of a plane

struct PlaneArgs {
  int n;
  int Kx, Ky, Kz;
  double Lx, Ly, Lz;
  double iLx, iLy, iLz;
  double gx, gy, gz;  // grid points per A
  int gnx, gny, gnz;  // neighbour-list grid
  double wx;          // its cell width along x
  double margin;      // list skin/2 plus rounding slack
  int W;              // candidates examined per round (bounded by the LDS list of touching ones)
  int rec_cap;        // gather records per plane in global memory
};

struct GatherRec {  // 24 B (stored in an int buffer, 6 words per record)
  int atom;
  int yzk;          // by | bz << 12 | kx << 24
  float wx, wy, wz, q;
};
static_assert(sizeof(GatherRec) == 6 * sizeof(int), "gather record layout");

// weight k of bspline4 and its derivative; branch-free so lanes with different k do not diverge
__device__ __forceinline__ float sel4(int k, float a0, float a1, float a2, float a3) {
  return k == 0 ? a0 : (k == 1 ? a1 : (k == 2 ? a2 : a3));
}
__device__ __forceinline__ float bsp4(float w, int k) {
  float t[4];
  bspline4(w, t, nullptr);
  return sel4(k, t[0], t[1], t[2], t[3]);
}
__device__ __forceinline__ float dbsp4(float w, int k) {
  const float w2 = w * w, om = 1.f - w;
  return sel4(k, w2, -3.f * w2 + 2.f * w + 1.f, 3.f * w2 - 4.f * w, -om * om) * 0.5f;
}

// sorted-slot ranges [b0,e0) and [b1,e1) holding every atom that can touch plane x0
__device__ void plane_ranges(const PlaneArgs& a, const int* __restrict__ cell_start, int x0, int* b0, int* e0,
                             int* b1, int* e1) {
  const double h = a.Lx / a.Kx;
  const int lo = (int)floor((x0 * h - a.margin) / a.wx);
  const int hi = (int)floor(((x0 + 4) * h + a.margin) / a.wx);
  *b1 = *e1 = 0;
  if (hi - lo + 1 >= a.gnx) {
    *b0 = 0;
    *e0 = a.n;
    return;
  }
  const int first = ((lo % a.gnx) + a.gnx) % a.gnx;
  const int last = ((hi % a.gnx) + a.gnx) % a.gnx;
  const int per = a.gny * a.gnz;
  const int s_first = cell_start[first * per];
  const int e_last = last + 1 < a.gnx ? cell_start[(last + 1) * per] : a.n;
  if (first <= last) {
    *b0 = s_first;
    *e0 = e_last;
  } else {
    *b0 = s_first;
    *e0 = a.n;
    *b1 = 0;
    *e1 = e_last;
  }
}

// wave-aggregated slot reservation in an LDS counter
__device__ __forceinline__ int reserve_slot(bool keep, int* counter) {
  const unsigned long long m = __ballot(keep);
  const int lane = threadIdx.x & 63;
  int base = 0;
  const int leader = m ? __ffsll((long long)m) - 1 : 0;
  if (m && lane == leader) base = atomicAdd(counter, __popcll(m));
  base = __shfl(base, leader, 64);
  return base + __popcll(m & ((1ull << lane) - 1ull));
}

// the record of sorted slot s for plane x0: splines' offsets and kx (beyond 3: it does not touch the plane)
__device__ __forceinline__ GatherRec plane_record(const PlaneArgs& a, const int* __restrict__ sorted_orig,
                                                  const double* __restrict__ pos_sorted, const float4* __restrict__ xq,
                                                  int s, int x0, int* by, int* bz, int* kx) {
  const double x = pos_sorted[3 * s], y = pos_sorted[3 * s + 1], z = pos_sorted[3 * s + 2];
  GatherRec g;
  g.q = xq[s].w;
  g.atom = sorted_orig[s];
  int bx;
  frac_coord(x, a.iLx, a.Kx, &bx, &g.wx);
  frac_coord(y, a.iLy, a.Ky, by, &g.wy);
  frac_coord(z, a.iLz, a.Kz, bz, &g.wz);
  *kx = bx - x0;
  *kx += *kx < 0 ? a.Kx : 0;
  g.yzk = *by | (*bz << 12) | (*kx << 24);
  return g;
}

// candidates examined per lane per round of phase 1 (independent loads in flight), and gather
// records held ahead per lane
#define PLANE_U 4
#define GATHER_U 2

// complex elements of one of the two transform buffers of a plane: (Ky + 1)/2 packed lines of
// stride Kz | 1, or Ky rows of the Kz/2 + 1 half spectrum
__host__ __device__ __forceinline__ int plane_buf(int Ky, int Kz) {
  const int packed = ((Ky + 1) / 2) * (Kz | 1), half = Ky * (Kz / 2 + 1);
  return packed > half ? packed : half;
}

// spread q*sqrt(ke) of every atom touching plane x0 into an LDS int64 plane (integer sums, so the
// result is independent of the order of the atomics), then forward FFT along z (two real rows per
// complex line) and y; the half spectrum goes to cg[x0][y][kz], kz <= Kz/2.  LDS: twiddles
// (Kz + Ky), then the int64 plane and the list of touching atoms, which two transform buffers overlay.
__device__ __forceinline__ void plane_fwd_body(const PlaneArgs& a, const FftPlan& plz, const FftPlan& ply,
                               const float2* __restrict__ twz_g, const float2* __restrict__ twy_g,
                               const int* __restrict__ sorted_orig, const int* __restrict__ cell_start,
                               const double* __restrict__ pos_sorted, const float4* __restrict__ xq,
                               float2* __restrict__ cg, GatherRec* __restrict__ grec, int* __restrict__ grec_n,
                               DevState* st, int x0, float2* lds) {
  __shared__ int ntouch;
  const int S = plane_buf(a.Ky, a.Kz);
  float2* twz = lds;
  float2* twy = lds + a.Kz;
  float2* A = twy + a.Ky;
  float2* Bf = A + S;
  const int ls = a.Kz | 1;  // row stride of the fixed-point plane and of the packed lines (odd: the
                            // four rows of a stencil fall on distinct banks)
  long long* plane = (long long*)A;
  int* list = (int*)(plane + a.Ky * ls);
  load_twiddles(twz, twz_g, a.Kz);
  load_twiddles(twy, twy_g, a.Ky);
  for (int i = threadIdx.x; i < a.Ky * ls; i += blockDim.x) plane[i] = 0;
  GatherRec* gout = grec + (long long)x0 * a.rec_cap;
  int b0, e0, b1, e1;
  plane_ranges(a, cell_start, x0, &b0, &e0, &b1, &e1);
  const int len0 = e0 - b0, total = len0 + (e1 - b1);
  int done = 0;  // records written by earlier rounds
  for (int w0 = 0; w0 < total; w0 += a.W) {
    if (threadIdx.x == 0) ntouch = 0;
    __syncthreads();
    const int wend = min(total, w0 + a.W);
    // uniform trip count so every lane reaches the ballots
    for (int c0 = w0; c0 < wend; c0 += PLANE_U * blockDim.x) {
      int sl[PLANE_U];
      double px[PLANE_U];
#pragma unroll
      for (int u = 0; u < PLANE_U; ++u) {
        const int ci = c0 + u * blockDim.x + threadIdx.x;
        sl[u] = ci < wend ? (ci < len0 ? b0 + ci : b1 + (ci - len0)) : -1;
        px[u] = pos_sorted[3 * max(sl[u], 0)];
      }
#pragma unroll
      for (int u = 0; u < PLANE_U; ++u) {
        int bx;
        float wx;
        frac_coord(px[u], a.iLx, a.Kx, &bx, &wx);
        int kx = bx - x0;
        kx += kx < 0 ? a.Kx : 0;
        const bool touch = sl[u] >= 0 && kx <= 3;
        const int slot = reserve_slot(touch, &ntouch);
        if (touch) list[slot] = sl[u];
      }
    }
    __syncthreads();
    const int nt = ntouch;
    for (int e = threadIdx.x; e < nt; e += blockDim.x) {
      int by, bz, kx;
      const GatherRec g = plane_record(a, sorted_orig, pos_sorted, xq, list[e], x0, &by, &bz, &kx);
      const float q = g.q;
      // the gather's record (zero charges included: the gather writes their slot, so every atom
      // owns exactly four)
      if (done + e < a.rec_cap) gout[done + e] = g;
      if (q == 0.f) continue;
      float ty[4], tz[4];
      bspline4(g.wy, ty, nullptr);
      bspline4(g.wz, tz, nullptr);
      const float qx = q * bsp4(g.wx, kx);
      int gz[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) gz[k] = bz - k + (bz < k ? a.Kz : 0);
#pragma unroll
      for (int ky = 0; ky < 4; ++ky) {
        long long* row = plane + (by - ky + (by < ky ? a.Ky : 0)) * ls;
        const float qxy = qx * ty[ky];
#pragma unroll
        for (int kz = 0; kz < 4; ++kz)
          atomicAdd((unsigned long long*)&row[gz[kz]], (unsigned long long)to_fix_f(qxy * tz[kz]));
      }
    }
    done += nt;
    __syncthreads();
  }
  __syncthreads();
  if (threadIdx.x == 0) grec_n[x0] = done;  // beyond rec_cap: the gather walks the candidates itself
  // Rows 2m and 2m + 1 become the real and imaginary part of packed line m (stride Kz | 1). The
  // packed lines overlay the fixed-point plane: every value is in registers before the first
  // store (pairs * Kz <= PLANE_REG * lanes, plane_lanes_ok).
  const int pairs = (a.Ky + 1) >> 1, nz = a.Kz / 2 + 1;
  {
    float2 v[PLANE_REG];
    const float iKz = 1.f / (float)a.Kz;
#pragma unroll
    for (int q = 0; q < PLANE_REG; ++q) {
      const int idx = threadIdx.x + q * blockDim.x;
      if (idx < pairs * a.Kz) {
        const int m = (int)(((float)idx + 0.5f) * iKz), k = idx - m * a.Kz;
        const long long lo = plane[2 * m * ls + k], hi = 2 * m + 1 < a.Ky ? plane[(2 * m + 1) * ls + k] : 0;
        v[q] = make_float2((float)((double)lo * kFixInv), (float)((double)hi * kFixInv));
      }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < PLANE_REG; ++q) {
      const int idx = threadIdx.x + q * blockDim.x;
      if (idx < pairs * a.Kz) {
        const int m = (int)(((float)idx + 0.5f) * iKz);
        A[m * ls + idx - m * a.Kz] = v[q];
      }
    }
  }
  __syncthreads();
  float2* r = A;
  float2* o = Bf;
  const float inz = 1.f / (float)nz;
#pragma unroll 1
  for (int axis = 0; axis < 2; ++axis) {
    float2* f = lds_fft(r, o, axis ? ply : plz, axis ? nz : pairs, axis ? twy : twz, axis ? 1 : ls, axis ? nz : 1, -1.f);
    o = f == r ? o : r;
    r = f;
    if (axis) break;
    // separate the two rows' spectra: X_2m = (Z_k + conj Z_-k)/2, X_2m+1 = (Z_k - conj Z_-k)/2i
    for (int idx = threadIdx.x; idx < pairs * nz; idx += blockDim.x) {
      const int m = (int)(((float)idx + 0.5f) * inz), k = idx - m * nz;
      const float2 p = r[m * ls + k], q = r[m * ls + (k ? a.Kz - k : 0)];
      o[2 * m * nz + k] = make_float2(0.5f * (p.x + q.x), 0.5f * (p.y - q.y));
      if (2 * m + 1 < a.Ky) o[(2 * m + 1) * nz + k] = make_float2(0.5f * (p.y + q.y), 0.5f * (q.x - p.x));
    }
    __syncthreads();
    float2* h = o;
    o = r;
    r = h;
  }
  float2* out = cg + (long long)x0 * (a.Ky * nz);
  for (int i = threadIdx.x; i < a.Ky * nz; i += blockDim.x) out[i] = r[i];
}

__global__ __launch_bounds__(PLANE_THREADS) void k_pme_plane_fwd(
    PlaneArgs a, FftPlan plz, FftPlan ply, const float2* __restrict__ twz_g, const float2* __restrict__ twy_g,
    const int* __restrict__ sorted_orig, const int* __restrict__ cell_start, const double* __restrict__ pos_sorted,
    const float4* __restrict__ xq, float2* __restrict__ cg, GatherRec* __restrict__ grec, int* __restrict__ grec_n,
    DevState* st) {
  extern __shared__ float2 lds[];
  plane_fwd_body(a, plz, ply, twz_g, twy_g, sorted_orig, cell_start, pos_sorted, xq, cg, grec, grec_n, st,
                 blockIdx.x, lds);
}

// inverse FFT along y and z of plane x0, then for every atom touching the plane its share of
// the reciprocal force, -q (dtheta_x theta_y theta_z, ...) . conv over this plane's 4x4 (y,z)
// stencil, written to fpart[kx][3*atom + d] (each slot once per evaluation).
// LDS: twiddles and two transform buffers (plane_buf); the convolved plane is left in packed lines.
__device__ __forceinline__ void plane_gather_body(const PlaneArgs& a, const FftPlan& plz, const FftPlan& ply,
                                  const float2* __restrict__ twz_g, const float2* __restrict__ twy_g,
                                  const int* __restrict__ sorted_orig, const int* __restrict__ cell_start,
                                  const double* __restrict__ pos_sorted, const float4* __restrict__ xq,
                                  const float2* __restrict__ cg, const GatherRec* __restrict__ grec,
                                  const int* __restrict__ grec_n, double* __restrict__ fpart, DevState* st, int x0,
                                  float2* lds) {
  const int S = plane_buf(a.Ky, a.Kz);
  const int pairs = (a.Ky + 1) >> 1, ls = a.Kz | 1, nz = a.Kz / 2 + 1;
  float2* twz = lds;
  float2* twy = lds + a.Kz;
  float2* A = twy + a.Ky;
  float2* Bf = A + S;
  load_twiddles(twz, twz_g, a.Kz);
  load_twiddles(twy, twy_g, a.Ky);
  // the records of the atoms touching this plane, written by the forward kernel; each lane's first
  // ones are loaded with the grid, the others GATHER_U at a time ahead of their use
  const int touching = grec_n[x0];
  const int nr = touching <= a.rec_cap ? touching : 0;
  const GatherRec* gin = grec + (long long)x0 * a.rec_cap;
  GatherRec rec[GATHER_U];
  auto fetch = [&](int e0) {
#pragma unroll
    for (int u = 0; u < GATHER_U; ++u) {
      const int e = e0 + u * (int)blockDim.x;
      if (e < nr) rec[u] = gin[e];
    }
  };
  fetch(threadIdx.x);
  const float2* in = cg + (long long)x0 * (a.Ky * nz);
  for (int i = threadIdx.x; i < a.Ky * nz; i += blockDim.x) A[i] = in[i];
  __syncthreads();
  float2* r = A;
  float2* o = Bf;
  const float inz = 1.f / (float)nz;
#pragma unroll 1
  for (int axis = 0; axis < 2; ++axis) {
    float2* f = lds_fft(r, o, axis ? plz : ply, axis ? pairs : nz, axis ? twz : twy, axis ? ls : 1, axis ? 1 : nz, 1.f);
    o = f == r ? o : r;
    r = f;
    if (axis) break;
    // rows 2m and 2m + 1 again as one packed line, Z = X_2m + i X_2m+1 over the whole period. The
    // coefficients of k = 0 and k = Kz/2 are real but for rounding; packed, the imaginary part of one row's
    // would go to the other, with opposite signs, which a force along y sees in full (reciprocal
    // forces of 30,021 atoms, 72^3: 3.2e-6 of their size off, 0.9e-6 without it)
    for (int idx = threadIdx.x; idx < pairs * nz; idx += blockDim.x) {
      const int m = (int)(((float)idx + 0.5f) * inz), k = idx - m * nz;
      const float2 p = r[2 * m * nz + k], q = 2 * m + 1 < a.Ky ? r[(2 * m + 1) * nz + k] : make_float2(0.f, 0.f);
      const bool real = k == 0 || 2 * k == a.Kz;
      o[m * ls + k] = real ? make_float2(p.x, q.x) : make_float2(p.x - q.y, p.y + q.x);
      if (!real) o[m * ls + a.Kz - k] = make_float2(p.x + q.y, q.x - p.y);
    }
    __syncthreads();
    float2* h = o;
    o = r;
    r = h;
  }
  const float* convr = (const float*)r;  // real parts: row 2m, imaginary parts: row 2m + 1
  const long long n3 = 3LL * a.n;
  // one lane per record; zero charges give zero forces (their slot is still written)
  auto share = [&](const GatherRec& r) {
    const int by = r.yzk & 4095, bz = (r.yzk >> 12) & 4095, kx = r.yzk >> 24;
    float ty[4], dy[4], tz[4], dz[4];
    bspline4(r.wy, ty, dy);
    bspline4(r.wz, tz, dz);
    int gz[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) gz[k] = 2 * (bz - k + (bz < k ? a.Kz : 0));
    float sx = 0.f, sy = 0.f, sz = 0.f;
#pragma unroll
    for (int ky = 0; ky < 4; ++ky) {
      const int gy = by - ky + (by < ky ? a.Ky : 0);
      const float* row = convr + 2 * (gy >> 1) * ls + (gy & 1);
      float c = 0.f, cz = 0.f;
#pragma unroll
      for (int kz = 0; kz < 4; ++kz) {
        const float cv = row[gz[kz]];
        c += tz[kz] * cv;
        cz += dz[kz] * cv;
      }
      sx += ty[ky] * c;
      sy += dy[ky] * c;
      sz += ty[ky] * cz;
    }
    const float tx = bsp4(r.wx, kx), dx = dbsp4(r.wx, kx);
    double* dst = fpart + kx * n3 + 3LL * r.atom;
    const double q = -(double)r.q;
    dst[0] = r.q == 0.f ? 0.0 : q * (double)(dx * sx) * a.gx;
    dst[1] = r.q == 0.f ? 0.0 : q * (double)(tx * sy) * a.gy;
    dst[2] = r.q == 0.f ? 0.0 : q * (double)(tx * sz) * a.gz;
  };
  for (int e0 = threadIdx.x; e0 < nr; e0 += GATHER_U * blockDim.x) {
    GatherRec now[GATHER_U];
#pragma unroll
    for (int u = 0; u < GATHER_U; ++u) now[u] = rec[u];
    fetch(e0 + GATHER_U * blockDim.x);
#pragma unroll
    for (int u = 0; u < GATHER_U; ++u)
      if (e0 + u * (int)blockDim.x < nr) share(now[u]);
  }
  if (touching > a.rec_cap) {
    // more atoms than records (a dense slab along x): every candidate again, as the forward kernel does
    int b0, e0, b1, e1;
    plane_ranges(a, cell_start, x0, &b0, &e0, &b1, &e1);
    const int len0 = e0 - b0, total = len0 + (e1 - b1);
    for (int c = threadIdx.x; c < total; c += blockDim.x) {
      int by, bz, kx;
      const GatherRec g = plane_record(a, sorted_orig, pos_sorted, xq, c < len0 ? b0 + c : b1 + (c - len0), x0, &by,
                                       &bz, &kx);
      if (kx <= 3) share(g);
    }
  }
  // every atom owns exactly one slot per kx: the grid-wide count must be 4 n. One 64-bit add per
  // workgroup carries its slots (40 bits) and its arrival (above); the last of the Kx plane
  // workgroups (launches may hold others) checks the total and re-arms the counter.
  if (threadIdx.x == 0) {
    const unsigned long long mine = (1ull << 40) + (unsigned)touching;
    const unsigned long long all = atomicAdd(&st->pme_count, mine) + mine;
    if (all >> 40 == (unsigned)a.Kx) {
      if ((all & ((1ull << 40) - 1ull)) != 4ull * (unsigned)a.n) atomicOr(&st->flags, MDX_FLAG_PME_COVERAGE);
      atomicExch(&st->pme_count, 0ull);
    }
  }
}

__global__ __launch_bounds__(PLANE_THREADS) void k_pme_plane_inv_gather(
    PlaneArgs a, FftPlan plz, FftPlan ply, const float2* __restrict__ twz_g, const float2* __restrict__ twy_g,
    const int* __restrict__ sorted_orig, const int* __restrict__ cell_start, const double* __restrict__ pos_sorted,
    const float4* __restrict__ xq, const float2* __restrict__ cg, const GatherRec* __restrict__ grec,
    const int* __restrict__ grec_n, double* __restrict__ fpart, DevState* st) {
  extern __shared__ float2 lds[];
  plane_gather_body(a, plz, ply, twz_g, twy_g, sorted_orig, cell_start, pos_sorted, xq, cg, grec, grec_n, fpart, st,
                    blockIdx.x, lds);
}

// Grid-wide barrier of a kernel whose blocks are all resident at once (at most one block per
// compute unit, grid no larger than the device). The last block to arrive resets the count and
// advances the generation; the others wait for that with a bounded spin, so a launch whose
// blocks cannot all be resident raises MDX_FLAG_SYNC and finishes instead of hanging. One
// thread per block fences on each side (device-scope fences act on whole caches: a fence per
// thread would repeat the same cache write-back a thousand times).
__device__ void grid_barrier(DevState* st) {
  __syncthreads();  // every thread's global stores issued and complete at workgroup scope
  if (threadIdx.x == 0) {
    __threadfence();  // release for the whole block: the cache write-back covers all its stores
    const unsigned gen = atomicAdd(&st->bar_gen, 0u);
    const unsigned arrived = atomicAdd(&st->bar_count, 1u);
    if (arrived == gridDim.x - 1) {
      atomicExch(&st->bar_count, 0u);
      __threadfence();
      atomicAdd(&st->bar_gen, 1u);
    } else {
      for (unsigned spin = 0; atomicAdd(&st->bar_gen, 0u) == gen; ++spin) {
        if (spin > (1u << 18)) {
          atomicOr(&st->flags, MDX_FLAG_SYNC);
          break;
        }
        __builtin_amdgcn_s_sleep(2);
      }
    }
    __threadfence();  // acquire: invalidates this compute unit's caches for the whole block
  }
  __syncthreads();
}

// The whole reciprocal-space evaluation in one launch of Kx blocks: block x0 spreads and
// transforms plane x0; after a grid barrier the blocks share the x-axis pass (pencils of the
// Ky x Kz plane, influence function, energy); after a second barrier block x0 transforms plane
// x0 back and gathers its forces. The blocks keep their compute units for the whole
// evaluation, so kernels running concurrently on other streams cannot delay the later phases.
__global__ __launch_bounds__(PLANE_THREADS) void k_pme_fused(
    PlaneArgs a, FftPlan plz, FftPlan ply, XPass xp, const float2* __restrict__ twz_g,
    const float2* __restrict__ twy_g, const float2* __restrict__ twx_g, const int* __restrict__ sorted_orig,
    const int* __restrict__ cell_start, const double* __restrict__ pos_sorted, const float4* __restrict__ xq,
    float2* __restrict__ cg, const float* __restrict__ bc, long long* __restrict__ eslot,
    GatherRec* __restrict__ grec, int* __restrict__ grec_n, double* __restrict__ fpart, DevState* st) {
  extern __shared__ float2 lds[];
  plane_fwd_body(a, plz, ply, twz_g, twy_g, sorted_orig, cell_start, pos_sorted, xq, cg, grec, grec_n, st,
                 blockIdx.x, lds);
  grid_barrier(st);
  const int nchunks = (xp.nl + xp.B - 1) / xp.B;
  for (int ch = blockIdx.x; ch < nchunks; ch += gridDim.x) {
    fft_x_body(xp, twx_g, cg, bc, eslot, ch * xp.B, lds);
    __syncthreads();
  }
  grid_barrier(st);
  plane_gather_body(a, plz, ply, twz_g, twy_g, sorted_orig, cell_start, pos_sorted, xq, cg, grec, grec_n, fpart, st,
                    blockIdx.x, lds);
}

// Phase launches of one force evaluation, on one stream: workgroups [0, npme) run a PME
// reciprocal phase (0: spread + 2D forward FFT per x-plane, 1: x-axis pass with the influence
// function, 2: 2D inverse FFT + gather per x-plane), the next nbn run nonbonded workgroups
// nb0 .. nb0 + nbn - 1 (PLANE_THREADS lanes each), the rest the bonded terms. The PME
// workgroups come first, so they take compute units before the nonbonded ones; the nonbonded
// shares are sized to end with their phase. This replaces the side stream of the three-kernel
// path and its fork and join.
struct PhaseArgs {
  PlaneArgs a;
  FftPlan plz, ply;
  XPass xp;
  const float2 *twz, *twy, *twx;
  const int* sorted_orig;
  const int* cell_start;
  const double* pos_sorted;
  const float4* xq;
  float2* cg;
  const float* bc;
  long long* eslot;
  GatherRec* grec;
  int* grec_n;
  double* fpart;
  DevState* st;
};

template <bool ENERGY, int G>
__global__ __launch_bounds__(PLANE_THREADS) void k_force_phase(int phase, int npme, int nb0, int nbn, PhaseArgs p,
                                                               NbArgs na, NbPtrs P, BondedArgs ba) {
  extern __shared__ float2 lds[];
  const int b = blockIdx.x;
  if (b < npme) {
    if (phase == 0)
      plane_fwd_body(p.a, p.plz, p.ply, p.twz, p.twy, p.sorted_orig, p.cell_start, p.pos_sorted, p.xq, p.cg, p.grec,
                     p.grec_n, p.st, b, lds);
    else if (phase == 1)
      fft_x_body(p.xp, p.twx, p.cg, p.bc, p.eslot, b * p.xp.B, lds);
    else
      plane_gather_body(p.a, p.plz, p.ply, p.twz, p.twy, p.sorted_orig, p.cell_start, p.pos_sorted, p.xq, p.cg,
                        p.grec, p.grec_n, p.fpart, p.st, b, lds);
    return;
  }
  const int vb = b - npme;
  if (vb < nbn) {
    nb_block<true, true, ENERGY, G, PLANE_THREADS, true>(na, P, nb0 + vb);
    return;
  }
  bonded_block(ba, vb - nbn);
}

typedef void (*PhaseKernel)(int, int, int, int, PhaseArgs, NbArgs, NbPtrs, BondedArgs);
static PhaseKernel phase_kernel(bool energy, int G) {
  if (G == 16) return energy ? k_force_phase<true, 16> : k_force_phase<false, 16>;
  if (G == 64) return energy ? k_force_phase<true, 64> : k_force_phase<false, 64>;
  return energy ? k_force_phase<true, 32> : k_force_phase<false, 32>;
}

// LDS bytes of the two plane kernels (the forward one for a window of W candidates)
static inline size_t plane_fwd_lds(int Ky, int Kz, int W) {
  return (size_t)(Ky + Kz) * 8 +
         std::max(2 * (size_t)plane_buf(Ky, Kz) * 8, (size_t)Ky * (Kz | 1) * 8 + (size_t)W * sizeof(int));
}
static inline size_t plane_gather_lds(int Ky, int Kz) {
  return (size_t)(Ky + Kz) * 8 + 2 * (size_t)plane_buf(Ky, Kz) * 8;
}
// the forward kernel holds a plane's packed values in PLANE_REG registers a lane
static inline bool plane_lanes_ok(int Ky, int Kz, int threads) {
  return (long long)((Ky + 1) / 2) * Kz <= (long long)PLANE_REG * threads;
}
static inline size_t x_pass_lds(int K, int B) { return (2 * (size_t)(B | 1) * K + K) * sizeof(float2); }

// ---------------------------------------------------------------- host
// K as a product of the fewest radices (every pass is a round trip through LDS and a barrier), the
// largest one as small as possible among those (fewer registers, more butterflies)
static bool split_radices(int k, int passes, int largest, int* out, int* n) {
  static const int radices[] = {2, 3, 4, 5, 6, 8, 9, 10, 12, 16};
  if (passes == 0) return k == 1;
  for (int q = 9; q >= 0; --q) {
    const int r = radices[q];
    if (r > largest || k % r) continue;
    const int m = *n;
    out[(*n)++] = r;
    if (split_radices(k / r, passes - 1, r, out, n)) return true;
    *n = m;
  }
  return false;
}
static int factorize(int K, FftPlan* pl) {
  static const int radices[] = {2, 3, 4, 5, 6, 8, 9, 10, 12, 16};
  pl->K = K;
  pl->nrad = 0;
  pl->code = 0;
  for (int passes = 1; passes <= MAX_RADICES; ++passes)
    for (int largest : radices) {
      int r[MAX_RADICES], n = 0;
      if (!split_radices(K, passes, largest, r, &n)) continue;
      for (int q = 0; q < n; ++q) pl->code |= (unsigned long long)r[q] << (8 * q);
      pl->nrad = n;
      return 0;
    }
  return -1;
}

// |b(m)|^-2 of Essmann eq. 4.4 for order 4: M4(1)=1/6, M4(2)=2/3, M4(3)=1/6
static void bspline_moduli(int K, std::vector<double>& out) {
  const double M[3] = {1.0 / 6.0, 2.0 / 3.0, 1.0 / 6.0};
  out.assign(K, 0.0);
  std::vector<double> mod(K);
  for (int m = 0; m < K; ++m) {
    double re = 0, im = 0;
    for (int k = 0; k < 3; ++k) {
      double a = 2.0 * M_PI * m * k / K;
      re += M[k] * cos(a);
      im += M[k] * sin(a);
    }
    mod[m] = re * re + im * im;
  }
  for (int m = 0; m < K; ++m)
    if (mod[m] < 1e-10) mod[m] = 0.5 * (mod[(m - 1 + K) % K] + mod[(m + 1) % K]);
  for (int m = 0; m < K; ++m) out[m] = 1.0 / mod[m];
}

extern "C" int mdx_pme_config(mdx_ctx* c, const int* h_grid, int order, double beta) {
  MDX_CHECK(c && c->pos, MDX_ERR_INVALID, "mdx_pme_config: no system bound");
  MDX_CHECK(order == 4, MDX_ERR_INVALID, "only B-spline order 4 is implemented");
  MDX_CHECK(beta > 0, MDX_ERR_INVALID, "beta must be positive");
  FftPlan pl;
  for (int d = 0; d < 3; ++d) {
    MDX_CHECK(h_grid[d] >= 4 && factorize(h_grid[d], &pl) == 0, MDX_ERR_INVALID,
              "PME grid %d must be >= 4 with prime factors 2, 3, 5 only", h_grid[d]);
    c->K[d] = h_grid[d];
  }
  c->order = order;
  c->beta = beta;
  mdx_invalidate_graph(c);
  size_t G = (size_t)c->K[0] * c->K[1] * c->K[2];
  int rc;
  if ((rc = c->qfix.ensure(G)) || (rc = c->cgrid.ensure(G)) || (rc = c->conv.ensure(G)) || (rc = c->bc.ensure(G)) ||
      (rc = c->bch.ensure((size_t)c->K[0] * c->K[1] * (c->K[2] / 2 + 1))) || (rc = c->fpart.ensure(12 * (size_t)c->n)))
    return rc;
  MDX_HIP(hipMemset(c->qfix.p, 0, G * sizeof(long long)));
  // influence function B(m) C(m), C(0) = 0
  std::vector<double> Bm[3];
  for (int d = 0; d < 3; ++d) bspline_moduli(c->K[d], Bm[d]);
  double V = c->box[0] * c->box[1] * c->box[2];
  std::vector<float> h_bc(G);
  for (int x = 0; x < c->K[0]; ++x) {
    double mx = (x <= c->K[0] / 2 ? x : x - c->K[0]) / c->box[0];
    for (int y = 0; y < c->K[1]; ++y) {
      double my = (y <= c->K[1] / 2 ? y : y - c->K[1]) / c->box[1];
      for (int z = 0; z < c->K[2]; ++z) {
        double mz = (z <= c->K[2] / 2 ? z : z - c->K[2]) / c->box[2];
        double m2 = mx * mx + my * my + mz * mz;
        size_t g = ((size_t)x * c->K[1] + y) * c->K[2] + z;
        if (m2 == 0) {
          h_bc[g] = 0.f;
          continue;
        }
        double C = exp(-M_PI * M_PI * m2 / (beta * beta)) / (M_PI * V * m2);
        h_bc[g] = (float)(Bm[0][x] * Bm[1][y] * Bm[2][z] * C);
      }
    }
  }
  MDX_HIP(hipMemcpy(c->bc.p, h_bc.data(), G * sizeof(float), hipMemcpyHostToDevice));
  const int nz = c->K[2] / 2 + 1;  // the plane path's half spectrum
  std::vector<float> h_bch((size_t)c->K[0] * c->K[1] * nz);
  for (size_t row = 0; row < (size_t)c->K[0] * c->K[1]; ++row)
    std::memcpy(&h_bch[row * nz], &h_bc[row * c->K[2]], nz * sizeof(float));
  MDX_HIP(hipMemcpy(c->bch.p, h_bch.data(), h_bch.size() * sizeof(float), hipMemcpyHostToDevice));
  int Kmax = std::max(c->K[0], std::max(c->K[1], c->K[2]));
  if ((rc = c->twiddle.ensure(3 * (size_t)Kmax))) return rc;
  std::vector<float2> tw(3 * (size_t)Kmax);
  for (int d = 0; d < 3; ++d)
    for (int k = 0; k < c->K[d]; ++k) {
      double a = -2.0 * M_PI * k / c->K[d];
      tw[(size_t)d * Kmax + k] = make_float2((float)cos(a), (float)sin(a));
    }
  MDX_HIP(hipMemcpy(c->twiddle.p, tw.data(), tw.size() * sizeof(float2), hipMemcpyHostToDevice));
  // the plane kernels hold twiddles, the fixed-point plane and a window of touching atoms (forward),
  // or two half-spectrum planes (gather) in LDS: up to 128 x 128 points on 160 KB. The window is
  // as large as the device allows (at most 8192 candidates)
  int lds_max = 0;
  MDX_HIP(hipDeviceGetAttribute(&lds_max, hipDeviceAttributeMaxSharedMemoryPerBlock, c->device));
  const size_t budget = lds_max > 1024 ? (size_t)lds_max - 1024 : 0;  // static LDS of the kernels
  c->pme_x_lines = FFTX_B;  // fewer where that many long lines don't fit (grids elongated along x)
  while (c->pme_x_lines > 1 && x_pass_lds(c->K[0], c->pme_x_lines) > budget) c->pme_x_lines /= 2;
  c->pme_wf = 0;
  for (int W = 8192; W >= PLANE_THREADS; W -= PLANE_THREADS)
    if (!c->pme_wf && plane_fwd_lds(c->K[1], c->K[2], W) <= budget) c->pme_wf = W;
  c->pme_planes = c->pme_wf > 0 && plane_gather_lds(c->K[1], c->K[2]) <= budget &&
                  plane_lanes_ok(c->K[1], c->K[2], PLANE_THREADS) && c->K[1] < 4096 && c->K[2] < 4096;
  // gather records: each atom touches 4 of the Kx planes; room for twice the mean plus slack (planes that
  // more atoms touch do without)
  c->pme_rec_cap = (int)std::min<long long>(c->n, 8LL * c->n / c->K[0] + 4096);
  if ((rc = c->pme_grec.ensure((size_t)c->K[0] * c->pme_rec_cap * 6)) || (rc = c->pme_grec_n.ensure(c->K[0])))
    return rc;
  if (c->pme_planes) {  // the whole budget, so contexts with other grids stay launchable
    MDX_HIP(hipFuncSetAttribute((const void*)k_pme_plane_fwd, hipFuncAttributeMaxDynamicSharedMemorySize, (int)budget));
    MDX_HIP(hipFuncSetAttribute((const void*)k_pme_plane_inv_gather, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)budget));
    MDX_HIP(hipFuncSetAttribute((const void*)k_pme_fused, hipFuncAttributeMaxDynamicSharedMemorySize, (int)budget));
    MDX_HIP(hipFuncSetAttribute((const void*)k_fft_x, hipFuncAttributeMaxDynamicSharedMemorySize, (int)budget));
  }
  // one-launch kernel: Kx blocks that must all be resident together (one per compute unit);
  // the x-axis pass takes ceil(Ky Kz / Kx) pencils per block if the LDS allows
  int ncu = 0;
  MDX_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, c->device));
  c->pme_fused_B = 0;
  if (c->pme_planes && c->K[0] <= ncu) {
    const int nl = c->K[1] * nz;
    int B = (nl + c->K[0] - 1) / c->K[0];
    while (B > 1 && x_pass_lds(c->K[0], B) > budget) B = (B + 1) / 2;
    const size_t lds_x = x_pass_lds(c->K[0], B);
    c->pme_fused_B = lds_x <= budget ? B : 0;
    c->pme_fused_lds = std::max(lds_x, std::max(plane_fwd_lds(c->K[1], c->K[2], c->pme_wf),
                                                plane_gather_lds(c->K[1], c->K[2])));
  }
  // phase launches: their static LDS (the nonbonded workgroups' table) comes off the budget
  c->pme_wf_phase = 0;
  if (c->pme_planes && c->pme_fused_B > 0) {
    size_t st_max = 0;
    for (int e = 0; e < 2; ++e)
      for (int G = 16; G <= 64; G *= 2) {
        hipFuncAttributes fa;
        MDX_HIP(hipFuncGetAttributes(&fa, (const void*)phase_kernel(e != 0, G)));
        st_max = std::max(st_max, (size_t)fa.sharedSizeBytes);
      }
    const size_t pb = (size_t)lds_max > st_max + 256 ? (size_t)lds_max - st_max - 256 : 0;
    for (int W = 8192; W >= PLANE_THREADS; W -= PLANE_THREADS)
      if (!c->pme_wf_phase && plane_fwd_lds(c->K[1], c->K[2], W) <= pb) c->pme_wf_phase = W;
    const size_t lx = x_pass_lds(c->K[0], c->pme_fused_B);
    if (plane_gather_lds(c->K[1], c->K[2]) > pb || lx > pb) c->pme_wf_phase = 0;
    if (c->pme_wf_phase)
      for (int e = 0; e < 2; ++e)
        for (int G = 16; G <= 64; G *= 2)
          MDX_HIP(hipFuncSetAttribute((const void*)phase_kernel(e != 0, G),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)pb));
  }
  if ((rc = mdx_coulomb_table_update(c))) return rc;
  c->pme_configured = true;
  return 0;
}

extern "C" int mdx_pme_set_fused(mdx_ctx* c, int enable) {
  MDX_CHECK(c, MDX_ERR_INVALID, "mdx_pme_set_fused: null context");
  c->pme_fused_on = enable != 0;
  mdx_invalidate_graph(c);
  return 0;
}

// one axis pass of a context's grid: its transform plan, line layout, twiddles and dynamic LDS
static void fft_axis_of(const mdx_ctx* c, int axis, FftPlan* plo, FftLines* lno, const float2** two, size_t* ldso) {
  const int Kx = c->K[0], Ky = c->K[1], Kz = c->K[2];
  FftPlan& pl = *plo;
  FftLines& ln = *lno;
  int Kmax = std::max(Kx, std::max(Ky, Kz));
  if (axis == 2) {
    factorize(Kz, &pl);
    ln.nlines = Kx * Ky;
    ln.inner = ln.nlines;
    ln.inner_stride = Kz;
    ln.outer_stride = 0;
    ln.estride = 1;
    ln.B = std::max(1, 1024 / Kz);
  } else if (axis == 1) {
    factorize(Ky, &pl);
    ln.nlines = Kx * Kz;
    ln.inner = Kz;
    ln.inner_stride = 1;
    ln.outer_stride = Ky * Kz;
    ln.estride = Kz;
    ln.B = std::min(16, Kz);
  } else {
    factorize(Kx, &pl);
    ln.nlines = Ky * Kz;
    ln.inner = ln.nlines;
    ln.inner_stride = 1;
    ln.outer_stride = 0;
    ln.estride = Ky * Kz;
    ln.B = std::min(16, Kz);
  }
  *two = c->twiddle.p + (size_t)axis * Kmax;
  *ldso = (2 * (size_t)ln.B * (pl.K | 1) + pl.K) * sizeof(float2);
}

// the plane path's x-axis pass, B lines per workgroup
static XPass x_pass_of(const mdx_ctx* c, int B) {
  XPass xp;
  factorize(c->K[0], &xp.pl);
  xp.nz = c->K[2] / 2 + 1;
  xp.nl = c->K[1] * xp.nz;
  xp.kz_even = c->K[2] % 2 == 0;
  xp.B = B;
  return xp;
}

static int fft_pass(mdx_ctx* c, int axis, int dir, int mode) {
  FftPlan pl;
  FftLines ln;
  const float2* tw;
  size_t lds;
  fft_axis_of(c, axis, &pl, &ln, &tw, &lds);
  dim3 grid(div_up(ln.nlines, ln.B));
#define FFT_L(D, M)                                                                                    \
  k_fft_axis<D, M><<<grid, FFT_THREADS, lds, c->stream>>>(pl, ln, tw, c->cgrid.p, c->qfix.p, c->conv.p, c->bc.p, \
                                                          c->efix.p + 2)
  if (mode == 1) FFT_L(-1, 1);
  else if (mode == 3) FFT_L(-1, 3);
  else if (mode == 2) FFT_L(1, 2);
  else if (dir < 0) FFT_L(-1, 0);
  else FFT_L(1, 0);
#undef FFT_L
  MDX_LAUNCH_CHECK();
  return 0;
}

// plane path: spread + 2D forward FFT per x-plane, x-axis pass with the influence function,
// 2D inverse FFT + gather per x-plane. Needs the cell-sorted atom order of the neighbour-list
// grid (current for this evaluation) and two complex planes in LDS.
// parts: bit 0 the plane forward kernel, bit 1 the x-axis transform pass, bit 2 the inverse +
// gather kernel (all three for an evaluation; one at a time for timing)
// the plane kernels' arguments of a context (a.W: the forward kernel's record window)
static void plane_args_of(const mdx_ctx* c, PlaneArgs* out) {
  const int Kx = c->K[0], Ky = c->K[1], Kz = c->K[2];
  PlaneArgs& a = *out;
  a.n = c->n;
  a.Kx = Kx;
  a.Ky = Ky;
  a.Kz = Kz;
  a.Lx = c->box[0];
  a.Ly = c->box[1];
  a.Lz = c->box[2];
  a.iLx = 1.0 / c->box[0];
  a.iLy = 1.0 / c->box[1];
  a.iLz = 1.0 / c->box[2];
  a.gx = Kx / c->box[0];
  a.gy = Ky / c->box[1];
  a.gz = Kz / c->box[2];
  a.gnx = c->gn[0];
  a.gny = c->gn[1];
  a.gnz = c->gn[2];
  a.wx = c->box[0] / c->gn[0];
  a.margin = 0.5 * c->skin + 1e-6 * c->box[0] + 1e-9;
  a.rec_cap = c->pme_rec_cap;
  a.W = c->pme_wf;
}

static int pme_enqueue_planes(mdx_ctx* c, unsigned parts = 7u) {
  const int Kx = c->K[0], Ky = c->K[1], Kz = c->K[2];
  PlaneArgs a;
  plane_args_of(c, &a);
  MDX_CHECK(c->pme_grec.n >= (size_t)Kx * a.rec_cap * 6, MDX_ERR_INVALID, "PME configured for another system size");
  GatherRec* grec = (GatherRec*)c->pme_grec.p;
  FftPlan plz, ply;
  factorize(Kz, &plz);
  factorize(Ky, &ply);
  const int Kmax = std::max(Kx, std::max(Ky, Kz));
  const float2* twy = c->twiddle.p + (size_t)Kmax;
  const float2* twz = c->twiddle.p + 2 * (size_t)Kmax;
  if (parts == 7u && c->pme_fused_B > 0 && c->pme_fused_on && !c->in_batch) {
    a.W = c->pme_wf;
    k_pme_fused<<<Kx, PLANE_THREADS, c->pme_fused_lds, c->stream>>>(
        a, plz, ply, x_pass_of(c, c->pme_fused_B), twz, twy, c->twiddle.p, c->sorted_orig.p, c->cell_start.p,
        c->pos_sorted.p, c->xq.p, c->cgrid.p, c->bch.p, c->efix.p + 2, grec, c->pme_grec_n.p, c->fpart.p, c->dstate.p);
    MDX_LAUNCH_CHECK();
    return 0;
  }
  a.W = c->pme_wf;
  if (parts & 1u) {
    k_pme_plane_fwd<<<Kx, PLANE_THREADS, plane_fwd_lds(Ky, Kz, a.W), c->stream>>>(
        a, plz, ply, twz, twy, c->sorted_orig.p, c->cell_start.p, c->pos_sorted.p, c->xq.p, c->cgrid.p, grec,
        c->pme_grec_n.p, c->dstate.p);
    MDX_LAUNCH_CHECK();
  }
  if (parts & 2u) {  // x forward, * B C, energy, x inverse
    const XPass xp = x_pass_of(c, c->pme_x_lines);
    k_fft_x<<<div_up(xp.nl, xp.B), FFTX_THREADS, x_pass_lds(Kx, xp.B), c->stream>>>(xp, c->twiddle.p, c->cgrid.p,
                                                                                   c->bch.p, c->efix.p + 2);
    MDX_LAUNCH_CHECK();
  }
  if (parts & 4u) {
    k_pme_plane_inv_gather<<<Kx, PLANE_THREADS, plane_gather_lds(Ky, Kz), c->stream>>>(
        a, plz, ply, twz, twy, c->sorted_orig.p, c->cell_start.p, c->pos_sorted.p, c->xq.p, c->cgrid.p, grec,
        c->pme_grec_n.p, c->fpart.p, c->dstate.p);
    MDX_LAUNCH_CHECK();
  }
  return 0;
}

// One of the plane path's three launches alone (part 0, 1 or 2 of pme_enqueue_planes), for
// timing: each reads only what the previous evaluation's launches left in place.
int mdx_pme_enqueue_part(mdx_ctx* c, int part) {
  MDX_CHECK(c->pme_configured && c->pme_planes && c->nb_configured && part >= 0 && part <= 2, MDX_ERR_INVALID,
            "PME part timing needs the plane path");
  return pme_enqueue_planes(c, 1u << part);
}

bool mdx_force_phases_ok(const mdx_ctx* c) {
  return c->phases_on && c->pme_configured && c->pme_planes && c->pme_wf_phase > 0 && c->pme_fused_B > 0 &&
         c->nb_configured && c->has_lj && c->has_charges;
}

int mdx_force_phases_enqueue(mdx_ctx* c, bool energy, unsigned bonded_terms) {
  MDX_CHECK(mdx_force_phases_ok(c), MDX_ERR_INVALID, "phase launches not available for this context");
  MDX_CHECK(c->fpart.p && c->fpart.n >= 12 * (size_t)c->n, MDX_ERR_INVALID, "PME configured for another system size");
  const int Kx = c->K[0], Ky = c->K[1], Kz = c->K[2];
  PhaseArgs p;
  PlaneArgs& a = p.a;
  plane_args_of(c, &a);
  a.W = c->pme_wf_phase;
  MDX_CHECK(c->pme_grec.n >= (size_t)Kx * a.rec_cap * 6, MDX_ERR_INVALID, "PME configured for another system size");
  factorize(Kz, &p.plz);
  factorize(Ky, &p.ply);
  p.xp = x_pass_of(c, c->pme_fused_B);
  const int Kmax = std::max(Kx, std::max(Ky, Kz));
  p.twx = c->twiddle.p;
  p.twy = c->twiddle.p + (size_t)Kmax;
  p.twz = c->twiddle.p + 2 * (size_t)Kmax;
  p.sorted_orig = c->sorted_orig.p;
  p.cell_start = c->cell_start.p;
  p.pos_sorted = c->pos_sorted.p;
  p.xq = c->xq.p;
  p.cg = c->cgrid.p;
  p.bc = c->bch.p;
  p.eslot = c->efix.p + 2;
  p.grec = (GatherRec*)c->pme_grec.p;
  p.grec_n = c->pme_grec_n.p;
  p.fpart = c->fpart.p;
  p.st = c->dstate.p;
  const NbArgs na = nb_args(c);
  const NbPtrs P = nb_ptrs(c);
  MDX_CHECK(na.ctab && c->ctab_beta == c->beta && c->ctab_rc == c->rc, MDX_ERR_INVALID,
            "Ewald-correction table not built for the current beta and cutoff");
  BondedArgs ba{};
  const int nbo = bonded_terms ? mdx_bonded_args(c, bonded_terms, &ba, PLANE_THREADS) : 0;
  const int G = mdx_nb_lanes(c);
  const int nbt = (int)div_up((long long)c->n * G, PLANE_THREADS);
  const int n0 = std::min(nbt, (int)(c->phase_frac[0] * nbt + 0.5));
  const int n1 = std::min(nbt - n0, (int)(c->phase_frac[1] * nbt + 0.5));
  const int n2 = nbt - n0 - n1;
  const int nx = div_up(p.xp.nl, p.xp.B);  // x-pass workgroups
  const size_t lx = x_pass_lds(Kx, p.xp.B);
  PhaseKernel k = phase_kernel(energy, G);
  k<<<Kx + n0, PLANE_THREADS, plane_fwd_lds(Ky, Kz, a.W), c->stream>>>(0, Kx, 0, n0, p, na, P, ba);
  MDX_LAUNCH_CHECK();
  k<<<nx + n1, PLANE_THREADS, lx, c->stream>>>(1, nx, n0, n1, p, na, P, ba);
  MDX_LAUNCH_CHECK();
  k<<<Kx + n2 + nbo, PLANE_THREADS, plane_gather_lds(Ky, Kz), c->stream>>>(2, Kx, n0 + n1, n2, p, na, P, ba);
  MDX_LAUNCH_CHECK();
  c->fpart_live = true;
  return 0;
}

extern "C" int mdx_force_phases_config(mdx_ctx* c, int enable, double frac0, double frac1) {
  MDX_CHECK(c, MDX_ERR_INVALID, "mdx_force_phases_config: no context");
  MDX_CHECK(frac0 >= 0 && frac1 >= 0 && frac0 + frac1 <= 1, MDX_ERR_INVALID,
            "nonbonded shares must be >= 0 and sum to at most 1");
  c->phases_on = enable != 0;
  c->phase_frac[0] = frac0;
  c->phase_frac[1] = frac1;
  mdx_invalidate_graph(c);
  return 0;
}

int mdx_pme_enqueue(mdx_ctx* c, bool energy) {
  (void)energy;
  MDX_CHECK(c->pme_configured, MDX_ERR_INVALID, "PME not configured");
  if (c->pme_planes && c->nb_configured) {
    MDX_CHECK(c->fpart.p && c->fpart.n >= 12 * (size_t)c->n, MDX_ERR_INVALID, "PME configured for another system size");
    int rc;
    if ((rc = pme_enqueue_planes(c))) return rc;
    c->fpart_live = true;
    return 0;
  }
  c->fpart_live = false;
  PmeArgs a;
  a.n = c->n;
  a.Kx = c->K[0];
  a.Ky = c->K[1];
  a.Kz = c->K[2];
  a.Lx = c->box[0];
  a.Ly = c->box[1];
  a.Lz = c->box[2];
  a.iLx = 1.0 / c->box[0];
  a.iLy = 1.0 / c->box[1];
  a.iLz = 1.0 / c->box[2];
  k_spread<<<div_up(16LL * c->n, PME_BLOCK), PME_BLOCK, 0, c->stream>>>(a, c->pos, c->charge_s.p, c->qfix.p);
  MDX_LAUNCH_CHECK();
  int rc;
  if ((rc = fft_pass(c, 2, -1, 1))) return rc;  // z forward, from the fixed-point grid
  if ((rc = fft_pass(c, 1, -1, 0))) return rc;  // y forward
  if ((rc = fft_pass(c, 0, -1, 3))) return rc;  // x forward, * B C, energy, x inverse
  if ((rc = fft_pass(c, 1, 1, 0))) return rc;   // y inverse
  if ((rc = fft_pass(c, 2, 1, 2))) return rc;   // z inverse, real part out
  k_gather<<<div_up(c->n, PME_BLOCK), PME_BLOCK, 0, c->stream>>>(a, c->pos, c->charge_s.p, c->conv.p, c->ffix.p);
  MDX_LAUNCH_CHECK();
  return 0;
}


// ---------------------------------------------------------------- batched replicas
// The three plane-path launches of every replica of a batch: each replica's arguments are the
// record a single-context launch passes by value.
struct PlaneCall {
  PlaneArgs a;
  FftPlan plz, ply;
  const float2* twz;
  const float2* twy;
  const int* sorted_orig;
  const int* cell_start;
  const double* pos_sorted;
  const float4* xq;
  float2* cg;
  GatherRec* grec;
  int* grec_n;
  double* fpart;
  DevState* st;
};
struct FftCall {
  XPass xp;
  const float2* tw;
  float2* cg;
  const float* bc;
  long long* eslot;
};

// Batched plane kernels of BS lanes: PLANE_THREADS, or fewer when every replica's planes are small.
template <int BS>
__global__ __launch_bounds__(BS) void k_pme_plane_fwd_batch(BatchMap map, const PlaneCall* __restrict__ calls) {
  extern __shared__ float2 lds[];
  int x0;
  const PlaneCall& p = calls[batch_replica(map, &x0)];
  plane_fwd_body(p.a, p.plz, p.ply, p.twz, p.twy, p.sorted_orig, p.cell_start, p.pos_sorted, p.xq, p.cg, p.grec,
                 p.grec_n, p.st, x0, lds);
}
__global__ __launch_bounds__(FFTX_THREADS) __attribute__((amdgpu_waves_per_eu(4))) void k_fft_x_batch(BatchMap map, const FftCall* __restrict__ calls) {
  extern __shared__ float2 lds[];
  int ch;
  const FftCall& f = calls[batch_replica(map, &ch)];
  fft_x_body(f.xp, f.tw, f.cg, f.bc, f.eslot, ch * f.xp.B, lds);
}
template <int BS>
__global__ __launch_bounds__(BS) void k_pme_plane_inv_gather_batch(BatchMap map, const PlaneCall* __restrict__ calls) {
  extern __shared__ float2 lds[];
  int x0;
  const PlaneCall& p = calls[batch_replica(map, &x0)];
  plane_gather_body(p.a, p.plz, p.ply, p.twz, p.twy, p.sorted_orig, p.cell_start, p.pos_sorted, p.xq, p.cg, p.grec,
                    p.grec_n, p.fpart, p.st, x0, lds);
}
// The batched forward kernel runs 256-lane workgroups with a window of 1,024 candidates where every
// replica's planes fit their registers (plane_lanes_ok: 2,048 packed values, 64 x 64 points): more planes
// in flight, 54 us against 113 with PLANE_THREADS lanes over 64 water replicas (321,897 atoms), 4.35
// against 4.07e8 atom-steps/s. The gather keeps PLANE_THREADS lanes: alone 71 us, 35 with 256 lanes and
// 40 with 512, but a whole step waits for the nonbonded kernel beside it (4.35, 4.36 and 4.32e8).
#define PLANE_BATCH_SMALL 256
#define PLANE_BATCH_W 1024

int mdx_batch_prepare_pme(mdx_ctx* const* cs, int n, BatchKind* fwd, BatchKind* fft, BatchKind* gat) {
  std::vector<PlaneCall> pc;
  std::vector<FftCall> fc;
  std::vector<int> bp, bf;
  size_t lf = 0, lx = 0, lg = 0;
  bool small = true;
  for (int r = 0; r < n; ++r) small &= plane_lanes_ok(cs[r]->K[1], cs[r]->K[2], PLANE_BATCH_SMALL);
  const int fthreads = small ? PLANE_BATCH_SMALL : PLANE_THREADS;
  for (int r = 0; r < n; ++r) {
    mdx_ctx* c = cs[r];
    MDX_CHECK(c->pme_configured && c->pme_planes && c->nb_configured && c->has_charges, MDX_ERR_INVALID,
              "replica %d: batched steps need the PME plane path", r);
    PlaneCall p;
    plane_args_of(c, &p.a);
    if (small) p.a.W = std::min(p.a.W, PLANE_BATCH_W);
    MDX_CHECK(c->pme_grec.n >= (size_t)c->K[0] * p.a.rec_cap * 6 && c->fpart.p && c->fpart.n >= 12 * (size_t)c->n,
              MDX_ERR_INVALID, "replica %d: PME configured for another system size", r);
    factorize(c->K[2], &p.plz);
    factorize(c->K[1], &p.ply);
    const int Kmax = std::max(c->K[0], std::max(c->K[1], c->K[2]));
    p.twy = c->twiddle.p + (size_t)Kmax;
    p.twz = c->twiddle.p + 2 * (size_t)Kmax;
    p.sorted_orig = c->sorted_orig.p;
    p.cell_start = c->cell_start.p;
    p.pos_sorted = c->pos_sorted.p;
    p.xq = c->xq.p;
    p.cg = c->cgrid.p;
    p.grec = (GatherRec*)c->pme_grec.p;
    p.grec_n = c->pme_grec_n.p;
    p.fpart = c->fpart.p;
    p.st = c->dstate.p;
    pc.push_back(p);
    bp.push_back(c->K[0]);
    lf = std::max(lf, plane_fwd_lds(c->K[1], c->K[2], p.a.W));
    lg = std::max(lg, plane_gather_lds(c->K[1], c->K[2]));
    FftCall f;
    f.xp = x_pass_of(c, c->pme_x_lines);
    f.tw = c->twiddle.p;
    f.cg = c->cgrid.p;
    f.bc = c->bch.p;
    f.eslot = c->efix.p + 2;
    fc.push_back(f);
    bf.push_back(div_up(f.xp.nl, f.xp.B));
    lx = std::max(lx, x_pass_lds(c->K[0], f.xp.B));
  }
  const void* kf = fthreads == PLANE_THREADS ? (const void*)k_pme_plane_fwd_batch<PLANE_THREADS>
                                             : (const void*)k_pme_plane_fwd_batch<PLANE_BATCH_SMALL>;
  MDX_HIP(hipFuncSetAttribute(kf, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lf));
  MDX_HIP(hipFuncSetAttribute((const void*)k_fft_x_batch, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lx));
  MDX_HIP(hipFuncSetAttribute((const void*)k_pme_plane_inv_gather_batch<PLANE_THREADS>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lg));
  int rc;
  if ((rc = batch_kind_upload(fwd, pc, bp, lf)) || (rc = batch_kind_upload(fft, fc, bf, lx)) ||
      (rc = batch_kind_upload(gat, pc, bp, lg)))
    return rc;
  fwd->threads = fthreads;
  fft->threads = FFTX_THREADS;
  gat->threads = PLANE_THREADS;
  return 0;
}

int mdx_batch_launch_pme(const BatchKind& fwd, const BatchKind& fft, const BatchKind& gat, hipStream_t s,
                         unsigned parts) {
  const bool big = fwd.threads == PLANE_THREADS;
  if (parts & 1u) {
    if (big)
      k_pme_plane_fwd_batch<PLANE_THREADS><<<fwd.blocks, PLANE_THREADS, fwd.lds, s>>>(fwd.map, (const PlaneCall*)fwd.calls);
    else
      k_pme_plane_fwd_batch<PLANE_BATCH_SMALL><<<fwd.blocks, PLANE_BATCH_SMALL, fwd.lds, s>>>(fwd.map,
                                                                                          (const PlaneCall*)fwd.calls);
    MDX_LAUNCH_CHECK();
  }
  if (parts & 2u) {
    k_fft_x_batch<<<fft.blocks, FFTX_THREADS, fft.lds, s>>>(fft.map, (const FftCall*)fft.calls);
    MDX_LAUNCH_CHECK();
  }
  if (parts & 4u) {
    k_pme_plane_inv_gather_batch<PLANE_THREADS><<<gat.blocks, PLANE_THREADS, gat.lds, s>>>(
        gat.map, (const PlaneCall*)gat.calls);
    MDX_LAUNCH_CHECK();
  }
  return 0;
}
