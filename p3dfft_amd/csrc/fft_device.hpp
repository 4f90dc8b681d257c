// fft_device.hpp -- device-side building blocks of the gfx950 FFT engine.
//
// Complex numbers are (re, im) pairs of float or double.  A transform of length
// n = r_0 r_1 ... r_{S-1} is run as S stages over data held in LDS; each stage
// reads R values per butterfly into registers, applies the stage twiddles, runs
// a length-R DFT in registers and writes the results in place (positions in
// mixed radix, one side digit-reversed) or, where both sides are in natural
// order, to their autosorted position.  Twiddles are FP64-generated tables; the FP32
// engine stores each twiddle as a hi+lo pair of floats and multiplies with
// both (compensated twiddle multiply).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace p3amd {

template <class T>
struct alignas(2 * sizeof(T)) cpx {
  T x, y;
};

template <class T>
__device__ __forceinline__ cpx<T> mk(T a, T b) { cpx<T> r; r.x = a; r.y = b; return r; }
template <class T>
__device__ __forceinline__ cpx<T> add(cpx<T> a, cpx<T> b) { return mk<T>(a.x + b.x, a.y + b.y); }
template <class T>
__device__ __forceinline__ cpx<T> sub(cpx<T> a, cpx<T> b) { return mk<T>(a.x - b.x, a.y - b.y); }
template <class T>
__device__ __forceinline__ cpx<T> scl(cpx<T> a, T s) { return mk<T>(a.x * s, a.y * s); }
// multiply by -i (forward) or +i (backward)
template <bool FWD, class T>
__device__ __forceinline__ cpx<T> rot(cpx<T> a) { return FWD ? mk<T>(a.y, -a.x) : mk<T>(-a.y, a.x); }

// ---------------------------------------------------------------------------
// twiddle storage
//   double : double2 w = exp(-2 pi i e / M)
//   float  : float4 (hi.re, hi.im, lo.re, lo.im) with hi = fl32(w), lo = fl32(w - hi)
// Backward transforms use the conjugate.
// ---------------------------------------------------------------------------
template <class T> struct TwT;
template <> struct TwT<double> { typedef double2 type; };
template <> struct TwT<float> { typedef float4 type; };

template <bool FWD>
__device__ __forceinline__ cpx<double> twmul(cpx<double> a, double2 w) {
  double wy = FWD ? w.y : -w.y;
  return mk<double>(fma(a.x, w.x, -a.y * wy), fma(a.x, wy, a.y * w.x));
}
template <bool FWD>
__device__ __forceinline__ cpx<float> twmul(cpx<float> a, float4 w) {
  float hy = FWD ? w.y : -w.y;
  float ly = FWD ? w.w : -w.w;
  float tr = fmaf(a.x, w.z, -a.y * ly);
  float ti = fmaf(a.x, ly, a.y * w.z);
  return mk<float>(fmaf(a.x, w.x, fmaf(-a.y, hy, tr)), fmaf(a.x, hy, fmaf(a.y, w.x, ti)));
}

// exp(-2 pi i e / M) = (c, -s) as a twiddle of either type, from FP64 constants
template <class T>
__device__ __forceinline__ typename TwT<T>::type tw_const(double c, double s) {
  if constexpr (sizeof(T) == 4) {
    const float hx = (float)c, hy = (float)-s;
    return make_float4(hx, hy, (float)(c - (double)hx), (float)(-s - (double)hy));
  } else {
    return make_double2(c, -s);
  }
}

// ---------------------------------------------------------------------------
// small DFTs in registers
// ---------------------------------------------------------------------------
template <bool FWD, class T>
__device__ __forceinline__ void dft2(cpx<T>* v) {
  cpx<T> a = v[0], b = v[1];
  v[0] = add(a, b);
  v[1] = sub(a, b);
}

template <bool FWD, class T>
__device__ __forceinline__ void dft4(cpx<T>* v) {
  cpx<T> t0 = add(v[0], v[2]), t1 = sub(v[0], v[2]);
  cpx<T> t2 = add(v[1], v[3]), t3 = rot<FWD>(sub(v[1], v[3]));
  v[0] = add(t0, t2);
  v[2] = sub(t0, t2);
  v[1] = add(t1, t3);
  v[3] = sub(t1, t3);
}

template <bool FWD, class T>
__device__ __forceinline__ void dft8(cpx<T>* v) {
  const T h = (T)0.70710678118654752440;
  cpx<T> e[4] = {v[0], v[2], v[4], v[6]};
  cpx<T> o[4] = {v[1], v[3], v[5], v[7]};
  dft4<FWD>(e);
  dft4<FWD>(o);
  // o[k] *= W8^k  (W8 = exp(-i pi/4) forward, conjugate backward)
  cpx<T> o1, o3;
  if (FWD) {
    o1 = mk<T>((o[1].x + o[1].y) * h, (o[1].y - o[1].x) * h);
    o3 = mk<T>((o[3].y - o[3].x) * h, -(o[3].x + o[3].y) * h);
  } else {
    o1 = mk<T>((o[1].x - o[1].y) * h, (o[1].x + o[1].y) * h);
    o3 = mk<T>(-(o[3].x + o[3].y) * h, (o[3].x - o[3].y) * h);
  }
  cpx<T> o2 = rot<FWD>(o[2]);
  v[0] = add(e[0], o[0]);
  v[4] = sub(e[0], o[0]);
  v[1] = add(e[1], o1);
  v[5] = sub(e[1], o1);
  v[2] = add(e[2], o2);
  v[6] = sub(e[2], o2);
  v[3] = add(e[3], o3);
  v[7] = sub(e[3], o3);
}

// 16 points as 4 x 4: DFT4 over the stride-4 subsequences n1 + 4 n2, the
// twiddles W16^(n1 k1), DFT4 over n1; output in natural order
template <bool FWD, class T>
__device__ __forceinline__ void dft16(cpx<T>* v) {
  const T c1 = (T)0.92387953251128675613, s1 = (T)0.38268343236508977173;
  const T h = (T)0.70710678118654752440;
  cpx<T> y[4][4];
#pragma unroll
  for (int n1 = 0; n1 < 4; n1++) {
    cpx<T> t[4] = {v[n1], v[n1 + 4], v[n1 + 8], v[n1 + 12]};
    dft4<FWD>(t);
#pragma unroll
    for (int k1 = 0; k1 < 4; k1++) y[n1][k1] = t[k1];
  }
  // W16^m (forward exp(-2 pi i m / 16), backward its conjugate), m = n1 k1
  auto w = [&](cpx<T> a, int m) -> cpx<T> {
    T c, sn;
    switch (m) {
      case 1: c = c1; sn = s1; break;
      case 2: c = h; sn = h; break;
      case 3: c = s1; sn = c1; break;
      case 4: c = 0; sn = 1; break;
      case 6: c = -h; sn = h; break;
      default: c = -c1; sn = -s1; break;  // m = 9
    }
    const T sy = FWD ? -sn : sn;
    return mk<T>(a.x * c - a.y * sy, a.x * sy + a.y * c);
  };
  y[1][1] = w(y[1][1], 1);
  y[1][2] = w(y[1][2], 2);
  y[1][3] = w(y[1][3], 3);
  y[2][1] = w(y[2][1], 2);
  y[2][2] = rot<FWD>(y[2][2]);
  y[2][3] = w(y[2][3], 6);
  y[3][1] = w(y[3][1], 3);
  y[3][2] = w(y[3][2], 6);
  y[3][3] = w(y[3][3], 9);
#pragma unroll
  for (int k1 = 0; k1 < 4; k1++) {
    cpx<T> t[4] = {y[0][k1], y[1][k1], y[2][k1], y[3][k1]};
    dft4<FWD>(t);
#pragma unroll
    for (int k2 = 0; k2 < 4; k2++) v[k1 + 4 * k2] = t[k2];
  }
}

template <bool FWD, class T>
__device__ __forceinline__ void dft3(cpx<T>* v) {
  const T c3 = (T)0.86602540378443864676;
  cpx<T> s = add(v[1], v[2]);
  cpx<T> d = scl(rot<FWD>(sub(v[1], v[2])), c3);
  cpx<T> m = sub(v[0], scl(s, (T)0.5));
  v[0] = add(v[0], s);
  v[1] = add(m, d);
  v[2] = sub(m, d);
}

template <bool FWD, class T>
__device__ __forceinline__ void dft5(cpx<T>* v) {
  const T c1 = (T)0.30901699437494742410, c2 = (T)-0.80901699437494742410;
  const T s1 = (T)0.95105651629515357212, s2 = (T)0.58778525229247312917;
  cpx<T> s14 = add(v[1], v[4]), d14 = sub(v[1], v[4]);
  cpx<T> s23 = add(v[2], v[3]), d23 = sub(v[2], v[3]);
  cpx<T> a0 = v[0];
  cpx<T> m1 = mk<T>(a0.x + c1 * s14.x + c2 * s23.x, a0.y + c1 * s14.y + c2 * s23.y);
  cpx<T> m2 = mk<T>(a0.x + c2 * s14.x + c1 * s23.x, a0.y + c2 * s14.y + c1 * s23.y);
  cpx<T> n1 = rot<FWD>(mk<T>(s1 * d14.x + s2 * d23.x, s1 * d14.y + s2 * d23.y));
  cpx<T> n2 = rot<FWD>(mk<T>(s2 * d14.x - s1 * d23.x, s2 * d14.y - s1 * d23.y));
  v[0] = add(a0, add(s14, s23));
  v[1] = add(m1, n1);
  v[4] = sub(m1, n1);
  v[2] = add(m2, n2);
  v[3] = sub(m2, n2);
}

// odd-prime DFT (of 7) by the pairwise (a_p +- a_{P-p}) form; tables hold
// cos(2 pi j/P), sin(2 pi j/P) for j = 1..(P-1)/2.
template <int P> struct PrimeTab;
template <> struct PrimeTab<7> {
  static constexpr double c[4] = {1.0, 0.6234898018587336, -0.22252093395631434, -0.900968867902419};
  static constexpr double s[4] = {0.0, 0.7818314824680298, 0.9749279121818236, 0.43388373911755823};
};
template <int P, bool FWD, class T>
__device__ __forceinline__ void dftp(cpx<T>* v) {
  constexpr int H = (P - 1) / 2;
  cpx<T> sp[H + 1], dp[H + 1];
#pragma unroll
  for (int p = 1; p <= H; p++) {
    sp[p] = add(v[p], v[P - p]);
    dp[p] = sub(v[p], v[P - p]);
  }
  cpx<T> a0 = v[0];
  cpx<T> y0 = a0;
#pragma unroll
  for (int p = 1; p <= H; p++) y0 = add(y0, sp[p]);
#pragma unroll
  for (int q = 1; q <= H; q++) {
    cpx<T> m = a0, n = mk<T>(0, 0);
#pragma unroll
    for (int p = 1; p <= H; p++) {
      const int j = (p * q) % P;
      const T c = (T)PrimeTab<P>::c[j <= H ? j : P - j];
      const T s = j <= H ? (T)PrimeTab<P>::s[j] : -(T)PrimeTab<P>::s[P - j];
      m = mk<T>(m.x + c * sp[p].x, m.y + c * sp[p].y);
      n = mk<T>(n.x + s * dp[p].x, n.y + s * dp[p].y);
    }
    n = rot<FWD>(n);
    v[q] = add(m, n);
    v[P - q] = sub(m, n);
  }
  v[0] = y0;
}

template <int R, bool FWD, class T>
__device__ __forceinline__ void dft(cpx<T>* v);

// 9 points as 3 x 3, twiddles W9^(n1 k1), in FP32 hi + lo as the stage twiddles
// that they stand in for: with W9 rounded to FP32, 81, 729 and 243 points had
// errors 5 to 7% above 3 x 3 x .. stages.
template <bool FWD, class T>
__device__ __forceinline__ void dft9(cpx<T>* v) {
  constexpr double C[5] = {1.0, 0.76604444311897803520, 0.17364817766693034885, -0.5, -0.93969262078590838405};
  constexpr double S[5] = {0.0, 0.64278760968653932632, 0.98480775301220805937, 0.86602540378443864676,
                           0.34202014332566873304};
  cpx<T> y[3][3];
#pragma unroll
  for (int n1 = 0; n1 < 3; n1++) {
    cpx<T> t[3] = {v[n1], v[n1 + 3], v[n1 + 6]};
    dft3<FWD>(t);
#pragma unroll
    for (int k1 = 0; k1 < 3; k1++) {
      const int m = n1 * k1;
      y[n1][k1] = m == 0 ? t[k1] : twmul<FWD>(t[k1], tw_const<T>(C[m], S[m]));
    }
  }
#pragma unroll
  for (int k1 = 0; k1 < 3; k1++) {
    cpx<T> t[3] = {y[0][k1], y[1][k1], y[2][k1]};
    dft3<FWD>(t);
#pragma unroll
    for (int k2 = 0; k2 < 3; k2++) v[k1 + 3 * k2] = t[k2];
  }
}

// N1 x N2 points, N1 and N2 coprime, without twiddles (the prime-factor
// algorithm of Good and Thomas: the input index runs over N2 n1 + N1 n2, the
// output index is recovered by the Chinese remainder theorem)
constexpr int inv_mod(int a, int m) {
  for (int x = 1; x < m; x++)
    if (a % m * x % m == 1) return x;
  return 0;
}
template <int N1, int N2, bool FWD, class T>
__device__ __forceinline__ void dft_pfa(cpx<T>* v) {
  constexpr int N = N1 * N2;
  constexpr int E1 = N2 * inv_mod(N2, N1), E2 = N1 * inv_mod(N1, N2);
  cpx<T> y[N1][N2];
#pragma unroll
  for (int n1 = 0; n1 < N1; n1++) {
#pragma unroll
    for (int n2 = 0; n2 < N2; n2++) y[n1][n2] = v[(N2 * n1 + N1 * n2) % N];
    dft<N2, FWD>(y[n1]);
  }
#pragma unroll
  for (int k2 = 0; k2 < N2; k2++) {
    cpx<T> t[N1];
#pragma unroll
    for (int n1 = 0; n1 < N1; n1++) t[n1] = y[n1][k2];
    dft<N1, FWD>(t);
#pragma unroll
    for (int k1 = 0; k1 < N1; k1++) v[(E1 * k1 + E2 * k2) % N] = t[k1];
  }
}

template <int R, bool FWD, class T>
__device__ __forceinline__ void dft(cpx<T>* v) {
  if constexpr (R == 1) return;
  else if constexpr (R == 2) dft2<FWD>(v);
  else if constexpr (R == 3) dft3<FWD>(v);
  else if constexpr (R == 4) dft4<FWD>(v);
  else if constexpr (R == 5) dft5<FWD>(v);
  else if constexpr (R == 6) dft_pfa<2, 3, FWD>(v);
  else if constexpr (R == 8) dft8<FWD>(v);
  else if constexpr (R == 9) dft9<FWD>(v);
  else if constexpr (R == 10) dft_pfa<2, 5, FWD>(v);
  else if constexpr (R == 12) dft_pfa<4, 3, FWD>(v);
  else if constexpr (R == 16) dft16<FWD>(v);
  else dftp<R, FWD>(v);
}

// ---------------------------------------------------------------------------
// exact small-integer division: q = (x * m) >> 32 with m = ceil(2^32 / d),
// valid for x, d < 2^16 (all in-workgroup indices are below 2^16).
// ---------------------------------------------------------------------------
struct FDiv {
  uint64_t m;
  int d;
};
__device__ __forceinline__ int fdiv(int x, const FDiv& f) {
  return (int)(((uint64_t)(uint32_t)x * f.m) >> 32);
}

// ---------------------------------------------------------------------------
// length descriptor (built by the host)
// ---------------------------------------------------------------------------
constexpr int kMaxStages = 24;
struct LenDesc {
  int n;
  int nst;                 // number of stages
  int radix[kMaxStages];   // radix of each stage
  int ns[kMaxStages];      // product of the radices of earlier stages
  int twoff[kMaxStages];   // offset of each stage's twiddles in the table
  int twcount;             // total entries
};

}  // namespace p3amd
