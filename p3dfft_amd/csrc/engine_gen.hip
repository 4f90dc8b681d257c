// engine_gen.hip -- gfx950 kernels for transform lengths whose radix schedule
// is a run-time value.
//
// A length n = R_0 R_1 ... R_{S-1} (radices up to 10, the composite ones as
// prime-factor butterflies in registers) is run in place over an LDS tile of
// B sequences.  Position p of the tile is written in mixed radix with R_0 the
// fastest digit; stage s combines the R_s values a stride Ns = R_0 ... R_{s-1}
// apart:
//   forward order (decimation in time): twiddle W_{Ns R}^{k r}, then the
//     butterfly, stages 0 .. S-1; input index e sits at the digit-reversed
//     position, the result is in natural order;
//   reverse order (decimation in frequency): butterfly, then the twiddle,
//     stages S-1 .. 0; natural order in, digit-reversed out.
// Both use one twiddle table.  A butterfly writes the positions it read, so
// a stage needs one barrier, one butterfly's registers and one tile, and the
// number of butterflies per thread is a run-time loop.  The digit reversal
// costs nothing on the side that addresses memory by rows: stage 0 there reads
// (or writes) global memory itself, one 128-byte row segment per value, and
// the reversal is one division per butterfly.
//
// 11 and 13 points run as such a butterfly too, by the symmetric pairs
// v_i +- v_{R-i} (half the multiplications of the direct sum).  A larger prime
// radix runs as a stage over LDS by those pairs, its outputs held in registers
// across a barrier.
//
// What bounds the passes: with 128-byte row segments they move each byte once
// per pass and run at 4-5.5 TB/s.  Counters of 200x300x250 FP32 / 1000x100x90
// FP64: 48-63% / 26-33% of the VALU slots busy (butterflies, compensated
// twiddles, run-time index arithmetic), the waves waiting for half of their
// cycles, 1-4% of them for LDS: the latencies of a tile's serial phases, and in
// FP32 the instruction issue beside them.
// Against a tile loaded to LDS, autosort stages and a direct sum for every
// prime: FP32 200x300x250 columns of 300 points 97 -> 30 us, of 250 102 -> 28,
// X r2c of 200 54 -> 28; FP64 1000x100x90 columns of 100 points 85 -> 26 us, of
// 90 100 -> 27, X r2c of 1000 80 -> 38.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <type_traits>

#include "engine_gen.hpp"

namespace p3amd {

typedef TwT<real_t>::type Tw;
static constexpr size_t kLdsMax = 160 * 1024;

struct GenStage {
  int R, Ns, tw;    // radix, product of the earlier radices, twiddle offset
  unsigned mNs;     // ceil(2^32 / Ns) (see gdiv)
  unsigned mR;
};
constexpr int kGenStages = 16;
// bytes before the twiddles that hold the columns' offsets (length-fastest views)
constexpr int kColTab = 32 * sizeof(unsigned long long);
struct GenDesc {
  int n, nst;
  GenStage st[kGenStages];
  int twcount;
};

// x / d for x, d < 2^16 with m = ceil(2^32 / d); d is uniform
__device__ __forceinline__ int gdiv(int x, unsigned m, int d) {
  return d == 1 ? x : (int)__umulhi((unsigned)x, m);
}

// address of position p: blocks of R_0 positions BP apart, the blocks R_0 BP +
// skew apart
struct GenTile {
  int BP, P0, skew, R0;
  unsigned mR0;
};

template <class F>
__device__ __forceinline__ void with_radix(int R, F f) {
#define P3_CASE(N) case N: f(std::integral_constant<int, N>{}); break;
  static_assert(kGenMaxRadix == 10, "one case per radix");
  switch (R) {
    P3_CASE(1) P3_CASE(2) P3_CASE(3) P3_CASE(4) P3_CASE(5) P3_CASE(6) P3_CASE(7) P3_CASE(8)
    P3_CASE(9) P3_CASE(10)
    default: break;
  }
#undef P3_CASE
}

// input index of stage 0's butterfly j (its R_0 values are n / R_0 apart)
__device__ __forceinline__ int gen_rev(const GenDesc& L, int j) {
  int acc = 0;
  for (int s = 1; s + 1 < L.nst; s++) {
    const int q = gdiv(j, L.st[s].mR, L.st[s].R);
    acc = acc * L.st[s].R + (j - q * L.st[s].R);
    j = q;
  }
  return L.nst > 1 ? acc * L.st[L.nst - 1].R + j : 0;
}

// the butterfly j whose input index is e (the inverse of gen_rev)
__device__ __forceinline__ int gen_unrev(const GenDesc& L, int e) {
  int acc = 0;
  for (int s = L.nst - 1; s > 1; s--) {
    const int q = gdiv(e, L.st[s].mR, L.st[s].R);
    acc = acc * L.st[s].R + (e - q * L.st[s].R);
    e = q;
  }
  return L.nst > 1 ? acc * L.st[1].R + e : 0;
}

// address of the first value of stage s's butterfly (block g, offset k) and
// the stride of its values
__device__ __forceinline__ int gen_base(const GenTile& t, const GenStage& st, int g, int k, int SP) {
  int a = g * st.R * SP + k * t.BP;
  if (t.skew) a += gdiv(k, t.mR0, t.R0) * t.skew;
  return a;
}
__device__ __forceinline__ int gen_stride(const GenTile& t, const GenStage& st) {
  return gdiv(st.Ns, t.mR0, t.R0) * t.P0;
}

// a butterfly of 11 or 13 points in place, its positions SP apart: the sums and
// differences of the symmetric pairs in registers, each pair of outputs written
// as soon as it is summed, so 13 FP64 points hold 13 values and not 26.  One
// barrier and 2 R LDS accesses a butterfly: 25600 columns of 143 points 35 us in
// FP64 and 28 us in FP32 (3.4 and 2.1 TB/s), 4096 of 2197 points 95 and 60 us; with
// the pairs' sums over LDS (gen_prime) 90 and 47, 170 and 142 us, slower than a
// direct radix 11 or 13 of autosort stages (77 and 43, 240 and 115 us).
template <int R>
struct PrimeConst;
template <>
struct PrimeConst<11> {
  static constexpr double c[6] = {1.0, 0.84125353283118116886, 0.41541501300188642553, -0.14231483827328514044,
                                  -0.65486073394528506406, -0.95949297361449738989};
  static constexpr double s[6] = {0.0, 0.54064081745559758211, 0.90963199535451837141, 0.98982144188093273238,
                                  0.75574957435425828377, 0.28173255684142969771};
};
template <>
struct PrimeConst<13> {
  static constexpr double c[7] = {1.0, 0.88545602565320989590, 0.56806474673115580251, 0.12053668025532305335,
                                  -0.35460488704253562597, -0.74851074817110109863, -0.97094181742605202716};
  static constexpr double s[7] = {0.0, 0.46472317204376854566, 0.82298386589365639458, 0.99270887409805399280,
                                  0.93501624268541482344, 0.66312265824079520238, 0.23931566428755776715};
};

// a + x * k, the constant hi + lo in FP32
template <class T>
__device__ __forceinline__ cpx<T> fma_const(cpx<T> x, double k, cpx<T> a) {
  if constexpr (sizeof(T) == 4) {
    const float h = (float)k, l = (float)(k - (double)h);
    return mk<T>(fmaf(x.x, h, fmaf(x.x, l, a.x)), fmaf(x.y, h, fmaf(x.y, l, a.y)));
  } else {
    return mk<T>(fma(x.x, k, a.x), fma(x.y, k, a.y));
  }
}

template <class T, bool FWD, bool DIF, int R>
__device__ __forceinline__ void gen_reg_prime(cpx<T>* p, int SP, const typename TwT<T>::type* w) {
  constexpr int H = (R - 1) / 2;
  const cpx<T> v0 = p[0];
  cpx<T> s[H], d[H], y0 = v0;
#pragma unroll
  for (int i = 0; i < H; i++) {
    cpx<T> u = p[(i + 1) * SP], v = p[(R - 1 - i) * SP];
    if constexpr (!DIF) {
      u = twmul<FWD>(u, w[i]);
      v = twmul<FWD>(v, w[R - 2 - i]);
    }
    s[i] = add(u, v);
    d[i] = sub(u, v);
    y0 = add(y0, s[i]);
  }
  p[0] = y0;
#pragma unroll
  for (int q = 1; q <= H; q++) {
    cpx<T> c = v0, e = mk<T>(0, 0);
#pragma unroll
    for (int i = 0; i < H; i++) {
      const int m = (i + 1) * q % R;
      c = fma_const(s[i], PrimeConst<R>::c[m <= H ? m : R - m], c);
      e = fma_const(d[i], m <= H ? PrimeConst<R>::s[m] : -PrimeConst<R>::s[R - m], e);
    }
    e = rot<FWD>(e);
    cpx<T> a = add(c, e), b = sub(c, e);
    if constexpr (DIF) {
      a = twmul<FWD>(a, w[q - 1]);
      b = twmul<FWD>(b, w[R - 1 - q]);
    }
    p[q * SP] = a;
    p[(R - q) * SP] = b;
  }
}

// a stage with a larger prime radix: outputs by symmetric pairs over LDS
constexpr int kPrimeItems = 8;
template <class T, bool FWD, bool DIF>
__device__ __forceinline__ void gen_prime(cpx<T>* lds, const GenDesc& L, const GenStage& st, const GenTile& t, int B,
                                          unsigned mB, const typename TwT<T>::type* tw) {
  typedef typename TwT<T>::type TwL;
  const int NT = blockDim.x, R = st.R, H = (R - 1) / 2;
  const int nj = gdiv(L.n, st.mR, R), nb = B * nj, SP = gen_stride(t, st);
  const unsigned mb = nb > 1 ? (unsigned)((0x100000000ull + nb - 1) / nb) : 0;
  // v_i, v_{R-i} -> their sum and difference, in place
  for (int it = threadIdx.x; it < nb * H; it += NT) {
    const int i0 = gdiv(it, mb, nb), w = it - i0 * nb, i = i0 + 1;
    const int j = gdiv(w, mB, B), b = w - j * B;
    const int g = gdiv(j, st.mNs, st.Ns), k = j - g * st.Ns;
    const int p = gen_base(t, st, g, k, SP) + b;
    cpx<T> u = lds[p + i * SP], v = lds[p + (R - i) * SP];
    if constexpr (!DIF) {
      const TwL* q = tw + st.tw + k * (R - 1);
      u = twmul<FWD>(u, q[i - 1]);
      v = twmul<FWD>(v, q[R - i - 1]);
    }
    lds[p + i * SP] = add(u, v);
    lds[p + (R - i) * SP] = sub(u, v);
  }
  __syncthreads();
  const TwL* wr = tw + st.tw + st.Ns * (R - 1);  // W_R^j
  cpx<T> ya[kPrimeItems], yb[kPrimeItems];
#pragma unroll
  for (int m = 0; m < kPrimeItems; m++) {
    const int it = threadIdx.x + m * NT;
    if (it < nb * (H + 1)) {
      const int q = gdiv(it, mb, nb), w = it - q * nb;
      const int j = gdiv(w, mB, B), b = w - j * B;
      const int g = gdiv(j, st.mNs, st.Ns), k = j - g * st.Ns;
      const int p = gen_base(t, st, g, k, SP) + b;
      cpx<T> c = lds[p], d = mk<T>(0, 0);
      int e = 0;
      for (int i = 1; i <= H; i++) {
        e += q;
        if (e >= R) e -= R;
        // cos and sin of 2 pi i q / R times the pair's sum and difference
        const TwL x = wr[e];
        const cpx<T> s = lds[p + i * SP], f = lds[p + (R - i) * SP];
        if constexpr (sizeof(T) == 4) {
          c.x = fmaf(s.x, x.x, fmaf(s.x, x.z, c.x));
          c.y = fmaf(s.y, x.x, fmaf(s.y, x.z, c.y));
          d.x = fmaf(f.x, -x.y, fmaf(f.x, -x.w, d.x));
          d.y = fmaf(f.y, -x.y, fmaf(f.y, -x.w, d.y));
        } else {
          c.x = fma(s.x, x.x, c.x);
          c.y = fma(s.y, x.x, c.y);
          d.x = fma(f.x, -x.y, d.x);
          d.y = fma(f.y, -x.y, d.y);
        }
      }
      d = rot<FWD>(d);
      ya[m] = add(c, d);
      yb[m] = sub(c, d);
      if constexpr (DIF) {
        const TwL* w2 = tw + st.tw + k * (R - 1);
        if (q > 0) {
          ya[m] = twmul<FWD>(ya[m], w2[q - 1]);
          yb[m] = twmul<FWD>(yb[m], w2[R - q - 1]);
        }
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int m = 0; m < kPrimeItems; m++) {
    const int it = threadIdx.x + m * NT;
    if (it < nb * (H + 1)) {
      const int q = gdiv(it, mb, nb), w = it - q * nb;
      const int j = gdiv(w, mB, B), b = w - j * B;
      const int g = gdiv(j, st.mNs, st.Ns), k = j - g * st.Ns;
      const int p = gen_base(t, st, g, k, SP) + b;
      lds[p + q * SP] = ya[m];
      if (q > 0) lds[p + (R - q) * SP] = yb[m];
    }
  }
  __syncthreads();
}

// The prime stages of a schedule: none, over LDS only (all of them above
// kGenRegPrime), or some in registers.  Each is compiled apart: the registers of a
// stage over LDS (FP32 X kernels 96-109 against 80) cost every stage a wave per
// SIMD (200-point FP32 X r2c of a 200x300x250 box 39.7 -> 28.6 us without,
// 1000-point FP64 of 1000x100x90 45.0 -> 41.6), and 11 and 13 points in registers
// beside it 8 to 48 bytes of scratch in FP64 (X r2c / c2r of 2^22 points in rows
// of 57 31.7 / 29.7 us with, 28.2 / 27.1 without, c2r in rows of 1360 34.0
// and 28.0; FP32, 2^23 points in columns of 127, 101 and 94).
enum { kPrimeNone = 0, kPrimeLds = 1, kPrimeAny = 2 };

// An in-place stage over the tile.  b: this thread's sequence, jt, js: its
// first butterfly and their stride
template <class T, bool FWD, bool DIF, int PM>
__device__ __forceinline__ void gen_mid(cpx<T>* lds, const GenDesc& L, int s, const GenTile& t, int B, unsigned mB,
                                        int b, int jt, int js, const typename TwT<T>::type* tw) {
  const GenStage st = L.st[s];
  if constexpr (PM != kPrimeNone) {
    if (st.R > kGenRegPrime) {
      gen_prime<T, FWD, DIF>(lds, L, st, t, B, mB, tw);
      return;
    }
  }
  const int nj = gdiv(L.n, st.mR, st.R), SP = gen_stride(t, st);
  if constexpr (PM == kPrimeAny) {
    if (st.R > kGenMaxRadix) {
      for (int j = jt; j < nj; j += js) {
        const int g = gdiv(j, st.mNs, st.Ns), k = j - g * st.Ns;
        cpx<T>* p = lds + gen_base(t, st, g, k, SP) + b;
        const typename TwT<T>::type* w = tw + st.tw + k * (st.R - 1);
        if (st.R == 11) gen_reg_prime<T, FWD, DIF, 11>(p, SP, w);
        else gen_reg_prime<T, FWD, DIF, 13>(p, SP, w);
      }
      __syncthreads();
      return;
    }
  }
  with_radix(st.R, [&](auto rc) {
    constexpr int R = decltype(rc)::value;
    for (int j = jt; j < nj; j += js) {
      const int g = gdiv(j, st.mNs, st.Ns), k = j - g * st.Ns;
      cpx<T>* p = lds + gen_base(t, st, g, k, SP) + b;
      cpx<T> v[R];
#pragma unroll
      for (int r = 0; r < R; r++) v[r] = p[r * SP];
      const typename TwT<T>::type* w = tw + st.tw + k * (R - 1);
      if constexpr (!DIF) {
#pragma unroll
        for (int r = 1; r < R; r++) v[r] = twmul<FWD>(v[r], w[r - 1]);
      }
      dft<R, FWD>(v);
      if constexpr (DIF) {
#pragma unroll
        for (int r = 1; r < R; r++) v[r] = twmul<FWD>(v[r], w[r - 1]);
      }
#pragma unroll
      for (int r = 0; r < R; r++) p[r * SP] = v[r];
    }
  });
  __syncthreads();
}

extern __shared__ __align__(16) unsigned char gen_smem[];

// the twiddle table, copied into LDS behind the tile where it fits (TL;
// complete at the next barrier).  A compile-time choice: with one pointer for
// either place the stages read it through the flat path (300-point FP32
// columns of a 200x300x250 box 31.6 us so, 29.8 us now).
template <class T, bool TL>
__device__ __forceinline__ const typename TwT<T>::type* gen_twiddles(const void* tw, int off, int count) {
  typedef typename TwT<T>::type TwL;
  const TwL* g = (const TwL*)tw;
  if constexpr (TL) {
    TwL* l = (TwL*)(gen_smem + off);
    for (int i = threadIdx.x; i < count; i += blockDim.x) l[i] = g[i];
    return l;
  } else {
    return g;
  }
}

// workgroup id -> tile: each XCD (id mod 8) owns a contiguous range
__device__ __forceinline__ int gen_tile_of(int rev, int xcd) {
  const int n = (int)gridDim.x, bid = (int)blockIdx.x;
  int t = bid;
  if (xcd) {
    const int q = n >> 3, rm = n & 7, x = bid & 7;
    t = x * q + (x < rm ? x : rm) + (bid >> 3);
  }
  return rev ? n - 1 - t : t;
}

// ---------------------------------------------------------------------------
// columns
// ---------------------------------------------------------------------------
struct GColArgs {
  const void* in;
  void* out;
  long long si_in, sl_in, so_in, si_out, sl_out, so_out;
  long long ncol;
  int n_inner;
  int lB;             // log2 of the columns per tile
  int kind, rows;     // ColKind, logical rows of a column
  int nld, ld_lo, ld_hi, ld_shift, nst, st_lo, st_shift;
  FDiv dld, dst;      // length-fastest sides: divide by the rows loaded / stored
  GenTile t;
  GenDesc L;
  const void* tw;
  int tw_lds, tw_off;
  int rev, xcd;
};

// input row of FFT row e (-1: zero); neg: with its sign changed
__device__ __forceinline__ int gen_src(const GColArgs& a, int e, bool& neg) {
  neg = false;
  int i = e;
  if (a.kind == COL_DCT1) {
    if (e >= a.rows) i = a.L.n - e;
  } else if (a.kind == COL_DST1) {
    if (e == 0 || e == a.rows + 1) return -1;
    neg = e > a.rows;
    i = neg ? a.L.n - e - 1 : e - 1;
  }
  if (i >= a.nld) return -1;
  return i < a.ld_lo ? i : (i >= a.ld_hi ? i - a.ld_shift : -1);
}
// output row of FFT row p (-1: not stored)
__device__ __forceinline__ int gen_dst(const GColArgs& a, int p) {
  const int i = a.kind == COL_DST1 ? p - 1 : p;
  const int e = i < a.st_lo ? i : (i >= a.st_lo + a.st_shift ? i - a.st_shift : -1);
  return e < a.nst ? e : -1;
}
template <class T>
__device__ __forceinline__ cpx<T> gen_out(const GColArgs& a, cpx<T> v) {
  return a.kind == COL_DST1 ? mk<T>(-v.y, v.x) : v;
}

// MAP: pruned rows, DCT-I / DST-I extensions.  LF: 0 rows on both sides, 1 the
// input is length-fastest (decimation in frequency), 2 the output is.  Off: the
// type of the byte offsets from the tile's first column.  Rows without maps have
// a form of either width, so that a view of 4 GiB gives the bits of a smaller one
// (the form with maps contracts its products differently) and is not slowed by
// the maps' arithmetic.
template <class T, bool FWD, bool MAP, int LF, class Off, bool TL, int PM>
__global__ __launch_bounds__(1024) void k_gcol(GColArgs a) {
  typedef cpx<T> C;
  constexpr long long E = sizeof(C);
  C* lds = (C*)gen_smem;
  const auto* tw = gen_twiddles<T, TL>(a.tw, a.tw_off, a.L.twcount);
  const int B = 1 << a.lB, NT = blockDim.x, S = a.L.nst;
  const unsigned mB = a.lB ? 1u << (32 - a.lB) : 0u;
  const int b = threadIdx.x & (B - 1), jt = threadIdx.x >> a.lB, js = NT >> a.lB;
  const long long c0 = (long long)gen_tile_of(a.rev, a.xcd) * B;
  const int nb = (int)(a.ncol - c0 < B ? a.ncol - c0 : B);
  const unsigned n_in = (unsigned)a.n_inner;
  const unsigned o0 = (unsigned)c0 / n_in, i0 = (unsigned)c0 - o0 * n_in;
  const char* in = (const char*)a.in + ((long long)o0 * a.so_in + (long long)i0 * a.si_in) * E;
  char* out = (char*)a.out + ((long long)o0 * a.so_out + (long long)i0 * a.si_out) * E;
  // columns past the last one repeat it and are not stored
  const unsigned c = (unsigned)c0 + (b < nb ? b : nb - 1);
  const unsigned o = c / n_in, i = c - o * n_in;
  const Off lin = (Off)((((long long)o - o0) * a.so_in + ((long long)i - i0) * a.si_in) * E);
  const Off lout = (Off)((((long long)o - o0) * a.so_out + ((long long)i - i0) * a.si_out) * E);
  const Off sin = (Off)(a.sl_in * E), sout = (Off)(a.sl_out * E);
  const bool valid = b < nb;
  const GenStage s0 = a.L.st[0];
  const int n0 = gdiv(a.L.n, s0.mR, s0.R);
  // values of a finished butterfly: FFT rows p0 + r * dp
  auto store = [&](auto rc, C* v, int p0, int dp) {
    constexpr int R = decltype(rc)::value;
    if (!valid) return;
    if constexpr (MAP) {
#pragma unroll
      for (int r = 0; r < R; r++) {
        const int e = gen_dst(a, p0 + r * dp);
        if (e >= 0) *(C*)(out + (lout + (Off)e * sout)) = gen_out(a, v[r]);
      }
    } else {
      Off q = lout + (Off)p0 * sout;
      const Off dq = (Off)dp * sout;
#pragma unroll
      for (int r = 0; r < R; r++, q += dq) *(C*)(out + q) = v[r];
    }
  };
  if constexpr (LF == 1) {
    // natural order into the tile, the lanes along the length
    const int m = a.L.n;
    unsigned long long* colb = (unsigned long long*)(gen_smem + a.tw_off - kColTab);
    if (threadIdx.x < B) colb[threadIdx.x] = (unsigned long long)lin;
    __syncthreads();
    for (int q = threadIdx.x; q < B * m; q += NT) {
      const int bb = fdiv(q, a.dld), e = q - bb * m;
      bool neg;
      const int src = gen_src(a, e, neg);
      C v = mk<T>(0, 0);
      if (src >= 0) v = *(const C*)(in + (colb[bb] + (unsigned long long)src * (unsigned long long)sin));
      lds[e * a.t.BP + bb] = neg ? mk<T>(-v.x, -v.y) : v;
    }
    __syncthreads();
    for (int s = S - 1; s > 0; s--) gen_mid<T, FWD, true, PM>(lds, a.L, s, a.t, B, mB, b, jt, js, tw);
    with_radix(s0.R, [&](auto rc) {
      constexpr int R = decltype(rc)::value;
      for (int j = jt; j < n0; j += js) {
        C v[R];
        const C* p = lds + j * a.t.P0 + b;
#pragma unroll
        for (int r = 0; r < R; r++) v[r] = p[r * a.t.BP];
        dft<R, FWD>(v);
        store(rc, v, gen_rev(a.L, j), n0);
      }
    });
    return;
  }
  with_radix(s0.R, [&](auto rc) {
    constexpr int R = decltype(rc)::value;
    for (int j = jt; j < n0; j += js) {
      const int e0 = gen_rev(a.L, j);
      C v[R];
      if constexpr (MAP) {
#pragma unroll
        for (int r = 0; r < R; r++) {
          bool neg;
          const int src = gen_src(a, e0 + r * n0, neg);
          // a row that is zero reads the column's first row instead, so no
          // load sits under a branch
          const C u = *(const C*)(in + (lin + (Off)(src >= 0 ? src : 0) * sin));
          v[r].x = src >= 0 ? (neg ? -u.x : u.x) : (T)0;
          v[r].y = src >= 0 ? (neg ? -u.y : u.y) : (T)0;
        }
      } else {
        Off q = lin + (Off)e0 * sin;
        const Off dq = (Off)n0 * sin;
#pragma unroll
        for (int r = 0; r < R; r++, q += dq) v[r] = *(const C*)(in + q);
      }
      dft<R, FWD>(v);
      if (S == 1 && LF == 0) {
        store(rc, v, 0, 1);
      } else {
        C* p = lds + j * a.t.P0 + b;
#pragma unroll
        for (int r = 0; r < R; r++) p[r * a.t.BP] = v[r];
      }
    }
  });
  if (S == 1 && LF == 0) return;
  __syncthreads();
  const int last = LF == 2 ? S : S - 1;
  for (int s = 1; s < last; s++) gen_mid<T, FWD, false, PM>(lds, a.L, s, a.t, B, mB, b, jt, js, tw);
  if constexpr (LF == 2) {
    unsigned long long* colb = (unsigned long long*)(gen_smem + a.tw_off - kColTab);
    if (threadIdx.x < B) colb[threadIdx.x] = (unsigned long long)lout;
    __syncthreads();
    for (int q = threadIdx.x; q < nb * a.nst; q += NT) {
      const int bb = fdiv(q, a.dst), e = q - bb * a.nst;
      const int p = (e < a.st_lo ? e : e + a.st_shift) + (a.kind == COL_DST1 ? 1 : 0);
      *(C*)(out + (colb[bb] + (unsigned long long)e * (unsigned long long)sout)) = gen_out(a, lds[p * a.t.BP + bb]);
    }
  } else {
    const GenStage st = a.L.st[S - 1];
    const int SP = gen_stride(a.t, st);
    with_radix(st.R, [&](auto rc) {
      constexpr int R = decltype(rc)::value;
      for (int j = jt; j < st.Ns; j += js) {
        C v[R];
        const C* p = lds + gen_base(a.t, st, 0, j, SP) + b;
#pragma unroll
        for (int r = 0; r < R; r++) v[r] = p[r * SP];
        const auto* w = tw + st.tw + j * (R - 1);
#pragma unroll
        for (int r = 1; r < R; r++) v[r] = twmul<FWD>(v[r], w[r - 1]);
        dft<R, FWD>(v);
        store(rc, v, j, st.Ns);
      }
    });
  }
}

// rows moved without a transform (row maps and the length-fastest layout),
// through an LDS tile so that both sides are read and written along their
// contiguous index
template <class T>
__global__ __launch_bounds__(1024) void k_gcopy(GColArgs a) {
  typedef cpx<T> C;
  C* lds = (C*)gen_smem;
  const int B = 1 << a.lB, NT = blockDim.x;
  const long long c0 = (long long)gen_tile_of(a.rev, a.xcd) * B;
  const int nb = (int)(a.ncol - c0 < B ? a.ncol - c0 : B);
  const bool lf_in = a.sl_in == 1 && a.si_in != 1, lf_out = a.sl_out == 1 && a.si_out != 1;
  const unsigned n_in = (unsigned)a.n_inner;
  auto col = [&](int b, long long si, long long so) {
    const unsigned c = (unsigned)c0 + b, o = c / n_in, i = c - o * n_in;
    return (long long)o * so + (long long)i * si;
  };
  for (int q = threadIdx.x; q < B * a.nld; q += NT) {
    int b, e;
    if (lf_in) { b = fdiv(q, a.dld); e = q - b * a.nld; }
    else { e = q >> a.lB; b = q & (B - 1); }
    const int src = e < a.ld_lo ? e : (e >= a.ld_hi ? e - a.ld_shift : -1);
    C v = mk<T>(0, 0);
    if (b < nb && src >= 0) v = ((const C*)a.in)[col(b, a.si_in, a.so_in) + (long long)src * a.sl_in];
    lds[e * a.t.BP + b] = v;
  }
  __syncthreads();
  for (int q = threadIdx.x; q < B * a.nst; q += NT) {
    int b, e;
    if (lf_out) { b = fdiv(q, a.dst); e = q - b * a.nst; }
    else { e = q >> a.lB; b = q & (B - 1); }
    if (b < nb) {
      const int p = e < a.st_lo ? e : e + a.st_shift;
      ((C*)a.out)[col(b, a.si_out, a.so_out) + (long long)e * a.sl_out] = lds[p * a.t.BP + b];
    }
  }
}

// ---------------------------------------------------------------------------
// rows along X: two real rows as one complex row (x_a + i x_b)
// ---------------------------------------------------------------------------
struct GXArgs {
  const void* in;
  void* out;
  long long nrows, si_row, so_row;
  int nk;         // r2c: kept modes; c2r: valid input modes
  int lB;         // log2 of the row pairs per tile
  FDiv dnk, dn0;  // divide by the modes, by n / R_0 (c2r of one stage: by n)
  GenTile t;
  GenDesc L;
  const void* tw;
  int tw_lds, tw_off;
  int rev;
};

// r2c: stage 0 reads the rows (lanes along the row), in-place stages, and the
// two half spectra separated from the natural-order result as they are stored.
// Bound by the latencies of a tile's serial phases (see the top of the file).
// Lanes along one row throughout: 16 lanes along each of 4 rows met fewer LDS
// conflicts, but their short runs cost more on the memory side: FP64 200x300x250
// r2c / c2r 51 / 70 -> 46 / 49 us (5.0 TB/s), FP32 30 / 34 -> 28 / 31 us.
template <class T, bool TL, int PM>
__global__ __launch_bounds__(1024) void k_gx_r2c(GXArgs a) {
  typedef cpx<T> C;
  C* lds = (C*)gen_smem;
  const auto* tw = gen_twiddles<T, TL>(a.tw, a.tw_off, a.L.twcount);
  const int B = 1 << a.lB, NT = blockDim.x, S = a.L.nst, n = a.L.n;
  const long long pair0 = (long long)gen_tile_of(a.rev, 1) * B;
  const int nr = (int)(a.nrows - 2 * pair0 < 2 * B ? a.nrows - 2 * pair0 : 2 * B);
  const char* in = (const char*)a.in + 2 * pair0 * a.si_row * (long long)sizeof(T);
  const unsigned si = (unsigned)(a.si_row * sizeof(T));
  const GenStage s0 = a.L.st[0];
  const int n0 = gdiv(n, s0.mR, s0.R);
  with_radix(s0.R, [&](auto rc) {
    constexpr int R = decltype(rc)::value;
    for (int it = threadIdx.x; it < B * n0; it += NT) {
      const int b = fdiv(it, a.dn0), e0 = it - b * n0;
      const bool oka = 2 * b < nr, okb = 2 * b + 1 < nr;
      // rows past the last one read the tile's first row and are zeroed
      const char* pa = in + ((oka ? (unsigned)(2 * b) * si : 0u) + (unsigned)e0 * (unsigned)sizeof(T));
      const char* pb = in + ((okb ? (unsigned)(2 * b + 1) * si : 0u) + (unsigned)e0 * (unsigned)sizeof(T));
      C v[R];
      const unsigned d = (unsigned)n0 * (unsigned)sizeof(T);
#pragma unroll
      for (int r = 0; r < R; r++) {
        v[r].x = *(const T*)(pa + (unsigned)r * d);
        v[r].y = *(const T*)(pb + (unsigned)r * d);
      }
      if (!oka) {
#pragma unroll
        for (int r = 0; r < R; r++) v[r].x = (T)0;
      }
      if (!okb) {
#pragma unroll
        for (int r = 0; r < R; r++) v[r].y = (T)0;
      }
      dft<R, true>(v);
      C* p = lds + gen_unrev(a.L, e0) * a.t.P0 + b;
#pragma unroll
      for (int r = 0; r < R; r++) p[r * a.t.BP] = v[r];
    }
  });
  __syncthreads();
  const int b0 = threadIdx.x & (B - 1), jt = threadIdx.x >> a.lB, js = NT >> a.lB;
  const unsigned mB = a.lB ? 1u << (32 - a.lB) : 0u;
  for (int s = 1; s < S; s++)
    gen_mid<T, true, false, PM>(lds, a.L, s, a.t, B, mB, b0, jt, js, tw);
  char* out = (char*)a.out + 2 * pair0 * a.so_row * (long long)sizeof(C);
  const unsigned so = (unsigned)(a.so_row * sizeof(C));
  const T h = (T)0.5;
  for (int q = threadIdx.x; q < B * a.nk; q += NT) {
    const int b = fdiv(q, a.dnk), k = q - b * a.nk;
    const C zk = lds[k * a.t.BP + b], zn = lds[(k == 0 ? 0 : n - k) * a.t.BP + b];
    const unsigned off = (unsigned)(2 * b) * so + (unsigned)k * (unsigned)sizeof(C);
    if (2 * b < nr) *(C*)(out + off) = mk<T>((zk.x + zn.x) * h, (zk.y - zn.y) * h);
    if (2 * b + 1 < nr) *(C*)(out + off + so) = mk<T>((zk.y + zn.y) * h, (zn.x - zk.x) * h);
  }
}

// c2r: the mirror image: natural order in, decimation in frequency, stage 0
// stores the rows
template <class T, bool TL, int PM>
__global__ __launch_bounds__(1024) void k_gx_c2r(GXArgs a) {
  typedef cpx<T> C;
  C* lds = (C*)gen_smem;
  const auto* tw = gen_twiddles<T, TL>(a.tw, a.tw_off, a.L.twcount);
  const int B = 1 << a.lB, NT = blockDim.x, S = a.L.nst, n = a.L.n, K = n / 2 + 1;
  const long long pair0 = (long long)gen_tile_of(a.rev, 1) * B;
  const int nr = (int)(a.nrows - 2 * pair0 < 2 * B ? a.nrows - 2 * pair0 : 2 * B);
  const char* in = (const char*)a.in + 2 * pair0 * a.si_row * (long long)sizeof(C);
  const unsigned si = (unsigned)(a.si_row * sizeof(C));
  // the loads of LU items in flight at a time before their LDS writes (200x300x250
  // FP32, without the prime stage: 37.4 -> 31.3 us)
  constexpr int LU = 4;
  for (int q0 = threadIdx.x; q0 < B * K; q0 += LU * NT) {
    C A[LU], Bv[LU];
    int bb[LU], kk[LU];
#pragma unroll
    for (int u = 0; u < LU; u++) {
      const int q = q0 + u * NT;
      const int b = bb[u] = q < B * K ? fdiv(q, a.dnk) : B;
      const int k = kk[u] = q - b * K;
      // items outside the tile or past the valid modes read its first element
      // and are zeroed, so no load sits under a branch
      const bool oka = q < B * K && k < a.nk && 2 * b < nr, okb = oka && 2 * b + 1 < nr;
      const unsigned off = (unsigned)(2 * b) * si + (unsigned)k * (unsigned)sizeof(C);
      A[u] = *(const C*)(in + (oka ? off : 0u));
      Bv[u] = *(const C*)(in + (okb ? off + si : 0u));
      if (!oka) A[u] = mk<T>(0, 0);
      if (!okb) Bv[u] = mk<T>(0, 0);
      // FFTW c2r: the imaginary parts of k = 0 and k = n/2 (n even) do not
      // contribute; there both forms are the same value
      if (k == 0 || 2 * k == n) { A[u].y = 0; Bv[u].y = 0; }
    }
#pragma unroll
    for (int u = 0; u < LU; u++) {
      if (bb[u] < B) {
        const int b = bb[u], k = kk[u];
        lds[k * a.t.BP + b] = mk<T>(A[u].x - Bv[u].y, A[u].y + Bv[u].x);
        lds[(k == 0 ? 0 : n - k) * a.t.BP + b] = mk<T>(A[u].x + Bv[u].y, Bv[u].x - A[u].y);
      }
    }
  }
  __syncthreads();
  const int b0 = threadIdx.x & (B - 1), jt = threadIdx.x >> a.lB, js = NT >> a.lB;
  const unsigned mB = a.lB ? 1u << (32 - a.lB) : 0u;
  for (int s = S - 1; s > 0; s--)
    gen_mid<T, false, true, PM>(lds, a.L, s, a.t, B, mB, b0, jt, js, tw);
  char* out = (char*)a.out + 2 * pair0 * a.so_row * (long long)sizeof(T);
  const unsigned so = (unsigned)(a.so_row * sizeof(T));
  const GenStage s0 = a.L.st[0];
  if (S == 1) {
    // rows of one butterfly: stored by it, the lanes would write a value each of
    // 64 rows at a time (2^23 points in rows of 8, FP32 45 us, through the tile
    // 15 us; of 7 41 and 14.5)
    with_radix(s0.R, [&](auto rc) {
      constexpr int R = decltype(rc)::value;
      for (int b = threadIdx.x; b < B; b += NT) {
        C v[R];
#pragma unroll
        for (int r = 0; r < R; r++) v[r] = lds[r * a.t.BP + b];
        dft<R, false>(v);
#pragma unroll
        for (int r = 0; r < R; r++) lds[r * a.t.BP + b] = v[r];
      }
    });
    __syncthreads();
    for (int q = threadIdx.x; q < nr * n; q += NT) {
      const int row = fdiv(q, a.dn0), e = q - row * n;
      const C z = lds[e * a.t.BP + (row >> 1)];
      *(T*)(out + ((unsigned)row * so + (unsigned)e * (unsigned)sizeof(T))) = row & 1 ? z.y : z.x;
    }
    return;
  }
  const int n0 = gdiv(n, s0.mR, s0.R);
  with_radix(s0.R, [&](auto rc) {
    constexpr int R = decltype(rc)::value;
    for (int it = threadIdx.x; it < B * n0; it += NT) {
      const int b = fdiv(it, a.dn0), e0 = it - b * n0;
      C v[R];
      const C* p = lds + gen_unrev(a.L, e0) * a.t.P0 + b;
#pragma unroll
      for (int r = 0; r < R; r++) v[r] = p[r * a.t.BP];
      dft<R, false>(v);
      char* pa = out + ((unsigned)(2 * b) * so + (unsigned)e0 * (unsigned)sizeof(T));
      const unsigned d = (unsigned)n0 * (unsigned)sizeof(T);
      if (2 * b < nr) {
#pragma unroll
        for (int r = 0; r < R; r++) *(T*)(pa + (unsigned)r * d) = v[r].x;
      }
      if (2 * b + 1 < nr) {
#pragma unroll
        for (int r = 0; r < R; r++) *(T*)(pa + so + (unsigned)r * d) = v[r].y;
      }
    }
  });
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
// instructions of a butterfly of radix r per value, and of a stage's
// twiddles, addresses and LDS accesses per value, in units of one FP32
// instruction: the schedule with the smallest sum is taken
static double radix_cost(int r) {
  static const double c[kGenMaxRadix + 1] = {0, 0, 4, 12, 16, 34, 36, 66, 56, 90, 88};
  return c[r] / r;
}
constexpr double kStageCost = 16;

static void search(int m, int maxr, std::vector<int>& cur, double cost, std::vector<int>& best, double& bc) {
  if (cost >= bc) return;
  if (m == 1) {
    bc = cost;
    best = cur;
    return;
  }
  for (int r = std::min(maxr, m); r >= 2; r--) {
    if (m % r) continue;
    cur.push_back(r);
    search(m / r, r, cur, cost + radix_cost(r) + kStageCost, best, bc);
    cur.pop_back();
  }
}

std::vector<int> gen_factors(int n) {
  std::vector<int> big;
  int m = n;
  for (int p = 11; p <= m; p++) {
    bool prime = true;
    for (int q = 2; (long long)q * q <= p; q++)
      if (p % q == 0) { prime = false; break; }
    if (prime && !gen_in_registers(p))
      while (m % p == 0) { big.push_back(p); m /= p; }
  }
  std::vector<int> cur, best;
  double bc = 1e30;
  search(m, kGenMaxRadix, cur, 0, best, bc);
  // the factors in registers, largest first; the large primes in between
  best.insert(best.begin() + (best.empty() ? 0 : 1), big.begin(), big.end());
  return gen_wrap(best);
}

std::vector<int> gen_wrap(const std::vector<int>& f) {
  std::vector<int> g = f;
  if (g.empty() || !gen_in_registers(g.front())) g.insert(g.begin(), 1);
  if (!gen_in_registers(g.back())) g.push_back(1);
  return g;
}

static unsigned magic(int d) { return d > 1 ? (unsigned)(((1ull << 32) + d - 1) / d) : 0u; }
static FDiv make_fdiv(int d) {
  FDiv f;
  f.d = d;
  f.m = ((1ULL << 32) + (uint64_t)d - 1) / (uint64_t)d;
  return f;
}

static GenDesc make_desc(const Len1D& L) {
  GenDesc g;
  std::memset(&g, 0, sizeof(g));
  g.n = L.gd.n;
  g.nst = L.gd.nst;
  if (g.nst > kGenStages) throw Error{"transform length has too many factors", -1};
  for (int s = 0; s < g.nst; s++) {
    GenStage& t = g.st[s];
    t.R = L.gd.radix[s];
    t.Ns = L.gd.ns[s];
    t.tw = L.gd.twoff[s];
    t.mNs = magic(t.Ns);
    t.mR = magic(t.R);
  }
  g.twcount = L.gd.twcount;
  return g;
}

static int log2i(int x) {
  int l = 0;
  while ((1 << (l + 1)) <= x) l++;
  return l;
}

// LDS bytes of a tile of `data` bytes and its twiddle table, which joins the
// tile where that leaves room for as many workgroups per CU or at least two
static size_t place_twiddles(size_t data, const LenDesc& d, int* tw_lds, int* tw_off) {
  const size_t off = (data + 15) & ~(size_t)15, twb = (size_t)d.twcount * sizeof(Tw);
  *tw_off = (int)off;
  *tw_lds = d.twcount > 0 && (off + twb <= 80 * 1024 || (off > 80 * 1024 && off + twb <= kLdsMax)) ? 1 : 0;
  return *tw_lds ? off + twb : off;
}

// (butterfly, pair) items of a prime stage of B sequences, whose outputs a
// workgroup holds in registers, kPrimeItems a thread
static long long prime_items(const LenDesc& d, int s, int B) {
  const int R = d.radix[s];
  return (long long)B * (d.n / R) * ((R + 1) / 2);
}
static bool prime_stages_fit(const LenDesc& d, int B) {
  for (int s = 0; s < d.nst; s++)
    if (gen_over_lds(d.radix[s]) && prime_items(d, s, B) > 1024LL * kPrimeItems) return false;
  return true;
}

// threads of a workgroup: the count that finishes most tiles per unit of
// time, a butterfly of radix R counted as R + 3 and a CU as holding as many
// workgroups as the LDS, 16 waves (128 registers per lane; 24 in FP32, whose
// kernels need 80, measured slower: 240-point columns of 320x240x160 24.0 ->
// 26.1 us) and the number of tiles allow; 0 where no count holds the tile
static int pick_threads(const LenDesc& d, int B, size_t lds, long long tiles) {
  double best = -1;
  int bn = 0;
  for (int nt = 64; nt <= 1024; nt += 64) {
    long long wg = std::min<long long>((long long)(kLdsMax / std::max<size_t>(lds, 1)), 1024 / nt);
    wg = std::max<long long>(1, std::min<long long>(wg, (tiles + 255) / 256));
    double t = 0;
    bool ok = true;
    for (int s = 0; s < d.nst; s++) {
      const int R = d.radix[s];
      const long long nb = (long long)B * (d.n / R);
      if (!gen_over_lds(R)) {
        // (11 and 13 points by pairs: about as many operations as two of their size)
        t += (double)((nb + nt - 1) / nt) * (gen_in_registers(R) ? R + 3 : 2 * R);
      } else {
        const long long items = prime_items(d, s, B);
        if (items > (long long)nt * kPrimeItems) ok = false;
        t += (double)((items + nt - 1) / nt) * 2 * R;
      }
    }
    if (!ok) continue;
    const double rate = (double)wg / t;
    if (rate > best * 1.02) { best = rate; bn = nt; }
  }
  return bn;
}

static int prime_stages(const LenDesc& d) {
  int k = kPrimeNone;
  for (int s = 0; s < d.nst; s++)
    if (!gen_in_registers(d.radix[s])) k = std::max(k, gen_over_lds(d.radix[s]) ? (int)kPrimeLds : (int)kPrimeAny);
  return k;
}

// the tile of a launch: sequences, threads, LDS bytes and the layout
struct TileChoice {
  int B, nt;
  size_t bytes;
  GenTile t;
  int tw_lds, tw_off;
};

// column tile of m rows (d: the schedule, null: rows are copied): a 128-byte
// row segment (plan-time measurement may choose another) while the tile stays
// within the plan's bytes (0: 64 KiB), segments of 64 bytes as long as the tile
// fits at all; halved while there is not a tile for every CU
static TileChoice col_tile(const LenDesc* d, int m, bool lf, long long ncol, int plan_bytes, int seg) {
  const long long E = sizeof(cplx_t);
  const int tile_bytes = plan_bytes ? plan_bytes : 64 * 1024;
  const int R0 = d ? d->radix[0] : 1;
  // LDS bytes of a tile of b columns, sk elements between its blocks
  auto data_of = [&](int b, int sk) {
    const size_t x = (size_t)(((long long)m * (lf && b > 1 ? b + 1 : b) + (long long)(m / R0) * sk) * E);
    return lf && d ? ((x + 15) & ~(size_t)15) + kColTab : x;
  };
  auto above_want = [&](int b) {
    return ((long long)m * (lf && b > 1 ? b + 1 : b) + b) * E + 256 > (long long)tile_bytes + tile_bytes / 8;
  };
  int B = 1;
  while (B * 2 * E <= seg) B *= 2;
  while (B > 1 && ((above_want(B) && B * E > 64) || data_of(B, 0) > kLdsMax)) B /= 2;
  while (B > 1 && d && !prime_stages_fit(*d, B)) B /= 2;
  while (B * E > 32 && (ncol + B - 1) / B < 256) B /= 2;
  // fewer columns than one LDS access covers: blocks an odd multiple of B
  // apart, where the LDS has room for that.  Where it has not, the whole
  // segment counts for more than the bank conflicts: without the skew against
  // half the columns with it, FP64 2400 points x 4096 columns 79 / 73 us (4.0
  // TB/s) against 107 / 94, 5000 x 2048 108 / 88 against 166 / 141; FP32 42 / 42
  // against 51 / 52, 50 / 50 against 74 / 74
  int skew = !lf && B * E < 128 && R0 % 2 == 0 ? B : 0;
  if (data_of(B, skew) > kLdsMax) skew = 0;
  const size_t data = data_of(B, skew);
  TileChoice c;
  c.B = B;
  c.t.BP = lf && B > 1 ? B + 1 : B;
  c.t.R0 = R0;
  c.t.mR0 = magic(R0);
  c.t.skew = skew;
  c.t.P0 = R0 * c.t.BP + skew;
  c.tw_lds = c.tw_off = 0;
  c.bytes = data;
  // a copy has a tile or two per CU in flight and waits for its loads: four values
  // a thread (FP32 with op 'n', forward / backward: 3 fields of 3x192x2149,
  // length-fastest, 95 / 90 us with 256 threads, 51 / 50 so; 2 of 256x32x564, 176
  // modes kept, 66 / 61 -> 46 / 47; with sixteen a thread 63 / 61 and 50 / 49), and
  // at least 256 threads (FP64 forward 192x22x32, 21 modes kept, 14.2 us, 15.7 with
  // 64)
  c.nt = (int)std::max<long long>(256, std::min<long long>(1024, ((long long)m * B + 255) / 256 * 64));
  if (d) {
    c.bytes = place_twiddles(data, *d, &c.tw_lds, &c.tw_off);
    c.nt = pick_threads(*d, B, c.bytes, (ncol + B - 1) / B);
  }
  return c;
}

// the byte offsets of a tile of B columns from its first column stay below 2^32
static bool offsets_fit(const ColSpec& c, int B) {
  const long long nout = B / std::max(c.n_inner, 1) + 2;
  auto fits = [&](long long si, long long sl, long long so) {
    return (nout * so + (long long)c.n_inner * si + (long long)(std::max(c.nld, c.nst) + 1) * sl) *
               (long long)sizeof(cplx_t) < (1LL << 32);
  };
  return fits(c.si_in, c.sl_in, c.so_in) && fits(c.si_out, c.sl_out, c.so_out);
}

// f(TL, PM): the twiddle table in LDS, the schedule's prime stages
template <class F>
static void with_variant(bool tl, int pm, F f) {
  auto with_tl = [&](auto t) {
    if (pm == kPrimeAny) f(t, std::integral_constant<int, kPrimeAny>{});
    else if (pm == kPrimeLds) f(t, std::integral_constant<int, kPrimeLds>{});
    else f(t, std::integral_constant<int, kPrimeNone>{});
  };
  if (tl) with_tl(std::true_type{});
  else with_tl(std::false_type{});
}

template <bool FWD, bool MAP, int LF, class Off>
static void go_col(const GColArgs& a, int pm, unsigned g, int nt, size_t bytes, hipStream_t st) {
  with_variant(a.tw_lds != 0, pm, [&](auto tl, auto pr) {
    k_gcol<real_t, FWD, MAP, LF, Off, tl.value, pr.value><<<g, nt, bytes, st>>>(a);
  });
}

void gen_launch_col(const Len1D* L, const ColSpec& c, int xcd, bool wide, hipStream_t st) {
  const long long ncol = (long long)c.n_inner * c.n_outer;
  if (ncol > 0x7fffffffLL) throw Error{"grid too large", -1};
  GColArgs a;
  std::memset(&a, 0, sizeof(a));
  a.in = c.in; a.out = c.out;
  a.si_in = c.si_in; a.sl_in = c.sl_in; a.so_in = c.so_in;
  a.si_out = c.si_out; a.sl_out = c.sl_out; a.so_out = c.so_out;
  a.ncol = ncol;
  a.n_inner = c.n_inner;
  a.kind = c.kind;
  a.rows = c.n;
  a.nld = c.nld; a.ld_lo = c.ld_lo; a.ld_hi = c.ld_hi; a.ld_shift = c.ld_shift;
  a.nst = c.nst; a.st_lo = c.st_lo; a.st_shift = c.st_shift;
  a.rev = c.rev ? 1 : 0;
  a.xcd = xcd;
  const bool lf_in = c.sl_in == 1 && c.si_in != 1, lf_out = c.sl_out == 1 && c.si_out != 1;
  const bool lf = lf_in || lf_out;
  const int m = L ? L->gd.n : c.nld;
  const TileChoice tc =
      L ? col_tile(&L->gd, m, lf, ncol, L->tile_bytes, L->col_seg) : col_tile(nullptr, m, lf, ncol, 0, 128);
  const int B = tc.B;
  a.lB = log2i(B);
  a.t = tc.t;
  const long long nwg = (ncol + B - 1) / B;
  if (nwg > 0x7fffffffLL) throw Error{"grid too large", -1};
  if (!L) {
    if (tc.bytes > kLdsMax) throw Error{"column copy does not fit in LDS", -1};
    a.dld = make_fdiv(c.nld);
    a.dst = make_fdiv(c.nst);
    k_gcopy<real_t><<<(unsigned)nwg, tc.nt, tc.bytes, st>>>(a);
    check_hip(hipGetLastError(), "k_gcopy launch");
    return;
  }
  a.L = make_desc(*L);
  a.tw = L->gtw;
  a.dld = make_fdiv(m);
  a.dst = make_fdiv(std::max(c.nst, 1));
  a.tw_lds = tc.tw_lds; a.tw_off = tc.tw_off;
  const size_t bytes = tc.bytes;
  if (bytes > kLdsMax) throw Error{"column transform does not fit in LDS", -1};
  const int nt = tc.nt;
  if (!nt) throw Error{"transform tile exceeds the 1024-thread workgroup capacity", -1};
  const int pm = prime_stages(L->gd);
  const bool fwd = c.fwd || c.kind == COL_DCT1 || c.kind == COL_DST1;
  const bool ld_id = c.nld == m && (c.ld_lo >= m || (c.ld_hi <= c.ld_lo && c.ld_shift == 0));
  const bool st_id = c.nst == m && (c.st_lo >= m || c.st_shift == 0);
  const bool map = c.kind != COL_C2C || !(ld_id && st_id);
  const bool fits = !wide && offsets_fit(c, B);
  typedef unsigned U32;
  typedef unsigned long long U64;
  const unsigned g = (unsigned)nwg;
  if (fwd) {
    if (lf_in) go_col<true, true, 1, U64>(a, pm, g, nt, bytes, st);
    else if (lf_out) go_col<true, true, 2, U64>(a, pm, g, nt, bytes, st);
    else if (!fits && map) go_col<true, true, 0, U64>(a, pm, g, nt, bytes, st);
    else if (!fits) go_col<true, false, 0, U64>(a, pm, g, nt, bytes, st);
    else if (map) go_col<true, true, 0, U32>(a, pm, g, nt, bytes, st);
    else go_col<true, false, 0, U32>(a, pm, g, nt, bytes, st);
  } else {
    if (lf_in) go_col<false, true, 1, U64>(a, pm, g, nt, bytes, st);
    else if (lf_out) go_col<false, true, 2, U64>(a, pm, g, nt, bytes, st);
    else if (!fits && map) go_col<false, true, 0, U64>(a, pm, g, nt, bytes, st);
    else if (!fits) go_col<false, false, 0, U64>(a, pm, g, nt, bytes, st);
    else if (map) go_col<false, true, 0, U32>(a, pm, g, nt, bytes, st);
    else go_col<false, false, 0, U32>(a, pm, g, nt, bytes, st);
  }
  check_hip(hipGetLastError(), "k_gcol launch");
}

// tile of the X kernels, rows of at most `row` elements apart
static TileChoice x_row_tile(const LenDesc& d, long long nrows, long long row, int plan_bytes) {
  const long long pairs = (nrows + 1) / 2, E = sizeof(cplx_t);
  const int n = d.n;
  int B = 16;
  // short rows: tiles of more than 256 values, below which the launch of the
  // workgroups bounds the pass, up to 64 pairs (the lanes along them divide every
  // workgroup).  Not from 16 points on: FP32 c2r of 2^23 points in rows of 16 takes
  // 20.6 us with 16 pairs, 22.6 with 32; of 11 31 and 22 us
  while (B < 64 && 2LL * B * n < 512) B *= 2;
  // the plan's bytes, by default 64 KiB, in FP64 40 KiB (four workgroups per CU in
  // different phases; a prime stage wants the pairs): r2c / c2r 600x128x200 61 / 74 -> 48 / 50 us,
  // 720x240x200 155 / 165 -> 139 / 130.  FP32 measured no gain (1500x64x100 28
  // -> 29), its tiles hold twice the values per byte in flight.
  const long long def = sizeof(real_t) == 8 && prime_stages(d) == kPrimeNone ? 40 * 1024 : 64 * 1024;
  const long long lim = plan_bytes ? plan_bytes : def;
  while (B > 1 && ((long long)n * (B + 1) * E > lim || (2LL * B + 1) * row * E >= (1LL << 32))) B /= 2;
  while (B > 1 && !prime_stages_fit(d, B)) B /= 2;
  while (B > 2 && (pairs + B - 1) / B < 512) B /= 2;
  TileChoice c;
  c.B = B;
  c.t.BP = B > 1 ? B + 1 : 1;
  c.t.R0 = d.radix[0];
  c.t.mR0 = magic(c.t.R0);
  c.t.skew = 0;
  c.t.P0 = c.t.R0 * c.t.BP;
  c.bytes = place_twiddles((size_t)n * c.t.BP * E, d, &c.tw_lds, &c.tw_off);
  c.nt = pick_threads(d, B, c.bytes, (pairs + B - 1) / B);
  return c;
}

// the same for a launch; returns the LDS bytes
static size_t x_tile(GXArgs& a, const Len1D& L, long long nrows, long long row, int* nt, unsigned* nwg) {
  const TileChoice c = x_row_tile(L.gd, nrows, row, L.tile_bytes);
  a.lB = log2i(c.B);
  a.t = c.t;
  a.L = make_desc(L);
  a.tw = L.gtw;
  a.dn0 = make_fdiv(L.gd.n / c.t.R0);
  a.tw_lds = c.tw_lds; a.tw_off = c.tw_off;
  if (c.bytes > kLdsMax) throw Error{"X transform does not fit in LDS", -1};
  if (!c.nt) throw Error{"transform tile exceeds the 1024-thread workgroup capacity", -1};
  const long long g = ((nrows + 1) / 2 + c.B - 1) / c.B;
  if (g > 0x7fffffffLL) throw Error{"grid too large", -1};
  *nwg = (unsigned)g;
  *nt = c.nt;
  return c.bytes;
}

// launch shape of a length (host only): form 0 rows on both sides, 1 a
// length-fastest side, 2 rows along X, 3 and 4 as 0 and 1 of rows that are copied
void gen_tile_shape(const LenDesc& d, int form, long long count, int tile_bytes, int seg, bool wide, int* seqs,
                    int* threads, size_t* lds, int* offset_bytes) {
  const TileChoice c = form == 2   ? x_row_tile(d, count, d.n + 2, tile_bytes)
                       : form >= 3 ? col_tile(nullptr, d.n, form == 4, count, 0, 128)
                                   : col_tile(&d, d.n, form == 1, count, tile_bytes, seg);
  *seqs = c.B;
  *threads = c.nt;
  *lds = c.bytes;
  ColSpec v{};
  v.n_inner = (int)std::min<long long>(count, 0x7fffffff);
  v.n_outer = 1;
  v.si_in = v.si_out = 1;
  v.sl_in = v.sl_out = count;
  v.nld = v.nst = d.n;
  *offset_bytes = form == 2 || (form == 0 && !wide && offsets_fit(v, c.B)) ? 4 : 8;
}

void gen_launch_x_r2c(const Len1D& L, const real_t* in, cplx_t* out, long long nrows, long long si_row,
                      long long so_row, int nxo, bool rev, hipStream_t st) {
  GXArgs a;
  std::memset(&a, 0, sizeof(a));
  a.in = in; a.out = out; a.nrows = nrows; a.si_row = si_row; a.so_row = so_row;
  a.nk = nxo; a.dnk = make_fdiv(nxo);
  a.rev = rev ? 1 : 0;
  int nt;
  unsigned g;
  const size_t bytes = x_tile(a, L, nrows, std::max(si_row, so_row), &nt, &g);
  with_variant(a.tw_lds != 0, prime_stages(L.gd), [&](auto tl, auto pm) {
    k_gx_r2c<real_t, tl.value, pm.value><<<g, nt, bytes, st>>>(a);
  });
  check_hip(hipGetLastError(), "k_gx_r2c launch");
}

void gen_launch_x_c2r(const Len1D& L, const cplx_t* in, real_t* out, long long nrows, long long si_row,
                      long long so_row, int nxi, bool rev, hipStream_t st) {
  GXArgs a;
  std::memset(&a, 0, sizeof(a));
  a.in = in; a.out = out; a.nrows = nrows; a.si_row = si_row; a.so_row = so_row;
  a.nk = nxi; a.dnk = make_fdiv(L.gd.n / 2 + 1);
  a.rev = rev ? 1 : 0;
  int nt;
  unsigned g;
  const size_t bytes = x_tile(a, L, nrows, std::max(si_row, so_row), &nt, &g);
  if (L.gd.nst == 1) a.dn0 = make_fdiv(L.gd.n);
  with_variant(a.tw_lds != 0, prime_stages(L.gd), [&](auto tl, auto pm) {
    k_gx_c2r<real_t, tl.value, pm.value><<<g, nt, bytes, st>>>(a);
  });
  check_hip(hipGetLastError(), "k_gx_c2r launch");
}

template <class K>
static void allow_big_lds(K kernel) {
  (void)hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsMax);
  (void)hipGetLastError();  // a refused attribute leaves the default limit, not a pending error
}
template <bool FWD, bool TL, int PM>
static void prep_dir() {
  typedef unsigned U32;
  typedef unsigned long long U64;
  allow_big_lds(k_gcol<real_t, FWD, false, 0, U32, TL, PM>);
  allow_big_lds(k_gcol<real_t, FWD, true, 0, U32, TL, PM>);
  allow_big_lds(k_gcol<real_t, FWD, false, 0, U64, TL, PM>);
  allow_big_lds(k_gcol<real_t, FWD, true, 0, U64, TL, PM>);
  allow_big_lds(k_gcol<real_t, FWD, true, 1, U64, TL, PM>);
  allow_big_lds(k_gcol<real_t, FWD, true, 2, U64, TL, PM>);
  if (FWD) allow_big_lds(k_gx_r2c<real_t, TL, PM>);
  else allow_big_lds(k_gx_c2r<real_t, TL, PM>);
}
void gen_prep_kernels() {
  static std::once_flag once;
  std::call_once(once, [] {
    for (int tl = 0; tl < 2; tl++)
      for (int pm : {kPrimeNone, kPrimeLds, kPrimeAny})
        with_variant(tl != 0, pm, [](auto t, auto p) {
          prep_dir<true, t.value, p.value>();
          prep_dir<false, t.value, p.value>();
        });
    allow_big_lds(k_gcopy<real_t>);
  });
}

}  // namespace p3amd
