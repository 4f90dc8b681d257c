// engine_ct.hpp -- compile-time specialised engine.
//
// For the transform lengths the workloads use, the radix schedule, the tile
// width and the thread count are template parameters, so every index
// computation of a stage folds to shifts and constant multiplies and the
// per-thread register arrays have fixed size.  The LDS tile holds B sequences,
// element e of sequence b at lds[e*B + b] (columns), in rotated rows (lds_at:
// length-fastest columns) or in skewed ones (XLay: rows along X), each laid out
// so that the accesses along the sequences and along the elements both avoid
// bank conflicts.  The stages run in place wherever one side is addressed by
// row, and so can be digit-reversed at no cost.  Stage twiddles use the same
// table layout as the run-time engine (stage 0 has none; stage s holds
// Ns*(R-1) entries W_{Ns R}^{k r}, k < Ns, r = 1..R-1).
#pragma once
#include <type_traits>
#include "fft_device.hpp"

namespace p3amd {

template <int... Rs>
struct RList {};

template <int A, int... Rs>
struct RProd {
  static constexpr int value = A * RProd<Rs...>::value;
};
template <int A>
struct RProd<A> {
  static constexpr int value = A;
};

// element `row` of sequence b in a tile of B sequences: rows BP elements apart,
// or (BP = 0) rows of B elements rotated by the row, so that lanes along the
// rows and lanes along the sequences both meet distinct LDS banks without
// padding
template <int B, int BP>
__device__ __forceinline__ int lds_at(int row, int b) {
  if constexpr (BP == 0) return row * B + ((b + row) & (B - 1));
  else return row * BP + b;
}

// One stage: radix R, Ns = product of the earlier radices, twiddles at Off.
template <class T, int R, bool FWD, int N, int B, int BP, int NT, int Ns, int Off>
__device__ __forceinline__ void stage_ct(cpx<T>* lds, const typename TwT<T>::type* tw) {
  constexpr int nR = N / R;
  constexpr int total = B * nR;
  constexpr int IT = (total + NT - 1) / NT;
  cpx<T> v[IT][R];
#pragma unroll
  for (int m = 0; m < IT; m++) {
    const int it = threadIdx.x + m * NT;
    if ((total % NT) == 0 || it < total) {
      const int j = it / B, b = it % B;
#pragma unroll
      for (int r = 0; r < R; r++) v[m][r] = lds[lds_at<B, BP>(j + r * nR, b)];
      if constexpr (Ns > 1) {
        const int k = j % Ns;
        const typename TwT<T>::type* w = tw + Off + k * (R - 1);
#pragma unroll
        for (int r = 1; r < R; r++) v[m][r] = twmul<FWD>(v[m][r], w[r - 1]);
      }
      dft<R, FWD>(v[m]);
    }
  }
  __syncthreads();
#pragma unroll
  for (int m = 0; m < IT; m++) {
    const int it = threadIdx.x + m * NT;
    if ((total % NT) == 0 || it < total) {
      const int j = it / B, b = it % B;
      const int k = j % Ns;
      const int base = (j - k) * R + k;
#pragma unroll
      for (int r = 0; r < R; r++) lds[lds_at<B, BP>(base + r * Ns, b)] = v[m][r];
    }
  }
  __syncthreads();
}

// The same stage in place: positions in mixed radix, the first radix the
// fastest digit, so a butterfly writes the positions it read (see the first
// stage's Rev): one barrier, nothing held across it.
template <class T, int R, bool FWD, int N, int B, int BP, int NT, int Ns, int Off>
__device__ __forceinline__ void stage_ip(cpx<T>* lds, const typename TwT<T>::type* tw, int tid = threadIdx.x) {
  constexpr int total = B * (N / R);
  constexpr int IT = (total + NT - 1) / NT;
#pragma unroll
  for (int m = 0; m < IT; m++) {
    const int it = tid + m * NT;
    if ((total % NT) == 0 || it < total) {
      const int j = it / B, b = it % B;
      const int k = j % Ns, base = (j - k) * R + k;
      cpx<T> v[R];
#pragma unroll
      for (int r = 0; r < R; r++) v[r] = lds[lds_at<B, BP>(base + r * Ns, b)];
      const typename TwT<T>::type* w = tw + Off + k * (R - 1);
#pragma unroll
      for (int r = 1; r < R; r++) v[r] = twmul<FWD>(v[r], w[r - 1]);
      dft<R, FWD>(v);
#pragma unroll
      for (int r = 0; r < R; r++) lds[lds_at<B, BP>(base + r * Ns, b)] = v[r];
    }
  }
  __syncthreads();
}

template <class T, bool FWD, int N, int B, int BP, int NT, int Ns, int Off, int R, int... Rest>
__device__ __forceinline__ void stages_ip(cpx<T>* lds, const typename TwT<T>::type* tw) {
  stage_ip<T, R, FWD, N, B, BP, NT, Ns, Off>(lds, tw);
  if constexpr (sizeof...(Rest) > 0)
    stages_ip<T, FWD, N, B, BP, NT, Ns * R, Off + Ns * (R - 1), Rest...>(lds, tw);
}

// Input row of the first stage's butterfly j: j itself for the autosort
// stages; for the in-place ones the digits of j over the later radices
// (Rs..., the first of them the fastest digit of j) in reverse.
struct RowNatural {
  static __device__ __forceinline__ int at(int j) { return j; }
};
template <int... Rs>
struct RowRev {
  template <int R, int... Rest>
  static __device__ __forceinline__ int step(int j, int acc) {
    if constexpr (sizeof...(Rest) == 0) return acc * R + j;
    else return step<Rest...>(j / R, acc * R + j % R);
  }
  static __device__ __forceinline__ int at(int j) { return step<Rs...>(j, 0); }
};

// the inverse: the butterfly of the first stage that holds input row e < N/R0
template <int R, int... Rest>
struct RowInv {
  static __device__ __forceinline__ int at(int e) {
    if constexpr (sizeof...(Rest) == 0) return e;
    else return e / RProd<Rest...>::value + R * RowInv<Rest...>::at(e % RProd<Rest...>::value);
  }
};

// LDS tile of the X kernels: B row pairs, position p of pair b at
// lds[at(p) + b].  The tile is reached by lanes along the pairs (middle
// stages), along neighbouring positions (separation) and along neighbouring
// blocks of the digit-reversed order (first stage): where a row of the tile is
// at most half the banks wide, one element more every 4 positions and 3 more
// every R0 R1 keep all three within twice the conflict-free cycles (512 points
// FP32, counted: 1.1 / 1.2 conflict cycles per LDS access of r2c / c2r, which
// takes 4 without), else a padded row and one element more every R0 R1.
template <class T, int B, class RL>
struct XLay;
template <class T, int B, int R0, int R1, int... Rs>
struct XLay<T, B, RList<R0, R1, Rs...>> {
  static constexpr int N = RProd<R0, R1, Rs...>::value;
  static constexpr bool HALF = B * sizeof(cpx<T>) <= 128;
  static constexpr int BP = HALF ? B : B + 1, D = HALF ? 4 : N, S2 = HALF ? 3 : 1;
  static_assert(!HALF || R0 % 4 == 0, "blocks of whole skews");
  static __device__ __host__ constexpr int at(int p) { return p * BP + p / D + p / (R0 * R1) * S2; }
  static constexpr long long BYTES = (long long)(at(N - 1) + B) * (long long)sizeof(cpx<T>);
};

// an in-place stage of the X tile (as stage_ip), decimation in time (the
// twiddles before the butterfly) or in frequency (after it)
template <class T, int R, bool FWD, bool DIF, class Lay, int B, int NT, int Ns, int Off>
__device__ __forceinline__ void x_stage_ip(cpx<T>* lds, const typename TwT<T>::type* tw) {
  constexpr int total = B * (Lay::N / R);
  constexpr int IT = (total + NT - 1) / NT;
#pragma unroll
  for (int m = 0; m < IT; m++) {
    const int it = threadIdx.x + m * NT;
    if ((total % NT) == 0 || it < total) {
      const int j = it / B, b = it % B;
      const int k = j % Ns;
      cpx<T>* p = lds + Lay::at((j - k) * R + k) + b;
      cpx<T> v[R];
#pragma unroll
      for (int r = 0; r < R; r++) v[r] = p[Lay::at(r * Ns)];
      const typename TwT<T>::type* w = tw + Off + k * (R - 1);
      if constexpr (Ns > 1 && !DIF) {
#pragma unroll
        for (int r = 1; r < R; r++) v[r] = twmul<FWD>(v[r], w[r - 1]);
      }
      dft<R, FWD>(v);
      if constexpr (Ns > 1 && DIF) {
#pragma unroll
        for (int r = 1; r < R; r++) v[r] = twmul<FWD>(v[r], w[r - 1]);
      }
#pragma unroll
      for (int r = 0; r < R; r++) p[Lay::at(r * Ns)] = v[r];
    }
  }
  __syncthreads();
}

// the stages after the first: upwards in time, downwards in frequency
template <class T, bool FWD, bool DIF, class Lay, int B, int NT, int Ns, int Off, int R, int... Rest>
__device__ __forceinline__ void x_stages_ip(cpx<T>* lds, const typename TwT<T>::type* tw) {
  if constexpr (!DIF) x_stage_ip<T, R, FWD, DIF, Lay, B, NT, Ns, Off>(lds, tw);
  if constexpr (sizeof...(Rest) > 0)
    x_stages_ip<T, FWD, DIF, Lay, B, NT, Ns * R, Off + Ns * (R - 1), Rest...>(lds, tw);
  if constexpr (DIF) x_stage_ip<T, R, FWD, DIF, Lay, B, NT, Ns, Off>(lds, tw);
}

// r2c: two real rows per complex sequence, ld(row, e) element e of a row of
// the tile.  The first stage reads the rows itself, lanes along N/R0 elements,
// where those are at least 32 bytes; shorter ones are read row by row into
// the tile's digit-reversed order first.  The other stages run in place.
template <class T, class Lay, int B, int NT, class Tw, class LD, int R0, int... Rs>
__device__ __forceinline__ void x_fft_fwd(cpx<T>* lds, const Tw& ctw, LD ld, RList<R0, Rs...>) {
  constexpr int N = Lay::N, nR = N / R0;
  if constexpr (nR * sizeof(T) >= 32) {
    constexpr int total = B * nR, IT = (total + NT - 1) / NT;
    cpx<T> v[IT][R0];
#pragma unroll
    for (int m = 0; m < IT; m++) {
      const int it = threadIdx.x + m * NT;
      const bool ok = (total % NT) == 0 || it < total;
      const int b = ok ? it / nR : 0, e = it % nR;
#pragma unroll
      for (int r = 0; r < R0; r++) {
        v[m][r].x = ld(2 * b, e + r * nR);
        v[m][r].y = ld(2 * b + 1, e + r * nR);
      }
    }
#pragma unroll
    for (int m = 0; m < IT; m++) {
      const int it = threadIdx.x + m * NT;
      if ((total % NT) == 0 || it < total) {
        const int b = it / nR, e = it % nR;
        dft<R0, true>(v[m]);
        cpx<T>* p = lds + Lay::at(RowInv<Rs...>::at(e) * R0) + b;
#pragma unroll
        for (int r = 0; r < R0; r++) p[Lay::at(r)] = v[m][r];
      }
    }
    ctw.put();
    __syncthreads();
  } else {
    constexpr int LI = (B * N + NT - 1) / NT;
    cpx<T> v[LI];
#pragma unroll
    for (int i = 0; i < LI; i++) {
      const int q = threadIdx.x + i * NT;
      const bool ok = (B * N) % NT == 0 || q < B * N;
      const int b = ok ? q / N : 0, e = q % N;
      v[i].x = ld(2 * b, e);
      v[i].y = ld(2 * b + 1, e);
    }
#pragma unroll
    for (int i = 0; i < LI; i++) {
      const int q = threadIdx.x + i * NT;
      if ((B * N) % NT == 0 || q < B * N) {
        const int e = q % N;
        lds[Lay::at(RowInv<Rs...>::at(e % nR) * R0 + e / nR) + q / N] = v[i];
      }
    }
    ctw.put();
    __syncthreads();
    x_stage_ip<T, R0, true, false, Lay, B, NT, 1, 0>(lds, ctw.table());
  }
  x_stages_ip<T, true, false, Lay, B, NT, R0, 0, Rs...>(lds, ctw.table());
}

// c2r, the mirror image: natural order in the tile, the stages downwards in
// place, the first radix last; st(pair, e, z) stores element e of a pair's
// rows.  From the last stage itself where N/R0 elements are at least 64 bytes:
// below (FP32, 48 points) the short runs of the stores cost more than the
// pass through the tile.
template <class T, class Lay, int B, int NT, class ST, int R0, int... Rs>
__device__ __forceinline__ void x_fft_bwd(cpx<T>* lds, const typename TwT<T>::type* tw, ST st, RList<R0, Rs...>) {
  constexpr int N = Lay::N, nR = N / R0;
  x_stages_ip<T, false, true, Lay, B, NT, R0, 0, Rs...>(lds, tw);
  if constexpr (nR * sizeof(T) >= 64) {
    constexpr int total = B * nR, IT = (total + NT - 1) / NT;
#pragma unroll
    for (int m = 0; m < IT; m++) {
      const int it = threadIdx.x + m * NT;
      if ((total % NT) == 0 || it < total) {
        const int b = it / nR, e = it % nR;
        const cpx<T>* p = lds + Lay::at(RowInv<Rs...>::at(e) * R0) + b;
        cpx<T> v[R0];
#pragma unroll
        for (int r = 0; r < R0; r++) v[r] = p[Lay::at(r)];
        dft<R0, false>(v);
#pragma unroll
        for (int r = 0; r < R0; r++) st(b, e + r * nR, v[r]);
      }
    }
  } else {
    x_stage_ip<T, R0, false, true, Lay, B, NT, 1, 0>(lds, tw);
    constexpr int LI = (B * N + NT - 1) / NT;
#pragma unroll
    for (int i = 0; i < LI; i++) {
      const int q = threadIdx.x + i * NT;
      if ((B * N) % NT == 0 || q < B * N) {
        const int e = q % N;
        st(q / N, e, lds[Lay::at(RowInv<Rs...>::at(e % nR) * R0 + e / nR) + q / N]);
      }
    }
  }
}

template <class T, bool FWD, int N, int B, int BP, int NT, int Ns, int Off, int R, int... Rest>
__device__ __forceinline__ void stages_ct(cpx<T>* lds, const typename TwT<T>::type* tw) {
  stage_ct<T, R, FWD, N, B, BP, NT, Ns, Off>(lds, tw);
  if constexpr (sizeof...(Rest) > 0)
    stages_ct<T, FWD, N, B, BP, NT, Ns * R, (Ns > 1 ? Off + Ns * (R - 1) : Off), Rest...>(lds, tw);
}

template <class T, bool FWD, int B, int BP, int NT, int... Rs>
__device__ __forceinline__ void run_fft_ct(cpx<T>* lds, const typename TwT<T>::type* tw, RList<Rs...>) {
  constexpr int N = RProd<Rs...>::value;
  stages_ct<T, FWD, N, B, BP, NT, 1, 0, Rs...>(lds, tw);
}

// Twiddle table entries used by a radix list (all stages after the first).
template <int... Rs>
struct TwCount;
template <int R0, int... Rs>
struct TwCount<R0, Rs...> {
  template <int Ns, int R, int... Rest>
  static constexpr int tail() {
    if constexpr (sizeof...(Rest) == 0) return Ns * (R - 1);
    else return Ns * (R - 1) + tail<Ns * R, Rest...>();
  }
  static constexpr int value() {
    if constexpr (sizeof...(Rs) == 0) return 0;
    else return tail<R0, Rs...>();
  }
};

// The twiddle table of a workgroup, in LDS (L) or where it is.  Its loads are
// issued here, ahead of the tile's, and written to LDS by put() when the
// tile's first stage is done, so that a workgroup waits for memory once and
// not twice before its first stage.
template <class T, int NT, bool L, class RL>
struct CtTw;
template <class T, int NT, bool L, int... Rs>
struct CtTw<T, NT, L, RList<Rs...>> {
  typedef typename TwT<T>::type TwL;
  static constexpr int COUNT = TwCount<Rs...>::value(), K = L ? (COUNT + NT - 1) / NT : 1;
  const TwL* src;
  TwL* dst;
  TwL v[K];
  __device__ __forceinline__ CtTw(const void* tw, unsigned char* smem, int off) {
    src = (const TwL*)tw;
    dst = (TwL*)(smem + off);
    if constexpr (L) {
#pragma unroll
      for (int i = 0; i < K; i++) {
        const int e = threadIdx.x + i * NT;
        v[i] = src[e < COUNT ? e : 0];
      }
    }
  }
  // before the barrier that ends the first stage
  __device__ __forceinline__ void put() const {
    if constexpr (L) {
#pragma unroll
      for (int i = 0; i < K; i++) {
        const int e = threadIdx.x + i * NT;
        if (e < COUNT) dst[e] = v[i];
      }
    }
  }
  __device__ __forceinline__ const TwL* table() const {
    if constexpr (L) return dst;
    else return src;
  }
};

// ---------------------------------------------------------------------------
// Column transforms with the first stage fed straight from global memory and
// the last stage stored straight to global memory (one LDS round trip fewer
// at each end; every thread keeps IT*R independent loads in flight).
// Addresses are a wave-uniform 64-bit tile base plus 32-bit per-lane byte
// offsets (Off = unsigned), so an element access costs one 32-bit add; views
// whose offsets do not fit use 64-bit offsets (Off = unsigned long long).
// With PR the rows are
// remapped on load (pruning zero-fill) and on store (pruning selection);
// without it both maps are the identity.
// ---------------------------------------------------------------------------
constexpr int kSepIT = 2, kSepR = 16;
struct ColIO {
  const char* in;             // input tile base
  char* out;                  // output tile base
  unsigned long long lane_in, lane_out;  // this lane's column, bytes from the tile bases
  unsigned long long sl_in, sl_out;      // row strides, bytes
  int nb;                     // valid columns of this tile
  int ld_lo, ld_hi, ld_shift; // PR: LDS row e <- input row e (e<ld_lo), e-ld_shift (e>=ld_hi), else 0
  int nst, st_lo, st_shift;   // PR: output row e <- FFT row e (e<st_lo) or e+st_shift
  int mirror;                 // PR, > 0: DCT-I even extension, row e <- input e (e<mirror) or 2(mirror-1)-e
  // table-addressed rows (Off = TabRows): row e of this lane's column at
  // element ltab[e].x + lane_o * ltab[e].y + lane_i of `in` (zero when
  // ltab[e].x < 0), FFT row p stored at stab[p] likewise (skipped when < 0)
  const int2* ltab;
  const int2* stab;
  unsigned lane_o, lane_i;    // this lane's outer and inner column index
  // separable rows (Off = TabSep): row e0 + r n/R of this lane's column at
  // byte lane_in + sa_in[m] + sb_in[r], e0 the first row of this thread's m-th
  // first-stage butterfly; FFT row j + r Ns likewise at lane_out + sa_out[m] +
  // sb_out[r]
  unsigned sa_in[kSepIT], sa_out[kSepIT], sb_in[kSepR], sb_out[kSepR];
};

// offset types selecting the table-addressed rows: some rows missing, none
// missing, or none missing and the table a sum of a part per butterfly and a
// part per value (peers with equal blocks), which needs no table in LDS
struct TabRows {};
struct TabAll {};
struct TabSep {};
template <class Off>
constexpr bool is_tab = std::is_same<Off, TabRows>::value || std::is_same<Off, TabAll>::value;

template <int R, int N, int B, int NT>
struct Stage0 {
  static constexpr int nR = N / R;
  static constexpr int total = B * nR;
  static constexpr int IT = (total + NT - 1) / NT;
};

template <class T, class Off>
__device__ __forceinline__ cpx<T> ld_at(const char* base, Off off) {
  return *(const cpx<T>*)(base + off);
}

template <class T, class Off>
__device__ __forceinline__ void st_at(char* base, Off off, cpx<T> v) {
  *(cpx<T>*)(base + off) = v;
}

// the first stage's values of one tile, held in registers between the loads
// and the butterflies
template <class T, int R, int N, int B, int NT>
struct Stage0Regs {
  cpx<T> v[Stage0<R, N, B, NT>::IT][R];
};

// first stage, loads: the tile's values of every butterfly of this thread.
// Lanes past the tile's last column repeat it (col_io with CL), so a loaded
// value is left alone until the butterflies: a select on it would wait for it
// where it is issued.
template <class T, int R, int N, int B, int NT, class Off, class Row>
__device__ __forceinline__ void stage0_load(Stage0Regs<T, R, N, B, NT>& rg, const ColIO& io, int tid) {
  static_assert(NT % B == 0, "one column per thread");
  typedef Stage0<R, N, B, NT> S;
  static_assert(!std::is_same<Off, TabSep>::value || (S::IT <= kSepIT && R <= kSepR), "separable rows");
#pragma unroll
  for (int m = 0; m < S::IT; m++) {
    const int it = tid + m * NT;
    if ((S::total % NT) == 0 || it < S::total) {
      const int j = Row::at(it / B);
#pragma unroll
      for (int r = 0; r < R; r++) {
        const int e = j + r * S::nR;
        if constexpr (std::is_same<Off, TabSep>::value) {
          rg.v[m][r] = ld_at<T, unsigned>(io.in, (unsigned)io.lane_in + io.sa_in[m] + io.sb_in[r]);
        } else if constexpr (is_tab<Off>) {
          const int2 t = io.ltab[e];
          const unsigned el = (unsigned)t.x + io.lane_o * (unsigned)t.y + io.lane_i;
          if constexpr (std::is_same<Off, TabAll>::value) {
            rg.v[m][r] = ((const cpx<T>*)io.in)[el];
          } else {
            const cpx<T> u = ((const cpx<T>*)io.in)[t.x >= 0 ? el : 0u];
            rg.v[m][r] = t.x >= 0 ? u : mk<T>(0, 0);
          }
        } else {
          rg.v[m][r] = ld_at<T, Off>(io.in, (Off)io.lane_in + (Off)e * (Off)io.sl_in);
        }
      }
    }
  }
}

// first stage, butterflies (no twiddles) and results into the LDS tile
template <class T, int R, bool FWD, int N, int B, int NT>
__device__ __forceinline__ void stage0_put(cpx<T>* lds, Stage0Regs<T, R, N, B, NT>& rg, int tid) {
  typedef Stage0<R, N, B, NT> S;
#pragma unroll
  for (int m = 0; m < S::IT; m++) {
    const int it = tid + m * NT;
    if ((S::total % NT) == 0 || it < S::total) {
      const int j = it / B, b = it % B;
      dft<R, FWD>(rg.v[m]);
#pragma unroll
      for (int r = 0; r < R; r++) lds[(j * R + r) * B + b] = rg.v[m][r];
    }
  }
  __syncthreads();
}

// first stage: loads of one tile into registers, butterflies (no twiddles),
// results into the LDS tile (the loads as stage0_load, written out here so
// that every load of the tile is issued back to back: composed of the two
// steps, the compiler interleaved them with address arithmetic and waited
// before the last one).  pre() runs before the barrier: it writes what the later
// stages read from LDS and was loaded ahead of the tile (CtTw).
template <class T, int R, bool FWD, int N, int B, int NT, bool PR, class Off, class Row, int BP = B, class Pre>
__device__ __forceinline__ void stage0_global(cpx<T>* lds, const ColIO& io, Pre pre) {
  static_assert(NT % B == 0, "one column per thread");
  constexpr bool TB = is_tab<Off>;
  typedef Stage0<R, N, B, NT> S;
  const bool valid = (int)(threadIdx.x % B) < io.nb;
  cpx<T> v[S::IT][R];
#pragma unroll
  for (int m = 0; m < S::IT; m++) {
    const int it = threadIdx.x + m * NT;
    if ((S::total % NT) == 0 || it < S::total) {
      const int j = Row::at(it / B);
#pragma unroll
      for (int r = 0; r < R; r++) {
        const int e = j + r * S::nR;
        // items outside the tile load its first element (always valid) and
        // are zeroed, so no load sits under a branch
        if constexpr (TB) {
          const int2 t = io.ltab[e];
          const bool ok = valid && (std::is_same<Off, TabAll>::value || t.x >= 0);
          const unsigned el = ok ? (unsigned)t.x + io.lane_o * (unsigned)t.y + io.lane_i : 0u;
          const cpx<T> u = ((const cpx<T>*)io.in)[el];
          v[m][r] = ok ? u : mk<T>(0, 0);
        } else if constexpr (PR) {
          const int src = io.mirror ? (e < io.mirror ? e : 2 * (io.mirror - 1) - e)
                                    : (e < io.ld_lo ? e : (e >= io.ld_hi ? e - io.ld_shift : -1));
          const bool ok = valid && src >= 0;
          const cpx<T> u = ld_at<T, Off>(io.in, ok ? (Off)io.lane_in + (Off)src * (Off)io.sl_in : (Off)0);
          v[m][r] = ok ? u : mk<T>(0, 0);
        } else {
          const cpx<T> u = ld_at<T, Off>(io.in, valid ? (Off)io.lane_in + (Off)e * (Off)io.sl_in : (Off)0);
          v[m][r] = valid ? u : mk<T>(0, 0);
        }
      }
    }
  }
#pragma unroll
  for (int m = 0; m < S::IT; m++) {
    const int it = threadIdx.x + m * NT;
    if ((S::total % NT) == 0 || it < S::total) {
      const int j = it / B, b = it % B;
      dft<R, FWD>(v[m]);
#pragma unroll
      for (int r = 0; r < R; r++) lds[lds_at<B, BP>(j * R + r, b)] = v[m][r];
    }
  }
  pre();
  __syncthreads();
}

// last stage: Ns * R == N, so every butterfly index j < Ns and k == j.  CL:
// lanes past the last column repeat it and store its values again, so that no
// store sits under a branch
template <class T, int R, bool FWD, int N, int B, int BP, int NT, int Ns, int TwOff, bool PR, class Off, bool CL>
__device__ __forceinline__ void stageL_global(const cpx<T>* lds, const typename TwT<T>::type* tw,
                                              const ColIO& io, int tid) {
  static_assert(Ns * R == N, "last stage");
  static_assert(NT % B == 0, "one column per thread");
  constexpr bool TB = is_tab<Off>;
  constexpr int total = B * Ns;
  constexpr int IT = (total + NT - 1) / NT;
  const bool valid = CL || (int)(tid % B) < io.nb;
#pragma unroll
  for (int m = 0; m < IT; m++) {
    const int it = tid + m * NT;
    if ((total % NT) == 0 || it < total) {
      const int j = it / B, b = it % B;
      cpx<T> v[R];
#pragma unroll
      for (int r = 0; r < R; r++) v[r] = lds[lds_at<B, BP>(j + r * Ns, b)];
      const typename TwT<T>::type* w = tw + TwOff + j * (R - 1);
#pragma unroll
      for (int r = 1; r < R; r++) v[r] = twmul<FWD>(v[r], w[r - 1]);
      dft<R, FWD>(v);
      // table-addressed rows: every entry and address first, so the table
      // reads issue together instead of one read and wait per store
      unsigned el[TB ? R : 1];
      bool st[TB ? R : 1];
      if constexpr (TB) {
#pragma unroll
        for (int r = 0; r < R; r++) {
          const int2 t = io.stab[j + r * Ns];
          el[r] = (unsigned)t.x + io.lane_o * (unsigned)t.y + io.lane_i;
          st[r] = std::is_same<Off, TabAll>::value || t.x >= 0;
        }
      }
      if (valid) {
#pragma unroll
        for (int r = 0; r < R; r++) {
          const int p = j + r * Ns;
          if constexpr (std::is_same<Off, TabSep>::value) {
            st_at<T, unsigned>(io.out, (unsigned)io.lane_out + io.sa_out[m] + io.sb_out[r], v[r]);
          } else if constexpr (TB) {
            if (st[r]) ((cpx<T>*)io.out)[el[r]] = v[r];
          } else if constexpr (PR) {
            const int e = p < io.st_lo ? p : p - io.st_shift;
            if (p < io.st_lo || (p >= io.st_lo + io.st_shift && e < io.nst))
              st_at<T, Off>(io.out, (Off)io.lane_out + (Off)e * (Off)io.sl_out, v[r]);
          } else {
            st_at<T, Off>(io.out, (Off)io.lane_out + (Off)p * (Off)io.sl_out, v[r]);
          }
        }
      }
    }
  }
}

// the stages from Ns on, the last one stored; IP: in place (after a first
// stage with RowRev), else autosort
template <class T, bool FWD, int N, int B, int BP, int NT, int Ns, int TwOff, bool PR, class Off, bool IP, bool CL,
          int R, int... Rest>
__device__ __forceinline__ void mid_and_last(cpx<T>* lds, const typename TwT<T>::type* tw, const ColIO& io,
                                             int tid = threadIdx.x) {
  if constexpr (sizeof...(Rest) == 0) {
    stageL_global<T, R, FWD, N, B, BP, NT, Ns, TwOff, PR, Off, CL>(lds, tw, io, tid);
  } else {
    if constexpr (IP) stage_ip<T, R, FWD, N, B, BP, NT, Ns, TwOff>(lds, tw, tid);
    else stage_ct<T, R, FWD, N, B, BP, NT, Ns, TwOff>(lds, tw);
    mid_and_last<T, FWD, N, B, BP, NT, Ns * R, (Ns > 1 ? TwOff + Ns * (R - 1) : TwOff), PR, Off, IP, CL, Rest...>(
        lds, tw, io, tid);
  }
}

template <class T, bool FWD, int B, int NT, bool PR, class Off, class Tw, int R0, int... Rs>
__device__ __forceinline__ void run_fft_io(cpx<T>* lds, const Tw& ctw, const ColIO& io, RList<R0, Rs...>) {
  static_assert(sizeof...(Rs) >= 1, "at least two stages");
  constexpr int N = R0 * RProd<Rs...>::value;
  stage0_global<T, R0, FWD, N, B, NT, PR, Off, RowRev<Rs...>>(lds, io, [&] { ctw.put(); });
  mid_and_last<T, FWD, N, B, B, NT, R0, 0, PR, Off, true, false, Rs...>(lds, ctw.table(), io);
}

// run_fft_io over the tiles t0, t0 + dt, ... below t1 of one workgroup: the
// next tile's first-stage loads are issued before the current tile's later
// stages and its stores, so they are in flight while those run.  The loop is
// turned so that the wait for them stands behind the stores in straight-line
// code: the memory counter retires in order, so it then waits for the loads
// only and the stores drain during the next tile.  make_io(t) gives tile t's
// addressing (lanes past the last column clamped).
template <class T, bool FWD, int B, int NT, class Off, class Tw, class MakeIO, int R0, int... Rs>
__device__ __forceinline__ void run_fft_io_pipe(cpx<T>* lds, const Tw& ctw, int t0, int t1, int dt, MakeIO make_io,
                                                RList<R0, Rs...>) {
  static_assert(sizeof...(Rs) >= 1, "at least two stages");
  constexpr int N = R0 * RProd<Rs...>::value;
  if (t0 >= t1) return;
  Stage0Regs<T, R0, N, B, NT> rg;
  ColIO io = make_io(t0);
  int tid = threadIdx.x;
  stage0_load<T, R0, N, B, NT, Off, RowRev<Rs...>>(rg, io, tid);
  ctw.put();
  const auto* tw = ctw.table();
  stage0_put<T, R0, FWD, N, B, NT>(lds, rg, tid);
  for (int t = t0 + dt; t < t1; t += dt) {
    // the thread index is opaque in the loop: hoisted out of it, the LDS and
    // row addresses take the registers the loads in flight need
    asm volatile("" : "+v"(tid));
    __builtin_assume(tid >= 0 && tid < NT);
    const ColIO nx = make_io(t);
    stage0_load<T, R0, N, B, NT, Off, RowRev<Rs...>>(rg, nx, tid);
    // the scheduler would sink the loads to save registers, and lift the first
    // butterflies (and their wait for the loads) above the later stages
    __builtin_amdgcn_sched_barrier(0);
    mid_and_last<T, FWD, N, B, B, NT, R0, 0, false, Off, true, true, Rs...>(lds, tw, io, tid);
    // the last stage's LDS reads before the next tile's first-stage writes
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
    stage0_put<T, R0, FWD, N, B, NT>(lds, rg, tid);
    io = nx;
  }
  mid_and_last<T, FWD, N, B, B, NT, R0, 0, false, Off, true, true, Rs...>(lds, tw, io, tid);
}

// Forward FFT of a tile whose first stage is fed from global memory (with
// the PR row maps, e.g. a DCT-I mirror) and whose result stays in the LDS
// tile (natural order, element e of column b at lds[e*B + b]).
template <class T, int B, int NT, class Off, class Tw, int R0, int... Rs>
__device__ __forceinline__ void run_fft_in_io(cpx<T>* lds, const Tw& ctw, const ColIO& io, RList<R0, Rs...>) {
  static_assert(sizeof...(Rs) >= 1, "at least two stages");
  constexpr int N = R0 * RProd<Rs...>::value;
  stage0_global<T, R0, true, N, B, NT, true, Off, RowRev<Rs...>>(lds, io, [&] { ctw.put(); });
  stages_ip<T, true, N, B, B, NT, R0, 0, Rs...>(lds, ctw.table());
}

// Table-addressed rows (Off = TabRows or TabAll) with the row tables staged in LDS at
// `tl` (n int2): the load table before the first stage, the store table
// after it, so every table read is an LDS read.
template <class T, bool FWD, int B, int NT, class Off, class Tw, int R0, int... Rs>
__device__ __forceinline__ void run_fft_io_tab(cpx<T>* lds, int2* tl, const Tw& ctw, ColIO io, const int2* ltab,
                                               const int2* stab, RList<R0, Rs...>) {
  static_assert(sizeof...(Rs) >= 1, "at least two stages");
  constexpr int N = R0 * RProd<Rs...>::value;
  for (int i = threadIdx.x; i < N; i += NT) tl[i] = ltab[i];
  __syncthreads();
  io.ltab = tl;
  stage0_global<T, R0, FWD, N, B, NT, false, Off, RowRev<Rs...>>(lds, io, [&] { ctw.put(); });
  for (int i = threadIdx.x; i < N; i += NT) tl[i] = stab[i];
  __syncthreads();
  io.stab = tl;
  mid_and_last<T, FWD, N, B, B, NT, R0, 0, false, Off, true, false, Rs...>(lds, ctw.table(), io);
}

// Spectral solve along the column: forward FFT, per-mode multiply by
// -scale/|k|^2 (k=0 -> 0), inverse FFT, all in one LDS tile.  Column i0 + b
// of the tile is kx + nxh * ky_index; the row is the kz index.  The inverse
// runs the forward stages backwards (decimation in frequency), so the last
// forward butterfly, the multiply and the first inverse butterfly are one pass
// over the same positions, and the last inverse stage stores the rows: 2 S - 2
// passes through the tile with a barrier each for S radices, against a forward
// transform, a multiply pass and an autosort inverse.  Bound by the latencies of
// that chain: the five lengths of 64 FP32 solves with axes 32 to 128 took 9.5,
// 13.6, 9.3, 12.4, 19.0 us, now 8.4, 12.1, 8.5, 11.9, 17.6 us.
struct SolveCtx {
  int nxh, ny, nz;
  double scale;
};

template <class T, int N, int B, int NT, int Ns, int Off, int R, int... Rest>
__device__ __forceinline__ void solve_mid(cpx<T>* lds, const typename TwT<T>::type* tw, long long i0,
                                          const SolveCtx& sc) {
  static_assert(NT % B == 0, "one column per thread");
  constexpr bool LAST = sizeof...(Rest) == 0;
  if constexpr (!LAST) {
    stage_ip<T, R, true, N, B, B, NT, Ns, Off>(lds, tw);
    solve_mid<T, N, B, NT, Ns * R, Off + Ns * (R - 1), Rest...>(lds, tw, i0, sc);
  }
  double kxy = 0;
  if constexpr (LAST) {
    const unsigned i = (unsigned)i0 + threadIdx.x % B;  // below 2^31 + B
    const int y = (int)(i / (unsigned)sc.nxh), kx = (int)(i - (unsigned)y * (unsigned)sc.nxh);
    const double ky = y <= sc.ny / 2 ? y : y - sc.ny;
    kxy = (double)kx * kx + ky * ky;
  }
  constexpr int total = B * (N / R), IT = (total + NT - 1) / NT;
#pragma unroll
  for (int m = 0; m < IT; m++) {
    const int it = threadIdx.x + m * NT;
    if ((total % NT) == 0 || it < total) {
      const int j = it / B, b = it % B;
      const int k = j % Ns, base = (j - k) * R + k;
      cpx<T> v[R];
#pragma unroll
      for (int r = 0; r < R; r++) v[r] = lds[(base + r * Ns) * B + b];
      const typename TwT<T>::type* w = tw + Off + k * (R - 1);
      if constexpr (LAST) {
#pragma unroll
        for (int r = 1; r < R; r++) v[r] = twmul<true>(v[r], w[r - 1]);
        dft<R, true>(v);
#pragma unroll
        for (int r = 0; r < R; r++) {
          const int e = base + r * Ns;
          const double kz = e <= sc.nz / 2 ? e : e - sc.nz;
          const double k2 = kxy + kz * kz;
          const double f = k2 > 0.0 ? -sc.scale / k2 : 0.0;
          v[r] = mk<T>((T)(v[r].x * f), (T)(v[r].y * f));
        }
      }
      dft<R, false>(v);
#pragma unroll
      for (int r = 1; r < R; r++) v[r] = twmul<false>(v[r], w[r - 1]);
#pragma unroll
      for (int r = 0; r < R; r++) lds[(base + r * Ns) * B + b] = v[r];
    }
  }
  __syncthreads();
}

template <class T, int B, int NT, class Tw, int R0, int... Rs>
__device__ __forceinline__ void run_fft_solve(cpx<T>* lds, const Tw& ctw, const ColIO& io, long long i0,
                                              const SolveCtx& sc, RList<R0, Rs...>) {
  static_assert(sizeof...(Rs) >= 1, "at least two stages");
  constexpr int N = R0 * RProd<Rs...>::value, nR = N / R0;
  stage0_global<T, R0, true, N, B, NT, false, unsigned, RowRev<Rs...>>(lds, io, [&] { ctw.put(); });
  solve_mid<T, N, B, NT, R0, 0, Rs...>(lds, ctw.table(), i0, sc);
  constexpr int total = B * nR, IT = (total + NT - 1) / NT;
  const bool valid = (int)(threadIdx.x % B) < io.nb;
#pragma unroll
  for (int m = 0; m < IT; m++) {
    const int it = threadIdx.x + m * NT;
    if ((total % NT) == 0 || it < total) {
      const int j = it / B, b = it % B;
      cpx<T> v[R0];
#pragma unroll
      for (int r = 0; r < R0; r++) v[r] = lds[(j * R0 + r) * B + b];
      dft<R0, false>(v);
      const int e = RowRev<Rs...>::at(j);
      if (valid) {
#pragma unroll
        for (int r = 0; r < R0; r++)
          st_at<T, unsigned>(io.out, (unsigned)io.lane_out + (unsigned)(e + r * nR) * (unsigned)io.sl_out, v[r]);
      }
    }
  }
}

// Columns whose input (IN) or output is length-fastest, the other side being
// rows, through a tile with rotated rows (a padded one costs the FP64 lengths
// 256 and 1024 a workgroup per CU: 256^3 82.4 us against 74.6 us of the kernel
// that met bank conflicts).  colb[b]:
// byte offset of column b of the length-fastest side from the tile's first.
template <class T, bool FWD, int B, int NT, bool IN, class Tw, int R0, int... Rs>
__device__ __forceinline__ void run_fft_lenfast(cpx<T>* lds, const Tw& ctw, const ColIO& io,
                                                const unsigned long long* colb, RList<R0, Rs...>) {
  static_assert(sizeof...(Rs) >= 1, "at least two stages");
  constexpr int N = R0 * RProd<Rs...>::value, BP = 0;
  constexpr int LI = (B * N + NT - 1) / NT;
  if constexpr (IN) {
    cpx<T> v[LI];
#pragma unroll
    for (int u = 0; u < LI; u++) {
      const int q = threadIdx.x + u * NT, b = q / N, e = q % N;
      const int src = e < io.ld_lo ? e : (e >= io.ld_hi ? e - io.ld_shift : -1);
      const bool ok = ((B * N) % NT == 0 || q < B * N) && b < io.nb && src >= 0;
      // items outside the tile load its first element (always valid) and are
      // zeroed, so no load sits under a branch
      const cpx<T> t = *(const cpx<T>*)(io.in + (ok ? colb[b] + (unsigned)src * (unsigned)sizeof(cpx<T>) : 0ull));
      v[u] = ok ? t : mk<T>(0, 0);
    }
#pragma unroll
    for (int u = 0; u < LI; u++) {
      const int q = threadIdx.x + u * NT;
      if ((B * N) % NT == 0 || q < B * N) lds[lds_at<B, BP>(q % N, q / N)] = v[u];
    }
    ctw.put();
    __syncthreads();
    mid_and_last<T, FWD, N, B, BP, NT, 1, 0, false, unsigned, false, false, R0, Rs...>(lds, ctw.table(), io);
  } else {
    stage0_global<T, R0, FWD, N, B, NT, false, unsigned, RowRev<Rs...>, BP>(lds, io, [&] { ctw.put(); });
    stages_ip<T, FWD, N, B, BP, NT, R0, 0, Rs...>(lds, ctw.table());
#pragma unroll
    for (int u = 0; u < LI; u++) {
      const int q = threadIdx.x + u * NT, b = q / N, p = q % N;
      const int e = p < io.st_lo ? p : p - io.st_shift;
      const bool kept = p < io.st_lo || (p >= io.st_lo + io.st_shift && e < io.nst);
      if (((B * N) % NT == 0 || q < B * N) && b < io.nb && kept)
        *(cpx<T>*)(io.out + (colb[b] + (unsigned)e * (unsigned)sizeof(cpx<T>))) = lds[lds_at<B, BP>(p, b)];
    }
  }
}

}  // namespace p3amd

namespace p3amd {
template <class RL>
struct RL_N;
template <int... Rs>
struct RL_N<RList<Rs...>> {
  static constexpr int value = RProd<Rs...>::value;
};
}  // namespace p3amd
