// engine_gen.hpp -- transforms of any length up to max_len() whose radix
// schedule is a run-time value (lengths without compile-time specialised
// kernels); the kernels are in engine_gen.hip.
#pragma once
#include "engine.hpp"

namespace p3amd {

// the radix schedule of a length: factors of at most kGenMaxRadix where the
// length has such a form, a larger prime otherwise stands between two factors
// (1 if there is none), since the first and the last stage hold a whole
// butterfly in registers
std::vector<int> gen_factors(int n);
// the same for factors in a given order (a plan-time candidate)
std::vector<int> gen_wrap(const std::vector<int>& f);
// the largest radix held in registers: with radices up to 16 the kernels with
// row maps need 544 to 880 bytes of scratch per lane, with 10 none (the FP64
// kernels with a length-fastest side 68 bytes, spilled scalar registers)
constexpr int kGenMaxRadix = 10;
inline bool gen_in_registers(int r) { return r <= kGenMaxRadix; }
// a prime radix above that (the specialised schedules also hold 16), never first
// or last; up to kGenRegPrime the pairs of a butterfly sit in registers, above
// they are summed over LDS
constexpr int kGenRegPrime = 13;
inline bool gen_is_prime_stage(int r) { return r > kGenMaxRadix && r % 2 == 1; }
inline bool gen_over_lds(int r) { return r > kGenRegPrime && r % 2 == 1; }

// the launchers of engine.hpp for these kernels
void gen_launch_x_r2c(const Len1D& L, const real_t* in, cplx_t* out, long long nrows, long long si_row,
                      long long so_row, int nxo, bool rev, hipStream_t st);
void gen_launch_x_c2r(const Len1D& L, const cplx_t* in, real_t* out, long long nrows, long long si_row,
                      long long so_row, int nxi, bool rev, hipStream_t st);
// L: the plan of the transform length (null: COL_COPY); wide: 64-bit offsets
// even where 32-bit ones fit
void gen_launch_col(const Len1D* L, const ColSpec& c, int xcd, bool wide, hipStream_t st);
// the launch shape of a schedule (host only): sequences per tile, threads (0:
// no count holds the tile) and LDS bytes of `count` columns (form 0 rows on both
// sides, 1 a length-fastest side; 3 and 4 the same of copied rows) or rows along X
// (form 2), and the width of the offsets into such contiguous columns or rows
void gen_tile_shape(const LenDesc& d, int form, long long count, int tile_bytes, int seg, bool wide, int* seqs,
                    int* threads, size_t* lds, int* offset_bytes);
// raise the kernels' dynamic-LDS limits (once, when a length is planned)
void gen_prep_kernels();

}  // namespace p3amd
