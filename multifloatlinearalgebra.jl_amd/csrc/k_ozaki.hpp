// Host-side interface of the Ozaki-split INT8 MFMA products (k_ozaki.hip).
#pragma once
#include "mf_common.hpp"

namespace mfk {

// Digits per operand for an N-limb result: of 7 bits (34 for Float64x4), and
// gemm!'s for a reduction of (padded) length K, of 8 bits up to 4096 (30).
int oz_digits(int N);
int oz_gemm_digits(int N, int64_t K);
int oz_chunks();
// digit rows are padded to a multiple of this many bytes
int oz_row_align();
// e[i] = ilogb(max_k |hi(X(i, k))|) + 3 (or a zero-row sentinel); part:
// oz_chunks() * m doubles of scratch. uplo 0 general, 1 / 2: X symmetric
// stored in its lower / upper triangle.
hipError_t oz_exponents(hipStream_t s, int64_t m, int64_t K, const DV &X, int uplo, int *e, double *part);
// S balanced digits (a count of oz_digits or oz_gemm_digits, of B = 7 or 8
// bits) of X(i, k) 2^(BS - e_i) in the fragment layout
// (16-row blocks of 64-deep k steps of S 1 KB fragments: oz_bytes(m, ld, S)
// bytes), ld a multiple of 64 >= K (padding digits zero).
int64_t oz_bytes(int64_t m, int64_t ld, int S);
hipError_t oz_split(int N, hipStream_t s, int64_t m, int64_t K, const DV &X, int uplo, const int *e, int S, int8_t *dig, int64_t ld);
// Rounds the binary64 columns D(:, j) in place to 7T-bit fixed point (scale
// 2^(e_j - 7T)) and writes their T digits dig[t*plane + j*ld + k].
hipError_t oz_round_fp64(hipStream_t s, int64_t K, int64_t ncols, const DV &D, const int *e, int T, int8_t *dig, int64_t ld,
                         int64_t plane);
// C = alpha*A*B (+ beta*C unless beta_zero): sum over digit pairs s + t <= S
// of 2^(ea_i + eb_j - B(s + t + 2)) sum_k dA_s(i, k) dB_t(j, k) in N limbs, dA
// and dB the S = oz_gemm_digits(N, K) digits of A's rows and B's columns. K =
// the ld of the splits (<= 8192).
hipError_t oz_gemm(int N, hipStream_t s, int64_t m, int64_t n, int64_t K, int S, const int8_t *dA, const int8_t *dB, const int *ea,
                   const int *eb, const DV &C, const double *alpha, const double *beta, int beta_zero);
// out[u][j][i] (int32, m x n column-major per u) = sum over digit pairs s + t
// = u of sum_k dA_s(i, k) dB_t(j, k), u = 0 .. SA + oz_narrow_digits() - 2: A's
// digits in the fragment layout (K = the ld of the split), B with
// oz_narrow_digits() digits: the refinement's product A * D.
int oz_narrow_digits();
hipError_t oz_gemm_narrow(hipStream_t s, int64_t m, int64_t n, int64_t K, const int8_t *dA, int SA, const int8_t *dB, int64_t ldb,
                          int64_t planeB, int32_t *out);
// C -= sum_u planes[u] 2^(ea_i + eb_j - 7(u + 2)) in N limbs (u ascending)
hipError_t oz_combine(int N, hipStream_t s, int64_t m, int64_t n, int U, const int32_t *planes, const int *ea, const int *eb,
                      const DV &C);

}  // namespace mfk
