// Ozaki-split products on the INT8 matrix cores (v_mfma_i32_16x16x64_i8).
//
// A Float64xN operand row (or column) is scaled by a power of two 2^e with
// |value| < 2^(e-2) over the row, converted exactly (up to truncation below
// 2^(e - BS)) to a two's complement fixed-point integer Z of BS bits, and
// split into S balanced digits d_s of B bits in [-2^(B-1), 2^(B-1) - 1] (most
// significant first):   value ~ 2^(e - BS) * Z,   Z = sum_s d_s 2^(B(S-1-s)).
// Then
//   sum_k A(i,k) B(k,j) = sum_{s,t} 2^(ea_i + eb_j - B(s+t+2)) C_{s,t}(i,j),
//   C_{s,t}(i,j) = sum_k dA_s(i,k) dB_t(j,k)          (exact int32)
// Digit products are at most 2^(2B-2) in magnitude, so a group of P pairs over
// K terms stays below 2^31 for B = 7 up to K = 8192 (P <= 34), for B = 8 up to
// K = 4096 (P <= 30). Eight bits need a fifth fewer digit pairs (x4: 30 digits
// of 8 bits hold 240 bits, 34 of 7 hold 238), so gemm! takes them up to K =
// 4096; the refinement's A * D keeps 7.
//
//  * k_oz_exp_part / k_oz_exp_finish: e_i = ilogb(max_k |hi(X(i,k))|) + 3
//    (chunked max, fixed order), or a sentinel for all-zero rows.
//  * k_oz_split<N>: the exact fixed-point conversion (each limb's 53-bit
//    mantissa shifted into a 256-bit two's complement accumulator, truncated
//    toward zero) and the balanced digit extraction.
//  * k_oz_round_fp64: a binary64 correction rounded to 7T-bit fixed point per
//    column (the rounded value is written back, so the caller uses exactly
//    the value whose digits are multiplied) and split into T digits.
//  * k_oz_gemm: C = alpha*A*B + beta*C; every wave keeps the sums C_u of all
//    u in [0, S] of one 16 x 16 block in registers and recombines them itself.
//  * k_oz_gemm_narrow / k_oz_combine<N>: the refinement's A * D as int32
//    planes C_u, then R = R - acc.
//  Recombination: acc(i,j) = sum_u C_u(i,j) 2^(ea_i + eb_j - 7(u+2)) in
//    Float64xN arithmetic, u ascending, four sums at a time (exact in 53 bits).
#include <climits>
#include <type_traits>
#include "mf_common.hpp"
#include "k_ozaki.hpp"

namespace mfk {

constexpr int OZ_CHUNKS = 32;
constexpr int OZ_ZERO_ROW = INT_MIN / 2;

// ------------------------------------------------------------ exponents
// view X(i, k): rows i in [0, m), k in [0, K); part[c * m + i] = max over
// chunk c of |hi(X(i, k))|.
// uplo 1 / 2: X is symmetric and only its lower / upper triangle is read.
__device__ __forceinline__ const double *oz_at(const DV &X, int uplo, int64_t i, int64_t k) {
    if ((uplo == 1 && i < k) || (uplo == 2 && i > k)) { const int64_t q = i; i = k; k = q; }
    return X.p + i * X.rs + k * X.cs;
}

__global__ void k_oz_exp_part(int64_t m, int64_t K, DV X, int uplo, double *part) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= m) return;
    const int64_t c = blockIdx.y, per = (K + OZ_CHUNKS - 1) / OZ_CHUNKS;
    const int64_t klo = c * per, khi = (klo + per < K) ? klo + per : K;
    double mx = 0.0;
    for (int64_t k = klo; k < khi; ++k) mx = fmax(mx, fabs(*oz_at(X, uplo, i, k)));
    part[c * m + i] = mx;
}

__global__ void k_oz_exp_finish(int64_t m, const double *part, int *e) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= m) return;
    double mx = 0.0;
    for (int c = 0; c < OZ_CHUNKS; ++c) mx = fmax(mx, part[c * m + i]);
    e[i] = (mx > 0.0 && __builtin_isfinite(mx)) ? ilogb(mx) + 3 : OZ_ZERO_ROW;
}

// ------------------------------------------------------ fixed point
// 256-bit two's complement accumulator, little-endian 64-bit words.
struct Acc256 {
    uint64_t w[4];
};

__device__ __forceinline__ void acc_add_shifted(Acc256 &a, uint64_t mag, int sh, bool neg) {
    // value = (neg ? -1 : 1) * floor-toward-zero(mag * 2^sh), |result| < 2^255
    uint64_t t[4] = {0, 0, 0, 0};
    if (sh >= 0) {
        const int wq = sh >> 6, bq = sh & 63;
        if (wq < 4) {
            t[wq] = mag << bq;
            if (bq != 0 && wq + 1 < 4) t[wq + 1] = mag >> (64 - bq);
        }
    } else {
        const int r = -sh;
        t[0] = r >= 64 ? 0 : (mag >> r);
    }
    if (neg) {   // two's complement negation of t
        uint64_t carry = 1;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint64_t v = ~t[q] + carry;
            carry = (carry && v == 0) ? 1 : 0;
            t[q] = v;
        }
    }
    uint64_t carry = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const uint64_t s1 = a.w[q] + t[q];
        const uint64_t c1 = s1 < a.w[q] ? 1 : 0;
        const uint64_t s2 = s1 + carry;
        const uint64_t c2 = s2 < s1 ? 1 : 0;
        a.w[q] = s2;
        carry = c1 | c2;
    }
}

// The S digits of B bits of a value held in a 256-bit accumulator, balanced,
// least significant first into d[S-1], ..., most significant into d[0]. S
// and B are constants, so every word index and shift is static.
template <int S, int B>
__device__ __forceinline__ void acc_digits(const Acc256 &a, int8_t *d, int64_t stride) {
    static_assert(B * S <= 250, "the accumulator holds the digits");
    constexpr int BASE = 1 << B;
    int carry = 0;
#pragma unroll
    for (int q = 0; q < S; ++q) {
        const int bit = B * q;
        const int wq = bit >> 6, bq = bit & 63;
        uint64_t chunk = a.w[wq] >> bq;
        if (bq > 64 - B && wq + 1 < 4) chunk |= a.w[wq + 1] << (64 - bq);
        int b = (int)(chunk & (BASE - 1)) + carry;
        int dig;
        if (b >= BASE / 2) { dig = b - BASE; carry = 1; } else { dig = b; carry = 0; }
        d[(int64_t)(S - 1 - q) * stride] = (int8_t)dig;
    }
}

// Digits of X(i, k) as MFMA fragments: 16-row blocks, each a sequence of
// 64-deep k steps, each the S digits' 16x16x64 fragments of 1 KB, laid out
// exactly as the lanes of a wave read one (lane l = 16 * (k % 64 / 16) + i %
// 16 takes 16 consecutive k). A wave's load is one contiguous 1 KB and the
// digits it multiplies together are adjacent. Offset of digit 0:
constexpr int64_t OZ_FRAG = 1024;
__device__ __forceinline__ int64_t oz_off(int64_t i, int64_t k, int64_t ld, int S) {
    return ((i >> 4) * (ld >> 6) + (k >> 6)) * S * OZ_FRAG + ((((k & 63) >> 4) << 4) + (i & 15)) * 16 + (k & 15);
}

// digits s = 0..S-1 of X(i, k); the padding columns k in [K, ld) get zero
// digits, the rows that fill the last block of 16 are left as they are (they
// reach only outputs that are not stored).
template <int N, int S, int B>
__global__ void k_oz_split(int64_t m, int64_t K, DV X, int uplo, const int *e, int8_t *dig, int64_t ld) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= m * ld) return;
    const int64_t k = idx % ld, i = idx / ld;        // k fastest: coalesced digit stores
    int8_t *d = dig + oz_off(i, k, ld, S);
    const int ei = e[i];
    Acc256 a{{0, 0, 0, 0}};
    if (ei != OZ_ZERO_ROW && k < K) {
        const double *p = oz_at(X, uplo, i, k);
#pragma unroll
        for (int l = 0; l < N; ++l) {
            const double x = p[l * X.ls];
            if (x == 0.0 || !__builtin_isfinite(x)) continue;
            int ex;
            const double f = frexp(fabs(x), &ex);                 // |x| = f 2^ex, f in [0.5, 1)
            const uint64_t mag = (uint64_t)ldexp(f, 53);            // 53-bit integer mantissa
            acc_add_shifted(a, mag, ex - 53 + B * S - ei, x < 0.0);
        }
    }
    acc_digits<S, B>(a, d, OZ_FRAG);
}

// binary64 correction D(k, j) (k in [0, K), column j): per-column exponent
// e_j from the column max; D(k, j) <- round(D 2^(7T - e_j)) 2^(e_j - 7T), and
// its T digits into dig[t * plane + j * ld + k].
__global__ void k_oz_round_fp64(int64_t K, int64_t ncols, DV D, const int *e, int T, int8_t *dig, int64_t ld, int64_t plane) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= ld * ncols) return;
    const int64_t k = idx % ld, j = idx / ld;
    if (k >= K) {                                   // zero padding digits
        for (int t = 0; t < T; ++t) dig[(int64_t)t * plane + j * ld + k] = 0;
        return;
    }
    double *p = D.p + k * D.rs + j * D.cs;
    const int ej = e[j];
    int64_t q = 0;
    if (ej != OZ_ZERO_ROW && __builtin_isfinite(*p)) {
        q = (int64_t)rint(ldexp(*p, 7 * T - ej));                 // |q| < 2^(7T - 2)
        *p = ldexp((double)q, ej - 7 * T);
    } else {
        *p = 0.0;
    }
    int carry = 0;
    const uint64_t u = (uint64_t)q;
    for (int t = 0; t < T; ++t) {
        int b = (int)((u >> (7 * t)) & 127) + carry;
        int dg;
        if (b >= 64) { dg = b - 128; carry = 1; } else { dg = b; carry = 0; }
        dig[(int64_t)(T - 1 - t) * plane + j * ld + k] = (int8_t)dg;
    }
}

// ----------------------------------------------------------- INT8 GEMM
typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int OZ_NARROW_TB = 6;   // B digits of the narrow kernel (binary64 corrections)

// Sums of U + 1 digit planes (B-bit digits) to Float64xN: c(u) weighs
// 2^(base - B(u + 2)). As many consecutive planes as stay below 2^53 together
// (|c| < 2^31) are one integer, so they enter the Float64xN sum exactly and
// as one binary64 value.
template <int N, int B, typename C> __device__ __forceinline__ mf::V<N> oz_sum(int U, int base, const C &c) {
    constexpr int G = 1 + 21 / B;
    mf::V<N> acc = mf::zero<N>();
    int u = 0;
#pragma unroll
    for (; u + G - 1 <= U; u += G) {
        int64_t v = c(u);
#pragma unroll
        for (int g = 1; g < G; ++g) v = (v << B) + c(u + g);
        acc = mf::add(acc, mf::from<N>(ldexp((double)v, base - B * (u + G + 1))));
    }
#pragma unroll
    for (; u <= U; ++u) acc = mf::add(acc, mf::from<N>(ldexp((double)c(u), base - B * (u + 2))));
    return acc;
}

// C = alpha*A*B + beta*C from the digits of A's rows and B's columns (both in
// the fragment layout, S digits each, `steps` k steps). A wave computes WN
// 16 x 16 blocks side by side with the sums C_u of all u <= S in registers
// (S + 1 fragments of 4 each: 124 for S = 30) beside A's S fragments of a k
// step: the 60 KB of digits of a step feed (S + 1)(S + 2) / 2 - 2 = 494 MFMAs
// (7900 cycles), so the operands stream from L2 at 8 bytes a cycle and wave
// (6 with WN = 2) and need neither LDS nor barriers. (One plane u per pass over
// 128 x 128 LDS tiles read 128 bytes of LDS a cycle, its peak, for MFMAs that
// ran at 28 % of theirs, and wrote the planes out for another kernel to sum:
// whole gemm! x4 2048^3 7.82 ms, x3 4.97, x2 2.68; so 3.84, 2.42, 1.55, the
// x4 kernel at 2400 TOP/s where a large bf16 matrix product reaches 54 % of
// its nominal rate on the same card and this 48 % of 5.0 POP/s.)
// B's fragments run OZ_AHEAD ahead; a fragment of A is replaced by the next
// step's after its last MFMA, the first OZ_EARLY (whose last MFMAs end the
// step) are fetched into registers of their own.
// KS = 1: the four waves of a workgroup take a tile of 2 x 2 wave blocks.
// KS = 4: they share one and take every fourth k step each, add their sums
// (integers: any order) through LDS and finish every fourth column each.
template <int N, int B, int S, int KS, int WN, int OZ_AHEAD, int OZ_EARLY>
__global__ __launch_bounds__(256, 1) void k_oz_gemm(int64_t m, int64_t n, int steps, const int8_t *dA, const int8_t *dB, const int *ea,
                                                    const int *eb, DV C, mfk::S<N> alpha, mfk::S<N> beta, int beta_zero, int tiles_m, int tiles_n,
                                                    int per_xcd) {
    constexpr int U = S;
    static_assert(2 * OZ_EARLY <= S - 1 && OZ_AHEAD < S, "the prefetches stay within one step");
    constexpr int64_t STEP = S * OZ_FRAG;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    // workgroup b runs on XCD b % 8: each XCD takes a contiguous run of tiles,
    // enumerated in bands of 8 tile rows, so the ~32 tiles it holds at once
    // share rows and columns in its L2
    const int64_t tile = (int64_t)(blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (tile >= (int64_t)tiles_m * tiles_n) return;
    const int64_t band = tile / (8 * tiles_n), in = tile - band * 8 * tiles_n;
    const int64_t high = tiles_m - band * 8 < 8 ? tiles_m - band * 8 : 8;
    const int64_t bi = band * 8 + in % high, bj = in / high;
    const int64_t ib = KS == 1 ? bi * 2 + (w & 1) : bi, jb = (KS == 1 ? bj * 2 + (w >> 1) : bj) * WN;   // 16-row / 16-column blocks
    if (ib * 16 >= m || jb * 16 >= n) return;            // KS == 1 only: no barrier follows
    v4i acc[WN][U + 1];
#pragma unroll
    for (int h = 0; h < WN; ++h)
#pragma unroll
        for (int u = 0; u <= U; ++u) acc[h][u] = v4i{0, 0, 0, 0};
    const int first = KS == 1 ? 0 : w;
    if (first < steps) {
        static_assert(WN <= 2, "one block may be missing at the right edge");
        const int64_t bcol = (jb + 1) * 16 < n ? steps * STEP : 0;   // to the second column block, if B has one
        const int8_t *pa = dA + (ib * steps + first) * STEP + lane * 16, *pb = dB + (jb * steps + first) * STEP + lane * 16;
        auto frag = [](const int8_t *p, int s) { return *(const v4i *)(p + s * OZ_FRAG); };
        v4i fa[S], fb[WN][OZ_AHEAD], early[OZ_EARLY];
#pragma unroll
        for (int s = S - 1; s >= 0; --s) fa[s] = frag(pa, s);
#pragma unroll
        for (int q = 0; q < OZ_AHEAD; ++q)
#pragma unroll
            for (int h = 0; h < WN; ++h) fb[h][q] = frag(pb + h * bcol, q);
        for (int ks = first; ks < steps; ks += KS) {
            // the last step fetches its own fragments again instead of a step past the end
            const int8_t *na = ks + KS < steps ? pa + KS * STEP : pa, *nb = ks + KS < steps ? pb + KS * STEP : pb;
#pragma unroll
            for (int q = 0; q < S; ++q) {
                v4i b[WN];
#pragma unroll
                for (int h = 0; h < WN; ++h) {
                    b[h] = fb[h][0];
#pragma unroll
                    for (int x = 0; x + 1 < OZ_AHEAD; ++x) fb[h][x] = fb[h][x + 1];
                    fb[h][OZ_AHEAD - 1] = q + OZ_AHEAD < S ? frag(pb + h * bcol, q + OZ_AHEAD) : frag(nb + h * bcol, q + OZ_AHEAD - S);
                }
                if (q >= S - 1 - 2 * OZ_EARLY && q < S - 1 - OZ_EARLY) early[q - (S - 1 - 2 * OZ_EARLY)] = frag(na, q - (S - 1 - 2 * OZ_EARLY));
#pragma unroll
                for (int x = S - 1; x >= 0; --x)
#pragma unroll
                    for (int h = 0; h < WN; ++h)
                        if (x + q <= U) acc[h][x + q] = __builtin_amdgcn_mfma_i32_16x16x64_i8(b[h], fa[x], acc[h][x + q], 0, 0, 0);
                if (q >= 1 && U - q >= OZ_EARLY) fa[U - q] = frag(na, U - q);
            }
#pragma unroll
            for (int x = 0; x < OZ_EARLY; ++x) fa[x] = early[x];
            pa = na;
            pb = nb;
        }
    }
    const mf::V<N> al = sv(alpha), be = sv(beta);
    // item v of lane l: row l % 16, column 4 (l / 16) + v of the block
    const int64_t i = ib * 16 + (lane & 15);
    auto finish = [&](int h, int v, auto sums) {
        const int64_t j = (jb + h) * 16 + 4 * (lane >> 4) + v;
        if (i >= m || j >= n) return;
        const int xa = ea[i], xb = eb[j];
        const mf::V<N> p = xa == OZ_ZERO_ROW || xb == OZ_ZERO_ROW ? mf::zero<N>() : oz_sum<N, B>(U, xa + xb, sums);
        stv<N>(C, i, j, beta_zero ? mf::mul(al, p) : mf::add(mf::mul(al, p), mf::mul(be, ld<N>(C, i, j))));
    };
    if constexpr (KS == 1) {
#pragma unroll
        for (int h = 0; h < WN; ++h)
#pragma unroll
            for (int v = 0; v < 4; ++v) finish(h, v, [&](int u) { return acc[h][u][v]; });
    } else {
        __shared__ int32_t part[3][U + 1][64];
#pragma unroll
        for (int h = 0; h < WN; ++h) {
            int32_t mine[U + 1];
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                if (w != v) {
#pragma unroll
                    for (int u = 0; u <= U; ++u) part[w < v ? w : w - 1][u][lane] = acc[h][u][v];
                }
                __syncthreads();
                if (w == v) {
#pragma unroll
                    for (int u = 0; u <= U; ++u) mine[u] = acc[h][u][v] + part[0][u][lane] + part[1][u][lane] + part[2][u][lane];
                }
                __syncthreads();
            }
            finish(h, w, [&](int u) { return mine[u]; });
        }
    }
}

// Narrow products (the refinement's A * D: few columns, TB = 6 digits of a
// binary64 correction): every wave owns one 16 x 16 output block and keeps
// the partial sums of all SMAX + TB - 1 planes in registers, so each digit
// plane of A is streamed once per 64-column group. A's digits are in the
// fragment layout (one contiguous 1 KB load per wave and 64-deep k step);
// the TB digit rows of the wave's 16 columns are few and stay in L2. Per k
// step the wave loads its TB B fragments once and multiplies every A digit
// s into the planes s .. s + TB - 1. A workgroup is 16 rows x 64 columns
// (four waves side by side); grid.y runs over 64-column groups.
template <int SA, int TB>
__global__ __launch_bounds__(256) void k_oz_gemm_narrow(int64_t m, int64_t n, int64_t K, const int8_t *dA, const int8_t *dB, int64_t ldb, int64_t planeB, int32_t *out) {
    constexpr int NP = SA + TB - 1;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int64_t i0 = (int64_t)blockIdx.x * 16, j0 = (int64_t)blockIdx.y * 64 + (int64_t)w * 16;
    const int64_t ia = i0 + (lane & 15), jb = j0 + (lane & 15);
    const bool rowok = ia < m, colok = jb < n;
    // the fragment layout pads the rows to 16, so every A load is in bounds
    const int8_t *pa = dA + (int64_t)blockIdx.x * (K >> 6) * SA * OZ_FRAG + lane * 16;
    const int8_t *pb = dB + (colok ? jb : 0) * ldb + (lane >> 4) * 16;
    v4i acc[NP];
#pragma unroll
    for (int u = 0; u < NP; ++u) acc[u] = v4i{0, 0, 0, 0};
    // all A fragments of a k step in registers; each slot is reloaded for
    // the next step right after its MFMAs are issued
    v4i fa[SA], fb[TB];
#pragma unroll
    for (int s = 0; s < SA; ++s) fa[s] = *(const v4i *)(pa + s * OZ_FRAG);
#pragma unroll
    for (int q = 0; q < TB; ++q) fb[q] = *(const v4i *)(pb + q * planeB);
    const v4i zero{0, 0, 0, 0};
    for (int64_t k0 = 0; k0 < K; k0 += 64) {
        const bool more = k0 + 64 < K;
        const int8_t *pn = pa + ((k0 + 64) >> 6) * SA * OZ_FRAG;
        v4i gb[TB];
#pragma unroll
        for (int q = 0; q < TB; ++q) gb[q] = colok ? fb[q] : zero;
        if (more) {
#pragma unroll
            for (int q = 0; q < TB; ++q) fb[q] = *(const v4i *)(pb + q * planeB + k0 + 64);
        }
#pragma unroll
        for (int s = 0; s < SA; ++s) {
            const v4i a = fa[s];
#pragma unroll
            for (int q = 0; q < TB; ++q) acc[s + q] = __builtin_amdgcn_mfma_i32_16x16x64_i8(gb[q], a, acc[s + q], 0, 0, 0);
            if (more) fa[s] = *(const v4i *)(pn + s * OZ_FRAG);
        }
    }
    // item v of lane l: row (lane % 16), column 4 (lane / 16) + v of the block
#pragma unroll
    for (int u = 0; u < NP; ++u) {
        int32_t *o = out + (int64_t)u * m * n;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int64_t j = j0 + 4 * (lane >> 4) + v;
            if (rowok && j < n) o[j * m + ia] = acc[u][v];
        }
    }
}

// -------------------------------------------------------------- combine
// C -= sum_u C_u 2^(ea_i + eb_j - 7(u + 2)), u ascending, in N limbs (four
// planes an addition: 39 additions took 50 us for x4 4096 x 64, ten take
// 20)
template <int N>
__global__ void k_oz_combine(int64_t m, int64_t n, int U, const int32_t *planes, const int *ea, const int *eb, DV C) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= m * n) return;
    const int64_t i = idx % m, j = idx / m;
    mf::V<N> acc = mf::zero<N>();
    if (ea[i] != OZ_ZERO_ROW && eb[j] != OZ_ZERO_ROW)
        acc = oz_sum<N, 7>(U, ea[i] + eb[j], [&](int u) { return planes[(int64_t)u * m * n + j * m + i]; });
    stv<N>(C, i, j, mf::sub(ld<N>(C, i, j), acc));
}

// ---------------------------------------------------------- launchers
#define OZ_DISPATCH(N, ...)                                        \
    switch (N) {                                                   \
        case 1: { constexpr int NN = 1; __VA_ARGS__; } break;      \
        case 2: { constexpr int NN = 2; __VA_ARGS__; } break;      \
        case 3: { constexpr int NN = 3; __VA_ARGS__; } break;      \
        case 4: { constexpr int NN = 4; __VA_ARGS__; } break;      \
        default: return hipErrorInvalidValue;                      \
    }

template <int N> static S<N> mk_oz(const double *a) { S<N> s; for (int l = 0; l < N; ++l) s.x[l] = a ? a[l] : 0.0; return s; }

int oz_digits(int N) { return N >= 4 ? 34 : (N == 3 ? 27 : (N == 2 ? 19 : 11)); }
int oz_chunks() { return OZ_CHUNKS; }

hipError_t oz_exponents(hipStream_t s, int64_t m, int64_t K, const DV &X, int uplo, int *e, double *part) {
    if (m == 0) return hipSuccess;
    hipLaunchKernelGGL(k_oz_exp_part, dim3((unsigned)cdiv(m, 256), OZ_CHUNKS), dim3(256), 0, s, m, K, X, uplo, part);
    hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
    hipLaunchKernelGGL(k_oz_exp_finish, dim3((unsigned)cdiv(m, 256)), dim3(256), 0, s, m, part, e);
    return hipGetLastError();
}

int64_t oz_bytes(int64_t m, int64_t ld, int S) { return cdiv(m, 16) * 16 * ld * S; }

// gemm!'s digits: 8 bits while the int32 sums hold them
int oz_gemm_digits(int N, int64_t K) {
    if (K > 4096) return oz_digits(N);
    return N >= 4 ? 30 : (N == 3 ? 24 : (N == 2 ? 17 : 10));
}

hipError_t oz_split(int N, hipStream_t s, int64_t m, int64_t K, const DV &X, int uplo, const int *e, int S, int8_t *dig, int64_t ld) {
    if (m * ld == 0) return hipSuccess;
    if (ld % 64 != 0 || ld < K) return hipErrorInvalidValue;
    const dim3 grid((unsigned)cdiv(m * ld, 256));
#define OZ_SPLIT(SC, B) OZ_DISPATCH(N, hipLaunchKernelGGL((k_oz_split<NN, SC, B>), grid, dim3(256), 0, s, m, K, X, uplo, e, dig, ld))
    switch (S) {   // the digit counts of oz_digits and oz_gemm_digits
        case 11: OZ_SPLIT(11, 7); break;
        case 19: OZ_SPLIT(19, 7); break;
        case 27: OZ_SPLIT(27, 7); break;
        case 34: OZ_SPLIT(34, 7); break;
        case 10: OZ_SPLIT(10, 8); break;
        case 17: OZ_SPLIT(17, 8); break;
        case 24: OZ_SPLIT(24, 8); break;
        case 30: OZ_SPLIT(30, 8); break;
        default: return hipErrorInvalidValue;
    }
#undef OZ_SPLIT
    return hipGetLastError();
}

int oz_narrow_digits() { return OZ_NARROW_TB; }

hipError_t oz_gemm_narrow(hipStream_t s, int64_t m, int64_t n, int64_t K, const int8_t *dA, int SA, const int8_t *dB, int64_t ldb,
                          int64_t planeB, int32_t *out) {
    if (m == 0 || n == 0) return hipSuccess;
    if (K > 8192 || K % 64 != 0 || ldb % 16 != 0) return hipErrorInvalidValue;
    const dim3 grid((unsigned)cdiv(m, 16), (unsigned)cdiv(n, 64)), block(256);
    switch (SA) {   // the digit counts of oz_digits(N)
        case 34: hipLaunchKernelGGL((k_oz_gemm_narrow<34, OZ_NARROW_TB>), grid, block, 0, s, m, n, K, dA, dB, ldb, planeB, out); break;
        case 27: hipLaunchKernelGGL((k_oz_gemm_narrow<27, OZ_NARROW_TB>), grid, block, 0, s, m, n, K, dA, dB, ldb, planeB, out); break;
        case 19: hipLaunchKernelGGL((k_oz_gemm_narrow<19, OZ_NARROW_TB>), grid, block, 0, s, m, n, K, dA, dB, ldb, planeB, out); break;
        case 11: hipLaunchKernelGGL((k_oz_gemm_narrow<11, OZ_NARROW_TB>), grid, block, 0, s, m, n, K, dA, dB, ldb, planeB, out); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t oz_round_fp64(hipStream_t s, int64_t K, int64_t ncols, const DV &D, const int *e, int T, int8_t *dig, int64_t ld,
                         int64_t plane) {
    if (ld * ncols == 0) return hipSuccess;
    if (T < 1 || T > 8 || ld % 64 != 0 || ld < K) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_oz_round_fp64, dim3((unsigned)cdiv(ld * ncols, 256)), dim3(256), 0, s, K, ncols, D, e, T, dig, ld, plane);
    return hipGetLastError();
}

// Workgroup shapes, by the number of 16 x 16 blocks (the gemm kernel alone,
// 512^3 / 1024^3 / 2048^3 / 4096^3): four limbs share two blocks side by side
// from 4096 blocks on (0.086 / 0.495 / 3.54 / 28.3 ms), give each wave a block
// from 1024 on, one block for each SIMD (0.072 / 0.473 / 4.02 / 31.0), and
// share one block below (0.097 / 0.601 / 4.65 / 37.9, but four times the
// workgroups). Fewer limbs share one block at every size (x3 0.049 / 0.284 /
// 2.08 / 17.8 against 0.055 / 0.334 / 2.21 / 19.6 for two, x2 0.029 / 0.177 /
// 1.34 / 11.5 against 0.033 / 0.224 / 1.60 / 15.1). The four-limb two-block
// shape spills 19 registers, 80 bytes a lane, and is the faster one all the
// same; with two blocks of three limbs' 27 digits nothing spills, and A's digits
// are read half as often (whole gemm!, 512 x 8192 x 512 1.12 against 1.81 ms, 2000
// x 6000 x 1000 5.03 against 8.65, 4096 x 4160 x 4096 26.0 against 52.0; 300 x 5000
// x 70 0.383 against 0.380).
template <int N, int B, int S, int KS, int WN, int AHEAD, int EARLY>
static hipError_t oz_launch(hipStream_t s, int64_t m, int64_t n, int64_t K, const int8_t *dA, const int8_t *dB, const int *ea, const int *eb,
                            const DV &C, const double *alpha, const double *beta, int beta_zero) {
    const int64_t bm = cdiv(m, 16), bn = cdiv(n, 16 * WN);
    const int64_t tm = KS == 1 ? cdiv(bm, 2) : bm, tn = KS == 1 ? cdiv(bn, 2) : bn, per = cdiv(tm * tn, 8);
    if (per * 8 > INT32_MAX) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_oz_gemm<N, B, S, KS, WN, AHEAD, EARLY>), dim3((unsigned)(per * 8)), dim3(256), 0, s, m, n, (int)(K / 64), dA, dB, ea,
                       eb, C, mk_oz<N>(alpha), mk_oz<N>(beta), beta_zero, (int)tm, (int)tn, (int)per);
    return hipGetLastError();
}

hipError_t oz_gemm(int N, hipStream_t s, int64_t m, int64_t n, int64_t K, int S, const int8_t *dA, const int8_t *dB, const int *ea,
                   const int *eb, const DV &C, const double *alpha, const double *beta, int beta_zero) {
    if (m == 0 || n == 0) return hipSuccess;
    if (K > 8192 || K % 64 != 0 || S != oz_gemm_digits(N, K)) return hipErrorInvalidValue;
    const int64_t blocks = cdiv(m, 16) * cdiv(n, 16);
#define OZ_GO(...) return oz_launch<__VA_ARGS__>(s, m, n, K, dA, dB, ea, eb, C, alpha, beta, beta_zero)
    switch (S) {
        case 30:
            if (blocks >= 4096) OZ_GO(4, 8, 30, 4, 2, 3, 6);
            if (blocks >= 1024) OZ_GO(4, 8, 30, 1, 1, 4, 6);
            OZ_GO(4, 8, 30, 4, 1, 8, 6);
        case 24: OZ_GO(3, 8, 24, 4, 1, 8, 6);
        case 17: OZ_GO(2, 8, 17, 4, 1, 8, 6);
        case 10: OZ_GO(1, 8, 10, 4, 1, 4, 4);
        case 34: OZ_GO(4, 7, 34, 4, 1, 8, 6);
        case 27: OZ_GO(3, 7, 27, 4, 2, 6, 6);
        case 19: OZ_GO(2, 7, 19, 4, 1, 8, 6);
        case 11: OZ_GO(1, 7, 11, 4, 1, 4, 5);
    }
#undef OZ_GO
    return hipErrorInvalidValue;
}

int oz_row_align() { return 64; }

hipError_t oz_combine(int N, hipStream_t s, int64_t m, int64_t n, int U, const int32_t *planes, const int *ea, const int *eb,
                      const DV &C) {
    if (m * n == 0) return hipSuccess;
    OZ_DISPATCH(N, hipLaunchKernelGGL(k_oz_combine<NN>, dim3((unsigned)cdiv(m * n, 256)), dim3(256), 0, s, m, n, U, planes, ea, eb, C));
    return hipGetLastError();
}

}  // namespace mfk
