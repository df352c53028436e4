// recon_core.hpp — Scheme II step-4 arithmetic shared by the single-problem and grouped
// reconstruction kernels: exact CRT reconstruction of one element from its digits, and the
// block body that reconstructs a 32 x 32 block of C from the blocked digit planes.
#pragma once

#include "oza_device.hpp"
#include "oza_internal.hpp"

namespace oza {
namespace core {

template <int S>
struct CrtShape {
    static constexpr int BITS = bitlen_M(S);
    static constexpr int G = (S + 2) / 3;            // groups of three moduli
    static constexpr int LR = (BITS + 31) / 32;      // words of R_g
    static constexpr int L = (BITS + 1 + 31) / 32;   // words of the signed Y, |Y| < 0.56 M
    static_assert(L <= kWords, "word budget");
};

// Byte b of w (b a compile-time constant: a byte select of the 24-bit multiply that uses it).
__device__ __forceinline__ uint32_t byte_of(uint32_t w, int b) { return (w >> (8 * b)) & 0xffu; }

// Adds k * v to Y, words modulo 2^(32 L), k = +1 or -1.
template <int L, bool SUB>
__device__ __forceinline__ void add_words(uint32_t (&y)[L], const uint32_t* __restrict__ v) {
    uint32_t carry = SUB ? 1 : 0;
#pragma unroll
    for (int l = 0; l < L; ++l) y[l] = __builtin_addc(y[l], SUB ? ~v[l] : v[l], carry, &carry);
}

// Signed reconstruction of one element from its digits, byte b of w[s] = c_s, as the reference's
// double.  With the groups of CrtSet:
//   X = sum_g u_g R_g in LR 64-bit columns (u_g < 2^25.4, at most 7 groups: every column < 2^61);
//   q estimates floor(X/M + 1/2) from h = 2^31 + sum_g u_g F_g, which is short of 2^32 (X/M + 1/2)
//     by less than sum_g u_g: q is that floor, or one less when the fraction of h is at or above
//     cs->amb (sum of the u_g bounds from the top, with a margin of 1/(2M));
//   Y = X - q M: the columns get q times the words of 2^160 - M, then one carry pass.
// The reference maps X mod M >= floor(M/2) to X mod M - M.  Away from the ambiguous fractions that
// is the Y above (|Y| < M/2, M odd); at them the exact comparison with floor(M/2) decides.
// What bounds it: VALU issue and the digits' and C's bytes about equally (every instruction here, the
// 64-bit multiply-add included, issues in four cycles per wave).  Groups of three, because u_g must
// fit the 32-bit operand of the multiply-add: three digits then cost 3 byte-select multiplies, one
// three-way add and LR multiply-adds.  16-bit limbs of X by v_dot4_u32_u8 (18 limbs at S = 17, five
// dot products each, a carry and a sign pass over every limb) took 239 instructions per element and
// 1.26 ms for the 512-GEMM batch's step 4 against 0.99 ms here (156 per element at S = 17, the
// ambiguous path included).
template <int S>
__device__ __forceinline__ double crt_value(const uint32_t (&w)[S], int b, const CrtSet* __restrict__ cs) {
    constexpr int G = CrtShape<S>::G, LR = CrtShape<S>::LR, L = CrtShape<S>::L;
    uint64_t col[L];
    uint64_t h = 1ull << 31;
#pragma unroll
    for (int l = 0; l < L; ++l) col[l] = 0;
#pragma unroll
    for (int g = 0; g < G; ++g) {
        uint32_t u = __umul24(byte_of(w[3 * g], b), cs->E[3 * g]);
        if (3 * g + 1 < S) u += __umul24(byte_of(w[3 * g + 1], b), cs->E[3 * g + 1]);
        if (3 * g + 2 < S) u += __umul24(byte_of(w[3 * g + 2], b), cs->E[3 * g + 2]);
        h += (uint64_t)u * cs->F[g];
#pragma unroll
        for (int l = 0; l < LR; ++l) col[l] += (uint64_t)u * cs->R[g][l];
    }
    const uint32_t q = (uint32_t)(h >> 32);
    uint32_t y[L];
    uint32_t carry = 0;
#pragma unroll
    for (int l = 0; l < L; ++l) {
        col[l] += (uint64_t)q * cs->Mneg[l];
        y[l] = l == 0 ? (uint32_t)col[0]
                      : __builtin_addc((uint32_t)col[l], (uint32_t)(col[l > 0 ? l - 1 : 0] >> 32), carry, &carry);
    }
    if (__builtin_expect((uint32_t)h >= cs->amb, 0)) {
        uint32_t d[L];
#pragma unroll
        for (int l = 0; l < L; ++l) d[l] = y[l];
        add_words<L, true>(d, cs->Mhalf32);
        if ((int32_t)d[L - 1] >= 0) add_words<L, true>(y, cs->M32);
    }
    // |Y| and the sign
    const uint32_t neg = (uint32_t)((int32_t)y[L - 1] >> 31);
    carry = neg & 1u;
#pragma unroll
    for (int l = 0; l < L; ++l) y[l] = __builtin_addc(y[l] ^ neg, 0u, carry, &carry);
    // to_double_256 (crt_math.hpp:73-80): the 64-bit word d_i = y[2i+1] 2^32 + y[2i] converted with one
    // rounding, as one fma of its exact halves, already scaled by its power of two 2^(64 i) (exact);
    // then the reference's additions in its order (0 + RN(d0) is RN(d0); the word d3 is zero).
    double f = (double)y[0];
    if (L > 1) f = fma((double)y[L > 1 ? 1 : 0], 0x1p32, f);
    if (L > 2) {
        double d1 = (double)y[L > 2 ? 2 : 0] * 0x1p64;
        if (L > 3) d1 = fma((double)y[L > 3 ? 3 : 0], 0x1p96, d1);
        f = f + d1;
    }
    if (L > 4) f = f + (double)y[L > 4 ? 4 : 0] * 0x1p128;
    // Y = 0 is +0 as in the reference: neg is 0 there
    return __longlong_as_double(__double_as_longlong(f) ^ ((int64_t)((uint64_t)(neg & 0x80000000u) << 32)));
}

// C[row * ldc + col] = alpha * x + beta * C[...] as fma(alpha, x, beta * C); beta == 0 does not
// read C, and alpha == 1 with beta == 0 stores x itself.
__device__ __forceinline__ void store_c(double* __restrict__ C, int64_t idx, double x, double alpha, double beta) {
    if (beta == 0.0) C[idx] = alpha == 1.0 ? x : alpha * x;
    else C[idx] = fma(alpha, x, beta * C[idx]);
}

// Partial digits of a call whose items past `whole` ran in parts (S2Plan): part j > 0 of item l at partial
// tile (j - 1) * tail + (l - whole).
struct DigitParts {
    const uint8_t* part;
    int64_t whole, tail;
    int parts, tiles_m, tiles_n, gm;  // gm: tile rows per group of the GEMM's tile order
};

// Four digits each of two words, added modulo m byte by byte (digits below m).
__device__ __forceinline__ uint32_t add_digits(uint32_t a, uint32_t b, uint32_t m) {
    typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
    const u16x2 mm = {(unsigned short)m, (unsigned short)m};
    auto add = [&](uint32_t x, uint32_t y) {
        const u16x2 s = __builtin_bit_cast(u16x2, x) + __builtin_bit_cast(u16x2, y);
        return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(s, s - mm));  // s - m wraps above s when s < m
    };
    const uint32_t lo = add(a & 0x00ff00ffu, b & 0x00ff00ffu);
    const uint32_t hi = add((a >> 8) & 0x00ff00ffu, (b >> 8) & 0x00ff00ffu);
    return lo | (hi << 8);
}

// Adds the parts' digits of element block (R, Q), byte offset `off` in the block, to w and to the digit
// planes, where w[s] came from dg + s * plane.
template <int S>
__device__ __forceinline__ void add_parts(uint32_t (&w)[S], const DigitParts& d, const CrtSet* __restrict__ cs,
                                          int64_t R, int64_t Q, int off, uint8_t* dg, int64_t plane) {
    // The block's tile in the GEMM's order: groups of gm tile rows, column by column.  (Inverse of
    // grouped_tile.)
    const int tm = (int)(R >> 3), tn = (int)(Q >> 3);
    const int first = tm / d.gm * d.gm, rows = min(d.tiles_m - first, d.gm);
    const int64_t t = (int64_t)first * d.tiles_n + (int64_t)tn * rows + (tm - first);
    const int64_t tiles = (int64_t)d.tiles_m * d.tiles_n;
    const int s0 = d.whole > t ? (int)((d.whole - t + tiles - 1) / tiles) : 0;  // the moduli that ran in parts
    if (s0 >= S) return;
    const uint8_t* base = d.part + (t - d.whole) * kTileBytes + ((((R & 7) << 3) + (Q & 7)) << 10) + off;
    for (int j = 1; j < d.parts; ++j, base += d.tail * kTileBytes) {
        uint32_t x[S];
#pragma unroll
        for (int s = 0; s < S; ++s) {
            x[s] = 0;
            if (s >= s0) x[s] = *reinterpret_cast<const uint32_t*>(base + s * tiles * kTileBytes);
        }
#pragma unroll
        for (int s = 0; s < S; ++s)
            if (s >= s0) w[s] = add_digits(w[s], x[s], cs->m[s]);
    }
#pragma unroll
    for (int s = 0; s < S; ++s)
        if (s >= s0) *reinterpret_cast<uint32_t*>(dg + s * plane) = w[s];
}

// One 32 x 32 element block (R, Q) of C from blocked digit planes (layout of store_digits:
// block (R, Q) at byte (R * Np/32 + Q) * 1024 of each plane, MFMA 32x32 order inside).
// 256 threads; thread t reads dword t of the block in every plane (4 elements of one column).
// PLAIN: alpha = 1, beta = 0 (C = X), compiled without the output rule.  PARTS: some items ran in parts.
template <int S, bool PLAIN = true, bool PARTS = false>
__device__ __forceinline__ void recon_digits_block(const uint8_t* __restrict__ dg, int64_t plane, int64_t Np,
                                                   const int32_t* __restrict__ shA, const int32_t* __restrict__ shB,
                                                   int64_t M, int64_t N, const CrtSet* __restrict__ cs,
                                                   double* __restrict__ Cout, int64_t ldc, double alpha, double beta,
                                                   int64_t R, int64_t Q, const DigitParts* parts = nullptr) {
    const int t = threadIdx.x;
    const int lane = t >> 2, wd = t & 3;
    const int64_t col = Q * 32 + (lane & 31);
    const int64_t row0 = R * 32 + 8 * wd + 4 * (lane >> 5);
    if (col >= N || row0 >= M) return;
    const uint8_t* base = dg + ((R * (Np >> 5) + Q) << 10) + t * 4;
    uint32_t w[S];
#pragma unroll
    for (int s = 0; s < S; ++s) w[s] = *reinterpret_cast<const uint32_t*>(base + s * plane);
    const int32_t sb = shB[col];
    if (PARTS) add_parts<S>(w, *parts, cs, R, Q, t * 4, const_cast<uint8_t*>(base), plane);
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        const int64_t row = row0 + b;
        if (row < M) {
            const double x = ldexp(crt_value<S>(w, b, cs), -(shA[row] + sb));
            if (PLAIN) Cout[row * ldc + col] = x;
            else store_c(Cout, row * ldc + col, x, alpha, beta);
        }
    }
}

}  // namespace core
}  // namespace oza
