// slice_core.hpp — step-2 block bodies (256 threads) shared by the single-problem and grouped
// kernels.  Operands with K-contiguous rows are read in blocks of 32 rows x 128 K, operands with
// row-contiguous storage in blocks of 64 rows x 128 K; see k_slice.hip for the arithmetic and the
// output layout.
#pragma once

#include "oza_device.hpp"
#include "oza_internal.hpp"

namespace oza {
namespace core {

constexpr int kSliceThreads = 256;

// Constants of sym_residue: byte weights per word, the word bias' share, m and m^-1 mod 2^32.
struct ResidueConsts {
    uint32_t wt[kMaxSlices][3];
    uint32_t init[kMaxSlices][3];  // by word count - 1
    uint32_t m[kMaxSlices], minv[kMaxSlices];
};

inline ResidueConsts make_residue_consts() {
    ResidueConsts rc;
    for (int s = 0; s < kMaxSlices; ++s) {
        const uint64_t m = kModuli[s];
        uint64_t p = (uint64_t(1) << 32) % m;  // 2^32 2^(8 i) mod m
        const uint64_t p256 = 256 % m;
        uint64_t w[13];
        for (int i = 0; i < 13; ++i) {
            w[i] = p;
            p = p * p256 % m;
        }
        for (int n = 0; n < 3; ++n) {
            rc.wt[s][n] = 0;
            for (int k = 0; k < 4; ++k) rc.wt[s][n] |= (uint32_t)((m - w[4 * n + k]) % m) << (8 * k);
            rc.init[s][n] = (uint32_t)(w[4 * n + 3] * 128 % m);  // 2^32 times the bias 2^(32 (n + 1) - 1)
        }
        uint32_t inv = 1;  // Newton: correct bits of m^-1 mod 2^32 double each time
        for (int i = 0; i < 6; ++i) inv *= 2u - (uint32_t)m * inv;
        rc.m[s] = (uint32_t)m;
        rc.minv[s] = inv;
    }
    return rc;
}

// Words sym_residue needs for |t| <= 2^kparam (K_param is at most 75: S = 20 and K <= 2).
inline int residue_words(int kparam) { return kparam <= 30 ? 1 : kparam <= 62 ? 2 : 3; }

template <int ND>
struct Words16 {
    uint32_t w[16][ND];
};

// rint(2^sh a) of 16 values as words.
template <int ND>
__device__ __forceinline__ void scaled_words16(const double (&a)[16], int sh, Words16<ND>& t) {
#pragma unroll
    for (int j = 0; j < 16; ++j) int_words<ND>(rint(ldexp(a[j], sh)), t.w[j]);
}

// Symmetric residues of 16 integers modulo m_s, packed into 16 bytes.
template <int ND>
__device__ __forceinline__ uint4 residues16(const Words16<ND>& t, const ResidueConsts& rc, int s) {
    uint32_t wt[ND];
#pragma unroll
    for (int n = 0; n < ND; ++n) wt[n] = rc.wt[s][n];
    int r[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) r[j] = sym_residue<ND>(t.w[j], wt, rc.init[s][ND - 1], rc.m[s], rc.minv[s]);
    return make_uint4(pack4_lo(r[0], r[1], r[2], r[3]), pack4_lo(r[4], r[5], r[6], r[7]),
                      pack4_lo(r[8], r[9], r[10], r[11]), pack4_lo(r[12], r[13], r[14], r[15]));
}

// 16 values of row `row` from K-byte 16c on, zero past K.  Ragged or unaligned: every load
// unconditional (clamped index), padding zeroed after.
__device__ __forceinline__ void load_row16(const double* __restrict__ A, int64_t lda, int64_t row, int64_t k0,
                                           int64_t K, double (&a)[16]) {
    const double* p = A + row * lda + k0;
    if (k0 + 16 <= K && ((reinterpret_cast<uintptr_t>(p) & 15) == 0)) {
#pragma unroll
        for (int j = 0; j < 16; j += 2) {
            const double2 v = *reinterpret_cast<const double2*>(p + j);
            a[j] = v.x;
            a[j + 1] = v.y;
        }
    } else {
        const double* row_p = A + row * lda;
#pragma unroll
        for (int j = 0; j < 16; ++j) a[j] = row_p[min(k0 + j, K - 1)];
#pragma unroll
        for (int j = 0; j < 16; ++j) a[j] = k0 + j < K ? a[j] : 0.0;
    }
}

// The shift of row r for a block of 256 threads, 256 / G of them (consecutive, the same rows) in each of
// its G groups.  Every thread of the block calls it; 0 past the last row.  From partial maxima, the
// block with `store` also writes the shift.
template <int G>
__device__ __forceinline__ int shift_of_row(const Shifts& s, int64_t r, int64_t rows, bool store) {
    if (!s.part) return r < rows ? s.shift[r] : 0;
    constexpr int T = kSliceThreads / G;
    __shared__ uint32_t s_key[kSliceThreads];
    const int g = threadIdx.x / T;
    const int64_t rr = min(r, rows - 1);
    uint32_t v[kStatParts / G], key = 0;
#pragma unroll
    for (int i = 0; i < kStatParts / G; ++i) v[i] = s.part[(int64_t)min(g + i * G, s.parts - 1) * s.rows + rr];
#pragma unroll
    for (int i = 0; i < kStatParts / G; ++i) key = max(key, v[i]);
    s_key[threadIdx.x] = key;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < G; ++i) key = max(key, s_key[i * T + threadIdx.x % T]);
    const int sh = s.offset - exp_from_key(key);
    if (store && g == 0 && r < rows) s.shift[r] = sh;
    return r < rows ? sh : 0;
}

// ---------------------------------------------------------------- Scheme II, K-contiguous rows
// Operand element (row, k) at A[row * lda + k] (the reference's A; also op(B) = B^T stored N x K).
// Block = 32 rows x 128 K; thread = row (tid % 32), 16-byte K chunk (tid / 32).  The 64 lanes of a
// wave cover one whole 1 KiB fragment block.
template <int ND, bool NT = false>
__device__ __forceinline__ void slice_s2_A_block(const double* __restrict__ A, int64_t lda,
                                                 const Shifts& shift, int64_t M, int64_t K, int64_t Mp, int64_t Kp,
                                                 int S, const ResidueConsts& rc, int8_t* __restrict__ out, int64_t bx,
                                                 int64_t by) {
    const int64_t row = bx * 32 + (threadIdx.x & 31);
    const int64_t c = by * 8 + (threadIdx.x >> 5);
    const int64_t k0 = c * 16;
    double a[16] = {};
    if (row < M) load_row16(A, lda, row, k0, K, a);
    const int sh = shift_of_row<8>(shift, row, M, by == 0);
    drop_non_finite(a);
    Words16<ND> t;
    scaled_words16(a, sh, t);
    const int64_t plane = Mp * Kp;
    int8_t* o = out + frag_off16(row, c, Kp);
    for (int s = 0; s < S; ++s) store_unit16<NT>(o + s * plane, residues16(t, rc, s));
}

// ---------------------------------------------------------------- Scheme II, row-contiguous columns
// Operand element (col, k) at B[k * ldb + col] (the reference's B; also op(A) = A^T stored K x M).
// Block = 64 columns x 4 groups of 32 K rows; thread = one column, 32 consecutive k.
template <int ND, bool NT = false>
__device__ __forceinline__ void slice_s2_B_block(const double* __restrict__ B, int64_t ldb,
                                                 const Shifts& shift, int64_t K, int64_t N, int64_t Np, int64_t Kp,
                                                 int S, const ResidueConsts& rc, int8_t* __restrict__ out, int64_t bx,
                                                 int64_t by) {
    const int64_t col = bx * 64 + (threadIdx.x & 63);
    const int64_t kbase = by * 128 + (threadIdx.x >> 6) * 32;
    const int64_t plane = Np * Kp;
    const int sh = shift_of_row<4>(shift, col, N, by == 0);
    const int64_t cc = min(col, N - 1);  // clamped: every load unconditional, padding zeroed after
#pragma unroll 1
    for (int half = 0; half < 2; ++half) {
        const int64_t k0 = kbase + half * 16;
        double a[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) a[j] = B[min(k0 + j, K - 1) * ldb + cc];
#pragma unroll
        for (int j = 0; j < 16; ++j) a[j] = col < N && k0 + j < K ? a[j] : 0.0;
        drop_non_finite(a);
        Words16<ND> t;
        scaled_words16(a, sh, t);
        int8_t* o = out + frag_off16(col, k0 >> 4, Kp);
        for (int s = 0; s < S; ++s) store_unit16<NT>(o + s * plane, residues16(t, rc, s));
    }
}

// ---------------------------------------------------------------- Scheme I
// Slices of 16 values sharing one exponent e (row of A or column of B); slices below s0 are formed (each
// takes its part off the values) but not stored.
__device__ __forceinline__ void slice_s1_16(double (&a)[16], int e, int beta, int S, int8_t* o, int64_t plane,
                                            int s0 = 0) {
#pragma clang fp contract(off)  // every operation rounds where the reference's does
    const double scale = ldexp(1.0, e + 1 - beta);
    const double inv_scale = ldexp(1.0, -(e + 1 - beta));
    for (int s = 0; s < S; ++s) {
        const double sigma = 0.75 * ldexp(scale, 53 - beta * s);
        int r[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            // (a + sigma) - sigma: contraction and reassociation are off in this file.
            const double tmp = a[j] + sigma;
            const double a_s = tmp - sigma;
            const double normalized = a_s * inv_scale;
            const double scaled = ldexp(normalized, beta * s);
            r[j] = (int)scaled;
            a[j] = a[j] - a_s;
        }
        if (s >= s0)
            *reinterpret_cast<uint4*>(o + s * plane) =
                make_uint4(pack4_lo(r[0], r[1], r[2], r[3]), pack4_lo(r[4], r[5], r[6], r[7]),
                           pack4_lo(r[8], r[9], r[10], r[11]), pack4_lo(r[12], r[13], r[14], r[15]));
    }
}

__device__ __forceinline__ void slice_s1_A_block(const double* __restrict__ A, int64_t lda,
                                                 const Shifts& neg_exp, int64_t M, int64_t K, int64_t Mp, int64_t Kp,
                                                 int S, int beta, int8_t* __restrict__ out, int64_t bx, int64_t by) {
    const int64_t row = bx * 32 + (threadIdx.x & 31);
    const int64_t c = by * 8 + (threadIdx.x >> 5);
    const int64_t k0 = c * 16;
    int8_t* o = out + frag_off16(row, c, Kp);
    double a[16];
    if (row < M) load_row16(A, lda, row, k0, K, a);
    const int e = -shift_of_row<8>(neg_exp, row, M, by == 0);
    if (row < M) {
        slice_s1_16(a, e, beta, S, o, Mp * Kp);
    } else {
        for (int s = 0; s < S; ++s) *reinterpret_cast<uint4*>(o + s * Mp * Kp) = make_uint4(0, 0, 0, 0);
    }
}

__device__ __forceinline__ void slice_s1_B_block(const double* __restrict__ B, int64_t ldb,
                                                 const Shifts& neg_exp, int64_t K, int64_t N, int64_t Np, int64_t Kp,
                                                 int S, int beta, int8_t* __restrict__ out, int64_t bx, int64_t by) {
    const int64_t col = bx * 64 + (threadIdx.x & 63);
    const int64_t kbase = by * 128 + (threadIdx.x >> 6) * 32;
    const int64_t plane = Np * Kp;
    const int e = -shift_of_row<4>(neg_exp, col, N, by == 0);
#pragma unroll 1
    for (int half = 0; half < 2; ++half) {
        const int64_t k0 = kbase + half * 16;
        int8_t* o = out + frag_off16(col, k0 >> 4, Kp);
        if (col < N) {
            double a[16];  // every load unconditional (clamped index), padding zeroed after
#pragma unroll
            for (int j = 0; j < 16; ++j) a[j] = B[min(k0 + j, K - 1) * ldb + col];
#pragma unroll
            for (int j = 0; j < 16; ++j) a[j] = k0 + j < K ? a[j] : 0.0;
            slice_s1_16(a, e, beta, S, o, plane);
        } else {
            for (int s = 0; s < S; ++s) *reinterpret_cast<uint4*>(o + s * plane) = make_uint4(0, 0, 0, 0);
        }
    }
}

// One operand of step 2: logical rows (padded to rows_p in the plane) of K values, element (r, k)
// at p[r * ld + k] (kcontig: 32-row blocks) or p[k * ld + r] (64-row blocks); nblk blocks of
// 128 K each, over the blocks that hold a logical row.  The plane's blocks past the last logical
// row are left unwritten: they only meet product rows (or columns) past M (or N), whose digits
// nothing reads, while the K padding inside the written blocks is zero.
struct SliceOp {
    const double* p;
    int64_t rows, rows_p, ld;
    int32_t kcontig;
    Shifts shift;
    int8_t* out;
    int64_t nblk;
};

inline SliceOp make_slice_op(const double* p, int64_t rows, int64_t rows_p, int64_t ld, bool kcontig,
                             int64_t Kp, const Shifts& shift, int8_t* out) {
    SliceOp o;
    o.p = p;
    o.rows = rows;
    o.rows_p = rows_p;
    o.ld = ld;
    o.kcontig = kcontig;
    o.shift = shift;
    o.out = out;
    const int64_t rb = kcontig ? 32 : 64;
    o.nblk = ((rows + rb - 1) / rb) * (Kp / 128);
    return o;
}

template <int ND>
__device__ __forceinline__ void slice_s2_op_block(const SliceOp& o, int64_t K, int64_t Kp, int S,
                                                  const ResidueConsts& rc, int64_t blk) {
    const int64_t kb = Kp / 128;
    const int64_t bx = blk / kb, by = blk - bx * kb;
    if (o.kcontig) slice_s2_A_block<ND>(o.p, o.ld, o.shift, o.rows, K, o.rows_p, Kp, S, rc, o.out, bx, by);
    else slice_s2_B_block<ND>(o.p, o.ld, o.shift, K, o.rows, o.rows_p, Kp, S, rc, o.out, bx, by);
}

__device__ __forceinline__ void slice_s1_op_block(const SliceOp& o, int64_t K, int64_t Kp, int S, int beta,
                                                  int64_t blk) {
    const int64_t kb = Kp / 128;
    const int64_t bx = blk / kb, by = blk - bx * kb;
    if (o.kcontig) slice_s1_A_block(o.p, o.ld, o.shift, o.rows, K, o.rows_p, Kp, S, beta, o.out, bx, by);
    else slice_s1_B_block(o.p, o.ld, o.shift, K, o.rows, o.rows_p, Kp, S, beta, o.out, bx, by);
}

// ---------------------------------------------------------------- steps 1 and 2 in one pass, both operands
// Single calls with Kp <= kPassMaxKp: a block of T threads (pass_threads: 256, 512 or 1024 by K) holds R
// whole rows (columns of a row-contiguous operand) in registers, takes their exponent maxima, writes
// the shifts and then the slices of the values it still holds.  Unit u = (row u % R, 16-byte K chunk u / R)
// of the block; thread t takes units t + T i, i < NU, all of row t % R.  With R = 16 a wave reads a
// row-contiguous operand in 128-byte runs and writes 256-byte runs of a fragment block; R grows to 64
// for short K so that the threads have units, and is 8 past K = 2048, whose runs of 64 and 128 bytes are
// the better choice only where the blocks run at once (one_pass).  Values and results are those of the
// separate kernels.
// A block's planes may be dealt to `parts` blocks that each read the rows again (part j stores planes
// [S j / parts, S (j + 1) / parts), part 0 the shifts): more blocks for small operands, whose second
// reads come from the XCD's L2 (the parts of a row block are 8 block indices apart, on one XCD).
// Small calls are bound by launches (4.7 us of stream time each) and latency: this takes the place of
// two launches (four before: keys cleared, maxima, keys to shifts, slices).  One or two units per thread
// and many threads, not four units in 256 threads (184 registers, 8 waves per CU instead of 16):
// 2048^3, S = 6 111 us per call in two kernels, 101 in one pass (37 us for the launch with four units in 512
// threads); 1024^3, S = 16 54 and 45; 8192^2 x 1024, S = 16 1.551 and 1.523 ms; 256^3, S = 4 24 and 15 us.
constexpr int64_t kPassMaxKp = 4096, kGroupPassMaxKp = 2048;

inline int pass_threads(int64_t Kp) { return Kp <= 256 ? 256 : Kp <= 512 ? 512 : 1024; }
inline int pass_units(int64_t Kp) { return Kp <= 1024 ? 1 : 2; }
inline int pass_rows(int64_t Kp) {
    int r = 64;
    while (r > 8 && r * (Kp / 16) > pass_threads(Kp) * pass_units(Kp)) r >>= 1;
    return r;
}

// Row blocks of an operand: the rows its planes hold, whole 32-row fragment blocks.
inline int64_t pass_row_blocks(int64_t rows, int R) { return ((rows + 31) / 32 * 32 + R - 1) / R; }

struct PassOp {
    const double* p;
    int64_t rows, rows_p, ld;
    int32_t kcontig;
    int32_t* shift;
    int8_t* out;
    int64_t nrow;  // row blocks
};

struct PassArgs {
    PassOp op[2];
    int64_t K, Kp;
    int S, R, parts, offset;  // offset: K_param (Scheme II) or beta (Scheme I)
    uint32_t* zero;           // words cleared by the first block (the GEMM's work counters)
    int nzero;
};

// ND: words per value (Scheme II), or 0 for Scheme I.
// NT: nontemporal plane stores (store_unit16).
template <int ND, int T, int NU, bool KC, bool NT = false>
__device__ __forceinline__ void pass_block(const PassOp& o, const PassArgs& g, const ResidueConsts& rc, int64_t rb,
                                           int part, uint32_t* s_key, int32_t* s_shift) {
    const int R = g.R;
    const int t = threadIdx.x;
    const int rl = t & (R - 1), c0 = t / R, cstep = T / R;
    const int64_t row = rb * R + rl;
    const int U = (int)(g.Kp / 16);
    double a[NU][16];
    uint32_t key = 0;
#pragma unroll
    for (int i = 0; i < NU; ++i) {
        const int c = c0 + i * cstep;
        if (c < U && row < o.rows) {
            const int64_t k0 = (int64_t)c * 16;
            if (KC) {
                load_row16(o.p, o.ld, row, k0, g.K, a[i]);
            } else {
#pragma unroll
                for (int j = 0; j < 16; ++j) a[i][j] = o.p[min(k0 + j, g.K - 1) * o.ld + row];
#pragma unroll
                for (int j = 0; j < 16; ++j) a[i][j] = k0 + j < g.K ? a[i][j] : 0.0;
            }
        } else {
#pragma unroll
            for (int j = 0; j < 16; ++j) a[i][j] = 0.0;
        }
    }
#pragma unroll
    for (int i = 0; i < NU; ++i) {
        key = max(key, max_key(a[i]));
        if (ND > 0) drop_non_finite(a[i]);
    }
    for (int d = R; d < 64; d <<= 1) key = max(key, (uint32_t)__shfl_xor((int)key, d));
    if ((t & 63) < R) s_key[(t >> 6) * 64 + (t & 63)] = key;
    __syncthreads();
    if (t < R) {
        uint32_t k = 0;
#pragma unroll
        for (int w = 0; w < T / 64; ++w) k = max(k, s_key[w * 64 + t]);
        const int32_t sh = (ND == 0 ? 0 : g.offset) - exp_from_key(k);  // key_to_shift
        s_shift[t] = sh;
        if (part == 0 && row < o.rows) o.shift[row] = sh;
    }
    __syncthreads();
    if (row >= (o.rows + 31) / 32 * 32) return;  // the planes' blocks past the last logical row stay unwritten
    const int sh = s_shift[rl];
    const int64_t plane = o.rows_p * g.Kp;
    const int s0 = g.S * part / g.parts, s1 = g.S * (part + 1) / g.parts;
#pragma unroll
    for (int i = 0; i < NU; ++i) {
        const int c = c0 + i * cstep;
        if (c >= U) break;
        int8_t* out = o.out + frag_off16(row, c, g.Kp);
        if constexpr (ND == 0) {
            if (row < o.rows) {
                slice_s1_16(a[i], -sh, g.offset, s1, out, plane, s0);
            } else {
                for (int s = s0; s < s1; ++s) *reinterpret_cast<uint4*>(out + s * plane) = make_uint4(0, 0, 0, 0);
            }
        } else {
            Words16<ND> v;
            scaled_words16(a[i], sh, v);
            for (int s = s0; s < s1; ++s) store_unit16<NT>(out + s * plane, residues16(v, rc, s));
        }
    }
}

// Grouped problems with Kp <= kGroupPassMaxKp: blocks of 512 threads with up to two units each, any K.  A group's
// launch is bound by memory, not by latency, and two such blocks share a CU, so that one reads while the
// other computes and writes.  Two units in 1024 threads, one in 512 and four in 512 or 256 were slower (the
// whole group of 512 problems, M, N, K log-uniform on [64, 2048]: 5.07, 5.15, 5.12 ms; two in 512 4.96 ms for
// B, 4.92 ms for both operands; before, with B read by step 1 and again by step 2, 5.17 ms).
constexpr int kGroupPassThreads = 512, kGroupPassUnits = 2;
__host__ __device__ inline int group_pass_rows(int64_t Kp) {
    int r = 64;
    while (r > 8 && r * (Kp / 16) > kGroupPassThreads * kGroupPassUnits) r >>= 1;
    return r;
}

}  // namespace core
}  // namespace oza
