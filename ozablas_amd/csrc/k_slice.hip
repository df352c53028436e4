// k_slice.hip — step 2: split FP64 operands into INT8 planes laid out for the MFMA GEMM.
//
// Scheme II (reference: src/pipeline/step2_slicing.hpp:29-38, 110-206): x = ldexp(a, shift),
// t = rint(x) (round-half-even, which is what both the reference's llrint fast path and its
// rint/fmod heavy path round to), residue r_s = symmetric residue of t mod m_s.  Any exact
// method yields the same bytes; sym_residue works on t as one to three 32-bit words.
//
// Scheme I (reference: step2_slicing.hpp:20-25, 44-100): the reference's exact sequence of
// FP64 operations, sigma = 0.75 * 2^(E+1-beta+53-beta*s), a_s = (a + sigma) - sigma,
// slice = int(ldexp(a_s * 2^-(E+1-beta), beta*s)), a -= a_s.  Contraction is off in this file
// so every operation rounds where the reference's does.
//
// Output layout: A planes (Mp x Kp) and B planes (Np x Kp, B transposed so that both MFMA
// operands are K-contiguous) in the fragment-tiled order of frag_off16.  Padding is zero.  Each
// thread produces 16 consecutive K values of one row/column, i.e. one 16-byte unit per plane, and
// a wave's 64 units form contiguous runs of the tiled layout.
#pragma clang fp contract(off)

#include <algorithm>

#include "slice_core.hpp"

namespace oza {
namespace {

using namespace core;

// Blocks of a one-pass launch that run at once when K is long (one 1024-thread block per CU).
constexpr int64_t kPassResident = 256;

// Blocks [0, a.nblk) slice operand a into its planes, the rest operand b.
template <int ND>
__global__ void __launch_bounds__(kSliceThreads)
    k_slice_s2(SliceOp a, SliceOp b, int64_t K, int64_t Kp, int S, ResidueConsts rc) {
    if ((int64_t)blockIdx.x < a.nblk) slice_s2_op_block<ND>(a, K, Kp, S, rc, blockIdx.x);
    else slice_s2_op_block<ND>(b, K, Kp, S, rc, (int64_t)blockIdx.x - a.nblk);
}

__global__ void __launch_bounds__(kSliceThreads)
    k_slice_s1(SliceOp a, SliceOp b, int64_t K, int64_t Kp, int S, int beta) {
    if ((int64_t)blockIdx.x < a.nblk) slice_s1_op_block(a, K, Kp, S, beta, blockIdx.x);
    else slice_s1_op_block(b, K, Kp, S, beta, (int64_t)blockIdx.x - a.nblk);
}

// Steps 1 and 2 of both operands in one launch (pass_block).  Block b -> part and row block: sets of 8
// consecutive row blocks (of operand 0, then operand 1), each set's parts after one another.
template <int ND, int T, int NU>
__global__ void __launch_bounds__(T) k_pass(PassArgs g, ResidueConsts rc) {
    __shared__ uint32_t s_key[T];
    __shared__ int32_t s_shift[64];
    if (blockIdx.x == 0 && (int)threadIdx.x < g.nzero) g.zero[threadIdx.x] = 0;
    const int64_t set = blockIdx.x / (8 * g.parts);
    const int in = (int)(blockIdx.x - set * 8 * g.parts);
    const int part = in >> 3;
    int64_t rb = set * 8 + (in & 7);
    const int w = rb >= g.op[0].nrow;
    if (w) rb -= g.op[0].nrow;
    const PassOp& o = g.op[w];
    if (rb >= o.nrow) return;  // past the last set's row blocks (whole block)
    if (o.kcontig) pass_block<ND, T, NU, true>(o, g, rc, rb, part, s_key, s_shift);
    else pass_block<ND, T, NU, false>(o, g, rc, rb, part, s_key, s_shift);
}

template <int ND>
hipError_t launch_pass_words(const PassArgs& g, const ResidueConsts& rc, unsigned grid, hipStream_t st) {
    switch (pass_threads(g.Kp) * pass_units(g.Kp)) {
        case 256: k_pass<ND, 256, 1><<<grid, 256, 0, st>>>(g, rc); break;
        case 512: k_pass<ND, 512, 1><<<grid, 512, 0, st>>>(g, rc); break;
        case 1024: k_pass<ND, 1024, 1><<<grid, 1024, 0, st>>>(g, rc); break;
        default: k_pass<ND, 1024, 2><<<grid, 1024, 0, st>>>(g, rc); break;
    }
    return hipGetLastError();
}

// ---------------------------------------------------------------- unpack to planar layout
__global__ void k_unpack_A(const int8_t* __restrict__ in, int64_t M, int64_t K, int64_t Mp, int64_t Kp, int S,
                           int8_t* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t tot = (int64_t)S * M * K;
    if (i >= tot) return;
    const int64_t s = i / (M * K);
    const int64_t r = (i / K) % M;
    const int64_t k = i % K;
    out[i] = in[s * Mp * Kp + frag_off16(r, k >> 4, Kp) + (k & 15)];
}

__global__ void k_unpack_B(const int8_t* __restrict__ in, int64_t K, int64_t N, int64_t Np, int64_t Kp, int S,
                           int8_t* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t tot = (int64_t)S * K * N;
    if (i >= tot) return;
    const int64_t s = i / (K * N);
    const int64_t k = (i / N) % K;
    const int64_t n = i % N;
    out[i] = in[s * Np * Kp + frag_off16(n, k >> 4, Kp) + (k & 15)];
}

}  // namespace

hipError_t launch_slice_s2(const Dims& d, const Operand& A, const Operand& B, const Shifts& shift_A,
                           const Shifts& shift_B, int8_t* A_sl, int8_t* B_sl, hipStream_t st, int words) {
    const ResidueConsts rc = make_residue_consts();
    const SliceOp a = make_slice_op(A.p, d.M, d.Mp, A.ld, A.kcontig, d.Kp, shift_A, A_sl);
    const SliceOp b = make_slice_op(B.p, d.N, d.Np, B.ld, B.kcontig, d.Kp, shift_B, B_sl);
    const unsigned grid = (unsigned)(a.nblk + b.nblk);
    switch (words) {
        case 1: k_slice_s2<1><<<grid, kSliceThreads, 0, st>>>(a, b, d.K, d.Kp, d.S, rc); break;
        case 2: k_slice_s2<2><<<grid, kSliceThreads, 0, st>>>(a, b, d.K, d.Kp, d.S, rc); break;
        default: k_slice_s2<3><<<grid, kSliceThreads, 0, st>>>(a, b, d.K, d.Kp, d.S, rc); break;
    }
    return hipGetLastError();
}

hipError_t launch_slice_s1(const Dims& d, int beta, const Operand& A, const Operand& B, const Shifts& shift_A,
                           const Shifts& shift_B, int8_t* A_sl, int8_t* B_sl, hipStream_t st) {
    const SliceOp a = make_slice_op(A.p, d.M, d.Mp, A.ld, A.kcontig, d.Kp, shift_A, A_sl);
    const SliceOp b = make_slice_op(B.p, d.N, d.Np, B.ld, B.kcontig, d.Kp, shift_B, B_sl);
    k_slice_s1<<<(unsigned)(a.nblk + b.nblk), kSliceThreads, 0, st>>>(a, b, d.K, d.Kp, d.S, beta);
    return hipGetLastError();
}

// Not when one more round of 1024-thread blocks would hold a few blocks only, which take as long as a full
// round, unless there are many rounds: 200 x 8000 x 900, S = 16 (514 row blocks) 120 us per call in one
// pass, 114 us in two kernels; 200 x 7800 x 900 (502) 102 against 109, 200 x 6000 x 900 (389) 88 against 93.
// Past K = 2048 (8 rows per block) up to one round, or two that are well filled; us per call in one pass and in
// two kernels: 512^2 x 4096, S = 14 (128 row blocks) 55 and 62; 1000^2 x 3000, S = 12 (250) 73 and 85;
// 1300 x 700 x 3500, S = 16 (251) 109 and 122; 1500 x 900 x 4000, S = 12 (304) 147 and 144; 1500^2 x 3000, S = 10
// (376) 131 and 132; 3000 x 1000 x 2050, S = 16 (504) 161 and 173; 2100^2 x 2100, S = 15 (528) 220 and 220; 4096^3,
// S = 17 (1024) 1261 and 1249; 300 x 8000 x 2304, S = 12 (1040) 228 and 200.  Past K = 4096 blocks of 4 rows would be
// needed: 512^2 x 8192, S = 14 124 and 98.
bool one_pass(const Dims& d) {
    if (d.Kp > kPassMaxKp) return false;
    const int R = pass_rows(d.Kp);
    const int64_t n = pass_row_blocks(d.M, R) + pass_row_blocks(d.N, R), over = n % kPassResident;
    if (d.Kp > 2048) return n <= kPassResident || (n >= kPassResident * 11 / 8 && n <= 2 * kPassResident);
    return !(pass_threads(d.Kp) == 1024 && n > kPassResident && n < 4 * kPassResident && over > 0 &&
             over < kPassResident / 8);
}

hipError_t launch_one_pass(int scheme, const Dims& d, int offset, const Operand& A, const Operand& B, int32_t* shift_A,
                           int32_t* shift_B, int8_t* A_sl, int8_t* B_sl, hipStream_t st, uint32_t* zero, int nzero) {
    PassArgs g;
    g.K = d.K;
    g.Kp = d.Kp;
    g.S = d.S;
    g.R = pass_rows(d.Kp);
    g.offset = offset;
    g.zero = zero;
    g.nzero = nzero;
    if (nzero > 256) return hipErrorInvalidValue;
    auto op = [&](const Operand& X, int64_t rows, int64_t rows_p, int32_t* shift, int8_t* out) {
        return PassOp{X.p, rows, rows_p, X.ld, X.kcontig, shift, out, pass_row_blocks(rows, g.R)};
    };
    g.op[0] = op(A, d.M, d.Mp, shift_A, A_sl);
    g.op[1] = op(B, d.N, d.Np, shift_B, B_sl);
    const int64_t nrow = g.op[0].nrow + g.op[1].nrow;
    // Parts while the blocks still run at once: 1024^3, S = 16 (128 row blocks) 49 us per call undivided,
    // 45 in two parts, 51 in four; 500 x 500 x 1000 (64) 39, 34 and 33; 777 x 1501 x 1003 (146) 60, 62 and 65.
    g.parts = 1;
    while (2 * g.parts <= std::min(d.S, 8) && nrow * g.parts * 2 <= kPassResident) g.parts *= 2;
    const int64_t grid = (nrow + 7) / 8 * 8 * g.parts;
    if (grid * pass_threads(d.Kp) > (int64_t)UINT32_MAX) return hipErrorInvalidValue;
    const ResidueConsts rc = make_residue_consts();
    if (scheme == 1) return launch_pass_words<0>(g, rc, (unsigned)grid, st);
    switch (residue_words(offset)) {
        case 1: return launch_pass_words<1>(g, rc, (unsigned)grid, st);
        case 2: return launch_pass_words<2>(g, rc, (unsigned)grid, st);
        default: return launch_pass_words<3>(g, rc, (unsigned)grid, st);
    }
}

hipError_t launch_unpack_A(const Dims& d, const int8_t* A_sl, int8_t* out, hipStream_t st) {
    const int64_t tot = (int64_t)d.S * d.M * d.K;
    if (tot == 0) return hipSuccess;
    k_unpack_A<<<(unsigned)((tot + 255) / 256), 256, 0, st>>>(A_sl, d.M, d.K, d.Mp, d.Kp, d.S, out);
    return hipGetLastError();
}

hipError_t launch_unpack_B(const Dims& d, const int8_t* B_sl, int8_t* out, hipStream_t st) {
    const int64_t tot = (int64_t)d.S * d.K * d.N;
    if (tot == 0) return hipSuccess;
    k_unpack_B<<<(unsigned)((tot + 255) / 256), 256, 0, st>>>(B_sl, d.K, d.N, d.Np, d.Kp, d.S, out);
    return hipGetLastError();
}

}  // namespace oza
