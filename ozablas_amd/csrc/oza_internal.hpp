// oza_internal.hpp — definitions shared by the gfx950 kernels and the C-ABI layer.
//
// HBM layout of one Ozaki workspace (all planes dense, device memory):
//   shift_A   int32[M]                   row shifts (reference semantics, step1_statistics.hpp:23-76)
//   shift_B   int32[N]                   column shifts
//   A_slices  int8 [S][Mp][Kp]           A residues/slices, K contiguous, fragment-tiled (frag_off16)
//   B_slices  int8 [S][Np][Kp]           B residues/slices TRANSPOSED (column n is a K-contiguous row)
//   C_tc      Scheme II: uint8 [S][Mp][Np] digits C_s mod m_s in 32 x 32 element blocks,
//                        then the partial tiles of items that ran in K parts (S2Plan)
//             Scheme I : int32 [S][Mp][Np] group products T_g in 32 x 32 element blocks, then the planes of
//                        groups that ran in parts (S1Plan) (the stage entry point writes the reference's
//                        planar int32 [S][M][N] instead)
// with Mp = roundup(M, 256), Np = roundup(N, 256), Kp = roundup(K, 128).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace oza {

constexpr int kMaxSlices = 20;
constexpr int kPadMN = 256;  // row padding of the operand planes (largest GEMM tile edge)
constexpr int kPadK = 128;   // K padding of the operand planes (largest K stage)

inline size_t round_up(size_t x, size_t m) { return (x + m - 1) / m * m; }

// The Scheme II moduli, identical to the reference list (src/common/crt_tables.hpp:13-16).
inline constexpr uint8_t kModuli[kMaxSlices] = {251, 241, 239, 233, 229, 227, 223, 211, 199, 197,
                                                193, 191, 181, 179, 173, 167, 163, 157, 151, 149};

// Bit length of M(S) = m_0 * ... * m_{S-1}, at compile time.
constexpr int bitlen_M(int S) {
    uint64_t d[4] = {1, 0, 0, 0};  // 256-bit little-endian
    for (int s = 0; s < S; ++s) {
        unsigned __int128 carry = 0;
        for (int i = 0; i < 4; ++i) {
            const unsigned __int128 p = (unsigned __int128)d[i] * kModuli[s] + carry;
            d[i] = (uint64_t)p;
            carry = p >> 64;
        }
    }
    for (int i = 3; i >= 0; --i)
        if (d[i]) {
            int b = 64 * i;
            for (uint64_t v = d[i]; v; v >>= 1) ++b;
            return b;
        }
    return 0;
}
static_assert(bitlen_M(8) == 63 && bitlen_M(16) == 124 && bitlen_M(20) == 153, "moduli products");

// Per-S CRT constants used by the kernels.  Big integers are little-endian 32-bit words.
//
// The moduli s = 0..S-1 are taken in groups of three, g = s / 3 (the last one may be shorter), with
// P_g the product of a group's moduli (< 2^24).  With the group sums
//   u_g = sum_{s in g} c_s (P_g / m_s)            (24-bit operands, u_g < 3 * 2^24)
// and the constants R_g = w_g (M / P_g), w_g < P_g with w_g (M / m_s) = 1 mod m_s for every s in g,
//   X = sum_g u_g R_g = C (mod M)   whenever   c_s = C mod m_s for all s.
constexpr int kWords = 5;                          // 160 bits: M < 2^153 and a sign
constexpr int kGroups = (kMaxSlices + 2) / 3;
struct CrtSet {
    int S;
    uint32_t E[kMaxSlices];           // P_g / m_s (< 2^16; 1 in a group of one)
    uint32_t F[kGroups];              // floor(2^32 R_g / M) = floor(2^32 w_g / P_g)
    uint32_t amb;                     // fractional part of the quotient estimate from which on it may be one short
    uint32_t R[kGroups][kWords];
    uint32_t Mneg[kWords];            // 2^160 - M
    uint32_t M32[kWords], Mhalf32[kWords];  // M and floor(M/2)
    // product_digit: m_s, m_s^-1 mod 2^32, the byte weights, and m_s + 2^8 (2^63 mod m_s) in one word
    uint32_t m[kMaxSlices], minv[kMaxSlices], wt[kMaxSlices], m_init[kMaxSlices];
    uint64_t M64[4];                  // M in 64-bit words
};

// All S = 1..20, computed on the host from the moduli (closed forms).
struct CrtTables {
    CrtSet set[kMaxSlices];  // set[S-1]
};
const CrtTables& host_crt_tables();

// Host-side parameters (reference: step1_statistics.hpp:12-20, pipeline.hip:205-207).
int scheme1_beta(size_t K);
int scheme2_kparam(int S, size_t K);
int scheme2_slices_for_digits(size_t K, double digits);
double scheme2_spread_shortfall(double spread);
int scheme2_slices_for_accuracy(size_t K, double digits, double spread);

// ------------------------------------------------------------------------------------------
// Launchers (each enqueues on `stream`, returns hipError_t from hipGetLastError()).
// ------------------------------------------------------------------------------------------
struct Dims {
    int64_t M, N, K;
    int64_t Mp, Np, Kp;
    int S;
};
Dims make_dims(size_t M, size_t N, size_t K, int S);

// An FP64 operand as steps 1 and 2 read it: logical rows (M rows of op(A), or the N columns of
// op(B)) of K values each, element (r, k) at p[r * ld + k] when kcontig, else at p[k * ld + r].
// The reference's dense row-major A is {A, K, true}, its B is {B, N, false}.
struct Operand {
    const double* p;
    int64_t ld;
    bool kcontig;
};
// The output of step 4: C[i * ldc + j] = alpha * X_ij + beta * C[i * ldc + j], evaluated as
// fma(alpha, X, beta * C); with beta == 0, C is not read and alpha == 1 stores X itself.
struct OutC {
    double* p;
    int64_t ldc;
    double alpha, beta;
};

// C = beta * C over an M x N block with leading dimension ldc (beta == 0 writes zeros).
hipError_t launch_scale_c(const OutC& c, int64_t M, int64_t N, hipStream_t st);

// Step 1: shift_A[i] = offset - E_i, shift_B[j] = offset - F_j.
hipError_t launch_stats(const Dims& d, const Operand& A, const Operand& B, int32_t offset, int32_t* shift_A,
                        int32_t* shift_B, hipStream_t st);

// Where a slicing block finds its rows' shifts: in `shift`, or (part != null) from step 1's partial
// maxima, `parts` (at most kStatParts) planes of `rows` exponent keys, whose maximum it turns into
// offset - exponent and stores in `shift`.
constexpr int kStatParts = 32;
struct Shifts {
    int32_t* shift;
    const uint32_t* part;
    int32_t parts, offset;
    int64_t rows;
};
// Step 1 into partial maxima at `scratch`, at most 128 (M + N) bytes (the digit planes hold S Mp Np, with
// Mp and Np at least 256); out: the shifts for step 2.  The launch also clears nzero words at `zero` (the
// work counters of the call's step-3 GEMMs).
hipError_t launch_stats_parts(const Dims& d, const Operand& A, const Operand& B, int32_t offset, int32_t* shift_A,
                              int32_t* shift_B, void* scratch, Shifts out[2], hipStream_t st, uint32_t* zero,
                              int nzero);

// Step 2.  words: 32-bit words per scaled value, |rint(2^shift a)| <= 2^(32 words - 2)
// (core::residue_words(K_param) with step 1's shifts).
hipError_t launch_slice_s2(const Dims& d, const Operand& A, const Operand& B, const Shifts& shift_A,
                           const Shifts& shift_B, int8_t* A_sl, int8_t* B_sl, hipStream_t st, int words);
hipError_t launch_slice_s1(const Dims& d, int beta, const Operand& A, const Operand& B, const Shifts& shift_A,
                           const Shifts& shift_B, int8_t* A_sl, int8_t* B_sl, hipStream_t st);
// Steps 1 and 2 in one launch, for shapes with one_pass(d): offset is K_param (scheme 2) or beta
// (scheme 1); zero / nzero as in launch_stats_parts.
bool one_pass(const Dims& d);
hipError_t launch_one_pass(int scheme, const Dims& d, int offset, const Operand& A, const Operand& B, int32_t* shift_A,
                           int32_t* shift_B, int8_t* A_sl, int8_t* B_sl, hipStream_t st, uint32_t* zero, int nzero);
// Unpack product-layout operand planes to the reference's planar layout [s][rows][cols].
hipError_t launch_unpack_A(const Dims& d, const int8_t* A_sl, int8_t* out, hipStream_t st);
hipError_t launch_unpack_B(const Dims& d, const int8_t* B_sl, int8_t* out, hipStream_t st);

// Division of 32-bit numbers by d in five scalar instructions (div_fast): inv = floor(2^32 / d), so that
// mulhi(n, inv) is the quotient or one less (for d = 1, inv = 2^32 - 1 gives n - 1).
struct FastDiv {
    uint32_t d, inv;
};
inline FastDiv fast_div(int64_t d) {
    return FastDiv{(uint32_t)d, d > 1 ? (uint32_t)((uint64_t(1) << 32) / (uint64_t)d) : UINT32_MAX};
}
// The order of a GEMM's tiles: groups of gm tile rows (IgemmCfg::GM), column by column (grouped_tile).
struct TileOrder {
    int32_t tiles_m, tiles_n;
    FastDiv tiles, group, last;  // all tiles; a group's tiles; the rows of the last, smaller group
};
inline TileOrder tile_order(int64_t tiles_m, int64_t tiles_n, int gm) {
    return TileOrder{(int32_t)tiles_m, (int32_t)tiles_n, fast_div(tiles_m * tiles_n), fast_div(gm * tiles_n),
                     fast_div(tiles_m % gm ? tiles_m % gm : gm)};
}

// How a single call's GEMM is cut into items (plan_host.cpp).
constexpr int kS2TileRows = 256;
constexpr int kTileBytes = kS2TileRows * kS2TileRows;  // digits of one tile
constexpr int kMaxParts = 32;
constexpr int kMaxS1Planes = 128;
// Scheme II: items l (modulus-major, then tile) below `whole` run whole, the others in `parts` parts of
// `kts` K steps (the last one may be shorter).  edge: 64 or 128 for small calls, whose tiles of that size
// all run whole.
struct S2Plan {
    int edge = kS2TileRows, parts = 1, kts = 0;
    int64_t whole = 0;
};
S2Plan scheme2_plan(const Dims& d);
// Whether the 256 x 256 tiles of a plan (or of none: S2Plan{}) run on a ring of four slots.
bool s2_deep_ring(const Dims& d, const S2Plan& p);
// Digit tiles that a plan writes (65536 bytes each).
int64_t s2_plan_tiles(const Dims& d, const S2Plan& p);
// Scheme I: group g + 2 (g + 1 pairs) runs in parts[g] equal runs of its stages; the first part's INT32
// plane is plane g, the other parts' follow the S planes, group after group.  edge: as in S2Plan.
struct S1Plan {
    int edge = kS2TileRows;
    int parts[kMaxSlices] = {};
    int planes = 0;
};
S1Plan scheme1_plan(const Dims& d);
// C_tc tiles (of digits, of INT32) that hold the plan of this shape and of every smaller one.
int64_t s2_most_tiles(const Dims& d);
int64_t s1_most_tiles(const Dims& d);

// Step 3 (+ fused epilogues).
enum class S2Out { Digits, Int32 };
// Tile rows [tm0, tm0 + tms) of BM = 256 rows (tms < 0: to the last tile row).
// plan (Digits only, or null: every item whole): items past plan->whole run in plan->parts parts of
// plan->kts K steps; part 0 writes the digits of its partial product to the S digit planes, part j > 0
// to the partial tiles behind them, tile (j - 1) * tail + (item - whole) in the blocked layout of one tile.
hipError_t launch_igemm_s2(const Dims& d, const int8_t* A_sl, const int8_t* B_sl, S2Out mode, void* out,
                           const CrtSet* crt_dev, hipStream_t st, int tm0 = 0, int tms = -1,
                           const S2Plan* plan = nullptr);
// Scheme I: group products T_g, g = 2..S+1, into blocked INT32 planes (32 x 32 blocks), one per group,
// or per part of a group with a plan: [planes][Mp][Np].
// Tile rows [tm0, tm0 + tms) of 256 rows (tms < 0: to the last tile row).  queue: 8 device counters for
// the dynamic work order, zero when the launch starts, or null (static order).
hipError_t launch_igemm_s1_blocked(const Dims& d, const int8_t* A_sl, const int8_t* B_sl, int32_t* T, hipStream_t st,
                                   const S1Plan& plan, unsigned* queue = nullptr, int tm0 = 0, int tms = -1);
// Scheme I: group products T_g only, int32 [S][M][N] (reference C_tc semantics per group).
hipError_t launch_igemm_s1_groups(const Dims& d, const int8_t* A_sl, const int8_t* B_sl, int32_t* T,
                                  hipStream_t st);

// Step 4.
// Rows [row0, row0 + rows) of C (row0 a multiple of 32; rows < 0: to the last row).  narrow: one
// workgroup per CU walks the blocks, leaving room on each CU for a concurrent step-3 workgroup.  plan:
// launch_igemm_s2's; the parts' digits are added modulo m_s first, in place.
hipError_t launch_recon_s2_digits(const Dims& d, uint8_t* digits, const int32_t* shift_A,
                                  const int32_t* shift_B, const CrtSet* crt_dev, const OutC& C, hipStream_t st,
                                  int64_t row0 = 0, int64_t rows = -1, bool narrow = false,
                                  const S2Plan* plan = nullptr);
hipError_t launch_recon_s2_int32(const Dims& d, const int32_t* C_tc, const int32_t* shift_A,
                                 const int32_t* shift_B, const CrtSet* crt_dev, double* C, hipStream_t st);
// Blocked digit planes <-> planar [s][M][N] digits in [0, m_s) (pack reduces its input mod m_s).
hipError_t launch_digits_unpack(const Dims& d, const uint8_t* digits, uint8_t* out, hipStream_t st);
hipError_t launch_digits_pack(const Dims& d, const uint8_t* planar, const CrtSet* crt_dev, uint8_t* digits,
                              hipStream_t st);
// Scheme I step 4 from blocked planes: T_g = the sum of its parts' planes (left in the first of them),
// C = fma(T_g, scale_g, C) for g ascending, then the output rule.
hipError_t launch_recon_s1_blocked(const Dims& d, int beta, int32_t* T, const int32_t* shift_A,
                                   const int32_t* shift_B, const OutC& C, hipStream_t st, const S1Plan& plan,
                                   int64_t row0 = 0, int64_t rows = -1, bool narrow = false);
hipError_t launch_recon_s1_groups(const Dims& d, int beta, const int32_t* T, const int32_t* shift_A,
                                  const int32_t* shift_B, double* C, hipStream_t st);

// Accuracy helpers: double-double GEMM (C_hi = the dd dot product rounded to FP64, optional
// C_abs = |A||B| in FP64) and error statistics of `actual` against `exact`.
hipError_t launch_dd_gemm(int64_t M, int64_t N, int64_t K, const double* A, const double* B, double* C_hi,
                          double* C_abs, hipStream_t st);
// stats (device, 4 doubles, zeroed by the launcher): max |d|, max |d|/|e| (|d| when e == 0),
// max |d|/absab (absab optional), count of mismatching bit patterns.
hipError_t launch_error_stats(int64_t n, const double* exact, const double* actual, const double* absab,
                              double* stats, hipStream_t st);
// INT8 MFMA rate with operands in registers (random residues or zeros), `grid` workgroups of 8 waves;
// acc4 (device, 4 x 64-bit, zeroed by the launcher) receives the summed shader-clock cycles and
// 100 MHz ticks of thread 0 of every workgroup.
hipError_t launch_mfma_ceiling(int iters, bool zero, unsigned grid, double* acc4, hipStream_t st);

}  // namespace oza
