// oza_device.hpp — device helpers shared by the gfx950 kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace oza {

// ---- exponent statistics -------------------------------------------------------------------
// The reference takes E = max(-1023, max_k e_k) where frexp(|a|) = f * 2^e, f in [1/2, 1),
// zeros and NaNs skipped (step1_statistics.hpp:33-42).  E depends only on the high word of
// |a|: for normal numbers e = biased_exponent - 1022; a subnormal gives -1022 when mantissa
// bit 51 is set and something <= -1023 otherwise; +-Inf has frexp exponent 0.  E is monotone
// in that high word, so a row maximum of the high word (after mapping NaN -> 0 and
// Inf -> 0x3FE00000, a word whose exponent is 0) gives the row's E.
__device__ __forceinline__ uint32_t exp_key(double x) {
    const uint64_t ab = (uint64_t)__double_as_longlong(x) & 0x7fffffffffffffffull;
    uint32_t hi = (uint32_t)(ab >> 32);
    if (ab > 0x7ff0000000000000ull) hi = 0;                // NaN
    else if (ab == 0x7ff0000000000000ull) hi = 0x3FE00000u;  // Inf: frexp exponent 0
    return hi;
}

__host__ __device__ __forceinline__ int exp_from_key(uint32_t key) {
    const int be = (int)(key >> 20);
    if (be == 0) return (key & 0x80000u) ? -1022 : -1023;
    return be - 1022;
}

// The largest exponent key of N values.  Finite values' keys are their high words without the sign;
// anything else is rare and takes the exact form.
constexpr uint32_t kNonFinite = 0x7ff00000u;
template <int N>
__device__ __forceinline__ uint32_t max_high(const double (&a)[N]) {
    uint32_t m = 0;
#pragma unroll
    for (int j = 0; j < N; ++j) m = max(m, (uint32_t)((uint64_t)__double_as_longlong(a[j]) >> 32) & 0x7fffffffu);
    return m;
}
template <int N>
__device__ __forceinline__ uint32_t max_key(const double (&a)[N]) {
    uint32_t m = max_high(a);
    if (m >= kNonFinite) {
        m = 0;
#pragma unroll
        for (int j = 0; j < N; ++j) m = max(m, exp_key(a[j]));
    }
    return m;
}
// Infinities and NaNs have residue 0 for every modulus.
__device__ __forceinline__ void drop_non_finite(double (&a)[16]) {
    if (max_high(a) >= kNonFinite) {
#pragma unroll
        for (int j = 0; j < 16; ++j)
            if (((uint64_t)__double_as_longlong(a[j]) >> 32 & kNonFinite) == kNonFinite) a[j] = 0.0;
    }
}

// Wave-wide max of a 32-bit unsigned value: DPP within each 16-lane row (quad permutes,
// half-row and row mirrors), then two cross-row exchanges.  All 64 lanes must be active.
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
    v = max(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xF, 0xF, false));   // quad_perm 1,0,3,2
    v = max(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x4E, 0xF, 0xF, false));   // quad_perm 2,3,0,1
    v = max(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x141, 0xF, 0xF, false));  // row_half_mirror
    v = max(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x140, 0xF, 0xF, false));  // row_mirror
    v = max(v, (uint32_t)__shfl_xor((int)v, 16));
    v = max(v, (uint32_t)__shfl_xor((int)v, 32));
    return v;
}

// ---- Scheme II residues and digits ---------------------------------------------------------------
// Integer-valued t, |t| <= 2^(32 ND - 2), as the ND 32-bit words of t + 2^(32 ND - 1) (word 0 lowest).
template <int ND>
__device__ __forceinline__ void int_words(double t, uint32_t (&w)[ND]) {
    static_assert(ND >= 1 && ND <= 3, "one to three words");
#pragma unroll
    for (int n = 0; n + 1 < ND; ++n) {  // exact: t has at most 53 bits, so t - floor(t 2^-32) 2^32 < 2^32 does too
        const double top = floor(t * 0x1p-32);
        w[n] = (uint32_t)fma(-top, 0x1p32, t);
        t = top;
    }
    w[ND - 1] = (uint32_t)(int)t;
    w[ND - 1] ^= 0x80000000u;
}

// Symmetric residue of t mod an odd m < 256, in [-(m-1)/2, (m-1)/2], from t's words: d, the sum of the
// 4 ND bytes times wt (byte k of wt[n] = -2^32 2^(8(4n+k)) mod m) plus init, which takes the words'
// bias off, is congruent to -2^32 t and below 2^20.  With p = d m^-1 mod 2^32 taken as a signed number,
// p m = r 2^32 + d for r = floor(p m / 2^32), so r is congruent to -2^-32 d = t, and |p| <= 2^31
// bounds r to the symmetric range: r + d / 2^32 = p m / 2^32 is in [-m/2, m/2) and d < 2^31 / m keeps
// r > -m/2.  ND + 2 full-rate integer operations against five in FP64 (fma, multiply, rint, fma,
// convert), on ND registers per value instead of four.
template <int ND>
__device__ __forceinline__ int sym_residue(const uint32_t (&w)[ND], const uint32_t (&wt)[ND], uint32_t init, uint32_t m,
                                           uint32_t minv) {
    uint32_t d = init;
#pragma unroll
    for (int n = 0; n < ND; ++n) d = __builtin_amdgcn_udot4(w[n], wt[n], d, false);
    return __mulhi((int)(d * minv), (int)m);
}

// CRT digit v mod m of any INT32 product v, in [0, m), from u = v + 2^31 in [0, 2^32); the addition costs
// nothing, the accumulators start from it (kProductBias).  As in sym_residue: d, the sum of u's four bytes times wt
// (byte k = -2^32 2^(8k) mod m) plus init = 2^32 2^31 mod m, is congruent to -2^32 v and below 2^18 + 2^8; with
// p = d m^-1 mod 2^32 the product p m = r 2^32 + d for r = floor(p m / 2^32) < m, so r is congruent to v.
// Three 32-bit instructions (full rate, four cycles per wave like every instruction here) against five for
// an FP64 quotient.  With a multiple of m for the 2^31 there would be no init, but the products past
// 2^32 minus it, up to 250 of them, would wrap.
constexpr uint32_t kProductBias = 0x80000000u;
__device__ __forceinline__ uint32_t product_digit(uint32_t u, uint32_t wt, uint32_t init, uint32_t m, uint32_t minv) {
    return __umulhi(__builtin_amdgcn_udot4(u, wt, init, false) * minv, m);
}

// ---- MFMA-fragment-tiled operand planes -------------------------------------------------------
// An operand plane (rows x Kp bytes, rows = M or N padded to 256, K contiguous) is stored as 1 KiB
// blocks of 32 rows x 32 K-bytes, block (rb, kb) at ((rb * Kp/32) + kb) * 1024.  Inside a block the
// 16-byte unit of lane l holds row l%32, K-bytes 16*(l/32) .. +15: exactly the register operand
// of lane l for v_mfma_i32_32x32x32_i8, so one wave moves a fragment with a single contiguous
// 1 KiB load (global -> LDS -> registers).  frag_off16 gives the byte offset of the 16-byte unit
// holding row `row`, K-bytes 16*c .. 16*c+15.
__host__ __device__ __forceinline__ int64_t frag_off16(int64_t row, int64_t c, int64_t Kp) {
    return (((row >> 5) * (Kp >> 5) + (c >> 1)) << 10) + (((row & 31) + ((c & 1) << 5)) << 4);
}

// ---- address spaces -------------------------------------------------------------------------------
// A 16-byte store through a global (address space 1) pointer.  Through a generic pointer the
// compiler emits a flat store, which may address LDS, and so first waits for every direct
// global->LDS load in flight (vmcnt(0)); a global store carries no such wait.
// NT: nontemporal (a wave instruction writes whole lines, and the data is not read back soon).
template <bool NT = false>
__device__ __forceinline__ void store_global16(void* p, uint32_t x, uint32_t y, uint32_t z, uint32_t w) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    const u32x4 v = {x, y, z, w};
    if (NT) __builtin_nontemporal_store(v, (__attribute__((address_space(1))) u32x4*)p);
    else *(__attribute__((address_space(1))) u32x4*)p = v;
}

// Read-only data in global memory seen as constant (address space 4): uniform reads become scalar
// loads, which are counted apart from the vector loads (lgkmcnt, not vmcnt), so waiting for them
// does not also wait for the direct loads in flight.
template <class T>
__device__ __forceinline__ const __attribute__((address_space(4))) T* as_constant(const T* p) {
    return (const __attribute__((address_space(4))) T*)p;
}

// Streaming loads of operands read once per pass (nontemporal: not kept in the caches).  Only for
// accesses whose wave covers whole cache lines in one instruction: a line read piecewise by
// several nontemporal loads is fetched from memory each time (slicing's 16-byte-per-lane row
// reads ran 25 % slower with them; the statistics' contiguous wave reads 11 % faster).
__device__ __forceinline__ double2 load_stream2(const double* p) {
    typedef double d2 __attribute__((ext_vector_type(2)));
    const d2 v = __builtin_nontemporal_load(reinterpret_cast<const d2*>(p));
    return make_double2(v.x, v.y);
}
__device__ __forceinline__ double load_stream(const double* p) { return __builtin_nontemporal_load(p); }

// 16-byte store of a plane unit, nontemporal with NT (every use writes a whole 1 KiB fragment block
// or half of one per wave instruction, so whole lines).  The grouped pipeline uses NT: its many
// small planes are not read again while still cached (grouped steps 2 and 3 -2.5 % and -5 %),
// whereas at 8192^3 it was neutral (slower slicing, slightly faster GEMM).
template <bool NT>
__device__ __forceinline__ void store_unit16(void* p, uint4 v) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    const u32x4 x = {v.x, v.y, v.z, v.w};
    if (NT) __builtin_nontemporal_store(x, reinterpret_cast<u32x4*>(p));
    else *reinterpret_cast<u32x4*>(p) = x;
}

// ---- byte packing ---------------------------------------------------------------------------------
// Low bytes of four values (any sign) into one word (byte 0 = a): v_perm_b32 picks byte 0 of each
// source (selector 0-3: second source, 4-7: first source, 0x0c: zero).
__device__ __forceinline__ uint32_t pack4_lo(int a, int b, int c, int d) {
    const uint32_t ab = __builtin_amdgcn_perm((uint32_t)b, (uint32_t)a, 0x0c0c0400u);
    const uint32_t cd = __builtin_amdgcn_perm((uint32_t)d, (uint32_t)c, 0x04000c0cu);
    return ab | cd;
}

}  // namespace oza
