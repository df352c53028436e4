// k_igemm.hip — step 3: INT8 x INT8 -> INT32 GEMMs on gfx950 matrix cores, with fused epilogues.
//
// Operands come from step 2 as fragment-tiled INT8 planes (A [s][Mp][Kp], B transposed
// [s][Np][Kp]), so every MFMA operand fragment is one contiguous 1 KiB block.  A workgroup owns a
// BM x BN output tile; each of its waves owns a (BM/NWM) x (BN/NWN) sub-tile made of 32x32
// v_mfma_i32_32x32x32_i8 fragments with exact INT32 accumulation (mainloop in igemm_core.hpp).
//
//   Scheme II (reference: rocblas_gemm_strided_batched_ex, src/hip/pipeline.hip:237-245):
//     one launch covers every (tile, modulus); the epilogue reduces C_s to its CRT digit
//     modulo m_s (product_digit) and stores it as one byte (layout below), or stores
//     the raw INT32 C_s planes in the reference's [s][M][N] layout.
//   Scheme I (reference: rocblas_gemm_ex loop, pipeline.hip:110-135): one launch covers every
//     (group g, tile); the pairs of group g = s + t accumulate into one INT32 fragment set and
//     T_g is stored as a blocked INT32 plane; step 4 (k_recon.hip) sums the groups in FP64 in
//     the reference's ascending order.  The planar form for the stage entry point walks all
//     pairs per tile and writes [g-2][M][N].
//
// Digit layout (Scheme II, C_tc workspace): planes [s] of Mp x Np bytes in 32 x 32 element
// blocks, row-major over blocks, each block in the MFMA 32x32 output order (see store_digits);
// Scheme I's T planes use the same blocking with INT32 elements (store_i32_blocked).
#include <algorithm>

#include "igemm_core.hpp"
#include "recon_core.hpp"

namespace oza {
namespace {

using namespace core;

// ------------------------------------------------------------------------------------------
// Work order of the persistent GEMMs (one workgroup per CU).  Scheme II's items are all of one length:
// workgroup b takes positions b, b + gridDim.x, ... of the item list through xcd_remap, so that each XCD
// (workgroup b runs on XCD b % 8) works through a contiguous run and its tiles in flight share their
// operand panels in L2.  Taking positions from per-XCD counters instead, to keep them neighbours when
// CUs drift apart, fetched 13.4 GB at 8192^3 unbanded (13.8 in this order), and the
// claim's wait costs 0.6 % (8192^3, S = 17: 8.715 against 8.667 ms; 4096^2 x 1024, S = 16: 415 against
// 410 us).  Scheme I's items differ in length and do take them from counters (Claims below).
// ------------------------------------------------------------------------------------------

// ------------------------------------------------------------------------------------------
// Scheme II
// ------------------------------------------------------------------------------------------
struct S2Args {
    const int8_t* A;
    const int8_t* B;
    int64_t M, N, Mp, Np, Kp;
    int S, KT;
    TileOrder order;       // of the tile rows [tm0, tm0 + order.tiles_m)
    int tm0;
    void* out;             // digits or int32 planes
    const CrtSet* crt;     // device copy (m_init, minv, wt used)
    // SPLIT only: items [0, whole) run whole, the `tail` others in `parts` parts of kts K steps
    uint32_t items, whole, tail;
    FastDiv by_tail;
    int parts, kts;
    uint8_t* part;         // partial tiles of parts 1..
};

// Work items (modulus, tile) in logical order l = 0..total-1: modulus-major; inside a modulus,
// tiles in groups of GM tile rows.  SPLIT: the whole items first, then the others' parts, part-major, part
// j over K steps [j kts, min((j + 1) kts, KT)).
template <class C, bool DIGITS, bool SPLIT = false>
__global__ void __launch_bounds__(C::NT) k_igemm_s2(S2Args p) {
    __shared__ __attribute__((aligned(1024))) int8_t smem[C::LDS_BYTES];
    uint32_t w = blockIdx.x;
    if (w >= p.items) return;  // whole workgroup leaves together
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave_part<C>(wave).m, wn = wave_part<C>(wave).n;
    struct Item {
        int s, tm, tn, j, k0, KT;
        uint32_t l;
        StageSrc src;  // this wave's blocks of stage 0
        uint32_t m_init, minv, wt;
    };
    auto decode = [&](uint32_t wi) {
        Item t;
        uint32_t l = SPLIT && wi >= p.whole ? p.whole + xcd_remap(wi - p.whole, p.items - p.whole)
                                            : xcd_remap(wi, SPLIT ? p.whole : p.items);
        t.j = 0;
        t.k0 = 0;
        t.KT = p.KT;
        if (SPLIT && l >= p.whole) {
            uint32_t item;
            t.j = (int)div_fast(l - p.whole, p.by_tail, item);
            l = p.whole + item;
            t.k0 = t.j * p.kts;
            t.KT = min(p.kts, p.KT - t.k0);
        }
        t.l = l;
        uint32_t tile;
        t.s = (int)div_fast(l, p.order.tiles, tile);
        grouped_tile<C>(tile, p.order, t.tm, t.tn);
        t.tm += p.tm0;
        // tile (tm, tn) starts at block-row tm*BM/32 of the fragment-tiled planes (BM*Kp bytes)
        t.src = wave_src<C>(p.A + (int64_t)t.s * p.Mp * p.Kp + (int64_t)t.tm * C::BM * p.Kp + (int64_t)t.k0 * C::STEP,
                            p.B + (int64_t)t.s * p.Np * p.Kp + (int64_t)t.tn * C::BN * p.Kp + (int64_t)t.k0 * C::STEP, p.Kp,
                            wave, (int)((p.M - (int64_t)t.tm * C::BM - 1) >> 5), (int)((p.N - (int64_t)t.tn * C::BN - 1) >> 5));
        // scalar loads: counted by lgkmcnt, so the epilogue does not wait for the direct loads
        t.m_init = as_constant(p.crt)->m_init[t.s];
        t.minv = as_constant(p.crt)->minv[t.s];
        t.wt = as_constant(p.crt)->wt[t.s];
        return t;
    };
    auto stage = [](const Item& t, int i) {  // stage i of an item; its last one past that
        const int64_t o = (int64_t)min(i, t.KT - 1) * C::STEP;
        return StageSrc{t.src.a + o, t.src.b + o};
    };
    auto step = [](StageSrc& c) {
        c.a += C::STEP;
        c.b += C::STEP;
    };
    Item cur = decode(w);
    if constexpr (C::STAGES == 2) chain_start<C>(smem, 0, cur.KT, stage(cur, 0), stage(cur, 1));
    else chain_start_deep<C>(smem, cur.KT, cur.src, step);
    int base = 0;  // ring slot of the current item's stage 0
    for (;;) {
        w += gridDim.x;
        const bool more = w < p.items;
        Item nxt = cur;
        auto entry = [&] {
            if (more) nxt = decode(w);
            if constexpr (C::STAGES == 2) return NextSrc{stage(nxt, 0), stage(nxt, 1)};
            else return nxt.src;
        };
        const int s = cur.s;
        const int64_t row0 = (int64_t)cur.tm * C::BM + wm * C::WTM, col0 = (int64_t)cur.tn * C::BN + wn * C::WTN;
        for_part<C>(
            p.M - row0, p.N - col0,
            [&]<class P>() {
                v16i acc[P::FM][P::FN];
                if (DIGITS) fill_acc<P>(acc, (int)kProductBias);
                else zero_acc<P>(acc);
                mainloop_chain<P>(acc, smem, base, cur.KT, stage(cur, C::STAGES), step, entry);
                if (DIGITS) {
                    const bool part = SPLIT && cur.j > 0;  // a partial tile: the blocks of one tile, row-major
                    uint8_t* plane = part ? p.part + (int64_t)((cur.j - 1) * p.tail + cur.l - p.whole) * kTileBytes
                                          : reinterpret_cast<uint8_t*>(p.out) + (int64_t)s * p.Mp * p.Np;
                    store_digits<P, false>(acc, plane, part ? C::BN : p.Np, part ? wm * C::WTM : row0,
                                           part ? wn * C::WTN : col0, p.M, p.N, cur.wt, cur.m_init, cur.minv, lane);
                } else {
                    int32_t* o = reinterpret_cast<int32_t*>(p.out) + (int64_t)s * p.M * p.N;
#pragma unroll
                    for (int fm = 0; fm < P::FM; ++fm)
#pragma unroll
                        for (int fn = 0; fn < P::FN; ++fn) {
                            const int64_t col = col0 + fn * 32 + (lane & 31);
#pragma unroll
                            for (int j = 0; j < 16; ++j) {
                                const int64_t row = row0 + fm * 32 + frag_row(j, lane);
                                if (row < p.M && col < p.N) o[row * p.N + col] = acc[fm][fn][j];
                            }
                        }
                }
            },
            [&] { mainloop_idle<C>(smem, base, cur.KT, stage(cur, C::STAGES), step, entry); });
        if (!more) break;
        base = (base + cur.KT) & (C::STAGES - 1);
        cur = nxt;
    }
    wait_vmcnt<0>();  // no direct load in flight into LDS when the workgroup leaves
}

// ------------------------------------------------------------------------------------------
// Scheme I
// ------------------------------------------------------------------------------------------
struct Claims {
    uint32_t w, w1;  // positions of the current and the next item
};

// First two positions of a workgroup.  Dynamic order: the first position is the workgroup's index
// among those of its XCD (blockIdx.x / 8), so that the first round runs the first items of the
// XCD's run side by side -- neighbours, which share operand panels (and, for Scheme I, the pair
// sequence of one group) -- and every later position comes from the XCD's counter, past that first
// round (publish_claim adds the same offset).  Two claims from the counter up front would hand the
// first claimants every other item of the first two rounds and leave the later ones with nothing
// when the run is short.  Positions only grow, so when the first is past the end so is the second.
template <bool DYN>
__device__ __forceinline__ Claims first_claims(unsigned* queue, int xcd, unsigned* s_pos) {
    Claims c;
    if (DYN) {
        if (threadIdx.x == 0) s_pos[1] = (gridDim.x >> 3) + atomicAdd(&queue[xcd], 1u);
        __syncthreads();
        c.w = blockIdx.x >> 3;
        c.w1 = __builtin_amdgcn_readfirstlane(s_pos[1]);
    } else {
        c.w = blockIdx.x;
        c.w1 = 2 * gridDim.x - 1 - c.w;
    }
    return c;
}

// Position of the item after next, from the ticket thread 0 took (dynamic order).  Every wave read
// s_pos[1] at the previous publication and has passed the current item's barriers since; the
// barrier here makes the new value visible.
__device__ __forceinline__ uint32_t publish_claim(unsigned ticket, unsigned* s_pos) {
    if (threadIdx.x == 0) s_pos[1] = (gridDim.x >> 3) + ticket;
    wait_lgkmcnt0();
    block_sync_lds();
    return __builtin_amdgcn_readfirstlane(s_pos[1]);
}

struct S1Args {
    const int8_t* A;
    const int8_t* B;
    int64_t M, N, Mp, Np, Kp;
    int S, KT;
    TileOrder order;         // of the tile rows [tm0, tm0 + order.tiles_m)
    int tm0;                 // blocked form only, else 0
    FastDiv by_KT;
    FastDiv by_share, by_share1;  // an XCD's share of the tiles, rounded down, and one more (dynamic order)
    int32_t* T;              // group products: int32 [S][M][N], or blocked [planes][Mp][Np]
    unsigned* queue;         // 8 work counters, zero at launch (dynamic order), or null (static order)
};

// A wave's place in the stages of group g of a tile (pairs s = 1..g-1, t = g - s, in the reference's
// ascending-s order, KT stages each), moved on stage by stage: the next K step, or the next pair's first.
struct S1Cursor {
    const int8_t* a;
    const int8_t* b;
    int kt;
};
template <class C>
struct S1Walk {
    int64_t wrapA, wrapB;  // from a pair's last stage to the next pair's first
    int KT;
    FastDiv by_KT;
    __device__ __forceinline__ S1Walk(const S1Args& p)
        : wrapA(p.Mp * p.Kp - (int64_t)(p.KT - 1) * C::STEP), wrapB(-p.Np * p.Kp - (int64_t)(p.KT - 1) * C::STEP), KT(p.KT), by_KT(p.by_KT) {}
    // Stage i of group g; abase, bbase: the wave's blocks of the tile in slice 1's planes.
    __device__ __forceinline__ S1Cursor at(const StageSrc& base, const S1Args& p, int g, int i) const {
        uint32_t k;
        const int pr = (int)div_fast((uint32_t)i, by_KT, k), kt = (int)k;  // s = pr + 1, t = g - s
        return S1Cursor{base.a + pr * p.Mp * p.Kp + (int64_t)kt * C::STEP,
                        base.b + (g - pr - 2) * p.Np * p.Kp + (int64_t)kt * C::STEP, kt};
    }
    __device__ __forceinline__ void operator()(S1Cursor& c) const {
        const bool wrap = c.kt + 1 == KT;
        c.a += wrap ? wrapA : (int64_t)C::STEP;
        c.b += wrap ? wrapB : (int64_t)C::STEP;
        c.kt = wrap ? 0 : c.kt + 1;
    }
    __device__ __forceinline__ NextSrc next(const StageSrc& base, const S1Args& p, int g, int i0, int nit) const {
        const S1Cursor s0 = at(base, p, g, i0);
        S1Cursor s1 = s0;
        if (nit >= 2) (*this)(s1);
        return NextSrc{{s0.a, s0.b}, {s1.a, s1.b}};
    }
};

// The items of one tile in the blocked form, longest first: stages [i0, i0 + nit) of group g into plane
// `plane`.  32-bit fields: read by scalar loads, while bytes would take vector loads, and a wait for those
// is one for the ring's loads too.
struct S1Entry {
    uint32_t g_plane;  // g | plane << 16
    uint32_t i0, nit;
};
struct S1List {
    int n;
    S1Entry e[kMaxS1Planes];
};

// Scheme I group products in the reference's planar layout (the stage entry point): one
// workgroup per tile; its items are the groups g = s + t = 2..S+1 in ascending order
// (src/hip/pipeline.hip:110-135), chained through the ring; each finished T_g is stored to
// int32 [g-2][M][N].
template <class C>
__global__ void __launch_bounds__(C::NT) k_igemm_s1(S1Args p) {
    __shared__ __attribute__((aligned(1024))) int8_t smem[C::LDS_BYTES];
    int tm, tn;
    grouped_tile<C>(xcd_remap(blockIdx.x, p.order.tiles.d), p.order, tm, tn);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave_part<C>(wave).m, wn = wave_part<C>(wave).n;
    const StageSrc src =
        wave_src<C>(p.A + (int64_t)tm * C::BM * p.Kp, p.B + (int64_t)tn * C::BN * p.Kp, p.Kp, wave);
    const S1Walk<C> walk(p);
    const NextSrc first = walk.next(src, p, 2, 0, p.KT);
    chain_start<C>(smem, 0, p.KT, first.s0, first.s1);
    int base = 0;
    for (int g = 2; g <= p.S + 1; ++g) {
        const int nit = (g - 1) * p.KT;
        auto entry = [&] {  // the next group, or this one again (a refetch)
            return g <= p.S ? walk.next(src, p, g + 1, 0, nit + p.KT) : walk.next(src, p, g, 0, nit);
        };
        v16i acc[C::FM][C::FN];
        zero_acc<C>(acc);
        mainloop_chain<C>(acc, smem, base, nit, walk.at(src, p, g, min(2, nit - 1)), walk, entry);
        int32_t* o = p.T + (int64_t)(g - 2) * p.M * p.N;
#pragma unroll
        for (int fm = 0; fm < C::FM; ++fm)
#pragma unroll
            for (int fn = 0; fn < C::FN; ++fn) {
                const int64_t col = (int64_t)tn * C::BN + wn * C::WTN + fn * 32 + (lane & 31);
#pragma unroll
                for (int j = 0; j < 16; ++j) {
                    const int64_t row = (int64_t)tm * C::BM + wm * C::WTM + fm * 32 + frag_row(j, lane);
                    if (row < p.M && col < p.N) o[row * p.N + col] = acc[fm][fn][j];
                }
            }
        base = (base + nit) & 1;
    }
    wait_vmcnt<0>();  // no direct load in flight into LDS when the workgroup leaves
}

// Scheme I group products with the 256 x 256 tile of the Scheme II GEMM: work item = (group g,
// tile); the pairs s = 1..g-1 (t = g - s) of the group accumulate in INT32 through one pass of
// the chained mainloop, and T_g is stored as a blocked INT32 plane (store_i32_blocked).  The
// FP64 sum over groups is step 4 (k_recon_s1_blocked).
// A group may run in parts (S1List), each over its own stages into its own plane; step 4 adds them.
// Work order: items differ in length, so the XCDs split the tiles, not the items: XCD x (workgroups b
// with b % 8 == x) owns the tiles [x*T/8, (x+1)*T/8) of the grouped tile order in every list entry, and
// walks its items longest entry first, then tile -- every XCD gets the same mix of work and its CUs share
// A and B panels in L2.  The workgroups of XCD x take the positions of its sequence in the order they ask
// for them (counter queue[x]).  Without counters (few tiles, whose shares would be uneven, or few items,
// see the launcher) the workgroups walk one list over all tiles, longest first, back and forth: round r
// takes position r * G + b of G workgroups, or (r + 1) * G - 1 - b when r is odd, so that a workgroup with
// a long item gets a short one next.  (Runs of 32 consecutive positions per XCD instead, whose tiles share
// panels in its L2, were slower: 1500^3, S = 8 199 against 186 us.)
template <class C, bool DYN>
__global__ void __launch_bounds__(C::NT) k_igemm_s1g(S1Args p, S1List list) {
    // The claim words lie behind the ring in one array: with a second LDS variable the compiler tells the
    // direct loads' LDS writes apart and waits for all of them before each read of the ring that may alias.
    __shared__ __attribute__((aligned(1024))) int8_t smem[C::LDS_BYTES + (DYN ? 16 : 0)];
    unsigned* s_pos = reinterpret_cast<unsigned*>(smem + (DYN ? C::LDS_BYTES : 0));
    const uint32_t tiles = p.order.tiles.d;
    const uint32_t xcd = blockIdx.x & 7;
    const uint32_t t0 = DYN ? tiles * xcd / 8 : 0, ntile = DYN ? tiles * (xcd + 1) / 8 - t0 : tiles;
    const FastDiv by_ntile = !DYN ? p.order.tiles : ntile == p.by_share.d ? p.by_share : p.by_share1;
    const uint32_t nwork = ntile * list.n;
    Claims c = first_claims<DYN>(p.queue, xcd, s_pos);
    if (c.w >= nwork) return;  // whole workgroup leaves together
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave_part<C>(wave).m, wn = wave_part<C>(wave).n;
    struct Item {
        int g, tm, tn, i0, nit, plane;
        StageSrc src;
    };
    auto decode = [&](uint32_t k) {
        Item t;
        uint32_t tile;
        const uint32_t e = div_fast(k, by_ntile, tile);
        t.g = (int)(list.e[e].g_plane & 0xffffu);
        t.plane = (int)(list.e[e].g_plane >> 16);
        t.i0 = (int)list.e[e].i0;
        t.nit = (int)list.e[e].nit;
        grouped_tile<C>(t0 + tile, p.order, t.tm, t.tn);
        t.tm += p.tm0;
        t.src = wave_src<C>(p.A + (int64_t)t.tm * C::BM * p.Kp, p.B + (int64_t)t.tn * C::BN * p.Kp, p.Kp, wave,
                            (int)((p.M - (int64_t)t.tm * C::BM - 1) >> 5), (int)((p.N - (int64_t)t.tn * C::BN - 1) >> 5));
        return t;
    };
    const S1Walk<C> walk(p);
    Item cur = decode(c.w);
    if constexpr (C::STAGES == 2) {
        const NextSrc first = walk.next(cur.src, p, cur.g, cur.i0, cur.nit);
        chain_start<C>(smem, 0, cur.nit, first.s0, first.s1);
    } else {
        chain_start_deep<C>(smem, cur.nit, walk.at(cur.src, p, cur.g, cur.i0), walk);
    }
    int base = 0;
    for (;;) {
        const bool more = c.w1 < nwork;
        Item nxt = cur;
        auto entry = [&] {
            if (more) nxt = decode(c.w1);
            if constexpr (C::STAGES == 2) return walk.next(nxt.src, p, nxt.g, nxt.i0, nxt.nit);
            else return walk.at(nxt.src, p, nxt.g, nxt.i0);
        };
        unsigned ticket;  // the item after next (dynamic order); thread 0's only: a value merged from both
        // paths would be copied, and so waited for behind the next item's loads, as soon as it returns
        auto claim = [&] {
            if (DYN && more && threadIdx.x == 0) ticket = atomicAdd(&p.queue[xcd], 1u);
        };
        const int64_t row0 = (int64_t)cur.tm * C::BM + wm * C::WTM, col0 = (int64_t)cur.tn * C::BN + wn * C::WTN;
        const S1Cursor stage2 = walk.at(cur.src, p, cur.g, cur.i0 + min(C::STAGES, cur.nit - 1));
        for_part<C>(
            p.M - row0, p.N - col0,
            [&]<class P>() {
                v16i acc[P::FM][P::FN];
                zero_acc<P>(acc);
                mainloop_chain<P>(acc, smem, base, cur.nit, stage2, walk, entry);
                claim();
                store_i32_blocked<P>(acc, p.T + (int64_t)cur.plane * p.Mp * p.Np, p.Np, row0, col0, lane);
            },
            [&] { mainloop_idle<C>(smem, base, cur.nit, stage2, walk, entry); });  // never thread 0's wave: part (0, 0)
        if (!more) break;
        const uint32_t w2 = DYN ? publish_claim(ticket, s_pos) : c.w + 2 * gridDim.x;
        base = (base + cur.nit) & (C::STAGES - 1);
        c.w = c.w1;
        c.w1 = w2;
        cur = nxt;
    }
    wait_vmcnt<0>();  // no direct load in flight into LDS when the workgroup leaves
}

// One resident workgroup per CU for the persistent GEMMs (the 128 KiB LDS ring allows no more).
hipError_t persistent_grid(int64_t total, unsigned& grid) {
    int dev = 0, cus = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    grid = (unsigned)std::min<int64_t>(total, std::max(cus, 1));
    return e;
}

}  // namespace

// ------------------------------------------------------------------------------------------
// Launchers
// ------------------------------------------------------------------------------------------
using CfgS2 = IgemmCfgS2;
using CfgS1 = IgemmCfgS1;

// Four slots of 64 K-bytes instead of two of 128, where s2_deep_ring says.
using CfgS2Deep = IgemmCfg<256, 256, 64, 4, 2, 4, 8>;

// Small calls (S2Plan::edge): 64 x 64 or 128 x 128 tiles, one item per workgroup, two workgroups per CU, four
// slots.  Few 256 x 256 tiles leave CUs idle, and one of them alone spends more on its epilogue (128 digits
// per thread) and on waiting for one stage at a time than on the products.  Lines and figures: scheme2_plan.
using CfgS2Small64 = IgemmCfg<64, 64, 128, 2, 2, 4, 4>;
using CfgS2Small128 = IgemmCfg<128, 128, 64, 2, 2, 4, 4>;
template <class C>
static hipError_t launch_small(const Dims& d, S2Args p, hipStream_t st) {
    p.order = tile_order((d.M + C::BM - 1) / C::BM, (d.N + C::BN - 1) / C::BN, C::GM);
    const int64_t items = (int64_t)p.order.tiles_m * p.order.tiles_n * d.S;
    if (items > INT32_MAX) return hipErrorInvalidValue;
    p.items = p.whole = (uint32_t)items;
    p.KT = p.kts = (int)(d.Kp / C::BK);
    k_igemm_s2<C, true><<<p.items, C::NT, 0, st>>>(p);
    return hipGetLastError();
}

hipError_t launch_igemm_s2(const Dims& d, const int8_t* A_sl, const int8_t* B_sl, S2Out mode, void* out,
                           const CrtSet* crt_dev, hipStream_t st, int tm0, int tms, const S2Plan* plan) {
    const bool split = plan && plan->parts > 1;
    const bool small = plan && plan->edge != CfgS2::BM;
    if ((split || small) && (mode != S2Out::Digits || tm0 != 0 || tms >= 0)) return hipErrorInvalidValue;
    S2Args p;
    p.A = A_sl;
    p.B = B_sl;
    p.M = d.M;
    p.N = d.N;
    p.Mp = d.Mp;
    p.Np = d.Np;
    p.Kp = d.Kp;
    p.S = d.S;
    p.KT = (int)(d.Kp / CfgS2::BK);
    const int tiles_m = (int)((d.M + CfgS2::BM - 1) / CfgS2::BM);
    if (tm0 < 0 || tm0 > tiles_m) return hipErrorInvalidValue;
    p.tm0 = tm0;
    const int rows = tms < 0 ? tiles_m - tm0 : std::min(tms, tiles_m - tm0);
    const int tiles_n = (int)((d.N + CfgS2::BN - 1) / CfgS2::BN);
    p.order = tile_order(rows, tiles_n, CfgS2::GM);
    p.out = out;
    p.crt = crt_dev;
    int64_t total = (int64_t)rows * tiles_n * d.S;
    const int64_t whole = split ? plan->whole : total, tail = total - whole;
    p.parts = split ? plan->parts : 1;
    p.kts = split ? plan->kts : p.KT;
    p.part = static_cast<uint8_t*>(out) + (int64_t)d.S * d.Mp * d.Np;
    if (split) total = whole + tail * p.parts;
    if (total == 0) return hipSuccess;
    if (total > INT32_MAX) return hipErrorInvalidValue;  // 2^47 bytes of digits
    p.items = (uint32_t)total;
    p.whole = (uint32_t)whole;
    p.tail = (uint32_t)tail;
    p.by_tail = fast_div(tail);
    if (small) return plan->edge == 64 ? launch_small<CfgS2Small64>(d, p, st) : launch_small<CfgS2Small128>(d, p, st);
    unsigned grid = 0;
    if (hipError_t e = persistent_grid(total, grid)) return e;
    if (mode == S2Out::Digits && s2_deep_ring(d, split ? *plan : S2Plan{})) {
        constexpr int kStages = CfgS2::BK / CfgS2Deep::BK;
        p.KT *= kStages;
        p.kts *= kStages;
        if (split) k_igemm_s2<CfgS2Deep, true, true><<<grid, CfgS2Deep::NT, 0, st>>>(p);
        else k_igemm_s2<CfgS2Deep, true><<<grid, CfgS2Deep::NT, 0, st>>>(p);
        return hipGetLastError();
    }
    if (split)
        k_igemm_s2<CfgS2, true, true><<<grid, CfgS2::NT, 0, st>>>(p);
    else if (mode == S2Out::Digits)
        k_igemm_s2<CfgS2, true><<<grid, CfgS2::NT, 0, st>>>(p);
    else
        k_igemm_s2<CfgS2, false><<<grid, CfgS2::NT, 0, st>>>(p);
    return hipGetLastError();
}

template <class C>
static S1Args make_s1(const Dims& d, const int8_t* A_sl, const int8_t* B_sl, int tm0, int rows) {
    S1Args p;
    p.A = A_sl;
    p.B = B_sl;
    p.M = d.M;
    p.N = d.N;
    p.Mp = d.Mp;
    p.Np = d.Np;
    p.Kp = d.Kp;
    p.S = d.S;
    p.KT = (int)(d.Kp / C::BK);
    p.order = tile_order(rows, (d.N + C::BN - 1) / C::BN, C::GM);
    p.tm0 = tm0;
    p.by_KT = fast_div(p.KT);
    p.by_share = fast_div(p.order.tiles.d / 8);
    p.by_share1 = fast_div(p.order.tiles.d / 8 + 1);
    p.T = nullptr;
    p.queue = nullptr;
    return p;
}

// The items of one tile, with kt stages per pair.
static bool make_s1_list(const S1Plan& plan, int S, int kt, S1List& list) {
    list.n = 0;
    for (int g = 0, extra = S; g < S; ++g) {
        const int stages = (g + 1) * kt, parts = plan.parts[g];
        for (int j = 0; j < parts; ++j) {
            if (list.n == kMaxS1Planes) return false;
            const int i0 = (int)((int64_t)stages * j / parts), i1 = (int)((int64_t)stages * (j + 1) / parts);
            list.e[list.n++] = S1Entry{(uint32_t)(g + 2) | (uint32_t)(j == 0 ? g : extra++) << 16, (uint32_t)i0, (uint32_t)(i1 - i0)};
        }
    }
    std::stable_sort(list.e, list.e + list.n, [](const S1Entry& a, const S1Entry& b) {
        return a.nit != b.nit ? a.nit > b.nit : (a.g_plane & 0xffffu) > (b.g_plane & 0xffffu);
    });
    return true;
}

// S1Plan::edge = 64 or 128: as launch_small.
template <class C>
static hipError_t launch_s1_small(const Dims& d, const int8_t* A_sl, const int8_t* B_sl, int32_t* T, hipStream_t st,
                                  const S1Plan& plan) {
    S1Args p = make_s1<C>(d, A_sl, B_sl, 0, (int)((d.M + C::BM - 1) / C::BM));
    p.T = T;
    S1List list;
    if (!make_s1_list(plan, d.S, p.KT, list)) return hipErrorInvalidValue;
    const int64_t total = (int64_t)p.order.tiles_m * p.order.tiles_n * list.n;
    if (total == 0) return hipSuccess;
    if (total > INT32_MAX) return hipErrorInvalidValue;
    k_igemm_s1g<C, false><<<(unsigned)total, C::NT, 0, st>>>(p, list);
    return hipGetLastError();
}

hipError_t launch_igemm_s1_blocked(const Dims& d, const int8_t* A_sl, const int8_t* B_sl, int32_t* T, hipStream_t st,
                                   const S1Plan& plan, unsigned* queue, int tm0, int tms) {
    const int tiles_m = (int)((d.M + CfgS2::BM - 1) / CfgS2::BM);
    if (tm0 < 0 || tm0 > tiles_m) return hipErrorInvalidValue;
    if (plan.edge != CfgS2::BM) {
        if (tm0 != 0 || tms >= 0) return hipErrorInvalidValue;
        return plan.edge == 64 ? launch_s1_small<CfgS2Small64>(d, A_sl, B_sl, T, st, plan)
                               : launch_s1_small<CfgS2Small128>(d, A_sl, B_sl, T, st, plan);
    }
    S1Args p = make_s1<CfgS2>(d, A_sl, B_sl, tm0, tms < 0 ? tiles_m - tm0 : std::min(tms, tiles_m - tm0));
    p.T = T;
    S1List list;
    if (!make_s1_list(plan, d.S, p.KT, list)) return hipErrorInvalidValue;
    const int64_t tiles = (int64_t)p.order.tiles_m * p.order.tiles_n, total = tiles * list.n;
    if (total == 0) return hipSuccess;
    if (total > INT32_MAX) return hipErrorInvalidValue;  // 2^49 bytes of products
    unsigned grid = 0;
    if (hipError_t e = persistent_grid(total, grid)) return e;
    // A workgroup of the dynamic order claims two positions before it starts, so with fewer than two
    // items per workgroup the first claimants would take them all and the others none; and with few
    // tiles the XCDs' shares of them are uneven (30 tiles: three or four each).
    p.queue = queue && grid % 8 == 0 && total >= 2 * (int64_t)grid && tiles >= 64 ? queue : nullptr;  // zeroed by the caller
    if (p.queue) k_igemm_s1g<CfgS2, true><<<grid, CfgS2::NT, 0, st>>>(p, list);
    else k_igemm_s1g<CfgS2, false><<<grid, CfgS2::NT, 0, st>>>(p, list);
    return hipGetLastError();
}

hipError_t launch_igemm_s1_groups(const Dims& d, const int8_t* A_sl, const int8_t* B_sl, int32_t* T,
                                  hipStream_t st) {
    S1Args p = make_s1<CfgS1>(d, A_sl, B_sl, 0, (int)((d.M + CfgS1::BM - 1) / CfgS1::BM));
    p.T = T;
    const int64_t grid = (int64_t)p.order.tiles_m * p.order.tiles_n;
    if (grid == 0) return hipSuccess;
    k_igemm_s1<CfgS1><<<(unsigned)grid, CfgS1::NT, 0, st>>>(p);
    return hipGetLastError();
}

}  // namespace oza
