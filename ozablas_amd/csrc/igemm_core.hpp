// igemm_core.hpp — the INT8 MFMA GEMM mainloop shared by the single-problem and grouped kernels.
//
// A workgroup owns a BM x BN output tile; each wave owns a (BM/NWM) x (BN/NWN) sub-tile made of
// 32x32 v_mfma_i32_32x32x32_i8 fragments with exact INT32 accumulation.  K advances in BK-byte
// stages through an LDS ring filled by direct global->LDS loads.
#pragma once

#include <utility>

#include "oza_device.hpp"
#include "oza_internal.hpp"
#include "k_igemm_cfg.hpp"

namespace oza {
namespace core {


// ------------------------------------------------------------------------------------------
// LDS ring filled by direct global->LDS loads (global_load_lds_dwordx4).  The operand planes are
// fragment-tiled (frag_off16): every 1 KiB block is one 32x32 MFMA operand fragment in lane order,
// so a wave-wide direct load copies one block contiguously from HBM/L2 into LDS and a wave reads a
// fragment back with one contiguous, bank-conflict-free ds_read_b128.  In LDS a stage holds A blocks
// [BM/32][kb] followed by B blocks [BN/32][kb]; wave w always loads the same few blocks of a stage,
// consecutive in memory and in LDS, so two waves never write the same LDS bytes.
// ------------------------------------------------------------------------------------------
#define OZA_LDS_PTR(p) ((__attribute__((address_space(3))) void*)(p))

// Waits until at most N vector-memory operations of this wave are outstanding (gfx9 s_waitcnt
// encoding: vmcnt bits [3:0] and [15:14]; expcnt and lgkmcnt left at their no-wait maxima).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// Waits for this wave's LDS reads and writes (lgkmcnt(0); vmcnt and expcnt left at their maxima).
__device__ __forceinline__ void wait_lgkmcnt0() { __builtin_amdgcn_s_waitcnt(0xC07F); }

__device__ __forceinline__ void block_sync_lds() {
    // s_barrier without the release/acquire fence of __syncthreads(): the fence would wait for
    // every outstanding load, including the prefetch of later stages.  The empty asm statements
    // keep the compiler from moving LDS accesses across the barrier.
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// Loads of one stage by one wave: LPA consecutive A blocks from `a` on and LPB B blocks from `b` on (the
// wave's own, see wave_src).  The pointers are wave-uniform and lane * 16 is the only lane part, and the
// instruction's offset moves both the memory and the LDS address, so a stage costs one scalar base and
// one M0 per operand.  (With a 64-bit address per load and blocks interleaved over the waves, about 45
// scalar and 10 vector instructions stood between a stage's barrier and its last k-step's MFMAs: Scheme I
// 8192^3, S = 8 16.76 against 15.96 ms, 4096^3, S = 6 1.393 against 1.347 ms; Scheme II 8192^3, S = 17
// 8.55 against 8.37 ms.)
template <class C>
__device__ __forceinline__ void issue_stage(int8_t* stage, const int8_t* __restrict__ a, const int8_t* __restrict__ b,
                                            int wave, unsigned lane) {
    const unsigned off = lane * 16;
    int8_t* sa = stage + wave * (C::LPA * 1024);
    int8_t* sb = stage + C::BM * C::BK + wave * (C::LPB * 1024);
    auto load = [&]<int... I>(const int8_t* p, int8_t* l, std::integer_sequence<int, I...>) {
        (__builtin_amdgcn_global_load_lds(p + off, OZA_LDS_PTR(l), 16, I * 1024, 0), ...);
    };
    load(a, sa, std::make_integer_sequence<int, C::LPA>{});
    load(b, sb, std::make_integer_sequence<int, C::LPB>{});
}

struct WavePart {
    int m, n;
};
// A wave's part of the tile.  At the product's edges the parts with nothing to compute leave their SIMD to
// others (for_part), so the order spreads the rest over the four SIMDs (a workgroup's wave w runs on SIMD
// w % 4): of 4 x 2 parts the first two rows, or the first column, lie on different SIMDs; of 2 x 2 parts
// the workgroups of a CU (one per 256 blocks) each take another order.
template <class C>
__device__ __forceinline__ WavePart wave_part(int wave) {
    if (C::NWM == 4 && C::NWN == 2) {
        const int n = wave >> 2;
        return {(wave & 3) ^ (n << 1), n};
    }
    if (C::NWM == 2 && C::NWN == 2) wave ^= (blockIdx.x >> 8) & 3;
    return {wave / C::NWN, wave % C::NWN};
}

// Sources of one K stage for one wave.
struct StageSrc {
    const int8_t* a;
    const int8_t* b;
};

// The wave's blocks of stage 0 of the operand tiles at a and b (fragment-tiled planes, ldk K-bytes per
// row); stage i lies i * C::STEP bytes further.  A block-row past last_a / last_b, the last that holds a row
// of the operand, is read as that one: nothing uses it, and it is at hand (the plane's memory there would
// come from HBM: groups 0.7 to 2.3 % slower).
template <class C>
__device__ __forceinline__ StageSrc wave_src(const int8_t* a, const int8_t* b, int64_t ldk, int wave,
                                             int last_a = C::BM / 32 - 1, int last_b = C::BN / 32 - 1) {
    const int64_t kblocks = ldk >> 5;  // fragment blocks per block-row of a plane
    constexpr int KB = C::KB;
    return StageSrc{a + ((min(wave * C::LPA / KB, last_a) * kblocks + wave * C::LPA % KB) << 10),
                    b + ((min(wave * C::LPB / KB, last_b) * kblocks + wave * C::LPB % KB) << 10)};
}

// What a wave loads after its current item's stages: the next item's stages 0 and 1 (any valid source
// where there is no such stage: nothing reads it, and the next chain start's vmcnt(0) completes it
// before its slot is loaded again).
struct NextSrc {
    StageSrc s0, s1;
};

template <class C>
struct Frags {
    v4i a[C::FM];
    v4i b[C::FN];
};

template <class C>
__device__ __forceinline__ void load_frags(Frags<C>& f, const int8_t* stage, int kk, int wm, int wn, int lane) {
    const int8_t* sb = stage + C::BM * C::BK;
#pragma unroll
    for (int fm = 0; fm < C::FM; ++fm)
        f.a[fm] = *reinterpret_cast<const v4i*>(stage + (((wm * (C::WTM / 32) + fm) * C::KB + kk) << 10) + lane * 16);
#pragma unroll
    for (int fn = 0; fn < C::FN; ++fn)
        f.b[fn] = *reinterpret_cast<const v4i*>(sb + (((wn * (C::WTN / 32) + fn) * C::KB + kk) << 10) + lane * 16);
}

template <class C>
__device__ __forceinline__ void mma_frags(v16i (&acc)[C::FM][C::FN], const Frags<C>& f) {
#pragma unroll
    for (int fm = 0; fm < C::FM; ++fm)
#pragma unroll
        for (int fn = 0; fn < C::FN; ++fn)
            acc[fm][fn] = __builtin_amdgcn_mfma_i32_32x32x32_i8(f.a[fm], f.b[fn], acc[fm][fn], 0, 0, 0);
}

// Scheduling hint for one k-step: interleave the next step's LDS fragment reads between the
// current step's MFMAs so that LDS latency hides behind matrix-core work.
template <class C>
__device__ __forceinline__ void interleave_hint() {
    constexpr int NMFMA = C::FM * C::FN;
    constexpr int NREAD = C::FM + C::FN;
#pragma unroll
    for (int i = 0; i < NMFMA; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                 // 1 MFMA
        if (i < NREAD) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // 1 DS read
    }
}

// Last k-step of an iteration: also spread the direct loads of a later stage between the MFMAs.
template <class C>
__device__ __forceinline__ void interleave_hint_last() {
    constexpr int NMFMA = C::FM * C::FN;
    constexpr int NREAD = C::FM + C::FN;
    constexpr int NLOAD = C::LPS;
#pragma unroll
    for (int i = 0; i < NMFMA; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                 // 1 MFMA
        if (i < NREAD) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // 1 DS read
        if (i < NLOAD) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // 1 VMEM (direct load)
    }
}

// ------------------------------------------------------------------------------------------
// Mainloop of one work item in a chain of items that share one 2-slot LDS ring.  A workgroup's
// items (tiles of one or several problems, moduli, or Scheme I groups) run back to back: item
// stage i sits in slot (base + i) & 1, and the next item's stage j is the chain's stage nit + j,
// so the next item's first two stages are issued during this item's last two iterations and land
// while its last MFMAs and its epilogue run.
//
// Ring protocol (tests/test_ring_model.py checks these rules on a transcription of the loops):
//  R1 a wave reads a stage only after every wave waited vmcnt(0) for its loads of that stage and
//     then passed a workgroup barrier;
//  R2 a wave loads into a slot only after every wave waited lgkmcnt(0) for its reads of that slot
//     and then passed a barrier;
//  R3 a wave loads into a slot only after a vmcnt(0) that follows its previous load into the same
//     slot: the ring never depends on two direct loads into one LDS address landing in issue order;
//  R4 the caller waits vmcnt(0) after its last item, so no load is in flight into LDS that a later
//     workgroup may be given.
//
// Per iteration `it` (k-steps 0..KSTEPS-1 of stage it):
//   k-steps 0..KSTEPS-2: MFMAs on the fragments in registers while the next k-step's fragments are
//     read from LDS;
//   then (it < nit-1) vmcnt(0) -- stage it+1, issued one iteration ago --, lgkmcnt(0), barrier; the
//     first fragments of stage it+1 are read and stage it+2 is issued into slot it, which every
//     wave has finished reading at that barrier, both interleaved with the last k-step's MFMAs;
//   the last iteration waits for no load: lgkmcnt(0), barrier, and chain stage nit+1 is issued into
//     its slot before the last k-step's MFMAs.
//   Wave priority: the section after each stage barrier (the direct loads and the last k-step's
//     MFMAs) runs at priority 1, everything else at 0.  Same-box A/B: Scheme II step 3 -4.5 % and
//     Scheme I -3 % against no priorities; priority 1 over all MFMA sections gave -2.4 % (Scheme
//     II), over the first k-step only +4 %.
//
//   The first wait lets LPS later operations stay outstanding: stage 1's loads, or the stores of the
//   previous item's epilogue, which would otherwise be waited for at every item (R1 needs stage 0 only;
//   with nit == 1 slot 1 is loaded at once, so there everything is waited for, R3).  Scheme II GEMM alone,
//   S = 8: 4096^2 x 256 69.8 -> 64.1 us, 4096^2 x 1024 138.7 -> 137.0 us (with the static order).
//
//   On entry this item's stage 0 has been issued, and its stage 1 too when nit >= 2 (chain_start
//   for a chain's first item; the previous item's last two iterations otherwise).  With nit == 1 no
//   earlier iteration can take chain stage 1, so it is issued after the first barrier.
//   `cur` is this item's stage 2 (if it has one) and step(cur) moves it on by a stage.  entry() runs after
//   the first barrier and returns the next item's sources.  The source is selected, so no branch
//   separates the loads from the MFMAs they are interleaved with.
//
//   With Q = STAGES > 2 slots every item has at least Q stages; Q stages are issued before an item starts,
//   stage i + Q when stage i has been read, `cur` starts at stage Q, entry() returns the next item's stage 0,
//   and the waits leave the Q - 2 (at an item's start Q - 1) later stages outstanding.
// ------------------------------------------------------------------------------------------
// More than two slots.
template <class C, class Cur, class Step>
__device__ __forceinline__ void chain_start_deep(int8_t* smem, int nit, Cur cur, Step step) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (int i = 0; i < C::STAGES; ++i) {
        issue_stage<C>(smem + i * C::STAGE_BYTES, cur.a, cur.b, wave, lane);
        if (i + 1 < nit) step(cur);
    }
}

template <class C>
__device__ __forceinline__ void chain_start(int8_t* smem, int base, int nit, const StageSrc& s0, const StageSrc& s1) {
    static_assert(C::STAGES == 2, "the chain keeps two slots");
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    issue_stage<C>(smem + (base & 1) * C::STAGE_BYTES, s0.a, s0.b, wave, lane);
    if (nit >= 2) issue_stage<C>(smem + ((base + 1) & 1) * C::STAGE_BYTES, s1.a, s1.b, wave, lane);
}

// The source of the next chain stage: this item's at cur, or the next item's at nx; moves it on.
template <class C, class Cur, class Next, class Step>
__device__ __forceinline__ void next_stage(bool own, Cur& cur, Next& nx, Step step, const int8_t*& a, const int8_t*& b) {
    if constexpr (C::STAGES == 2) {
        a = own ? cur.a : nx.s0.a;
        b = own ? cur.b : nx.s0.b;
        step(cur);
    } else {
        a = own ? cur.a : nx.a;
        b = own ? cur.b : nx.b;
        if (own) step(cur);
        else step(nx);
    }
}
template <class C, class Next>
__device__ __forceinline__ auto last_next(const Next& nx) {
    if constexpr (C::STAGES == 2) return nx.s1;
    else return nx;
}

template <class C, class Cur, class Step, class Entry>
__device__ __forceinline__ void mainloop_chain(v16i (&acc)[C::FM][C::FN], int8_t* smem, int base, int nit, Cur cur,
                                               Step step, Entry entry) {
    constexpr int KSTEPS = C::BK / 32, Q = C::STAGES;
    static_assert((Q & (Q - 1)) == 0, "slots by a mask");
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave_part<C>(wave).m, wn = wave_part<C>(wave).n;
    auto slot = [&](int i) { return smem + ((base + i) & (Q - 1)) * C::STAGE_BYTES; };
    auto lds_barrier = [] {
        wait_lgkmcnt0();  // this wave's LDS reads are done
        block_sync_lds();
    };
    Frags<C> f[2];
    // Stage 0 is the oldest of this wave's outstanding operations; the loads of Q - 1 chain stages and the
    // previous item's stores (if any) follow it.
    if (Q > 2 || nit >= 2) wait_vmcnt<(Q - 1) * C::LPS>();
    else wait_vmcnt<0>();
    lds_barrier();
    load_frags<C>(f[0], slot(0), 0, wm, wn, lane);
    auto nx = entry();
    if constexpr (Q == 2)
        if (nit == 1) issue_stage<C>(slot(1), nx.s0.a, nx.s0.b, wave, lane);
    for (int it = 0; it + 1 < nit; ++it) {
        const int8_t* now = slot(it);
        const bool own = it + Q < nit;  // chain stage it + Q: this item's, or the next item's
        const int8_t *pa, *pb;
        next_stage<C>(own, cur, nx, step, pa, pb);
#pragma unroll
        for (int kk = 0; kk + 1 < KSTEPS; ++kk) {
            load_frags<C>(f[(kk + 1) & 1], now, kk + 1, wm, wn, lane);
            mma_frags<C>(acc, f[kk & 1]);
            interleave_hint<C>();
        }
        wait_vmcnt<(Q - 2) * C::LPS>();  // stage it+1, issued Q - 1 iterations ago
        lds_barrier();
        load_frags<C>(f[KSTEPS & 1], slot(it + 1), 0, wm, wn, lane);
        __builtin_amdgcn_s_setprio(1);
        issue_stage<C>(slot(it + Q), pa, pb, wave, lane);
        mma_frags<C>(acc, f[(KSTEPS - 1) & 1]);
        interleave_hint_last<C>();
        __builtin_amdgcn_s_setprio(0);
        if (KSTEPS % 2 == 1) {  // keep the fragments of the next iteration in f[0]
#pragma unroll
            for (int i = 0; i < C::FM; ++i) f[0].a[i] = f[1].a[i];
#pragma unroll
            for (int i = 0; i < C::FN; ++i) f[0].b[i] = f[1].b[i];
        }
    }
    {  // last iteration: its slot is freed at the barrier for chain stage nit + Q - 1
        const int8_t* now = slot(nit - 1);
#pragma unroll
        for (int kk = 0; kk + 1 < KSTEPS; ++kk) {
            load_frags<C>(f[(kk + 1) & 1], now, kk + 1, wm, wn, lane);
            mma_frags<C>(acc, f[kk & 1]);
            interleave_hint<C>();
        }
        lds_barrier();
        __builtin_amdgcn_s_setprio(1);
        issue_stage<C>(slot(nit + Q - 1), last_next<C>(nx).a, last_next<C>(nx).b, wave, lane);
        mma_frags<C>(acc, f[(KSTEPS - 1) & 1]);
        __builtin_amdgcn_s_setprio(0);
    }
}

// mainloop_chain for a wave whose part of the tile holds no element of the product: its loads, waits and
// barriers, without fragments.
template <class C, class Cur, class Step, class Entry>
__device__ __forceinline__ void mainloop_idle(int8_t* smem, int base, int nit, Cur cur, Step step, Entry entry) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    constexpr int Q = C::STAGES;
    auto slot = [&](int i) { return smem + ((base + i) & (Q - 1)) * C::STAGE_BYTES; };
    if (Q > 2 || nit >= 2) wait_vmcnt<(Q - 1) * C::LPS>();
    else wait_vmcnt<0>();
    block_sync_lds();
    auto nx = entry();
    if constexpr (Q == 2)
        if (nit == 1) issue_stage<C>(slot(1), nx.s0.a, nx.s0.b, wave, lane);
    for (int it = 0; it + 1 < nit; ++it) {
        const int8_t *pa, *pb;
        next_stage<C>(it + Q < nit, cur, nx, step, pa, pb);
        wait_vmcnt<(Q - 2) * C::LPS>();
        block_sync_lds();
        issue_stage<C>(slot(it + Q), pa, pb, wave, lane);
    }
    block_sync_lds();
    issue_stage<C>(slot(nit + Q - 1), last_next<C>(nx).a, last_next<C>(nx).b, wave, lane);
}

// Edge tiles.  A wave that computes only the first FM_ x FN_ fragments of its part: the padding's products
// cost time and, in a kernel that is bound by power, the other waves' clock.  Groups of 64, M, N, K log-uniform
// on [64, 700]: 194 -> 187 us per call, 512 on [64, 2048] 4.95 -> 4.84 ms (4.87 with whole parts only); single
// calls 300 x 5000 x 3000, S = 12 187 -> 178 us, 100 x 100 x 20000, S = 10 85 -> 74 us; 8192^3 unchanged.
template <class C, int FM_, int FN_>
struct PartCfg : C {
    static constexpr int FM = FM_, FN = FN_;
};

// Runs full.operator()<P>() with the least of C, its half in either direction and its quarter that covers
// the `rows` x `cols` elements from the wave's first on that belong to the product, or idle() where
// none does.
template <class C, class Full, class Idle>
__device__ __forceinline__ void for_part(int64_t rows, int64_t cols, Full full, Idle idle) {
    constexpr int HM = (C::FM + 1) / 2, HN = (C::FN + 1) / 2;
    if (rows <= 0 || cols <= 0) {
        idle();
    } else if (C::FM > HM && rows <= HM * 32) {
        if (C::FN > HN && cols <= HN * 32) full.template operator()<PartCfg<C, HM, HN>>();
        else full.template operator()<PartCfg<C, HM, C::FN>>();
    } else if (C::FN > HN && cols <= HN * 32) {
        full.template operator()<PartCfg<C, C::FM, HN>>();
    } else {
        full.template operator()<C>();
    }
}

template <class C>
__device__ __forceinline__ void zero_acc(v16i (&acc)[C::FM][C::FN]) {
#pragma unroll
    for (int fm = 0; fm < C::FM; ++fm)
#pragma unroll
        for (int fn = 0; fn < C::FN; ++fn)
#pragma unroll
            for (int j = 0; j < 16; ++j) acc[fm][fn][j] = 0;
}

// Every accumulator element starts from the uniform value v (kProductBias; the MFMA adds
// modulo 2^32).  One move per element in asm: from plain assignments the compiler keeps one copy of
// the 16 values alive through the mainloop to start the first fragments from (+60 registers, spills).
// The mainloop's barrier lies between these moves and the first MFMA that reads them.
template <class C>
__device__ __forceinline__ void fill_acc(v16i (&acc)[C::FM][C::FN], int v) {
#pragma unroll
    for (int fm = 0; fm < C::FM; ++fm)
#pragma unroll
        for (int fn = 0; fn < C::FN; ++fn)
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                int x;
                asm volatile("v_mov_b32 %0, %1" : "=v"(x) : "s"(v));
                acc[fm][fn][j] = x;
            }
}

// Row of accumulator element j of lane l inside a 32x32 fragment.
__device__ __forceinline__ int frag_row(int j, int lane) { return 8 * (j >> 2) + 4 * (lane >> 5) + (j & 3); }

// Work index -> (s, tm, tn).  Consecutive workgroups are dealt round-robin to the 8 XCDs; the
// remap gives each XCD a contiguous run of work items so that neighbouring tiles (which share
// A rows and B columns) meet in the same L2.
__device__ __forceinline__ uint32_t xcd_remap(uint32_t id, uint32_t total) {
    const uint32_t per = total / 8;
    return id >= per * 8 ? id : (id % 8) * per + id / 8;
}

// n / f.d and n % f.d.
__device__ __forceinline__ uint32_t div_fast(uint32_t n, const FastDiv& f, uint32_t& rem) {
    uint32_t q = __umulhi(n, f.inv);
    rem = n - q * f.d;
    if (rem >= f.d) {
        ++q;
        rem -= f.d;
    }
    return q;
}

// Tile index t in [0, tiles_m*tiles_n) -> (tm, tn), GM tile-rows at a time.
template <class C>
__device__ __forceinline__ void grouped_tile(uint32_t t, const TileOrder& o, int& tm, int& tn) {
    static_assert((C::GM & (C::GM - 1)) == 0, "full groups divide by a shift");
    uint32_t r, row;
    const int first = (int)div_fast(t, o.group, r) * C::GM;
    if (o.tiles_m - first >= C::GM) {
        row = r % C::GM;
        tn = (int)(r / C::GM);
    } else {
        tn = (int)div_fast(r, o.last, row);
    }
    tm = first + (int)row;
}

// CRT-digit epilogue of one tile: the digit of C_s per accumulator element (product_digit; the accumulators
// started from kProductBias), one 16-byte store per fragment and lane.  Digit planes are blocked in
// 32 x 32 element blocks: block (R, Q) of a plane with Np columns starts at byte (R * (Np/32) + Q) * 1024, and inside it lane
// l's 16 bytes j = 0..15 sit at l*16 + j, holding element (row 8*(j/4) + 4*(l/32) + j%4,
// column l%32) of the block, i.e. the MFMA 32x32 output layout.  The layout does not depend on
// the tile shape, so every GEMM configuration feeds the same reconstruction.  With SKIP_PAD,
// blocks that hold no element of the M x N product (tile padding) are neither computed nor stored
// (the reconstruction never reads them); the grouped GEMM, whose small problems pad much, uses it,
// while the single-problem GEMM keeps the branch-free epilogue (0.3 % faster at 8192^3).  NT
// makes the stores nontemporal (store_unit16).  Four digits are packed by byte selects (three instructions;
// shifts and ors took seven, since the compiler does not know that a digit is below 256: 2048^3, S = 6 96.8 and
// 95.5 us, 512 grouped products 4881 and 4828 us).
template <class C, bool SKIP_PAD, bool NT = false>
__device__ __forceinline__ void store_digits(const v16i (&acc)[C::FM][C::FN], uint8_t* plane, int64_t Np,
                                             int64_t row0, int64_t col0, int64_t M, int64_t N, uint32_t wt,
                                             uint32_t m_init, uint32_t minv, int lane) {
    const int64_t qn = Np >> 5;
    // An instruction takes one scalar register.  From a plain use of a second one the compiler moved the whole
    // item descriptor to vector registers (185 -> 205 of them).
    uint32_t vinit;
    asm("v_mov_b32 %0, %1" : "=v"(vinit) : "s"(m_init >> 8));
    const uint32_t m = m_init & 0xffu;
    // row0 and col0 are the same for the whole wave
    const int64_t fm_end = (M - (int64_t)__builtin_amdgcn_readfirstlane((int)(row0 >> 5)) * 32 + 31) >> 5;
    const int64_t fn_end = (N - (int64_t)__builtin_amdgcn_readfirstlane((int)(col0 >> 5)) * 32 + 31) >> 5;
#pragma unroll
    for (int fm = 0; fm < C::FM; ++fm)
#pragma unroll
        for (int fn = 0; fn < C::FN; ++fn) {
            if (SKIP_PAD && (fm >= fm_end || fn >= fn_end)) continue;
            int d[16];
#pragma unroll
            for (int j = 0; j < 16; ++j) d[j] = (int)product_digit((uint32_t)acc[fm][fn][j], wt, vinit, m, minv);
            const int64_t blk = ((row0 >> 5) + fm) * qn + (col0 >> 5) + fn;
            store_global16<NT>(plane + (blk << 10) + lane * 16, pack4_lo(d[0], d[1], d[2], d[3]),
                               pack4_lo(d[4], d[5], d[6], d[7]), pack4_lo(d[8], d[9], d[10], d[11]),
                               pack4_lo(d[12], d[13], d[14], d[15]));
        }
}

// Split-K digit reduction of 16 digits: dg[off..off+15] = (dg + sum_{j < parts} part_j) mod m, with
// part_j at dgp + j * stride + off.  Every digit is below m, so one conditional subtraction per
// part keeps the running sum reduced.  off is a multiple of 16.
__device__ __forceinline__ void reduce_digits16(uint8_t* __restrict__ dg, const uint8_t* __restrict__ dgp,
                                                int64_t stride, int parts, uint32_t m, int64_t off) {
    uint4* dst = reinterpret_cast<uint4*>(dg + off);
    const uint4 d0 = *dst;
    uint32_t w[4] = {d0.x, d0.y, d0.z, d0.w};
    uint32_t r[16];
#pragma unroll
    for (int b = 0; b < 16; ++b) r[b] = (w[b >> 2] >> (8 * (b & 3))) & 0xffu;
    for (int j = 0; j < parts; ++j) {
        const uint4 v = *reinterpret_cast<const uint4*>(dgp + (int64_t)j * stride + off);
        const uint32_t u[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int b = 0; b < 16; ++b) {
            const uint32_t x = r[b] + ((u[b >> 2] >> (8 * (b & 3))) & 0xffu);
            r[b] = x >= m ? x - m : x;
        }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) w[q] = r[4 * q] | (r[4 * q + 1] << 8) | (r[4 * q + 2] << 16) | (r[4 * q + 3] << 24);
    *dst = make_uint4(w[0], w[1], w[2], w[3]);
}

// INT32 epilogue of one tile into a blocked plane: 32 x 32 element blocks of 4 KiB, block (R, Q)
// at element (R * (Np/32) + Q) * 1024, lane l's 16 values j at l*16 + j (the layout of
// store_digits with 4-byte elements).
template <class C>
__device__ __forceinline__ void store_i32_blocked(const v16i (&acc)[C::FM][C::FN], int32_t* plane, int64_t Np,
                                                  int64_t row0, int64_t col0, int lane) {
    const int64_t qn = Np >> 5;
#pragma unroll
    for (int fm = 0; fm < C::FM; ++fm)
#pragma unroll
        for (int fn = 0; fn < C::FN; ++fn) {
            const int64_t blk = ((row0 >> 5) + fm) * qn + (col0 >> 5) + fn;
            int4* o = reinterpret_cast<int4*>(plane + (blk << 10) + lane * 16);
            const v16i& a = acc[fm][fn];
            o[0] = make_int4(a[0], a[1], a[2], a[3]);
            o[1] = make_int4(a[4], a[5], a[6], a[7]);
            o[2] = make_int4(a[8], a[9], a[10], a[11]);
            o[3] = make_int4(a[12], a[13], a[14], a[15]);
        }
}

}  // namespace core
}  // namespace oza
