// Ping-pong form of the LDS-tiled GEMM for gfx950 (fp32 accumulation): the two
// wavefronts that share a SIMD take turns.  While one of them issues nothing
// but the 32 MFMAs of a k-step (a "compute cluster", 512 cycles of matrix-core
// time), the other one runs its "memory cluster": it reads its fragments of the
// next k-step from LDS into registers and issues its share of the direct-to-LDS
// loads that refill the ring.  A workgroup barrier ends every cluster and the
// two swap roles.  The matrix cores never wait for an LDS read or for the issue
// of a load (a wavefront alone on its SIMD loses 15-20 cycles of MFMA issue per
// 1 KiB load it issues), and the two wavefronts never compete for them.
//
// Wavefronts 0-3 of the workgroup sit on SIMDs 0-3 and wavefronts 4-7 join
// them in the same order; the second group enters the loop one barrier late, so
// that it runs one cluster behind the first for the whole K loop.
//
// Same canonical problem, tile mapping and LDS chunk layouts as gemm_tiled.hpp
// (P = X * Y, I contiguous in P).  What differs is how the ring is cut:
//   I-major operand: four entries of 32 k-values (one k-step).  The loads of
//       step t+3 are issued in the memory cluster of step t.
//   K-major operand: three slots of 64 k-values (rows of 128 bytes, so that
//       every direct-to-LDS load still fetches full 128-byte lines).  The loads
//       of pair p+2 are issued in the two memory clusters of pair p, half each.
// Either way a wavefront waits, at the end of memory cluster t, for the loads
// it issued in cluster t-2 and earlier (s_waitcnt vmcnt(2 * loads per cluster)):
// a load has two full clusters of both groups (about 2000 cycles) to land
// before anyone waits for it, and the barriers between that wait and the first
// read publish it to the other wavefronts.
//   Two K-major operands: three slots each would be 192 KiB.  X keeps three, Y
//       gets two (160 KiB).  A slot of Y is free once both groups have read its
//       second k-step, which is when group 0 starts the memory cluster after
//       that; so the first cluster of pair p+1 requests all of Y's pair p+2
//       into the slot of pair p, and the wait at the end of the second cluster
//       of pair p+1 must cover it: that cluster leaves only its own loads in
//       flight, and those are X's (all of X's pair p+3, into the slot of pair
//       p).  Y's loads have one compute and one memory cluster to land, X's two
//       of each as before.
#pragma once
#include "gemm_tiled.hpp"

namespace miw {

// (The measurement switch MIW_PP_ABLATE of gemm_tiled.hpp applies to the loops of these kernels too.)


// Second measurement switch (off in every shipped build; gemm_kernels.hip must be compiled with it
// too): with MIW_PP_TS the ping-pong kernels record, per wavefront, the shader clock at kernel
// entry [0], after the prologue's loads have landed [1], at the middle of the loop [2], one pair
// of k-steps later [3], at the end of the pairs that do not fold C [9], at the end of the loop [4],
// when the last store is issued [5] and when the stores have drained [6], plus the 100 MHz wall
// clock at exit [7] and entry [8], into the buffer whose device address the environment variable
// MIW_TS holds (cudanative.jl_amd/timestamps.py sets it and prints the phases).
#ifdef MIW_PP_TS
#define MIW_PP_STAMP(i) { __builtin_amdgcn_sched_barrier(0); ts[i] = clock64(); __builtin_amdgcn_sched_barrier(0); }
// (in the unrolled part of the loop: the ring of pairs that holds pair NPM / 2 stamps its first pair)
#define MIW_PP_MIDDLE(pr) { stamp_pair = (pr) <= NPM / 2 && NPM / 2 < (pr) + NSLOT; if (stamp_pair) MIW_PP_STAMP(2) }
#else
#define MIW_PP_STAMP(i)
#define MIW_PP_MIDDLE(pr)
#endif

constexpr int PP_KMAJOR_SLOTS = 3;
constexpr int PP_IMAJOR_ENTRIES = 4;
constexpr int PP_SPREAD_SLEEP = 64;  // units of 64 cycles between the starts of workgroups, see tiled_params::c_spread
constexpr int PP_FOLD_STEPS = 32;  // k-steps of 32 over which k_gemm_pp_fold adds C: one MFMA tile of the wavefront's 8 x 4 each

// Slots of a K-major Y: two when X is K-major as well (see above), else three.
constexpr int pp_y_slots(bool xk) { return xk ? 2 : PP_KMAJOR_SLOTS; }
constexpr int pp_operand_bytes(int rows, bool kmajor, int kslots)
{
    return kmajor ? kslots * rows * KGRAN * 2 : PP_IMAJOR_ENTRIES * rows * BKS * 2;
}
constexpr int pp_lds_bytes(int bi, int bj, bool xk, bool yk)
{
    return pp_operand_bytes(bi, xk, PP_KMAJOR_SLOTS) + pp_operand_bytes(bj, yk, pp_y_slots(xk));
}
constexpr bool pp_fits(int bi, int bj, bool xk, bool yk) { return pp_lds_bytes(bi, bj, xk, yk) <= 160 * 1024; }

// One operand of the ping-pong kernel: its ring in LDS, the loads that fill it
// and the fragment reads.  R rows (or columns) of the tile, NT threads.
template <int R, bool KMAJOR, int NT, int KSLOTS = PP_KMAJOR_SLOTS>
struct pp_operand {
    // loads per thread: per 64-k slot (K-major) or per 32-k entry (I-major)
    static constexpr int NL = KMAJOR ? R * KGRAN / 8 / NT : R * BKS / 8 / NT;
    // loads per thread and memory cluster (a K-major operand: half a slot, unless both operands are K-major)
    static constexpr int PER_CLUSTER = KMAJOR ? NL / 2 : NL;
    static constexpr int UNIT_BYTES = KMAJOR ? R * KGRAN * 2 : R * BKS * 2;
    static constexpr int UNITS = KMAJOR ? KSLOTS : PP_IMAJOR_ENTRIES;
    static constexpr int BYTES = UNITS * UNIT_BYTES;
    static_assert(NL >= 1 && (!KMAJOR || NL % 2 == 0), "operand must divide over the workgroup");
    static_assert(NT == 512 || NT == 256, "lane offsets below assume 256 or 512 threads");

    __device__ static inline unsigned lane_offset(int tid, int ld)
    {
        if constexpr (KMAJOR) {
            return slot_loader<R, true, NT>::lane_offset(tid, ld);
        } else {
            // chunk tid of the entry: i-block tid / 256, k-row (tid / 8) % 32, chunk position tid % 8
            const int k = (tid >> 3) & 31, cpos = tid & 7, iblk = tid >> 8;
            const int c = cpos ^ (2 * i_major_swizzle(k));
            return 2u * (unsigned)(k * ld + iblk * 64 + c * 8);
        }
    }
    // Element offset of load i of a unit relative to load 0 (uniform).
    __device__ static inline long load_delta(int i, long ld)
    {
        if constexpr (KMAJOR) return (long)i * (NT / 8) * ld;
        else return (long)i * (NT / 256) * 64;
    }

    // Fragment reads.  K-major: the reader of gemm_tiled.hpp on a 64-k slot.
    // I-major: the same transpose reads on an entry of 32 k-rows (i-blocks of
    // 64 i are 4 KiB apart instead of 8).
    frag_reader<R, true> kr;
    int ibase[4];
    __device__ inline void init(int wave_row0, int lane)
    {
        if constexpr (KMAJOR) {
            kr.init(wave_row0, lane);
        } else {
            const int j = lane & 15, q = lane >> 4;
            const int jq = j >> 2, jr = j & 3;
            const int g = ((jq >> 1) & 1) | ((q & 1) << 1);
            const int w16 = wave_row0 / 16;
#pragma unroll
            for (int m = 0; m < 4; m++)
                ibase[m] = (w16 / 4) * 4096 + (8 * q + jq) * 128 + jr * 8 + ((((w16 & 3) + m) & 3) ^ g) * 32;
        }
    }
    // Fragment T of k-step H (0/1: which half of the slot; ignored for I-major) out of the unit at `unit`.
    template <int T, int H>
    __device__ inline half8_t read(MIW_LDS const char *unit) const
    {
        if constexpr (KMAJOR) {
            return kr.template read<T, H>(unit);
        } else {
            const int off = ibase[T & 3] + (T >> 2) * 4096;
            fp16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4f16((MIW_LDS fp16x4_t *)(unit + off));
            fp16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4f16((MIW_LDS fp16x4_t *)(unit + off + 512));
            uint2_t l2 = __builtin_bit_cast(uint2_t, lo), h2 = __builtin_bit_cast(uint2_t, hi);
            uint4_t v = {l2[0], l2[1], h2[0], h2[1]};
            return __builtin_bit_cast(half8_t, v);
        }
    }
};

// Where the tiles outnumber the CUs a workgroup walks several (tiled_params::work), and the ring runs on from one
// tile into the next: behind the last unit of a tile the first ones of the next are requested, so that they land
// under the epilogue.  One workgroup per tile pays for a start of 2 to 3 us and for the dispatch, which hands
// workgroups to the shader engines in turn and waits for the slowest, 1 to 5 us, in every round; what is left is the
// store of D, whose acknowledgements the loads of the next tile's third k-step wait for (vmcnt counts in order).
// 8192x8192x1024, alpha = -1, operands from HBM: 188 us with one tile per workgroup, 180 like this; without C 143
// and 127; 6144^3 425 and 414; 8192^3 level (784, 779), which is bound by energy.
// FOLD: a Float32 C is added in the K loop; otherwise C, if any, in the epilogue.  They are kernels of their own: in
// one kernel the accumulators of both forms meet in the last pair, and that spills.
template <int BI, int BJ, int WI, int WJ, bool XK, bool YK, class CT, class DT, bool FOLD>
__device__ __attribute__((always_inline)) inline void gemm_pp(const tiled_params &p)
{
    constexpr int NT = WI * WJ * 64;
    static_assert(NT == 512, "two wavefronts per SIMD");
    constexpr int WTI = BI / WI, WTJ = BJ / WJ;
    constexpr int TI = WTI / 16, TJ = WTJ / 16;
    constexpr bool KK = XK && YK;  // two K-major operands: Y has two slots, clusters alternate between Y's loads and X's
    using xop = pp_operand<BI, XK, NT>;
    using yop = pp_operand<BJ, YK, NT, pp_y_slots(XK)>;
    constexpr int XB = xop::BYTES;
    constexpr int ND = xop::PER_CLUSTER + yop::PER_CLUSTER;  // loads per thread and memory cluster
    static_assert(!KK || (xop::NL == ND && yop::NL == ND), "alternating clusters carry equal loads");
    static_assert(pp_fits(BI, BJ, XK, YK), "ring does not fit in LDS");

#ifdef MIW_PP_TS
    long long ts[10] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    ts[0] = clock64();
    ts[8] = wall_clock64();
#endif
    extern __shared__ __attribute__((aligned(128))) char smem[];
    MIW_LDS char *lds = (MIW_LDS char *)smem;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wi = wave % WI, wj = wave / WI;
    const bool late_group = wave >= 4;

    // What only the start of a tile needs is read from the arguments again there: held through the K loop it
    // would take more scalar registers than there are.
    auto arguments = [] MIW_INLINE {
        auto a = (const __attribute__((address_space(4))) tiled_params *)__builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+s"(a));
        return a;
    };
    auto x_origin = [](auto a, int bt, int i0) MIW_INLINE { return a->X + (long)bt * a->sx + (XK ? (long)i0 * a->ldx : (long)i0); };
    auto y_origin = [](auto a, int bt, int j0) MIW_INLINE { return a->Y + (long)bt * a->sy + (YK ? (long)j0 * a->ldy : (long)j0); };
    fetch_arguments(p);  // (what is read again later is then in the scalar cache)
    int tile = blockIdx.x + blockIdx.y * (unsigned)p.span;
    tile_place at = tile_at(p, tile, blockIdx.y, BI, BJ);  // (the first tile's: already in registers)
    const half_t *X = x_origin(&p, at.bt, at.i0);
    const half_t *Y = y_origin(&p, at.bt, at.j0);
    const unsigned xoff = xop::lane_offset(tid, (int)p.ldx);
    const unsigned yoff = yop::lane_offset(tid, (int)p.ldy);

    xop xr;
    yop yr;
    // (the wavefront's place in the tile is added to the unit's address, a scalar: two operands of one kind
    // then share their lane offsets)
    static_assert(WTI % 64 == 0 && WTJ % 64 == 0, "wave tile");
    xr.init(0, lane);
    yr.init(0, lane);
    const unsigned xwave = wi * WTI * (XK ? 128 : 64), ywave = wj * WTJ * (YK ? 128 : 64);

    const int q = lane >> 4, r = lane & 15;
    float4_t acc[TI][TJ];

    const int NP = (p.K + KGRAN - 1) / KGRAN;  // pairs of k-steps
    const int NS = 2 * NP;                     // k-steps
    // K tail: the last pair starts at K - 64; tail_skip of its k-values repeat the pair before
    const int tail_skip = NP * KGRAN - p.K;
    const unsigned lds0 = (unsigned)(uintptr_t)lds;
    const unsigned wave_dst = lds0 + (unsigned)wave * 1024u;

    // ---- ring state (uniform).  I-major operand: the pair's two entries sit at `pair` and
    // pair + UNIT_BYTES, pair toggling between 0 and 2 UNIT_BYTES.  K-major operand: `pair` is the
    // slot of the current pair and `prev` the slot of the pair before it, which is the one being
    // refilled (with pair pr + 2).
    unsigned xpair = 0, xprev = 2 * xop::UNIT_BYTES, ypair = 0, yprev = (yop::UNITS - 1) * yop::UNIT_BYTES;
    // Lane offsets of the loads of one unit: K-major loads differ by whole rows (a per-load lane
    // offset keeps one uniform base address), I-major loads by 256 bytes (the instruction's offset field).
    unsigned xvo[XK ? xop::NL : 1], yvo[YK ? yop::NL : 1];
#pragma unroll
    for (int i = 0; i < (XK ? xop::NL : 1); i++) xvo[i] = xoff + 2u * (unsigned)xop::load_delta(i, p.ldx);
#pragma unroll
    for (int i = 0; i < (YK ? yop::NL : 1); i++) yvo[i] = yoff + 2u * (unsigned)yop::load_delta(i, p.ldy);
    // Load I of the unit at ring offset `unit` (bytes from the operand's region).
    auto x_load = [&]<int I>(unsigned unit, std::integral_constant<int, I>) MIW_INLINE {
        if constexpr (XK) lds_dma16_at<I * NT * 16, 0>(X, xvo[I], wave_dst + unit);
        else lds_dma16_at<I * NT * 16, I * 256>(X, xvo[0], wave_dst + unit);
    };
    auto y_load = [&]<int I>(unsigned unit, std::integral_constant<int, I>) MIW_INLINE {
        if constexpr (YK) lds_dma16_at<XB + I * NT * 16, 0>(Y, yvo[I], wave_dst + unit);
        else lds_dma16_at<XB + I * NT * 16, I * 256>(Y, yvo[0], wave_dst + unit);
    };
    // Elements from one unit to the next; the first unit of the last pair (pair NP - 1, or entry NS - 2)
    // lies tail_skip k-values short of where it would follow on (a step back for an entry of 32 when 48
    // repeat).  The steps are kept as 64-bit values: computed per request, the multiplication by the
    // leading dimension is a chain of scalar instructions at the end of every memory cluster, which is
    // the longer of the two clusters.
    constexpr int XUK = XK ? KGRAN : BKS, YUK = YK ? KGRAN : BKS;
    long xunit = XK ? (long)XUK : (long)XUK * p.ldx, xtail = XK ? (long)(XUK - tail_skip) : (long)(XUK - tail_skip) * p.ldx;
    long yunit = YK ? (long)YUK : (long)YUK * p.ldy, ytail = YK ? (long)(YUK - tail_skip) : (long)(YUK - tail_skip) * p.ldy;
    // The requests run on past the end of K: unit XN of a tile is unit 0 of the workgroup's next tile,
    // xjump elements from the last unit.  A workgroup without a next tile requests its last unit again (no
    // step), into a unit nobody reads any more.
    const int XN = XK ? NP : NS, YN = YK ? NP : NS;
    int xnext = 0, ynext = 0;                                // unit to request next (step index for I-major, pair index for K-major)
    long xjump = 0, yjump = 0;
    bool has_next = false;
    auto one_of = [](int next, int last, int end, long unit, long tail, long jump) MIW_INLINE {
        return next == last ? tail : next == end ? jump : unit;
    };
    // ANY: the step may lead to the last pair or beyond; otherwise it is the plain one and xnext is not kept.
    auto x_advance = [&]<bool ANY>(std::bool_constant<ANY>) MIW_INLINE {
        if constexpr (ANY) {
            xnext++;
            X += one_of(xnext, XK ? NP - 1 : NS - 2, XN, xunit, xtail, xjump);
            if (xnext >= XN && !has_next) xunit = 0;
        } else {
            X += xunit;
        }
    };
    auto y_advance = [&]<bool ANY>(std::bool_constant<ANY>) MIW_INLINE {
        if constexpr (ANY) {
            ynext++;
            Y += one_of(ynext, YK ? NP - 1 : NS - 2, YN, yunit, ytail, yjump);
            if (ynext >= YN && !has_next) yunit = 0;
        } else {
            Y += yunit;
        }
    };
    // Units requested when a tile's pair pr begins (both kinds of operand are ahead by that much).
    auto next_units = [&](int pr) MIW_INLINE {
        xnext = XK ? 2 + pr : 3 + 2 * pr;
        ynext = KK ? 1 + pr : YK ? 2 + pr : 3 + 2 * pr;
    };
    // Request number N (0 .. ND-1) of the memory cluster of k-step 2 pr + H: the X loads, then the Y loads.
    auto cluster_request = [&]<int H, int N>(std::integral_constant<int, H>, std::integral_constant<int, N>) MIW_INLINE {
        if constexpr (KK) {
            // first cluster of a pair: all of Y's pair after next, into the slot of the pair before
            // (read to the end one barrier ago); second cluster: all of X's, likewise
            if constexpr (H == 0) y_load(yprev, std::integral_constant<int, N>{});
            else x_load(xprev, std::integral_constant<int, N>{});
        } else if constexpr (N < xop::PER_CLUSTER) {
            if constexpr (XK) x_load(xprev, std::integral_constant<int, H * xop::NL / 2 + N>{});
            else x_load(H == 0 ? (xpair ^ (2u * xop::UNIT_BYTES)) + xop::UNIT_BYTES : xpair, std::integral_constant<int, N>{});
        } else {
            constexpr int M = N - xop::PER_CLUSTER;
            if constexpr (YK) y_load(yprev, std::integral_constant<int, H * yop::NL / 2 + M>{});
            else y_load(H == 0 ? (ypair ^ (2u * yop::UNIT_BYTES)) + yop::UNIT_BYTES : ypair, std::integral_constant<int, M>{});
        }
    };
    auto cluster_advance = [&]<int H, bool ANY>(std::integral_constant<int, H>, std::bool_constant<ANY> any) MIW_INLINE {
        if constexpr (!XK || H == 1) x_advance(any);
        if constexpr (!YK || H == (KK ? 0 : 1)) y_advance(any);
    };
    auto pair_advance = [&]() MIW_INLINE {
        if constexpr (XK) {
            xprev = xpair;
            xpair = xpair + xop::UNIT_BYTES == xop::BYTES ? 0 : xpair + xop::UNIT_BYTES;
        } else {
            xpair ^= 2u * xop::UNIT_BYTES;
        }
        if constexpr (YK) {
            yprev = ypair;
            ypair = ypair + yop::UNIT_BYTES == yop::BYTES ? 0 : ypair + yop::UNIT_BYTES;
        } else {
            ypair ^= 2u * yop::UNIT_BYTES;
        }
    };

    // Prologue: K-major operands request pairs 0 and 1, I-major operands steps 0, 1 and 2, in the order
    // in which the loop needs them: what step 0 reads (unit 0 of each operand), then step 1 (entry 1 of
    // an I-major operand), then step 2 (entry 2, pair 1).  The loop starts as soon as the units of step
    // 0 have landed; the rest arrives under the first clusters.  The loop's own wait covers it: at the
    // end of memory cluster t it leaves 2 ND loads in flight, and the units of step 2 are at least ND
    // loads, so after cluster 0 the units of step 1 have landed and after cluster 1 those of step 2.
    auto prologue_unit = [&]<int U>(std::integral_constant<int, U>, bool is_x) MIW_INLINE {
        if (is_x) {
            [&]<int... I>(std::integer_sequence<int, I...>) {
                (x_load((unsigned)(U * xop::UNIT_BYTES), std::integral_constant<int, I>{}), ...);
            }(std::make_integer_sequence<int, xop::NL>{});
            x_advance(std::true_type{});
        } else {
            [&]<int... I>(std::integer_sequence<int, I...>) {
                (y_load((unsigned)(U * yop::UNIT_BYTES), std::integral_constant<int, I>{}), ...);
            }(std::make_integer_sequence<int, yop::NL>{});
            y_advance(std::true_type{});
        }
    };
    // Workgroups that all end their loops at once leave HBM idle during the loops and share it in the epilogues.  Where C and D
    // take longer than the loop (tiled_params::c_spread) they start at four different times over 25000 cycles, eight tiles of one
    // column together (see spread_phase), so that some loop while others read C and store D; every start waits a fixed time and
    // nobody waits for another workgroup.  alpha = -1, all at once, by rows of tiles and by columns: 8192x8192x1024 180.2 us,
    // 168.8 and 165.8; 8192x8192x208 115.4, 113.1 and 104.1; two tiles each: 8192x4096x512 75.9, 86.0 and 69.6, 4096x8192x512
    // 73.9, 71.5 and 67.1; 8000x4400x208 81.7, 84.3 and 71.6.
    if constexpr (!FOLD && __is_same(CT, float) && __is_same(DT, float)) {
        if (p.c_spread)
            for (int phase = spread_phase() & 6; phase > 0; phase--) __builtin_amdgcn_s_sleep(PP_SPREAD_SLEEP);
    }
    constexpr std::integral_constant<int, 0> unit0{};
    constexpr std::integral_constant<int, 1> unit1{};
    constexpr std::integral_constant<int, 2> unit2{};
    prologue_unit(unit0, true);
    prologue_unit(unit0, false);
    if constexpr (!XK) prologue_unit(unit1, true);
    if constexpr (!YK) prologue_unit(unit1, false);
    if constexpr (XK) prologue_unit(unit1, true);
    else prologue_unit(unit2, true);
    if constexpr (!YK) prologue_unit(unit2, false);
    else if constexpr (!KK) prologue_unit(unit1, false);  // (two K-major operands: cluster 0 requests Y's pair 1)
    constexpr int PROLOGUE_LOADS = (XK ? 2 : 3) * xop::NL + (KK ? 1 : YK ? 2 : 3) * yop::NL;
    static_assert(xop::NL + yop::NL >= ND, "the units of step 2 must cover one cluster's requests");
    wait_loads_and_barrier<PROLOGUE_LOADS - xop::NL - yop::NL>();

    half8_t fx[TI], fy[TJ];
    if constexpr (MIW_PP_ABLATE & 2) {
        [&]<int... U>(std::integer_sequence<int, U...>) { ((fx[U] = xr.template read<U, 0>(lds)), ...); }(std::make_integer_sequence<int, TI>{});
        [&]<int... U>(std::integer_sequence<int, U...>) { ((fy[U] = yr.template read<U, 0>(lds + XB)), ...); }(std::make_integer_sequence<int, TJ>{});
    }
    // Memory cluster of step 2 pr + H: the fragments of the step, with the cluster's requests
    // issued at even distances between the reads (the reads are bound by the LDS, which the four
    // wavefronts that are in their memory cluster share: a load issued between two of them costs
    // no extra time).
    constexpr int NFRAG = TI + TJ;
    // Fragment unit U of a step (the TI x-fragments, then the TJ y-fragments), preceded by the
    // requests that go out before it: request N before unit N * NFRAG / ND.
    auto cluster_unit = [&]<int H, int U>(MIW_LDS const char *xu, MIW_LDS const char *yu, std::integral_constant<int, H> h,
                                          std::integral_constant<int, U>) MIW_INLINE {
        [&]<int... N>(std::integer_sequence<int, N...>) {
            (([&] {
                 // (Y's loads of a two-K-major kernel have the least time to land: they go out first)
                 if constexpr ((KK && H == 0 ? N : N * NFRAG / ND) == U && !(MIW_PP_ABLATE & 1)) {
                     cluster_request(h, std::integral_constant<int, N>{});
                     __builtin_amdgcn_sched_barrier(0);
                 }
             }()),
             ...);
        }(std::make_integer_sequence<int, ND>{});
        if constexpr (MIW_PP_ABLATE & 2) {
            asm volatile("" : "+v"(fx[U % TI]), "+v"(fy[U % TJ]));
        } else {
            if constexpr (U < TI) fx[U] = xr.template read<U, H>(xu);
            else fy[U - TI] = yr.template read<U - TI, H>(yu);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto memory_cluster = [&]<int H, bool ANY>(std::integral_constant<int, H> h, std::bool_constant<ANY> any) MIW_INLINE {
        MIW_LDS const char *xu = lds + xwave + xpair + (XK ? 0 : H * xop::UNIT_BYTES);
        MIW_LDS const char *yu = lds + XB + ywave + ypair + (YK ? 0 : H * yop::UNIT_BYTES);
        [&]<int... U>(std::integer_sequence<int, U...>) {
            (cluster_unit(xu, yu, h, std::integral_constant<int, U>{}), ...);
        }(std::make_integer_sequence<int, NFRAG>{});
        // The ring state and the operand pointers move on here, behind the last fragment read and under its
        // latency.  (Measured: the same scalar instructions between the first MFMAs of the compute cluster
        // hold the matrix core up for 65 cycles per cluster; between the fragment reads, for 19.)
        cluster_advance(h, any);
        if constexpr (H == 1) pair_advance();
        __builtin_amdgcn_sched_barrier(0);
    };
    auto compute_cluster = [&]() MIW_INLINE {
        __builtin_amdgcn_sched_barrier(0);
        // serpentine order: every MFMA changes exactly one of its two operand fragments
#pragma unroll
        for (int a = 0; a < TI; a++)
#pragma unroll
            for (int bb = 0; bb < TJ; bb++) {
                const int b = serpentine_column(a * TJ + bb, TJ);
                if constexpr (!(MIW_PP_ABLATE & 4)) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fx[a], fy[b], acc[a][b], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
    };

    // Folding C.  The C operand is added into the accumulators during the last NFOLD k-steps, one MFMA tile per
    // step, so that the memory system delivers C while the matrix cores run and the epilogue only stores.  The
    // tile of fold step S is requested at the start of the step with an ordinary load into registers (the lane
    // fetches the 16 bytes it owns); the wait at the end of the memory cluster two steps later covers it, and that
    // cluster adds it in: C has two clusters of both wavefront groups to arrive, and what it takes longer stalls the
    // loop, since loads return in order.  (Requested behind the cluster's own loads, or two tiles every other step,
    // 8192x8192x1024 with C folded takes 3 % longer.)  Three register stages rotate.  Tiles go in the order of their
    // addresses: 16 rows (64 bytes, the instruction's offset field) further down a column block, then the next 16
    // columns.  The accumulators are registers, so the folding steps are unrolled.
    constexpr int NTILE = TI * TJ;
    constexpr int NFOLD = NTILE;
    static_assert(!FOLD || (__is_same(CT, float) && NFOLD == PP_FOLD_STEPS && NFOLD % 2 == 0), "fold steps");
    float4_t cst[3];
    const char *cnext = nullptr;
    // (the lane offset into the tile of C is kept in 32 bits)
    const unsigned coff = 4u * (unsigned)((wj * WTJ + r) * (int)p.ldc + wi * WTI + 4 * q);
    auto fold_request = [&]<int S>(std::integral_constant<int, S>) MIW_INLINE {
        constexpr int a = S % TI;
        asm volatile("global_load_dwordx4 %0, %1, %2 offset:%3" : "=v"(cst[S % 3]) : "v"(coff), "s"(cnext), "n"(64 * a) : "memory");
        if constexpr (a == TI - 1) cnext += 64 * p.ldc;
    };
    auto fold_add = [&]<int S>(std::integral_constant<int, S>) MIW_INLINE {
        constexpr int a = S % TI, b = S / TI;
#pragma unroll
        for (int e = 0; e < 4; e++) acc[a][b][e] = __builtin_fmaf(p.beta, cst[S % 3][e], acc[a][b][e]);
    };
    // Zeroes the repeated k-values in the fragments of step H of the shifted last pair.
    auto mask_tail = [&]<int H>(std::integral_constant<int, H>) MIW_INLINE {
        int skip = tail_skip;
        asm volatile("" : "+s"(skip));  // (the mask is made here, not kept through the tiles)
        const unsigned keep = tail_keep<H>(skip);
#pragma unroll
        for (int a = 0; a < TI; a++) tail_apply(fx[a], keep);
#pragma unroll
        for (int b = 0; b < TJ; b++) tail_apply(fy[b], keep);
    };
    // One k-step: memory cluster, barrier, compute cluster, barrier.  FS: fold step, or -1; ANY: see x_advance; LAST:
    // a step of the last pair.  slack: a step of the first pair of a workgroup's second or later tile.  The NSTORE
    // stores of the tile before are then younger than the loads that the wait is for and may stay in flight.
    constexpr std::integral_constant<int, -1> no_fold{};
    constexpr int NSTORE = TI * TJ;
    auto wait_vm = [&]<int N>(std::integral_constant<int, N>) MIW_INLINE {
        static_assert(N < 64, "vmcnt");
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (0 << 8) | ((N >> 4) << 14));
        asm volatile("" ::: "memory");
    };
    auto step_wait = [&]<int H, int FS>(std::integral_constant<int, H>, std::integral_constant<int, FS>, bool slack) MIW_INLINE {
        // What may stay in flight: the cluster's own loads and, unless they have to land too, those of the cluster
        // before; a fold step issues a load of C ahead of the cluster's.
        constexpr bool BOTH = !(KK && H == 1);
        constexpr int YOUNGER = (BOTH ? 2 : 1) * ND + (FS >= 0 ? (BOTH && FS >= 1 ? 2 : 1) : 0);
        // (the second cluster of two K-major operands waits for loads that were issued behind the stores)
        if (slack && BOTH) wait_vm(std::integral_constant<int, YOUNGER + NSTORE>{});
        else wait_vm(std::integral_constant<int, YOUNGER>{});
    };
    auto barrier = [&]() {
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    auto step = [&]<int H, int FS, bool ANY, bool LAST>(std::integral_constant<int, H> h, std::integral_constant<int, FS> fs,
                                                        std::bool_constant<ANY> any, std::bool_constant<LAST>, bool slack) MIW_INLINE {
        if constexpr (FS >= 0) {
            fold_request(fs);
            __builtin_amdgcn_sched_barrier(0);
        }
        memory_cluster(h, any);
        step_wait(h, fs, slack);
        if constexpr (FS >= 2) {
            __builtin_amdgcn_sched_barrier(0);
            fold_add(std::integral_constant<int, FS - 2>{});
            __builtin_amdgcn_sched_barrier(0);
        }
        barrier();
        if constexpr (LAST) mask_tail(h);
        compute_cluster();
        __builtin_amdgcn_s_barrier();
    };
    constexpr std::true_type last_pair{};
    constexpr std::false_type inner{};
    constexpr std::integral_constant<int, 0> first_half{};
    constexpr std::integral_constant<int, 1> second_half{};
    constexpr std::true_type any{};     // the cluster's requests may reach the last pair
    constexpr std::false_type plain{};

    for (bool later = false;;) {  // tiles of this workgroup
    // Does another tile follow (then NP >= 4, see tiled_params::work), and how do the operands get there?
    auto first_args = arguments();
    has_next = tile + (int)gridDim.x < first_args->work;
    if (has_next) {
        const tile_place next = tile_at(*first_args, tile + (int)gridDim.x, 0, BI, BJ);
        xjump = x_origin(first_args, next.bt, next.i0) - x_origin(first_args, at.bt, at.i0) - ((XN - 2) * xunit + xtail);
        yjump = y_origin(first_args, next.bt, next.j0) - y_origin(first_args, at.bt, at.j0) - ((YN - 2) * yunit + ytail);
    } else {
        xjump = yjump = 0;
    }
    const int i0 = at.i0, j0 = at.j0;
    const long bt = at.bt;
    if constexpr (FOLD) cnext = (const char *)((const CT *)first_args->C + bt * first_args->sc + (long)j0 * first_args->ldc + i0);
    float zero = 0.f;
    asm volatile("" : "+s"(zero));  // (otherwise a zero vector is kept in registers through the tiles)
#pragma unroll
    for (int a = 0; a < TI; a++)
#pragma unroll
        for (int b = 0; b < TJ; b++) acc[a][b] = float4_t{zero, zero, zero, zero};

    MIW_PP_STAMP(1)
    if (late_group) __builtin_amdgcn_s_barrier();
    // the pairs before NPM neither fold nor are the last one; those from NP - 4 on may request the last
    // pair or the next tile
    const int NPM = FOLD ? NP - NFOLD / 2 : NP - 1;
    next_units(0);
    if (NPM > 0) {
        step(first_half, no_fold, any, inner, later);
        step(second_half, no_fold, any, inner, later);
    }
    int pr = 1;
    for (; pr < min(NPM, NP - 4); pr++) {
#ifdef MIW_PP_TS
        if (pr == NPM / 2) MIW_PP_STAMP(2)
        if (pr == NPM / 2 + 1) MIW_PP_STAMP(3)
#endif
        step(first_half, no_fold, plain, inner, false);
        step(second_half, no_fold, plain, inner, false);
    }
    next_units(pr);
    for (; pr < NPM; pr++) {
        step(first_half, no_fold, any, inner, false);
        step(second_half, no_fold, any, inner, false);
    }
    MIW_PP_STAMP(9)
    if constexpr (FOLD) {
        constexpr int GANY = NFOLD / 2 - 4;  // first pair of the last four
        [&]<int... G>(std::integer_sequence<int, G...>) {
            (([&] {
                 if constexpr (G == GANY) next_units(NP - 4);
                 constexpr std::bool_constant<(G >= GANY)> a{};
                 const bool slack = G == 0 && later && NPM == 0;
                 step(first_half, std::integral_constant<int, 2 * G>{}, a, inner, slack);
                 step(second_half, std::integral_constant<int, 2 * G + 1>{}, a, inner, slack);
             }()),
             ...);
        }(std::make_integer_sequence<int, NFOLD / 2 - 1>{});
    }
    step(first_half, std::integral_constant<int, FOLD ? NFOLD - 2 : -1>{}, any, last_pair, false);
    step(second_half, std::integral_constant<int, FOLD ? NFOLD - 1 : -1>{}, any, last_pair, false);
    if (FOLD || !has_next) wait_vm(std::integral_constant<int, 0>{});  // the last tiles of C; no load may outlive the workgroup's LDS
    if constexpr (FOLD) {
        fold_add(std::integral_constant<int, NFOLD - 2>{});
        fold_add(std::integral_constant<int, NFOLD - 1>{});
    }
    if (!late_group) __builtin_amdgcn_s_barrier();
    MIW_PP_STAMP(4)

    // Epilogue: each lane owns 4 consecutive i of one column j per MFMA tile.  Pairs of tiles are exchanged between
    // neighbouring lanes before C is added, so that C is read as D is stored, in pieces of whole lines.
    static_assert(TI % 2 == 0, "the epilogue stores pairs of tiles");
    auto args = arguments();
    const long ldd = args->ldd, ldc = args->ldc;
    int lane = tid & 63;
    asm volatile("" : "+v"(lane));  // (what is made of it is made here, not kept through the K loop)
    const bool odd = lane & 1;
    const float alpha = args->alpha, beta = args->beta;
    DT *D = (DT *)args->D + bt * args->sd + (long)(j0 + wj * WTJ) * ldd + (i0 + wi * WTI) + pair_place(lane, ldd);
    auto store = [](DT *to, float4_t v) MIW_INLINE {
        if constexpr (__is_same(DT, float)) __builtin_nontemporal_store(v, (float4_t *)to);
        else *(half4_t *)to = half4_t{(half_t)v[0], (half_t)v[1], (half_t)v[2], (half_t)v[3]};
    };
    // C_AT 0: no C, 1: laid out as D, 2: the other way round; EDGE: see own_from
    auto epilogue = [&]<int C_AT, bool STREAM, bool EDGE = false>(std::integral_constant<int, C_AT>, std::bool_constant<STREAM>,
                                                                  std::bool_constant<EDGE> = {}) MIW_INLINE {
        const int row = i0 + wi * WTI + 16 * odd, first_row = own_from<BI>(i0), col = j0 + wj * WTJ, first_col = own_from<BJ>(j0);
        const CT *C = nullptr;
        if constexpr (C_AT == 1) C = (const CT *)args->C + bt * args->sc + (long)(j0 + wj * WTJ) * ldc + (i0 + wi * WTI) + pair_place(lane, ldc);
        // (columns r - odd and the next, rows 16 odd + 4 q ..)
        if constexpr (C_AT == 2) C = (const CT *)args->C + bt * args->sc + (long)(i0 + wi * WTI + 16 * odd + 4 * (lane >> 4)) * ldc + (j0 + wj * WTJ + (lane & 14));
#pragma unroll
        for (int b = 0; b < TJ; b++)
#pragma unroll
            for (int a = 0; a < TI; a += 2) {
                float4_t v[2] = {acc[a][b], acc[a + 1][b]};
#pragma unroll
                for (int t = 0; t < 2; t++)
#pragma unroll
                    for (int e = 0; e < 4; e++) v[t][e] *= alpha;
                if constexpr (C_AT == 0) {
                    store_pair_at<STREAM>(D + 16 * b * ldd + 16 * a, ldd, odd, v[0], v[1],
                                          !EDGE || (row + 16 * a >= first_row && col + 16 * b >= first_col));
                } else {
                    pair_exchange(odd, v[0], v[1]);
#pragma unroll
                    for (int t = 0; t < 2; t++) {
                        float4_t c;
                        if constexpr (C_AT == 2) {
#pragma unroll
                            for (int e = 0; e < 4; e++) c[e] = (float)C[(16 * a + e) * ldc + 16 * b + t];
                        } else if constexpr (__is_same(CT, float)) {
                            c = *(const float4_t *)(C + (16 * b + t) * ldc + 16 * a);
                        } else {
                            const half4_t h = *(const half4_t *)(C + (16 * b + t) * ldc + 16 * a);
                            c = float4_t{(float)h[0], (float)h[1], (float)h[2], (float)h[3]};
                        }
#pragma unroll
                        for (int e = 0; e < 4; e++) v[t][e] = __builtin_fmaf(beta, c[e], v[t][e]);
                    }
                    store(D + 16 * b * ldd + 16 * a, v[0]);
                    store(D + (16 * b + 1) * ldd + 16 * a, v[1]);
                }
            }
    };
    // A Float32 D is written past the L2 where C or the operands of more tiles come through it at the same time
    // (4096x4096x512 with C from HBM: 34 us, 42 through the L2; 8192x8192x1024 without C 126 and 134), and through it
    // where nothing follows in the launch (4096x4096x512 without C: 26 us, 28 past it).
    const bool edge = FOLD && (i0 % BI || j0 % BJ);
    if (edge) epilogue(std::integral_constant<int, 0>{}, std::true_type{}, std::true_type{});
    else if (FOLD) epilogue(std::integral_constant<int, 0>{}, std::true_type{});
    else if (args->use_c && args->c_trans) epilogue(std::integral_constant<int, 2>{}, std::true_type{});
    else if (args->use_c) epilogue(std::integral_constant<int, 1>{}, std::true_type{});
    else if (args->work) epilogue(std::integral_constant<int, 0>{}, std::true_type{});
    else epilogue(std::integral_constant<int, 0>{}, std::false_type{});
#ifdef MIW_PP_TS
    MIW_PP_STAMP(5)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    MIW_PP_STAMP(6)
    ts[7] = wall_clock64();
    if (p.ts && lane == 0)
        for (int i = 0; i < 10; i++) p.ts[(launch_tile(tile, p.span, blockIdx.y, gridDim.x) * 8 + wave) * 10 + i] = ts[i];
    ts[0] = clock64();
    ts[8] = wall_clock64();
#endif
    if (!has_next) break;
    later = !edge;  // (a tile at the edge may have stored less)
    tile += (int)gridDim.x;
    at = tile_at(*arguments(), tile, 0, BI, BJ);
    }
}

// C, if any, is read in the epilogue.
template <int BI, int BJ, int WI, int WJ, bool XK, bool YK, class CT, class DT>
__global__ __launch_bounds__(WI *WJ * 64) __attribute__((amdgpu_waves_per_eu(2)))
void k_gemm_pp(tiled_params p)
{
    gemm_pp<BI, BJ, WI, WJ, XK, YK, CT, DT, false>(p);
}

// A Float32 C is folded into the K loop.
template <int BI, int BJ, int WI, int WJ, bool XK, bool YK, class DT>
__global__ __launch_bounds__(WI *WJ * 64) __attribute__((amdgpu_waves_per_eu(2)))
void k_gemm_pp_fold(tiled_params p)
{
    gemm_pp<BI, BJ, WI, WJ, XK, YK, float, DT, true>(p);
}

// ---------------------------------------------------------------------------
// Ping-pong kernel with clusters of 64 k-values (one LDS slot), for the tiles whose rings of whole
// slots fit in LDS: 256x128, 128x256 (three slots) and 128x128 (four).  A wavefront's memory
// cluster reads the fragments of both k-steps of pair p out of the pair's slot and requests pair
// p + NSLOT - 1 into the slot of pair p - 1 (which the other group finished reading one barrier
// ago); its compute cluster issues the pair's 2 * TI * TJ MFMAs.  At the end of the memory cluster
// the wavefront lets the NSLOT - 2 youngest pairs stay in flight: pair p + 1 has landed, and the
// two barriers that follow publish it before anyone reads it.  Both operand kinds use the slot
// layouts, loaders and fragment readers of gemm_tiled.hpp.
//
// A wavefront issues one instruction in four to five cycles, whatever the instruction, and only one
// instruction rides for nothing behind each MFMA.  So both clusters are as long as their instruction
// counts: the memory cluster is kept to the fragment reads, three instructions per load and a handful
// of scalar ones (the part of the loop that needs no look at the end of K is unrolled over the ring,
// so that slots are compile-time offsets, and advances the operand origins behind MFMAs of the compute
// cluster), and the compute cluster to the MFMAs and what must follow them.
//
// fp16 accumulation rounds once per slot (64 k-values), two MFMAs after a tile's last MFMA of the pair,
// inside the compute cluster, except the cluster's last two tiles, which the wavefront rounds at the
// end of its next memory cluster (more there, or the conversions between the fragment reads, lengthen
// the memory cluster beyond the compute cluster: measured, up to 25 % of the launch).  With alpha == 1
// the accumulators start as half(beta * C) and the MFMAs accumulate onto the rounded sum in place,
// otherwise the running sum is kept beside accumulators that restart from zero in every slot:
// run = half(run + alpha * slot sum).  C is requested before anything else and converted once the
// first pair's loads have landed.  With Float32 accumulation C waits in registers for the end of the loop.
template <int BI, int BJ, int WI, int WJ, int NSLOT, bool XK, bool YK, class CT, class DT, bool F16ACC>
__global__ __launch_bounds__(WI *WJ * 64) __attribute__((amdgpu_waves_per_eu(2)))
void k_gemm_pp64(tiled_params p)
{
    constexpr int NT = WI * WJ * 64;
    static_assert(NT == 512, "two wavefronts per SIMD");
    constexpr int WTI = BI / WI, WTJ = BJ / WJ;
    constexpr int TI = WTI / 16, TJ = WTJ / 16;
    constexpr int XBYTES = BI * KGRAN * 2, YBYTES = BJ * KGRAN * 2, SLOT = XBYTES + YBYTES;
    static_assert(NSLOT >= 3 && NSLOT * SLOT <= 160 * 1024, "ring does not fit in LDS");
    using xload = slot_loader<BI, XK, NT>;
    using yload = slot_loader<BJ, YK, NT>;
    constexpr int NLX = xload::NLOAD, NLY = yload::NLOAD, LPAIR = NLX + NLY;  // loads per thread and pair
    constexpr int NTILE = TI * TJ;
    constexpr int NFRAG = 2 * (TI + TJ);  // fragment units of a memory cluster

#ifdef MIW_PP_TS
    long long ts[10] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    ts[0] = clock64();
    ts[8] = wall_clock64();
#endif
    extern __shared__ __attribute__((aligned(128))) char smem[];
    MIW_LDS char *lds = (MIW_LDS char *)smem;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wi = wave % WI, wj = wave / WI;
    const bool late_group = wave >= 4;

    // (with Float16 accumulation C is requested ahead of the operands: one wait for all arguments)
    if constexpr (F16ACC) fetch_arguments(p);
    else fetch_operand_arguments(p);
    const tile_place at = workgroup_tile(p, BI, BJ);
    const int i0 = at.i0, j0 = at.j0;
    const long bt = at.bt;

    const half_t *X = p.X + bt * p.sx + (XK ? (long)i0 * p.ldx : (long)i0);
    const half_t *Y = p.Y + bt * p.sy + (YK ? (long)j0 * p.ldy : (long)j0);
    const unsigned xoff = xload::lane_offset(tid, (int)p.ldx);
    const unsigned yoff = yload::lane_offset(tid, (int)p.ldy);

    frag_reader<BI, XK> xr;
    frag_reader<BJ, YK> yr;
    xr.init(wi * WTI, lane);
    yr.init(wj * WTJ, lane);

    const int q = lane >> 4, r = lane & 15;
    const int row = i0 + wi * WTI + 4 * q;  // + 16*ti
    const int col = j0 + wj * WTJ + r;      // + 16*tj
    const CT *C = (const CT *)p.C + bt * p.sc;
    DT *D = (DT *)p.D + bt * p.sd;

    float4_t acc[TI][TJ];
#pragma unroll
    for (int a = 0; a < TI; a++)
#pragma unroll
        for (int b = 0; b < TJ; b++) acc[a][b] = float4_t{0.f, 0.f, 0.f, 0.f};

    auto read_c_across = [&](int a, int b) -> float4_t {
        float4_t c;
#pragma unroll
        for (int v = 0; v < 4; v++) c[v] = (float)C[(long)(row + 16 * a + v) * p.ldc + (col + 16 * b)];
        return c;
    };

    const int K = has_slices<CT, DT, F16ACC> ? member_k(p, at.bt) : p.K;
    const int NP = (K + KGRAN - 1) / KGRAN;
    // K tail: the last pair starts at K - 64; tail_skip of its k-values repeat the pair before
    const int tail_skip = NP * KGRAN - K;
    const unsigned wave_dst = (unsigned)(uintptr_t)lds + (unsigned)wave * 1024u;
    int next = 0;          // next pair to request
    unsigned woff = 0;     // byte offset in the ring of the slot it goes to
    unsigned dma_dst = 0;  // this wavefront's first destination byte in that slot
    // A wavefront issues little more than one instruction in four to five cycles, whatever the
    // instruction, and its memory cluster is a chain of some sixty of them: every scalar instruction
    // spent on addresses there lengthens the cluster as much as a fragment read does.  So a load is
    // three instructions (M0 written by the addition that forms the LDS address; the global address is
    // the slot's uniform origin plus a lane offset, the loads of a K-major operand, whose origins lie
    // a multiple of the leading dimension apart, each with a lane offset of their own, the others with
    // the instruction's offset field), the ring positions are kept as byte offsets, and the pairs whose
    // request needs no look at the end of K (FAST) advance the origins by a loop-invariant step.
    unsigned xvo[XK ? NLX : 1], yvo[YK ? NLY : 1];
#pragma unroll
    for (int i = 0; i < (XK ? NLX : 1); i++) xvo[i] = xoff + 2u * (unsigned)xload::load_delta(i, p.ldx);
#pragma unroll
    for (int i = 0; i < (YK ? NLY : 1); i++) yvo[i] = yoff + 2u * (unsigned)yload::load_delta(i, p.ldy);
    auto begin_request = [&]() { dma_dst = wave_dst + woff; };
    // the same for a pair that reads slot SL, known at compile time: its request goes to the slot before
    auto begin_request_at = [&]<int SL>(std::integral_constant<int, SL>) { dma_dst = wave_dst + (unsigned)((SL + NSLOT - 1) % NSLOT * SLOT); };
    auto request_one = [&]<int I>(std::integral_constant<int, I>) {
        if constexpr (I < NLX) {
            if constexpr (XK) lds_dma16_at<I * NT * 16, 0>(X, xvo[I], dma_dst);
            else lds_dma16_at<I * NT * 16, I * (NT / 512) * 128>(X, xvo[0], dma_dst);  // load_delta: 64 rows further along i
        } else {
            constexpr int J = I - NLX;
            if constexpr (YK) lds_dma16_at<XBYTES + J * NT * 16, 0>(Y, yvo[J], dma_dst);
            else lds_dma16_at<XBYTES + J * NT * 16, J * (NT / 512) * 128>(Y, yvo[0], dma_dst);
        }
    };
    // Past the end of K the last pair is requested again, into a slot nobody reads any more.
    auto end_request = [&]() {
        next++;
        woff = woff + SLOT == NSLOT * SLOT ? 0 : woff + SLOT;
        const int kstep = next < NP - 1 ? KGRAN : next == NP - 1 ? KGRAN - tail_skip : 0;
        // (64 leading dimensions fit in 32 bits: the host checks that 256 do)
        X += XK ? kstep : kstep * (int)p.ldx;
        Y += YK ? kstep : kstep * (int)p.ldy;
    };
    // FAST pairs: one origin per call, issued behind an MFMA of the compute cluster
    auto advance_fast = [&](int which) {
        if (which == 0) X += XK ? KGRAN : KGRAN * (int)p.ldx;
        else Y += YK ? KGRAN : KGRAN * (int)p.ldy;
    };

    // fp16 accumulation: the C operand is requested first, as raw bits that no instruction touches
    // before the prologue's wait (a conversion here would make the compiler wait for the loads
    // before the first direct-to-LDS load is issued).  C laid out as D: the lane's four halves in two
    // registers; C stored across D: one zero-extended half per register.
    //
    // Where LDS has room for the workgroup's whole tile of C beside the ring (128 x 128: 32 KiB), a C laid
    // out as D comes through LDS instead: the accumulator layout reads 32 contiguous bytes per column
    // and instruction, which costs the 128 x 128 kernel 6000 cycles of prologue, whereas direct-to-LDS
    // loads fetch whole 256-byte columns (16 lanes per column).  Chunk (column j, 16-byte piece c) sits at
    // chunk index j * 16 + (c ^ (j & 15)), so that the 16 lanes that later read 16 columns at one row
    // offset hit 16 different 16-byte slots.
    constexpr bool C_STAGE_FITS = F16ACC && NSLOT * SLOT + BI * BJ * 2 <= 160 * 1024 && (BI * 2) % 256 == 0;
    constexpr int C_STAGE = NSLOT * SLOT;                         // byte offset of the staged tile
    constexpr int C_CHUNKS_PER_COL = BI * 2 / 16, NLC = C_STAGE_FITS ? BI * BJ * 2 / 16 / NT : 0;
    const bool c_staged = C_STAGE_FITS && p.use_c && !p.c_trans && p.ldc < (1l << 22);  // (32-bit lane offsets)
    if constexpr (C_STAGE_FITS) {
        if (c_staged) {
            const char *ctile = (const char *)(C + (long)j0 * p.ldc + i0);
#pragma unroll
            for (int n = 0; n < NLC; n++) {
                const int g = n * NT + tid;
                const int j = g / C_CHUNKS_PER_COL, c = (g % C_CHUNKS_PER_COL) ^ (j & 15);
                lds_dma16(ctile, (unsigned)(j * (int)p.ldc * 2 + c * 16), wave_dst + (unsigned)(C_STAGE + n * NT * 16));
            }
        }
    }
    unsigned craw[F16ACC ? TI : 1][F16ACC ? TJ : 1][4];
    if constexpr (F16ACC) {
        if (p.use_c && !c_staged) {
            auto fetch = [&]<bool TRANS>(std::bool_constant<TRANS>) {
#pragma unroll
                for (int a = 0; a < TI; a++)
#pragma unroll
                    for (int b = 0; b < TJ; b++) {
                        const int ii = row + 16 * a, jj = col + 16 * b;
                        if constexpr (TRANS) {
#pragma unroll
                            for (int v = 0; v < 4; v++) craw[a][b][v] = *(const unsigned short *)(C + (long)(ii + v) * p.ldc + jj);
                        } else {
                            const uint2_t two = *(const uint2_t *)(C + (long)jj * p.ldc + ii);
                            craw[a][b][0] = two[0];
                            craw[a][b][1] = two[1];
                        }
                    }
            };
            if (p.c_trans) fetch(std::true_type{});
            else fetch(std::false_type{});
        }
    }
    // Prologue: the first NSLOT - 1 pairs are requested.
#pragma unroll
    for (int s = 0; s < NSLOT - 1; s++) {
        begin_request();
        [&]<int... I>(std::integer_sequence<int, I...>) { (request_one(std::integral_constant<int, I>{}), ...); }
        (std::make_integer_sequence<int, LPAIR>{});
        end_request();
    }
    if constexpr (!F16ACC) fetch_result_arguments(p);
    // Float32 accumulation: C laid out as D goes into registers while the loop runs (request_c), in the whole lines in which D
    // is stored.  (Added to the sums in the loop's last pairs, as k_gemm_pp_fold does, it costs those pairs a quarter more each,
    // and read behind the loop two loads at a time it waits for memory once per pair of tiles: 8192x1024x4096 from HBM
    // 73.1 us -> 68.0, with the times of tiled_params::c_spread, 7120x1024x720 with a Float16 C 18.9 -> 17.9, 2048x2048x128
    // 11.1 -> 8.9.  128x128 tiles in one round with a Float32 C, alpha of 1 and K above 1024 are 1 to 2.5 % behind the
    // folded form, whose sums are further from the exact result: 2048x2048x2048 20.4 -> 20.9, 1600x2064x2048 18.6 -> 19.0.)
    using cpieces = c_pieces<TI, TJ, CT>;
    cpieces cp;
    // Problems without C have instances of their own, without C's registers: 1280x5168x1408 23.0 us -> 22.6, 8192x768x1024
    // 17.9 -> 17.7, 1024x3072x1024 11.5 -> 11.0 (2048^3 level).
    constexpr bool HAS_C = !__is_same(CT, no_c_t);
    const bool early = HAS_C && !F16ACC && p.use_c && !p.c_trans;
    auto request_c = [&]() MIW_INLINE { cp.request(C + (long)(j0 + wj * WTJ) * p.ldc + (i0 + wi * WTI) + pair_place(lane, p.ldc), p.ldc); };
    // The loop starts when pair 0 (and, with Float16 accumulation, the C operand, requested before it) has landed: the
    // wait at the end of memory cluster p leaves NSLOT - 2 pairs in flight, so pair p + 1 has landed by then, the
    // first time as every other.
    wait_loads_and_barrier<(NSLOT - 2) * LPAIR>();
    float4_t cinit[F16ACC ? TI : 1][F16ACC ? TJ : 1];
    if constexpr (F16ACC) {
        auto convert = [&]<bool TRANS>(std::bool_constant<TRANS>) {
#pragma unroll
            for (int a = 0; a < TI; a++)
#pragma unroll
                for (int b = 0; b < TJ; b++)
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        const unsigned bits = TRANS ? craw[a][b][v] : craw[a][b][v >> 1] >> (16 * (v & 1));
                        const float c = (float)__builtin_bit_cast(half_t, (unsigned short)bits);
                        cinit[a][b][v] = round_through_half(p.beta * c);
                    }
        };
        if (!p.use_c) {
#pragma unroll
            for (int a = 0; a < TI; a++)
#pragma unroll
                for (int b = 0; b < TJ; b++) cinit[a][b] = float4_t{0.f, 0.f, 0.f, 0.f};
        } else if (c_staged) {
            if constexpr (C_STAGE_FITS) {
#pragma unroll
                for (int a = 0; a < TI; a++)
#pragma unroll
                    for (int b = 0; b < TJ; b++) {
                        const int j = wj * WTJ + 16 * b + r, i = wi * WTI + 16 * a + 4 * q;
                        const int at = C_STAGE + (j * C_CHUNKS_PER_COL + ((i >> 3) ^ (j & 15))) * 16 + (i & 7) * 2;
                        const half4_t h = *(MIW_LDS const half4_t *)(lds + at);
#pragma unroll
                        for (int v = 0; v < 4; v++) cinit[a][b][v] = round_through_half(p.beta * (float)h[v]);
                    }
            }
        } else if (p.c_trans) {
            convert(std::true_type{});
        } else {
            convert(std::false_type{});
        }
    }

    half8_t fx[2][TI], fy[2][TJ];
    if constexpr (MIW_PP_ABLATE & 2) {
        [&]<int... U>(std::integer_sequence<int, U...>) { ((fx[0][U] = fx[1][U] = xr.template read<U, 0>(lds)), ...); }(std::make_integer_sequence<int, TI>{});
        [&]<int... U>(std::integer_sequence<int, U...>) { ((fy[0][U] = fy[1][U] = yr.template read<U, 0>(lds + XBYTES)), ...); }(std::make_integer_sequence<int, TJ>{});
    }
    // fp16 accumulation: rounding of tile t = a * TJ + b after its pair's MFMAs.
    // RMODE 1 (alpha == 1): the accumulators start as half(beta * C), the MFMAs accumulate onto the
    //     rounded running sum, and it is rounded in place once per slot.
    // RMODE 3 (any alpha): `cinit` is the running sum (a Float16 value held as Float32), the MFMA
    //     accumulators restart from zero in every slot and run = half(run + alpha * slot sum).
    auto round_tile = [&]<int RMODE>(int t, std::integral_constant<int, RMODE>) {
        const int a = t / TJ, b = t % TJ;
        float4_t v = acc[a][b];
        if constexpr (RMODE == 3) {
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] = __builtin_fmaf(p.alpha, v[e], cinit[a][b][e]);
        }
        half4_t h = __builtin_convertvector(v, half4_t);
        if constexpr (RMODE == 3) cinit[a][b] = __builtin_convertvector(h, float4_t);
        else acc[a][b] = __builtin_convertvector(h, float4_t);
    };
    // Fragment unit U of a memory cluster (step 0: the TI x-fragments, then the TJ y-fragments; then
    // step 1), preceded by the direct-to-LDS loads that go out before it (load n before unit
    // n * NFRAG / LPAIR).
    auto cluster_unit = [&]<int U>(MIW_LDS const char *xs, std::integral_constant<int, U>) {
        [&]<int... N>(std::integer_sequence<int, N...>) {
            (([&] {
                 if constexpr (N * NFRAG / LPAIR == U && !(MIW_PP_ABLATE & 1)) {
                     request_one(std::integral_constant<int, N>{});
                     __builtin_amdgcn_sched_barrier(0);
                 }
             }()),
             ...);
        }(std::make_integer_sequence<int, LPAIR>{});
        constexpr int H = U / (TI + TJ), V = U % (TI + TJ);
        if constexpr (MIW_PP_ABLATE & 2) {
            asm volatile("" : "+v"(fx[H][V % TI]), "+v"(fy[H][V % TJ]));
        } else {
            if constexpr (V < TI) fx[H][V] = xr.template read<V, H>(xs);
            else fy[H][V - TI] = yr.template read<V - TI, H>(xs + XBYTES);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    unsigned roff = 0;  // byte offset in the ring of the slot that is read next
    // SL: -2: any pair; -1: a FAST pair; >= 0: a FAST pair that reads slot SL, known at compile time (the
    // loop is unrolled over the ring there: no ring position to keep, and the slot's offset is part of
    // the instructions' offset fields).  FAST pairs advance the origins in their compute cluster.
    auto memory_cluster = [&]<int SL>(std::integral_constant<int, SL> sl) {
        MIW_LDS const char *xs = SL >= 0 ? lds + SL * SLOT : lds + roff;
        if constexpr (SL >= 0) begin_request_at(sl);
        else begin_request();
        [&]<int... U>(std::integer_sequence<int, U...>) {
            (cluster_unit(xs, std::integral_constant<int, U>{}), ...);
        }(std::make_integer_sequence<int, NFRAG>{});
        if constexpr (SL == -2) end_request();
        if constexpr (SL == -1) woff = woff + SLOT == NSLOT * SLOT ? 0 : woff + SLOT;
        if constexpr (SL < 0) roff = roff + SLOT == NSLOT * SLOT ? 0 : roff + SLOT;
        __builtin_amdgcn_sched_barrier(0);
    };
    // ZERO (fp16 accumulation with alpha != 1): the accumulators restart from zero in every slot.
    auto tile_of_mfma = [](int m) { return m / TJ * TJ + serpentine_column(m, TJ); };
    // (fp16 accumulation, measured: with both k-steps of a tile back to back, so that the tiles finish
    // one after the other and the conversions spread over the whole cluster, the second MFMA of a tile
    // waits for the first and the launch takes 6 to 15 % longer.)
    constexpr int ROUND_LAG = 2;
    // The tiles whose last MFMA closes the compute cluster would be rounded behind it, with no MFMA to hide
    // the conversions and the other group waiting at the barrier: the last ROUND_DEFER tiles are rounded
    // at the end of the wavefront's next memory cluster instead (round_deferred), behind its last
    // fragment read and before the next compute cluster touches them.  (Measured on 2048^3: 1 or 2 tiles
    // 3 % faster than none, 3 and more slower again: the memory cluster must stay the shorter one.)
    constexpr int ROUND_DEFER = F16ACC ? 2 : 0;
    static_assert(ROUND_DEFER <= NTILE && ROUND_DEFER <= ROUND_LAG, "deferred tiles are the cluster's last");
    auto compute_cluster = [&]<bool ZERO, bool ADVANCE>(std::bool_constant<ZERO>, std::bool_constant<ADVANCE>) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int m = 0; m < NTILE; m++) {
                // serpentine order: every MFMA changes exactly one of its two operand fragments
                const int a = m / TJ, b = serpentine_column(m, TJ);
                if constexpr (!(MIW_PP_ABLATE & 4)) {
                    if (ZERO && h == 0) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fx[h][a], fy[h][b], float4_t{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                    else acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fx[h][a], fy[h][b], acc[a][b], 0, 0, 0);
                }
                // fp16 accumulation: a tile is rounded ROUND_LAG MFMAs after its last MFMA of the pair
                if constexpr (ADVANCE)
                    if (h == 0 && m < 2) advance_fast(m);
                if constexpr (F16ACC)
                    if (h == 1 && m >= ROUND_LAG && m - ROUND_LAG < NTILE - ROUND_DEFER) round_tile(tile_of_mfma(m - ROUND_LAG), std::integral_constant<int, ZERO ? 3 : 1>{});
                __builtin_amdgcn_sched_barrier(0);
            }
        if constexpr (F16ACC)
#pragma unroll
            for (int m = NTILE > ROUND_LAG ? NTILE - ROUND_LAG : 0; m < NTILE - ROUND_DEFER; m++) round_tile(tile_of_mfma(m), std::integral_constant<int, ZERO ? 3 : 1>{});
    };
    // The first memory cluster rounds sums that are Float16 values already, which changes nothing, and
    // the last compute cluster's tiles are rounded behind the loop.
    auto round_deferred = [&]<bool ZERO>(std::bool_constant<ZERO>) {
#pragma unroll
        for (int m = NTILE - ROUND_DEFER; m < NTILE; m++) round_tile(tile_of_mfma(m), std::integral_constant<int, ZERO ? 3 : 1>{});
    };

    // Zeroes the repeated k-values in the fragments of the shifted last pair.
    auto mask_tail = [&]() {
        const unsigned keep0 = tail_keep<0>(tail_skip), keep1 = tail_keep<1>(tail_skip);
#pragma unroll
        for (int a = 0; a < TI; a++) { tail_apply(fx[0][a], keep0); tail_apply(fx[1][a], keep1); }
#pragma unroll
        for (int b = 0; b < TJ; b++) { tail_apply(fy[0][b], keep0); tail_apply(fy[1][b], keep1); }
    };
    // One pair: memory cluster, barrier, compute cluster, barrier.  LAST: its fragments are masked.  RMODE: how the
    // compute cluster rounds its sums (0: fp32 accumulation; 1, 3: see round_tile).  fresh: C, requested behind the
    // first NSLOT - 1 pairs, may still be in flight.
    auto pair = [&]<bool LAST, int RMODE, int SL = -2>(std::bool_constant<LAST>, std::integral_constant<int, RMODE>, std::integral_constant<int, SL> sl = {}, bool fresh = false) {
        memory_cluster(sl);
        if constexpr (RMODE != 0) {
            round_deferred(std::bool_constant<RMODE == 3>{});
            __builtin_amdgcn_sched_barrier(0);
        }
        if (fresh) wait_loads_and_barrier<(NSLOT - 2) * LPAIR + cpieces::LOADS>();
        else wait_loads_and_barrier<(NSLOT - 2) * LPAIR>();
        if constexpr (LAST) mask_tail();
        compute_cluster(std::bool_constant<RMODE == 3>{}, std::bool_constant<SL != -2>{});
        __builtin_amdgcn_s_barrier();
    };
    constexpr std::false_type inner{};
    constexpr std::true_type last_pair{};
    constexpr std::integral_constant<int, -1> fast_pair{};
    // NSLOT pairs that need no look at the end of K, the first of which reads slot 0
#ifdef MIW_PP_TS
    bool stamp_pair = false;
#endif
    // fresh: C has been asked for in front of them
    auto ring_of_pairs = [&]<int RMODE>(std::integral_constant<int, RMODE> rmode, bool fresh = false) {
        [&]<int... S>(std::integer_sequence<int, S...>) {
            (([&] {
#ifdef MIW_PP_TS
                 if constexpr (S == 1)
                     if (stamp_pair) MIW_PP_STAMP(3)
#endif
                 pair(inner, rmode, std::integral_constant<int, S>{}, S < NSLOT - 2 && fresh);
             }()),
             ...);
        }(std::make_integer_sequence<int, NSLOT>{});
    };
    constexpr std::integral_constant<int, 0> plain{};

    MIW_PP_STAMP(1)
    if (late_group) __builtin_amdgcn_s_barrier();
    const int NPM = NP - 1;  // pairs but the last
    // the request of pair pr is pair pr + NSLOT - 1; the pairs before NP - 1 lie a full step apart
    const int NFAST = min(NPM, max(0, NP - 1 - NSLOT));
    const bool separate_sum = F16ACC && p.alpha != 1.0f;
    if constexpr (F16ACC) {
        // The running sum starts as half(beta * C): with alpha == 1 in the accumulators, which the MFMAs
        // add onto; otherwise beside them.
        constexpr std::integral_constant<int, 1> rolling{};
        constexpr std::integral_constant<int, 3> separate{};
        if (separate_sum) {
            int pr = 0;
            for (; pr + NSLOT <= NFAST; pr += NSLOT) ring_of_pairs(separate);
            for (; pr < NFAST; pr++) pair(inner, separate, fast_pair);
            next = NSLOT - 1 + pr;
            for (; pr < NPM; pr++) pair(inner, separate);
            pair(last_pair, separate);
            round_deferred(std::true_type{});
        } else {
#pragma unroll
            for (int a = 0; a < TI; a++)
#pragma unroll
                for (int b = 0; b < TJ; b++) acc[a][b] = cinit[a][b];
            int pr = 0;
            for (; pr + NSLOT <= NFAST; pr += NSLOT) {
                MIW_PP_MIDDLE(pr)
                ring_of_pairs(rolling);
            }
            for (; pr < NFAST; pr++) pair(inner, rolling, fast_pair);
            next = NSLOT - 1 + pr;
            for (; pr < NPM; pr++) pair(inner, rolling);
            MIW_PP_STAMP(9)
            pair(last_pair, rolling);
            round_deferred(std::false_type{});
        }
    } else {
        int pr = 0;
        // The ring of pairs that C is asked for in front of (see tiled_params::c_spread); behind all rings, in front of the last
        // pair.  Without a ring it is there in any case: so few pairs end before C arrives, and C's loads would hold theirs up.
        const int rings = max(0, NFAST / NSLOT);
        const int c_ring = BI * BJ > 128 * 128 && p.c_spread ? max(2, rings) * spread_phase() >> 3 : 0, c_at = c_ring * NSLOT;
        const bool late = c_ring >= rings;
        for (; pr + NSLOT <= NFAST; pr += NSLOT) {
            MIW_PP_MIDDLE(pr)
            const bool now = early && pr == c_at;
            if (now) request_c();
            ring_of_pairs(plain, now);
        }
        for (; pr < NFAST; pr++) pair(inner, plain, fast_pair);
        next = NSLOT - 1 + pr;
        for (; pr < NPM; pr++) pair(inner, plain);
        if (early && late) request_c();
        MIW_PP_STAMP(9)
        pair(last_pair, plain, std::integral_constant<int, -2>{}, early && late);  // (nothing that it reads is on the way any more)
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no load may outlive the workgroup's LDS
    if (!late_group) __builtin_amdgcn_s_barrier();
    MIW_PP_STAMP(4)

    // Epilogue: each lane owns 4 consecutive i of one column j per MFMA tile; tiles go out in pairs.
    static_assert(TI % 2 == 0, "the epilogue stores pairs of tiles");
    const bool odd = lane & 1;
    DT *to = D + (long)(j0 + wj * WTJ) * p.ldd + (i0 + wi * WTI) + pair_place(lane, p.ldd);
    // C_AT 0: nothing to add, 1: C laid out as D, in registers, 2: C laid out the other way round
    auto epilogue = [&]<int C_AT>(std::integral_constant<int, C_AT>) {
#pragma unroll
        for (int b = 0; b < TJ; b++)
#pragma unroll
            for (int a = 0; a < TI; a += 2) {
                float4_t v[2];
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    v[t] = separate_sum ? cinit[a + t][b] : acc[a + t][b];
                    if constexpr (!F16ACC) v[t] *= p.alpha;
                    if constexpr (C_AT == 2) {
                        const float4_t c = read_c_across(a + t, b);
#pragma unroll
                        for (int e = 0; e < 4; e++) v[t][e] = __builtin_fmaf(p.beta, c[e], v[t][e]);
                    }
                }
                DT *at = to + 16 * b * p.ldd + 16 * a;
                if constexpr (C_AT == 1) {
                    pair_exchange(odd, v[0], v[1]);
                    cp.add(a, b, p.beta, v[0], v[1]);
                    store_pieces_at<DT>(at, p.ldd, v[0], v[1]);
                } else {
                    store_pair_at(at, p.ldd, odd, v[0], v[1]);
                }
            }
    };
    if (F16ACC || !HAS_C || !p.use_c) epilogue(std::integral_constant<int, 0>{});
    else if (p.c_trans) epilogue(std::integral_constant<int, 2>{});
    else epilogue(std::integral_constant<int, 1>{});
#ifdef MIW_PP_TS
    MIW_PP_STAMP(5)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    MIW_PP_STAMP(6)
    ts[7] = wall_clock64();
    if (p.ts && lane == 0)
        for (int i = 0; i < 10; i++) p.ts[((long)(blockIdx.y * gridDim.x + blockIdx.x) * 8 + wave) * 10 + i] = ts[i];
#endif
}

}  // namespace miw
