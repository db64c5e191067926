// GEMM on tiles of 16x32 to 64x32 whose wavefronts share K: for problems whose small tiles take one round over the CUs.
#include "gemm_tiled.hpp"

#include <algorithm>

namespace miw {

constexpr int KWAVES = 4;

template <int BI, int BJ>
struct kwave_shape {
    static constexpr int SLOT = (BI + BJ) * KGRAN * 2;
    static constexpr int SLOTS = 160 * 1024 / (KWAVES * SLOT);  // per wavefront
    static_assert(SLOTS >= 2, "one slot is read while another is on the way");
    static constexpr int PITCH = BI + 4;  // floats from one column of a partial sum to the next: 16 columns fall on 64 banks
    static constexpr int RING = KWAVES * SLOTS * SLOT > KWAVES * PITCH * BJ * 4 ? KWAVES * SLOTS * SLOT : KWAVES * PITCH * BJ * 4;
};

// One wavefront's slot of an operand, R rows (or columns) of 64 k-values, and its fragments.
//   K-major, and I-major with 64 rows: the layout of gemm_tiled.hpp, which frag_reader reads.  Load i fetches eight
//     rows of 128 bytes.
//   I-major with 32 rows: 64 k-rows of 64 bytes, their two halves swapped where bit 3 of k is set, so that the row pieces
//     of one transposing read fall on all banks.  Load i fetches sixteen rows.
template <int R, bool KMAJOR>
struct wave_operand {
    static constexpr bool HALF_LINES = !KMAJOR && R == 32;
    static constexpr int NLOAD = R / 8;
    static_assert(KMAJOR || R == 64 || R == 32, "an operand with i contiguous is fetched in rows of 64 or 32 i");
    unsigned off[NLOAD];
    frag_reader<R, KMAJOR> whole;
    int half[2];
    __device__ inline void init(int lane, int ld)
    {
#pragma unroll
        for (int i = 0; i < NLOAD; i++) {
            if constexpr (HALF_LINES) {
                const int k = 16 * i + (lane >> 2), c = (lane & 3) ^ (2 * ((k >> 3) & 1));
                off[i] = 2u * (unsigned)(k * ld + c * 8);
            } else {
                const int row = 8 * i + (lane >> 3);  // K-major: row of the operand, else k
                const int c = (lane & 7) ^ (KMAJOR ? (row >> 1) & 7 : 2 * i_major_swizzle(row));
                off[i] = 2u * (unsigned)(row * ld + c * 8);
            }
        }
        if constexpr (HALF_LINES) {
            // k-row 8 q + (lane / 4) % 4 of a k-step, eight bytes of the tile's sixteen i
            const int j = lane & 15, q = lane >> 4;
#pragma unroll
            for (int t = 0; t < 2; t++) half[t] = (8 * q + (j >> 2)) * 64 + (t ^ (q & 1)) * 32 + (j & 3) * 8;
        } else {
            whole.init(0, lane);
        }
    }
    template <int I, int DST>
    __device__ inline void issue(const half_t *base, unsigned lds_addr) const
    {
        lds_dma16_at<DST + I * 1024, 0>(base, off[I], lds_addr);
    }
    // Fragment of MFMA tile T, k-step H.
    template <int T, int H>
    __device__ inline half8_t read(MIW_LDS const char *slot) const
    {
        if constexpr (HALF_LINES) {
            const int at = half[T] + H * 2048;
            fp16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4f16((MIW_LDS fp16x4_t *)(slot + at));
            fp16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4f16((MIW_LDS fp16x4_t *)(slot + at + 256));
            uint2_t l2 = __builtin_bit_cast(uint2_t, lo), h2 = __builtin_bit_cast(uint2_t, hi);
            uint4_t v = {l2[0], l2[1], h2[0], h2[1]};
            return __builtin_bit_cast(half8_t, v);
        } else {
            return whole.template read<T, H>(slot);
        }
    }
};

// One workgroup per tile of D, one tile per CU.  With so little work the time is the launch (2.8 us) and how fast one CU
// takes in its two panels of K: about 96 bytes per ns, from the last-level cache, with enough requests in flight.
//   - So the tile is the smallest that one round holds: the bytes of a CU go with BI + BJ.
//   - The four wavefronts split K, not the tile: wavefront w takes slots w, w + 4, ... of 64 k-values into a ring of its
//     own, and the 160 KiB of LDS are all in flight (64x64 tiles with a ring for the workgroup have 64).  No barrier in the
//     K loop: a wavefront waits only for its own loads, by count.  Every wavefront reads all fragments of its slots,
//     2 (BI + BJ) / 16 of them for BI BJ / 128 MFMAs, twice what four quarters of the tile would: LDS has the time.
//     Eight wavefronts with half the ring each: the same time.
//   - The partial sums meet in LDS after the loop and are added in wavefront order.
// With Float16 D and no C: 256x256x2048 9.9 us -> 6.3, 128x4096x4096 15.3 -> 12.3, 48x4096x4096 17.4 -> 9.9, against
// the 64x64 tile and k_gemm_skinny.
template <int BI, int BJ, bool XK, bool YK, class CT, class DT, bool SHORT>
__device__ __attribute__((always_inline)) inline void gemm_kwave(const tiled_params &p)
{
    constexpr bool HAS_C = !__is_same(CT, no_c_t);
    using shape = kwave_shape<BI, BJ>;
    constexpr int TI = BI / 16, TJ = BJ / 16, NS = shape::SLOTS, XBYTES = BI * KGRAN * 2;
    using xoperand = wave_operand<BI, XK>;
    using yoperand = wave_operand<BJ, YK>;
    constexpr int LOADS = xoperand::NLOAD + yoperand::NLOAD;

    extern __shared__ __attribute__((aligned(128))) char smem[];
    MIW_LDS char *lds = (MIW_LDS char *)smem;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    fetch_arguments(p);
    const tile_place at = workgroup_tile(p, BI, BJ);
    const int i0 = at.i0, j0 = at.j0;
    const long bt = at.bt;

    // This thread's share of D: four consecutive i of column j0 + tid / (BI / 4), then of every (1024 / BI)-th.
    // Its C is on the way while the K loop runs.
    constexpr int UNITS = BI * BJ / 4 <= 64 * KWAVES ? 1 : BI * BJ / 4 / (64 * KWAVES), STEP = 64 * KWAVES / (BI / 4);
    const bool takes = BI * BJ / 4 >= 64 * KWAVES || tid < BI * BJ / 4;
    const long oi = i0 + 4 * (tid % (BI / 4)), oj = j0 + tid / (BI / 4);
    using c4_t = CT __attribute__((ext_vector_type(4)));
    using d4_t = DT __attribute__((ext_vector_type(4)));
    c4_t cv[UNITS];
    if (HAS_C && takes && !p.c_trans) {
        const CT *at = (const CT *)p.C + bt * p.sc + oj * p.ldc + oi;
#pragma unroll
        for (int u = 0; u < UNITS; u++) cv[u] = *(const c4_t *)(at + (long)u * STEP * p.ldc);
    }

    const int K = SHORT ? member_k(p, at.bt) : p.K;
    const half_t *X = p.X + bt * p.sx + (XK ? (long)i0 * p.ldx : (long)i0);
    const half_t *Y = p.Y + bt * p.sy + (YK ? (long)j0 * p.ldy : (long)j0);
    const long xk = XK ? 1 : p.ldx, yk = YK ? 1 : p.ldy;  // elements from one k to the next
    xoperand xl;
    yoperand yl;
    xl.init(lane, (int)p.ldx);
    yl.init(lane, (int)p.ldy);

    // Slots wave, wave + 4, ... of 64 k-values; the k-values that 64 leaves are the last slot, shifted back to
    // end at K, of the wavefront whose turn it is.
    const int whole = K / KGRAN, tail_skip = whole * KGRAN == K ? 0 : (whole + 1) * KGRAN - K;
    const int own = (whole - wave + KWAVES - 1) / KWAVES;
    const bool has_tail = tail_skip && wave == whole % KWAVES;
    const int total = own + (has_tail ? 1 : 0);
    const unsigned ring = (unsigned)(uintptr_t)lds + (unsigned)(wave * NS * shape::SLOT);
    const half_t *xn, *yn;  // the slot being requested
    unsigned dst;
    auto begin_request = [&](int n, int slot) MIW_INLINE {
        const long k = n < own ? (long)(wave + KWAVES * n) * KGRAN : (long)K - KGRAN;
        xn = X + k * xk;
        yn = Y + k * yk;
        dst = ring + (unsigned)(slot * shape::SLOT);
    };
    auto request_one = [&]<int I>(std::integral_constant<int, I>) MIW_INLINE {
        if constexpr (I < xoperand::NLOAD) xl.template issue<I, 0>(xn, dst);
        else yl.template issue<I - xoperand::NLOAD, XBYTES>(yn, dst);
    };
    auto each = [&]<int... U>(std::integer_sequence<int, U...>, auto f) MIW_INLINE { (f(std::integral_constant<int, U>{}), ...); };
    float4_t acc[TI][TJ];
#pragma unroll
    for (int a = 0; a < TI; a++)
#pragma unroll
        for (int b = 0; b < TJ; b++) acc[a][b] = float4_t{0.f, 0.f, 0.f, 0.f};

    constexpr int NFRAG = 2 * (TI + TJ), NM = 2 * TI * TJ;
    struct fragments { half8_t x[2][TI], y[2][TJ]; };
    fragments f0, f1;
    // Fragment U of a slot in the order in which the MFMAs need them: both operands' first k-step, then the second.
    auto fetch = [&]<int U>(fragments &f, MIW_LDS const char *xs, std::integral_constant<int, U>) MIW_INLINE {
        constexpr int h = U / (TI + TJ), v = U % (TI + TJ);
        if constexpr (v < TJ) f.y[h][v] = yl.template read<v, h>(xs + XBYTES);
        else f.x[h][v - TJ] = xl.template read<v - TJ, h>(xs);
    };
    auto wait_vm = [&]<int N>(std::integral_constant<int, N>) MIW_INLINE { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); };
    // Lets the youngest n slots stay in flight (n < NS).
    auto wait_slots = [&](int n) MIW_INLINE {
        bool done = false;
        each(std::make_integer_sequence<int, NS>{}, [&](auto u) MIW_INLINE {
            constexpr int m = NS - 1 - decltype(u)::value;
            if (!done && n >= m) {
                wait_vm(std::integral_constant<int, m * LOADS>{});
                done = true;
            }
        });
        if (!done) wait_vm(std::integral_constant<int, 0>{});
    };
    auto slot_at = [&](int slot) MIW_INLINE { return (MIW_LDS const char *)(lds + (wave * NS + slot) * shape::SLOT); };
    auto mfma = [&](const fragments &f, int m) MIW_INLINE {
        const int h = m / (TI * TJ), a = m / TJ % TI, b = serpentine_column(m % (TI * TJ), TJ);
        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(f.x[h][a], f.y[h][b], acc[a][b], 0, 0, 0);
    };
    int slot = 0, n = 0;
    // The MFMAs of slot n out of `cur`; between them, first the requests of slot n + NS into the place of slot n
    // (whose fragments have all been read), then the fragments of slot n + 1 into `nxt` (behind the last slot, of
    // whatever is there: nobody uses them).
    auto pass = [&](const fragments &cur, fragments &nxt) MIW_INLINE {
        constexpr int PER_DMA = (LOADS + NM / 2 - 1) / (NM / 2);                // loads behind one MFMA
        constexpr int WAIT = NM / 4;                                            // MFMA ahead of the first read
        constexpr int AHEAD = WAIT * PER_DMA < LOADS ? WAIT * PER_DMA : LOADS;  // loads issued before it
        constexpr int PER_READ = (NFRAG + NM - WAIT - 1) / (NM - WAIT);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(15 | (7 << 4) | (0 << 8) | (3 << 14));  // lgkmcnt(0): slot n has been read
        asm volatile("" ::: "memory");
        const bool ask = n + NS < total;
        begin_request(n + NS, slot);
        slot = slot + 1 == NS ? 0 : slot + 1;
        MIW_LDS const char *xs = slot_at(slot);
        each(std::make_integer_sequence<int, NM>{}, [&](auto mc) MIW_INLINE {
            constexpr int m = decltype(mc)::value;
            if constexpr (m == WAIT) {
                // slot n + 1 has landed; behind it slots n + 2 .. and what this pass has requested
                if (ask) wait_vm(std::integral_constant<int, (NS - 2) * LOADS + AHEAD>{});
                else wait_slots(total - 2 - n);
            }
            mfma(cur, m);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (m * PER_DMA < LOADS) {
                if (ask)
                    each(std::make_integer_sequence<int, PER_DMA>{}, [&](auto u) MIW_INLINE {
                        constexpr int i = m * PER_DMA + decltype(u)::value;
                        if constexpr (i < LOADS) request_one(std::integral_constant<int, i>{});
                    });
            }
            if constexpr (m >= WAIT)
                each(std::make_integer_sequence<int, PER_READ>{}, [&](auto u) MIW_INLINE {
                    constexpr int i = (m - WAIT) * PER_READ + decltype(u)::value;
                    if constexpr (i < NFRAG) fetch(nxt, xs, std::integral_constant<int, i>{});
                });
            __builtin_amdgcn_sched_barrier(0);
        });
        n++;
    };
#pragma unroll
    for (int u = 0; u < NS; u++)
        if (u < total) {
            begin_request(u, u);
            each(std::make_integer_sequence<int, LOADS>{}, request_one);
        }
    if (own > 0) {
        wait_slots(min(total, NS) - 1);
        each(std::make_integer_sequence<int, NFRAG>{}, [&](auto u) MIW_INLINE { fetch(f0, slot_at(0), u); });
        for (;;) {
            pass(f0, f1);
            if (n >= own) break;
            pass(f1, f0);
            if (n >= own) break;
        }
    }
    if (has_tail) {
        wait_vm(std::integral_constant<int, 0>{});
        each(std::make_integer_sequence<int, NFRAG>{}, [&](auto u) MIW_INLINE { fetch(f0, slot_at(slot), u); });
        const unsigned keep[2] = {tail_keep<0>(tail_skip), tail_keep<1>(tail_skip)};
#pragma unroll
        for (int h = 0; h < 2; h++) {
#pragma unroll
            for (int a = 0; a < TI; a++) tail_apply(f0.x[h][a], keep[h]);
#pragma unroll
            for (int b = 0; b < TJ; b++) tail_apply(f0.y[h][b], keep[h]);
        }
#pragma unroll
        for (int m = 0; m < NM; m++) mfma(f0, m);
    }

    // The wavefronts' sums, added in wavefront order: no dependence on timing.
    __syncthreads();  // (every wavefront has waited for its loads and read its last slot)
    MIW_LDS float *part = (MIW_LDS float *)lds;
    {
        const int q = lane >> 4, r = lane & 15;
        MIW_LDS float *mine = part + wave * shape::PITCH * BJ + r * shape::PITCH + 4 * q;
#pragma unroll
        for (int b = 0; b < TJ; b++)
#pragma unroll
            for (int a = 0; a < TI; a++) *(MIW_LDS float4_t *)(mine + 16 * b * shape::PITCH + 16 * a) = acc[a][b];
    }
    __syncthreads();
    if (!takes) return;
#pragma unroll
    for (int u = 0; u < UNITS; u++) {
        MIW_LDS const float *src = part + (tid / (BI / 4) + u * STEP) * shape::PITCH + 4 * (tid % (BI / 4));
        float4_t v = *(MIW_LDS const float4_t *)src;
#pragma unroll
        for (int w = 1; w < KWAVES; w++) {
            const float4_t y = *(MIW_LDS const float4_t *)(src + w * shape::PITCH * BJ);
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] += y[e];
        }
        const long j = oj + (long)u * STEP;
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] *= p.alpha;
        if constexpr (HAS_C) {
            float4_t c;
            if (p.c_trans) {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    c[e] = (float)((const CT *)p.C)[bt * p.sc + (oi + e) * p.ldc + j];
                }
            } else {
                c = __builtin_convertvector(cv[u], float4_t);
            }
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] = __builtin_fmaf(p.beta, c[e], v[e]);
        }
        const long at = bt * p.sd + j * p.ldd + oi;
        *(d4_t *)((DT *)p.D + at) = __builtin_convertvector(v, d4_t);
    }
}

// A launch pays for the instructions it passes by, which it fetches from a cold cache: so the types, and whether there is a C,
// are the instance's.  With both asked for at run time decode 16x4096x4096 takes 8.17 us, 8.02 like this, 128x4096x4096
// 11.5 and 11.1, 640x576x1840 8.3 and 8.0, 720x656x784 with a Float32 C 6.24 and 5.99.
// Float32 C and D.
template <int BI, int BJ, bool XK, bool YK>
__global__ __launch_bounds__(64 * KWAVES) __attribute__((amdgpu_waves_per_eu(2)))
void k_gemm_kwave(tiled_params p)
{
    gemm_kwave<BI, BJ, XK, YK, float, float, false>(p);
}

// Other types of C and D, or no C.
template <int BI, int BJ, bool XK, bool YK, class CT, class DT>
__global__ __launch_bounds__(64 * KWAVES) __attribute__((amdgpu_waves_per_eu(2)))
void k_gemm_kwave_types(tiled_params p)
{
    gemm_kwave<BI, BJ, XK, YK, CT, DT, false>(p);
}

// Slices of K of which the last one is shorter.  (The question alone, in front of the first request, makes a launch of 8.14 us 8.19.)
template <int BI, int BJ, bool XK, bool YK>
__global__ __launch_bounds__(64 * KWAVES) __attribute__((amdgpu_waves_per_eu(2)))
void k_gemm_kwave_slices(tiled_params p)
{
    gemm_kwave<BI, BJ, XK, YK, no_c_t, float, true>(p);
}

template <int BI, int BJ, bool XK, bool YK>
static const void *kwave_types(int c_type, int d_type, bool slices)
{
    if (slices) return (const void *)k_gemm_kwave_slices<BI, BJ, XK, YK>;
    if (c_type == NO_C && d_type == 0) return (const void *)k_gemm_kwave_types<BI, BJ, XK, YK, no_c_t, half_t>;
    if (c_type == NO_C) return (const void *)k_gemm_kwave_types<BI, BJ, XK, YK, no_c_t, float>;
    if (c_type == 0 && d_type == 0) return (const void *)k_gemm_kwave_types<BI, BJ, XK, YK, half_t, half_t>;
    if (c_type == 0) return (const void *)k_gemm_kwave_types<BI, BJ, XK, YK, half_t, float>;
    if (d_type == 0) return (const void *)k_gemm_kwave_types<BI, BJ, XK, YK, float, half_t>;
    return (const void *)k_gemm_kwave<BI, BJ, XK, YK>;
}

// Kernel for a tile, operand layouts and types (c_type NO_C: no C), or null when there is none; slices: of K, the last one
// shorter (no C, Float32).
const void *kwave_kernel(int bi, int bj, bool xk, bool yk, int c_type, int d_type, bool slices, int *lds_bytes)
{
    auto is = [&](int i, int j, bool x, bool y) { return bi == i && bj == j && xk == x && yk == y; };
#define MIW_KWAVE(I, J, X, Y)                                        \
    if (is(I, J, X, Y)) {                                            \
        *lds_bytes = kwave_shape<I, J>::RING;                        \
        return kwave_types<I, J, X, Y>(c_type, d_type, slices);      \
    }
    MIW_KWAVE(64, 32, true, true)
    MIW_KWAVE(64, 32, false, true)
    MIW_KWAVE(64, 32, false, false)
    MIW_KWAVE(32, 64, true, false)
    MIW_KWAVE(32, 32, true, true)
    MIW_KWAVE(32, 32, false, true)
    MIW_KWAVE(32, 32, true, false)
    MIW_KWAVE(32, 32, false, false)
    MIW_KWAVE(32, 16, true, true)
    MIW_KWAVE(16, 32, true, true)
#undef MIW_KWAVE
    return nullptr;
}

static bool multiple16(const void *x) { return ((uintptr_t)x & 15) == 0; }

constexpr kwave_tile kwave_tiles[] = {{32, 16}, {16, 32}, {32, 32}, {64, 32}, {32, 64}};

// Operands' layouts in canonical form.
static void layouts(const gemm_params &g, bool *xk, bool *yk)
{
    *xk = g.d_row ? g.b_row == 0 : g.a_row != 0;
    *yk = g.d_row ? g.a_row != 0 : g.b_row == 0;
}

// What the 16-byte loads and the 8- and 16-byte stores assume, and 32-bit offsets inside a slot.
static bool kwave_runs(const gemm_params &g, int c_type, int d_type)
{
    const long cper = c_type == 0 ? 8 : 4, dper = d_type == 0 ? 8 : 4;
    if (g.K < 2 * KGRAN || g.K > (1l << 30) || g.M > (1l << 30) || g.N > (1l << 30)) return false;
    if (!multiple16(g.A) || !multiple16(g.B) || !multiple16(g.D) || g.lda % 8 || g.ldb % 8 || g.sa % 8 || g.sb % 8) return false;
    if (g.ldd % dper || g.sd % dper || (g.use_c && (!multiple16(g.C) || g.ldc % cper || g.sc % cper))) return false;
    return g.lda * 256 < (1l << 31) && g.ldb * 256 < (1l << 31);
}

// Workgroups on a tile, 0 where the kernel does not run the problem on it.
static long kwave_groups(const gemm_params &g, kwave_tile t, bool in_place)
{
    const long I = g.d_row ? g.N : g.M, J = g.d_row ? g.M : g.N;
    bool xk, yk;
    layouts(g, &xk, &yk);
    int lds;
    if (I < t.bi || J < t.bj || !kwave_kernel(t.bi, t.bj, xk, yk, 1, 1, false, &lds)) return 0;
    if (in_place && (I % t.bi || J % t.bj)) return 0;  // (edge tiles overlap their neighbours)
    return (I + t.bi - 1) / t.bi * ((J + t.bj - 1) / t.bj) * g.batch;
}

kwave_tile kwave_fits(const gemm_params &g, int c_type, int d_type, bool in_place, int cus)
{
    kwave_tile best = {0, 0};
    if (!kwave_runs(g, c_type, d_type)) return best;
    for (const kwave_tile t : kwave_tiles) {
        const long groups = kwave_groups(g, t, in_place);
        if (groups == 0 || groups / g.batch * 64 * KWAVES >= (1l << 32)) continue;
        best = t;
        if (groups <= cus) break;
    }
    return best;
}

// The smallest of the kernel's tiles that covers D in one round over the CUs: the fewer bytes a CU has to fetch the
// shorter the launch, and a second round costs more than any tile saves (1.3 to 1.7 times the time of the 64x64 tile).
// Measured against the kernels that run them otherwise, on operands from the last-level cache and from HBM:
//   32x16, 16x32, 32x32: 0.41 to 1.02 of the 64x64 tile's time from K = 128 on (256x256x2048 9.9 -> 6.3 us).
//   64x32, 32x64 with a C operand, whose reading the K loop here hides: 0.74 to 1.0 from K = 512 on with k contiguous in
//     both operands, 0.8 to 1.0 from 768 on otherwise.  Without C: 0.7 to 1.07 from K = 1024 on (128x4096x4096 15.3 ->
//     12.3 us), below that 1.0 to 1.1 (720x656x832 6.5, 5.8 on the tile), but where whatever has k contiguous starts its
//     rows off whole cache lines, which slows the tiles' loads: 0.92 to 1.06 from 512 (both operands) or 768 on.  Slices of
//     K go by the lines for a C.
//   Less than 64 rows or columns, against k_gemm_skinny and the fragment-op kernels: with k contiguous in both operands,
//     and rows on whole cache lines, which these loads need and those do not (16x4096x2064: 1.2 to 1.4), 0.34 to 0.96 where
//     those take a second round, and from K = 1024 (16 rows) or 512 on where they take one (48x4096x4096 17.4 -> 9.9;
//     16x4096 0.77 to 1.03 from the cache, 1.05 to 1.13 from HBM).  In other layouts 0.4 to 1.0 with 1024 or more of the
//     long extent, K from 1024 on, or 512 with 2048; shorter ones with k contiguous in one operand, the long one's up to
//     1024, the other up to 512: 1.0 to 1.2 below K = 3072, 0.6 to 1.02 from there (48x64x1280 5.7, 4.9 on fragment ops).
//   64 to 128 rows off whole cache lines, where k_gemm_skinny beats the 64x64 tile: up to 32x32 0.76 to 0.95 of its time
//     from K = 768 on.
kwave_tile kwave_pays(const gemm_params &g, int c_type, int d_type, bool in_place, int cus)
{
    constexpr kwave_tile none = {0, 0};
    if (!kwave_runs(g, c_type, d_type)) return none;
    bool xk, yk;
    layouts(g, &xk, &yk);
    const bool both = xk && yk, a_k = g.a_row != 0, b_k = g.b_row == 0;
    const long wide = std::max(g.M, g.N), thin = std::min(g.M, g.N);
    const bool narrow_wins = skinny_beats_tiles(g, d_type, false);
    if (thin < 64) {
        if (both && (g.lda % 64 || g.ldb % 64)) return none;
        const bool rounds = wide / 16 * g.batch > cus, wide_k = g.M >= g.N ? a_k : b_k;
        const long least = both ? (rounds ? 0 : thin == 16 ? 1024 : 512)
                           : wide >= 2048 ? 512
                           : (a_k || b_k) && wide < (wide_k ? 1024 : 512) ? 3072
                                                                          : 1024;
        if (g.K < least) return none;
    } else if (narrow_wins && g.K < 768) {
        return none;
    }
    // rows of whatever has k contiguous start off whole cache lines
    const bool off_lines = (a_k || b_k) && (!a_k || g.lda % 64) && (!b_k || g.ldb % 64);
    const long least_64 = !g.use_c && g.batch == 1 && !off_lines ? 1024 : both ? 512 : 768;
    for (const kwave_tile t : kwave_tiles) {
        const long groups = kwave_groups(g, t, in_place);
        if (groups == 0 || groups > cus) continue;
        if (t.bi * t.bj > 32 * 32 && (g.K < least_64 || (thin >= 64 && narrow_wins))) continue;
        return t;
    }
    return none;
}

// Estimated duration in microseconds, for the planner: what a CU fetches, at the pace of one workgroup's requests (within
// 20 % on nine of ten of the same problems).
double kwave_estimate_us(const gemm_params &g, int c_type, int d_type, kwave_tile t)
{
    const bool both = g.a_row != 0 && g.b_row == 0;
    const double mn = (double)g.M * (double)g.N * (double)g.batch;
    const double cd_bytes = mn * ((d_type == 0 ? 2 : 4) + (g.use_c ? (c_type == 0 ? 2 : 4) : 0));
    return 3.5 + cd_bytes / 5.5e6 + 2.0 * (double)(t.bi + t.bj) * (double)g.K / (both ? 90e3 : 70e3);
}

}  // namespace miw
