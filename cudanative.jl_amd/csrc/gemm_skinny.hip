// GEMM with at most 128 rows (or columns) on one side and k contiguous in both operands: one decoding
// step, or a short prefill, of a projection.
#include "gemm_tiled.hpp"

namespace miw {

struct skinny_params {
    const half_t *W, *S;  // wide operand (one row per entry of D's long dimension) and narrow one, k contiguous in both
    const void *C;
    void *D;
    int wide, K;
    long ldw, lds, sw, ss, sc, sd;  // row pitches and batch strides in elements
    long cw, cn, dw, dn;            // element strides of C and D along the long and the short dimension
    int use_c, c_f32, d_f32;
    float alpha, beta;
};

constexpr int SKINNY_WAVES = 8;

// What bounds this is the one read of the wide operand from HBM, so nothing goes through LDS on the
// way in: a lane loads its fragments of v_mfma_f32_16x16x32_f16 (16 contiguous bytes of one row) straight
// into registers, two buffers of UN chunks each, and the next buffer is requested before the
// MFMAs of this one.  A workgroup owns 16 * WT entries of the long dimension and all 16 * MT of the short
// one; its eight wavefronts take the 64-k chunks (128 bytes of a row) in turn, so that together they
// walk each row in 1 KiB pieces, and add their partial sums in wavefront order through LDS: no second
// kernel, no workspace, no dependence on timing.  The narrow operand is read again by every workgroup,
// from the caches; WT = 2 halves those reads.
// Below K of about 2048 a wavefront has fewer chunks than a buffer, and what bounds it is the requests
// that go through the CU's L1: each chunk is asked for once (16 x 4096 x 512: 3.5 us; 5.5 us when a buffer
// that K does not fill asks for its last chunk again; 32 x 4096 x 2048: 8.8 and 11.2).  From there on the
// wide operand's bytes count: 16 x 4096 x 8192 in 19.3 us is 3.5 TB/s.
template <int MT, int WT>
__global__ __launch_bounds__(64 * SKINNY_WAVES) void k_gemm_skinny(skinny_params p)
{
    constexpr int UN = MT + WT <= 2 ? 4 : MT + WT == 3 ? 3 : MT + WT <= 5 ? 2 : 1;  // two buffers stay below 256 VGPRs
    __shared__ float4_t part[SKINNY_WAVES][MT][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int r = lane & 15, q = lane >> 4;
    const long w0 = (long)blockIdx.x * (16 * WT), bt = blockIdx.y;
    const half_t *W = p.W + bt * p.sw + (w0 + r) * p.ldw + 8 * q;
    const half_t *S = p.S + bt * p.ss + (long)r * p.lds + 8 * q;
    const int chunks = p.K / 64, tail = p.K % 64;
    const int own = (chunks - wave + SKINNY_WAVES - 1) / SKINNY_WAVES;  // chunks wave, wave + 8, ... (K >= 64: none below zero)
    const int full = own / UN, rem = own % UN;

    float4_t acc[WT][MT];
#pragma unroll
    for (int t = 0; t < WT; t++)
#pragma unroll
        for (int m = 0; m < MT; m++) acc[t][m] = float4_t{0.f, 0.f, 0.f, 0.f};

    half8_t w[2][UN][WT][2], s[2][UN][MT][2];
    const half_t *w_next = W + 64l * wave, *s_next = S + 64l * wave;
    auto load = [&](auto buf, auto at) {
        constexpr int b = decltype(buf)::value, u = decltype(at)::value, k0 = 64 * SKINNY_WAVES * u;
#pragma unroll
        for (int h = 0; h < 2; h++) {
#pragma unroll
            for (int t = 0; t < WT; t++) w[b][u][t][h] = *(const half8_t *)(w_next + 16l * t * p.ldw + k0 + 32 * h);
#pragma unroll
            for (int m = 0; m < MT; m++) s[b][u][m][h] = *(const half8_t *)(s_next + 16l * m * p.lds + k0 + 32 * h);
        }
    };
    auto multiply = [&](auto buf, auto at) {
        constexpr int b = decltype(buf)::value, u = decltype(at)::value;
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int t = 0; t < WT; t++)
#pragma unroll
                for (int m = 0; m < MT; m++)
                    acc[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[b][u][t][h], s[b][u][m][h], acc[t][m], 0, 0, 0);
    };
    auto each = [&]<int... U>(std::integer_sequence<int, U...>, auto f) { (f(std::integral_constant<int, U>{}), ...); };
    constexpr std::make_integer_sequence<int, UN> all{};
    constexpr std::integral_constant<int, 0> b0{};
    constexpr std::integral_constant<int, 1> b1{};
    auto request = [&](auto buf) {
        each(all, [&](auto u) { load(buf, u); });
        w_next += 64l * SKINNY_WAVES * UN;
        s_next += 64l * SKINNY_WAVES * UN;
        __builtin_amdgcn_sched_barrier(0);  // the requests go out before the MFMAs of the other buffer
    };
    auto compute = [&](auto buf) { each(all, [&](auto u) { multiply(buf, u); }); };
    // The chunks that UN does not divide go first, through the second buffer and together with the first
    // whole one: no chunk is asked for twice, and the loop has no condition inside its steps.
    each(all, [&](auto u) { if (u < rem) load(b1, u); });
    w_next += 64l * SKINNY_WAVES * rem;
    s_next += 64l * SKINNY_WAVES * rem;
    if (full > 0) request(b0);
    each(all, [&](auto u) { if (u < rem) multiply(b1, u); });
    for (int i = 0; i < full; i += 2) {
        if (i + 1 < full) request(b1);
        compute(b0);
        if (i + 1 >= full) break;
        if (i + 2 < full) request(b0);
        compute(b1);
    }
    // The 16, 32 or 48 k-values that 64 leaves, by the wavefront whose turn it is; what lies past K is zero in both operands.
    if (tail && wave == chunks % SKINNY_WAVES) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const bool in = 32 * h + 8 * q < tail;
            half8_t a[WT], b[MT];
#pragma unroll
            for (int t = 0; t < WT; t++) {
                a[t] = half8_t{};
                if (in) a[t] = *(const half8_t *)(W + 16l * t * p.ldw + 64l * chunks + 32 * h);
            }
#pragma unroll
            for (int m = 0; m < MT; m++) {
                b[m] = half8_t{};
                if (in) b[m] = *(const half8_t *)(S + 16l * m * p.lds + 64l * chunks + 32 * h);
            }
#pragma unroll
            for (int t = 0; t < WT; t++)
#pragma unroll
                for (int m = 0; m < MT; m++) acc[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[t], b[m], acc[t][m], 0, 0, 0);
        }
    }
    // Lane (q, r) of a tile holds entries 4q .. 4q + 3 of the long dimension, entry r of the short one.
    for (int t = 0; t < WT; t++) {
        if (t) __syncthreads();
#pragma unroll
        for (int m = 0; m < MT; m++) part[wave][m][lane] = WT == 1 || t == 0 ? acc[0][m] : acc[WT - 1][m];
        __syncthreads();
        if (wave >= MT) continue;  // (MT <= 8: one tile per wavefront)
        float4_t v = part[0][wave][lane];
#pragma unroll
        for (int x = 1; x < SKINNY_WAVES; x++) {
            const float4_t y = part[x][wave][lane];
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] += y[e];
        }
        const long i = w0 + 16 * t + 4 * q, j = 16 * wave + r;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            v[e] *= p.alpha;
            if (p.use_c) {
                const long at = bt * p.sc + (i + e) * p.cw + j * p.cn;
                v[e] = __builtin_fmaf(p.beta, p.c_f32 ? ((const float *)p.C)[at] : (float)((const half_t *)p.C)[at], v[e]);
            }
        }
        const long at = bt * p.sd + i * p.dw + j * p.dn;
        if (p.d_f32) {
            float *d = (float *)p.D + at;
            if (p.dw == 1) *(float4_t *)d = v;
            else for (int e = 0; e < 4; e++) d[e * p.dw] = v[e];
        } else {
            half_t *d = (half_t *)p.D + at;
            if (p.dw == 1) *(half4_t *)d = half4_t{(half_t)v[0], (half_t)v[1], (half_t)v[2], (half_t)v[3]};
            else for (int e = 0; e < 4; e++) d[e * p.dw] = (half_t)v[e];
        }
    }
}

constexpr long SKINNY_CUS = 256;  // (one workgroup per CU: the registers of eight wavefronts)

// Tiles of 16 of the long dimension that a workgroup takes: two, with 64 or more of the short one, where
// one tile each would need a second round over the CUs.  The wavefronts' requests through the L1 are what
// takes the time then, and two tiles share the narrow operand's (128 x 8192 x 2048: 23 us, 39 with one
// tile); within one round it is the other way round (128 x 4096 x 2048: 22 and 20).
static int skinny_width(const gemm_params &g)
{
    const long wide = g.M <= g.N ? g.N : g.M, narrow = g.M <= g.N ? g.M : g.N;
    return wide % 32 == 0 && narrow >= 64 && wide / 16 * g.batch > SKINNY_CUS ? 2 : 1;
}

// Can k_gemm_skinny run this problem?  One extent of at most 128, k contiguous in both operands, at
// least one chunk of K, what its 16-byte loads and 8- or 16-byte stores assume of the alignment, and fewer than 2^32
// threads along x (the long extent of a problem that is thin enough to fit in memory can exceed that).
bool skinny_fits(const gemm_params &g, int d_type, bool f16acc)
{
    const long wide = g.M <= g.N ? g.N : g.M, narrow = g.M <= g.N ? g.M : g.N;
    if (f16acc || narrow > 128 || g.K < 64 || !g.a_row || g.b_row || g.K > (1l << 30) || wide > (1l << 30)) return false;
    if (((uintptr_t)g.A & 15) || ((uintptr_t)g.B & 15) || g.lda % 8 || g.ldb % 8 || g.sa % 8 || g.sb % 8) return false;
    if (wide / (16 * skinny_width(g)) * (64 * SKINNY_WAVES) >= 1l << 32) return false;
    const long dper = d_type == 0 ? 8 : 4;
    return !((uintptr_t)g.D & 15) && g.ldd % dper == 0 && g.sd % dper == 0;
}

// Rounds of workgroups over `cus` CUs.
static long skinny_rounds(const gemm_params &g, long cus)
{
    const long wide = g.M <= g.N ? g.N : g.M;
    return (wide / (16 * skinny_width(g)) * g.batch + cus - 1) / cus;
}

// Does k_gemm_skinny run this problem faster than the fragment-op kernels (k_gemm_fragops on one wavefront per
// tile, or k_gemm_fragops_ksplit on 4 to 16)?  Measured over 16 to 128 x 64 to 131072 x 80 to 8192 and batches up
// to 256: where the rule says yes the time is 0.16 to 1.06 of the other kernel's (median 0.77), and where it says
// no it would be 0.86 or more.
//   K < 256: the others give a tile to one wavefront, and its chain of steps takes longer than a round of
//     workgroups here (16 x 4096 x 128: 2.8 us against 4.7).  With more than two rounds the six of eight
//     wavefronts that have no chunk cost more than the chain (16 x 32768 x 128: 10.7 against 7.5), unless
//     three tiles or more share the wide operand.
//   K >= 256, one wavefront per tile there (more than 2048 workgroups): only 16 rows with a short K are faster there
//     (16 x 65536 x 256: 1.2 times; at K = 512 this kernel takes 0.89, at 1024 0.72).
//   K >= 256, K split there: the tile reads per CU, the bound of both, decide.  Without tiles of the short
//     dimension in one workgroup the other kernel spreads few tiles over more CUs (48 x 512 x 4096: 16.6 against
//     10.0).  Within one round of workgroups this kernel is ahead (16 x 4096 x 512: 3.5 against 3.9; 32 x 4096 x
//     4096: 14.3 against 17.1); each further round shows its start and its reduction, which a K per round of 1024,
//     384 or 256 for one, two or three tiles of the short dimension makes up for (16 x 16384: 0.97 at K = 4096,
//     1.03 at 2048; 32 x 16384: 0.93 at 1536, 1.0 at 1024; 48 x 16384: 0.98 at 1024).
bool skinny_pays(const gemm_params &g, int d_type, bool f16acc)
{
    if (!skinny_fits(g, d_type, f16acc)) return false;
    const long wide = g.M <= g.N ? g.N : g.M, mt = (g.M <= g.N ? g.M : g.N) / 16;
    const long rounds = skinny_rounds(g, SKINNY_CUS);
    if (g.K < 256) return rounds <= 2 || (mt >= 3 && g.K >= 128);
    int together;
    if (fragops_ksplit(g, f16acc, &together) == 1) return mt >= 2 || g.K >= 512;
    if (together == 1 && rounds * (mt + skinny_width(g)) > 2 * ((mt * (wide / 16) * g.batch + SKINNY_CUS - 1) / SKINNY_CUS)) return false;
    return rounds == 1 || mt >= 4 || g.K >= (mt == 1 ? 1024 : mt == 2 ? 384 : 256) * rounds;
}

// Does k_gemm_skinny run this problem faster than the LDS tile it would get?  Where the rows of both operands start on
// whole cache lines, never (64 to 128 x 256 to 16384 x 256 to 4096: 0.99 to 2.3 times the tile's time; a tile of 64 x 64
// reads 64 rows of each operand once, a workgroup here 16 of one and all of the other).  Pitches that 64 elements, 128
// bytes, do not divide slow the tiles' direct-to-LDS loads down (64 x 4096: 17.7 us at K = 3072, 26.2 at 3088) and
// leave these alone (17.6 and 17.0); with one operand on whole lines the two are level.  The tile rows of 16 that a CU
// reads here then decide: up to 6, i.e. 64 and 80 in one round of workgroups, 0.60 to 1.04 of the tile's time; 7 and 8,
// i.e. 96 and 112, only where rows also straddle 64-byte halves and K makes up for the start (96 x 4096 x 528: 0.98; 112 x 4096 x 1040: 0.93; 112 x 2064: 1.02 at K = 1040, 0.91 at 3088).
// Rows that all start at the same place inside a line cost the tiles less: 0.7 to 0.95 at 64, 0.83 to 1.13 at 80.
bool skinny_beats_tiles(const gemm_params &g, int d_type, bool f16acc)
{
    const long wide = g.M <= g.N ? g.N : g.M, narrow = g.M <= g.N ? g.M : g.N;
    if (narrow < 64 || g.K < 256 || !skinny_fits(g, d_type, f16acc)) return false;
    // 0: rows start on cache lines, 1: at one place inside a line, 2: at several, 3: also inside 64-byte halves
    auto straddles = [](const half_t *x, long ld) { return ld % 32 ? 3 : ld % 64 ? 2 : (uintptr_t)x & 127 ? 1 : 0; };
    const int a = straddles(g.A, g.lda), b = straddles(g.B, g.ldb), worst = a < b ? a : b;
    const long rows = skinny_rounds(g, SKINNY_CUS) * (narrow / 16 + skinny_width(g));
    if (worst < 2) return worst == 1 && rows <= 5;
    if (rows <= 6) return true;
    if (worst != 3) return false;
    return rows == 7 ? g.K >= 512 : rows == 8 && g.K >= 1024 && wide * g.batch >= (g.K >= 3072 ? 1024 : 4096);
}

// Estimated duration in microseconds, for the planner: launch, start and reduction of each round of
// workgroups, and the larger of a CU's requests through its L1 (0.96 ns per tile row of 16 and k-value) and the
// operands at 3.7 TB/s.  Fitted to the launches of the same sweep that skinny_pays takes: within 20 % on nine of ten.
double skinny_estimate_us(const gemm_params &g, int cus)
{
    const long rounds = skinny_rounds(g, cus), narrow = g.M <= g.N ? g.M : g.N;
    const double l1 = 0.96e-3 * (double)rounds * (double)(narrow / 16 + skinny_width(g)) * (double)g.K;
    const double hbm = 2.0 * (double)(g.M + g.N) * (double)g.K * (double)g.batch / 3.7e6;
    return 3.0 + 1.1 * (double)rounds + (l1 > hbm ? l1 : hbm);
}

hipError_t launch_gemm_skinny(const gemm_params &g, int c_type, int d_type, hipStream_t s)
{
    skinny_params p;
    const bool nm = g.M <= g.N;  // the short dimension is M
    p.W = nm ? g.B : g.A; p.S = nm ? g.A : g.B;
    p.ldw = nm ? g.ldb : g.lda; p.lds = nm ? g.lda : g.ldb;
    p.sw = nm ? g.sb : g.sa; p.ss = nm ? g.sa : g.sb;
    p.wide = (int)(nm ? g.N : g.M); p.K = (int)g.K;
    const bool d_wide = (g.d_row != 0) == nm, c_wide = (g.c_row != 0) == nm;  // contiguous along the long dimension
    p.dw = d_wide ? 1 : g.ldd; p.dn = d_wide ? g.ldd : 1;
    p.cw = c_wide ? 1 : g.ldc; p.cn = c_wide ? g.ldc : 1;
    p.C = g.C; p.D = g.D; p.sc = g.sc; p.sd = g.sd;
    p.use_c = g.use_c; p.c_f32 = c_type; p.d_f32 = d_type;
    p.alpha = g.alpha; p.beta = g.beta;
    const int mt = (int)((nm ? g.M : g.N) / 16), wt = skinny_width(g);
    const dim3 grid((unsigned)(p.wide / (16 * wt)), (unsigned)g.batch), block(64 * SKINNY_WAVES);
    auto go = [&]<int MT>(std::integral_constant<int, MT>) {
        if (wt == 1) hipLaunchKernelGGL((k_gemm_skinny<MT, 1>), grid, block, 0, s, p);
        else if constexpr (MT >= 4) hipLaunchKernelGGL((k_gemm_skinny<MT, 2>), grid, block, 0, s, p);
    };
    switch (mt) {
    case 1: go(std::integral_constant<int, 1>{}); break;
    case 2: go(std::integral_constant<int, 2>{}); break;
    case 3: go(std::integral_constant<int, 3>{}); break;
    case 4: go(std::integral_constant<int, 4>{}); break;
    case 5: go(std::integral_constant<int, 5>{}); break;
    case 6: go(std::integral_constant<int, 6>{}); break;
    case 7: go(std::integral_constant<int, 7>{}); break;
    case 8: go(std::integral_constant<int, 8>{}); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace miw
