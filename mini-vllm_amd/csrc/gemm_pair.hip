// The gated pair for prompts, rows by the hundred and thousand (bfloat16 in and out, float sums, MFMA):
//     C[M, I] = pair(A Wg^T (+ bias), A Wu^T (+ bias)),  A [M, K],  W = [Wg | Wu] of [2 I, K]
// with the activation on the float sums, so that the two products never go to memory.
//
// A workgroup of eight waves makes a tile of 64 to 256 rows by 64 to 192 weight rows (half gate, half up) and has a compute unit to itself;
// operands come through an LDS ring as in gemm_tile.hip, their reads run under the products. What bounds it: a chunk of 64 columns takes
// 0.15 us (the barrier, and waves that wait for the last of them) and 0.385 us for every 128 x 128 of the tile, 1.39 PFLOP/s, half of it
// the matrix unit, the rest LDS and issue; and a workgroup takes 3.5 us to its first products and from its last. So tiles are large, and
// which of the twelve shapes depends on how many whole rounds of compute units they make (mv_gemm_pair_shape): 2,048 x 6144 x 1024
// is one of 256 x 192. There 36.4 us with the library's product and the activation behind it, 27.2 here; 1,536 rows 34.7 (gemm_tile.hip)
// and 21.8; 1,024 23.5 and 17.6; 512 17.2 and 12.9; 1,024 x 12288 x 2048 72 and 47; 4,096 x 6144 x 1024 66 and 52.8. Large products of a long K
// stay with the library (4,096 x 24576 x 4096: 593 us with the activation, 700 here).
//
// The same kernel without the activation is mv_gemm_round: plain products whose tiles are one round of the compute units, which the
// library is behind at where its own tiles leave units idle, above all for N that are no multiple of 256 (projections packed beside
// one another). us, the library / here: 224 x 3104 x 1024 12.0 / 8.0, 1,024 16.7 / 14.3, 2,048 23.0 / 21.0; 2,048 x 5184 x 1024 33.5 / 29.3, 552
// 15.4 / 13.9; 1,000 x 592 x 1024 9.1 / 6.4; 2,048 x 2080 x 512 15.5 / 10.3. A tile takes what its operands take
// through the compute unit, 192 KB of a 128 x 64 tile with K of 1,024 in 8 us; long K (2,048 x 1024 x 3072 22.8 / 23.5), N that fill the chip
// with the library's 256 x 128 (2,048 x 4096 x 1024 21.5 / 23.0) and more than one round (4,096 x 3104 x 1024 37.6 / 38.5) stay where they were, and
// so do some that the rule takes for slower than they are (1,424 x 1024 x 1024 10.7 / 8.3, 1,100 x 2048 x 2048 23.1 / 18.3).
#include "gemm_deep.h"
#include "gemm_ring.h"

#include <cmath>
#include <type_traits>

struct PairArgs {
    const bf16* A;
    long lda;
    const bf16* W;
    const bf16* bias;
    bf16* C;
    long ldc;
    int M, I, K;                       // plain: I = N
    int tiles, fast, by_columns, wide_stores;    // fast: tiles of the side that changes fastest
    GatedPair pair;
    // rows behind a folded norm: P partial sums of squares each; PAIR_FOLD writes them
    float* partial;
    int P;
    float eps;
    // PAIR_FOLD
    float* resid;
    long ldr;
    WeightPtr norm_weight;
    int unit_offset;
    bf16* weighted;
    long ldw;
};

// PAIR_FOLD: the product in front of a residual add and a norm; _SCALED: behind one (see gemm_deep.hip for both)
enum PairForm { PAIR_PLAIN = 0, PAIR_GATED = 1, PAIR_FOLD = 2, PAIR_PLAIN_SCALED = 3, PAIR_GATED_SCALED = 4 };

// Eight waves, four down the rows and two along the columns, each with WM x WN products of 16 x 16.
// Gated: half of the weight rows are gates and half are ups, else C is the product itself.
// Rows and weight rows have rings of their own, of SA and SB chunks (SB >= SA). A tile of 256 x 192 has room for no third chunk of both, but
// for two of the rows and four of the weight, which comes from memory. A load's address is one scalar base an operand, advanced by a
// chunk, and 32 bits a lane that do not change (64 bits a lane: two vector additions a load). With both, and the epilogue's forms apart,
// us, weights that take turns, in turn with the kernel before: gated 6144 x 1024, 512 / 1,024 / 1,536 / 2,048 / 4,096 rows 13.2 -> 12.9, 18.2 -> 17.6,
// 22.9 -> 21.8, 27.8 -> 27.2, 55.0 -> 52.8; plain 1,024 x 3104 x 1024 14.8 -> 14.3, 2,048 x 1024 x 2048 16.7 -> 16.2, x 3072 and 2,048 x 5184 x 1024 level.
template <int WM, int WN, int SA, int SB, int FORM>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
gemm_pair_kernel(PairArgs a) {
    constexpr bool GATED = FORM == PAIR_GATED || FORM == PAIR_GATED_SCALED, SCALED = FORM == PAIR_PLAIN_SCALED || FORM == PAIR_GATED_SCALED;
    constexpr bool FOLD = FORM == PAIR_FOLD;
    constexpr int BM = 64 * WM, BN = 32 * WN, WAVES = 8;
    constexpr int LA = WM, GROUPS = BN / 8, LB = (GROUPS + WAVES - 1) / WAVES, LEAST = GROUPS / WAVES;      // a wave's loads of a chunk (of the weight: or LEAST)
    constexpr int STAGE_A = BM * 8, STAGE_B = BN * 8;
    static_assert(!GATED || WN % 2 == 0, "a wave's weight tiles are half gate, half up");
    static_assert(SA >= 2 && SB >= SA && (SA * STAGE_A + SB * STAGE_B) * 16 <= 163840, "the rings do not fit");
    static_assert((SA - 1) * LA + (SB - 1) * LB <= 63, "more loads on their way than the counter holds");
    __shared__ uint4 ring[SA * STAGE_A + SB * STAGE_B];
    uint4* const ring_b = ring + SA * STAGE_A;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / MV_WAVE), lane = tid % MV_WAVE, i = lane % 16, g = lane / 16;
    const int wm = wave / 2, wn = wave % 2;
    // An XCD has a run of tiles. Rows change fastest, so that a band of the weight goes into one L2; with more rows than weight rows
    // columns do, and it is a band of the rows: else every L2 reads all of the larger operand (5,564 x 736 x 1024 19.6 us, so 15.8).
    const int run = (a.tiles + GT_XCDS - 1) / GT_XCDS, id = blockIdx.x % GT_XCDS * run + blockIdx.x / GT_XCDS;
    if ((int)blockIdx.x / GT_XCDS >= run || id >= a.tiles) return;
    const int quick = id % a.fast, slow = id / a.fast, tm = a.by_columns ? slow : quick, tn = a.by_columns ? quick : slow;
    const int m0 = tm * BM, n0 = tn * (GATED ? BN / 2 : BN), n = a.K / GT_KC;

    // what the end needs from memory is asked for here, in front of everything
    // The sums of squares of the tile's rows: SHARE threads a row, of whose quads thread j of eight (a thread is 8 / SHARE of them) adds up
    // number j, j + 8, .. and the eight are added in pairs, in one order for every tile.
    constexpr int SHARE = BM == 64 ? 8 : BM == 128 ? 4 : 2, MINE = 8 / SHARE;
    float4 sq[SCALED ? MINE : 1];
    const float4* sq_row = nullptr;
    int quads = 0;
    if constexpr (SCALED) {
        quads = a.P / 4;
        sq_row = reinterpret_cast<const float4*>(a.partial + (size_t)min(m0 + tid / SHARE, a.M - 1) * a.P);
#pragma unroll
        for (int e = 0; e < MINE; ++e) {
            const int q = tid % SHARE * MINE + e;
            sq[e] = q < quads ? sq_row[q] : float4{0.f, 0.f, 0.f, 0.f};
        }
    }
    float4 old[FOLD ? WN : 1][FOLD ? WM : 1];
    float nw[FOLD ? WN : 1][4];
    if constexpr (FOLD) {
#pragma unroll
        for (int t = 0; t < WN; ++t) {
            const int col = min(n0 + 16 * (WN * wn + t) + 4 * g, a.I - 4);
            a.norm_weight.at_few<4>(col, nw[t]);
#pragma unroll
            for (int u = 0; u < WM; ++u)
                old[t][u] = *reinterpret_cast<const float4*>(a.resid + (size_t)min(m0 + 16 * (WM * wm + u) + i, a.M - 1) * a.ldr + col);
        }
    }

    // this lane's share of the loads (eight rows of a chunk an instruction, pieces swizzled as in gemm_tile.hip); the entry points have made
    // sure that the offsets fit into 32 bits
    const int lrow = lane / 8, piece = (lane % 8) ^ lrow;
    uint32_t off_a[LA], off_b[LB];
#pragma unroll
    for (int r = 0; r < LA; ++r) off_a[r] = ((uint32_t)min(8 * (wave + WAVES * r) + lrow, a.M - 1 - m0) * (uint32_t)a.lda + 8 * piece) * 2;
#pragma unroll
    for (int r = 0; r < LB; ++r) {
        const int row = 8 * (wave + WAVES * r) + lrow;
        const int w = !GATED || row < BN / 2 ? min(n0 + row, a.I - 1) : min(a.I + n0 + row - BN / 2, 2 * a.I - 1);
        off_b[r] = ((uint32_t)w * (uint32_t)a.K + 8 * piece) * 2;
    }
    const char* const from_a = reinterpret_cast<const char*>(a.A + (size_t)m0 * a.lda);
    const char* const from_b = reinterpret_cast<const char*>(a.W);
    auto fetch_a = [&](int c, int stage) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < LA; ++r)
            gt_load_to_lds_from(from_a + (size_t)c * (GT_KC * sizeof(bf16)), off_a[r],
                                (__attribute__((address_space(3))) void*)(ring + stage * STAGE_A + (wave + WAVES * r) * 64));
    };
    auto fetch_b = [&](int c, int stage) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < LB; ++r)
            if (GROUPS % WAVES == 0 || r < LEAST || wave < GROUPS % WAVES)
                gt_load_to_lds_from(from_b + (size_t)c * (GT_KC * sizeof(bf16)), off_b[r],
                                    (__attribute__((address_space(3))) void*)(ring_b + stage * STAGE_B + (wave + WAVES * r) * 64));
    };
    int a_off[WM], w_off[WN];
#pragma unroll
    for (int t = 0; t < WM; ++t) a_off[t] = (16 * (WM * wm + t) + i) * 8;
#pragma unroll
    for (int t = 0; t < WN; ++t) {
        const int group = !GATED ? WN * wn + t : t < WN / 2 ? (WN / 2) * wn + t : (WN / 2) * (2 + wn) + (t - WN / 2);
        w_off[t] = (16 * group + i) * 8;
    }
    const int sw0 = g ^ (i & 7), sw1 = (4 + g) ^ (i & 7);
    floatx4_t acc[WN][WM];
#pragma unroll
    for (int t = 0; t < WN; ++t)
#pragma unroll
        for (int u = 0; u < WM; ++u) acc[t][u] = floatx4_t{0.f, 0.f, 0.f, 0.f};
    struct Operands {
        TFrag a[WM], w[WN];
    };
    auto read = [&](int sa, int sb, int sw, Operands& o) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < WN; ++t) o.w[t].u = ring_b[sb * STAGE_B + w_off[t] + sw];
#pragma unroll
        for (int u = 0; u < WM; ++u) o.a[u].u = ring[sa * STAGE_A + a_off[u] + sw];
    };
    auto multiply = [&](const Operands& o) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < WM; ++u)
#pragma unroll
            for (int t = 0; t < WN; ++t) acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(o.w[t].v, o.a[u].v, acc[t][u], 0, 0, 0);
    };
    // Chunk k lives in stages k % SA and k % SB; its operands are read in two halves of 32 columns, each while the products of the half
    // before run. The barrier stands between the halves: then everybody's reads of chunk k are back, so chunks k + SA of the rows and
    // k + SB of the weight may come into its stages, and everybody's loads of chunk k + 1 have landed. A wave's loads behind those of
    // chunk k + 1 are then, with all there are to ask for, SA - 2 whole chunks, and the weight's of the turn that asked for the
    // chunk's rows where its own were asked for before; at the end, where some are missing, all are waited for.
    constexpr int STEADY = (SA - 2) * (LA + LEAST) + (SB > SA ? LEAST : 0);
    for (int j = -SB; j < 0; ++j) {                    // (as the turns in front of the first would)
        if (j + SA >= 0 && j + SA < n) fetch_a(j + SA, j + SA);
        if (j + SB < n) fetch_b(j + SB, j + SB);
    }
    Operands even, odd;
    if (n > SB) GT_WAIT_VMCNT((SA - 1) * (LA + LEAST));
    else GT_WAIT_VMCNT(0);
    __builtin_amdgcn_s_barrier();
    read(0, 0, sw0, even);
    int sa = 0, sb = 0;
    for (int k = 0; k < n; ++k) {
        const int old_a = sa, old_b = sb;
        sa = sa + 1 == SA ? 0 : sa + 1;
        sb = sb + 1 == SB ? 0 : sb + 1;
        read(old_a, old_b, sw1, odd);
        multiply(even);
        // (a read, then some products, in turn: as the compiler has them, all reads first, 3 % slower)
#pragma unroll
        for (int x = 0; x < WM + WN; ++x) {
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, WM * WN / (WM + WN) > 0 ? WM * WN / (WM + WN) : 1, 0);
        }
        if (k + SB <= n) GT_WAIT_VMCNT(STEADY);
        else GT_WAIT_VMCNT(0);
        __builtin_amdgcn_s_waitcnt(0xc07f);
        __builtin_amdgcn_s_barrier();
        if (k + SA < n) fetch_a(k + SA, old_a);
        if (k + SB < n) fetch_b(k + SB, old_b);
        if (k + 1 < n) read(sa, sb, sw0, even);
        multiply(odd);
    }

    // lane l holds C[row 16 u + l % 16][columns 4 (l / 16) .. + 3 of tile t]
    constexpr int TOUT = GATED ? WN / 2 : WN;
    if constexpr (FOLD) {
        // resid += bf16(product (+ bias)), as the add behind a rounded product makes it; a wave's columns leave each row's sum of squares
        const float off = a.unit_offset ? 1.f : 0.f;
        float ssq[WM];
#pragma unroll
        for (int u = 0; u < WM; ++u) ssq[u] = 0.f;
#pragma unroll
        for (int t = 0; t < WN; ++t) {
            const int col = n0 + 16 * (WN * wn + t) + 4 * g;
            float b[4] = {0.f, 0.f, 0.f, 0.f};
            if (a.bias != nullptr) {
#pragma unroll
                for (int e = 0; e < 4; ++e) b[e] = to_f(a.bias[min(col + e, a.I - 1)]);
            }
#pragma unroll
            for (int u = 0; u < WM; ++u) {
                const int row = m0 + 16 * (WM * wm + u) + i;
                if (row >= a.M || col >= a.I) continue;                 // (columns beyond the last come in fours)
                const float was[4] = {old[t][u].x, old[t][u].y, old[t][u].z, old[t][u].w};
                float x[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    x[e] = was[e] + __uint_as_float((uint32_t)f32_to_bf16_bits(acc[t][u][e] + b[e]) << 16);
                    ssq[u] = fmaf(x[e], x[e], ssq[u]);
                }
                *reinterpret_cast<float4*>(a.resid + (size_t)row * a.ldr + col) = float4{x[0], x[1], x[2], x[3]};
                *reinterpret_cast<uint2*>(a.weighted + (size_t)row * a.ldw + col) =
                    uint2{f32x2_to_bf16x2_bits(x[0] * (nw[t][0] + off), x[1] * (nw[t][1] + off)),
                          f32x2_to_bf16x2_bits(x[2] * (nw[t][2] + off), x[3] * (nw[t][3] + off))};
            }
        }
        const int part = n0 / (16 * WN) + wn;
#pragma unroll
        for (int u = 0; u < WM; ++u) {
            ssq[u] += __shfl_xor(ssq[u], 16, MV_WAVE);
            ssq[u] += __shfl_xor(ssq[u], 32, MV_WAVE);
            const int row = m0 + 16 * (WM * wm + u) + i;
            if (g == 0 && row < a.M && part < a.P) a.partial[(size_t)row * a.P + part] = ssq[u];
        }
        return;
    }
    float rinv[WM];
    if constexpr (SCALED) {
        float s[MINE];
#pragma unroll
        for (int e = 0; e < MINE; ++e) {
            for (int q = tid % SHARE * MINE + e + 8; q < quads; q += 8) {
                const float4 v = sq_row[q];
                sq[e].x += v.x; sq[e].y += v.y; sq[e].z += v.z; sq[e].w += v.w;
            }
            s[e] = (sq[e].x + sq[e].y) + (sq[e].z + sq[e].w);
        }
#pragma unroll
        for (int o = 1; o < MINE; o <<= 1)
#pragma unroll
            for (int e = 0; e < MINE; e += 2 * o) s[e] += s[e + o];
#pragma unroll
        for (int o = 1; o < SHARE; o <<= 1) s[0] += __shfl_xor(s[0], o, MV_WAVE);
        float* const sh = reinterpret_cast<float*>(ring);               // (behind the last barrier nobody reads the rings)
        if (tid % SHARE == 0 && tid / SHARE < BM) sh[tid / SHARE] = rsqrtf(s[0] / (float)a.K + a.eps);
        __syncthreads();
#pragma unroll
        for (int u = 0; u < WM; ++u) rinv[u] = sh[16 * (WM * wm + u) + i];
    }
    // The forms that are in use have code of their own, with nothing in it to be jumped over: what a wave fetches of it for the first time
    // is on its way (2,048 x 6144 x 1024: all in one 29.4 us, apart 27.2).
    auto store = [&](auto bias, auto clamped, auto whole) __attribute__((always_inline)) {
        constexpr bool BIAS = decltype(bias)::value, WHOLE = decltype(whole)::value;
#pragma unroll
        for (int t = 0; t < TOUT; ++t) {
            const int col = n0 + 16 * (TOUT * wn + t) + 4 * g;
            float bv[4] = {0.f, 0.f, 0.f, 0.f}, bu[4] = {0.f, 0.f, 0.f, 0.f};
            if constexpr (BIAS) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int c = min(col + e, a.I - 1);
                    bv[e] = a.bias != nullptr ? to_f(a.bias[c]) : 0.f;
                    bu[e] = GATED && a.bias != nullptr ? to_f(a.bias[a.I + c]) : 0.f;
                }
            }
#pragma unroll
            for (int u = 0; u < WM; ++u) {
                const int row = m0 + 16 * (WM * wm + u) + i;
                if (row >= a.M || col >= a.I) continue;
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    auto sum = [&](float x, float b) __attribute__((always_inline)) {
                        if constexpr (SCALED) return fmaf(x, rinv[u], BIAS ? b : 0.f);
                        else return BIAS ? x + b : x;
                    };
                    v[e] = sum(acc[t][u][e], bv[e]);
                    if constexpr (GATED) v[e] = a.pair.of_short<decltype(clamped)::value>(v[e], sum(acc[t + TOUT][u][e], bu[e]));
                }
                bf16* to = a.C + (size_t)row * a.ldc + col;
                if (WHOLE || (a.wide_stores && col + 3 < a.I)) {
                    *reinterpret_cast<uint2*>(to) = uint2{f32x2_to_bf16x2_bits(v[0], v[1]), f32x2_to_bf16x2_bits(v[2], v[3])};
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (col + e < a.I) to[e] = from_f<bf16>(v[e]);
                }
            }
        }
    };
    constexpr std::true_type yes{};
    constexpr std::false_type no{};
    const bool whole = a.wide_stores && a.I % 4 == 0;
    if (GATED && a.pair.limit > 0.f) {
        if (!whole) store(yes, yes, no);
        else if (a.bias != nullptr) store(yes, yes, yes);
        else store(no, yes, yes);
    } else {
        if (!whole) store(yes, no, no);
        else if (a.bias != nullptr) store(yes, no, yes);
        else store(no, no, yes);
    }
}

// 1: a tile's rows, lda apart, and the weight lie within the 32 bits of a lane's offset (what does not is left to the other kernels)
extern "C" int mv_gemm_pair_reaches(long lda, int N, int K) { return lda < 1L << 23 && (long)N * K < 1L << 31; }

struct PairTile {
    int tile;            // rows << 16 | weight rows
    double time, other;  // us, estimated: with that tile, and with what serves where this product does not
};

// Times in us, ours as said above (tiles wider than tall a little behind, rounds beyond the first 6 % longer each: the rows no longer come
// from L2); the library's with the activation behind it 8.5, the products at 1.1 to 1.5 PFLOP/s by K or the weight at 4.2 TB/s, and 6 bytes
// a result at 5 TB/s. Below the size where the library would serve (1,536 rows) the tiled product would, level at 128
// rows and behind from there.
static PairTile pair_tile(int M, int N, int K, int units) {
    const double chunks = K / GT_KC, memory = 2.0 * N * K / 5e6;
    PairTile best{0, 0, 0};
    for (int bm = 64; bm <= 256; bm += 64)
        for (int bn = 64; bn <= 192; bn += 64) {
            const double tiles = (double)((M + bm - 1) / bm) * ((N / 2 + bn / 2 - 1) / (bn / 2)), rounds = ceil(tiles / units);
            const double one = 3.5 + chunks * (0.15 + 0.385 * bm * bn / 16384.0 + (bn > bm ? 0.01 * (bn - bm) / 64 : 0.0));
            const double time = 2.0 + fmax(rounds * one * (1.0 + 0.06 * (rounds - 1)), memory);
            if (best.tile == 0 || time < best.time) {
                best.tile = bm << 16 | bn;
                best.time = time;
            }
        }
    const double rate = 1.1e9 + 0.4e9 * fmin(1.0, K / 4096.0);
    best.other = 8.5 + fmax(2.0 * M * N * K / rate, 2.0 * N * K / 4.2e6) + 3.0 * M * N / 5e6;
    return best;
}

// rows << 16 | weight rows of the tile that M rows against a pair [N = 2 I, K] have on a device of so many compute units; 0: the pair is left to
// the other kernels. Over 68 shapes, 129 to 8,192 rows, K of 512 to 4,096, the choice is 1 % behind the best on average; above 6,144 rows the
// library is ahead again. Above 1,536 rows a pair may be estimated up to 5 % behind the library with its activation (98 pairs of 1,552 to 6,144
// rows: 1.0 to 2.1 times as fast) but for N of its tiles, where the estimate is too high for it and has to be 3 % ahead: 4,096 x 4096 x 2048
// 66.8 us there and 75.6 here, 5,120 x 6144 x 1024 78 and 81, 4,096 x 8192 x 1024 81 and 84; 2,560 x 6144 x 1024 43.4 both. Weights of 64 MB and
// more are left to it at every number of rows: there a pair is two calls, the product and its activation. Whether the pair comes here is decided by
// the rows that a recorded step is padded to (the library rounds gate and up in front of the activation), the tile by the rows there
// are: every tile adds in one order.
extern "C" int mv_gemm_pair_shape(int M, int N, int K, int units) {
    if (M <= 128 || M > 6144 || N % 2 || K % GT_KC || N <= 0 || K <= 0 || 2.0 * N * K >= 64.0 * 1024 * 1024) return 0;
    const int padded = mv_class_rows(M);
    const PairTile p = pair_tile(padded, N, K, units);
    if (p.time >= (padded <= 1536 ? 1.0 : N % 256 ? 1.05 : 0.97) * p.other) return 0;
    return M == padded ? p.tile : pair_tile(M, N, K, units).tile;
}

static int check_pair(const char* what, const void* A, long lda, const void* W, int M, int N, int K) {
    MV_REQUIRE(M > 0 && N > 0 && K > 0 && K % GT_KC == 0, "%s: bad sizes M=%d N=%d K=%d", what, M, N, K);
    MV_REQUIRE(A && W && lda >= K && lda % 8 == 0 && ((uintptr_t)A | (uintptr_t)W) % 16 == 0, "%s: operands not aligned or pitches too small", what);
    MV_REQUIRE(mv_gemm_pair_reaches(lda, N, K), "%s: rows %ld apart or a weight of %d x %d are too long", what, lda, N, K);
    return 0;
}

// the tile's sides, and how an XCD's run goes through the tiles
static int place_tiles(const char* what, PairArgs& a, int N, bool gated, int bm, int bn, dim3& grid) {
    const int wide = gated ? bn / 2 : bn, tiles_m = (a.M + bm - 1) / bm, tiles_n = (a.I + wide - 1) / wide;
    const long tiles = (long)tiles_m * tiles_n;
    MV_REQUIRE(tiles < (1L << 30), "%s: too many tiles", what);
    a.tiles = (int)tiles;
    a.by_columns = a.M > N;
    a.fast = a.by_columns ? tiles_n : tiles_m;
    a.wide_stores = a.ldc % 4 == 0 && (uintptr_t)a.C % 8 == 0;
    grid = dim3((unsigned)((tiles + GT_XCDS - 1) / GT_XCDS * GT_XCDS));
    return 0;
}

template <int FORM>
static int launch_pair(const char* what, PairArgs& a, int N, int tile, hipStream_t stream) {
    const int bm = tile >> 16, bn = tile & 0xffff;
    MV_REQUIRE(bm >= 64 && bm <= 256 && bm % 64 == 0 && (bn == 64 || bn == 128 || bn == 192), "%s: no tile of %d x %d", what, bm, bn);
    dim3 grid;
    if (place_tiles(what, a, N, true, bm, bn, grid)) return 1;
#define GP_LAUNCH(WM, WN, SA, SB) hipLaunchKernelGGL((gemm_pair_kernel<WM, WN, SA, SB, FORM>), grid, dim3(512), 0, stream, a)
    if (bn == 192) {
        if (bm == 256) GP_LAUNCH(4, 6, 2, 4);
        else if (bm == 192) GP_LAUNCH(3, 6, 3, 3);
        else if (bm == 128) GP_LAUNCH(2, 6, 4, 4);
        else GP_LAUNCH(1, 6, 4, 4);
    } else if (bn == 128) {
        if (bm == 256) GP_LAUNCH(4, 4, 3, 3);
        else if (bm == 192) GP_LAUNCH(3, 4, 4, 4);
        else if (bm == 128) GP_LAUNCH(2, 4, 4, 4);
        else GP_LAUNCH(1, 4, 4, 4);
    } else {
        if (bm == 256) GP_LAUNCH(4, 2, 4, 4);
        else if (bm == 192) GP_LAUNCH(3, 2, 4, 4);
        else if (bm == 128) GP_LAUNCH(2, 2, 4, 4);
        else GP_LAUNCH(1, 2, 4, 4);
    }
#undef GP_LAUNCH
    return mv_check_launch(what);
}

// C [M, I] bf16 (pitch ldc) = pair(A Wg^T (+ bias), A Wu^T (+ bias)) for the packed weight [N = 2 I, K]: K a multiple of 64, A and W at
// 16-byte addresses, pitch lda a multiple of eight. `tile`: as mv_gemm_pair_shape says, or another of 64, 128, 192, 256 rows by 64, 128, 192.
extern "C" int mv_gemm_pair(const void* A, long lda, const void* W, const void* bias, void* C, long ldc, int M, int N, int K, float limit, float slope,
                            int tile, hipStream_t stream) {
    if (check_pair("gemm_pair", A, lda, W, M, N, K)) return 1;
    MV_REQUIRE(C && N % 2 == 0 && ldc >= N / 2, "gemm_pair: N=%d is odd or ldc=%ld too small", N, ldc);
    PairArgs a{(const bf16*)A, lda, (const bf16*)W, (const bf16*)bias, (bf16*)C, ldc, M, N / 2, K, 0, 0, 0, 0, GatedPair{limit, slope}};
    return launch_pair<PAIR_GATED>("gemm_pair", a, N, tile, stream);
}

// Columns of the plain product's tiles, and its time in us with tiles of bm x bn in one round, fitted to 671 of 130 to 4,096 rows, K of 256 to
// 4,096, before the kernel's loads had a scalar base: of the kernel now 37 such took 3 % less, with a standard deviation of 6 %: operands into LDS (bm + bn), out of it and through the matrix unit (bm bn), both slower
// the more units are at it.
static const int kRoundColumns[] = {64, 96, 128, 192};
static double round_time(int bm, int bn, int K, double tiles, int units) {
    const double chunks = K / GT_KC, sides = (bm + bn) / 256.0;
    return 0.46 + 4.41 * sides + chunks * (0.204 - 0.080 * sides + 0.311 * bm * bn / 16384.0 + 0.165 * sides * tiles / units);
}
static PairTile round_tile(int M, int N, int K, int units) {
    PairTile best{0, 0, 0};
    for (int bm = 64; bm <= 256; bm += 64)
        for (int bn : kRoundColumns) {
            const double tiles = (double)((M + bm - 1) / bm) * ((N + bn - 1) / bn), time = round_time(bm, bn, K, tiles, units);
            if (tiles <= units && (best.tile == 0 || time < best.time)) {
                best.tile = bm << 16 | bn;
                best.time = time;
            }
        }
    best.other = N % 256 ? 10.2 + 2.0 * M * N * K / 1.15e9 : 7.5 + 2.0 * M * N * K / 1.3e9;
    return best;
}

// rows << 16 | columns of the tile that M rows against a plain weight [N, K] have, 0: the library's (or gemm_deep.hip's). The library's
// times are taken as its better ones, 1.15 PFLOP/s behind 10.2 us, 1.3 behind 7.5 where N is a multiple of its tiles: over 133 shapes, 160 to
// 4,096 rows, of the 95 that come here one is 4 % behind it and the others up to 43 % ahead. Decided by the rows of the step's class, as above.
extern "C" int mv_gemm_round_shape(int M, int N, int K, int units) {
    if (M <= 128 || M > 8192 || N <= 0 || K <= 0 || K % GT_KC || (double)N * K >= 240e6 || mv_gemm_deep_shape(M, N, K, 0)) return 0;
    const int padded = mv_class_rows(M);
    const PairTile p = round_tile(padded, N, K, units);
    if (p.tile == 0 || p.time >= p.other) return 0;
    return M == padded ? p.tile : round_tile(M, N, K, units).tile;
}

template <int FORM>
static int launch_round(const char* what, PairArgs& a, int tile, hipStream_t stream) {
    const int bm = tile >> 16, bn = tile & 0xffff;
    MV_REQUIRE(bm >= 64 && bm <= 256 && bm % 64 == 0 && (bn == 64 || bn == 96 || bn == 128 || bn == 192), "%s: no tile of %d x %d", what, bm, bn);
    dim3 grid;
    if (place_tiles(what, a, a.I, false, bm, bn, grid)) return 1;
#define GR_LAUNCH(WM, WN, SA, SB) hipLaunchKernelGGL((gemm_pair_kernel<WM, WN, SA, SB, FORM>), grid, dim3(512), 0, stream, a)
    if (bn == 192) {
        if (bm == 256) GR_LAUNCH(4, 6, 2, 4);
        else if (bm == 192) GR_LAUNCH(3, 6, 3, 3);
        else if (bm == 128) GR_LAUNCH(2, 6, 4, 4);
        else GR_LAUNCH(1, 6, 4, 4);
    } else if (bn == 128) {
        if (bm == 256) GR_LAUNCH(4, 4, 3, 3);
        else if (bm == 192) GR_LAUNCH(3, 4, 4, 4);
        else if (bm == 128) GR_LAUNCH(2, 4, 4, 4);
        else GR_LAUNCH(1, 4, 4, 4);
    } else if (bn == 96) {
        if (bm == 256) GR_LAUNCH(4, 3, 3, 3);
        else if (bm == 192) GR_LAUNCH(3, 3, 4, 4);
        else if (bm == 128) GR_LAUNCH(2, 3, 4, 4);
        else GR_LAUNCH(1, 3, 4, 4);
    } else {
        if (bm == 256) GR_LAUNCH(4, 2, 4, 4);
        else if (bm == 192) GR_LAUNCH(3, 2, 4, 4);
        else if (bm == 128) GR_LAUNCH(2, 2, 4, 4);
        else GR_LAUNCH(1, 2, 4, 4);
    }
#undef GR_LAUNCH
    return mv_check_launch(what);
}

// C [M, N] bf16 (pitch ldc) = A W^T (+ bias), operands as above. `tile`: 64 to 256 rows by 64, 96, 128, 192 columns.
extern "C" int mv_gemm_round(const void* A, long lda, const void* W, const void* bias, void* C, long ldc, int M, int N, int K, int tile,
                             hipStream_t stream) {
    if (check_pair("gemm_round", A, lda, W, M, N, K)) return 1;
    MV_REQUIRE(C && ldc >= N, "gemm_round: ldc=%ld too small for N=%d", ldc, N);
    PairArgs a{(const bf16*)A, lda, (const bf16*)W, (const bf16*)bias, (bf16*)C, ldc, M, N, K, 0, 0, 0, 0, GatedPair{0.f, 1.f}};
    return launch_round<PAIR_PLAIN>("gemm_round", a, tile, stream);
}

// ---- the norms between two products taken apart (see gemm_deep.hip), for prompts and steps with prompts in them, 129 to 1,024 rows:
// there an add and a norm of their own are 3.5 to 4.5 us, most of it what any kernel costs. What serves is decided by the rows of a step's
// class, and the sums of squares are added in an order that the rows there are have no part in.
// us, weights of the 0.6B sizes that take turns, before / with it: output projection and add + norm, 256 rows 10.2 / 7.2, 512 12.9 / 9.1, 552 15.2 / 12.7,
// 1,000 16.1 / 13.9; down and add + norm 12.1 / 8.8, 15.8 / 11.2, 18.8 / 17.1, 20.1 / 17.8; the gated pair 9.5 / 10.0, 12.5 / 12.9, 12.9 / 13.6,
// 17.5 / 18.3; queries, keys and values, 512 rows 10.8 / 10.1, 552 14.0 / 12.1, 1,000 14.3 both. With more rows the sums' way through memory
// at the products' ends costs what the norm's kernel does: 2,048 rows, all four, 98.5 / 98.4.
#define PN_MIN_ROWS 128
#define PN_MAX_ROWS 1024

// Behind the norm: the tile of gemm_pair.hip, or 1 for a tile of gemm_deep.hip, or 0: not served.
static int behind_norm_tile(int M, int N, int K, bool gated, int units) {
    if (M <= PN_MIN_ROWS || M > PN_MAX_ROWS || N <= 0 || K <= 0 || K % GT_KC || (gated && N % 2)) return 0;
    const int padded = mv_class_rows(M);
    if (padded > PN_MAX_ROWS) return 0;
    if (mv_gemm_deep_shape(padded, N, K, gated)) return 1;
    if (gated) return mv_gemm_pair_shape(M, N, K, units);
    return round_tile(padded, N, K, units).tile ? round_tile(M, N, K, units).tile : 0;
}
extern "C" int mv_gemm_behind_norm_serves(int M, int N, int K, int gated, int units) { return behind_norm_tile(M, N, K, gated != 0, units) != 0; }

// C [M, N] bf16 = A W^T / rms (+ bias), or the gated pair of it [M, N / 2], rms[m] = sqrt(sum_p partial[m][p] / K + eps); operands as above,
// partial at a 16-byte address, P a multiple of four.
extern "C" int mv_gemm_behind_norm(const void* A, long lda, const void* W, const void* bias, void* C, long ldc, int M, int N, int K, int gated, float limit,
                                   float slope, const float* partial, int P, float eps, hipStream_t stream) {
    if (check_pair("gemm_behind_norm", A, lda, W, M, N, K)) return 1;
    MV_REQUIRE(C && (!gated || N % 2 == 0) && ldc >= (gated ? N / 2 : N), "gemm_behind_norm: N=%d is odd or ldc=%ld too small", N, ldc);
    MV_REQUIRE(partial != nullptr && (uintptr_t)partial % 16 == 0 && P > 0 && P % 4 == 0 && eps > 0.f,
               "gemm_behind_norm: the partial sums (P=%d, in fours) or eps are missing or not aligned", P);
    const int tile = behind_norm_tile(M, N, K, gated != 0, mv_compute_units());
    MV_REQUIRE(tile != 0, "gemm_behind_norm: M=%d N=%d K=%d is not served", M, N, K);
    if (tile == 1)
        return mv_gemm_deep(A, lda, W, bias, C, ldc, MV_BF16, M, N, K, gated, partial, P, eps, limit, slope, 0, mv_gemm_deep_shape(mv_class_rows(M), N, K, gated),
                            stream);
    PairArgs a{(const bf16*)A, lda, (const bf16*)W, (const bf16*)bias, (bf16*)C, ldc, M, gated ? N / 2 : N, K, 0, 0, 0, 0, GatedPair{limit, slope},
               const_cast<float*>(partial), P, eps};
    return gated ? launch_pair<PAIR_GATED_SCALED>("gemm_behind_norm", a, N, tile, stream) : launch_round<PAIR_PLAIN_SCALED>("gemm_behind_norm", a, tile, stream);
}

extern "C" int mv_gemm_into_norm_rows() { return PN_MAX_ROWS; }
// In front of it: partial sums a row, 0: not served. One round of tiles of 64 x 64 where gemm_deep.hip takes no more rows.
extern "C" int mv_gemm_into_norm_parts(int M, int N, int K, int units) {
    if (M <= PN_MIN_ROWS || M > PN_MAX_ROWS || N <= 0 || K <= 0 || N % 128 || K % GT_KC || (long)N * K >= 8L << 20) return 0;
    const int padded = mv_class_rows(M);
    if (padded > PN_MAX_ROWS) return 0;
    if (mv_gemm_deep_shape(padded, N, K, 0)) return mv_gemm_deep_fold_parts(N);
    return (long)((padded + 63) / 64) * (N / 64) <= units ? N / 32 : 0;
}

// resid [M, N] += bf16(A W^T (+ bias)), weighted = bf16(resid * norm_weight (+ 1 with unit_offset)), partial [M, P] = sums of resid^2 over N / P columns each.
extern "C" int mv_gemm_into_norm(const void* A, long lda, const void* W, const void* bias, float* resid, long ldr, const void* norm_weight,
                                 int norm_weight_dtype, int unit_offset, void* weighted, long ldw, float* partial, int P, int M, int N, int K,
                                 hipStream_t stream) {
    if (check_pair("gemm_into_norm", A, lda, W, M, N, K)) return 1;
    MV_REQUIRE(P > 0 && P == mv_gemm_into_norm_parts(M, N, K, mv_compute_units()), "gemm_into_norm: M=%d N=%d K=%d is not served with %d partial sums", M, N, K, P);
    if (mv_gemm_deep_shape(mv_class_rows(M), N, K, 0))
        return mv_gemm_deep_fold(A, lda, W, bias, resid, ldr, norm_weight, norm_weight_dtype, unit_offset, weighted, ldw, partial, P, M, N, K,
                                 mv_gemm_deep_shape(mv_class_rows(M), N, K, 0), stream);
    MV_REQUIRE(resid != nullptr && weighted != nullptr && partial != nullptr && ldr >= N && ldw >= N && ldr % 4 == 0 && ldw % 4 == 0
               && (uintptr_t)resid % 16 == 0 && (uintptr_t)weighted % 8 == 0,
               "gemm_into_norm: the residual, the weighted rows or the partial sums are missing or not aligned (ldr=%ld, ldw=%ld)", ldr, ldw);
    MV_REQUIRE(mv_valid_dtype(norm_weight_dtype) && norm_weight != nullptr && (uintptr_t)norm_weight % 16 == 0,
               "gemm_into_norm: the norm weight is missing, of an unknown type or not 16-byte aligned");
    PairArgs a{(const bf16*)A, lda, (const bf16*)W, (const bf16*)bias, nullptr, 0, M, N, K, 0, 0, 0, 0, GatedPair{0.f, 1.f}, partial, P, 0.f,
               resid, ldr, WeightPtr{norm_weight, norm_weight_dtype}, unit_offset, (bf16*)weighted, ldw};
    dim3 grid;
    if (place_tiles("gemm_into_norm", a, N, false, 64, 64, grid)) return 1;
    hipLaunchKernelGGL((gemm_pair_kernel<1, 2, 4, 4, PAIR_FOLD>), grid, dim3(512), 0, stream, a);
    return mv_check_launch("gemm_into_norm");
}
