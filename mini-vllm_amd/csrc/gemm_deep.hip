// C[M, N] = A[M, K] * W[N, K]^T (+ bias) or its gated pair in bf16 for products whose tiles hardly fill the chip once (up to a few hundred
// rows against the weights of a small model, up to 16 against larger ones), so that their time is that of one tile: how often a
// workgroup goes to memory and back, and how many lines it asks for.
//
// A chunk is 256 values of k, 32 for each of the eight waves: the waves split K, not the tile, and K = 2048 is eight steps of a
// ring of LDS stages, all of which are asked for at once where K is short (the tiled product of gemm_tile.hip with its chunks
// of 64 takes 32 steps, each with a barrier and a wait; the weight-streaming one loads sixteen rows an instruction, half lines
// or single ones, and every workgroup all activation rows). A row's 512 bytes of a chunk are loaded as whole lines straight
// into LDS; a wave has the operands of its next block in registers before the products of the current one. At the end the
// waves' sums are added in the order ((0+4)+(2+6))+((1+5)+(3+7)) through LDS, in float, and rounded once. Against weights of 8 Mi
// elements and more a wave adds up even and odd chunks apart (CHAINS), so that a sum has sixteen chains, as it has in the weight-streaming
// product there, and no larger an error (16 rows of N(0, 1) operands, weight-streaming / eight chains / sixteen: K = 4096 1.06e-7 / 1.34e-7 /
// 1.02e-7, 12288 1.68e-7 / 2.34e-7 / 1.65e-7). Below that its sums have eight, and so has this one (K = 1024 8.2e-8 / 7.6e-8, 3072 1.21e-7 /
// 1.18e-7): two accumulators a tile cost 2 % where tiles are many.
// LDS: rows of 512 bytes, 16-byte piece p of row r in place p ^ (r & 15): sixteen lanes that read one piece of sixteen rows
// meet in no bank.
//
// Like the weight-streaming product it takes the norms between two products apart: behind a folded norm (`partial`) row m is
// divided by sqrt(sum_p partial[m][p] / K + eps) before the bias; in front of one (FOLD) the product, rounded, is added to the
// float residual, the sum times the norm's weight is stored beside it, and a tile's columns leave each row's sum of squares. What
// these read besides (sums, residual, weights) is asked for before the first chunk and used behind the last.
//
// What bounds it: the operands of a tile, (rows + columns) x K, that a compute unit can pull from the caches, and a fixed 3 to
// 4 us. Measured alone (us; weight-streaming, tiled or the library's, whichever served / here; what is faster alone is not always so in
// a model, see the rule): 8 x 4096 x 1024 behind a norm 5.6 / 4.8,
// 8 x 6144 x 1024 gated behind a norm 7.5 / 6.2, 8 x 1024 x 3072 in front of one 6.2 / 5.6, 8 x 6144 x 4096 14.1 / 11.8; 64 x 4096 x 1024
// 7.4 / 4.9, 64 x 1024 x 3072 in front of a norm 8.7 / 7.2; 512 x 1024 x 2048 9.8 / 7.7, 512 x 1024 x 3072 12.5 / 9.6.
#include "gemm_ring.h"
#include "gemm_deep.h"

#define GD_WAVES 8
#define GD_KC 256                   // columns of a chunk

struct DeepArgs {
    const bf16* A;
    long lda;
    const bf16* W;
    const bf16* bias;
    void* C;
    long ldc;
    int c_float, c_vec, M, N, K, half, tiles_m, tiles;   // half: columns of the result of a gated pair, else 0; c_vec: four columns a store
    GatedPair pair;
    int square_relu;
    // rows behind a folded norm: P partial sums of squares each; FOLD writes them
    float* partial;
    int P;
    float eps;
    float* resid;
    long ldr;
    WeightPtr norm_weight;
    int unit_offset;
    bf16* weighted;
    long ldw;
};

enum DeepForm { DEEP_PLAIN = 0, DEEP_GATED = 1, DEEP_FOLD = 2 };

// RM x RN tiles of 16 tokens x 16 weight rows a workgroup; gated: the second half of the weight rows are the up rows of the
// first half's columns
template <int RM, int RN, int STAGES, int FORM, int CHAINS>
__global__ void __launch_bounds__(64 * GD_WAVES)
gemm_deep_kernel(DeepArgs p) {
    constexpr bool GATED = FORM == DEEP_GATED, FOLD = FORM == DEEP_FOLD;
    constexpr int ROWS = 16 * (RM + RN), LOADS = RM + RN, TILES = RM * RN;
    constexpr int OC = GATED ? RN / 2 : RN;          // tiles of output columns
    static_assert(TILES * 8192 <= STAGES * ROWS * 512 && RM * OC <= GD_WAVES, "the sums fit where the ring was, an output tile a wave");
    __shared__ uint4 ring[STAGES][ROWS][32];
    __shared__ float sh_rinv[16 * RM];
    const int tid = threadIdx.x, lane = tid % MV_WAVE, wave = __builtin_amdgcn_readfirstlane(tid / MV_WAVE), i = lane % 16, g = lane / 16;
    // workgroups go to the XCDs in turn: an XCD takes neighbouring tiles, which share weight rows (row tiles follow each other)
    const int xcd = blockIdx.x % GT_XCDS;
    const int tile = (int)((long)p.tiles * xcd / GT_XCDS) + blockIdx.x / GT_XCDS;
    if (tile >= (int)((long)p.tiles * (xcd + 1) / GT_XCDS)) return;
    const int m0 = tile % p.tiles_m * (16 * RM), n0 = tile / p.tiles_m * (16 * OC), last = (GATED ? p.half : p.N) - 1;
    const int chunks = p.K / GD_KC;

    // this wave's output tile: token i, columns col .. col + 3 of a lane
    const int orow = wave / OC, ocol = wave % OC, tok = m0 + 16 * orow + i, col = n0 + 16 * ocol + 4 * g;
    const bool owns = wave < RM * OC && tok < p.M && col <= last;
    float4 old{0.f, 0.f, 0.f, 0.f};
    float nw[4] = {0.f, 0.f, 0.f, 0.f};
    if constexpr (FOLD) {
        if (owns) {
            old = *reinterpret_cast<const float4*>(p.resid + (size_t)tok * p.ldr + col);
            p.norm_weight.at_few<4>(col, nw);
        }
    }
    // the sums of squares of the tile's rows: SHARE threads a row
    constexpr int SHARE = 64 * GD_WAVES / (16 * RM), FIRST = 256 / SHARE;
    const bool scaled = !FOLD && p.partial != nullptr;
    float sq[FIRST];
    const float* sq_row = nullptr;
    if (scaled) {
        sq_row = p.partial + (size_t)min(m0 + tid / SHARE, p.M - 1) * p.P;
#pragma unroll
        for (int e = 0; e < FIRST; ++e) {
            const int at = tid % SHARE + e * SHARE;
            sq[e] = at < p.P ? sq_row[at] : 0.f;
        }
    }

    const bf16* src[LOADS];                          // this lane's place in the rows that it brings in, two rows an instruction
#pragma unroll
    for (int j = 0; j < LOADS; ++j) {
        const int r = 2 * (wave * LOADS + j) + lane / 32, piece = lane % 32 ^ (r & 15);
        const bf16* row;
        if (r < 16 * RM) {
            row = p.A + (size_t)min(m0 + r, p.M - 1) * p.lda;
        } else {
            const int c = r - 16 * RM, up = GATED && c >= 16 * OC;
            row = p.W + (size_t)(min(n0 + c - (up ? 16 * OC : 0), last) + (up ? p.half : 0)) * p.K;
        }
        src[j] = row + 8 * piece;
    }
    auto fetch = [&](int stage) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < LOADS; ++j) {
            gt_load_to_lds(src[j], (__attribute__((address_space(3))) void*)&ring[stage][2 * (wave * LOADS + j)][0]);
            src[j] += GD_KC;
        }
    };
    TFrag a[2][RM], w[2][RN];
    auto take = [&](int stage, int to) __attribute__((always_inline)) {
        const int slot = (4 * wave + g) ^ i;
#pragma unroll
        for (int r = 0; r < RM; ++r) a[to][r].u = ring[stage][16 * r + i][slot];
#pragma unroll
        for (int c = 0; c < RN; ++c) w[to][c].u = ring[stage][16 * (RM + c) + i][slot];
    };
    floatx4_t acc[CHAINS][RM][RN];                   // two: of the even chunks, of the odd ones
#pragma unroll
    for (int r = 0; r < RM; ++r)
#pragma unroll
        for (int c = 0; c < RN; ++c) acc[0][r][c] = acc[CHAINS - 1][r][c] = floatx4_t{0.f, 0.f, 0.f, 0.f};
    // this wave's loads have landed but for those of the newest `left` chunks, and what it read of LDS has arrived; then all waves'
    auto meet = [&](int left) __attribute__((always_inline)) {
#define GD_WAIT(N) __builtin_amdgcn_s_waitcnt(0x0070 | (((N) * LOADS) & 15) | ((((N) * LOADS) >> 4) << 14))
        switch (left) {
            case 0: GD_WAIT(0); break;
            case 1: GD_WAIT(1); break;
            case 2: GD_WAIT(2); break;
            case 3: GD_WAIT(3); break;
            case 4: GD_WAIT(4); break;
            default: GD_WAIT(5); break;
        }
#undef GD_WAIT
        asm volatile("s_barrier" ::: "memory");
    };
    static_assert(STAGES <= 6 && 5 * LOADS < 64, "meet knows five chunks on their way");
    const int ahead = min(STAGES, chunks);
    for (int s = 0; s < ahead; ++s) fetch(s);
    meet(ahead - 1);
    take(0, 0);
    int stage = 0;
    auto turn = [&](int c, int cur) __attribute__((always_inline)) {
        // behind the barrier this chunk is in registers everywhere: its stage is free
        if (c + 1 < chunks) {
            meet(min(STAGES - 2, chunks - 2 - c));
            if (c + STAGES < chunks) fetch(stage);
            if (++stage == STAGES) stage = 0;
            take(stage, 1 - cur);
        }
#pragma unroll
        for (int r = 0; r < RM; ++r)
#pragma unroll
            for (int k = 0; k < RN; ++k) acc[cur % CHAINS][r][k] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[cur][k].v, a[cur][r].v, acc[cur % CHAINS][r][k], 0, 0, 0);
    };
    for (int c = 0; c < chunks; c += 2) {
        turn(c, 0);
        if (c + 1 < chunks) turn(c + 1, 1);
    }
    // the waves' sums; a lane holds token i, weight rows 4 g .. 4 g + 3 of a tile
    __builtin_amdgcn_s_waitcnt(0x0070);
    asm volatile("s_barrier" ::: "memory");
    floatx4_t* part = reinterpret_cast<floatx4_t*>(&ring[0][0][0]);
#pragma unroll
    for (int r = 0; r < RM; ++r)
#pragma unroll
        for (int c = 0; c < RN; ++c) part[((r * RN + c) * GD_WAVES + wave) * MV_WAVE + lane] = CHAINS == 1 ? acc[0][r][c] : acc[0][r][c] + acc[CHAINS - 1][r][c];
    if (scaled) {
        float t = 0.f;
#pragma unroll
        for (int e = 0; e < FIRST; ++e) t += sq[e];
        for (int at = tid % SHARE + 256; at < p.P; at += SHARE) t += sq_row[at];
#pragma unroll
        for (int o = 1; o < SHARE; o <<= 1) t += __shfl_xor(t, o, MV_WAVE);
        if (tid % SHARE == 0) sh_rinv[tid / SHARE] = rsqrtf(t / (float)p.K + p.eps);
    }
    __syncthreads();
    if (wave >= RM * OC) return;
    auto sum = [&](int t) -> floatx4_t {
        const floatx4_t* s = part + t * GD_WAVES * MV_WAVE + lane;
        return ((s[0] + s[4 * MV_WAVE]) + (s[2 * MV_WAVE] + s[6 * MV_WAVE])) +
               ((s[MV_WAVE] + s[5 * MV_WAVE]) + (s[3 * MV_WAVE] + s[7 * MV_WAVE]));
    };
    floatx4_t o = sum(orow * RN + ocol), u{0.f, 0.f, 0.f, 0.f};
    if constexpr (GATED) u = sum(orow * RN + OC + ocol);
    if constexpr (FOLD) {
        // resid += bf16(product (+ bias)), as the add behind a rounded product makes it
        const float was[4] = {old.x, old.y, old.z, old.w}, off = p.unit_offset ? 1.f : 0.f;
        float x[4], ssq = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float v = p.bias != nullptr ? o[e] + to_f(p.bias[min(col + e, last)]) : o[e];
            x[e] = was[e] + __uint_as_float((uint32_t)f32_to_bf16_bits(v) << 16);
            ssq += x[e] * x[e];
        }
        if (owns) {
            *reinterpret_cast<float4*>(p.resid + (size_t)tok * p.ldr + col) = float4{x[0], x[1], x[2], x[3]};
            *reinterpret_cast<uint2*>(p.weighted + (size_t)tok * p.ldw + col) =
                uint2{f32x2_to_bf16x2_bits(x[0] * (nw[0] + off), x[1] * (nw[1] + off)), f32x2_to_bf16x2_bits(x[2] * (nw[2] + off), x[3] * (nw[3] + off))};
        } else {
            ssq = 0.f;                               // (columns beyond the last come in fours)
        }
        ssq += __shfl_xor(ssq, 16, MV_WAVE);
        ssq += __shfl_xor(ssq, 32, MV_WAVE);
        if (g == 0 && owns) p.partial[(size_t)tok * p.P + (n0 / 16 + ocol)] = ssq;
        return;
    }
    if (!owns) return;
    const float rinv = scaled ? sh_rinv[16 * orow + i] : 1.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int n = min(col + e, last);
        const float b = p.bias != nullptr ? to_f(p.bias[n]) : 0.f;
        if constexpr (GATED) {
            o[e] = p.pair.of(fmaf(o[e], rinv, b), fmaf(u[e], rinv, p.bias != nullptr ? to_f(p.bias[p.half + n]) : 0.f));
        } else {
            o[e] = o[e] * rinv + b;
            if (p.square_relu) o[e] = o[e] > 0.f ? o[e] * o[e] : 0.f;
        }
    }
    const size_t at = (size_t)tok * p.ldc + col;
    if (col + 3 <= last && p.c_vec) {
        if (p.c_float) *reinterpret_cast<floatx4_t*>((float*)p.C + at) = o;
        else *reinterpret_cast<uint2*>((bf16*)p.C + at) = uint2{f32x2_to_bf16x2_bits(o[0], o[1]), f32x2_to_bf16x2_bits(o[2], o[3])};
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (col + e <= last) {
                if (p.c_float) ((float*)p.C)[at + e] = o[e];
                else ((bf16*)p.C)[at + e] = from_f<bf16>(o[e]);
            }
    }
}

// Shapes: 11: 16 x 16, 12: 16 x 32, 22: 32 x 32, 24: 32 x 64 (gated: half as many output columns, the other half of the weight rows are the up rows)
static long deep_tiles(int shape, int M, int columns, bool gated) {
    const int rm = shape / 10, rn = shape % 10, wide = 16 * (gated ? rn / 2 : rn);
    return (long)((M + 16 * rm - 1) / (16 * rm)) * ((columns + wide - 1) / wide);
}

// Which products come here, and with which tile: the smallest of which every compute unit gets at most one. (The more units pull at a
// weight that comes from memory, the faster it is there: 64 rows against 1024 columns in front of a norm, 0.6B-sized steps, 8.8 us
// with 64 tiles and 6.9 with 256; a second round costs more than it saves: 192 x 4096 x 1024 9.6 us in two, the library 7.2.)
// Weights of 1 to 8 Mi elements from 9 rows on (below 1 Mi everything takes the fixed cost, 4 to 5 us): for fewer rows the
// weight-streaming product, whose workgroups take four
// columns, reads them as fast or faster (a step of one request 1,000 us with it, 1,043 here; of eight 1,130 and 1,135), at 16, 24,
// 40 and 64 requests steps take 1,355 / 1,214, 1,515 / 1,314, 1,812 / 1,552 and 3,117 / 2,819. Larger weights up to 16 rows, where
// 16 columns a unit cover them, or 32 up to 32 Mi elements, from the first row on
// (steps of the 8B sizes at 1,024 tokens, before / with it: 1 request 3,545 / 3,515, 2 3,579 / 3,543, 4 3,710 / 3,656, 8 4,005 / 3,860;
// one request of Dutilix 5,271 / 5,183, Bolapel 4,558 / 4,532, Sorulix 4,883 / 4,844, Zedudra 4,587 / 4,531, Furanex 5,795 / 5,774,
// Setirax 4,775 / 4,801), so a row's bits are the same for 1 to 16 rows; from 17 rows on the tiled product with its split of K is
// ahead (32 x 4096 x 12288 23.0 us against 33.1). A K of one chunk stays where it was: there is nothing to walk, and the others are as fast to 1 us.
// What stays with the library's split of K and the tiled product (us, these / here): above 96 rows a K of more than 4096 (500 x 128 x
// 8192 11.0 / 14.8, 800 x 512 x 16384 44.0 / 51.5; 200 x 768 x 8192 would be 19.9 / 15.4), and one of 4096 in tiles of 32 x 64 or above 512
// rows (800 x 576 x 4096 15.2 / 16.5, 800 x 256 x 4096 11.8 / 12.6; but 100 x 1024 x 4096 11.9 / 9.0, 300 x 576 x 4096 11.8 / 9.7); and
// two chunks in tiles of 32 x 64 above 32 rows (128 x 4096 x 512 5.8 / 5.9, gated 64 x 8192 x 512 6.4 / 6.6; 32 x 16384 x 512 8.6 / 7.4). Gated
// pairs of a longer K have no such end: 500 x 1024 x 8192 56.7 / 27.1.
// The other kernels add in other orders, so which one serves is decided by the rows that a recorded step is padded to (all shapes
// here add a weight up in one order): a step gives the same bits recorded and not.
static int served_shape(int M, int N, int K, bool gated) {
    if (M <= 0 || N <= 0 || K < 2 * GD_KC || K % GD_KC || (gated && N % 2)) return 0;
    const int columns = gated ? N / 2 : N;
    const long units = mv_compute_units(), weight = (long)N * K;
    if (weight > 8L << 20) {
        if (M > 16) return 0;
        if (!gated && deep_tiles(11, M, columns, false) <= units) return 11;
        return deep_tiles(12, M, columns, gated) <= units && weight <= 32L << 20 ? 12 : 0;
    }
    if (M <= 8 || weight < 1L << 20) return 0;
    if (!gated && M > 96 && (K > 4096 || (K == 4096 && M > 512))) return 0;
    for (const int shape : {11, 12, 22, 24}) {
        if ((gated && shape == 11) || deep_tiles(shape, M, columns, gated) > units) continue;
        const bool slow = shape == 24 && (K <= 2 * GD_KC ? M > 32 : !gated && K == 4096 && M > 96);
        return slow ? 0 : shape;
    }
    return 0;
}

static int deep_shape(int M, int N, int K, bool gated) {
    return M < (1 << 24) && served_shape(mv_class_rows(M), N, K, gated) ? served_shape(M, N, K, gated) : 0;
}

extern "C" int mv_gemm_deep_shape(int M, int N, int K, int gated) { return deep_shape(M, N, K, gated != 0); }
extern "C" int mv_gemm_deep_fold_parts(int N) { return (N + 15) / 16; }

template <int FORM>
static int deep_launch(const char* what, DeepArgs p, int shape, hipStream_t stream) {
    const bool gated = FORM == DEEP_GATED;
    MV_REQUIRE(p.M > 0 && p.N > 0 && p.K > 0 && p.K % GD_KC == 0, "%s: K=%d must be a positive multiple of %d (M=%d, N=%d)", what, p.K, GD_KC, p.M, p.N);
    MV_REQUIRE(p.lda >= p.K && p.lda % 8 == 0 && (uintptr_t)p.A % 16 == 0 && (uintptr_t)p.W % 16 == 0,
               "%s: rows must start at 16-byte addresses and hold K=%d (lda=%ld)", what, p.K, p.lda);
    MV_REQUIRE(!gated || p.N % 2 == 0, "%s: the gated form takes an even N", what);
    if (shape == 0) shape = deep_shape(p.M, p.N, p.K, gated);
    MV_REQUIRE(shape == 12 || shape == 22 || shape == 24 || (shape == 11 && !gated), "%s: no tile for M=%d N=%d K=%d (shape %d)", what, p.M, p.N, p.K, shape);
    p.half = gated ? p.N / 2 : 0;
    p.tiles_m = (p.M + 16 * (shape / 10) - 1) / (16 * (shape / 10));
    const long tiles = deep_tiles(shape, p.M, gated ? p.half : p.N, gated);
    MV_REQUIRE(tiles < (1L << 24), "%s: too many tiles", what);
    p.tiles = (int)tiles;
    const dim3 grid((p.tiles + GT_XCDS - 1) / GT_XCDS * GT_XCDS), block(64 * GD_WAVES);
    const bool chains = (long)p.N * p.K >= 8L << 20;
#define GD_LAUNCH(RM, RN, STAGES)                                                                                                   \
    do {                                                                                                                            \
        if (chains) hipLaunchKernelGGL((gemm_deep_kernel<RM, RN, STAGES, FORM, 2>), grid, block, 0, stream, p);                     \
        else hipLaunchKernelGGL((gemm_deep_kernel<RM, RN, STAGES, FORM, 1>), grid, block, 0, stream, p);                            \
    } while (0)
    if constexpr (!(FORM == DEEP_GATED))
        if (shape == 11) GD_LAUNCH(1, 1, 6);
    if (shape == 12) GD_LAUNCH(1, 2, 6);
    else if (shape == 22) GD_LAUNCH(2, 2, 4);
    else if (shape == 24) GD_LAUNCH(2, 4, 3);
#undef GD_LAUNCH
    return mv_check_launch(what);
}

// C[M, N] = A W^T (+ bias), or with `gated` C[M, N / 2] = pair(A Wg^T (+ bias), A Wu^T (+ bias)) for the packed weight [N, K]; bf16 A
// (row stride lda) and W (contiguous rows of K), C bf16 or float (the entry points in front of this one keep float outputs). With `partial` [M, P] output row m is first divided by
// sqrt(sum_p partial[m][p] / K + eps). square_relu: C = max(., 0)^2. shape: see deep_tiles; 0 lets the rule choose.
extern "C" int mv_gemm_deep(const void* A, long lda, const void* W, const void* bias, void* C, long ldc, int c_dtype, int M, int N, int K,
                            int gated, const float* partial, int P, float eps, float limit, float slope, int square_relu, int shape,
                            hipStream_t stream) {
    MV_REQUIRE(c_dtype == MV_F32 || c_dtype == MV_BF16, "gemm_deep: bad output dtype %d", c_dtype);
    MV_REQUIRE(C != nullptr && ldc >= (gated ? N / 2 : N), "gemm_deep: ldc=%ld too small for N=%d", ldc, N);
    MV_REQUIRE(partial == nullptr || (P > 0 && eps > 0.f), "gemm_deep: bad partial sums (P=%d) or eps", P);
    MV_REQUIRE(!square_relu || !gated, "gemm_deep: the squared ReLU needs no gated pair");
    DeepArgs p{};
    p.A = (const bf16*)A; p.lda = lda; p.W = (const bf16*)W; p.bias = (const bf16*)bias; p.C = C; p.ldc = ldc;
    p.c_float = c_dtype == MV_F32;
    p.c_vec = ldc % 4 == 0 && (uintptr_t)C % (p.c_float ? 16 : 8) == 0;
    p.M = M; p.N = N; p.K = K;
    p.pair = GatedPair{limit, slope};
    p.square_relu = square_relu;
    p.partial = const_cast<float*>(partial); p.P = P; p.eps = eps;
    return gated ? deep_launch<DEEP_GATED>("gemm_deep", p, shape, stream) : deep_launch<DEEP_PLAIN>("gemm_deep", p, shape, stream);
}

// The product in front of a residual add and an RMSNorm (see mv_gemm_skinny_fold): resid[M, N] += bf16(A W^T (+ bias)), weighted =
// bf16(resid * norm_weight (+ 1 with unit_offset)), partial[M, P] = sums of resid^2 over 16 columns each, P = mv_gemm_deep_fold_parts(N).
extern "C" int mv_gemm_deep_fold(const void* A, long lda, const void* W, const void* bias, float* resid, long ldr, const void* norm_weight,
                                 int norm_weight_dtype, int unit_offset, void* weighted, long ldw, float* partial, int P, int M, int N, int K,
                                 int shape, hipStream_t stream) {
    MV_REQUIRE(resid != nullptr && weighted != nullptr && partial != nullptr && ldr >= N && ldw >= N,
               "gemm_deep_fold: the residual, the weighted rows or the partial sums are missing (ldr=%ld)", ldr);
    MV_REQUIRE(mv_valid_dtype(norm_weight_dtype) && norm_weight != nullptr && ((uintptr_t)norm_weight % 16) == 0,
               "gemm_deep_fold: the norm weight is missing, of an unknown type or not 16-byte aligned");
    MV_REQUIRE(N % 4 == 0 && ldr % 4 == 0 && ldw % 4 == 0 && ((uintptr_t)resid % 16) == 0 && ((uintptr_t)weighted % 8) == 0,
               "gemm_deep_fold: N=%d and the row pitches %ld / %ld must be multiples of four, the rows aligned", N, ldr, ldw);
    MV_REQUIRE(P == mv_gemm_deep_fold_parts(N), "gemm_deep_fold: %d partial sums a row, the launch makes %d", P, mv_gemm_deep_fold_parts(N));
    DeepArgs p{};
    p.A = (const bf16*)A; p.lda = lda; p.W = (const bf16*)W; p.bias = (const bf16*)bias;
    p.M = M; p.N = N; p.K = K;
    p.resid = resid; p.ldr = ldr; p.norm_weight = WeightPtr{norm_weight, norm_weight_dtype}; p.unit_offset = unit_offset;
    p.weighted = (bf16*)weighted; p.ldw = ldw; p.partial = partial; p.P = P;
    return deep_launch<DEEP_FOLD>("gemm_deep_fold", p, shape, stream);
}
