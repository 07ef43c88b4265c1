// A mixture's products over the chosen (token, expert) pairs only (bfloat16, MFMA; see moe.hip for what the mixture is),
// through the LDS ring of gemm_tile.hip: the rows of a tile are pairs of one expert, gathered by the addresses their loads
// take, so that a weight is read once for up to 160 pairs.
//
//   moe_pairs     lays the pairs out expert by expert (`sorted`: pair numbers, a pair is token * top + place; a shared expert
//                 that every token uses is one more expert, its pairs n * top + token) and cuts every expert's run into tiles
//                 of `rows` (`tile_expert`, `tile_row0`, `tile_rows`, `n_tiles` of them). Identity experts
//                 and pairs without an expert are left out. Within an expert the order of the pairs is whatever the counters
//                 gave; no result depends on it (a row's products read only its own row).
//   moe_tile<GATED>  act[pair] = weight[pair] * pair(x W_gate^T, x W_up^T), rounded once
//   moe_tile      out[pair] = act[pair] W_down^T as floats
//   moe_combine   y[token] = its places' out rows in order, the shared expert's, (identity weights) * x[token], added in float
//
// What bounds it: the bytes of the weights that were chosen, and how evenly tiles fill the compute units: 32 experts of 768 x 1024, 4 a
// token, are 151 MB, worth 30 us. With tiles of 128 x 128 and two workgroups a compute unit 1,000 tokens (125 pairs an expert, so every third
// expert had a second tile, nearly empty) beside a shared expert took 89 us a layer, 2,048 tokens 109, 500 62; with tiles of up to 160
// rows and 256 columns, one workgroup of eight waves a unit, chosen so that no round is nearly empty (mt_rows), and an activation of few
// instructions (GatedPair::of_short; alone 4 us of 89) 67.5, 97 and 56, of which 6 to 9 are moe_pairs and 5 to 8 the combination. Every
// expert for every token took 110 + 154 + 26 at 1,000. Eight rows: 47 us a layer with the routing against 55 (the unchosen experts' weights
// are not read).
#include "gemm_ring.h"

#include <cmath>

#define MT_MAX_E 1024

struct PairTables {
    int* sorted;
    int* tile_expert;
    int* tile_row0;
    int* tile_rows;
    int* n_tiles;
    int max_tiles;
};

// exclusive prefix sums of two numbers over the workgroup's 1024 threads; scratch holds 32 ints
__device__ __forceinline__ void mt_prefix(int& a, int& b, int* scratch) {
    const int lane = threadIdx.x % MV_WAVE, wave = threadIdx.x / MV_WAVE;
    int incl_a = a, incl_b = b;
#pragma unroll
    for (int o = 1; o < MV_WAVE; o <<= 1) {
        const int t = __shfl_up(incl_a, o, MV_WAVE), u = __shfl_up(incl_b, o, MV_WAVE);
        if (lane >= o) {
            incl_a += t;
            incl_b += u;
        }
    }
    if (lane == MV_WAVE - 1) {
        scratch[wave] = incl_a;
        scratch[16 + wave] = incl_b;
    }
    __syncthreads();
    int before_a = lane % 16 < wave ? scratch[lane % 16] : 0, before_b = lane % 16 < wave ? scratch[16 + lane % 16] : 0;
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) {
        before_a += __shfl_xor(before_a, o, MV_WAVE);
        before_b += __shfl_xor(before_b, o, MV_WAVE);
    }
    a = before_a + incl_a - a;
    b = before_b + incl_b - b;
}

// One workgroup; what bounds it is the number of waits one behind the other. A thread keeps its first MT_KEEP pairs: their experts are all
// asked for at once, and the count that a pair finds is its place in the expert's run, so that nothing is read or counted again. Pairs
// beyond are counted, and placed behind those, in a loop. 2,048 rows of 4 among 32 experts 7.5 us, here 6.2; 4,096 12.0 and 10.9; 2,048
// of 8 among 128 14.6 and 13.4; 1,000 and fewer alike, 3.6 to 5.5.
#define MT_KEEP 8
__global__ void __launch_bounds__(1024)
moe_pairs_kernel(const int* __restrict__ ids, int n_pairs, int n_real, int shared_pairs, int rows, PairTables t) {
    __shared__ int count[MT_MAX_E], start[MT_MAX_E], scratch[32];
    const int tid = threadIdx.x;
    int expert[MT_KEEP], place[MT_KEEP];
#pragma unroll
    for (int u = 0; u < MT_KEEP; ++u) expert[u] = ids[min(tid + 1024 * u, n_pairs - 1)];
    count[tid] = tid == n_real ? shared_pairs : 0;             // (n_real < MT_MAX_E)
    __syncthreads();
#pragma unroll
    for (int u = 0; u < MT_KEEP; ++u) {
        if (tid + 1024 * u >= n_pairs || expert[u] >= n_real) expert[u] = -1;
        place[u] = expert[u] >= 0 ? atomicAdd(&count[expert[u]], 1) : 0;
    }
    __syncthreads();
    const int kept = count[tid];
    if (n_pairs > 1024 * MT_KEEP) {
        __syncthreads();
        for (int p = tid + 1024 * MT_KEEP; p < n_pairs; p += 1024) {
            const int e = ids[p];
            if (e >= 0 && e < n_real) atomicAdd(&count[e], 1);
        }
        __syncthreads();
    }
    const int c = count[tid];
    int first = c, tile = (c + rows - 1) / rows;
    mt_prefix(first, tile, scratch);
    start[tid] = first;
    count[tid] = first + kept;                                 // (its own alone, which nobody else reads in front of the barrier)
    for (int r = 0; r < c && tile < t.max_tiles; r += rows, ++tile) {
        t.tile_expert[tile] = tid;
        t.tile_row0[tile] = first + r;
        t.tile_rows[tile] = min(rows, c - r);
    }
    if (tid == 1023) *t.n_tiles = tile;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < MT_KEEP; ++u)
        if (expert[u] >= 0) t.sorted[start[expert[u]] + place[u]] = tid + 1024 * u;
    for (int p = tid + 1024 * MT_KEEP; p < n_pairs; p += 1024) {
        const int e = ids[p];
        if (e >= 0 && e < n_real) t.sorted[atomicAdd(&count[e], 1)] = p;
    }
    for (int s = tid; s < shared_pairs; s += 1024) t.sorted[start[n_real] + s] = n_pairs + s;
}

struct MoeTileArgs {
    const bf16* A;                 // GATED: the tokens' rows; else the pairs' activations
    long lda;
    const bf16* W;                 // GATED: [E gate blocks of F rows | E up blocks | gate of the shared expert (FS rows) | its up]
    long ldw;                      // else: [N rows], the experts' F columns side by side, the shared expert's FS behind them
    PairTables t;
    const float* weights;          // GATED: of the pairs; a shared expert's weigh one
    int top, n_pairs, n_real, F, FS, N;
    bf16* act;                     // GATED: [pairs][ld_act]
    float* out;                    // else: [pairs][N]
    long ld_act;
    int K;                         // GATED: columns of W
    int tiles_n;
    GatedPair pair;
};

// Waves stand GM down the rows and GN along the columns, each with WM x WN products of 16 x 16.
template <int WM, int WN, int GM, int GN, bool GATED, int STAGES>
__global__ void __launch_bounds__(64 * GM * GN) __attribute__((amdgpu_waves_per_eu(2, 2)))
moe_tile_kernel(MoeTileArgs a) {
    constexpr int BM = 16 * WM * GM, BN = 16 * WN * GN, WAVES = GM * GN;
    constexpr int ROWS = BM + BN, INSTR = ROWS / 8, REPS = (INSTR + WAVES - 1) / WAVES, LEAST = INSTR / WAVES;
    static_assert((!GATED || WN % 2 == 0) && STAGES >= 2 && STAGES <= 4 && (STAGES - 2) * REPS <= 63, "");
    constexpr int STAGE = ROWS * 8;
    __shared__ uint4 ring[STAGES * STAGE];

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid / MV_WAVE);
    const int lane = tid % MV_WAVE, i = lane % 16, g = lane / 16;
    const int wm = wave / GN, wn = wave % GN;
    // An XCD walks a run of tiles with all their columns: an expert's tiles stand side by side, so its weights go into one L2.
    // The runs are cut from the tiles that there are, not from the most there could be (what the grid is sized for): so cut, the
    // last XCDs had none: 2,048 tokens, 32 experts, 4 a token 70.2 -> 53.6 us (gate and up), 42.2 -> 40.9 (down); 1,000 tokens
    // beside a shared expert 54 -> 53.5 and 38 -> 28; 64 rows beside one 66 -> 59 us a layer.
    const int total = *a.t.n_tiles * a.tiles_n, run = (total + GT_XCDS - 1) / GT_XCDS, at = blockIdx.x / GT_XCDS;
    const int id = blockIdx.x % GT_XCDS * run + at;
    if (at >= run || id >= total) return;
    const int tile = id / a.tiles_n, tn = id % a.tiles_n;
    const int expert = a.t.tile_expert[tile];
    const bool is_shared = expert == a.n_real;
    const int width = is_shared ? a.FS : a.F;                  // of the expert
    const int n_out = GATED ? width : a.N;
    const int n0 = tn * (GATED ? BN / 2 : BN);
    if (n0 >= n_out) return;
    const int row0 = a.t.tile_row0[tile], count = a.t.tile_rows[tile];
    const int n = (GATED ? a.K : width) / GT_KC;               // chunks

    const int lrow = lane / 8, piece = (lane % 8) ^ lrow;
    const char* src[REPS];
    int slot[REPS];
#pragma unroll
    for (int rep = 0; rep < REPS; ++rep) {
        const int j = wave + WAVES * rep, row = 8 * j + lrow;
        slot[rep] = j * 64;
        if (row < BM) {
            const int p = a.t.sorted[row0 + (row < count ? row : 0)];          // rows past the end: some pair; never stored
            const long row_of = GATED ? (p < a.n_pairs ? p / a.top : p - a.n_pairs) : p;
            src[rep] = reinterpret_cast<const char*>(a.A + row_of * a.lda + 8 * piece);
        } else {
            const int r = row - BM;
            long w;
            if (GATED) {
                const int c = r < BN / 2 ? n0 + r : n0 + (r - BN / 2);
                const long gate0 = is_shared ? 2L * a.n_real * a.F : (long)expert * a.F;
                const long up0 = is_shared ? gate0 + a.FS : (long)(a.n_real + expert) * a.F;
                w = ((r < BN / 2 ? gate0 : up0) + (c < width ? c : width - 1)) * a.ldw;
            } else {
                const int c = n0 + r;
                w = (long)(c < a.N ? c : a.N - 1) * a.ldw + (is_shared ? (long)a.n_real * a.F : (long)expert * a.F);
            }
            src[rep] = reinterpret_cast<const char*>(a.W + w + 8 * piece);
        }
    }
    auto fetch = [&](int c, uint4* stage) {
#pragma unroll
        for (int rep = 0; rep < REPS; ++rep)
            if (INSTR % WAVES == 0 || rep < LEAST || wave < INSTR % WAVES)
                gt_load_to_lds(src[rep] + (size_t)c * (GT_KC * sizeof(bf16)), (__attribute__((address_space(3))) void*)(stage + slot[rep]));
    };
    int a_off[WM], w_off[WN];
#pragma unroll
    for (int t = 0; t < WM; ++t) a_off[t] = (16 * (WM * wm + t) + i) * 8;
#pragma unroll
    for (int t = 0; t < WN; ++t) {
        int group;
        if (GATED) group = t < WN / 2 ? (WN / 2) * wn + t : (WN / 2) * (GN + wn) + (t - WN / 2);
        else group = WN * wn + t;
        w_off[t] = (BM + 16 * group + i) * 8;
    }
    const int sw0 = g ^ (i & 7), sw1 = (4 + g) ^ (i & 7);
    floatx4_t acc[WN][WM];
#pragma unroll
    for (int t = 0; t < WN; ++t)
#pragma unroll
        for (int u = 0; u < WM; ++u) acc[t][u] = floatx4_t{0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](const uint4* stage) {
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const int sw = ks ? sw1 : sw0;
            TFrag af[WM], wf[WN];
#pragma unroll
            for (int u = 0; u < WM; ++u) af[u].u = stage[a_off[u] + sw];
#pragma unroll
            for (int t = 0; t < WN; ++t) wf[t].u = stage[w_off[t] + sw];
#pragma unroll
            for (int t = 0; t < WN; ++t)
#pragma unroll
                for (int u = 0; u < WM; ++u)
                    acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[t].v, af[u].v, acc[t][u], 0, 0, 0);
        }
    };
    // the ring: see gemm_tile.hip. (The loads of `sorted` above have been waited for: addresses depend on them.)
#pragma unroll
    for (int k = 0; k < STAGES - 1; ++k)
        if (k < n) fetch(k, ring + k * STAGE);
    int st = 0, st_fetch = STAGES - 1;
    for (int k = 0; k < n; ++k) {
        const int later = n - k - 1 < STAGES - 2 ? n - k - 1 : STAGES - 2;
        // (a wave has LEAST or one more loads a chunk on their way; a wait for the fewer covers both)
        switch (later) {
            case 0: GT_WAIT_VMCNT(0); break;
            case 1: GT_WAIT_VMCNT(LEAST); break;
            default: GT_WAIT_VMCNT(2 * LEAST); break;
        }
        __builtin_amdgcn_s_barrier();
        if (k + STAGES - 1 < n) fetch(k + STAGES - 1, ring + st_fetch * STAGE);
        multiply(ring + st * STAGE);
        st = st + 1 == STAGES ? 0 : st + 1;
        st_fetch = st_fetch + 1 == STAGES ? 0 : st_fetch + 1;
    }
    // lane l holds C[pair row 16 u + l%16][weight row of tile t + 4 (l/16) + 0..3]
    constexpr int TOUT = GATED ? WN / 2 : WN;
#pragma unroll
    for (int u = 0; u < WM; ++u) {
        const int row = 16 * (WM * wm + u) + i;
        if (row >= count) continue;
        const int p = a.t.sorted[row0 + row];
        const float weight = !GATED || p >= a.n_pairs ? 1.f : a.weights[p];
#pragma unroll
        for (int t = 0; t < TOUT; ++t) {
            const int col = n0 + 16 * ((GATED ? WN / 2 : WN) * wn + t) + 4 * g;
            if (col >= n_out) continue;                        // (n_out is a multiple of four)
            if constexpr (GATED) {
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = weight * a.pair.of_short(acc[t][u][e], acc[t + WN / 2][u][e]);
                *reinterpret_cast<uint2*>(a.act + (size_t)p * a.ld_act + col) =
                    uint2{f32x2_to_bf16x2_bits(v[0], v[1]), f32x2_to_bf16x2_bits(v[2], v[3])};
            } else {
                *reinterpret_cast<float4*>(a.out + (size_t)p * a.N + col) = float4{acc[t][u][0], acc[t][u][1], acc[t][u][2], acc[t][u][3]};
            }
        }
    }
}

// four columns a thread (width a multiple of four, rows of x and y at addresses that four elements can be moved at)
__global__ void __launch_bounds__(256)
moe_pairs_combine_kernel(const float* __restrict__ out, const int* __restrict__ ids, int top, int n_pairs, int n_real, int shared,
                         const bf16* __restrict__ x, long ldx, const float* __restrict__ dense, int ld_dense, int identity,
                         bf16* __restrict__ y, long ldy, int width) {
    const int t = blockIdx.x;
    float idw = 0.f;
    for (int e = 0; e < identity; ++e) idw += dense[(size_t)t * ld_dense + n_real + e];
    for (int c = threadIdx.x * 4; c < width; c += 1024) {
        float4 v{0.f, 0.f, 0.f, 0.f};
        auto add = [&](size_t pair) {
            const float4 o = *reinterpret_cast<const float4*>(out + pair * width + c);
            v.x += o.x; v.y += o.y; v.z += o.z; v.w += o.w;
        };
        for (int k = 0; k < top; ++k) {
            const int e = ids[(size_t)t * top + k];
            if (e >= 0 && e < n_real) add((size_t)t * top + k);
        }
        if (shared) add((size_t)n_pairs + t);
        if (idw != 0.f) {
            const uint2 u = *reinterpret_cast<const uint2*>(x + (size_t)t * ldx + c);
            v.x = fmaf(idw, __uint_as_float(u.x << 16), v.x);
            v.y = fmaf(idw, __uint_as_float(u.x & 0xffff0000u), v.y);
            v.z = fmaf(idw, __uint_as_float(u.y << 16), v.z);
            v.w = fmaf(idw, __uint_as_float(u.y & 0xffff0000u), v.w);
        }
        *reinterpret_cast<uint2*>(y + (size_t)t * ldy + c) = uint2{f32x2_to_bf16x2_bits(v.x, v.y), f32x2_to_bf16x2_bits(v.z, v.w)};
    }
}

template <bool GATED>
static int launch_moe_tiles(MoeTileArgs& a, int wm, int columns, hipStream_t stream) {
    const int n_out = GATED ? (a.F > a.FS ? a.F : a.FS) : a.N, bn = columns / (GATED ? 2 : 1);
    a.tiles_n = (n_out + bn - 1) / bn;
    const long blocks = ((long)a.t.max_tiles * a.tiles_n + GT_XCDS - 1) / GT_XCDS * GT_XCDS;
    MV_REQUIRE(blocks < (1L << 31), "moe_tile: too many tiles");
#define MT_LAUNCH(WM, WN, GN, STAGES) \
    hipLaunchKernelGGL((moe_tile_kernel<WM, WN, 2, GN, GATED, STAGES>), dim3((unsigned)blocks), dim3(128 * GN), 0, stream, a)
    if (columns == 256) {
        if (wm == 1) MT_LAUNCH(1, 4, 4, 4);
        else if (wm == 2) MT_LAUNCH(2, 4, 4, 4);
        else if (wm == 3) MT_LAUNCH(3, 4, 4, 3);
        else if (wm == 4) MT_LAUNCH(4, 4, 4, 3);
        else MT_LAUNCH(5, 4, 4, 3);
    } else if (columns == 64) MT_LAUNCH(1, 2, 2, 4);
    else if (wm == 1) MT_LAUNCH(1, 4, 2, 4);
    else if (wm == 2) MT_LAUNCH(2, 4, 2, 3);
    else if (wm == 3) MT_LAUNCH(3, 4, 2, 2);
    else if (wm == 4) MT_LAUNCH(4, 4, 2, 2);
    else MT_LAUNCH(5, 4, 2, 2);
#undef MT_LAUNCH
    return mv_check_launch("moe_tile");
}

// Tiles of `rows` pairs that `experts` runs of `mean` pairs on average have in all: a run's length taken as normal around its mean, a
// third wider than dice would make it.
static double mt_tiles(int experts, double mean, int rows) {
    const double width = 1.3 * sqrt(mean) * 1.41421356;
    double tiles = 0;
    for (int k = 0; k * (double)rows < mean + 5 * width; ++k) tiles += 0.5 * erfc((k * (double)rows + 0.5 - mean) / width);
    return experts * (tiles < mean ? tiles : mean);
}

// Columns of a tile (W's rows) where a product has so many tiles of rows and columns: 256, one workgroup of eight waves a compute unit,
// where those find work for more than half of the units; else 128, two workgroups of four waves each.
static int mt_columns(double row_tiles, int n_out, int halves, int units) {
    return row_tiles * ((n_out * halves + 255) / 256) >= 0.55 * units ? 256 : 128;
}

// Rows of a tile, in 32s. A tile takes as long as its operands take through its compute unit, 77 KB a us: (rows + columns) * 128 bytes a
// chunk of 64 columns of K; tiles come in rounds; and the weights come from memory whatever the tiles. Of 1 to 5 the one with the least
// sum over both products: 1.5 % behind the best of all shapes on average over 98 mixtures (0.25 to 512 pairs an expert, 8 to 128 experts, 256 x 512
// to 1536 x 4096), the worst one 13 %, where rounds are estimated nearly even (8 experts of 1024 x 2048, 2 a token, and a shared one, 2,048 tokens:
// 160 rows 149 us, 128 rows 132). 32 experts of 768 x 1024, 4 a token, and a shared one: 256 tokens tiles of 64
// rows 50 us, of 128 55; 1,000 tokens (125 pairs an expert) 160 rows 66.5, 128 rows 78, the last tiles of the experts with more than 128
// being a round of their own; 1,500 tokens 128 rows 96, 160 rows 103; 2,048 tokens 160 rows 112, 128 rows 118.
static int mt_rows(int n, long n_pairs, int n_real, int hidden, int F, int FS, int units) {
    const double mean = (double)n_pairs / n_real, used = n_pairs < n_real ? n_pairs : n_real;
    int best = 1;
    double least = 0;
    for (int wm = 1; wm <= 5; ++wm) {
        const int rows = 32 * wm;
        const double tiles = mt_tiles(n_real, mean, rows) + (FS ? (n + rows - 1) / rows : 0);
        double cost = 0;
        for (int gated = 0; gated < 2; ++gated) {
            const int K = gated ? hidden : F, n_out = gated ? (F > FS ? F : FS) : hidden;
            const int columns = mt_columns(tiles, n_out, gated ? 2 : 1, units);
            const double rounds = tiles * ((n_out * (gated ? 2 : 1) + columns - 1) / columns) / units;
            const double whole = fmax(1.0, 0.5 * (rounds + ceil(rounds)));
            const double port = whole * (rows + columns + (columns == 256 ? 100 : 150)) * (K / 64.0) * 128 / 77e3;
            const double memory = (used * F + FS) * hidden * (gated ? 4.0 : 2.0) / 6.2e6;
            cost += fmax(port, memory) + 0.3 * fmin(port, memory);
        }
        if (wm == 1 || cost < least) {
            best = wm;
            least = cost;
        }
    }
    return best;
}

// The same where the rows of a tile are known. Tiles of up to 64 rows wait for the weights: there a workgroup to itself has less on its way
// at the ends of a long K, and a second round that few units have costs as much as the first; the smaller tiles share units and end more
// evenly. us, with 256 columns / 128: 64 experts of 768 x 2048, 8 a token, 8 rows 135 / 118, 64 rows 157 / 143; 128 of 384 x 1024, 33 rows 73 / 66; 16 of
// 1536 x 4096, 2 a token, 256 rows 150 / 141. One round of short tiles stays wide: 32 of 768 x 1024 beside a shared one, 100 rows 45 / 48.
static int mt_columns_of(int wm, double row_tiles, int n_out, int halves, int K, int units) {
    const double wide = row_tiles * ((n_out * halves + 255) / 256);
    return wm <= 2 && (wide > units || K > 1024) ? 128 : mt_columns(row_tiles, n_out, halves, units);
}

struct MtShape {
    int wm, in, down;          // rows of a tile in 32s, columns of a tile of the first product and of the second
};
static MtShape mt_shape(int n, int top, int n_real, int hidden, int F, int FS, int units) {
    const long n_pairs = (long)n * top, busy = n_pairs < n_real ? n_pairs : n_real;      // tiles, at most, of a step of few rows
    const int wm = mt_rows(n, n_pairs, n_real, hidden, F, FS, units), rows = 32 * wm;
    const double tiles = mt_tiles(n_real, (double)n_pairs / n_real, rows) + (FS ? (n + rows - 1) / rows : 0);
    // (a step of few rows whose tiles leave compute units idle has narrow ones)
    return MtShape{wm, wm == 1 && busy * ((F + 63) / 64) < units ? 64 : mt_columns_of(wm, tiles, F > FS ? F : FS, 2, hidden, units),
                   wm == 1 && busy * ((hidden + 127) / 128) < units ? 64 : mt_columns_of(wm, tiles, hidden, 1, F, units)};
}
// rows | columns << 10 | columns of the second product << 20 of the tiles that mv_moe_pairs has on a device of so many compute units
extern "C" int mv_moe_pairs_shape(int n, int top, int n_real, int hidden, int F, int FS, int units) {
    const MtShape s = mt_shape(n, top, n_real, hidden, F, FS, units);
    return 32 * s.wm | s.in << 10 | s.down << 20;
}

// ints of scratch: sorted pairs, the three tile tables, for tiles of 32 rows, and the number of tiles
extern "C" long mv_moe_pairs_ints(int n, int top, int n_real, int shared) {
    const long pairs = (long)n * (top + (shared ? 1 : 0));
    return pairs + 3L * (pairs / 32 + n_real + 2);
}

// y[t] = sum over t's chosen experts of weight * down_e(pair(gate_e x, up_e x)) + the shared expert's (FS > 0) + (identity weights) * x[t].
// act: bf16 [pairs][max(F, FS)], out: float [pairs][hidden] with pairs = n * top, and n more with a shared expert.
// Returns 2 (nothing done) for sizes it does not serve.
extern "C" int mv_moe_pairs(const void* x, long ldx, int n, int hidden, const void* w_gate_up, const void* w_down, int n_real,
                            int identity, int F, int FS, const int* ids, const float* weights, int top, const float* dense, int ld_dense,
                            int* ints, void* act, float* out, void* y, long ldy, float limit, float slope, hipStream_t stream) {
    MV_REQUIRE(n >= 0 && hidden > 0 && n_real > 0 && F > 0 && FS >= 0 && top > 0 && identity >= 0 && limit >= 0.f, "moe_pairs: bad sizes");
    if (hidden % GT_KC || F % GT_KC || FS % GT_KC || ldx % 8 || ldy % 4 || (uintptr_t)x % 16 || (uintptr_t)y % 8 || (uintptr_t)w_gate_up % 16
        || (uintptr_t)w_down % 16 || (uintptr_t)act % 16 || (uintptr_t)out % 16 || n_real >= MT_MAX_E)
        return 2;
    MV_REQUIRE(x && w_gate_up && w_down && ids && weights && ints && act && out && y && ldx >= hidden && ldy >= hidden
               && (identity == 0 || (dense && ld_dense >= n_real + identity)), "moe_pairs: missing operand");
    if (n == 0) return 0;
    const long n_pairs = (long)n * top, pairs = n_pairs + (FS ? n : 0);
    MV_REQUIRE(pairs < (1L << 30), "moe_pairs: too many pairs");
    const MtShape shape = mt_shape(n, top, n_real, hidden, F, FS, mv_compute_units());
    const int rows = 32 * shape.wm;
    PairTables t;
    t.max_tiles = (int)(pairs / rows + (n_real < n_pairs ? n_real : n_pairs) + 1);
    t.sorted = ints;
    t.tile_expert = ints + pairs;
    t.tile_row0 = t.tile_expert + t.max_tiles;
    t.tile_rows = t.tile_row0 + t.max_tiles;
    t.n_tiles = t.tile_rows + t.max_tiles;
    hipLaunchKernelGGL(moe_pairs_kernel, dim3(1), dim3(1024), 0, stream, ids, (int)n_pairs, n_real, FS ? n : 0, rows, t);
    if (mv_check_launch("moe_pairs")) return 1;
    MoeTileArgs a{(const bf16*)x, ldx, (const bf16*)w_gate_up, (long)hidden, t, weights, top, (int)n_pairs, n_real, F, FS, hidden,
                  (bf16*)act, out, (long)(F > FS ? F : FS), hidden, 0, GatedPair{limit, slope}};
    if (launch_moe_tiles<true>(a, shape.wm, shape.in, stream)) return 1;
    a.A = (const bf16*)act;
    a.lda = a.ld_act;
    a.W = (const bf16*)w_down;
    a.ldw = (long)n_real * F + FS;
    if (launch_moe_tiles<false>(a, shape.wm, shape.down, stream)) return 1;
    hipLaunchKernelGGL(moe_pairs_combine_kernel, dim3(n), dim3(256), 0, stream, out, ids, top, (int)n_pairs, n_real, FS ? 1 : 0, (const bf16*)x,
                       ldx, dense, ld_dense, identity, (bf16*)y, ldy, hidden);
    return mv_check_launch("moe_pairs_combine");
}
