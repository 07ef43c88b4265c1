// C[M, N] = A[M, K] * W[N, K]^T (+ bias[N]) with float operands and float accumulation in a fixed order.
//
// This is the exact matrix product of the engine: every output element is the sum of GF_WAVES partial sums, partial w over
// the blocks of 16 values of k whose number is w modulo GF_WAVES, in the order of k, added pairwise at the end; whatever M
// is and wherever the row lies in the batch, so a row's result never depends on what else is in the step. It serves the
// float32 path entirely, and the bfloat16 path wherever a weight is stored in float or no faster kernel takes the shape.
// Inputs are converted to float on load (exact for bf16) and multiplied as floats (v_mfma_f32_16x16x4_f32); there is no
// reduced-precision mode.
//
// What bounds it: the float matrix unit (256 flops a cycle and compute unit) where M is large, the bytes of W where it is
// small. A wave of 16x16x4 products needs an operand value only once in 8 cycles, so the operands come straight from the
// caches into registers, a block ahead of the products, without LDS (gemm_nt_kernel), or through an LDS ring where rows and K
// allow whole lines (gemm_nt_ring_kernel); the waves of a workgroup split K instead of the tile, so that a few hundred rows
// against a narrow weight still give every compute unit a tile with eight waves on it.
// Measured (float, us at 224 rows; a 64x64 tile of scalar multiply-adds a workgroup -> registers -> ring): N x K of 1024 x 2048
// 405 -> 23 -> 13.5, 1024 x 3072 405 -> 30 -> 19, 4096 x 1024 164 -> 35 -> 24, 6144 x 1024 169 -> 54 -> 36; at 1,024 rows
// 24576 x 4096 runs at 127 TFLOP/s, where a large library product reaches 135.
#include "gemm_ring.h"

typedef float gf_acc_t __attribute__((ext_vector_type(4)));

#define GF_WAVES 8                  // of a workgroup; they split K

// four neighbours of a row from k on; beyond K (TAIL) zeros
template <typename T, bool VEC, bool TAIL>
__device__ __forceinline__ float4 gf_load(const T* __restrict__ row, int k, int K) {
    if constexpr (VEC && !TAIL) {
        if constexpr (sizeof(T) == 4) {
            return *reinterpret_cast<const float4*>(row + k);
        } else {
            const uint2 u = *reinterpret_cast<const uint2*>(row + k);
            return float4{__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u), __uint_as_float(u.y << 16),
                          __uint_as_float(u.y & 0xffff0000u)};
        }
    } else if constexpr (!TAIL) {
        return float4{to_f(row[k]), to_f(row[k + 1]), to_f(row[k + 2]), to_f(row[k + 3])};
    } else {
        if constexpr (VEC) {
            if (K % 4 == 0) {                        // all four or none
                const float4 v = gf_load<T, true, false>(row, k < K ? k : 0, K);
                return k < K ? v : float4{0.f, 0.f, 0.f, 0.f};
            }
        }
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float x = to_f(row[k + e < K ? k + e : 0]);
            v[e] = k + e < K ? x : 0.f;
        }
        return float4{v[0], v[1], v[2], v[3]};
    }
}

template <typename TW, typename TC, int RM, int RN>
__device__ __forceinline__ void gf_store(const gf_acc_t (&acc)[RM][RN], const TW* __restrict__ bias, TC* __restrict__ C, long ldc, int m0,
                                         int n0, int i, int g, int M, int N) {
#pragma unroll
    for (int c = 0; c < RN; ++c) {
        const int n = n0 + 16 * c + i;
        if (n >= N) continue;
        const float add = bias ? to_f(bias[n]) : 0.f;
#pragma unroll
        for (int r = 0; r < RM; ++r)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int m = m0 + 16 * r + 4 * g + e;
                if (m < M) C[(size_t)m * ldc + n] = from_f<TC>(bias ? acc[r][c][e] + add : acc[r][c][e]);
            }
    }
}

// RM x RN: tiles of 16 rows and 16 columns a workgroup. VEC: rows of both operands start at addresses that four elements
// can be loaded from at once.
template <typename TA, typename TW, typename TC, int RM, int RN, int AHEAD, bool VEC>
__global__ void __launch_bounds__(64 * GF_WAVES)
gemm_nt_kernel(const TA* __restrict__ A, long lda, const TW* __restrict__ W, long ldw, const TW* __restrict__ bias,
               TC* __restrict__ C, long ldc, int M, int N, int K) {
    __shared__ gf_acc_t part[GF_WAVES / 2][RM * RN][64];
    const int lane = threadIdx.x % MV_WAVE, wave = threadIdx.x / MV_WAVE, i = lane % 16, g = lane / 16;
    const int m0 = blockIdx.y * (16 * RM), n0 = blockIdx.x * (16 * RN);
    const TA* a_row[RM];
    const TW* w_row[RN];
#pragma unroll
    for (int r = 0; r < RM; ++r) a_row[r] = A + (size_t)min(m0 + 16 * r + i, M - 1) * lda;      // (rows beyond the last are not stored)
#pragma unroll
    for (int c = 0; c < RN; ++c) w_row[c] = W + (size_t)min(n0 + 16 * c + i, N - 1) * ldw;
    gf_acc_t acc[RM][RN];
#pragma unroll
    for (int r = 0; r < RM; ++r)
#pragma unroll
        for (int c = 0; c < RN; ++c) acc[r][c] = gf_acc_t{0.f, 0.f, 0.f, 0.f};
    float4 a[RM], w[RN];
    // a lane takes four neighbours in k for four products; they then sum over k in another order, the same for both operands
    auto products = [&]() {
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int r = 0; r < RM; ++r)
#pragma unroll
                for (int c = 0; c < RN; ++c)
                    acc[r][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(reinterpret_cast<const float*>(&a[r])[e],
                                                                     reinterpret_cast<const float*>(&w[c])[e], acc[r][c], 0, 0, 0);
    };
    const int whole = K / 16;                        // blocks of 16; the wave's own: wave, wave + GF_WAVES, ...
    float4 an[AHEAD][RM], wn[AHEAD][RN];
    auto fetch = [&](int d, int b) {                 // (always issued, from a block that exists)
        const int k = 16 * (b < whole ? b : 0) + 4 * g;
#pragma unroll
        for (int r = 0; r < RM; ++r) an[d][r] = gf_load<TA, VEC, false>(a_row[r], k, K);
#pragma unroll
        for (int c = 0; c < RN; ++c) wn[d][c] = gf_load<TW, VEC, false>(w_row[c], k, K);
    };
    if (whole > 0) {
#pragma unroll
        for (int d = 0; d < AHEAD; ++d)
            if (VEC || wave + d * GF_WAVES < whole) fetch(d, wave + d * GF_WAVES);       // (a scalar form has loads to spare)
    }
    for (int b0 = wave; b0 < whole; b0 += AHEAD * GF_WAVES) {
#pragma unroll
        for (int d = 0; d < AHEAD; ++d) {
            const int b = b0 + d * GF_WAVES;
            if (b < whole) {
#pragma unroll
                for (int r = 0; r < RM; ++r) a[r] = an[d][r];
#pragma unroll
                for (int c = 0; c < RN; ++c) w[c] = wn[d][c];
                if (VEC || b + AHEAD * GF_WAVES < whole) fetch(d, b + AHEAD * GF_WAVES);      // flies under the products of the blocks between
                products();
            }
        }
    }
    if (K % 16 != 0 && whole % GF_WAVES == wave) {
#pragma unroll
        for (int r = 0; r < RM; ++r) a[r] = gf_load<TA, VEC, true>(a_row[r], 16 * whole + 4 * g, K);
#pragma unroll
        for (int c = 0; c < RN; ++c) w[c] = gf_load<TW, VEC, true>(w_row[c], 16 * whole + 4 * g, K);
        products();
    }
    // the waves' sums, pairwise: 4..7 into 0..3, 2..3 into 0..1, 1 into 0
#pragma unroll
    for (int half = GF_WAVES / 2; half >= 1; half /= 2) {
        if (K <= 16 * half) continue;                // (they hold zeros, which change no sum)
        if (wave >= half && wave < 2 * half)
#pragma unroll
            for (int t = 0; t < RM * RN; ++t) part[wave - half][t][lane] = acc[t / RN][t % RN];
        __syncthreads();
        if (wave < half)
#pragma unroll
            for (int t = 0; t < RM * RN; ++t) acc[t / RN][t % RN] += part[wave][t][lane];
        __syncthreads();
    }
    if (wave == 0) gf_store<TW, TC, RM, RN>(acc, bias, C, ldc, m0, n0, i, g, M, N);
}

// The same sums again for float operands with more than 16 rows and a K of whole chunks: the operands come through a ring of LDS
// stages. A chunk is 128 values of k, a block for each of the eight waves, so a row's 512 bytes are loaded as whole lines, and
// once for all waves. (Straight into registers, a load touches sixteen half lines of 64 bytes. A compute unit asks its cache for
// about one line in four cycles, and that, not the matrix unit, was what a tile took.)
// A workgroup has a compute unit to itself and walks its tiles without a pause in the loads: the stream of chunks goes on into
// the next tile while the sums of this one are added up. A wave has the operands of its next block in registers before the
// products of the current one, so that reading LDS costs the matrix unit nothing.
// LDS: rows of 512 bytes, 16-byte piece p of row r in place p ^ (r & 15): sixteen lanes that read one piece of sixteen rows
// meet in no bank.
template <int RM, int RN, int STAGES>
struct RingShape {
    static constexpr int ROWS = 16 * (RM + RN), LOADS = RM + RN;       // load instructions (two rows each) of a wave and chunk
    static constexpr int TILES = RM * RN, LEFT = 160 * 1024 - STAGES * ROWS * 512;
    static constexpr int PASS = LEFT / 8192 >= TILES ? TILES : LEFT / 8192 >= TILES / 2 ? TILES / 2 : TILES / 4;   // tiles added up at a time
    static_assert(PASS >= 1 && PASS * 8192 <= LEFT && TILES % PASS == 0, "the sums of a pass fit beside the ring");
};

template <int RM, int RN, int STAGES>
__global__ void __launch_bounds__(64 * GF_WAVES)
gemm_nt_ring_kernel(const float* __restrict__ A, long lda, const float* __restrict__ W, long ldw, const float* __restrict__ bias,
                    float* __restrict__ C, long ldc, int M, int N, int K, int m_tiles, int tiles) {
    typedef RingShape<RM, RN, STAGES> S;
    __shared__ uint4 ring[STAGES][S::ROWS][32];
    __shared__ float part[GF_WAVES][S::PASS][4][MV_WAVE];
    const int lane = threadIdx.x % MV_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / MV_WAVE), i = lane % 16, g = lane / 16;
    // workgroups go to the XCDs in turn: an XCD walks neighbouring tiles, which share weight rows (row tiles follow each other)
    const int xcd = blockIdx.x % GT_XCDS, step = gridDim.x / GT_XCDS;
    const int first = (int)((long)tiles * xcd / GT_XCDS) + blockIdx.x / GT_XCDS, end = (int)((long)tiles * (xcd + 1) / GT_XCDS);
    if (first >= end) return;
    const int chunks = K / 128, total = (end - first + step - 1) / step * chunks;

    const float* src[S::LOADS];                      // this lane's place in the rows that it brings in
    int f_tile = first, f_chunk = 0, f_count = 0;
    auto point = [&]() __attribute__((always_inline)) {
        const int m0 = f_tile % m_tiles * (16 * RM), n0 = f_tile / m_tiles * (16 * RN);
#pragma unroll
        for (int j = 0; j < S::LOADS; ++j) {
            const int r = 2 * (wave * S::LOADS + j) + lane / 32, piece = lane % 32 ^ (r & 15);
            const float* row = r < 16 * RM ? A + (size_t)min(m0 + r, M - 1) * lda : W + (size_t)min(n0 + r - 16 * RM, N - 1) * ldw;
            src[j] = row + 4 * piece;
        }
    };
    point();
    auto fetch = [&](int stage) __attribute__((always_inline)) {         // the next chunk of the stream; behind its end the last one again
#pragma unroll
        for (int j = 0; j < S::LOADS; ++j)
            gt_load_to_lds(src[j], (__attribute__((address_space(3))) void*)&ring[stage][2 * (wave * S::LOADS + j)][0]);
        if (++f_count >= total) return;
        if (++f_chunk == chunks) {
            f_chunk = 0;
            f_tile += step;
            point();
        } else {
#pragma unroll
            for (int j = 0; j < S::LOADS; ++j) src[j] += 128;
        }
    };
    float4 a[2][RM], w[2][RN];
    auto take = [&](int stage, int to) __attribute__((always_inline)) {
        const int slot = (4 * wave + g) ^ i;
#pragma unroll
        for (int r = 0; r < RM; ++r) a[to][r] = *reinterpret_cast<const float4*>(&ring[stage][16 * r + i][slot]);
#pragma unroll
        for (int c = 0; c < RN; ++c) w[to][c] = *reinterpret_cast<const float4*>(&ring[stage][16 * (RM + c) + i][slot]);
    };
    gf_acc_t acc[RM][RN];
    auto clear = [&]() {
#pragma unroll
        for (int r = 0; r < RM; ++r)
#pragma unroll
            for (int c = 0; c < RN; ++c) acc[r][c] = gf_acc_t{0.f, 0.f, 0.f, 0.f};
    };
    clear();
    // a wave's own loads have landed but for the newest LEFT chunks', and what it read of LDS has arrived; then the same for all waves
#define GF_MEET(LEFT)                                                                                               \
    do {                                                                                                            \
        __builtin_amdgcn_s_waitcnt(0x0070 | (((LEFT) * S::LOADS) & 15) | ((((LEFT) * S::LOADS) >> 4) << 14));       \
        asm volatile("s_barrier" ::: "memory");                                                                     \
    } while (0)
#pragma unroll
    for (int s = 0; s < STAGES; ++s) fetch(s);
    GF_MEET(STAGES - 1);
    take(0, 0);
    int tile = first, chunk = 0, stage = 0;
    auto turn = [&](int cur) __attribute__((always_inline)) {
        // the stage of this chunk is in registers everywhere behind the barrier: the stream goes on into it, between products
        // (a load holds up the instructions behind it, and the matrix unit would wait for all of them)
        GF_MEET(STAGES - 2);
        const int free = stage;
        if (++stage == STAGES) stage = 0;
        auto products = [&](int e) __attribute__((always_inline)) {
#pragma unroll
            for (int r = 0; r < RM; ++r)
#pragma unroll
                for (int c = 0; c < RN; ++c)
                    acc[r][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(reinterpret_cast<const float*>(&a[cur][r])[e],
                                                                     reinterpret_cast<const float*>(&w[cur][c])[e], acc[r][c], 0, 0, 0);
        };
        products(0);
        fetch(free);
        products(1);
        take(stage, 1 - cur);
        products(2);
        products(3);
        if (++chunk < chunks) return;
        // the waves' sums, added pairwise as above; every thread adds up one element (or a few) of a pass
        const int m0 = tile % m_tiles * (16 * RM), n0 = tile / m_tiles * (16 * RN);
#pragma unroll
        for (int pass = 0; pass < S::TILES / S::PASS; ++pass) {
#pragma unroll
            for (int t = 0; t < S::PASS; ++t)
#pragma unroll
                for (int e = 0; e < 4; ++e) part[wave][t][e][lane] = acc[(pass * S::PASS + t) / RN][(pass * S::PASS + t) % RN][e];
            __builtin_amdgcn_s_waitcnt(0xc07f);      // (LDS alone)
            asm volatile("s_barrier" ::: "memory");
#pragma unroll
            for (int u = 0; u < S::PASS * 4; u += GF_WAVES) {
                if (S::PASS * 4 < GF_WAVES && wave >= S::PASS * 4) break;
                const int t = (u + wave) / 4, e = (u + wave) % 4, at = pass * S::PASS + t;
                float p[GF_WAVES];
#pragma unroll
                for (int v = 0; v < GF_WAVES; ++v) p[v] = part[v][t][e][lane];
                float sum = ((p[0] + p[4]) + (p[2] + p[6])) + ((p[1] + p[5]) + (p[3] + p[7]));
                const int m = m0 + 16 * (at / RN) + 4 * g + e, n = n0 + 16 * (at % RN) + i;
                if (m < M && n < N) C[(size_t)m * ldc + n] = bias != nullptr ? sum + bias[n] : sum;
            }
            __builtin_amdgcn_s_waitcnt(0xc07f);
            asm volatile("s_barrier" ::: "memory");
        }
        clear();
        chunk = 0;
        tile += step;
    };
    for (int c = 0; c < total; c += 2) {
        turn(0);
        if (c + 1 < total) turn(1);
    }
    __builtin_amdgcn_s_waitcnt(0x0070);              // nothing is on its way into LDS any more
#undef GF_MEET
}

// The same sums, all GF_WAVES of a tile by one wave one after the other: for products of many rows and a short K, where a
// split leaves every wave a block or two and one of eight the tile's output (4096 x 1024 x 16: 28 us -> 10).
template <typename TA, typename TW, typename TC, int RM, int RN, bool VEC>
struct WaveTile {
    const TA* a_row[RM];
    const TW* w_row[RN];
    int K, g;
    struct Sums { gf_acc_t t[RM][RN]; };

    template <bool TAIL>
    __device__ __forceinline__ void add(Sums& s, int b) const {
        float4 a[RM], w[RN];
#pragma unroll
        for (int r = 0; r < RM; ++r) a[r] = gf_load<TA, VEC, TAIL>(a_row[r], 16 * b + 4 * g, K);
#pragma unroll
        for (int c = 0; c < RN; ++c) w[c] = gf_load<TW, VEC, TAIL>(w_row[c], 16 * b + 4 * g, K);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int r = 0; r < RM; ++r)
#pragma unroll
                for (int c = 0; c < RN; ++c)
                    s.t[r][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(reinterpret_cast<const float*>(&a[r])[e],
                                                                     reinterpret_cast<const float*>(&w[c])[e], s.t[r][c], 0, 0, 0);
    }
    // partial sums FIRST, FIRST + STEP, ..., added up as the waves' are
    template <int FIRST, int STEP>
    __device__ __forceinline__ void sum(Sums& s) const {
        if constexpr (STEP == GF_WAVES) {
#pragma unroll
            for (int r = 0; r < RM; ++r)
#pragma unroll
                for (int c = 0; c < RN; ++c) s.t[r][c] = gf_acc_t{0.f, 0.f, 0.f, 0.f};
            const int whole = K / 16;
            int b = FIRST;
            for (; b < whole; b += GF_WAVES) add<false>(s, b);
            if (b == whole && K % 16 != 0) add<true>(s, b);
        } else {
            sum<FIRST, 2 * STEP>(s);
            if (16 * (FIRST + STEP) < K) {           // (the others are zero)
                Sums o;
                sum<FIRST + STEP, 2 * STEP>(o);
#pragma unroll
                for (int r = 0; r < RM; ++r)
#pragma unroll
                    for (int c = 0; c < RN; ++c) s.t[r][c] += o.t[r][c];
            }
        }
    }
};

template <typename TA, typename TW, typename TC, int RM, int RN, bool VEC>
__global__ void __launch_bounds__(256)
gemm_nt_wave_kernel(const TA* __restrict__ A, long lda, const TW* __restrict__ W, long ldw, const TW* __restrict__ bias,
                    TC* __restrict__ C, long ldc, int M, int N, int K) {
    const int lane = threadIdx.x % MV_WAVE, i = lane % 16, g = lane / 16;
    const int m0 = (blockIdx.y * 4 + threadIdx.x / MV_WAVE) * (16 * RM), n0 = blockIdx.x * (16 * RN);
    if (m0 >= M) return;
    WaveTile<TA, TW, TC, RM, RN, VEC> tile;
    tile.K = K;
    tile.g = g;
#pragma unroll
    for (int r = 0; r < RM; ++r) tile.a_row[r] = A + (size_t)min(m0 + 16 * r + i, M - 1) * lda;
#pragma unroll
    for (int c = 0; c < RN; ++c) tile.w_row[c] = W + (size_t)min(n0 + 16 * c + i, N - 1) * ldw;
    typename WaveTile<TA, TW, TC, RM, RN, VEC>::Sums s;
    tile.template sum<0, 1>(s);
    gf_store<TW, TC, RM, RN>(s.t, bias, C, ldc, m0, n0, i, g, M, N);
}

template <typename TA, typename TW, typename TC, int RM, int RN, int AHEAD>
static void launch_tiles(const void* A, long lda, const void* W, long ldw, const void* bias, void* C, long ldc, int M, int N, int K,
                         hipStream_t stream) {
    const bool vec = lda % 4 == 0 && ldw % 4 == 0 && (uintptr_t)A % (4 * sizeof(TA)) == 0 && (uintptr_t)W % (4 * sizeof(TW)) == 0;
    dim3 grid((N + 16 * RN - 1) / (16 * RN), (M + 16 * RM - 1) / (16 * RM));
    if (vec)
        hipLaunchKernelGGL((gemm_nt_kernel<TA, TW, TC, RM, RN, AHEAD, true>), grid, dim3(64 * GF_WAVES), 0, stream, (const TA*)A, lda,
                           (const TW*)W, ldw, (const TW*)bias, (TC*)C, ldc, M, N, K);
    else
        hipLaunchKernelGGL((gemm_nt_kernel<TA, TW, TC, RM, RN, AHEAD, false>), grid, dim3(64 * GF_WAVES), 0, stream, (const TA*)A, lda,
                           (const TW*)W, ldw, (const TW*)bias, (TC*)C, ldc, M, N, K);
}

template <int RM, int RN, int STAGES>
static void launch_ring(const void* A, long lda, const void* W, long ldw, const void* bias, void* C, long ldc, int M, int N, int K,
                        hipStream_t stream) {
    const int m_tiles = (M + 16 * RM - 1) / (16 * RM), n_tiles = (N + 16 * RN - 1) / (16 * RN), tiles = m_tiles * n_tiles;   // (below 2^31)
    const int most = mv_compute_units() / GT_XCDS, share = (tiles + GT_XCDS - 1) / GT_XCDS;
    const int each = share < most ? share : most > 0 ? most : 1;                   // workgroups of an XCD
    hipLaunchKernelGGL((gemm_nt_ring_kernel<RM, RN, STAGES>), dim3(each * GT_XCDS), dim3(64 * GF_WAVES), 0, stream, (const float*)A, lda,
                       (const float*)W, ldw, (const float*)bias, (float*)C, ldc, M, N, K, m_tiles, tiles);
}

template <typename TA, typename TW, typename TC, int RM, int RN>
static void launch_waves(const void* A, long lda, const void* W, long ldw, const void* bias, void* C, long ldc, int M, int N, int K,
                         hipStream_t stream) {
    const bool vec = lda % 4 == 0 && ldw % 4 == 0 && (uintptr_t)A % (4 * sizeof(TA)) == 0 && (uintptr_t)W % (4 * sizeof(TW)) == 0;
    dim3 grid((N + 16 * RN - 1) / (16 * RN), (M + 64 * RM - 1) / (64 * RM));
    if (vec)
        hipLaunchKernelGGL((gemm_nt_wave_kernel<TA, TW, TC, RM, RN, true>), grid, dim3(256), 0, stream, (const TA*)A, lda, (const TW*)W, ldw,
                           (const TW*)bias, (TC*)C, ldc, M, N, K);
    else
        hipLaunchKernelGGL((gemm_nt_wave_kernel<TA, TW, TC, RM, RN, false>), grid, dim3(256), 0, stream, (const TA*)A, lda, (const TW*)W, ldw,
                           (const TW*)bias, (TC*)C, ldc, M, N, K);
}

// The tile of float operands that go through the ring, in sixteens (rows x columns: 22, 24 or 44), 0: they don't. Rows that start at
// 16-byte addresses and a K of whole chunks of 128 do, from 17 rows on, and
// below that where the columns give half of the compute units a tile (us, registers / ring: 16 x 4096 x 1024 10.4 / 8.2,
// 16 x 151936 x 1024 195 / 123; but 1 x 1024 x 3072 13.1 / 16.5, 16 x 1024 x 3072 16.8 / 16.7). Its tile is the one whose rounds
// of the chip take the least time. Measured (us, registers / 32 x 32 / 32 x 64 / 64 x 64): 224 x 4096 x 1024 35 / 25.8 / 25.4 / 23.8,
// 224 x 6144 x 1024 54 / 36.9 / 36.2 / 42.7, 224 x 1024 x 3072 30 / 18.7 / 31 / 54, 64 x 6144 x 1024 25 / 14.7 / 14.4 / 22,
// 1024 x 24576 x 4096 2073 / 1898 / 1742 / 1627 (127 TFLOP/s).
// Where one wave would make a tile alone (below) the ring is ahead too (one wave / ring: 500 x 1024 x 128 10.4 / 6.4, 200 x 4096 x 128
// 10.6 / 8.6, 1000 x 1024 x 256 15.3 / 11.4, 4096 x 1024 x 256 36.0 / 33.2, x 512 57.9 / 48.8, 8192 x 4096 x 512 420 / 350), but for a
// single chunk and eight tiles a compute unit or more: then there is nothing to walk (2048 x 1024 x 128 13.9 / 14.1, 4096 x 1024 x 128
// 25.0 / 25.2, 200 x 151936 x 128 166 / 170).
static int ring_shape(int M, int N, int K) {
    const long units = mv_compute_units();
    auto tiles = [&](int rm, int rn) { return ((M + 16L * rm - 1) / (16 * rm)) * ((N + 16L * rn - 1) / (16 * rn)); };
    if (M <= 0 || N <= 0 || K <= 0 || K % 128 || (M <= 16 && 2 * tiles(2, 2) < units) || (K == 128 && tiles(2, 2) >= 8 * units)) return 0;
    // us of a chunk and of a tile's end, per shape, fitted to what they take alone and in rounds
    auto cost = [&](int rm, int rn, double chunk, double last) {
        return (double)((tiles(rm, rn) + units - 1) / units) * (K / 128 * chunk + last);
    };
    const double c22 = cost(2, 2, 0.57, 1.2), c24 = cost(2, 4, 1.07, 2.0), c44 = cost(4, 4, 2.0, 3.0);
    return c44 <= c24 && c44 <= c22 ? 44 : c24 <= c22 ? 24 : 22;
}

extern "C" int mv_gemm_ref_ring_shape(int M, int N, int K) { return ring_shape(M, N, K); }

// The others (rows at any address, another K, types of 16 bits):
// The largest tile that still gives every compute unit one, since a larger one reads less a product; the bits do not depend
// on it. Tiles of 32 x 64 where whole rounds of the chip by 64 x 64 leave it a quarter idle or more (224 x 6144 x 1024: 1.5
// rounds, 61 us against 55), but not below 64 rows, where they are all of it (40 x 24576 x 4096: 235 us against 177).
// Up to 512 values of k one wave makes a tile alone where that gives the chip two waves a compute unit, or fewer where K has
// few blocks (us, eight waves / one: 64 x 256 x 32 8.5 / 7.9, 500 x 1024 x 128 13.4 / 11.5, 4096 x 1024 x 128 46 / 26, x 256 56 / 39,
// 16384 x 4096 x 48 392 / 125; but 200 x 1024 x 128 10.2 / 11.2, 2000 x 1024 x 1024 64 / 70), in tiles of 32 x 64 from 128 values
// on where these are enough (4096 x 1024 x 512 63 against 74).
template <typename TA, typename TW, typename TC>
static void launch_gemm(const void* A, long lda, const void* W, long ldw, const void* bias, void* C, long ldc,
                        int M, int N, int K, hipStream_t stream) {
    const long units = mv_compute_units();
    auto tiles = [&](int rm, int rn) { return ((M + 16L * rm - 1) / (16 * rm)) * ((N + 16L * rn - 1) / (16 * rn)); };
    // work of the unit that gets the most tiles, in tiles of 16 x 16
    auto rounds = [&](int rm, int rn) { return (tiles(rm, rn) + units - 1) / units * rm * rn; };
    if constexpr (sizeof(TA) == 4 && sizeof(TW) == 4 && sizeof(TC) == 4) {
        const bool vec = lda % 4 == 0 && ldw % 4 == 0 && (uintptr_t)A % 16 == 0 && (uintptr_t)W % 16 == 0;
        const int shape = vec ? ring_shape(M, N, K) : 0;
        if (shape) {
            if (shape == 44) launch_ring<4, 4, 2>(A, lda, W, ldw, bias, C, ldc, M, N, K, stream);
            else if (shape == 24) launch_ring<2, 4, 3>(A, lda, W, ldw, bias, C, ldc, M, N, K, stream);
            else launch_ring<2, 2, 4>(A, lda, W, ldw, bias, C, ldc, M, N, K, stream);
            return;
        }
    }
    if (M > 16 && M <= 65535 * 32 && K <= 512 && (K <= 32 || tiles(2, 2) >= (K <= 64 ? units / 2 : 2 * units))) {
        if (K > 128 && tiles(2, 4) > 4 * units) launch_waves<TA, TW, TC, 2, 4>(A, lda, W, ldw, bias, C, ldc, M, N, K, stream);
        else launch_waves<TA, TW, TC, 2, 2>(A, lda, W, ldw, bias, C, ldc, M, N, K, stream);
    } else if (M > 65535 * 32 || (M > 32 && tiles(4, 4) >= units && (M <= 64 || 4 * rounds(4, 4) <= 5 * rounds(2, 4))))
        launch_tiles<TA, TW, TC, 4, 4, 1>(A, lda, W, ldw, bias, C, ldc, M, N, K, stream);
    else if (M > 64 && tiles(2, 4) >= units)
        launch_tiles<TA, TW, TC, 2, 4, 2>(A, lda, W, ldw, bias, C, ldc, M, N, K, stream);
    else if (M > 16)
        launch_tiles<TA, TW, TC, 2, 2, 3>(A, lda, W, ldw, bias, C, ldc, M, N, K, stream);
    else if (tiles(1, 4) >= units)
        launch_tiles<TA, TW, TC, 1, 4, 4>(A, lda, W, ldw, bias, C, ldc, M, N, K, stream);
    else
        launch_tiles<TA, TW, TC, 1, 1, 8>(A, lda, W, ldw, bias, C, ldc, M, N, K, stream);
}

// a_dtype: activations; w_dtype: weight and bias as stored; c_dtype: a_dtype or float.
extern "C" int mv_gemm_ref(const void* A, long lda, int a_dtype, const void* W, long ldw, int w_dtype,
                           const void* bias, void* C, long ldc, int c_dtype, int M, int N, int K,
                           hipStream_t stream) {
    MV_REQUIRE(M >= 0 && N > 0 && K > 0, "gemm: bad sizes M=%d N=%d K=%d", M, N, K);
    MV_REQUIRE(lda >= K && ldw >= K && ldc >= N, "gemm: leading dimensions lda=%ld ldw=%ld ldc=%ld too small for "
               "M=%d N=%d K=%d", lda, ldw, ldc, M, N, K);
    MV_REQUIRE(mv_valid_dtype(w_dtype), "gemm: bad weight dtype %d", w_dtype);
    MV_REQUIRE(c_dtype == a_dtype || c_dtype == MV_F32, "gemm: output dtype %d must be the activation dtype %d "
               "or float", c_dtype, a_dtype);
    if (M == 0) return 0;
    MV_REQUIRE((M + 63) / 64 <= 65535, "gemm: M=%d too large for one launch", M);
    MV_DISPATCH_T(a_dtype, "gemm", {
        if (w_dtype == MV_F32) {
            if (c_dtype == MV_F32) launch_gemm<T, float, float>(A, lda, W, ldw, bias, C, ldc, M, N, K, stream);
            else launch_gemm<T, float, T>(A, lda, W, ldw, bias, C, ldc, M, N, K, stream);
        } else {
            if (c_dtype == MV_F32) launch_gemm<T, bf16, float>(A, lda, W, ldw, bias, C, ldc, M, N, K, stream);
            else launch_gemm<T, bf16, T>(A, lda, W, ldw, bias, C, ldc, M, N, K, stream);
        }
    });
    return mv_check_launch("gemm");
}
