// Attention over a cached latent for steps with prompt portions (bfloat16, MFMA; see attention_latent.hip for what is computed
// and for the page layouts). A workgroup takes ALP_TOKENS neighbouring tokens of a request and 16 heads, each of its waves
// a token: 16 rows that all read the same key rows. Blocks of 32 keys go from the pages straight into LDS (global_load_lds),
// one block ahead of the computation, so a key row is read from the caches once for the workgroup.
//
// What bounds it: the kernel that gives every (row, 16 heads) a wave of its own (attention_latent_mfma_kernel) reads 36 KB of
// keys and latents for 36 products of 16 x 16 x 32, which is what the L2 can deliver; here a workgroup's 288 products share
// them, and what is left is LDS, 288 KB of operands a block. (Two tokens a wave share the operands too, but their 128
// accumulators and 80 registers of queries do not fit beside anything else: the moves between the register files took
// 4.7 us a block, 305 us for 2,048 tokens.) One request of 2,048 tokens, 16 heads, a latent of 256 and 64 rotary channels:
// 290 us a launch with a wave a (row, 16 heads), 143 us here, 270 TFLOP/s of what causality leaves. Short contexts, and steps
// whose many decoding requests would need rounds of workgroups with one busy wave each, stay there (Ops.latent_shares).
//
// Blocks lie at multiples of 32 positions, so the order of additions depends on a query's position (and window) alone. Keys are
// masked in S; a block's slots outside the keys that the workgroup's tokens see (they may hold anything) are zeroed in LDS.
// A wave issues an instruction in four cycles or so, and two waves share a SIMD: beyond the products it is the number of
// instructions a block costs that counts. So a load instruction's keys lie in one page (its address is one scalar base and
// an offset that a lane keeps), a column of scores is a lane's two neighbouring keys (one store for both weights), a row's
// sum is added up over its lanes at the end, exponentials are powers of two (the queries bring the factor), and only
// blocks that a token sees in part are masked.
// LDS, 16-byte pieces: key rows [eight keys g][eight pieces b][key][piece], piece p of key k in place p ^ k ^ (g & 1), and the
// latents slot-contiguous [eight keys g][channel]: sixteen lanes that read one piece of sixteen rows meet in no bank.
#include "gemm_ring.h"

#define ALP_TOKENS 8               // one a wave
#define ALP_THREADS (64 * ALP_TOKENS)
#define ALP_KEYS 32

union AlpFrag {
    uint4 u;
    bf16x8_t v;
};

// over the 16 lanes of a row, every lane gets the result
template <int CTRL>
__device__ __forceinline__ float alp_dpp(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ float alp_row_max(float v) {
    v = fmaxf(v, alp_dpp<0xB1>(v));           // neighbours
    v = fmaxf(v, alp_dpp<0x4E>(v));           // pairs of a quad
    v = fmaxf(v, alp_dpp<0x141>(v));          // mirror of 8
    return fmaxf(v, alp_dpp<0x140>(v));       // mirror of 16
}
__device__ __forceinline__ float alp_row_sum(float v) {
    v += alp_dpp<0xB1>(v);
    v += alp_dpp<0x4E>(v);
    v += alp_dpp<0x141>(v);
    return v + alp_dpp<0x140>(v);
}

struct AlpArgs {
    const float* q;
    long ldq;
    float* out;
    long ldo;
    const bf16* pages;
    const bf16* pages_t;
    const int* block_table;
    int bt_width, page_size;
    const int* positions;
    const int* cu_seqlens;
    int n_seqs, H;
    float scale;
    int window;
    const float* sink;
    const int* token_seq;      // null: no padding rows
    int n;
};

template <int NQ, int NR>
__global__ void __launch_bounds__(ALP_THREADS) __attribute__((amdgpu_waves_per_eu(2, 2)))
attention_latent_prompt_kernel(AlpArgs a) {
    constexpr int DK = NQ * 32, R = NR * 16, PIECES = DK / 8;
    constexpr int KI = 2 * NQ, LOADS = KI + NR;                // load instructions (1 KB each) of a block: key rows, latents
    constexpr int STAGE = LOADS * 64;                          // 16-byte units
    static_assert(DK % 64 == 0, "a row's pieces are permuted in groups of eight");
    __shared__ uint4 ring[2 * STAGE];
    __shared__ __attribute__((aligned(16))) uint16_t pl[ALP_TOKENS][16][40];       // a token's weights: [head][key], rows 80 bytes apart
    __shared__ int sh[8];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / MV_WAVE), lane = tid % MV_WAVE;
    const int r = lane % 16, kq = lane / 16, h0 = blockIdx.y * 16, nh = min(16, a.H - h0);

    // rows that belong to no request: zeros
    if (a.token_seq != nullptr)
        for (int row = blockIdx.x; row < a.n; row += gridDim.x)
            if (a.token_seq[row] < 0)
                for (int e = tid; e < nh * R; e += ALP_THREADS) a.out[(size_t)row * a.ldo + (size_t)h0 * R + e] = 0.f;

    // which request and tokens: units of ALP_TOKENS tokens, the last ones (with the most keys) first
    int seq = -1, row0 = 0, count = 0;
    {
        const int unit = gridDim.x - 1 - blockIdx.x;
        if (tid == 0) sh[4] = -1;
        int base = 0;
        for (int s0 = 0; s0 < a.n_seqs; s0 += 256) {
            const int s = s0 + tid;                        // (the first 256 threads search)
            const bool in = tid < 256 && s < a.n_seqs;
            const int first = in ? a.cu_seqlens[s] : 0, len = in ? a.cu_seqlens[s + 1] - first : 0;
            const int mine = (len + ALP_TOKENS - 1) / ALP_TOKENS;
            int incl = mine;
#pragma unroll
            for (int o = 1; o < MV_WAVE; o <<= 1) {
                const int t = __shfl_up(incl, o, MV_WAVE);
                if (lane >= o) incl += t;
            }
            __syncthreads();
            if (lane == MV_WAVE - 1 && wave < 4) sh[wave] = incl;
            __syncthreads();
            int before = base;
            for (int w = 0; w < wave && w < 4; ++w) before += sh[w];
            incl += before;
            if (unit < incl && unit >= incl - mine) {
                const int c = unit - (incl - mine);
                sh[4] = s;
                sh[5] = first + c * ALP_TOKENS;
                sh[6] = min(len - c * ALP_TOKENS, ALP_TOKENS);
            }
            base += sh[0] + sh[1] + sh[2] + sh[3];
            if (base > unit) break;                            // (the same for every thread)
        }
        __syncthreads();
        seq = sh[4];
        row0 = sh[5];
        count = sh[6];
    }
    if (seq < 0) return;
    const int* bt = a.block_table + (size_t)seq * a.bt_width;
    const int ps = a.page_size;
    const int first_pos = __builtin_amdgcn_readfirstlane(a.positions[row0]), last = first_pos + count - 1;    // a request's rows follow each other
    const int lowest = a.window >= 0 ? max(0, first_pos - a.window) : 0;      // the first key that any of the tokens sees
    // the wave's token: the last key it sees (-1: no such token) and the first
    const int pos = wave < count ? first_pos + wave : -1, lo = pos >= 0 && a.window >= 0 ? max(0, pos - a.window) : 0;

    AlpFrag qf[NQ];
    {
        // (heads and tokens that do not exist read another's row and count as zeros)
        const float* src = a.q + (size_t)(row0 + min(wave, count - 1)) * a.ldq + (size_t)(h0 + min(r, nh - 1)) * DK + 8 * kq;
        const float on = r < nh && pos >= 0 ? a.scale * 1.44269504f : 0.f;
#pragma unroll
        for (int c = 0; c < NQ; ++c) {
            float x[8];
            Vec8<float>::load(src + 32 * c, x);
            qf[c].u = uint4{f32x2_to_bf16x2_bits(x[0] * on, x[1] * on), f32x2_to_bf16x2_bits(x[2] * on, x[3] * on),
                            f32x2_to_bf16x2_bits(x[4] * on, x[5] * on), f32x2_to_bf16x2_bits(x[6] * on, x[7] * on)};
        }
    }
    float m[4], l[4];
    floatx4_t acc[NR];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        // (the sink is a key whose weight counts and whose value is zero)
        const bool has = a.sink != nullptr && 4 * kq + i < nh;
        m[i] = has ? a.sink[h0 + 4 * kq + i] * 1.44269504f : -INFINITY;
        l[i] = has && r == 0 ? 1.f : 0.f;
    }
#pragma unroll
    for (int d = 0; d < NR; ++d) acc[d] = floatx4_t{0.f, 0.f, 0.f, 0.f};

    // eight neighbouring keys lie in one page (page_size is a multiple of eight); those outside what the tokens see are
    // taken from the nearest eight inside
    const int low8 = lowest & ~7, high8 = last & ~7;
    // (lane l looks after the eight keys l % 4 of a block: their page, and in `slot` their first slot there)
    auto page_of = [&](int kb, int& slot) __attribute__((always_inline)) {
        const int key = min(max(kb + 8 * (lane & 3), low8), high8), entry = key / ps;
        slot = key - entry * ps;
        return bt[entry];
    };
    constexpr int MINE = (LOADS + ALP_TOKENS - 1) / ALP_TOKENS, PB = PIECES / 8, VB = R / 64;
    const int key_lane = (lane / 8) * DK + 8 * ((lane % 8) ^ (lane / 8)), key_odd = (lane / 8) * DK + 8 * ((lane % 8) ^ (lane / 8) ^ 1);
    const int value_lane = lane * ps;
    auto fetch = [&](int page, int slot, uint4* stage) __attribute__((always_inline)) {
#pragma unroll
        for (int y = 0; y < MINE; ++y) {
            const int x = y * ALP_TOKENS + wave;               // (scalar, like all that follows from it)
            if (x < LOADS) {
                const bf16* src;
                const int v = x - KI, g = x < KI ? x / PB : v / VB;
                const int pg = __builtin_amdgcn_readlane(page, g), sl = __builtin_amdgcn_readlane(slot, g);
                if (x < KI) src = a.pages + (((size_t)pg * ps + sl) * DK + 64 * (x % PB)) + ((g & 1) ? key_odd : key_lane);
                else src = a.pages_t + (((size_t)pg * R + 64 * (v % VB)) * ps + sl) + value_lane;
                gt_load_to_lds(src, (__attribute__((address_space(3))) void*)(stage + x * 64));
            }
        }
    };
    const int kb0 = lowest & ~(ALP_KEYS - 1);
    int slot_ahead, ahead = page_of(kb0, slot_ahead);
    fetch(ahead, slot_ahead, ring);
    ahead = page_of(kb0 + ALP_KEYS, slot_ahead);
    int st = 0;
    for (int kb = kb0; kb <= last; kb += ALP_KEYS, st ^= 1) {
        uint4* stage = ring + st * STAGE;
        GT_WAIT_VMCNT(0);                                      // the block's loads of this wave, and of the others behind the barrier
        __builtin_amdgcn_s_barrier();
        if (kb < lowest || kb + ALP_KEYS - 1 > last) {         // (the same for every wave)
            uint16_t* v = reinterpret_cast<uint16_t*>(stage + KI * 64);
            for (int e = tid; e < R * ALP_KEYS; e += ALP_THREADS) {
                const int d = e / ALP_KEYS, k = e % ALP_KEYS;
                if (kb + k < lowest || kb + k > last) v[((k / 8) * R + d) * 8 + k % 8] = 0;
            }
            __syncthreads();
        }
        if (kb + ALP_KEYS <= last) {
            fetch(ahead, slot_ahead, ring + (st ^ 1) * STAGE);
            ahead = page_of(kb + 2 * ALP_KEYS, slot_ahead);
        }
        if (kb > pos || kb + ALP_KEYS <= lo) continue;         // the wave's token sees none of these
        // column r of half `sub`: key 2 r + sub of the block
        floatx4_t s[2] = {floatx4_t{0.f, 0.f, 0.f, 0.f}, floatx4_t{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int c = 0; c < NQ; ++c)
#pragma unroll
            for (int sub = 0; sub < 2; ++sub) {
                const int row = 2 * r + sub, g = row / 8, k = row % 8, piece = 4 * c + kq;
                AlpFrag kf;
                kf.u = stage[((g * PB + piece / 8) * 8 + k) * 8 + ((piece % 8) ^ k ^ (g & 1))];
                s[sub] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qf[c].v, kf.v, s[sub], 0, 0, 0);
            }
        const bool in_part = kb + ALP_KEYS - 1 > pos || kb < lo;             // (the same for the wave)
        if (in_part) {
            const int k0 = kb + 2 * r;
            const bool ok0 = k0 <= pos && k0 >= lo, ok1 = k0 + 1 <= pos && k0 + 1 >= lo;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                s[0][i] = ok0 ? s[0][i] : -INFINITY;
                s[1][i] = ok1 ? s[1][i] : -INFINITY;
            }
        }
        float corr[4];
        bool moved = false;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float m_new = fmaxf(m[i], alp_row_max(fmaxf(s[0][i], s[1][i])));
            const float base = m_new == -INFINITY ? 0.f : m_new;            // (no key of this row so far)
            const float e0 = __builtin_amdgcn_exp2f(s[0][i] - base), e1 = __builtin_amdgcn_exp2f(s[1][i] - base);
            corr[i] = __builtin_amdgcn_exp2f(m[i] - base);
            moved |= m_new != m[i];
            l[i] = fmaf(l[i], corr[i], e0 + e1);               // this lane's share of the sum
            m[i] = m_new;
            *reinterpret_cast<uint32_t*>(&pl[wave][4 * kq + i][2 * r]) = f32x2_to_bf16x2_bits(e0, e1);
        }
        if (__any(moved)) {                                    // (a maximum that stands scales by one)
#pragma unroll
            for (int d = 0; d < NR; ++d)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[d][i] *= corr[i];
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        AlpFrag pf;
        pf.u = *reinterpret_cast<const uint4*>(&pl[wave][r][8 * kq]);
#pragma unroll
        for (int d = 0; d < NR; ++d) {
            AlpFrag vf;
            vf.u = stage[KI * 64 + kq * R + 16 * d + r];
            acc[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pf.v, vf.v, acc[d], 0, 0, 0);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    if (pos < 0) return;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int head = 4 * kq + i;
        if (head < nh) {
            const float inv = 1.f / alp_row_sum(l[i]);
            float* o = a.out + (size_t)(row0 + wave) * a.ldo + (size_t)(h0 + head) * R + r;
#pragma unroll
            for (int d = 0; d < NR; ++d) o[16 * d] = acc[d][i] * inv;
        }
    }
}

extern "C" int mv_attention_latent_prompt_tokens() { return ALP_TOKENS; }
// 1: a latent of R numbers and DR rotary channels is served
extern "C" int mv_attention_latent_prompt_serves(int R, int DR) {
    return (DR == 0 && (R == 64 || R == 128 || R == 192 || R == 256)) || (DR == 64 && (R == 128 || R == 256));
}

// `units`: the runs of ALP_TOKENS tokens of the step's requests, or an upper bound (the rest of the grid ends at once). A
// request's rows stand at neighbouring positions. `padding`: there may be rows of no request; they become zeros. Returns 2 (nothing done) for sizes it does not serve.
extern "C" int mv_attention_latent_prompt(const float* q, long ldq, float* out, long ldo, const void* pages, const void* pages_t,
                                          const int* block_table, int bt_width, int page_size, const int* positions, const int* token_seq,
                                          const int* cu_seqlens, int n_seqs, int units, int n, int padding, int H, int R, int DR, float scale,
                                          int window, const float* sink, hipStream_t stream) {
    MV_REQUIRE(n >= 0 && n_seqs >= 0 && units >= 0 && H > 0 && R > 0 && DR >= 0, "attention_latent_prompt: bad sizes n=%d H=%d R=%d DR=%d", n, H, R, DR);
    if (!mv_attention_latent_prompt_serves(R, DR) || page_size % 8 || !pages_t || (uintptr_t)pages % 16
        || (uintptr_t)pages_t % 16)
        return 2;
    MV_REQUIRE(bt_width > 0 && ldq >= (long)H * (R + DR) && ldo >= (long)H * R && H <= 65535 * 16, "attention_latent_prompt: pitches too small");
    MV_REQUIRE(q && out && pages && block_table && positions && token_seq && cu_seqlens && ((uintptr_t)q % 16) == 0 && ldq % 4 == 0,
               "attention_latent_prompt: missing operand or queries not aligned");
    if (n == 0) return 0;
    const AlpArgs a{q, ldq, out, ldo, (const bf16*)pages, (const bf16*)pages_t, block_table, bt_width, page_size, positions, cu_seqlens, n_seqs, H,
                    scale, window, sink, padding ? token_seq : nullptr, n};
    const dim3 grid(units > 0 ? units : 1, (H + 15) / 16);
#define ALP_LAUNCH(NQ, NR) hipLaunchKernelGGL((attention_latent_prompt_kernel<NQ, NR>), grid, dim3(ALP_THREADS), 0, stream, a)
    if (DR == 64) {
        if (R == 256) ALP_LAUNCH(10, 16);
        else ALP_LAUNCH(6, 8);
    } else if (R == 64) ALP_LAUNCH(2, 4);
    else if (R == 128) ALP_LAUNCH(4, 8);
    else if (R == 192) ALP_LAUNCH(6, 12);
    else ALP_LAUNCH(8, 16);
#undef ALP_LAUNCH
    return mv_check_launch("attention_latent_prompt");
}
