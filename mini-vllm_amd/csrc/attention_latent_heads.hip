// Attention over a cached latent for steps whose requests bring many tokens (bfloat16, MFMA; see attention_latent.hip for what is
// computed): the heads' own keys and values are made from the step's latents once, and attention runs on those.
//
// Carried into the latent's space a (query, key) pair costs R + DR products for the score and R for the sum, 576 at a latent of
// 256 and 64 rotary channels; with the head's own keys and values 128 + DR and 128, 320. Making them costs 256 R a key and head,
// what carrying the queries in and the sums out costs a query and head: they are the same maps. So a request whose tokens are
// about as many as its keys computes 1.8 times less (what is left to choose is Ops.latent_heads).
//
//   latent_expand_kernel           K_h = W_uk,h c and V_h = W_uv,h c of every key of the step's requests, in operand order
//   attention_latent_heads_kernel  causal softmax attention on them, the output gates in its epilogue
//
// Layout of the keys: the requests' keys in blocks of 32, each request from a block of its own on (the blocks' slots behind a
// request's end hold zeros). Of block b and head h, in pieces of 16 bytes a lane:
//   k   [b][h][tile t of 2][step s of 4][lane]      lane (g, rho) = 16 g + rho: channels 32 s + 8 g.. of key 8 (rho / 4) + 4 t + rho % 4
//   kr  [b][t][step s of DR / 32][lane]             the rotated channels, the same for all heads
//   v   [b][h][tile dt of 8][lane]                  channel 16 dt + rho of keys 8 g .. 8 g + 7
// What bounds it: a wave's block of 32 keys is a chain (scores, maximum, exponentials, sums) of 0.7 us, and a compute unit's two
// workgroups take 0.85 us for one each, LDS 60 % busy with the operands. 256 + 64, 16 heads, one request of 200 / 1,000 / 2,048 /
// 8,000 tokens, us by events around 30 calls: in the latent's space with its maps in and out 56 / 117 / 202 / 1,265, here 32 / 40 / 68 / 553
// (2,048: 11.5 for the keys and values).
//
// Precision: the keys and values are rounded to 16 bits here where the carried queries and the sums of latents are there, so two
// roundings that both have are taken out: the weights and the turned channels of the queries are two operands each, the rounded
// number and what that leaves (13 products more beside 21; 2,048 tokens 59.5 -> 68 us). Error against 64 bits over that of the
// latent's space, scores of a deviation of 0.3 / 1 / 3, 65 to 8,000 tokens and 100 to 300 behind 500 to 2,000: 0.76 to 0.92, 0.69 to
// 0.92, 0.90 to 0.91; with neither 0.90 to 1.03, 0.79 to 1.01, 1.00 to 1.04, with the weights' alone up to 1.01, with the queries' alone
// up to 1.02. Without a rotary part there is no turned channel, and sharp weights (a deviation of 3) are up to 4 % further off than in
// the latent's space: models of that kind stay there (LatentAttention.heads_operands).
//
// These are the operands of v_mfma_f32_16x16x32_bf16 as attention_prefill.hip holds them in LDS (the order of a tile's keys lets a
// lane's probabilities be the second product's operand as they are), so a load instruction is a kilobyte of whole lines.
#include "gemm_ring.h"

#define ALH_DIM 128                                            // plain channels of a head, and channels of its values
#define ALH_WAVES 4
#define ALH_THREADS (64 * ALH_WAVES)
#define ALH_TOKENS (16 * ALH_WAVES)                            // of a unit
#define ALH_KEYS 32
#define ALH_TILE 512                                           // pieces of a block's k, and of its v, a head
#define ALH_LOG2E 1.4426950408889634f

union AlhFrag {
    uint4 u;
    uint16_t h[8];
    bf16x8_t v;
};

__device__ __forceinline__ int alh_blocks(int len, int context) { return len > 0 ? (context + ALH_KEYS - 1) / ALH_KEYS : 0; }

// Which request the `at`-th of something lies in that request s has of_request(s) of: (request, how many of its own come before it,
// and the sum of alongside(s) of the requests in front). Every wave finds it by itself, 64 requests at a time. Request -1: none.
struct AlhPlace {
    int seq, in, before;
};
template <class Of, class Along>
__device__ __forceinline__ AlhPlace alh_find(int at, int n_seqs, Of of_request, Along alongside) {
    const int lane = threadIdx.x % MV_WAVE;
    int before = 0;
    for (int s0 = 0; s0 < n_seqs; s0 += MV_WAVE) {
        const int s = s0 + lane;
        const int mine = s < n_seqs ? of_request(s) : 0, along = s < n_seqs ? alongside(s) : 0;
        int incl = mine, incl_along = along;
#pragma unroll
        for (int o = 1; o < MV_WAVE; o <<= 1) {
            const int t = __shfl_up(incl, o, MV_WAVE), u = __shfl_up(incl_along, o, MV_WAVE);
            if (lane >= o) {
                incl += t;
                incl_along += u;
            }
        }
        const unsigned long long hit = __ballot(at < incl && at >= incl - mine);
        if (hit != 0) {
            const int l = __ffsll(hit) - 1;
            return AlhPlace{__builtin_amdgcn_readfirstlane(s0 + l), __builtin_amdgcn_readfirstlane(at - __shfl(incl - mine, l, MV_WAVE)),
                            __builtin_amdgcn_readfirstlane(before + __shfl(incl_along - along, l, MV_WAVE))};
        }
        at -= __shfl(incl, MV_WAVE - 1, MV_WAVE);
        before += __shfl(incl_along, MV_WAVE - 1, MV_WAVE);
    }
    return AlhPlace{-1, 0, 0};
}

// A workgroup makes one head's keys and values of two neighbouring blocks (64 keys). The latents come from the pages a quarter a
// wave, into LDS in operand order; each wave takes 32 of the 128 channels of K and of V, its weights straight from memory (in
// operand order too: [head][tile of 16 channels][32 inputs][lane]). `blocks` of a recording is what its size class may hold, up to
// some ten times what a step does: workgroups walk over the pairs of blocks, twice as many of them as stand on the chip at once, and end
// at the first pair that holds nothing (16 heads, 2,048 tokens, room for 1,000 blocks more: 14.7 us, 12.1 without them; with a workgroup for
// every pair 34.8 and 11.2).
template <int RS, int DRS>                                     // k-steps of the latent and of the rotary part
__global__ void __launch_bounds__(ALH_THREADS)
latent_expand_kernel(const bf16* __restrict__ pages, const int* __restrict__ block_table, int bt_width, int page_size,
                     const int* __restrict__ cu_seqlens, const int* __restrict__ context_lens, int n_seqs, const uint4* __restrict__ w_k,
                     const uint4* __restrict__ w_v, int H, uint4* __restrict__ k_out, uint4* __restrict__ kr_out, uint4* __restrict__ v_out,
                     int blocks) {
    constexpr int R = 32 * RS, DK = R + 32 * DRS;
    __shared__ uint4 lat[4 * RS * 64];                         // [16 keys][k-step][lane]
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / MV_WAVE), lane = tid % MV_WAVE;
    const int r = lane % 16, g = lane / 16, head = blockIdx.x;
    for (int pair = blockIdx.y; 2 * pair < blocks; pair += gridDim.y) {
        // this wave's sixteen keys: half `wave % 2` of block `wave / 2`
        int limit[2];                                          // keys of the two blocks that there are
        bool any = false;
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const int block = 2 * pair + b;
            limit[b] = -1;
            if (block < blocks) {
                const auto of = [&](int s) { return alh_blocks(cu_seqlens[s + 1] - cu_seqlens[s], context_lens[s]); };
                const AlhPlace at = alh_find(block, n_seqs, of, [](int) { return 0; });
                if (at.seq >= 0) {
                    const int left = context_lens[at.seq] - ALH_KEYS * at.in;
                    limit[b] = left < ALH_KEYS ? left : ALH_KEYS;
                    any = true;
                    if (wave / 2 == b) {
                        const int key = 16 * (wave % 2) + r, have = key < limit[b] ? key : limit[b] - 1;
                        const int pos = ALH_KEYS * at.in + have, entry = pos / page_size;
                        const bf16* row = pages + ((size_t)block_table[(size_t)at.seq * bt_width + entry] * page_size + (pos - entry * page_size)) * DK + 8 * g;
                        const bool on = key < limit[b];
                        AlhFrag c[RS];
#pragma unroll
                        for (int s = 0; s < RS; ++s) c[s].u = *reinterpret_cast<const uint4*>(row + 32 * s);
                        if (head == 0) {
                            const int t = (key / 4) % 2, rho = 4 * (key / 8) + key % 4;
#pragma unroll
                            for (int s = 0; s < DRS; ++s) {
                                const uint4 x = *reinterpret_cast<const uint4*>(row + R + 32 * s);
                                kr_out[(((size_t)block * 2 + t) * DRS + s) * 64 + 16 * g + rho] = on ? x : uint4{0u, 0u, 0u, 0u};
                            }
                        }
#pragma unroll
                        for (int s = 0; s < RS; ++s) lat[(wave * RS + s) * 64 + lane] = on ? c[s].u : uint4{0u, 0u, 0u, 0u};
                    }
                }
            }
            if (limit[b] < 0 && wave / 2 == b)
#pragma unroll
                for (int s = 0; s < RS; ++s) lat[(wave * RS + s) * 64 + lane] = uint4{0u, 0u, 0u, 0u};
        }
        if (!any) return;                                      // (the same for every wave; nor are there blocks behind)
        __syncthreads();
        int maps = 0;
        asm volatile("" : "+s"(maps));                         // (the maps are read again for every pair: kept, a wave has the unit to itself)
#pragma unroll
        for (int which = 0; which < 2; ++which) {
            const uint4* w = (which == 0 ? w_k : w_v) + maps + ((size_t)head * 8 + 2 * wave) * RS * 64 + lane;
            AlhFrag fw[2][RS];
#pragma unroll
            for (int dt = 0; dt < 2; ++dt)
#pragma unroll
                for (int s = 0; s < RS; ++s) fw[dt][s].u = w[(dt * RS + s) * 64];
            floatx4_t acc[4][2];
#pragma unroll
            for (int ct = 0; ct < 4; ++ct)
#pragma unroll
                for (int dt = 0; dt < 2; ++dt) acc[ct][dt] = floatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ct = 0; ct < 4; ++ct)
#pragma unroll
                for (int s = 0; s < RS; ++s) {
                    AlhFrag fc;
                    fc.u = lat[(ct * RS + s) * 64 + lane];
#pragma unroll
                    for (int dt = 0; dt < 2; ++dt)
                        acc[ct][dt] = which == 0 ? __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[dt][s].v, fc.v, acc[ct][dt], 0, 0, 0)
                                                 : __builtin_amdgcn_mfma_f32_16x16x32_bf16(fc.v, fw[dt][s].v, acc[ct][dt], 0, 0, 0);
                }
#pragma unroll
            for (int ct = 0; ct < 4; ++ct) {
                if (limit[ct / 2] < 0) continue;
                const size_t tile = ((size_t)(2 * pair + ct / 2) * H + head) * ALH_TILE;
#pragma unroll
                for (int dt = 0; dt < 2; ++dt) {
                    const int d16 = 2 * wave + dt;                 // which sixteen channels
                    uint2 bits{f32x2_to_bf16x2_bits(acc[ct][dt][0], acc[ct][dt][1]), f32x2_to_bf16x2_bits(acc[ct][dt][2], acc[ct][dt][3])};
                    uint2* to;
                    if (which == 0) {                              // four channels 16 d16 + 4 g.. of key r
                        const int key = 16 * (ct % 2) + r, t = (key / 4) % 2, rho = 4 * (key / 8) + key % 4;
                        to = reinterpret_cast<uint2*>(k_out + tile + (t * 4 + d16 / 2) * 64 + 16 * (2 * (d16 % 2) + g / 2) + rho) + g % 2;
                    } else {                                       // four keys 4 g.. of channel r
                        to = reinterpret_cast<uint2*>(v_out + tile + d16 * 64 + 16 * (2 * (ct % 2) + g / 2) + r) + g % 2;
                    }
                    *to = bits;
                }
            }
        }
        __syncthreads();                                       // (the latents have been read)
    }
}

struct AlhArgs {
    const bf16* q;             // [row][head][128 | DR], rotated here
    long ldq;
    bf16* out;                 // [row][head][128]
    long ldo;
    const uint4 *k, *kr, *v;
    const int *positions, *cu_seqlens, *context_lens;
    int n_seqs, H;
    float scale;
    const float* table;        // [position][cos DR / 2 | sin DR / 2]
    const float* sink;
    const bf16* gate;          // null: none; rows of H * 128 gates, or of one a head
    long ldg;
    int gate_per_head;
    const int* token_seq;      // null: no padding rows
    int n, fold;
};

// A workgroup of four waves serves one head of a unit, a run of 64 tokens of a request; each wave has 16 of them. Blocks of 32 keys
// walk through four LDS stages in two pairs as in attention_prefill.hip: two blocks to a barrier, which stands between the two;
// a block's operands come from LDS while the block before is computed. (32 tokens a wave read the operands half as often, but 100
// registers of them do not fit: 4,100 tokens of one request 439 us with its keys and values, 8,000 1,125, so 151 and 438.)
template <int DRS>
__global__ void __launch_bounds__(ALH_THREADS) __attribute__((amdgpu_waves_per_eu(2, 2)))
attention_latent_heads_kernel(AlhArgs a) {
    constexpr int DS = 4 + DRS, DT = 8;
    constexpr int KR0 = ALH_TILE, V0 = ALH_TILE + 2 * DRS * 64, STAGE = V0 + ALH_TILE;     // pieces
    __shared__ uint4 ring[4 * STAGE];                          // (80 KB with 64 rotary channels: two workgroups a compute unit)
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / MV_WAVE), lane = tid % MV_WAVE;
    const int i = lane % 16, g = lane / 16, head = blockIdx.x;

    // rows that belong to no request: zeros (a thread looks at a row, all of the workgroup's at once: one after the other they took
    // 6 us of 30 in front of the walk)
    if (a.token_seq != nullptr) {
        const int share = (a.n + gridDim.y - 1) / gridDim.y, end = min((int)(blockIdx.y + 1) * share, a.n);
        for (int row = blockIdx.y * share + tid; row < end; row += ALH_THREADS)
            if (a.token_seq[row] < 0)
                for (int d = 0; d < ALH_DIM; d += 4) *reinterpret_cast<uint2*>(a.out + (size_t)row * a.ldo + (size_t)head * ALH_DIM + d) = uint2{0u, 0u};
    }

    // units with the most keys first; where the whole grid is resident at once its second half runs from the lightest unit upwards
    const int n_all = gridDim.y, half = (n_all + 1) / 2, y = blockIdx.y;
    const int u = (!a.fold || y < half) ? n_all - 1 - y : y - half;
    const auto len_of = [&](int s) { return a.cu_seqlens[s + 1] - a.cu_seqlens[s]; };
    const AlhPlace at = alh_find(u, a.n_seqs, [&](int s) { return (len_of(s) + ALH_TOKENS - 1) / ALH_TOKENS; },
                                 [&](int s) { return alh_blocks(len_of(s), a.context_lens[s]); });
    if (at.seq < 0) return;
    const int first_row = __builtin_amdgcn_readfirstlane(a.cu_seqlens[at.seq]);
    const int t0 = first_row + at.in * ALH_TOKENS;
    const int left = __builtin_amdgcn_readfirstlane(len_of(at.seq)) - at.in * ALH_TOKENS, nt = left < ALH_TOKENS ? left : ALH_TOKENS;
    const int pos0 = __builtin_amdgcn_readfirstlane(a.positions[t0]);     // (a request's rows follow each other)
    const int last = (pos0 + nt - 1) / ALH_KEYS;                          // the walk's last block

    const int col = wave * 16 + i;
    const bool ok = col < nt;
    const int col_tok = t0 + (ok ? col : nt - 1);              // (columns that do not exist: another's, never stored)
    const int col_pos = ok ? pos0 + col : -1;
    AlhFrag qop[DS], qrest[DRS > 0 ? DRS : 1];                 // (rest: what the turned channels' rounding leaves)
    const bf16* row = a.q + (size_t)col_tok * a.ldq + (size_t)head * (ALH_DIM + 32 * DRS) + 8 * g;
#pragma unroll
    for (int s = 0; s < DS; ++s) qop[s].u = *reinterpret_cast<const uint4*>(row + 32 * s);
    if constexpr (DRS == 2) {                                  // channel c of the rotary part turns with c + 32: the same lane holds both
        const float* cs = a.table + (size_t)(pos0 + (ok ? col : nt - 1)) * 64 + 8 * g;
        float c[8], s[8];
        Vec8<float>::load(cs, c);
        Vec8<float>::load(cs + 32, s);
        AlhFrag lo = qop[4], hi = qop[5];
        float x[8], z[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float p = __uint_as_float((uint32_t)lo.h[e] << 16), n = __uint_as_float((uint32_t)hi.h[e] << 16);
            x[e] = p * c[e] - n * s[e];
            z[e] = n * c[e] + p * s[e];
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            qop[4].v[e] = (__bf16)x[e];
            qop[5].v[e] = (__bf16)z[e];
            qrest[0].v[e] = (__bf16)(x[e] - (float)qop[4].v[e]);
            qrest[1].v[e] = (__bf16)(z[e] - (float)qop[5].v[e]);
        }
    }
    // blocks up to bm need no mask: all the wave's columns exist and see all their keys
    const int wave0 = pos0 + wave * 16;
    const int bm = (wave + 1) * 16 <= nt && wave0 >= ALH_KEYS - 1 ? (wave0 - (ALH_KEYS - 1)) / ALH_KEYS : -1;

    float m_run = -INFINITY;
    floatx4_t acc[DT], l_run = floatx4_t{0.f, 0.f, 0.f, 0.f};  // (a row of ones times the weights: a lane's four are one number)
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) acc[dt] = floatx4_t{0.f, 0.f, 0.f, 0.f};
    const float sc = a.scale * ALH_LOG2E;
    AlhFrag ones;
    ones.u = uint4{0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};

    // a block's way into LDS: five loads of a kilobyte a wave (four without a rotary part)
    auto fetch = [&](int j, uint4* stage) __attribute__((always_inline)) {
        const int b = at.before + (j < last ? j : last);       // (past the end: the last block again, it does no harm)
        const size_t own = ((size_t)b * a.H + head) * ALH_TILE;
        const uint4 *k = a.k + own + lane, *v = a.v + own + lane;
#pragma unroll
        for (int x = 0; x < 2; ++x)
            gt_load_to_lds(k + (wave + 4 * x) * 64, (__attribute__((address_space(3))) void*)(stage + (wave + 4 * x) * 64));
        if constexpr (DRS > 0)
            gt_load_to_lds(a.kr + ((size_t)b * 2 * DRS + wave) * 64 + lane, (__attribute__((address_space(3))) void*)(stage + KR0 + wave * 64));
#pragma unroll
        for (int x = 0; x < 2; ++x)
            gt_load_to_lds(v + (wave + 4 * x) * 64, (__attribute__((address_space(3))) void*)(stage + V0 + (wave + 4 * x) * 64));
    };
    struct KOps {
        AlhFrag f[2][DS];
    };
    struct VOps {
        AlhFrag f[DT];
    };
    auto read_k = [&](const uint4* stage, KOps& o) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int s = 0; s < DS; ++s) o.f[t][s].u = s < 4 ? stage[(t * 4 + s) * 64 + lane] : stage[KR0 + (t * DRS + s - 4) * 64 + lane];
    };
    auto read_v = [&](const uint4* stage, VOps& o) __attribute__((always_inline)) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) o.f[dt].u = stage[V0 + dt * 64 + lane];
    };
    // the two products with the softmax between them; behind the score products, asks for the next block's keys and (now) this block's values
    auto compute = [&](int j, const KOps& ko, VOps& vo, const uint4* v_now, const uint4* k_next, KOps& kn, const bool ask_v) __attribute__((always_inline)) {
        const int base = ALH_KEYS * j;
        float p[2][4];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            floatx4_t s4 = floatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < DS; ++s) s4 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ko.f[t][s].v, qop[s].v, s4, 0, 0, 0);
#pragma unroll
            for (int s = 0; s < DRS; ++s) s4 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ko.f[t][4 + s].v, qrest[s].v, s4, 0, 0, 0);
#pragma unroll
            for (int e = 0; e < 4; ++e) p[t][e] = s4[e];
        }
        __builtin_amdgcn_sched_barrier(0);
        if (ask_v) read_v(v_now, vo);
        read_k(k_next, kn);
        __builtin_amdgcn_sched_barrier(0);
        if (j > bm) {                                          // (the same for the wave; kept a branch, see attention_prefill.hip)
            asm volatile("");
            const int hi = col_pos - base - 8 * g;
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int e = 0; e < 4; ++e) p[t][e] = 4 * t + e <= hi ? p[t][e] : -INFINITY;
        }
        AlhFrag pop, rest;
        float mx = -INFINITY;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e) mx = fmaxf(mx, p[t][e]);
        // (the exponentials' reference only follows a maximum that has overtaken it by 2^8: until then nothing is rescaled)
        if (__any(mx * sc > m_run + 8.f)) {
            mx = fmaxf(mx, __shfl_xor(mx, 16, MV_WAVE));
            mx = fmaxf(mx, __shfl_xor(mx, 32, MV_WAVE));
            const float m_new = fmaxf(m_run, mx * sc), ref = m_new == -INFINITY ? 0.f : m_new;
            const float corr = __builtin_amdgcn_exp2f(m_run - ref);
            l_run *= corr;
            m_run = m_new;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) acc[dt] *= corr;
        }
        const float ref = m_run == -INFINITY ? 0.f : m_run;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float w = __builtin_amdgcn_exp2f(fmaf(p[t][e], sc, -ref));
                pop.v[4 * t + e] = (__bf16)w;
                rest.v[4 * t + e] = (__bf16)(w - (float)pop.v[4 * t + e]);
            }
        // (the denominator too is a product, with a row of ones)
        l_run = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones.v, pop.v, l_run, 0, 0, 0);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) acc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vo.f[dt].v, pop.v, acc[dt], 0, 0, 0);
        l_run = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones.v, rest.v, l_run, 0, 0, 0);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) acc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vo.f[dt].v, rest.v, acc[dt], 0, 0, 0);
    };

    uint4 *s0 = ring, *s1 = ring + STAGE, *s2 = ring + 2 * STAGE, *s3 = ring + 3 * STAGE;
    KOps k_even, k_odd;
    VOps vals;
    // blocks j and j + 1 of one pair of stages, j + 2 and j + 3 landing in the other; past the walk's end blocks are computed with every key masked
    auto two_blocks = [&](int j, uint4* cur0, uint4* cur1, uint4* nxt0, uint4* nxt1) __attribute__((always_inline)) {
        compute(j, k_even, vals, cur0, cur1, k_odd, true);
        read_v(cur1, vals);
        GT_WAIT_VMCNT(0);
        __builtin_amdgcn_s_waitcnt(0xc07f);                    // this wave's reads of the pair are back
        __builtin_amdgcn_s_barrier();
        if (j + 4 <= last) {
            fetch(j + 4, cur0);
            fetch(j + 5, cur1);
        }
        compute(j + 1, k_odd, vals, nxt0, nxt0, k_even, false);
    };
    fetch(0, s0);
    fetch(1, s1);
    GT_WAIT_VMCNT(0);
    __builtin_amdgcn_s_barrier();
    fetch(2, s2);
    fetch(3, s3);
    read_k(s0, k_even);
    for (int j = 0; j <= last; j += 4) {
        two_blocks(j, s0, s1, s2, s3);
        if (j + 2 > last) break;
        two_blocks(j + 2, s2, s3, s0, s1);
    }
    GT_WAIT_VMCNT(0);                                          // (a workgroup ends with nothing on its way into its LDS)

    const float l = l_run[0];
    if (!ok) return;
    float inv = 1.f / l;
    if (a.sink != nullptr) {                                   // one more term of the denominator, without a value
        const float sk = a.sink[head] * ALH_LOG2E, m = fmaxf(m_run, sk), f = exp2f(m_run - m);
        inv = f / fmaf(f, l, exp2f(sk - m));
    }
    const bf16* gates = a.gate == nullptr ? nullptr : a.gate + (size_t)col_tok * a.ldg + (a.gate_per_head ? head : head * ALH_DIM);
    if (gates != nullptr && a.gate_per_head) inv *= 1.f / (1.f + expf(-to_f(*gates)));
    bf16* to = a.out + (size_t)col_tok * a.ldo + (size_t)head * ALH_DIM + 4 * g;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
        float o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = acc[dt][e] * inv;
        if (gates != nullptr && !a.gate_per_head)
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] *= 1.f / (1.f + expf(-to_f(gates[16 * dt + 4 * g + e])));
        *reinterpret_cast<uint2*>(to + 16 * dt) = uint2{f32x2_to_bf16x2_bits(o[0], o[1]), f32x2_to_bf16x2_bits(o[2], o[3])};
    }
}

extern "C" int mv_attention_latent_heads_tokens() { return ALH_TOKENS; }
extern "C" int mv_attention_latent_heads_keys() { return ALH_KEYS; }
// 1: heads of `plain` + DR channels and values of `vdim` over a latent of R are served
extern "C" int mv_attention_latent_heads_serves(int plain, int vdim, int R, int DR) {
    return plain == ALH_DIM && vdim == ALH_DIM && (DR == 0 || DR == 64) && (R == 128 || R == 256);
}

// `blocks`: blocks of 32 keys that the step's requests' contexts have in all, or an upper bound. Scratch, 16-byte aligned: k and v
// [blocks][H][4096] bfloat16 each, kr [blocks][32 DR]. w_k, w_v: [H][8 tiles of 16 channels][R / 32][4 groups of 8 inputs][16 channels][8 inputs].
extern "C" int mv_latent_expand(const void* pages, const int* block_table, int bt_width, int page_size, const int* cu_seqlens,
                                const int* context_lens, int n_seqs, const void* w_k, const void* w_v, int H, int R, int DR, void* k, void* kr,
                                void* v, int blocks, hipStream_t stream) {
    MV_REQUIRE(mv_attention_latent_heads_serves(ALH_DIM, ALH_DIM, R, DR) && H > 0 && bt_width > 0 && page_size > 0 && n_seqs >= 0 && blocks >= 0 && blocks <= 131070,
               "latent_expand: sizes R=%d DR=%d H=%d blocks=%d are not served", R, DR, H, blocks);
    MV_REQUIRE(pages && block_table && cu_seqlens && context_lens && w_k && w_v && k && (kr || DR == 0) && v
                   && ((uintptr_t)pages | (uintptr_t)w_k | (uintptr_t)w_v | (uintptr_t)k | (uintptr_t)kr | (uintptr_t)v) % 16 == 0,
               "latent_expand: missing or unaligned operand");
    if (blocks == 0 || n_seqs == 0) return 0;
    const int pairs = (blocks + 1) / 2, at_once = 4 * mv_compute_units() / H + 1;
    const dim3 grid(H, pairs < at_once ? pairs : at_once);
#define ALH_EXPAND(RS, DRS)                                                                                                            \
    hipLaunchKernelGGL((latent_expand_kernel<RS, DRS>), grid, dim3(ALH_THREADS), 0, stream, (const bf16*)pages, block_table, bt_width, page_size, \
                       cu_seqlens, context_lens, n_seqs, (const uint4*)w_k, (const uint4*)w_v, H, (uint4*)k, (uint4*)kr, (uint4*)v, blocks)
    if (R == 256 && DR == 64) ALH_EXPAND(8, 2);
    else if (R == 256) ALH_EXPAND(8, 0);
    else if (DR == 64) ALH_EXPAND(4, 2);
    else ALH_EXPAND(4, 0);
#undef ALH_EXPAND
    return mv_check_launch("latent_expand");
}

// `units`: runs of mv_attention_latent_heads_tokens() tokens of the step's requests, or an upper bound (the rest of the grid
// ends at once); `busy`: how many hold tokens, as far as the caller knows. A request's rows stand at neighbouring positions.
// `padding`: there may be rows of no request; they become zeros.
extern "C" int mv_attention_latent_heads(const void* q, long ldq, void* out, long ldo, const void* k, const void* kr, const void* v,
                                         const int* positions, const int* token_seq, const int* cu_seqlens, const int* context_lens, int n_seqs,
                                         int units, int busy, int n, int padding, int H, int DR, float scale, const float* table,
                                         const float* sink, const void* gate, long ldg, int gate_per_head, hipStream_t stream) {
    MV_REQUIRE(n >= 0 && n_seqs >= 0 && units >= 0 && units <= 65535 && H > 0 && (DR == 0 || DR == 64), "attention_latent_heads: bad sizes n=%d H=%d DR=%d units=%d", n, H, DR, units);
    MV_REQUIRE(ldq >= (long)H * (ALH_DIM + DR) && ldq % 8 == 0 && ldo >= (long)H * ALH_DIM && ldo % 4 == 0 && (!gate || ldg >= (gate_per_head ? H : (long)H * ALH_DIM)),
               "attention_latent_heads: pitches do not fit");
    MV_REQUIRE(q && out && k && v && (kr || DR == 0) && (table || DR == 0) && positions && token_seq && cu_seqlens && context_lens && (uintptr_t)q % 16 == 0
                   && (uintptr_t)out % 8 == 0 && ((uintptr_t)k | (uintptr_t)kr | (uintptr_t)v | (uintptr_t)table) % 16 == 0,
               "attention_latent_heads: missing or unaligned operand");
    if (n == 0) return 0;
    int cus = 0, dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) cus = 256;
    const int fold = (long)H * (busy > 0 && busy < units ? busy : units) <= 2L * cus;
    const AlhArgs a{(const bf16*)q, ldq, (bf16*)out, ldo, (const uint4*)k, (const uint4*)kr, (const uint4*)v, positions, cu_seqlens, context_lens, n_seqs, H,
                    scale, table, sink, (const bf16*)gate, ldg, gate_per_head, padding ? token_seq : nullptr, n, fold};
    const dim3 grid(H, units > 0 ? units : 1);
#define ALH_LAUNCH(DRS) hipLaunchKernelGGL(attention_latent_heads_kernel<DRS>, grid, dim3(ALH_THREADS), 0, stream, a)
    if (DR == 64) ALH_LAUNCH(2);
    else ALH_LAUNCH(0);
#undef ALH_LAUNCH
    return mv_check_launch("attention_latent_heads");
}
