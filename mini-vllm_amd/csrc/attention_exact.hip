// Paged causal attention in float on the float matrix unit (v_mfma_f32_16x16x4_f32), for the steps of the float32 engine with
// plain softmax attention: head sizes 64 and 128, no window, no gate, unchanged scores (attention_ref.hip takes the rest).
//
// A workgroup takes the 16 / (heads of a key/value head) neighbouring tokens of a request whose query rows of one key/value
// head fill 16 columns; its eight waves take the blocks of 16 keys in turn, wave w blocks w, w + 8, ..., and their partial
// results are merged through LDS in the order of the waves.
//   scores^T = K Q^T     lane i + 16 g holds column i, keys 4 g .. 4 g + 3 of the block,
//   out^T    = V^T P^T   which is what the second product takes: nothing is exchanged between the two.
// Maximum, sum and accumulator are float, and nothing is rounded between. Blocks lie at multiples of 16 positions and a wave's
// blocks do not depend on the request, so a row's bits depend on its position alone: what a unit's later tokens see beyond
// it adds zeros. (Where a later value of the block is no number, the products of the block are added up one by one instead: the
// row keeps its value to rounding.)
//
// What bounds it: the round trips of a workgroup's start (the request's place, page ids, keys), then the lines of keys that a
// compute unit asks for; the kernel of a workgroup a (token, head) reads every key row once for every query row. A prompt of
// 200 tokens (224 rows), 16 query and 8 key/value heads of 128: 41 us with that, 17 here; error against 64 bits 1.9e-7, 2.9e-7 with that
// (N(0, 1) operands).
#include "dispatch.h"

typedef float ax_acc_t __attribute__((ext_vector_type(4)));

#define AX_WAVES 8
#define AX_KEYS 16

// The unit (up to `tokens` neighbouring tokens of a request) number `unit` of the step; every wave looks by itself.
__device__ __forceinline__ void ax_find(const int* __restrict__ cu, int n_seqs, int tokens, int unit, int& seq, int& row0, int& count) {
    const int lane = threadIdx.x % MV_WAVE;
    int base = 0;
    seq = -1;
    row0 = count = 0;
    for (int s0 = 0; s0 < n_seqs; s0 += MV_WAVE) {
        const int s = s0 + lane;
        const int first = s < n_seqs ? cu[s] : 0, len = s < n_seqs ? cu[s + 1] - first : 0;
        const int mine = (len + tokens - 1) / tokens;
        int upto = mine;
#pragma unroll
        for (int o = 1; o < MV_WAVE; o <<= 1) {
            const int t = __shfl_up(upto, o, MV_WAVE);
            if (lane >= o) upto += t;
        }
        const unsigned long long here = __ballot(base + upto > unit);
        if (here) {
            const int l = __builtin_ctzll(here);
            const int c = unit - (base + __shfl(upto, l, MV_WAVE) - __shfl(mine, l, MV_WAVE));
            seq = s0 + l;
            row0 = __shfl(first, l, MV_WAVE) + c * tokens;
            count = min(__shfl(len, l, MV_WAVE) - c * tokens, tokens);
            return;
        }
        base += __shfl(upto, MV_WAVE - 1, MV_WAVE);
    }
}

template <int D>
__global__ void __launch_bounds__(64 * AX_WAVES)
attention_exact_kernel(const float* __restrict__ q, long q_stride, float* __restrict__ out, long out_stride, const float* __restrict__ k_pages,
                       const float* __restrict__ v_pages, const int* __restrict__ block_table, int bt_width, int page_size,
                       const int* __restrict__ positions, const int* __restrict__ cu_seqlens, int n_seqs, const int* __restrict__ token_seq,
                       int n, int padded, int H, int Hkv, float scale) {
    constexpr int DT = D / 16;
    __shared__ float sm_m[AX_WAVES][16], sm_l[AX_WAVES][16];
    __shared__ ax_acc_t sm_o[AX_WAVES][DT][MV_WAVE];
    const int lane = threadIdx.x % MV_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / MV_WAVE), i = lane % 16, g = lane / 16;
    const int unit = blockIdx.x / Hkv, kvh = blockIdx.x - unit * Hkv, G = H / Hkv, tokens = 16 / G;
    int seq, row0, count;
    ax_find(cu_seqlens, n_seqs, tokens, unit, seq, row0, count);
    if (padded)                                       // rows that belong to no request: zeros
        for (int row = unit; row < n; row += gridDim.x / Hkv)
            if (row >= cu_seqlens[n_seqs] && token_seq[row] < 0)
                for (int e = threadIdx.x; e < G * D; e += 64 * AX_WAVES) out[(size_t)row * out_stride + (size_t)kvh * G * D + e] = 0.f;
    if (seq < 0 || count <= 0) return;
    const bool live = i < count * G;
    const int row = row0 + (live ? i / G : 0), head = kvh * G + (live ? i % G : 0);
    const int pos = live ? positions[row] : -1;       // of this lane's column
    const int lo = positions[row0], hi = positions[row0 + count - 1];
    const int* bt = block_table + (size_t)seq * bt_width;
    // Page ids are asked for before it is known which keys there are: behind the newest key a lane takes page 0 instead of what
    // the table says there (its scores are masked and its values zeroed).
    struct Pages {
        int k, v;                                     // of this lane's key row, and of its four values a row
    };
    auto look = [&](int b) -> Pages {
        return Pages{bt[min((AX_KEYS * b + i) / page_size, bt_width - 1)], bt[min((AX_KEYS * b + 4 * g) / page_size, bt_width - 1)]};
    };
    Pages now = look(wave), next = look(wave + AX_WAVES);

    float4 qv[DT];
    const float* qrow = q + (size_t)row * q_stride + (size_t)head * D + 4 * g;
#pragma unroll
    for (int t = 0; t < DT; ++t) qv[t] = *reinterpret_cast<const float4*>(qrow + 16 * t);

    float4 x_v[DT];
    const int blocks = hi / AX_KEYS + 1;
    auto fetch_keys = [&](float4 (&k)[DT], int b, int page) {
        const int key = AX_KEYS * b + i;
        const float* kp = k_pages + (((size_t)(key <= hi ? page : 0) * Hkv + kvh) * page_size + key % page_size) * D + 4 * g;
#pragma unroll
        for (int t = 0; t < DT; ++t) k[t] = *reinterpret_cast<const float4*>(kp + 16 * t);
    };
    auto fetch_values = [&](int b, int page) {
        const int key = AX_KEYS * b + 4 * g;
        const float* vp = v_pages + (((size_t)(key <= hi ? page : 0) * Hkv + kvh) * D + i) * page_size + key % page_size;
#pragma unroll
        for (int t = 0; t < DT; ++t) x_v[t] = *reinterpret_cast<const float4*>(vp + (size_t)16 * t * page_size);
    };
    auto mfma = [](ax_acc_t& acc, const float4& a, const float4& b) {
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b.x, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b.y, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, b.z, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, b.w, acc, 0, 0, 0);
    };

    float m = -INFINITY, l = 0.f;
    ax_acc_t acc[DT];
#pragma unroll
    for (int t = 0; t < DT; ++t) acc[t] = ax_acc_t{0.f, 0.f, 0.f, 0.f};
    auto compute = [&](const float4 (&x_k)[DT], int b) {
        ax_acc_t even{0.f, 0.f, 0.f, 0.f}, odd{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < DT; t += 2) {
            mfma(even, x_k[t], qv[t]);
            mfma(odd, x_k[t + 1], qv[t + 1]);
        }
        const int key0 = AX_KEYS * b + 4 * g;
        float p[4], mx = -INFINITY;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            p[r] = key0 + r <= pos ? (even[r] + odd[r]) * scale : -INFINITY;
            mx = fmaxf(mx, p[r]);
        }
        mx = fmaxf(mx, __shfl_xor(mx, 16, MV_WAVE));
        mx = fmaxf(mx, __shfl_xor(mx, 32, MV_WAVE));
        const float m_new = fmaxf(m, mx), safe = m_new == -INFINITY ? 0.f : m_new;
        const float corr = expf(m - safe);            // exp(-inf) = 0
        float sum = 0.f;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            p[r] = expf(p[r] - safe);
            sum += p[r];
        }
        l = l * corr + sum;
        m = m_new;
#pragma unroll
        for (int t = 0; t < DT; ++t) acc[t] *= corr;
        if (AX_KEYS * b + AX_KEYS - 1 > lo) {         // (the same for the workgroup) some column does not see all keys of the block
            // slots behind the newest key may hold anything
            bool odd_value = false;
#pragma unroll
            for (int t = 0; t < DT; ++t) {
                float* v = reinterpret_cast<float*>(&x_v[t]);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (key0 + r > hi) v[r] = 0.f;
                    odd_value |= !(fabsf(v[r]) < INFINITY);
                }
            }
            // and a value that is no number must not reach the columns that do not see it: zero times it is none either
            if (__ballot(odd_value)) {
                for (int key = AX_KEYS * b; key < AX_KEYS * (b + 1) && key <= hi; ++key) {
                    const float* v = v_pages + ((size_t)bt[key / page_size] * Hkv + kvh) * D * page_size + key % page_size;
                    const int from = i + 16 * ((key % AX_KEYS) / 4), r = key % 4;
                    const float p0 = __shfl(p[0], from, MV_WAVE), p1 = __shfl(p[1], from, MV_WAVE), p2 = __shfl(p[2], from, MV_WAVE),
                                p3 = __shfl(p[3], from, MV_WAVE);
                    const float w = r == 0 ? p0 : r == 1 ? p1 : r == 2 ? p2 : p3;
                    if (key <= pos)
#pragma unroll
                        for (int t = 0; t < DT; ++t)
#pragma unroll
                            for (int e = 0; e < 4; ++e) acc[t][e] = fmaf(w, v[(size_t)(16 * t + 4 * g + e) * page_size], acc[t][e]);
                }
                return;
            }
        }
        const float4 pv{p[0], p[1], p[2], p[3]};
#pragma unroll
        for (int t = 0; t < DT; ++t) mfma(acc[t], x_v[t], pv);
    };

    // keys come a block ahead of their products, page ids a block ahead of that, values behind the scores' products
    if (wave < blocks) {
        float4 ka[DT], kb[DT];
        fetch_keys(ka, wave, now.k);
        for (int b = wave; b < blocks; b += 2 * AX_WAVES) {
            fetch_values(b, now.v);
            fetch_keys(kb, b + AX_WAVES, next.k);
            now = next;
            next = look(b + 2 * AX_WAVES);
            compute(ka, b);
            if (b + AX_WAVES >= blocks) break;
            fetch_values(b + AX_WAVES, now.v);
            fetch_keys(ka, b + 2 * AX_WAVES, next.k);
            now = next;
            next = look(b + 3 * AX_WAVES);
            compute(kb, b + AX_WAVES);
        }
    }
    l += __shfl_xor(l, 16, MV_WAVE);
    l += __shfl_xor(l, 32, MV_WAVE);

    if (g == 0) {
        sm_m[wave][i] = m;
        sm_l[wave][i] = l;
    }
#pragma unroll
    for (int t = 0; t < DT; ++t) sm_o[wave][t][lane] = acc[t];
    __syncthreads();
    if (wave >= DT || !live) return;                  // tile `wave` of the head's elements
    float top = -INFINITY, total = 0.f;
#pragma unroll
    for (int w = 0; w < AX_WAVES; ++w) top = fmaxf(top, sm_m[w][i]);
    ax_acc_t o{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < AX_WAVES; ++w) {
        // No key of this wave's is seen. (Its maximum does not say so: fmaxf passes over scores that are no numbers, and a wave that
        // sees nothing else keeps minus infinity, with the sum that has to come through.)
        if (AX_KEYS * w > pos) continue;
        const float f = expf(sm_m[w][i] - top);
        total += f * sm_l[w][i];
        o += f * sm_o[w][wave][lane];
    }
    const float inv = 1.f / total;
    *reinterpret_cast<float4*>(out + (size_t)row * out_stride + (size_t)head * D + 16 * wave + 4 * g) =
        float4{o[0] * inv, o[1] * inv, o[2] * inv, o[3] * inv};
}

// Neighbouring tokens of a request that share a workgroup, 0: heads or pages of these sizes are not served
extern "C" int mv_attention_exact_unit(int H, int Hkv, int D, int page_size) {
    if (H <= 0 || Hkv <= 0 || H % Hkv || H / Hkv > 16 || (D != 64 && D != 128) || page_size <= 0 || page_size % 4) return 0;
    return 16 / (H / Hkv);
}

// units: at least the runs of mv_attention_exact_unit tokens that cu_seqlens [n_seqs + 1] holds. padded: there
// are rows that belong to no request (token_seq < 0); they are written as zeros.
extern "C" int mv_attention_exact(const void* q, long q_stride, void* out, long out_stride, const void* k_pages, const void* v_pages,
                                  const int* block_table, int bt_width, int page_size, const int* positions, const int* cu_seqlens, int n_seqs,
                                  int units, const int* token_seq, int n, int padded, int H, int Hkv, int D, float scale, hipStream_t stream) {
    MV_REQUIRE(n >= 0 && n_seqs >= 0 && units >= 0 && bt_width > 0, "attention_exact: bad sizes n=%d seqs=%d", n, n_seqs);
    MV_REQUIRE(mv_attention_exact_unit(H, Hkv, D, page_size) > 0, "attention_exact: %d / %d heads of %d on pages of %d are not served", H, Hkv, D, page_size);
    MV_REQUIRE(q_stride >= (long)H * D && q_stride % 4 == 0 && out_stride >= (long)H * D && out_stride % 4 == 0 && (uintptr_t)q % 16 == 0 &&
                   (uintptr_t)out % 16 == 0 && (uintptr_t)k_pages % 16 == 0 && (uintptr_t)v_pages % 16 == 0,
               "attention_exact: rows of queries, outputs and pages start at 16-byte addresses");
    MV_REQUIRE(q && out && k_pages && v_pages && block_table && positions && cu_seqlens && token_seq, "attention_exact: missing operand");
    MV_REQUIRE((long)units * Hkv <= 8388607L, "attention_exact: too many units %d", units);
    if (n == 0 || units == 0) return 0;
    if (D == 128)
        hipLaunchKernelGGL((attention_exact_kernel<128>), dim3((unsigned)units * Hkv), dim3(64 * AX_WAVES), 0, stream, (const float*)q, q_stride, (float*)out,
                           out_stride, (const float*)k_pages, (const float*)v_pages, block_table, bt_width, page_size, positions, cu_seqlens, n_seqs,
                           token_seq, n, padded, H, Hkv, scale);
    else
        hipLaunchKernelGGL((attention_exact_kernel<64>), dim3((unsigned)units * Hkv), dim3(64 * AX_WAVES), 0, stream, (const float*)q, q_stride, (float*)out,
                           out_stride, (const float*)k_pages, (const float*)v_pages, block_table, bt_width, page_size, positions, cu_seqlens, n_seqs,
                           token_seq, n, padded, H, Hkv, scale);
    return mv_check_launch("attention_exact");
}
