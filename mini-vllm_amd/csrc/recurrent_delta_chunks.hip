// The recurrences of recurrent.hip and recurrent_channel.hip for requests that bring many tokens in a step: a request's
// tokens are cut into chunks of DC_TOKENS, everything that concerns one chunk alone is a product of small matrices on the
// MFMA units (float operands, v_mfma_f32_16x16x4_f32), chunks and heads side by side, and only a walk along the chunks
// with one product each is left in a row. All four rules are, per head with S [key size DK][columns DV],
//     p = a^T S;   S <- diag(w) S + b p^T + x v^T;   o = S^T r
//   RULE_GENERAL  Bolapel's delta rule: w the decay, a = u, b = -(rate u), x = k
//   RULE_CHANNEL  the gated delta rule with a decay g per key channel: w = g, a = g k, x = beta k, b = -x
//   RULE_GATED    the same with one decay per head
//   RULE_SUM      the mLSTM's matrix memory: w the forget gate, no p, x = k, v times the input gate
// With tokens s, t counted inside a chunk, P_t = w_0 .. w_t per channel, P_{-1} = 1 and S_0 the state in front of the chunk,
//     A[t][s] = sum_i a_t (P_{t-1} / P_s) x_s (s < t),  B[t][s] = sum_i r_t (P_t / P_s) x_s (s <= t),  A', B' with b for x,
//     T = (I - A')^-1,  W = T (a_t P_{t-1})_t,  U = T A V        (then p = W S_0 + U)
//     S_1 = M S_0 + N,  M = diag(P_last) + B_e W,  N = X_e V + B_e U,  X_e = (x_s P_last / P_s)^T, B_e with b
//     o   = Q S_0 + O,  Q = (r_t P_t)_t + B' W,     O = B V + B' U
// The first kernel leaves M, N, Q and (in the output's rows) O; the second walks S <- M S + N and adds Q S to the output.
// Only quotients P_t / P_s with s <= t occur, as products of decays (never a division, so decays down to zero and chunks
// that forget everything are exact): inside a run of DC_RUN tokens term by term, between the two runs of a chunk as (what
// is left of s at its run's end) times (what is left of that at t), which is a product on the MFMA units again.
//
// What bounded these before was one chain of about 0.2 us a token for every (request, head, 16 columns), 64 workgroups
// for a head count of 16; the chunks' work is spread over every compute unit and the chain is one product of DK x DK with
// DK x 16 a chunk. Measured on one prompt of
// 2,048 tokens, 16 heads of 64 x 64 (us, scan against the two kernels here): GENERAL 438 -> 48 + 37, GATED 477 -> 40 + 37,
// SUM with 65 columns 411 -> 30 + 26; CHANNEL on prompts of 941 and 483 tokens 215 -> 36 + 21. The chunk kernel waits for
// its own phases (eight waves a workgroup hide that best: four took 90, 49, 36 and 45; of GENERAL's 48 us the loads are 12, the products inside
// the runs 10, what makes T, W and U 9 and the maps, which are 50 MB to write, 16), the walk for a round of matrix unit, LDS and barrier a chunk,
// 0.53 us.
//
// Layouts are those of the scans: states [..][H][DV][DK] (a head's matrix column by column), out [n][H][DV]. M [chunks][H][DK][DK],
// N [chunks][H][DV][DK] and Q [n][H][DK] pass from one kernel to the other in the order of quad_of.
#include "recurrent_chunk.h"

#define DC_TOKENS 32
#define DC_RUN 16                  // half a chunk: two runs
// Requests with fewer tokens of a step are left to the scans. There a token's bits do not depend on how the request was cut;
// here they depend on where the chunks lie, and which steps come here depends on all of a step's requests and heads
// (parts/matrix_state.py weighs both paths), so a bfloat16 request's sums may be added in another order in other company.
// The float32 engine scans. One request of 128 tokens, 16 heads of 64, takes the scan 33 us (28 to 34 by rule) and the two
// kernels 28 (19 to 28): the line lies where there is something to gain.
#define DC_LINE 128

enum DeltaRule { RULE_GENERAL = 0, RULE_CHANNEL = 1, RULE_GATED = 2, RULE_SUM = 3 };

struct DeltaChunkArgs {
    const float* vec;              // GENERAL: coef [n][H][5][DK] (w, rate u, u, k, r); else qk [n][G][2][DK]
    const float* gates;            // CHANNEL: beta [n][H]; GATED, SUM: [n][H][4] (decay, strength, ..)
    const float* decay; long ldz;  // CHANNEL: rows whose first H*DK columns are the decays
    int decay4;                    // ... whose rows start at addresses that four floats can be loaded from at once
    const void* vals; long ldv;    // GENERAL: packed rows, the values in columns 2*H*DK ..; else [n][H][DV] floats
    int H, G, DV;
    const int* cu_seqlens; int n_seqs;
    float* M; float* N; float* Q; float* out;
    // ROWS: what the general rule's vectors are made of beside the rows (see delta_prepare_kernel)
    int rank; const void* w2t; const void* w0; const void* a_bias; int weights_f32; float decay_rate, key_eps;
    // ... and those of the channel and gated rules (see channel_prepare_kernel, gdelta_prepare_kernel); `decay` are the rows in front of the exponentials then
    const void* conv_w; const void* a_log; const void* dt_bias; const void* conv_state; const int* state_slots; int gate_off; float unit_eps;
};

#define DC_MAX_RANK 64             // of the decays' products: a lane holds its operands of all of it
template <typename T>
__device__ __forceinline__ float4 four_of(const T* p) {
    if constexpr (sizeof(T) == 4) {
        return *reinterpret_cast<const float4*>(p);
    } else {
        const uint2 u = *reinterpret_cast<const uint2*>(p);
        return float4{__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u), __uint_as_float(u.y << 16), __uint_as_float(u.y & 0xffff0000u)};
    }
}

#define DC_THREADS 512

// find_chunk, for requests of at least DC_LINE tokens and DC_THREADS threads (the first 256 search)
__device__ __forceinline__ void find_long_chunk(const int* __restrict__ cu, int n_seqs, int unit, int* sh, int& seq, int& row0, int& count) {
    const int tid = threadIdx.x, lane = tid % MV_WAVE, wave = tid / MV_WAVE;
    if (tid == 0) sh[4] = -1;
    int base = 0;
    for (int s0 = 0; s0 < n_seqs; s0 += 256) {
        const int s = s0 + tid;
        const int first = s < n_seqs ? cu[s] : 0, len = s < n_seqs ? cu[s + 1] - first : 0;
        const int mine = tid < 256 && len >= DC_LINE ? (len + DC_TOKENS - 1) / DC_TOKENS : 0;
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
            sh[5] = first + c * DC_TOKENS;
            sh[6] = min(len - c * DC_TOKENS, DC_TOKENS);
        }
        base += sh[0] + sh[1] + sh[2] + sh[3];
        if (base > unit) break;                        // (the same for every thread)
    }
    __syncthreads();
    seq = sh[4];
    row0 = sh[5];
    count = seq >= 0 ? sh[6] : 0;
}

// acc += A B over 16 values of k: A's rows hold neighbouring k side by side, B's rows are k
__device__ __forceinline__ void mfma_row_col(floatx4_t& acc, const float* a_row, const float* b_k0, int pitch, int g) {
    const float4 a = *reinterpret_cast<const float4*>(a_row + 4 * g);
    const float* b = b_k0 + (size_t)(4 * g) * pitch;
    mfma4(acc, a, float4{b[0], b[pitch], b[2 * pitch], b[3 * pitch]});
}
// acc += A^T B over 16 values of k: the rows of both are k
__device__ __forceinline__ void mfma_col_col(floatx4_t& acc, const float* a_k0, int pa, const float* b_k0, int pb, int g) {
    const float* a = a_k0 + (size_t)(4 * g) * pa;
    const float* b = b_k0 + (size_t)(4 * g) * pb;
    mfma4(acc, float4{a[0], a[pa], a[2 * pa], a[3 * pa]}, float4{b[0], b[pb], b[2 * pb], b[3 * pb]});
}

// acc += A^T B^T over 16 values of k: the rows of A are k, B's rows hold neighbouring k side by side
__device__ __forceinline__ void mfma_col_row(floatx4_t& acc, const float* a_k0, int pa, const float* b_row, int g) {
    const float* a = a_k0 + (size_t)(4 * g) * pa;
    mfma4(acc, float4{a[0], a[pa], a[2 * pa], a[3 * pa]}, *reinterpret_cast<const float4*>(b_row + 4 * g));
}

// ---- how M, N and Q lie in memory: a tile of 16 x 16 is what one load of the walk's matrix operands takes, lane after lane
// (lane i + 16 g: row i, columns 4 g .. 4 g + 3), so that a load asks for whole lines. (Row by row, a load touched sixteen
// half lines, and the number of lines a compute unit asks for was what a step of the walk took: 0.9 us against 0.6; the
// walk of 2,048 tokens, 16 heads of 64, 57 -> 42 us.) A tile of fewer
// rows is packed: quad g of row i is number g * rows + i.
//   M: tiles (16 rows, 16 columns) of a (chunk, head), row tile by row tile
//   N: tiles (16 value columns as rows, 16 channels); Q: tiles (16 tokens, 16 channels), a chunk's heads one after the other
__device__ __forceinline__ size_t quad_of(int tile_row, int rows, int k_tile, int width, int i, int g) {
    return (size_t)tile_row * 16 * width + ((size_t)(4 * k_tile + g) * rows + i) * 4;
}

// ---- what concerns one chunk alone: workgroup (chunk, head)
// ROWS (general rule, heads of 64): the vectors are made here from the packed rows [r | k | v | g | a | w1], the decays' products over the rank on the
// MFMA units, and not by a kernel that leaves them in memory as floats: 42 MB written and read again for 2,048 rows of 16 heads.
// us, prepare + chunks / this: 2,048 rows 21.0 + 47.4 / 52.5, 552 rows 15.4 + 24.5 / 27.5. Where a step has requests for the scan too, those want the vectors.
// The mLSTM's (heads of 64 x 64) too: prepare + chunks / this at 2,048 rows of 16 heads 14.7 + 29.6 / 25.6.
// ROWS of 2 to 4 (channel and gated rules, heads of 64 x 64): so many taps of the convolution that queries, keys and values pass first;
// a token's four rows are read by four threads each, from L1. us, prepare + chunks / this: gated, 2,048 rows, 16 heads in 8 groups 21.5 + 41.1 / 47.1;
// channel, 941 and 483 rows, 16 heads in 8 groups 29.2 + 36.5 / 41.4.
// Heads of 128 have their vectors laid out still: a thread makes four channels of one token here, the workgroup 32 x 64, which is what
// the designs' heads are at 0.6B and above.
template <typename T, int DK, int RULE, int ROWS>
__global__ void __launch_bounds__(DC_THREADS)
delta_chunk_kernel(DeltaChunkArgs A) {
    constexpr int C = DC_TOKENS, R16 = DC_RUN;
    constexpr bool PAIR = RULE == RULE_GENERAL;                // b is not -x: sources of two kinds
    constexpr bool READ = RULE != RULE_SUM;
    constexpr int P = DK + 4;                                  // pitch of rows of key channels
    constexpr int DVMAX = PAIR ? DK : DK + 16, PV = DVMAX + 4; // of value columns (the general rule's heads are square)
    constexpr int PC = C + 4;                                  // of tokens
    __shared__ __attribute__((aligned(16))) float sA[READ ? C : 1][P], sX[C][P], sR[C][P], sW[C][P], sB[PAIR ? C : 1][P];
    __shared__ __attribute__((aligned(16))) float sV[C][PV];
    __shared__ __attribute__((aligned(16))) float mB[C][PC], mB2[PAIR ? C : 1][PC], mG[READ ? C : 1][PC];
    // U comes when A, A' and T have been used up, and takes their place: with a general rule's heads of 64 two workgroups share a
    // compute unit then (80 KB of LDS; 93 KB and one alone: 67 us a launch at 2,048 tokens and 16 heads against 48)
    constexpr int MROWS = READ ? C : 1, M2ROWS = PAIR ? C : 1;
    __shared__ __attribute__((aligned(16))) float once[(2 * MROWS + M2ROWS) * PC > MROWS * PV ? (2 * MROWS + M2ROWS) * PC : MROWS * PV];
    float (*mA)[PC] = reinterpret_cast<float (*)[PC]>(once), (*mT)[PC] = mA + MROWS, (*mA2)[PC] = mT + MROWS;
    float (*sU)[PV] = reinterpret_cast<float (*)[PV]>(once);
    __shared__ float full[2][DK];                              // a run's decays multiplied
    __shared__ int sh[8];
    int seq, row0, count;
    find_long_chunk(A.cu_seqlens, A.n_seqs, blockIdx.x, sh, seq, row0, count);
    if (count <= 0) return;
    const int head = blockIdx.y, H = A.H, DV = A.DV;
    const int tid = threadIdx.x, lane = tid % MV_WAVE, wave = tid / MV_WAVE, i = lane % 16, g = lane / 16;
    const int NT = (DV + 15) / 16;                             // tiles of value columns

    // the chunk's vectors; rows beyond its tokens change nothing (decay one, everything else zero)
    const int group = RULE == RULE_GENERAL ? head : head / (H / A.G);
    if constexpr (ROWS == 1 && RULE == RULE_SUM) {
        // (the scan's floats, bit for bit: the gates are there, the values have a column of ones behind them)
        static_assert(C * (DK / 4) == DC_THREADS && DVMAX == DK + 16, "four channels a thread");
        const int t = tid / 16, c = (tid % 16) * 4;
        const bool ok = t < count;
        const size_t row = row0 + (ok ? t : 0);
        const T* p = (const T*)A.vals + row * A.ldv + (size_t)head * DK + c;
        const size_t inner = (size_t)H * DK;
        const float4 q = four_of(p), k = four_of(p + inner), v = four_of(p + 2 * inner);
        const float w = A.gates[(row * H + head) * 4], b = A.gates[(row * H + head) * 4 + 1], qs = 1.f / sqrtf((float)DK);
        auto put = [&](float* to, float x, float y, float z, float e, float none) __attribute__((always_inline)) {
            *reinterpret_cast<float4*>(to) = ok ? float4{x, y, z, e} : float4{none, none, none, none};
        };
        put(&sW[t][c], w, w, w, w, 1.f);
        put(&sX[t][c], k.x, k.y, k.z, k.w, 0.f);
        put(&sR[t][c], q.x * qs, q.y * qs, q.z * qs, q.w * qs, 0.f);
        put(&sV[t][c], v.x * b, v.y * b, v.z * b, v.w * b, 0.f);
        if (c < 16) put(&sV[t][DK + c], c == 0 ? b : 0.f, 0.f, 0.f, 0.f, 0.f);
    } else if constexpr (ROWS == 1) {
        static_assert(RULE == RULE_GENERAL && C * (DK / 4) == DC_THREADS && DK / 4 == 16 && 2 * (DK / 16) == DC_THREADS / 64, "four channels a thread, a tile of decays a wave");
        constexpr int PT = DC_MAX_RANK + 4;
        static_assert(C * PT <= (2 * MROWS + M2ROWS) * PC, "no room for the rows of the decays' products");
        float (*th)[PT] = reinterpret_cast<float (*)[PT]>(once);               // (used up before A and A' come)
        const int t = tid / 16, c = (tid % 16) * 4, inner = H * DK, col = head * DK + c;
        const bool ok = t < count;
        const T* row = (const T*)A.vals + (size_t)(row0 + (ok ? t : 0)) * A.ldv;
        const float4 r = four_of(row + col), k = four_of(row + inner + col), v = four_of(row + 2 * (size_t)inner + col), az = four_of(row + 4 * (size_t)inner + col);
        const float4 z = four_of(row + 5 * (size_t)inner + (c < A.rank ? c : 0));
        // the wave's tile of decays: tokens 16 rt .., channels 16 ct ..; its weights are on their way meanwhile
        const int rt = wave % 2, ct = wave / 2, ch = head * DK + 16 * ct + i;
        float4 w2[DC_MAX_RANK / 16];
        float4 ab;
        float b0;
        auto weights = [&](const auto* w2t, const auto* w0, const auto* a_bias) __attribute__((always_inline)) {
#pragma unroll
            for (int b = 0; b < DC_MAX_RANK / 16; ++b) {
                const auto* at = w2t + (size_t)min(16 * b + 4 * g, A.rank - 4) * inner + ch;       // (the rank is a multiple of 16)
                w2[b] = float4{to_f(at[0]), to_f(at[inner]), to_f(at[2 * inner]), to_f(at[3 * inner])};
            }
            b0 = to_f(w0[ch]);
            ab = four_of(a_bias + col);
        };
        if (A.weights_f32) weights((const float*)A.w2t, (const float*)A.w0, (const float*)A.a_bias);
        else weights((const bf16*)A.w2t, (const bf16*)A.w0, (const bf16*)A.a_bias);
        const float inv = 1.f / sqrtf(lanes_sum<16>(fmaf(k.x, k.x, fmaf(k.y, k.y, fmaf(k.z, k.z, k.w * k.w)))) + A.key_eps);
        const float4 u{k.x * inv, k.y * inv, k.z * inv, k.w * inv};
        const float4 b{-sigmoid_f(az.x + ab.x) * u.x, -sigmoid_f(az.y + ab.y) * u.y, -sigmoid_f(az.z + ab.z) * u.z, -sigmoid_f(az.w + ab.w) * u.w};
        // (two names for the choice would be a choice between addresses, and both in scratch)
        auto there = [&](const float4& x) __attribute__((always_inline)) { return ok ? x : float4{0.f, 0.f, 0.f, 0.f}; };
        *reinterpret_cast<float4*>(&sX[t][c]) = there(k);
        *reinterpret_cast<float4*>(&sR[t][c]) = there(r);
        *reinterpret_cast<float4*>(&sA[t][c]) = there(u);
        *reinterpret_cast<float4*>(&sB[t][c]) = there(b);
        *reinterpret_cast<float4*>(&sV[t][c]) = there(v);
        if (c < A.rank) *reinterpret_cast<float4*>(&th[t][c]) = float4{tanhf(z.x), tanhf(z.y), tanhf(z.z), tanhf(z.w)};
        __syncthreads();
        floatx4_t acc{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int b = 0; b < DC_MAX_RANK / 16; ++b)
            if (16 * b < A.rank)
                mfma4(acc, *reinterpret_cast<const float4*>(&th[16 * rt + i][16 * b + 4 * g]), w2[b]);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int at = 16 * rt + 4 * g + q;
            sW[at][16 * ct + i] = at < count ? expf(-A.decay_rate * sigmoid_f(acc[q] + b0)) : 1.f;
        }
    } else if constexpr (ROWS > 1) {
        static_assert((RULE == RULE_CHANNEL || RULE == RULE_GATED) && C * (DK / 4) == DC_THREADS && DK / 4 == 16, "four channels a thread");
        constexpr int TAPS = ROWS;
        const int t = tid / 16, c = (tid % 16) * 4, G = A.G, width = 2 * G * DK + H * DK;
        const bool ok = t < count;
        const int row = row0 + (ok ? t : 0), first = A.cu_seqlens[seq];
        const T* const rows = (const T*)A.vals;
        const T* const kept = (const T*)A.conv_state + (size_t)A.state_slots[seq] * (TAPS - 1) * width;
        const T* in[TAPS];                             // the inputs' rows: of the step, or what was kept from before it
#pragma unroll
        for (int j = 0; j < TAPS; ++j) {
            const int r = row - (TAPS - 1) + j;
            in[j] = r >= first ? rows + (size_t)r * A.ldv : kept + (size_t)(TAPS - 1 + r - first) * width;
        }
        const T* const gates = rows + (size_t)row * A.ldv + A.gate_off + head;
        const float beta = sigmoid_f(to_f(gates[0]));
        auto make = [&](const auto* conv_w, const auto* a_log, const auto* dt_bias) __attribute__((always_inline)) {
            auto conv = [&](int col) __attribute__((always_inline)) {
                float w[4 * TAPS], acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int x = 0; x < TAPS; ++x) {
                    const float4 f = four_of(conv_w + (size_t)col * TAPS + 4 * x);
                    w[4 * x] = f.x; w[4 * x + 1] = f.y; w[4 * x + 2] = f.z; w[4 * x + 3] = f.w;
                }
#pragma unroll
                for (int j = 0; j < TAPS; ++j) {
                    const float4 f = four_of(in[j] + col);
                    acc[0] = fmaf(w[j], f.x, acc[0]);
                    acc[1] = fmaf(w[TAPS + j], f.y, acc[1]);
                    acc[2] = fmaf(w[2 * TAPS + j], f.z, acc[2]);
                    acc[3] = fmaf(w[3 * TAPS + j], f.w, acc[3]);
                }
                return float4{silu_f(acc[0]), silu_f(acc[1]), silu_f(acc[2]), silu_f(acc[3])};
            };
            auto inverse_length = [&](const float4& x) __attribute__((always_inline)) {
                return 1.f / sqrtf(lanes_sum<16>(fmaf(x.x, x.x, fmaf(x.y, x.y, fmaf(x.z, x.z, x.w * x.w)))) + A.unit_eps);
            };
            const float4 q = conv(group * DK + c), k = conv(G * DK + group * DK + c), v = conv(2 * G * DK + head * DK + c);
            float w[4];
            const float rate = -expf(to_f(a_log[head]));
            if constexpr (RULE == RULE_CHANNEL) {
                const float4 z = *reinterpret_cast<const float4*>(A.decay + (size_t)row * A.ldz + (size_t)head * DK + c), bias = four_of(dt_bias + head * DK + c);
                w[0] = expf(rate * softplus_f(z.x + bias.x));
                w[1] = expf(rate * softplus_f(z.y + bias.y));
                w[2] = expf(rate * softplus_f(z.z + bias.z));
                w[3] = expf(rate * softplus_f(z.w + bias.w));
            } else {
                w[0] = w[1] = w[2] = w[3] = expf(rate * softplus_f(to_f(gates[H]) + to_f(dt_bias[head])));
            }
            const float iq = 1.f / sqrtf((float)DK) * inverse_length(q), ik = inverse_length(k);
            const float4 u{k.x * ik, k.y * ik, k.z * ik, k.w * ik};
            auto put = [&](float (*to)[P], float x, float y, float z, float e, float none) __attribute__((always_inline)) {
                *reinterpret_cast<float4*>(&to[t][c]) = ok ? float4{x, y, z, e} : float4{none, none, none, none};
            };
            put(sW, w[0], w[1], w[2], w[3], 1.f);
            put(sR, q.x * iq, q.y * iq, q.z * iq, q.w * iq, 0.f);
            put(sA, w[0] * u.x, w[1] * u.y, w[2] * u.z, w[3] * u.w, 0.f);
            put(sX, beta * u.x, beta * u.y, beta * u.z, beta * u.w, 0.f);
            *reinterpret_cast<float4*>(&sV[t][c]) = ok ? float4{v.x, v.y, v.z, v.w} : float4{0.f, 0.f, 0.f, 0.f};
        };
        if (A.weights_f32) make((const float*)A.conv_w, (const float*)A.a_log, (const float*)A.dt_bias);
        else make((const bf16*)A.conv_w, (const bf16*)A.a_log, (const bf16*)A.dt_bias);
    } else {
        for (int x = tid; x < C * (DK / 4); x += DC_THREADS) {
            const int t = x / (DK / 4), c = (x % (DK / 4)) * 4;
            const bool ok = t < count;
            const size_t row = row0 + (ok ? t : 0);
            const float4 zero{0.f, 0.f, 0.f, 0.f};
            auto at = [&](const float* p) __attribute__((always_inline)) { return *reinterpret_cast<const float4*>(p + c); };
            float4 w, a = zero, xx, r, b = zero;
            if constexpr (RULE == RULE_GENERAL) {
                const float* v = A.vec + (row * H + head) * 5 * DK;
                w = at(v); b = at(v + DK); a = at(v + 2 * DK); xx = at(v + 3 * DK); r = at(v + 4 * DK);
                b = float4{-b.x, -b.y, -b.z, -b.w};
            } else {
                const float* v = A.vec + (row * A.G + group) * 2 * DK;
                r = at(v);
                xx = at(v + DK);
                if constexpr (RULE == RULE_CHANNEL) {
                    const float* d = A.decay + row * A.ldz + (size_t)head * DK;
                    w = A.decay4 ? at(d) : float4{d[c], d[c + 1], d[c + 2], d[c + 3]};
                } else {
                    const float d = A.gates[(row * H + head) * 4];
                    w = float4{d, d, d, d};
                }
                if constexpr (READ) {
                    const float beta = RULE == RULE_CHANNEL ? A.gates[row * H + head] : A.gates[(row * H + head) * 4 + 1];
                    a = float4{w.x * xx.x, w.y * xx.y, w.z * xx.z, w.w * xx.w};
                    xx = float4{beta * xx.x, beta * xx.y, beta * xx.z, beta * xx.w};
                }
            }
            *reinterpret_cast<float4*>(&sW[t][c]) = ok ? w : float4{1.f, 1.f, 1.f, 1.f};
            *reinterpret_cast<float4*>(&sX[t][c]) = ok ? xx : float4{0.f, 0.f, 0.f, 0.f};
            *reinterpret_cast<float4*>(&sR[t][c]) = ok ? r : float4{0.f, 0.f, 0.f, 0.f};
            if constexpr (READ) *reinterpret_cast<float4*>(&sA[t][c]) = ok ? a : float4{0.f, 0.f, 0.f, 0.f};
            if constexpr (PAIR) *reinterpret_cast<float4*>(&sB[t][c]) = ok ? b : float4{0.f, 0.f, 0.f, 0.f};
        }
        for (int x = tid; x < C * DVMAX; x += DC_THREADS) {
            const int t = x / DVMAX, j = x % DVMAX;
            const bool ok = t < count && j < DV;
            const size_t row = row0 + (ok ? t : 0);
            const int jj = ok ? j : 0;
            float v;
            if constexpr (RULE == RULE_GENERAL) v = to_f(((const T*)A.vals)[row * A.ldv + 2 * (size_t)H * DK + (size_t)head * DK + jj]);
            else v = ((const float*)A.vals)[(row * H + head) * DV + jj];
            if constexpr (RULE == RULE_SUM) v *= A.gates[(row * H + head) * 4 + 1];
            sV[t][j] = ok ? v : 0.f;
        }
    }
    __syncthreads();

    // A and B inside a run: LP lanes share a source token s and walk t along its run with what is left of x_s
    constexpr int LP = 16, CH = DK / LP;                       // channels of a lane
    static_assert(C * LP == DC_THREADS, "a source token for every sixteen lanes");
    {
        const int src = tid / LP, first = src / R16 * R16, s = src % R16, c = (tid % LP) * CH;
        float d[CH], e[CH];
        auto take = [&](float (&v)[CH], const float* p) __attribute__((always_inline)) {
#pragma unroll
            for (int q = 0; q < CH; q += 4) {
                const float4 x = *reinterpret_cast<const float4*>(p + q);
                v[q] = x.x; v[q + 1] = x.y; v[q + 2] = x.z; v[q + 3] = x.w;
            }
        };
        take(d, &sX[src][c]);
        if constexpr (PAIR) take(e, &sB[src][c]);
#pragma unroll 4
        for (int t = 0; t < R16; ++t) {
            const int row = first + t;
            float w[CH], r[CH], da = 0.f, db = 0.f, ea = 0.f, eb = 0.f;
            take(w, &sW[row][c]);
            take(r, &sR[row][c]);
            const bool behind = t > s;
            if constexpr (READ) {
                float a[CH];
                take(a, &sA[row][c]);
#pragma unroll
                for (int q = 0; q < CH; ++q) {
                    da = fmaf(a[q], d[q], da);
                    if constexpr (PAIR) ea = fmaf(a[q], e[q], ea);
                }
            }
#pragma unroll
            for (int q = 0; q < CH; ++q) {
                d[q] = behind ? d[q] * w[q] : d[q];
                db = fmaf(r[q], d[q], db);
                if constexpr (PAIR) {
                    e[q] = behind ? e[q] * w[q] : e[q];
                    eb = fmaf(r[q], e[q], eb);
                }
            }
            if constexpr (READ) da = lanes_sum<LP>(da);
            db = lanes_sum<LP>(db);
            if constexpr (PAIR) { ea = lanes_sum<LP>(ea); eb = lanes_sum<LP>(eb); }
            if (tid % LP == 0) {
                if constexpr (READ) mA[row][src] = behind ? da : 0.f;
                mB[row][src] = t >= s ? db : 0.f;
                if constexpr (PAIR) {
                    mA2[row][src] = behind ? ea : 0.f;
                    mB2[row][src] = t >= s ? eb : 0.f;
                }
            }
        }
    }
    __syncthreads();

    // what is left of a token's sources at its run's end, and of a run's start at a token
    for (int x = tid; x < 4 * DK; x += DC_THREADS) {
        const int c = x % DK, run = (x / DK) % 2, first = run * R16;
        float f = 1.f;
        if (x < 2 * DK) {
            for (int t = 0; t < R16; ++t) {
                if constexpr (READ) sA[first + t][c] *= f;
                f *= sW[first + t][c];
                sR[first + t][c] *= f;
            }
            full[run][c] = f;
        } else {
            for (int t = R16 - 1; t >= 0; --t) {
                sX[first + t][c] *= f;
                if constexpr (PAIR) sB[first + t][c] *= f;
                f *= sW[first + t][c];
            }
        }
    }
    // (no token of the first run sees the second)
    if (tid < R16 * R16) {
        const int t = tid / R16, s = R16 + tid % R16;
        mB[t][s] = 0.f;
        if constexpr (READ) mA[t][s] = 0.f;
        if constexpr (PAIR) mA2[t][s] = mB2[t][s] = 0.f;
        if constexpr (READ) mT[t][s] = 0.f;
    }
    __syncthreads();

    // between the runs, and (first wave) the inverses of the two runs' own blocks, a column a lane
    auto between = [&](float (*dst)[PC], const float (&rows)[C][P], const float (&cols)[C][P]) __attribute__((always_inline)) {
        floatx4_t acc{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < DK; k += 16)
            mfma4(acc, *reinterpret_cast<const float4*>(&rows[R16 + i][k + 4 * g]), *reinterpret_cast<const float4*>(&cols[i][k + 4 * g]));
#pragma unroll
        for (int q = 0; q < 4; ++q) dst[R16 + 4 * g + q][i] = acc[q];
    };
    if (wave == 1) between(mB, sR, sX);
    if constexpr (READ) {
        if (wave == 2) between(mA, sA, sX);
        if constexpr (PAIR) {
            if (wave == 3) between(mA2, sA, sB);
            if (wave == 5) between(mB2, sR, sB);
        }
        if (wave == 0 && lane < C) {
            const int first = lane / R16 * R16, c = lane % R16;
            float col[R16];
#pragma unroll
            for (int t = 0; t < R16; ++t) {
                float acc = t == c ? 1.f : 0.f;
#pragma unroll
                for (int s = 0; s < t; ++s) {
                    if constexpr (PAIR) acc = fmaf(mA2[first + t][first + s], col[s], acc);
                    else acc = fmaf(-mA[first + t][first + s], col[s], acc);
                }
                col[t] = acc;
                mT[first + t][first + c] = acc;
            }
        }
    }
    __syncthreads();
    // the inverse's block between the runs: T22 (A'21 T11); the sources of the first run reach the chunk's end, the
    // second run's tokens the chunk's start
    if constexpr (READ) {
        if (wave == 0) {
            floatx4_t acc{0.f, 0.f, 0.f, 0.f};
            mfma_row_col(acc, PAIR ? &mA2[R16 + i][0] : &mA[R16 + i][0], &mT[0][i], PC, g);
#pragma unroll
            for (int q = 0; q < 4; ++q) mG[4 * g + q][i] = PAIR ? acc[q] : -acc[q];
        }
    }
    for (int x = tid; x < R16 * DK; x += DC_THREADS) {
        const int t = x / DK, c = x % DK;
        sR[R16 + t][c] *= full[0][c];
        if constexpr (READ) sA[R16 + t][c] *= full[0][c];
        sX[t][c] *= full[1][c];
        if constexpr (PAIR) sB[t][c] *= full[1][c];
    }
    __syncthreads();
    if constexpr (READ) {
        if (wave == 0) {
            floatx4_t acc{0.f, 0.f, 0.f, 0.f};
            mfma_row_col(acc, &mT[R16 + i][R16], &mG[0][i], PC, g);
#pragma unroll
            for (int q = 0; q < 4; ++q) mT[R16 + 4 * g + q][i] = acc[q];
        }
        __syncthreads();
        // W = T (a P) over the decays' rows, which are used up; G = T A
        for (int job = wave; job < 2 * (DK / 16) + 4; job += DC_THREADS / 64) {
            const bool is_w = job < 2 * (DK / 16);
            const int rt = is_w ? job % 2 : (job - 2 * (DK / 16)) % 2, ct = is_w ? job / 2 : (job - 2 * (DK / 16)) / 2;
            floatx4_t acc{0.f, 0.f, 0.f, 0.f};
            for (int k = 0; k <= 16 * rt; k += 16)
                mfma_row_col(acc, &mT[16 * rt + i][k], is_w ? &sA[k][16 * ct + i] : &mA[k][16 * ct + i], is_w ? P : PC, g);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (is_w) sW[16 * rt + 4 * g + q][16 * ct + i] = acc[q];
                else mG[16 * rt + 4 * g + q][16 * ct + i] = acc[q];
            }
        }
        __syncthreads();
        // U = G V, or what replaces V where b = -x: V - U
        for (int job = wave; job < 2 * NT; job += DC_THREADS / 64) {
            const int rt = job % 2, ct = job / 2;
            floatx4_t acc{0.f, 0.f, 0.f, 0.f};
            for (int k = 0; k <= 16 * rt; k += 16) mfma_row_col(acc, &mG[16 * rt + i][k], &sV[k][16 * ct + i], PV, g);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int t = 16 * rt + 4 * g + q;
                sU[t][16 * ct + i] = PAIR ? acc[q] : sV[t][16 * ct + i] - acc[q];
            }
        }
        __syncthreads();
    }
    // what the walk needs
    const size_t unit = (size_t)blockIdx.x * H + head;
    float* q_out = A.Q + ((size_t)row0 * H + (size_t)head * count) * DK;
    const float (*E)[PV] = (READ && !PAIR) ? sU : sV;          // the values the sources x carry
    constexpr int KT = DK / 16;
    const int jobs_n = NT * KT, jobs_m = READ ? KT * KT : 0, jobs_q = READ ? 2 * KT : 0, jobs_o = 2 * NT;
    for (int job = wave; job < jobs_n + jobs_m + jobs_q + jobs_o; job += DC_THREADS / 64) {
        floatx4_t acc{0.f, 0.f, 0.f, 0.f};
        int j = job;
        if (j < jobs_n) {                                      // N: columns of the product are value columns
            const int vt = j / KT, kt = j % KT, rows = min(16, DV - 16 * vt);
#pragma unroll
            for (int k = 0; k < C; k += 16) {
                mfma_col_col(acc, &sX[k][16 * kt + i], P, &E[k][16 * vt + i], PV, g);
                if constexpr (PAIR) mfma_col_col(acc, &sB[k][16 * kt + i], P, &sU[k][16 * vt + i], PV, g);
            }
            if (i < rows) *reinterpret_cast<floatx4_t*>(A.N + unit * DV * DK + quad_of(vt, rows, kt, DK, i, g)) = acc;
            continue;
        }
        j -= jobs_n;
        if (j < jobs_m) {
            const int rt = j / KT, ct = j % KT;
#pragma unroll
            for (int k = 0; k < C; k += 16)
                mfma_col_col(acc, &sW[k][16 * ct + i], P, PAIR ? &sB[k][16 * rt + i] : &sX[k][16 * rt + i], P, g);
#pragma unroll
            for (int q = 0; q < 4; ++q) {                      // (columns of the product are rows of M)
                const int r = 16 * rt + i, c = 16 * ct + 4 * g + q;
                const float m = PAIR ? acc[q] : -acc[q];
                acc[q] = r == c ? full[0][c] * full[1][c] + m : m;
            }
            *reinterpret_cast<floatx4_t*>(A.M + unit * DK * DK + quad_of(rt, 16, ct, DK, i, g)) = acc;
            continue;
        }
        j -= jobs_m;
        if (j < jobs_q) {
            const int rt = j % 2, ct = j / 2, rows = min(16, count - 16 * rt);
            for (int k = 0; k <= 16 * rt; k += 16)
                mfma_col_row(acc, &sW[k][16 * ct + i], P, PAIR ? &mB2[16 * rt + i][k] : &mB[16 * rt + i][k], g);
            const float4 r = *reinterpret_cast<const float4*>(&sR[16 * rt + i][16 * ct + 4 * g]);
            const floatx4_t left{r.x, r.y, r.z, r.w};
            acc = PAIR ? left + acc : left - acc;
            if (i < rows) *reinterpret_cast<floatx4_t*>(q_out + quad_of(rt, rows, ct, DK, i, g)) = acc;
            continue;
        }
        j -= jobs_q;
        const int rt = j % 2, ct = j / 2;
        for (int k = 0; k <= 16 * rt; k += 16) {
            mfma_row_col(acc, &mB[16 * rt + i][k], &E[k][16 * ct + i], PV, g);
            if constexpr (PAIR) mfma_row_col(acc, &mB2[16 * rt + i][k], &sU[k][16 * ct + i], PV, g);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int t = 16 * rt + 4 * g + q, v = 16 * ct + i;
            if (t < count && v < DV) A.out[((size_t)(row0 + t) * H + head) * DV + v] = acc[q];
        }
    }
    if constexpr (!READ) {                                     // M is the one decay of the chunk, Q the queries as they are left
        if (tid == 0) A.M[unit] = full[0][0] * full[1][0];
        for (int x = tid; x < C * (DK / 4); x += DC_THREADS) {
            const int t = x % C, quad = x / C, rows = min(16, count - t / 16 * 16);
            if (t < count)
                *reinterpret_cast<float4*>(q_out + quad_of(t / 16, rows, quad / 4, DK, t % 16, quad % 4)) = *reinterpret_cast<const float4*>(&sR[t][4 * quad]);
        }
    }
}

// ---- the walk: workgroup (request, head, 16 value columns). The first KT waves own 16 rows of the state each, the last
// four the output: waves of one SIMD unit then share its matrix unit evenly. An output wave owns 16 tokens and half of
// the key channels; the two halves of a tile meet in LDS a step later. What a step reads of memory is asked for DEPTH
// steps ahead, and always asked for, also by steps beyond the last chunk (DEPTH divides the number of steps) and by
// lanes that have no use for it; what they would store falls outside the window of the buffer instruction, which drops it.
// So no load or store stands under a condition (behind one, the wait for an older load becomes a wait for newer ones
// too), and a step's addresses are one scalar base each: the lanes' offsets hardly change. (Addresses of 64 bits a lane
// and stores under conditions were two thirds of the output waves' instructions; mLSTM, 2,048 tokens, 36 -> 30 us, and 26 with the operands in order.)
template <int DK, bool READ>
__global__ void __launch_bounds__((DK / 16 + 4) * 64)
delta_chunk_walk_kernel(DeltaChunkArgs A, float* __restrict__ state, const int* __restrict__ state_slots) {
    constexpr int KT = DK / 16, DEPTH = DK <= 64 ? 4 : 2, P = DK + 4;
    constexpr uint32_t NOWHERE = 0x80000000u;                              // beyond every window
    __shared__ __attribute__((aligned(16))) float sS[2][16][P];            // the state in front of the chunk, column by column
    __shared__ floatx4_t sO[2][4][MV_WAVE];                                // the output waves' tiles
    __shared__ int part[8];
    const int seq = blockIdx.x, head = blockIdx.y, v0 = blockIdx.z * 16, H = A.H, DV = A.DV;
    const int begin = A.cu_seqlens[seq], len = A.cu_seqlens[seq + 1] - begin;
    if (len < DC_LINE) return;
    const int tid = threadIdx.x, lane = tid % MV_WAVE, i = lane % 16, g = lane / 16;
    const int wave = __builtin_amdgcn_readfirstlane(tid / MV_WAVE);
    int before = 0;                                                        // chunks in front of the request's
    for (int s = tid; s < seq; s += 256) {
        const int l = A.cu_seqlens[s + 1] - A.cu_seqlens[s];
        if (tid < 256 && l >= DC_LINE) before += (l + DC_TOKENS - 1) / DC_TOKENS;
    }
#pragma unroll
    for (int o = MV_WAVE / 2; o > 0; o >>= 1) before += __shfl_xor(before, o, MV_WAVE);
    if (lane == 0 && wave < 4) part[wave] = before;
    __syncthreads();
    const int c0 = __builtin_amdgcn_readfirstlane(part[0] + part[1] + part[2] + part[3]);
    const int chunks = (len + DC_TOKENS - 1) / DC_TOKENS;
    const int v = v0 + i;
    const bool live = v < DV;
    const int vc = live ? v : 0;
    const int steps = (chunks + DEPTH - 1) / DEPTH * DEPTH;

    // A step: what the step before left in LDS is asked for, then, while it comes, what a later step reads of memory, into the registers that
    // the step before has used; then the products, and the workgroup meets. (Asked for at a step's end, with addresses made anew from the chunk's number, it
    // stood between the state and the barrier: 2,048 tokens, 16 heads of 64 42 -> 37 us, 8 heads of 128 73 -> 66, two requests of 4,096 86 -> 76.)
    if (wave < KT) {
        float* st = state + (((size_t)state_slots[seq] * H + head) * DV + vc) * DK + 16 * wave + 4 * g;
        float4 s = *reinterpret_cast<const float4*>(st);
        if (!live) s = float4{0.f, 0.f, 0.f, 0.f};
        *reinterpret_cast<float4*>(&sS[0][i][16 * wave + 4 * g]) = s;
        float4 m[DEPTH][READ ? KT : 1], nn[DEPTH];
        float decay[DEPTH];
        const uint32_t m_at = 4u * quad_of(wave, 16, 0, DK, i, g);
        const uint32_t n_at = live ? 4u * quad_of(v0 / 16, min(16, DV - v0), wave, DK, i, g) : NOWHERE;
        const size_t unit0 = (size_t)c0 * H + head, step_m = (size_t)H * (READ ? DK * DK : 1), step_n = (size_t)H * DV * DK;
        const float *next_m = A.M + unit0 * (READ ? DK * DK : 1), *next_n = A.N + unit0 * DV * DK;
        int left = chunks - 1;                                              // chunks behind the next one to ask for
        auto fetch = [&](int d) __attribute__((always_inline)) {
            if constexpr (READ) {
                const BufferWindow w(next_m, 4u * DK * DK);
#pragma unroll
                for (int k = 0; k < KT; ++k) m[d][k] = w.load4(m_at, 1024 * k);
            } else {
                decay[d] = *next_m;
            }
            nn[d] = BufferWindow(next_n, 4u * DV * DK).load4(n_at, 0);
            next_m += left > 0 ? step_m : 0;                                // (behind the last chunk the last again)
            next_n += left > 0 ? step_n : 0;
            --left;
        };
#pragma unroll
        for (int d = 0; d < DEPTH - 1; ++d) fetch(d);
        __builtin_amdgcn_s_setprio(2);                                      // (the chain of the states is what the walk waits for)
        __syncthreads();
        for (int b = 0; b < steps; b += DEPTH) {
#pragma unroll
            for (int d = 0; d < DEPTH; ++d) {
                const int c = b + d;
                float4 sv[READ ? KT : 1];
                if constexpr (READ) {
#pragma unroll
                    for (int k = 0; k < KT; ++k) sv[k] = *reinterpret_cast<const float4*>(&sS[d % 2][i][16 * k + 4 * g]);
                }
                fetch((d + DEPTH - 1) % DEPTH);
                __builtin_amdgcn_sched_barrier(0);
                floatx4_t acc{nn[d].x, nn[d].y, nn[d].z, nn[d].w}, acc2{0.f, 0.f, 0.f, 0.f};
                if constexpr (READ) {
#pragma unroll
                    for (int k = 0; k < KT; k += 2) {
                        mfma4(acc, m[d][k], sv[k]);
                        mfma4(acc2, m[d][k + 1], sv[k + 1]);
                    }
                    acc += acc2;
                } else {
                    acc[0] = fmaf(decay[d], s.x, acc[0]);
                    acc[1] = fmaf(decay[d], s.y, acc[1]);
                    acc[2] = fmaf(decay[d], s.z, acc[2]);
                    acc[3] = fmaf(decay[d], s.w, acc[3]);
                }
                const bool moves = live && c < chunks;
                s = float4{moves ? acc[0] : s.x, moves ? acc[1] : s.y, moves ? acc[2] : s.z, moves ? acc[3] : s.w};
                *reinterpret_cast<float4*>(&sS[(d + 1) % 2][i][16 * wave + 4 * g]) = s;
                __syncthreads();
            }
        }
        if (live) *reinterpret_cast<float4*>(st) = s;
        __syncthreads();
    } else {
        const int ow = wave - KT, tile = ow % 2, half = ow / 2;             // 16 tokens, half of the key channels
        const int last = len - (chunks - 1) * DC_TOKENS;                    // tokens of the last chunk
        float4 qv[DEPTH][KT / 2];
        float ov[DEPTH][4];
        // rows of a chunk behind the request's last fall outside the windows: they read zero and store nothing
        const uint32_t o_row = 4u * H * DV;
        uint32_t o_at[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) o_at[q] = half == 0 && live ? (16 * tile + 4 * g + q) * o_row + 4u * v : NOWHERE;
        const uint32_t o_bytes = (DC_TOKENS - 1) * o_row + 4u * DV, o_last = (last - 1) * o_row + 4u * DV;
        const int rows_last = max(0, min(16, last - 16 * tile));
        const uint32_t q_at = 4u * quad_of(tile, 16, half * (KT / 2), DK, i, g);
        const uint32_t q_last = 4u * quad_of(tile, rows_last, half * (KT / 2), DK, i, g);
        const size_t step_q = (size_t)DC_TOKENS * H * DK, step_o = (size_t)DC_TOKENS * H * DV;
        const float* next_q = A.Q + ((size_t)begin * H + (size_t)head * (chunks > 1 ? DC_TOKENS : last)) * DK;
        const float* next_o = A.out + ((size_t)begin * H + head) * DV;
        float* store_o = A.out + ((size_t)begin * H + head) * DV;
        int left = chunks - 1;
        auto fetch = [&](int d) __attribute__((always_inline)) {
            const bool end = left <= 0;
            const BufferWindow w(next_q, 4u * (end ? last : DC_TOKENS) * DK);
            const uint32_t at = end ? q_last : q_at, more = end ? 64u * rows_last : 1024u;
#pragma unroll
            for (int k = 0; k < KT / 2; ++k) qv[d][k] = w.load4(at + more * k, 0);
            const BufferWindow o(next_o, end ? o_last : o_bytes);
#pragma unroll
            for (int q = 0; q < 4; ++q) ov[d][q] = o.load(o_at[q], 0);
            // (the last chunk's heads lie closer together)
            next_q += end ? 0 : left == 1 ? step_q - (size_t)head * (DC_TOKENS - last) * DK : step_q;
            next_o += end ? 0 : step_o;
            --left;
        };
#pragma unroll
        for (int d = 0; d < DEPTH - 1; ++d) fetch(d);
        floatx4_t held{0.f, 0.f, 0.f, 0.f};                                 // this wave's half of the step before
        auto store = [&](int c, const floatx4_t& other) __attribute__((always_inline)) {    // the tile of chunk c
            const floatx4_t o = held + other;
            const bool there = c >= 0 && c < chunks;
            const BufferWindow w(store_o, there ? (c == chunks - 1 ? o_last : o_bytes) : 0u);
#pragma unroll
            for (int q = 0; q < 4; ++q) w.store(o[q], o_at[q]);
            store_o += there ? step_o : 0;
        };
        sO[1][ow][lane] = held;                                             // (what the first step reads; it stores nothing)
        __syncthreads();
        for (int b = 0; b < steps; b += DEPTH) {
#pragma unroll
            for (int d = 0; d < DEPTH; ++d) {
                const int c = b + d;
                float4 sv[KT / 2];
#pragma unroll
                for (int k = 0; k < KT / 2; ++k)
                    sv[k] = *reinterpret_cast<const float4*>(&sS[d % 2][i][half * (DK / 2) + 16 * k + 4 * g]);
                const floatx4_t other = sO[(d + 1) % 2][ow ^ 2][lane];
                fetch((d + DEPTH - 1) % DEPTH);
                __builtin_amdgcn_sched_barrier(0);
                floatx4_t acc{ov[d][0], ov[d][1], ov[d][2], ov[d][3]};      // (zero for the second half)
#pragma unroll
                for (int k = 0; k < KT / 2; ++k) mfma4(acc, qv[d][k], sv[k]);
                store(c - 1, other);
                held = acc;
                sO[d % 2][ow][lane] = acc;
                __syncthreads();
            }
        }
        __syncthreads();
        store(steps - 1, sO[1][ow ^ 2][lane]);
    }
}

extern "C" int mv_delta_chunk_tokens() { return DC_TOKENS; }
extern "C" int mv_delta_chunk_line() { return DC_LINE; }
// 1: heads of these sizes are served
extern "C" int mv_delta_chunks_serve(int rule, int DK, int DV) {
    return rule >= RULE_GENERAL && rule <= RULE_SUM && (DK == 64 || DK == 128) && DV >= 1 && DV <= DK + 16;
}

template <typename T, int DK, int RULE, int ROWS = 0>
static int launch_delta_chunks(const DeltaChunkArgs& A, float* state, const int* state_slots, int chunks, hipStream_t stream) {
    hipLaunchKernelGGL((delta_chunk_kernel<T, DK, RULE, ROWS>), dim3(chunks, A.H), dim3(DC_THREADS), 0, stream, A);
    if (mv_check_launch("delta_chunk")) return 1;
    hipLaunchKernelGGL((delta_chunk_walk_kernel<DK, RULE != RULE_SUM>), dim3(A.n_seqs, A.H, (A.DV + 15) / 16), dim3((DK / 16 + 4) * 64), 0,
                       stream, A, state, state_slots);
    return mv_check_launch("delta_chunk_walk");
}

// The requests of at least mv_delta_chunk_line() tokens; `chunks`: an upper bound of their chunks (the rest of the grid
// ends at once). M [chunks][H][DK][DK] (RULE_SUM: [chunks][H]), N [chunks][H][DV][DK] and Q [n][H][DK] are scratch.
extern "C" int mv_delta_chunks(int rule, const float* vec, const float* gates, const float* decay, long ldz, const void* vals, long ldv,
                               float* state, const int* cu_seqlens, const int* state_slots, int n_seqs, int n, int H, int G, int DK, int DV,
                               int chunks, float* M, float* N, float* Q, float* out, int dtype, hipStream_t stream) {
    MV_REQUIRE(n >= 0 && n_seqs >= 0 && H > 0 && G > 0 && H % G == 0 && chunks >= 0, "delta_chunks: bad sizes n=%d seqs=%d H=%d G=%d", n, n_seqs, H, G);
    MV_REQUIRE(mv_delta_chunks_serve(rule, DK, DV), "delta_chunks: rule %d with heads of %d x %d is not served", rule, DK, DV);
    MV_REQUIRE(vec && vals && state && cu_seqlens && state_slots && M && N && Q && out, "delta_chunks: missing operand");
    MV_REQUIRE(rule != RULE_GENERAL || (G == H && DV == DK && ldv >= 3L * H * DK && mv_valid_dtype(dtype)), "delta_chunks: rows do not hold r, k and v");
    MV_REQUIRE(rule == RULE_GENERAL || gates, "delta_chunks: missing gates");
    MV_REQUIRE(rule != RULE_CHANNEL || (decay && ldz >= (long)H * DK), "delta_chunks: decays do not fit");
    MV_REQUIRE((uintptr_t)vec % 16 == 0 && (uintptr_t)state % 16 == 0 && (uintptr_t)M % 16 == 0 && (uintptr_t)N % 16 == 0 && (uintptr_t)Q % 16 == 0,
               "delta_chunks: operands must be 16-byte aligned");
    MV_REQUIRE(H <= 65535, "delta_chunks: too many heads");
    if (n == 0 || n_seqs == 0 || chunks == 0) return 0;
    const int decay4 = ldz % 4 == 0 && (uintptr_t)decay % 16 == 0;
    const DeltaChunkArgs A{vec, gates, decay, ldz, decay4, vals, ldv, H, G, DV, cu_seqlens, n_seqs, M, N, Q, out, 0, nullptr, nullptr, nullptr, 0, 0.f, 0.f,
                           nullptr, nullptr, nullptr, nullptr, nullptr, 0, 0.f};
#define DC_LAUNCH(T, RULE)                                                                                   \
    return DK == 64 ? launch_delta_chunks<T, 64, RULE>(A, state, state_slots, chunks, stream)               \
                    : launch_delta_chunks<T, 128, RULE>(A, state, state_slots, chunks, stream)
    switch (rule) {
        case RULE_GENERAL: MV_DISPATCH_T(dtype, "delta_chunks", { DC_LAUNCH(T, RULE_GENERAL); }); break;
        case RULE_CHANNEL: DC_LAUNCH(float, RULE_CHANNEL);
        case RULE_GATED: DC_LAUNCH(float, RULE_GATED);
        default: DC_LAUNCH(float, RULE_SUM);
    }
#undef DC_LAUNCH
    return 0;
}

// 1: mv_delta_chunks_rows serves heads of this size and decays of this rank, rows this far apart
extern "C" int mv_delta_chunks_rows_serve(int D, int rank, long ld) { return D == 64 && rank > 0 && rank <= DC_MAX_RANK && rank % 16 == 0 && ld % 8 == 0; }

// mv_delta_chunks under the general rule straight from the packed rows, without the vectors of mv_delta_prepare (ROWS above).
extern "C" int mv_delta_chunks_rows(const void* packed, long ld, int rank, const void* w2t, const void* w0, const void* a_bias, int weight_dtype,
                                    float decay_rate, float key_eps, float* state, const int* cu_seqlens, const int* state_slots, int n_seqs, int n, int H,
                                    int D, int chunks, float* M, float* N, float* Q, float* out, int dtype, hipStream_t stream) {
    MV_REQUIRE(n >= 0 && n_seqs >= 0 && H > 0 && H <= 65535 && chunks >= 0, "delta_chunks_rows: bad sizes n=%d seqs=%d H=%d", n, n_seqs, H);
    MV_REQUIRE(mv_delta_chunks_rows_serve(D, rank, ld) && ld >= 5L * H * D + rank, "delta_chunks_rows: heads of %d, rank %d, rows of %ld columns are not served", D, rank, ld);
    MV_REQUIRE(packed && w2t && w0 && a_bias && state && cu_seqlens && state_slots && M && N && Q && out, "delta_chunks_rows: missing operand");
    MV_REQUIRE(mv_valid_dtype(weight_dtype) && key_eps > 0.f, "delta_chunks_rows: an unknown weight type, or key_eps is not positive");
    MV_REQUIRE((uintptr_t)packed % 16 == 0 && (uintptr_t)a_bias % 16 == 0 && (uintptr_t)state % 16 == 0 && (uintptr_t)M % 16 == 0 && (uintptr_t)N % 16 == 0
               && (uintptr_t)Q % 16 == 0, "delta_chunks_rows: operands must be 16-byte aligned");
    if (n == 0 || n_seqs == 0 || chunks == 0) return 0;
    const DeltaChunkArgs A{nullptr, nullptr, nullptr, 0, 0, packed, ld, H, H, D, cu_seqlens, n_seqs, M, N, Q, out, rank, w2t, w0, a_bias,
                           weight_dtype == MV_F32, decay_rate, key_eps, nullptr, nullptr, nullptr, nullptr, nullptr, 0, 0.f};
    MV_DISPATCH_T(dtype, "delta_chunks_rows", { return (launch_delta_chunks<T, 64, RULE_GENERAL, 1>(A, state, state_slots, chunks, stream)); });
    return 0;
}

// 1: mv_delta_chunks_conv serves heads of these sizes, so many taps, rows this far apart (ldz: the decays', 0: none)
extern "C" int mv_delta_chunks_conv_serve(int DK, int DV, int taps, long ld, long ldz) {
    return DK == 64 && DV == 64 && taps >= 2 && taps <= 4 && ld % 8 == 0 && ldz % 4 == 0;
}

// mv_delta_chunks under the channel or the gated rule straight from the packed rows, without the vectors of mv_channel_prepare and mv_gdelta_prepare
// (ROWS above), and the convolution's kept inputs moved on behind it. gate_off: the column of the strengths, the gated rule's decays H behind them;
// z: the channel rule's decays in front of bias and exponential, rows ldz apart, left as they are.
extern "C" int mv_delta_chunks_conv(int rule, const void* packed, long ld, int gate_off, int taps, const void* conv_w, const void* a_log, const void* dt_bias,
                                    int weight_dtype, void* conv_state, float unit_eps, const float* z, long ldz, float* state, const int* cu_seqlens,
                                    const int* state_slots, int n_seqs, int n, int H, int G, int DK, int DV, int chunks, float* M, float* N, float* Q, float* out,
                                    int dtype, hipStream_t stream) {
    const bool channel = rule == RULE_CHANNEL;
    MV_REQUIRE(n >= 0 && n_seqs >= 0 && H > 0 && H <= 65535 && G > 0 && H % G == 0 && chunks >= 0, "delta_chunks_conv: bad sizes n=%d seqs=%d H=%d G=%d", n, n_seqs, H, G);
    MV_REQUIRE((channel || rule == RULE_GATED) && mv_delta_chunks_conv_serve(DK, DV, taps, ld, channel ? ldz : 0),
               "delta_chunks_conv: rule %d with heads of %d x %d, %d taps, rows of %ld is not served", rule, DK, DV, taps, ld);
    const long width = 2L * G * DK + (long)H * DV;
    MV_REQUIRE(gate_off >= width && ld >= (long)gate_off + (channel ? 1 : 2) * H, "delta_chunks_conv: rows of %ld columns are too short", ld);
    MV_REQUIRE(packed && conv_w && a_log && dt_bias && conv_state && state && cu_seqlens && state_slots && M && N && Q && out
               && (!channel || (z && ldz >= (long)H * DK)), "delta_chunks_conv: missing operand");
    MV_REQUIRE(mv_valid_dtype(weight_dtype) && unit_eps > 0.f && (width + 255) / 256 <= 65535, "delta_chunks_conv: bad constants");
    MV_REQUIRE(((uintptr_t)packed | (uintptr_t)conv_w | (uintptr_t)dt_bias | (uintptr_t)conv_state | (uintptr_t)z | (uintptr_t)state | (uintptr_t)M | (uintptr_t)N
                | (uintptr_t)Q) % 16 == 0, "delta_chunks_conv: operands must be 16-byte aligned");
    if (n == 0 || n_seqs == 0 || chunks == 0) return 0;
    const DeltaChunkArgs A{nullptr, nullptr, z, ldz, 1, packed, ld, H, G, DV, cu_seqlens, n_seqs, M, N, Q, out, 0, nullptr, nullptr, nullptr,
                           weight_dtype == MV_F32, 0.f, 0.f, conv_w, a_log, dt_bias, conv_state, state_slots, gate_off, unit_eps};
    int rc = 1;
#define DC_CONV(RULE)                                                                                                            \
    MV_DISPATCH_T(dtype, "delta_chunks_conv", {                                                                                  \
        rc = taps == 4   ? launch_delta_chunks<T, 64, RULE, 4>(A, state, state_slots, chunks, stream)                            \
             : taps == 3 ? launch_delta_chunks<T, 64, RULE, 3>(A, state, state_slots, chunks, stream)                            \
                         : launch_delta_chunks<T, 64, RULE, 2>(A, state, state_slots, chunks, stream);                           \
    })
    if (channel) {
        DC_CONV(RULE_CHANNEL);
    } else {
        DC_CONV(RULE_GATED);
    }
#undef DC_CONV
    if (rc) return rc;
    MV_DISPATCH_T(dtype, "conv_state",
                  hipLaunchKernelGGL(conv_state_kernel<T>, dim3(n_seqs, (unsigned)((width + 255) / 256)), dim3(256), 0, stream, (const T*)packed, ld, (int)width,
                                     taps, (T*)conv_state, cu_seqlens, state_slots));
    return mv_check_launch("conv_state");
}

// mv_delta_chunks under the mLSTM's rule straight from the packed rows [q | k | v | ..] of heads of 64 x 64 and the gates that mv_mlstm_prepare
// leaves; DV = 65 columns, the last one the normaliser. Rows ld apart, a multiple of eight.
extern "C" int mv_delta_chunks_sum_rows(const void* packed, long ld, const float* gates, float* state, const int* cu_seqlens, const int* state_slots, int n_seqs,
                                        int n, int H, int chunks, float* M, float* N, float* Q, float* out, int dtype, hipStream_t stream) {
    MV_REQUIRE(n >= 0 && n_seqs >= 0 && H > 0 && H <= 65535 && chunks >= 0, "delta_chunks_sum_rows: bad sizes n=%d seqs=%d H=%d", n, n_seqs, H);
    MV_REQUIRE(ld >= 3L * H * 64 && ld % 8 == 0, "delta_chunks_sum_rows: rows of %ld columns are not served", ld);
    MV_REQUIRE(packed && gates && state && cu_seqlens && state_slots && M && N && Q && out, "delta_chunks_sum_rows: missing operand");
    MV_REQUIRE(((uintptr_t)packed | (uintptr_t)state | (uintptr_t)N | (uintptr_t)Q) % 16 == 0, "delta_chunks_sum_rows: operands must be 16-byte aligned");
    if (n == 0 || n_seqs == 0 || chunks == 0) return 0;
    const DeltaChunkArgs A{nullptr, gates, nullptr, 0, 0, packed, ld, H, H, 65, cu_seqlens, n_seqs, M, N, Q, out, 0, nullptr, nullptr, nullptr, 0, 0.f, 0.f,
                           nullptr, nullptr, nullptr, nullptr, nullptr, 0, 0.f};
    MV_DISPATCH_T(dtype, "delta_chunks_sum_rows", { return (launch_delta_chunks<T, 64, RULE_SUM, 1>(A, state, state_slots, chunks, stream)); });
    return 0;
}
