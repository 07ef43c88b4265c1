// Device helpers shared by the kernels of mixers that carry a matrix state per head: the gates' functions,
// the lanes' share of a column of the state, the causal convolution's inputs in front of a step.
#pragma once
#include "dispatch.h"

__device__ __forceinline__ float sigmoid_f(float z) { return 1.f / (1.f + expf(-z)); }

__device__ __forceinline__ float silu_f(float z) { return z / (1.f + expf(-z)); }
__device__ __forceinline__ float softplus_f(float z) { return z > 20.f ? z : log1pf(expf(z)); }
// log(sigmoid(z)) without overflow
__device__ __forceinline__ float logsigmoid_f(float z) { return fminf(z, 0.f) - log1pf(expf(-fabsf(z))); }

// NT sums over j in [j0, j1) of w2t[j][c] * th[t][j] (th rows `pitch` floats apart), the weight's element
// type known at compile time and eight loads in flight at a time; the additions run in the order of j
template <typename W, int NT>
__device__ __forceinline__ void decay_dots(const W* __restrict__ w2t_c, size_t inner, const float* th, int pitch, int j0,
                                           int j1, float (&acc)[NT]) {
    int j = j0;
    for (; j + 8 <= j1; j += 8) {
        W raw[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) raw[e] = w2t_c[(size_t)(j + e) * inner];
        __builtin_amdgcn_sched_barrier(0);                     // (16-bit loads would be waited for one by one)
        float w[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) w[e] = to_f(raw[e]);
#pragma unroll
        for (int e = 0; e < 8; ++e)
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[t] = fmaf(w[e], th[t * pitch + j + e], acc[t]);
    }
    for (; j < j1; ++j) {
        const float w = to_f(w2t_c[(size_t)j * inner]);
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t] = fmaf(w, th[t * pitch + j], acc[t]);
    }
}

// the sum of a value over the L lanes that share a column (L = 4, 8 or 16 neighbouring lanes of a row
// of 16): exchanges inside the row by data-parallel moves; every lane ends with the sum
template <int L>
__device__ __forceinline__ float lanes_sum(float v) {
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, true));   // quad [1,0,3,2]
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x4E, 0xF, 0xF, true));   // quad [2,3,0,1]
    if constexpr (L >= 8)
        v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x141, 0xF, 0xF, true));  // mirror of 8
    if constexpr (L >= 16)
        v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x140, 0xF, 0xF, true));  // mirror of 16
    return v;
}

// a lane's R rows of its column, between registers and the column's D floats in memory (rows
// sub*R .. sub*R+R-1; rows beyond D are zero and are not stored)
template <int R, bool STORE>
__device__ __forceinline__ void delta_state_io(float (&s)[R], float* column, int sub, int D, bool live) {
    const int i0 = sub * R;
    if ((D & 3) == 0) {
#pragma unroll
        for (int e = 0; e < R; e += 4) {
            const bool ok = live && i0 + e < D;
            float4* p = reinterpret_cast<float4*>(column + (i0 + e < D ? i0 + e : 0));
            if constexpr (STORE) {
                if (ok) *p = float4{s[e], s[e + 1], s[e + 2], s[e + 3]};
            } else {
                const float4 v = *p;                  // always issued (a valid address either way), dropped where it does not count
                s[e] = ok ? v.x : 0.f; s[e + 1] = ok ? v.y : 0.f; s[e + 2] = ok ? v.z : 0.f; s[e + 3] = ok ? v.w : 0.f;
            }
        }
    } else {
#pragma unroll
        for (int e = 0; e < R; ++e) {
            const bool ok = live && i0 + e < D;
            if constexpr (STORE) {
                if (ok) column[i0 + e] = s[e];
            } else {
                const float v = column[i0 + e < D ? i0 + e : 0];
                s[e] = ok ? v : 0.f;
            }
        }
    }
}

// how a head of size D is dealt out: (rows a lane keeps, lanes a column); 0 when D is not served
static inline void delta_scan_shape(int D, int& R, int& L) {
    // few rows a lane and many lanes a column: a token costs the fewest instructions of the one wave a
    // SIMD runs, and a head is spread over the most workgroups
    if (D <= 16) { R = 4; L = 4; }
    else if (D <= 32) { R = 4; L = 8; }
    else if (D <= 64) { R = 4; L = 16; }
    else if (D <= 128) { R = 8; L = 16; }
    else { R = 16; L = 16; }
}

// most taps of a causal convolution over time
#define MS_MAX_TAPS 16

// One input of the causal convolution: row r of the step when the request's rows reach back that far,
// else the request's kept inputs (hist[slot][taps-1][C], the last one the newest).
template <typename T>
__device__ __forceinline__ float conv_input(const T* __restrict__ rows, long ld, const T* __restrict__ hist, int C, int taps,
                                            int first, int r, int c) {
    if (r >= first) return to_f(rows[(size_t)r * ld + c]);
    return to_f(hist[(size_t)(taps - 1 + (r - first)) * C + c]);
}

// The convolution's kept inputs after the step: the last taps-1 inputs of each request, from the step's
// rows and, where the step brought fewer, from what was kept before. Thread (request, channel) reads all
// it needs before it writes, and no other thread touches its channel.
template <typename T>
static __global__ void __launch_bounds__(256)
conv_state_kernel(const T* __restrict__ packed, long ld, int C, int taps, T* __restrict__ conv_state,
                  const int* __restrict__ cu_seqlens, const int* __restrict__ state_slots) {
    const int seq = blockIdx.x;
    const int c = blockIdx.y * 256 + threadIdx.x;
    const int first = cu_seqlens[seq], end = cu_seqlens[seq + 1];
    if (end <= first || c >= C) return;
    T* hist = conv_state + (size_t)state_slots[seq] * (taps - 1) * C;
    T keep[MS_MAX_TAPS];
    for (int i = 0; i < taps - 1; ++i) {
        const int r = end - (taps - 1) + i;
        keep[i] = r >= first ? packed[(size_t)r * ld + c] : hist[(size_t)(taps - 1 + (r - first)) * C + c];
    }
    for (int i = 0; i < taps - 1; ++i) hist[(size_t)i * C + c] = keep[i];
}

// ---------------------------------------------------------------------------------------
// The causal convolution and SiLU of CP_ROWS neighbouring rows by one wave, a channel a lane: a lane's filter stays in
// registers and a row's input is read once for all the taps it falls under. The sums are those of one row alone, term by term.
// A prompt's rows are bound by how many loads are on their way, not by their bytes: a workgroup a (row, head) took 63 us for
// 2,048 rows of 24 heads (gated delta rule) and 8 rows by a workgroup of 128, half of them idle at 64 channels, 38 us for
// 1,536 rows of 16 heads in 16 groups (channel decays); a wave for 8 rows of a head takes 18.7 and 28.4 us.
// ---------------------------------------------------------------------------------------
#define CP_ROWS 8

// taps and head sizes these serve, where they give every compute unit eight waves. Fewer rows fill the chip only one a
// workgroup; both forms, 16 heads in 16 groups, channel decays: 15.9 us one a workgroup against 16.6 at 256 rows of 64
// channels (12,288 rows x jobs), 19.1 against 17.1 at 384, 88.2 against 38.7 at 2,048; 128 channels 25.7 against 26.3 at 384,
// 99.3 against 55.8 at 2,048; 8 heads of 128: 17.6 against 22.8 at 512, 31.9 against 25.8 at 1,024; 4 of 256: 31.2 against
// 37.3 at 1,024, 51.3 against 43.3 at 2,048 (with the kept inputs' kernel behind, about 5 us).
static inline bool conv_rows_serve(int taps, int DK, int n, int jobs) {
    return taps >= 2 && taps <= 4 && DK <= 256 && (long)n * jobs >= 8L * CP_ROWS * mv_compute_units();
}

template <int TAPS>
struct ConvRows {
    int first[CP_ROWS], slot[CP_ROWS];       // of a row's request: its first row of the step, its row of the kept inputs
    bool live[CP_ROWS];
    __device__ __forceinline__ ConvRows(const int* __restrict__ token_seq, const int* __restrict__ cu_seqlens,
                                        const int* __restrict__ state_slots, int t0, int n) {
#pragma unroll
        for (int r = 0; r < CP_ROWS; ++r) {
            // (a row that does not count is computed as if its request began far in front of it, and not stored)
            const int seq = t0 + r < n ? token_seq[t0 + r] : -1;
            live[r] = seq >= 0;
            first[r] = live[r] ? cu_seqlens[seq] : -TAPS;
            slot[r] = live[r] ? state_slots[seq] : 0;
        }
    }
};

// x[r] = silu(convolution) of channel c (of C) in row t0 + r
template <typename T, int TAPS>
__device__ __forceinline__ void conv_rows(float (&x)[CP_ROWS], const ConvRows<TAPS>& rows, const T* __restrict__ packed, long ld,
                                          const WeightPtr& conv_w, const T* __restrict__ conv_state, int t0, int n, int C, int c) {
    float w[TAPS], in[CP_ROWS + TAPS - 1];
#pragma unroll
    for (int j = 0; j < TAPS; ++j) w[j] = conv_w.at((size_t)c * TAPS + j);
#pragma unroll
    for (int i = 0; i < CP_ROWS + TAPS - 1; ++i) in[i] = to_f(packed[(size_t)min(max(t0 - (TAPS - 1) + i, 0), n - 1) * ld + c]);
#pragma unroll
    for (int r = 0; r < CP_ROWS; ++r) {
        float acc = 0.f;
        if (t0 + r - (TAPS - 1) >= rows.first[r]) {
#pragma unroll
            for (int j = 0; j < TAPS; ++j) acc = fmaf(w[j], in[r + j], acc);
        } else {
            const T* hist = conv_state + (size_t)rows.slot[r] * (TAPS - 1) * C;
#pragma unroll
            for (int j = 0; j < TAPS; ++j)
                acc = fmaf(w[j], conv_input(packed, ld, hist, C, TAPS, rows.first[r], t0 + r - (TAPS - 1) + j, c), acc);
        }
        x[r] = silu_f(acc);
    }
}

// job 2 * group: unit queries (times DK^-1/2), 2 * group + 1: unit keys, into qk [n][G][2][DK]; lane d keeps channels d, d + 64 ..
// (UNITS of them). The squares are added up as the kernels of one row do with their 128 threads.
template <typename T, int TAPS, int UNITS>
__device__ __forceinline__ void conv_unit_rows(const ConvRows<TAPS>& rows, const T* __restrict__ packed, long ld, const WeightPtr& conv_w,
                                               const T* __restrict__ conv_state, int t0, int n, int C, int G, int DK, int job, int d,
                                               float unit_eps, float* __restrict__ qk) {
    const int group = job / 2, which = job % 2;
    float x[UNITS][CP_ROWS];
#pragma unroll
    for (int u = 0; u < UNITS; ++u) {
        const int c = u * MV_WAVE + d;
        conv_rows<T, TAPS>(x[u], rows, packed, ld, conv_w, conv_state, t0, n, C, which * G * DK + group * DK + (c < DK ? c : 0));
#pragma unroll
        for (int r = 0; r < CP_ROWS; ++r) x[u][r] = c < DK ? x[u][r] : 0.f;
    }
    const float scale = which == 0 ? 1.f / sqrtf((float)DK) : 1.f;
#pragma unroll
    for (int r = 0; r < CP_ROWS; ++r) {
        float even = fmaf(x[0][r], x[0][r], 0.f), odd = 0.f;         // (as there: a bare product could be fused into the sum)
        if constexpr (UNITS >= 2) odd = fmaf(x[1][r], x[1][r], 0.f);
        if constexpr (UNITS == 4) {
            even = fmaf(x[2][r], x[2][r], even);
            odd = fmaf(x[3][r], x[3][r], odd);
        }
        float ss = wave_sum(even);
        if constexpr (UNITS >= 2) ss += wave_sum(odd);
        const float inv = scale / sqrtf(ss + unit_eps);
        float* o = qk + (((size_t)(t0 + r) * G + group) * 2 + which) * DK;
#pragma unroll
        for (int u = 0; u < UNITS; ++u)
            if (rows.live[r] && u * MV_WAVE + d < DK) o[u * MV_WAVE + d] = x[u][r] * inv;
    }
}

// a head's values, vals [n][H][DV], from column c0 on
template <typename T, int TAPS>
__device__ __forceinline__ void conv_value_rows(const ConvRows<TAPS>& rows, const T* __restrict__ packed, long ld, const WeightPtr& conv_w,
                                                const T* __restrict__ conv_state, int t0, int n, int C, int c0, int H, int DV, int head, int lane,
                                                float* __restrict__ vals) {
    for (int d = lane; d < DV; d += MV_WAVE) {
        float x[CP_ROWS];
        conv_rows<T, TAPS>(x, rows, packed, ld, conv_w, conv_state, t0, n, C, c0 + head * DV + d);
#pragma unroll
        for (int r = 0; r < CP_ROWS; ++r)
            if (rows.live[r]) vals[((size_t)(t0 + r) * H + head) * DV + d] = x[r];
    }
}

// LAUNCH(taps, units) for what conv_rows_serve accepts
#define CONV_ROWS_DISPATCH(taps, DK, LAUNCH)                        \
    switch ((taps) * 8 + ((DK) <= 64 ? 1 : (DK) <= 128 ? 2 : 4)) {  \
        case 2 * 8 + 1: LAUNCH(2, 1); break;                        \
        case 2 * 8 + 2: LAUNCH(2, 2); break;                        \
        case 2 * 8 + 4: LAUNCH(2, 4); break;                        \
        case 3 * 8 + 1: LAUNCH(3, 1); break;                        \
        case 3 * 8 + 2: LAUNCH(3, 2); break;                        \
        case 3 * 8 + 4: LAUNCH(3, 4); break;                        \
        case 4 * 8 + 1: LAUNCH(4, 1); break;                        \
        case 4 * 8 + 2: LAUNCH(4, 2); break;                        \
        default: LAUNCH(4, 4);                                      \
    }
