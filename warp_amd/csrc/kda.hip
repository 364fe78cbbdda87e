// kda.hip — the Kimi Delta Attention recurrence on the device: the
// kda_step slot of the reference's dispatch table (src/waste_backend.h:69-72,
// src/kda.c:26-68) and a T-step forward that keeps the state on chip.
//
// Per head h, with state S [K][V]: q and k are L2-normalised (k by
// 1/sqrt(sum k^2 + 1e-12), q by the same and by 1/sqrt(K)); pass A decays
// every row kk of S by exp(g[kk]) and accumulates u = S^T k; then
// d = beta (v - u); pass B adds k d^T to S and accumulates o = S^T q. Every
// column i of S depends only on per-row scalars. The arithmetic is the
// reference's, operation by operation (separate multiplies and adds in row
// order, IEEE sqrt and division, glibc's expf), so S and o are bit-identical
// to waste_kda_step.

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "warp_internal.h"

#define WARP_EXPF_QUAL __device__ __forceinline__
#include "expf_glibc.h"

constexpr int KDA_MAX_K = 256;
constexpr int KDA_NT = 256;                   // 4 waves of 4 columns each

// The value of the lane before this one in its row of 16 lanes (0 in the
// row's first lane), and the row's last lane's value in every lane.
__device__ __forceinline__ float kda_prev(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x111, 0xf, 0xf, true));
}
__device__ __forceinline__ float kda_last(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x15f, 0xf, 0xf, true));
}

// T steps of 16 columns of one head per block. What bounds a step is the
// reference's summation order: u and o are each one chain of K dependent
// adds per column, and u's must end before the state can be updated. A row
// of 16 lanes owns a column, lane g its rows [g R, g R + R) in registers for
// the whole call, so the decay, the products and the update take R
// instructions instead of K; the chain runs in K / R phases of R adds by all
// lanes at once, each phase starting from the lane before (a DPP row shift),
// so that after the last phase lane 15 holds the sum in row order. The o
// chain of a step is interleaved with the u chain of the next (neither waits
// for the other), which hides the adds' latency. Rows are aligned to the
// end: pad = 16 R - K rows before the first are zeros, whole lanes of them
// are skipped by the phase count, and the rest add +0 (no sum here is ever
// -0, so that changes nothing).
// The per-row scalars (exp(g), normalised k and q) are made once per block
// and tile of TT steps, the two norms' sequential sums one step per lane;
// the next tile's rows are loaded while this one's steps run.
// 32 heads of 128 x 128, 256 steps: 5,085 us with a thread per column, the
// state in LDS and one thread's norms; 216 us now (0.84 us a step, where
// the 256 adds and the rest of a step's 300 instructions issue in 0.5 us).
template <int R, bool FULL>
__global__ __launch_bounds__(KDA_NT) void k_kda(int T, int H, int K, int V, int units, const float *__restrict__ q,
                                                const float *__restrict__ k, const float *__restrict__ v,
                                                const float *__restrict__ g, const float *__restrict__ beta,
                                                float *__restrict__ S, float *__restrict__ o) {
    constexpr int RS = 16 * R, LS = RS + 4;       // rows per column; LDS stride (steps on different banks)
    constexpr int TT = R == 16 ? 16 : 32, NE = TT * RS / KDA_NT;
    __shared__ __attribute__((aligned(16))) float kv[TT * LS], qv[TT * LS];
    __shared__ float dk[TT * LS], vt[TT * 16], bt[TT], nrm[2 * TT];
    static_assert(LS % 4 == 0 && __alignof__(kv) >= 16 && __alignof__(qv) >= 16, "their rows are read as float4");
    // blocks reach the XCDs in turn: each takes a contiguous eighth of the
    // units, so a head's blocks share one L2
    const int per = (int)gridDim.x >> 3, unit = ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
    if (unit >= units) return;
    const int ncg = (V + 15) >> 4, h = unit / ncg, c0 = (unit % ncg) * 16;
    const int tid = threadIdx.x, lane = tid & 63, col = (tid >> 6) * 4 + (lane >> 4), gl = lane & 15;
    const int i = c0 + col, pad = FULL ? 0 : RS - K, np = FULL ? 16 : (K + R - 1) / R, r0 = gl * R - pad;
    const bool live = i < V;
    float *Sh = S + (size_t)h * K * V;
    float s[R], w[R];
#pragma unroll
    for (int j = 0; j < R; j++) {
        const int kk = r0 + j;
        s[j] = live && (FULL || kk >= 0) ? Sh[(size_t)kk * V + i] : 0.0f;
        w[j] = 0.0f;
    }
    const float qscale = __fdiv_rn(1.0f, sqrtf((float)K));
    float tq[NE], tk[NE], tg[NE], tv[(TT * 16 + KDA_NT - 1) / KDA_NT], tb = 0.0f;
    // this thread's elements of the tile of n steps from t0
    auto load = [&](int t0, int n) {
#pragma unroll
        for (int e = 0; e < NE; e++) {
            const int x = tid + e * KDA_NT, t = x / RS, kk = x % RS - pad;
            const bool in = t < n && (FULL || kk >= 0);
            const size_t at = in ? ((size_t)(t0 + t) * H + h) * K + kk : 0;
            tq[e] = in ? q[at] : 0.0f;
            tk[e] = in ? k[at] : 0.0f;
            tg[e] = in ? g[at] : 0.0f;
        }
#pragma unroll
        for (int e = 0; e < TT * 16 / KDA_NT; e++) {
            const int x = tid + e * KDA_NT, t = x >> 4, c = c0 + (x & 15);
            tv[e] = t < n && c < V ? v[((size_t)(t0 + t) * H + h) * V + c] : 0.0f;
        }
        if (tid < n) tb = beta[(size_t)(t0 + tid) * H + h];
    };
    load(0, min(TT, T));
    for (int t0 = 0; t0 < T; t0 += TT) {
        const int n = min(TT, T - t0);
        __syncthreads();                          // the last tile's rows are read
#pragma unroll
        for (int e = 0; e < NE; e++) {
            const int x = tid + e * KDA_NT, t = x / RS, c = x % RS;
            if (t < n) {
                qv[t * LS + c] = tq[e];
                kv[t * LS + c] = tk[e];
                dk[t * LS + c] = warp_expf(tg[e]);
            }
        }
#pragma unroll
        for (int e = 0; e < TT * 16 / KDA_NT; e++) vt[tid + e * KDA_NT] = tv[e];
        if (tid < n) bt[tid] = tb;
        __syncthreads();
        // 1 / sqrt(sum x^2 + 1e-12), the sum sequential in index order
        // (l2_rnorm, src/kda.c:19-24): a lane per step, q then k. (sqrtf is
        // correctly rounded here; __fsqrt_rn may become the bare v_sqrt_f32,
        // off by an ulp.)
        if (tid < 2 * TT && (tid & (TT - 1)) < n) {
            const float *x = (tid < TT ? qv : kv) + (tid & (TT - 1)) * LS;
            float a = 0.0f;
#pragma unroll 8
            for (int c = FULL ? 0 : pad >> 2; c < RS / 4; c++) {
                const float4 y = *(const float4 *)(x + 4 * c);
                a = __fadd_rn(a, __fmul_rn(y.x, y.x));
                a = __fadd_rn(a, __fmul_rn(y.y, y.y));
                a = __fadd_rn(a, __fmul_rn(y.z, y.z));
                a = __fadd_rn(a, __fmul_rn(y.w, y.w));
            }
            const float rn = __fdiv_rn(1.0f, sqrtf(__fadd_rn(a, 1e-12f)));
            nrm[tid] = tid < TT ? __fmul_rn(rn, qscale) : rn;
        }
        __syncthreads();
#pragma unroll
        for (int e = 0; e < NE; e++) {
            const int x = tid + e * KDA_NT, t = x / RS, c = x % RS;
            if (t < n) {
                qv[t * LS + c] = __fmul_rn(tq[e], nrm[t]);
                kv[t * LS + c] = __fmul_rn(tk[e], nrm[TT + t]);
            }
        }
        __syncthreads();
        if (t0 + TT < T) load(t0 + TT, min(TT, T - t0 - TT));
        for (int t = 0; t < n; t++) {
            const float *pd = dk + t * LS + gl * R, *pk = kv + t * LS + gl * R, *pq = qv + t * LS + gl * R;
            float kr[R], p[R];
            // pass A: decay the rows, u = sum over rows of row * kv
#pragma unroll
            for (int j = 0; j < R; j++) {
                kr[j] = pk[j];
                s[j] = __fmul_rn(s[j], pd[j]);
                p[j] = __fmul_rn(s[j], kr[j]);
            }
            float u = 0.0f, acc = 0.0f;
            // (and the step before's o = sum over rows of row * qv)
            auto phase = [&]() {
                u = __fadd_rn(kda_prev(u), p[0]);
                acc = __fadd_rn(kda_prev(acc), w[0]);
#pragma unroll
                for (int j = 1; j < R; j++) {
                    u = __fadd_rn(u, p[j]);
                    acc = __fadd_rn(acc, w[j]);
                }
            };
            if (FULL) {
#pragma unroll
                for (int ph = 0; ph < 16; ph++) phase();
            } else {
                for (int ph = 0; ph < np; ph++) phase();
            }
            if (live && gl == 15 && t0 + t > 0) o[((size_t)(t0 + t - 1) * H + h) * V + i] = acc;
            const float d = __fmul_rn(bt[t], __fsub_rn(vt[t * 16 + col], kda_last(u)));
            // pass B: the rank-1 update of the column
#pragma unroll
            for (int j = 0; j < R; j++) {
                s[j] = __fadd_rn(s[j], __fmul_rn(d, kr[j]));
                if (!FULL && r0 + j < 0) s[j] = 0.0f;       // (an infinite d makes a NaN of a zero row)
                w[j] = __fmul_rn(s[j], pq[j]);
            }
        }
    }
    float acc = 0.0f;
    for (int ph = 0; ph < np; ph++) {
        acc = __fadd_rn(kda_prev(acc), w[0]);
#pragma unroll
        for (int j = 1; j < R; j++) acc = __fadd_rn(acc, w[j]);
    }
    if (live) {
        if (gl == 15) o[((size_t)(T - 1) * H + h) * V + i] = acc;
#pragma unroll
        for (int j = 0; j < R; j++)
            if (FULL || r0 + j >= 0) Sh[(size_t)(r0 + j) * V + i] = s[j];
    }
}

extern "C" int wk_kda(int T, int H, int K, int V, const float *q, const float *k, const float *v, const float *g,
                      const float *beta, float *S, float *o, void *stream) {
    if (T <= 0 || H <= 0 || K <= 0 || K > KDA_MAX_K || V <= 0 || V > 1024) return -1;
    // (the header's bound on K V, which callers test and fall back by; nothing
    // here needs it since the state left LDS)
    if ((size_t)K * V * sizeof(float) > 150 * 1024) return -1;
    const int units = H * ((V + 15) / 16);
    const dim3 grid((unsigned)((units + 7) / 8 * 8));
#define KDA(R, FULL)                                                                                              \
    hipLaunchKernelGGL((k_kda<R, FULL>), grid, dim3(KDA_NT), 0, (hipStream_t)stream, T, H, K, V, units, q, k, v, g, \
                       beta, S, o)
    // the fewest rows per lane that hold the column: the chain is K adds
    // either way, the rest of a step R
    if (K == 64) KDA(4, true);
    else if (K < 64) KDA(4, false);
    else if (K == 128) KDA(8, true);
    else if (K < 128) KDA(8, false);
    else if (K == 256) KDA(16, true);
    else KDA(16, false);
#undef KDA
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : -(int)e - 1000;
}
