// model.hip -- the non-attention kernels of a device-resident Model::forward
// (/root/reference/src/model.rs:420-516): matrix-vector products with fused
// RMSNorm prologues and residual / SwiGLU / q-k-v epilogues, the embedding
// gather and the greedy sampler.
//
// Decode (t = 1) is HBM-bound: every weight is read once per token.  One wave
// owns one output row, streams it with float4 loads (a wave reads 1 KiB of the
// row per instruction) and reduces its 64 partial sums with a fixed butterfly,
// so results are deterministic run to run.  2 or 3 tokens of a small model go
// through one such weight pass together; more run on the matrix cores
// (gemm_kernel).
#include <hip/hip_runtime.h>

#include <math.h>

#include <algorithm>

#include "gemm_tiles.h"
#include "model_kernels.h"
#include "wave_ops.h"

namespace wick {

namespace {

typedef float f4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float dot4(const f4 w, const f4 x, float acc) {
    acc = fmaf(w.x, x.x, acc);
    acc = fmaf(w.y, x.y, acc);
    acc = fmaf(w.z, x.z, acc);
    return fmaf(w.w, x.w, acc);
}

// Keeps (v, i) when v is larger, or equal at a smaller index: the first index
// of the maximum over the non-NaN values (NaN never compares greater).
__device__ __forceinline__ void arg_better(float v, int i, float &bv, int &bi) {
    if (v > bv || (v == bv && i < bi)) {
        bv = v;
        bi = i;
    }
}

}  // namespace

// One wave per R output rows (rows R*wave .. R*wave+R-1), NT tokens per wave
// (token group blockIdx.y).  Column c4 (a float4 index) of a row is handled by
// lane c4 % 64; a pass covers 64*UNR float4s of every row.  All loads a pass
// needs -- weight rows, input rows, norm weight, and the residual being added
// to -- are issued before the first arithmetic on them, so a kernel whose rows
// fit one pass waits for memory once.
template <int NT, int R, int UNR, int EPI, bool NORM>
__global__ __launch_bounds__(256) void gemv_kernel(const GemvArgs a) {
    static_assert(EPI != kEpiSwiglu || R == 1, "SwiGLU pairs one gate row with one up row");
    const int lane = threadIdx.x & 63;
    const int row0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * R;
    if (row0 >= a.rows) return;  // whole waves only; no barriers below
    const int tok0 = blockIdx.y * NT;
    const int nt = min(NT, a.t - tok0);
    const int C4 = a.cols >> 2;
    const f4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    const f4 *X[NT];
#pragma unroll
    for (int tk = 0; tk < NT; tk++) X[tk] = reinterpret_cast<const f4 *>(a.x + (size_t)(tok0 + min(tk, nt - 1)) * a.cols);
    const f4 *W[R];
#pragma unroll
    for (int r = 0; r < R; r++) W[r] = reinterpret_cast<const f4 *>(a.w + (size_t)min(row0 + r, a.rows - 1) * a.cols);
    const f4 *W2 = EPI == kEpiSwiglu ? reinterpret_cast<const f4 *>(a.w2 + (size_t)row0 * a.cols) : W[0];
    const f4 *G = reinterpret_cast<const f4 *>(a.norm);

    // the first pass's weights go out before anything waits on memory
    f4 wv[R][UNR], wv2[UNR];
#pragma unroll
    for (int u = 0; u < UNR; u++) {
        const int c = lane + 64 * u;
#pragma unroll
        for (int r = 0; r < R; r++) wv[r][u] = c < C4 ? __builtin_nontemporal_load(W[r] + c) : zero;
        if (EPI == kEpiSwiglu) wv2[u] = c < C4 ? __builtin_nontemporal_load(W2 + c) : zero;
    }
    // the values the residual epilogue adds to (lane tk: token tk, one per row)
    float resid[EPI == kEpiResid ? R : 1];
    if constexpr (EPI == kEpiResid) {
        const float *src = a.resid ? a.resid : a.out0;
#pragma unroll
        for (int r = 0; r < R; r++)
            resid[r] = (lane < nt && row0 + r < a.rows) ? src[(size_t)(tok0 + lane) * a.ld0 + row0 + r] : 0.0f;
    }

    // rmsnorm (src/kernels.rs:343-349) of each input row: xn = x * scale * g
    float scale[NT];
    if (NORM) {
#pragma unroll
        for (int tk = 0; tk < NT; tk++) {
            float ss = 0.0f;
            for (int c = lane; c < C4; c += 64) {
                const f4 v = X[tk][c];
                ss = dot4(v, v, ss);
            }
            ss = wave_sum(ss);
            scale[tk] = 1.0f / sqrtf(ss / (float)a.cols + a.eps);
        }
    }

    float acc[R][NT], acc2[NT];
#pragma unroll
    for (int tk = 0; tk < NT; tk++) {
        acc2[tk] = 0.0f;
#pragma unroll
        for (int r = 0; r < R; r++) acc[r][tk] = 0.0f;
    }
    for (int base = 0; base < C4; base += 64 * UNR) {
        if (base > 0) {
#pragma unroll
            for (int u = 0; u < UNR; u++) {
                const int c = base + lane + 64 * u;
#pragma unroll
                for (int r = 0; r < R; r++) wv[r][u] = c < C4 ? __builtin_nontemporal_load(W[r] + c) : zero;
                if (EPI == kEpiSwiglu) wv2[u] = c < C4 ? __builtin_nontemporal_load(W2 + c) : zero;
            }
        }
        f4 xv[NT][UNR], gv[UNR];
#pragma unroll
        for (int u = 0; u < UNR; u++) {
            const int c = base + lane + 64 * u;
            if (NORM) gv[u] = c < C4 ? G[c] : zero;
#pragma unroll
            for (int tk = 0; tk < NT; tk++) xv[tk][u] = c < C4 ? X[tk][c] : zero;
        }
#pragma unroll
        for (int u = 0; u < UNR; u++) {
#pragma unroll
            for (int tk = 0; tk < NT; tk++) {
                f4 x = xv[tk][u];
                if (NORM) x = x * scale[tk] * gv[u];
#pragma unroll
                for (int r = 0; r < R; r++) acc[r][tk] = dot4(wv[r][u], x, acc[r][tk]);
                if (EPI == kEpiSwiglu) acc2[tk] = dot4(wv2[u], x, acc2[tk]);
            }
        }
    }
#pragma unroll
    for (int tk = 0; tk < NT; tk++) {
#pragma unroll
        for (int r = 0; r < R; r++) acc[r][tk] = wave_sum(acc[r][tk]);
        if (EPI == kEpiSwiglu) acc2[tk] = wave_sum(acc2[tk]);
    }
    // lane tk writes token tk's values
#pragma unroll
    for (int tk = 0; tk < NT; tk++) {
        if (lane != tk || tk >= nt) continue;
        const size_t tok = (size_t)tok0 + tk;
#pragma unroll
        for (int r = 0; r < R; r++) {
            const int row = row0 + r;
            if (row >= a.rows) break;
            const float d = acc[r][tk];
            if (EPI == kEpiStore || EPI == kEpiArgmax) {
                a.out0[tok * a.ld0 + row] = d;
            } else if (EPI == kEpiResid) {
                a.out0[tok * a.ld0 + row] = resid[r] + d;
            } else if (EPI == kEpiQkv) {
                if (row < a.split0)
                    a.out0[tok * a.ld0 + row] = d;
                else if (row < a.split1)
                    a.out1[tok * a.ld1 + (row - a.split0)] = d;
                else
                    a.out2[tok * a.ld2 + (row - a.split1)] = d;
            } else {  // silu_mul: g / (1 + exp(-g)) * u
                a.out0[tok * a.ld0 + row] = d / (1.0f + expf(-d)) * acc2[tk];
            }
        }
    }
    if constexpr (EPI == kEpiArgmax) {
        // the wave's rows in increasing order; argmax_kernel reduces the pairs
        static_assert(NT == 1 && R == kArgmaxRows, "one token, one pair per kArgmaxRows rows");
        if (lane == 0) {
            float bv = -INFINITY;
            int bi = 0x7fffffff;
#pragma unroll
            for (int r = 0; r < R; r++)
                if (row0 + r < a.rows) arg_better(acc[r][0], row0 + r, bv, bi);
            reinterpret_cast<float2 *>(a.out1)[row0 / R] = make_float2(bv, __int_as_float(bi));
        }
    }
}

// One token, rows of up to 64 * UNR float4s (one pass): the input row is
// staged through LDS once per workgroup instead of being read by every wave.
// Thread t owns float4s t, t + 256, ... of the row: it loads x (plus, with
// NP > 0, the a.nparts partial vectors added in order -- the fused decode's
// per-unit output projections, the residual add of src/model.rs:486-487 --
// and the block-0 threads write that sum to a.xout), the norm weight, and its
// share of the sum of squares; the 4 waves' sums meet in LDS in a fixed order.
// Each wave owns R output rows, whose weights it requests first, so the
// kernel waits for memory once; epilogues as gemv_kernel's.
template <int R, int UNR, int EPI, bool NORM, int NP>
__global__ __launch_bounds__(256) void gemv1_kernel(const GemvArgs a) {
    static_assert(EPI != kEpiSwiglu || R == 1, "SwiGLU pairs one gate row with one up row");
    constexpr int XK = (64 * UNR + 255) / 256;  // float4s of the row per thread
    __shared__ f4 sx[256 * XK];
    __shared__ f4 sg[NORM ? 256 * XK : 1];
    __shared__ float sss[4];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, t = threadIdx.x;
    const int row0 = (blockIdx.x * 4 + w) * R;
    const bool live = row0 < a.rows;  // every wave reaches the barrier
    const int C4 = a.cols >> 2;
    const f4 zero = {0.0f, 0.0f, 0.0f, 0.0f};

    // Loads from clamped, in-bounds indices with no condition, and selects
    // afterwards: a load under a per-lane condition becomes an exec-mask
    // branch of its own, which serialises the issue of the loads.
    f4 wv[R][UNR], wv2[UNR];
#pragma unroll
    for (int r = 0; r < R; r++) {
        const f4 *W = reinterpret_cast<const f4 *>(a.w + (size_t)min(row0 + r, a.rows - 1) * a.cols);
#pragma unroll
        for (int u = 0; u < UNR; u++) wv[r][u] = __builtin_nontemporal_load(W + min(lane + 64 * u, C4 - 1));
    }
    if constexpr (EPI == kEpiSwiglu) {
        const f4 *W2 = reinterpret_cast<const f4 *>(a.w2 + (size_t)min(row0, a.rows - 1) * a.cols);
#pragma unroll
        for (int u = 0; u < UNR; u++) wv2[u] = __builtin_nontemporal_load(W2 + min(lane + 64 * u, C4 - 1));
    }
    float resid[EPI == kEpiResid ? R : 1];
    if constexpr (EPI == kEpiResid) {
        const float *src = a.resid ? a.resid : a.out0;
#pragma unroll
        for (int r = 0; r < R; r++) resid[r] = src[min(row0 + r, a.rows - 1)];
    }
    f4 xv[XK], gv[XK], pv[NP > 0 ? NP : 1][XK];
#pragma unroll
    for (int k = 0; k < XK; k++) {
        const int c = min(t + 256 * k, C4 - 1);
        xv[k] = reinterpret_cast<const f4 *>(a.x)[c];
        if (NORM) gv[k] = reinterpret_cast<const f4 *>(a.norm)[c];
#pragma unroll
        for (int p = 0; p < NP; p++)
            pv[p][k] = reinterpret_cast<const f4 *>(a.parts + (size_t)min(p, a.nparts - 1) * a.cols)[c];
    }
#pragma unroll
    for (int u = 0; u < UNR; u++) {
        const bool in = lane + 64 * u < C4;
#pragma unroll
        for (int r = 0; r < R; r++) wv[r][u] = in ? wv[r][u] : zero;
        if (EPI == kEpiSwiglu) wv2[u] = in ? wv2[u] : zero;
    }
    float ss = 0.0f;
#pragma unroll
    for (int k = 0; k < XK; k++) {
        const bool in = t + 256 * k < C4;
        xv[k] = in ? xv[k] : zero;
        if (NORM) gv[k] = in ? gv[k] : zero;
#pragma unroll
        for (int p = 0; p < NP; p++)
            if (p < a.nparts) xv[k] += in ? pv[p][k] : zero;
        const int c = t + 256 * k;
        sx[c] = xv[k];
        if (NORM) {
            sg[c] = gv[k];
            ss = dot4(xv[k], xv[k], ss);
        }
        if (NP > 0 && blockIdx.x == 0 && c < C4) reinterpret_cast<f4 *>(a.xout)[c] = xv[k];
    }
    if (NORM) {
        ss = wave_sum(ss);
        if (lane == 0) sss[w] = ss;
    }
    __syncthreads();
    float scale = 1.0f;
    if (NORM) {
        // rmsnorm (src/kernels.rs:343-349): xn = x * scale * g
        ss = (sss[0] + sss[1]) + (sss[2] + sss[3]);
        scale = 1.0f / sqrtf(ss / (float)a.cols + a.eps);
    }
    if (!live) return;
    float acc[R], acc2 = 0.0f;
#pragma unroll
    for (int r = 0; r < R; r++) acc[r] = 0.0f;
#pragma unroll
    for (int u = 0; u < UNR; u++) {
        const int c = lane + 64 * u;
        if (c >= C4) break;
        f4 x = sx[c];
        if (NORM) x = x * scale * sg[c];
#pragma unroll
        for (int r = 0; r < R; r++) acc[r] = dot4(wv[r][u], x, acc[r]);
        if (EPI == kEpiSwiglu) acc2 = dot4(wv2[u], x, acc2);
    }
#pragma unroll
    for (int r = 0; r < R; r++) acc[r] = wave_sum(acc[r]);
    if (EPI == kEpiSwiglu) acc2 = wave_sum(acc2);
    if (lane == 0) {
#pragma unroll
        for (int r = 0; r < R; r++) {
            const int row = row0 + r;
            if (row >= a.rows) break;
            const float d = acc[r];
            if (EPI == kEpiStore || EPI == kEpiArgmax) {
                a.out0[row] = d;
            } else if (EPI == kEpiResid) {
                a.out0[row] = resid[r] + d;
            } else if (EPI == kEpiQkv) {
                if (row < a.split0)
                    a.out0[row] = d;
                else if (row < a.split1)
                    a.out1[row - a.split0] = d;
                else
                    a.out2[row - a.split1] = d;
            } else {  // silu_mul: g / (1 + exp(-g)) * u
                a.out0[row] = d / (1.0f + expf(-d)) * acc2;
            }
        }
        if constexpr (EPI == kEpiArgmax) {
            // the wave's rows in increasing order; argmax_kernel reduces the pairs
            static_assert(R == kArgmaxRows, "one pair per kArgmaxRows rows");
            float bv = -INFINITY;
            int bi = 0x7fffffff;
#pragma unroll
            for (int r = 0; r < R; r++)
                if (row0 + r < a.rows) arg_better(acc[r], row0 + r, bv, bi);
            reinterpret_cast<float2 *>(a.out1)[row0 / R] = make_float2(bv, __int_as_float(bi));
        }
    }
}

// One token, rows too long for gemv1_kernel: HBM-bound, and gemv_kernel's waves
// each read the input row again for every row of weights (twice with a norm)
// through the L1 that the weights come through.  Here a workgroup stages the
// row in LDS once, times the norm's weight (its factor multiplies the sums), and
// its waves stream R rows of weights after R rows, the next U float4s of each
// requested while these are multiplied, across row ends too.  A layer of 4096 x
// 14336 (8B size): q/k/v 23.4 -> 17.8 us, gate/up 79.4 -> 69.5 (6.8 TB/s), down
// 38.7 -> 37.0; a head of 32000 rows 95.4 -> 91.4.
constexpr int kWideWaves = 8;

template <int R, int U, int EPI, bool NORM>
__global__ __launch_bounds__(64 * kWideWaves) void gemv_wide_kernel(const GemvArgs a) {
    static_assert(EPI != kEpiArgmax || R == kArgmaxRows, "one pair per kArgmaxRows rows");
    constexpr int M = EPI == kEpiSwiglu ? 2 : 1, NW = kWideWaves;
    extern __shared__ f4 sx[];  // the row, zero-padded to whole passes
    __shared__ float sss[NW];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int C4 = a.cols >> 2, passes = (C4 + 64 * U - 1) / (64 * U);
    const int groups = (a.rows + R - 1) / R, step = gridDim.x * NW;
    const f4 zero = {0.f, 0.f, 0.f, 0.f};
    f4 wv[2][M][R][U];
    const auto load = [&](f4 (&b)[M][R][U], int g, int p) {
#pragma unroll
        for (int r = 0; r < R; r++) {
            const size_t row = (size_t)min(g * R + r, a.rows - 1) * a.cols;
            const f4 *W = reinterpret_cast<const f4 *>(a.w + row);
            const f4 *W2 = reinterpret_cast<const f4 *>((M == 2 ? a.w2 : a.w) + row);
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int c = min(64 * (p * U + u) + lane, C4 - 1);
                b[0][r][u] = __builtin_nontemporal_load(W + c);
                if (M == 2) b[M - 1][r][u] = __builtin_nontemporal_load(W2 + c);
            }
        }
    };
    int g = blockIdx.x * NW + w, p = 0;
    load(wv[0], min(g, groups - 1), 0);
    float ss = 0.f;
    for (int c = threadIdx.x; c < passes * 64 * U; c += 64 * NW) {
        f4 x = c < C4 ? reinterpret_cast<const f4 *>(a.x)[c] : zero;
        if (NORM) {
            ss = dot4(x, x, ss);
            x = c < C4 ? x * reinterpret_cast<const f4 *>(a.norm)[c] : zero;
        }
        sx[c] = x;
    }
    if (NORM) {
        ss = wave_sum(ss);
        if (lane == 0) sss[w] = ss;
    }
    __syncthreads();
    float scale = 1.f;
    if (NORM) {
        ss = 0.f;
#pragma unroll
        for (int j = 0; j < NW; j++) ss += sss[j];
        scale = 1.0f / sqrtf(ss / (float)a.cols + a.eps);
    }
    float acc[M][R];
#pragma unroll
    for (int m = 0; m < M; m++)
#pragma unroll
        for (int r = 0; r < R; r++) acc[m][r] = 0.f;
    // this batch's products while the next one's weights (the row's next pass, or
    // the next row's first) are on their way
    const auto turn = [&](f4 (&b)[M][R][U], f4 (&next)[M][R][U]) {
        const bool last = p + 1 == passes;
        const int ng = last ? g + step : g, np = last ? 0 : p + 1;
        load(next, min(ng, groups - 1), np);
        __builtin_amdgcn_sched_barrier(0);
        const bool tail = 64 * U * (p + 1) > C4;
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int c = 64 * (p * U + u) + lane;
            const f4 x = sx[c];
#pragma unroll
            for (int m = 0; m < M; m++)
#pragma unroll
                for (int r = 0; r < R; r++) acc[m][r] = dot4(tail && c >= C4 ? zero : b[m][r][u], x, acc[m][r]);
        }
        if (last) {
#pragma unroll
            for (int m = 0; m < M; m++)
#pragma unroll
                for (int r = 0; r < R; r++) acc[m][r] = wave_sum(acc[m][r]) * scale;
            if (lane == 0) {
                float bv = -INFINITY;
                int bi = 0x7fffffff;
#pragma unroll
                for (int r = 0; r < R; r++) {
                    const int row = g * R + r;
                    if (row >= a.rows) break;
                    const float d = acc[0][r];
                    if (EPI == kEpiStore || EPI == kEpiArgmax) {
                        a.out0[row] = d;
                    } else if (EPI == kEpiResid) {
                        a.out0[row] = (a.resid ? a.resid : a.out0)[row] + d;
                    } else if (EPI == kEpiQkv) {
                        if (row < a.split0)
                            a.out0[row] = d;
                        else if (row < a.split1)
                            a.out1[row - a.split0] = d;
                        else
                            a.out2[row - a.split1] = d;
                    } else {  // silu_mul: g / (1 + exp(-g)) * u
                        a.out0[row] = d / (1.0f + expf(-d)) * acc[M - 1][r];
                    }
                    if (EPI == kEpiArgmax) arg_better(d, row, bv, bi);
                }
                if (EPI == kEpiArgmax) reinterpret_cast<float2 *>(a.out1)[g] = make_float2(bv, __int_as_float(bi));
            }
#pragma unroll
            for (int m = 0; m < M; m++)
#pragma unroll
                for (int r = 0; r < R; r++) acc[m][r] = 0.f;
        }
        g = ng;
        p = np;
    };
    while (g < groups) {
        turn(wv[0], wv[1]);
        if (g >= groups) break;
        turn(wv[1], wv[0]);
    }
}

// The o product of a split single-token decode with the merge of its chunks'
// states (DecodeStates) as the prologue: gemv1_kernel<1, UNR, kEpiResid> whose
// input row every workgroup merges for itself.  Thread t owns float4s t, t + 256,
// ... of the row: it requests all NC states of its float4 (slots past nchunks
// repeat the last and weigh 0) next to the weights, so the kernel waits for
// memory once (figures at kStateChunks).
template <int UNR, int NC>
__global__ __launch_bounds__(256) void gemv1_states_kernel(const GemvArgs a, const DecodeStates st) {
    constexpr int XK = (64 * UNR + 255) / 256;
    __shared__ f4 sx[256 * XK];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, t = threadIdx.x;
    const int row = blockIdx.x * 4 + w;
    const int C4 = a.cols >> 2;
    const f4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    f4 wv[UNR];
    const f4 *W = reinterpret_cast<const f4 *>(a.w + (size_t)min(row, a.rows - 1) * a.cols);
#pragma unroll
    for (int u = 0; u < UNR; u++) wv[u] = __builtin_nontemporal_load(W + min(lane + 64 * u, C4 - 1));
    const float resid = (a.resid ? a.resid : a.out0)[min(row, a.rows - 1)];
#pragma unroll
    for (int k = 0; k < XK; k++) {
        const int c = min(t + 256 * k, C4 - 1), h = 4 * c / st.head_dim, d = 4 * c % st.head_dim;
        const int kvh = h / st.group, hh = h % st.group;
        const size_t base = (size_t)((kvh * st.hslices + hh / 16) * 16 + hh % 16) * st.stride;
        f4 o[NC];
        float m[NC], l[NC];
#pragma unroll
        for (int j = 0; j < NC; j++) {
            const size_t at = base + min(j, st.nchunks - 1);
            m[j] = st.m[at];
            l[j] = st.l[at];
            o[j] = *reinterpret_cast<const f4 *>(st.o + at * st.head_dim + d);
        }
        float M = m[0];
#pragma unroll
        for (int j = 1; j < NC; j++) M = fmaxf(M, m[j]);
        f4 acc = zero;
        float L = 0.0f;
#pragma unroll
        for (int j = 0; j < NC; j++) {
            const float e = j < st.nchunks ? __builtin_amdgcn_exp2f(m[j] - M) : 0.0f;
            acc += o[j] * e;
            L += l[j] * e;
        }
        sx[t + 256 * k] = acc / L;
    }
    __syncthreads();
    if (row >= a.rows) return;
    float acc = 0.0f;
#pragma unroll
    for (int u = 0; u < UNR; u++) {
        const int c = lane + 64 * u;
        if (c >= C4) break;
        acc = dot4(wv[u], sx[c], acc);
    }
    acc = wave_sum(acc);
    if (lane == 0) a.out0[row] = resid + acc;
}

// Several tokens: out rows of W . X^T on the f32 matrix cores
// (v_mfma_f32_16x16x4_f32: A = 16 weight rows x 4 k, B = 4 k x 16 tokens).  The
// contraction index is permuted so each lane loads whole float4s: MFMA e of
// k-step s uses k = 16s + 4*(lane/16) + e for both operands.  Lane l then holds
// rows row0 + 4*(l/16) + r of token tok0 + 16b + l%16.
//
// A workgroup computes one tile of 16*RB rows x 16*TB tokens; its NW waves deal
// the k-steps out in batches of KU (wave w takes batches w, w + NW, ...: the
// waves together read whole cache lines of every row) and their partial tiles
// are summed through LDS in wave order.  The next batch's loads are in flight
// during this one's products.
//
// What bounds it: chunks hold at most a few hundred tokens, so a CU's share of
// the output is one small tile and every CU reads its rows and tokens at full
// length from L2.  In the MFMA lane layout consecutive lanes are consecutive
// rows, and the L1 then serves one lane (16 bytes) a cycle: 65 cache accesses
// per load instruction counted, 13 to 15 bytes per cycle and CU whatever the tile
// (13 to 16 accesses as loaded here).
// So a wave loads 16 rows x 32 k with 8 consecutive lanes on one row's 128-byte
// line (4 lanes on 64 bytes: 5 to 20% slower) and passes it through its own
// piece of LDS.  251 tokens of a 2048-wide layer (hidden 2048, FFN 5632): q/k/v
// 60 -> 27.5 us, o and down 180 together -> 20.7 + 47.3 (122 TFLOP/s; the
// library's largest f32 products reach 152), gate/up 194 -> 110; straight to
// registers 31, 27 + 69, 115.  251 tokens at hidden 576, FFN 1536: 10.8 -> 5.8,
// 6.3, 21.6 -> 14.1, 9.5 us.  Reading the next fragments from LDS ahead of the
// products gained nothing.
__device__ __forceinline__ f4 mfma4(float a, float b, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

__device__ __forceinline__ __amdgpu_buffer_rsrc_t gemm_rsrc(const float *base, unsigned bytes) {
    const unsigned long long p = (unsigned long long)base;
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)p);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(p >> 32));
    return __builtin_amdgcn_make_buffer_rsrc((void *)(((unsigned long long)hi << 32) | lo), (short)0,
                                             (int)__builtin_amdgcn_readfirstlane(bytes), 0x00020000);
}

__device__ __forceinline__ f4 gemm_load(__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff) {
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    const u4 x = __builtin_amdgcn_raw_buffer_load_b128(r, (int)voff, (int)soff, 0);
    return f4{__uint_as_float(x[0]), __uint_as_float(x[1]), __uint_as_float(x[2]), __uint_as_float(x[3])};
}

template <int EPI, int RB, int TB, int NW, int KU>
__global__ __launch_bounds__(64 * NW) void gemm_kernel(const GemmArgs a) {
    constexpr int M = EPI == kEpiSwiglu ? 2 : 1;  // weight matrices
    constexpr int NB = RB * TB;                   // 16 x 16 blocks of the tile
    constexpr int NT = 16 * TB;                   // tokens of the tile
    constexpr int PG = 64 * NW / NT;              // threads sharing a token's sum-of-squares parts
    constexpr int BPW = (NB + NW - 1) / NW;       // blocks each wave finishes
    constexpr int WL = 64 * (M * NB > KU * (M * RB + TB) ? M * NB : KU * (M * RB + TB));  // a wave's LDS, float4s
    __shared__ f4 sm[NW][WL];
    __shared__ float sss[PG][NT];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // Workgroup ids go round the 8 XCDs: all token tiles of a row tile run on
    // one XCD, one after another, so its L2 reads each weight once.
    const int nrt = (a.rows + 16 * RB - 1) / (16 * RB), ntt = (a.t + NT - 1) / NT;
    const int slot = blockIdx.x >> 3;
    const int rt = (blockIdx.x & 7) + 8 * (slot / ntt), tt = slot % ntt;
    if (rt >= nrt) return;
    const int row0 = 16 * RB * rt, tok0 = NT * tt;
    const int i = lane & 15, g = lane >> 4;
    // Rows and tokens past the end read as zero: within a 16-row block through
    // the resource's bound, a whole block past it as block 0 (never stored).
    // The k position is a lane's own offset, the row block a scalar one, so a
    // batch costs one select per k-step: a k past the row reads out of bounds,
    // as zero, without a branch (behind a branch the compiler waits for every
    // load in flight, the next batch's too).
    const unsigned pitch = (unsigned)a.cols * 4u;
    const int wrows = min(16 * RB, a.rows - row0), toks = min(NT, a.t - tok0);
    const __amdgpu_buffer_rsrc_t rw = gemm_rsrc(a.w + (size_t)row0 * a.cols, (unsigned)wrows * pitch);
    const __amdgpu_buffer_rsrc_t rw2 =
        M == 2 ? gemm_rsrc(a.w2 + (size_t)row0 * a.cols, (unsigned)wrows * pitch) : rw;
    const __amdgpu_buffer_rsrc_t rx = gemm_rsrc(a.x + (size_t)tok0 * a.cols, (unsigned)toks * pitch);
    unsigned so_w[RB], so_x[TB];
#pragma unroll
    for (int r = 0; r < RB; r++) so_w[r] = __builtin_amdgcn_readfirstlane(16 * r < wrows ? 16u * r * pitch : 0u);
#pragma unroll
    for (int t = 0; t < TB; t++) so_x[t] = __builtin_amdgcn_readfirstlane(16 * t < toks ? 16u * t * pitch : 0u);
    // the row (of the first 8, or of the last 8) and 16-byte chunk this lane
    // loads of 16 rows x 32 k
    static_assert(KU % 2 == 0, "batches of whole cache lines");
    const int lr = lane >> 3, lc = (lane & 7) ^ lr;  // (row & 7 is lr in both halves)
    const unsigned vrow = (unsigned)lr * pitch + 16u * lc;

    struct Batch {
        f4 w[M][KU][RB], x[KU][TB];
    };
    auto load = [&](Batch &b, int n) {
#pragma unroll
        for (int u = 0; u < KU; u++) {
            const int k = 16 * (KU * n + (u & ~1));
            const unsigned vo = (k + 4 * lc < a.cols ? vrow + 4u * (unsigned)k : 0x80000000u) + (u & 1) * 8u * pitch;
#pragma unroll
            for (int r = 0; r < RB; r++) {
                b.w[0][u][r] = gemm_load(rw, vo, so_w[r]);
                if (M == 2) b.w[M - 1][u][r] = gemm_load(rw2, vo, so_w[r]);
            }
#pragma unroll
            for (int t = 0; t < TB; t++) b.x[u][t] = gemm_load(rx, vo, so_x[t]);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // through the wave's own LDS: stored as loaded, read in the product's lane
    // layout (one wave's LDS operations run in order, so no barrier)
    f4 *const mine = &sm[w][0];
    const int rd[2] = {8 * i + (g ^ (i & 7)), 8 * i + ((4 + g) ^ (i & 7))};
    auto turn = [&](Batch &b) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int u = 0; u < KU; u++) {
            f4 *q = mine + 64 * ((u & ~1) * (M * RB + TB) + (u & 1));
#pragma unroll
            for (int m = 0; m < M; m++)
#pragma unroll
                for (int r = 0; r < RB; r++) q[128 * (m * RB + r) + lane] = b.w[m][u][r];
#pragma unroll
            for (int t = 0; t < TB; t++) q[128 * (M * RB + t) + lane] = b.x[u][t];
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    auto frags = [&](Batch &b) {
#pragma unroll
        for (int u = 0; u < KU; u++) {
            const f4 *q = mine + 64 * (u & ~1) * (M * RB + TB) + rd[u & 1];
#pragma unroll
            for (int m = 0; m < M; m++)
#pragma unroll
                for (int r = 0; r < RB; r++) b.w[m][u][r] = q[128 * (m * RB + r)];
#pragma unroll
            for (int t = 0; t < TB; t++) b.x[u][t] = q[128 * (M * RB + t)];
        }
    };
    f4 acc[M][RB][TB];
#pragma unroll
    for (int m = 0; m < M; m++)
#pragma unroll
        for (int r = 0; r < RB; r++)
#pragma unroll
            for (int t = 0; t < TB; t++) acc[m][r][t] = f4{0.f, 0.f, 0.f, 0.f};
    auto step = [&](const Batch &b) {
#pragma unroll
        for (int u = 0; u < KU; u++)
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int m = 0; m < M; m++)
#pragma unroll
                    for (int r = 0; r < RB; r++)
#pragma unroll
                        for (int t = 0; t < TB; t++) acc[m][r][t] = mfma4(b.w[m][u][r][e], b.x[u][t][e], acc[m][r][t]);
    };

    const int nbat = (a.cols + 16 * KU - 1) / (16 * KU), iters = (nbat + NW - 1) / NW;
    Batch ba, bb;
    load(ba, w);
    // the values the epilogue needs, requested behind the first batch
    f4 resid[EPI == kEpiResid ? BPW : 1];
    if constexpr (EPI == kEpiResid) {
#pragma unroll
        for (int q = 0; q < BPW; q++) {
            const int bl = min(w + NW * q, NB - 1);
            const int tok = min(tok0 + 16 * (bl % TB) + i, a.t - 1), row = min(row0 + 16 * (bl / TB) + 4 * g, a.rows - 4);
            resid[q] = *reinterpret_cast<const f4 *>(a.out0 + (size_t)tok * a.ld0 + row);
        }
    }
    constexpr int SQ = 8;  // sum-of-squares parts a thread requests up front
    const int pg = threadIdx.x / NT, ptk = threadIdx.x % NT;
    const float *sp = a.ssq ? a.ssq + min(tok0 + ptk, a.t - 1) : nullptr;
    float sq[SQ];
    if (a.ssq) {
#pragma unroll
        for (int p = 0; p < SQ; p++) sq[p] = sp[(size_t)min(pg + p * PG, a.nssq - 1) * a.t];
    }
    __builtin_amdgcn_sched_barrier(0);
    for (int it = 0; it < iters; it++) {
        turn(ba);
        load(ba, w + NW * (it + 1));
        frags(bb);
        step(bb);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int m = 0; m < M; m++)
#pragma unroll
        for (int r = 0; r < RB; r++)
#pragma unroll
            for (int t = 0; t < TB; t++) sm[w][64 * (m * NB + r * TB + t) + lane] = acc[m][r][t];
    if (a.ssq) {
        float ssum = 0.f;
#pragma unroll
        for (int p = 0; p < SQ; p++) ssum += pg + p * PG < a.nssq ? sq[p] : 0.f;
        for (int p = pg + SQ * PG; p < a.nssq; p += PG) ssum += sp[(size_t)p * a.t];
        sss[pg][ptk] = ssum;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < BPW; q++) {
        const int bl = w + NW * q;
        if (bl >= NB) break;
        const int tk = 16 * (bl % TB) + i, tok = tok0 + tk, row = row0 + 16 * (bl / TB) + 4 * g;
        f4 d[M];
#pragma unroll
        for (int m = 0; m < M; m++) {
            d[m] = sm[0][64 * (m * NB + bl) + lane];
#pragma unroll
            for (int ww = 1; ww < NW; ww++) d[m] += sm[ww][64 * (m * NB + bl) + lane];
        }
        if (a.ssq) {
            // rmsnorm's factor of the token (src/kernels.rs:343-349); its weight is in x
            float ss = 0.f;
#pragma unroll
            for (int p = 0; p < PG; p++) ss += sss[p][tk];
            const float scale = 1.0f / sqrtf(ss / (float)a.cols + a.eps);
#pragma unroll
            for (int m = 0; m < M; m++) d[m] *= scale;
        }
        const bool live = tok < a.t && row < a.rows;
        const size_t tkn = (size_t)tok;
        if constexpr (EPI == kEpiStore) {
            if (live) {
#pragma unroll
                for (int r = 0; r < 4; r++)
                    if (row + r < a.rows) a.out0[tkn * a.ld0 + row + r] = d[0][r];
            }
        } else if constexpr (EPI == kEpiResid) {
            const f4 x = resid[q] + d[0];
            if (live) {
                *reinterpret_cast<f4 *>(a.out0 + tkn * a.ld0 + row) = x;
                if (a.xg) *reinterpret_cast<f4 *>(a.xg + tkn * a.ld0 + row) = x * *reinterpret_cast<const f4 *>(a.xnorm + row);
            }
            if (a.xg) {
                // the block's share of the token's sum of squares, rows in order
                float ss = live ? dot4(x, x, 0.f) : 0.f;
                ss = rows_sum(ss);
                const int part = row0 / 16 + bl / TB;
                if (g == 0 && tok < a.t && 16 * part < a.rows) a.xssq[(size_t)part * a.t + tok] = ss;
            }
        } else if constexpr (EPI == kEpiQkv) {
            // the splits are multiples of 16: a float4 lies in one output
            if (live) {
                float *o = row < a.split0   ? a.out0 + tkn * a.ld0 + row
                           : row < a.split1 ? a.out1 + tkn * a.ld1 + (row - a.split0)
                                            : a.out2 + tkn * a.ld2 + (row - a.split1);
                *reinterpret_cast<f4 *>(o) = d[0];
            }
        } else {  // silu_mul: g / (1 + exp(-g)) * u
            if (live) {
                f4 h;
#pragma unroll
                for (int r = 0; r < 4; r++) h[r] = d[0][r] / (1.0f + expf(-d[0][r])) * d[M - 1][r];
                *reinterpret_cast<f4 *>(a.out0 + tkn * a.ld0 + row) = h;
            }
        }
    }
}

// step (graph-replayed decode loop): the token is tokens[*step + i].
// xg: also x * xnorm (the first layer's norm weight) and the row's sum of
// squares, for the products that apply the norm's factor (GemmArgs::ssq).
__global__ __launch_bounds__(256) void embed_kernel(const float *__restrict__ embed, const uint32_t *__restrict__ tokens,
                                                    const int *__restrict__ step, float *__restrict__ x, int hidden,
                                                    float *__restrict__ xg, const float *__restrict__ xnorm,
                                                    float *__restrict__ xssq) {
    __shared__ float red[4];
    const int i = blockIdx.x;
    const int at = (step ? *step : 0) + i;
    const f4 *src = reinterpret_cast<const f4 *>(embed + (size_t)tokens[at] * hidden);
    f4 *dst = reinterpret_cast<f4 *>(x + (size_t)i * hidden);
    if (!xg) {
        for (int c = threadIdx.x; c < hidden / 4; c += blockDim.x) dst[c] = src[c];
        return;
    }
    f4 *dg = reinterpret_cast<f4 *>(xg + (size_t)i * hidden);
    float ss = 0.0f;
    for (int c = threadIdx.x; c < hidden / 4; c += blockDim.x) {
        const f4 v = src[c];
        dst[c] = v;
        dg[c] = v * reinterpret_cast<const f4 *>(xnorm)[c];
        ss = dot4(v, v, ss);
    }
    ss = wave_sum(ss);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
    __syncthreads();
    if (threadIdx.x == 0) xssq[i] = (red[0] + red[1]) + (red[2] + red[3]);
}

// sampler::argmax (src/sampler.rs:129-137): best = 0; for i: if x[i] > x[best]
// { best = i }.  That is the first index of the maximum over the non-NaN
// values (NaN never compares greater), except that a NaN at index 0 is never
// replaced.  One workgroup; each thread issues 8 float4 loads per pass before
// comparing.  Ties resolve to the smaller index.  With parts (the LM head's
// kEpiArgmax pairs, one per kArgmaxRows rows) the workgroup reduces those
// instead: a quarter of the values, each 2 floats, and every pair's index the
// smallest among its rows' maxima, so the result is the same.

// step, len (graph-replayed decode loop): the id goes to out[*step + 1], then
// *step and *len advance to the next forward's token and cache length.
// embed (greedy decode loop): the workgroup also copies the chosen id's
// embedding row (hidden floats) to xe, the next forward's input row, in place
// of that forward's embed_kernel launch.
__global__ __launch_bounds__(1024) void argmax_kernel(const float *__restrict__ x, int n, uint32_t *__restrict__ out,
                                                      int *__restrict__ step, int *__restrict__ len,
                                                      const float *__restrict__ parts, const float *__restrict__ embed,
                                                      float *__restrict__ xe, int hidden) {
    constexpr int U = 8;
    __shared__ float sv[16];
    __shared__ int si[16];
    __shared__ int sbest;
    float bv = -INFINITY;
    int bi = 0x7fffffff;
    // x[0] (wick keeps index 0 when it is NaN) is requested with the rest
    const float x0 = threadIdx.x == 0 ? x[0] : 0.f;
    if (parts) {
        // two pairs per float4
        const int np = argmax_parts(n), np2 = np >> 1;
        const f4 *p4 = reinterpret_cast<const f4 *>(parts);
        for (int base = threadIdx.x; base < np2; base += U * 1024) {
            f4 v[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int c = base + 1024 * u;
                if (c < np2) v[u] = p4[c];
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int c = base + 1024 * u;
                if (c < np2) {
                    arg_better(v[u].x, __float_as_int(v[u].y), bv, bi);
                    arg_better(v[u].z, __float_as_int(v[u].w), bv, bi);
                }
            }
        }
        if ((np & 1) && threadIdx.x == 0) arg_better(parts[2 * np - 2], __float_as_int(parts[2 * np - 1]), bv, bi);
    } else {
        const int n4 = n >> 2;
        const f4 *x4 = reinterpret_cast<const f4 *>(x);
        for (int base = threadIdx.x; base < n4; base += U * 1024) {
            f4 v[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int c = base + 1024 * u;
                v[u] = c < n4 ? x4[c] : f4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int c = base + 1024 * u;
                if (c < n4) {
                    arg_better(v[u].x, 4 * c, bv, bi);
                    arg_better(v[u].y, 4 * c + 1, bv, bi);
                    arg_better(v[u].z, 4 * c + 2, bv, bi);
                    arg_better(v[u].w, 4 * c + 3, bv, bi);
                }
            }
        }
        for (int i = 4 * n4 + threadIdx.x; i < n; i += 1024) arg_better(x[i], i, bv, bi);
    }
    // the wave's best pair on lane moves (no lane holds a NaN as its best, so
    // "better of two" is commutative and every lane ends with the wave's best)
    arg_better(dpp_f<kDppQuadXor1>(bv), dpp_i<kDppQuadXor1>(bi), bv, bi);
    arg_better(dpp_f<kDppQuadXor2>(bv), dpp_i<kDppQuadXor2>(bi), bv, bi);
    arg_better(dpp_f<kDppRowHalfMirror>(bv), dpp_i<kDppRowHalfMirror>(bi), bv, bi);
    arg_better(dpp_f<kDppRowMirror>(bv), dpp_i<kDppRowMirror>(bi), bv, bi);
    {
        const auto pv = __builtin_amdgcn_permlane16_swap(__float_as_uint(bv), __float_as_uint(bv), false, false);
        const auto pi = __builtin_amdgcn_permlane16_swap((unsigned)bi, (unsigned)bi, false, false);
        arg_better(__uint_as_float(pv[0]), (int)pi[0], bv, bi);
        arg_better(__uint_as_float(pv[1]), (int)pi[1], bv, bi);
    }
    {
        const auto pv = __builtin_amdgcn_permlane32_swap(__float_as_uint(bv), __float_as_uint(bv), false, false);
        const auto pi = __builtin_amdgcn_permlane32_swap((unsigned)bi, (unsigned)bi, false, false);
        arg_better(__uint_as_float(pv[0]), (int)pi[0], bv, bi);
        arg_better(__uint_as_float(pv[1]), (int)pi[1], bv, bi);
    }
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        sv[w] = bv;
        si[w] = bi;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < 16; k++) arg_better(sv[k], si[k], bv, bi);
        // all values NaN (bi unset) or x[0] NaN: wick keeps index 0
        if (bi == 0x7fffffff || isnan(x0)) bi = 0;
        if (step) {
            const int k = *step;
            out[k + 1] = (uint32_t)bi;
            *step = k + 1;
            *len += 1;
        } else {
            *out = (uint32_t)bi;
        }
        sbest = bi;
    }
    if (embed) {
        __syncthreads();
        const f4 *src = reinterpret_cast<const f4 *>(embed + (size_t)sbest * hidden);
        f4 *dst = reinterpret_cast<f4 *>(xe);
        for (int c = threadIdx.x; c < hidden / 4; c += blockDim.x) dst[c] = src[c];
    }
}

// ------------------------------------------------------------------ launchers

namespace {

template <int NT, int R, int UNR, int EPI>
hipError_t gemv_launch(const GemvArgs &a, hipStream_t s) {
    const int waves = (a.rows + R - 1) / R;
    const dim3 grid((unsigned)((waves + 3) / 4), (unsigned)((a.t + NT - 1) / NT)), block(256);
    if (a.norm)
        hipLaunchKernelGGL((gemv_kernel<NT, R, UNR, EPI, true>), grid, block, 0, s, a);
    else
        hipLaunchKernelGGL((gemv_kernel<NT, R, UNR, EPI, false>), grid, block, 0, s, a);
    return hipGetLastError();
}

template <int R, int UNR, int EPI>
hipError_t gemv1_launch_unr(const GemvArgs &a, hipStream_t s) {
    const int waves = (a.rows + R - 1) / R;
    const dim3 grid((unsigned)((waves + 3) / 4)), block(256);
    if (a.parts)
        hipLaunchKernelGGL((gemv1_kernel<R, UNR, EPI, true, kMaxParts>), grid, block, 0, s, a);
    else if (a.norm)
        hipLaunchKernelGGL((gemv1_kernel<R, UNR, EPI, true, 0>), grid, block, 0, s, a);
    else
        hipLaunchKernelGGL((gemv1_kernel<R, UNR, EPI, false, 0>), grid, block, 0, s, a);
    return hipGetLastError();
}

// The unroll that covers the row (64 lanes x UNR float4s) with the fewest
// spare slots: every slot is a load (clamped in bounds), so spare ones cost
// load instructions (576 floats: 3; 1536: 6).
template <int R, int EPI>
hipError_t gemv1_launch(const GemvArgs &a, hipStream_t s) {
    const int need = ((a.cols >> 2) + 63) / 64;
    if (need <= 2) return gemv1_launch_unr<R, 2, EPI>(a, s);
    if (need <= 3) return gemv1_launch_unr<R, 3, EPI>(a, s);
    if (need <= 4) return gemv1_launch_unr<R, 4, EPI>(a, s);
    if (need <= 6) return gemv1_launch_unr<R, 6, EPI>(a, s);
    if (need <= 8) return gemv1_launch_unr<R, 8, EPI>(a, s);
    return hipErrorInvalidValue;
}

// Where gemv_wide_kernel is the faster one: 16 MB of weights or more, and the row
// (padded to passes of 2048 columns) and the waves' sums within 64 KiB of LDS.
// Its workgroups of 8 waves fill the CUs in coarser steps than gemv_kernel's 4, so
// past that the lines lie where its rounds are full (weights not in cache, us):
//   o / down (no norm): rows of 12288 columns and more, over three quarters to one
//     round of 512 workgroups (3716 x 14336 40.6 -> 36.7, 4096 x 14336 40.1 -> 39.3;
//     3072 x 14336 31.1 against 32.1, 4612 x 12288 40.9 / 42.1, 8192 columns 13.5 / 14.7)
//   gate/up: not from 2048 to 3072 rows (2436 x 3072 16.4 / 17.1), nor rows a multiple
//     of 32 KB apart (8192 x 8192 96.1 / 101.2); else 5 to 40% faster
//   the head: more than 4096 rows, and past 8192 rounds of 8192 rows at least seven
//     eighths full, up to 8 of them (4228 x 4096 23.3 -> 20.3, 32000 x 4096 104 -> 98;
//     3072 x 3072 13.2 / 13.9, 10244 x 4096 37.7 / 40.8, 20484 x 3072 43.7 / 45.5,
//     128256 x 3072 238 / 244)
//   q/k/v: always (5 to 60% faster).
template <int EPI>
bool gemv_wide(const GemvArgs &a) {
    if ((long long)a.rows * a.cols < (4 << 20) || a.cols > 7 * 2048) return false;
    if (EPI == kEpiResid) return !a.norm && a.cols >= 12288 && a.rows > 3072 && a.rows <= 4096;
    if (!a.norm || a.cols <= 2048) return false;
    if (EPI == kEpiSwiglu) return a.cols % 8192 != 0 && (a.rows <= 2048 || a.rows > 3072);
    if (EPI == kEpiStore || EPI == kEpiArgmax) {
        const long long rounds = (a.rows + 8191LL) / 8192;
        return a.rows > 4096 && rounds <= 8 && (rounds == 1 || 8LL * a.rows >= 7 * 8192 * rounds);
    }
    return true;
}

template <int R, int U, int EPI>
hipError_t gemv_wide_launch(const GemvArgs &a, hipStream_t s) {
    const int groups = (a.rows + R - 1) / R, passes = ((a.cols >> 2) + 64 * U - 1) / (64 * U);
    const dim3 grid((unsigned)std::min((groups + kWideWaves - 1) / kWideWaves, 512)), block(64 * kWideWaves);
    const size_t lds = (size_t)passes * 64 * U * sizeof(f4);
    hipLaunchKernelGGL((gemv_wide_kernel<R, U, EPI, EPI != kEpiResid>), grid, block, lds, s, a);
    return hipGetLastError();
}

// One token: one row per wave (the LM head, kEpiStore / kEpiArgmax, 4 rows per
// wave to keep more of its 100+ MB in flight per wave), the input row through
// LDS when it fits one pass (64 * 8 float4s), else gemv_kernel.  Several
// tokens: 4 per wave, 4 float4s per lane per pass.
template <int EPI>
hipError_t gemv_epi(const GemvArgs &a, hipStream_t s) {
    const bool one_pass = a.cols <= 4 * 64 * 8;
    if constexpr (EPI == kEpiArgmax) {
        if (a.t != 1 || !a.out1) return hipErrorInvalidValue;
        if (a.cols <= 4 * 64 * 4) return gemv1_launch<kArgmaxRows, EPI>(a, s);
        if (gemv_wide<EPI>(a)) return gemv_wide_launch<kArgmaxRows, 2, EPI>(a, s);
        return gemv_launch<1, kArgmaxRows, 4, EPI>(a, s);
    } else {
        if (a.t > 1) return gemv_launch<4, 1, 4, EPI>(a, s);
        if constexpr (EPI == kEpiStore) {
            if (a.cols <= 4 * 64 * 4) return gemv1_launch<4, EPI>(a, s);
            if (gemv_wide<EPI>(a)) return gemv_wide_launch<4, 2, EPI>(a, s);
            return gemv_launch<1, 4, 4, EPI>(a, s);
        }
        if (gemv_wide<EPI>(a)) return gemv_wide_launch<1, EPI == kEpiSwiglu ? 4 : 8, EPI>(a, s);
        if (one_pass) return gemv1_launch<1, EPI>(a, s);
        return gemv_launch<1, 1, 8, EPI>(a, s);
    }
}

}  // namespace

template <int UNR>
static hipError_t gemv1_states_launch(const GemvArgs &a, const DecodeStates &st, hipStream_t s) {
    const dim3 grid((unsigned)((a.rows + 3) / 4)), block(256);
    if (st.nchunks <= 4)
        hipLaunchKernelGGL((gemv1_states_kernel<UNR, 4>), grid, block, 0, s, a, st);
    else if (st.nchunks <= 8)
        hipLaunchKernelGGL((gemv1_states_kernel<UNR, 8>), grid, block, 0, s, a, st);
    else
        hipLaunchKernelGGL((gemv1_states_kernel<UNR, kStateChunks>), grid, block, 0, s, a, st);
    return hipGetLastError();
}

hipError_t launch_gemv_states(const GemvArgs &a, const DecodeStates &st, hipStream_t s) {
    if (a.rows <= 0) return hipSuccess;
    if (a.t != 1 || a.norm || a.cols > kStateCols || st.nchunks < 1 || st.nchunks > kStateChunks)
        return hipErrorInvalidValue;
    // the fewest spare slots of a row's float4s (gemv1_launch)
    const int need = ((a.cols >> 2) + 63) / 64;
    if (need <= 2) return gemv1_states_launch<2>(a, st, s);
    if (need <= 3) return gemv1_states_launch<3>(a, st, s);
    return gemv1_states_launch<4>(a, st, s);
}

hipError_t launch_gemv(int epi, const GemvArgs &a, hipStream_t s) {
    if (a.rows <= 0 || a.t <= 0) return hipSuccess;
    if (a.parts) {
        // the gate/up product after the fused decode + output projection
        if (epi != kEpiSwiglu || a.t != 1 || !a.norm || !a.xout || a.nparts < 1 || a.nparts > kMaxParts ||
            a.cols > 4 * 64 * 8)
            return hipErrorInvalidValue;
        return gemv1_launch<1, kEpiSwiglu>(a, s);
    }
    switch (epi) {
    case kEpiStore: return gemv_epi<kEpiStore>(a, s);
    case kEpiResid: return gemv_epi<kEpiResid>(a, s);
    case kEpiQkv: return gemv_epi<kEpiQkv>(a, s);
    case kEpiSwiglu: return gemv_epi<kEpiSwiglu>(a, s);
    case kEpiArgmax: return gemv_epi<kEpiArgmax>(a, s);
    default: return hipErrorInvalidValue;
    }
}

namespace {

template <int EPI, int RB, int TB, int NW, int KU>
hipError_t gemm_launch(const GemmArgs &a, hipStream_t s) {
    const int nrt = (a.rows + 16 * RB - 1) / (16 * RB), ntt = (a.t + 16 * TB - 1) / (16 * TB);
    hipLaunchKernelGGL((gemm_kernel<EPI, RB, TB, NW, KU>), dim3(8u * ((nrt + 7) / 8) * ntt), dim3(64 * NW), 0, s, a);
    return hipGetLastError();
}

template <int EPI>
hipError_t gemm_epi(const GemmArgs &a, hipStream_t s) {
    const GemmTile x = gemm_tile(EPI == kEpiSwiglu, a.rows, a.cols, a.t);
    const auto is = [&](int rb, int tb, int waves, int ku) {
        return x.rb == rb && x.tb == tb && x.waves == waves && x.ku == ku;
    };
    if (is(1, 1, 6, 2)) return gemm_launch<EPI, 1, 1, 6, 2>(a, s);
    if (is(1, 1, 8, 2)) return gemm_launch<EPI, 1, 1, 8, 2>(a, s);
    if (is(1, 2, 8, 2)) return gemm_launch<EPI, 1, 2, 8, 2>(a, s);
    if constexpr (EPI == kEpiSwiglu) {
        if (is(1, 2, 4, 2)) return gemm_launch<EPI, 1, 2, 4, 2>(a, s);
    } else {
        if (is(1, 1, 8, 4)) return gemm_launch<EPI, 1, 1, 8, 4>(a, s);
        if (is(1, 2, 6, 2)) return gemm_launch<EPI, 1, 2, 6, 2>(a, s);
        if (is(2, 2, 6, 2)) return gemm_launch<EPI, 2, 2, 6, 2>(a, s);
        if (is(2, 2, 8, 2)) return gemm_launch<EPI, 2, 2, 8, 2>(a, s);
        if (is(2, 4, 8, 2)) return gemm_launch<EPI, 2, 4, 8, 2>(a, s);
        if (is(5, 2, 8, 2)) return gemm_launch<EPI, 5, 2, 8, 2>(a, s);
    }
    return hipErrorInvalidValue;
}

}  // namespace

hipError_t launch_gemm(int epi, const GemmArgs &a, hipStream_t s) {
    if (a.rows <= 0 || a.t <= 0) return hipSuccess;
    if (a.cols % 4 != 0 || a.cols > kGemmCols || a.norm) return hipErrorInvalidValue;
    switch (epi) {
    case kEpiStore: return gemm_epi<kEpiStore>(a, s);
    case kEpiResid: return gemm_epi<kEpiResid>(a, s);
    case kEpiQkv: return gemm_epi<kEpiQkv>(a, s);
    case kEpiSwiglu: return gemm_epi<kEpiSwiglu>(a, s);
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_embed(const float *embed, const uint32_t *tokens, float *x, int t, int hidden, hipStream_t s,
                        const int *step, float *xg, const float *xnorm, float *xssq) {
    if (t <= 0) return hipSuccess;
    hipLaunchKernelGGL(embed_kernel, dim3((unsigned)t), dim3(256), 0, s, embed, tokens, step, x, hidden, xg, xnorm,
                       xssq);
    return hipGetLastError();
}

__global__ void set_step_kernel(int *counters, int step, int len) {
    counters[0] = step;
    counters[1] = len;
}

hipError_t launch_set_step(int *counters, int step, int len, hipStream_t s) {
    hipLaunchKernelGGL(set_step_kernel, dim3(1), dim3(1), 0, s, counters, step, len);
    return hipGetLastError();
}

hipError_t launch_argmax(const float *x, int n, uint32_t *out, hipStream_t s, int *step, int *len, const float *parts,
                         const float *embed, float *xe, int hidden) {
    hipLaunchKernelGGL(argmax_kernel, dim3(1), dim3(1024), 0, s, x, n, out, step, len, parts, embed, xe, hidden);
    return hipGetLastError();
}

}  // namespace wick
