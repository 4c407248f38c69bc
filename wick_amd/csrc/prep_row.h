// prep_row.h -- one row of the per-token input preparation, shared by the
// decode kernel's prologue (attention.hip) and the chunk kernel (prep.hip).
#pragma once

#include "wave_ops.h"

namespace wick {

typedef float f4 __attribute__((ext_vector_type(4)));

// The per-token preparation of src/model.rs:464-480 for one row of D floats,
// bit-identical to wick's CPU arithmetic (and to prep_kernel): bias add;
// rmsnorm_inplace (src/kernels.rs:351-357) -- a sequential f32 sum of squares
// from -0.0, ss / D, 1 / sqrt(ss + eps) with IEEE divide and square root, then
// (x * scale) * w; rope (src/model.rs:404-414) -- two rounded products and a
// rounded sum per output, (sin, cos) from the host-filled table row.
// A group of D/8 lanes (or 16, the rest idle) owns a row: lane l of the group
// holds the rotation quad j = 4l (< D/2), i.e. elements j..j+3 and
// j+D/2..j+D/2+3, so all loads go out at once; the sum of squares is carried
// through the lanes in element order (first half, then second half), each step
// a lane move within the row of 16.  rowbase is the group's first lane; every
// lane of the group must call this with the same row.
// prep_load16 requests a row's inputs as one lane of its 16 holds them and
// prep_finish16 does the arithmetic, so that a caller can request several
// rows' inputs before it waits for any.
struct PrepIn {
    f4 u, w, bu, bw, nu, nw, c, sn;
};

template <int D>
__device__ __forceinline__ PrepIn prep_load16(const float *src, const float *bias, const float *norm,
                                              const float *cosr, const float *sinr, int l16) {
    constexpr int H = D / 2, NQ = H / 4;
    const int j = l16 < NQ ? 4 * l16 : 0;
    PrepIn in;
    in.u = *reinterpret_cast<const f4 *>(src + j);
    in.w = *reinterpret_cast<const f4 *>(src + j + H);
    in.bu = in.bw = in.nu = in.nw = in.c = in.sn = f4{0.f, 0.f, 0.f, 0.f};
    if (bias) {
        in.bu = *reinterpret_cast<const f4 *>(bias + j);
        in.bw = *reinterpret_cast<const f4 *>(bias + j + H);
    }
    if (norm) {
        in.nu = *reinterpret_cast<const f4 *>(norm + j);
        in.nw = *reinterpret_cast<const f4 *>(norm + j + H);
    }
    if (cosr) {
        in.c = *reinterpret_cast<const f4 *>(cosr + j);
        in.sn = *reinterpret_cast<const f4 *>(sinr + j);
    }
    return in;
}

// The arithmetic of prep_row16 on loaded inputs; bias / norm / rot say which
// steps apply (the pointers prep_load16 was given were non-null).
template <int D>
__device__ __forceinline__ void prep_finish16(PrepIn in, float *dst, bool bias, bool norm, float eps, bool rot,
                                              int l16, int rowbase) {
#pragma clang fp contract(off)
    constexpr int H = D / 2, NQ = H / 4;
    const bool mine = l16 < NQ;
    const int j = mine ? 4 * l16 : 0;
    f4 u = in.u, w = in.w;
    if (bias) {
        u = u + in.bu;
        w = w + in.bw;
    }
    if (norm) {
        // at step i lane i of the group holds the sum so far and hands it on
        const f4 uu = u * u, ww = w * w;
        float run = -0.0f, m = 0.0f;
#pragma unroll
        for (int i = 0; i < NQ; i++) {
            m = run + uu.x;
            m = m + uu.y;
            m = m + uu.z;
            m = m + uu.w;
            run = dpp_f<kDppRowShr1>(m);
        }
        run = __shfl(m, rowbase + NQ - 1, 64);
#pragma unroll
        for (int i = 0; i < NQ; i++) {
            m = run + ww.x;
            m = m + ww.y;
            m = m + ww.z;
            m = m + ww.w;
            run = dpp_f<kDppRowShr1>(m);
        }
        run = __shfl(m, rowbase + NQ - 1, 64);
        run = run / (float)D;
        const float scale = 1.0f / sqrtf(run + eps);
        u = u * scale * in.nu;
        w = w * scale * in.nw;
    }
    if (rot) {
        const f4 a = u * in.c - w * in.sn;
        const f4 b = w * in.c + u * in.sn;
        u = a;
        w = b;
    }
    if (mine) {
        *reinterpret_cast<f4 *>(dst + j) = u;
        *reinterpret_cast<f4 *>(dst + j + H) = w;
    }
}

template <int D>
__device__ __forceinline__ void prep_row16(const float *src, float *dst, const float *bias, const float *norm,
                                           float eps, const float *cosr, const float *sinr, int l16, int rowbase) {
    const PrepIn in = prep_load16<D>(src, bias, norm, cosr, sinr, l16);
    prep_finish16<D>(in, dst, bias != nullptr, norm != nullptr, eps, cosr != nullptr, l16, rowbase);
}

}  // namespace wick
