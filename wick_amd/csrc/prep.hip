// prep.hip -- the per-token input preparation of wick's Model::forward on the
// device: bias add, per-head RMSNorm of q and k (QK-norm), rotate-half RoPE of
// q and k, and the append of k and v to the device KV cache
// (/root/reference/src/model.rs:464-484).
//
// The output is bit-identical to wick's CPU arithmetic, so the cache the
// attention kernels read holds exactly the bits the CPU path would hold
// (prep_row.h): the sum of squares is the CPU's sequential sum, floating-point
// contraction is off, the (sin, cos) pairs come from a table the host fills
// with the C library's sinf / cosf of the f32 angle pos * inv_freq[i].
#include <hip/hip_runtime.h>

#include <algorithm>

#include "attn_kernels.h"
#include "prep_row.h"

namespace wick {

// D/8 lanes per row r of t * (heads + 2 * kv_heads): token i = r / R, slot
// s = r % R; slots [0, heads) are q heads (rewritten in place), the next
// kv_heads are k heads and the last kv_heads are v heads (written to the
// cache at position start + i).
//
// A few bytes per row and a serial sum of D squares: bound by latency, so the
// rows are spread over as many waves as they fill and read whole.  (One thread
// per row read 16 bytes of 64 rows per load and filled a quarter of the CUs:
// 512 tokens of the Qwen3-0.6B shape, QK-norm, attention and a 4 MB copy
// included, 32.2 against 23.8 us.)
template <int D>
__global__ __launch_bounds__(256) void prep_kernel(const PrepArgs a) {
    constexpr int LANES = D / 8;
    const unsigned R = a.heads + 2 * a.kv_heads;
    const unsigned idx = blockIdx.x * 256u + threadIdx.x, r = idx / LANES;
    const int l = idx % LANES, rowbase = (threadIdx.x & 63) - l;
    if (r >= (unsigned)a.t * R) return;  // whole groups
    const int i = (int)(r / R), s = (int)(r % R), pos = a.start + i;
    const float *src, *bias = nullptr, *norm = nullptr;
    const float *cosr = a.rope_cos + (size_t)pos * (D / 2), *sinr = a.rope_sin + (size_t)pos * (D / 2);
    float *dst;
    if (s < a.heads) {
        src = dst = a.q + ((size_t)i * a.heads + s) * D;
        if (a.bq) bias = a.bq + (size_t)s * D;
        norm = a.qn;
    } else if (s < a.heads + a.kv_heads) {
        const int h = s - a.heads;
        src = a.ksrc + ((size_t)i * a.kv_heads + h) * D;
        dst = a.k + ((size_t)h * a.capacity + pos) * D;
        if (a.bk) bias = a.bk + (size_t)h * D;
        norm = a.kn;
    } else {
        const int h = s - a.heads - a.kv_heads;
        src = a.vsrc + ((size_t)i * a.kv_heads + h) * D;
        dst = a.v + ((size_t)h * a.capacity + pos) * D;
        if (a.bv) bias = a.bv + (size_t)h * D;
        cosr = sinr = nullptr;
    }
    prep_row16<D>(src, dst, bias, norm, a.eps, cosr, sinr, l, rowbase);
}

hipError_t launch_prep(int head_dim, const PrepArgs &all, hipStream_t s) {
    const long long R = all.heads + 2LL * all.kv_heads, lanes = head_dim / 8;
    // tokens per launch: lane indexes of one launch stay within 30 bits
    const int most = (int)std::max(1LL, std::min((long long)all.t, (1LL << 30) / (R * lanes)));
    for (int i = 0; i < all.t; i += most) {
        PrepArgs a = all;
        a.t = std::min(most, all.t - i);
        a.start += i;
        a.q += (size_t)i * all.heads * head_dim;
        a.ksrc += (size_t)i * all.kv_heads * head_dim;
        a.vsrc += (size_t)i * all.kv_heads * head_dim;
        const dim3 grid((unsigned)((a.t * R * lanes + 255) / 256)), block(256);
        switch (head_dim) {
        case 16: hipLaunchKernelGGL(prep_kernel<16>, grid, block, 0, s, a); break;
        case 32: hipLaunchKernelGGL(prep_kernel<32>, grid, block, 0, s, a); break;
        case 64: hipLaunchKernelGGL(prep_kernel<64>, grid, block, 0, s, a); break;
        case 128: hipLaunchKernelGGL(prep_kernel<128>, grid, block, 0, s, a); break;
        default: return hipErrorInvalidValue;
        }
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace wick
