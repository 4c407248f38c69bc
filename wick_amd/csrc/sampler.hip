// sampler.hip -- Sampler::sample (/root/reference/src/sampler.rs:73-127) as two
// kernels per draw, next to the logits the LM head wrote: a split kernel over
// up to kSampleParts slices of the vocabulary (one workgroup streams only a
// few tens of GB/s, so passes over the whole vocabulary are shared out), then
// one workgroup that finishes the draw.  Larger candidate sets than the split
// kernel's are sorted by many workgroups instead (launch_sorted).
//
// Phases (every branch that encloses a barrier depends only on kernel
// arguments or on LDS values read after a barrier, so all threads take it):
//   1. repetition penalty (:75-83) through a device bitset of seen ids, each
//      slice's ids by its workgroup;
//   2. temperature <= 0: argmax (:84-86, :129-137) per slice, then merged;
//   3. top-k (:87-94) on keys in f32::total_cmp order.  For k <= kFastK each
//      slice keeps its k best (key, id) pairs and the final kernel merges them
//      by rank.  Otherwise (or when a slice holds too many ties) an
//      11/11/10-bit radix select over the whole vocabulary finds the smallest
//      key bound whose candidate set holds the k best logits (the set ends at
//      a bin boundary, so it can hold more);
//   4. sort of that set by (key, id): bitonic in LDS up to kList entries, else
//      a stable LSD radix sort of the whole vocabulary in global memory; the
//      first k entries are the candidates, equal logits ordered by id;
//   5. softmax at the temperature (:95-98), min-p (:99-104), top-p (:105-115),
//      the draw (:116-125): f32 operations in wick's order (exp with the bits
//      of the C library's expf, exp_f32.h), the running sums and the draw
//      walked one element at a time by one wave.
// The sums stop early once the next term is at most a quarter ulp of the sum:
// the terms only shrink (the list is sorted), so no later term can change it.
#include <hip/hip_runtime.h>

#include <climits>
#include <cmath>

#include "exp_f32.h"
#include "sampler_kernels.h"
#include "wave_ops.h"

namespace wick {
namespace {

constexpr int kT = 1024, kW = kT / 64;
constexpr int kCopies = 16;            // histogram copies, indexed by lane % 16
constexpr int kStride = kCopies + 1;   // words per bin: odd, so a bin per lane reads 32 banks
constexpr int kMaxBins = 2048;         // 11-bit digits
constexpr int kList = 4096;            // largest candidate set sorted in LDS
constexpr int kSlicePer = kSliceMax / kT;  // slice entries per thread in the split kernel
constexpr int kPartCand = 1024;        // candidates one slice may hold at its k-th key
constexpr int kQuickCand = 256;        // candidates placed by rank behind quick_bound; past these a radix select is cheaper
// the slices' merge: past these one slice's k-th best is tried as the bound (logits
// sorted by id, 49152 of them: k 40 21.6 -> 18.5 us, k 20 19.0 -> 17.1)
constexpr int kOneCand = 192;

typedef float f4 __attribute__((ext_vector_type(4)));

struct SampleLds {
    union {
        uint32_t hist[kMaxBins * kStride];  // 136 KiB: radix select and sort histograms
        struct {
            unsigned long long cand[kList];  // (key << 32) | id
            float prob[kList];
        } l;
        uint32_t wcnt[kW * 256];  // global sort: per-wave digit counts, then offsets
    };
    uint32_t tot[kMaxBins];  // per-bin totals of the copies
    uint32_t run[256];       // global sort: next free slot per digit
    uint32_t wsum[kW];
    uint32_t sel_bin, sel_before, sel_count, count, min_pos;
    int any_nan, bad, fast;
    int pcount[kSampleParts];
    unsigned long long top[kFastK];  // the merged list of the split path
    float fv[kW];
    int fi[kW];
    float sum;
};

// f32::total_cmp order as an unsigned key, complemented so that ascending keys
// are descending logits.
__device__ __forceinline__ uint32_t desc_key(float x) {
    const uint32_t u = __float_as_uint(x);
    return ~((u & 0x80000000u) ? ~u : (u | 0x80000000u));
}

// acc + p == acc for every 0 <= p' <= p (round to nearest): p is at most a
// quarter of the spacing above acc (a margin of 2x over the exact half).
__device__ __forceinline__ bool negligible(float acc, float p) {
    const uint32_t e = (__float_as_uint(acc) >> 23) & 0xffu;
    if ((__float_as_uint(acc) >> 31) || e <= 25u || e == 255u) return false;
    return p <= __uint_as_float((e - 25u) << 23);
}

// The logit a desc_key came from (the key is a bijection of the bits).
__device__ __forceinline__ float key_value(uint32_t key) {
    const uint32_t ord = ~key;
    return __uint_as_float((ord & 0x80000000u) ? (ord & 0x7fffffffu) : ~ord);
}

__device__ __forceinline__ void arg_better(float v, int i, float &bv, int &bi) {
    if (v > bv || (v == bv && i < bi)) {
        bv = v;
        bi = i;
    }
}

// f(i, x[i]) for every i < n, by every thread of the block; 32 floats per
// thread in flight per pass.
template <class F>
__device__ __forceinline__ void for_each_logit(const float *__restrict__ x, int n, F &&f) {
    constexpr int U = 8;
    const int n4 = n >> 2;
    const f4 *x4 = reinterpret_cast<const f4 *>(x);
    for (int base = threadIdx.x; base < n4; base += U * kT) {
        f4 v[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int c = base + u * kT;
            v[u] = c < n4 ? x4[c] : f4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int c = base + u * kT;
            if (c < n4) {
                f(4 * c, v[u].x);
                f(4 * c + 1, v[u].y);
                f(4 * c + 2, v[u].z);
                f(4 * c + 3, v[u].w);
            }
        }
    }
    for (int i = 4 * n4 + (int)threadIdx.x; i < n; i += kT) f(i, x[i]);
}

// Exclusive prefix over the block of one value per thread; *total = the sum.
__device__ __forceinline__ uint32_t block_exclusive_scan(uint32_t v, SampleLds &s, uint32_t *total) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t inc = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t t = __shfl_up(inc, o, 64);
        if (lane >= o) inc += t;
    }
    if (lane == 63) s.wsum[w] = inc;
    __syncthreads();
    uint32_t before = 0, all = 0;
#pragma unroll
    for (int j = 0; j < kW; j++) {
        const uint32_t t = s.wsum[j];
        before += j < w ? t : 0u;
        all += t;
    }
    __syncthreads();
    *total = all;
    return before + inc - v;
}

// The walks below run in one whole wave with wave-uniform arguments.  A chunk
// of 64 terms is loaded one per lane and the running f32 value takes term j
// (broadcast by readlane) in order, the same in every lane.  The running sum
// only grows and the draw's remainder only shrinks (the terms are >= 0), so
// without NaNs a crossing shows in the chunk's last value; only that chunk is
// walked again keeping the value after term j in lane j, and one ballot finds
// the first term where the condition holds (with NaNs every chunk is, and the
// last chunk is walked that way directly).  Early
// exits of the sums are tested once per chunk: terms past the exit point are
// at most a quarter ulp of the running sum and would leave it unchanged.
__device__ __forceinline__ float lane_value(float v, int j) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), j));
}

// The first m (<= 64) terms of a chunk: all 64 unrolled, or in steps of 8 for
// a partial chunk (lanes past the valid terms hold zeros, which leave the
// value unchanged).
template <bool SUB>
__device__ __forceinline__ float chunk_end(float v, float acc, int m) {
    if (m == 64) {
#pragma unroll
        for (int j = 0; j < 64; j++) acc = SUB ? acc - lane_value(v, j) : acc + lane_value(v, j);
        return acc;
    }
    for (int j0 = 0; j0 < m; j0 += 8) {
#pragma unroll
        for (int j = j0; j < j0 + 8; j++) acc = SUB ? acc - lane_value(v, j) : acc + lane_value(v, j);
    }
    return acc;
}

template <bool SUB>
__device__ __forceinline__ float chunk_record(float v, float acc, int m) {
    const int lane = threadIdx.x & 63;
    float rec = 0.0f;
    if (m == 64) {
#pragma unroll
        for (int j = 0; j < 64; j++) {
            acc = SUB ? acc - lane_value(v, j) : acc + lane_value(v, j);
            rec = lane == j ? acc : rec;
        }
        return rec;
    }
    for (int j0 = 0; j0 < m; j0 += 8) {
#pragma unroll
        for (int j = j0; j < j0 + 8; j++) {
            acc = SUB ? acc - lane_value(v, j) : acc + lane_value(v, j);
            rec = lane == j ? acc : rec;
        }
    }
    return rec;
}

// The running f32 sum of p[0..n) in order, from acc.
__device__ __forceinline__ float sequential_sum(const float *p, int n, float acc, bool no_nan) {
    const int lane = threadIdx.x & 63;
    for (int base = 0; base < n; base += 64) {
        const float v = base + lane < n ? p[base + lane] : 0.0f;
        if (no_nan && negligible(acc, lane_value(v, 0))) break;
        acc = chunk_end<false>(v, acc, min(64, n - base));
    }
    return acc;
}

// top-p (src/sampler.rs:105-115): the running sum over p[0..*keep) from 0.0;
// *keep becomes i + 1 for the first i where it reaches top_p.  Returns the sum
// over the kept prefix (the total of :116).
__device__ __forceinline__ float top_p_cut(const float *p, int *keep, float top_p, bool no_nan) {
    const int lane = threadIdx.x & 63, n = *keep;
    float acc = 0.0f;
    for (int base = 0; base < n; base += 64) {
        const float v = base + lane < n ? p[base + lane] : 0.0f;
        if (no_nan && negligible(acc, lane_value(v, 0))) break;
        const int m = min(64, n - base);
        // the last chunk (or any, with NaNs) is walked keeping every value
        const bool last = base + 64 >= n;
        const float end = last || !no_nan ? 0.0f : chunk_end<false>(v, acc, m);
        if (last || !no_nan || end >= top_p) {
            const float run = chunk_record<false>(v, acc, m);
            const unsigned long long hit = __ballot(run >= top_p && base + lane < n);
            if (hit) {
                const int j = __builtin_ctzll(hit);
                *keep = base + j + 1;
                return lane_value(run, j);
            }
            acc = lane_value(run, m - 1);
        } else {
            acc = end;
        }
    }
    return acc;
}

// The draw (src/sampler.rs:118-125): r -= p[i] in order until r <= 0.
__device__ __forceinline__ int draw_index(const float *p, int keep, float r, bool no_nan) {
    const int lane = threadIdx.x & 63;
    for (int base = 0; base < keep; base += 64) {
        const float v = base + lane < keep ? p[base + lane] : 0.0f;
        const int m = min(64, keep - base);
        const bool last = base + 64 >= keep;
        const float end = last || !no_nan ? 0.0f : chunk_end<true>(v, r, m);
        if (last || !no_nan || end <= 0.0f) {
            const float run = chunk_record<true>(v, r, m);
            const unsigned long long hit = __ballot(run <= 0.0f && base + lane < keep);
            if (hit) return base + __builtin_ctzll(hit);
            r = lane_value(run, m - 1);
        } else {
            r = end;
        }
    }
    return keep - 1;
}

// Bitonic sort of one key per lane, ascending with the lane index.  The partner
// at a stride of 1 to 8 lanes comes by DPP, at 16 and 32 as the pair of a
// permlane swap, whose order does not matter to min and max: the 21 steps wait
// for no LDS (figures at quick_bound).
__device__ __forceinline__ unsigned long long wave_sort(unsigned long long v) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int size = 2; size <= 64; size <<= 1) {
#pragma unroll
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            const uint32_t vl = (uint32_t)v, vh = (uint32_t)(v >> 32);
            uint32_t lo, hi;
            if (stride >= 16) {
                const auto pl = stride == 16 ? __builtin_amdgcn_permlane16_swap(vl, vl, false, false)
                                             : __builtin_amdgcn_permlane32_swap(vl, vl, false, false);
                const auto ph = stride == 16 ? __builtin_amdgcn_permlane16_swap(vh, vh, false, false)
                                             : __builtin_amdgcn_permlane32_swap(vh, vh, false, false);
                v = ((unsigned long long)ph[0] << 32) | pl[0];
                lo = pl[1];
                hi = ph[1];
            } else if (stride == 8) {
                lo = dpp_i<kDppRowRor8>(vl);
                hi = dpp_i<kDppRowRor8>(vh);
            } else if (stride == 4) {  // lane ^ 7, then ^ 3
                lo = dpp_i<kDppQuadXor3>(dpp_i<kDppRowHalfMirror>(vl));
                hi = dpp_i<kDppQuadXor3>(dpp_i<kDppRowHalfMirror>(vh));
            } else if (stride == 2) {
                lo = dpp_i<kDppQuadXor2>(vl);
                hi = dpp_i<kDppQuadXor2>(vh);
            } else {
                lo = dpp_i<kDppQuadXor1>(vl);
                hi = dpp_i<kDppQuadXor1>(vh);
            }
            const unsigned long long o = ((unsigned long long)hi << 32) | lo;
            const bool keep_min = ((lane & stride) == 0) == ((lane & size) == 0);
            v = keep_min ? (v < o ? v : o) : (v < o ? o : v);
        }
    }
    return v;
}

// Rng::next_u64 (src/sampler.rs:45-55), xoshiro256**.
__device__ __forceinline__ uint64_t rotl64(uint64_t x, int k) { return (x << k) | (x >> (64 - k)); }
__device__ __forceinline__ uint64_t next_u64(uint64_t (&s)[4]) {
    const uint64_t out = rotl64(s[1] * 5u, 7) * 9u;
    const uint64_t t = s[1] << 17;
    s[2] ^= s[0];
    s[3] ^= s[1];
    s[1] ^= s[2];
    s[0] ^= s[3];
    s[2] ^= t;
    s[3] = rotl64(s[3], 45);
    return out;
}

// Radix select over the keys each(f) visits (f(key) once per element, by every
// thread of the block), most significant digit first with the digit widths
// WIDTHS (summing to 32, each at most 11): the candidate set {key <= *bound}
// of the k smallest keys; returns its size (>= k; above `limit` only after the
// last digit).
template <int... WIDTHS, class Each>
__device__ __forceinline__ uint32_t select_bound(Each &&each, uint32_t k, uint32_t limit, SampleLds &s, uint32_t *bound) {
    const int lane = threadIdx.x & 63;
    constexpr int NP = sizeof...(WIDTHS);
    const int widths[NP] = {WIDTHS...};
    uint32_t prefix = 0, pmask = 0, need = k, below = 0;
    int shift = 32;
    for (int pass = 0; pass < NP; pass++) {
        shift -= widths[pass];
        const int nb = 1 << widths[pass];
        for (int i = threadIdx.x; i < nb * kStride; i += kT) s.hist[i] = 0u;
        __syncthreads();
        const uint32_t dmask = (uint32_t)nb - 1u;
        each([&](uint32_t key) {
            if ((key & pmask) == prefix) atomicAdd(&s.hist[((key >> shift) & dmask) * kStride + (lane & 15)], 1u);
        });
        __syncthreads();
        // fold the copies (bin b by thread b % kT), then thread t owns bins
        // [t * per, (t + 1) * per) for the scan
        for (int b = threadIdx.x; b < nb; b += kT) {
            uint32_t c = 0u;
#pragma unroll
            for (int r = 0; r < kCopies; r++) c += s.hist[b * kStride + r];
            s.tot[b] = c;
        }
        __syncthreads();
        const int per = nb >= kT ? nb / kT : 1;
        uint32_t c[2] = {0u, 0u}, mine = 0u;
        if ((int)threadIdx.x * per < nb) {
            for (int j = 0; j < per; j++) {
                c[j] = s.tot[threadIdx.x * per + j];
                mine += c[j];
            }
        }
        uint32_t total;
        const uint32_t before = block_exclusive_scan(mine, s, &total);
        if (before < need && need <= before + mine) {
            uint32_t acc = before;
            for (int j = 0; j < per; j++) {
                if (need <= acc + c[j]) {
                    s.sel_bin = (uint32_t)(threadIdx.x * per + j);
                    s.sel_before = acc;
                    s.sel_count = c[j];
                    break;
                }
                acc += c[j];
            }
        }
        __syncthreads();
        const uint32_t bin = s.sel_bin, sb = s.sel_before, sc = s.sel_count;
        __syncthreads();
        const uint32_t le = below + sb + sc;
        if (le <= limit || pass == NP - 1) {
            *bound = prefix | (bin << shift) | ((1u << shift) - 1u);
            return le;
        }
        prefix |= bin << shift;
        pmask |= dmask << shift;
        need -= sb;
        below += sb;
    }
    return 0;  // not reached
}

// Stable LSD radix sort of (key0, idx0) over n entries, 8 bits per pass; the
// result ends in (key0, idx0).
__device__ void global_sort(uint32_t *key0, uint32_t *idx0, uint32_t *key1, uint32_t *idx1, int n, SampleLds &s) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const unsigned long long below_me = (1ull << lane) - 1ull;
    for (int pass = 0; pass < 4; pass++) {
        const int shift = 8 * pass;
        const uint32_t *sk = (pass & 1) ? key1 : key0, *si = (pass & 1) ? idx1 : idx0;
        uint32_t *dk = (pass & 1) ? key0 : key1, *di = (pass & 1) ? idx0 : idx1;
        for (int i = threadIdx.x; i < 256 * kStride; i += kT) s.hist[i] = 0u;
        __syncthreads();
        for (int i = threadIdx.x; i < n; i += kT) atomicAdd(&s.hist[((sk[i] >> shift) & 255u) * kStride + (lane & 15)], 1u);
        __syncthreads();
        uint32_t cnt = 0u;
        if (threadIdx.x < 256) {
#pragma unroll
            for (int r = 0; r < kCopies; r++) cnt += s.hist[threadIdx.x * kStride + r];
        }
        uint32_t total;
        const uint32_t base = block_exclusive_scan(cnt, s, &total);
        if (threadIdx.x < 256) s.run[threadIdx.x] = base;
        for (int i = threadIdx.x; i < kW * 256; i += kT) s.wcnt[i] = 0u;
        __syncthreads();
        for (int tile = 0; tile < n; tile += kT) {
            const int i = tile + (int)threadIdx.x;
            const bool valid = i < n;
            const uint32_t key = valid ? sk[i] : 0u, id = valid ? si[i] : 0u;
            const uint32_t d = (key >> shift) & 255u;
            // lanes of this wave holding the same digit
            unsigned long long peers = __ballot(valid);
#pragma unroll
            for (int b = 0; b < 8; b++) {
                const bool bit = (d >> b) & 1u;
                const unsigned long long m = __ballot(bit);
                peers &= bit ? m : ~m;
            }
            const uint32_t rank = (uint32_t)__popcll(peers & below_me);
            if (valid && rank == 0u) s.wcnt[w * 256 + d] = (uint32_t)__popcll(peers);
            __syncthreads();
            if (threadIdx.x < 256) {
                uint32_t off = s.run[threadIdx.x];
#pragma unroll
                for (int ww = 0; ww < kW; ww++) {
                    const uint32_t c = s.wcnt[ww * 256 + threadIdx.x];
                    s.wcnt[ww * 256 + threadIdx.x] = off;
                    off += c;
                }
                s.run[threadIdx.x] = off;
            }
            __syncthreads();
            if (valid) {
                const uint32_t pos = s.wcnt[w * 256 + d] + rank;
                if (pos < (uint32_t)n) {
                    dk[pos] = key;
                    di[pos] = id;
                } else {
                    s.bad = 2;
                }
            }
            __syncthreads();
            for (int j = threadIdx.x; j < kW * 256; j += kT) s.wcnt[j] = 0u;
            __syncthreads();
        }
    }
}

// Block-wide reduction of (bv, bi) with arg_better; the result in thread 0.
__device__ __forceinline__ void block_argmax(float &bv, int &bi, SampleLds &s) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const float ov = __shfl_xor(bv, off, 64);
        const int oi = __shfl_xor(bi, off, 64);
        arg_better(ov, oi, bv, bi);
    }
    if (lane == 0) {
        s.fv[w] = bv;
        s.fi[w] = bi;
    }
    __syncthreads();
    if (threadIdx.x == 0)
        for (int j = 1; j < kW; j++) arg_better(s.fv[j], s.fi[j], bv, bi);
}

// The number of keys[0..n) below c (the keys are distinct); the reads are
// broadcasts, eight in flight.
__device__ __forceinline__ int rank_of(unsigned long long c, const unsigned long long *keys, int n) {
    int r = 0, j = 0;
    for (; j + 8 <= n; j += 8) {
        unsigned long long v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = keys[j + u];
#pragma unroll
        for (int u = 0; u < 8; u++) r += v[u] < c ? 1 : 0;
    }
    for (; j < n; j++) r += keys[j] < c ? 1 : 0;
    return r;
}

__host__ __device__ inline uint32_t top_k_of(const SampleArgs &a) {
    return (a.top_k == 0u || a.top_k > (uint32_t)a.vocab) ? (uint32_t)a.vocab : a.top_k;
}

// A bound with at least k of the block's keys at or below it, so the k best are
// among those: every wave's ceil(k / kW)-th smallest of its lanes' smallest keys
// (`least`; ~0 for none), the largest of these over the waves.  A tight one needs
// the radix select, whose digits cost seven barriers and an LDS histogram each;
// this costs one barrier and leaves a few times k candidates to be ranked.  With
// the slices merged behind the same kind of bound and wave_sort off LDS, one draw
// with top-k 40 over 32000 ids 19.1 -> 13.6 us, 49152 18.4 -> 14.1, 151936 20.3 ->
// 15.8; top-k 50 over 128256 20.7 -> 17.5.  Sets s.count to 0.
__device__ __forceinline__ uint32_t quick_bound(uint32_t least, uint32_t k, SampleLds &s) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t b = 0u;
    for (uint32_t r = 0; r < (k + kW - 1) / kW; r++) {
        b = wave_min(least);
        if (lane == __builtin_ctzll(__ballot(least == b))) least = 0xffffffffu;
    }
    if (lane == 0) s.wsum[w] = b;
    if (threadIdx.x == 0) s.count = 0u;
    __syncthreads();
    b = s.wsum[0];
#pragma unroll
    for (int j = 1; j < kW; j++) b = max(b, s.wsum[j]);
    return b;
}

// The first kernel of a draw: workgroup g owns the slice [g * slice, +slice)
// of the vocabulary (slices are whole bitset words).  It applies the
// repetition penalty to its ids (src/sampler.rs:75-83, each distinct id once),
// then writes its slice's argmax (greedy) or, for k <= kFastK, its k best
// (key, id) pairs in order: the k best of the vocabulary are among these.
__global__ __launch_bounds__(kT) void sample_split_kernel(SampleArgs a) {
    __shared__ SampleLds s;
    const int g = blockIdx.x, tid = threadIdx.x;
    float *__restrict__ x = a.logits;
    const int lo = g * a.slice, hi = max(lo, min(a.vocab, lo + a.slice));
    if (a.penalty != 1.0f) {
        for (int i = tid; i < a.n_history; i += kT) {
            const uint32_t t = a.history[i];
            if (t >= (uint32_t)lo && t < (uint32_t)hi) {
                const uint32_t bit = 1u << (t & 31u);
                if (!(atomicOr(&a.flags[t >> 5], bit) & bit)) {
                    const float l = x[t];
                    x[t] = l > 0.0f ? l / a.penalty : l * a.penalty;
                }
            }
        }
        __syncthreads();
        for (int i = tid; i < a.n_history; i += kT) {
            const uint32_t t = a.history[i];
            if (t >= (uint32_t)lo && t < (uint32_t)hi) a.flags[t >> 5] = 0u;
        }
        __syncthreads();
    }
    if (a.temperature <= 0.0f) {
        float bv = -INFINITY;
        int bi = INT_MAX;
        for_each_logit(x + lo, hi - lo, [&](int i, float v) { arg_better(v, lo + i, bv, bi); });
        block_argmax(bv, bi, s);
        if (tid == 0) {
            a.part_val[g] = bv;
            a.part_id[g] = (uint32_t)bi;
        }
        return;
    }
    const uint32_t k = top_k_of(a);
    if (!a.split_top_k || k > (uint32_t)kFastK) return;
    uint32_t key[kSlicePer], least = 0xffffffffu;
#pragma unroll
    for (int j = 0; j < kSlicePer; j++) {
        const int i = lo + j * kT + tid;
        key[j] = i < hi ? desc_key(x[i]) : 0xffffffffu;
        least = min(least, key[j]);
    }
    auto gather = [&](uint32_t bound) {
#pragma unroll
        for (int j = 0; j < kSlicePer; j++) {
            const int i = lo + j * kT + tid;
            if (i < hi && key[j] <= bound) {
                const uint32_t pos = atomicAdd(&s.count, 1u);
                if (pos < (uint32_t)kPartCand) s.l.cand[pos] = ((unsigned long long)key[j] << 32) | (uint32_t)i;
            }
        }
        __syncthreads();
    };
    gather(quick_bound(least, k, s));
    uint32_t nset = s.count;
    if (nset > (uint32_t)kQuickCand) {  // many ties, or a few waves hold the best ids
        __syncthreads();
        uint32_t bound = 0xffffffffu;
        nset = (uint32_t)(hi - lo);
        if (k < nset)
            nset = select_bound<8, 8, 8, 8>(
                [&](auto &&f) {
#pragma unroll
                    for (int j = 0; j < kSlicePer; j++)
                        if (lo + j * kT + tid < hi) f(key[j]);
                },
                k, 64u, s, &bound);
        if (tid == 0) s.count = 0u;
        __syncthreads();
        if (nset > (uint32_t)kPartCand) {  // too many ties: the final kernel takes the whole vocabulary
            if (tid == 0) a.part_count[g] = -1;
            return;
        }
        gather(bound);
    }
    const int n = (int)min(s.count, (uint32_t)kPartCand);
    if (n <= 64) {  // one wave sorts them
        if (tid < 64) {
            const unsigned long long c = wave_sort(tid < n ? s.l.cand[tid] : ~0ull);
            if (tid < min(n, (int)k)) a.part_cand[g * kFastK + tid] = c;
        }
    } else if (tid < n) {
        const unsigned long long c = s.l.cand[tid];
        const int r = rank_of(c, s.l.cand, n);
        if (r < (int)k) a.part_cand[g * kFastK + r] = c;
    }
    if (tid == 0) a.part_count[g] = s.count == nset ? min(n, (int)k) : -1;
}

// The second kernel: one workgroup finishes the draw.
__global__ __launch_bounds__(kT) void sample_kernel(SampleArgs a) {
    __shared__ SampleLds s;
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    float *__restrict__ x = a.logits;
    const int vocab = a.vocab;

    // 2. greedy (src/sampler.rs:84-86): the first index of the maximum over the
    // slices' results; a NaN at index 0 (or no value above NaN) keeps index 0,
    // as argmax (:129-137)
    if (a.temperature <= 0.0f) {
        if (tid == 0) {
            float bv = -INFINITY;
            int bi = INT_MAX;
            for (int g = 0; g < a.parts; g++) arg_better(a.part_val[g], (int)a.part_id[g], bv, bi);
            if (bi == INT_MAX || isnan(x[0])) bi = 0;
            *a.out = (uint32_t)bi;
            a.res_meta[0] = 0;
            a.res_meta[1] = 0;
            a.res_meta[2] = 0;
        }
        return;
    }

    // 3./4. the k best logits, sorted (src/sampler.rs:87-94)
    const uint32_t k = top_k_of(a);
    const bool try_fast = a.split_top_k && k <= (uint32_t)kFastK;
    if (tid == 0) {
        s.count = 0u;
        s.bad = 0;
        s.fast = try_fast ? 1 : 0;
    }
    __syncthreads();
    if (try_fast && tid < a.parts) {
        const int c = a.part_count[tid];
        s.pcount[tid] = c;
        if (c < 0) s.fast = 0;
    }
    __syncthreads();
    const bool fast = s.fast != 0;
    bool in_lds = true;
    if (fast) {
        // Each thread holds at most one of the slices' pairs; those up to a bound
        // are sorted by one wave, or placed by rank where they are more.
        const int slots = a.parts * kFastK;
        unsigned long long mine = ~0ull;
        bool have = false;
        if (tid < slots) {
            const int g = tid / kFastK;
            have = tid - g * kFastK < min(s.pcount[g], kFastK);
            if (have) mine = a.part_cand[tid];
        }
        // every slice's ceil(k / parts)-th best, the largest of these: at least k
        // pairs up to it, where every slice has as many
        const int q = ((int)k + a.parts - 1) / a.parts - 1;
        uint32_t b = 0u;
        if (lane < a.parts)
            b = q < s.pcount[lane] ? (uint32_t)(a.part_cand[lane * kFastK + q] >> 32) : 0xffffffffu;
        uint32_t bound = ~wave_min(~b);
        if (have && (uint32_t)(mine >> 32) <= bound) s.l.cand[atomicAdd(&s.count, 1u)] = mine;
        __syncthreads();
        if (s.count > (uint32_t)kOneCand) {  // a few slices hold the best ids: up to one's own k-th best
            b = 0xffffffffu;
            if (lane < a.parts && (int)k <= s.pcount[lane]) b = (uint32_t)(a.part_cand[lane * kFastK + k - 1] >> 32);
            bound = wave_min(b);
            __syncthreads();
            if (tid == 0) s.count = 0u;
            __syncthreads();
            if (have && (uint32_t)(mine >> 32) <= bound) s.l.cand[atomicAdd(&s.count, 1u)] = mine;
            __syncthreads();
        }
        if (s.count > (uint32_t)kQuickCand) {  // hundreds of equal ids
            const uint32_t total = (uint32_t)__syncthreads_count(have);
            bound = 0xffffffffu;
            if (k < total)
                select_bound<8, 8, 8, 8>([&](auto &&f) { if (have) f((uint32_t)(mine >> 32)); }, k, 64u, s, &bound);
            if (tid == 0) s.count = 0u;
            __syncthreads();
            if (have && (uint32_t)(mine >> 32) <= bound) s.l.cand[atomicAdd(&s.count, 1u)] = mine;
            __syncthreads();
        }
        const int n = (int)s.count;
        if (n < (int)k && tid == 0) s.bad = 4;
        if (n <= 64) {
            if (w == 0) s.top[lane] = wave_sort(lane < n ? s.l.cand[lane] : ~0ull);
        } else {
            for (int t = tid; t < n; t += kT) {
                const unsigned long long c = s.l.cand[t];
                const int r = rank_of(c, s.l.cand, n);
                if (r < (int)k) s.top[r] = c;
            }
        }
        __syncthreads();
        for (int i = tid; i < (int)k; i += kT) a.res_idx[i] = (uint32_t)s.top[i];
    } else {
        uint32_t bound = 0xffffffffu, nset = (uint32_t)vocab;
        if (k < (uint32_t)vocab)
            nset = select_bound<11, 11, 10>(
                [&](auto &&f) { for_each_logit(x, vocab, [&](int, float v) { f(desc_key(v)); }); }, k,
                (uint32_t)kList, s, &bound);
        in_lds = nset <= (uint32_t)kList;
        if (in_lds) {
            for_each_logit(x, vocab, [&](int i, float v) {
                const uint32_t key = desc_key(v);
                if (key <= bound) {
                    const uint32_t pos = atomicAdd(&s.count, 1u);
                    if (pos < (uint32_t)kList) s.l.cand[pos] = ((unsigned long long)key << 32) | (uint32_t)i;
                }
            });
            __syncthreads();
            const uint32_t got = s.count;
            if (got != nset && tid == 0) s.bad = 1;
            const int n = (int)min(got, (uint32_t)kList);
            int n2 = 2;
            while (n2 < n) n2 <<= 1;
            for (int i = n + tid; i < n2; i += kT) s.l.cand[i] = ~0ull;
            __syncthreads();
            if (n2 <= 64) {
                if (w == 0) s.l.cand[lane] = wave_sort(lane < n ? s.l.cand[lane] : ~0ull);
                __syncthreads();
            } else {
                for (int size = 2; size <= n2; size <<= 1) {
                    for (int stride = size >> 1; stride > 0; stride >>= 1) {
                        for (int t = tid; t < (n2 >> 1); t += kT) {
                            const int lo = 2 * t - (t & (stride - 1)), hi = lo + stride;
                            const unsigned long long p = s.l.cand[lo], q = s.l.cand[hi];
                            if ((p > q) == ((lo & size) == 0)) {
                                s.l.cand[lo] = q;
                                s.l.cand[hi] = p;
                            }
                        }
                        __syncthreads();
                    }
                }
            }
            for (int i = tid; i < (int)k; i += kT) a.res_idx[i] = (uint32_t)s.l.cand[i];
        } else {
            for (int i = tid; i < vocab; i += kT) {
                a.key0[i] = desc_key(x[i]);
                a.res_idx[i] = (uint32_t)i;
            }
            __syncthreads();
            global_sort(a.key0, a.res_idx, a.key1, a.idx1, vocab, s);
        }
    }
    __syncthreads();

    // 5. probabilities (src/sampler.rs:95-98); the logits are read back from
    // the sorted keys
    float *prob = in_lds ? s.l.prob : a.res_prob;
    const unsigned long long *sorted = fast ? s.top : s.l.cand;
    auto logit = [&](int i) { return key_value(in_lds ? (uint32_t)(sorted[i] >> 32) : a.key0[i]); };
    const float mx = logit(0);
    if (tid == 0) s.any_nan = 0;
    __syncthreads();
    for (int i = tid; i < (int)k; i += kT) {
        const float p = exp_f32((logit(i) - mx) / a.temperature);
        prob[i] = p;
        if (isnan(p)) s.any_nan = 1;
    }
    __syncthreads();
    const bool any_nan = s.any_nan != 0;
    if (w == 0) {
        const float sum = sequential_sum(prob, (int)k, -0.0f, !any_nan);
        if (lane == 0) s.sum = sum;
    }
    if (tid == 0) s.min_pos = k;
    __syncthreads();
    const float sum = s.sum;
    for (int i = tid; i < (int)k; i += kT) {
        const float p = prob[i] / sum;
        prob[i] = p;
        if (in_lds) a.res_prob[i] = p;
    }
    __syncthreads();
    // min-p (src/sampler.rs:99-104): the first position below probs[0] * min_p
    if (a.min_p > 0.0f) {
        const float floor_p = prob[0] * a.min_p;
        for (int i = tid; i < (int)k; i += kT)
            if (prob[i] < floor_p) atomicMin(&s.min_pos, (uint32_t)i);
        __syncthreads();
    }
    if (w == 0) {
        int keep = max((int)s.min_pos, 1);
        // top-p (:105-115); the total (:116) is the same running sum over the kept prefix
        const float total = a.top_p < 1.0f ? top_p_cut(prob, &keep, a.top_p, !any_nan)
                                           : sequential_sum(prob, keep, 0.0f, !any_nan);
        uint64_t st[4] = {a.rng[0], a.rng[1], a.rng[2], a.rng[3]};
        const uint64_t u = next_u64(st);
        const float r = (float)(uint32_t)(u >> 40) / 16777216.0f * total;
        const int pick = draw_index(prob, keep, r, !any_nan);
        if (lane == 0) {
            a.rng[0] = st[0];
            a.rng[1] = st[1];
            a.rng[2] = st[2];
            a.rng[3] = st[3];
            const uint32_t id = in_lds ? (uint32_t)sorted[pick] : a.res_idx[pick];
            *a.out = min(id, (uint32_t)vocab - 1u);
            a.res_meta[0] = (int)k;
            a.res_meta[1] = keep;
            a.res_meta[2] = s.bad;
        }
    }
}

// ---------------------------------------------------------------- large candidate sets
//
// Thousands of candidates or all ids (sorts_vocabulary).  One workgroup took
// 2.3 ms a draw over all of 151936 ids: it sorted them at a few tens of GB/s
// and added the probabilities one at a time.  Here the whole vocabulary is sorted by a
// stable radix sort over as many workgroups as it fills, and the three walks in
// wick's order take thousands of terms at once where that gives the same bits
// (walk): 100 us a draw in 9 launches, each bound by its own latency (under the
// profiler: histograms 5-6 us, moves 12-14, sum 16, draw 23).
//
// Radix sort, 11 + 11 + 10 bits: per pass a histogram of every tile of kTile
// entries (sort_hist_kernel), then every tile finds its digits' places from all
// tiles' histograms and moves its entries (sort_move_kernel).  A wave owns 256
// consecutive entries of the tile and ranks equal digits by ballots, so the
// order among them is kept.  The first pass reads the logits, the last leaves
// the candidates' ids and exp terms.

constexpr int kSortE = 4, kTile = kT * kSortE;
static_assert(kTile == kSampleTile, "the sampler's buffers hold one histogram per tile");

// the lanes of this wave with the same BITS-bit digit
template <int BITS>
__device__ __forceinline__ unsigned long long same_digit(uint32_t d, bool valid) {
    unsigned long long peers = __ballot(valid);
#pragma unroll
    for (int b = 0; b < BITS; b++) {
        const bool bit = (d >> b) & 1u;
        const unsigned long long m = __ballot(bit);
        peers &= bit ? m : ~m;
    }
    return peers;
}

__device__ __forceinline__ int tile_entry(int e) {
    return (int)blockIdx.x * kTile + (int)(threadIdx.x >> 6) * 64 * kSortE + 64 * e + (int)(threadIdx.x & 63);
}

// PASS 0 takes key bits 0..10, PASS 1 bits 11..21, PASS 2 bits 22..31.
template <int PASS>
__global__ __launch_bounds__(kT) void sort_hist_kernel(SampleArgs a) {
    constexpr int BITS = PASS < 2 ? 11 : 10, NB = 1 << BITS, SHIFT = 11 * PASS;
    __shared__ uint32_t cnt[NB];
    __shared__ uint32_t least[kW];
    const uint2 *src = reinterpret_cast<const uint2 *>(PASS == 1 ? a.key0 : a.key1);
    uint32_t key[kSortE], best = 0xffffffffu;
#pragma unroll
    for (int e = 0; e < kSortE; e++) {
        const int i = min(tile_entry(e), a.vocab - 1);
        key[e] = PASS == 0 ? desc_key(a.logits[i]) : src[i].x;
        best = min(best, key[e]);
    }
    for (int b = threadIdx.x; b < NB; b += kT) cnt[b] = 0u;
    if (PASS == 0) {
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) best = min(best, (uint32_t)__shfl_xor((int)best, off, 64));
        if ((threadIdx.x & 63) == 0) least[threadIdx.x >> 6] = best;
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < kSortE; e++) {
        const bool valid = tile_entry(e) < a.vocab;
        const uint32_t d = (key[e] >> SHIFT) & (NB - 1);
        const unsigned long long peers = same_digit<BITS>(d, valid);
        if (valid && (peers & ((1ull << (threadIdx.x & 63)) - 1ull)) == 0ull) atomicAdd(&cnt[d], (uint32_t)__popcll(peers));
    }
    __syncthreads();
    for (int b = threadIdx.x; b < NB; b += kT) a.tile_hist[(size_t)blockIdx.x * NB + b] = (uint16_t)cnt[b];
    if (PASS == 0 && threadIdx.x == 0) {
        for (int j = 1; j < kW; j++) best = min(best, least[j]);
        a.tile_least[blockIdx.x] = best;
    }
}

template <int PASS>
__global__ __launch_bounds__(kT) void sort_move_kernel(SampleArgs a) {
    constexpr int BITS = PASS < 2 ? 11 : 10, NB = 1 << BITS, SHIFT = 11 * PASS, U = 16;
    __shared__ __attribute__((aligned(16))) uint16_t wcnt[kW][NB];  // a wave's digit counts, then its places within the tile's
    __shared__ uint32_t base[NB];
    __shared__ uint32_t wsum[kW];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, tiles = gridDim.x;
    const uint2 *src = reinterpret_cast<const uint2 *>(PASS == 1 ? a.key0 : a.key1);
    uint32_t key[kSortE], id[kSortE], pos[kSortE];
#pragma unroll
    for (int e = 0; e < kSortE; e++) {
        const int i = min(tile_entry(e), a.vocab - 1);
        const uint2 in = PASS == 0 ? make_uint2(desc_key(a.logits[i]), (uint32_t)i) : src[i];
        key[e] = in.x;
        id[e] = in.y;
    }
    // the thread's two bins over all tiles, and over the tiles before this one
    const bool owner = 2 * tid < NB;
    uint32_t tot0 = 0u, tot1 = 0u, bef0 = 0u, bef1 = 0u;
    if (owner) {
        // 16-bit counts: every tile reads all of them, 27 GB/s a CU
        const uint32_t *h = reinterpret_cast<const uint32_t *>(a.tile_hist) + tid;
        for (int t0 = 0; t0 < tiles; t0 += U) {
            uint32_t c[U];
#pragma unroll
            for (int u = 0; u < U; u++) c[u] = h[(size_t)min(t0 + u, tiles - 1) * (NB / 2)];
#pragma unroll
            for (int u = 0; u < U; u++) {
                c[u] = t0 + u < tiles ? c[u] : 0u;
                if (t0 + u == (int)blockIdx.x) {
                    bef0 = tot0;
                    bef1 = tot1;
                }
                tot0 += c[u] & 0xffffu;
                tot1 += c[u] >> 16;
            }
        }
    }
    for (int b = tid; b < kW * NB / 2; b += kT) reinterpret_cast<uint32_t *>(&wcnt[0][0])[b] = 0u;
    // exclusive prefix of the bins' totals over the threads
    uint32_t inc = tot0 + tot1;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t t = __shfl_up(inc, o, 64);
        if (lane >= o) inc += t;
    }
    if (lane == 63) wsum[w] = inc;
    __syncthreads();
    uint32_t excl = inc - tot0 - tot1;
#pragma unroll
    for (int j = 0; j < kW; j++) excl += j < w ? wsum[j] : 0u;
    if (owner) {
        base[2 * tid] = excl + bef0;
        base[2 * tid + 1] = excl + tot0 + bef1;
    }
#pragma unroll
    for (int e = 0; e < kSortE; e++) {
        const bool valid = tile_entry(e) < a.vocab;
        const uint32_t d = (key[e] >> SHIFT) & (NB - 1);
        const unsigned long long peers = same_digit<BITS>(d, valid);
        const uint32_t rank = (uint32_t)__popcll(peers & ((1ull << lane) - 1ull)), before = wcnt[w][d];
        pos[e] = before + rank;
        __builtin_amdgcn_wave_barrier();
        if (valid && rank == 0u) wcnt[w][d] = (uint16_t)(before + (uint32_t)__popcll(peers));
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    // a wave's counts become its places among the tile's (two 16-bit bins at a
    // time: none passes kTile)
    if (owner) {
        uint32_t c[kW], off = 0u;
#pragma unroll
        for (int j = 0; j < kW; j++) c[j] = *reinterpret_cast<const uint32_t *>(&wcnt[j][2 * tid]);
#pragma unroll
        for (int j = 0; j < kW; j++) {
            *reinterpret_cast<uint32_t *>(&wcnt[j][2 * tid]) = off;
            off += c[j];
        }
    }
    float mx = 0.0f;
    if (PASS == 2) {
        uint32_t best = 0xffffffffu;
        for (int t = lane; t < tiles; t += 64) best = min(best, a.tile_least[t]);
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) best = min(best, (uint32_t)__shfl_xor((int)best, o, 64));
        mx = key_value(best);
    }
    __syncthreads();
    const uint32_t k = top_k_of(a);
#pragma unroll
    for (int e = 0; e < kSortE; e++) {
        if (tile_entry(e) >= a.vocab) continue;
        const uint32_t d = (key[e] >> SHIFT) & (NB - 1), to = base[d] + wcnt[w][d] + pos[e];
        if (PASS == 2) {
            // src/sampler.rs:95-98, the terms before their sum
            if (to < k) {
                a.res_idx[to] = id[e];
                a.res_prob[to] = exp_f32((key_value(key[e]) - mx) / a.temperature);
            }
        } else if (to < (uint32_t)a.vocab) {
            reinterpret_cast<uint2 *>(PASS == 0 ? a.key0 : a.key1)[to] = make_uint2(key[e], id[e]);
        }
    }
}

// wick's running f32 sums, term by term in order, by the whole workgroup:
//   kWalkSum   acc + p[0] + p[1] + ...
//   kWalkReach the same until the sum reaches limit (>=): *hit is that term
//   kWalkDrain acc - p[0] - p[1] - ... until it is <= 0: *hit is that term
// (*hit = -1 where it never does), the value there or at the end returned in
// every thread.  No NaNs; p >= 0 and never grows by more than a rounding.
//
// While acc stays within one power of two, acc = R u with u its ulp and R an
// integer, acc + p rounds to (R + rint(p/u)) u -- but for p/u exactly half way
// between two integers, where it depends on R.  So a run of terms none of which
// ties, that does not leave the power of two, changes R by the sum of the
// rint(p/u), integers that add up exactly in any order.  Every wave adds up 1024
// consecutive terms at acc's ulp; the waves' sums are taken in order, and a wave
// whose terms tie or leave the power of two (or hold the hit) takes them in
// chunks of 64 the same way, one term at a time where even that fails.  A sum
// must end below 2^24 u, a remainder at 2^23 + 1 or above: then no value on the
// way, before its rounding, was past the power of two.
constexpr int kWalkU = 16, kWalkTerms = 64 * kWalkU;
static_assert(kW == 16 && kWalkU == 16, "16 waves of 16 chunks: a row of 16 lanes holds one sum of each");
enum WalkMode { kWalkSum, kWalkReach, kWalkDrain };

struct WalkLds {
    __attribute__((aligned(16))) float v[kWalkTerms];  // of the wave that walks its terms
    float sum[kW], csum[kWalkU];                       // of the waves, of that wave's chunks
    int tie[kW], ctie[kWalkU];
    float acc;
    int hit;
};

// u, 1/u for acc's ulp u; false where acc is negative, zero, tiny or not finite
__device__ __forceinline__ bool ulp_of(float acc, float &u, float &inv) {
    const uint32_t b = __float_as_uint(acc), e = b >> 23;
    if (e < 25u || e >= 255u) return false;
    u = __uint_as_float((e - 23u) << 23);
    inv = __uint_as_float((277u - e) << 23);
    return true;
}

// Takes the sums [next, n) of 16 runs of terms (lane l holds run l % 16's) into
// R in order, as far as they need no closer look; returns the first not taken.
template <WalkMode MODE>
__device__ __forceinline__ int take_runs(float &R, float sum, bool tie, int next, int n, float u, float limit) {
    const int l = threadIdx.x & 15;
    const bool mine = l >= next;
    float inc = mine ? sum : 0.0f;  // the sum of runs [next, l]
    inc += dpp_f<0x111>(inc);       // row_shr 1, 2, 4, 8
    inc += dpp_f<0x112>(inc);
    inc += dpp_f<0x114>(inc);
    inc += dpp_f<0x118>(inc);
    const float R2 = MODE == kWalkDrain ? R - inc : R + inc;
    bool ok = !tie && (MODE == kWalkDrain ? R2 >= 8388609.0f : R2 < 16777216.0f);
    if (MODE == kWalkReach) ok = ok && R2 * u < limit;
    const unsigned stop = (unsigned)__ballot(mine && !ok) & 0xffffu;
    const int first = min(stop ? (int)__builtin_ctz(stop) : 16, n);
    if (first > next) R = lane_value(R2, first - 1);
    return first;
}

// the integers a lane's 4 consecutive terms change R by
__device__ __forceinline__ float run_units(const f4 &v, float inv, bool &tie) {
    float sum = 0.0f;
#pragma unroll
    for (int c = 0; c < 4; c++) {
        const float t = v[c] * inv, r = rintf(t);
        tie |= fabsf(t - r) == 0.5f;
        sum += r;  // exact up to 2^24, not below it past that
    }
    return sum;
}

template <WalkMode MODE>
__device__ __forceinline__ float walk(const float *__restrict__ p, int n, float acc, float limit, int *hit, WalkLds &s) {
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    *hit = -1;
    f4 ahead[kWalkU / 4];
    const auto fetch = [&](int base) {
#pragma unroll
        for (int j = 0; j < kWalkU / 4; j++) {
            const int i = base + w * kWalkTerms + 256 * j + 4 * lane;
            ahead[j] = *reinterpret_cast<const f4 *>(p + min(i, (n - 1) & ~3));
        }
    };
    fetch(0);
    for (int base = 0; base < n; base += kW * kWalkTerms) {
        // terms that cannot change the sum any more
        if (MODE != kWalkDrain && negligible(acc, p[base])) break;
        const int wb = base + w * kWalkTerms, nw = min(kW, (n - base + kWalkTerms - 1) / kWalkTerms);
        // the next round's terms are on their way while this one's are added
        f4 v[kWalkU / 4];
#pragma unroll
        for (int j = 0; j < kWalkU / 4; j++) {
            const int i = wb + 256 * j + 4 * lane;
            v[j] = ahead[j];
#pragma unroll
            for (int c = 0; c < 4; c++) v[j][c] = i + c < n ? v[j][c] : 0.0f;  // adds nothing
        }
        fetch(base + kW * kWalkTerms);
        int next = 0;  // the first wave whose terms are not in acc
        while (next < nw) {
            float u, inv;
            if (ulp_of(acc, u, inv)) {
                float sum = 0.0f;
                bool tie = false;
#pragma unroll
                for (int j = 0; j < kWalkU / 4; j++) sum += run_units(v[j], inv, tie);
                sum = wave_sum(sum);
                const bool any = __any(tie);
                if (lane == 0) {
                    s.sum[w] = sum;
                    s.tie[w] = any;
                }
                __syncthreads();
                float R = acc * inv;
                next = take_runs<MODE>(R, s.sum[lane & 15], s.tie[lane & 15] != 0, next, nw, u, limit);
                acc = R * u;
            }
            if (next < nw && w == next) {
                int h = -1;
#pragma unroll
                for (int j = 0; j < kWalkU / 4; j++) *reinterpret_cast<f4 *>(&s.v[256 * j + 4 * lane]) = v[j];
                const int nc = min(kWalkU, (n - wb + 63) / 64);
                for (int c = 0; c < nc && h < 0; c++) {
                    float cu, cinv;
                    if (ulp_of(acc, cu, cinv)) {
                        // chunk 4j + lane / 16: a row of 16 lanes' float4 j
#pragma unroll
                        for (int j = 0; j < kWalkU / 4; j++) {
                            bool tie = false;
                            float sum = run_units(v[j], cinv, tie);
                            sum += dpp_f<kDppQuadXor1>(sum);
                            sum += dpp_f<kDppQuadXor2>(sum);
                            sum += dpp_f<kDppRowHalfMirror>(sum);
                            sum += dpp_f<kDppRowMirror>(sum);
                            const unsigned ties = (unsigned)(__ballot(tie) >> (lane & 48)) & 0xffffu;
                            if ((lane & 15) == 0) {
                                s.csum[4 * j + (lane >> 4)] = sum;
                                s.ctie[4 * j + (lane >> 4)] = ties != 0u;
                            }
                        }
                        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                        __builtin_amdgcn_wave_barrier();
                        float R = acc * cinv;
                        c = take_runs<MODE>(R, s.csum[lane & 15], s.ctie[lane & 15] != 0, c, nc, cu, limit);
                        acc = R * cu;
                        if (c >= nc) break;
                    }
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    __builtin_amdgcn_wave_barrier();
                    const float x = s.v[64 * c + lane];
                    if (MODE == kWalkSum) {
                        acc = chunk_end<false>(x, acc, 64);
                    } else {
                        const float run = chunk_record<MODE == kWalkDrain>(x, acc, 64);
                        const unsigned long long at = __ballot((MODE == kWalkDrain ? run <= 0.0f : run >= limit) &&
                                                               wb + 64 * c + lane < n);
                        const int stop = at ? (int)__builtin_ctzll(at) : 63;
                        if (at) h = wb + 64 * c + stop;
                        acc = lane_value(run, stop);
                    }
                }
                if (lane == 0) {
                    s.acc = acc;
                    s.hit = h;
                }
            }
            __syncthreads();
            if (next < nw) {
                acc = s.acc;
                *hit = s.hit;
                next++;
            }
            // The next turn writes what was just read; so does the first turn of a
            // next walk on the same LDS, before any other barrier where it starts
            // from zero.
            __syncthreads();
            if (*hit >= 0) return acc;
        }
    }
    return acc;
}

// The sum of the terms (src/sampler.rs:97) to walk[0], the first term to
// walk[1].  NaN logits sort first or last (f32::total_cmp) and make an end term
// NaN, as does an infinite maximum; then every probability is NaN.
__global__ __launch_bounds__(kT) void sample_sum_kernel(SampleArgs a) {
    __shared__ WalkLds s;
    const int k = (int)top_k_of(a);
    const float first = a.res_prob[0], last = a.res_prob[k - 1];
    int hit;
    const float sum = isnan(first) || isnan(last) ? first + last : walk<kWalkSum>(a.res_prob, k, -0.0f, 0.0f, &hit, s);
    if (threadIdx.x == 0) {
        a.walk[0] = sum;
        a.walk[1] = first;
    }
}

// The terms over their sum, and each workgroup's first position below min-p's
// floor (src/sampler.rs:98-104).
__global__ __launch_bounds__(kT) void sample_normalise_kernel(SampleArgs a) {
    __shared__ int below;
    const int k = (int)top_k_of(a), i = blockIdx.x * kT + threadIdx.x;
    const float sum = a.walk[0], floor_p = a.walk[1] / sum * a.min_p;
    if (threadIdx.x == 0) below = INT_MAX;
    __syncthreads();
    if (i < k) {
        const float p = a.res_prob[i] / sum;
        a.res_prob[i] = p;
        if (a.min_p > 0.0f && p < floor_p) atomicMin(&below, i);
    }
    __syncthreads();
    if (threadIdx.x == 0) a.tile_below[blockIdx.x] = below;
}

// top-p and the draw (src/sampler.rs:105-125).
__global__ __launch_bounds__(kT) void sample_draw_kernel(SampleArgs a) {
    __shared__ WalkLds s;
    __shared__ int below;
    const int k = (int)top_k_of(a);
    if (threadIdx.x == 0) below = k;
    uint64_t st[4] = {a.rng[0], a.rng[1], a.rng[2], a.rng[3]};
    __syncthreads();
    for (int b = threadIdx.x; b < (k + kT - 1) / kT; b += kT) atomicMin(&below, a.tile_below[b]);
    __syncthreads();
    int keep = max(below, 1), hit = -1;
    const uint64_t u = next_u64(st);
    if (!isnan(a.walk[0])) {
        float total;
        if (a.top_p < 1.0f) {
            total = walk<kWalkReach>(a.res_prob, keep, 0.0f, a.top_p, &hit, s);
            if (hit >= 0) keep = hit + 1;
        } else {
            total = walk<kWalkSum>(a.res_prob, keep, 0.0f, 0.0f, &hit, s);
        }
        const float r = (float)(uint32_t)(u >> 40) / 16777216.0f * total;
        walk<kWalkDrain>(a.res_prob, keep, r, 0.0f, &hit, s);
    }
    const int pick = hit >= 0 ? hit : keep - 1;
    __syncthreads();  // every thread has read the generator
    if (threadIdx.x == 0) {
        for (int j = 0; j < 4; j++) a.rng[j] = st[j];
        *a.out = min(a.res_idx[pick], (uint32_t)a.vocab - 1u);
        a.res_meta[0] = k;
        a.res_meta[1] = keep;
        a.res_meta[2] = 0;
    }
}

hipError_t launch_sorted(const SampleArgs &a, hipStream_t s) {
    const dim3 tiles((unsigned)((a.vocab + kTile - 1) / kTile)), block(kT);
    hipLaunchKernelGGL(sort_hist_kernel<0>, tiles, block, 0, s, a);
    hipLaunchKernelGGL(sort_move_kernel<0>, tiles, block, 0, s, a);
    hipLaunchKernelGGL(sort_hist_kernel<1>, tiles, block, 0, s, a);
    hipLaunchKernelGGL(sort_move_kernel<1>, tiles, block, 0, s, a);
    hipLaunchKernelGGL(sort_hist_kernel<2>, tiles, block, 0, s, a);
    hipLaunchKernelGGL(sort_move_kernel<2>, tiles, block, 0, s, a);
    hipLaunchKernelGGL(sample_sum_kernel, dim3(1), block, 0, s, a);
    hipLaunchKernelGGL(sample_normalise_kernel, dim3((top_k_of(a) + kT - 1) / kT), block, 0, s, a);
    hipLaunchKernelGGL(sample_draw_kernel, dim3(1), block, 0, s, a);
    return hipGetLastError();
}

}  // namespace

// Draws that launch_sorted serves: more candidates than one workgroup selects
// and sorts faster.  The workgroup's time steps up where its sort goes from 1024
// to 2048 slots, at a k that depends on the logits (those that share their high
// bits latest).  One workgroup against the sort, top-p 0.9: 20000 ids, k 1025 46
// / 62 us, 1600 52 / 61, 2049 72 / 62, all of them 341 / 68; 32000 ids, k 1800,
// logits of one exponent, 76 / 85; 65536, the same, 82 / 84, k 2048 103 / 81;
// 100000 ids, the same, k 1400 78 / 84, 1600 99 / 88; 151936 ids, k 1025 69 / 74,
// 1600 98 / 75, all of them 2267 / 101; 16384 ids, k 2049 73 / 64.  Up to kList
// ids every set fits the workgroup's LDS.
bool sorts_vocabulary(const SampleArgs &a) {
    const uint32_t k = top_k_of(a);
    return !(a.temperature <= 0.0f) && a.vocab > kList && k > (a.vocab >= 100000 ? 1600u : 2048u);
}

hipError_t launch_sample(const SampleArgs &a, hipStream_t s) {
    // the split kernel is needed for the penalty, greedy, and the split top-k
    if (a.penalty != 1.0f || a.temperature <= 0.0f || (a.split_top_k && top_k_of(a) <= (uint32_t)kFastK)) {
        hipLaunchKernelGGL(sample_split_kernel, dim3(a.parts), dim3(kT), 0, s, a);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    if (sorts_vocabulary(a)) return launch_sorted(a, s);
    hipLaunchKernelGGL(sample_kernel, dim3(1), dim3(kT), 0, s, a);
    return hipGetLastError();
}

}  // namespace wick
