// ACT-SHAVE `mvn1`: per normalisation group, y = (x - mean) / sqrt(var + eps) (eps inside the
// square root) or x - mean; group = (C,H,W) of one batch element when across_channels, else (H,W)
// of one channel (VPU.MVN, src/vpux_compiler/tblgen/vpux/compiler/dialect/VPU/ops.td:3600-3652).
//
// Statistics are fp32: mean and centred sum of squares in two passes over values that stay on chip, or in one about a first mean where that is
// as exact (slice_moments).  Where a group is more than one workgroup's, each publishes the moments {count, mean, M2} of its part and the parts
// meet in a fixed order -- pairwise with the update of Chan et al., or all at once about their common mean -- so results do not depend on scheduling.  This is the
// decomposition the compiler itself uses when a group does not fit local memory
// (MVN1Sum -> MVN1MeanVar -> MVN1Normalize,
// src/vpux_compiler/src/NPU37XX/dialect/VPU/transforms/passes/decompose_mvn.cpp:82-129), with
// centred partial sums instead of raw sum / sum of squares.
//
// Groups that one wavefront or workgroup holds (registers or LDS) take one launch without any exchange.  Up to 16 longer
// groups that the chip's registers hold take one launch whose workgroups exchange their moments (mvn_fused_kernel): tagged
// records that each polls for its own group, 2.9 us, where an arrival counter for the whole device took about 30.  What is
// left -- more or longer groups, input and output in one place -- takes two launches over 4096-element chunks, the second
// of which reads the tensor again.
#include <atomic>
#include <type_traits>

#include "vpx_common.h"

namespace vpx {

namespace {

typedef _Float16 half_t;
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef half_t halfx8 __attribute__((ext_vector_type(8)));
typedef u32x4 __attribute__((aligned(2))) u32x4_any;  // a 128-bit access at any fp16 address

constexpr int kThreads = 256;
constexpr int kVecPerThread = 2;                           // 128-bit loads per lane
constexpr int kChunk = kThreads * kVecPerThread * 8;       // fp16 elements per workgroup
constexpr int kMergeInKernel = 256;                        // most chunks per group merged inside the normalise kernel

struct Moments {
    float n, mean, m2;
};

// A published record: 16 bytes, so that it moves as one access.
struct __attribute__((aligned(16))) Record {
    float n, mean, m2, pad;
};
__device__ __forceinline__ Moments unpack(const Record& r) {
    return Moments{r.n, r.mean, r.m2};
}

// Chan/Golub/LeVeque pairwise combination of two sample sets.
__device__ __forceinline__ Moments merge(Moments a, Moments b) {
    const float n = a.n + b.n;
    if (n == 0.f) return Moments{0.f, 0.f, 0.f};
    const float d = b.mean - a.mean;
    const float w = b.n * __builtin_amdgcn_rcpf(n);  // 1 ulp; the same everywhere, so still deterministic
    Moments r;
    r.n = n;
    r.mean = a.mean + d * w;
    r.m2 = a.m2 + b.m2 + d * d * a.n * w;
    return r;
}

template <int CTRL>
__device__ __forceinline__ float dppf(float v) {
    const int i = __builtin_bit_cast(int, v);
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(i, i, CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float swz16(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_ds_swizzle(__builtin_bit_cast(int, v), 0x401F));
}
__device__ __forceinline__ float lane_bcast(float v, int lane) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}

__device__ __forceinline__ float wave_sum(float v) {
    v += dppf<0xB1>(v);
    v += dppf<0x4E>(v);
    v += dppf<0x141>(v);
    v += dppf<0x140>(v);
    v += swz16(v);
    return lane_bcast(v, 0) + lane_bcast(v, 32);
}
// The same bits with a lane of each row of 16 read instead of the trip through LDS: shorter where a workgroup waits for its sum ([3,144,82,56] across
// channels 6.93 -> 6.54 us, layer norm [25 x 3008] 3.74 -> 3.54), more vector instructions where many wavefronts hide the trip ([6052 x 576] 6.10 -> 6.37).
__device__ __forceinline__ float wave_sum_soon(float v) {
    v += dppf<0xB1>(v);
    v += dppf<0x4E>(v);
    v += dppf<0x141>(v);
    v += dppf<0x140>(v);
    return (lane_bcast(v, 0) + lane_bcast(v, 16)) + (lane_bcast(v, 32) + lane_bcast(v, 48));
}

// a / n where 1 / n, correctly rounded, was at hand before a was: two fused operations behind the product in place of the dozen of a division, whose
// result this is.  An infinite a stays infinite.
__device__ __forceinline__ float over(float a, float n, float inv_n) {
    const float q = a * inv_n;
    return __builtin_fabsf(q) < __builtin_inff() ? __builtin_fmaf(__builtin_fmaf(-q, n, a), inv_n, q) : q;
}

// 1 / sqrt(v): the hardware's approximation and one Newton step, within an ulp as a rounded root and a rounded quotient are, in a fifth of their
// instructions.  Outside the normal numbers those.
__device__ __forceinline__ float inv_root(float v) {
    if (!(v >= 0x1p-126f && v < __builtin_inff())) return 1.0f / __builtin_sqrtf(v);
    const float y = __builtin_amdgcn_rsqf(v);
    return __builtin_fmaf(0.5f * y, __builtin_fmaf(-v * y, y, 1.0f), y);
}

template <class Shuffle>
__device__ __forceinline__ Moments merge_with(Moments m, Shuffle sh) {
    return merge(m, Moments{sh(m.n), sh(m.mean), sh(m.m2)});
}

// Combines the moments held by the 64 lanes of a wavefront in a fixed butterfly order.  The
// pairwise update is not exactly commutative, so lanes may end a few ulps apart: lane 0's value
// is taken for all.
__device__ __forceinline__ Moments wave_merge(Moments m) {
    m = merge_with(m, [](float v) { return dppf<0xB1>(v); });
    m = merge_with(m, [](float v) { return dppf<0x4E>(v); });
    m = merge_with(m, [](float v) { return dppf<0x141>(v); });
    m = merge_with(m, [](float v) { return dppf<0x140>(v); });
    m = merge_with(m, [](float v) { return swz16(v); });
    const Moments lo{lane_bcast(m.n, 0), lane_bcast(m.mean, 0), lane_bcast(m.m2, 0)};
    const Moments hi{lane_bcast(m.n, 32), lane_bcast(m.mean, 32), lane_bcast(m.m2, 32)};
    return merge(lo, hi);
}

struct Chunk {
    float x[kVecPerThread][8];
    int cnt;  // valid elements held by this lane
};

template <bool ALIGNED>
__device__ __forceinline__ void load_chunk(const half_t* __restrict__ g, int64_t base, int64_t size, Chunk& c) {
    c.cnt = 0;
#pragma unroll
    for (int j = 0; j < kVecPerThread; j++) {
        const int64_t e0 = base + (int64_t)(j * kThreads + threadIdx.x) * 8;
        if (ALIGNED && e0 + 8 <= size) {
            const u32x4 q = *reinterpret_cast<const u32x4*>(g + e0);
            const half_t* p = reinterpret_cast<const half_t*>(&q);
#pragma unroll
            for (int k = 0; k < 8; k++) c.x[j][k] = (float)p[k];
            c.cnt += 8;
        } else {
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const bool ok = e0 + k < size;
                c.x[j][k] = ok ? (float)g[ok ? e0 + k : 0] : 0.f;
                c.cnt += ok ? 1 : 0;
            }
        }
    }
}

// Chunk statistics.  Each wavefront finds the mean and centred sum of squares of its own 1024
// elements with lane shuffles only; the four results meet in local memory once and every lane
// merges them in the same order.  Padded slots hold 0 and are excluded through the counts.
__device__ __forceinline__ Moments chunk_moments(const Chunk& c, int64_t base, int64_t size, Moments* smem) {
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < kVecPerThread; j++)
#pragma unroll
        for (int k = 0; k < 8; k++) s += c.x[j][k];
    const float n = wave_sum((float)c.cnt);
    const float mean = n > 0.f ? wave_sum(s) / n : 0.f;
    float q = 0.f;
#pragma unroll
    for (int j = 0; j < kVecPerThread; j++)
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const int64_t e = base + (int64_t)(j * kThreads + threadIdx.x) * 8 + k;
            const float d = c.x[j][k] - mean;
            q += e < size ? d * d : 0.f;
        }
    q = wave_sum(q);
    if ((threadIdx.x & 63) == 0) smem[threadIdx.x >> 6] = Moments{n, mean, q};
    __syncthreads();
    return merge(merge(smem[0], smem[1]), merge(smem[2], smem[3]));
}

template <bool ALIGNED>
__device__ __forceinline__ void store_chunk(half_t* __restrict__ g, int64_t base, int64_t size, const Chunk& c,
                                            float mean, float inv) {
#pragma unroll
    for (int j = 0; j < kVecPerThread; j++) {
        const int64_t e0 = base + (int64_t)(j * kThreads + threadIdx.x) * 8;
        if (ALIGNED && e0 + 8 <= size) {
            u32x4 q;
            half_t* p = reinterpret_cast<half_t*>(&q);
#pragma unroll
            for (int k = 0; k < 8; k++) p[k] = (half_t)((c.x[j][k] - mean) * inv);
            __builtin_nontemporal_store(q, reinterpret_cast<u32x4*>(g + e0));
        } else {
#pragma unroll
            for (int k = 0; k < 8; k++)
                if (e0 + k < size) g[e0 + k] = (half_t)((c.x[j][k] - mean) * inv);
        }
    }
}

__device__ __forceinline__ float inv_std(Moments m, bool normalize_variance, float eps) {
    return normalize_variance ? 1.0f / __builtin_sqrtf(m.m2 / m.n + eps) : 1.0f;
}

// Fixed-order merge of up to 256 published partials of one group.  Every wavefront does the
// whole merge on its own (lane l folds partials l, l+64, l+128, l+192 in sequence -- a wave reads
// 64 consecutive records at a time --, then the butterfly), so all wavefronts of all workgroups get
// the same bits.  `get(i)` returns partial i.
template <class Get>
__device__ __forceinline__ Moments merge_partials(Get get, int chunks) {
    const int lane = threadIdx.x & 63;
    Moments acc{0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < kMergeInKernel / 64; k++) {
        const int i = k * 64 + lane;
        if (i < chunks) acc = merge(acc, get(i));
    }
    return wave_merge(acc);
}

// Fixed-order tree merge of one partial per lane of the workgroup; every lane returns the total.
__device__ __forceinline__ Moments block_merge(Moments m, Moments* smem) {
    __syncthreads();
    smem[threadIdx.x] = m;
    __syncthreads();
    for (int step = kThreads / 2; step > 0; step >>= 1) {
        if ((int)threadIdx.x < step) smem[threadIdx.x] = merge(smem[threadIdx.x], smem[threadIdx.x + step]);
        __syncthreads();
    }
    return smem[0];
}

// One workgroup per (group, chunk).  MODE 0: the group is a single chunk, normalise at once.
// MODE 1: publish the chunk's moments.  MODE 2: merge the group's published moments (all of them
// when `merged` is null, else read the finished result) and normalise.
template <int MODE, bool ALIGNED>
__global__ __launch_bounds__(kThreads) void mvn_chunk_kernel(const half_t* __restrict__ in, half_t* __restrict__ out,
                                                             int64_t group_size, int chunks, Record* partial,
                                                             const Record* merged, int normalize_variance, float eps) {
    __shared__ Moments red[4];
    const int64_t group = blockIdx.x / chunks;
    const int chunk = blockIdx.x % chunks;
    const int64_t base = (int64_t)chunk * kChunk;
    const half_t* gin = in + group * group_size;
    Chunk c;
    load_chunk<ALIGNED>(gin, base, group_size, c);
    if (MODE == 0) {
        const Moments m = chunk_moments(c, base, group_size, red);
        store_chunk<ALIGNED>(out + group * group_size, base, group_size, c, m.mean, inv_std(m, normalize_variance, eps));
    } else if (MODE == 1) {
        const Moments m = chunk_moments(c, base, group_size, red);
        if (threadIdx.x == 0) partial[blockIdx.x] = Record{m.n, m.mean, m.m2, 0.f};
    } else {
        const Record* mine = partial + group * chunks;
        const Moments total = merged ? unpack(merged[group]) : merge_partials([&](int i) { return unpack(mine[i]); }, chunks);
        store_chunk<ALIGNED>(out + group * group_size, base, group_size, c, total.mean,
                             inv_std(total, normalize_variance, eps));
    }
}

// Groups with more than kMergeInKernel chunks: one workgroup per group folds its partials.
__global__ __launch_bounds__(kThreads) void mvn_merge_kernel(const Record* partial, Record* merged, int chunks) {
    __shared__ Moments tree[kThreads];
    const int64_t group = blockIdx.x;
    Moments acc{0.f, 0.f, 0.f};
    // lane t folds chunks t, t+256, ... in order, then the lanes are merged by the fixed tree
    for (int c = threadIdx.x; c < chunks; c += kThreads) acc = merge(acc, unpack(partial[group * chunks + c]));
    const Moments total = block_merge(acc, tree);
    if (threadIdx.x == 0) merged[group] = Record{total.n, total.mean, total.m2, 0.f};
}

// Many short groups that follow one another in memory (per-channel statistics of small planes, 15 x 15 or 7 x 7; rows
// of a few hundred values): a workgroup takes a run of whole groups of at most kSmallChunk values, moves it between
// global memory and LDS in aligned 128-bit words whatever the group length (the values of neighbouring groups that
// share its first and last word are read too, but never written), and half-wavefronts normalise one group each in LDS:
// sum, centred sum of squares, scale -- three passes over at most 512 values.
constexpr int kSmallChunk = 4096;   // values per workgroup, at most
__device__ __forceinline__ float half_wave_sum(float v) {
    v += dppf<0xB1>(v);
    v += dppf<0x4E>(v);
    v += dppf<0x141>(v);
    v += dppf<0x140>(v);
    return v + swz16(v);
}
template <int K>  // values per lane: a group has at most 32 K
__global__ __launch_bounds__(kThreads) void mvn_small_groups_kernel(const half_t* __restrict__ in, half_t* __restrict__ out,
                                                                    int64_t groups, int len, int per_wg, int normalize_variance,
                                                                    int eps_mode, float eps) {
    __shared__ __attribute__((aligned(16))) half_t buf[kSmallChunk + 16];
    const int64_t g0 = (int64_t)blockIdx.x * per_wg;
    const int ng = groups - g0 < per_wg ? (int)(groups - g0) : per_wg;
    const int64_t e0 = g0 * len, e1 = e0 + (int64_t)ng * len, total = groups * len;
    const int64_t a0 = e0 & ~7ll;                  // first aligned word that holds a value of the run
    const int words = (int)((e1 - a0 + 7) >> 3);
    for (int w = threadIdx.x; w < words; w += kThreads) {
        const int64_t at = a0 + (int64_t)w * 8;
        if (at + 8 <= total) {
            *reinterpret_cast<u32x4*>(buf + w * 8) = *reinterpret_cast<const u32x4*>(in + at);
        } else {
            for (int k = 0; k < 8; k++) buf[w * 8 + k] = at + k < total ? in[at + k] : (half_t)0.f;
        }
    }
    __syncthreads();
    const int lane = threadIdx.x & 31, team = threadIdx.x >> 5;
    const float n = (float)len;
    for (int g = team; g < ng; g += kThreads / 32) {   // uniform per half-wavefront
        half_t* x = buf + (int)(e0 - a0) + g * len;
        float v[K];  // the lane's values stay in registers between the passes
        float sum = 0.f;
#pragma unroll
        for (int k = 0; k < K; k++) {
            const int i = lane + 32 * k;
            v[k] = i < len ? (float)x[i] : 0.f;
            sum += v[k];
        }
        const float mean = half_wave_sum(sum) / n;
        float q = 0.f;
#pragma unroll
        for (int k = 0; k < K; k++) {
            const float d = v[k] - mean;
            q += lane + 32 * k < len ? d * d : 0.f;
        }
        const float inv = !normalize_variance ? 1.0f
                          : (eps_mode == 0 ? 1.0f / __builtin_sqrtf(half_wave_sum(q) / n + eps) : 1.0f / (__builtin_sqrtf(half_wave_sum(q) / n) + eps));
#pragma unroll
        for (int k = 0; k < K; k++) {
            const int i = lane + 32 * k;
            if (i < len) x[i] = (half_t)((v[k] - mean) * inv);
        }
    }
    __syncthreads();
    for (int w = threadIdx.x; w < words; w += kThreads) {
        const int64_t at = a0 + (int64_t)w * 8;
        if (at >= e0 && at + 8 <= e1) {
            __builtin_nontemporal_store(*reinterpret_cast<const u32x4*>(buf + w * 8), reinterpret_cast<u32x4*>(out + at));
        } else {
            for (int k = 0; k < 8; k++)
                if (at + k >= e0 && at + k < e1) out[at + k] = buf[w * 8 + k];
        }
    }
}

// Groups of a few thousand to some 75 000 values (112 x 112 or 224 x 224 planes), many of them: one workgroup of
// 1024 lanes keeps its whole group in LDS, so the tensor is read once and written once where the chunked form reads
// it twice.  Sum on the way in, centred sum of squares and the scaled values from LDS.  Groups of any length at any
// address: whole words at 2-byte alignment, the last few values one per lane (two launches with an element per access took
// 47.9 us for 384 groups of 33233, 25.5 MB).
// Between 17 groups (fewer share the chip's workgroups) and 128 it pays while one compute unit moves a group faster than
// the chip launches twice.
constexpr int kFusedMaxGroups = 16;  // groups that several workgroups share in one launch (see there)
constexpr int kLdsGroupMax = 76800;  // values: 150 KiB of the 160 KiB a compute unit has
__global__ __launch_bounds__(1024) void mvn_lds_group_kernel(const half_t* __restrict__ in, half_t* __restrict__ out, int64_t len,
                                                             int normalize_variance, int eps_mode, float eps) {
    extern __shared__ __attribute__((aligned(16))) u32x4 grp[];
    __shared__ float red[16];
    const half_t* px = in + (int64_t)blockIdx.x * len;
    half_t* py = out + (int64_t)blockIdx.x * len;
    const int nvec = (int)(len / 8), rem = (int)(len % 8), lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    auto block_sum = [&](float v) {
        v = wave_sum(v);
        __syncthreads();
        if (lane == 0) red[wave] = v;
        __syncthreads();
        float t = 0.f;
#pragma unroll
        for (int w = 0; w < 16; w++) t += red[w];
        return t;
    };
    float sum = 0.f;
    const float last = (int)threadIdx.x < rem ? (float)px[nvec * 8 + threadIdx.x] : 0.f;  // of the partial word
    for (int v = threadIdx.x; v < nvec; v += 1024) {
        const u32x4 q = reinterpret_cast<const u32x4_any*>(px)[v];
        grp[v] = q;
        const half_t* h = reinterpret_cast<const half_t*>(&q);
#pragma unroll
        for (int k = 0; k < 8; k++) sum += (float)h[k];
    }
    const float n = (float)len;
    const float mean = block_sum(sum + last) / n;
    float sq = (int)threadIdx.x < rem ? (last - mean) * (last - mean) : 0.f;
    for (int v = threadIdx.x; v < nvec; v += 1024) {
        const u32x4 q = grp[v];
        const half_t* h = reinterpret_cast<const half_t*>(&q);
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const float d = (float)h[k] - mean;
            sq += d * d;
        }
    }
    const float var = block_sum(sq) / n;
    const float inv = !normalize_variance ? 1.0f : (eps_mode == 0 ? 1.0f / __builtin_sqrtf(var + eps) : 1.0f / (__builtin_sqrtf(var) + eps));
    for (int v = threadIdx.x; v < nvec; v += 1024) {
        const u32x4 q = grp[v];
        const half_t* h = reinterpret_cast<const half_t*>(&q);
        u32x4 o;
        half_t* ho = reinterpret_cast<half_t*>(&o);
#pragma unroll
        for (int k = 0; k < 8; k++) ho[k] = (half_t)(((float)h[k] - mean) * inv);
        __builtin_nontemporal_store(o, reinterpret_cast<u32x4_any*>(py) + v);
    }
    if ((int)threadIdx.x < rem) py[nvec * 8 + threadIdx.x] = (half_t)((last - mean) * inv);
}
static bool lds_groups_ok(int64_t groups, int64_t len) {
    return len > kChunk && len <= kLdsGroupMax && (groups >= 128 || (groups > kFusedMaxGroups && len <= 40000)) && groups < (1ll << 31);
}
static int launch_lds_groups(const half_t* in, half_t* out, int64_t groups, int64_t len, int nv, int eps_mode, float eps, hipStream_t s) {
    const size_t lds = (size_t)(len / 8) * 16;
    // more than 64 KiB of dynamic LDS is an opt-in per device and function; asking again costs little
    VPX_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(mvn_lds_group_kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                      kLdsGroupMax * (int)sizeof(half_t)));
    VPX_LAUNCH(mvn_lds_group_kernel, dim3((unsigned)groups), dim3(1024), lds, s, in, out, len, nv, eps_mode, eps);
    return VPX_RESULT_SUCCESS;
}

// Packed, aligned groups of 8, 16, ... 256 values (a power of two): T = len / 8 adjacent lanes hold a group, one
// 128-bit word each, and its sums cross the T lanes by DPP (one 16-lane swap for T = 32).
template <int T>
__global__ __launch_bounds__(kThreads) void mvn_tiny_groups_kernel(const half_t* __restrict__ in, half_t* __restrict__ out, int64_t n_vec,
                                                                   int normalize_variance, int eps_mode, float eps) {
    const int64_t v = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (v >= n_vec) return;  // n_vec is a multiple of T and so is the workgroup: a group's lanes leave together
    const u32x4 q = reinterpret_cast<const u32x4*>(in)[v];
    const half_t* h = reinterpret_cast<const half_t*>(&q);
    auto across = [](float a) {
        if (T >= 2) a += dppf<0xB1>(a);
        if (T >= 4) a += dppf<0x4E>(a);
        if (T >= 8) a += dppf<0x141>(a);
        if (T >= 16) a += dppf<0x140>(a);
        if (T >= 32) a += swz16(a);
        return a;
    };
    float x[8];
    float sum = 0.f;
#pragma unroll
    for (int k = 0; k < 8; k++) {
        x[k] = (float)h[k];
        sum += x[k];
    }
    constexpr float n = (float)(8 * T);
    const float mean = across(sum) / n;
    float sq = 0.f;
#pragma unroll
    for (int k = 0; k < 8; k++) {
        x[k] -= mean;
        sq += x[k] * x[k];
    }
    const float var = across(sq) / n;
    const float inv = !normalize_variance ? 1.0f : (eps_mode == 0 ? 1.0f / __builtin_sqrtf(var + eps) : 1.0f / (__builtin_sqrtf(var) + eps));
    u32x4 o;
    half_t* ho = reinterpret_cast<half_t*>(&o);
#pragma unroll
    for (int k = 0; k < 8; k++) ho[k] = (half_t)(x[k] * inv);
    __builtin_nontemporal_store(o, reinterpret_cast<u32x4*>(out) + v);
}
static bool tiny_groups_ok(const half_t* in, const half_t* out, int64_t groups, int64_t len) {
    return (len == 8 || len == 16 || len == 32 || len == 64 || len == 128 || len == 256) && groups * (len / 8) < (1ll << 39) &&
           ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) & 15) == 0;
}
static int launch_tiny_groups(const half_t* in, half_t* out, int64_t groups, int64_t len, int nv, int eps_mode, float eps, hipStream_t s) {
    const int64_t n_vec = groups * (len / 8);
    const dim3 grid((unsigned)((n_vec + kThreads - 1) / kThreads));
#define VPX_TINY(T) VPX_LAUNCH(mvn_tiny_groups_kernel<T>, grid, dim3(kThreads), 0, s, in, out, n_vec, nv, eps_mode, eps)
    if (len == 8) VPX_TINY(1);
    else if (len == 16) VPX_TINY(2);
    else if (len == 32) VPX_TINY(4);
    else if (len == 64) VPX_TINY(8);
    else if (len == 128) VPX_TINY(16);
    else VPX_TINY(32);
#undef VPX_TINY
    return VPX_RESULT_SUCCESS;
}

// Groups a workgroup takes: what its eight half-wavefronts walk one after another.  As many as fill kSmallChunk, 37 of 110 values, left a small
// tensor to a few workgroups with a long walk each and a large one waiting for it too (us, that many / these): [512 x 7] 24.6 / 3.3,
// [16384 x 21] 12.9 / 4.4, [65536 x 110] 12.1 / 9.6, [65536 x 361] 22.8 / 19.7, [131072 x 49] 16.5 / 12.6.  Sixteen in place of eight where groups of up to 256
// values are many: eight / these [308452 x 130] 41.2 / 36.3, [237176 x 217] 37.1 / 32.8, [176306 x 166] 25.7 / 23.6.
static int small_groups_run(int64_t groups, int64_t len) {
    const int64_t fits = kSmallChunk / len, most = len <= 64 ? (groups < 16384 ? 8 : 32) : len > 128 ? (len <= 256 && groups >= (1 << 17) ? 16 : 8) : groups < (1 << 18) ? 16 : fits;
    return (int)(fits < most || groups / most >= (1 << 24) - 1 ? fits : most);  // (a launch holds fewer than 2^32 lanes)
}
// Whether the short-group form applies, and its launch.  It serves what the registers of mvn6_rows_kernel do not, groups of fewer than eight
// values, and many groups of up to 512 that are no whole number of words: a row of those leaves most of a team's lanes idle or ends in a word that
// two lanes take.  us in a HIP graph, that kernel / this one: [448 x 110] 3.2 / 3.3, [1024 x 390] 3.3 / 4.2, [8192 x 361] 5.85 / 5.83,
// [65536 x 110] 12.3 / 9.6, [131072 x 390] 25.6 / 20.6 a half of them, [131072 x 49] 20.0 / 12.6; but [16384 x 675] 11.6 / 13.7, [16384 x 784] 10.1 / 14.2.
// Of whole words it serves up to twelve, which leave two thirds of that kernel's lanes idle, where they are so many that memory does not hide it:
// [315392 x 24] 25.7 / 20.0, [1056847 x 24] 83.8 / 60.1, [494619 x 56] 41.2 / 32.4, [648482 x 72] 53.9 / 48.5, [403511 x 96] 35.7 / 33.5; even at 2^18.
static bool small_groups_ok(const half_t* in, const half_t* out, int64_t groups, int64_t len) {
    const int64_t run = len >= 1 ? small_groups_run(groups, len) : 1;
    return len >= 1 && groups >= 64 && (len < 8 || (groups > 8192 && len <= 512 && len % 8 != 0) || (groups >= (1 << 18) && len <= 96)) &&
           ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) & 15) == 0 && (groups + run - 1) / run < (1ll << 31);
}
static int launch_small_groups(const half_t* in, half_t* out, int64_t groups, int64_t len, int nv, int eps_mode, float eps, hipStream_t s) {
    const int per_wg = small_groups_run(groups, len);
    const unsigned blocks = (unsigned)((groups + per_wg - 1) / per_wg);
#define VPX_SMALL(K) VPX_LAUNCH(mvn_small_groups_kernel<K>, dim3(blocks), dim3(kThreads), 0, s, in, out, groups, (int)len, per_wg, nv, eps_mode, eps)
    if (len <= 64) VPX_SMALL(2);
    else if (len <= 128) VPX_SMALL(4);
    else if (len <= 256) VPX_SMALL(8);
    else VPX_SMALL(16);
#undef VPX_SMALL
    return VPX_RESULT_SUCCESS;
}

// position (counted from the innermost memory dimension) of logical dimension `logical`
int mem_pos_of(uint64_t order, int nd, int logical) {
    for (int i = 0; i < nd; i++)
        if ((int)((order >> (4 * i)) & 0xf) == logical + 1) return nd - 1 - i;
    return -1;
}

// ------------------------------------------------------------------------------------------------
// A few long groups in ONE launch, the tensor read once: as many workgroups as the device has compute units, each
// keeps a slice of one group in registers and publishes the slice's {mean, M2}, each word tagged, with write-through
// stores; the first wavefront then polls the records of ITS group (not of the whole grid) with loads that bypass the
// caches until every tag names this launch, merges them in a fixed order and hands the result to the other wavefronts,
// which normalise the slice from the registers.  No read-modify-write is involved: arrivals do not queue at a counter.
// The tag is the launch count + 1.  Every workgroup has counts of its own in the zero-initialised sync area (the group's kMergeInKernel
// are dealt out in turn, and a launch moves all of them on, however many workgroups it has): nobody else writes them during a
// launch, so a workgroup finds the launch's tag however late it starts, and no record of an earlier launch carries it.
// The wait is bounded: a workgroup that does not see its group complete in time (the others are not resident: the device is
// shared) computes missing slices with the same arithmetic and publishes them for their owners and for everyone else, one
// at a time, each time one that nobody has published yet.  So the result is the same bits, the missing slices are computed
// about once among those that wait, whoever starts later finds the group complete, and every wave exits: a workgroup
// computes a slice at most once.  (Each computing all slices for itself took 29 ms for 52 M values beside a launch that held
// 224 of 256 compute units, eight rounds of workgroups that wait and read the tensor 32 times; now 0.9: the wait, 0.1 for the missing slices, eight rounds.)
// What bounds a small tensor is the chain of trips to memory: arguments, slice, tag, publication, the others' records; in between nothing waits for a
// division by a count that was known before, and moments meet all at once.  us in a HIP graph, with the tag in front of the slice, records
// polled a round of 64 at a time and pairwise merges / now: [1,128,57,73] 7.1 / 5.6, [1,16,142,176] 6.6 / 5.1, [4,256,64,64] among other calls 6.5 / 6.0.
constexpr int kFusedMaxVec = 52;           // 128-bit words per lane of 512, 208 of its 256 registers: the chip holds 54 M values
constexpr int kSyncStride = 4;             // words between launch counts
// kFusedMaxGroups groups at most: each owns a fixed run of kMergeInKernel launch counts and as many record slots
constexpr size_t kSyncRecords = sizeof(unsigned) * kSyncStride * kFusedMaxGroups * kMergeInKernel;  // byte offset of the records
static_assert(kSyncRecords + sizeof(Record) * kFusedMaxGroups * kMergeInKernel <= kSyncCminor, "sync area layout");

// A published slice: two 64-bit words, {mean, tag} and {M2, tag}, each written and read as one access that goes
// through to memory (agent scope), so neither needs the other to be valid; the count of a slice follows from its index.
struct __attribute__((aligned(16))) Tagged {
    unsigned long long mean, m2;
};
__device__ __forceinline__ unsigned long long tagged(float v, unsigned tag) {
    return (unsigned long long)__builtin_bit_cast(unsigned, v) | ((unsigned long long)tag << 32);
}

// A slice in registers: V words of 128 bits for each of T lanes, plus the group's last few values, one per lane, where the
// group is no whole number of words (groups of any length at any address).
// Slices for 512 lanes are summed while they arrive, kFusedAhead words a lane under way at a time: all at once, up to 400 KB a compute unit,
// they reach the memory in an order that costs a third of its rate.
constexpr int kFusedAhead = 12;
template <int V>
struct Slice {
    u32x4 q[V];
    int have;    // words of this lane
    float last;  // its value of the partial word
    bool has_last;
    float wave_count, count;  // values of the wavefront, of the slice
    const half_t* from;       // of the word to load next: the group's values, and its place among them
    uint32_t at;
};

template <int V, int T>
__device__ __forceinline__ void load_word(Slice<V>& sl, int j) {
    sl.q[j] = *reinterpret_cast<const u32x4_any*>(sl.from + (j < sl.have ? sl.at : 0));
    sl.at += T * 8;
    asm volatile("" : "+v"(sl.at));  // one running offset, not V of them
}
template <int V, int T>
__device__ __forceinline__ void load_slice(const half_t* __restrict__ g, uint32_t base, uint32_t end, uint32_t group_size, Slice<V>& sl) {
    const uint32_t words = (end - base) / 8;  // (only the group's last slice is not whole words)
    sl.have = threadIdx.x < words ? (int)((words - threadIdx.x + T - 1) / T) : 0;
    sl.from = g;
    sl.at = base + threadIdx.x * 8;
#pragma unroll
    for (int j = 0; j < (V <= kFusedAhead ? V : kFusedAhead); j++) load_word<V, T>(sl, j);
    if (T < 512) {
#pragma unroll
        for (int j = 0; j < V; j++) sl.q[j] = j < sl.have ? sl.q[j] : u32x4{0, 0, 0, 0};
    }
    const uint32_t rest = base + words * 8 + threadIdx.x;
    sl.has_last = rest < end && threadIdx.x < 8;
    sl.last = sl.has_last ? (float)g[rest] : 0.f;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), more = (int)(words % T) - 64 * wave;
    sl.count = (float)(end - base);
    sl.wave_count = (float)(8 * (64 * (int)(words / T) + (more < 0 ? 0 : more < 64 ? more : 64)) + (wave == 0 ? (int)(end - base - words * 8) : 0));
}

// The eight values of a word in single precision (the conversion is exact).  KEEP: both passes of the moments and the
// normalisation share one conversion; else, with many words, the asm keeps the compiler from holding converted values.
template <bool KEEP>
__device__ __forceinline__ void widen_word(u32x4& q, float (&f)[8]) {
    if (!KEEP) asm volatile("" : "+v"(q));
    const halfx8 h = __builtin_bit_cast(halfx8, q);
#pragma unroll
    for (int k = 0; k < 8; k++) f[k] = (float)h[k];
}

// Moments of the slice held by the workgroup: per wavefront by lane shuffles, the wavefronts' results met by every lane.
// Long slices (T == 512): one pass while the words arrive, over values less the mean of the wavefront's first kFirst words.  That is rounded to
// half precision, so that a difference is exact and the sum of differences as good as one of the values, whose grid they are on.  Where the first
// words say little about the others the squares about their mean are up to V / kFirst = 13 times those about the mean, and so is what
// rounding does to them: from an eighth of them on the wavefront sums the squares again, about the mean, from its registers.  Relative errors of the
// variance against 64 bits (worst of 16 tensors of eight slices, the kernel's arithmetic on a host), two passes / this: values of one distribution 1.8e-7 /
// 1.0e-7, the mean 40 deviations away 1.5e-7 / 1.2e-7, constant first words at another level 2.0e-6 / 1.8e-6 (8.0e-6 without the second sum).  us
// across channels, all words at once and two passes behind the last one / this, where the second sum is not taken / where every wavefront takes it:
// [3,128,124,88] 9.2 / 7.7 / 8.3, [2,202,224,80] 9.9 / 8.5 / 9.3, [1,368,182,224] 16.0 / 14.8 / 15.9, [2,181,194,308] 23.5 / 21.3 / 23.2,
// [2,452,175,218] 34.1 / 29.0 / 31.9, [5,146,180,352] 50.6 / 39.7 / 44.3.  With 256 lanes, whose words
// arrive together, the second pass is shorter than what this adds in front of it: [1,176,113,145] 7.0 / 7.6.
template <int V, int T>
__device__ __forceinline__ Moments slice_moments(Slice<V>& sl, Moments* red) {
    constexpr int kFirst = V > 8 ? 4 : 1;
    const float n = sl.wave_count, inv_n = 1.f / n;  // (of loads that are still on their way)
    float mean, q;
    if constexpr (T == 512) {
        float shift = 0.f;
        int firsts = sl.have < kFirst ? sl.have : kFirst;
#pragma unroll
        for (int j = 0; j < kFirst; j++) {
            float f[8], sum = 0.f;
            widen_word<false>(sl.q[j], f);
#pragma unroll
            for (int k = 0; k < 8; k++) sum += f[k];
            shift += j < sl.have ? sum : 0.f;
        }
        const float of = wave_sum_soon((float)(8 * firsts));
        shift = wave_sum_soon(shift);
        shift = of > 0.f ? (float)(half_t)(shift / of) : 0.f;
        float sum = sl.has_last ? sl.last - shift : 0.f;
        q = sum * sum;
#pragma unroll
        for (int j = 0; j < V; j++) {
            // word after word: the values of V words at once are more than the registers hold
            asm volatile("" : "+v"(sl.q[j]), "+v"(sum), "+v"(q));
            if (j + kFusedAhead < V) load_word<V, T>(sl, j + kFusedAhead);
            float f[8], sj = 0.f, qj = 0.f;
            widen_word<false>(sl.q[j], f);
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const float d = f[k] - shift;
                sj += d;
                qj = __builtin_fmaf(d, d, qj);
            }
            sum += j < sl.have ? sj : 0.f;
            q += j < sl.have ? qj : 0.f;
        }
        sum = wave_sum_soon(sum);
        const float off = n > 0.f ? over(sum, n, inv_n) : 0.f;
        mean = shift + off;
        q = wave_sum_soon(q);
        if (sum * off > 0.125f * q) {  // (the same for the wavefront)
            q = sl.has_last ? (sl.last - mean) * (sl.last - mean) : 0.f;
#pragma unroll
            for (int j = 0; j < V; j++) {
                asm volatile("" : "+v"(sl.q[j]), "+v"(q));
                float f[8], qj = 0.f;
                widen_word<false>(sl.q[j], f);
#pragma unroll
                for (int k = 0; k < 8; k++) {
                    const float d = f[k] - mean;
                    qj = __builtin_fmaf(d, d, qj);
                }
                q += j < sl.have ? qj : 0.f;
            }
            q = wave_sum_soon(q);
        } else {
            q -= sum * off;
        }
    } else {
        float sum = sl.last;
#pragma unroll
        for (int j = 0; j < V; j++) {
            float f[8];
            widen_word<true>(sl.q[j], f);
#pragma unroll
            for (int k = 0; k < 8; k++) sum += f[k];
        }
        mean = n > 0.f ? over(wave_sum_soon(sum), n, inv_n) : 0.f;
        q = sl.has_last ? (sl.last - mean) * (sl.last - mean) : 0.f;
#pragma unroll
        for (int j = 0; j < V; j++) {
            float f[8], qj = 0.f;
            widen_word<true>(sl.q[j], f);
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const float d = f[k] - mean;
                qj += d * d;
            }
            q += j < sl.have ? qj : 0.f;
        }
        q = wave_sum_soon(q);
    }
    __syncthreads();  // the previous use of `red` is over
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = Moments{n, mean, q};
    __syncthreads();
    // all at once (a tree of pairwise merges is three reciprocals in a row), about their mean, which the distances to it then correct by what was rounded off
    Moments w[T / 64];
#pragma unroll
    for (int k = 0; k < T / 64; k++) w[k] = red[k];
    const float count = sl.count, inv_count = 1.f / count;
    float all = 0.f, rest = 0.f, m2 = 0.f;
#pragma unroll
    for (int k = 0; k < T / 64; k++) all += w[k].n * w[k].mean;
    mean = over(all, count, inv_count);
#pragma unroll
    for (int k = 0; k < T / 64; k++) {
        const float d = w[k].mean - mean;
        rest += w[k].n * d;
        m2 += w[k].m2 + w[k].n * d * d;
    }
    return Moments{count, mean + over(rest, count, inv_count), m2};
}

template <int V, int T>
__global__ __launch_bounds__(T) void mvn_fused_kernel(const half_t* __restrict__ in, half_t* __restrict__ out,
                                                      uint32_t group_size, int wpg, uint32_t slice, unsigned* sync,
                                                      int normalize_variance, float eps, unsigned long long spin_ticks) {
    __shared__ Moments red[8];
    __shared__ Moments shared_total;
    __shared__ int complete, pick;
    __shared__ unsigned char helped[kMergeInKernel];
    const int64_t group = blockIdx.y;
    const int part = (int)blockIdx.x;
    const int lane = threadIdx.x & 63;
    // this workgroup's launch counts: every wpg-th of the group's, from its own place on
    unsigned* counts = sync + group * (kMergeInKernel * kSyncStride);
    Tagged* records = reinterpret_cast<Tagged*>(reinterpret_cast<char*>(sync) + kSyncRecords) + group * kMergeInKernel;
    const half_t* gin = in + group * group_size;
    const uint32_t base = (uint32_t)part * slice;
    const uint32_t end = part + 1 < wpg ? base + slice : group_size;
    Slice<V> sl;
    load_slice<V, T>(gin, base, end, group_size, sl);
    // The launch's tag, asked for behind the slice: loads return in order, and this one goes through to memory.  (In front of them, in a branch that
    // works with it at once or moved to a scalar register as uniform, every launch paid its way, 0.6 of 6.7 us at [3,48,76,60].)
    int here = 0;
    asm("" : "+v"(here));
    const unsigned counted = __hip_atomic_load(counts + part * kSyncStride + here, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const float group_count = (float)group_size, inv_count = 1.f / group_count;
    Moments total = slice_moments<V, T>(sl, red);
    if (wpg > 1) {
        const unsigned tag = counted + 1u == 0u ? 1u : counted + 1u;
        const auto publish = [&](int p, const Moments& m) {  // by one lane of the first wavefront
            __hip_atomic_store(&records[p].mean, tagged(m.mean, tag), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&records[p].m2, tagged(m.m2, tag), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        };
        unsigned long long rm[kMergeInKernel / 64], rq[kMergeInKernel / 64];
        const auto poll = [&](int k) {  // record k * 64 + lane; true if it is this launch's, or none
            const int i = k * 64 + lane;
            rm[k] = rq[k] = 0;
            if (i >= wpg) return true;
            rm[k] = __hip_atomic_load(&records[i].mean, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            rq[k] = __hip_atomic_load(&records[i].m2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return (unsigned)(rm[k] >> 32) == tag && (unsigned)(rq[k] >> 32) == tag;
        };
        const auto collect = [&](bool waits) {  // the first wavefront: reads the group's records and merges them
            const unsigned long long t0 = wall_clock64();
            bool ok;
            // (records asked for together, places past the last one reading that again: a branch around each round waits for it)
            const auto poll_rounds = [&](auto rounds_c) {
                constexpr int ROUNDS = decltype(rounds_c)::value;
#pragma unroll
                for (int k = 0; k < ROUNDS; k++) {
                    const Tagged* r = &records[k * 64 + lane < wpg ? k * 64 + lane : wpg - 1];
                    rm[k] = __hip_atomic_load(&r->mean, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    rq[k] = __hip_atomic_load(&r->m2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
                bool ready = true;
#pragma unroll
                for (int k = 0; k < ROUNDS; k++) ready &= (unsigned)(rm[k] >> 32) == tag && (unsigned)(rq[k] >> 32) == tag;
                return __builtin_amdgcn_ballot_w64(!ready) == 0;
            };
            constexpr int kRounds = kMergeInKernel / 64;
            for (;;) {
                if (wpg <= 64) ok = poll_rounds(std::integral_constant<int, 1>{});
                else if (wpg <= 128) ok = poll_rounds(std::integral_constant<int, 2>{});
                else ok = poll_rounds(std::integral_constant<int, kRounds>{});
                if (ok || !waits || wall_clock64() - t0 >= spin_ticks) break;  // (pausing between polls measured slower)
            }
            if (ok || !waits) {
                // All at once, about the first slice's mean, in a fixed order (a butterfly of pairwise merges: six reciprocals in a row).  Where that lies
                // further than a deviation from the whole's, about the latter, which the distances to it correct by what was rounded off (for
                // every launch: 0.1 us).
                const auto value = [&](int k) { return __builtin_bit_cast(float, (unsigned)rm[k]); };
                const float first = lane_bcast(value(0), 0);
                float shift = 0.f, m2 = 0.f;
                const auto count = [&](int i) { return i >= wpg ? 0.f : i + 1 < wpg ? (float)slice : (float)(group_size - (uint32_t)i * slice); };
                const auto off = [&](int k, float from) { return k * 64 + lane < wpg ? value(k) - from : 0.f; };
                const auto squares = [&](int k, float d) { return k * 64 + lane < wpg ? __builtin_bit_cast(float, (unsigned)rq[k]) + count(k * 64 + lane) * d * d : 0.f; };
#pragma unroll
                for (int k = 0; k < kMergeInKernel / 64; k++) shift += count(k * 64 + lane) * off(k, first);
                shift = over(wave_sum_soon(shift), group_count, inv_count);
#pragma unroll
                for (int k = 0; k < kMergeInKernel / 64; k++) m2 += squares(k, off(k, first) - shift);
                m2 = wave_sum_soon(m2);
                float mean = first + shift;
                if (shift * shift * group_count > m2) {  // (the same for the wavefront)
                    float rest = 0.f;
                    m2 = 0.f;
#pragma unroll
                    for (int k = 0; k < kMergeInKernel / 64; k++) {
                        const float d = off(k, mean);
                        rest += count(k * 64 + lane) * d;
                        m2 += squares(k, d);
                    }
                    m2 = wave_sum_soon(m2);
                    mean += over(wave_sum_soon(rest), group_count, inv_count);
                }
                if (lane == 0) shared_total = Moments{group_count, mean, m2};
            }
            return ok;
        };
        if (threadIdx.x < 64) {
            if (lane == 0) publish(part, total);
            // (here and not behind the meeting: their way to memory then ends under the wait, 0.2 of 8.3 us at [4,256,64,64])
            for (int i = part + lane * wpg; i < kMergeInKernel; i += 64 * wpg)
                __hip_atomic_store(counts + i * kSyncStride, tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const bool ok = collect(true);
            if (lane == 0) complete = ok ? 1 : 0;
        }
        __syncthreads();
        if (!complete) {
            for (int i = threadIdx.x; i < wpg; i += T) helped[i] = 0;
            __syncthreads();
            for (int n = 0; n < wpg; n++) {
                if (threadIdx.x < 64) {
                    // of the slices that nobody has published: the one at this workgroup's place among them
                    unsigned long long missing[kMergeInKernel / 64];
                    int count = 0;
#pragma unroll
                    for (int k = 0; k < kMergeInKernel / 64; k++) {
                        const bool there = poll(k) || helped[k * 64 + lane];
                        missing[k] = __builtin_amdgcn_ballot_w64(!there);
                        count += __builtin_popcountll(missing[k]);
                    }
                    int at = count ? part % count : 0, p = -1;
#pragma unroll
                    for (int k = 0; k < kMergeInKernel / 64; k++) {
                        unsigned long long m = missing[k];
                        const int c = __builtin_popcountll(m);
                        if (p < 0 && at < c) {
                            for (; at > 0; at--) m &= m - 1;
                            p = k * 64 + __builtin_ctzll(m);
                        }
                        at -= c;
                    }
                    if (lane == 0) pick = p;
                }
                __syncthreads();
                const int p = pick;
                if (p < 0) break;
                const uint32_t b = (uint32_t)p * slice;
                load_slice<V, T>(gin, b, p + 1 < wpg ? b + slice : group_size, group_size, sl);
                const Moments mp = slice_moments<V, T>(sl, red);
                if (threadIdx.x == 0) {
                    publish(p, mp);
                    __threadfence();
                    helped[p] = 1;
                }
            }
            if (threadIdx.x < 64) collect(false);
            load_slice<V, T>(gin, base, end, group_size, sl);  // its own again
            if (V > kFusedAhead) slice_moments<V, T>(sl, red);  // (which asks for the rest)
            __syncthreads();
        }
        total = shared_total;
    }
    const float mean = total.mean, inv = normalize_variance ? inv_root(over(total.m2, group_count, inv_count) + eps) : 1.0f;
    half_t* gout = out + group * group_size;
    uint32_t at = base + threadIdx.x * 8;
#pragma unroll
    for (int j = 0; j < V; j++, at += T * 8) {
        float f[8];
        widen_word<V <= 8>(sl.q[j], f);
        asm volatile("" : "+v"(at));
        if (j >= sl.have) continue;
        halfx8 r;
#pragma unroll
        for (int k = 0; k < 8; k++) r[k] = (half_t)((f[k] - mean) * inv);
        __builtin_nontemporal_store(__builtin_bit_cast(u32x4, r), reinterpret_cast<u32x4_any*>(gout + at));
    }
    if (sl.has_last) gout[group_size / 8 * 8 + threadIdx.x] = (half_t)((sl.last - mean) * inv);
}

// Takes the launch when the groups are few and the tensor fits the registers of one workgroup per compute unit.
// *done is set when the kernel was launched.
int launch_fused_groups(const half_t* in, half_t* out, int64_t groups, int64_t group_size, int nv, float eps, hipStream_t s,
                        bool* done) {
    *done = false;
    const int mode = tuning_mvn_fused();  // 0: never, 1: default, 2: spin limit 0 (a workgroup computes what it finds missing at once)
    if (mode == 0) return VPX_RESULT_SUCCESS;
    int cus = 0;
    int rc = device_compute_units(&cus);
    if (rc) return rc;
    if (groups > cus || groups > kFusedMaxGroups) return VPX_RESULT_SUCCESS;
    // In place (or any overlap of the two tensors): a workgroup whose wait runs out reads slices of others, which
    // by then may have stored their normalised values over them.  The two-launch kernels finish every
    // read of the statistics before the first store, so overlapping tensors go there.
    {
        const uintptr_t ib = reinterpret_cast<uintptr_t>(in), ob = reinterpret_cast<uintptr_t>(out);
        const uintptr_t bytes = (uintptr_t)(groups * group_size) * sizeof(half_t);
        if (ib < ob + bytes && ob < ib + bytes) return VPX_RESULT_SUCCESS;
    }
    int64_t wpg = cus / groups;  // (two workgroups per compute unit measured 1.2 us slower at [4,256,64,64])
    if (wpg > kMergeInKernel) wpg = kMergeInKernel;
    const int64_t words = group_size / 8;
    const int64_t most = (words + kThreads - 1) / kThreads;  // at least one word per lane
    if (words == 0 || group_size >= (1ll << 31)) return VPX_RESULT_SUCCESS;
    if (wpg > most) wpg = most;
    const int64_t slice = (words + wpg - 1) / wpg * 8;
    wpg = (words * 8 + slice - 1) / slice;  // no empty slices (the last one takes the partial word's values along)
    const int64_t lane_words = slice / 8;
    if (lane_words > (int64_t)kFusedMaxVec * 512) return VPX_RESULT_SUCCESS;
    void* sync = nullptr;
    rc = get_sync_area(s, &sync);
    if (rc) return rc;
    const unsigned long long spin = mode == 2 ? 0ull : 50000ull;  // 0.5 ms of the 100 MHz counter
    const dim3 grid((unsigned)wpg, (unsigned)groups);
#define VPX_FUSED(V, T)                                                                                                        \
    VPX_LAUNCH((mvn_fused_kernel<V, T>), grid, dim3(T), 0, s, in, out, (uint32_t)group_size, (int)wpg, (uint32_t)slice,         \
               (unsigned*)sync, nv, eps, spin)
    // up to eight words per lane four wavefronts do (eight measured 0.3 us slower there)
    if (lane_words <= kThreads) VPX_FUSED(1, 256);
    else if (lane_words <= 2 * kThreads) VPX_FUSED(2, 256);
    else if (lane_words <= 4 * kThreads) VPX_FUSED(4, 256);
    else if (lane_words <= 8 * kThreads) VPX_FUSED(8, 256);
    else if (lane_words <= 8 * 512) VPX_FUSED(8, 512);
    else if (lane_words <= 12 * 512) VPX_FUSED(12, 512);
    else if (lane_words <= 16 * 512) VPX_FUSED(16, 512);
    else if (lane_words <= 20 * 512) VPX_FUSED(20, 512);
    else if (lane_words <= 24 * 512) VPX_FUSED(24, 512);
    else if (lane_words <= 28 * 512) VPX_FUSED(28, 512);
    else if (lane_words <= 32 * 512) VPX_FUSED(32, 512);
    else if (lane_words <= 36 * 512) VPX_FUSED(36, 512);
    else if (lane_words <= 40 * 512) VPX_FUSED(40, 512);
    else if (lane_words <= 44 * 512) VPX_FUSED(44, 512);
    else if (lane_words <= 48 * 512) VPX_FUSED(48, 512);
    else VPX_FUSED(kFusedMaxVec, 512);
#undef VPX_FUSED
    *done = true;
    return VPX_RESULT_SUCCESS;
}

template <bool ALIGNED>
int launch_groups(const half_t* in, half_t* out, int64_t groups, int64_t group_size, int nv, float eps, hipStream_t s) {
    const int64_t chunks64 = (group_size + kChunk - 1) / kChunk;
    VPX_REQUIRE(chunks64 * groups < (1ll << 31), VPX_RESULT_ERROR_UNSUPPORTED_FEATURE,
                "mvn1: %lld groups of %lld elements exceed the launch limit", (long long)groups, (long long)group_size);
    const int chunks = (int)chunks64;
    const unsigned blocks = (unsigned)(groups * chunks);
    if (chunks > 1) {
        bool done = false;
        const int rc = launch_fused_groups(in, out, groups, group_size, nv, eps, s, &done);
        if (rc || done) return rc;
    }
    if (chunks == 1) {
        VPX_LAUNCH((mvn_chunk_kernel<0, ALIGNED>), dim3(blocks), dim3(kThreads), 0, s, in, out, group_size, 1,
                   (Record*)nullptr, (const Record*)nullptr, nv, eps);
        return VPX_RESULT_SUCCESS;
    }
    void* ws = nullptr;
    const size_t need = sizeof(Record) * ((size_t)blocks + (size_t)groups);
    int rc = get_workspace(s, need, &ws);
    if (rc) return rc;
    Record* partial = (Record*)ws;
    Record* merged = partial + blocks;

    VPX_LAUNCH((mvn_chunk_kernel<1, ALIGNED>), dim3(blocks), dim3(kThreads), 0, s, in, out, group_size, chunks,
               partial, (const Record*)nullptr, nv, eps);
    const Record* use_merged = nullptr;
    if (chunks > kMergeInKernel) {
        VPX_LAUNCH(mvn_merge_kernel, dim3((unsigned)groups), dim3(kThreads), 0, s, partial, merged, chunks);
        use_merged = merged;
    }
    VPX_LAUNCH((mvn_chunk_kernel<2, ALIGNED>), dim3(blocks), dim3(kThreads), 0, s, in, out, group_size, chunks,
               partial, use_merged, nv, eps);
    return VPX_RESULT_SUCCESS;
}


// ------------------------------------------------------------------------------------------------
// The compiler's three-step decomposition of MVN-1 for tensors that do not fit local memory
// (src/vpux_compiler/src/NPU37XX/dialect/VPU/transforms/passes/decompose_mvn.cpp:82-129;
// operator definitions src/vpux_compiler/tblgen/vpux/compiler/dialect/VPU/ops.td:3659-3845):
//   mvn1_sum      x[N,C,H,W] -> f32 {sum, sum of squares} [N, C or 1, parts, 2 or 1], channel-minor
//   mvn1_mean_var those partial sums -> {mean, 1/sqrt(var + eps)} [N, C or 1, 1, 2 or 1]
//   mvn1_norm     x, {mean, 1/std} -> (x - mean) * 1/std
// `parts` (the output height of mvn1_sum) is the number of partial sums per group; a single call
// here splits the group's elements into that many consecutive ranges, so that their sum is the
// group's total whatever the count.

// fp32 value -> fp16, round to nearest even.  The empty asm keeps the compiler from folding the preceding
// multiply into a mixed-precision multiply that rounds the exact product once: the result is defined as
// the fp32 product rounded again.
__device__ __forceinline__ half_t round_f16(float v) {
    asm volatile("" : "+v"(v));
    return (half_t)v;
}

struct SumOut {
    float* out;
    int parts, out_w;
    int64_t out_c;
    __device__ __forceinline__ void put(int64_t group, int part, float s, float q) const {
        const int64_t n = group / out_c, c = group % out_c;
        float* o = out + ((n * parts + part) * out_w) * out_c + c;
        o[0] = s;
        if (out_w == 2) o[out_c] = q;
    }
};

__device__ __forceinline__ float2 add2(float2 a, float2 b) {
    return float2{a.x + b.x, a.y + b.y};
}

// One workgroup per (group, chunk) of a contiguous group: raw fp32 sum and sum of squares.
template <bool ALIGNED>
__global__ __launch_bounds__(kThreads) void mvn_sum_chunk_kernel(const half_t* __restrict__ in, int64_t group_size,
                                                                 int chunks, float2* __restrict__ partial, SumOut o,
                                                                 int direct) {
    __shared__ float2 red[4];
    const int64_t group = blockIdx.x / chunks;
    const int chunk = blockIdx.x % chunks;
    Chunk c;
    load_chunk<ALIGNED>(in + group * group_size, (int64_t)chunk * kChunk, group_size, c);
    float sum = 0.f, sq = 0.f;
#pragma unroll
    for (int j = 0; j < kVecPerThread; j++)
#pragma unroll
        for (int k = 0; k < 8; k++) {
            sum += c.x[j][k];
            sq += c.x[j][k] * c.x[j][k];
        }
    sum = wave_sum(sum);
    sq = wave_sum(sq);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = float2{sum, sq};
    __syncthreads();
    if (threadIdx.x == 0) {
        const float2 t = add2(add2(red[0], red[1]), add2(red[2], red[3]));
        if (direct) o.put(group, 0, t.x, t.y);
        else partial[blockIdx.x] = t;
    }
}

// One workgroup per (group, part): folds that part's chunk sums in a fixed order.
__global__ __launch_bounds__(kThreads) void mvn_sum_finish_kernel(const float2* __restrict__ partial, int chunks, SumOut o) {
    __shared__ float2 tree[kThreads];
    const int64_t group = blockIdx.x / o.parts;
    const int part = blockIdx.x % o.parts;
    const int c0 = (int)((int64_t)part * chunks / o.parts), c1 = (int)((int64_t)(part + 1) * chunks / o.parts);
    float2 acc{0.f, 0.f};
    for (int c = c0 + threadIdx.x; c < c1; c += kThreads) acc = add2(acc, partial[group * chunks + c]);
    tree[threadIdx.x] = acc;
    __syncthreads();
    for (int step = kThreads / 2; step > 0; step >>= 1) {
        if ((int)threadIdx.x < step) tree[threadIdx.x] = add2(tree[threadIdx.x], tree[threadIdx.x + step]);
        __syncthreads();
    }
    if (threadIdx.x == 0) o.put(group, part, tree[0].x, tree[0].y);
}

// Per-channel sums of a channel-minor layout: a workgroup takes 64 channels of one spatial range
// of one batch element (lane (r, c) walks positions r, r+4, ...).  With SHIFT the sums are of
// x - x[first position of the channel], which keeps the sum of squares free of cancellation when a
// channel's mean is far from zero (used where the variance is taken from these sums).
template <bool SHIFT>
__global__ __launch_bounds__(kThreads) void mvn_sum_cminor_kernel(const half_t* __restrict__ in, int64_t S, int64_t C,
                                                                  int subparts, int64_t cpad, float2* __restrict__ partial) {
    __shared__ float2 red[4][64];
    const int cl = threadIdx.x & 63, r = threadIdx.x >> 6;
    const int64_t ctiles = cpad / 64;
    const int64_t ct = blockIdx.x % ctiles;
    const int sp = (int)((blockIdx.x / ctiles) % subparts);
    const int64_t n = blockIdx.x / (ctiles * subparts);
    const int64_t s0 = sp * S / subparts, s1 = (sp + 1) * S / subparts;
    const int64_t c = ct * 64 + cl;
    float sum = 0.f, sq = 0.f;
    if (c < C) {
        const half_t* px = in + n * S * C + c;
        const float shift = SHIFT ? (float)px[0] : 0.f;
        for (int64_t i = s0 + r; i < s1; i += 4) {
            const float x = (float)px[i * C] - shift;
            sum += x;
            sq += x * x;
        }
    }
    red[r][cl] = float2{sum, sq};
    __syncthreads();
    if (r == 0) partial[(n * subparts + sp) * cpad + c] = add2(add2(red[0][cl], red[1][cl]), add2(red[2][cl], red[3][cl]));
}

// The same sums with eight adjacent channels per lane (channel counts that are a multiple of eight, up to 2048): a
// lane's 128-bit loads walk the positions of its channel octet, the workgroup's lanes cover 256 / (C / 8) positions
// at a time, and the lanes that share an octet meet in LDS.  Same partial layout as the kernel above.
template <bool SHIFT>
__global__ __launch_bounds__(kThreads) void mvn_sum_cminor8_kernel(const half_t* __restrict__ in, int64_t S, int64_t C,
                                                                   int subparts, int64_t cpad, float2* __restrict__ partial) {
    extern __shared__ float2 red8[];  // [slots][C]
    const int cv = (int)(C / 8), slots = kThreads / cv;
    const int sp = (int)(blockIdx.x % subparts);
    const int64_t n = blockIdx.x / subparts;
    const int64_t s0 = sp * S / subparts, s1 = (sp + 1) * S / subparts;
    const int slot = threadIdx.x / cv, oct = threadIdx.x % cv;
    float sum[8], sq[8];
#pragma unroll
    for (int k = 0; k < 8; k++) sum[k] = sq[k] = 0.f;
    if (slot < slots) {
        const half_t* px = in + n * S * C + oct * 8;
        float shift[8];
        {
            const u32x4 q = *reinterpret_cast<const u32x4*>(px);
            const half_t* h = reinterpret_cast<const half_t*>(&q);
#pragma unroll
            for (int k = 0; k < 8; k++) shift[k] = SHIFT ? (float)h[k] : 0.f;
        }
        for (int64_t i = s0 + slot; i < s1; i += slots) {
            const u32x4 q = *reinterpret_cast<const u32x4*>(px + i * C);
            const half_t* h = reinterpret_cast<const half_t*>(&q);
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const float x = (float)h[k] - shift[k];
                sum[k] += x;
                sq[k] += x * x;
            }
        }
#pragma unroll
        for (int k = 0; k < 8; k++) red8[(int64_t)slot * C + oct * 8 + k] = float2{sum[k], sq[k]};
    }
    __syncthreads();
    for (int c = threadIdx.x; c < C; c += kThreads) {
        float2 t = red8[c];
        for (int r = 1; r < slots; r++) t = add2(t, red8[(int64_t)r * C + c]);
        partial[(n * subparts + sp) * cpad + c] = t;
    }
}

// Launches whichever sum kernel fits; `subparts` spatial ranges per image, partials [N][subparts][cpad].
template <bool SHIFT>
static int launch_sum_cminor(const half_t* in, int64_t N, int64_t S, int64_t C, int64_t subparts, int64_t cpad, float2* partial,
                             hipStream_t s) {
    if (C % 8 == 0 && C >= 8 && C <= 2048 && (reinterpret_cast<uintptr_t>(in) & 15) == 0) {
        const int slots = kThreads / (int)(C / 8);
        const size_t lds = sizeof(float2) * (size_t)slots * (size_t)C;  // at most 16 KiB
        VPX_LAUNCH(mvn_sum_cminor8_kernel<SHIFT>, dim3((unsigned)(N * subparts)), dim3(kThreads), lds, s, in, S, C, (int)subparts,
                   cpad, partial);
    } else {
        VPX_LAUNCH(mvn_sum_cminor_kernel<SHIFT>, dim3((unsigned)(N * subparts * (cpad / 64))), dim3(kThreads), 0, s, in, S, C,
                   (int)subparts, cpad, partial);
    }
    return VPX_RESULT_SUCCESS;
}

__global__ __launch_bounds__(kThreads) void mvn_sum_cminor_finish_kernel(const float2* __restrict__ partial, int64_t total,
                                                                         int64_t C, int64_t cpad, int subparts, int isplit,
                                                                         SumOut o) {
    const int64_t idx = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (idx >= total) return;
    const int64_t c = idx % C;
    const int part = (int)((idx / C) % o.parts);
    const int64_t n = idx / (C * o.parts);
    float2 acc{0.f, 0.f};
#pragma unroll 8
    for (int j = 0; j < isplit; j++) acc = add2(acc, partial[(n * subparts + part * isplit + j) * cpad + c]);
    o.put(n * C + c, part, acc.x, acc.y);
}

// mvn1 on a channel-minor layout with per-channel statistics: folds the shifted partial sums of one
// (n, c) and leaves {mean, 1/std} as fp32 in the layout mvn_norm_cminor_kernel reads.
__global__ __launch_bounds__(kThreads) void mvn_cminor_stats_kernel(const half_t* __restrict__ in, const float2* __restrict__ partial,
                                                                    float* __restrict__ stats, int64_t total, int64_t S, int64_t C,
                                                                    int64_t cpad, int subparts, int normalize_variance, float eps) {
    const int64_t idx = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (idx >= total) return;
    const int64_t c = idx % C, n = idx / C;
    float2 acc{0.f, 0.f};
#pragma unroll 8
    for (int j = 0; j < subparts; j++) acc = add2(acc, partial[(n * subparts + j) * cpad + c]);
    const float shift = (float)in[n * S * C + c];
    const float cnt = (float)S;
    const float m = acc.x / cnt;
    const float var = fmaxf(acc.y / cnt - m * m, 0.f);
    stats[(n * 2) * C + c] = shift + m;
    stats[(n * 2 + 1) * C + c] = normalize_variance ? 1.0f / __builtin_sqrtf(var + eps) : 1.0f;
}

// One lane per output statistic; the handful of partial sums is folded in double.
template <typename TO>
__global__ __launch_bounds__(kThreads) void mvn_mean_var_kernel(const float* __restrict__ sum, TO* __restrict__ out, int64_t N,
                                                                int64_t c_in, int parts, int in_w, int64_t out_c, int out_w,
                                                                int across, int64_t group_c, double count, float eps) {
    const int64_t idx = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (idx >= N * out_c) return;
    const int64_t n = idx / out_c, c = idx % out_c;
    int64_t c0 = 0, c1 = c_in;
    if (!across) {
        c0 = (c / group_c) * group_c;
        c1 = c0 + group_c < c_in ? c0 + group_c : c_in;
    }
    double s = 0.0, q = 0.0;
    for (int p = 0; p < parts; p++) {
        const float* row = sum + ((n * parts + p) * in_w) * c_in;
        for (int64_t ci = c0; ci < c1; ci++) {
            s += (double)row[ci];
            if (in_w == 2) q += (double)row[c_in + ci];
        }
    }
    const double mean = s / count;
    out[(n * out_w) * out_c + c] = (TO)(float)mean;
    if (out_w == 2) {
        double var = q / count - mean * mean;
        var = var > 0.0 ? var : 0.0;
        out[(n * out_w + 1) * out_c + c] = (TO)(float)(1.0 / __builtin_sqrt(var + (double)eps));
    }
}

// x and y in runs of `run` elements that share one statistic (a (n,c) plane, or a whole batch
// element when across channels): one workgroup per 2048-element piece of a run.
template <typename TS, bool ALIGNED>
__global__ __launch_bounds__(kThreads) void mvn_norm_runs_kernel(const half_t* __restrict__ in, half_t* __restrict__ out,
                                                                 const TS* __restrict__ mv, int64_t run, int pieces,
                                                                 int64_t rows_per_n, int64_t out_c, int out_w) {
    const int64_t row = blockIdx.x / pieces;
    const int piece = blockIdx.x % pieces;
    const int64_t n = row / rows_per_n, c = row % rows_per_n;  // rows_per_n = 1 when across channels
    const float mean = (float)mv[(n * out_w) * out_c + c];
    const float inv = out_w == 2 ? (float)mv[(n * out_w + 1) * out_c + c] : 1.0f;
    const int64_t e0 = (int64_t)piece * (kThreads * 8) + threadIdx.x * 8;
    const half_t* gi = in + row * run;
    half_t* go = out + row * run;
    if (ALIGNED && e0 + 8 <= run) {
        const u32x4 q = *reinterpret_cast<const u32x4*>(gi + e0);
        const half_t* p = reinterpret_cast<const half_t*>(&q);
        u32x4 y;
        half_t* py = reinterpret_cast<half_t*>(&y);
#pragma unroll
        for (int k = 0; k < 8; k++) py[k] = round_f16(((float)p[k] - mean) * inv);
        __builtin_nontemporal_store(y, reinterpret_cast<u32x4*>(go + e0));
    } else {
        for (int k = 0; k < 8; k++)
            if (e0 + k < run) go[e0 + k] = round_f16(((float)gi[e0 + k] - mean) * inv);
    }
}

// Channel-minor layout with per-channel statistics: element e of batch element n has channel e % C.
// VEC: the channel count is a multiple of 8 and everything is 16-byte aligned, so a lane's 8 elements are 8
// consecutive channels and their statistics two contiguous runs.
template <typename TS, bool VEC>
__global__ __launch_bounds__(kThreads) void mvn_norm_cminor_kernel(const half_t* __restrict__ in, half_t* __restrict__ out,
                                                                   const TS* __restrict__ mv, int64_t per_n, int64_t C,
                                                                   int pieces, int out_w) {
    const int64_t n = blockIdx.x / pieces;
    const int64_t e0 = (int64_t)(blockIdx.x % pieces) * (kThreads * 8) + threadIdx.x * 8;
    const TS* mean = mv + (n * out_w) * C;
    const TS* inv = mean + C;
    const half_t* gi = in + n * per_n;
    half_t* go = out + n * per_n;
    uint32_t c = (uint32_t)(e0 % C);
    if (VEC) {
        if (e0 >= per_n) return;
        const u32x4 q = *reinterpret_cast<const u32x4*>(gi + e0);
        const half_t* p = reinterpret_cast<const half_t*>(&q);
        TS m[8], iv[8];
        typedef uint32_t words_t __attribute__((ext_vector_type(sizeof(TS) * 2)));  // 8 statistics = 16 or 32 bytes
        *reinterpret_cast<words_t*>(m) = *reinterpret_cast<const words_t*>(mean + c);
        if (out_w == 2) *reinterpret_cast<words_t*>(iv) = *reinterpret_cast<const words_t*>(inv + c);
        u32x4 y;
        half_t* py = reinterpret_cast<half_t*>(&y);
#pragma unroll
        for (int k = 0; k < 8; k++) py[k] = round_f16(((float)p[k] - (float)m[k]) * (out_w == 2 ? (float)iv[k] : 1.0f));
        __builtin_nontemporal_store(y, reinterpret_cast<u32x4*>(go + e0));
        return;
    }
    for (int k = 0; k < 8; k++) {
        if (e0 + k < per_n) {
            const float i = out_w == 2 ? (float)inv[c] : 1.0f;
            go[e0 + k] = round_f16(((float)gi[e0 + k] - (float)mean[c]) * i);
        }
        c = c + 1 == (uint32_t)C ? 0 : c + 1;
    }
}

struct MvnShape {
    int64_t N, C, S;
    bool channel_minor;
};

int mvn_shape(const char* what, const MemRef& in, MvnShape& sh) {
    VPX_REQUIRE(in.nd == 4, VPX_RESULT_ERROR_INVALID_ARGUMENT, "%s: expects a 4-D tensor, got rank %d", what, in.nd);
    VPX_REQUIRE(in.order == VPX_ORDER_NCHW || in.order == VPX_ORDER_NCWH || in.order == VPX_ORDER_NHWC ||
                        in.order == VPX_ORDER_NWHC,
                VPX_RESULT_ERROR_UNSUPPORTED_FEATURE, "%s: unsupported order 0x%llx", what, (unsigned long long)in.order);
    VPX_REQUIRE(in.compact, VPX_RESULT_ERROR_UNSUPPORTED_FEATURE, "%s: only compact tensors are supported", what);
    const int pn = mem_pos_of(in.order, 4, 0), pc = mem_pos_of(in.order, 4, 1);
    VPX_REQUIRE(pn == 3, VPX_RESULT_ERROR_UNSUPPORTED_FEATURE, "%s: batch must be the outermost dimension", what);
    sh.N = in.dims[pn];
    sh.C = in.dims[pc];
    sh.S = sh.N * sh.C ? in.numel() / (sh.N * sh.C) : 0;
    sh.channel_minor = pc != 2;
    return VPX_RESULT_SUCCESS;
}

// Logical [N, C, H, W] of a 4-D channel-minor (NHWC) statistics tensor.
int stats_shape(const char* what, const MemRef& m, int64_t dims[4]) {
    VPX_REQUIRE(m.nd == 4 && m.order == VPX_ORDER_NHWC && m.compact, VPX_RESULT_ERROR_INVALID_ARGUMENT,
                "%s: the statistics tensor must be a compact 4-D NHWC tensor", what);
    for (int l = 0; l < 4; l++) dims[l] = m.dims[mem_pos_of(m.order, 4, l)];
    return VPX_RESULT_SUCCESS;
}


// ------------------------------------------------------------------------------------------------
// mvn6: OpenVINO MVN-6 over an arbitrary set of axes with the eps inside or outside the square
// root, and the compiler's fused `* scale + bias` (VPU.MVN6,
// src/vpux_compiler/tblgen/vpux/compiler/dialect/VPU/ops.td:3850-3900;
// src/vpux_compiler/src/dialect/IE/transforms/passes/fuse_mvn6_scale_bias.cpp).  A row is one
// combination of the kept (not normalised) coordinates.

struct Mvn6Geom {
    int nk, nr;
    int32_t kdim[kMaxDims], rdim[kMaxDims];
    int64_t k_in[kMaxDims], k_out[kMaxDims], k_sc[kMaxDims], k_bi[kMaxDims];
    int64_t r_in[kMaxDims], r_out[kMaxDims], r_sc[kMaxDims], r_bi[kMaxDims];
    int64_t rows;
    uint32_t row_len;
    int sc_along_row, bi_along_row;  // contiguous-row kernels: 1 = the operand has the row's elements, 0 = one value per row
};

struct RowBase {
    int64_t in, out, sc, bi;
};

__device__ __forceinline__ RowBase row_base(const Mvn6Geom& g, int64_t row) {
    RowBase b{0, 0, 0, 0};
    uint32_t r = (uint32_t)row;  // the host keeps the row count below 2^31
    for (int d = 0; d < g.nk; d++) {
        const bool last = d == g.nk - 1;  // what is left indexes the outermost kept dimension: no division
        const int64_t c = last ? r : r % (uint32_t)g.kdim[d];
        if (!last) r /= (uint32_t)g.kdim[d];
        b.in += c * g.k_in[d];
        b.out += c * g.k_out[d];
        b.sc += c * g.k_sc[d];
        b.bi += c * g.k_bi[d];
    }
    return b;
}

// The same with at most one kept dimension: what a launch says fits two lines of its argument block, read at once.  (Mvn6Geom's eleven lines are read
// one after another as the walk over its dimensions comes to them, each a trip to memory in front of the first row.)
struct FlatGeom {
    int64_t in, out, sc, bi;  // from row to row
    int64_t rows;
    uint32_t row_len;
    int sc_along_row, bi_along_row;
};
__device__ __forceinline__ RowBase row_base(const FlatGeom& g, int64_t row) {
    return RowBase{row * g.in, row * g.out, row * g.sc, row * g.bi};
}

__device__ __forceinline__ float mvn6_inv(float var, int normalize_variance, int eps_mode, float eps) {
    if (!normalize_variance) return 1.0f;
    return eps_mode == 0 ? inv_root(var + eps) : 1.0f / (__builtin_sqrtf(var) + eps);
}

// Sum over the TEAM lanes that share a row: half a wavefront, a wavefront, or the whole workgroup.
template <int TEAM>
__device__ __forceinline__ float team_sum(float v, float* smem) {
    if (TEAM == 32) {  // the row operations and the 16-lane swap stay inside each half
        v += dppf<0xB1>(v);
        v += dppf<0x4E>(v);
        v += dppf<0x141>(v);
        v += dppf<0x140>(v);
        return v + swz16(v);
    }
    if (TEAM == 64) return wave_sum(v);
    v = wave_sum_soon(v);
    // one barrier: each sum of a workgroup's lifetime has slots of its own
    if ((threadIdx.x & 63) == 0) smem[threadIdx.x >> 6] = v;
    __syncthreads();
    if (TEAM == 256) return (smem[0] + smem[1]) + (smem[2] + smem[3]);
    constexpr int WAVES = TEAM / 64;  // 8 or 16, one per lane of a row of 16
    v = smem[threadIdx.x & (WAVES - 1)];
    v += dppf<0xB1>(v);
    v += dppf<0x4E>(v);
    v += dppf<0x141>(v);
    return WAVES == 16 ? v + dppf<0x140>(v) : v;
}

// Rows that are contiguous in memory: the row lives in the registers of half a wavefront (TEAM = 32, eight rows per
// workgroup), of a wavefront (64) or of the workgroup (256).
// WORDS: rows start on 128-bit words and are a whole number of them.  Else (rows of at least eight values, at any
// address) the accesses are the same 128-bit ones at 2-byte alignment, and the lane with the row's last, partial word
// takes the row's last eight values: those it shares with its neighbour stay out of its sums, and both store them alike.
// Element-per-lane accesses and three passes over such rows took 21.1 us for [14187 x 173] (1.9 us of traffic).
__device__ __forceinline__ uint32_t row_at(uint32_t e0, uint32_t row_len) {
    return e0 + 8 <= row_len ? e0 : row_len - 8;
}
template <bool WORDS>
__device__ __forceinline__ u32x4 row_word(const half_t* row, uint32_t e0, uint32_t row_len) {
    if (WORDS) return *reinterpret_cast<const u32x4*>(row + e0);
    return *reinterpret_cast<const u32x4_any*>(row + row_at(e0, row_len));
}
// how many of a word's values belong to the word before
template <bool WORDS>
__device__ __forceinline__ int row_again(uint32_t e0, uint32_t row_len) {
    return WORDS ? 0 : e0 >= row_len ? 8 : (int)(e0 - row_at(e0, row_len));
}
constexpr int kMvn6MaxRegRow = 16384;  // longest row a workgroup keeps in registers (64 values per lane)
constexpr int team_threads(int team) { return team > kThreads ? team : kThreads; }
// Wavefronts a SIMD that the registers are cut for: the words and their values, with RPT > 1 a scale and a bias beside them.  (Left to itself the compiler
// takes 250 registers for eight words: [3808 x 10640] 45 us in place of 35.)
constexpr int row_waves(int vpt, int rpt) {
    return rpt > 1 ? (vpt == 1 ? 8 : vpt == 2 ? 5 : vpt == 3 ? 4 : vpt == 4 ? 3 : 2) : vpt <= 2 ? 8 : vpt <= 4 ? 7 : vpt == 5 ? 6 : vpt == 6 ? 5 : 4;
}
template <class GEOM, int TEAM, int VPT, int RPT = 1, bool WORDS = true>  // RPT: consecutive rows a team walks, keeping a scale / bias that runs along the row in registers
__global__ __launch_bounds__(team_threads(TEAM)) __attribute__((amdgpu_waves_per_eu(row_waves(VPT, RPT)))) void mvn6_rows_kernel(const half_t* __restrict__ in, half_t* __restrict__ out,
                                                             const half_t* __restrict__ sc, const half_t* __restrict__ bi,
                                                             GEOM g, int normalize_variance, int eps_mode, float eps) {
    constexpr int T = team_threads(TEAM);
    __shared__ float red[32];
    static_assert(TEAM < 256 || RPT == 1, "the workgroup-wide sums have slots for one row");
    const int t = (int)(threadIdx.x % TEAM);
    const int64_t row0 = ((int64_t)blockIdx.x * (T / TEAM) + threadIdx.x / TEAM) * RPT;
    // The words of a row are asked for all at once (but see AHEAD), and before they are used the scale and the bias that run along it: asked for
    // where they are needed, behind both sums, they cost a trip to the caches per row ([16384 x 4096] 56.7 -> 51.9 us, [16384 x
    // 1024] 17.1 -> 15.9, [1 x 4096] 3.2 -> 2.7).  They stay late where nothing is gained, of one word per lane of a workgroup or
    // of half a wavefront, and where their registers cost a wavefront per SIMD, from three words of half a wavefront or four of
    // one on ([16384 x 768] 11.2 us late, 13.1 early, [8192 x 2048] 14.2 and 17.2).
    constexpr bool EARLY = RPT > 1 || (TEAM == 64 ? VPT <= 3 : TEAM == 512 ? VPT <= 2 : VPT == 2);
    // Three to five words per lane of a workgroup are converted each as it comes: all asked for first they gain from memory
    // ([800 x 6480] 7.83 -> 6.98 us) what they lose from the cache that the writer of the rows left them in ([1280 x 4324] 8.51 ->
    // 8.76 us, [800 x 8100] 9.12 -> 9.57); from six on there is a gain in both ([512 x 12544] 9.53 -> 7.45 and 8.01 -> 7.70).
    constexpr bool AHEAD = RPT > 1 || TEAM != 256 || VPT <= 2 || VPT >= 6;
    const auto fetch = [&](const RowBase& at, bool real, u32x4(&w)[VPT]) {
#pragma unroll
        for (int j = 0; j < VPT; j++) {
            const uint32_t e0 = (uint32_t)(j * TEAM + t) * 8;
            if (real && e0 < g.row_len) w[j] = row_word<WORDS>(in + at.in, e0, g.row_len);
        }
    };
    bool live = row0 < g.rows;  // uniform per team; dead teams skip memory only
    RowBase b = row_base(g, live ? row0 : 0);
    u32x4 words[VPT];
    if (AHEAD) fetch(b, live, words);
    // scale and bias that run along the row, asked for beside it; with RPT > 1 they do not depend on it and are loaded once
    u32x4 scv[VPT], biv[VPT];
    if (EARLY) {
#pragma unroll
        for (int j = 0; j < VPT; j++) {
            const uint32_t e0 = (uint32_t)(j * TEAM + t) * 8;
            if (e0 < g.row_len) {
                if (sc && g.sc_along_row) scv[j] = row_word<WORDS>(sc + b.sc, e0, g.row_len);
                if (bi && g.bi_along_row) biv[j] = row_word<WORDS>(bi + b.bi, e0, g.row_len);
            }
        }
    }
    const float n = (float)g.row_len, inv_n = 1.0f / n;  // (under the loads)
#pragma unroll 1
    for (int rr = 0; rr < RPT; rr++) {
    float x[VPT][8];
    float sum = 0.f;
#pragma unroll
    for (int j = 0; j < VPT; j++) {
        const uint32_t e0 = (uint32_t)(j * TEAM + t) * 8;
        if (live && e0 < g.row_len) {
            const u32x4 q = AHEAD ? words[j] : row_word<WORDS>(in + b.in, e0, g.row_len);
            const half_t* p = reinterpret_cast<const half_t*>(&q);
            const int again = row_again<WORDS>(e0, g.row_len);
#pragma unroll
            for (int k = 0; k < 8; k++) {
                x[j][k] = (float)p[k];
                sum += k >= again ? x[j][k] : 0.f;
            }
        } else {
#pragma unroll
            for (int k = 0; k < 8; k++) x[j][k] = 0.f;
        }
    }
    const RowBase here = b;
    const bool real = live;
    if (RPT > 1 && rr + 1 < RPT) {  // the next row is on its way while this one is summed and stored
        live = row0 + rr + 1 < g.rows;
        b = row_base(g, live ? row0 + rr + 1 : 0);
        fetch(b, live, words);
    }
    const float mean = over(team_sum<TEAM>(sum, red), n, inv_n);
    float q = 0.f;
#pragma unroll
    for (int j = 0; j < VPT; j++) {
        const uint32_t e0 = (uint32_t)(j * TEAM + t) * 8;
        const int again = row_again<WORDS>(e0, g.row_len);  // (8 past the row's end)
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const float d = x[j][k] - mean;
            q += (WORDS ? e0 < g.row_len : k >= again) ? d * d : 0.f;
        }
    }
    const float var = over(team_sum<TEAM>(q, red + 16), n, inv_n);
    const float inv = mvn6_inv(var, normalize_variance, eps_mode, eps);
    const float sc_row = sc && !g.sc_along_row ? (float)sc[here.sc] : 1.0f;
    const float bi_row = bi && !g.bi_along_row ? (float)bi[here.bi] : 0.0f;
#pragma unroll
    for (int j = 0; j < VPT; j++) {
        const uint32_t e0 = (uint32_t)(j * TEAM + t) * 8;
        if (!(real && e0 < g.row_len)) continue;
        float y[8];
#pragma unroll
        for (int k = 0; k < 8; k++) y[k] = (x[j][k] - mean) * inv;
        if (sc) {
            if (g.sc_along_row) {
                const u32x4 v = EARLY ? scv[j] : row_word<WORDS>(sc + here.sc, e0, g.row_len);
                const half_t* p = reinterpret_cast<const half_t*>(&v);
#pragma unroll
                for (int k = 0; k < 8; k++) y[k] *= (float)p[k];
            } else {
#pragma unroll
                for (int k = 0; k < 8; k++) y[k] *= sc_row;
            }
        }
        if (bi) {
            if (g.bi_along_row) {
                const u32x4 v = EARLY ? biv[j] : row_word<WORDS>(bi + here.bi, e0, g.row_len);
                const half_t* p = reinterpret_cast<const half_t*>(&v);
#pragma unroll
                for (int k = 0; k < 8; k++) y[k] += (float)p[k];
            } else {
#pragma unroll
                for (int k = 0; k < 8; k++) y[k] += bi_row;
            }
        }
        u32x4 o;
        half_t* po = reinterpret_cast<half_t*>(&o);
#pragma unroll
        for (int k = 0; k < 8; k++) po[k] = (half_t)y[k];
        if (WORDS) __builtin_nontemporal_store(o, reinterpret_cast<u32x4*>(out + here.out + e0));
        else *reinterpret_cast<u32x4_any*>(out + here.out + row_at(e0, g.row_len)) = o;
    }
    }
}

struct ElemOff {
    int64_t in, out, sc, bi;
};
__device__ __forceinline__ ElemOff elem_off(const Mvn6Geom& g, uint32_t e) {
    ElemOff o{0, 0, 0, 0};
    for (int d = 0; d < g.nr; d++) {
        const uint32_t c = e % (uint32_t)g.rdim[d];
        e /= (uint32_t)g.rdim[d];
        o.in += c * g.r_in[d];
        o.out += c * g.r_out[d];
        o.sc += c * g.r_sc[d];
        o.bi += c * g.r_bi[d];
    }
    return o;
}

// The innermost dimension is kept and contiguous (normalising over channels of a channel-major tensor,
// say): a workgroup takes P adjacent positions of it, so that every access covers a contiguous run, and
// splits the reduced elements over its 256 / P lane groups (group r walks elements r, r + G, ...; three
// passes, the later ones from cache).  Smaller P gives more workgroups when the tensor has few positions.
template <int P>
__global__ __launch_bounds__(kThreads) void mvn6_inner_kernel(const half_t* __restrict__ in, half_t* __restrict__ out,
                                                              const half_t* __restrict__ sc, const half_t* __restrict__ bi,
                                                              Mvn6Geom g, int normalize_variance, int eps_mode, float eps) {
    constexpr int G = kThreads / P;
    __shared__ float red[G][P];
    const int cl = threadIdx.x % P;
    const uint32_t r = P == 64 ? (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x / P)) : threadIdx.x / P;
    const int64_t tiles = (g.kdim[0] + P - 1) / P;
    int64_t o = blockIdx.x / tiles;
    const int64_t i0 = (blockIdx.x % tiles) * P + cl;
    const bool ok = i0 < g.kdim[0];
    RowBase b{0, 0, 0, 0};
    for (int d = 1; d < g.nk; d++) {
        const int64_t c = o % g.kdim[d];
        o /= g.kdim[d];
        b.in += c * g.k_in[d];
        b.out += c * g.k_out[d];
        b.sc += c * g.k_sc[d];
        b.bi += c * g.k_bi[d];
    }
    const int64_t i = ok ? i0 : 0;
    b.in += i * g.k_in[0];
    b.out += i * g.k_out[0];
    b.sc += i * g.k_sc[0];
    b.bi += i * g.k_bi[0];
    const float n = (float)g.row_len;
    const auto total = [&](float v) {
        __syncthreads();
        red[r][cl] = v;
        __syncthreads();
        float t = 0.f;
#pragma unroll
        for (int k = 0; k < G; k++) t += red[k][cl];
        return t;
    };
    float sum = 0.f;
    for (uint32_t e = r; e < g.row_len; e += G) sum += (float)in[b.in + elem_off(g, e).in];
    const float mean = total(sum) / n;
    float q = 0.f;
    if (normalize_variance)
        for (uint32_t e = r; e < g.row_len; e += G) {
            const float d = (float)in[b.in + elem_off(g, e).in] - mean;
            q += d * d;
        }
    const float var = total(q) / n;
    const float inv = mvn6_inv(var, normalize_variance, eps_mode, eps);
    if (!ok) return;
    for (uint32_t e = r; e < g.row_len; e += G) {
        const ElemOff off = elem_off(g, e);
        float y = ((float)in[b.in + off.in] - mean) * inv;
        if (sc) y *= (float)sc[b.sc + off.sc];
        if (bi) y += (float)bi[b.bi + off.bi];
        out[b.out + off.out] = (half_t)y;
    }
}

// Any layout, any row length: one workgroup per row, three passes over the row (the second and
// third come from cache).
__global__ __launch_bounds__(kThreads) void mvn6_generic_kernel(const half_t* __restrict__ in, half_t* __restrict__ out,
                                                                const half_t* __restrict__ sc, const half_t* __restrict__ bi,
                                                                Mvn6Geom g, int normalize_variance, int eps_mode, float eps) {
    __shared__ float red[8];
    const RowBase b = row_base(g, blockIdx.x);
    float sum = 0.f;
    for (uint32_t e = threadIdx.x; e < g.row_len; e += kThreads) sum += (float)in[b.in + elem_off(g, e).in];
    const float n = (float)g.row_len;
    const float mean = team_sum<256>(sum, red) / n;
    float q = 0.f;
    if (normalize_variance)
        for (uint32_t e = threadIdx.x; e < g.row_len; e += kThreads) {
            const float d = (float)in[b.in + elem_off(g, e).in] - mean;
            q += d * d;
        }
    const float var = team_sum<256>(q, red + 4) / n;
    const float inv = mvn6_inv(var, normalize_variance, eps_mode, eps);
    for (uint32_t e = threadIdx.x; e < g.row_len; e += kThreads) {
        const ElemOff o = elem_off(g, e);
        float y = ((float)in[b.in + o.in] - mean) * inv;
        if (sc) y *= (float)sc[b.sc + o.sc];
        if (bi) y += (float)bi[b.bi + o.bi];
        out[b.out + o.out] = (half_t)y;
    }
}


// Contiguous rows of 8 ... kMvn6MaxRegRow values (see mvn6_rows_kernel); words: the rows are whole, aligned 128-bit words.
template <class GEOM>
int launch_rows_of(const half_t* pi, half_t* po, const half_t* ps, const half_t* pb, const GEOM& g, bool shared_rows, bool words, int nv, int eps_mode,
                   float eps, hipStream_t s) {
    const int64_t row_len = g.row_len;
    const bool half768 = shared_rows && row_len == 768;  // 32 lanes x 3 words, none idle: pays with scale / bias
    const int team = row_len <= 256 || half768 ? 32 : 64;
    const int64_t team_rows = g.rows / (kThreads / team);
    // (two rows of three words a lane and more only where they are whole words: with the values that words share the registers run out, and a row at a time is ahead;
    // us, two / one: [40382 x 1233] 42.6 / 35.8, [62548 x 1322] 75.3 / 58.8, [39878 x 1606] 55.0 / 43.8, [58293 x 2031] 109.4 / 108.3)
    const int rpt = !shared_rows ? 1 : team_rows >= 4 * 4096 ? 4 : team_rows >= 2 * 4096 && (words || (row_len <= 1024 && !half768)) ? 2 : 1;
#define VPX_MVN6_ROWS_R(TEAM, VPT, RPT)                                                                                      \
    do {                                                                                                                     \
        constexpr int T = team_threads(TEAM), PER = RPT * (T / TEAM);                                                        \
        const dim3 grid((unsigned)((g.rows + PER - 1) / PER));                                                               \
        if (words)                                                                                                           \
            VPX_LAUNCH((mvn6_rows_kernel<GEOM, TEAM, VPT, RPT, true>), grid, dim3(T), 0, s, pi, po, ps, pb, g, nv,                 \
                       eps_mode, eps);                                                                                       \
        else if constexpr (RPT != 2 || VPT <= 2)                                                                             \
            VPX_LAUNCH((mvn6_rows_kernel<GEOM, TEAM, VPT, RPT, false>), grid, dim3(T), 0, s, pi, po, ps, pb, g, nv,                \
                       eps_mode, eps);                                                                                       \
    } while (0)
#define VPX_MVN6_ROWS(TEAM, VPT) VPX_MVN6_ROWS_R(TEAM, VPT, 1)
#define VPX_MVN6_SHORT(TEAM, VPT)                         \
    do {                                                  \
        if (rpt == 4) VPX_MVN6_ROWS_R(TEAM, VPT, 4);      \
        else if (rpt == 2) VPX_MVN6_ROWS_R(TEAM, VPT, 2); \
        else VPX_MVN6_ROWS(TEAM, VPT);                    \
    } while (0)
    // Rows too few to give every SIMD several wavefronts: the whole workgroup takes a row, one or two words per lane in
    // place of up to six one after another ([1024 x 2752] 7.5 -> 5.0 us, [2048 x 2304] 7.9 -> 6.4, [64 x 1280] 4.4 -> 3.3;
    // with twice the rows the wavefront form is ahead again, 6.7 against 7.6 us for [4096 x 1280]).
    const bool few = row_len > 640 && g.rows <= (row_len > 1024 ? 2048 : 1024);
    // A row or less per compute unit: 512 lanes take it, at most half as many words each ([128 x 8640] 4.53 -> 4.03 us in a HIP graph, [9 x
    // 9216] 4.33 -> 3.79; with scale and bias [16 x 2050] 3.88 -> 3.59, [256 x 3136] 3.94 -> 3.79, [1 x 1088] 3.20 -> 3.11; of up to 2048 values without them
    // nothing is gained, [128 x 1200] 3.47 / 3.52).  With two rows a unit it is even ([512 x 4096] 3.97 / 4.01), with four slower ([1024 x 4096] 4.73 / 5.20);
    // 1024 lanes are behind 512 but for [512 x 16384] (8.17 / 7.80, 1024 rows 11.7 / 12.9).
    int cus = 0;
    const int rc = device_compute_units(&cus);
    if (rc) return rc;
    const bool wide = g.rows <= cus && row_len > (ps || pb ? 640 : 2048);
    if (wide && row_len <= 4096) VPX_MVN6_ROWS(512, 1);
    else if (wide && row_len <= 8192) VPX_MVN6_ROWS(512, 2);
    else if (wide && row_len <= 12288) VPX_MVN6_ROWS(512, 3);
    else if (wide) VPX_MVN6_ROWS(512, 4);
    else if (few && row_len <= 2048) VPX_MVN6_ROWS(256, 1);
    else if (few && row_len <= 4096) VPX_MVN6_ROWS(256, 2);
    else if (row_len <= 256) VPX_MVN6_SHORT(32, 1);
    else if (row_len <= 512) VPX_MVN6_SHORT(64, 1);
    else if (half768) VPX_MVN6_SHORT(32, 3);
    else if (row_len <= 1024) VPX_MVN6_SHORT(64, 2);
    else if (row_len <= 1536) VPX_MVN6_SHORT(64, 3);
    else if (row_len <= 2048) VPX_MVN6_SHORT(64, 4);
    else if (row_len <= 2560) VPX_MVN6_SHORT(64, 5);
    else if (row_len <= 3072) VPX_MVN6_SHORT(64, 6);
    else if (row_len <= 4096) VPX_MVN6_ROWS(256, 2);  // one wavefront per 4096-element row measured 9 % slower
    else if (row_len <= 6144) VPX_MVN6_ROWS(256, 3);
    else if (row_len <= 8192) VPX_MVN6_ROWS(256, 4);
    else if (row_len <= 10240) VPX_MVN6_ROWS(256, 5);
    else if (row_len <= 12288) VPX_MVN6_ROWS(256, 6);
    else if (row_len <= 14336) VPX_MVN6_ROWS(256, 7);
    else VPX_MVN6_ROWS(256, 8);
#undef VPX_MVN6_ROWS
#undef VPX_MVN6_ROWS_R
#undef VPX_MVN6_SHORT
    return VPX_RESULT_SUCCESS;
}

// A launch holds fewer than 2^32 lanes, a row of many takes 32, 64 or 256 of them: several launches from 2^31 on (2^26 rows of 24 values, 2^25 of 520).
int launch_flat_rows(const half_t* pi, half_t* po, const half_t* ps, const half_t* pb, const FlatGeom& g, bool shared_rows, bool words, int nv, int eps_mode,
                     float eps, hipStream_t s) {
    const int64_t most = (1ll << 31) / (g.row_len <= 256 ? 32 : g.row_len <= 3072 ? 64 : 256);
    for (int64_t r0 = 0; r0 < g.rows; r0 += most) {
        FlatGeom part = g;
        part.rows = g.rows - r0 < most ? g.rows - r0 : most;
        const int rc = launch_rows_of(pi + r0 * g.in, po + r0 * g.out, ps ? ps + r0 * g.sc : nullptr, pb ? pb + r0 * g.bi : nullptr, part, shared_rows, words, nv,
                                      eps_mode, eps, s);
        if (rc) return rc;
    }
    return VPX_RESULT_SUCCESS;
}

// rows of a tensor with any kept dimensions
int launch_rows(const half_t* pi, half_t* po, const half_t* ps, const half_t* pb, const Mvn6Geom& g, bool words, int nv, int eps_mode,
                float eps, hipStream_t s) {
    // A scale / bias shared by all rows stays in registers while a team walks 2 or 4 consecutive rows, as long
    // as that leaves 4096 workgroups (two rounds of the chip) or more.
    bool shared_rows = (ps && g.sc_along_row) || (pb && g.bi_along_row);
    for (int d = 0; d < g.nk; d++)
        if ((ps && g.sc_along_row && g.k_sc[d] != 0) || (pb && g.bi_along_row && g.k_bi[d] != 0)) shared_rows = false;
    // kept dimensions that every operand walks as one
    int nk = g.nk > 0 ? 1 : 0;
    for (; nk < g.nk; nk++) {
        const int64_t n = g.kdim[nk - 1];
        if (g.k_in[nk] != n * g.k_in[nk - 1] || g.k_out[nk] != n * g.k_out[nk - 1] || (ps && g.k_sc[nk] != n * g.k_sc[nk - 1]) ||
            (pb && g.k_bi[nk] != n * g.k_bi[nk - 1]))
            break;
    }
    if (nk < g.nk) return launch_rows_of(pi, po, ps, pb, g, shared_rows, words, nv, eps_mode, eps, s);
    const bool kept = g.nk > 0;
    const FlatGeom f{kept ? g.k_in[0] : 0, kept ? g.k_out[0] : 0, kept && ps ? g.k_sc[0] : 0, kept && pb ? g.k_bi[0] : 0, g.rows, g.row_len,
                     g.sc_along_row, g.bi_along_row};
    return launch_flat_rows(pi, po, ps, pb, f, shared_rows, words, nv, eps_mode, eps, s);
}

// mvn1 over groups that follow one another in memory, as rows
int launch_group_rows(const half_t* in, half_t* out, int64_t groups, int64_t len, int nv, float eps, hipStream_t s) {
    const bool words = len % 8 == 0 && ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) & 15) == 0;
    return launch_flat_rows(in, out, nullptr, nullptr, FlatGeom{len, len, 0, 0, groups, (uint32_t)len, 0, 0}, false, words, nv, 0, eps, s);
}

// mvn1 with per-channel statistics on a channel-minor layout: shifted partial sums over spatial ranges,
// a fold to {mean, 1/std}, then the element-wise pass.
int launch_channel_minor(const half_t* in, half_t* out, int64_t N, int64_t S, int64_t C, int nv, float eps, hipStream_t s) {
    const int64_t ctiles = (C + 63) / 64, cpad = ctiles * 64;
    // spatial ranges per image: enough workgroups to fill the chip (the eight-channel kernel has no channel tiles)
    const bool octets = C % 8 == 0 && C >= 8 && C <= 2048 && (reinterpret_cast<uintptr_t>(in) & 15) == 0;
    const int64_t per_range = octets ? N : N * ctiles;
    int64_t subparts = ((octets ? 2048 : 1024) + per_range - 1) / per_range;
    if (subparts > S / 64) subparts = S / 64;
    if (subparts < 1) subparts = 1;
    const int64_t per_n = S * C, piece = kThreads * 8, pieces = (per_n + piece - 1) / piece;
    VPX_REQUIRE(N * subparts * ctiles < (1ll << 31) && N * pieces < (1ll << 31) && C < (1ll << 31), VPX_RESULT_ERROR_UNSUPPORTED_FEATURE,
                "mvn1: tensor exceeds the launch limit");
    void* ws = nullptr;
    const size_t partial_bytes = sizeof(float2) * (size_t)(N * subparts * cpad);
    int rc = get_workspace(s, partial_bytes + sizeof(float) * (size_t)(N * 2 * C), &ws);
    if (rc) return rc;
    float2* partial = (float2*)ws;
    float* stats = (float*)((char*)ws + partial_bytes);
    rc = launch_sum_cminor<true>(in, N, S, C, subparts, cpad, partial, s);
    if (rc) return rc;
    VPX_LAUNCH(mvn_cminor_stats_kernel, dim3((unsigned)((N * C + kThreads - 1) / kThreads)), dim3(kThreads), 0, s, in,
               (const float2*)partial, stats, N * C, S, C, cpad, (int)subparts, nv, eps);
    const bool vec = C % 8 == 0 && ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) & 15) == 0 &&
                     (reinterpret_cast<uintptr_t>(stats) & 31) == 0;
    if (vec)
        VPX_LAUNCH((mvn_norm_cminor_kernel<float, true>), dim3((unsigned)(N * pieces)), dim3(kThreads), 0, s, in, out,
                   (const float*)stats, per_n, C, (int)pieces, 2);
    else
        VPX_LAUNCH((mvn_norm_cminor_kernel<float, false>), dim3((unsigned)(N * pieces)), dim3(kThreads), 0, s, in, out,
                   (const float*)stats, per_n, C, (int)pieces, 2);
    return VPX_RESULT_SUCCESS;
}

}  // namespace

int launch_mvn(const MemRef& in, const MemRef& out, bool across_channels, bool normalize_variance, float eps,
               hipStream_t s) {
    VPX_REQUIRE(in.dtype == VPX_NN_FP16 && out.dtype == VPX_NN_FP16, VPX_RESULT_ERROR_UNSUPPORTED_FEATURE,
                "mvn1: only FP16 input/output is implemented, got %s -> %s", dtype_name(in.dtype), dtype_name(out.dtype));
    VPX_REQUIRE(in.nd == 4 && out.nd == 4, VPX_RESULT_ERROR_INVALID_ARGUMENT, "mvn1: expects 4-D tensors, got rank %d",
                in.nd);
    VPX_REQUIRE(in.order == out.order, VPX_RESULT_ERROR_INVALID_ARGUMENT, "mvn1: input and output layouts differ");
    // Same layouts as the reference kernel (sw_kernel.cpp:946-953); compact operands only.
    VPX_REQUIRE(in.order == VPX_ORDER_NCHW || in.order == VPX_ORDER_NCWH || in.order == VPX_ORDER_NHWC ||
                        in.order == VPX_ORDER_NWHC,
                VPX_RESULT_ERROR_UNSUPPORTED_FEATURE, "mvn1: unsupported order 0x%llx", (unsigned long long)in.order);
    VPX_REQUIRE(in.compact && out.compact, VPX_RESULT_ERROR_UNSUPPORTED_FEATURE, "mvn1: only compact tensors are supported");
    for (int d = 0; d < 4; d++)
        VPX_REQUIRE(in.dims[d] == out.dims[d], VPX_RESULT_ERROR_INVALID_ARGUMENT, "mvn1: input and output shapes differ");
    const int pn = mem_pos_of(in.order, 4, 0), pc = mem_pos_of(in.order, 4, 1);
    VPX_REQUIRE(pn == 3, VPX_RESULT_ERROR_UNSUPPORTED_FEATURE, "mvn1: batch must be the outermost dimension");
    const int64_t N = in.dims[pn], C = in.dims[pc];
    const int64_t total = in.numel();
    if (total == 0) return VPX_RESULT_SUCCESS;
    const int64_t S = total / (N * C);
    const half_t* pi = (const half_t*)in.data;
    half_t* po = (half_t*)out.data;
    const int nv = normalize_variance ? 1 : 0;
    {   // in place is served (every kernel reads a value before it stores that value's result); any other overlap is not
        const uintptr_t ib = reinterpret_cast<uintptr_t>(pi), ob = reinterpret_cast<uintptr_t>(po);
        const uintptr_t bytes = (uintptr_t)total * sizeof(half_t);
        VPX_REQUIRE(ib == ob || ib + bytes <= ob || ob + bytes <= ib, VPX_RESULT_ERROR_INVALID_ARGUMENT,
                    "mvn1: input and output overlap without being the same tensor");
    }

    int64_t groups, group_size;
    if (across_channels) {
        groups = N;
        group_size = C * S;
    } else if (pc == 2) {  // channel-major: each (n,c) plane is contiguous
        groups = N * C;
        group_size = S;
    } else {  // channel-minor layout, per-channel statistics
        bool done = false;
        const int rc = launch_mvn_cminor_resident(pi, po, N, S, C, nv, eps, s, &done);
        return rc || done ? rc : launch_channel_minor(pi, po, N, S, C, nv, eps, s);
    }
    if (tiny_groups_ok(pi, po, groups, group_size)) return launch_tiny_groups(pi, po, groups, group_size, nv, 0, eps, s);
    if (small_groups_ok(pi, po, groups, group_size)) return launch_small_groups(pi, po, groups, group_size, nv, 0, eps, s);
    if (group_size >= 8 && group_size <= kMvn6MaxRegRow && groups < (1ll << 31))
        return launch_group_rows(pi, po, groups, group_size, nv, eps, s);
    if (lds_groups_ok(groups, group_size)) return launch_lds_groups(pi, po, groups, group_size, nv, 0, eps, s);
    const bool aligned = group_size % 8 == 0 && (reinterpret_cast<uintptr_t>(pi) & 15) == 0 &&
                         (reinterpret_cast<uintptr_t>(po) & 15) == 0;
    return aligned ? launch_groups<true>(pi, po, groups, group_size, nv, eps, s)
                   : launch_groups<false>(pi, po, groups, group_size, nv, eps, s);
}

int launch_mvn_sum(const MemRef& in, const MemRef& out, bool across_channels, bool normalize_variance, hipStream_t s) {
    VPX_REQUIRE(in.dtype == VPX_NN_FP16 && out.dtype == VPX_NN_FP32, VPX_RESULT_ERROR_UNSUPPORTED_FEATURE,
                "mvn1_sum: FP16 input and FP32 sums are implemented, got %s -> %s", dtype_name(in.dtype), dtype_name(out.dtype));
    MvnShape sh;
    int rc = mvn_shape("mvn1_sum", in, sh);
    if (rc) return rc;
    int64_t od[4];
    rc = stats_shape("mvn1_sum", out, od);
    if (rc) return rc;
    const int64_t out_c = across_channels ? 1 : sh.C;
    const int out_w = normalize_variance ? 2 : 1;
    VPX_REQUIRE(od[0] == sh.N && od[1] == out_c && od[2] >= 1 && od[3] == out_w, VPX_RESULT_ERROR_INVALID_ARGUMENT,
                "mvn1_sum: output shape [%lld,%lld,%lld,%lld] does not match [%lld,%lld,parts,%d]", (long long)od[0],
                (long long)od[1], (long long)od[2], (long long)od[3], (long long)sh.N, (long long)out_c, out_w);
    VPX_REQUIRE(od[2] <= 4096, VPX_RESULT_ERROR_UNSUPPORTED_FEATURE, "mvn1_sum: %lld partial sums per group", (long long)od[2]);
    if (in.numel() == 0) return VPX_RESULT_SUCCESS;
    const SumOut o{(float*)out.data, (int)od[2], out_w, out_c};
    const half_t* pi = (const half_t*)in.data;

    if (!across_channels && sh.channel_minor) {
        const int64_t ctiles = (sh.C + 63) / 64, cpad = ctiles * 64;
        // enough spatial ranges to spread over the device, at least 64 positions each
        int64_t isplit = (1024 + sh.N * ctiles * o.parts - 1) / (sh.N * ctiles * o.parts);
        const int64_t most = sh.S / (64 * (int64_t)o.parts);
        if (isplit > most) isplit = most;
        if (isplit < 1) isplit = 1;
        const int64_t subparts = isplit * o.parts;
        const int64_t blocks = sh.N * subparts * ctiles, total = sh.N * o.parts * sh.C;
        VPX_REQUIRE(blocks < (1ll << 31) && total < (1ll << 31) * kThreads, VPX_RESULT_ERROR_UNSUPPORTED_FEATURE,
                    "mvn1_sum: tensor exceeds the launch limit");
        void* ws = nullptr;
        rc = get_workspace(s, sizeof(float2) * (size_t)(sh.N * subparts * cpad), &ws);
        if (rc) return rc;
        rc = launch_sum_cminor<false>(pi, sh.N, sh.S, sh.C, subparts, cpad, (float2*)ws, s);
        if (rc) return rc;
        VPX_LAUNCH(mvn_sum_cminor_finish_kernel, dim3((unsigned)((total + kThreads - 1) / kThreads)), dim3(kThreads), 0,
                   s, (const float2*)ws, total, sh.C, cpad, (int)subparts, (int)isplit, o);
        return VPX_RESULT_SUCCESS;
    }

    const int64_t groups = across_channels ? sh.N : sh.N * sh.C;
    const int64_t group_size = across_channels ? sh.C * sh.S : sh.S;
    const int64_t chunks64 = (group_size + kChunk - 1) / kChunk;
    VPX_REQUIRE(chunks64 * groups < (1ll << 31) && groups * o.parts < (1ll << 31), VPX_RESULT_ERROR_UNSUPPORTED_FEATURE,
                "mvn1_sum: %lld groups of %lld elements exceed the launch limit", (long long)groups, (long long)group_size);
    const int chunks = (int)chunks64;
    const bool direct = chunks == 1 && o.parts == 1;
    void* ws = nullptr;
    if (!direct) {
        rc = get_workspace(s, sizeof(float2) * (size_t)(groups * chunks), &ws);
        if (rc) return rc;
    }
    const bool aligned = group_size % 8 == 0 && (reinterpret_cast<uintptr_t>(pi) & 15) == 0;
    const dim3 grid((unsigned)(groups * chunks));
    if (aligned)
        VPX_LAUNCH((mvn_sum_chunk_kernel<true>), grid, dim3(kThreads), 0, s, pi, group_size, chunks, (float2*)ws, o,
                   direct ? 1 : 0);
    else
        VPX_LAUNCH((mvn_sum_chunk_kernel<false>), grid, dim3(kThreads), 0, s, pi, group_size, chunks, (float2*)ws, o,
                   direct ? 1 : 0);
    if (!direct) {
        VPX_LAUNCH(mvn_sum_finish_kernel, dim3((unsigned)(groups * o.parts)), dim3(kThreads), 0, s, (const float2*)ws,
                   chunks, o);
    }
    return VPX_RESULT_SUCCESS;
}

int launch_mvn_mean_var(const MemRef& sum, const MemRef& out, const int64_t orig_shape[4], bool across_channels,
                        bool normalize_variance, int64_t group_c, float eps, hipStream_t s) {
    VPX_REQUIRE(sum.dtype == VPX_NN_FP32 && (out.dtype == VPX_NN_FP16 || out.dtype == VPX_NN_FP32),
                VPX_RESULT_ERROR_UNSUPPORTED_FEATURE, "mvn1_mean_var: FP32 sums and FP16/FP32 output are implemented, got %s -> %s",
                dtype_name(sum.dtype), dtype_name(out.dtype));
    int64_t id[4], od[4];
    int rc = stats_shape("mvn1_mean_var", sum, id);
    if (rc) return rc;
    rc = stats_shape("mvn1_mean_var", out, od);
    if (rc) return rc;
    for (int i = 0; i < 4; i++)
        VPX_REQUIRE(orig_shape[i] >= 1, VPX_RESULT_ERROR_INVALID_ARGUMENT, "mvn1_mean_var: orig_shape[%d] = %lld", i,
                    (long long)orig_shape[i]);
    const int64_t N = orig_shape[0], C = orig_shape[1];
    const int64_t out_c = across_channels ? 1 : C;
    const int out_w = normalize_variance ? 2 : 1;
    VPX_REQUIRE(id[0] == N && id[3] >= out_w && id[3] <= 2 && id[1] == out_c, VPX_RESULT_ERROR_INVALID_ARGUMENT,
                "mvn1_mean_var: sums of shape [%lld,%lld,%lld,%lld] do not fit the original shape [%lld,%lld,..] (%s channels)",
                (long long)id[0], (long long)id[1], (long long)id[2], (long long)id[3], (long long)N, (long long)C,
                across_channels ? "across" : "per");
    VPX_REQUIRE(od[0] == N && od[1] == out_c && od[2] == 1 && od[3] == out_w, VPX_RESULT_ERROR_INVALID_ARGUMENT,
                "mvn1_mean_var: output shape [%lld,%lld,%lld,%lld] does not match [%lld,%lld,1,%d]", (long long)od[0],
                (long long)od[1], (long long)od[2], (long long)od[3], (long long)N, (long long)out_c, out_w);
    VPX_REQUIRE(group_c >= 1 && C % group_c == 0, VPX_RESULT_ERROR_INVALID_ARGUMENT,
                "mvn1_mean_var: %lld channels per group does not divide %lld channels", (long long)group_c, (long long)C);
    VPX_REQUIRE(eps >= 0.f, VPX_RESULT_ERROR_INVALID_ARGUMENT, "mvn1_mean_var: eps must not be negative, got %g", (double)eps);
    const double count = (double)orig_shape[2] * (double)orig_shape[3] * (double)(across_channels ? C : group_c);
    const dim3 grid((unsigned)((N * out_c + kThreads - 1) / kThreads));
    if (out.dtype == VPX_NN_FP16)
        VPX_LAUNCH((mvn_mean_var_kernel<half_t>), grid, dim3(kThreads), 0, s, (const float*)sum.data, (half_t*)out.data, N,
                   id[1], (int)id[2], (int)id[3], out_c, out_w, across_channels ? 1 : 0, group_c, count, eps);
    else
        VPX_LAUNCH((mvn_mean_var_kernel<float>), grid, dim3(kThreads), 0, s, (const float*)sum.data, (float*)out.data, N,
                   id[1], (int)id[2], (int)id[3], out_c, out_w, across_channels ? 1 : 0, group_c, count, eps);
    return VPX_RESULT_SUCCESS;
}

template <typename TS>
static int mvn_norm_impl(const MemRef& in, const MemRef& mv, const MemRef& out, const MvnShape& sh, bool across_channels, int out_w,
                         hipStream_t s) {
    const half_t* pi = (const half_t*)in.data;
    half_t* po = (half_t*)out.data;
    const TS* pm = (const TS*)mv.data;
    const int64_t piece = kThreads * 8;
    if (!across_channels && sh.channel_minor) {
        const int64_t per_n = sh.S * sh.C;
        const int64_t pieces = (per_n + piece - 1) / piece;
        VPX_REQUIRE(sh.N * pieces < (1ll << 31) && sh.C < (1ll << 31), VPX_RESULT_ERROR_UNSUPPORTED_FEATURE,
                    "mvn1_norm: tensor exceeds the launch limit");
        const bool vec = sh.C % 8 == 0 && ((reinterpret_cast<uintptr_t>(pi) | reinterpret_cast<uintptr_t>(po)) & 15) == 0 &&
                         (reinterpret_cast<uintptr_t>(pm) & 31) == 0;
        if (vec)
            VPX_LAUNCH((mvn_norm_cminor_kernel<TS, true>), dim3((unsigned)(sh.N * pieces)), dim3(kThreads), 0, s, pi, po, pm,
                       per_n, sh.C, (int)pieces, out_w);
        else
            VPX_LAUNCH((mvn_norm_cminor_kernel<TS, false>), dim3((unsigned)(sh.N * pieces)), dim3(kThreads), 0, s, pi, po, pm,
                       per_n, sh.C, (int)pieces, out_w);
        return VPX_RESULT_SUCCESS;
    }
    const int64_t rows = across_channels ? sh.N : sh.N * sh.C;
    const int64_t run = across_channels ? sh.C * sh.S : sh.S;
    const int64_t pieces = (run + piece - 1) / piece;
    VPX_REQUIRE(rows * pieces < (1ll << 31), VPX_RESULT_ERROR_UNSUPPORTED_FEATURE, "mvn1_norm: tensor exceeds the launch limit");
    const bool aligned = run % 8 == 0 && (reinterpret_cast<uintptr_t>(pi) & 15) == 0 && (reinterpret_cast<uintptr_t>(po) & 15) == 0;
    const int64_t rows_per_n = across_channels ? 1 : sh.C;
    const int64_t out_c = across_channels ? 1 : sh.C;
    const dim3 grid((unsigned)(rows * pieces));
    if (aligned)
        VPX_LAUNCH((mvn_norm_runs_kernel<TS, true>), grid, dim3(kThreads), 0, s, pi, po, pm, run, (int)pieces, rows_per_n,
                   out_c, out_w);
    else
        VPX_LAUNCH((mvn_norm_runs_kernel<TS, false>), grid, dim3(kThreads), 0, s, pi, po, pm, run, (int)pieces, rows_per_n,
                   out_c, out_w);
    return VPX_RESULT_SUCCESS;
}

int launch_mvn_norm(const MemRef& in, const MemRef& mean_var, const MemRef& out, bool across_channels, bool normalize_variance,
                    hipStream_t s) {
    VPX_REQUIRE(in.dtype == VPX_NN_FP16 && out.dtype == VPX_NN_FP16, VPX_RESULT_ERROR_UNSUPPORTED_FEATURE,
                "mvn1_norm: only FP16 input/output is implemented, got %s -> %s", dtype_name(in.dtype), dtype_name(out.dtype));
    VPX_REQUIRE(mean_var.dtype == VPX_NN_FP16 || mean_var.dtype == VPX_NN_FP32, VPX_RESULT_ERROR_UNSUPPORTED_FEATURE,
                "mvn1_norm: statistics must be FP16 or FP32, got %s", dtype_name(mean_var.dtype));
    MvnShape sh;
    int rc = mvn_shape("mvn1_norm", in, sh);
    if (rc) return rc;
    VPX_REQUIRE(out.nd == 4 && out.order == in.order && out.compact, VPX_RESULT_ERROR_INVALID_ARGUMENT,
                "mvn1_norm: output must be a compact tensor of the input's layout");
    for (int d = 0; d < 4; d++)
        VPX_REQUIRE(in.dims[d] == out.dims[d], VPX_RESULT_ERROR_INVALID_ARGUMENT, "mvn1_norm: input and output shapes differ");
    int64_t md[4];
    rc = stats_shape("mvn1_norm", mean_var, md);
    if (rc) return rc;
    const int out_w = normalize_variance ? 2 : 1;
    VPX_REQUIRE(md[0] == sh.N && md[1] == (across_channels ? 1 : sh.C) && md[2] == 1 && md[3] == out_w,
                VPX_RESULT_ERROR_INVALID_ARGUMENT, "mvn1_norm: statistics of shape [%lld,%lld,%lld,%lld] do not match [%lld,%lld,1,%d]",
                (long long)md[0], (long long)md[1], (long long)md[2], (long long)md[3], (long long)sh.N,
                (long long)(across_channels ? 1 : sh.C), out_w);
    if (in.numel() == 0) return VPX_RESULT_SUCCESS;
    if (mean_var.dtype == VPX_NN_FP16) return mvn_norm_impl<half_t>(in, mean_var, out, sh, across_channels, out_w, s);
    return mvn_norm_impl<float>(in, mean_var, out, sh, across_channels, out_w, s);
}

namespace {

// How an optional operand varies along a row whose reduced dimensions have element strides `stride`:
// 1 = laid out like the contiguous row, 0 = constant along the row, -1 = neither.
int along_row(bool present, const int32_t* rdim, const int64_t* stride, int nr) {
    if (!present) return 0;
    bool constant = true, full = true;
    int64_t expect = 1;
    for (int d = 0; d < nr; d++) {
        if (stride[d] != 0) constant = false;
        if (stride[d] != expect) full = false;
        expect *= rdim[d];
    }
    return constant ? 0 : (full ? 1 : -1);
}

bool aligned_rows(const void* p, const int64_t* kstride, int nk) {
    if (reinterpret_cast<uintptr_t>(p) & 15) return false;
    for (int d = 0; d < nk; d++)
        if (kstride[d] % 8 != 0) return false;
    return true;
}

}  // namespace

int launch_mvn6(const MemRef& in, const MemRef* scale, const MemRef* bias, const MemRef& out, bool normalize_variance, int eps_mode,
                float eps, const int64_t* mem_axes, int n_axes, hipStream_t s) {
    VPX_REQUIRE(in.dtype == VPX_NN_FP16 && out.dtype == VPX_NN_FP16, VPX_RESULT_ERROR_UNSUPPORTED_FEATURE,
                "mvn6: only FP16 input/output is implemented, got %s -> %s", dtype_name(in.dtype), dtype_name(out.dtype));
    VPX_REQUIRE(in.nd == out.nd && in.nd <= kMaxDims, VPX_RESULT_ERROR_INVALID_ARGUMENT, "mvn6: ranks %d / %d (at most %d)", in.nd,
                out.nd, kMaxDims);
    for (int d = 0; d < in.nd; d++)
        VPX_REQUIRE(in.dims[d] == out.dims[d], VPX_RESULT_ERROR_INVALID_ARGUMENT, "mvn6: input and output shapes differ");
    VPX_REQUIRE(eps_mode == 0 || eps_mode == 1, VPX_RESULT_ERROR_INVALID_ARGUMENT, "mvn6: unknown eps mode %d", eps_mode);
    VPX_REQUIRE(eps >= 0.f, VPX_RESULT_ERROR_INVALID_ARGUMENT, "mvn6: eps must not be negative, got %g", (double)eps);
    VPX_REQUIRE(n_axes >= 1 && n_axes <= in.nd, VPX_RESULT_ERROR_INVALID_ARGUMENT, "mvn6: %d axes for rank %d", n_axes, in.nd);
    bool reduced[kMaxDims] = {};
    for (int i = 0; i < n_axes; i++) {
        VPX_REQUIRE(mem_axes[i] >= 0 && mem_axes[i] < in.nd && !reduced[mem_axes[i]], VPX_RESULT_ERROR_INVALID_ARGUMENT,
                    "mvn6: axis %lld is outside rank %d or repeated", (long long)mem_axes[i], in.nd);
        reduced[mem_axes[i]] = true;
    }
    const MemRef* extra[2] = {scale, bias};
    for (const MemRef* m : extra) {
        if (!m) continue;
        VPX_REQUIRE(m->dtype == VPX_NN_FP16 && m->nd == in.nd, VPX_RESULT_ERROR_INVALID_ARGUMENT,
                    "mvn6: scale / bias must be FP16 tensors of the input's rank");
        for (int d = 0; d < in.nd; d++)
            VPX_REQUIRE(m->dims[d] == in.dims[d] || m->dims[d] == 1, VPX_RESULT_ERROR_INVALID_ARGUMENT,
                        "mvn6: scale / bias dimension %d is %lld, input has %lld", d, (long long)m->dims[d], (long long)in.dims[d]);
    }
    if (in.numel() == 0) return VPX_RESULT_SUCCESS;

    Mvn6Geom g{};
    int64_t row_len = 1;
    g.rows = 1;
    bool innermost = true;   // the reduced dimensions are the innermost ones
    bool inner_kept = false;  // the innermost dimension (of more than one element) is kept
    for (int d = 0; d < in.nd; d++) {
        if (in.dims[d] == 1) continue;
        if (g.nk + g.nr == 0) inner_kept = !reduced[d];
        const int64_t ssc = scale && scale->dims[d] != 1 ? scale->strides[d] : 0;
        const int64_t sbi = bias && bias->dims[d] != 1 ? bias->strides[d] : 0;
        if (reduced[d]) {
            if (g.nk > 0) innermost = false;
            g.rdim[g.nr] = (int32_t)in.dims[d];
            g.r_in[g.nr] = in.strides[d];
            g.r_out[g.nr] = out.strides[d];
            g.r_sc[g.nr] = ssc;
            g.r_bi[g.nr] = sbi;
            g.nr++;
            row_len *= in.dims[d];
        } else {
            g.kdim[g.nk] = (int32_t)in.dims[d];
            g.k_in[g.nk] = in.strides[d];
            g.k_out[g.nk] = out.strides[d];
            g.k_sc[g.nk] = ssc;
            g.k_bi[g.nk] = sbi;
            g.nk++;
            g.rows *= in.dims[d];
        }
    }
    // Kept dimensions that every operand walks as one (stride of the outer = stride x extent of the inner) fold
    // into one, so a packed tensor's rows are found without a division.
    for (int d = 0; d + 1 < g.nk;) {
        const int64_t e = g.kdim[d];
        if (g.k_in[d + 1] == g.k_in[d] * e && g.k_out[d + 1] == g.k_out[d] * e && g.k_sc[d + 1] == g.k_sc[d] * e &&
            g.k_bi[d + 1] == g.k_bi[d] * e && e * g.kdim[d + 1] < (1ll << 31)) {
            g.kdim[d] = (int32_t)(e * g.kdim[d + 1]);
            for (int k = d + 1; k + 1 < g.nk; k++) {
                g.kdim[k] = g.kdim[k + 1];
                g.k_in[k] = g.k_in[k + 1];
                g.k_out[k] = g.k_out[k + 1];
                g.k_sc[k] = g.k_sc[k + 1];
                g.k_bi[k] = g.k_bi[k + 1];
            }
            g.nk--;
        } else {
            d++;
        }
    }
    VPX_REQUIRE(row_len < (1ll << 31) && g.rows < (1ll << 31), VPX_RESULT_ERROR_UNSUPPORTED_FEATURE,
                "mvn6: %lld rows of %lld elements exceed the launch limit", (long long)g.rows, (long long)row_len);
    g.row_len = (uint32_t)row_len;
    const half_t* pi = (const half_t*)in.data;
    half_t* po = (half_t*)out.data;
    const half_t* ps = scale ? (const half_t*)scale->data : nullptr;
    const half_t* pb = bias ? (const half_t*)bias->data : nullptr;
    const int nv = normalize_variance ? 1 : 0;

    // Long contiguous rows of a compact tensor, eps inside the root, no scale or bias: the chunked two-launch
    // scheme of mvn1 (a row is a group there).
    if (innermost && row_len > kMvn6MaxRegRow && !scale && !bias && in.compact && out.compact && lds_groups_ok(g.rows, row_len))
        return launch_lds_groups(pi, po, g.rows, row_len, nv, eps_mode, eps, s);
    if (innermost && row_len > kMvn6MaxRegRow && !scale && !bias && eps_mode == 0 && in.compact && out.compact) {
        const bool aligned = row_len % 8 == 0 && ((reinterpret_cast<uintptr_t>(pi) | reinterpret_cast<uintptr_t>(po)) & 15) == 0;
        return aligned ? launch_groups<true>(pi, po, g.rows, row_len, nv, eps, s) : launch_groups<false>(pi, po, g.rows, row_len, nv, eps, s);
    }
    // Short contiguous rows whose length is not a multiple of eight (7 x 7 planes, rows of 100): runs of whole rows
    // per workgroup, as for mvn1's short groups.
    if (innermost && !scale && !bias && in.compact && out.compact && tiny_groups_ok(pi, po, g.rows, row_len))
        return launch_tiny_groups(pi, po, g.rows, row_len, nv, eps_mode, eps, s);
    if (innermost && row_len % 8 != 0 && !scale && !bias && in.compact && out.compact && small_groups_ok(pi, po, g.rows, row_len))
        return launch_small_groups(pi, po, g.rows, row_len, nv, eps_mode, eps, s);
    bool fast = innermost && row_len >= 8 && row_len <= kMvn6MaxRegRow, words = false;
    if (fast) {
        fast = along_row(true, g.rdim, g.r_in, g.nr) == 1 && along_row(true, g.rdim, g.r_out, g.nr) == 1;
        g.sc_along_row = along_row(scale != nullptr, g.rdim, g.r_sc, g.nr);
        g.bi_along_row = along_row(bias != nullptr, g.rdim, g.r_bi, g.nr);
        fast = fast && g.sc_along_row >= 0 && g.bi_along_row >= 0;
        words = row_len % 8 == 0 && aligned_rows(pi, g.k_in, g.nk) && aligned_rows(po, g.k_out, g.nk);
        if (words && scale && g.sc_along_row) words = aligned_rows(ps, g.k_sc, g.nk);
        if (words && bias && g.bi_along_row) words = aligned_rows(pb, g.k_bi, g.nk);
    }
    if (fast) {
        return launch_rows(pi, po, ps, pb, g, words, nv, eps_mode, eps, s);
    } else if (inner_kept && g.k_in[0] == 1 && g.k_out[0] == 1) {
        const int64_t outer = g.rows / g.kdim[0];
        const auto blocks = [&](int p) { return outer * ((g.kdim[0] + p - 1) / p); };
        if (blocks(64) >= 512)
            VPX_LAUNCH(mvn6_inner_kernel<64>, dim3((unsigned)blocks(64)), dim3(kThreads), 0, s, pi, po, ps, pb, g, nv, eps_mode, eps);
        else if (blocks(32) >= 512)
            VPX_LAUNCH(mvn6_inner_kernel<32>, dim3((unsigned)blocks(32)), dim3(kThreads), 0, s, pi, po, ps, pb, g, nv, eps_mode, eps);
        else
            VPX_LAUNCH(mvn6_inner_kernel<16>, dim3((unsigned)blocks(16)), dim3(kThreads), 0, s, pi, po, ps, pb, g, nv, eps_mode, eps);
    } else {
        VPX_LAUNCH(mvn6_generic_kernel, dim3((unsigned)g.rows), dim3(kThreads), 0, s, pi, po, ps, pb, g, nv, eps_mode, eps);
    }
    return VPX_RESULT_SUCCESS;
}

}  // namespace vpx
