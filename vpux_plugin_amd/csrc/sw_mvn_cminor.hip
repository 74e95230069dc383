// ACT-SHAVE `mvn1` with per-channel statistics on a channel-minor layout (NHWC), in one launch with the tensor in registers.
//
// What bounds it is memory: the sums need every value before the first result can be written.  Sums, a fold of the partial
// sums and a second pass over the tensor are three launches and two reads (58 us for [16,112,112,256], of which the fold
// alone 9; 11 us for tensors of a few hundred KB, all of it launches).  Here a workgroup keeps its part of the tensor in
// registers -- 512 lanes of up to 50 words of 128 bits, 400 KB of the 512 KB a compute unit has -- between the sums and the
// normalisation, and the workgroups that share a channel exchange their partial sums inside the launch.
//
// Deal.  A lane owns one word of a row and walks rows, so each of its eight values belongs to one channel throughout and its
// sums are eight registers.  Octets: a row is a position, a workgroup takes `ob` adjacent octets of its channels (eight of them are
// 128 bytes); of a channel count that is no multiple of eight the last octet begins inside the one before, both hold those channels
// and store them alike.  Rows: R positions are a row of `words` whole 128-bit words, R the least count that makes it so (1 for a multiple of
// 8 channels, else 2, 4 or 8), and a workgroup takes whole rows, whose sums fold through LDS; they serve fewer than eight channels, odd channel
// counts in place, and where they cost less.  (Octets of odd channel counts against rows or the three launches, us: [1,15,10,349] 4.0 / 11.6,
// [7,10,14,359] 4.2 / 11.5, [3,141,122,426] 21 / 138, [2,211,167,511] 36 / 238; 250 drawn tensors of them take 0.58 of the time, 500 of whole octets 0.92.)
#include "vpx_common.h"

namespace vpx {

namespace {

typedef _Float16 half_t;
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef half_t halfx8 __attribute__((ext_vector_type(8)));
typedef u32x4 __attribute__((aligned(2))) u32x4_any;  // images of an odd number of values start off the words

constexpr int kT = 512;
constexpr int kMostWords = 50;        // words per lane: 200 of the 256 registers of a lane at two wavefronts per SIMD
constexpr int kAhead = 12;            // words per lane under way: 96 KB a compute unit
constexpr int kMostGroups = 128;      // groups of workgroups that exchange partial sums
constexpr int kMostParts = 256;       // workgroups of a group
constexpr int kCountStride = 4;       // words between launch counts
constexpr int kMostRowGroups = 16;    // the same for the form that deals whole rows, with more records each
constexpr int kMostRowRecords = 16384;
constexpr int kMostRecords = 2048;    // partial sums a workgroup reads from the workgroups it shares channels with: four per lane

struct Geom {
    uint32_t C, S, per_n;             // channels, positions and values of an image
    uint32_t R, words, rows;          // positions and words of a row, rows of an image (the last one may be cut short)
    uint32_t pitch;                   // values from row to row
    uint32_t ob, ob_log, nb;          // words a workgroup takes of each row, and how many such blocks make the row
    uint32_t parts, rows_per_part;    // workgroups that share a block's rows
    uint32_t units;                   // images x parts
};

// A partial sum in memory: two 64-bit words, {value, tag} each, written and read as one access that goes through to memory
// (agent scope), so that the tag vouches for the value beside it.
struct __attribute__((aligned(16))) Tagged {
    unsigned long long sum, sq;
};
static_assert(kSyncCminor + sizeof(unsigned) * kCountStride * kMostParts * (kMostGroups + kMostRowGroups) +
                      sizeof(Tagged) * ((size_t)kMostGroups * kMostRecords + (size_t)kMostRowGroups * kMostRowRecords) <=
                  kSyncBytes, "sync area layout");
__device__ __forceinline__ unsigned long long tagged(float v, unsigned tag) {
    return (unsigned long long)__builtin_bit_cast(unsigned, v) | ((unsigned long long)tag << 32);
}
__device__ __forceinline__ float untagged(unsigned long long w) {
    return __builtin_bit_cast(float, (unsigned)w);
}

// The result is the fp32 product rounded again; the empty asm keeps it from being folded into one mixed-precision multiply.
__device__ __forceinline__ half_t round_f16(float v) {
    asm volatile("" : "+v"(v));
    return (half_t)v;
}

// Tags.  The workgroups that share a block of channels of an image are a group with launch counts and a run of records of
// its own, so that a record only ever carries tags of its own group's counts; a launch's tag is the count + 1, and it is the
// device that counts, as a replayed graph needs.  Every workgroup has counts of its own (the group's kMostParts are dealt out in
// turn, and a launch moves all of them on, however many workgroups it has): nobody else writes them during a launch, so a workgroup finds
// the launch's tag however late it starts, and no record of an earlier launch carries it.  No read-modify-write is involved:
// 192 arrivals at one counter took 1.5 us.
// The wait is bounded: a workgroup whose partners do not show up in time (they are not resident: the device is shared)
// computes missing partial sums with the same arithmetic and publishes them for their owners and for everyone else, part by
// part, each time one that nobody has published yet.  So the result is the same bits, the missing parts are computed about
// once among those that wait, whoever starts later finds its group complete, and every wave exits: a workgroup computes a
// part at most once.  (Each computing all parts for itself took 6.5 ms for [1,448,448,256] beside a launch that held 224 of 256
// compute units; now 1.4.)
//
// How the sums meet.  With OCTETS ob is a power of two: lanes that own the same word are ob apart
// in a wavefront and add up by rotations and swaps, and so do a channel's partial sums of other workgroups; eight wavefronts
// meet in LDS.  (A fold through LDS alone, group after group of lanes, took 4 us of a small tensor's 9.)  Rows of several
// positions, whose channels lie anywhere in the words, fold through LDS.
template <int CTRL>
__device__ __forceinline__ float dppf(float v) {
    const int i = __builtin_bit_cast(int, v);
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(i, i, CTRL, 0xf, 0xf, true));
}
// sums over the lanes of a row of 16 that are a multiple of `stride` (a power of two, uniform) apart, N values at a time
template <int N>
__device__ __forceinline__ void stride_sums(float (&v)[N], uint32_t stride) {
#define VPX_STEP(S, CTRL)                                  \
    if (stride <= S) {                                     \
        _Pragma("unroll") for (int k = 0; k < N; k++) v[k] += dppf<CTRL>(v[k]); \
    }
    VPX_STEP(1, 0x121)  // rotations
    VPX_STEP(2, 0x122)
    VPX_STEP(4, 0x124)
    VPX_STEP(8, 0x128)
#undef VPX_STEP
}
// D = 32: a + its other half's in the lower half of the wavefront, b + its other half's in the upper one; D = 16: the same
// of the even and the odd rows
template <int D>
__device__ __forceinline__ float swap_add(float a, float b) {
    // (this compiler's builtins for the two hand back the first register twice; the waits are those it puts around them)
    if (D == 32) asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
    else asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
    return a + b;
}

//
// Results are written past the caches (a plain store of [16,112,112,256] costs 8 of its 49 us), except (kShort) in runs of 16 or 32 bytes and in runs
// that end within lines, which the neighbouring workgroups' runs complete to lines there: of 700 drawn tensors, those with such runs that hold 12 M
// values or more take 0.60 ... 0.88 of the time of stores past the caches.  A kernel of its own, because one branch with either store is compiled
// to plain ones.
enum Form { kRows, kOctets, kShort };
template <int V, Form FORM>
__global__ __launch_bounds__(kT) void mvn_cminor_resident(const half_t* __restrict__ in, half_t* __restrict__ out, Geom g, unsigned* sync,
                                                          int normalize_variance, float eps, unsigned long long spin_ticks) {
    constexpr bool OCTETS = FORM != kRows;
    __shared__ float2 red[OCTETS ? 8 * 64 : kT * 8];  // [wavefront or slot][column] sums
    __shared__ float2 folded[OCTETS ? 1 : kT];             // [group of lanes][channel]
    __shared__ float s_mean[OCTETS ? 64 : kT], s_inv[OCTETS ? 64 : kT];
    __shared__ float2 s_tail[8];
    __shared__ unsigned s_tag, s_pick;
    __shared__ unsigned char helped[kMostParts];

    // the blocks of one part are neighbours on one die, whose L2 then holds the lines they share
    const uint32_t seq = blockIdx.x >> 3, b = seq % g.nb, u = seq / g.nb * 8 + (blockIdx.x & 7);
    if (u >= g.units) return;
    const uint32_t n = u / g.parts, part = u % g.parts;
    const int t = (int)threadIdx.x;
    const half_t* img = in + (int64_t)n * g.per_n;
    half_t* oimg = out + (int64_t)n * g.per_n;
    asm volatile("" ::"s"(out), "s"(sync), "s"(g.S), "s"(g.C), "s"(g.per_n), "s"(g.rows), "s"(normalize_variance), "s"(eps));  // (one trip to the arguments)
    const uint32_t w0 = b * g.ob, nw = g.words - w0 < g.ob ? g.words - w0 : g.ob;
    // OCTETS: a last block of fewer words leaves lanes idle
    const uint32_t slots = OCTETS ? kT >> g.ob_log : kT / nw, slot = OCTETS ? (uint32_t)t >> g.ob_log : (uint32_t)t / nw;
    const uint32_t wl = OCTETS ? (uint32_t)t & (g.ob - 1) : (uint32_t)t - slot * nw;
    const bool active = OCTETS ? wl < nw : slot < slots;
    // first value of a word in its row; OCTETS: a last word that is not whole takes the last eight channels, which the word before has in part
    const auto word_at = [&](uint32_t word) { return OCTETS && word * 8 + 8 > g.C ? g.C - 8 : word * 8; };
    const uint32_t at = word_at(OCTETS && !active ? w0 : w0 + wl);
    const uint32_t cols = OCTETS ? g.ob * 8 : nw * 8, nch = OCTETS ? cols : g.C, ch0 = w0 * 8;  // (R > 1: ch0 is 0)
    const uint32_t G = kT / nch, gi = (uint32_t)t / nch, c = (uint32_t)t - gi * nch;
    // of the channel whose statistics this lane finishes
    const half_t own_first = img[OCTETS ? ((uint32_t)t < nch && w0 + t / 8 < g.words ? word_at(w0 + t / 8) + t % 8 : 0) : (uint32_t)t < nch && ch0 + t < g.C ? ch0 + t : 0];
    const uint32_t rem = OCTETS ? 0 : g.per_n % 8;  // values of the image's last, partial word
    const uint32_t group = OCTETS ? n * g.nb + b : kMostGroups + n;
    // this workgroup's launch counts: every parts-th of the group's, from its own place on
    unsigned* counts = sync + (size_t)group * (kMostParts * kCountStride);
    Tagged* records = reinterpret_cast<Tagged*>(sync + (size_t)(kMostGroups + kMostRowGroups) * (kMostParts * kCountStride)) +
                      (OCTETS ? (size_t)group * kMostRecords : (size_t)kMostGroups * kMostRecords + (size_t)n * kMostRowRecords);
    // sums are of x - x[first position of the channel]: no cancellation where a channel's mean is far from zero
    halfx8 first;
    if (OCTETS) {
        first = __builtin_bit_cast(halfx8, *reinterpret_cast<const u32x4_any*>(img + at));
    } else {
#pragma unroll
        for (int k = 0; k < 8; k++) first[k] = img[(at + k) % g.C];
    }
    u32x4 q[V];
    uint32_t have = 0;  // words of this lane
    // The sums of part p over channel t, for the lanes below nch; its words stay in q.
    const auto part_sums = [&](uint32_t p, auto behind_first) __attribute__((always_inline)) -> float2 {
        const uint32_t r0 = p * g.rows_per_part, r1 = r0 + g.rows_per_part < g.rows ? r0 + g.rows_per_part : g.rows;
        const uint32_t r = r0 + slot;
        have = active && r < r1 ? (r1 - r + slots - 1) / slots : 0;
        uint32_t f = r * g.pitch + at;
        const uint32_t step = slots * g.pitch;
        // the last row's words past the image, and the partial one, are not among a lane's words
        if (have && (uint64_t)f + (uint64_t)(have - 1) * step + 8 > g.per_n) have--;
        // No branch around a load (lanes without a word read the image's first one), and kAhead of them under way while
        // the words before are summed: all V at once, 400 KB a compute unit, reach the memory in an order that costs a
        // third of its rate.
        const auto load = [&](int j) {
            q[j] = *reinterpret_cast<const u32x4_any*>(img + ((uint32_t)j < have ? f : 0));
            f += step;
            asm volatile("" : "+v"(f));  // one running offset, not V of them
        };
#pragma unroll
        for (int j = 0; j < (V < kAhead ? V : kAhead); j++) load(j);
        behind_first();
        float sum[8], sq[8], shift[8];
#pragma unroll
        for (int k = 0; k < 8; k++) {
            sum[k] = sq[k] = 0.f;
            shift[k] = (float)first[k];
        }
#pragma unroll
        for (int j = 0; j < V; j++) {
            // word after word: the values of V words at once are more than the registers hold
            asm volatile("" : "+v"(q[j]), "+v"(sum[0]), "+v"(sum[1]), "+v"(sum[2]), "+v"(sum[3]), "+v"(sum[4]), "+v"(sum[5]), "+v"(sum[6]),
                         "+v"(sum[7]));
            asm volatile("" : "+v"(sq[0]), "+v"(sq[1]), "+v"(sq[2]), "+v"(sq[3]), "+v"(sq[4]), "+v"(sq[5]), "+v"(sq[6]), "+v"(sq[7]));
            if (j + kAhead < V) load(j + kAhead);
            if ((uint32_t)j >= have) q[j] = __builtin_bit_cast(u32x4, first);  // adds nothing to the shifted sums
            const halfx8 h = __builtin_bit_cast(halfx8, q[j]);
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const float x = (float)h[k] - shift[k];
                sum[k] += x;
                sq[k] = __builtin_fmaf(x, x, sq[k]);
            }
        }
        if (OCTETS) {
            // across the halves and the rows of 16 lanes two registers become one: the odd one's sums end up in the
            // upper half, in the odd rows
            float s4[4], q4[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                s4[i] = swap_add<32>(sum[2 * i], sum[2 * i + 1]);
                q4[i] = swap_add<32>(sq[2 * i], sq[2 * i + 1]);
            }
            float v[4];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                v[i] = swap_add<16>(s4[2 * i], s4[2 * i + 1]);
                v[2 + i] = swap_add<16>(q4[2 * i], q4[2 * i + 1]);
            }
            stride_sums(v, g.ob);
            __syncthreads();  // the last use of red is over
            if ((uint32_t)(t & 15) < g.ob) {
                const int k = (t & 16 ? 2 : 0) + (t & 32 ? 1 : 0);
                red[(t >> 6) * 64 + wl * 8 + k] = float2{v[0], v[2]};
                red[(t >> 6) * 64 + wl * 8 + k + 4] = float2{v[1], v[3]};
            }
            __syncthreads();
            float2 a{0.f, 0.f};
            if ((uint32_t)t < nch) {
#pragma unroll
                for (int k = 0; k < 8; k++) {
                    const float2 v = red[k * 64 + t];
                    a.x += v.x;
                    a.y += v.y;
                }
            }
            return a;
        }
        __syncthreads();  // the last use of red and folded is over
        if (active) {
#pragma unroll
            for (int k = 0; k < 8; k++) red[slot * cols + wl * 8 + k] = float2{sum[k], sq[k]};
        }
        if ((uint32_t)t < rem && p == g.parts - 1) {
            const uint32_t f = g.per_n - rem + t;
            const float x = (float)img[f] - (float)img[f % g.C];
            s_tail[t] = float2{x, x * x};
        }
        __syncthreads();
        if (gi < G) {
            float2 a{0.f, 0.f};
            for (uint32_t m = 0; m < g.R; m++)
#pragma unroll 4
                for (uint32_t s = gi; s < slots; s += G) {
                    const float2 v = red[s * cols + c + m * g.C];
                    a.x += v.x;
                    a.y += v.y;
                }
            if (gi == 0 && p == g.parts - 1)
                for (uint32_t e = 0; e < rem; e++)
                    if ((g.per_n - rem + e) % g.C == c) {
                        a.x += s_tail[e].x;
                        a.y += s_tail[e].y;
                    }
            folded[t] = a;
        }
        __syncthreads();
        float2 a{0.f, 0.f};
        if ((uint32_t)t < nch)
#pragma unroll 8
            for (uint32_t k = 0; k < G; k++) {
                a.x += folded[k * nch + t].x;
                a.y += folded[k * nch + t].y;
            }
        return a;
    };

    // The launch's tag, asked for by one lane behind its first words (in front of them, worked with at once, it was a trip to memory before the first
    // load) and dealt out behind the sums: workgroups that publish later for it, but all of whose wavefronts start to poll together, are ahead of
    // those where seven poll while the first sums up (all lanes asking, no barrier: [8,69,106,64] 8.9 us, so 8.4).
    unsigned counted = 0;
    const auto ask_tag = [&]() __attribute__((always_inline)) {
        if (g.parts > 1 && t == 0) counted = __hip_atomic_load(counts + part * kCountStride, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    float2 total = part_sums(part, ask_tag);
    if (g.parts > 1) {
        asm volatile("" : "+v"(counted));  // (what is done with it stays here)
        if (t == 0) s_tag = counted + 1u == 0u ? 1u : counted + 1u;
        __syncthreads();
        const unsigned tag = s_tag;
        const uint32_t count = g.parts * nch;
        const auto publish = [&](uint32_t p, float2 v) {
            if ((uint32_t)t < nch) {
                __hip_atomic_store(&records[p * nch + t].sum, tagged(v.x, tag), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(&records[p * nch + t].sq, tagged(v.y, tag), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        };
        publish(part, total);
        // (here and not at the end: their way to memory then ends under the wait, 1.2 of 43 us at [16,112,112,256])
        if (part + t * g.parts < kMostParts)
            __hip_atomic_store(counts + (part + t * g.parts) * kCountStride, tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const unsigned long long began = wall_clock64();
        const auto poll = [&](uint32_t i, unsigned long long& rs, unsigned long long& rq) {
            rs = __hip_atomic_load(&records[i].sum, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            rq = __hip_atomic_load(&records[i].sq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return (unsigned)(rs >> 32) == tag && (unsigned)(rq >> 32) == tag;
        };
        constexpr int kAtOnce = 4;
        static_assert(kMostRecords == kAtOnce * kT, "records a workgroup reads at once");
        // adds up this lane's records in `a`; false if one of them was not this launch's when the wait ran out
        float2 a;
        const auto collect = [&](bool waits) {
            a = float2{0.f, 0.f};
            bool ready = true;
            if (OCTETS) {
                // a lane's records are all of channel t % nch
                unsigned long long rs[kAtOnce], rq[kAtOnce];
                do {
                    ready = true;
#pragma unroll
                    for (int k = 0; k < kAtOnce; k++)
                        if ((uint32_t)(k * kT + t) < count) ready &= poll(k * kT + t, rs[k], rq[k]);
                } while (waits && __builtin_amdgcn_ballot_w64(!ready) != 0 && wall_clock64() - began < spin_ticks);
#pragma unroll
                for (int k = 0; k < kAtOnce; k++)
                    if ((uint32_t)(k * kT + t) < count) {
                        a.x += untagged(rs[k]);
                        a.y += untagged(rq[k]);
                    }
            } else {
                // lane (gi, c) adds up channel c of the parts gi, gi + G, ...
                constexpr int kRowsAtOnce = V >= 32 ? 4 : 12;  // (more would not leave the words their registers)
                for (uint32_t p = gi; p < g.parts && gi < G && ready; p += kRowsAtOnce * G) {
                    unsigned long long rs[kRowsAtOnce], rq[kRowsAtOnce];
                    do {
                        ready = true;
#pragma unroll
                        for (int k = 0; k < kRowsAtOnce; k++) ready &= poll((p + k * G < g.parts ? p + k * G : p) * nch + c, rs[k], rq[k]);
                    } while (waits && !ready && wall_clock64() - began < spin_ticks);
#pragma unroll
                    for (int k = 0; k < kRowsAtOnce; k++)
                        if (p + k * G < g.parts) {
                            a.x += untagged(rs[k]);
                            a.y += untagged(rq[k]);
                        }
                }
            }
            return ready;
        };
        if (!__syncthreads_and(collect(true))) {
            if (t < kMostParts) helped[t] = 0;
            for (uint32_t k = 0; k < g.parts; k++) {
                // of the parts that nobody has published: the first one from a place of this workgroup's own on
                const uint32_t from = (part * 2654435761u >> 8) % g.parts;
                if (t == 0) s_pick = g.parts;
                __syncthreads();
                for (uint32_t i = t; i < count; i += kT) {
                    unsigned long long rs, rq;
                    const uint32_t p = i / nch;
                    if (!poll(i, rs, rq) && !helped[p]) atomicMin(&s_pick, (p + g.parts - from) % g.parts);
                }
                __syncthreads();
                const uint32_t pick = s_pick, p = (from + pick) % g.parts;
                if (pick == g.parts) break;
                publish(p, part_sums(p, [] {}));
                __threadfence();
                if (t == 0) helped[p] = 1;
                __syncthreads();
            }
            collect(false);
            part_sums(part, [] {});  // its own words again
            __syncthreads();
        }
        if (OCTETS) {
            float both[2] = {a.x, a.y};
            stride_sums(both, nch);
            if (nch <= 16) {
                both[0] += __shfl_xor(both[0], 16);
                both[1] += __shfl_xor(both[1], 16);
            }
            if (nch <= 32) {
                both[0] += __shfl_xor(both[0], 32);
                both[1] += __shfl_xor(both[1], 32);
            }
            if ((uint32_t)(t & 63) < nch) red[(t >> 6) * 64 + (t & 63)] = float2{both[0], both[1]};  // (read last before the records were published)
            __syncthreads();
            total = float2{0.f, 0.f};
            if ((uint32_t)t < nch) {
#pragma unroll
                for (int k = 0; k < 8; k++) {
                    total.x += red[k * 64 + t].x;
                    total.y += red[k * 64 + t].y;
                }
            }
        } else {
            folded[t] = a;
            __syncthreads();
            total = float2{0.f, 0.f};
            if ((uint32_t)t < nch) {
#pragma unroll 8
                for (uint32_t k = 0; k < G; k++) {
                    total.x += folded[k * nch + t].x;
                    total.y += folded[k * nch + t].y;
                }
            }
        }
    }
    if ((uint32_t)t < nch) {
        const float count = (float)g.S, m = total.x / count, var = fmaxf(total.y / count - m * m, 0.f);
        s_mean[t] = (float)own_first + m;
        s_inv[t] = normalize_variance ? 1.0f / __builtin_sqrtf(var + eps) : 1.0f;
    }
    __syncthreads();
    float mean[8], inv[8];
#pragma unroll
    for (int k = 0; k < 8; k++) {
        uint32_t ch = wl * 8 + k;
        if (!OCTETS) ch %= g.C;
        mean[k] = s_mean[ch];
        inv[k] = s_inv[ch];
    }
    uint32_t f = (part * g.rows_per_part + slot) * g.pitch + at;
    const uint32_t step = slots * g.pitch;
#pragma unroll
    for (int j = 0; j < V; j++) {
        asm volatile("" : "+v"(q[j]), "+v"(f));  // (values converted for the sums are not kept: twice the registers)
        if ((uint32_t)j < have) {
            const halfx8 h = __builtin_bit_cast(halfx8, q[j]);
            halfx8 y;
#pragma unroll
            for (int k = 0; k < 8; k++) y[k] = round_f16(((float)h[k] - mean[k]) * inv[k]);
            if constexpr (FORM == kShort) *reinterpret_cast<u32x4_any*>(oimg + f) = __builtin_bit_cast(u32x4, y);
            else __builtin_nontemporal_store(__builtin_bit_cast(u32x4, y), reinterpret_cast<u32x4_any*>(oimg + f));
        }
        f += step;
    }
    if ((uint32_t)t < rem && part == g.parts - 1) {
        const uint32_t f = g.per_n - rem + t, ch = f % g.C;
        oimg[f] = round_f16(((float)img[f] - s_mean[ch]) * s_inv[ch]);
    }
}

uint32_t ceil_div(uint64_t a, uint64_t b) {
    return (uint32_t)((a + b - 1) / b);
}

}  // namespace

// Microseconds of a form: the launch, a word of a lane, the way of the fullest die's share of the tensor (of eight: a unit's workgroups are on one) at the
// rate of a copy (runs of 16 ... 64 bytes cross the caches several times), more of both where that die is dealt more workgroups than it has compute units
// (1.3 ... 1.8 times where a lane holds more than 16 words), a partial sum that is exchanged, a channel of the fold through LDS.  Fitted to 1095 drawn
// tensors under each form that serves them (8500 times, median error 4 %, one tenth beyond 8 to 20): the least of these takes 1.2 % more than the best
// form of each; without the crowding, 4.6 %.  The kernels that run take 0.87 of that alone with up to 16 words a lane, 0.94 with an exchange and 1.04 in rows (medians of 4500
// tensors).  Of 6400 drawn ones 60 are more than 3 % slower than under the rule that knew no runs of 16 or 32 bytes with more than 16 words, 1.2 us at
// most but for [8,54,54,544], 12.4 / 15.4; unscaled it would be twice as many.
struct FormTime {
    float launch, word, copy, crowded, exchange, channel;
};
// by whether workgroups exchange sums, octets a workgroup takes of each position (1, 2, 4, 8), whether C is no multiple of 8, one of 8, or one of
// the workgroup's run (every run of a position is then as far from a line as the first one)
constexpr FormTime kOctetTime[2][4][3] = {{{{3.27f, 0.425f, 1.80f, 0, 0, 0}, {3.27f, 0.274f, 1.73f, 0, 0, 0}, {3.27f, 0.274f, 1.73f, 0, 0, 0}},
                                           {{3.29f, 0.423f, 0.90f, 0.48f, 0, 0}, {3.32f, 0.295f, 1.03f, 0, 0, 0}, {3.26f, 0.265f, 0.86f, 0.13f, 0, 0}},
                                           {{3.40f, 0.318f, 0.66f, 0, 0, 0}, {3.23f, 0.273f, 0.60f, 0, 0, 0}, {3.27f, 0.249f, 0.48f, 0, 0, 0}},
                                           {{3.30f, 0.312f, 0.47f, 0, 0, 0}, {3.20f, 0.276f, 0.49f, 0, 0, 0}, {3.34f, 0.265f, 0.14f, 0, 0, 0}}},
                                          {{{2.56f, 1.143f, 1.09f, 0.75f, 0, 0}, {3.72f, 0.652f, 1.27f, 0.47f, 0, 0}, {3.72f, 0.652f, 1.27f, 0.47f, 0, 0}},
                                           {{3.98f, 0.598f, 0.94f, 2.15f, 0.50e-3f, 0}, {4.12f, 0.562f, 0.79f, 2.31f, 0, 0}, {4.45f, 0.376f, 0.82f, 0.78f, 0.59e-3f, 0}},
                                           {{4.49f, 0.389f, 0.78f, 1.71f, 0.72e-3f, 0}, {4.60f, 0.285f, 0.75f, 1.23f, 0.84e-3f, 0}, {4.28f, 0.393f, 0.52f, 1.14f, 0.63e-3f, 0}},
                                           {{4.72f, 0.284f, 0.78f, 4.89f, 0.78e-3f, 0}, {4.73f, 0.228f, 0.75f, 4.53f, 0.76e-3f, 0}, {4.81f, 0.211f, 0.60f, 1.30f, 0.59e-3f, 0}}}};
constexpr FormTime kRowTime[2] = {{4.98f, 0.257f, 0.46f, 0, 2.30e-3f, 0}, {8.27f, 0.146f, 0.66f, 0, 0.26e-3f, 2.94e-3f}};

// Takes the launch when the tensor fits the registers of one workgroup per compute unit; *done is set when it has.
int launch_mvn_cminor_resident(const void* in, void* out, int64_t N, int64_t S, int64_t C, int nv, float eps, hipStream_t s, bool* done) {
    *done = false;
    const int mode = tuning_mvn_fused();  // 0: never, 1: default, 2: no waiting (every workgroup computes all partial sums)
    int cus = 0;
    int rc = device_compute_units(&cus);
    if (rc) return rc;
    if (mode == 0 || S * C < 8 || S * C >= (1ll << 31) || N >= (1 << 16)) return VPX_RESULT_SUCCESS;
    Geom best{};
    uint32_t best_v = 0;
    float best_cost = 0.f;
    bool best_rows = false;
    const uint32_t R = C % 8 == 0 ? 1 : C % 4 == 0 ? 2 : C % 2 == 0 ? 4 : 8, words = (uint32_t)(R * C / 8), rows = ceil_div(S, R);
    const uint32_t octets = ceil_div(C, 8);
    const float copied = 4.0f / 5.9e6f * (float)N * (float)S * (float)C;
    const uint32_t cus_of_die = (uint32_t)cus >= 8 ? (uint32_t)cus / 8 : 1;
    // What the three launches of the general form take, which read the tensor twice and whose sums of few large images are long chains: this is 0.77 ... 1.08 of it for
    // nine tenths of 212 of whole octets and 3 M values or more.
    const float many = 0.6e-3f * (float)S, few = 80.0f / (float)N;
    const float launches_us = 8.0f + (C % 8 == 0 ? 0.95e-6f : 5.4e-6f) * (float)N * (float)S * (float)C + (many < few ? many : few);
    const auto consider = [&](bool whole, uint32_t ob, uint32_t ob_log, uint32_t nb, uint32_t parts, bool ahead) {
        const uint32_t of = whole ? rows : (uint32_t)S, slots = kT / ob, per_part = ceil_div(of, parts), v = ceil_div(per_part, slots);
        if (v > kMostWords) return;
        parts = ceil_div(of, per_part);
        const FormTime& f = whole ? kRowTime[parts > 1] : kOctetTime[parts > 1][ob_log][C % 8 != 0 ? 0 : C % (8 * ob) != 0 ? 1 : 2];
        const uint32_t units = (uint32_t)N * parts, of_die = ceil_div(units, 8), dealt = of_die * nb;
        const float crowd = dealt > cus_of_die ? (float)dealt / (float)cus_of_die : 1.0f, share = copied * 8.0f * (float)of_die / (float)units;
        const float cost = (f.launch + f.word * (float)v * crowd + (f.copy + f.crowded * (crowd - 1.0f)) * share +
                            f.exchange * (float)(parts * (whole ? (uint32_t)C : ob * 8)) + (whole ? f.channel * (float)C : 0.0f)) *
                           (whole ? 1.04f : parts > 1 ? 0.94f : v <= 16 ? 0.87f : 1.0f);
        // Runs of 16 or 32 bytes and many words a lane are few workgroups, each with the whole image of its channels, dealt a second time: [4,155,155,560] 157
        // us, in three launches 72, [9,137,138,312] 126 / 67, [6,118,136,480] 79 / 59; but [3,110,111,600] 18 / 47.
        if ((ahead || (ob < 4 && v > 16)) && cost >= launches_us) return;
        if (best_v != 0 && cost >= best_cost) return;
        best = Geom{(uint32_t)C, (uint32_t)S, (uint32_t)(S * C), whole ? R : 1, whole ? words : octets, of, whole ? words * 8 : (uint32_t)C, ob, ob_log, nb, parts, per_part,
                    (uint32_t)N * parts};
        best_v = v;
        best_cost = cost;
        best_rows = whole;
    };
    // Workgroups that share channels: as many as are resident together, with two words per lane or more, and no more
    // partial sums than there are records.
    const auto most_parts = [&](uint32_t of, uint32_t ob, uint32_t blocks, uint32_t records) {
        uint32_t parts = (uint32_t)cus / blocks;
        if (parts > kMostParts) parts = kMostParts;
        if (parts > of / (2 * (kT / ob))) parts = of / (2 * (kT / ob));
        return parts < records ? parts : records;
    };
    // exchange: forms whose workgroups exchange sums too; ahead: only what takes less than the three launches
    const auto pick = [&](bool exchange, bool ahead) {
        best_v = 0;
        // Octets of channels, where a channel count that is no multiple of eight has a last one that begins inside the one before: in place, the workgroup
        // of either could find results of the other's.
        if (C >= 8 && (C % 8 == 0 || in != out))
            for (int k = 3; k >= 0; k--) {
                const uint32_t ob = 1u << k, nb = ceil_div(octets, ob);
                if (ob > 1 && ob / 2 >= octets) continue;
                consider(false, ob, (uint32_t)k, nb, 1, ahead);
                const uint32_t parts = most_parts((uint32_t)S, ob, (uint32_t)N * nb, kMostRecords / (ob * 8));
                if (exchange && parts > 1 && N * nb <= kMostGroups) {
                    consider(false, ob, (uint32_t)k, nb, parts, ahead);
                    // (as many as leave no die with more workgroups than compute units: the others would wait for those that are dealt a second time)
                    const uint32_t even = 8 * (cus_of_die / nb) / (uint32_t)N;
                    if (even > 1 && even < parts) consider(false, ob, (uint32_t)k, nb, even, ahead);
                }
            }
        if (words <= kT && C <= kT) {
            consider(true, words, 0, 1, 1, ahead);
            // (all that are resident read each other's partial sums of every channel: half and a quarter of them less)
            const uint32_t parts = most_parts(rows, words, (uint32_t)N, kMostRowRecords / (uint32_t)C);
            for (uint32_t div = 1; exchange && div <= 4 && parts / div > 1 && N <= kMostRowGroups; div *= 2) consider(true, words, 0, 1, parts / div, ahead);
        }
    };
    pick(true, false);
    // In place, a workgroup that computes a partner's partial sums could find results there: those launches take a workgroup alone with its channels, which
    // reads everything before it writes, or the kernels that finish all reads first.
    if (best_v != 0 && best.parts > 1 && in == out) pick(false, true);
    void* sync = nullptr;
    if (best_v != 0 && best.parts > 1) {
        bool absent = false;
        rc = get_sync_area(s, &sync, &absent);
        if (rc) return rc;
        sync = (char*)sync + kSyncCminor;
        if (absent) pick(false, false);  // (a capture on a stream without one)
    }
    if (best_v == 0) return VPX_RESULT_SUCCESS;
    // A launch holds fewer than 2^32 lanes; small images of many channels ask for more from N * nb = 2^23 on.
    const uint64_t blocks = ((uint64_t)best.units + 7) / 8 * best.nb * 8;
    if (blocks * kT >= (1ull << 32)) return VPX_RESULT_SUCCESS;
    const unsigned long long spin = mode == 2 ? 0ull : 50000ull;  // 0.5 ms of the 100 MHz counter
    const dim3 grid((unsigned)blocks);
#define VPX_CMINOR_AS(V, FORM) \
    VPX_LAUNCH((mvn_cminor_resident<V, FORM>), grid, dim3(kT), 0, s, (const half_t*)in, (half_t*)out, best, (unsigned*)sync, nv, eps, spin)
#define VPX_CMINOR(V)                           \
    do {                                        \
        if (best_rows) VPX_CMINOR_AS(V, kRows);   \
        else if (plain) VPX_CMINOR_AS(V, kShort); \
        else VPX_CMINOR_AS(V, kOctets);         \
    } while (0)
    const bool plain = best.ob < 4 || C % (8 * best.ob) != 0;
    if (best_v <= 2) VPX_CMINOR(2);
    else if (best_v <= 4) VPX_CMINOR(4);
    else if (best_v <= 8) VPX_CMINOR(8);
    else if (best_v <= 16) VPX_CMINOR(16);
    else if (best_v <= 24) VPX_CMINOR(24);
    else if (best_v <= 32) VPX_CMINOR(32);
    else if (best_v <= 40) VPX_CMINOR(40);
    else VPX_CMINOR(kMostWords);
#undef VPX_CMINOR
#undef VPX_CMINOR_AS
    *done = true;
    return VPX_RESULT_SUCCESS;
}

}  // namespace vpx
