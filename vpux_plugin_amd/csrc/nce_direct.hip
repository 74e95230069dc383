// nce_direct: convolutions and matmuls that would leave most of the chip idle or are over before a tile is staged -- the
// layers of one image, a classifier's few rows, narrow layers -- as an implicit product with nothing staged: fragments of
// weights and activations go from global memory straight into `v_mfma_i32_16x16x64_i8`.
//
// What bounds such a layer is a chain of latencies (launch, operands, a K loop that one or two waves per SIMD walk alone, the
// waves' meeting, PPE, stores), not bytes or MFMAs.  So the tile of a workgroup is small (16*TM channels x 16*TN positions), its K
// steps of 64 bytes are dealt to its S waves, each wave asks for as many steps' fragments at once as its registers hold, and the
// partial sums meet in LDS once (SPLIT); where tiles are many enough to fill the chip by themselves (not SPLIT) a wave keeps a
// tile to itself.  What the chain still holds is kept short: the channels' words of the weight table are asked for before
// the operands and prepared by the first wave while those travel (asked for at the end they cost a trip to memory of their own, and
// every lane prepared four channels or more); the meeting gives every lane one channel of up to four positions, a byte transpose within
// a quad turns that into whole pieces of rows; a walk of few steps leaves its unrolled loops by one branch (one skipped branch per step
// asked for cost 0.3 us).  us a launch, back to back in a HIP graph, before / after: [529 x 288] -> 32, 3x3: 3.21 / 2.80, [512 x 1728] -> 192,
// 3x3: 5.88 / 4.86, [29744 x 288] -> 32, 3x3: 6.48 / 4.92, [46818 x 144] -> 16, 3x3 stride 2: 5.20 / 4.04, [8 x 896] . [896 x 3552]
// 4.48 / 3.81, [3724 x 512] . [512 x 128] 6.22 / 5.51; an empty kernel 2.1.
//
// Weights are the first operand: a lane's four accumulators are four channels of one position (quarter c4 of the wave: rows
// 4*c4 ... 4*c4+3 of a tile).  Row i of tile j is channel 4*TM*(i/4) + 4*j + i%4: a quarter's 4*TM channels of a position lie
// side by side in the output and leave in one store, at any address.
// The zero-point term corr * sum_k w comes from one more MFMA per weight fragment, against a fragment of ones: it lands
// in the accumulators' own layout and takes part in the meeting of the waves, no pass over the weights, no lane exchange.
// K is walked as the flat run of 16-byte chunks the weights hold (tap, then channel).  Where a pixel's channels fill whole steps the tap
// is the step's, worked out once per wave; else a lane's chunk 4*step + c4 names its tap, and chunks past the end multiply
// zero weights.  Taps outside the image hold the zero-point byte.
#include "nce_common.h"

namespace vpx {
namespace nce {
namespace {

constexpr int kMaxWaves = 8;

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef u32x2 u32x2_any __attribute__((aligned(1)));
typedef uint32_t u32_any __attribute__((aligned(1)));

// K steps asked for at once: what about 70 registers hold.
constexpr int direct_depth(int tm, int tn) { return tm + tn == 2 ? 8 : (tm + tn == 3 ? 6 : (tm + tn == 4 ? 4 : (tm + tn == 6 ? 3 : 2))); }

// Waves per SIMD the register budget is cut for.
constexpr int direct_waves_per_simd(int tm, int tn) { return tm * tn <= 4 ? 4 : (tm * tn == 8 ? 3 : 2); }

// How a step finds its activations: the pixel itself (1x1), a tap per lane, or (a pixel's channels fill whole steps) a tap per step.
enum DirectTaps { kNoTaps = 0, kTapPerLane = 1, kTapPerStep = 2 };

template <int TM, int TN, DirectTaps TAPS, bool SPLIT>
__global__ __launch_bounds__(SPLIT ? 64 * kMaxWaves : 256) void nce_direct(const int8_t* __restrict__ in, const int8_t* __restrict__ w,
                                                                           const int32_t* __restrict__ wt, uint8_t* __restrict__ out, ConvGeom g,
                                                                           GemmPpe ppe, DirectGeom d, int pad, int flip) {
    constexpr int DEPTH = direct_depth(TM, TN), CH = 16 * TM;
    constexpr bool CONV = TAPS != kNoTaps;
    extern __shared__ __attribute__((aligned(16))) i32x4 s_part[];  // SPLIT: [wave][tile][lane]
    __shared__ ChanPrep s_prep[CH];
    __shared__ int s_general;
    // (a value of every line of the launch's arguments: one trip to memory for all, see vpx_common.h)
    asm volatile("" ::"s"(in), "s"(w), "s"(wt), "s"(out), "s"(g.SX), "s"(g.ish), "s"(ppe.corr), "s"(d.noc), "s"(d.ow), "s"(flip));
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n16 = lane & 15, c4 = lane >> 4;
    const int noc = d.noc;
    // (Everything up to the first load is a chain: divisions are products with what the host has worked out, a dozen dependent instructions less each.
    // us in a HIP graph, divided / this: [4,14,14,96] -> 96 3x3 3.49 / 3.31, [1,14,14,256] -> 256 4.76 / 4.56, [1,112,112,16] -> 16 7x7 3.03 / 2.89.)
    const unsigned pos = quotient(blockIdx.x, (unsigned)noc, d.noc_magic);
    const int oct = (int)(blockIdx.x - pos * (unsigned)noc);
    const int post = (int)pos * (SPLIT ? 1 : 4) + (SPLIT ? 0 : wave);
    const int oc0 = oct * CH, P = d.P, OC = (int)g.OC;
    const int chunks = d.chunks;
    const int steps = (chunks + 3) >> 2;
    const int s0 = SPLIT ? wave * d.share : 0, s1 = SPLIT ? (s0 + d.share < steps ? s0 + d.share : steps) : (post * 16 * TN < P ? steps : 0);

    // The first wave prepares the tile's channels; their words of the table are asked for before anything else.
    int2 words = int2{0, 0};
    if (wave == 0) {
        const int ch = oc0 + (lane & (CH - 1));
        words = *reinterpret_cast<const int2*>(wt + (int64_t)(ch < OC ? ch : OC - 1) * 4 + 2);
    }

    // channel of row i of tile j
    const auto channel = [&](int i, int j) { return oc0 + 4 * TM * (i >> 2) + 4 * j + (i & 3); };
    unsigned wofs[TM];
#pragma unroll
    for (int j = 0; j < TM; j++) {
        int ch = channel(n16, j);
        ch = ch < OC ? ch : OC - 1;  // (rows past the last channel repeat it and are not stored)
        wofs[j] = ((unsigned)ch * (unsigned)chunks + (TAPS == kTapPerStep ? (unsigned)c4 : 0u)) * 16u;
    }
    int iy0[TN], ix0[TN];
    int pofs[TN];  // byte offset of the pixel under tap (0, 0); CONV: may lie outside the image
#pragma unroll
    for (int j = 0; j < TN; j++) {
        int m = (post * TN + j) * 16 + n16;
        m = m < P ? m : P - 1;
        if (CONV || !d.flat_in) {
            const unsigned img = quotient((unsigned)m, (unsigned)d.ohow, d.ohow_magic), rem = (unsigned)m - img * (unsigned)d.ohow,
                           oy = quotient(rem, (unsigned)d.ow, d.ow_magic), ox = rem - oy * (unsigned)d.ow;
            iy0[j] = (int)oy * g.SY - g.PT;
            ix0[j] = (int)ox * g.SX - g.PL;
            pofs[j] = (int)img * (int)g.isn + iy0[j] * (int)g.ish + ix0[j] * (int)g.isw;
        } else {
            pofs[j] = m * (int)g.isw;
        }
        if (TAPS == kTapPerStep) pofs[j] += 16 * c4;
    }

    struct Step {
        i32x4 wf[TM], af[TN];
        unsigned inside;  // bit j: the lane's chunk of position tile j lies inside the image
    };
    const auto load = [&](int s, Step& f) {
        if constexpr (TAPS == kTapPerStep) {  // (four chunks a step: no last step is short)
            const int tap = fdiv(4 * s, d.cpp), c = 4 * s - tap * (int)d.cpp.d;
            const int ky = fdiv(tap, d.kx), kx = tap - ky * (int)d.kx.d;
            const int ofs = ky * (int)g.ish + kx * (int)g.isw + c * 16;
#pragma unroll
            for (int j = 0; j < TM; j++) f.wf[j] = *reinterpret_cast<const i32x4*>(w + (wofs[j] + (unsigned)s * 64u));
            f.inside = 0;
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const bool hit = (unsigned)(iy0[j] + ky) < (unsigned)d.H && (unsigned)(ix0[j] + kx) < (unsigned)d.W;
                f.inside |= hit ? 1u << j : 0u;
                f.af[j] = *reinterpret_cast<const i32x4*>(in + (unsigned)(hit ? pofs[j] + ofs : 0));
            }
            return;
        }
        const int u = 4 * s + c4;
        const bool real = u < chunks;
        const unsigned uc = (unsigned)(real ? u : 0);
#pragma unroll
        for (int j = 0; j < TM; j++) f.wf[j] = *reinterpret_cast<const i32x4*>(w + (wofs[j] + uc * 16u));
        f.inside = 0;
        if constexpr (CONV) {
            const int tap = fdiv((int)uc, d.cpp), c = (int)uc - tap * (int)d.cpp.d;
            const int ky = fdiv(tap, d.kx), kx = tap - ky * (int)d.kx.d;
            const int ofs = ky * (int)g.ish + kx * (int)g.isw + c * 16;
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const bool hit = (unsigned)(iy0[j] + ky) < (unsigned)d.H && (unsigned)(ix0[j] + kx) < (unsigned)d.W;
                f.inside |= hit ? 1u << j : 0u;
                f.af[j] = *reinterpret_cast<const i32x4*>(in + (unsigned)(hit ? pofs[j] + ofs : 0));
            }
        } else {
#pragma unroll
            for (int j = 0; j < TN; j++) f.af[j] = *reinterpret_cast<const i32x4*>(in + (unsigned)(pofs[j] + (int)uc * 16));
        }
        f.inside |= real ? 0x80000000u : 0u;
    };

    i32x4 acc[TM][TN], sums[TM];
#pragma unroll
    for (int i = 0; i < TM; i++) {
        sums[i] = i32x4{0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = i32x4{0, 0, 0, 0};
    }
    const bool corrects = ppe.corr != 0, ragged = (chunks & 3) != 0;
    const auto use = [&](Step& f) {
        if (TAPS != kTapPerStep && ragged) {
            const bool real = (int)f.inside < 0;
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int q = 0; q < 4; q++) f.wf[i][q] = real ? f.wf[i][q] : 0;
        }
#pragma unroll
        for (int j = 0; j < TN; j++) {
            if (CONV) {
                const bool hit = (f.inside >> j) & 1u;
#pragma unroll
                for (int q = 0; q < 4; q++) f.af[j][q] = hit ? f.af[j][q] : pad;
            }
            f.af[j] = f.af[j] ^ flip;
#pragma unroll
            for (int i = 0; i < TM; i++) acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(f.wf[i], f.af[j], acc[i][j], 0, 0, 0);
        }
        if (corrects) {
            const i32x4 ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101};
#pragma unroll
            for (int i = 0; i < TM; i++) sums[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(f.wf[i], ones, sums[i], 0, 0, 0);
        }
    };

    const PpePack pk = make_ppe_pack(ppe.zp_out, ppe.lo, ppe.hi, ppe.out_signed != 0);
    {
        Step f[DEPTH];
        int s = s0;
        asm volatile("" : "+s"(s));  // (known to be zero, the steps' addresses would all be worked out ahead and held in registers)
        const bool long_walk = s1 - s >= DEPTH;
        if (long_walk) {
#pragma unroll
            for (int p = 0; p < DEPTH; p++) load(s + p, f[p]);
        } else {
#pragma unroll
            for (int p = 0; p < DEPTH - 1; p++) {  // (a walk that ends early leaves by one branch)
                if (s + p >= s1) break;
                load(s + p, f[p]);
            }
        }
        if (wave == 0) {  // (while the operands travel)
            const ChanPrep c = ppe_prepare_packed((int)(int16_t)((uint32_t)words.x >> 16), (int)(((uint32_t)words.x >> 8) & 0xffu), words.y,
                                                  ppe.prelu_mult, ppe.prelu_shift);
            const bool clip = c.bmax_pos != 0x7fffffff || c.bmax_neg != 0x7fffffff;
            const int general = __builtin_amdgcn_ballot_w64(clip) != 0 || pk.odd != 0 ? 1 : 0;
            if (lane < CH) s_prep[lane] = c;
            if (lane == 0) s_general = general;
        }
        if (long_walk) {
            // (no branch between a load and the waits of the steps before it, or those waits would cover the load too)
            for (; s + 2 * DEPTH <= s1; s += DEPTH) {
#pragma unroll
                for (int p = 0; p < DEPTH; p++) {
                    use(f[p]);
                    load(s + p + DEPTH, f[p]);
                }
            }
#pragma unroll
            for (int p = 0; p < DEPTH; p++) use(f[p]);
            s += DEPTH;
#pragma unroll
            for (int p = 0; p < DEPTH - 1; p++) {
                if (s + p >= s1) break;
                load(s + p, f[p]);
            }
        }
#pragma unroll
        for (int p = 0; p < DEPTH - 1; p++) {
            if (s + p >= s1) break;
            use(f[p]);
        }
    }
    // The first reader of an MFMA's result has to come eight issue slots behind it.  Behind the branches of the walk the compiler keeps them only on the paths
    // that it takes to be possible -- this condition is the one in use(); on the others there were four with one tile of one block --, so
    // they are kept here: everything read below goes through the second of these, which come in order.
    if constexpr (TM * TN == 1) {
        asm volatile("" : "+v"(acc[0][0]), "+v"(sums[0]));
        asm volatile("s_nop 7" : "+v"(acc[0][0]), "+v"(sums[0]));
    }
    if (corrects) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) acc[i][j] += sums[i] * ppe.corr;
    }

    // element offset of output position m
    const auto position = [&](int m) -> int64_t {
        if (g.out_flat == 2) return (int64_t)m * g.osw;
        const unsigned img = quotient((unsigned)m, (unsigned)d.ohow, d.ohow_magic), rem = (unsigned)m - img * (unsigned)d.ohow,
                       oy = quotient(rem, (unsigned)d.ow, d.ow_magic), ox = rem - oy * (unsigned)d.ow;
        return (int64_t)img * g.osn + (int64_t)oy * g.osh + (int64_t)ox * g.osw;
    };
    // 4 * TM channels from ch on of one position
    const auto store = [&](uint8_t* dst, const unsigned (&v)[TM], int ch) {
        if (TM == 4 && ch + 16 <= OC) {  // (at any address)
            *reinterpret_cast<i32x4_any*>(dst) = i32x4{(int)v[0], (int)v[1], (int)v[TM > 2 ? 2 : 0], (int)v[TM > 3 ? 3 : 0]};
        } else if (TM == 2 && ch + 8 <= OC) {
            *reinterpret_cast<u32x2_any*>(dst) = u32x2{v[0], v[TM > 1 ? 1 : 0]};
        } else {
#pragma unroll
            for (int i = 0; i < TM; i++) {
                if (ch + 4 * i + 4 <= OC) {
                    *reinterpret_cast<u32_any*>(dst + 4 * i) = v[i];
                } else {
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        if (ch + 4 * i + r < OC) dst[4 * i + r] = (uint8_t)(v[i] >> (8 * r));
                }
            }
        }
    };

    if constexpr (SPLIT) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) s_part[(wave * TM * TN + i * TN + j) * 64 + lane] = acc[i][j];
        __syncthreads();
        // A value per lane and tile: lane (position lane / 4, channel lane % 4) of quarter q of every tile, summed over the
        // waves; after the transpose lane t of a quad has position tile t's 4 * TM channels.
        const int* const part = reinterpret_cast<const int*>(s_part);
        const int S = d.S;
        const QuadTranspose transpose(lane);
        const auto finish = [&](auto general_c) {
            for (int q = wave; q < 4; q += S) {
                int term[TN];
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    const int m = (post * TN + j) * 16 + (lane >> 2);
                    term[j] = ppe.rowterm ? ppe.rowterm[m < P ? m : P - 1] : 0;
                }
                unsigned v[TM];
#pragma unroll
                for (int i = 0; i < TM; i++) {
                    const ChanPrep c = s_prep[4 * TM * q + 4 * i + (lane & 3)];
                    unsigned bytes = 0;
#pragma unroll
                    for (int j = 0; j < TN; j++) {
                        const int at = (i * TN + j) * 256 + q * 64 + lane;
                        int x[kMaxWaves];
#pragma unroll
                        for (int k = 0; k < 4; k++) x[k] = part[(k < S ? k : 0) * (TM * TN * 256) + at];
                        int sum = term[j] + x[0] + x[1] + (S > 2 ? x[2] : 0) + (S > 3 ? x[3] : 0);  // (2 waves at least)
                        if (S > 4) {
#pragma unroll
                            for (int k = 4; k < kMaxWaves; k++) x[k] = part[(k < S ? k : 0) * (TM * TN * 256) + at];
                            sum += x[4] + (S > 5 ? x[5] : 0) + (S > 6 ? x[6] : 0) + (S > 7 ? x[7] : 0);
                        }
                        bytes |= ppe_one<false, decltype(general_c)::value>(sum, c, pk) << (8 * j);
                    }
                    v[i] = transpose(bytes) ^ pk.flip;
                }
                const int j = lane & 3, m = (post * TN + j) * 16 + (lane >> 2), ch = oc0 + 4 * TM * q;
                if (j < TN && m < P && ch < OC) store(out + (position(m) + ch), v, ch);
            }
        };
        if (s_general != 0) finish(std::true_type{});
        else finish(std::false_type{});
    } else {
        __syncthreads();  // (the prepared channels)
        const int ch = oc0 + 4 * TM * c4;
        const auto finish = [&](auto general_c) {
            unsigned v[TN][TM];
            int term[TN];
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const int m = (post * TN + j) * 16 + n16;
                term[j] = ppe.rowterm ? ppe.rowterm[m < P ? m : P - 1] : 0;
#pragma unroll
                for (int i = 0; i < TM; i++) v[j][i] = 0;
            }
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const ChanPrep c = s_prep[4 * TM * c4 + 4 * i + r];
#pragma unroll
                    for (int j = 0; j < TN; j++) v[j][i] |= ppe_one<false, decltype(general_c)::value>(acc[i][j][r] + term[j], c, pk) << (8 * r);
                }
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const int m = (post * TN + j) * 16 + n16;
                if (m >= P || ch >= OC) continue;
#pragma unroll
                for (int i = 0; i < TM; i++) v[j][i] ^= pk.flip;
                store(out + (position(m) + ch), v[j], ch);
            }
        };
        if (s_general != 0) finish(std::true_type{});
        else finish(std::false_type{});
    }
}

}  // namespace

// The tile and the number of waves for a layer, and the time to expect.  The terms were fitted (non-negative least squares,
// median error 7 %, back to back in a HIP graph over rotating buffers) to 330 layers of P 1 ... 370 000, K 16 ... 4608,
// OC 16 ... 9500 with every tile here and 1, 2, 4 and 8 waves: a launch and its first operands 2.2 us; the meeting of the waves; rounds of
// resident waves; operand loads through a compute unit's cache; rounds of asked-for steps and the steps one wave walks; MFMAs
// of the fullest SIMD; the PPE of the fullest compute unit's tiles; memory, and output in pieces of 4 or 8 bytes.  The tile is the one
// that would be shortest with 0.17 us for a step of a walk and 0.025 for a wave's value at the meeting: of 327 layers that takes 0.8 % over
// the best of all combinations, 17 more than 5 % (by the time itself 1.4 %, 37: [600 x 256] . [256 x 64] without a split 3.5 us, with
// one 2.9; 7x7 x 16 -> 64 of one image of [139,257] 6.5 and 5.9).
// (Every layer asks, so the arithmetic is whole numbers of 32 bits and divisions by constants as far as it goes.)
DirectShape direct_shape(int64_t P, int64_t OC, int64_t K, int64_t in_bytes, int cus) {
    const uint32_t steps = (uint32_t)((K / 16 + 3) / 4);
    const double mbytes = 1e-6 * ((double)P * (double)OC + (double)OC * (double)K + (double)in_bytes), mout = 1e-6 * (double)P * (double)OC;
    struct Walk {
        uint32_t share, S;  // steps of a wave, waves that have any
    };
    const auto walk = [&](uint32_t most) {
        const uint32_t waves = most < steps ? most : steps, share = (steps + waves - 1) / waves;
        return Walk{share, (steps + share - 1) / share};
    };
    const Walk by1{steps, 1}, by4 = walk(4), by8 = walk(8);
    DirectShape best{0, 0, 0, 0.0};
    double least = 0.0;
    const auto consider = [&](auto tm_c, auto tn_c, auto waves_c) {
        constexpr int tm = decltype(tm_c)::value, tn = decltype(tn_c)::value, most = decltype(waves_c)::value;
        constexpr uint32_t depth = direct_depth(tm, tn);
        const int64_t noc = (OC + 16 * tm - 1) / (16 * tm), npos = (P + 16 * tn - 1) / (16 * tn), tiles = noc * npos;
        const Walk& w = most == 1 ? by1 : (most == 4 ? by4 : by8);
        const uint32_t share = w.share, S = w.S;
        const bool split = S > 1;
        const int64_t wgs = split ? tiles : noc * ((npos + 3) / 4);
        if (wgs >= (1ll << 31)) return;
        const uint64_t fullest = (uint64_t)(((uint32_t)wgs + (uint32_t)cus - 1) / (uint32_t)cus) * (split ? 1 : 4);  // tiles of the fullest compute unit
        const uint64_t of_simd = (fullest * S + 3) / 4;
        const double cu_tiles = (double)fullest, simd_waves = (double)of_simd, values = cu_tiles * tm * tn;
        const double rounds = (double)(tm * tn <= 4 ? (of_simd + 3) / 4 : (of_simd + 1) / 2);
        const double us = 2.2 + (split ? 0.484 : 0.0) + 0.491 * (rounds - 1.0) + 0.0066 * (double)tiles / cus * (double)steps * (tm + tn) +
                          0.07 * (double)((share + depth - 1) / depth) + 0.126 * (double)share + 0.0174 * simd_waves * (double)share * tm * (tn + 1) +
                          values * (split ? 0.0122 + 0.0295 * (double)S : 0.0259) + kDirectPerMByte * mbytes + mout * (tm == 1 ? 0.913 : (tm == 2 ? 0.18 : 0.0));
        const double rank = us + 0.044 * (double)share - (split ? 0.0045 * values * (double)S : 0.0);
        const double shortest = best.tm == 0 || us < best.us ? us : best.us;
        if (best.tm == 0 || rank < least) {
            least = rank;
            best = DirectShape{tm, tn, most, shortest};
        }
        best.us = shortest;
    };
    const std::integral_constant<int, 1> one;
    const std::integral_constant<int, 2> two;
    const std::integral_constant<int, 4> four;
    const std::integral_constant<int, 8> eight;
    consider(one, one, one), consider(one, one, four), consider(one, one, eight);
    consider(two, one, one), consider(two, one, four), consider(two, one, eight);
    consider(two, two, one), consider(two, two, four), consider(two, two, eight);
    consider(two, four, one);
    consider(four, four, one);
    return best;
}

int launch_direct(const DirectLaunch& a, hipStream_t s) {
    const int flip = a.in_u8 ? (int)0x80808080 : 0, pad = (int)(0x01010101u * (unsigned)(a.pad_byte & 0xff));
    const int npos = (a.d.P + 16 * a.tn - 1) / (16 * a.tn);
    const bool split = a.d.S > 1;
    const int64_t blocks = (int64_t)a.d.noc * (split ? npos : (npos + 3) / 4);
    const dim3 grid((unsigned)blocks), block(split ? 64 * a.d.S : 256);
    const size_t lds = split ? (size_t)a.d.S * a.tm * a.tn * 1024 : 0;
    VPX_REQUIRE(a.d.S <= kMaxWaves, VPX_RESULT_ERROR_UNKNOWN, "nce_direct has no form of %d waves", a.d.S);
    const auto launch = [&](auto kernel) -> int {
        const int rc = set_dyn_lds(kernel, lds);
        if (rc) return rc;
        VPX_LAUNCH(kernel, grid, block, lds, s, a.in, a.w, a.wt, a.out, a.g, a.ppe, a.d, pad, flip);
        return VPX_RESULT_SUCCESS;
    };
    const auto by_taps = [&](auto tm_c, auto tn_c) -> int {
        constexpr int TM = decltype(tm_c)::value, TN = decltype(tn_c)::value;
        constexpr bool kSplits = TM <= 2 && TN <= 2;
        VPX_REQUIRE(kSplits || !split, VPX_RESULT_ERROR_UNKNOWN, "nce_direct splits K in tiles of one or two by one or two only");
        if (!a.conv) return split ? launch(nce_direct<TM, TN, kNoTaps, kSplits>) : launch(nce_direct<TM, TN, kNoTaps, false>);
        if (a.g.IC % 64 == 0) return split ? launch(nce_direct<TM, TN, kTapPerStep, kSplits>) : launch(nce_direct<TM, TN, kTapPerStep, false>);
        return split ? launch(nce_direct<TM, TN, kTapPerLane, kSplits>) : launch(nce_direct<TM, TN, kTapPerLane, false>);
    };
    const auto one = std::integral_constant<int, 1>{};
    const auto two = std::integral_constant<int, 2>{};
    const auto four = std::integral_constant<int, 4>{};
    int rc;
    switch (a.tm * 10 + a.tn) {
    case 11: rc = by_taps(one, one); break;
    case 21: rc = by_taps(two, one); break;
    case 22: rc = by_taps(two, two); break;
    case 24: rc = by_taps(two, four); break;
    case 44: rc = by_taps(four, four); break;
    default: return fail(VPX_RESULT_ERROR_UNKNOWN, "nce_direct has no tile of %d x %d", a.tm, a.tn);
    }
    if (rc) return rc;
    return VPX_RESULT_SUCCESS;
}

}  // namespace nce
}  // namespace vpx
