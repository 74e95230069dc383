// nce_gemm_regb: A[M][K] x B[N][K]^T with the PPE fused, for a short K (up to 256, any multiple of 16) and many rows -- the 1x1
// layers of a network's early stages, where a row of the result costs more vector work in the PPE than matrix work and
// the tile kernel (nce_gemm.hip) is all prologue and epilogue.
//
// No workgroup barrier after the set-up, and neither operand goes through LDS.  A wave owns CBW blocks of 16*NT output
// channels for the whole launch and keeps their weights in registers (CBW x NT x KS fragments of
// `v_mfma_i32_16x16x64_i8`, KS = K/64 rounded up, 64 registers at most); it walks blocks of 16 rows: one 16-byte load per
// lane and 64 of K straight from global memory (the 16 rows of a block are one contiguous piece when K = 64), then per
// channel block NT x KS MFMAs that start from the bias and the short PPE.  The loads run kPrefetch blocks ahead of the
// arithmetic.  The part of the last fragment past K holds zero weights, against the row's first bytes.
//
// The weights are the FIRST operand of the MFMA: the product is the transposed block, channels down and rows of the
// matrix across, so a lane's four accumulators of a tile are four channels of one row -- the bytes of a dword of the
// output as it lies in memory, no transpose.  Row i of tile j is channel 4*NT*(i/4) + 4*j + i%4 of its block: lane
// (row n16, quarter c4) then holds channels 4*NT*c4 .. 4*NT*c4 + 4*NT-1 of row n16 in its NT result dwords.
// The PPE factors of a lane's 4*NT channels per block come from a table in LDS that the workgroup prepares once
// (one channel per thread); in registers they would be 32 to 64 per block.
//
// Output: the wave collects its 16 rows x CBW x 16*NT bytes in an LDS tile of its own and writes them as whole pieces of
// rows, neighbouring lanes neighbouring 16-byte pieces (measured at [401408 x 64] . [64 x 256]: 64-byte pieces of
// 256-byte rows, one per lane quarter, 34 us; a row per sixteen lanes 28 us).
//
// The set-up is half of a launch.  Weights, then the words of the weight table, are asked for together, and the rows behind the barriers:
// asked for in front, they stand between every workgroup and its weights ([3380 x 128] . [128 x 512], a block of rows for each wave, 5.25 us
// on one set of buffers, now 4.69; 4.84 with the words behind a barrier of their own).  Four waves with the same channels and a K beyond 64
// have few weights and deal one contiguous fetch out through LDS: there the first rows' way begins before it.  Channel sums come from MFMAs
// against ones.  us in a HIP graph over rotating buffers, with the words behind the sums and a copy of the weights for each wave / now:
// [100352 x 256] . [256 x 64] 12.6 / 9.0, [20216 x 256] . [256 x 64] 7.9 / 5.3, [100352 x 128] . [128 x 32] 8.3 / 6.0, [100352 x 64] . [64 x
// 256] 14.2 / 13.1, [401408 x 64] . [64 x 256] 39.0 / 33.6, [18928 x 192] . [192 x 48] 5.1 / 4.1, [2890 x 192] . [192 x 768] 6.0 / 5.7,
// [5547 x 32] . [32 x 128] 4.1 / 2.9.
// What is left at K = 64: a SIMD's vector instructions (115 a block of 16 x 64, 64 of them the PPE) as long as its memory time.
//
// Work is dealt by wave.  The four waves of a workgroup serve GW different groups of CBW channel blocks (4 / GW row
// streams each): with GW > 1 the waves that share a row block are neighbours, so its rows come from memory once.  A
// workgroup's index modulo the number of its kind picks the channels; wave s of those that share them takes row blocks
// s, s + S, ...
#include <algorithm>

#include "nce_common.h"

namespace vpx {
namespace nce {
namespace {

constexpr int kRegbWaves = 4;

// Waves per SIMD the register budget is cut for (512 registers / 4, 3, 2 waves): the launch is bound by the memory
// system and by vector instructions, both of which want waves.
constexpr int regb_waves_per_simd(bool same_f, int ks, int cbw, int nt) {
    const int wregs = ks * cbw * nt * 4;  // registers of weights
    return wregs <= 16 ? 4 : (wregs <= 32 ? (same_f && ks == 1 ? 4 : 3) : (wregs < 48 || (same_f && (wregs == 48 || ks <= 2)) ? 3 : 2));
}

template <bool SAME_F, int KS, int CBW, int GW, int NT>
__global__ __launch_bounds__(64 * kRegbWaves) __attribute__((amdgpu_waves_per_eu(regb_waves_per_simd(SAME_F, KS, CBW, NT)))) void nce_gemm_regb(
    const int8_t* __restrict__ A, const int8_t* __restrict__ B, const int32_t* __restrict__ wt, uint8_t* __restrict__ out, int64_t M, int N,
    int chunks, int64_t lda, int64_t ldc, GemmPpe ppe, int supers, int sign_flip, int past_cache) {
    constexpr int BCH = 16 * NT, NCH = CBW * BCH, RSW = kRegbWaves / GW, TCH = GW * NCH;
    static_assert(TCH <= 64 * kRegbWaves, "one thread prepares one channel");
    constexpr int kPrefetch = KS == 4 ? 1 : (KS == 1 && CBW < 4 ? 3 : 2);  // row blocks ahead; (kPrefetch + 1) x KS x 4 registers
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int gw = w / RSW, super = (int)blockIdx.x % supers;
    const int stream = ((int)blockIdx.x / supers) * RSW + w % RSW, streams = ((int)gridDim.x / supers) * RSW;
    const int n16 = lane & 15, c4 = lane >> 4;
    const int n0 = (super * GW + gw) * NCH;  // this wave's first channel
    const int tb = gw * NCH;                 // ... and its place in the workgroup's tables

    const bool tail = (KS - 1) * 4 + c4 < chunks;  // the last fragment's chunk of this lane exists
    const int nblk = (int)((M + 15) >> 4);
    const int tail_at = tail ? (KS - 1) * 64 + c4 * 16 : 0;
    auto fetch = [&](int b, i32x4 (&a)[KS]) {
        int64_t row = (int64_t)b * 16 + n16;
        row = row < M ? row : M - 1;
        const int8_t* src = A + row * lda;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) a[ks] = *reinterpret_cast<const i32x4*>(src + (ks < KS - 1 ? c4 * 16 + ks * 64 : tail_at));
    };
    // ---- what the set-up waits for, asked for in the order it is used: the weights (from the caches: every workgroup reads them), this
    // thread's words of the weight table, then the rows.  (No branch around the words: at its end the compiler waits for what was asked for
    // inside, which cost a trip to memory in front of the weights.)
    constexpr bool SHARE = GW == 1 && KS >= 2;  // the four waves serve the same channels and K is long
    i32x4 a[kPrefetch + 1][KS];
    const auto fetch_ahead = [&](int from) __attribute__((always_inline)) {  // (blocks that there are: repeating the last row for the others cost 2 %)
#pragma unroll
        for (int p = 0; p < kPrefetch; p++)
            if (p >= from && (p == 0 || stream + p * streams < nblk)) fetch(stream + p * streams, a[p]);
    };
    int2 words;
    const auto fetch_words = [&]() __attribute__((always_inline)) {
        const int ch = super * TCH + (tid < TCH ? tid : 0);
        words = *reinterpret_cast<const int2*>(wt + (int64_t)(ch < N ? ch : N - 1) * 4 + 2);
    };
    if (SHARE) {  // (their weights are few: the first rows' longer way begins before)
        fetch(stream, a[0]);
        fetch_words();
    }
    // Fragment (cbl, j) of the weights: row n16 of tile j of block cbl, 16 of K per quarter.  SHARE: the workgroup fetches them once, a
    // contiguous piece, and deals them out through LDS.
    i32x4 wb[CBW][NT][KS];
    if constexpr (SHARE) {
        constexpr int ROW = KS * 64 + 16, PIECES = NCH * KS * 4, PER = (PIECES + 64 * kRegbWaves - 1) / (64 * kRegbWaves);
        __shared__ __attribute__((aligned(16))) uint8_t s_w[NCH * ROW];
        i32x4 v[PER];
#pragma unroll
        for (int u = 0; u < PER; u++) {
            const int q0 = u * 64 * kRegbWaves + tid, q = q0 < PIECES ? q0 : PIECES - 1, row = q / (KS * 4), c = q % (KS * 4);
            const int ch = n0 + row < N ? n0 + row : N - 1;  // channels past the end repeat the last one (never stored)
            v[u] = *reinterpret_cast<const i32x4*>(B + ((int64_t)ch * chunks + (c < chunks ? c : 0)) * 16);
        }
#pragma unroll
        for (int u = 0; u < PER; u++) {
            const int q0 = u * 64 * kRegbWaves + tid, q = q0 < PIECES ? q0 : PIECES - 1, row = q / (KS * 4), c = q % (KS * 4);
            *reinterpret_cast<i32x4*>(s_w + row * ROW + c * 16) = v[u];
        }
        __syncthreads();
#pragma unroll
        for (int cbl = 0; cbl < CBW; cbl++)
#pragma unroll
            for (int j = 0; j < NT; j++)
#pragma unroll
                for (int ks = 0; ks < KS; ks++)
                    wb[cbl][j][ks] = *reinterpret_cast<const i32x4*>(s_w + (cbl * BCH + (n16 >> 2) * (4 * NT) + j * 4 + (n16 & 3)) * ROW + ks * 64 + c4 * 16);
    } else {
#pragma unroll
        for (int cbl = 0; cbl < CBW; cbl++)
#pragma unroll
            for (int j = 0; j < NT; j++) {
                int ch = n0 + cbl * BCH + (n16 >> 2) * (4 * NT) + j * 4 + (n16 & 3);
                ch = ch < N ? ch : N - 1;
#pragma unroll
                for (int ks = 0; ks < KS; ks++)
                    wb[cbl][j][ks] = *reinterpret_cast<const i32x4*>(B + ((int64_t)ch * chunks + (ks < KS - 1 || tail ? ks * 4 + c4 : 0)) * 16);
            }
        fetch_words();
    }
#pragma unroll
    for (int cbl = 0; cbl < CBW; cbl++)
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int q = 0; q < 4; q++) wb[cbl][j][KS - 1][q] = tail ? wb[cbl][j][KS - 1][q] : 0;

    // ---- PPE parameters: thread t prepares channel t of the workgroup's TCH into tables in LDS
    __shared__ double s_fpos[TCH], s_fneg[TCH];
    __shared__ __attribute__((aligned(16))) int s_bias[TCH], s_sum[TCH];
    __shared__ int s_w2[TCH], s_general[kRegbWaves];
    if (ppe.corr != 0) {
        // the column sums by MFMAs against ones: a lane's four of a tile are four channels (waves that serve the same channels write the same)
        const i32x4 ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101};
#pragma unroll
        for (int cbl = 0; cbl < CBW; cbl++)
#pragma unroll
            for (int j = 0; j < NT; j++) {
                i32x4 sum = i32x4{0, 0, 0, 0};
#pragma unroll
                for (int ks = 0; ks < KS; ks++) sum = __builtin_amdgcn_mfma_i32_16x16x64_i8(wb[cbl][j][ks], ones, sum, 0, 0, 0);
                if (n16 == 0) *reinterpret_cast<i32x4*>(&s_sum[tb + cbl * BCH + c4 * (4 * NT) + j * 4]) = sum;
            }
        __syncthreads();
    }
    const PpePack pk = make_ppe_pack(ppe.zp_out, ppe.lo, ppe.hi, ppe.out_signed != 0);
    bool clip = false;
    if (tid < TCH) {
        const int sum = ppe.corr != 0 ? s_sum[tid] : 0;
        const uint32_t w2 = (uint32_t)words.x;
        const ChanPrep c = ppe_prepare((int)(int16_t)(w2 >> 16), (int)((w2 >> 8) & 0xffu), (int)((unsigned)words.y + (unsigned)(ppe.corr * sum)),
                                       ppe.prelu_mult, ppe.prelu_shift);
        clip = c.bmax_pos != 0x7fffffff || c.bmax_neg != 0x7fffffff;
        s_fpos[tid] = c.f_pos;
        s_fneg[tid] = c.f_neg;
        s_bias[tid] = c.bias;
        s_w2[tid] = (int)w2;
    }
    // the short PPE serves slopes in [0, 1] (ReLU, LeakyReLU), an even zero-point offset and scales up to 1/2
    const bool slope_ok = SAME_F || (ppe.prelu_mult >= 0 && (ppe.prelu_shift >= 31 || ppe.prelu_mult <= (1 << ppe.prelu_shift)));
    const bool special = __builtin_amdgcn_ballot_w64(clip) != 0 || pk.odd != 0 || !slope_ok;
    if (lane == 0) s_general[w] = special ? 1 : 0;
    __syncthreads();
    const bool general = (s_general[0] | s_general[1] | s_general[2] | s_general[3]) != 0;  // (one answer for the workgroup)
    fetch_ahead(SHARE ? 1 : 0);
    if (n0 >= N) return;  // (a wave past the last block)
    const int32_t* const rt = ppe.rowterm;

    // the sums of channel block cbl of a row block: from the bias (short PPE) or from zero, the row term added
    auto multiply = [&](int cbl, const i32x4 (&f)[KS], int rowterm, i32x4 (&acc)[NT], bool from_bias) {
#pragma unroll
        for (int j = 0; j < NT; j++)
            acc[j] = from_bias ? *reinterpret_cast<const i32x4*>(&s_bias[tb + cbl * BCH + c4 * (4 * NT) + j * 4]) : i32x4{0, 0, 0, 0};
#pragma unroll
        for (int ks = 0; ks < KS; ks++)
#pragma unroll
            for (int j = 0; j < NT; j++) acc[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wb[cbl][j][ks], f[ks], acc[j], 0, 0, 0);
        // (a condition between MFMAs and the first reader of their results, which has to come eight issue slots behind: a unit has two MFMAs at the least, the
        // second of which the matrix unit takes when it is through with the first, and the compiler keeps the slots of the last on both sides of the branch)
        if (rt) {
#pragma unroll
            for (int j = 0; j < NT; j++) acc[j] += rowterm;
        }
    };
    // The wave's tile: 16 rows of NCH bytes, padded to 2 mod 4 sixteen-byte pieces per row (the 16-row x 4-piece pattern
    // of a wave's writes without bank conflicts).  Piece p of the tile is piece p % PPR of row p / PPR; lane L writes pieces
    // L, L + 64, ...
    // (the host sends layers here whose output rows are a fixed pitch apart, 16-byte aligned, N a multiple of 16)
    constexpr int kTileStride = NCH + 32, PPR = NCH / 16;
    __shared__ __attribute__((aligned(16))) uint8_t s_tile[kRegbWaves][16 * kTileStride];
    uint8_t* const tile_w = &s_tile[w][n16 * kTileStride + c4 * (4 * NT)];
    auto write_out = [&](int b) {
#pragma unroll
        for (int p = lane; p < 16 * PPR; p += 64) {
            const int row = p / PPR, piece = p % PPR;
            const i32x4 v = *reinterpret_cast<const i32x4*>(&s_tile[w][row * kTileStride + piece * 16]);  // (LDS serves a wave's accesses in order)
            const int64_t m = (int64_t)b * 16 + row;
            const int col = n0 + piece * 16;
            i32x4* const dst = reinterpret_cast<i32x4*>(out + (m * ldc + col));
            if (m < M && col < N) {
                if (past_cache) {
                    __builtin_nontemporal_store(v, dst);
                } else {
                    asm volatile("");  // (without the two, both stores are compiled to one plain one)
                    *dst = v;
                    asm volatile("");
                }
            }
        }
    };
    auto one_block = [&](int b, const i32x4 (&a)[KS], auto general_c) {
        constexpr bool GENERAL = decltype(general_c)::value;
        i32x4 f[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ks++) f[ks] = a[ks] ^ sign_flip;  // unsigned input: the top bit of every byte
        const int rowterm = rt ? rt[(int64_t)b * 16 + n16] : 0;  // (padded past the last row: an edge block may read ahead)
#pragma unroll
        for (int cbl = 0; cbl < CBW; cbl++) {
            i32x4 acc[NT];
            multiply(cbl, f, rowterm, acc, !GENERAL);
            if constexpr (GENERAL) {
                // Every PPE setting, in the integer form the compiler programs.  Rare (scales above 1/2, odd zero
                // points, slopes above one) and long: one copy of the arithmetic walks the lane's sums through LDS.
                __shared__ int sums[kRegbWaves][4 * NT][64];
#pragma unroll
                for (int j = 0; j < NT; j++)
#pragma unroll
                    for (int r = 0; r < 4; r++) sums[w][j * 4 + r][lane] = acc[j][r];
                const Ppe p{ppe.prelu_mult, ppe.prelu_shift, ppe.zp_out, ppe.lo, ppe.hi, 0.f, 0.f};
#pragma unroll 1
                for (int i = 0; i < 4 * NT; i++) {  // channel n0 + BCH * cbl + 4 * NT * c4 + i
                    const uint32_t w2 = (uint32_t)s_w2[tb + cbl * BCH + c4 * (4 * NT) + i];
                    const ChanParams c{s_bias[tb + cbl * BCH + c4 * (4 * NT) + i], (int)(int16_t)(w2 >> 16), (int)((w2 >> 8) & 0xffu)};
                    tile_w[cbl * BCH + i] = (uint8_t)ppe_requant(sums[w][i][lane], c, p);
                }
            } else {
                unsigned o[NT];
#pragma unroll
                for (int j = 0; j < NT; j++) {
                    unsigned v = 0;
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const int ci = tb + cbl * BCH + c4 * (4 * NT) + j * 4 + r;
                        v |= ppe_one_biased<!SAME_F>(acc[j][r], s_fpos[ci], SAME_F ? 0.0 : s_fneg[ci], pk) << (8 * r);
                    }
                    o[j] = v ^ pk.flip;
                }
                if constexpr (NT == 4) {
                    *reinterpret_cast<i32x4*>(tile_w + cbl * BCH) = i32x4{(int)o[0], (int)o[1], (int)o[2], (int)o[3]};
                } else {
#pragma unroll
                    for (int j = 0; j < NT; j++) *reinterpret_cast<unsigned*>(tile_w + cbl * BCH + j * 4) = o[j];
                }
            }
        }
        write_out(b);
    };
    if (general) {  // (nothing fetched ahead)
        for (int b = stream; b < nblk; b += streams) {
            fetch(b, a[0]);
            one_block(b, a[0], std::true_type{});
        }
    } else {
        for (int b = stream; b < nblk; b += (kPrefetch + 1) * streams) {
#pragma unroll
            for (int p = 0; p <= kPrefetch; p++) {
                const int bb = b + p * streams;
                if (bb >= nblk) break;
                if (bb + kPrefetch * streams < nblk) fetch(bb + kPrefetch * streams, a[(p + kPrefetch) % (kPrefetch + 1)]);
                one_block(bb, a[p], std::false_type{});
            }
        }
    }
}

}  // namespace

// The shape of the work: blocks of 16 * `nt` channels, `cbw` of them per wave, `gw` groups of those per workgroup.
// nt and gw: what leaves least of the launch empty -- a lane's PPE runs over the empty part of a last block too, and the
// last workgroup's waves past the last block idle -- where a gw of two or four counts for a good deal, since the waves of
// a workgroup then share its rows ([24341 x 64] . [64 x 464]: fifteen blocks of 32 channels one to a workgroup 12.1 us,
// eight of 64 four to a workgroup 7.0).
// cbw: as many as keep the weights within 64 registers and divide the number of blocks -- whole pieces of output rows
// per store -- where the rows are many enough for units of that size to fill the waves evenly (about six row blocks per
// wave: [401408 x 64] . [64 x 256] 30.5 us with four blocks per wave, 34.1 with one; [100352 x 64] . [64 x 256] 11.8
// against 10.2 us); else one.
// us: what the launch should take, fitted (non-negative least squares, median error 5 %, one tenth beyond 15) to 986 layers of 200 ...
// 30 000 rows, K 16 ... 256, 16 ... 1024 channels, the mean of one set of buffers and of rotating ones: the launch and the weights, the busiest
// wave's walk, the compute unit's share of the arithmetic, of the row loads and of the weight loads, memory.
RegbShape gemm_regb_shape(int64_t M, int64_t N, int64_t K, int cus, bool same_f, bool widest) {
    const int ks = (int)((K + 63) / 64);
    const int64_t nblk = (M + 15) / 16;
    const auto finish = [&](RegbShape r) {
        const int64_t tiles = (int64_t)r.nt * r.cbw, per = 16 * tiles * r.gw, supers = (N + per - 1) / per, blocks = supers * r.gw;
        const int64_t wgs = ((int64_t)cus * regb_waves_per_simd(same_f, ks, r.cbw, r.nt) + supers - 1) / supers * supers;
        const int64_t streams = wgs / supers * (kRegbWaves / r.gw), walks = (nblk + streams - 1) / streams;
        const int64_t per_cu = (std::min(wgs, (nblk + kRegbWaves / r.gw - 1) / (kRegbWaves / r.gw) * supers) + cus - 1) / cus;
        const bool shared = r.gw == 1 && ks >= 2;  // (SHARE above)
        r.us = 2.13 + 0.036 * (double)(ks * tiles) + (double)walks * (0.059 * ks + 0.061 * (double)tiles) +
               (double)(nblk * blocks) / cus * (0.0165 * (double)tiles + 0.028 * ks / r.gw) + 0.0125 * (double)(per_cu * ks * tiles * (shared ? 1 : 4)) +
               0.035e-6 * (double)(M * (K + N));
        return r;
    };
    const int64_t cb_total = (N + 63) / 64;
    int cbw = K > 128 ? 1 : (K > 64 ? 2 : 4);
    while (cb_total % cbw) cbw /= 2;
    const int64_t streams = (int64_t)cus * 3 * kRegbWaves / (cb_total / cbw);
    if (cbw > 1 && N % 64 == 0 && ((M + 15) / 16 >= 6 * streams || widest)) {
        int gw = 4 / cbw;
        while (cb_total / cbw % gw) gw /= 2;
        return finish(RegbShape{4, cbw, gw, 0.0});
    }
    RegbShape best{4, 1, 1, 0.0};
    double least = 0;
    for (int nt = 4; nt >= 2; nt--)
        for (int gw = 4; gw >= 1; gw /= 2) {
            const int64_t blocks = (N + 16 * nt - 1) / (16 * nt), padded = (blocks + gw - 1) / gw * gw;
            const double cost = (double)(padded * nt) * (gw == 4 || blocks <= gw ? 1.0 : gw == 2 ? 1.12 : 1.35);
            if (least == 0 || cost < least) {
                least = cost;
                best = RegbShape{nt, 1, gw, 0.0};
            }
        }
    return finish(best);
}

// Workgroups (of one wave per SIMD) a compute unit holds at once.
int gemm_regb_workgroups_per_cu(bool same_f, int64_t K, const RegbShape& r) { return regb_waves_per_simd(same_f, (int)((K + 63) / 64), r.cbw, r.nt); }

int launch_gemm_regb(const GemmLaunch& a, const RegbShape& r, int workgroups, hipStream_t s) {
    const int per = 16 * r.nt * r.cbw * r.gw, supers = (int)((a.N + per - 1) / per);
    const bool same_f = a.ppe.prelu_mult == 1 && a.ppe.prelu_shift == 0;
    const int ks = (int)((a.K + 63) / 64);
    const int sign_flip = a.in_u8 ? (int)0x80808080 : 0;
    // Stores go past the cache where the waves of a workgroup fill whole 128-byte lines and the result is up to 16 MB.  Through
    // the cache / past it, us, alone: [25088 x 64] . [64 x 256] 6.0 / 5.2, [100352 x 64] . [64 x 128] 9.2 / 7.4, [25088 x 128] . [128
    // x 512] 12.3 / 10.5; with the eltwise that reads the result 11.4 / 10.9, 18.7 / 17.6, 21.7 / 21.2.  A larger one is found in the
    // Infinity Cache by the next call, which gains what the store lost: [100352 x 64] . [64 x 256] 13.7 / 10.7 alone, but in a
    // residual block (three convolutions and the eltwise) 41.2 / 42.5; [401408 x 64] . [64 x 256] 39.3 / 36.3, with the eltwise 84 / 87.
    // Rows that begin inside a line share it with their neighbours and are left to the cache to put together ([100352 x 64] .
    // [64 x 192] 11.8 / 11.8, with the eltwise 23.6 / 24.3).
    const int nch = 16 * r.nt * r.cbw;
    const int past_cache = nch % 64 == 0 && ((a.dst.sw & 127) == 0 || a.dst.sw == nch) && a.M * a.N <= (16ll << 20) ? 1 : 0;
    if (supers < 1 || workgroups % supers != 0 || a.K % 16 != 0) return VPX_RESULT_ERROR_UNKNOWN;
    const auto launch = [&](auto kernel) -> int {
        VPX_LAUNCH(kernel, dim3((unsigned)workgroups), dim3(64 * kRegbWaves), 0, s, a.A, a.B, a.wt, a.out, a.M, (int)a.N, (int)(a.K / 16),
                   a.rows.lda, a.dst.sw, a.ppe, supers, sign_flip, past_cache);
        return VPX_RESULT_SUCCESS;
    };
    const auto unknown = [&] {
        return fail(VPX_RESULT_ERROR_UNKNOWN, "nce_gemm_regb has no form for K = %lld in blocks of %d x %d channels", (long long)a.K, r.cbw, 16 * r.nt);
    };
    const auto by_groups = [&](auto same_c, auto ks_c, auto cbw_c, auto nt_c) {
        constexpr bool SAME = decltype(same_c)::value;
        constexpr int KS = decltype(ks_c)::value, CBW = decltype(cbw_c)::value, NT = decltype(nt_c)::value;
        if (r.gw == 1) return launch(nce_gemm_regb<SAME, KS, CBW, 1, NT>);
        if constexpr (CBW <= 2) {
            if (r.gw == 2) return launch(nce_gemm_regb<SAME, KS, CBW, 2, NT>);
        }
        if constexpr (CBW == 1) {
            if (r.gw == 4) return launch(nce_gemm_regb<SAME, KS, 1, 4, NT>);
        }
        return unknown();
    };
    const auto by_blocks = [&](auto same_c, auto ks_c) {
        constexpr int KS = decltype(ks_c)::value;
        const auto one = std::integral_constant<int, 1>{};
        const auto four = std::integral_constant<int, 4>{};
        if (r.nt == 2 && r.cbw == 1) return by_groups(same_c, ks_c, one, std::integral_constant<int, 2>{});
        if (r.nt == 3 && r.cbw == 1) return by_groups(same_c, ks_c, one, std::integral_constant<int, 3>{});
        if (r.nt == 4 && r.cbw == 1) return by_groups(same_c, ks_c, one, four);
        if constexpr (KS <= 2) {
            if (r.nt == 4 && r.cbw == 2) return by_groups(same_c, ks_c, std::integral_constant<int, 2>{}, four);
        }
        if constexpr (KS == 1) {
            if (r.nt == 4 && r.cbw == 4) return by_groups(same_c, ks_c, four, four);
        }
        return unknown();
    };
    const auto by_length = [&](auto same_c) {
        if (ks == 1) return by_blocks(same_c, std::integral_constant<int, 1>{});
        if (ks == 2) return by_blocks(same_c, std::integral_constant<int, 2>{});
        if (ks == 3) return by_blocks(same_c, std::integral_constant<int, 3>{});
        if (ks == 4) return by_blocks(same_c, std::integral_constant<int, 4>{});
        return unknown();
    };
    return same_f ? by_length(std::true_type{}) : by_length(std::false_type{});
}

}  // namespace nce
}  // namespace vpx
