// nce_conv_strips: the row-patch convolution of nce_conv_rows.hip (same implicit product, same LDS layouts of rows and weights)
// with a patch per wave: for layers of more than 32 output channels with taps, byte output, whose weights and eight small
// patches fit LDS together.
//
// There the eight waves of a workgroup share one patch and go through load, MFMA loop, PPE and stores in step, two barriers a
// tile; MFMA loops were half of a stem's time.  Here a wave owns a tile of 64 positions (16 columns x 4 rows, 8 x 8, or 32 x 2) with
// the input rows under it, walks its own run of tiles down a column of tiles and meets nobody after the weights are staged, so
// that one wave's MFMAs cover the other's PPE, stores and row writes.  The next tile's rows travel in registers while a tile
// is computed (a row per load: its first byte is a scalar, the lane's offset the same for every row and tile).
// What bounds it (7x7 x 16 channels -> 64, stride 2, 401 408 positions, clocks of a wave): launch to the first MFMA 11 000, most of it the first
// rows and the weights on their way; then 10 000 for the two tiles of a SIMD, of which the MFMAs are 6 400; 3 or 4 tiles a wave.
// Tiles of 128 positions need half the weight reads but leave no registers for rows that travel ahead (their waits, 13 000
// clocks a tile, cost more: 45 us); weights in registers and the PPE of one tile between the MFMAs of the next, one wave a SIMD, 91 us.
// us against nce_conv_rows16 (HIP graph, rotating buffers): [32,224,224,16] -> 64 7x7 stride 2 33 / 42 (on images, whose padding channels are
// constant, 27 / 38), [8,521,314,16] -> 64 3x3 stride 2 19.9 / 26.3, [32,112,112,32] -> 64 3x3 23.6 / 31.8, [1,640,640,16] -> 64 7x7 stride 2
// 14.3 / 18.7, [16,56,56,48] -> 96 3x3 11.5 / 13.6; layers of 32 channels have half the MFMAs per patch read (17.0 / 15.8) and 1x1 layers no
// rows to share (12.5 / 12.2 at [32,28,28,96] -> 200): both stay there.
#include "nce_common.h"

namespace vpx {
namespace nce {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
constexpr int kStripRows = 14;  // rows that travel ahead, in registers

template <bool IN_U8, bool REST>
__global__ __launch_bounds__(64 * kStripWaves) void nce_conv_strips(const int8_t* __restrict__ in, const int8_t* __restrict__ w,
                                                                     const int32_t* __restrict__ wt, uint8_t* __restrict__ out, StripGeom g, GemmPpe ppe) {
    constexpr int TM = 2, TN = 2, BN = 32 * TN, NT = 64 * kStripWaves;  // blocks of 32 positions and of 32 channels per tile
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    uint8_t* const wlds = smem;                                             // [BN][WS], rows in tile order
    ChanPrep* const sprep = reinterpret_cast<ChanPrep*>(smem + BN * g.WS);  // [BN], by channel
    int* const sbias = reinterpret_cast<int*>(sprep + BN);                  // [BN] biases, [BN] row sums, one flag
    int* const csum = sbias + BN;
    int* const sflag = csum + BN;
    int* const stab = sflag + 4;                                            // [S + 8][2] fragment offsets, by step and lane half

    const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int S = g.S, kc = 2 * S, nchunks = g.nchunks, OC = g.OC;
    uint8_t* const patch = reinterpret_cast<uint8_t*>(stab + (kc + 19) / 4 * 4) + wave * g.patch_bytes;  // [PH][RB], this wave's own
    const int oc0 = blockIdx.y * BN;
    const int nwg = (int)gridDim.x;
    // Every wave walks its own run of tiles, down a column of tiles; workgroups of one die are neighbours in their order.
    const int per_die = nwg >> 3, b = (nwg & 7) == 0 ? (int)(blockIdx.x & 7) * per_die + (int)(blockIdx.x >> 3) : (int)blockIdx.x;
    // (`every` tiles each and one more for `more` waves, dealt out a wave of every workgroup at a time)
    const int q = g.more / nwg, r = g.more - q * nwg, extra = q + (b < r ? 1 : 0);
    const int first = (b * kStripWaves + wave) * g.every + b * q + (b < r ? b : r) + (wave < extra ? wave : extra);
    const int last = first + g.every + (wave < extra ? 1 : 0);

    // ---- a tile's input rows -> this wave's patch, a row per instruction (two where a row has more than 64 chunks); padding
    // and the sign flip applied here.  What a lane holds of a row does not depend on the tile: worked out once.
    constexpr int GROUPS = REST ? 2 : 1, ROWS = kStripRows;
    const int flip = IN_U8 ? (int)0x80808080 : 0, pad = g.pad32 ^ flip;
    int lsrc[GROUPS], ldst[GROUPS], lcol[GROUPS];
#pragma unroll
    for (int u = 0; u < GROUPS; u++) {
        int q = lane + 64 * u;
        q = q < g.row_chunks ? q : g.row_chunks - 1;  // (lanes past the end repeat the last chunk)
        const int px = fdiv(q, g.cpp), qd = fdiv(q, g.fm);
        lcol[u] = px;
        lsrc[u] = px * g.isw + (q - px * (int)g.cpp.d) * 16;
        ldst[u] = ((q - qd * g.m) * g.plane + qd) * 16;
    }
    struct TilePos {
        int img, oy0, ox0;
    };
    const auto tile_pos = [&](int tile_) {  // tiles in the order (image, column of tiles, tile)
        const int tc = fdiv(tile_, g.tiles_y), ty = tile_ - tc * (int)g.tiles_y.d;
        const int img = fdiv(tc, g.tiles_x);
        return TilePos{img, ty * g.R, (tc - img * (int)g.tiles_x.d) << g.cw_log};
    };
    i32x4 ahead[ROWS];
    // (A row's place in its image is wave-uniform, the lane's offset the same for all rows: a scalar and a vector offset of a buffer that is the
    // image.  As one address per lane the compiler multiplies 64 bits wide for every row.  Rows outside the image read the border row.)
    const auto image = [&](int img) __attribute__((always_inline)) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(in) + (int64_t)img * g.isn, (short)0, -1, 0x00020000);
    };
    const auto load_row = [&](const __amdgpu_buffer_rsrc_t& img, int y, int col) __attribute__((always_inline)) {
        const int row = (y < 0 ? 0 : (y < g.H ? y : g.H - 1)) * g.ish;
        return __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(img, col, row, 0));
    };
    // byte offset of group u's chunk in a row, from the row's first pixel; a column outside the image reads the pixel at the border
    const auto column = [&](int ix0, auto u_c) __attribute__((always_inline)) {
        constexpr int u = decltype(u_c)::value;
        const int x = ix0 + lcol[u];
        return ix0 * g.isw + lsrc[u] + ((unsigned)x < (unsigned)g.W ? 0 : (x < 0 ? -x : g.W - 1 - x) * g.isw);
    };
    constexpr std::integral_constant<int, 0> g0{};
    constexpr std::integral_constant<int, 1> g1{};
    const auto load_patch = [&](const TilePos& tp) __attribute__((always_inline)) {
        const int iy0 = tp.oy0 * g.SY - g.PT, col = column(tp.ox0 * g.SX - g.PL, g0);
        const auto img = image(tp.img);
#pragma unroll
        for (int r = 0; r < ROWS; r++) ahead[r] = load_row(img, iy0 + (r < g.PH ? r : 0), col);
    };
    const auto store_patch = [&](const TilePos& tp) __attribute__((always_inline)) {
        const int iy0 = tp.oy0 * g.SY - g.PT, ix0 = tp.ox0 * g.SX - g.PL;
        const auto img = image(tp.img);
        const auto put_rows = [&](auto border_c) __attribute__((always_inline)) {
            constexpr bool BORDER = decltype(border_c)::value;
            const bool ok0 = (unsigned)(ix0 + lcol[0]) < (unsigned)g.W;
            uint8_t* dst = patch + ldst[0];
#pragma unroll
            for (int r = 0; r < ROWS; r++) {
                if (r >= g.PH) break;
                i32x4 v = ahead[r] ^ flip;
                if (BORDER) {
                    const bool ok = ok0 && (unsigned)(iy0 + r) < (unsigned)g.H;
#pragma unroll
                    for (int q = 0; q < 4; q++) v[q] = ok ? v[q] : pad;
                }
                *reinterpret_cast<i32x4*>(dst) = v;
                dst += g.RB;
            }
        };
        if (iy0 >= 0 && ix0 >= 0 && iy0 + g.PH <= g.H && ix0 + g.PW <= g.W) put_rows(std::false_type{});
        else put_rows(std::true_type{});
        const auto rest = [&](int r0, auto u_c) __attribute__((always_inline)) {  // what does not travel ahead: four rows a round trip
            constexpr int u = decltype(u_c)::value;
            const int col = column(ix0, u_c);
            const bool ok0 = (unsigned)(ix0 + lcol[u]) < (unsigned)g.W;
            for (; r0 < g.PH; r0 += 4) {
                i32x4 v[4];
#pragma unroll
                for (int r = 0; r < 4; r++) v[r] = load_row(img, iy0 + r0 + r, col);
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const bool ok = ok0 && (unsigned)(iy0 + r0 + r) < (unsigned)g.H;
                    i32x4 x = v[r] ^ flip;
#pragma unroll
                    for (int q = 0; q < 4; q++) x[q] = ok ? x[q] : pad;
                    if (r0 + r < g.PH) *reinterpret_cast<i32x4*>(patch + ((r0 + r) * g.RB + ldst[u])) = x;
                }
            }
        };
        if constexpr (REST) {
            if (g.PH > ROWS) rest(ROWS, g0);
            if (g.row_chunks > 64) rest(0, g1);
        }
    };

    int wt2 = 0, wt3 = 0;  // this thread's channel of the weight table, asked for before anything else
    if (tid < BN) {
        const int n = oc0 + tid < OC ? oc0 + tid : OC - 1;
        wt2 = wt[n * 4 + 2];
        wt3 = wt[n * 4 + 3];
    }
    TilePos tp = tile_pos(first < last ? first : 0);

    // ---- weights -> LDS, once; the table of fragment offsets
    for (int q0 = tid; q0 < BN * kc || q0 == tid; q0 += 8 * NT) {  // (the batch's loads before the first write; what is past the end repeats the first chunk)
        i32x4 v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int q = q0 + u * NT < BN * kc ? q0 + u * NT : 0, n = fdiv(q, g.kc), c = q - n * kc;
            const int oc = oc0 + n < OC ? oc0 + n : OC - 1;  // channels past the end repeat the last one
            v[u] = *reinterpret_cast<const i32x4*>(w + ((int64_t)oc * nchunks + (c < nchunks ? c : 0)) * 16);
            if (c >= nchunks) v[u] = i32x4{0, 0, 0, 0};
        }
        if (q0 == tid) load_patch(tp);  // (behind the first batch)
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int q = q0 + u * NT < BN * kc ? q0 + u * NT : 0, n = fdiv(q, g.kc), c = q - n * kc;
            const int lrow = (n & ~31) + 8 * ((n >> 2) & 3) + 4 * ((n >> 4) & 1) + (n & 3);
            *reinterpret_cast<i32x4*>(wlds + lrow * g.WS + c * 16) = v[u];
        }
    }
    for (int c = tid; c < kc + 16; c += NT) {
        const int ky = fdiv(c, g.rin), e = c - ky * (int)g.rin.d;
        const int ed = fdiv(e, g.fm);
        stab[c] = c < nchunks ? ky * g.RB + ((e - ed * g.m) * g.plane + ed) * 16 : 0;  // (chunks past the end: zero weights, any bytes)
    }
    __syncthreads();
    {  // the sums of the weight rows, for the zero-point term
        constexpr int PER = NT / BN;  // threads a row
        const int n = tid / PER, part = tid % PER;
        const int lrow = (n & ~31) + 8 * ((n >> 2) & 3) + 4 * ((n >> 4) & 1) + (n & 3);
        int sum = 0;
        if (ppe.corr != 0) {
#pragma unroll 4
            for (int c = part; c < kc; c += PER) {
                const i32x4 q = *reinterpret_cast<const i32x4*>(wlds + lrow * g.WS + c * 16);
#pragma unroll
                for (int j = 0; j < 4; j++) sum = __builtin_amdgcn_sdot4(q[j], 0x01010101, sum, false);
            }
#pragma unroll
            for (int o = 1; o < PER; o *= 2) sum += __shfl_xor(sum, o);
        }
        if (part == 0) csum[n] = sum;
    }
    __syncthreads();
    const PpePack pk = make_ppe_pack(ppe.zp_out, ppe.lo, ppe.hi, ppe.out_signed != 0);
    if (tid < BN) {
        const uint32_t w2 = (uint32_t)wt2;
        const ChanPrep c = ppe_prepare((int)(int16_t)(w2 >> 16), (int)((w2 >> 8) & 0xffu), (int)((unsigned)wt3 + (unsigned)(ppe.corr * csum[tid])),
                                       ppe.prelu_mult, ppe.prelu_shift);
        sprep[tid] = c;
        sbias[tid] = c.bias;
        // the short PPE serves slopes in [0, 1] (ReLU, LeakyReLU), an even zero-point offset and scales up to 1/2
        const bool slope_ok = (ppe.prelu_mult >= 0 && (ppe.prelu_shift >= 31 || ppe.prelu_mult <= (1 << ppe.prelu_shift)));
        const bool clip = c.bmax_pos != 0x7fffffff || c.bmax_neg != 0x7fffffff;
        const bool general = __builtin_amdgcn_ballot_w64(clip) != 0 || pk.odd != 0 || !slope_ok;
        if (tid == 0) sflag[0] = general ? 1 : 0;
    }
    __syncthreads();  // (the last one: from here on every wave walks its own tiles)
    if (first >= last) return;
    store_patch(tp);
    // PPE kinds.  0: the general form; 1: two factors, the short form (see ppe_pack4_biased); 2: one factor (no PReLU stage, or a
    // slope of zero, which the host turns into a clamp)
    const int kind = __builtin_amdgcn_readfirstlane(sflag[0]) != 0 ? 0 : (ppe.prelu_mult == 1 && ppe.prelu_shift == 0 ? 2 : 1);
    const int q16 = oc0 + half * 16;  // first of the 16 channels this lane stores in channel tile 0
    const int lr = (lane & 31) >> g.cw_log, lc = (lane & 31) & ((1 << g.cw_log) - 1), rows_per_block = 32 >> g.cw_log;
    const uint8_t* pl[TM];
#pragma unroll
    for (int i = 0; i < TM; i++) pl[i] = patch + ((lr + i * rows_per_block) * g.SY * g.RB + lc * 16);
    const uint8_t* wl[TN];
#pragma unroll
    for (int j = 0; j < TN; j++) wl[j] = wlds + ((lane & 31) + 32 * j) * g.WS + half * 16;

    for (int tile = first;;) {
        // the next tile's rows travel while this one is computed (after the last tile: the same rows once more, no branch around the loads)
        const TilePos next = tile_pos(tile + 1 < last ? tile + 1 : tile);
        load_patch(next);
        i32x16 acc[TM][TN];
        {
            // Three fragment buffers: a step's fragments are read two steps ahead of its MFMAs (one step, 128 clocks, is less than
            // an LDS read takes beside the other waves'), their offsets in the patch three steps earlier still.  Past the end
            // the reads go on, at offset 0 of the patch and into the bytes behind the weight rows, and are never used.
            const int* tab = stab + half;
            const uint8_t* wp[TN];
#pragma unroll
            for (int j = 0; j < TN; j++) wp[j] = wl[j];
            i32x4 fa[3][TN], fb[3][TM];
            int poff[3] = {tab[0], tab[2], tab[4]};
            const auto read = [&](auto buf_c, auto at_c) __attribute__((always_inline)) {  // the fragments of step `at` from the pointers
                constexpr int buf = decltype(buf_c)::value, at = decltype(at_c)::value;
#pragma unroll
                for (int j = 0; j < TN; j++) fa[buf][j] = *reinterpret_cast<const i32x4*>(wp[j] + 32 * at);
#pragma unroll
                for (int i = 0; i < TM; i++) fb[buf][i] = *reinterpret_cast<const i32x4*>(pl[i] + poff[buf]);
                poff[buf] = tab[2 * (at + 3)];
                __builtin_amdgcn_sched_barrier(0);
            };
            const auto multiply = [&](auto buf_c) __attribute__((always_inline)) {
                constexpr int buf = decltype(buf_c)::value;
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[buf][j], fb[buf][i], acc[i][j], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            };
            constexpr std::integral_constant<int, 0> k0{};
            constexpr std::integral_constant<int, 1> k1{};
            constexpr std::integral_constant<int, 2> k2{};
            constexpr std::integral_constant<int, 3> k3{};
            constexpr std::integral_constant<int, 4> k4{};
            read(k0, k0);
            read(k1, k1);
            // the accumulators start from the bias
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const i32x4 b4 = *reinterpret_cast<const i32x4*>(sbias + 32 * j + 16 * half + 4 * q);
#pragma unroll
                    for (int r = 0; r < 4; r++)
#pragma unroll
                        for (int i = 0; i < TM; i++) acc[i][j][4 * q + r] = b4[r];
                }
            int s = S;
            for (; s >= 3; s -= 3) {
                read(k2, k2);
                multiply(k0);
                read(k0, k3);
                multiply(k1);
                read(k1, k4);
                multiply(k2);
                tab += 6;
#pragma unroll
                for (int j = 0; j < TN; j++) wp[j] += 96;
            }
            if (s >= 1) multiply(k0);
            if (s >= 2) multiply(k1);
        }
        const int oy = tp.oy0 + lr, ox = tp.ox0 + lc;
        if (ppe.rowterm) {
            const int32_t* const rt = ppe.rowterm + (int64_t)tp.img * g.OH * g.OW;
#pragma unroll
            for (int i = 0; i < TM; i++) {
                const int y = oy + i * rows_per_block;
                const int v = rt[y < g.OH && ox < g.OW ? y * g.OW + ox : 0];
#pragma unroll
                for (int j = 0; j < TN; j++)
#pragma unroll
                    for (int r = 0; r < 16; r++) acc[i][j][r] += v;
            }
        }
        uint8_t* const dst0 = out + (int64_t)tp.img * g.osn + (oy * g.osh + ox * g.osw + q16);
        // Without REST: the image as a buffer that drops what lies past its end, so that no branch makes the number of stores under way unknown (the
        // wait for the next tile's rows would be one for these stores too).
        const auto dst_image = __builtin_amdgcn_make_buffer_rsrc(out + (int64_t)tp.img * g.osn, (short)0, (g.OH - 1) * g.osh + (g.OW - 1) * g.osw + OC, 0x00020000);
        const auto finish = [&](auto kind_c) __attribute__((always_inline)) {
            constexpr int KIND = decltype(kind_c)::value;
#pragma unroll
            for (int j = 0; j < TN; j++) {
                i32x4 o[TM];
#pragma unroll
                for (int i = 0; i < TM; i++) o[i] = i32x4{0, 0, 0, 0};
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const ChanPrep* cpp = sprep + 32 * j + 16 * half + r;
                    if constexpr (KIND == 0) {
                        ChanPrep c = *cpp;  // the form ppe_one takes: sign flip in the bias (which the sums contain), factors swapped for a negative multiplier
                        c.bias = (int)0x80000000u;
                        if (c.sgn) {
                            const double f = c.f_pos;
                            c.f_pos = c.f_neg;
                            c.f_neg = f;
                            const int bm = c.bmax_pos;
                            c.bmax_pos = c.bmax_neg;
                            c.bmax_neg = bm;
                        }
#pragma unroll
                        for (int i = 0; i < TM; i++) o[i][r >> 2] |= (int)(ppe_one<false, true>(acc[i][j][r], c, pk) << (8 * (r & 3)));
                        __builtin_amdgcn_sched_barrier(0);  // (a channel at a time: hoisted, the parameters of all sixteen fill the register file)
                    } else {
                        const double f_pos = cpp->f_pos, f_neg = KIND == 2 ? 0.0 : cpp->f_neg;
#pragma unroll
                        for (int i = 0; i < TM; i++)
                            o[i][r >> 2] |= (int)(ppe_one_biased<KIND == 1>(acc[i][j][r], f_pos, f_neg, pk) << (8 * (r & 3)));
                    }
                }
                const int qc = q16 + 32 * j;
#pragma unroll
                for (int i = 0; i < TM; i++) {
                    o[i] ^= (int)pk.flip;
                    const bool there = (oy + i * rows_per_block < g.OH) & (ox < g.OW) & (qc < OC);
                    if (!REST) {
                        const unsigned at = (unsigned)((oy + i * rows_per_block) * g.osh + ox * g.osw + qc);
                        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, o[i]), dst_image, there ? (int)at : (int)0x80000000, 0, 0);
                        continue;
                    }
                    if (!there) continue;
                    uint8_t* const dst = dst0 + (i * rows_per_block * g.osh + 32 * j);
                    if (qc + 16 <= OC) *reinterpret_cast<i32x4_any*>(dst) = o[i];
                    else
                        for (int e = 0; qc + e < OC; e++) dst[e] = (uint8_t)(o[i][e >> 2] >> (8 * (e & 3)));
                }
            }
        };
        if (kind == 2) finish(std::integral_constant<int, 2>{});
        else if (kind == 1) finish(std::integral_constant<int, 1>{});
        else finish(std::integral_constant<int, 0>{});
        if (++tile >= last) break;
        tp = next;
        __builtin_amdgcn_wave_barrier();  // (the patch is this wave's own: LDS serves a wave's accesses in order)
        store_patch(tp);
        __builtin_amdgcn_wave_barrier();
    }
}

}  // namespace

int launch_conv_strips(const StripLaunch& a, hipStream_t s) {
    const auto launch = [&](auto kernel) -> int {
        const int rc = set_dyn_lds(kernel, a.lds);
        if (rc) return rc;
        VPX_LAUNCH(kernel, a.grid, dim3(64 * kStripWaves), a.lds, s, a.in, a.w, a.wt, a.out, a.sg, a.ppe);
        return VPX_RESULT_SUCCESS;
    };
    // What few layers have is a kernel of its own (REST): patches of more than 14 rows or 64 chunks a row, last chunks of fewer than 16 channels, rows
    // of the output that do not start on words, images of 2^31 elements and more.  In one kernel with the rest it made every tile begin with a wait for
    // the last one's stores.  us, one kernel / two, and row addresses of 64 bits a lane / two offsets: [32,224,224,16] -> 64 7x7 stride 2 30.9 / 29.8,
    // [8,243,563,16] -> 64 3x3 stride 2 16.7 / 15.6, [8,521,314,16] -> 64 5x5 stride 2 22.0 / 21.1, [30,160,37,16] -> 64 3x3 13.5 / 12.7.
    const StripGeom& g = a.sg;
    const int64_t extent = (int64_t)(g.OH - 1) * g.osh + (int64_t)(g.OW - 1) * g.osw + g.OC;
    const bool rest = g.PH > kStripRows || g.row_chunks > 64 || g.OC % 16 != 0 || (g.out_bits & 3) != 0 || extent >= (1ll << 31);
    const int rc = a.in_u8 ? (rest ? launch(nce_conv_strips<true, true>) : launch(nce_conv_strips<true, false>))
                           : (rest ? launch(nce_conv_strips<false, true>) : launch(nce_conv_strips<false, false>));
    if (rc) return rc;
    return VPX_RESULT_SUCCESS;
}

}  // namespace nce
}  // namespace vpx
