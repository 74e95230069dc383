// nce_conv_regb: convolutions of a short K onto few output channels (16 to 64) at many positions -- the first layers of image networks, 16, 32 or 48 channels
// under square taps, and wider inputs under few taps (80 under 3x3, 368 under 1x2) -- as nce_gemm_regb.hip's product, with the taps of a position in
// the place of a row of the matrix.
//
// A wave keeps the weights of all its 16 * NT output channels in registers (NT x KS fragments of `v_mfma_i32_16x16x64_i8`, first operand, so that a
// lane's accumulators are neighbouring bytes of the output) and walks blocks of 16 output positions: KS 16-byte loads a lane straight from global
// memory, PF blocks ahead of the arithmetic; no patch, no barrier after the set-up.  A lane's chunk of K step ks is the same tap for
// every block, so its offset under the window is worked out once; a position's place in the input and the output is stepped on from block to block by
// additions.  Only blocks with a tap outside the image look at taps one by one: those read the tensor's first bytes and become padding.
//
// What bounds it is the rate at which the first-level cache serves the fragments (KS kilobytes a block; 7x7 taps, 13 KB, take twice the time of a
// staged patch's reads, which is why more than 16 channels of those stay with the patch kernels), for 3x3 taps memory.  Pairs of fragments dealt so that the
// lanes of a quad read neighbouring words where positions are 32 bytes apart: 4 % slower, it is not the cache's banks.
// us in a HIP graph, nce_conv_rows16 or nce_conv_strips / here: [14,338,585,16] -> 16 3x3 stride 2 24.5 / 12.0, [8,521,314,16] -> 32 13.8 / 9.5,
// [32,224,224,16] -> 32 14.4 / 10.9, [6,349,320,48] -> 32 19.3 / 10.0, [5,593,523,16] -> 16 7x7 stride 2 23.4 / 19.2, [18,88,88,48] -> 48 3x3
// 13.3 / 11.1, [9,367,486,16] -> 64 3x3 stride 2 19.9 / 17.9; nce_direct / here: [3,376,640,16] -> 16 3x3 stride 2 8.0 / 6.0.  Wider inputs, nce_conv_rows16
// or nce_direct / here: [14,109,164,80] -> 16 2x2 12.7 / 8.1, [13,168,87,240] -> 16 3x1 stride 2 25.0 / 7.9, [26,268,159,80] -> 48 2x2 stride 2 34.2 / 20.2, [30,74,79,96]
// -> 16 2x1 8.1 / 6.1; 150 drawn layers of 80 to 368 channels take 0.82 of the time, one is more than 3 % slower ([2,233,391,144] -> 16 1x2 stride 2 4.6 / 4.8).
#include <algorithm>

#include "nce_common.h"

namespace vpx {
namespace nce {
namespace {

constexpr int kWaves = 4;

template <bool SAME_F, int KS, int NT, int PF, int EU>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(EU))) void nce_conv_regb(
    const int8_t* __restrict__ in, const int8_t* __restrict__ wts, const int32_t* __restrict__ wt, uint8_t* __restrict__ out, RegbConvGeom g, GemmPpe ppe,
    int sign_flip) {
    constexpr int TCH = 16 * NT;
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n16 = lane & 15, c4 = lane >> 4;
    // Every die has a run of blocks of its own, which its waves walk side by side: the rows that neighbouring blocks share are in its cache.
    const int nwg = (int)gridDim.x, dies = (nwg & 7) == 0 ? 8 : 1;
    const int die = (int)blockIdx.x & (dies - 1), step = nwg / dies * kWaves;
    const int every = g.nblk / dies, more = g.nblk - every * dies;
    const int last = (die + 1) * every + (die + 1 < more ? die + 1 : more);
    const int first = die * every + (die < more ? die : more) + ((int)blockIdx.x / dies) * kWaves + w;

    // ---- the taps: chunk 4 * ks + c4 of a position is this lane's piece of K step ks
    __shared__ int s_tap[4 * KS];  // its row and column under the window
    int toff[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
        const int c = ks * 4 + c4 < g.chunks ? ks * 4 + c4 : 0;  // (past the end: zero weights)
        const int tap = fdiv(c, g.cpp), ky = fdiv(tap, g.kx), kx = tap - ky * (int)g.kx.d;
        toff[ks] = ky * g.ish + kx * g.isw + (c - tap * (int)g.cpp.d) * 16;
        if (tid < 64 && n16 == 0) s_tap[ks * 4 + c4] = ky | kx << 16;
    }
    i32x4 wb[NT][KS];
#pragma unroll
    for (int j = 0; j < NT; j++) {
        const int ch = (n16 >> 2) * (4 * NT) + j * 4 + (n16 & 3);
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const int c = ks * 4 + c4;
            wb[j][ks] = *reinterpret_cast<const i32x4*>(wts + ((int64_t)ch * g.chunks + (c < g.chunks ? c : 0)) * 16);
        }
    }
    const int2 words = *reinterpret_cast<const int2*>(wt + (tid < TCH ? tid : 0) * 4 + 2);
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
        for (int ks = 0; ks < KS; ks++)
#pragma unroll
            for (int q = 0; q < 4; q++) wb[j][ks][q] = ks * 4 + c4 < g.chunks ? wb[j][ks][q] : 0;

    __shared__ double s_fpos[TCH], s_fneg[TCH];
    __shared__ __attribute__((aligned(16))) int s_bias[TCH], s_sum[TCH];
    __shared__ int s_w2[TCH], s_general;
    if (ppe.corr != 0) {
        const i32x4 ones = i32x4{0x01010101, 0x01010101, 0x01010101, 0x01010101};
#pragma unroll
        for (int j = 0; j < NT; j++)
            if (j % kWaves == w) {
                i32x4 sum = i32x4{0, 0, 0, 0};
#pragma unroll
                for (int ks = 0; ks < KS; ks++) sum = __builtin_amdgcn_mfma_i32_16x16x64_i8(wb[j][ks], ones, sum, 0, 0, 0);
                if (n16 == 0) *reinterpret_cast<i32x4*>(&s_sum[c4 * (4 * NT) + j * 4]) = sum;
            }
        __syncthreads();
    }
    const PpePack pk = make_ppe_pack(ppe.zp_out, ppe.lo, ppe.hi, ppe.out_signed != 0);
    if (tid < 64) {
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
        if (tid == 0) s_general = special ? 1 : 0;
    }
    __syncthreads();
    const bool general = __builtin_amdgcn_readfirstlane(s_general) != 0;
    const int32_t* const rt = ppe.rowterm;
    const int pad = g.pad32 ^ sign_flip;

    // What a block of 16 positions needs from its fetch to its result: the fragments, the lane's place in the output (-1: none), which of
    // its chunks are inside the image, and whether any lane's are not.
    struct Block {
        i32x4 a[KS];
        int at;
        unsigned inside;
        bool border;
    };
    // This lane's position of the block to fetch next, and where it lies in the operands: stepped on from block to block, no divisions.
    int p = first * 16 + n16, oy, ox;
    unsigned src, dst;  // (past the last position: any value, not used)
    {
        const int q = p < g.P ? p : 0;
        const unsigned img = quotient((unsigned)q, (unsigned)g.ohow, g.ohow_magic), rem = (unsigned)q - img * (unsigned)g.ohow;
        oy = (int)quotient(rem, (unsigned)g.ow, g.ow_magic);
        ox = (int)rem - oy * g.ow;
        src = img * (unsigned)g.isn + (unsigned)((oy * g.SY - g.PT) * g.ish + (ox * g.SX - g.PL) * g.isw);
        dst = img * (unsigned)g.osn + (unsigned)(oy * g.osh + ox * g.osw + c4 * (4 * NT));
    }
    const unsigned by = (unsigned)step * 16, by_img = by / (unsigned)g.ohow, by_rem = by - by_img * (unsigned)g.ohow, by_oy = by_rem / (unsigned)g.ow,
                   by_ox = by_rem - by_oy * (unsigned)g.ow;
    const unsigned isy = (unsigned)(g.SY * g.ish), isx = (unsigned)(g.SX * g.isw);
    const unsigned src_step = by_img * (unsigned)g.isn + by_oy * isy + by_ox * isx, src_row = isy - (unsigned)g.ow * isx, src_img = (unsigned)g.isn - (unsigned)g.OH * isy;
    const unsigned dst_step = by_img * (unsigned)g.osn + by_oy * (unsigned)g.osh + by_ox * (unsigned)g.osw, dst_row = (unsigned)(g.osh - g.ow * g.osw),
                   dst_img = (unsigned)(g.osn - g.OH * g.osh);
    auto fetch = [&](Block& k) __attribute__((always_inline)) {
        const bool there = p < g.P;
        k.at = there ? (int)dst : -1;
        k.border = __builtin_amdgcn_ballot_w64(!(there & ((unsigned)(oy - g.oy_lo) < (unsigned)g.oy_n) & ((unsigned)(ox - g.ox_lo) < (unsigned)g.ox_n))) != 0;
        unsigned off[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ks++) off[ks] = src + (unsigned)toff[ks];
        if (k.border) {
            const int iy0 = oy * g.SY - g.PT, ix0 = ox * g.SX - g.PL;
            k.inside = 0;
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {
                const int t = s_tap[ks * 4 + c4];
                const bool ok = there & ((unsigned)(iy0 + (t & 0xffff)) < (unsigned)g.H) & ((unsigned)(ix0 + (t >> 16)) < (unsigned)g.W);
                off[ks] = ok ? off[ks] : 0;
                k.inside |= ok ? 1u << ks : 0u;
            }
        }
        p += (int)by;
        oy += (int)by_oy;
        ox += (int)by_ox;
        src += src_step;
        dst += dst_step;
        const bool row = ox >= g.ow;
        ox -= row ? g.ow : 0;
        oy += row ? 1 : 0;
        src += row ? src_row : 0u;
        dst += row ? dst_row : 0u;
        const bool img = oy >= g.OH;
        oy -= img ? g.OH : 0;
        src += img ? src_img : 0u;
        dst += img ? dst_img : 0u;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) k.a[ks] = *reinterpret_cast<const i32x4*>(in + off[ks]);
    };
    auto one_block = [&](int b, Block& k, auto general_c) __attribute__((always_inline)) {
        constexpr bool GENERAL = decltype(general_c)::value;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) k.a[ks] = k.a[ks] ^ sign_flip;
        if (k.border) {
#pragma unroll
            for (int ks = 0; ks < KS; ks++)
#pragma unroll
                for (int q = 0; q < 4; q++) k.a[ks][q] = (k.inside >> ks & 1) != 0 ? k.a[ks][q] : pad;
        }
        i32x4 acc[NT];
#pragma unroll
        for (int j = 0; j < NT; j++) acc[j] = GENERAL ? i32x4{0, 0, 0, 0} : *reinterpret_cast<const i32x4*>(&s_bias[c4 * (4 * NT) + j * 4]);
        // (In front of the MFMAs.  Behind them the branch came, from the compiler, without the wait states that the first reader of a result needs:
        // with one MFMA in the last step the first of a lane's four sums was read too early.)
        if (rt) {
            const int v = rt[(int64_t)b * 16 + n16];  // (padded past the last position)
#pragma unroll
            for (int j = 0; j < NT; j++) acc[j] += v;
        }
#pragma unroll
        for (int ks = 0; ks < KS; ks++)
#pragma unroll
            for (int j = 0; j < NT; j++) acc[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wb[j][ks], k.a[ks], acc[j], 0, 0, 0);
        unsigned o[NT];
        if constexpr (GENERAL) {
            // Every PPE setting, in the integer form the compiler programs: rare and long, one copy walks the lane's sums through LDS.
            __shared__ int sums[kWaves][4 * NT][64];
#pragma unroll
            for (int j = 0; j < NT; j++)
#pragma unroll
                for (int r = 0; r < 4; r++) sums[w][j * 4 + r][lane] = acc[j][r];
            const Ppe p{ppe.prelu_mult, ppe.prelu_shift, ppe.zp_out, ppe.lo, ppe.hi, 0.f, 0.f};
#pragma unroll 1
            for (int i = 0; i < 4 * NT; i++) {
                const uint32_t w2 = (uint32_t)s_w2[c4 * (4 * NT) + i];
                const ChanParams c{s_bias[c4 * (4 * NT) + i], (int)(int16_t)(w2 >> 16), (int)((w2 >> 8) & 0xffu)};
                sums[w][i][lane] = ppe_requant(sums[w][i][lane], c, p);
            }
#pragma unroll
            for (int j = 0; j < NT; j++) {
                o[j] = 0;
#pragma unroll
                for (int r = 0; r < 4; r++) o[j] |= ((unsigned)sums[w][j * 4 + r][lane] & 0xffu) << (8 * r);
            }
        } else {
#pragma unroll
            for (int j = 0; j < NT; j++) {
                unsigned v = 0;
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int ci = c4 * (4 * NT) + j * 4 + r;
                    v |= ppe_one_biased<!SAME_F>(acc[j][r], s_fpos[ci], SAME_F ? 0.0 : s_fneg[ci], pk) << (8 * r);
                }
                o[j] = v ^ pk.flip;
            }
        }
        if (k.at >= 0) {
            typedef unsigned Word __attribute__((aligned(1)));
            typedef unsigned Pair __attribute__((ext_vector_type(2), aligned(1)));
            uint8_t* const to = out + (unsigned)k.at;
            if constexpr (NT == 1) *reinterpret_cast<Word*>(to) = o[0];
            else if constexpr (NT == 2) *reinterpret_cast<Pair*>(to) = Pair{o[0], o[1]};
            else if constexpr (NT == 3) {
                *reinterpret_cast<Pair*>(to) = Pair{o[0], o[1]};
                *reinterpret_cast<Word*>(to + 8) = o[2];
            } else *reinterpret_cast<i32x4_any*>(to) = i32x4{(int)o[0], (int)o[1], (int)o[2], (int)o[NT - 1]};
        }
    };
    Block k[PF + 1];
    if (general) {  // (nothing fetched ahead)
        for (int b = first; b < last; b += step) {
            fetch(k[0]);
            one_block(b, k[0], std::true_type{});
        }
    } else {
#pragma unroll
        for (int u = 0; u < PF; u++)
            if (first + u * step < last) fetch(k[u]);
        for (int b = first; b < last; b += (PF + 1) * step) {
#pragma unroll
            for (int u = 0; u <= PF; u++) {
                const int bb = b + u * step;
                if (bb >= last) break;
                if (bb + PF * step < last) fetch(k[(u + PF) % (PF + 1)]);
                one_block(bb, k[u], std::false_type{});
            }
        }
    }
}

}  // namespace

int launch_conv_regb(const RegbConvLaunch& a, hipStream_t s) {
    const bool same_f = a.ppe.prelu_mult == 1 && a.ppe.prelu_shift == 0;
    const int sign_flip = a.in_u8 ? (int)0x80808080 : 0, ks = (a.g.chunks + 3) / 4;
    const auto launch = [&](auto kernel, int per_cu) -> int {
        // as many as are resident at once, or one for every four blocks; whole dies
        const int64_t wgs = std::min<int64_t>((int64_t)a.cus * per_cu, ((int64_t)a.g.nblk + 8 * kWaves - 1) / (8 * kWaves) * 8);
        VPX_LAUNCH(kernel, dim3((unsigned)wgs), dim3(64 * kWaves), 0, s, a.in, a.w, a.wt, a.out, a.g, a.ppe, sign_flip);
        return VPX_RESULT_SUCCESS;
    };
    const auto by_taps = [&](auto same_c, auto nt_c) -> int {
        constexpr bool SAME = decltype(same_c)::value;
        constexpr int NT = decltype(nt_c)::value;
        if constexpr (NT != 3) {
            constexpr int EU = NT == 4 ? 2 : (SAME ? 6 - NT : 3);
            if (ks <= 3) return launch(nce_conv_regb<SAME, 3, NT, 2, EU>, EU);
        }
        if constexpr (NT <= 2) {
            if (ks <= 5) return launch(nce_conv_regb<SAME, 5, NT, NT == 1 ? 2 : 1, 3>, 3);
        }
        if constexpr (NT <= 3) {
            if (ks <= 7) return launch(nce_conv_regb<SAME, 7, NT, 1, NT == 1 ? 3 : 2>, NT == 1 ? 3 : 2);
        }
        if constexpr (NT == 1) {
            if (ks <= 13) return launch(nce_conv_regb<SAME, 13, 1, 1, 2>, 2);
        }
        return fail(VPX_RESULT_ERROR_UNKNOWN, "nce_conv_regb has no form for %d chunks", a.g.chunks);
    };
    const auto by_channels = [&](auto same_c) -> int {
        if (a.nt == 1) return by_taps(same_c, std::integral_constant<int, 1>{});
        if (a.nt == 2) return by_taps(same_c, std::integral_constant<int, 2>{});
        if (a.nt == 3) return by_taps(same_c, std::integral_constant<int, 3>{});
        return by_taps(same_c, std::integral_constant<int, 4>{});
    };
    return same_f ? by_channels(std::true_type{}) : by_channels(std::false_type{});
}

}  // namespace nce
}  // namespace vpx
