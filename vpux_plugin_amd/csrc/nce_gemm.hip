// nce_gemm_mfma: 1x1 kernel, no padding (this is how NCE.MatMul arrives; a stride picks rows from the input), and as nce_conv_gemm
// convolutions of 64 channels and more that fill the chip a few times at most: a plain
// A[M][K] x B[N][K]^T GEMM.  256 x 256, 128 x 128 or 64 x 64 output tile per workgroup, v_mfma_i32_32x32x32_i8, K panels from
// global memory straight into XOR-swizzled LDS (global_load_lds, no register staging), a ring of buffers, the integer PPE
// fused into the epilogue.
#include "nce_common.h"

namespace vpx {
namespace nce {
namespace {

// Sixteen bytes of every value, for the taps of a convolution that lie outside the image.
struct PadTable {
    uint8_t bytes[256][16];
    constexpr PadTable() : bytes{} {
        for (int v = 0; v < 256; v++)
            for (int i = 0; i < 16; i++) bytes[v][i] = (uint8_t)v;
    }
};
__device__ const PadTable g_pads{};

// What a form of the kernel keeps in LDS: the tables of column sums in the head, behind them the panel buffers, which the staging tile
// reuses.  The tables share no byte with the rest: the waves write and read them while panels are still arriving, and while
// faster waves already fill the staging tile.
template <bool IN_U8, int OUT, int NW, int TILE = 256, bool SHORTK = false, bool PP = false, int NS = 4, bool CONV = false>
struct GemmLds {
    // panels of 128 bytes (see WIDE below); else of 64
    static constexpr bool kWide = (TILE == 128 && NW == 8) || TILE == 64 || (TILE == 256 && NS == 2);
    static constexpr int kSumTables = kWide ? 2 : 1;  // one per row of waves that sums columns
    static constexpr int kPanel = 2 * TILE * (kWide ? 128 : 64);
    static constexpr int kStaging = OUT == OUT_F16 ? (TILE == 256 ? 128 : TILE) * (2 * TILE + 32) : TILE * kOutStride;
    static_assert(kSumTables * TILE * (int)sizeof(int) <= kGemmLdsHead, "the column sums end in front of the panel buffers");
    static_assert(SHORTK || kStaging <= NS * kPanel, "the staging tile fits the panel buffers");
    static size_t bytes(int64_t K) {  // of a launch; a short K asks for the panels there are or for the staging tile
        const size_t panels = SHORTK ? (size_t)(K / 64) * kPanel : (size_t)NS * kPanel;
        return kGemmLdsHead + (panels > kStaging ? panels : (size_t)kStaging);
    }
};

// A[M][K] x B[N][K]^T with the PPE fused; see the file header.  K must be a multiple of 64.
//
// Pipeline of the forms below that walk K in panels of 64 bytes (K <= 192, and two that are only run when asked for: the 256 tile
// with four waves, and PP): a panel of A and B (32 KiB of the 256 tile) goes from global memory straight into one of four LDS
// buffers.  In iteration kt the waves multiply panel kt, fetch panel kt+3 (DMA instructions spread between the MFMAs) and read
// the fragments one sub-step ahead; the only wait is for panel kt+1, which was requested two iterations earlier, and it sits
// with the workgroup barrier in the middle of the iteration, between the two sub-steps,
// so that the MFMAs of the second sub-step cover the first fragment reads of panel kt+1.  The column sums of B that the
// zero-point term needs are taken from the fragments as they pass, and the per-column PPE parameters are unpacked from the
// weight table in the epilogue.
//
// PP (eight waves, large tile, K a multiple of four panels): the two waves of a SIMD take turns.  While one runs the
// sixteen MFMAs of a panel back to back at raised priority, the other issues everything else it has to -- the twelve
// fragment reads of its next panel, its four panel loads, the column sums -- and at a workgroup barrier they swap,
// twice per panel.  (With both waves running the same interleaved stream their loads and reads fall on the same
// moments and the MFMA pipe waits for both.)
//
// WIDE (the 256 tile with eight waves of 128 x 64, the 128 tile with eight of 64 x 32, the 64 tile with four of 32 x 32): panels of
// 128 bytes, whole cache lines -- of 64-byte pieces the second of a line came after the first had left the first-level cache, and
// every line was read from the second level twice -- with one barrier each.  The 256 tile has LDS for two such panels, and asks
// for one whenever it has read the last fragment of the one before the last: its panel's MFMAs take 2 048 clocks, and between
// 192.4 us (panels of 64 bytes, four buffers) and 172.0 at [4096 x 4096] . [4096 x 11008], 497 and 451 at 8192^3, 71.3
// and 63.8 at 4096^3 lies only the order of its loads (back to back, the clock settled; beside a dequantize and an add a program sees 243 and 234 in all).  The smaller tiles' loads stand in line far ahead and nobody
// waits for them; a tile of 128 takes about 850 clocks for a panel whose MFMAs take 512, bound by the LDS (96 KiB of
// fragments and 32 KiB of loads), one of 64 about 400, bound likewise.  Four waves of 64 x 64 on
// panels of 64, 24.5 us at [2080 x 3456] . [3456 x 608] whether or not fragments were read a panel ahead or twice the
// panels were in flight, now take 20.2, 16.2 with the 64 tile; [512 x 4096] . [4096 x 4096] 26.9, now 22.0 and 20.7;
// [1024 x 1024] . [1024 x 1024] 9.7, now 8.6 and 6.2.  (Eight waves of 64 x 64 with K split over two groups read a third less
// but hand 64 KiB of sums over: 21.3 at the first.)  Summing the columns in one row of waves only cost 260 clocks a panel
// on the SIMDs that held them; now the waves that share columns take a half of each panel each.
//
// CONV (WIDE, 64 and 128 tiles): a convolution as a matmul over (tap, channel) with nothing laid out for it: row m is an output
// position, and a lane keeps where its 16 bytes of the next panel lie -- tap, chunk of the tap, offset -- and steps them by a panel,
// seven vector instructions; what lies outside the image it fetches from sixteen bytes of padding, what lies past the end of
// K, of the weights, from sixteen zeros.  A panel costs a fifth more than the matmul's ([2000 x 2880] . [2880 x 320] 9.3 us,
// [20,10,10,320] -> 320 3x3 11.0), bound by the LDS as there.
template <bool IN_U8, int OUT, int NW, int TILE = 256, bool SHORTK = false, bool PP = false, int NS = 4, bool CONV = false>
__global__ __launch_bounds__(64 * NW, SHORTK ? 3 : 1) void nce_gemm_mfma(const int8_t* __restrict__ A, const int8_t* __restrict__ B,
                                                     const int32_t* __restrict__ wt, const int32_t* __restrict__ colsum,
                                                     uint8_t* __restrict__ out,
                                                     int64_t M, int64_t N, int64_t K, int tiles_m, int tiles_n, unsigned group_magic,
                                                     GemmPpe ppe, GemmRows rows, GemmOut dst, GemmConv cv) {
    // NW = 4: waves 2 x 2, 128 x 128 each, one per SIMD.  NW = 8: waves 2 x 4, 128 x 64 each, two per SIMD,
    // so that one wave's loads and address arithmetic issue while the other's MFMAs run.
    // TILE = 128 and 64 serve problems with too few 256 x 256 tiles.
    // SHORTK (K <= 192, three panels at most): all panels are fetched up front, nothing is pipelined and no panel buffer
    // is reused, so the workgroup asks only for the LDS it touches and more of them fit a CU (a matmul this short is
    // bound by its epilogue and stores, not by the MFMAs).  Three waves a SIMD are asked for: left to itself the compiler keeps the
    // sums in accumulation registers beside 124 others, two waves, and [15514 x 64] . [64 x 584] took 10.1 us, now 8.6.
    using Lds = GemmLds<IN_U8, OUT, NW, TILE, SHORTK, PP, NS, CONV>;
    constexpr bool WIDE = Lds::kWide;
    constexpr bool SPLIT_RINGS = WIDE && TILE == 256;  // a ring of buffers per operand, so that an instruction's offset reaches both of its buffers
    constexpr int BM = TILE, BN = TILE, BK = WIDE ? 128 : 64, WM = BM / 2, WN = BN / (NW / 2), TM = WM / 32, TN = WN / 32;
    constexpr int MFMA_PER_DMA = WIDE ? 1 : TM * TN / (BM * BK / 1024 / NW);  // MFMAs between two DMA instructions of a sub-step
    static_assert(WIDE || (TM * TN >= TM + TN && MFMA_PER_DMA >= 1), "fragment reads and DMA instructions are interleaved with the MFMAs");
    constexpr int NT = 64 * NW;
    constexpr int CPR = BK / 16;                      // 16-byte chunks per tile row
    constexpr int RPI = 64 / CPR;                     // tile rows one 1 KiB DMA instruction covers
    constexpr int DMA_PER_WAVE = BM * BK / 1024 / NW;  // per operand, per panel
    constexpr int STAGE = (BM + BN) * BK;
    static_assert(STAGE == Lds::kPanel, "the launch asks for the panels there are");

    extern __shared__ __attribute__((aligned(16))) uint8_t smem_raw[];
    int* const colsums = reinterpret_cast<int*>(smem_raw);  // [Lds::kSumTables][TILE] column sums of B, handed from wave to wave
    uint8_t* const smem = smem_raw + kGemmLdsHead;          // the panel buffers, later the output staging tile

    // Grouped matmul: blockIdx.y is the group; every operand holds the groups one after the other.
    if (const int64_t grp = CONV ? 0 : blockIdx.y) {
        A += grp * M * K;
        B += grp * N * K;
        wt += grp * N * 4;
        if (colsum) colsum += grp * N;
        out += grp * M * N * (OUT == OUT_F16 ? 2 : 1);
        if (ppe.rowterm) ppe.rowterm += grp * M;
    }

    // Workgroup ids are dealt round-robin to the 8 XCDs.  Give each XCD a contiguous run of tile
    // ids and walk tiles in groups of 4 tile-rows, so that workgroups resident on one XCD at the
    // same time share A and B panels in that XCD's L2.
    // (Everything up to the first load is a chain of instructions fetched for the first time: no division, 32 bits where they do.)
    const unsigned total = (unsigned)tiles_m * (unsigned)tiles_n;
    const unsigned per_xcd = (total + 7) / 8;
    const unsigned id = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if (id >= total) return;
    constexpr int GM = 4;
    const unsigned group = quotient(id, GM * (unsigned)tiles_n, group_magic);
    const int gm0 = (int)group * GM;
    const int gsz = tiles_m - gm0 < GM ? tiles_m - gm0 : GM;
    const unsigned in_group = id - group * (GM * (unsigned)tiles_n);
    const unsigned tn = gsz == 4 ? in_group / 4 : (gsz == 3 ? in_group / 3 : (gsz == 2 ? in_group / 2 : in_group));
    const unsigned tm = (unsigned)gm0 + (in_group - tn * (unsigned)gsz);
    const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm0 = NW == 4 ? (wave >> 1) * WM : (wave >> 2) * WM, wn0 = NW == 4 ? (wave & 1) * WN : (wave & 3) * WN;

    // Source addresses of this lane's DMA chunks.  Instruction q of a panel fills LDS bytes
    // [q*1024, q*1024+1024) of the operand's tile = rows q*RPI .. ; the lane sitting at chunk slot p
    // of row r fetches source chunk p ^ swz(r), which is what puts the swizzle in place.
    const int mrows = (int)(M - m0 < BM ? M - m0 : BM), nrows = (int)(N - n0 < BN ? N - n0 : BN);
    unsigned oa[DMA_PER_WAVE], ob[DMA_PER_WAVE];  // byte offsets from the tile's first row
    [[maybe_unused]] int iy[DMA_PER_WAVE], ix[DMA_PER_WAVE];  // CONV: the row's first tap
#pragma unroll
    for (int i = 0; i < DMA_PER_WAVE; i++) {
        const int q = wave + NW * i;
        const int r = q * RPI + lane / CPR, p = lane % CPR;
        const int c = p ^ lds_swz<BK>(r);
        const unsigned rm = (unsigned)(r < mrows ? r : mrows - 1);  // rows past the edge repeat the last one; their outputs are not stored
        const unsigned rn = (unsigned)(r < nrows ? r : nrows - 1);
        ob[i] = rn * (unsigned)K + (unsigned)(c * 16);
        if constexpr (CONV) {
            const unsigned mm = (unsigned)m0 + rm, img = quotient(mm, (unsigned)cv.ohow, cv.ohow_magic), rem = mm - img * (unsigned)cv.ohow;
            const unsigned oy = quotient(rem, (unsigned)cv.ow, cv.ow_magic), ox = rem - oy * (unsigned)cv.ow;
            iy[i] = (int)oy * cv.SY - cv.PT;
            ix[i] = (int)ox * cv.SX - cv.PL;
            oa[i] = (unsigned)((int)img * cv.isn + iy[i] * cv.ish + ix[i] * cv.isw);  // (of a pixel that may lie outside the image)
        } else {
            oa[i] = rm * (unsigned)rows.lda + (unsigned)(c * 16);
        }
    }
    if (!CONV && rows.strided) {  // (offsets from the tensor's first byte; the host has checked that they fit 32 bits)
#pragma unroll
        for (int i = 0; i < DMA_PER_WAVE; i++) {
            const int r = (wave + NW * i) * RPI + lane / CPR, c = (lane % CPR) ^ lds_swz<BK>(r);
            const int mm = (int)m0 + (r < mrows ? r : mrows - 1), img = mm / rows.ohow, rem = mm - img * rows.ohow, oy = rem / rows.ow, ox = rem - oy * rows.ow;
            oa[i] = (unsigned)img * rows.pimg + (unsigned)oy * rows.py + (unsigned)ox * rows.px + (unsigned)(c * 16);
        }
    }
    const int8_t* abase = CONV || rows.strided ? A : A + m0 * rows.lda;
    const int8_t* bbase = B + n0 * K;
    const unsigned lds0 = lds_address(smem);
    const int nk = (int)((K + BK - 1) / BK);
    const bool half = WIDE && !CONV && (K & 64) != 0;  // the last panel is half a panel
    const unsigned past_half = WIDE && (((lane % CPR) ^ lds_swz<BK>(wave * RPI + lane / CPR)) & 4) != 0 ? 64u : 0u;
    // CONV: the chunk of K this lane fetches of the panel asked for next, the same for all its rows (their swizzle is): the chunk
    // of the tap's channels, the tap, and its offset from the row's first tap.
    [[maybe_unused]] int cc = 0, ky = 0, kx = 0, koff = 0;
    [[maybe_unused]] const int kc = ((lane % CPR) ^ lds_swz<BK>(wave * RPI + lane / CPR)) * 16;  // byte of the panel
    if constexpr (CONV) {
        static_assert(!CONV || (lds_swz<BK>(NW * RPI) == lds_swz<BK>(0)), "a lane's rows share their swizzle");
        const int tap = (kc / 16) / cv.cpt;
        cc = kc / 16 - tap * cv.cpt;
        ky = tap / cv.KX;
        kx = tap - ky * cv.KX;
        koff = ky * cv.ish + kx * cv.isw + cc * 16;
    }
    [[maybe_unused]] const int8_t* const pad16 = reinterpret_cast<const int8_t*>(g_pads.bytes[CONV ? cv.pad : 0]);
    [[maybe_unused]] const int8_t* const zero16 = reinterpret_cast<const int8_t*>(g_pads.bytes[0]);
    [[maybe_unused]] const auto next_tap = [&]() {
        const bool wrap = cc >= cv.cpt;
        cc -= wrap ? cv.cpt : 0;
        koff += wrap ? cv.isw - cv.cpt * 16 : 0;
        kx += wrap ? 1 : 0;
        const bool down = kx == cv.KX;
        kx = down ? 0 : kx;
        ky += down ? 1 : 0;
        koff += down ? cv.ish - cv.KX * cv.isw : 0;
    };
    [[maybe_unused]] const auto next_panel = [&]() {
        cc += CPR;
        koff += CPR * 16;
        next_tap();
        if (cv.cpt < CPR) next_tap();  // (a tap is at least half a panel)
    };
    // d-th DMA instruction (first half A, second half B) of panel p.  Panels past the end keep the number of loads
    // in flight the same in every iteration: every lane re-fetches the tile's first 16 bytes (one cache line for
    // the whole instruction) into a buffer nobody reads.
    auto dma_one = [&](auto known_real, int p, int d) {
        const unsigned base = lds0 + (unsigned)((p % NS) * (SPLIT_RINGS ? BM * BK : STAGE));
        constexpr unsigned B0 = SPLIT_RINGS ? NS * BM * BK : BM * BK;  // of the first B panel
        if constexpr (CONV) {
            if (d < DMA_PER_WAVE) {  // (past the end of K the walk goes on, on pixels inside the image or on padding)
                const bool in = (unsigned)(iy[d] + ky) < (unsigned)cv.H && (unsigned)(ix[d] + kx) < (unsigned)cv.W;
                dma16_at(in ? A + (int64_t)(int)(oa[d] + (unsigned)koff) : pad16, base + (unsigned)((wave + NW * d) * 1024));
                if (d == DMA_PER_WAVE - 1) next_panel();
            } else {
                const int8_t* from = bbase + (int64_t)p * BK + ob[d - DMA_PER_WAVE];
                if (!decltype(known_real)::value && (int64_t)p * BK + kc >= K) from = zero16;
                dma16_at(from, base + (unsigned)(BM * BK + (wave + NW * (d - DMA_PER_WAVE)) * 1024));
            }
            return;
        }
        const bool real = decltype(known_real)::value || p < nk;  // (known: no select instructions in the loop body)
        const int64_t k0 = real ? (int64_t)p * BK : 0;
        unsigned off = d < DMA_PER_WAVE ? oa[d] : ob[d - DMA_PER_WAVE];
        if (WIDE && !decltype(known_real)::value && half && p == nk - 1) off -= past_half;  // (its second half: the first again, not multiplied)
        if (d < DMA_PER_WAVE) dma16(abase + k0, real ? off : 0u, base + (unsigned)((wave + NW * d) * 1024));
        else dma16(bbase + k0, real ? off : 0u, base + B0 + (unsigned)((wave + NW * (d - DMA_PER_WAVE)) * 1024));
    };

    i32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0;

    i32x4 fa[2][TM], fb[2][TN];
    auto load_frag = [&](const uint8_t* pa, int kk, int slot, int n) {
        const int chunk = kk * 2 + (lane >> 5);
        if (n == 0) fa[slot][0] = *reinterpret_cast<const i32x4*>(pa + lds_offset<BK>(wm0 + (lane & 31), chunk));
        else if (n <= TN) fb[slot][n - 1] = *reinterpret_cast<const i32x4*>(pa + BM * BK + lds_offset<BK>(wn0 + (n - 1) * 32 + (lane & 31), chunk));
        else fa[slot][n - TN] = *reinterpret_cast<const i32x4*>(pa + lds_offset<BK>(wm0 + (n - TN) * 32 + (lane & 31), chunk));
    };
    // The same reads for a panel buffer known at compile time: the lane's part of the address is one of eight registers
    // that do not change over the K loop (operand, sub-step, lower or upper pair of buffers) and everything else is the
    // instruction's immediate offset, so the unrolled loop below computes no LDS address.
    typedef const __attribute__((address_space(3))) uint8_t* lds_bytes_t;  // 32-bit LDS addresses: one register each
    typedef const __attribute__((address_space(3))) i32x4* lds_v4_t;
    lds_bytes_t frag_base[2][2][2];  // [buffer pair][operand: 0 = A, 1 = B][sub-step]
#pragma unroll
    for (int hi = 0; hi < 2; hi++)
#pragma unroll
        for (int kk = 0; kk < 2; kk++) {
            if (WIDE) continue;
            const int chunk = kk * 2 + (lane >> 5);
            frag_base[hi][0][kk] = (lds_bytes_t)(smem + hi * 2 * STAGE + lds_offset<BK>(wm0 + (lane & 31), chunk));
            frag_base[hi][1][kk] = (lds_bytes_t)(smem + hi * 2 * STAGE + BM * BK + lds_offset<BK>(wn0 + (lane & 31), chunk));
            asm volatile("" : "+v"(frag_base[hi][0][kk]), "+v"(frag_base[hi][1][kk]));  // keep them: re-deriving costs vector ALU slots per read
        }
    auto load_frag_static = [&](auto stage_c, int kk, int slot, int n) {
        constexpr int stage = decltype(stage_c)::value;
        constexpr int imm = (stage & 1) * STAGE;
        // rows 32 apart are 32 * BK bytes apart and share their swizzle
        if (n == 0) fa[slot][0] = *(lds_v4_t)(frag_base[(stage >> 1) & 1][0][kk] + imm);
        else if (n <= TN) fb[slot][n - 1] = *(lds_v4_t)(frag_base[(stage >> 1) & 1][1][kk] + imm + (n - 1) * 32 * BK);
        else fa[slot][n - TN] = *(lds_v4_t)(frag_base[(stage >> 1) & 1][0][kk] + imm + (n - TN) * 32 * BK);
    };
    // One sub-step: the TM x TN MFMAs on fragment slot `cur`; between them, the TM + TN fragment reads of the
    // next sub-step (panel at pnext, sub-step knext) into the other slot and this wave's DMA instructions
    // dma0.. of panel dma_p.
    // Column sums of B for the zero-point term, from the fragments as they pass: lane l sums the 16-byte chunks it
    // holds of column l % 32 (lanes l and l ^ 32 hold alternate chunks), four dot instructions per fragment.  Vector
    // ALU instructions between the MFMAs are not free (they take issue slots of the SIMD), so only the waves of the
    // tile's upper half (SUM) do this -- the lower half reads the same columns -- and hand the sums over through LDS.
    int cs[TN];
#pragma unroll
    for (int j = 0; j < TN; j++) cs[j] = 0;
    auto substep = [&](auto sum_c, auto next_stage_c, int cur, const uint8_t* pnext, int knext, int dma_p, int dma0) {
        constexpr bool SUM = decltype(sum_c)::value;
        constexpr int NEXT_STAGE = decltype(next_stage_c)::value;  // buffer the next sub-step's panel sits in, -1: see pnext
        auto load_next = [&](int n) {
            if constexpr (NEXT_STAGE >= 0) load_frag_static(next_stage_c, knext, cur ^ 1, n);
            else load_frag(pnext, knext, cur ^ 1, n);
        };
#pragma unroll
        for (int i = 0; i < TM; i++) {
            i32x4 a = fa[cur][i];
            if (IN_U8) a ^= (int32_t)0x80808080;  // u8 -> s8 (value - 128)
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const int idx = i * TN + j;
                acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, fb[cur][j], acc[i][j], 0, 0, 0);
                if (SUM && i == TM - 1) {  // behind the last MFMA that reads the fragment
#pragma unroll
                    for (int d = 0; d < 4; d++) cs[j] = __builtin_amdgcn_sdot4(fb[cur][j][d], 0x01010101, cs[j], false);
                }
                // all fragment reads of the next sub-step behind the first two MFMAs: the reads of the eight waves
                // queue at the LDS, and the last one issued must be back before this sub-step's MFMAs are through
                constexpr int FH = (TM + TN + 1) / 2;
                if (idx == 0) {
#pragma unroll
                    for (int n = 0; n < FH; n++) load_next(n);
                } else if (idx == 1) {
#pragma unroll
                    for (int n = FH; n < TM + TN; n++) load_next(n);
                }
                if (!SHORTK && idx % MFMA_PER_DMA == MFMA_PER_DMA - 1)
                    dma_one(std::integral_constant<bool, (NEXT_STAGE >= 0)>{}, dma_p, dma0 + idx / MFMA_PER_DMA);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };

    // per-column PPE words, fetched now so that the epilogue does not start with a memory round trip
    int w2r[TN], w3r[TN], csr[TN];
#pragma unroll
    for (int j = 0; j < TN; j++) {
        const int r = wn0 + j * 32 + (lane & 31);
        const int2 words = *reinterpret_cast<const int2*>(wt + n0 * 4 + (unsigned)((r < nrows ? r : nrows - 1) * 4 + 2));
        csr[j] = 0;
        w2r[j] = words.x;
        w3r[j] = words.y;
    }
    // (Nobody waits for these words here: they are the oldest loads in flight, so every count waited for below covers them.)

    constexpr std::integral_constant<int, -1> kDynamicStage{};
    auto main_loop = [&](auto sum_c) {
        if constexpr (WIDE && TILE == 256) {
            constexpr int HALF = decltype(sum_c)::value;  // the half of each panel whose column sums this wave takes, or neither (2)
            i32x4 pa[2][TM], pb[2][TN];
            lds_bytes_t base[2][4];  // [operand][sub-step of a panel]
#pragma unroll
            for (int o = 0; o < 2; o++)
#pragma unroll
                for (int kk = 0; kk < 4; kk++) {
                    base[o][kk] = (lds_bytes_t)(smem + o * NS * BM * BK + lds_offset<BK>((o ? wn0 : wm0) + (lane & 31), kk * 2 + (lane >> 5)));
                    asm volatile("" : "+v"(base[o][kk]));
                }
            auto read_one = [&](int stage, int kk, int slot, int n) {
                if (n == 0) pa[slot][0] = *(lds_v4_t)(base[0][kk] + stage * BM * BK);
                else if (n <= TN) pb[slot][n - 1] = *(lds_v4_t)(base[1][kk] + stage * BN * BK + (n - 1) * 32 * BK);
                else pa[slot][n - TN] = *(lds_v4_t)(base[0][kk] + stage * BM * BK + (n - TN) * 32 * BK);
            };
            // Sub-step kk of a panel; the next one's fragments come from `stage`.  Panel p is asked for in the last sub-step of panel
            // p - 2, all of it: with half its loads in the next sub-step [4096 x 4096] . [4096 x 11008] takes 186 us, not 176.
            auto step = [&](auto kk_c, int stage, auto real_c, int p) {
                constexpr int kk = decltype(kk_c)::value, slot = kk & 1;
#pragma unroll
                for (int i = 0; i < TM; i++) {
                    i32x4 a = pa[slot][i];
                    if (IN_U8) a ^= (int32_t)0x80808080;  // u8 -> s8 (value - 128)
#pragma unroll
                    for (int j = 0; j < TN; j++) {
                        const int idx = i * TN + j;
                        acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, pb[slot][j], acc[i][j], 0, 0, 0);
                        constexpr int FH = (TM + TN + 1) / 2;
                        if (idx == 0) {
#pragma unroll
                            for (int n = 0; n < FH; n++) read_one(stage, (kk + 1) & 3, slot ^ 1, n);
                        } else if (idx == 1) {
#pragma unroll
                            for (int n = FH; n < TM + TN; n++) read_one(stage, (kk + 1) & 3, slot ^ 1, n);
                        }
                        if (kk == 3) dma_one(real_c, p, idx);
                        if (kk / 2 == HALF && idx == TM * TN - 1) {
#pragma unroll
                            for (int d = 0; d < 4; d++)
#pragma unroll
                                for (int c = 0; c < TN; c++) cs[c] = __builtin_amdgcn_sdot4(pb[slot][c][d], 0x01010101, cs[c], false);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            };
            constexpr std::integral_constant<int, 0> s0{};
            constexpr std::integral_constant<int, 1> s1{};
            constexpr std::integral_constant<int, 2> s2{};
            constexpr std::integral_constant<int, 3> s3{};
            static_assert(TILE != 256 || !WIDE || 2 * DMA_PER_WAVE == TM * TN, "a load behind each MFMA of a panel's last sub-step");
            auto one_panel = [&](int u, auto real_c, int k) {
                step(s0, u, real_c, 0);
                step(s1, u, real_c, 0);
                if (!decltype(real_c)::value && half && k == nk - 1) return;
                step(s2, u, real_c, 0);
                asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");  // panel k + 1 is in, panel k has been read
                step(s3, u ^ 1, real_c, k + 2);
            };
#pragma unroll
            for (int p = 0; p < 2; p++)
#pragma unroll
                for (int d = 0; d < 2 * DMA_PER_WAVE; d++) dma_one(std::false_type{}, p, d);
            asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(2 * DMA_PER_WAVE) : "memory");  // panel 0 is in
#pragma unroll
            for (int n = 0; n < TM + TN; n++) read_one(0, 0, 0, n);
            int kt = 0;
            for (; kt + 4 < nk; kt += 2) {  // (every panel asked for whole)
                one_panel(0, std::true_type{}, kt);
                one_panel(1, std::true_type{}, kt + 1);
            }
            for (; kt < nk; kt += 2) {
                one_panel(0, std::false_type{}, kt);
                if (kt + 1 < nk) one_panel(1, std::false_type{}, kt + 1);
            }
        } else if constexpr (WIDE) {
            // The fragments of half a panel are read under the MFMAs of the half before it; behind the barrier between the two
            // everybody is through with the panel's buffer, which panel k + NS is then asked into.
            constexpr int HALF = decltype(sum_c)::value;  // the half of each panel whose column sums this wave takes, or neither (2)
            i32x4 pa[2][2][TM], pb[2][2];
            int cs1 = 0;
            lds_bytes_t base[2][4];  // [operand][sub-step of a panel]
#pragma unroll
            for (int o = 0; o < 2; o++)
#pragma unroll
                for (int kk = 0; kk < 4; kk++) {
                    base[o][kk] = (lds_bytes_t)(smem + o * BM * BK + lds_offset<BK>((o ? wn0 : wm0) + (lane & 31), kk * 2 + (lane >> 5)));
                    asm volatile("" : "+v"(base[o][kk]));
                }
            auto read_half = [&](int stage, auto h_c) {
                constexpr int h = decltype(h_c)::value;
#pragma unroll
                for (int kk = 0; kk < 2; kk++) {
                    pb[h][kk] = *(lds_v4_t)(base[1][h * 2 + kk] + stage * STAGE);
#pragma unroll
                    for (int i = 0; i < TM; i++) pa[h][kk][i] = *(lds_v4_t)(base[0][h * 2 + kk] + stage * STAGE + i * 32 * BK);
                }
                __builtin_amdgcn_sched_barrier(0);
            };
            auto mfma_half = [&](auto h_c, auto real_c, int p) {
                constexpr int h = decltype(h_c)::value;
#pragma unroll
                for (int kk = 0; kk < 2; kk++)
#pragma unroll
                    for (int i = 0; i < TM; i++) {
                        i32x4 a = pa[h][kk][i];
                        if (IN_U8) a ^= (int32_t)0x80808080;  // u8 -> s8 (value - 128)
                        acc[i][0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, pb[h][kk], acc[i][0], 0, 0, 0);
                        if (h == 1) {
#pragma unroll
                            for (int d = 0; d < DMA_PER_WAVE / TM; d++) dma_one(real_c, p, (kk * TM + i) * (DMA_PER_WAVE / TM) + d);
                        }
                        if (h == HALF && kk == 1 && i == 0) {  // (two chains: an instruction need not wait for the one before it)
#pragma unroll
                            for (int d = 0; d < 4; d++) {
                                cs[0] = __builtin_amdgcn_sdot4(pb[h][0][d], 0x01010101, cs[0], false);
                                cs1 = __builtin_amdgcn_sdot4(pb[h][1][d], 0x01010101, cs1, false);
                            }
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
            };
            static_assert(!WIDE || TILE == 256 || (DMA_PER_WAVE % TM == 0 && TN == 1), "the same number of loads behind each MFMA of a second half");
            constexpr std::integral_constant<int, 0> first{};
            constexpr std::integral_constant<int, 1> second{};
            auto one_panel = [&](int u, auto real_c, int k) {
                read_half(u, second);
                mfma_half(first, real_c, 0);
                asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((NS - 2) * 2 * DMA_PER_WAVE) : "memory");  // panel k + 1 is in
                read_half((u + 1) % NS, first);
                if (decltype(real_c)::value || k + 1 < nk || !half) mfma_half(second, real_c, k + NS);
            };
#pragma unroll
            for (int p = 0; p < NS; p++)
#pragma unroll
                for (int d = 0; d < 2 * DMA_PER_WAVE; d++) dma_one(std::false_type{}, p, d);
            asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((NS - 1) * 2 * DMA_PER_WAVE) : "memory");  // panel 0 is in
            read_half(0, first);
            int kt = 0;
            for (; kt + 2 * NS < nk; kt += NS) {  // (every panel asked for whole)
#pragma unroll
                for (int u = 0; u < NS; u++) one_panel(u, std::true_type{}, kt + u);
            }
            for (; kt < nk; kt += NS) {  // the last panels, at most two rounds
#pragma unroll
                for (int u = 0; u < NS; u++)
                    if (kt + u < nk) one_panel(u, std::false_type{}, kt + u);
            }
            cs[0] += cs1;
        } else if constexpr (SHORTK) {
#pragma unroll
            for (int p = 0; p < NS - 1; p++)
                if (p < nk) {
#pragma unroll
                    for (int d = 0; d < 2 * DMA_PER_WAVE; d++) dma_one(std::false_type{}, p, d);
                }
            dma_wait_all_and_barrier();
#pragma unroll
            for (int n = 0; n < TM + TN; n++) load_frag(smem, 0, 0, n);
            for (int kt = 0; kt < nk; kt++) {
                const uint8_t* pcur = smem + kt * STAGE;
                const uint8_t* pnxt = kt + 1 < nk ? pcur + STAGE : pcur;  // the last step prefetches fragments nobody uses
                substep(sum_c, kDynamicStage, 0, pcur, 1, 0, 0);
                substep(sum_c, kDynamicStage, 1, pnxt, 0, 0, 0);
            }
        } else {
#pragma unroll
            for (int p = 0; p < NS - 1; p++)
#pragma unroll
                for (int d = 0; d < 2 * DMA_PER_WAVE; d++) dma_one(std::false_type{}, p, d);
            asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(4 * DMA_PER_WAVE) : "memory");  // panel 0 is in
#pragma unroll
            for (int n = 0; n < TM + TN; n++) load_frag(smem, 0, 0, n);
            int kt = 0;
            // Four panels per trip while all loads are real ones: the panel buffers are then known by number, the
            // fragment reads take immediate offsets and the loads need no selects.
            if ((nk & (NS - 1)) == 0) {
                auto one_panel = [&](auto u_c, int k) {
                    constexpr int u = decltype(u_c)::value;
                    substep(sum_c, std::integral_constant<int, u>{}, 0, nullptr, 1, k + NS - 1, 0);
                    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(3 * DMA_PER_WAVE) : "memory");
                    substep(sum_c, std::integral_constant<int, (u + 1) & (NS - 1)>{}, 1, nullptr, 0, k + NS - 1, DMA_PER_WAVE);
                };
                for (; kt + 2 * NS <= nk; kt += NS) {
                    one_panel(std::integral_constant<int, 0>{}, kt);
                    one_panel(std::integral_constant<int, 1>{}, kt + 1);
                    one_panel(std::integral_constant<int, 2>{}, kt + 2);
                    one_panel(std::integral_constant<int, 3>{}, kt + 3);
                }
            }
            for (; kt < nk; kt++) {
                const uint8_t* pcur = smem + (kt & (NS - 1)) * STAGE;
                const uint8_t* pnxt = smem + ((kt + 1) & (NS - 1)) * STAGE;
                substep(sum_c, kDynamicStage, 0, pcur, 1, kt + NS - 1, 0);
                // Loads in flight here, oldest first: panel kt+1, panel kt+2 (2 * DMA_PER_WAVE each), half of panel kt+3.
                // Behind the barrier panel kt+1 is complete for every wave and nobody reads panel kt-1 any
                // more, whose buffer panel kt+3 is being written to.
                asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(3 * DMA_PER_WAVE) : "memory");
                substep(sum_c, kDynamicStage, 1, pnxt, 0, kt + NS - 1, DMA_PER_WAVE);
            }
        }
    };
    // Waves w and w + 4 share a SIMD.  Half-steps are counted from 0; in half-step h the first four waves (the tile's upper
    // half) multiply panel h / 2 when h is even and do their memory work when it is odd, the other four the other way
    // round, one half-step behind.  Panel p sits in buffer p % 4, and its loads are issued three panels ahead: by the
    // lower waves in half-step 2 (p - 3), by the upper ones in 2 (p - 3) + 1; the buffer they write held panel p - 4, whose
    // last fragment reads were consumed by MFMAs two half-steps earlier.  Before the barrier that ends an even
    // half-step 2 k every wave waits for its own loads of panel k + 1, so behind that barrier the panel is complete.
    auto pingpong_loop = [&]() {
        static_assert(!PP || (NW == 8 && TILE == 256 && !SHORTK), "wave roles alternate on the eight-wave large tile");
        auto read_panel = [&](auto stage_c) {
#pragma unroll
            for (int kk = 0; kk < 2; kk++)
#pragma unroll
                for (int n = 0; n < TM + TN; n++) load_frag_static(stage_c, kk, kk, n);
        };
        auto dma_panel = [&](int p) {
#pragma unroll
            for (int d = 0; d < 2 * DMA_PER_WAVE; d++) dma_one(std::false_type{}, p, d);
        };
        auto mfma_panel = [&]() {
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int kk = 0; kk < 2; kk++)
#pragma unroll
                for (int i = 0; i < TM; i++) {
                    i32x4 a = fa[kk][i];
                    if (IN_U8) a ^= (int32_t)0x80808080;  // u8 -> s8 (value - 128)
#pragma unroll
                    for (int j = 0; j < TN; j++) acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, fb[kk][j], acc[i][j], 0, 0, 0);
                }
            __builtin_amdgcn_s_setprio(0);
            __builtin_amdgcn_sched_barrier(0);
        };
        auto sum_panel = [&]() {  // the column sums of B from the fragments of the panel just multiplied
#pragma unroll
            for (int kk = 0; kk < 2; kk++)
#pragma unroll
                for (int j = 0; j < TN; j++)
#pragma unroll
                    for (int d = 0; d < 4; d++) cs[j] = __builtin_amdgcn_sdot4(fb[kk][j][d], 0x01010101, cs[j], false);
            __builtin_amdgcn_sched_barrier(0);
        };
#pragma unroll
        for (int p = 0; p < NS - 1; p++) dma_panel(p);
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(4 * DMA_PER_WAVE) : "memory");  // panel 0 is in
        // (two loops, one per role: the same number of barriers in each)
        if (wm0 == 0) {
            read_panel(std::integral_constant<int, 0>{});
            auto one_panel = [&](auto u_c, int k) {
                constexpr int u = decltype(u_c)::value;
                mfma_panel();
                asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(2 * DMA_PER_WAVE) : "memory");  // this wave's share of panel k + 1 is in
                sum_panel();
                if (k + 1 < nk) read_panel(std::integral_constant<int, (u + 1) & (NS - 1)>{});
                dma_panel(k + NS - 1);
                asm volatile("s_barrier" ::: "memory");
            };
            for (int k = 0; k < nk; k += NS) {
                one_panel(std::integral_constant<int, 0>{}, k);
                one_panel(std::integral_constant<int, 1>{}, k + 1);
                one_panel(std::integral_constant<int, 2>{}, k + 2);
                one_panel(std::integral_constant<int, 3>{}, k + 3);
            }
        } else {
            auto one_panel = [&](auto u_c, int k) {
                read_panel(u_c);
                dma_panel(k + NS - 1);
                asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(4 * DMA_PER_WAVE) : "memory");  // likewise, with panel k + 3 just asked for
                mfma_panel();
                asm volatile("s_barrier" ::: "memory");
            };
            for (int k = 0; k < nk; k += NS) {
                one_panel(std::integral_constant<int, 0>{}, k);
                one_panel(std::integral_constant<int, 1>{}, k + 1);
                one_panel(std::integral_constant<int, 2>{}, k + 2);
                one_panel(std::integral_constant<int, 3>{}, k + 3);
            }
        }
    };
    if constexpr (PP) {
        pingpong_loop();
    } else {
        // (a matmul of at most three panels is all epilogue: there every wave sums its own columns and nothing is handed over)
        if constexpr (WIDE) {  // (of the two waves on the same columns each sums half of every panel)
            if (ppe.corr == 0) main_loop(std::integral_constant<int, 2>{});
            else if (wm0 == 0) main_loop(std::integral_constant<int, 0>{});
            else main_loop(std::integral_constant<int, 1>{});
        } else {
            if (ppe.corr != 0 && (SHORTK || wm0 == 0)) main_loop(std::true_type{});
            else main_loop(std::false_type{});
        }
    }
#pragma unroll
    for (int j = 0; j < TN; j++) {
        csr[j] = cs[j] + __shfl_xor(cs[j], 32, 64);  // every lane takes part
        if (!SHORTK && (WIDE || wm0 == 0) && lane < 32) colsums[(WIDE && wm0 != 0 ? TILE : 0) + wn0 + j * 32 + lane] = csr[j];
    }
    dma_wait_all_and_barrier();  // every wave is done with the panels: LDS becomes the output staging tile
    if (!SHORTK) {
#pragma unroll
        for (int j = 0; j < TN; j++) {
            csr[j] = colsums[wn0 + j * 32 + (lane & 31)];  // sum_k B[n][k] of column n of block j
            if (WIDE) csr[j] += colsums[TILE + wn0 + j * 32 + (lane & 31)];
        }
    }
    // Epilogue.  Accumulator register r of lane l is C[8*(r/4) + 4*(l/32) + r%4][l%32] of its 32x32 tile.
    if constexpr (OUT == OUT_F16) {
        // fp16 output: through the staging tile like the bytes below, half of a 256-row tile at a time (128 rows x 544
        // bytes), so that the tile leaves in whole rows of 16-byte stores (two-byte stores straight from the registers,
        // 64 bytes of a row per half-wavefront, cost the [4096 x 4096] . [4096 x 11008] matmul 60 us).
        constexpr int PASSES = TILE == 256 ? 2 : 1, ROWS = BM / PASSES, STR = BN * 2 + 32;
        static_assert(ROWS * STR == Lds::kStaging, "the fp16 staging tile is what the launch has room for");
        uint16_t* out16 = reinterpret_cast<uint16_t*>(out);
        if (ppe.rowterm) {  // (padded past the last row: edge tiles may read ahead)
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const i32x4 v = *reinterpret_cast<const i32x4*>(ppe.rowterm + m0 + wm0 + i * 32 + 8 * g + 4 * (lane >> 5));
#pragma unroll
                    for (int j = 0; j < TN; j++)
#pragma unroll
                        for (int q = 0; q < 4; q++) acc[i][j][g * 4 + q] += v[q];
                }
        }
        const bool vec_ok = (dst.bits & 15) == 0;
#pragma unroll
        for (int pass = 0; pass < PASSES; pass++) {
            if (wm0 / ROWS == pass) {
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    const uint32_t w2 = (uint32_t)w2r[j];
                    const ChanPrep c = ppe_prepare((int)(int16_t)(w2 >> 16), (int)((w2 >> 8) & 0xffu) - 15,
                                                   (int)((unsigned)w3r[j] + (unsigned)(ppe.corr * csr[j])), ppe.prelu_mult, ppe.prelu_shift);
                    uint8_t* const col = smem + (wm0 - pass * ROWS + 4 * (lane >> 5)) * STR + (wn0 + j * 32 + (lane & 31)) * 2;
#pragma unroll
                    for (int i = 0; i < TM; i++)
#pragma unroll
                        for (int r = 0; r < 16; r++)
                            *reinterpret_cast<uint16_t*>(col + (i * 32 + 8 * (r / 4) + (r % 4)) * STR) = ppe_fast_f16(acc[i][j][r], c, ppe.f16_lo, ppe.f16_hi);
                }
            }
            __syncthreads();
            for (int it = 0; it < ROWS * (BN / 8) / NT; it++) {
                const int cid = tid + NT * it;
                const int row = cid / (BN / 8), c8 = cid % (BN / 8);
                const int64_t m = m0 + pass * ROWS + row, n = n0 + c8 * 8;
                if (m >= M || n >= N) continue;
                const i32x4 v = *reinterpret_cast<const i32x4*>(smem + row * STR + c8 * 16);
                uint16_t* const to = out16 + dst.row(m) + n;
                if (vec_ok && n + 8 <= N) {
                    __builtin_nontemporal_store(v, reinterpret_cast<i32x4*>(to));
                } else if (n + 8 <= N) {
                    *reinterpret_cast<i32x4_any*>(to) = v;
                } else if (c8 > 0) {  // (the row's last eight: those before n twice, alike)
                    *reinterpret_cast<i32x4_any*>(out16 + dst.row(m) + N - 8) = *reinterpret_cast<const i32x4_any*>(smem + row * STR + (int)(N - 8 - n0) * 2);
                } else {
                    store_tail16(reinterpret_cast<uint8_t*>(to), v, (int)(N - n < 8 ? N - n : 8) * 2, out_align(dst.bits));
                }
            }
            if (pass + 1 < PASSES) __syncthreads();  // the other half overwrites the staging tile
        }
        return;
    }
    constexpr bool OUT_SIGNED = OUT == OUT_I8;
    ChanPrep cp[TN];
    bool clip = false;
#pragma unroll
    for (int j = 0; j < TN; j++) {
        const uint32_t w2 = (uint32_t)w2r[j];
        cp[j] = ppe_prepare_packed((int)(int16_t)(w2 >> 16), (int)((w2 >> 8) & 0xffu),
                                   (int)((unsigned)w3r[j] + (unsigned)(ppe.corr * csr[j])), ppe.prelu_mult, ppe.prelu_shift);
        clip = clip || cp[j].bmax_pos != 0x7fffffff || cp[j].bmax_neg != 0x7fffffff;
        // keep the prepared factors in registers: without this the compiler re-derives them per element
        asm volatile("" : "+v"(cp[j].f_pos), "+v"(cp[j].f_neg));
    }
    const PpePack pk = make_ppe_pack(ppe.zp_out, ppe.lo, ppe.hi, OUT_SIGNED);
    if (ppe.rowterm) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const i32x4 v = *reinterpret_cast<const i32x4*>(ppe.rowterm + m0 + wm0 + i * 32 + 8 * g + 4 * (lane >> 5));
#pragma unroll
                for (int j = 0; j < TN; j++)
#pragma unroll
                    for (int q = 0; q < 4; q++) acc[i][j][g * 4 + q] += v[q];
            }
    }
    // kind 0: every PPE setting; 1: no clipping, even zero-point offset, slope in [0, 1] (ReLU, LeakyReLU): no sign
    // test, see ppe_pack4_biased; 2: the same with slope 1 (no PReLU stage)
    auto requant_tile = [&](auto kind_c) {
        constexpr int KIND = decltype(kind_c)::value;
#pragma unroll
        for (int j = 0; j < TN; j++) {
            const int col4 = wn0 + j * 32 + ((lane & 31) & ~3);
            const int pb = (int)((unsigned)cp[j].bias - 0x80000000u);  // the bias without the sign flip of the packed form
#pragma unroll
            for (int i = 0; i < TM; i++) {
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    unsigned w;
                    if constexpr (KIND == 0)
                        w = ppe_pack4<false, true>(acc[i][j][g * 4], acc[i][j][g * 4 + 1], acc[i][j][g * 4 + 2], acc[i][j][g * 4 + 3], cp[j], pk);
                    else  // (the larger of the two products is the same whichever way a negative multiplier swapped the factors)
                        w = ppe_pack4_biased<KIND == 1>(acc[i][j][g * 4] + pb, acc[i][j][g * 4 + 1] + pb, acc[i][j][g * 4 + 2] + pb,
                                                        acc[i][j][g * 4 + 3] + pb, cp[j].f_pos, cp[j].f_neg, pk);
                    w = quad_transpose_bytes(w, lane);
                    const int row = wm0 + i * 32 + 8 * g + 4 * (lane >> 5) + (lane & 3);
                    *reinterpret_cast<unsigned*>(smem + row * kOutStride + col4) = w;
                }
            }
        }
    };
    // scale factors above 1/2 are rare (shift < 15), as are odd zero-point offsets and slopes outside [0, 1]
    const bool slope_ok = ppe.prelu_mult >= 0 && (ppe.prelu_shift >= 31 || ppe.prelu_mult <= (1 << ppe.prelu_shift));
    if (__builtin_amdgcn_ballot_w64(clip) != 0 || pk.odd != 0 || !slope_ok) requant_tile(std::integral_constant<int, 0>{});
    else if (ppe.prelu_mult == 1 && ppe.prelu_shift == 0) requant_tile(std::integral_constant<int, 2>{});
    else requant_tile(std::integral_constant<int, 1>{});
    __syncthreads();
    // Rows that start at any byte leave in 16-byte stores as well (their last one overlaps the one before): in pieces of what their
    // alignment allows, bytes for odd lengths, [4000 x 1024] . [1024 x 3001] took 41.5 us, now 24.8; [349 x 320] . [320 x 10317]
    // 14.9, now 9.1; 3008 columns, whose stores are aligned and go past the caches, 22.6.
    const bool vec_ok = (dst.bits & 15) == 0;
    for (int it = 0; it < BM * (BN / 16) / NT; it++) {
        const int cid = tid + NT * it;
        const int row = cid / (BN / 16), c16 = cid % (BN / 16);
        const int64_t m = m0 + row, n = n0 + c16 * 16;
        if (m >= M || n >= N) continue;
        const i32x4 v = *reinterpret_cast<const i32x4*>(smem + row * kOutStride + c16 * 16);
        uint8_t* const to = out + dst.row(m) + n;
        if (vec_ok && n + 16 <= N) {
            __builtin_nontemporal_store(v, reinterpret_cast<i32x4*>(to));
        } else if (n + 16 <= N) {
            *reinterpret_cast<i32x4_any*>(to) = v;
        } else if (c16 > 0) {  // (the row's last sixteen: those before n twice, alike)
            *reinterpret_cast<i32x4_any*>(out + dst.row(m) + N - 16) = *reinterpret_cast<const i32x4_any*>(smem + row * kOutStride + (int)(N - 16 - n0));
        } else {
            store_tail16(to, v, (int)(N - n < 16 ? N - n : 16), out_align(dst.bits));
        }
    }
}

}  // namespace

int launch_gemm_mfma(const GemmLaunch& a, hipStream_t s) {
    const int tile = a.tile, nw = tile == 64 ? 4 : (tile == 128 ? (a.shortk ? 4 : 8) : a.waves);
    const bool out_f16 = a.out_kind == OUT_F16;
    const int tiles_m = (int)((a.M + tile - 1) / tile), tiles_n = (int)((a.N + tile - 1) / tile);
    const int per_xcd = (tiles_m * tiles_n + 7) / 8;
    const dim3 grid((unsigned)(per_xcd * 8), (unsigned)a.G);
    const int64_t nk = a.K / 64;
    const bool shortk = a.shortk;
    const int32_t* colsum = nullptr;  // the kernel sums the columns of B itself, from the fragments it reads
    int rc = VPX_RESULT_SUCCESS;
    // the form in which the waves of a SIMD take turns: K a whole number of panel-buffer rounds
    const bool pingpong = a.pingpong && tile == 256 && nw == 8 && nk % 4 == 0 && nk >= 4 && !out_f16;
#define VPX_GEMM_K(...)                                                                                              \
    do {                                                                                                             \
        auto kern = nce_gemm_mfma<__VA_ARGS__>;                                                                      \
        const size_t lds = GemmLds<__VA_ARGS__>::bytes(a.K);                                                         \
        rc = set_dyn_lds(kern, lds);                                                                                 \
        if (rc) return rc;                                                                                           \
        VPX_LAUNCH(kern, grid, dim3(64 * nw), lds, s, a.A, a.B, a.wt, colsum, a.out, a.M, a.N, a.K, tiles_m,          \
                   tiles_n, quotient_magic(4 * (unsigned)tiles_n), a.ppe, a.rows, a.dst, a.conv);                                                           \
    } while (0)
    // the tiles of 64 and 128, any kind of output
#define VPX_GEMM_SMALL(U8, SGN)                                                                                      \
    do {                                                                                                             \
        if (tile == 64) VPX_GEMM_K(U8, SGN, 4, 64, false, false, 4);                                                 \
        else if (a.stages == 3) VPX_GEMM_K(U8, SGN, 8, 128, false, false, 3);                                        \
        else VPX_GEMM_K(U8, SGN, 8, 128, false, false, 2);                                                           \
    } while (0)
    // a convolution: byte outputs
#define VPX_GEMM_CONV(U8, SGN)                                                                                       \
    do {                                                                                                             \
        if (tile == 64) VPX_GEMM_K(U8, SGN, 4, 64, false, false, 4, true);                                           \
        else if (a.stages == 3) VPX_GEMM_K(U8, SGN, 8, 128, false, false, 3, true);                                  \
        else VPX_GEMM_K(U8, SGN, 8, 128, false, false, 2, true);                                                     \
    } while (0)
#define VPX_GEMM(U8, SGN)                                                                                            \
    do {                                                                                                             \
        if (shortk) VPX_GEMM_K(U8, SGN, 4, 128, true);                                                               \
        else if (tile < 256) VPX_GEMM_SMALL(U8, SGN);                                                                \
        else if (nw == 4) VPX_GEMM_K(U8, SGN, 4, 256);                                                               \
        else if (pingpong) VPX_GEMM_K(U8, SGN, 8, 256, false, true);                                                 \
        else VPX_GEMM_K(U8, SGN, 8, 256, false, false, 2);                                                           \
    } while (0)
    if (a.is_conv) {
        if (a.in_u8 && a.out_kind == OUT_I8) VPX_GEMM_CONV(true, OUT_I8);
        else if (a.in_u8) VPX_GEMM_CONV(true, OUT_U8);
        else if (a.out_kind == OUT_I8) VPX_GEMM_CONV(false, OUT_I8);
        else VPX_GEMM_CONV(false, OUT_U8);
    } else if (out_f16) {
        // fp16 output: of the large tile the eight-wave form only (the host passes waves = 8)
        if (a.in_u8) { if (tile < 256) VPX_GEMM_SMALL(true, OUT_F16); else VPX_GEMM_K(true, OUT_F16, 8, 256, false, false, 2); }
        else { if (tile < 256) VPX_GEMM_SMALL(false, OUT_F16); else VPX_GEMM_K(false, OUT_F16, 8, 256, false, false, 2); }
    }
    else if (a.in_u8 && a.out_kind == OUT_I8) VPX_GEMM(true, OUT_I8);
    else if (a.in_u8) VPX_GEMM(true, OUT_U8);
    else if (a.out_kind == OUT_I8) VPX_GEMM(false, OUT_I8);
    else VPX_GEMM(false, OUT_U8);
#undef VPX_GEMM
#undef VPX_GEMM_SMALL
#undef VPX_GEMM_CONV
#undef VPX_GEMM_K
    return VPX_RESULT_SUCCESS;
}

}  // namespace nce
}  // namespace vpx
