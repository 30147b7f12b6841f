// gemm_ksplit.hip -- the fp16 MFMA Linear for every size between the GEMV and
// the 256x256 tiles: X (fp16 or fp32) . W^T (fp16, as stored), any N and K,
// fused gate/up included.
//
// What bounds these sizes is bytes into the CUs (W and X each pass through LDS
// once per workgroup) and how many CUs have work, not MFMA rate: a full grid of
// 32x32 tiles moves 50 bytes a cycle and CU (8.7 us per MB of a workgroup's
// operands); where a CU has one workgroup of four waves (M = 61: 160 tiles of
// 32x64; X fp32, M = 500: 256 of 64x64) it moves 21-24, its waves issuing 40% of
// the time, waiting for their copies 36-40% and for an issue slot 20-23%, the
// matrix cores 13% busy. So the output is cut into small tiles (32x32 to
// 128x128, chosen by gemm_ksplit_plan so that the tiles fill the CUs), and the
// 4 or 8 waves of a workgroup split K instead of the tile: every wave runs the
// whole tile over its own 64- or 32-wide k chunks, dealt out in turn, so each
// staged byte is written to LDS once and read from it once (a 2x2 split of the
// tile reads each operand twice), no wave waits for another in the K loop,
// and small tiles still keep four to eight waves' copies in flight. Each wave
// has its own ring of stages filled by buffer_load ... lds (whole 64- to
// 256-byte row pieces, 16-byte chunks XOR-swizzled by row); the partial tiles
// meet in LDS at the end. fp32 X is copied as fp32 and rounded to fp16 when
// its fragments are read (once, since no two waves read the same k), the
// rounding the tile path's fp16 staging always made.
//
// Tiles of 64x128 up are quadrants of four waves over one shared ring instead:
// their partial tiles would not fit LDS, and 64 k of both operands a wave only
// once each. The copies are spread over the MFMA steps (in one burst a stage
// took 0.56 us at 128x128, spread 0.40).
//
// Measured (back-to-back calls, us, against the kernels these sizes took
// before, register-staged 64x64 tiles or 256x256 packed tiles with a K split):
// X fp16 [61, 3072], N 5120 21.5 -> 10.7 (2.9 TB/s of W); fp32 [500, 2048],
// N 2048 62 -> 15.8; fp16 [300, 4096], N 1000 139 -> 11.4; fp16 [948, 2481],
// N 1216 (odd K) 206 -> 31; gated fp16 [500, 2048], H 2048 54 -> 17.3.
//
// fp32 X and W (F32): v_mfma_f32_32x32x2_f32, a sixteenth of the rate, so the
// matrix cores bound it and 64x64 quadrants are large enough (two workgroups a
// CU; four sums per output). Against the register-staged tiles that these sizes
// took: [1024, 768], N 3072 75.5 -> 48.9 us; [1000, 3072], N 4096 579 -> 216 (117
// of the 153 TFLOP/s that a large product reaches); [900, 767], N 3073 123 -> 49.7;
// [100, 1147], N 3000 31.6 -> 16.3.
//
// Rows that are not whole 16-byte chunks (K % 8 != 0, fp32 K % 4) or operands off a
// 16-byte boundary take the same kernel with the chunks loaded into registers
// (unaligned 16-byte loads, the last chunk of a row element by element) and
// written to LDS from there.
#include <algorithm>

#include "device_common.h"
#include "kernels.h"
#include "launch_once.h"

#define LDS_AS __attribute__((address_space(3)))

namespace vai_dev {

namespace ks {

// One variant: tile, waves, k per stage and ring depth for X of type TA.
// KSP: the waves split K, each with its own ring; otherwise four waves take a
// quadrant each of the tile and share one ring. DMA false: staged through
// registers (one stage per wave, or two shared ones), X in LDS as fp16. PK:
// the weight is gemm_pack_weight's copy, whose 16-byte pieces (8 k of one row,
// 32 rows of a block after each other) are staged in that order: whole
// contiguous copies, and fragment reads of 1 KB without a swizzle.
template <int BM_, int BN_, int NW_, int BK_, int S_, bool KSP_, typename TA_, bool DMA_, bool PK_, typename TB_ = half_t>
struct Cfg {
    static constexpr int BM = BM_, BN = BN_, NW = NW_, BK = BK_, S = DMA_ ? S_ : (KSP_ ? 1 : 2);
    static constexpr bool KSP = KSP_, DMA = DMA_, PK = PK_;
    typedef TA_ TA;
    static constexpr int WM = KSP ? BM : BM / 2, WN = KSP ? BN : BN / 2;   // a wave's part of the tile
    typedef TB_ TB;
    static constexpr bool F32 = sizeof(TB_) == 4;              // fp32 W (and X): v_mfma_f32_32x32x2_f32, 8 k a step
    static constexpr int KQ = F32 ? 8 : 16, KSTEPS = BK / KQ;
    // sums per output and wave (k steps in turn)
    static constexpr int AS = F32 ? (KSP ? 2 : 4) : !KSP ? 1 : WM * WN <= 32 * 64 ? (BK / 16 < 4 || NW == 8 ? 2 : 4) : 2;
    // Long K: sums per output and wave (fewer where the total takes their
    // registers), and the stages after which they go to the total: chains of at
    // most 256 k (fp32: 128).
    static constexpr int LAS = KSP && WM * WN == 32 * 64 ? (DMA ? 2 : 1) : WM * WN > 32 * 64 ? 1 : AS;
    static constexpr int CHAIN = (F32 ? 128 : 256) * LAS / BK;
    // The quadrants over fp16 X fit in 256 registers (accumulation registers would
    // cost a move per element and chain); with fp32 X 128x128 would spill.
    static constexpr int WPS = NW == 8 || (!KSP && DMA && sizeof(TA_) == 2) ? 2 : 1;
    // whether a wave's share of K is longer than its sums' chains
    static bool long_k(uint32_t K) { return K > (F32 ? 128u : 256u) * AS * (KSP ? NW : 1); }
    static constexpr int AES = DMA || F32 ? (int)sizeof(TA) : 2, BES = (int)sizeof(TB);   // element bytes in LDS
    static constexpr int AROW = BK * AES, BROW = BK * BES;       // row bytes in LDS
    static constexpr int ABYTES = BM * AROW, BBYTES = BN * BROW, STAGE = ABYTES + BBYTES;
    static constexpr int SHARE = KSP ? 1 : NW;                 // waves that fill a stage together
    static constexpr int ACOPIES = ABYTES / 1024 / SHARE, BCOPIES = BBYTES / 1024 / SHARE, COPIES = ACOPIES + BCOPIES;
    static constexpr int RING = (KSP ? NW : 1) * S * STAGE;
    // the final exchange: RB rows of every partial tile at a time
    static constexpr int PLANES = KSP ? NW : 1;
    static constexpr int RROW = BN * 4 + 16;
    static constexpr int RB = PLANES * BM * RROW <= 160 * 1024 ? BM : BM / 2;
    static constexpr int RED = PLANES * RB * RROW;
    static constexpr int LDS = RING > RED ? RING : RED;
    static_assert(LDS <= 160 * 1024 && RB % 32 == 0 && ACOPIES * SHARE * 1024 == ABYTES &&
                  BCOPIES * SHARE * 1024 == BBYTES && (KSP || (NW == 4 && RB == BM)), "fits");
};

// Physical 16-byte chunk of logical chunk c in row r, rows of ROWB bytes: the
// 16 rows one pass of a 16-byte fragment read touches land on 16 distinct
// chunks of the 256-byte bank window.
template <int ROWB>
__device__ __forceinline__ int swz(int r, int c)
{
    constexpr int CH = ROWB / 16, RPW = ROWB >= 256 ? 1 : 256 / ROWB;
    return c ^ ((r / RPW) % CH);
}

template <int N>
__device__ __forceinline__ void wait_vmcnt()
{
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}
__device__ __forceinline__ void wait_lgkmcnt0() { __builtin_amdgcn_s_waitcnt(15 | (7 << 4) | (0 << 8) | (3 << 14)); }

}   // namespace ks

template <typename C, bool GATED, bool LONG>
__global__ __launch_bounds__(64 * C::NW, C::WPS) void gemm_ksplit_kernel(GemmParams p, const half_t* __restrict__ packed)
{
    using namespace ks;
    constexpr int BM = C::BM, BN = C::BN, NW = C::NW, BK = C::BK, S = C::S;
    constexpr int FM = C::WM / 32, FN = C::WN / 32, KSTEPS = C::KSTEPS;
    typedef std::conditional_t<C::F32, float4v, half8> frag;   // 16 bytes of one row
    constexpr int BNO = GATED ? BN / 2 : BN;    // output columns per tile
    constexpr int TH = 64 * NW;
    typedef typename C::TA TA;
    typedef typename C::TB TB;
    extern __shared__ half8 ks_lds[];
    LDS_AS char* lds = (LDS_AS char*)(LDS_AS void*)ks_lds;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int fr = lane & 31, fk = lane >> 5;
    const uint32_t M = p.M, N = p.N, K = p.K, H = p.H, NO = GATED ? H : N;
    const uint32_t tiles_m = (M + BM - 1) / BM, tiles_n = (NO + BNO - 1) / BNO, tiles = tiles_m * tiles_n;

    // Workgroup -> tile. Workgroups go round-robin over the 8 XCDs; each XCD
    // takes a contiguous run of the tiles, ordered so that the
    // operand with more bytes is cut up among the XCDs and the other one is
    // what every XCD's L2 reads whole.
    const uint32_t w = blockIdx.x, x = w % 8, q8 = tiles / 8, r8 = tiles % 8;
    const uint32_t t = x * q8 + (x < r8 ? x : r8) + w / 8;
    const bool nmaj = (uint64_t)NO * (GATED ? 2 : 1) * sizeof(TB) >= (uint64_t)M * sizeof(TA);
    const uint32_t tm = __builtin_amdgcn_readfirstlane(nmaj ? t % tiles_m : t / tiles_n);
    const uint32_t tn = __builtin_amdgcn_readfirstlane(nmaj ? t / tiles_m : t % tiles_n);
    const uint32_t m0 = tm * BM, n0 = tn * BNO;
    const int chunks = (int)((K + BK - 1) / BK);
    // the chunks this wave runs: all, or wave, wave + NW, ..
    const int mine = C::KSP ? (chunks - wave + NW - 1) / NW : chunks;
    const int wm0 = C::KSP ? 0 : (wave >> 1) * C::WM, wn0 = C::KSP ? 0 : (wave & 1) * C::WN;

    const TA* A = (const TA*)p.A;
    const TB* B = (const TB*)p.B;
    // W row of the tile's logical column j (clamped into W; a column past the
    // output is never stored)
    const auto wrow = [&](uint32_t j) __attribute__((always_inline)) {
        if constexpr (GATED) {
            const uint32_t c = n0 + (j < BNO ? j : j - BNO);
            return std::min(c, H - 1) + (j < BNO ? 0u : H);
        } else {
            return std::min(n0 + j, N - 1);
        }
    };

    LDS_AS char* ring = lds + (C::KSP ? wave * S * C::STAGE : 0);
    const int cw = C::KSP ? 0 : wave;   // which share of a stage's copies is this wave's

    // ---- staging ----
    // Copy slot s of an operand (16 bytes) holds row s / CH, physical chunk
    // s % CH. Rows past M read as zero (out of the resource's range), chunks
    // past the row's end too (an offset past any range).
    constexpr int ACH = C::AROW / 16, BCH = C::BROW / 16;
    constexpr int AEC = 16 / C::AES, BEC = 16 / C::BES;   // elements per chunk
    uint32_t aoff[C::ACOPIES], boff[C::BCOPIES];
    __amdgpu_buffer_rsrc_t ra, rb;
    frag sa[C::DMA ? 1 : C::ACOPIES], sb[C::DMA ? 1 : C::BCOPIES];
    if constexpr (C::DMA) {
        ra = __builtin_amdgcn_make_buffer_rsrc((void*)uniform_ptr(A + (size_t)m0 * K), (short)0,
                                               (int)__builtin_amdgcn_readfirstlane((M - m0) * K * (uint32_t)sizeof(TA)),
                                               0x00020000);
        // packed: the tile's 32-row blocks from block nb0 on (a block is K * 64
        // bytes; padding blocks fill the tile), the k steps by scalar offset
        const uint32_t nb0 = GATED ? n0 / 32 * 2 : n0 / 32;
        if constexpr (C::PK)
            rb = __builtin_amdgcn_make_buffer_rsrc((void*)uniform_ptr(packed + (size_t)nb0 * K * 32), (short)0,
                                                   (int)__builtin_amdgcn_readfirstlane((GATED && BN < 64 ? 2 : BN / 32) * K * 64),
                                                   0x00020000);
        else
            rb = __builtin_amdgcn_make_buffer_rsrc((void*)uniform_ptr(B), (short)0,
                                                   (int)__builtin_amdgcn_readfirstlane((GATED ? 2 * H : N) * K * (uint32_t)sizeof(TB)), 0x00020000);
#pragma unroll
        for (int i = 0; i < C::ACOPIES; ++i) {
            const int s = (cw * C::ACOPIES + i) * 64 + lane, row = s / ACH, ch = swz<C::AROW>(row, s % ACH);
            aoff[i] = ((uint32_t)row * K + ch * AEC) * sizeof(TA);
        }
#pragma unroll
        for (int i = 0; i < C::BCOPIES; ++i) {
            const int s = (cw * C::BCOPIES + i) * 64 + lane;
            if constexpr (C::PK) {
                // slot s: chunk s / BN, tile column s % BN
                const uint32_t ch = s / BN, j = s % BN;
                const uint32_t jo = GATED ? n0 % 32 + (j < (uint32_t)BNO ? j : j - BNO) : j;   // row within the tile's blocks
                const uint32_t blk = GATED ? jo / 32 * 2 + (j < (uint32_t)BNO ? 0 : 1) : jo / 32;
                boff[i] = blk * K * 64 + (ch * 32 + jo % 32) * 16;
            } else {
                const int row = s / BCH, ch = swz<C::BROW>(row, s % BCH);
                boff[i] = (wrow(row) * K + ch * BEC) * (uint32_t)sizeof(TB);
            }
        }
    }
    // Part q of KSTEPS of this wave's copies of chunk c into a slot, spread over
    // the MFMA steps (a burst holds the wave about 100 cycles a copy on the
    // vector memory path). Chunks past the range copy zeros, so that the
    // number of copies in flight stays fixed.
    const auto issue_part = [&](int slot, int c, int q) __attribute__((always_inline)) {
        const uint32_t k0 = (uint32_t)c * BK;
        const uint32_t left = c < chunks ? K - k0 : 0u;
        LDS_AS char* adst = ring + slot * C::STAGE + cw * C::ACOPIES * 1024;
        LDS_AS char* bdst = ring + slot * C::STAGE + C::ABYTES + cw * C::BCOPIES * 1024;
#pragma unroll
        for (int i = C::ACOPIES * q / KSTEPS; i < C::ACOPIES * (q + 1) / KSTEPS; ++i) {
            const int s = (cw * C::ACOPIES + i) * 64 + lane, ch = swz<C::AROW>(s / ACH, s % ACH);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (LDS_AS void*)(adst + i * 1024), 16,
                                                     (int)((uint32_t)ch * AEC < left ? aoff[i] : 0x80000000u),
                                                     (int)(k0 * sizeof(TA)), 0, 0);
        }
#pragma unroll
        for (int i = C::BCOPIES * q / KSTEPS; i < C::BCOPIES * (q + 1) / KSTEPS; ++i) {
            const int s = (cw * C::BCOPIES + i) * 64 + lane, ch = C::PK ? s / BN : swz<C::BROW>(s / BCH, s % BCH);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (LDS_AS void*)(bdst + i * 1024), 16,
                                                     (int)((uint32_t)ch * BEC < left ? boff[i] : 0x80000000u),
                                                     (int)(k0 * (C::PK ? 64 : (int)sizeof(TB))), 0, 0);
        }
    };
    const auto issue = [&](int slot, int c) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < KSTEPS; ++q) issue_part(slot, c, q);
    };
    // Register staging of chunk c, and its write into a stage. Rows past M
    // read row M - 1 (their outputs are never stored); a piece past the row's
    // last PE elements reads those and moves them down.
    constexpr int PE = C::F32 ? 4 : 8;          // elements per piece
    const auto fetch = [&](int c) __attribute__((always_inline)) {
        const uint32_t k0 = (uint32_t)c * BK;
        const bool whole = k0 + BK <= K;
        const auto piece = [&](const auto* row, uint32_t k) __attribute__((always_inline)) {
            if constexpr (C::F32) return load4f(row + std::min(k, K - PE));
            else return load8(row + std::min(k, K - PE));
        };
#pragma unroll
        for (int i = 0; i < C::ACOPIES; ++i) {
            const int s = (cw * C::ACOPIES + i) * 64 + lane;
            sa[i] = piece(A + (size_t)std::min(m0 + s / ACH, M - 1) * K, k0 + (s % ACH) * PE);
        }
#pragma unroll
        for (int i = 0; i < C::BCOPIES; ++i) {
            const int s = (cw * C::BCOPIES + i) * 64 + lane;
            sb[i] = piece(B + (size_t)wrow(s / BCH) * K, k0 + (s % BCH) * PE);
        }
        if (!whole) {
#pragma unroll
            for (int i = 0; i < C::ACOPIES; ++i) {
                const uint32_t k = k0 + (((cw * C::ACOPIES + i) * 64 + lane) % ACH) * PE;
                sa[i] = shift_down(sa[i], std::min<uint32_t>(k - std::min(k, K - PE), PE));
            }
#pragma unroll
            for (int i = 0; i < C::BCOPIES; ++i) {
                const uint32_t k = k0 + (((cw * C::BCOPIES + i) * 64 + lane) % BCH) * PE;
                sb[i] = shift_down(sb[i], std::min<uint32_t>(k - std::min(k, K - PE), PE));
            }
        }
    };
    const auto place = [&](int slot) __attribute__((always_inline)) {
        LDS_AS char* st = ring + slot * C::STAGE;
#pragma unroll
        for (int i = 0; i < C::ACOPIES; ++i) {
            const int s = (cw * C::ACOPIES + i) * 64 + lane, row = s / ACH;
            *(LDS_AS frag*)(st + row * C::AROW + swz<C::AROW>(row, s % ACH) * 16) = sa[i];
        }
#pragma unroll
        for (int i = 0; i < C::BCOPIES; ++i) {
            const int s = (cw * C::BCOPIES + i) * 64 + lane, row = s / BCH;
            *(LDS_AS frag*)(st + C::ABYTES + row * C::BROW + swz<C::BROW>(row, s % BCH) * 16) = sb[i];
        }
    };

    // ---- fragments: row i*32 + fr of the wave's part, k step q (lane half fk:
    // 8 of its 16, or 4 of its 8 fp32) ----
    const auto read_x = [&](const LDS_AS char* st, int i, int q) __attribute__((always_inline)) {
        const int row = wm0 + i * 32 + fr;
        if constexpr (C::AES == 2 || C::F32) {
            return *(const LDS_AS frag*)(st + row * C::AROW + swz<C::AROW>(row, q * 2 + fk) * 16);
        } else {
            const float4v lo = *(const LDS_AS float4v*)(st + row * C::AROW + swz<C::AROW>(row, q * 4 + 2 * fk) * 16);
            const float4v hi = *(const LDS_AS float4v*)(st + row * C::AROW + swz<C::AROW>(row, q * 4 + 2 * fk + 1) * 16);
            return __builtin_shufflevector(__builtin_convertvector(lo, half4), __builtin_convertvector(hi, half4), 0, 1,
                                           2, 3, 4, 5, 6, 7);
        }
    };
    const auto read_w = [&](const LDS_AS char* st, int j, int q) __attribute__((always_inline)) {
        const int row = wn0 + j * 32 + fr;
        if constexpr (C::PK) return *(const LDS_AS half8*)(st + C::ABYTES + ((q * 2 + fk) * BN + row) * 16);
        else return *(const LDS_AS frag*)(st + C::ABYTES + row * C::BROW + swz<C::BROW>(row, q * 2 + fk) * 16);
    };

    // This thread's output columns in the final exchange (the same for each of
    // its rows), and their bias, loaded ahead of the K loop.
    constexpr int CG = BNO / 4;                 // 4-column groups per output row
    const uint32_t cg = threadIdx.x % CG, col = n0 + 4 * cg;
    const bool row_bias = !p.bias || p.bias_repeat == (GATED ? 2 * H : N);
    float bg[4] = {0.f, 0.f, 0.f, 0.f}, bu[4] = {0.f, 0.f, 0.f, 0.f};
    if (p.bias && row_bias) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const uint32_t c = std::min(col + e, NO - 1);
            bg[e] = ld(p.bias, p.bias_dtype, c);
            if constexpr (GATED) bu[e] = ld(p.bias, p.bias_dtype, H + c);
        }
    }

    // D = W X^T: lane (fr, fk) holds X row i*32 + fr at columns j*32 + 8 g + 4 fk .. +3.
    // The k steps go to AS sums in turn. LONG: no sum runs over more than 256 k
    // (fp32 128), the shortest split of the split-K launches whose place this
    // kernel takes, before it goes to the total, so that the error is no larger
    // than theirs (K = 4096: one chain 4.1e-7 relative, 8 splits 1.6e-7, this
    // 1.3e-7; K = 8192 in 16 sums 1.6e-7, this 1.3e-7). A chain's first MFMA
    // starts from a zero operand; the additions run beside the MFMAs before it
    // (fp16 X, us, one chain / this: [500, 4096], N 4096 31.8 / 32.8; [400,
    // 4096], N 8192 42.5 / 45; [61, 8192], N 5120 21.9 / 22.3).
    constexpr int AS = LONG ? C::LAS : C::AS;
    float16v acc[AS][FM][FN], total[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            total[i][j] = (float16v)0.f;
#pragma unroll
            for (int a = 0; a < AS; ++a) acc[a][i][j] = (float16v)0.f;
        }

    // A stage's MFMAs; step(q) runs after those of k step q. KSP reads all of
    // the stage's fragments first (so that its slot can be refilled during the
    // MFMAs), the shared ring's waves read one step ahead. NEW: new chains start.
    const auto stage_mfma = [&](const LDS_AS char* st, auto NEW, auto&& step) __attribute__((always_inline)) {
        constexpr int AHEAD = C::KSP ? KSTEPS : 1, SETS = C::KSP ? KSTEPS : 2;
        frag xf[SETS][FM], wf[SETS][FN];
#pragma unroll
        for (int q = 0; q < AHEAD; ++q) {
#pragma unroll
            for (int i = 0; i < FM; ++i) xf[q][i] = read_x(st, i, q);
#pragma unroll
            for (int j = 0; j < FN; ++j) wf[q][j] = read_w(st, j, q);
        }
        if constexpr (C::KSP && C::DMA) wait_lgkmcnt0();
#pragma unroll
        for (int q = 0; q < KSTEPS; ++q) {
            if (q + AHEAD < KSTEPS) {
#pragma unroll
                for (int i = 0; i < FM; ++i) xf[(q + AHEAD) % SETS][i] = read_x(st, i, q + AHEAD);
#pragma unroll
                for (int j = 0; j < FN; ++j) wf[(q + AHEAD) % SETS][j] = read_w(st, j, q + AHEAD);
            }
            // the next MFMA of a sum: its chain so far, or nothing as that joins the total
            const auto chain = [&](int a, int i, int j, bool first) __attribute__((always_inline)) {
                if (!first) return acc[a][i][j];
                total[i][j] += acc[a][i][j];
                return (float16v)0.f;
            };
            if constexpr (C::F32) {
                // element e of both halves' pieces is one k pair (the same on both operands)
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int i = 0; i < FM; ++i)
#pragma unroll
                        for (int j = 0; j < FN; ++j)
                            acc[e % AS][i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(
                                wf[q % SETS][j][e], xf[q % SETS][i][e], chain(e % AS, i, j, NEW && q == 0 && e < AS), 0, 0, 0);
            } else {
#pragma unroll
                for (int i = 0; i < FM; ++i)
#pragma unroll
                    for (int j = 0; j < FN; ++j)
                        acc[q % AS][i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                            wf[q % SETS][j], xf[q % SETS][i], chain(q % AS, i, j, NEW && q < AS), 0, 0, 0);
            }
            if constexpr (C::DMA) __builtin_amdgcn_sched_barrier(0);
            step(q);
            if constexpr (C::DMA) __builtin_amdgcn_sched_barrier(0);
        }
    };
    // stage(r, NEW) for r = 0 .. mine - 1
    // (128x128 replaced at most 7 splits: 512 k and more each from K = 3584 up)
    const uint32_t chain = C::CHAIN * (BM == 128 && K >= 7 * 512 ? 2u : 1u);
    const auto stages = [&](auto&& stage) __attribute__((always_inline)) {
        for (int r = 0; r < mine;) {
            const int end = LONG ? std::min(r + (int)chain, mine) : mine;
            if constexpr (LONG) stage(r++, std::true_type{});
            for (; r < end; ++r) stage(r, std::false_type{});
        }
    };

    if constexpr (C::DMA && C::KSP) {
        // Stage r of this wave is its chunk wave + r NW. S stages are in
        // flight or being read: at the top of trip r stages r .. r + S - 1 are
        // issued, so once at most (S - 1) COPIES copies are outstanding stage r
        // has landed. Its slot is refilled when every read of it returned.
#pragma unroll
        for (int r = 0; r < S; ++r) issue(r, wave + r * NW);
        int slot = 0;
        stages([&](int r, auto NEW) __attribute__((always_inline)) {
            wait_vmcnt<(S - 1) * C::COPIES>();
            stage_mfma(ring + slot * C::STAGE, NEW, [&](int q) __attribute__((always_inline)) {
                issue_part(slot, wave + (r + S) * NW, q);
            });
            slot = slot + 1 == S ? 0 : slot + 1;
        });
        wait_vmcnt<0>();   // the copies past the range land before LDS is reused
    } else if constexpr (C::DMA) {
        // Stages r .. r + S - 2 are issued at the top of trip r: once at most
        // (S - 2) COPIES of this wave's copies are outstanding its share of
        // stage r has landed, after the barrier every wave's has, and every
        // wave is done reading stage r - 1 (its reads returned before the
        // barrier), whose slot takes stage r + S - 1.
#pragma unroll
        for (int r = 0; r < S - 1; ++r) issue(r, r);
        int slot = 0;
        stages([&](int r, auto NEW) __attribute__((always_inline)) {
            wait_vmcnt<(S - 2) * C::COPIES>();
            wait_lgkmcnt0();
            __builtin_amdgcn_s_barrier();
            const int free = slot == 0 ? S - 1 : slot - 1;
            stage_mfma(ring + slot * C::STAGE, NEW,
                       [&](int q) __attribute__((always_inline)) { issue_part(free, r + S - 1, q); });
            slot = slot + 1 == S ? 0 : slot + 1;
        });
        wait_vmcnt<0>();   // the copies past the range land before LDS is reused
    } else if constexpr (C::KSP) {
        if (mine > 0) fetch(wave);
        stages([&](int r, auto NEW) __attribute__((always_inline)) {
            place(0);
            if (r + 1 < mine) fetch(wave + (r + 1) * NW);
            stage_mfma(ring, NEW, [](int) {});
        });
    } else {
        // A wave that writes stage r + 2 has passed the barrier of trip
        // r + 1, so every wave is done reading stage r from the same slot.
        fetch(0);
        stages([&](int r, auto NEW) __attribute__((always_inline)) {
            place(r & 1);
            if (r + 1 < mine) fetch(r + 1);
            __syncthreads();
            stage_mfma(ring + (r & 1) * C::STAGE, NEW, [](int) {});
        });
    }

#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int a = 0; a < AS; ++a) total[i][j] += acc[a][i][j];

    // ---- the partial tiles meet in LDS, RB rows at a time ----
    // U rows of a thread's four columns at a time, the residual of the next U
    // loaded ahead; as vectors where rows are whole aligned groups of four
    // (`al`). A bias or residual with its own repeat goes element by element.
    const bool al = NO % 4 == 0 && ((uintptr_t)p.C % 16) == 0 && ((uintptr_t)p.residual % 16) == 0;
    const bool batch = row_bias && (!p.residual || p.residual_repeat == 0);
    const bool res = !GATED && p.residual;
    constexpr int RSTEP = TH / CG, RT = C::RB > RSTEP ? C::RB / RSTEP : 1;   // rows per thread and round
    constexpr int U = RT < 4 ? RT : 4;
    static_assert(RT % U == 0, "whole groups of rows");
    const uint32_t r0 = threadIdx.x / CG;
#pragma unroll
    for (int h = 0; h < BM / C::RB; ++h) {
        float4v rv[U];
        const auto residual = [&](int t0) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < U; ++i) {
                const uint32_t row = std::min(m0 + h * C::RB + r0 + (t0 + i) * RSTEP, M - 1);
                const size_t o = (size_t)row * NO + (al ? std::min(col, NO - 4) : 0u);
                if (!al) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) rv[i][e] = ld(p.residual, p.residual_dtype, o + std::min(col + e, NO - 1));
                } else if (p.residual_dtype == DT_F16)
                    rv[i] = __builtin_convertvector(*(const half4*)((const half_t*)p.residual + o), float4v);
                else
                    rv[i] = *(const float4v*)((const float*)p.residual + o);
            }
        };
        if (batch && res) residual(0);
        __syncthreads();
#pragma unroll
        for (int i = C::KSP ? h * (C::RB / 32) : 0; i < (C::KSP ? (h + 1) * (C::RB / 32) : FM); ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const int row = (C::KSP ? wave * C::RB : wm0) + i * 32 + fr - h * C::RB;
                    *(LDS_AS float4v*)(lds + row * C::RROW + (wn0 + j * 32 + 8 * g + 4 * fk) * 4) =
                        float4v{total[i][j][4 * g], total[i][j][4 * g + 1], total[i][j][4 * g + 2], total[i][j][4 * g + 3]};
                }
        __syncthreads();
        const auto sums = [&](uint32_t rr, float4v& v, float4v& up) __attribute__((always_inline)) {
            v = up = (float4v)0.f;
#pragma unroll
            for (int w2 = 0; w2 < C::PLANES; ++w2) {
                const LDS_AS char* src = lds + (w2 * C::RB + rr) * C::RROW + cg * 16;
                v += *(const LDS_AS float4v*)src;
                if constexpr (GATED) up += *(const LDS_AS float4v*)(src + BNO * 4);
            }
        };
        if (batch) {
#pragma unroll 1
            for (int t0 = 0; t0 < RT; t0 += U) {
                float4v v[U], up[U], rc[U];
#pragma unroll
                for (int i = 0; i < U; ++i) {
                    sums(std::min<uint32_t>(r0 + (t0 + i) * RSTEP, C::RB - 1), v[i], up[i]);
                    rc[i] = res ? rv[i] : (float4v)0.f;
                }
                if (res && t0 + U < RT) residual(t0 + U);
                const auto rows = [&](auto&& put) __attribute__((always_inline)) {
#pragma unroll
                    for (int i = 0; i < U; ++i) {
                        const uint32_t rr = r0 + (t0 + i) * RSTEP, row = m0 + h * C::RB + rr;
                        if (rr < C::RB && row < M && col < NO) put(i, row);
                    }
                };
                const auto act = [&](auto EPI) __attribute__((always_inline)) {
#pragma unroll
                    for (int i = 0; i < U; ++i)
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            if constexpr (GATED) v[i][e] = epilogue(v[i][e] + bg[e], EPI) * (up[i][e] + bu[e]);
                            else v[i][e] = finish(v[i][e] + bg[e], rc[i][e], EPI, p.residual_order, p.scalar_scale);
                        }
                };
                switch (p.epilogue) {
                case 0: act(std::integral_constant<uint32_t, 0>{}); break;
                case 1: act(std::integral_constant<uint32_t, 1>{}); break;
                case 2: act(std::integral_constant<uint32_t, 2>{}); break;
                case 3: act(std::integral_constant<uint32_t, 3>{}); break;
                case 4: act(std::integral_constant<uint32_t, 4>{}); break;
                default: act(std::integral_constant<uint32_t, 5>{}); break;
                }
                if (!al)
                    rows([&](int i, uint32_t row) __attribute__((always_inline)) {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (col + e < NO) st(p.C, p.c_dtype, (size_t)row * NO + col + e, v[i][e]);
                    });
                else if (p.c_dtype == DT_F16)
                    rows([&](int i, uint32_t row) __attribute__((always_inline)) {
                        *(half4*)((half_t*)p.C + (size_t)row * NO + col) = __builtin_convertvector(v[i], half4);
                    });
                else
                    rows([&](int i, uint32_t row) __attribute__((always_inline)) {
                        *(float4v*)((float*)p.C + (size_t)row * NO + col) = v[i];
                    });
            }
        } else {
#pragma unroll 1
            for (uint32_t rr = r0; rr < C::RB; rr += RSTEP) {
                const uint32_t row = m0 + h * C::RB + rr;
                if (row >= M) break;
                float4v v, up;
                sums(rr, v, up);
#pragma unroll 1
                for (uint32_t e = 0; e < 4 && col + e < NO; ++e) {
                    const float x = e == 0 ? v[0] : e == 1 ? v[1] : e == 2 ? v[2] : v[3];
                    const float y = e == 0 ? up[0] : e == 1 ? up[1] : e == 2 ? up[2] : up[3];
                    const uint32_t c = col + e;
                    const size_t o = (size_t)row * NO + c;
                    if constexpr (GATED) {
                        const float g0 = p.bias ? ld(p.bias, p.bias_dtype, c) : 0.f;
                        const float u0 = p.bias ? ld(p.bias, p.bias_dtype, H + c) : 0.f;
                        st(p.C, p.c_dtype, o, epilogue(x + g0, p.epilogue) * (y + u0));
                    } else {
                        store_output_general(OutputSpec{p.C, p.bias, p.residual, p.c_dtype, p.bias_dtype, p.bias_repeat,
                                                        p.residual_repeat, p.epilogue, p.residual_order, p.scalar_scale},
                                             o, x);
                    }
                }
            }
        }
    }
}

// fp16 W with fp16 or fp32 X, or both fp32 (ungated); 32-bit buffer offsets.
bool gemm_ksplit_ok(const GemmParams& p, bool gated)
{
    const uint64_t as = p.a_dtype == DT_F16 ? 2 : 4, bs = p.b_dtype == DT_F16 ? 2 : 4;
    return (p.b_dtype == DT_F16 || (p.a_dtype == DT_F32 && !gated)) && p.batch == 1 &&
           (uint64_t)p.M * p.K * as < (1ull << 31) && (uint64_t)p.N * p.K * bs < (1ull << 31) &&
           (uint64_t)p.M * p.N < (1ull << 31) && p.K >= 32 && p.K < (1u << 22) && (!gated || p.H > 0);
}

// The tiles offered. A launch takes about 2.5 us plus, per round of tiles over
// the CUs, `fixed` plus `chunk` per 64 k (us; index 0: fp16 X, 1: fp32 X, 2:
// fp32 X and W; measured on full grids at K = 768 and 2048). fp32 products run
// at 1/16 of the fp16 rate: operands take a quarter of the time and only the
// smallest quadrants and K-split tiles are of use.
namespace ks {
struct Tile { int bm, bn; float fixed[3], chunk[3]; };
constexpr float NONE = 1e9f;
constexpr Tile TILES[] = {
    {32, 32, {2.2f, 1.7f, 1.5f}, {.091f, .165f, .31f}},     // 8 waves split K
    {32, 64, {2.2f, 2.3f, NONE}, {.14f, .18f, 0.f}},        // 4 waves split K
    {64, 64, {2.85f, 1.7f, 2.3f}, {.17f, .37f, 1.1f}},      // (fp32: quadrants)
    {64, 128, {2.3f, 2.7f, NONE}, {.39f, .465f, 0.f}},      // quadrants
    {128, 128, {4.0f, 2.3f, NONE}, {.55f, .84f, 0.f}},
};
constexpr int NTILES = sizeof(TILES) / sizeof(TILES[0]);

// Whole 16-byte chunks everywhere: the copies go straight to LDS.
inline bool dma_ok(const GemmParams& p)
{
    return p.K % (p.b_dtype == DT_F16 ? 8 : 4) == 0 && ((uintptr_t)p.A % 16) == 0 && ((uintptr_t)p.B % 16) == 0;
}
}

void gemm_ksplit_tile(int tile, uint32_t& bm, uint32_t& bn)
{
    bm = ks::TILES[tile].bm;
    bn = ks::TILES[tile].bn;
}

float gemm_ksplit_tile_us(const GemmParams& p, bool gated, uint32_t cus, int tile)
{
    const int x = p.b_dtype == DT_F32 ? 2 : p.a_dtype == DT_F16 ? 0 : 1;
    // (register staging: fp16 1.5-1.9; fp32 measured alike, 15.2 us a tile at K = 767 and 768)
    const float chunks = (float)((p.K + 63) / 64) * (ks::dma_ok(p) || x == 2 ? 1.f : 1.7f);
    const uint32_t cols = gated ? 2 * p.H : p.N;
    const ks::Tile& k = ks::TILES[tile];
    const uint64_t tiles = (uint64_t)((p.M + k.bm - 1) / k.bm) * ((cols + k.bn - 1) / k.bn);
    // (fp32 quadrants alone on a CU, one wave per SIMD: 22 us where a pair takes 2 x 19)
    const float rounds = (float)((tiles + cus - 1) / cus) * (x == 2 && k.bm == 64 && tiles <= cus ? 1.15f : 1.f);
    return 2.5f + rounds * (k.fixed[x] + chunks * k.chunk[x]);
}

int gemm_ksplit_plan(const GemmParams& p, bool gated, uint32_t cus, float* us)
{
    int best = 0;
    *us = 1e30f;
    for (int t = 0; t < ks::NTILES; ++t) {
        const float cost = gemm_ksplit_tile_us(p, gated, cus, t);
        if (cost < *us) { *us = cost; best = t; }
    }
    return best;
}

// The 32x32 tile's time where its tiles are far fewer than the CUs: more bytes a
// cycle for each than on a full grid (8 and 32 tiles, K = 2048 to 32768; fp32
// operands alike).
float gemm_ksplit_few_us(const GemmParams& p)
{
    const float chunks = (float)((p.K + 63) / 64);
    if (p.b_dtype == DT_F32) return 4.f + .31f * chunks;
    // (fp32 X in rows off 128-byte lines: 234 x 7080 25.3 us)
    if (p.a_dtype == DT_F32)
        return 4.2f + (!ks::dma_ok(p) ? .16f : p.K % 32 == 0 || p.M <= 32 ? .135f : .175f) * chunks;
    return 4.7f + (ks::dma_ok(p) ? .08f : .125f) * chunks;
}

template <typename C, bool GATED, bool LONG>
static hipError_t launch_long(const GemmParams& p, const void* packed, hipStream_t s)
{
    static PerDevice lds_once;
    hipError_t e = set_max_lds(lds_once, (const void*)gemm_ksplit_kernel<C, GATED, LONG>, C::LDS);
    if (e != hipSuccess) return e;
    const uint32_t no = GATED ? p.H : p.N, bno = GATED ? C::BN / 2 : C::BN;
    const uint32_t tiles = ((p.M + C::BM - 1) / C::BM) * ((no + bno - 1) / bno);
    hipLaunchKernelGGL((gemm_ksplit_kernel<C, GATED, LONG>), dim3(tiles), dim3(64 * C::NW), C::LDS, s, p,
                       (const half_t*)packed);
    return hipGetLastError();
}

template <typename C, bool GATED>
static hipError_t launch_cfg(const GemmParams& p, const void* packed, hipStream_t s)
{
    // (an fp16 quadrant's one sum is 256 k long at once; fp32 quadrants keep four
    // sums, more than the splits the same sizes had: they take 61 and more tiles
    // of 64x64, and so at most 4)
    if constexpr (C::F32 && !C::KSP) {
        return launch_long<C, GATED, false>(p, packed, s);
    } else {
        if constexpr (C::KSP)
            if (!C::long_k(p.K)) return launch_long<C, GATED, false>(p, packed, s);
        return launch_long<C, GATED, true>(p, packed, s);
    }
}

template <typename TA, bool DMA, bool PK, bool GATED>
static hipError_t launch_tile(const GemmParams& p, const void* packed, int tile, hipStream_t s)
{
    constexpr bool H = sizeof(TA) == 2 || !DMA;   // X is fp16 in LDS
    switch (tile) {
    case 0: return launch_cfg<ks::Cfg<32, 32, 8, H ? 64 : 32, H ? 2 : 3, true, TA, DMA, PK>, GATED>(p, packed, s);
    case 1: return launch_cfg<ks::Cfg<32, 64, 4, 64, H ? 3 : 2, true, TA, DMA, PK>, GATED>(p, packed, s);
    case 2: return launch_cfg<ks::Cfg<64, 64, 4, H ? 64 : 32, H ? 2 : 3, true, TA, DMA, PK>, GATED>(p, packed, s);
    case 3: return launch_cfg<ks::Cfg<64, 128, 4, 64, 4, false, TA, DMA, PK>, GATED>(p, packed, s);
    case 4: return launch_cfg<ks::Cfg<128, 128, 4, 64, H ? 4 : 3, false, TA, DMA, PK>, GATED>(p, packed, s);
    default: return hipErrorInvalidValue;
    }
}

template <typename TA, bool DMA, bool PK>
static hipError_t launch_gate(const GemmParams& p, const void* packed, bool gated, int tile, hipStream_t s)
{
    return gated ? launch_tile<TA, DMA, PK, true>(p, packed, tile, s) : launch_tile<TA, DMA, PK, false>(p, packed, tile, s);
}

template <bool DMA>
static hipError_t launch_f32(const GemmParams& p, int tile, hipStream_t s)
{
    if (tile == 0) return launch_cfg<ks::Cfg<32, 32, 8, 32, 2, true, float, DMA, false, float>, false>(p, nullptr, s);
    return launch_cfg<ks::Cfg<64, 64, 4, 32, 4, false, float, DMA, false, float>, false>(p, nullptr, s);
}

hipError_t gemm_ksplit_launch(const GemmParams& p, const void* packed, bool gated, int tile, hipStream_t s)
{
    const bool dma = ks::dma_ok(p);
    if (p.b_dtype == DT_F32) return dma ? launch_f32<true>(p, tile, s) : launch_f32<false>(p, tile, s);
    if (p.a_dtype == DT_F16) {
        // (the packed form has K % 128 == 0: no short chunk). The weight itself
        // is then not read, as in the 256x256 kernel over the packed form.
        if (packed && ((uintptr_t)packed % 16) == 0 && ((uintptr_t)p.A % 16) == 0)
            return launch_gate<half_t, true, true>(p, packed, gated, tile, s);
        return dma ? launch_gate<half_t, true, false>(p, nullptr, gated, tile, s)
                   : launch_gate<half_t, false, false>(p, nullptr, gated, tile, s);
    }
    return dma ? launch_gate<float, true, false>(p, nullptr, gated, tile, s)
               : launch_gate<float, false, false>(p, nullptr, gated, tile, s);
}

}   // namespace vai_dev
