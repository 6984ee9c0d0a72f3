// Pipelined tile GEMM of tall tiles, 16 R x 256 outputs (R = 9 .. 16), for weights in MFMA operand order.
// Workgroup = 4 wavefronts side by side: each walks all 16 R token rows and owns 64 columns, R x 4 accumulators of
// v_mfma_f32_16x16x128_f8f6f4.  Its weights are its own, so they go global -> registers through a ring of four register
// sets; LDS carries the activations only, through a ring of four stages of 128 bytes of K that the wavefronts hand to each
// other through progress words instead of meeting at a barrier per stage.  Any number of row blocks: the planner takes the
// height that fills the rounds of 256 workgroups best (4800 rows x 2048 columns: 30 x 8 tiles of 160 rows, one round).
//
// What bounds it: with so many accumulators there is one wavefront per SIMD, and nothing overlaps what it does outside its
// main loop.  A tile of 224 rows used to be 6 k cycles of opening (all CUs ask at once), 34 k of main loop for 28.7 k of MFMAs
// at K = 2048, 10 k of GeGLU arithmetic and 2.5 k of stores, 53 k in all.  So:
//  * one workgroup per CU for the whole launch takes tile after tile (every 32nd of its XCD's), and asks for the next tile's
//    first two stage-loads, scales and bias in between the pieces of the present one's epilogue;
//  * the last two stage-loads are multiplied row block by row block, and the epilogue of the block before goes in between: the
//    matrix pipe runs under VALU work of three times its length;
//  * the first MFMA of a sum takes zero in place of it: no accumulators are cleared;
//  * requests are spread over all MFMAs of a stage (weights in its first half, activations in the second): in one half they
//    kept the CU's address unit busy for longer than that (main loop of 208 rows 28.4 -> 27.3 k cycles).
// 47 k cycles a tile at 224 rows, K = 2048, GeGLU: main loop 29.4 k for 25.1 k of MFMAs, last two stages and epilogue 15.4 k (9.4 k
// without an activation, 28.3 k with GELU), 2 k from there to the next tile's first stage; the first tile's opening 6 - 10 k.
// us of a GEMM on ready codes, the shape that was taken before / this kernel: 816 x 32768 x 2048 + GeGLU (208 rows) 60.5 / 52.3,
// 13056 x 32768 x 2048 + GeGLU 752 / 706, 4800 x 6144 x 2048 (240) 58.4 / 48.1, 4800 x 8192 x 2048 + GELU (208) 92.8 / 87.4,
// 4800 x 2048 x 8192 (160) 67 / 57.5, 4800 x 2048 x 2048 21.5 / 17.6, 3264 x 2560 x 2048 (144) 21.4 / 17.2, 6528 x 2048 x 2048
// (208) 28.5 / 22.3, 13056 x 2048 x 16384 297 / 288.
// Row-major weights are not served: straight into registers they come in 64-byte pieces of 16 rows per instruction, and the same
// kernel is then slower than tiles with staged weights (4800 x 2048 x 8192 78 against 60 us on operand order).
#include "gemm_big.h"
#include "stamps.h"
#include "weight_layout.h"
#include <stdlib.h>
#include <type_traits>
#include <utility>

namespace phyai {

// (debug build only; of a workgroup's last tile: 1 first stage published, 2 main loop done but for the last two stages,
// 3 everyone there, 4 those and the epilogue done)
PHYAI_STAMP_SINK(g_tall_stamps)

constexpr uint32_t kNowhere = 0x80000000u;   // an offset that no resource of the epilogue reaches
typedef unsigned int v4u __attribute__((ext_vector_type(4)));
constexpr int TALL_COLS = 256, TALL_GRID = 256;   // columns of a tile; workgroups of a launch of more tiles than that

// f(0), ..., f(N - 1) with the index as a type: register arrays are indexed by it, whatever the unroller thinks of the size.
template <class F, int... I>
__device__ __forceinline__ void tall_each_of(F&& f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }
template <int N, class F>
__device__ __forceinline__ void tall_each(F&& f) { tall_each_of(f, std::make_integer_sequence<int, N>{}); }

template <int R, int EPI, bool RES>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1)))
void gemm_fp8_tall_kernel(
    const uint8_t* __restrict__ a_a, const uint8_t* __restrict__ a_b, int a_K, int a_M, int a_N, int a_m_tiles, int a_order,
    const float* __restrict__ a_a_scale, const float* __restrict__ a_b_scale, const uint16_t* __restrict__ a_bias,
    uint16_t* __restrict__ a_out, int64_t a_ldo, const ResidualArgs a_res) {
    PHYAI_STAMP_BEGIN
    constexpr bool GATED = epi_is_gated(EPI);
    constexpr int BM = 16 * R, BN = TALL_COLS, WN = 64;
    constexpr int H0 = (R + 1) / 2, H1 = R / 2;      // row blocks of the two halves of a stage-load's MFMAs
    constexpr int CA = (R + 1) / 2;                  // copies of 8 activation rows per wavefront and stage-load
    constexpr int BL = 8;                            // 16-byte weight loads per lane and stage-load: 4 blocks of 16 columns x 2
    constexpr int COPIES = CA + BL;
    constexpr int STAGE_BYTES = CA * 32 * BIG_BK;
    constexpr int DEPTH = 4, LEAD = 3, CLAIM = 2, SLACK = 1;   // (see hand_over)
    constexpr int SLOTS_AFTER = 4 * (H1 - 1);        // MFMAs of a stage-load behind its hand-over
    static_assert(R >= 9 && R <= 16, "144 to 256 rows");
    // a staged row block of the epilogue; two per wavefront
    constexpr int TNO = GATED ? 1 : 2;               // output column blocks of 32 per wavefront
    constexpr int ROWB = TNO * 64, SLOTS = ROWB / 16, ROWS_PER_PASS = 16 / SLOTS, LEAVES = TNO;
    constexpr int STAGING_AT = DEPTH * STAGE_BYTES, RING_END = STAGING_AT + 8 * 16 * ROWB;
    // row scales, weight scales and bias of two tiles, in blocks of 64 words
    constexpr int XBLOCKS = (BM + 63) / 64, WBLOCKS = BN / 64, BBLOCKS = BN / 128, BLOCKS = XBLOCKS + WBLOCKS + BBLOCKS;
    constexpr int CONSTS = (BLOCKS + 3) / 4;         // copies of a wavefront
    constexpr int CONST_AT = RING_END + 16, CONST_BYTES = BLOCKS * 256;
    __shared__ __attribute__((aligned(1024))) uint8_t lds[CONST_AT + 2 * CONST_BYTES];

    // (pointers that say "LDS": through a generic pointer the accesses would be flat ones, counted with the copies)
    typedef __attribute__((address_space(3))) int lds_int_t;
    typedef __attribute__((address_space(3))) v4i lds_v4i_t;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wn = __builtin_amdgcn_readfirstlane(wave);
    const int l16 = lane & 15, q = lane >> 4;
    const int M = a_M, N = a_N, K = a_K, half_n = a_N / 2;
    const int band = a_order & 255, by_rows = (a_order >> 8) & 1, one_scale = (a_order >> 11) & 1;
    const int n_tiles_all = ((GATED ? half_n : N) + (GATED ? BN / 2 : BN) - 1) / (GATED ? BN / 2 : BN);
    const int n_loads = K / BIG_BK;
    const uint32_t lane16 = (uint32_t)lane * 16;
    const uint32_t lds_base = (uint32_t)(uintptr_t)lds;
    const uint32_t wave_a = __builtin_amdgcn_readfirstlane(lds_base + wave * (CA * 1024));

    // What depends on the lane alone would be computed once in front of the loop over the tiles and kept, in more registers than
    // there are: `here` makes a value opaque, so that what is derived from it is computed where it is used.
    auto here = [](int v) __attribute__((always_inline)) { asm volatile("" : "+v"(v)); return v; };
    auto here_s = [](int v) __attribute__((always_inline)) { asm volatile("" : "+s"(v)); return v; };

    // ---- tiles -------------------------------------------------------------------------------------
    int m0, n0;
    uint32_t aoff[CA];
    const uint8_t* bsrc[4];                          // weight block jj (16 columns; gated: 8 gate columns and their up columns), K step 0
    // This workgroup's tiles: every 32nd of its XCD's (workgroups go to the 8 XCDs in turn), from its own place there on.
    int at = blockIdx.x >> 3, tile_m = 0, tile_n = 0;
    auto next_tile = [&]() -> bool {   // false: none left
        const int m_tiles = here_s(a_m_tiles), n_tiles = here_s(n_tiles_all);
        const BigTile t = big_tile_of_xcd(blockIdx.x & 7, at, by_rows ? n_tiles : m_tiles, by_rows ? m_tiles : n_tiles, band);
        at += TALL_GRID / 8;
        tile_m = by_rows ? t.n : t.m;   // (by_rows: an XCD takes tile rows)
        tile_n = by_rows ? t.m : t.n;
        return by_rows ? tile_m < m_tiles : tile_n < n_tiles;
    };
    // step 0 .. CA: the places that the next tile's requests read from
    auto take_tile = [&](int step) __attribute__((always_inline)) {
        if (step == 0) {
            m0 = tile_m * BM;
            n0 = GATED ? tile_n * (BN / 2) : tile_n * BN;
            const uint32_t unit0 = GATED ? (uint32_t)n0 >> 3 : (uint32_t)n0 >> 4, units = (uint32_t)N >> 4;
#pragma unroll
            for (int jj = 0; jj < 4; ++jj) {
                const uint32_t u = unit0 + (uint32_t)(wn * 4 + jj);
                bsrc[jj] = a_b + (size_t)(u < units ? u : units - 1) * ((size_t)K << 4);
            }
        } else if (step <= CA) {
            const int ln = here(lane), rt = (wn * CA + step - 1) * 8 + (ln >> 3);
            const int r = m0 + rt < M ? m0 + rt : M - 1;
            aoff[step - 1] = (uint32_t)r * (uint32_t)K + (((ln & 7) ^ big_swizzle(rt)) << 4);
        }
    };

    // ---- requests ----------------------------------------------------------------------------------
    v4i bring[DEPTH][4][2];                          // [set][block][chunk pair]
    // Stage-load d of a tile lies in stage (ring + d) % 4 of LDS: the ring goes on from tile to tile, whatever K leaves over
    // beyond a multiple of four.  Register sets have to be named at compile time: see `turn`.
    int ring = 0;
    auto stage_at = [&](int base, int d) __attribute__((always_inline)) { return (uint32_t)__builtin_amdgcn_readfirstlane(((base + d) & 3) * STAGE_BYTES); };
    // (SGPRs are short here: the compiler keeps some in VGPR lanes, the base pointers of copies among them, and reads them back right
    // in front of a copy.  Hence kBaseSettles, and an MFMA among the wait states where copies are many: multiply_copy and `tail`.)
    auto copy = [&](int d, int c, uint32_t at) __attribute__((always_inline)) { copy16_to_lds<kBaseSettles>(a_a + d * BIG_BK, aoff[c], wave_a + at + c * 1024); };
    auto load = [&](int d, int e, auto set) __attribute__((always_inline)) {
        bring[decltype(set)::value][e >> 1][e & 1] = *reinterpret_cast<const v4i*>(bsrc[e >> 1] + ((size_t)d << 11) + (e & 1) * 1024 + lane16);
    };
    const bool bias_rides = a_bias != nullptr && (reinterpret_cast<uintptr_t>(a_bias) & 3) == 0;
    // Blocks of the constants: row scales of the tile, the weight scales of its columns (gated: gate columns, then up
    // columns), then their bias values, two to a word; past the matrix its last ones.  Every wavefront makes CONSTS copies (the
    // waits count them): with fewer blocks than that one of them again.  No bias, or one that is not a row of words: its
    // place is filled by hand.
    auto constants = [&](int c, int at_byte) __attribute__((always_inline)) {   // copy c of this wavefront
        const int ln = here(lane);
        const int w = __builtin_amdgcn_readfirstlane(c * 4 + wn);
        int blk = w < BLOCKS - 1 ? w : BLOCKS - 1;
        if (blk >= XBLOCKS + WBLOCKS && !bias_rides) blk = XBLOCKS;
        const void* base;
        uint32_t at;
        if (blk < XBLOCKS) {
            const int m = m0 + blk * 64 + ln;
            base = a_a_scale;
            at = one_scale ? 0u : (uint32_t)(m < M ? m : M - 1) * 4;
        } else {
            // column j of the tile; bias: the even one of the pair
            const bool of_bias = blk >= XBLOCKS + WBLOCKS;
            const int j = of_bias ? (blk - XBLOCKS - WBLOCKS) * 128 + 2 * ln : (blk - XBLOCKS) * 64 + ln;
            int n;
            if constexpr (GATED) {
                const int up = j >= BN / 2 ? 1 : 0;
                n = n0 + j - up * (BN / 2);
                n = (n < half_n ? n : half_n - 2) + up * half_n;
            } else {
                n = n0 + j;
                n = n < N ? n : N - 2;
            }
            base = of_bias ? static_cast<const void*>(a_bias) : a_b_scale;
            at = (uint32_t)n * (of_bias ? 2u : 4u);
        }
        const uint64_t b64 = reinterpret_cast<uint64_t>(base);   // (uniform, which the compiler does not see)
        const uint64_t b_lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b64);
        const uint64_t b_hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(b64 >> 32));
        copy4_to_lds<kBaseSettles>(reinterpret_cast<const uint8_t*>(b_lo | b_hi << 32), at, __builtin_amdgcn_readfirstlane(lds_base + at_byte + blk * 256));
    };
    auto fill_bias = [&](int at_byte) __attribute__((always_inline)) {
        if (bias_rides) return;
        const int tid = wn * 64 + here(lane);
        uint16_t v = 0;
        if (a_bias != nullptr) {
            const int up = GATED && tid >= BN / 2 ? 1 : 0, n = n0 + tid - up * (BN / 2), lim = GATED ? half_n : N;
            v = a_bias[(n < lim ? n : lim - 1) + up * half_n];
        }
        reinterpret_cast<uint16_t*>(lds + at_byte + (XBLOCKS + WBLOCKS) * 256)[tid] = v;
    };
    using S0 = std::integral_constant<int, 0>; using S1 = std::integral_constant<int, 1>;
    using S2 = std::integral_constant<int, 2>; using S3 = std::integral_constant<int, 3>;
    // Request n of a tile's opening, stage-loads 0 and 1: first what stage 0 waits for - its weights come from HBM - and the
    // activations that progress word -1 vouches for (0 .. CLAIM - 1), then the constants and the weights of stage-load 1.
    constexpr int OPENING = 2 * COPIES + CONSTS;
    auto opening = [&](auto n_, int const_at, int base) __attribute__((always_inline)) {
        constexpr int n = decltype(n_)::value;
        if constexpr (n < BL) load(0, n, S0{});
        else if constexpr (n < BL + CA) copy(0, n - BL, stage_at(base, 0));
        else if constexpr (n < BL + 2 * CA) copy(1, n - BL - CA, stage_at(base, 1));
        else if constexpr (n < BL + 2 * CA + CONSTS) constants(n - BL - 2 * CA, const_at);
        else load(1, n - BL - 2 * CA - CONSTS, S1{});
    };

    // ---- hand-over ---------------------------------------------------------------------------------
    // Word w = d says: wavefront w has issued all its LDS reads of stage-loads <= d, and its own copies of stage-loads
    // <= d + CLAIM have landed.  At its hand-over point of stage d a wavefront publishes d and goes on once every word is
    // >= d - SLACK: then stage-load d + 1 is complete in LDS (SLACK <= CLAIM - 1) and the stage that stage-load d + LEAD
    // refills has been read by everyone (it held stage-load d + LEAD - DEPTH = d - SLACK).  The slowest wavefront never waits,
    // so the scheme cannot lock up; the spin is bounded all the same (a wavefront that gave up would read a stage early:
    // wrong numbers, never a hang).  The words are read BEFORE the second half's operand reads and looked at behind its first
    // MFMAs (LDS answers in order: read at the hand-over point they would queue behind that batch); a value that old can only
    // be too small, and then they are read again.
    volatile lds_int_t* const progress = (volatile lds_int_t*)(lds + RING_END);
    auto progress_words = [&]() -> v4i { return *(const volatile lds_v4i_t*)(lds + RING_END); };
    auto hand_over = [&](int d, v4i seen) {
        if (lane == 0) progress[wave] = d;
        auto behind = [&](const v4i& w) {
            return __builtin_amdgcn_readfirstlane(min(min(w[0], w[1]), min(w[2], w[3]))) < d - SLACK;
        };
        if (__builtin_expect(behind(seen), 0)) {   // (its own block: the wait for `seen` above stays a counted one)
#pragma nounroll
            for (int spin = 0; spin < (1 << 18); ++spin) {
                __builtin_amdgcn_s_sleep(1);
                const v4i now = progress_words();
                if (!behind(now)) break;
            }
        }
    };

    // ---- sums --------------------------------------------------------------------------------------
    // In inline assembly and AGPRs, with the sum in place: left to the compiler, a sum may land in other registers than it
    // came from, which ends in copies and spills.  The s_nop covers a VALU write of an operand just before.
    v4f acc[R][4];
    // (first: the sum begins here)
    auto multiply = [&](v8i w, v8i x, v4f& c, auto first) __attribute__((always_inline)) {
        if constexpr (decltype(first)::value) asm volatile("s_nop 1\n\tv_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, 0" : "=a"(c) : "v"(w), "v"(x));
        else asm volatile("s_nop 1\n\tv_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, %0" : "+a"(c) : "v"(w), "v"(x));
    };
    using No = std::integral_constant<int, 0>; using Yes = std::integral_constant<int, 1>;
    // The same with copy(d, k, at) behind it: the MFMA and its s_nop are among the wait states between what wrote the copy's base and
    // the copy, at no cost in time (with kBaseSettles behind the MFMA instead 2441 x 13312 x 2048 + GeGLU took 65.8 us for 63.9).
    auto multiply_copy = [&](v8i w, v8i x, v4f& c, auto first, int d, int k, uint32_t at) __attribute__((always_inline)) {
        const uint8_t* const base = a_a + d * BIG_BK;
        const uint32_t from = aoff[k], to = wave_a + at + k * 1024;
        if constexpr (decltype(first)::value)
            asm volatile("s_mov_b32 m0, %5\n\ts_nop 0\n\tv_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, 0\n\ts_nop 1\n\tglobal_load_lds_dwordx4 %3, %4"
                         : "=a"(c) : "v"(w), "v"(x), "v"(from), "s"(base), "s"(to) : "memory", "m0");
        else
            asm volatile("s_mov_b32 m0, %5\n\ts_nop 0\n\tv_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, %0\n\ts_nop 1\n\tglobal_load_lds_dwordx4 %3, %4"
                         : "+a"(c) : "v"(w), "v"(x), "v"(from), "s"(base), "s"(to) : "memory", "m0");
    };
    v8i fa[2][H0];
    constexpr int AHEAD = 2;   // blocks of a half that are read during the half before it
    // Lane (l16, q) of row block b reads chunks q and 4 + q of its row: frag_lo and frag_hi beyond the stage's place and the block.
    uint32_t frag_lo = lds_base + l16 * BIG_BK + ((q ^ big_swizzle(l16)) << 4), frag_hi = lds_base + l16 * BIG_BK + (((q + 4) ^ big_swizzle(l16)) << 4);
    asm volatile("" : "+v"(frag_lo), "+v"(frag_hi));
    auto frag = [&](uint32_t lo, uint32_t hi, int b) __attribute__((always_inline)) {
        return big_join(*(const lds_v4i_t*)(lo + b * (16 * BIG_BK)), *(const lds_v4i_t*)(hi + b * (16 * BIG_BK)));
    };
    // Half P of stage-load d (register set S): row blocks P * H0 .. of it against all four weight blocks.  The blocks that open a
    // half are read during the half before it, the others behind the first MFMAs' issue; the hand-over comes behind the first
    // row block of half 1.  Requests go out between the MFMAs, spread over both halves - four wavefronts that send theirs in one
    // half keep each other waiting for the CU's address unit: the weights of stage-load d + 2 in half 0, behind the hand-over of
    // half 1 the activation copies of stage-load d + LEAD.
    // next: stage-load d + 1 follows in the main loop; ask: 1 as said, 2 (half 0 of a tile's first stage-load) copies and weights
    // both, 0 nothing; first: that stage-load; beside(n): other work behind MFMA n.
    auto half = [&](int d, auto set, auto p_, auto next, auto ask, auto first, auto beside) __attribute__((always_inline)) {
        constexpr int S = decltype(set)::value, P = decltype(p_)::value, HP = P ? H1 : H0, ASK = decltype(ask)::value;
        constexpr bool NEXT = decltype(next)::value;
        constexpr int OPEN_NEXT = HP - AHEAD < 3 ? HP - AHEAD : 3;
        const uint32_t here_at = stage_at(ring, d), next_at = P ? stage_at(ring, d + 1) : here_at;   // ... whose block opens the next half
        const uint32_t lo = frag_lo + here_at, hi = frag_hi + here_at, next_lo = P ? frag_lo + next_at : lo, next_hi = P ? frag_hi + next_at : hi;
        const uint32_t copies_at = stage_at(ring, d + 2 + P);
        v4i seen = {0, 0, 0, 0};
        if constexpr (P == 1 && NEXT) seen = progress_words();
#pragma unroll
        for (int i = 0; i < HP; ++i) {
            if (i == 0) {
#pragma unroll
                for (int b = AHEAD; b < HP; ++b) fa[P][b] = frag(lo, hi, P * H0 + b);
            }
            if (i >= OPEN_NEXT && i < OPEN_NEXT + AHEAD && (P == 0 || NEXT)) fa[1 - P][i - OPEN_NEXT] = frag(next_lo, next_hi, (1 - P) * H0 + i - OPEN_NEXT);
#pragma unroll
            for (int jj = 0; jj < 4; ++jj) {
                const int slot_n = P ? (i - 1) * 4 + jj : i * 4 + jj;
                constexpr int REQUESTS = P ? CA : BL, MFMAS = P ? SLOTS_AFTER : 4 * H0;
                const int n = ASK == 2 ? slot_n : slot_n * REQUESTS / MFMAS;   // the request behind this MFMA, if there is one
                const bool asks = ASK == 2 ? n < COPIES : ASK == 1 && (slot_n == 0 || (slot_n > 0 && n != (slot_n - 1) * REQUESTS / MFMAS));
                const bool copies = asks && (ASK == 2 ? n < CA : P == 1);
                const v8i weights = big_join(bring[S][jj][0], bring[S][jj][1]);
                if (copies) multiply_copy(weights, fa[P][i], acc[P * H0 + i][jj], first, ASK == 2 ? d + 2 : d + LEAD, n, copies_at);
                else multiply(weights, fa[P][i], acc[P * H0 + i][jj], first);
                if (asks && !copies) load(d + 2, ASK == 2 ? n - CA : n, std::integral_constant<int, (S + 2) % DEPTH>{});
                beside(i * 4 + jj);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (P == 1 && i == 0 && NEXT) {
                wait_copies<BL>();   // my activation copies of d + CLAIM have landed; its weights may be in flight
                hand_over(d, seen);
                asm volatile("" ::: "memory");
            }
        }
    };
    static_assert(COPIES <= 4 * H0, "the first stage-load's first half asks for stage-load 2");
    static_assert(CA <= SLOTS_AFTER && BL <= 4 * H0, "one request behind an MFMA");
    using Two = std::integral_constant<int, 2>;
    auto nothing = [](int) __attribute__((always_inline)) {};
    auto stage = [&](int d, auto set) __attribute__((always_inline)) {
        half(d, set, No{}, Yes{}, Yes{}, No{}, nothing);
        half(d, set, Yes{}, Yes{}, Yes{}, No{}, nothing);
    };
    // The loop over stage-loads names sets 0 .. 3 in turn and ends with sets 2 and 3.  Up to three stage-loads beyond a multiple of
    // four come before it, each in set 1, the two behind it moving up.  (The move waits for weights that were asked for half a stage
    // ago.  K = 128, 256, 384 mod 512 are 1.09, 1.09, 1.08 times as fast as staged tiles all the same, the rest 1.10, in 325 linears.)
    auto turn = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            bring[1][e >> 1][e & 1] = bring[2][e >> 1][e & 1];
            bring[2][e >> 1][e & 1] = bring[3][e >> 1][e & 1];
        }
    };

    // ---- the last two stage-loads and the epilogue -------------------------------------------------
    // Row block by row block: the eight MFMAs that end block r's sums between the pieces of block r - 1's epilogue, which is
    // several times as much VALU work.  (One wavefront per SIMD: nothing else would multiply meanwhile.)  Two stages of the ring and
    // two register sets are free by now: the next tile's opening goes out in between, a request behind each piece
    // (asked for all at once, by all CUs, it would hold up the wavefront for 6 k cycles).
    // The weight block is the MFMA's first operand: register e of lane (l16, q) of block (r, jj) is token row 16 r + l16, column
    // 16 jj + 4 q + e of the wavefront (gated operand order: registers 0, 1 are gate and 2, 3 up of output columns 8 jj + 2 q,
    // + 1).  A finished row block passes through the wavefront's own two slots of LDS (16-byte slots XOR-swizzled with the row)
    // and leaves row-wise, 16 bytes per lane, two blocks later.  Output is written once and never read here: non-temporal.
    auto tail = [&](const int em0, const int en0, const int const_at, const int next_const_at, const int next_ring, const bool more) __attribute__((always_inline)) {
        const int lane = here(threadIdx.x & 63), l16 = lane & 15, q = lane >> 4;
        const float* const const_x = reinterpret_cast<const float*>(lds + const_at);
        const float* const const_w = const_x + XBLOCKS * 64;
        const uint16_t* const const_bias = reinterpret_cast<const uint16_t*>(const_w + BN);
        uint8_t* const stg = lds + STAGING_AT + wn * (2 * 16 * ROWB);
        const int n_lim = GATED ? half_n : N, nbase = en0 + wn * (GATED ? WN / 2 : WN);
        // [block][register]; beside a residual's rows there is room for the bias as it lies only, two values to a word, and for the
        // scales of one block and the next
        float sc[RES ? 1 : 4][4], bi[RES ? 1 : 4][4];
        uint2 bi_packed[RES ? 4 : 1];
        v4f sc_now, sc_next;
        if constexpr (RES) sc_next = *reinterpret_cast<const v4f*>(const_w + wn * WN + 4 * q);
#pragma unroll
        for (int jj = 0; jj < 4; ++jj)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int c = GATED ? wn * 32 + 8 * jj + 2 * q + (e & 1) + (e >> 1) * (BN / 2) : wn * WN + 16 * jj + 4 * q + e;
                if constexpr (!RES) {
                    sc[jj][e] = const_w[c];
                    bi[jj][e] = bf16_bits_to_f32(const_bias[c]);
                } else if (e == 0) {
                    bi_packed[jj] = *reinterpret_cast<const uint2*>(const_bias + c);
                }
            }
        const int sw = (l16 / ROWS_PER_PASS) & (SLOTS - 1);
        const uint32_t at0 = stage_at(ring, n_loads - 2), at1 = stage_at(ring, n_loads - 1);
        const uint32_t lo0 = frag_lo + at0, hi0 = frag_hi + at0, lo1 = frag_lo + at1, hi1 = frag_hi + at1;
        v8i f0 = frag(lo0, hi0, 0), f1 = frag(lo1, hi1, 0);
        float s_next = const_x[l16];
        // Where lane's 16 bytes of a row block go.  Through a buffer resource that ends with the matrix's last row, so that rows
        // past it are not written (nor the residual's read); lanes of columns past the matrix stay beyond the resource.  (A
        // compare, a mask and a branch per store otherwise, and 64-bit addresses.)
        const int rows_here = M - em0 < BM ? M - em0 : BM;
        const auto out_rsrc = __builtin_amdgcn_make_buffer_rsrc(a_out + em0 * a_ldo, 0, rows_here * (int)a_ldo * 2, 0x00020000);
        // (the second kilobyte of a block, where it has one, is 8 rows further)
        const int leaf_row = lane * 16 / ROWB, leaf_n = nbase + lane * 16 % ROWB / 2;
        uint32_t leaves_to = leaf_n < n_lim ? (uint32_t)(leaf_row * (int)a_ldo + leaf_n) * 2 : kNowhere;
        // residual and gate the same way; a gate row for every `group` token rows, the first of them that this tile needs is first_gate
        const int ld_res = (int)a_res.ld_res, ld_gate = (int)a_res.ld_gate, group = a_res.gate_group;
        const int first_gate = RES && group < M ? big_div(em0, group) : 0;
        const auto res_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(RES ? a_res.residual + (int64_t)em0 * ld_res : nullptr), 0, RES ? rows_here * ld_res * 2 : 0, 0x00020000);
        const auto gate_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(RES ? a_res.gate + (int64_t)first_gate * ld_gate : nullptr), 0, RES ? 0x7FFFFFFF : 0, 0x00020000);
        uint32_t res_from = RES && leaf_n < n_lim ? (uint32_t)(leaf_row * ld_res + leaf_n) * 2 : kNowhere;
        const float one_by_group = RES ? __builtin_amdgcn_rcpf((float)group) : 0.f;
        v4i staged[LEAVES];
        v4u rs[LEAVES], gt[LEAVES];
        float s = 0.f;
        uint32_t g01 = 0, u01 = 0;
        tall_each<8 * (R + 3)>([&](auto piece_) __attribute__((always_inline)) {
                constexpr int piece = decltype(piece_)::value, r = piece / 8, e = piece % 8;
                if constexpr (e == 0 && r >= 1 && r <= R) s = s_next;
                // The request behind this piece (evenly over the pieces beside MFMAs).  If a copy's base has to be read back it is here:
                // the MFMA and its s_nop are wait states enough.  (kBaseSettles, three more each time, beside work that is VALU bound:
                // two projections of 13056 rows 1148 us, 1145 so, 1143 with none at all)
                constexpr int n = piece * OPENING / (8 * R);
                constexpr bool asks = r < R && (piece == 0 || n != (piece - 1) * OPENING / (8 * R)), copies = asks && n >= BL && n < BL + 2 * CA;
                constexpr int of_load = n < BL + CA ? 0 : 1;
                const uint8_t* base = a_a + of_load * BIG_BK;
                if constexpr (copies) asm volatile("" : "+s"(base));
                if constexpr (r < R) {
                    multiply(big_join(bring[2 + (e >> 2)][e & 3][0], bring[2 + (e >> 2)][e & 3][1]), e < 4 ? f0 : f1, acc[r][e & 3], No{});
                    if constexpr (e == 3 && r + 1 < R) f0 = frag(lo0, hi0, r + 1);
                    if constexpr (e == 7 && r + 1 < R) f1 = frag(lo1, hi1, r + 1);
                }
                if constexpr (e == 0 && r >= 3) {   // block r - 3 leaves
#pragma unroll
                    for (int i = 0; i < LEAVES; ++i) {
                        v4i v = staged[i];
                        if constexpr (RES) {   // out = residual + bf16(linear) * gate
#pragma unroll
                            for (int w = 0; w < 4; ++w) v[w] = (int)addcmul2((uint32_t)v[w], rs[i][w], gt[i][w]);
                        }
                        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, v), out_rsrc, (int)leaves_to + i * 16 * (int)a_ldo, 0, 2);   // (2: nt)
                    }
                    leaves_to += 32u * (uint32_t)a_ldo;
                }
                if constexpr (e == 2 && r + 1 <= R && r >= 1) s_next = const_x[16 * r + l16];
                if constexpr (e == 1 && r >= 2 && r < R + 2) {   // block r - 2 out of LDS
#pragma unroll
                    for (int i = 0; i < LEAVES; ++i) {
                        const int byte = i * 1024 + lane * 16, row = byte / ROWB, slot = (byte % ROWB) / 16;
                        staged[i] = *reinterpret_cast<const v4i*>(stg + (r & 1) * (16 * ROWB) + row * ROWB + ((slot ^ ((row / ROWS_PER_PASS) & (SLOTS - 1))) << 4));
                        if constexpr (RES) {
                            rs[i] = __builtin_amdgcn_raw_buffer_load_b128(res_rsrc, (int)res_from + i * 16 * ld_res, 0, 0);
                            if (i == LEAVES - 1) res_from += 32u * (uint32_t)ld_res;
                            uint32_t gate_at = 0;
                            if (group < M) {   // (uniform) the token row's quotient by the group, of values below 2^24
                                const int m = em0 + (r - 2) * 16 + row < M ? em0 + (r - 2) * 16 + row : M - 1;
                                int g = (int)((float)m * one_by_group);
                                g += m - g * group >= group ? 1 : 0;
                                g -= m - g * group < 0 ? 1 : 0;
                                gate_at = (uint32_t)((g - first_gate) * ld_gate) * 2;
                            }
                            gt[i] = __builtin_amdgcn_raw_buffer_load_b128(gate_rsrc, (int)(leaf_n < n_lim ? gate_at + 2 * leaf_n : kNowhere), 0, 0);
                        }
                    }
                }
                if constexpr (r >= 1 && r <= R) {
                    const int jj = e >> 1;
                    uint8_t* const at = stg + ((r - 1) & 1) * (16 * ROWB) + l16 * ROWB;
                    if constexpr ((e & 1) == 0) {
                        // (the sums' MFMAs are three and more MFMAs back; no read of them moves in front of this)
                        v4f& sum = acc[r - 1][jj];
                        float o[4];
                        asm volatile("" : "+a"(sum));
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            float b, w_scale;
                            if constexpr (RES) {
                                if (i == 0) sc_now = sc_next;
                                w_scale = sc_now[i];
                                const uint32_t two = i < 2 ? bi_packed[jj].x : bi_packed[jj].y;
                                b = __uint_as_float(i & 1 ? two & 0xFFFF0000u : two << 16);
                            } else {
                                b = bi[jj][i];
                                w_scale = sc[jj][i];
                            }
                            o[i] = __builtin_fmaf(sum[i], s * w_scale, b);
                        }
                        if constexpr (RES) sc_next = *reinterpret_cast<const v4f*>(const_w + wn * WN + 16 * ((jj + 1) & 3) + 4 * q);
                        // an activation's input passes through bf16 first, as the two-launch form materialises it
                        g01 = pack_bf16x2(o[0], o[1]);
                        u01 = pack_bf16x2(o[2], o[3]);
                    } else if constexpr (GATED) {
                        const float o0 = apply_act<EPI>(__uint_as_float(g01 << 16)) * __uint_as_float(u01 << 16);
                        const float o1 = apply_act<EPI>(__uint_as_float(g01 & 0xFFFF0000u)) * __uint_as_float(u01 & 0xFFFF0000u);
                        *reinterpret_cast<uint32_t*>(at + (jj ^ sw) * 16 + 4 * q) = pack_bf16x2(o0, o1);
                    } else {
                        uint2 w;
                        w.x = g01; w.y = u01;
                        if constexpr (EPI != EPI_NONE) {
                            w.x = pack_bf16x2(apply_act<EPI>(__uint_as_float(g01 << 16)), apply_act<EPI>(__uint_as_float(g01 & 0xFFFF0000u)));
                            w.y = pack_bf16x2(apply_act<EPI>(__uint_as_float(u01 << 16)), apply_act<EPI>(__uint_as_float(u01 & 0xFFFF0000u)));
                        }
                        *reinterpret_cast<uint2*>(at + ((2 * jj + (q >> 1)) ^ sw) * 16 + (q & 1) * 8) = w;
                    }
                }
                if constexpr (copies) {
                    constexpr int c = n - BL - of_load * CA;
                    if (more) copy16_to_lds(base, aoff[c], wave_a + stage_at(next_ring, of_load) + c * 1024);
                } else if constexpr (asks) {
                    if (more) opening(std::integral_constant<int, n>{}, next_const_at, next_ring);
                }
                __builtin_amdgcn_sched_barrier(0);
        });
    };
    static_assert(OPENING <= 8 * R, "the opening goes out beside the MFMAs");
    if (!next_tile()) return;
#pragma unroll
    for (int step = 0; step <= CA; ++step) take_tile(step);
    int parity = 0;
    tall_each<OPENING>([&](auto n) __attribute__((always_inline)) { opening(n, CONST_AT, 0); });
    fill_bias(CONST_AT);
#pragma unroll
    for (int c = 0; c < CA; ++c) copy(2, c, stage_at(0, 2));
#pragma unroll
    for (int e = 0; e < BL; ++e) load(2, e, S2{});
    for (bool first = true;; first = false) {
        // Stage-load 0 and the activations up to stage-load CLAIM - 1 have landed (what progress word -1 stands for; the
        // stores of the tile before, younger than all of these, only make the wait stricter).  The first tile's stage-load 2
        // has been asked for; a later one's, whose place was still in use, is asked for beside the first MFMAs.  (The two ways
        // meet in one set of registers, for which the compiler waits: a first tile for those weights before its first MFMA,
        // a later one for most of them before half 1.)
        if (first) wait_copies<COPIES + BL + CONSTS>();
        else wait_copies<BL + CONSTS>();
        if (lane == 0) progress[wave] = -1;
        __syncthreads();
        PHYAI_STAMP(1)
#pragma unroll
        for (int b = 0; b < AHEAD; ++b) fa[0][b] = frag(frag_lo + stage_at(ring, 0), frag_hi + stage_at(ring, 0), b);
        if (first) half(0, S0{}, No{}, Yes{}, No{}, Yes{}, nothing);
        else half(0, S0{}, No{}, Yes{}, Two{}, Yes{}, nothing);
        const bool more = next_tile();   // (behind MFMAs that are still to run)
        half(0, S0{}, Yes{}, Yes{}, Yes{}, Yes{}, nothing);
        int d = 0;
        for (; d < (n_loads & (DEPTH - 1)); ++d) {
            stage(d + 1, S1{});
            turn();
        }
        if (d < n_loads - DEPTH) {
            stage(d + 1, S1{});
            stage(d + 2, S2{});
            stage(d + 3, S3{});
            for (d += DEPTH; d < n_loads - DEPTH; d += DEPTH) {
                stage(d, S0{});
                stage(d + 1, S1{});
                stage(d + 2, S2{});
                stage(d + 3, S3{});
            }
            stage(d, S0{});
        }
        half(d + 1, S1{}, No{}, Yes{}, Yes{}, No{}, nothing);
        const int em0 = m0, en0 = n0, const_at = CONST_AT + parity * CONST_BYTES;
        half(d + 1, S1{}, Yes{}, No{}, No{}, No{}, take_tile);   // (nothing asks for this tile's places any more)
        PHYAI_STAMP(2)
        wait_copies<BL>();
        __syncthreads();   // the activations of the last two stage-loads and all constants have landed, everyone is done with those before
        parity ^= 1;
        const int next_const_at = CONST_AT + parity * CONST_BYTES;
        PHYAI_STAMP(3)
        const int next_ring = (ring + n_loads) & 3;
        tail(em0, en0, const_at, next_const_at, next_ring, more);
        ring = next_ring;
        PHYAI_STAMP(4)
        if (!more) break;
        fill_bias(next_const_at);
    }
    PHYAI_STAMP_END(g_tall_stamps, (size_t)blockIdx.x * 4 + wave, lane)
}

// ---- host side -------------------------------------------------------------------------------------

template <int R, int EPI, bool RES = false>
static void tall_launch(const GemmProblem& g, hipStream_t st) {
    constexpr bool gated = epi_is_gated(EPI);
    constexpr int BM = 16 * R, BN = gated ? TALL_COLS / 2 : TALL_COLS;
    const int n_tiles = big_ceil_div(gated ? g.N / 2 : g.N, BN), m_tiles = big_ceil_div(g.M, BM);
    double bytes;
    int busiest;
    int by_rows = big_takes_rows(g.M, g.N, g.K, m_tiles, n_tiles, 32, &bytes, &busiest);
    if (const char* e = tuning_env("PHYAI_FP8_BY_ROWS")) by_rows = atoi(e) != 0;
    const int band = big_band(by_rows, m_tiles, BM, g.K);
    const int busiest_of_order = by_rows ? big_max_tiles_per_xcd(n_tiles, m_tiles, band) : big_max_tiles_per_xcd(m_tiles, n_tiles, band);
    hipLaunchKernelGGL((gemm_fp8_tall_kernel<R, EPI, RES>), dim3(8 * busiest_of_order < TALL_GRID ? 8 * busiest_of_order : TALL_GRID), dim3(256), 0, st, g.xq, g.w, g.K, g.M, g.N, m_tiles,
                       big_order(band, by_rows, 1, g.x_scale_is_scalar, 0), g.x_scale, g.w_scale, g.bias, g.out, g.ldo, residual_of(g));
}

template <int R>
static int tall_launch_epi(const GemmProblem& g, hipStream_t st) {
    switch (g.epilogue) {
    case EPI_NONE:
        if (g.residual != nullptr) tall_launch<R, EPI_NONE, true>(g, st);
        else tall_launch<R, EPI_NONE>(g, st);
        return 0;
    case EPI_GEGLU_TANH: tall_launch<R, EPI_GEGLU_TANH>(g, st); return 0;
    case EPI_GEGLU_ERF: tall_launch<R, EPI_GEGLU_ERF>(g, st); return 0;
    case EPI_SWIGLU: tall_launch<R, EPI_SWIGLU>(g, st); return 0;
    case EPI_GELU_TANH: tall_launch<R, EPI_GELU_TANH>(g, st); return 0;
    case EPI_GELU_ERF: tall_launch<R, EPI_GELU_ERF>(g, st); return 0;
    default: return -2;
    }
}

// The epilogue's offsets from a tile's first row are 32-bit, and below 2^30.
bool tall_reaches(const GemmProblem& g) {
    constexpr int64_t far = 1 << 21;
    return g.ldo < far && (g.residual == nullptr || (g.ld_res < far && g.ld_gate < far));
}

int launch_gemm_tall(const GemmProblem& g, int rows, hipStream_t st) {
    if (g.weight_layout == W_ROW_MAJOR || g.K % BIG_BK != 0 || g.K < 4 * BIG_BK) return -2;
    if (g.ldo % 8 != 0 || (reinterpret_cast<uintptr_t>(g.out) & 15) != 0 || !tall_reaches(g)) return -2;   // (16 bytes per lane leave)
    switch (rows) {
    case 144: return tall_launch_epi<9>(g, st);
    case 160: return tall_launch_epi<10>(g, st);
    case 176: return tall_launch_epi<11>(g, st);
    case 192: return tall_launch_epi<12>(g, st);
    case 208: return tall_launch_epi<13>(g, st);
    case 224: return tall_launch_epi<14>(g, st);
    case 240: return tall_launch_epi<15>(g, st);
    case 256: return tall_launch_epi<16>(g, st);
    default: return -2;
    }
}

int launch_set_stamp_sink_tall(unsigned long long* buf, unsigned int records) {
#ifdef PHYAI_FP8_STAMPS
    const StampSink s = {buf, records};
    return hipMemcpyToSymbol(HIP_SYMBOL(g_tall_stamps), &s, sizeof(s)) == hipSuccess ? 0 : -4;
#else
    (void)buf; (void)records;
    return -2;
#endif
}

}  // namespace phyai
