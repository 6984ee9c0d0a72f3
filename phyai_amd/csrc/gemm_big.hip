// MFMA-bound fp8 GEMM for large M (prefix prefill, batched serving).
// Workgroup = 4 wavefronts, 2 x 2 or 1 x 4; a wavefront owns TM x TN blocks of 32 x 32 outputs: 256 x 256 (4 x 4
// blocks, one workgroup per CU) and 224 x 256 (7 x 2, wavefronts 1 x 4) for long K or many tiles, 192 x 128 (3 x 2, two
// workgroups per CU) when there are plenty of tiles and K is short, 128 x 128 (2 x 2, or 4 x 1 with wavefronts 1 x 4;
// ring of four stages, or of two with two workgroups per CU) for mid-sized problems, 96 x 128 (3 x 1, wavefronts 1 x 4)
// and 128 x 64 (2 x 1) when even those leave CUs idle.
//
// A 32 x 32 block is four v_mfma_f32_16x16x128_f8f6f4, 32 cycles each.  The chip runs these kernels at its power limit
// (13056 x 32768 x 2048 + GeGLU 581 us on zeros, 745 on real data; 816 x 32768 x 2048 49 / 58), and this MFMA takes less
// energy per product than the 32 x 32 x 64 one at the same rate: held in registers, on random codes, 4.5 against 4.1
// PFLOP/s (both 5.0 on zeros); 4800 x 6144 x 2048 60.0 -> 58.2 us, 3264 x 32768 x 2048 + GeGLU 203 -> 197.
//
// Why 4 x 4 blocks per wavefront for the large tile.  A wavefront with TM x TN blocks reads (TM + TN) operand blocks of
// 4 KB (32 rows x 128 bytes of K) from LDS per 4 TM TN MFMAs; LDS delivers 128 bytes per clock to the whole CU, so four
// wavefronts with 4 x 4 blocks ask for 64 bytes per clock, 2 x 2 blocks for 128.  The same ratio governs the bytes that
// must come from L2: (BM + BN) * K per tile, and L2 -> CU delivery (measured: 10-13 TB/s over all CUs inside these
// kernels) bounds the small tiles.  4 x 4 blocks of 16 accumulators are 256 registers: they live in AGPRs, one wavefront
// per SIMD, and latency is hidden inside the wavefront:
//
//  * global -> LDS copies bypass the register file (global_load_lds_dwordx4): lane i of a
//    wavefront fetches one 16-byte chunk and the hardware deposits chunk i at LDS base + 16*i.
//    An LDS row is 128 bytes of K - one L2 line per row per request; the XOR swizzle that keeps
//    the 128-bit operand reads conflict-free is therefore applied on the global side: lane i
//    (row i/8 of an 8-row group, slot i%8 of the row) fetches chunk (i%8) ^ swizzle(row).
//  * K is consumed in 128-byte stage-loads - one K step of the MFMA - through a ring of DEPTH LDS stages: the copies of
//    load d + DEPTH are requested while loads d and d + 1 are being multiplied, one copy instruction per MFMA, so the
//    wavefront never waits on the memory pipeline's issue queue with its MFMA pipe empty.
//  * a stage-load is multiplied in two halves, each with one 16-row half of the activation blocks and all of the
//    weights.  Staged weights are read once per stage-load, block by block into the registers that their predecessor's
//    last MFMA has just left; the activation blocks of a half are read during the half before it, so ds_read latency
//    overlaps MFMA time.  Sums stay in place through inline assembly (`multiply`).
//  * one barrier per stage-load, in its second half behind the first group of MFMAs: it publishes the next stage and
//    tells everyone that the stage about to be refilled is no longer read.  All wavefronts reach it at about the same
//    time, with MFMAs queued.  Where the weights are in MFMA operand order and a wavefront owns its column blocks
//    (128 x 128 tiles as 4 x 1 blocks per wavefront; 144 .. 256 x 256 in gemm_tall.hip) they do not go through
//    LDS at all - each wavefront loads its own weight blocks straight into a ring of register sets - and the barrier
//    gives way to a hand-over through one progress word per wavefront in LDS, which lets a wavefront run a stage or two
//    ahead of the slowest (see `hand_over` in the kernel).
//  * epilogue: the weight block is the MFMA's first operand, which gives a lane runs of four
//    consecutive output columns of one token row; each wavefront stages its bf16 tile in its own
//    slice of the (now idle) LDS and writes it out row-wise, 16 bytes per lane, whole row
//    segments per instruction.  It is straight-line arithmetic on LDS and registers: scales and bias are in LDS since
//    the prologue, the gated residual is added where the tile leaves row by row, and the sums of the tiles up to 128 x 128
//    are in VGPRs, which the arithmetic can read where they are.  A 128 x 64 tile's took 1.9 k cycles while each group of four columns
//    looked for a residual, and waited for its constants from memory; 0.8 k now, and its main loop 8.9 k instead of 9.4 k
//    (us: 816 x 2048 x 2048 7.7 -> 7.4, 816 x 2560 x 2048 9.9 -> 9.4, 777 x 4304 x 1168 + GELU 12.0 -> 11.1,
//    400 x 8192 x 1024 + GeGLU 8.2 -> 8.0, 1632 x 2048 x 2048 11.1 -> 10.0, 4800 x 6144 x 2048 59.3 -> 57.9; 816 x 32768 x 2048 level).
//
// The smaller tiles (192 x 128, and 128 x 128 with a ring of two) keep within the register and
// LDS budget of two workgroups per CU, so that one workgroup's prologue and epilogue run under
// the other's MFMAs.
//
// Gated epilogues: within a wavefront's 32*TN columns the first half are gate columns and the
// second half the matching up columns, so the pair sits in the same lane of two accumulators.
// Requires K >= 512 per split (the stage-loads must fill the ring).  K that is not a multiple of 128 (RAGGED
// instantiations, weights staged row-major): the last stage-load is partial, its missing chunks arrive as zeros
// (copy16_to_lds_checked), one extra VALU instruction per copy and nothing in the MFMA loop.  Such widths used to go
// to the generic tile kernel: the MLP 1168 -> 4304 -> 1168 at M = 777 took 43 + 37 us of GEMM there, 85 us in all;
// 31 us in all now (its second projection by the weight-streaming kernel, both on codes in padded rows).
#include "gemm_big.h"
#include "splitk.h"
#include "stamps.h"
#include "weight_layout.h"
#include <math.h>
#include <stdlib.h>
#include <type_traits>

namespace phyai {

// (debug build only: where the kernels below leave their time stamps - 1 first stage published, 2 main loop done,
// 3 split-K sums gathered, 4 epilogue arithmetic done and tile staged, 5 stores issued)
PHYAI_STAMP_SINK(g_big_stamps)

struct BigArgs {
    const uint8_t* __restrict__ a;   // xq [M, K]
    const uint8_t* __restrict__ b;   // w  [N, K]
    const float* __restrict__ a_scale;
    const float* __restrict__ b_scale;
    const uint16_t* __restrict__ bias;
    uint16_t* __restrict__ out;
    int64_t ldo;
    int M, N, K;
    int a_scale_scalar;
    // split-K (grid.z > 1): each split covers k_per_split bytes of K; see splitk.h
    int k_per_split;
    float* __restrict__ partials;
    int* __restrict__ counters;
    int m_tiles, n_tiles;            // tile grid; the launch is 1-D over it (see big_tile_of)
    int band;                        // tile rows per band of that order
    int by_rows;                     // the order with the roles of tile rows and columns exchanged
    int operand_w;                   // weights in MFMA operand order (weight_layout.h)
    ResidualArgs res;
};

// The same block out of weights staged in operand order (WMODE 1): chunk c of row r of a unit lies at c * 256 + r * 16, so
// the lanes read 1 KB in a row, twice.
__device__ __forceinline__ v8i big_frag_operand(const uint8_t* buf, int row, int q) {
    const uint8_t* r = buf + (row >> 4) * 2048 + (row & 15) * 16 + q * 256;
    return big_join(*reinterpret_cast<const v4i*>(r), *reinterpret_cast<const v4i*>(r + 1024));
}

// Variants held to the register and LDS budget of two workgroups per CU (two wavefronts per SIMD).
__host__ __device__ constexpr bool big_two_per_cu(int tm, int tn, int depth, int wmode) {
    // (... and the 128 x 128 tile as 4 x 1 blocks per wavefront with weights in registers and a ring of four: 64 KB of
    // LDS, 64 accumulators)
    return (depth == 2 && tm < 4) || (wmode == 2 && tm == 4 && tn == 1 && depth == 4);
}

// The epilogue's constants ride with the first stage-load, except in 192 x 128 tiles, two of which fill the LDS to the last
// byte.  Asked for in the epilogue they were a trip to memory that nothing overlapped.
__host__ __device__ constexpr bool big_constants_ride(int tm, int tn) { return !(tm == 3 && tn == 2); }

// DEPTH: stages of the LDS ring, each holding BIG_BK bytes of K for the whole tile.
// Variants whose ring leaves room for two workgroups per CU are held to the register budget of
// two wavefronts per SIMD: while one workgroup is in its prologue or epilogue the other one
// keeps the MFMA pipe busy.
//
// WGM x WGN: how the four wavefronts tile the workgroup's output (2 x 2, or 1 x 4 for the
// 224 x 256 tile: every wavefront then walks all the tile's token rows and a quarter of its columns).
//
// WMODE: how the weights are laid out and reach the MFMA.  0: row-major [N, K] (or operand order, gathered
// row by row into the same LDS layout: the slow way, kept for shapes without a dedicated variant), staged
// through LDS in 128-byte rows.  1: MFMA operand order (weight_layout.h), staged through LDS as they lie:
// a copy instruction moves 1 KB in a row, and lane (l16, q) finds chunk c of its row at
// unit * 2 KB + c * 256 + l16 * 16.  2: operand order and WGM == 1, so that a wavefront's weight
// blocks are its own: they go global -> registers, DEPTH stage-loads ahead through a ring of register
// sets, and LDS carries the activations only.
template <int TM, int TN, int DEPTH, int EPI, bool SPLIT, int WGM = 2, int WGN = 2, int WMODE = 0, bool RAGGED = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(big_two_per_cu(TM, TN, DEPTH, WMODE) ? 2 : 1)))
void gemm_fp8_big_kernel(
    const uint8_t* __restrict__ a_a, const uint8_t* __restrict__ a_b, int a_K, int a_M, int a_N, int a_m_tiles, int a_order,
    int a_k_per_split, const float* __restrict__ a_a_scale, const float* __restrict__ a_b_scale,
    const uint16_t* __restrict__ a_bias, uint16_t* __restrict__ a_out, int64_t a_ldo, float* __restrict__ a_partials,
    int* __restrict__ a_counters, const ResidualArgs a_res) {
    // scalar arguments, what the prologue needs first (the first 16 dwords, up to a_bias, are preloaded into SGPRs)
    BigArgs p;
    p.a = a_a; p.b = a_b; p.a_scale = a_a_scale; p.b_scale = a_b_scale; p.bias = a_bias; p.out = a_out;
    p.ldo = a_ldo; p.M = a_M; p.N = a_N; p.K = a_K;
    p.k_per_split = a_k_per_split; p.partials = a_partials; p.counters = a_counters; p.m_tiles = a_m_tiles; p.res = a_res;
    // a_order: see big_order
    p.band = a_order & 255; p.by_rows = (a_order >> 8) & 3;
    p.operand_w = __builtin_amdgcn_readfirstlane((a_order >> 10) & 1);
    p.a_scale_scalar = (a_order >> 11) & 1;
    {
        constexpr int bn_eff = (epi_is_gated(EPI) ? 16 : 32) * TN * WGN;
        p.n_tiles = ((epi_is_gated(EPI) ? p.N / 2 : p.N) + bn_eff - 1) / bn_eff;
    }
    PHYAI_STAMP_BEGIN
    constexpr bool GATED = epi_is_gated(EPI);
    constexpr bool OPW = WMODE != 0, BDIRECT = WMODE == 2;
    static_assert(WGM * WGN == 4, "four wavefronts per workgroup");
    static_assert(!RAGGED || WMODE == 0, "operand order exists for whole K steps only");
    static_assert(!BDIRECT || (WGM == 1 && TM == 4 && TN == 1 && (DEPTH == 4 || DEPTH == 8)), "weights go straight to registers only where a wavefront owns them");
    constexpr int BM = WGM * 32 * TM, BN = WGN * 32 * TN;   // workgroup tile
    constexpr int WM = 32 * TM, WN = 32 * TN;        // wavefront tile
    constexpr int STAGE_BYTES = (BM + (BDIRECT ? 0 : BN)) * BIG_BK;  // one stage: A rows, then B rows (if staged)
    constexpr int CA = BM / 32, CB = BDIRECT ? 0 : BN / 32;   // copy instructions (8 rows each) per wavefront per stage
    constexpr int BL = BDIRECT ? TN * 4 : 0;         // 16-byte weight loads per lane per stage: TN blocks x 2 K halves x 2
    constexpr int COPIES = CA + CB + BL;             // vector-memory instructions per wavefront per stage-load
    constexpr int SLOTS_PER_STAGE = 4 * TM * TN;     // MFMAs of a wavefront per stage
    constexpr int SLOTS_AFTER = BDIRECT ? 2 * TM * TN : (2 * TN - 1) * TM;   // ... behind its barrier / hand-over
    // Requests of a stage-load are numbered; request n goes out behind MFMA n / CPS counted from the barrier of
    // the stage that frees its target: CPS per MFMA.
    // LEAD: the barrier of stage d frees the target of stage-load d + LEAD.  Staged operands: LEAD = DEPTH - the
    // barrier waits for this wavefront's LDS reads of stage d, whose stage is then refilled.  Weights in registers:
    // LEAD = DEPTH - 1 - the targets (LDS stage and register set of stage d - 1) were last read by MFMAs that
    // every wavefront has issued before it reaches the barrier of stage d, so the barrier need not wait for the
    // LDS reads in flight (the activation blocks of the second K half, requested just before it), and no register
    // set is written while MFMAs of its stage are still to come.
    // Weights in registers, ring of eight (one column block per wavefront, stages of 8 MFMAs or fewer): LEAD = 6, so
    // that a wavefront may run two stages ahead of the slowest (see the hand-over below) with its weight loads six
    // stages and its activation copies three stages old when they are needed.
    constexpr int CPS = BDIRECT ? (COPIES + SLOTS_AFTER - 1) / SLOTS_AFTER : 1;
    constexpr int LEAD = BDIRECT ? (DEPTH == 8 ? 6 : DEPTH - 1) : DEPTH;
    // (weights in registers) progress word d of a wavefront vouches for its activation copies up to stage-load
    // d + CLAIM; SLACK: how many stages a wavefront may be ahead of the slowest one
    constexpr int CLAIM = DEPTH == 8 ? 3 : 2;
    constexpr int SLACK = CLAIM - 1 < DEPTH - LEAD ? CLAIM - 1 : DEPTH - LEAD;
    constexpr int LATE = SLOTS_AFTER * CPS;          // first request number that falls into the next stage
    constexpr int IDX_END = COPIES;
    static_assert(BDIRECT || COPIES <= SLOTS_PER_STAGE, "a stage-load's requests are out before the next barrier");
    static_assert(!BDIRECT || COPIES <= LATE, "with weights in registers every request goes out behind the barrier");
    static_assert((TM == TN && TM % 2 == 0) || (TM == 3 && TN == 2) || (TM == 7 && TN == 2) || (TM == 2 && TN == 1 && !GATED) ||
                  (TM == 3 && TN == 1 && !GATED) || (TM == 4 && TN == 1 && !GATED && BDIRECT), "supported wavefront tiles");
    static_assert(BM % 32 == 0 && BN % 32 == 0, "every wavefront copies whole groups of 8 rows");
    static_assert(DEPTH == 2 || DEPTH == 4 || (DEPTH == 8 && BDIRECT), "ring depth");
    // (the epilogue stages the bf16 tile in the same LDS; where the ring is smaller than that, the ring grows)
    constexpr int EPI_STAGING = 4 * WM * ((GATED ? TN / 2 : TN) * 64);
    constexpr int LDS_BYTES = DEPTH * STAGE_BYTES > EPI_STAGING ? DEPTH * STAGE_BYTES : EPI_STAGING;
    // What the epilogue multiplies with - BM row scales, BN weight scales, BN bias values - rides along with the first
    // stage-load into LDS of its own, a word per lane, in blocks of 64 words.
    constexpr bool RIDE = big_constants_ride(TM, TN);
    constexpr int XBLOCKS = (BM + 63) / 64, WBLOCKS = BN / 64, BBLOCKS = (BN + 127) / 128;
    constexpr int CONSTS = RIDE ? (XBLOCKS + WBLOCKS + BBLOCKS + 3) / 4 : 0;   // copies of a wavefront
    constexpr int CONST_AT = LDS_BYTES + (BDIRECT ? 16 : 0), CONST_BYTES = RIDE ? (XBLOCKS + WBLOCKS + BBLOCKS) * 256 : 0;
    // (weights in registers: 16 more bytes for the four wavefronts' progress words, see the main loop)
    __shared__ __attribute__((aligned(1024))) uint8_t lds[CONST_AT + CONST_BYTES];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave / WGN, wn = wave % WGN;
    const int l16 = lane & 15, q = lane >> 4;
    (void)wm;
    const int half_n = p.N / 2;
    BigTile tile_id;
    int split_z = SPLIT ? (int)blockIdx.z : 0, n_splits = SPLIT ? (int)gridDim.z : 1;
    if (SPLIT && p.by_rows == 2) {
        // Split-K with an XCD per K range: XCD x (= id % 8) works on K range x % S of the tile
        // columns of group x / S, all tile rows.  The workgroups of an XCD then march along the same
        // K range together: its L2 fetches that range of the activation rows once, not all of K.
        n_splits = p.band;   // the split count rides in `band`, which this order does not use
        const int x = blockIdx.x & 7, r = blockIdx.x >> 3, groups = 8 / n_splits;
        const int cols = (p.n_tiles + groups - 1) / groups;
        split_z = x % n_splits;
        tile_id.n = (x / n_splits) * cols + r % cols;
        tile_id.m = r / cols;
    } else if (p.by_rows) {   // an XCD takes tile rows: bands of tile columns, 8 neighbouring tile rows per 8 ids
        const BigTile t = big_tile_of(blockIdx.x, p.n_tiles, p.m_tiles, p.band);
        tile_id.m = t.n; tile_id.n = t.m;
    } else {
        tile_id = big_tile_of(blockIdx.x, p.m_tiles, p.n_tiles, p.band);
    }
    if (tile_id.n >= p.n_tiles || tile_id.m >= p.m_tiles) return;   // padding of the tile order
    const int m0 = tile_id.m * BM;
    const int n0 = GATED ? tile_id.n * (BN / 2) : tile_id.n * BN;

    // acc[i][j][p][b]: rows 32 i + 16 p .., columns 32 j + 16 b .. of the wavefront's tile
    v4f acc[TM][TN][2][2];
#pragma unroll
    for (int e = 0; e < TM * TN * 4; ++e) acc[e / (TN * 4)][e / 4 % TN][e / 2 % 2][e % 2] = v4f{0.f, 0.f, 0.f, 0.f};
    // The multiply in inline assembly, with the sum in place: left to the compiler, a sum may land in other registers than
    // it came from, and with 96 - 256 of them live that ends in copies and spills (3 x 2 blocks: 174 registers this way,
    // 256 the other; 7 x 2 did not fit).  AGPRs where the VGPRs do not hold them (the split kernels' epilogue wants those for the
    // other half).  The s_nop covers a VALU write of an operand just before (the hazards inside an asm are not the compiler's).
    constexpr bool ACC_IN_AGPR = TM * TN >= 14 || SPLIT;
    auto multiply = [&](v8i w, v8i x, v4f& c) {
        if constexpr (ACC_IN_AGPR) asm volatile("s_nop 1\n\tv_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, %0" : "+a"(c) : "v"(w), "v"(x));
        else asm volatile("s_nop 1\n\tv_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, %0" : "+v"(c) : "v"(w), "v"(x));
    };
    auto acc_of = [&](int blk, int e) -> float { return acc[blk / TN][blk % TN][e >> 3][(e >> 2) & 1][e & 3]; };   // e: 0 .. 15

    // ---- copy geometry: wavefront w moves 8-row groups w*CA .. of A and w*CB .. of B; lane i
    // fills slot i%8 of row i/8 of its group with the chunk that the swizzle assigns to it ------
    // (padded rows of codes begin on a line and end in zeros: nothing to check in them)
    const bool a_padded = RAGGED && ((a_order >> 12) & 1);
    const uint32_t lda = a_padded ? ((uint32_t)p.K + 127u) & ~127u : (uint32_t)p.K;
    uint32_t aoff[CA], boff[CB > 0 ? CB : 1];
#pragma unroll
    for (int i = 0; i < CA; ++i) {
        const int rt = (wave * CA + i) * 8 + (lane >> 3);         // row of the tile
        int r = m0 + rt;
        r = r < p.M ? r : p.M - 1;
        aoff[i] = (uint32_t)r * lda + (((lane & 7) ^ big_swizzle(rt)) << 4);
    }
    // first 16-row unit of the tile in an operand-order matrix (plain: 16 weight rows; gated: 8 gate
    // columns and the 8 up columns that pair with them), and the units the matrix has
    const uint32_t unit0 = GATED ? (uint32_t)n0 >> 3 : (uint32_t)n0 >> 4, units = (uint32_t)p.N >> 4;
#pragma unroll
    for (int i = 0; i < CB; ++i) {
        if constexpr (WMODE == 1) {
            // instruction i moves half a unit (1 KB) as it lies; units past the matrix repeat the last one
            const uint32_t hu = wave * CB + i, u = unit0 + (hu >> 1);
            boff[i] = (u < units ? u : units - 1) * ((uint32_t)p.K << 4) + (hu & 1) * 1024 + lane * 16;
            continue;
        }
        const int jj = (wave * CB + i) * 8 + (lane >> 3);         // column of the output tile
        int rb;
        uint32_t ob;   // the row's place in operand order
        if constexpr (GATED) {
            const int w_ = jj / WN, j = jj % WN;
            int g = n0 + w_ * (WN / 2) + (j % (WN / 2));
            g = g < half_n ? g : half_n - 1;
            rb = (j / (WN / 2)) * half_n + g;
            ob = operand_offset_gated((uint32_t)g, (uint32_t)(j / (WN / 2)), (uint32_t)p.K);
        } else {
            rb = n0 + jj;
            rb = rb < p.N ? rb : p.N - 1;
            ob = operand_offset_plain((uint32_t)rb, (uint32_t)p.K);
        }
        const uint32_t chunk = (uint32_t)((lane & 7) ^ big_swizzle(jj));
        boff[i] = !RAGGED && p.operand_w ? ob + chunk * kOperandChunkBytes : (uint32_t)rb * (uint32_t)p.K + (chunk << 4);
    }
    const int k_begin = SPLIT ? split_z * p.k_per_split : 0;
    // RAGGED: the last stage-load of the matrix holds K % 128 bytes per row; kCopyNothing for the lanes whose chunk is
    // not among them.  The chunk of a lane depends on its row's swizzle, which repeats every two 8-row groups.
    uint32_t a_gone[2] = {0, 0}, b_gone[2] = {0, 0};
    v4i a_source = {0, 0, 0, 0}, b_source = {0, 0, 0, 0};
    if constexpr (RAGGED) {
        const int tail = p.K & (BIG_BK - 1);
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int ra = (wave * CA + e) * 8 + (lane >> 3), rb = (wave * CB + e) * 8 + (lane >> 3);
            a_gone[e] = !a_padded && (((lane & 7) ^ big_swizzle(ra)) << 4) >= tail ? kCopyNothing : 0u;
            b_gone[e] = (((lane & 7) ^ big_swizzle(rb)) << 4) >= tail ? kCopyNothing : 0u;
        }
        a_source = copy_source(p.a, (uint32_t)p.M * lda);
        b_source = copy_source(p.b, (uint32_t)p.N * (uint32_t)p.K);
    }
    const int b_step_shift = (OPW || p.operand_w) ? 4 : 0;   // a K step of operand-order weights is 2 KB away, not 128 bytes
    // BDIRECT: unit b of weight block j, K step 0 (the same for the whole wavefront); lane i takes bytes 16 i of its first
    // KB (chunk q of row l16: the units' own order) and of its second, the next K step is 2 KB further
    const uint32_t lane16 = (uint32_t)lane * 16;
    const uint8_t* bsrc[BDIRECT ? TN : 1][2];
    v4i bring[BDIRECT ? DEPTH : 1][BDIRECT ? TN : 1][2][2];   // [stage-load % DEPTH][block][unit][chunk pair]
    if constexpr (BDIRECT) {
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                const uint32_t u = unit0 + (uint32_t)(__builtin_amdgcn_readfirstlane(wn) * (WN / 16) + 2 * j + b);
                bsrc[j][b] = p.b + (size_t)(u < units ? u : units - 1) * ((size_t)p.K << 4) + ((size_t)k_begin << 4);
            }
    }
    const uint32_t lds_base = (uint32_t)(uintptr_t)lds;
    const uint32_t const_base = __builtin_amdgcn_readfirstlane(lds_base + CONST_AT);
    const uint32_t wave_a = __builtin_amdgcn_readfirstlane(lds_base + wave * (CA * 1024));
    const uint32_t wave_b = __builtin_amdgcn_readfirstlane(lds_base + BM * BIG_BK + wave * (CB * 1024));
    // copy c (0 .. COPIES-1) of this wavefront's share of stage-load `d` (K bytes [128 d, 128 d + 128))
    // (slot: d % DEPTH as a compile-time value, needed where the target is a register set)
    auto issue = [&](int d, int c, auto slot) {
        const int k = k_begin + d * BIG_BK;
        const uint32_t stage_off = __builtin_amdgcn_readfirstlane((d % DEPTH) * STAGE_BYTES);   // (goes into m0: a scalar)
        if constexpr (RAGGED) {
            const uint32_t last = k + BIG_BK > p.K ? ~0u : 0u;   // (uniform)
            if (c < CA) copy16_to_lds_checked(a_source, aoff[c] | (a_gone[c & 1] & last), k, wave_a + stage_off + c * 1024);
            else copy16_to_lds_checked(b_source, boff[c - CA] | (b_gone[(c - CA) & 1] & last), k, wave_b + stage_off + (c - CA) * 1024);
            return;
        }
        if (c < CA) {
            copy16_to_lds(p.a + k, aoff[c], wave_a + stage_off + c * 1024);
        } else if constexpr (BDIRECT) {
            constexpr int S = decltype(slot)::value;
            const int e = c - CA, j = e >> 2, b = (e >> 1) & 1, pr = e & 1;   // half pr of unit b of block j
            bring[S][j][b][pr] = *reinterpret_cast<const v4i*>(bsrc[j][b] + ((size_t)d << 11) + pr * 1024 + lane16);
        } else {
            copy16_to_lds(p.b + ((size_t)k << b_step_shift), boff[c - CA], wave_b + stage_off + (c - CA) * 1024);
        }
    };
    using Slot0 = std::integral_constant<int, 0>;
    const bool bias_rides = p.bias != nullptr && (reinterpret_cast<uintptr_t>(p.bias) & 3) == 0;
    // Blocks of the constants: row scales of the tile, then the weight scales of its columns (gated: gate columns, then up
    // columns), then their bias values, two to a word; past the matrix its last ones.  Every wavefront makes CONSTS copies (the
    // waits count them): with fewer blocks than that one of them again.  No bias, or one that is not a row of words: its
    // place is filled by hand.
    const int M = p.M, N = p.N, one_scale = p.a_scale_scalar;
    auto issue_constants = [&, M, N, one_scale](const void* x_scale, const void* w_scale, const void* bias) {
#pragma unroll
        for (int c = 0; c < CONSTS; ++c) {
            constexpr int LAST = XBLOCKS + WBLOCKS + BBLOCKS - 1;
            const int w = __builtin_amdgcn_readfirstlane(c * 4 + wave);
            int blk = w < LAST ? w : LAST;
            if (blk >= XBLOCKS + WBLOCKS && !bias_rides) blk = XBLOCKS;
            const void* base;
            uint32_t at;
            if (blk < XBLOCKS) {
                const int m = m0 + blk * 64 + lane;
                base = x_scale;
                at = one_scale ? 0u : (uint32_t)(m < M ? m : M - 1) * 4;
            } else {
                // column j of the tile; bias: the even one of the pair
                const bool of_bias = blk >= XBLOCKS + WBLOCKS;
                int j = of_bias ? (blk - XBLOCKS - WBLOCKS) * 128 + 2 * lane : (blk - XBLOCKS) * 64 + lane;
                if (j >= BN) j = 0;
                int n;
                if constexpr (GATED) {
                    const int up = j >= BN / 2 ? 1 : 0;
                    n = n0 + j - up * (BN / 2);
                    n = (n < half_n ? n : half_n - 2) + up * half_n;
                } else {
                    n = n0 + j;
                    n = n < N ? n : N - 2;
                }
                base = of_bias ? bias : w_scale;
                at = (uint32_t)n * (of_bias ? 2u : 4u);
            }
            const uint64_t b64 = reinterpret_cast<uint64_t>(base);   // (uniform, which the compiler does not see)
            const uint64_t b_lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b64);
            const uint64_t b_hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(b64 >> 32));
            copy4_to_lds(reinterpret_cast<const uint8_t*>(b_lo | b_hi << 32), at, __builtin_amdgcn_readfirstlane(const_base + blk * 256));
        }
        if (CONSTS > 0 && !bias_rides && tid < BN) {
            uint16_t v = 0;
            if (bias != nullptr) {
                const int up = GATED && tid >= BN / 2 ? 1 : 0, n = n0 + tid - up * (BN / 2), lim = GATED ? half_n : N;
                v = static_cast<const uint16_t*>(bias)[(n < lim ? n : lim - 1) + up * half_n];
            }
            reinterpret_cast<uint16_t*>(lds + CONST_AT + (XBLOCKS + WBLOCKS) * 256)[tid] = v;
        }
    };

    // stage-loads in all, >= DEPTH
    const int n_loads = RAGGED && SPLIT ? ((k_begin + p.k_per_split < p.K ? p.k_per_split : p.K - k_begin) + BIG_BK - 1) / BIG_BK
                        : RAGGED        ? (p.K + BIG_BK - 1) / BIG_BK
                                        : (SPLIT ? p.k_per_split : p.K) / BIG_BK;
    const int arow = wm * WM + l16, brow = wn * WN + l16;
    auto stage_ptr = [&](int d) -> const uint8_t* { return lds + (d % DEPTH) * STAGE_BYTES; };
    // 16-row block jj of the wavefront's staged weight rows
    auto read_b = [&](const uint8_t* stage, int jj) -> v8i {
        const uint8_t* bbuf = stage + BM * BIG_BK;
        if constexpr (WMODE == 1) return big_frag_operand(bbuf, brow + jj * 16, q);
        else return big_frag(bbuf, brow + jj * 16, q);
    };

    // Weights in registers: LDS carries the activations only, and the wavefronts hand its stages to each other
    // through one progress word each instead of meeting at a barrier.  Word w = d says: wavefront w has issued all its
    // LDS reads of stage-loads <= d, and its own copies of stage-loads <= d + CLAIM have landed.  At its hand-over
    // point of stage d a wavefront publishes d and goes on once every word is >= d - SLACK: then stage-load d + 1 is
    // complete in LDS (SLACK <= CLAIM - 1) and the stage that stage-load d + LEAD refills has been read by everyone
    // (it held stage-load d + LEAD - DEPTH <= d - SLACK).  A wavefront may so run up to SLACK stages ahead of the
    // slowest instead of waiting for it at every stage: each stalls now and then on its own memory requests, and a
    // barrier per stage makes all four pay for every such stall (7 x 2 blocks per wavefront, K = 2048, earlier MFMA: 40.2 k
    // cycles with the barrier, 32.7 k with none at all and with this).  The slowest wavefront never waits, so the scheme cannot
    // lock up; the spin is bounded all the same (a wavefront that gave up would read a stage early: wrong numbers,
    // never a hang).
    // The words are read BEFORE the stage's last batch of operand reads and looked at behind the MFMAs that follow it
    // (LDS answers in order: read at the hand-over point they would queue behind that batch, several hundred cycles
    // with two MFMAs in the pipe); a value that old can only be too small, and then the words are read again.
    // (pointers that say "LDS": through a generic pointer the accesses would be flat ones, counted with the copies)
    typedef __attribute__((address_space(3))) int lds_int_t;
    typedef __attribute__((address_space(3))) v4i lds_v4i_t;
    volatile lds_int_t* const progress = (volatile lds_int_t*)(lds + LDS_BYTES);
    auto progress_words = [&]() -> v4i { return *(const volatile lds_v4i_t*)(lds + LDS_BYTES); };
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

    // A stage-load is multiplied in two halves, each with one 16-row half (p) of the wavefront's 32-row activation blocks
    // and all of its weights: TM x 2 TN MFMAs.  Activation blocks of half p are in fa[p]; staged weights (fb) are read
    // once per stage-load, block by block into the registers that its predecessor's last MFMA has just left.
    // (224-row tiles with staged weights read only the first three of a half's activation blocks ahead, the others where
    // the last group of MFMAs leaves their predecessors' registers: two whole sets of seven do not fit)
    constexpr int AHEAD_BLOCKS = TM == 7 ? 3 : TM;
    v8i fa[2][TM], fb[BDIRECT ? 1 : 2 * TN];

// LDS reads are issued long before their MFMAs: a batch of 128-bit reads takes several hundred cycles to land.
//
// One barrier per stage-load, in half 1 after the first group of MFMAs: by then a wavefront has issued every
// LDS read of stage-load D, so the barrier both publishes stage-load D+1 (own copies awaited
// first: AHEAD later stage-loads may stay in flight) and releases D's stage, which load D+DEPTH
// then refills.  Its copies are requested one or two at a time between the MFMAs that follow - a
// wavefront that queues them all at once sits in the memory pipeline's issue queue while its
// MFMA pipe runs dry.  ISSUE: load D+DEPTH exists (requests after the barrier); ISSUE_P: load
// D-1+DEPTH exists (requests still being spread before the barrier).  All flags are literals, so
// the steady-state loop body is straight-line code.
//
// PHYAI_MFMA_SLOT: one MFMA and the requests that go out behind it; SLOT_: MFMAs since the last barrier.
#define PHYAI_MFMA_SLOT(FB, FA, ACC, SLOT_)                                                                    \
    {                                                                                                          \
        multiply(FB, FA, ACC);                                                                                 \
        _Pragma("unroll") for (int c_ = 0; c_ < CPS; ++c_)                                                     \
            if (req_ && (SLOT_) * CPS + c_ < IDX_END) {                                                        \
                /* (register set of the load: its number modulo DEPTH) */                                      \
                if (after_) issue(load_, (SLOT_) * CPS + c_, std::integral_constant<int, (stage_slot_ + LEAD) % DEPTH>{});     \
                else issue(load_, (SLOT_) * CPS + c_, std::integral_constant<int, (stage_slot_ + LEAD - 1) % DEPTH>{}); \
            }                                                                                                  \
        __builtin_amdgcn_sched_barrier(0);                                                                     \
    }
// Half P of stage-load D with staged weights: weight block after weight block, so that a block's registers are free for
// the next stage-load's as soon as its own MFMAs are issued.
#define PHYAI_RUN_HALF_STAGED(D, SLOT, P, NEXT, AHEAD, ISSUE_P, ISSUE)                                         \
    {                                                                                                          \
        const int d_ = (D);                                                                                    \
        constexpr int stage_slot_ = (SLOT);                                                                    \
        const uint8_t* nbuf_ = (P) == 0 ? stage_ptr(d_) : stage_ptr(d_ + 1);                                   \
        if ((P) == 0) {                                                                                        \
            _Pragma("unroll") for (int a_ = 0; a_ < AHEAD_BLOCKS; ++a_)                                        \
                fa[1][a_] = big_frag(nbuf_, arow + a_ * 32 + 16, q);                                           \
        }                                                                                                      \
        _Pragma("unroll") for (int jj_ = 0; jj_ < 2 * TN; ++jj_) {                                             \
            const bool after_ = (P) == 1 && jj_ >= 1;   /* past this stage-load's barrier */                   \
            const bool req_ = after_ ? (ISSUE) : (ISSUE_P);                                                    \
            const int load_ = after_ ? d_ + LEAD : d_ - 1 + LEAD;                                              \
            const int slot0_ = after_ ? (jj_ - 1) * TM : SLOTS_AFTER + ((P) * 2 * TN + jj_) * TM;              \
            _Pragma("unroll") for (int i_ = 0; i_ < TM; ++i_) {                                                \
                PHYAI_MFMA_SLOT(fb[jj_], fa[P][i_], acc[i_][jj_ >> 1][P][jj_ & 1], slot0_ + i_)                \
                if (i_ >= AHEAD_BLOCKS && jj_ == 2 * TN - 1 && ((P) == 0 || (NEXT)))                           \
                    fa[1 - (P)][i_] = big_frag(nbuf_, arow + i_ * 32 + 16 * (1 - (P)), q);                     \
            }                                                                                                  \
            if ((P) == 1 && (NEXT)) {                                                                          \
                if (jj_ == 0) {                                                                                \
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); /* my reads of stage-load D have landed */ \
                    wait_copies<COPIES * (AHEAD)>();               /* ... my copies of D+1 too ... */          \
                    __syncthreads();  /* ... and so have everybody's */                                        \
                }                                                                                              \
                fb[jj_] = read_b(nbuf_, jj_);                                                                  \
                /* the activation blocks of the next half 0: one or two behind each of the first groups */     \
                _Pragma("unroll") for (int a_ = 0; a_ < AHEAD_BLOCKS; ++a_)                                    \
                    if (a_ * TN / TM == jj_) fa[0][a_] = big_frag(nbuf_, arow + a_ * 32, q);                   \
            }                                                                                                  \
        }                                                                                                      \
    }
// My activation copies of D+CLAIM have landed (AHEAD: the stage-loads from that one on that have been requested: its
// weight loads, which follow its copies, and all of the later ones may be in flight); published, and everybody's of D+1
// awaited.
#define PHYAI_HAND_OVER(D_, AHEAD)                                                                             \
    {                                                                                                          \
        wait_copies<(AHEAD) == 0 ? 0 : ((AHEAD) - 1) * COPIES + (COPIES - CA)>();                              \
        hand_over(D_, seen_);                                                                                  \
        asm volatile("" ::: "memory");                                                                         \
    }
// Half P of stage-load D with weights in registers: row block after row block.  All of a half's blocks are read during the
// half before, one behind each pair of MFMAs, so that the hand-over can open half 1 and the requests have all of it.
#define PHYAI_RUN_HALF_DIRECT(D, SLOT, P, NEXT, AHEAD, ISSUE_P, ISSUE)                                         \
    {                                                                                                          \
        const int d_ = (D);                                                                                    \
        constexpr int stage_slot_ = (SLOT);                                                                    \
        const uint8_t* abuf_ = stage_ptr(d_);                                                                  \
        const uint8_t* nbuf_ = (P) == 0 ? abuf_ : stage_ptr(d_ + 1);                                           \
        if ((P) == 1 && (NEXT)) PHYAI_HAND_OVER(d_, AHEAD)                                                     \
        _Pragma("unroll") for (int i_ = 0; i_ < TM; ++i_) {                                                    \
            if ((P) == 0 && i_ == TM - 1) seen_ = progress_words();                                            \
            if (NEXT) fa[1 - (P)][i_] = big_frag(nbuf_, arow + i_ * 32 + 16 * (1 - (P)), q);                   \
            const bool after_ = (P) == 1;   /* past this stage-load's hand-over */                             \
            const bool req_ = after_ ? (ISSUE) : (ISSUE_P);                                                    \
            const int load_ = after_ ? d_ + LEAD : d_ - 1 + LEAD;                                              \
            const int slot0_ = after_ ? i_ * 2 * TN : SLOTS_AFTER + ((P) * TM + i_) * 2 * TN;                  \
            _Pragma("unroll") for (int jj_ = 0; jj_ < 2 * TN; ++jj_)                                           \
                PHYAI_MFMA_SLOT(big_join(bring[SLOT][jj_ >> 1][jj_ & 1][0], bring[SLOT][jj_ >> 1][jj_ & 1][1]), \
                                fa[P][i_], acc[i_][jj_ >> 1][P][jj_ & 1], slot0_ + jj_)                        \
        }                                                                                                      \
    }
// a whole stage-load
#define PHYAI_RUN_STAGE(D, SLOT, NEXT, AHEAD, ISSUE_P, ISSUE)                                                  \
    if constexpr (BDIRECT) {                                                                                   \
        v4i seen_ = {0, 0, 0, 0};                                                                              \
        PHYAI_RUN_HALF_DIRECT(D, SLOT, 0, 1, 0, ISSUE_P, 0)                                                    \
        PHYAI_RUN_HALF_DIRECT(D, SLOT, 1, NEXT, AHEAD, ISSUE_P, ISSUE)                                         \
    } else {                                                                                                   \
        PHYAI_RUN_HALF_STAGED(D, SLOT, 0, 1, 0, ISSUE_P, 0)                                                    \
        PHYAI_RUN_HALF_STAGED(D, SLOT, 1, NEXT, AHEAD, ISSUE_P, ISSUE)                                         \
    }

    // prologue: stage-loads 0 .. DEPTH-2 and the copies of load DEPTH-1 that the row groups after
    // a barrier would have requested in flight (the rest of it is spread over stage-load 0 like
    // every later one), load 0 published, its opening blocks in registers.
    // (as request numbers up to LATE, and as the instructions they are)
    constexpr int HEAD_IDX = LATE < IDX_END ? LATE : IDX_END;
    constexpr int HEAD = BDIRECT ? 0 : HEAD_IDX;
    if constexpr (BDIRECT) {   // stage-loads 0 .. LEAD - 1; stage-load d fills register set d % DEPTH
        // First what the first stage waits for: the activations of the stage-loads that progress word -1 vouches
        // for (0 .. CLAIM - 1; they come from L2) and the weights of stage-load 0; then the other weights of those
        // stage-loads and the later stage-loads whole, in the order the waits of the main loop count on.
        auto part = [&](auto slot, int c0, int c1) {
#pragma unroll
            for (int c = c0; c < c1; ++c) issue(decltype(slot)::value, c, slot);
        };
        using S0 = std::integral_constant<int, 0>; using S1 = std::integral_constant<int, 1>;
        using S2 = std::integral_constant<int, 2>;
        part(S0{}, CA, IDX_END);   // (the weights of stage-load 0 come from HBM: out first)
        part(S0{}, 0, CA);
        part(S1{}, 0, CA);
        if constexpr (CLAIM == 3) part(S2{}, 0, CA);
        issue_constants(p.a_scale, p.b_scale, p.bias);
        part(S1{}, CA, IDX_END);
        if constexpr (CLAIM == 3) part(S2{}, CA, IDX_END);
        if constexpr (CLAIM == 2) part(S2{}, 0, IDX_END);
        if constexpr (LEAD == 6) {
            part(std::integral_constant<int, 3>{}, 0, IDX_END);
            part(std::integral_constant<int, 4>{}, 0, IDX_END);
            part(std::integral_constant<int, 5>{}, 0, IDX_END);
        }
    } else {
#pragma unroll
        for (int d = 0; d < DEPTH - 1; ++d) {
#pragma unroll
            for (int c = 0; c < COPIES; ++c) issue(d, c, Slot0{});
            if (d == 0) issue_constants(p.a_scale, p.b_scale, p.bias);
        }
#pragma unroll
        for (int c = 0; c < HEAD_IDX; ++c) issue(DEPTH - 1, c, Slot0{});
    }
    // (the large tiles' 224 - 256 accumulators are zeroed here, under the first stage-load's latency: left to the
    // compiler they are zeroed behind the wait, 1 - 2 k cycles in which nothing else happens)
    if constexpr (TM * TN >= 14) {
#pragma unroll
        for (int e = 0; e < TM * TN * 4; ++e) asm volatile("" : "+a"(acc[e / (TN * 4)][e / 4 % TN][e / 2 % 2][e % 2]));
    }
    if constexpr (BDIRECT) {
        // stage-load 0 and the activations up to stage-load CLAIM - 1 have landed (what progress word -1 stands for)
        wait_copies<(LEAD - CLAIM) * COPIES + (CLAIM - 1) * (COPIES - CA) + CONSTS>();
        if (lane == 0) progress[wave] = -1;
    } else {
        wait_copies<COPIES * (LEAD - 2) + HEAD + CONSTS>();   // stage-load 0 has landed
    }
    __syncthreads();
    PHYAI_STAMP(1)
    if constexpr (!BDIRECT) {
#pragma unroll
        for (int jj = 0; jj < 2 * TN; ++jj) fb[jj] = read_b(lds, jj);
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) fa[0][i] = big_frag(lds, arow + i * 32, q);
    int d = 0;
    if constexpr (BDIRECT) {
        // the register sets are named at compile time: DEPTH stage-loads per trip (the launcher sees to it
        // that their number is a multiple of DEPTH)
        // ring of four: at the hand-over of stage d stage-load d + 2 may be in flight; behind it d + 3 is requested
        for (; d < n_loads - DEPTH; d += DEPTH) {
            if constexpr (DEPTH == 4) {
                PHYAI_RUN_STAGE(d, 0, 1, 1, 0, 1)
                PHYAI_RUN_STAGE(d + 1, 1, 1, 1, 0, 1)
                PHYAI_RUN_STAGE(d + 2, 2, 1, 1, 0, 1)
                PHYAI_RUN_STAGE(d + 3, 3, 1, 1, 0, 1)
            } else {   // at the hand-over of stage d stage-loads d + 3 .. d + 5 may be in flight; d + 6 is requested behind it
                PHYAI_RUN_STAGE(d, 0, 1, 3, 0, 1)
                PHYAI_RUN_STAGE(d + 1, 1, 1, 3, 0, 1)
                PHYAI_RUN_STAGE(d + 2, 2, 1, 3, 0, 1)
                PHYAI_RUN_STAGE(d + 3, 3, 1, 3, 0, 1)
                PHYAI_RUN_STAGE(d + 4, 4, 1, 3, 0, 1)
                PHYAI_RUN_STAGE(d + 5, 5, 1, 3, 0, 1)
                PHYAI_RUN_STAGE(d + 6, 6, 1, 3, 0, 1)
                PHYAI_RUN_STAGE(d + 7, 7, 1, 3, 0, 1)
            }
        }
    } else {
        for (; d < n_loads - DEPTH; ++d) { PHYAI_RUN_STAGE(d, 0, 1, DEPTH - 2, 1, 1) }
    }
    // d == n_loads - DEPTH: the last requests are still being spread, then the ring drains
    if constexpr (BDIRECT && DEPTH == 8) {   // the last request goes out behind the hand-over of stage n - 7
        PHYAI_RUN_STAGE(d, 0, 1, 3, 0, 1)
        PHYAI_RUN_STAGE(d + 1, 1, 1, 3, 0, 1)
        PHYAI_RUN_STAGE(d + 2, 2, 1, 3, 0, 0)
        PHYAI_RUN_STAGE(d + 3, 3, 1, 2, 0, 0)
        PHYAI_RUN_STAGE(d + 4, 4, 1, 1, 0, 0)
        PHYAI_RUN_STAGE(d + 5, 5, 1, 0, 0, 0)
        PHYAI_RUN_STAGE(d + 6, 6, 1, 0, 0, 0)
        PHYAI_RUN_STAGE(d + 7, 7, 0, 0, 0, 0)
    } else if constexpr (BDIRECT) {   // the last request goes out behind the hand-over of stage n - 4
        PHYAI_RUN_STAGE(d, 0, 1, 1, 0, 1)
        PHYAI_RUN_STAGE(d + 1, 1, 1, 1, 0, 0)
        PHYAI_RUN_STAGE(d + 2, 2, 1, 0, 0, 0)
        PHYAI_RUN_STAGE(d + 3, 3, 0, 0, 0, 0)
    } else if constexpr (DEPTH == 2) {
        PHYAI_RUN_STAGE(d, 0, 1, 0, 1, 0)
        PHYAI_RUN_STAGE(d + 1, 0, 0, 0, 0, 0)
    } else {
        PHYAI_RUN_STAGE(d, 0, 1, 2, 1, 0)
        PHYAI_RUN_STAGE(d + 1, 1, 1, 1, 0, 0)
        PHYAI_RUN_STAGE(d + 2, 2, 1, 0, 0, 0)
        PHYAI_RUN_STAGE(d + 3, 3, 0, 0, 0, 0)
    }
#undef PHYAI_RUN_STAGE
#undef PHYAI_RUN_HALF_STAGED
#undef PHYAI_RUN_HALF_DIRECT
#undef PHYAI_HAND_OVER
#undef PHYAI_MFMA_SLOT
    // the last MFMAs' results, before anything else reads them (24 wait states; every sum passes behind them)
    asm volatile("s_nop 15\n\ts_nop 7");
#pragma unroll
    for (int e = 0; e < TM * TN * 4; ++e) {
        v4f& c = acc[e / (TN * 4)][e / 4 % TN][e / 2 % 2][e % 2];
        if constexpr (ACC_IN_AGPR) asm volatile("" : "+a"(c));
        else asm volatile("" : "+v"(c));
    }
    __builtin_amdgcn_sched_barrier(0);
    PHYAI_STAMP(2)

    // ---- split-K: publish partial sums; the last split to arrive adds them in split order --
    // Two blocks (32 floats per lane) at a time, so that the 4 x 4 variant never holds more than
    // that outside its accumulators.
    // (K split in two) this workgroup arrived second: the half that the first one wrote is added where the epilogue
    // reads the accumulators, block by block, the loads of the next block under the arithmetic of the current one
    bool add_other = false;
    const int sp_tile = tile_id.m * p.n_tiles + tile_id.n;
    if constexpr (SPLIT) {
        constexpr int FRAG = TM * TN * 16, CHUNK = 32;
        const int S = n_splits;
        const int tile = sp_tile;
        auto publish = [&]() {
#pragma unroll
            for (int c = 0; c < TM * TN / 2; ++c) {
                float frag[CHUNK];
#pragma unroll
                for (int r = 0; r < 32; ++r) frag[r] = acc_of(2 * c + r / 16, r % 16);
                splitk_publish_part<FRAG, 256, CHUNK>(p.partials, tile, S, split_z, c * CHUNK, frag);
            }
            wait_own_stores();
        };
        // gather: as much of the fragment per round trip as the registers allow
        constexpr int GCH = FRAG <= 64 ? FRAG : 32;
        if (S == 2) {   // (uniform) two splits: the first to arrive writes its half, the second adds it to its own
            const int found = splitk_arrive_early(p.counters, tile, reinterpret_cast<int*>(lds));
            if (found == 0) {
                publish();
                splitk_published(p.counters, tile);
                return;
            }
            splitk_await_published(p.counters, tile, found);
            add_other = true;
        } else {
            publish();
            // splitk_arrive opens with a barrier, after which nobody reads operands any more: a word
            // of the ring serves as its flag
            if (!splitk_arrive(p.counters, tile, S, reinterpret_cast<int*>(lds))) return;
#pragma unroll
            for (int c = 0; c < FRAG / GCH; ++c) {
                float frag[GCH];
                splitk_gather_part<FRAG, 256, GCH>(p.partials, tile, S, c * GCH, frag);
#pragma unroll
                for (int r = 0; r < GCH; ++r) {
                    const int blk = (c * GCH + r) / 16;
                    const int e = r % 16;
                    acc[blk / TN][blk % TN][e >> 3][(e >> 2) & 1][e & 3] = frag[r];
                }
            }
        }
        splitk_reset(p.counters, tile);
    }

    PHYAI_STAMP(3)
    // ---- epilogue ------------------------------------------------------------------------
    // The weight block is the MFMA's first operand, so accumulator r of lane (l16, q) of block
    // (i, j, p, b) is the output at token row i*32 + 16*p + l16, column j*32 + 16*b + 4*q + r: a lane
    // owns runs of four consecutive columns of one row.  A run becomes four bf16 with two packed
    // converts and goes to the wavefront's slice of the (now idle) LDS as one 8-byte write; the
    // staged tile leaves row-wise, 16 bytes per lane, whole row segments per instruction.  The
    // 16-byte slots of a staged row are XOR-swizzled with the row so that the 32 rows written by
    // one instruction spread over the banks.
    constexpr int TNO = GATED ? TN / 2 : TN;             // output column blocks per wavefront
    constexpr int ROWB = TNO * 64;                       // staged row length in bytes
    constexpr int SLOTS = ROWB / 16;
    constexpr int ROWS_PER_PASS = 16 / SLOTS > 0 ? 16 / SLOTS : 1;   // rows per 256 bytes of banks
    constexpr int STG_BYTES = WM * ROWB;                 // per wavefront
    static_assert(4 * STG_BYTES <= LDS_BYTES, "staging fits in the operand LDS");
    const int n_lim = GATED ? half_n : p.N;
    const int nbase = n0 + wn * (GATED ? WN / 2 : WN);
    const float* const const_x = reinterpret_cast<const float*>(lds + CONST_AT);   // where RIDE
    const float* const const_w = const_x + XBLOCKS * 64;
    const uint16_t* const const_bias = reinterpret_cast<const uint16_t*>(const_w + BN);
    // column constants are read 4 at a time when the arrays allow it (N is a multiple of 16, so
    // a run of four columns is valid or invalid as a whole)
    const bool vec_cols = (reinterpret_cast<uintptr_t>(p.b_scale) & 15) == 0 &&
                          (reinterpret_cast<uintptr_t>(p.bias) & 7) == 0;
    auto bias4 = [](uint2 b, v4f& bi) {
        bi[0] = bf16_bits_to_f32(b.x & 0xFFFFu); bi[1] = __uint_as_float(b.x & 0xFFFF0000u);
        bi[2] = bf16_bits_to_f32(b.y & 0xFFFFu); bi[3] = __uint_as_float(b.y & 0xFFFF0000u);
    };
    // four columns from n of the matrix, which are columns c .. of the constants that rode
    auto load_cols = [&](int n, int c, v4f& sc, v4f& bi) {
        if constexpr (RIDE) {
            sc = *reinterpret_cast<const v4f*>(const_w + c);
            bias4(*reinterpret_cast<const uint2*>(const_bias + c), bi);
        } else if (vec_cols) {
            sc = *reinterpret_cast<const v4f*>(p.b_scale + n);
            if (p.bias) {
                bias4(*reinterpret_cast<const uint2*>(p.bias + n), bi);
            } else {
                bi[0] = bi[1] = bi[2] = bi[3] = 0.f;
            }
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                sc[e] = p.b_scale[n + e];
                bi[e] = p.bias ? bf16_bits_to_f32(p.bias[n + e]) : 0.f;
            }
        }
    };
    float sa[TM][2];
    if constexpr (!RIDE) {
#pragma unroll
        for (int e = 0; e < 2 * TM; ++e) {
            const int m = m0 + wm * WM + e * 16 + l16;
            sa[e >> 1][e & 1] = p.a_scale[p.a_scale_scalar ? 0 : (m < p.M ? m : p.M - 1)];
        }
    }
    __syncthreads();  // every wavefront is done reading operands from LDS, and its share of the constants has landed
    if constexpr (RIDE) {
#pragma unroll
        for (int e = 0; e < 2 * TM; ++e) sa[e >> 1][e & 1] = const_x[wm * WM + e * 16 + l16];
    }
    uint8_t* stg = lds + wave * STG_BYTES;
    // the other workgroup's 16 partial sums of block (i, j) (element (i TN + j) 16 + r of its fragment, splitk.h)
    auto other_half = [&](int i, int j, float* po) {
        if constexpr (SPLIT) {
            if (add_other) splitk_load_part<TM * TN * 16, 256, 16>(p.partials, sp_tile, 2, 1 - split_z, (i * TN + j) * 16, po);
        }
    };
    // accumulator r of a block, with the other half where there is one (a + b: the sum in split order either way)
    auto summed = [&](float a, const float* po, int r) { return SPLIT && add_other ? a + po[r] : a; };
    if constexpr (OPW && GATED) {
        // Weights in the gated operand order: rows 4q .. 4q+3 of a 16-row unit are gate columns 2q, 2q+1 and up
        // columns 2q, 2q+1 of the unit's 8.  Accumulator 2t + c of lane (l16, q) of unit b of block j is gate (t = 0) /
        // up (t = 1) of output column 16 j + 8 b + 2 q + c of the wavefront - a lane holds both halves of two
        // neighbouring output columns per unit.  Same arithmetic as below, operation for operation.
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            float sgk[2][2], suk[2][2], bgk[2][2], buk[2][2];
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                const int n = nbase + 16 * j + 8 * b + 2 * q;
                const int n_safe = n < n_lim ? n : 0;
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    if constexpr (RIDE) {
                        sgk[b][c] = const_w[n - n0 + c];
                        suk[b][c] = const_w[BN / 2 + n - n0 + c];
                    } else {
                        sgk[b][c] = p.b_scale[n_safe + c];
                        suk[b][c] = p.b_scale[half_n + n_safe + c];
                    }
                    if constexpr (RIDE) {
                        bgk[b][c] = bf16_bits_to_f32(const_bias[n - n0 + c]);
                        buk[b][c] = bf16_bits_to_f32(const_bias[BN / 2 + n - n0 + c]);
                    } else {
                        bgk[b][c] = p.bias ? bf16_bits_to_f32(p.bias[n_safe + c]) : 0.f;
                        buk[b][c] = p.bias ? bf16_bits_to_f32(p.bias[half_n + n_safe + c]) : 0.f;
                    }
                }
            }
            float pn[16] = {};
            other_half(0, j, pn);
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                float po[16];
#pragma unroll
                for (int r = 0; r < 16; ++r) po[r] = pn[r];
                if (i + 1 < TM) other_half(i + 1, j, pn);
#pragma unroll
                for (int pb = 0; pb < 4; ++pb) {
                    const int half = pb >> 1, b = pb & 1, row = i * 32 + 16 * half + l16;
                    const int sw = (row / ROWS_PER_PASS) & (SLOTS - 1);
                    const v4f& a = acc[i][j][half][b];
                    const float s = sa[i][half];
                    const float g0 = __builtin_fmaf(summed(a[0], po, 4 * pb + 0), s * sgk[b][0], bgk[b][0]);
                    const float g1 = __builtin_fmaf(summed(a[1], po, 4 * pb + 1), s * sgk[b][1], bgk[b][1]);
                    const float u0 = __builtin_fmaf(summed(a[2], po, 4 * pb + 2), s * suk[b][0], buk[b][0]);
                    const float u1 = __builtin_fmaf(summed(a[3], po, 4 * pb + 3), s * suk[b][1], buk[b][1]);
                    // gate and up pass through bf16 first, as the two-launch form materialises them
                    const uint32_t g01 = pack_bf16x2(g0, g1), u01 = pack_bf16x2(u0, u1);
                    const float o0 = apply_act<EPI>(__uint_as_float(g01 << 16)) * __uint_as_float(u01 << 16);
                    const float o1 = apply_act<EPI>(__uint_as_float(g01 & 0xFFFF0000u)) * __uint_as_float(u01 & 0xFFFF0000u);
                    *reinterpret_cast<uint32_t*>(stg + row * ROWB + ((2 * j + b) ^ sw) * 16 + 4 * q) = pack_bf16x2(o0, o1);
                }
            }
        }
    } else {
#pragma unroll
    for (int j = 0; j < TNO; ++j) {
        v4f sg[2], bg[2], su[2], bu[2];
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const int n = nbase + j * 32 + 16 * b + 4 * q;
            const int n_safe = n < n_lim ? n : 0;
            load_cols(n_safe, n - n0, sg[b], bg[b]);
            if constexpr (GATED) load_cols(half_n + n_safe, BN / 2 + n - n0, su[b], bu[b]);
        }
        float pn[16] = {}, un[16] = {};
        other_half(0, j, pn);
        if constexpr (GATED) other_half(0, j + TN / 2, un);
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            float po[16], pu[16];
#pragma unroll
            for (int r = 0; r < 16; ++r) { po[r] = pn[r]; pu[r] = un[r]; }
            if (i + 1 < TM) {
                other_half(i + 1, j, pn);
                if constexpr (GATED) other_half(i + 1, j + TN / 2, un);
            }
#pragma unroll
            for (int pb = 0; pb < 4; ++pb) {
                const int half = pb >> 1, b = pb & 1, row = i * 32 + 16 * half + l16;
                const int sw = (row / ROWS_PER_PASS) & (SLOTS - 1);
                const float s = sa[i][half];
                float o[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = __builtin_fmaf(summed(acc[i][j][half][b][e], po, 4 * pb + e), s * sg[b][e], bg[b][e]);
                if constexpr (GATED) {
                    float u[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) u[e] = __builtin_fmaf(summed(acc[i][j + TN / 2][half][b][e], pu, 4 * pb + e), s * su[b][e], bu[b][e]);
                    // gate and up pass through bf16 first, as the two-launch form materialises them
                    const uint32_t g01 = pack_bf16x2(o[0], o[1]), g23 = pack_bf16x2(o[2], o[3]);
                    const uint32_t u01 = pack_bf16x2(u[0], u[1]), u23 = pack_bf16x2(u[2], u[3]);
                    o[0] = apply_act<EPI>(__uint_as_float(g01 << 16)) * __uint_as_float(u01 << 16);
                    o[1] = apply_act<EPI>(__uint_as_float(g01 & 0xFFFF0000u)) * __uint_as_float(u01 & 0xFFFF0000u);
                    o[2] = apply_act<EPI>(__uint_as_float(g23 << 16)) * __uint_as_float(u23 << 16);
                    o[3] = apply_act<EPI>(__uint_as_float(g23 & 0xFFFF0000u)) * __uint_as_float(u23 & 0xFFFF0000u);
                } else if constexpr (EPI != EPI_NONE) {
                    const uint32_t g01 = pack_bf16x2(o[0], o[1]), g23 = pack_bf16x2(o[2], o[3]);
                    o[0] = apply_act<EPI>(__uint_as_float(g01 << 16));
                    o[1] = apply_act<EPI>(__uint_as_float(g01 & 0xFFFF0000u));
                    o[2] = apply_act<EPI>(__uint_as_float(g23 << 16));
                    o[3] = apply_act<EPI>(__uint_as_float(g23 & 0xFFFF0000u));
                }
                uint2 w;
                w.x = pack_bf16x2(o[0], o[1]);
                w.y = pack_bf16x2(o[2], o[3]);
                *reinterpret_cast<uint2*>(stg + row * ROWB + ((j * 4 + 2 * b + (q >> 1)) ^ sw) * 16 + (q & 1) * 8) = w;
            }
        }
    }
    }
    PHYAI_STAMP(4)
    // write the staged tile out: 1 KB (whole rows) per instruction.  The output is written once
    // and never read here: non-temporal stores keep it from evicting the operands that the
    // neighbouring tiles still want from L2 (4800 x 8192 x 2048 + GELU: 113 -> 95 us;
    // 13056 x 2560 x 2048: 76.6 -> 70.1 us; same box, alternating builds of the earlier main loop).
    auto write_out = [&](auto residual) {
#pragma unroll 4
        for (int qd = 0; qd < STG_BYTES / 1024; ++qd) {
            const int byte = qd * 1024 + lane * 16;
            const int row = byte / ROWB, slot = (byte % ROWB) / 16;
            const int sw = (row / ROWS_PER_PASS) & (SLOTS - 1);
            v4i v = *reinterpret_cast<const v4i*>(stg + row * ROWB + ((slot ^ sw) << 4));
            const int m = m0 + wm * WM + row;
            const int n = nbase + slot * 8;
            if (m >= p.M || n >= n_lim) continue;
            if constexpr (decltype(residual)::value) {   // out = residual + bf16(linear) * gate, row-wise like the output
                const int grow = p.res.gate_group >= p.M ? 0 : m / p.res.gate_group;
                const uint4 rs = *reinterpret_cast<const uint4*>(p.res.residual + (int64_t)m * p.res.ld_res + n);
                const uint4 gt = *reinterpret_cast<const uint4*>(p.res.gate + (int64_t)grow * p.res.ld_gate + n);
                v[0] = (int)addcmul2((uint32_t)v[0], rs.x, gt.x); v[1] = (int)addcmul2((uint32_t)v[1], rs.y, gt.y);
                v[2] = (int)addcmul2((uint32_t)v[2], rs.z, gt.z); v[3] = (int)addcmul2((uint32_t)v[3], rs.w, gt.w);
            }
            __builtin_nontemporal_store(v, reinterpret_cast<v4i*>(p.out + (int64_t)m * p.ldo + n));
        }
    };
    if constexpr (EPI == EPI_NONE) {
        if (p.res.residual != nullptr) write_out(std::true_type{});
        else write_out(std::false_type{});
    } else {
        write_out(std::false_type{});
    }
    PHYAI_STAMP(5)
    PHYAI_STAMP_END(g_big_stamps, ((size_t)blockIdx.x + (size_t)gridDim.x * blockIdx.z) * 4 + wave, lane)
}

// ---- host side ---------------------------------------------------------------------------

static int big_tile_cols(int tile) { return (tile == 256 || tile == 224) ? 256 : 128; }

// Fraction of the tile slots that hold a tile, over all rounds of `slots` concurrent tiles.
static double big_fill(int tiles, int slots) {
    const int rounds = big_ceil_div(tiles, slots);
    return rounds > 0 ? (double)tiles / ((double)rounds * slots) : 1.0;
}

// (PHYAI_FP8_BIG_DIRECT=0: weights in operand order go through LDS in every tile shape)
static bool big_registers_allowed() {
    const char* e = tuning_env("PHYAI_FP8_BIG_DIRECT");
    return e == nullptr || atoi(e) != 0;
}
// The ring of register sets that a shape's weights in operand order go through (0: staged in LDS).
static int big_register_ring(const BigPlan& pl, int K, int epilogue) {
    if (!big_registers_allowed()) return 0;
    if (K % 128 != 0) return 0;
    if (pl.tile == 224 && pl.splits == 1 && K % 512 == 0) return 4;
    if (pl.tile == 128 && pl.cols == 128 && pl.depth == 4 && (K / pl.splits) % 1024 == 0 && !epi_is_gated(epilogue)) return 8;
    // (more tiles than CUs: two workgroups per CU, each with a ring of four)
    if (pl.tile == 128 && pl.cols == 128 && pl.depth == 2 && pl.splits == 1 && K % 512 == 0 && !epi_is_gated(epilogue)) return 4;
    return 0;
}

// Shapes that share a CU in pairs.
static bool big_two_of(const BigPlan& pl) { return pl.depth == 2 && pl.cols == 128 && (pl.tile == 192 || pl.tile == 128); }
// Shapes of gemm_tall.hip: 256 columns, weights in registers.
static bool big_tall(const BigPlan& pl) { return pl.regs == 4 && pl.cols == 256; }

// Tile shape, K splits, ring depth.  All times in here: graphs of weight sets beyond the Infinity Cache, every tile shape
// forced in turn at 988 shapes (M = 136 .. 13056, N = 1024 .. 32768, K = 1024 .. 16384, both layouts).  The lines were drawn on
// an earlier main loop (32 x 32 x 64 MFMAs) and epilogue, whose times these are; where another shape is ahead by now, the comment
// says so.  With the fitted costs below (launch_gemm's choice: the order of sums for every GEMM, the tile shape for codes that a
// linear stages) ready codes are 1.0 % behind the best of all shapes in the geometric mean, linears 0.6 %.
BigPlan big_plan(int M, int N, int K, int epilogue, bool operand_w) {
    BigPlan pl = {0, 0, 1, 0, 0, 0};
    if (K < 512) return pl;   // the stage-loads must fill the ring
    const bool ragged = K % 128 != 0;
    if (const char* e = tuning_env("PHYAI_FP8_TALL")) {   // rows of a tile of gemm_tall.hip, where it takes the problem
        const int rows = atoi(e);
        if (operand_w && K % 128 == 0 && rows >= 144 && rows <= 256 && rows % 16 == 0) return {rows, 256, 1, big_tiles(M, N, epilogue, rows, 256), 2, 4};
    }
    int forced = -1;
    if (const char* e = tuning_env("PHYAI_FP8_BIG")) forced = atoi(e);   // "0": never; "256"/"192"/"128": force
    if (forced == 0) return pl;
    if (forced == 256 || forced == 224 || forced == 192 || forced == 128) pl.tile = forced;   // ("96": 96 x 128, below)
    else if (forced == 12864 && !epi_is_gated(epilogue)) { pl.tile = 128; pl.cols = 64; }   // "12864": 128 rows x 64 columns
    else if (forced == 96 && !epi_is_gated(epilogue)) { pl.tile = 96; pl.cols = 128; }
    else if (M < 128) return pl;
    // 256 x 256 tiles need the fewest bytes from L2 per flop but run one workgroup per CU, so a
    // tile's prologue and epilogue leave the MFMA pipe idle; 192 x 128 tiles fit twice and overlap
    // them.  The small tile wins once there are enough of them and while K is short enough for
    // prologue and epilogue to matter (192 / 256, us: 4800 x 8192 x 2048 + GELU 93 / 118, 1632 x 32768 x 2048 +
    // GeGLU 108 / 122, 4800 x 2048 x 8192 76 / 89), unless M pads worse or its last round of 512 tiles would be much
    // emptier than the large tile's last round of 256 (6528 x 2048 x 2048: 544 small tiles 36.3, 208 large
    // ones 33.2).  Row-major weights from K = 4096 on: 224 x 256 tiles are now ahead of both (3264 x 8192 x 4096 192:
    // 102, 224: 92; 13056 x 2048 x 8192 193 / 170) and are not asked.
    else if (K <= 8192 && big_tiles(M, N, epilogue, 192, 128) >= 400 &&
             big_ceil_div(M, 192) * 192 <= big_ceil_div(M, 256) * 256 &&
             big_fill(big_tiles(M, N, epilogue, 192, 128), 512) >= big_fill(big_tiles(M, N, epilogue, 256, 256), 256) - 0.15)
        pl.tile = 192;
    // ... and also when it fits one round of two workgroups per CU while 128 x 128 tiles would just
    // spill into a second one (3264 x 2560 x 2048: 340 tiles of 192 x 128 take 24.1 us, 520 of
    // 128 x 128 29.6; with 416 of those, 3264 x 2048 x 2048, the smaller tile wins 18.5 to 23.0)
    else if (K <= 8192 && big_tiles(M, N, epilogue, 256, 256) < 200 && big_tiles(M, N, epilogue, 192, 128) > 256 &&
             big_tiles(M, N, epilogue, 192, 128) <= 512 && big_tiles(M, N, epilogue, 128, 128) > 512)
        pl.tile = 192;
    else if (big_tiles(M, N, epilogue, 256, 256) >= 200)
        // 224 x 256 tiles (every wavefront walks all 224 token rows) when they need no more tile
        // rows than 256 x 256: the same number of workgroups, fewer MFMAs on padding (816 rows:
        // 896 instead of 1024, gate_up 2048 -> 32768 at M = 816 64.7 -> 59.2 us row-major).  More tile rows
        // are not tried, though where they fit the same rounds they are 8 - 10 % ahead now (6528 x 2048 x 2048, 240
        // tiles against 208: 30.3 / 33.2; 1632 x 8192 x 2048 37.9 / 41.2).
        pl.tile = big_ceil_div(M, 224) == big_ceil_div(M, 256) ? 224 : 256;
    else if (big_tiles(M, N, epilogue, 128, 128) >= 32) pl.tile = 128;   // fewer: the weight-streaming kernel wins
    else return pl;
    if (pl.cols == 0) pl.cols = big_tile_cols(pl.tile);
    int tiles = big_tiles(M, N, epilogue, pl.tile, pl.cols);
    // Few 128 x 128 tiles and a plain epilogue: 128 x 64 tiles (2 x 1 blocks per wavefront) put twice
    // as many CUs to work; the narrow tile reads half as many bytes again per MFMA, so it pays only while the
    // 128 x 128 grid leaves at least half of the CUs idle (us: 816 x 2048 x 2048, 112 -> 224 tiles, 11.6 -> 8.6;
    // 816 x 2048 x 4096 18.1 -> 13.2; 1100 x 1024 x 4096 17.6 -> 13.1; 816 x 2560 x 2048, 140 -> 280 tiles, a second
    // round, 11.8 -> 14.2 and stays).  From K = 8192 on the 128 x 128 form with K split in two is taken: ahead at
    // K = 16384 (816 rows: 38.3 against 42.6), no longer at 8192 (24.0 against 22.2).
    if (forced < 0 && pl.tile == 128 && !epi_is_gated(epilogue) && tiles > 64 && tiles <= 128 && K < 8192) {
        pl.cols = 64;
        tiles = big_tiles(M, N, epilogue, 128, 64);
    }
    // Between 129 and 255 tiles of 128 x 128 (and a plain epilogue) 96 x 128 tiles - wavefronts 1 x 4, three row
    // blocks each - put up to 256 CUs to work in one round where the 128-row grid leaves a fifth to a half of them
    // idle and 128 x 64 tiles would need a second round (128 x 128 / 96 x 128, us: 816 x 2560 x 2048, 140 -> 180 tiles,
    // 11.8 / 10.2, 816 x 3072 x 2048 11.9 / 10.3, 1000 x 2304 x 2048 12.0 / 10.4, 816 x 2560 x 4096 + GELU 19.2 / 16.3,
    // 560 x 4096 x 2048 12.0 / 10.4).  Where the 128-row grid already fills the chip, or 128 x 64 tiles fit one round,
    // it loses (816 x 2048 x 2048: 10.2 against 8.6; 1632 x 2560 x 2048: 18.5 against 15.7).  From K = 8192 on the
    // split form is taken, and there 96 x 128 tiles are far ahead now (1100 x 2048 x 8192 40.2 / 26.4, 2400 x 1024 x 16384
    // 60.8 / 46.7): the line at K = 8192 is the old loop's.
    if (forced < 0 && pl.tile == 128 && pl.cols == 128 && !epi_is_gated(epilogue) && tiles > 128 && tiles < 256 && K < 8192) {
        const int t96 = big_tiles(M, N, epilogue, 96, 128);
        if (t96 > tiles && t96 <= 256) { pl.tile = 96; tiles = t96; }
    }
    pl.tiles = tiles;
    pl.depth = (pl.tile == 128 || pl.tile == 96) ? 4 : 2;
    bool to_224 = false;
    if (operand_w && forced < 0 && pl.tile != 224 && K >= 4096 && K % 512 == 0) {
        // Weights in operand order: tiles of 224 x 256 load them straight into registers and hand their activation
        // stages over without barriers (gemm_tall.hip).  The line was drawn with that kernel's predecessor, whose prologue and
        // epilogue stood alone, and whose times these are; GEMMs on ready codes keep to it, a linear's staged codes get
        // the height that the costs below choose.  Taken with at least 160 tiles that fill their rounds of 256
        // workgroups with useful rows and columns at least 0.8 times as well as the shape chosen above fills its own
        // (chosen above / this, us: 6528 x 2048 x 16384 173 / 154, 13056 x 2048 x 16384 340 / 300, 6528 x 2048 x 8192 93.9 /
        // 81.8, 1632 x 8192 x 8192 93.4 / 85.0, 6528 x 4096 x 4096 104 / 96, 13056 x 2048 x 4096 101 / 91, 3264 x 16384 x 4096 +
        // GeGLU 184 / 181, 4800 x 8192 x 4096 141 / 134, 3264 x 8192 x 4096 101 / 89; level: 4800 x 2048 x 8192 74.1 / 73.6; not
        // taken, and slower when forced: 2048 x 8192 x 8192 (320 tiles, two rounds) 101 / 147, 8000 x 1024 x 8192 (144
        // tiles) 57.3 / 70.3, 3264 x 2048 x 16384 (120 tiles) 106 / 125).  0.8 lets a second round in that is nearly empty:
        // 6528 x 2560 x 4096 (300 tiles) 64.9 / 88.7, 4800 x 4096 x 4096 (352) 78.4 / 90.3.  At K = 2048 the shapes that run
        // two workgroups per CU are level or ahead.
        const int t224 = big_tiles(M, N, epilogue, 224, 256);
        const int slots = big_two_per_cu(pl.tile == 192 ? 3 : pl.tile == 256 ? 4 : 2, 2, pl.depth, 0) ? 512 : 256;
        const double area_now = (double)big_ceil_div(tiles * pl.splits, slots) * slots * pl.tile * pl.cols;
        const double area_224 = (double)big_ceil_div(t224, 256) * 256 * 224 * 256;
        if (t224 >= 160 && pl.splits == 1 && area_now >= 0.8 * area_224) to_224 = true;
    }
    if (to_224) {
        pl.tile = 224; pl.cols = 256; pl.depth = 2;
        pl.tiles = tiles = big_tiles(M, N, epilogue, 224, 256);
    }
    if ((pl.tile == 128 && pl.cols == 64) || pl.tile == 96) {
        // always one round of at most 256 workgroups here, or forced: deep ring, no split
    } else if (pl.tile == 128) {
        // K split in two: the partial sums' round trip is worth 4 - 8 us (816 rows: 56.1 -> 38.3 us at K = 16384, 29.4 ->
        // 24.0 at 8192, but 18.1 -> 18.7 at 4096, 11.6 -> 16.8 at 2048).
        if (tiles < 200 && K >= 8192 && (K % 256 == 0 || ragged)) pl.splits = 2;
        // With more tiles than CUs a ring of two stages lets two workgroups share a CU instead of
        // queueing behind each other (1632 x 2560 x 2048, 260 tiles: 21.5 -> 15.7 us; 800 x 8192 x 1024 +
        // GeGLU, 448 tiles: 14.4 -> 11.4); up to one tile per CU the
        // deeper ring hides more latency (1632 x 2048 x 2048, 208 tiles: 12.0 against 14.3).
        else if (tiles > 256) pl.depth = 2;
    }
    if (const char* e = tuning_env("PHYAI_FP8_BIG_SPLITS")) {
        const int s = atoi(e);
        if (pl.tile == 128 && pl.cols == 128 && s >= 1 && (K % (s * 128) == 0 || (ragged && s <= 2)) && K / s >= 512 && tiles * s <= 4096) pl.splits = s;
    }
    if (const char* e = tuning_env("PHYAI_FP8_BIG_DEPTH")) {
        const int d = atoi(e);
        if (pl.tile == 128 && pl.cols == 128 && pl.splits == 1 && (d == 2 || d == 4)) pl.depth = d;
    }
    // Weights in operand order and a whole number of trips round the ring per K range: the wavefronts load their own
    // weight blocks straight into registers (PHYAI_FP8_BIG_DIRECT=0: stage them like the rest).  224 x 256 tiles: ring
    // of four, gemm_tall.hip.  128 x 128 tiles with a ring of four LDS stages and a plain epilogue: wavefronts 1 x 4 with one column
    // block each and a ring of eight.  (Not the 96 x 128 tile: its main loop gains what its longer prologue - six
    // stage-loads requested up front, at what the CU's vector-memory path passes - loses: 816 x 2560 x 2048 10.0 ->
    // 10.1 us on the earlier loop.  Up to K = 2048 the ring of eight is level with staged weights, and the ring of four of
    // two workgroups per CU up to 14 % ahead of it from 160 tiles up: 2048 x 2048 x 2048 15.5 / 13.6.)
    pl.regs = operand_w ? big_register_ring(pl, K, epilogue) : 0;
    return pl;
}

// ---- what a tile shape costs ----------------------------------------------------------------------------------------------
// Microseconds beyond what every linear pays (launches, quantizer), from the workgroups that the busiest XCD runs on its 32
// CUs: R rounds of them, x of a round each round's worth (R >= x > R - 1), S stages of 128 bytes of K.  A workgroup's life
// is prologue and epilogue plus S stages, and both depend on how many CUs are at work beside it:
//     one workgroup per CU    R round + x part + S (R round_step + x part_step)
//     two                     the same beyond one round of single workgroups; within it alone + x alone_part + S (alone_step + x alone_part_step)
// plus x S ragged where K is no multiple of 128, and the activation's arithmetic.  Least squares over 9800 linears drawn
// over M = 130 .. 13056, N = 256 .. 32768, K = 512 .. 16384 (every shape forced in turn, weight sets beyond the Infinity
// Cache): 3 - 7 % off a single time.
struct BigCost {
    double round, part, round_step, part_step, ragged, act, gated;
    double alone, alone_part, alone_step, alone_part_step;   // two per CU
};
static BigCost big_cost_of(const BigPlan& pl) {
    const bool regs = pl.regs != 0;
    switch (pl.tile) {
    case 256: return {4.59, 2.45, 1.240, 0.153, 0.258, 4.33, 1.07, 0, 0, 0, 0};
    case 224: return {3.30, 2.15, 1.161, 0.137, 0.264, 3.77, 1.25, 0, 0, 0, 0};
    case 192: return {2.30, 0.93, 0.616, 0.652, 0.102, 1.84, 0.37, 0.84, 1.06, 0.737, 0.472};
    case 96: return {-0.12, 1.56, 0.364, 0.049, 0.108, 0.79, 0, 0, 0, 0, 0};
    default: break;
    }
    if (pl.cols == 64) return {-0.52, 1.71, 0.288, 0.026, 0.062, 0.50, 0, 0, 0, 0, 0};
    if (pl.depth == 2)
        return regs ? BigCost{0.80, 1.24, 0.433, 0.440, 0, 1.28, 0, 0.08, 1.10, 0.464, 0.274} : BigCost{0.31, 1.56, 0.702, 0.211, 0.114, 1.29, 0.40, -0.34, 0.50, 0.647, 0.404};
    // (K split in two: the halves' round trip through memory)
    const double split = pl.splits > 1 ? 5.0 : 0.0;
    return regs ? BigCost{1.02 + split, 1.06, 0.356, 0.112, 0, 1.09, 0, 0, 0, 0, 0} : BigCost{0.63 + split, 1.23, 0.393, 0.095, 0.109, 1.06, 0.33, 0, 0, 0, 0};
}
// Rounds of `slots` workgroups that the busiest XCD runs of a shape, in fractions.
static double big_rounds(const BigPlan& pl, int M, int N, int K, int epilogue, int slots) {
    const bool gated = epi_is_gated(epilogue);
    double bytes;
    int busiest;
    big_takes_rows(M, N, K, big_ceil_div(M, pl.tile), big_ceil_div(gated ? N / 2 : N, gated ? pl.cols / 2 : pl.cols), slots, &bytes, &busiest);
    return (double)(busiest * pl.splits) / slots;
}
// The same for a tall tile of h x 256 rows: a round is its opening and its epilogue plus S stages, all of them longer with the
// rows.  Fitted to 2200 linears with weights in operand order (eight heights each, 2.4 % off a single time in the median); the
// height that it chooses is 0.2 % behind the best of the eight in the geometric mean.
static double tall_cost(const BigPlan& pl, int M, int N, int K, int epilogue) {
    const double S = K / 128, x = big_rounds(pl, M, N, K, epilogue, 32), R = ceil(x), h = pl.tile / 256.0;
    double act = 0;
    switch (epilogue) {
    case EPI_GEGLU_TANH: act = 2.68; break;
    case EPI_GEGLU_ERF: act = 5.21; break;
    case EPI_SWIGLU: act = 2.27; break;
    case EPI_GELU_TANH: act = 5.23; break;
    case EPI_GELU_ERF: act = 10.59; break;
    default: break;
    }
    return 1.28 + R * (1.23 + (3.05 + act) * h) + x * (0.32 - 0.72 * h) + S * (R * (0.004 + 0.933 * h) + x * (0.170 + 0.123 * h));
}
double big_cost(const BigPlan& pl, int M, int N, int K, int epilogue) {
    if (big_tall(pl)) return tall_cost(pl, M, N, K, epilogue);
    const BigCost c = big_cost_of(pl);
    const bool gated = epi_is_gated(epilogue), two = big_two_of(pl);
    const double S = (double)big_ceil_div(K, 128 * pl.splits), x = big_rounds(pl, M, N, K, epilogue, two ? 64 : 32), R = ceil(x);
    const double ragged = K % 128 != 0 ? c.ragged : 0.0, epi = gated ? c.gated : epilogue != EPI_NONE ? c.act : 0.0;
    if (!two) return R * (c.round + epi) + x * c.part + S * (R * c.round_step + x * (c.part_step + ragged));
    const double t = x <= 0.5 ? c.alone + x * c.alone_part + S * (c.alone_step + x * c.alone_part_step)
                            : R * c.round + x * c.part + S * (R * c.round_step + x * c.part_step);
    return t + (x > 1.0 ? x : 1.0) * (S * ragged + epi);
}

// The same for 192 x 128 tiles as far as the choice between them and tall ones goes, weights in operand order: activations told
// apart, and a shorter stage beside a longer start than the account over both layouts gives them.  Fitted to the difference of
// the two in 663 linears: 4.8 % off (9.1 % by the costs).
static double beside_tall_192(const BigPlan& pl, int M, int N, int K, int epilogue) {
    const double x = big_rounds(pl, M, N, K, epilogue, 64), rounds = x > 1.0 ? x : 1.0;
    double act = 0;
    switch (epilogue) {
    case EPI_GEGLU_TANH: act = -0.42; break;
    case EPI_GEGLU_ERF: act = 1.29; break;
    case EPI_SWIGLU: act = -0.22; break;
    case EPI_GELU_TANH: act = 1.54; break;
    case EPI_GELU_ERF: act = 5.86; break;
    default: break;
    }
    return big_cost(pl, M, N, K, EPI_NONE) + 1.62 + rounds * (act - 0.158 * (K / 128));
}

// The cheapest unsplit tile shape by that account, `rule` (big_plan's choice, or no tile at all) where nothing is 8 % ahead
// of it, `shared` being what all of them pay.  All unsplit shapes add in the same order of K.
BigPlan big_plan_by_cost(int M, int N, int K, int epilogue, bool operand_w, const BigPlan& rule, double shared, double* cost) {
    static const BigPlan shapes[] = {{256, 256, 1, 0, 2, 0}, {224, 256, 1, 0, 2, 0}, {192, 128, 1, 0, 2, 0}, {128, 128, 1, 0, 4, 0},
                                     {128, 128, 1, 0, 2, 0}, {128, 64, 1, 0, 4, 0}, {96, 128, 1, 0, 4, 0}};
    BigPlan best = rule;
    const double of_rule = rule.tile ? big_cost(rule, M, N, K, epilogue) + shared : 1e30;
    double lowest = 0.92 * of_rule;
    *cost = of_rule;
    for (BigPlan pl : shapes) {
        if (epi_is_gated(epilogue) && (pl.cols == 64 || pl.tile == 96)) continue;
        pl.regs = operand_w ? big_register_ring(pl, K, epilogue) : 0;
        const double t = big_cost(pl, M, N, K, epilogue) + shared;
        if (t < lowest) { *cost = lowest = t; best = pl; }
    }
    // Tall tiles where they are ahead of that (by 4 % below 60 us, where the costs are less sure): 325 of 1200 drawn linears,
    // 1.09 times as fast as the best staged shape in the geometric mean, more than 2 % slower in 10.  Against 192 x 128 tiles `beside_tall_192` is asked as well, with
    // 5.5 % in favour of the tall ones.  Cards differ there: on one, 68 of 1300 such linears were 3 % slower in tall tiles and more, 40 of
    // these against 192 x 128 (8689 x 11840 x 896 + GELU (tanh) 131.4 / 113.2 us, 5398 x 17856 x 768 + GeGLU 103.8 / 93.1), and
    // with 2 % in favour 24 of 900 others went back, 1.084 times as fast.  On another the same two are 128.7 / 122.6 and 94.8 / 90.9,
    // and of 52 that 2 % send back 6 are more than 2 % slower in tall tiles, 19 more than 2 % faster (2307 x 26336 x 640 + SwiGLU
    // 61.0 / 65.8); of the 23 that 5.5 % send back it is 5 and 6, level in the mean.
    // (The rest, 128 x 128 tiles two to a CU against a tall grid of less than a round, is a toss-up: asked to be 7 % ahead, in
    // the 900 as much is lost as won.)
    if (operand_w && K % 128 == 0 && big_registers_allowed()) {
        const bool against_192 = best.tile == 192 && best.cols == 128;
        lowest = (big_tall(best) || *cost - shared >= 60.0 ? 1.0 : 0.96) * *cost;
        if (against_192) {
            const double limit = 1.055 * (beside_tall_192(best, M, N, K, epilogue) + shared);
            lowest = limit < lowest ? limit : lowest;
        }
        for (int rows = 144; rows <= 256; rows += 16) {
            const BigPlan pl = {rows, 256, 1, 0, 2, 4};
            const double t = big_cost(pl, M, N, K, epilogue) + shared;
            if (t < lowest) { *cost = lowest = t; best = pl; }
        }
    }
    best.tiles = big_tiles(M, N, epilogue, best.tile, best.cols);
    return best;
}

size_t big_partial_bytes(int M, int N, int epilogue, const BigPlan& pl) {
    if (pl.splits <= 1) return 0;
    const int bn = pl.cols;
    return (size_t)big_tiles(M, N, epilogue, pl.tile, bn) * pl.splits * pl.tile * bn * sizeof(float);
}

template <int TM, int TN, int DEPTH, int EPI, int WGM = 2, int WGN = 2, int WMODE = 0, bool RAGGED = false>
static void big_launch(BigArgs a, const GemmProblem& g, int splits, hipStream_t st) {
    const bool gated = epi_is_gated(EPI);
    constexpr int BM = WGM * 32 * TM, BN = WGN * 32 * TN;
    const int bn_eff = gated ? BN / 2 : BN;
    a.n_tiles = big_ceil_div(gated ? g.N / 2 : g.N, bn_eff);
    a.m_tiles = big_ceil_div(g.M, BM);
    // which operand the XCDs share
    double chosen_bytes;
    int busiest;
    a.by_rows = big_takes_rows(g.M, g.N, g.K, a.m_tiles, a.n_tiles, 32 * (big_two_per_cu(TM, TN, DEPTH, WMODE) ? 2 : 1), &chosen_bytes, &busiest);
    if (const char* e = tuning_env("PHYAI_FP8_BY_ROWS")) a.by_rows = atoi(e) != 0;
    a.band = big_band(a.by_rows, a.m_tiles, BM, g.K);
    const int outer = a.by_rows ? a.n_tiles : a.m_tiles, inner = a.by_rows ? a.m_tiles : a.n_tiles;
    dim3 grid(big_grid_ids(outer, inner, a.band), 1, splits);
    // Split along K: an XCD per K range (see the kernel).  Every XCD then fetches 1 / splits of the
    // activation codes instead of all of them, and the weights of its tile columns once.  Taken when
    // that is the smaller estimate and the tile columns divide evenly among the 8 / splits groups
    // (816 x 2048 x 16384, K split in two: 155 -> 87 MB fetched, 36.8 -> 35.3 us row-major, 35.4 -> 34.2 in operand order).
    if (splits == 2 || splits == 4 || splits == 8) {
        const int groups = 8 / splits, cols = big_ceil_div(a.n_tiles, groups);
        const double by_k = (double)g.M * g.K * 8.0 / splits + (double)g.N * g.K;
        bool xcd_k = cols * groups == a.n_tiles && by_k < 0.8 * chosen_bytes;
        if (const char* e = tuning_env("PHYAI_FP8_XCD_SPLIT")) xcd_k = atoi(e) != 0;
        if (xcd_k) {
            a.by_rows = 2;
            a.band = splits;
            grid = dim3(8 * cols * a.m_tiles, 1, 1);
        }
    }
#define PHYAI_BIG_ARGS a.a, a.b, a.K, a.M, a.N, a.m_tiles, big_order(a.band, a.by_rows, a.operand_w, a.a_scale_scalar, g.xq_padded), a.k_per_split, \
                       a.a_scale, a.b_scale, a.bias, a.out, a.ldo, a.partials, a.counters, a.res
    if (splits > 1) {
        // (K splits: 128 x 128 tiles with a ring of four, staged or with weights in registers.  The 256 x 256 tile is
        // not built with them: its 256 accumulators leave the gather no registers, and a kernel that spills has
        // vector-memory instructions of the compiler's among the copies that the waits count by hand.)
        if constexpr ((TM == TN && TM == 2 && DEPTH == 4) || (WMODE == 2 && TN == 1 && !big_two_per_cu(TM, TN, DEPTH, WMODE)))
            hipLaunchKernelGGL((gemm_fp8_big_kernel<TM, TN, DEPTH, EPI, true, WGM, WGN, WMODE, RAGGED>), grid, dim3(256), 0, st, PHYAI_BIG_ARGS);
    } else {
        hipLaunchKernelGGL((gemm_fp8_big_kernel<TM, TN, DEPTH, EPI, false, WGM, WGN, WMODE, RAGGED>), grid, dim3(256), 0, st, PHYAI_BIG_ARGS);
    }
#undef PHYAI_BIG_ARGS
}

template <int TM, int TN, int DEPTH, int WGM = 2, int WGN = 2, int WMODE = 0, bool RAGGED = false>
static int big_launch_epi(const BigArgs& a, const GemmProblem& g, int splits, hipStream_t st) {
    switch (g.epilogue) {
    case EPI_NONE: big_launch<TM, TN, DEPTH, EPI_NONE, WGM, WGN, WMODE, RAGGED>(a, g, splits, st); return 0;
    case EPI_GEGLU_TANH: big_launch<TM, TN, DEPTH, EPI_GEGLU_TANH, WGM, WGN, WMODE, RAGGED>(a, g, splits, st); return 0;
    case EPI_GEGLU_ERF: big_launch<TM, TN, DEPTH, EPI_GEGLU_ERF, WGM, WGN, WMODE, RAGGED>(a, g, splits, st); return 0;
    case EPI_SWIGLU: big_launch<TM, TN, DEPTH, EPI_SWIGLU, WGM, WGN, WMODE, RAGGED>(a, g, splits, st); return 0;
    case EPI_GELU_TANH: big_launch<TM, TN, DEPTH, EPI_GELU_TANH, WGM, WGN, WMODE, RAGGED>(a, g, splits, st); return 0;
    case EPI_GELU_ERF: big_launch<TM, TN, DEPTH, EPI_GELU_ERF, WGM, WGN, WMODE, RAGGED>(a, g, splits, st); return 0;
    default: return -2;
    }
}

// (tiles with one column block per wavefront cannot hold a gate / up pair: plain epilogues only)
template <int TM, int TN, int DEPTH, int WGM = 2, int WGN = 2, int WMODE = 0, bool RAGGED = false>
static int big_launch_plain(const BigArgs& a, const GemmProblem& g, int splits, hipStream_t st) {
    switch (g.epilogue) {
    case EPI_NONE: big_launch<TM, TN, DEPTH, EPI_NONE, WGM, WGN, WMODE, RAGGED>(a, g, splits, st); return 0;
    case EPI_GELU_TANH: big_launch<TM, TN, DEPTH, EPI_GELU_TANH, WGM, WGN, WMODE, RAGGED>(a, g, splits, st); return 0;
    case EPI_GELU_ERF: big_launch<TM, TN, DEPTH, EPI_GELU_ERF, WGM, WGN, WMODE, RAGGED>(a, g, splits, st); return 0;
    default: return -2;
    }
}

// The same tile shape for row-major weights (or operand order gathered row by row) and for weights staged in
// operand order as they lie.
template <int TM, int TN, int DEPTH, int WGM = 2, int WGN = 2>
static int big_launch_layout(const BigArgs& a, const GemmProblem& g, int splits, hipStream_t st) {
    if (g.K % BIG_BK != 0) return big_launch_epi<TM, TN, DEPTH, WGM, WGN, 0, true>(a, g, splits, st);
    if (a.operand_w && !tuning_env("PHYAI_FP8_BIG_GATHER")) return big_launch_epi<TM, TN, DEPTH, WGM, WGN, 1>(a, g, splits, st);
    return big_launch_epi<TM, TN, DEPTH, WGM, WGN, 0>(a, g, splits, st);
}

int launch_set_stamp_sink_big(unsigned long long* buf, unsigned int records) {
#ifdef PHYAI_FP8_STAMPS
    const StampSink s = {buf, records};
    return hipMemcpyToSymbol(HIP_SYMBOL(g_big_stamps), &s, sizeof(s)) == hipSuccess ? 0 : -4;
#else
    (void)buf; (void)records;
    return -2;
#endif
}

int launch_gemm_big(const GemmProblem& g, const BigPlan& pl, hipStream_t st) {
    // the epilogue writes 16 bytes per lane (the caller chooses this kernel only for such outputs)
    if (g.ldo % 8 != 0 || (reinterpret_cast<uintptr_t>(g.out) & 15) != 0) return -2;
    BigArgs a;
    a.a = g.xq; a.b = g.w; a.a_scale = g.x_scale; a.b_scale = g.w_scale; a.bias = g.bias;
    a.out = g.out; a.ldo = g.ldo; a.M = g.M; a.N = g.N; a.K = g.K;
    a.a_scale_scalar = g.x_scale_is_scalar;
    a.res = residual_of(g);
    a.operand_w = g.weight_layout != W_ROW_MAJOR;
    // (K that is no multiple of 128: the ranges end on whole K steps, the last one is the shorter)
    a.k_per_split = g.K % BIG_BK == 0 ? g.K / pl.splits : big_ceil_div(big_ceil_div(g.K, BIG_BK), pl.splits) * BIG_BK;
    a.counters = static_cast<int*>(g.workspace);
    a.partials = g.workspace ? reinterpret_cast<float*>(static_cast<uint8_t*>(g.workspace) + kGemmHeaderBytes) : nullptr;
    if (pl.splits > 1 && (g.workspace == nullptr ||
                          g.workspace_bytes < kGemmHeaderBytes + big_partial_bytes(g.M, g.N, g.epilogue, pl)))
        return -3;
    if (big_tall(pl)) {
        if (pl.splits != 1) return -2;
        // (rows of output too far apart for it: another shape, which adds alike)
        return tall_reaches(g) ? launch_gemm_tall(g, pl.tile, st) : big_launch_layout<4, 4, 2>(a, g, 1, st);
    }
    if (pl.tile == 256) return pl.splits == 1 ? big_launch_layout<4, 4, 2>(a, g, 1, st) : -2;
    if (pl.regs != 0 && !a.operand_w) return -2;
    if (pl.tile == 224) {
        if (pl.splits != 1) return -2;
        return big_launch_layout<7, 2, 2, 1, 4>(a, g, 1, st);
    }
    if (pl.tile == 192 && pl.splits == 1) return big_launch_layout<3, 2, 2>(a, g, 1, st);
    if (pl.tile == 96) {   // 96 rows x 128 columns: wavefronts 1 x 4, three row blocks each; plain epilogues
        if (pl.splits != 1) return -2;
        if (g.K % BIG_BK != 0) return big_launch_plain<3, 1, 4, 1, 4, 0, true>(a, g, 1, st);
        return a.operand_w ? big_launch_plain<3, 1, 4, 1, 4, 1>(a, g, 1, st) : big_launch_plain<3, 1, 4, 1, 4, 0>(a, g, 1, st);
    }
    if (pl.tile == 128 && pl.cols == 64) {
        if (pl.splits != 1) return -2;
        if (g.K % BIG_BK != 0) return big_launch_plain<2, 1, 4, 2, 2, 0, true>(a, g, 1, st);
        return a.operand_w ? big_launch_plain<2, 1, 4, 2, 2, 1>(a, g, 1, st) : big_launch_plain<2, 1, 4, 2, 2, 0>(a, g, 1, st);
    }
    if (pl.tile == 128 && pl.depth == 4 && pl.regs == 8) return big_launch_plain<4, 1, 8, 1, 4, 2>(a, g, pl.splits, st);
    if (pl.tile == 128 && pl.depth == 2 && pl.regs == 4 && pl.splits == 1) return big_launch_plain<4, 1, 4, 1, 4, 2>(a, g, 1, st);
    if (pl.tile == 128 && pl.depth == 4) return big_launch_layout<2, 2, 4>(a, g, pl.splits, st);
    if (pl.tile == 128 && pl.splits == 1) return big_launch_layout<2, 2, 2>(a, g, 1, st);
    return -2;
}

}  // namespace phyai
