// gemm.hip -- grouped bf16 MFMA GEMMs over expert segments (gfx950).
//
// Replaces the reference's per-expert cuBLAS loops (tmt-cuda/src/moe.cu:431-436
// forward, :533-539 backward; wrappers tmt-cuda/src/linalg.cu:9-41) and the
// gather kernel (moe.cu:127-140): one launch covers all experts, tiles are
// found from the device-side offset table (no host sync, no 128-row padding),
// and the forward token gather is folded into the operand addressing.
//
// Tile: 256 x 256 outputs per 256-thread workgroup (one workgroup per CU),
// 4 waves in 2 x 2, each wave 128 x 128 = 4 x 4 v_mfma_f32_32x32x16_bf16
// tiles (256 fp32 accumulators per lane, held in AGPRs); 128 x 128 (64 x 64
// per wave) where the large tiles would leave CUs idle (gemm_tile).
//
// Operand staging: direct global -> LDS loads (global_load_lds_dwordx4, the
// data never passes through VGPRs). Two ring layouts:
//   * split rings (the activation GEMMs on 256 x 256 tiles): K = 64 tiles,
//     the A operand in a ring of 3 slots and B in a ring of 2 (32 KiB each,
//     160 KiB in all). Iteration kt loads B(kt+1) and A(kt+2). K = 64 makes
//     each K-contiguous row a full 128-byte segment: the CU accepts one
//     1 KiB load per 16 cycles when every row segment of the load is >= 128
//     bytes, but only one per 29-34 cycles with 64-byte segments from L2 or
//     HBM, so with K = 32 stages the loads alone filled the CU's load path;
//   * one ring of NST stages, issued NST - 1 tiles ahead (weight-gradient
//     GEMMs and 128 x 128 tiles; see Ring).
//   * K-contiguous operands (activations in every GEMM, weights in the
//     forward) land as [256 rows][32] bf16, 16-byte chunks XOR-swizzled by
//     (row >> 2) & 3, and are read with ds_read_b128.
//   * Row-contiguous operands (weights read as [K][N] in the backward, and
//     the token-major operands of the weight-gradient GEMMs) land as
//     [32 k][256] bf16, chunks swizzled by 4 * (k & 3), and are read with the
//     gfx950 transposing ds_read_b64_tr_b16: inside each 16-lane group, lane
//     r points at row k0 + r/4, columns c0 + 4(r%4) .. +3, and lane i receives
//     column c0 + i of rows k0 .. k0+3 -- a K-contiguous MFMA fragment.
// The loads are issued from inline asm with explicit vmcnt accounting: the
// compiler would otherwise wait for every outstanding LDS-DMA load before
// each LDS read. Masked rows/columns are clamped to valid addresses (they
// only feed outputs that are not stored), except the reduction tail of the
// weight-gradient GEMMs, which is zeroed in LDS.
//
// Epilogue: accumulators go through LDS (fp32, 16-byte chunks swizzled by
// row) so every global store is a 16-byte vector and each output row is
// written as one contiguous 256-byte (bf16) or 512-byte (fp32) run; the
// stores (and GEMM_DACT's pre-activation reads) are non-temporal.
#include <algorithm>
#include <cmath>

#include "device_util.hpp"
#include "moe_internal.hpp"

namespace tmt {
namespace {

constexpr int kLarge = kGemmTileRows;  // tile of the large-problem kernels

// Tile geometry: TILE x TILE outputs (256 or 128) on 4 waves in 2 x 2. BK_ is
// the K depth of one LDS stage (32 or 64), NST the number of stages in the
// ring.
template <int BK_, int NST, int TILE>
struct Geo {
    static constexpr int BM = TILE, BN = TILE;
    static constexpr int BK = BK_;
    static constexpr int NW = 4, NT = 64 * NW;         // waves, threads
    static constexpr int WTM = BM / 2, MI = WTM / 32;  // wave tile rows
    static constexpr int WTN = BN / 2, NJ = WTN / 32;  // wave tile columns
    static constexpr int EPR = 64;                     // epilogue rows per wave and pass
    static constexpr int KCH = BK / 8;                 // 16-byte chunks per K-contiguous row
    static constexpr int OPND_A = BM * BK;             // bf16 elements of the A tile
    static constexpr int OPND_B = BN * BK;             // bf16 elements of the B tile
    static constexpr int STAGE = OPND_A + OPND_B;      // A then B
    static constexpr int DMA_A = OPND_A * 2 / 1024 / NW;  // 1 KiB wave loads per wave, A tile
    static constexpr int DMA_B = OPND_B * 2 / 1024 / NW;  // ... B tile
    static constexpr int DMA_PER_TILE = DMA_A + DMA_B;
    static constexpr int KC_ROWS = 1024 / (2 * BK);    // K-contiguous rows per wave load
    static constexpr int STEPS = BK / 16;              // MFMA k16 steps per stage
    static constexpr int WGS = TILE == 256 || (BK == 64 && NST > 2) ? 1 : 2;  // workgroups per CU
    // the epilogue's fp32 staging ([EPR][WTN] per wave); the kernel sizes the
    // ring (single or split) and checks the total
    static constexpr int EPI = NW * EPR * WTN * 4;
    // K-contiguous rows: 16-byte chunk swizzle making 16 consecutive rows (the
    // lanes one ds_read_b128 cycle serves from the 64 banks = 256 bytes) hit
    // distinct banks: rows r and r + 4j share (r & 3) * 64 bytes of bank offset
    // (BK 32: 64-byte rows), so the chunk is XORed with (r >> 2) & 3; with
    // 128-byte rows (BK 64) rows r and r + 2j pair up, XOR with (r >> 1) & 7.
    static __device__ __forceinline__ int kc_swz(int r) {
        return KCH == 4 ? ((r >> 2) & 3) : ((r >> 1) & 7);
    }
    // Row-contiguous [BK][256 or 128] tiles (rows of 512 / 256 bytes, all
    // starting at bank 0): the 32 lanes of one ds_read_b64_tr_b16 cycle read
    // 4 k rows x 4 chunks; XOR with 4 * (k & 3) spreads them over 16 distinct
    // chunks (256 bytes).
    static __device__ __forceinline__ int mc_swz(int k) { return 4 * (k & 3); }
};

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

template <int KIND> struct Traits;
// C[slot][n] = X[perm[slot]] . W_up[e][n]              A: K-contig (gathered), B: K-contig
template <> struct Traits<GEMM_UP> {
    static constexpr bool group_k = false, a_kc = true, b_kc = true, gather = true, b_fp4 = false;
};
// C[slot][n] = A[slot] . W_down[e][n]
template <> struct Traits<GEMM_DOWN> {
    static constexpr bool group_k = false, a_kc = true, b_kc = true, gather = false, b_fp4 = false;
};
// C[slot][n] = (dO[slot] . W_down[e][:, n]) * silu'(U)  B: [K][N]; silu'(U) as the
// up GEMM wrote it (p.u)
template <> struct Traits<GEMM_DACT> {
    static constexpr bool group_k = false, a_kc = true, b_kc = false, gather = false, b_fp4 = false;
};
// C[slot][n] = dU[slot] . W_up[e][:, n]                 B: [K][N]
template <> struct Traits<GEMM_DX> {
    static constexpr bool group_k = false, a_kc = true, b_kc = false, gather = false, b_fp4 = false;
};
// dW_down[e][m][n] = sum_slot dO[slot][m] * A[slot][n]
template <> struct Traits<GEMM_DW_DOWN> {
    static constexpr bool group_k = true, a_kc = false, b_kc = false, b_fp4 = false;
};
// dW_up[e][m][n] = sum_slot dU[slot][m] * Xg[slot][n]   (Xg: X gathered to slot order)
template <> struct Traits<GEMM_DW_UP> {
    static constexpr bool group_k = true, a_kc = false, b_kc = false, b_fp4 = false;
};

// MXFP4 variants: same as GEMM_UP / GEMM_DOWN, B = e2m1 weights + e8m0 scales.
template <> struct Traits<GEMM_UP_FP4> {
    static constexpr bool group_k = false, a_kc = true, b_kc = true, gather = true, b_fp4 = true;
};
template <> struct Traits<GEMM_DOWN_FP4> {
    static constexpr bool group_k = false, a_kc = true, b_kc = true, gather = false, b_fp4 = true;
};

// 8 e2m1 codes (low nibble first) sharing one e8m0 scale -> 8 bf16, with the
// gfx950 scaled conversion (two codes per instruction). e2m1 values have at
// most two significant bits, so every product with 2^(scale - 127) inside
// bf16's exponent range is exact; the scale byte becomes the fp32 2^(s-127)
// (s = 0 is the subnormal 2^-127).
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint4 dequant8(uint32_t w, uint32_t scale) {
    const float sc = __uint_as_float(scale == 0 ? 0x00400000u : (scale << 23));
    return make_uint4(__builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, sc, 0)),
                      __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, sc, 1)),
                      __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, sc, 2)),
                      __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, sc, 3)));
}

// Streaming 16-byte accesses for the epilogue: outputs are written once
// (st16_nt) and read by a later kernel, so they should not displace the
// operand tiles the other workgroups are reusing from L2.
typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ uint4 ld16_nt(const uint16_t* p) {
    const u32x4_t v = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(p));
    return make_uint4(v[0], v[1], v[2], v[3]);
}

__device__ __forceinline__ uint32_t lds_addr(const void* p) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char*)p;
}

// One wave-wide 16-byte-per-lane load from global memory into LDS at
// lds_base + 16 * lane (lds_base must be wave-uniform).
// M0 is written here and declared clobbered (clang warns that it is reserved).
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void dma16(const void* g, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(g), "s"(lds_base) : "m0");
}
#pragma clang diagnostic pop
template <int N>
__device__ __forceinline__ void wait_vm() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N));
}

// Order of a launch's tiles. The hardware hands workgroup b to XCD b % 8, and
// the list of (M tile, N tile) is dealt to the XCDs in pieces of consecutive
// tiles, so that the tiles an XCD runs at a time are neighbours and its L2
// serves each operand slice to several workgroups. The list goes by blocks of `rows` M
// tiles, column by column inside a block, so that 32 (16) consecutive tiles
// cover 4 x 8 (2 x 8) tiles where there are 8 columns or more.
__device__ __forceinline__ void list_tile(int j, int mtiles, int ntn, int rows, int& mt, int& nt) {
    const int blk = j / (rows * ntn), rem = j - blk * (rows * ntn);
    const int in = min(rows, mtiles - blk * rows);  // the last block may be shorter
    nt = rem / in;
    mt = blk * rows + (rem - nt * in);
}
// M tiles per block of the activation GEMMs' list.
__device__ __forceinline__ int list_rows(int ntn) { return ntn >= 8 ? 4 : 32 / ntn; }

// Split-K of the last round (GEMM_DOWN / GEMM_DX, tiles 256 x 256, one
// workgroup per CU). Of the launch's tiles, F (a multiple of the W resident
// workgroups) fill whole rounds. The R tiles left would run as one short
// round on R CUs while the rest idle, so each is cut into S parts along K
// (S = W / R, at least 8 k tiles a part). Part q of tail tile j is workgroup
// F + j*S + q, after the whole rounds in launch order; it writes an fp32
// partial tile, and split_fixup_kernel adds a tile's S partials in part order
// and stores the bf16 result.
struct SplitPlan {
    int F = 0, R = 0, S = 1, chunk = 0;  // chunk: reduction length of a part
};
__device__ __forceinline__ int act_mtiles(const GemmParams& p) {
    int mt = 0;
    for (int ee = 0; ee < p.E; ++ee) mt += (p.offsets[ee + 1] - p.offsets[ee] + kLarge - 1) / kLarge;
    return mt;
}
template <int BK>
__device__ __forceinline__ SplitPlan split_plan(const GemmParams& p, int tiles) {
    SplitPlan sp;
    const int W = p.resident;
    if (p.part == nullptr || W <= 0 || W % 256 != 0) return sp;
    sp.F = tiles / W * W;
    sp.R = tiles - sp.F;
    const int nk = p.K / BK;
    int S = sp.R > 0 ? W / sp.R : 1;
    S = min(S, nk / 8);
    if (S < 2) return SplitPlan{};
    sp.S = S;
    sp.chunk = ((nk + S - 1) / S) * BK;
    return sp;
}
// Expert segment of activation M tile mt (256 rows per tile): expert, first
// slot, rows (e < 0: none).
__device__ __forceinline__ void act_tile(const GemmParams& p, int mt, int& e, int& row0, int& rows) {
    e = -1;
    int t0 = 0;
    for (int ee = 0; ee < p.E; ++ee) {
        const int beg = p.offsets[ee], end = p.offsets[ee + 1];
        const int tiles = (end - beg + kLarge - 1) / kLarge;
        if (mt < t0 + tiles) {
            e = ee;
            row0 = beg + (mt - t0) * kLarge;
            rows = min(kLarge, end - row0);
            return;
        }
        t0 += tiles;
    }
}

// Split rings (A in 3 slots, B in 2) of K = 64: the activation GEMMs on
// 256 x 256 tiles. Those kernels are persistent (every tile of a launch has
// the same K, so a static schedule stays balanced): one workgroup per CU
// walks the tiles vb = blockIdx.x, blockIdx.x + gridDim.x, ... . A tile's
// first operand loads then go out while the previous tile's epilogue stores
// drain, and the per-workgroup launch and set-up cost is paid once per CU
// instead of once per tile. vb keeps the launch-order meaning of blockIdx.x
// (gridDim.x is a multiple of 8 whenever it is below the tile count, so vb
// runs on XCD vb % 8 as the tile map assumes).
template <int KIND, int TILE>
constexpr bool split_ring() {
    return TILE == 256 && !Traits<KIND>::group_k;
}

// MXFP4 B operand (split rings of K = 64 only): per stage 256 rows x 32 bytes
// of codes, then one 1 KiB copy per wave of the tile's row scales (lanes 0-15
// load the first 32-block's, lanes 16-31 the second's).
constexpr int kFp4Codes = 256 * 32, kFp4Scales = 4 * 1024;
// bf16 elements of a B tile's slot.
template <int KIND, int BK, int NST, int TILE>
constexpr int b_slot_elems() {
    return Traits<KIND>::b_fp4 ? (kFp4Codes + kFp4Scales) / 2 : Geo<BK, NST, TILE>::OPND_B;
}
// LDS of one workgroup: the operand ring, or the epilogue's fp32 staging if
// larger.
template <int KIND, int BK, int NST, int TILE>
constexpr int gemm_lds_bytes() {
    using Gm = Geo<BK, NST, TILE>;
    constexpr int ring = split_ring<KIND, TILE>() ? (NST * Gm::OPND_A + (NST - 1) * b_slot_elems<KIND, BK, NST, TILE>()) * 2
                                                  : NST * Gm::STAGE * 2;
    return ring > Gm::EPI ? ring : Gm::EPI;
}

// One output tile (or split-K part) of the grouped GEMM: launch-order block
// index vb; returns without touching memory when vb maps to no tile. et: the
// experts' activation tiles (unused by the weight-gradient kinds). lds_raw:
// the workgroup's gemm_lds_bytes() of LDS, declared by the kernel (measured:
// DOWN and DX about 1% faster at c3 than with the array declared here).
template <int KIND, bool DUAL, int BK_, int NST, int TILE>
__device__ __forceinline__ void grouped_gemm_tile(const GemmParams& p, const int vb, const ExpertTiles& et,
                                                  uint4* lds_raw) {
    using Tr = Traits<KIND>;
    using Gm = Geo<BK_, NST, TILE>;
    constexpr int BM = Gm::BM;
    constexpr int BK = Gm::BK, BN = Gm::BN, WTN = Gm::WTN, NJ = Gm::NJ;
    constexpr int WTM = Gm::WTM, MI = Gm::MI, NT = Gm::NT, EPR = Gm::EPR;
    constexpr int OPND_A = Gm::OPND_A, STAGE = Gm::STAGE;
    constexpr int DMA_A = Gm::DMA_A, DMA_B = Gm::DMA_B, DMA_PER_TILE = Gm::DMA_PER_TILE;
    constexpr bool kSplit = split_ring<KIND, TILE>();
    static_assert(!kSplit || (NST == 3 && BK == 64), "split rings: 3 A slots and 2 B slots of K = 64");
    static_assert(!Tr::b_fp4 || kSplit, "MXFP4 tiles: split rings");
    // split rings: B slot size (bf16 elements) and wave loads per B tile
    constexpr int B_SLOT = b_slot_elems<KIND, BK_, NST, TILE>();
    constexpr int DMA_BT = Tr::b_fp4 ? kFp4Codes / 1024 / 4 + 1 : DMA_B;
    constexpr int KCH = Gm::KCH, KC_ROWS = Gm::KC_ROWS, STEPS = Gm::STEPS;
    static_assert(gemm_lds_bytes<KIND, BK_, NST, TILE>() * Gm::WGS <= 160 * 1024, "LDS ring too large");
    uint16_t* lds = reinterpret_cast<uint16_t*>(lds_raw);

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform (SGPR)
    // the wave's first row and column in the tile
    const int wrow = (wave >> 1) * WTM, wcol = (wave & 1) * WTN;
    const int ntn = (p.N + BN - 1) / BN;

    // ---- tile coordinates -------------------------------------------------
    int e = -1, mt = 0, nt = 0;
    int row0 = 0, rows = 0;   // activation GEMMs: slot range of this tile
    int kbeg = 0, kend = 0;   // reduction range (slots for dW GEMMs)
    int mlim = 0;             // valid output rows in this tile
    constexpr bool kSplitK = (KIND == GEMM_DOWN || KIND == GEMM_DX) && BM == 256;
    int part_unit = -1;  // split-K tail: index of this workgroup's partial tile
    if constexpr (!Tr::group_k) {
        kbeg = 0;
        kend = p.K;
        const int tiles = et.total * ntn;
        SplitPlan sp;
        if constexpr (kSplitK) {
            if (p.part != nullptr) sp = split_plan<BK>(p, tiles);
        }
        int j;
        if (sp.S >= 2 && vb >= sp.F) {
            const int u = vb - sp.F;
            if (u >= sp.R * sp.S) return;
            j = u / sp.S;
            const int q = u - j * sp.S;
            j += sp.F;
            kbeg = q * sp.chunk;
            kend = min(p.K, kbeg + sp.chunk);
            part_unit = u;
        } else {
            // Whole rounds of 256: workgroups 8i + x with i in [32t, 32t + 32)
            // are co-resident on XCD x and take 32 consecutive tiles; all
            // XCDs are near each other in the list, so they also share the
            // last-level cache. Where few rounds run, what is left of the last
            // one is cut into one run per XCD, so that every XCD gets the same
            // number of tiles (eleven columns, 715 tiles: UP 121.3 us, dealt
            // as another round 122.6; after 32 rounds the deal keeps the
            // neighbours together: UP at 8304 tiles 1244 against 1248 us).
            // (In fixed groups of 4 x 8 tiles, N = 2752's eleven
            // columns gave every second XCD 12 tiles for the others' 32: UP
            // and DACT at 15 K slots, K = 1024 took 150 and 138 us against
            // 122 and 119.)
            const int n = sp.S >= 2 ? sp.F : tiles, whole = n >= 8 * 256 ? (n + 255) & ~255 : n & ~255;
            const int per = (n - whole + 7) / 8, i = (vb - whole) >> 3;
            j = vb < whole ? (((vb >> 8) << 3) + (vb & 7)) * 32 + ((vb >> 3) & 31) : whole + (vb & 7) * per + i;
            if (j >= n || (vb >= whole && i >= per)) return;
        }
        list_tile(j, et.total, ntn, list_rows(ntn), mt, nt);
        if (!expert_tile<BM>(et, mt, e, row0, rows)) return;  // beyond the last tile of the last expert
        mlim = rows;
    } else {
        // A group's work is proportional to its expert's count, and groups
        // come in descending-count order. With G % 8 as the XCD, an expert
        // whose groups fill half of the XCDs sends every following expert to
        // the same halves in turn (c3: 74K against 57K slots per XCD).
        //  * 128 x 128 tiles (two workgroups per CU): round r hands its 8
        //    groups of 32 tiles to the XCDs in snake order (reversed on odd
        //    rounds), which keeps every XCD's sum of counts near the mean;
        //  * 256 x 256 tiles (one per CU): groups of 16 tiles, two per XCD
        //    and round, paired heaviest with lightest (XCD x runs groups
        //    16r + x and 16r + 15 - x). With 32-tile groups the XCD holding
        //    the heaviest expert's group could not be balanced.
        // The list runs expert by expert (descending count), in groups of
        // GSZ; a last round that is not full is cut into one run per XCD.
        constexpr int GSZ = BN == 256 ? 16 : 32;
        const int rnd = vb >> 8, xcd = vb & 7, sub = (vb >> 3) & 31;
        const int Gs = GSZ == 16 ? 16 * rnd + (sub < 16 ? xcd : 15 - xcd) : 8 * rnd + ((rnd & 1) ? 7 - xcd : xcd);
        const int ntm = (p.M + BM - 1) / BM;
        const int n = p.E * ntm * ntn, rest = n - (vb & ~255);  // tiles from this round on
        int j = Gs * GSZ + (sub & (GSZ - 1));
        if (rest < 256) {
            const int per = (rest + 7) / 8;
            if (sub >= per) return;
            j = (vb & ~255) + xcd * per + sub;
        }
        if (j >= n) return;
        const int ei = j / (ntm * ntn);
        list_tile(j - ei * (ntm * ntn), ntm, ntn, GSZ / min(ntn, 8), mt, nt);
        e = p.order[ei];
        kbeg = p.offsets[e];
        kend = p.offsets[e + 1];
        // the outputs may be narrower than the operands' padded widths (by
        // less than 64, so every tile keeps a row and a column)
        mlim = min(BM, p.m_out - mt * BM);
    }
    const int col0 = nt * BN;                // the tile's first output column
    const int nlim = min(BN, (Tr::group_k ? p.n_out : p.N) - col0);  // valid output columns in this tile
    const int nk = (kend - kbeg + BK - 1) / BK;

    // ---- DMA addressing -----------------------------------------------------
    // K-contiguous tile: wave load q covers rows KC_ROWS*q .. +KC_ROWS-1;
    // lane -> row KC_ROWS*q + lane/KCH, physical chunk lane%KCH, logical chunk
    // (lane%KCH) ^ kc_swz(row). Row-contiguous tile of C chunks per k row
    // (32 for 256 columns, 16 for 128): wave load q covers k rows
    // (64/C)q .. ; lane -> k = (64/C)q + lane/C, physical chunk lane%C,
    // logical chunk (lane%C) ^ mc_swz(k).
    // K-contiguous operands keep one source pointer per wave load; row-
    // contiguous ones keep a column pointer and the lane's k row, clamped to
    // the last valid reduction index when issued (the tail is zeroed in LDS).
    const uint16_t* a_ptr[DMA_A];
    const uint16_t* b_ptr[DMA_B];
    int a_k[DMA_A], b_k[DMA_B];
#pragma unroll
    for (int i = 0; i < DMA_A; ++i) {
        const int q = wave * DMA_A + i;
        if constexpr (Tr::a_kc) {
            const int r = KC_ROWS * q + lane / KCH;
            const int c = (lane % KCH) ^ Gm::kc_swz(r);
            const int slot = min(row0 + r, p.slots - 1);
            const int src = Tr::gather ? p.perm[slot] : slot;
            a_ptr[i] = p.a + (int64_t)src * p.lda + c * 8;
            a_k[i] = 0;
        } else {
            constexpr int C = BM / 8;  // 16-byte chunks per k row
            const int k = (64 / C) * q + lane / C;
            const int c = (lane % C) ^ Gm::mc_swz(k);
            a_ptr[i] = p.a + min(mt * BM + c * 8, p.M - 8);
            a_k[i] = k;
        }
    }
#pragma unroll
    for (int i = 0; i < DMA_B; ++i) {
        const int q = wave * DMA_B + i;
        if constexpr (Tr::b_fp4) {
            b_ptr[i] = nullptr;
            b_k[i] = 0;
        } else if constexpr (Tr::b_kc) {
            const int r = KC_ROWS * q + lane / KCH;
            const int c = (lane % KCH) ^ Gm::kc_swz(r);
            const int n = min(col0 + r, p.N - 1);
            b_ptr[i] = p.w[e] + (int64_t)n * p.ldb + c * 8;
            b_k[i] = 0;
        } else {
            constexpr int C = BN / 8;
            const int k = (64 / C) * q + lane / C;
            const int c = (lane % C) ^ Gm::mc_swz(k);
            const uint16_t* base = Tr::group_k ? p.b : p.w[e];
            b_ptr[i] = base + min(col0 + c * 8, p.N - 8);
            b_k[i] = k;
        }
    }
    // MXFP4: lane pair (2m, 2m+1) loads the 32 code bytes of row m (two 16-byte
    // halves, swapped in LDS when bit 3 of m is set); every wave loads its own
    // copy of the tile's 256 row scales of both 32-blocks (lane l: rows
    // 16(l%16)..+15 of block l/16; row groups past N are clamped to the tile's
    // first group).
    const uint8_t* q_ptr[2] = {nullptr, nullptr};
    const uint8_t* sc_ptr = nullptr;
    if constexpr (Tr::b_fp4) {
        const int g = nt * BN + 16 * (lane & 15);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int sl = (wave * 2 + i) * 64 + lane, m = sl >> 1;
            const int half = (sl & 1) ^ ((m >> 3) & 1);
            q_ptr[i] = p.wq[e] + (int64_t)min(nt * BN + m, p.N - 1) * (p.K / 2) + half * 16;
        }
        sc_ptr = p.wsc[e] + (int64_t)((lane >> 4) & 1) * p.N + (g < p.N ? g : nt * BN);
    }
    const uint32_t lds0 = lds_addr(lds);
    // bf16 element offsets of tile t's A and B operand tiles in LDS
    auto a_slot = [&](int t) -> int { return kSplit ? (t % NST) * OPND_A : (t % NST) * STAGE; };
    auto b_slot = [&](int t) -> int {
        return kSplit ? NST * OPND_A + (t % (NST - 1)) * B_SLOT : (t % NST) * STAGE + OPND_A;
    };
    // Wave load i of tile t's A / B operand (t clamped to the last real tile
    // so the per-tile load count stays constant).
    auto dma_a = [&](int t, int i) {
        const int k0 = kbeg + min(t, nk - 1) * BK;
        const uint16_t* ga = Tr::a_kc ? a_ptr[i] + k0 : a_ptr[i] + (int64_t)min(k0 + a_k[i], kend - 1) * p.lda;
        dma16(ga, lds0 + (uint32_t)a_slot(t) * 2u + (uint32_t)(wave * DMA_A + i) * 1024u);
    };
    auto dma_b = [&](int t, int i) {
        const int k0 = kbeg + min(t, nk - 1) * BK;
        if constexpr (Tr::b_fp4) {
            const uint32_t sb = lds0 + (uint32_t)b_slot(t) * 2u;
            if (i < DMA_BT - 1) dma16(q_ptr[i] + k0 / 2, sb + (uint32_t)(wave * (DMA_BT - 1) + i) * 1024u);
            else dma16(sc_ptr + (int64_t)(k0 / 32) * p.N, sb + kFp4Codes + (uint32_t)wave * 1024u);
        } else {
            const uint16_t* gb = Tr::b_kc ? b_ptr[i] + k0 : b_ptr[i] + (int64_t)min(k0 + b_k[i], kend - 1) * p.ldb;
            dma16(gb, lds0 + (uint32_t)b_slot(t) * 2u + (uint32_t)(wave * DMA_B + i) * 1024u);
        }
    };
    // One ring: issue the wave loads of K tile t (clamped to the last real tile
    // so the per-tile load count stays constant) into stage t % NST.
    auto dma_tile = [&](int t) {
        const int k0 = kbeg + min(t, nk - 1) * BK;  // first reduction index of the tile
        const uint32_t sbase = lds0 + (uint32_t)((t % NST) * STAGE) * 2u;
#pragma unroll
        for (int i = 0; i < DMA_A; ++i) {
            const uint32_t qoff = (uint32_t)(wave * DMA_A + i) * 1024u;
            const uint16_t* ga = Tr::a_kc ? a_ptr[i] + k0
                                          : a_ptr[i] + (int64_t)min(k0 + a_k[i], kend - 1) * p.lda;
            dma16(ga, sbase + qoff);
        }
#pragma unroll
        for (int i = 0; i < DMA_B; ++i) {
            const uint32_t qoff = (uint32_t)(wave * DMA_B + i) * 1024u;
            const uint16_t* gb = Tr::b_kc ? b_ptr[i] + k0
                                          : b_ptr[i] + (int64_t)min(k0 + b_k[i], kend - 1) * p.ldb;
            dma16(gb, sbase + OPND_A * 2u + qoff);
        }
    };
    // Load `idx` of dma_tile(t) on its own, for interleaving with the MFMAs.
    auto dma_one = [&](int t, int idx) {
        const int k0 = kbeg + min(t, nk - 1) * BK;
        const uint32_t sbase = lds0 + (uint32_t)((t % NST) * STAGE) * 2u;
        if (idx < DMA_A) {
            const uint32_t qoff = (uint32_t)(wave * DMA_A + idx) * 1024u;
            const uint16_t* ga = Tr::a_kc ? a_ptr[idx] + k0
                                          : a_ptr[idx] + (int64_t)min(k0 + a_k[idx], kend - 1) * p.lda;
            dma16(ga, sbase + qoff);
        } else {
            const int i = idx - DMA_A;
            const uint32_t qoff = (uint32_t)(wave * DMA_B + i) * 1024u;
            const uint16_t* gb = Tr::b_kc ? b_ptr[i] + k0
                                          : b_ptr[i] + (int64_t)min(k0 + b_k[i], kend - 1) * p.ldb;
            dma16(gb, sbase + OPND_A * 2u + qoff);
        }
    };
    // Reduction tail of the weight-gradient GEMMs: zero k rows >= kvalid of
    // the last tile in both operand tiles (rows of 512 bytes).
    auto zero_tail = [&](int t) {
        if constexpr (Tr::group_k) {
            const int kvalid = kend - (kbeg + t * BK);
            if (kvalid < BK) {
                uint16_t* st = lds + (t % NST) * STAGE;
                const int na = (BK - kvalid) * (BM / 8), nb = (BK - kvalid) * (BN / 8);  // 16-byte vectors
                for (int v = tid; v < na + nb; v += NT) {
                    if (v < na) *reinterpret_cast<uint4*>(st + kvalid * BM + v * 8) = make_uint4(0, 0, 0, 0);
                    else *reinterpret_cast<uint4*>(st + OPND_A + kvalid * BN + (v - na) * 8) = make_uint4(0, 0, 0, 0);
                }
            }
        }
    };

    // ---- fragments ----------------------------------------------------------
    struct Frag {
        uint4 a[MI], b[NJ];
    };
    // K-contiguous: lane reads row base + lane%32, chunk 2s + lane/32.
    auto read_kc = [&](const uint16_t* t, int rbase, int s) {
        const int r = rbase + (lane & 31);
        const int c = (2 * s + (lane >> 5)) ^ Gm::kc_swz(r);
        return *reinterpret_cast<const uint4*>(t + r * BK + c * 8);
    };
    // Row-contiguous: two transposing reads give k = 16s + 8(lane/32) + 0..7
    // for column cbase + lane%32.
    auto read_mc = [&](const uint16_t* t, int stride, int cbase, int s) {
        const int g = lane >> 4, r = lane & 15;
        const int col = cbase + 16 * (g & 1) + 4 * (r & 3);
        const int kb = 16 * s + 8 * (g >> 1) + (r >> 2);
        uint32_t w[4];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int k = kb + 4 * h;
            const int c = (col >> 3) ^ Gm::mc_swz(k);
            const s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (lds_s16x4*)(t + k * stride + c * 8 + (col & 7)));
            w[2 * h] = (uint32_t)(uint16_t)v[0] | ((uint32_t)(uint16_t)v[1] << 16);
            w[2 * h + 1] = (uint32_t)(uint16_t)v[2] | ((uint32_t)(uint16_t)v[3] << 16);
        }
        return make_uint4(w[0], w[1], w[2], w[3]);
    };
    // MXFP4: lane reads 4 bytes (8 codes: k = 16s + 8(lane/32) .. +7, byte
    // 8s + 4(lane/32) of the row's 32) of row rbase + lane%32 and that row's
    // scale from its wave's copy, and expands them to a bf16 fragment.
    auto read_fp4 = [&](const uint16_t* tB, int rbase, int s) {
        const uint8_t* codes = reinterpret_cast<const uint8_t*>(tB);
        const uint8_t* scales = codes + kFp4Codes + wave * 1024;
        const int r = rbase + (lane & 31);
        const int blk = s >> 1, within = (8 * s + 4 * (lane >> 5)) & 15;
        const uint32_t w = *reinterpret_cast<const uint32_t*>(
            codes + r * 32 + ((blk ^ ((lane >> 3) & 1)) * 16) + within);
        return dequant8(w, scales[blk * 256 + r]);
    };
    auto load_frag = [&](Frag& f, int t, int s) {
        const uint16_t* tA = lds + a_slot(t);
        const uint16_t* tB = lds + b_slot(t);
#pragma unroll
        for (int i = 0; i < MI; ++i)
            f.a[i] = Tr::a_kc ? read_kc(tA, wrow + 32 * i, s) : read_mc(tA, BM, wrow + 32 * i, s);
#pragma unroll
        for (int j = 0; j < NJ; ++j)
            f.b[j] = Tr::b_fp4 ? read_fp4(tB, wcol + 32 * j, s)
                               : (Tr::b_kc ? read_kc(tB, wcol + 32 * j, s) : read_mc(tB, BN, wcol + 32 * j, s));
    };

    f32x16 acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
    // The first k16 step of a tile with the loads of tile t spread over its
    // MFMAs (one after every MI*NJ / DMA_PER_TILE of them). A wave that issues
    // the eight loads back to back leaves its SIMD's MFMA unit idle while
    // they issue. Measured on the c3 shapes: DOWN 1.115 -> 1.070 ms, UP and
    // DACT about 0.5% faster; DX (+6.6%) and the weight-gradient GEMMs
    // (+1-2.5%) keep the loads in one batch.
    constexpr bool kSpreadDma = KIND == GEMM_DOWN || KIND == GEMM_UP || KIND == GEMM_DACT;
    auto mma_dma = [&](const Frag& f, int t) {
        constexpr int NM = MI * NJ;
        int dq = 0;
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                    __builtin_bit_cast(bf16x8, f.b[j]), __builtin_bit_cast(bf16x8, f.a[i]),
                    acc[i][j], 0, 0, 0);
                const int q = i * NJ + j;
                if (dq < DMA_PER_TILE && (q + 1) * DMA_PER_TILE >= (dq + 1) * NM) {
                    __builtin_amdgcn_sched_barrier(0);
                    dma_one(t, dq);
                    __builtin_amdgcn_sched_barrier(0);
                    ++dq;
                }
            }
        for (; dq < DMA_PER_TILE; ++dq) dma_one(t, dq);
    };
    auto mma = [&](const Frag& f) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                    __builtin_bit_cast(bf16x8, f.b[j]), __builtin_bit_cast(bf16x8, f.a[i]),
                    acc[i][j], 0, 0, 0);
    };

    // ---- main loop ----------------------------------------------------------
    // Iteration kt runs the STEPS k16 steps of tile kt. Every step first reads
    // the next step's fragments; the first step also issues the loads of
    // tile kt + NST - 1. Before the last step the wave waits for its loads
    // of tile kt+1 and the workgroup synchronises (all loads of tile kt+1 are
    // visible, and every wave is done reading the stage that the next
    // iteration refills); the last step then prefetches step 0 of tile kt+1.
    constexpr int VM_AHEAD = (NST - 2) * DMA_PER_TILE;
    if constexpr (kSplit) {
        // Split rings. Iteration kt multiplies tile kt in STEPS k16 steps;
        // the loads of B(kt+1) and then A(kt+2) are spread over the MFMAs of
        // the first STEPS - 1 steps (their slots were last read by tile kt-1,
        // before the previous barrier). Loads complete in issue order, so
        // waiting until only A(kt+2)'s loads are outstanding leaves all of
        // tile kt+1 in LDS at the barrier; the last step then prefetches
        // tile kt+1's first fragments.
        constexpr int ND = DMA_A + DMA_BT;
        auto mma_loads = [&](const Frag& f, int kt, int d0, int dn) {
            constexpr int NM = MI * NJ;
            int dq = 0;
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                        __builtin_bit_cast(bf16x8, f.b[j]), __builtin_bit_cast(bf16x8, f.a[i]),
                        acc[i][j], 0, 0, 0);
                    const int q = i * NJ + j;
                    if (dq < dn && (q + 1) * dn >= (dq + 1) * NM) {
                        const int d = d0 + dq;
                        __builtin_amdgcn_sched_barrier(0);
                        if (d < DMA_BT) dma_b(kt + 1, d);
                        else dma_a(kt + 2, d - DMA_BT);
                        __builtin_amdgcn_sched_barrier(0);
                        ++dq;
                    }
                }
        };
        auto dfirst = [](int s) { return s * ND / (STEPS - 1); };
        if (nk > 0) {
#pragma unroll
            for (int i = 0; i < DMA_A; ++i) dma_a(0, i);
#pragma unroll
            for (int i = 0; i < DMA_BT; ++i) dma_b(0, i);
#pragma unroll
            for (int i = 0; i < DMA_A; ++i) dma_a(1, i);
            wait_vm<DMA_A>();
            __syncthreads();
            Frag f[2];
            load_frag(f[0], 0, 0);
            for (int kt = 0; kt < nk; ++kt) {
#pragma unroll
                for (int s = 0; s < STEPS - 1; ++s) {
                    load_frag(f[(s + 1) & 1], kt, s + 1);
                    mma_loads(f[s & 1], kt, dfirst(s), dfirst(s + 1) - dfirst(s));
                }
                wait_vm<DMA_A>();
                __syncthreads();
                load_frag(f[0], min(kt + 1, nk - 1), 0);
                mma(f[(STEPS - 1) & 1]);
#pragma unroll
                for (int q = 0; q < MI * NJ / 2; ++q) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 1);  // MFMA
                    __builtin_amdgcn_sched_group_barrier(0x100, 2, 1);  // DS read
                }
                __builtin_amdgcn_sched_group_barrier(0x008, MI * NJ / 2, 1);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    } else if (nk > 0) {
#pragma unroll
        for (int t = 0; t < NST - 1; ++t) dma_tile(t);
        wait_vm<VM_AHEAD>();
        __syncthreads();
        if (nk == 1) {
            zero_tail(0);
            __syncthreads();
        }
        Frag f[2];
        load_frag(f[0], 0, 0);
        for (int kt = 0; kt < nk; ++kt) {
#pragma unroll
            for (int s = 0; s < STEPS - 1; ++s) {
                load_frag(f[(s + 1) & 1], kt, s + 1);
                if constexpr (kSpreadDma) {
                    if (s == 0) {
                        mma_dma(f[0], kt + NST - 1);
                        continue;
                    }
                } else {
                    if (s == 0) dma_tile(kt + NST - 1);
                }
                mma(f[s & 1]);
#pragma unroll
                for (int q = 0; q < MI * NJ / 2; ++q) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
                    __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);  // DS read
                }
                __builtin_amdgcn_sched_group_barrier(0x008, MI * NJ / 2, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
            wait_vm<VM_AHEAD>();
            __syncthreads();
            if (kt + 1 == nk - 1) {
                zero_tail(kt + 1);
                __syncthreads();
            }
            load_frag(f[0], min(kt + 1, nk - 1), 0);
            mma(f[1]);
#pragma unroll
            for (int q = 0; q < MI * NJ / 2; ++q) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 1);  // MFMA
                __builtin_amdgcn_sched_group_barrier(0x100, 2, 1);  // DS read
            }
            __builtin_amdgcn_sched_group_barrier(0x008, MI * NJ / 2, 1);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    wait_vm<0>();
    __syncthreads();

    // ---- epilogue ---------------------------------------------------------
    // acc[i][j][r] = C[m][n] with m = wrow + 32i + (lane&31) and
    // n = wcol + 32j + 8(r>>2) + 4(lane>>5) + (r&3) (n from the tile's col0).
    // Passes of EPR rows per wave go through an fp32 LDS region ([EPR][WTN],
    // 16-byte chunks swizzled by row), then leave as row-contiguous 16-byte
    // stores.
    constexpr int CH = WTN / 4;              // 16-byte fp32 chunks per staged row
    constexpr int LPR = WTN / 8, RPI = 64 / LPR;     // bf16 out: lanes per row, rows per instruction
    constexpr int FLPR = WTN / 4, FRPI = 64 / FLPR;  // fp32 out
    constexpr int FPP = EPR / 32, PASSES = MI / FPP;  // row fragments per pass, passes
    float* stage_f = reinterpret_cast<float*>(lds_raw) + wave * (EPR * WTN);
    const int mbase = wrow, nbase = wcol;
    // GEMM_DACT: silu'(U) of every pass is requested here, in one batch, so
    // the tile waits for one memory round trip instead of one per pass (the
    // mainloop's operand fragments are dead, which leaves room).
    constexpr int UPP = KIND == GEMM_DACT ? EPR / RPI : 1;  // U loads per lane and pass
    uint4 uin[KIND == GEMM_DACT ? PASSES : 1][UPP];
    if constexpr (KIND == GEMM_DACT && !Tr::group_k) {
        const int n = nbase + (lane % LPR) * 8;
#pragma unroll
        for (int pass = 0; pass < PASSES; ++pass)
#pragma unroll
            for (int k = 0; k < UPP; ++k) {
                const int m = mbase + pass * EPR + lane / LPR + RPI * k;
                const bool ok = m < mlim && n < nlim;
                const int64_t off = (int64_t)(row0 + (ok ? m : 0)) * p.ldc + col0 + (ok ? n : 0);
                uin[pass][k] = ld16_nt(p.u + off);
            }
    }
#pragma unroll
    for (int pass = 0; pass < PASSES; ++pass) {
#pragma unroll
        for (int ii = 0; ii < FPP; ++ii) {
            const int i = pass * FPP + ii;
            const int lr = ii * 32 + (lane & 31);
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int ch = j * 8 + 2 * q + (lane >> 5);
                    *reinterpret_cast<f32x4*>(stage_f + lr * WTN + ((ch ^ (lr & (CH - 1))) * 4)) =
                        f32x4{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2],
                              acc[i][j][4 * q + 3]};
                }
        }
        __syncthreads();
        if (kSplitK && part_unit >= 0) {
            // split-K part: the fp32 partial tile [BM][BN], rows < mlim, with
            // plain stores (split_fixup_kernel reads it right after, from
            // the caches; non-temporal stores measured 0.015 ms slower per GEMM)
            float* C = p.part + (int64_t)part_unit * BM * BN;
            const int cl = lane % FLPR;
#pragma unroll 4
            for (int rr = lane / FLPR; rr < EPR; rr += FRPI) {
                const int m = mbase + pass * EPR + rr;
                const int n = nbase + cl * 4;
                if (m >= mlim || n >= nlim) continue;
                const f32x4 v = *reinterpret_cast<const f32x4*>(stage_f + rr * WTN + ((cl ^ (rr & (CH - 1))) * 4));
                *reinterpret_cast<f32x4*>(C + (int64_t)m * BN + n) = v;
            }
        } else if constexpr (!Tr::group_k) {
            // LPR lanes per row (8 bf16 each), RPI rows per instruction
            uint16_t* C = reinterpret_cast<uint16_t*>(p.c);
            const int cl = lane % LPR;
            const int n = nbase + cl * 8;
            // element offset of the lane's first row in this pass, advanced by
            // RPI rows per store (no 64-bit multiply per store)
            const int64_t off0 = (int64_t)(row0 + mbase + pass * EPR + lane / LPR) * p.ldc + col0 + n;
            const int64_t rstep = (int64_t)RPI * p.ldc;
#pragma unroll
            for (int k = 0; k < EPR / RPI; ++k) {
                const int rr = lane / LPR + RPI * k;
                const int m = mbase + pass * EPR + rr;
                if (m >= mlim || n >= nlim) continue;
                const float* src = stage_f + rr * WTN;
                const f32x4 v0 = *reinterpret_cast<const f32x4*>(src + (((2 * cl) ^ (rr & (CH - 1))) * 4));
                const f32x4 v1 = *reinterpret_cast<const f32x4*>(src + (((2 * cl + 1) ^ (rr & (CH - 1))) * 4));
                float v[8] = {v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
                const int64_t off = off0 + k * rstep;
                if constexpr (DUAL) {
                    // U itself is not kept: C = silu'(U) (skipped when C is
                    // null, for forward-only handles), c2 = SiLU(U)
                    float a[8], da[8];
#pragma unroll
                    for (int t = 0; t < 8; ++t) silu_dsilu(v[t], a[t], da[t]);
                    if (C != nullptr) st16_nt(C + off, pack8(da));
                    st16_nt(p.c2 + off, pack8(a));
                } else {
                    if constexpr (KIND == GEMM_DACT) {
                        float ds[8];
                        unpack8(uin[pass][k], ds);  // silu'(U) from the up GEMM
#pragma unroll
                        for (int t = 0; t < 8; ++t) v[t] *= ds[t];
                    }
                    st16_nt(C + off, pack8(v));
                }
            }
        } else {
            // FLPR lanes per row (4 fp32 each), FRPI rows per instruction
            float* C = p.dw[e];
            const int cl = lane % FLPR;
            const int n = nbase + cl * 4;
            float* o0 = C + (int64_t)(mt * BM + mbase + pass * EPR) * p.ldc + col0 + n;
            auto staged = [&](int rr) {
                return *reinterpret_cast<const f32x4*>(stage_f + rr * WTN + ((cl ^ (rr & (CH - 1))) * 4));
            };
            // rows of any width: 16-byte stores at any float's address
            if (mlim == BM && nlim == BN) {  // uniform: a whole tile
#pragma unroll 4
                for (int rr = lane / FLPR; rr < EPR; rr += FRPI)
                    __builtin_nontemporal_store(staged(rr), reinterpret_cast<f32x4_any*>(o0 + (int64_t)rr * p.ldc));
            } else {
#pragma unroll 4
                for (int rr = lane / FLPR; rr < EPR; rr += FRPI) {
                    if (mbase + pass * EPR + rr >= mlim || n >= nlim) continue;
                    const f32x4 v = staged(rr);
                    float* o = o0 + (int64_t)rr * p.ldc;
                    if (n + 4 <= nlim) __builtin_nontemporal_store(v, reinterpret_cast<f32x4_any*>(o));
                    else
                        for (int t = 0; t < nlim - n; ++t) o[t] = v[t];
                }
            }
        }
        __syncthreads();
    }
}

template <int KIND, bool DUAL, int BK, int NST, int TILE>
__global__ __launch_bounds__(256, (Geo<BK, NST, TILE>::WGS)) void grouped_gemm_kernel(GemmParams p) {
    __shared__ uint4 lds_raw[gemm_lds_bytes<KIND, BK, NST, TILE>() / 16];
    // the experts' tiles, once per workgroup (before any tile's stores, so
    // the vector load of the offsets waits on nothing else)
    ExpertTiles et{};
    if constexpr (!Traits<KIND>::group_k) et = expert_tiles<TILE>(p.offsets, p.E, threadIdx.x & 63);
    if constexpr (split_ring<KIND, TILE>()) {
        for (int vb = blockIdx.x; vb < p.vblocks; vb += gridDim.x)
            grouped_gemm_tile<KIND, DUAL, BK, NST, TILE>(p, vb, et, lds_raw);
    } else {
        grouped_gemm_tile<KIND, DUAL, BK, NST, TILE>(p, blockIdx.x, et, lds_raw);
    }
}

// The split-K tail's second pass: tail tile j is the sum of its S partials
// in part order, rounded once to bf16. Work items are (tile, 8-row slab);
// thread t adds 8 columns of one row.
template <int BK>
__global__ __launch_bounds__(256) void split_fixup_kernel(GemmParams p) {
    constexpr int BM = kLarge, BN = kLarge;
    const int ntn = (p.N + BN - 1) / BN, mtiles = act_mtiles(p);
    const SplitPlan sp = split_plan<BK>(p, mtiles * ntn);
    if (sp.S < 2) return;
    constexpr int kSlabs = BM / 8;
    const int tid = threadIdx.x;
    const int rr = tid / (BN / 8), col = (tid % (BN / 8)) * 8;  // 8 rows x 32 lanes of 8 columns
    uint16_t* C = reinterpret_cast<uint16_t*>(p.c);
    for (int w = blockIdx.x; w < sp.R * kSlabs; w += gridDim.x) {
        const int j = w / kSlabs, slab = w % kSlabs;
        int mt, nt, e, row0 = 0, rows = 0;
        list_tile(sp.F + j, mtiles, ntn, list_rows(ntn), mt, nt);
        act_tile(p, mt, e, row0, rows);
        const int row = slab * 8 + rr;
        if (e < 0 || row >= rows || nt * BN + col >= p.N) continue;
        float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        const float* src = p.part + (int64_t)j * sp.S * BM * BN + (int64_t)row * BN + col;
        // the loads of up to 8 parts in flight together (one round trip per
        // 8 parts), then added in part order
        for (int q0 = 0; q0 < sp.S; q0 += 8) {
            f32x4 a[8], b[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int q = min(q0 + u, sp.S - 1);  // clamped: the extra loads are not added
                a[u] = *reinterpret_cast<const f32x4*>(src + (int64_t)q * BM * BN);
                b[u] = *reinterpret_cast<const f32x4*>(src + (int64_t)q * BM * BN + 4);
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                if (q0 + u >= sp.S) break;
                acc[0] += a[u][0]; acc[1] += a[u][1]; acc[2] += a[u][2]; acc[3] += a[u][3];
                acc[4] += b[u][0]; acc[5] += b[u][1]; acc[6] += b[u][2]; acc[7] += b[u][3];
            }
        }
        *reinterpret_cast<uint4*>(C + (int64_t)(row0 + row) * p.ldc + nt * BN + col) = pack8(acc);
    }
}

}  // namespace

// Ring of a kind and tile size:
//   256 x 256 (one workgroup per CU): split rings of K = 64 (activation
//   GEMMs), 4 stages of K = 32 (weight gradients);
//   128 x 128 activation tiles: 2 stages of K = 64, two workgroups per CU
//   (64 KiB each, the size of the epilogue's staging anyway), or DEEP, 4
//   stages, one workgroup per CU. With two stages a lone workgroup waits out
//   a memory round trip per K = 64 step (about 1.1 us); with four it is down
//   to 0.72 us, mostly its LDS reads. K = 64 makes 128-byte row segments,
//   which the CU's load path takes at twice the rate of 64-byte ones;
//   128 x 128 weight-gradient tiles: 4 stages of K = 32, two workgroups per CU.
template <int KIND, int TILE = kLarge, bool DEEP = false>
struct Ring {
    static constexpr bool k64 = !Traits<KIND>::group_k;
    static constexpr int BK = k64 ? 64 : 32;
    static constexpr int NST = split_ring<KIND, TILE>() ? 3 : k64 && !DEEP ? 2 : 4;
};

// grid: the launch-order blocks of the tile map. Persistent kinds run
// min(grid, CUs rounded down to a multiple of 8) workgroups over them.
template <int KIND, bool DUAL, int TILE = kLarge, bool DEEP = false>
hipError_t launch_kind(const GemmParams& p, unsigned grid, hipStream_t s) {
    using R = Ring<KIND, TILE, DEEP>;
    GemmParams q = p;
    q.vblocks = (int)grid;
    unsigned g = grid;
    if constexpr (split_ring<KIND, TILE>()) {
        const unsigned cus = (unsigned)(cu_count() / 8 * 8);
        if (cus >= 8 && g > cus) g = cus;
    }
    grouped_gemm_kernel<KIND, DUAL, R::BK, R::NST, TILE><<<g, 256, 0, s>>>(q);
    return hipGetLastError();
}

// Tiles of `rows` rows that the experts' segments make at even routing: one
// per expert while the mean is well below `rows`; above, half of each
// expert's last tile is empty on average, or, with few tiles per expert, the
// mean's own last tile where it lies clear of a multiple of `rows`.
static double act_tiles(const GemmParams& p, int rows) {
    const double used = std::min(p.E, p.slots), m = p.slots / (used > 0 ? used : 1.0) / rows;
    return used * (m <= 0.85 ? 1.0 : m < 3.0 ? std::min(m + 0.5, std::ceil(m + 0.15)) : m + 0.5);
}
// Estimated time (us) of an activation GEMM on each tile, from what the
// kernels measured on one MI355X over K = 256 .. 4096 and 0.2 .. 33 rounds
// (nk: K = 64 steps):
//   256 x 256, a round of one tile per CU: 17 + 1.24 nk where the epilogue
//     evaluates or multiplies by the SiLU terms (GEMM_UP with hidden > 0,
//     GEMM_DACT), else 9 + 1.56 nk; GEMM_DOWN and GEMM_DX split the last
//     round along K, which costs the partial tiles' write and fix-up (up to
//     28 us when it fills the chip);
//   128 x 128, a round of two per CU: 5 + 1.1 nk (full or not);
//   128 x 128 deep, one per CU: 4 + 0.72 nk, better than two per CU only
//     while every tile has a CU of its own.
// Small problems leave CUs idle or end in a nearly empty round on the large
// tiles. Measured (us; 256 x 256 / 128 x 128 / deep): 777 tokens on 16
// experts, top-4, N = 1024, K = 4096 70 / 77 / 52; 4096 slots, E = 8,
// N = K = 1280 35 / 25 / 30; 8192 slots, E = 8, N = 2048, K = 768 61 / 55 /
// 61; 32768 slots, E = 8, N = 2048, K = 512 146 / 133 / 164; 131072 slots,
// E = 16, N = 4096, K = 1024 1228 / 1456 / -.
static GemmTile act_tile_choice(GemmKind kind, const GemmParams& p) {
    const double cus = cu_count(), nk = p.K / 64.0;
    const bool silu = kind == GEMM_DACT || (kind == GEMM_UP && p.c2 != nullptr);
    const double t256 = act_tiles(p, 256) * ((p.N + 255) / 256), t128 = act_tiles(p, 128) * ((p.N + 127) / 128);
    const double round256 = silu ? 17.0 + 1.24 * nk : 9.0 + 1.56 * nk;
    double c256 = std::ceil(t256 / cus) * round256;
    if ((kind == GEMM_DOWN || kind == GEMM_DX) && p.part != nullptr) {
        const double whole = std::floor(t256 / cus), rest = std::ceil(t256 - whole * cus);
        const double parts = rest > 0 ? std::min(std::floor(cus / rest), std::floor(nk / 8)) : 1.0;
        if (parts >= 2) c256 = whole * round256 + 12.0 + 1.56 * nk / parts + 28.0 * rest * parts / cus;
    }
    const double c128 = std::ceil(t128 / (2 * cus)) * (5.0 + 1.1 * nk);
    const double cdeep = std::ceil(t128 / cus) * (4.0 + 0.72 * nk);
    if (c256 <= c128 && c256 <= cdeep) return GemmTile{256};
    return GemmTile{128, t128 <= cus && cdeep < c128};
}

GemmTile gemm_tile(GemmKind kind, const GemmParams& p) {
    if (kind == GEMM_UP_FP4 || kind == GEMM_DOWN_FP4) return GemmTile{256};
    if (kind == GEMM_DW_DOWN || kind == GEMM_DW_UP) {
        // Weight gradients: 128 x 128 tiles (two per CU) where the 256 x 256
        // ones fill at most half of the CUs. d = 512, h = 2048, E = 8 (128
        // large tiles): 113 -> 86 us each at 32768 slots; d = h = 1280, E = 8
        // (200 large tiles): 28 us on large, 30 on small ones.
        const int64_t tiles = (int64_t)p.E * ((p.M + 255) / 256) * ((p.N + 255) / 256);
        return GemmTile{2 * tiles <= cu_count() ? 128 : 256};
    }
    return act_tile_choice(kind, p);
}

hipError_t launch_gemm_tile(GemmKind kind, bool dual, const GemmParams& p, GemmTile tile, hipStream_t s) {
    const int m = tile.m;
    if (p.N % 8 != 0 || p.N <= 0) return hipErrorInvalidValue;
    if (m != 256 && m != 128) return hipErrorInvalidValue;
    const bool group_k = kind == GEMM_DW_DOWN || kind == GEMM_DW_UP;
    const bool fp4 = kind == GEMM_UP_FP4 || kind == GEMM_DOWN_FP4;
    if (tile.deep && (m != 128 || group_k)) return hipErrorInvalidValue;
    if (fp4 && m != 256) return hipErrorInvalidValue;
    const int64_t ntn = (p.N + m - 1) / m;
    int64_t grid;
    if (group_k) {
        if (p.M % 8 != 0 || p.M <= 0) return hipErrorInvalidValue;
        if (p.m_out > p.M || p.n_out > p.N || p.M - p.m_out >= 64 || p.N - p.n_out >= 64 || p.ldc < p.n_out)
            return hipErrorInvalidValue;
        // whole rounds of 8 XCDs x 32 workgroups keep the block -> tile map a bijection
        grid = ((int64_t)p.E * ((p.M + m - 1) / m) * ntn + 255) / 256 * 256;
    } else {
        if (p.K % 64 != 0) return hipErrorInvalidValue;
        // sum_e ceil(cnt_e / m) <= ceil(slots / m) + E - 1
        const int64_t tiles = (((int64_t)p.slots + m - 1) / m + p.E) * ntn;
        grid = tiles >= 8 * 256 ? (tiles + 255) / 256 * 256 : (tiles + 7) / 8 * 8;  // whole rounds, or eight equal runs
    }
    // split-K tail (GEMM_DOWN / GEMM_DX on 256 x 256 tiles): its parts are
    // the workgroups after the whole rounds, at most `resident` of them.
    const bool split = (kind == GEMM_DOWN || kind == GEMM_DX) && m == 256 && p.part != nullptr &&
                       p.resident > 0 && p.resident % 256 == 0;
    if (split) grid += p.resident;
    if (grid <= 0) return hipSuccess;
    if (grid > 0x7fffffff) return hipErrorInvalidValue;
    const unsigned g = (unsigned)grid;
    if (split) {
        hipError_t err = kind == GEMM_DOWN ? launch_kind<GEMM_DOWN, false>(p, g, s) : launch_kind<GEMM_DX, false>(p, g, s);
        if (err != hipSuccess) return err;
        static_assert(Ring<GEMM_DOWN>::BK == Ring<GEMM_DX>::BK, "one split plan for DOWN and DX");
        // 4 workgroups per CU: the (tile, 8-row slab) items are short and latency-bound
        split_fixup_kernel<Ring<GEMM_DOWN>::BK><<<p.resident * 4, 256, 0, s>>>(p);
        return hipGetLastError();
    }
#define TMT_ACT(KIND_, DUAL_)                                   \
    (m == 256     ? launch_kind<KIND_, DUAL_>(p, g, s)          \
     : !tile.deep ? launch_kind<KIND_, DUAL_, 128>(p, g, s)     \
                  : launch_kind<KIND_, DUAL_, 128, true>(p, g, s))
#define TMT_DW(KIND_) (m == 256 ? launch_kind<KIND_, false>(p, g, s) : launch_kind<KIND_, false, 128>(p, g, s))
    switch (kind) {
        case GEMM_UP: return dual ? TMT_ACT(GEMM_UP, true) : TMT_ACT(GEMM_UP, false);
        case GEMM_DOWN: return TMT_ACT(GEMM_DOWN, false);
        case GEMM_DACT: return TMT_ACT(GEMM_DACT, false);
        case GEMM_DX: return TMT_ACT(GEMM_DX, false);
        case GEMM_DW_DOWN: return TMT_DW(GEMM_DW_DOWN);
        case GEMM_DW_UP: return TMT_DW(GEMM_DW_UP);
        case GEMM_UP_FP4: return dual ? launch_kind<GEMM_UP_FP4, true>(p, g, s) : hipErrorInvalidValue;
        case GEMM_DOWN_FP4: return launch_kind<GEMM_DOWN_FP4, false>(p, g, s);
        default: return hipErrorInvalidValue;
    }
#undef TMT_ACT
#undef TMT_DW
}

hipError_t launch_gemm(GemmKind kind, bool dual, const GemmParams& p, hipStream_t s) {
    return launch_gemm_tile(kind, dual, p, gemm_tile(kind, p), s);
}

}  // namespace tmt
