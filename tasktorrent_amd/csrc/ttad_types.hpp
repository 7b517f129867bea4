// Shared host/device definitions of the tile DAG executor.
#pragma once
#include <stdint.h>

namespace ttad {

// Task kinds of the tiled Cholesky PTG (miniapp/dense_cholesky/2d_cholesky.cpp:316-608).
enum Kind : int32_t { K_POTRF = 0, K_TRSM = 1, K_SYRK = 2, K_GEMM = 3, K_ACCU = 4, K_NOP = 5 };
// Arithmetic of a task. Tiles are stored in FP64 (P_F64) or FP32 (the mixed variants).
enum Prec : int32_t { P_F64 = 0, P_F32 = 1, P_BF16 = 2, P_BF16X3 = 3 };

constexpr int NTHREADS = 256;  // one workgroup = 4 wave64
constexpr int GEMM_BM = 128;   // GEMM/SYRK work item = 128x128 output sub-tile
constexpr int GEMM_BS = 64;    // or a 64x64 one, where the items of 128 leave CUs idle (DevTask::sub)
// Rows of a TRSM work item. Up to TRSM_LDS_COLS columns the solved part of X stays in LDS: 16 FP64 or 32 FP32 rows of
// 512 columns (64 KB, so that two workgroups share a CU). Wider tiles re-read it: 32 and 64 rows.
constexpr int TRSM_LDS_COLS = 512;
constexpr int TRSM_BM = 32;
constexpr int TRSM_BM_F32 = 64;
__host__ __device__ constexpr int trsm_rows(int elem_bytes, bool in_lds) {
    return (elem_bytes == 8 ? TRSM_BM : TRSM_BM_F32) / (in_lds ? 2 : 1);
}
constexpr int DB = 64;         // diagonal sub-block size whose inverse POTRF leaves for TRSM

// Items of a raw GEMM (SYRK) of bm x bm of them.
__host__ __device__ inline long raw_gemm_items(int m, int n, bool syrk, int bm) {
    const long tr = ((long)m + bm - 1) / bm, tc = ((long)n + bm - 1) / bm;
    return syrk ? tr * (tr + 1) / 2 : tr * tc;
}
// Whether a raw GEMM takes 64x64 items: where 128x128 ones would leave CUs without work. Measured, us with 128 / with 64,
// by the number of 128x128 items: 4 (m = n = k = 256) FP64 48 / 19, FP32 25 / 11, bf16x3 17 / 10; 64 (m = n = 1000, k = 300)
// FP64 74 / 31, bf16x3 30 / 16; 144 (1536, 512) FP64 90 / 78, FP32 47 / 42, bf16x3 32 / 25; 256 (2048, 1024) FP64 175 / 191,
// FP32 92 / 97, bf16x3 62 / 53; 484 (2816, 512) FP64 158 / 191, FP32 81 / 97, bf16x3 44 / 54. Short products move mostly C,
// and from 512 64x64 items (two on each CU) on, those gain nothing on it: 144 items, k = 16 FP64 14.2 / 15.2, k = 48 18.7 / 18.7,
// k = 64 21.0 / 17.8; FP32 k = 16 9.1 / 11.2, k = 32 8.3 / 12.1, k = 48 11.5 / 13.2, k = 64 10.5 / 9.9 (121 items, k = 16 FP64
// 13.9 / 10.2). Long bf16 products are bound by their operands, which these items read twice as often: 256 items, k =
// 1024 37.8 / 37.2, 2048 66.0 / 67.0, 8192 238 / 255; 196 (1792) 1024 36.7 / 38.3, 8192 237 / 260, but ragged (1700) 4096 189 / 164.
__host__ __device__ inline bool raw_gemm_small(int prec, int m, int n, int K, bool syrk) {
    const long items = raw_gemm_items(m, n, syrk, GEMM_BM);
    if (prec == P_F64 || prec == P_F32) return items <= (K < 64 ? 128 : 192);
    if (prec == P_BF16 && K > 1024 && raw_gemm_items(m, n, syrk, GEMM_BS) > 768) return false;
    return items <= 256;
}

// Whether a raw TRSM of m rows and n columns takes the strips that keep X in LDS. These are half as high, so L is read twice
// as often: they pay while all strips run at once (two on each of 256 CUs), where the time is one strip's chain, and behind
// that as long as the chain is long. Measured, us of the other form / of this one: FP64 n = 512, 512 strips (m = 8192)
// 101 / 83, 768 130 / 119, 875 148 / 144, 1024 132 / 147, 4096 426 / 522; n = 256, 512 strips 36.7 / 36.6, 768 45.7 /
// 48.6, 1024 51.5 / 60.1; n = 64, 1024 17.4 / 19.9, 16384 98 / 130. FP32 n = 512, 512 strips (m = 16384) 108 / 84, 625 148
// / 123, 1250 230 / 187, 8192 1145 / 1064; n = 256, 512 40.5 / 37.1, 1024 55.6 / 62.0, 1250 88.9 / 74.4; n = 128, 512 22.9 /
// 22.2, 1024 27.2 / 32.1, 8192 143 / 160.
__host__ __device__ inline bool trsm_in_lds(int elem_bytes, int m, int n) {
    const int rows = trsm_rows(elem_bytes, true);
    const long strips = ((long)m + rows - 1) / rows;
    if (n > TRSM_LDS_COLS) return false;
    return strips <= 512 || (elem_bytes == 8 ? n > 256 && strips < 1024 : n >= 256);
}

// Addresses of the TRSM items that keep X in LDS: a wave-uniform 64-bit base and a lane's offset of 32 bits, which spans
// 16 columns of X, or 4 of L, whatever the column block (leading dimensions are below TRSM_LDS_MAX_LD).
constexpr long TRSM_LDS_MAX_LD = 1 << 24;
// The column of a block of cw columns at which wave w's part of the right-hand side begins (the last one for waves
// behind the block's end).
__host__ __device__ inline int trsm_wave_col(int w, int cw) { return 16 * w < cw ? 16 * w : cw - 1; }
// Bytes from there to row `row` of the wave's column c, 0 .. 15 (clamped to the block's last).
__host__ __device__ inline unsigned trsm_lane_offset(int row, int c, int w, int cw, long ldx, int elem_bytes) {
    const int left = cw - 1 - trsm_wave_col(w, cw);
    return ((unsigned)row + (unsigned)(c < left ? c : left) * (unsigned)ldx) * (unsigned)elem_bytes;
}
static_assert((15 * (TRSM_LDS_MAX_LD - 1) + TRSM_BM_F32) * 8 < (1LL << 32), "a lane's offset in X");
static_assert((3 * (TRSM_LDS_MAX_LD - 1) + TRSM_LDS_COLS) * 8 < (1LL << 32), "a lane's offset in L");

// The items of POTRF of an n x n tile (item_potrf), numbered row by row of 64x64 blocks: row r has r of them (row 0 one),
// the blocks (r, q), q < r - 1, and last its tail item, which owns (r, r-1) and (r, r).
__host__ __device__ inline int potrf_blocks(int n) { return (n + DB - 1) / DB; }
__host__ __device__ inline int potrf_items(int n) { return 1 + potrf_blocks(n) * (potrf_blocks(n) - 1) / 2; }
struct PotrfItem {
    int r, q;   // its off-diagonal block (row 0 has none: q = -1)
    bool tail;  // it owns the diagonal block (r, r) too
};
__host__ __device__ inline PotrfItem potrf_item(int it) {
    int r = 0, rem = it;
    while (rem >= (r > 1 ? r : 1)) {
        rem -= r > 1 ? r : 1;
        r++;
    }
    const bool tail = rem == (r > 1 ? r : 1) - 1;
    return {r, tail ? r - 1 : rem, tail};
}
// Flags of a tile: one per block, and behind them the count of finished items (the last one clears them for the next run).
__host__ __device__ inline int potrf_flag(int r, int q) { return r * (r + 1) / 2 + q; }
__host__ __device__ inline int potrf_fin(int n) { return potrf_flag(potrf_blocks(n), 0); }
__host__ __device__ inline int potrf_flags(int n) { return potrf_fin(n) + 1; }

// One tiled symmetric matrix in HBM. Tile (i,j), i >= j, is a column-major
// bsz[i] x bsz[j] array with leading dimension bsz[i] (block_sizes_lda,
// 2d_cholesky.cpp:86-89), reached through the pointer table.
struct DevMat {
    int32_t nt;
    int32_t storage;  // P_F64 or P_F32
    const int32_t* bsz;
    const int32_t* boff;
    void* const* tiles;    // [nt*nt], entry i + j*nt
    double* const* dinv;   // [nt]: inverses of the 64x64 diagonal blocks of L_jj (FP64, 64x64 each, ld 64)
    int32_t* info;         // first non-positive pivot, 1-based global column; 0 = none
    int32_t* pflags;       // [nt * pf_stride]: flags of the POTRF items of each diagonal tile (zero between runs)
    int32_t pf_stride;     // ints per tile: potrf_flags of the largest tile
    int32_t* locks;        // [nt * nt * 16]: accumulate-mode sub-tile locks of tile (i, j) (zero when free)
    // [nt*nt] or null: bf16 hi/lo planes of the off-diagonal FP32 tiles (i > j, bsz[j] % 32 == 0; other
    // entries null), written by the TRSM items that produce the tile and read by the bf16x3 GEMM items.
    // Tile (i, j) with m = bsz[i] rows: 16-byte granule ((c*2 + p)*4 + g)*m + r holds bf16 plane p
    // (0: hi = bf16(x), 1: lo = bf16(x - hi), both rounded to nearest even) of columns 32c + 8g ... +7 of row r.
    void* const* planes;
};
// bf16 split planes: granule of (chunk of 32 columns, plane, 8-column group, row) in a tile of m rows.
__host__ __device__ inline long plane_granule(int c, int p, int g, int r, int m) {
    return ((long)(c * 2 + p) * 4 + g) * m + r;
}

constexpr int KSPAN_MAX = 8;  // steps of one fused update at most

// The operands of a GEMM/SYRK task, C(i,j) -= A(i,k) B(j,k)^T, resolved from the matrix's tile tables
// before a run, so that an item finds them in one load with its task record instead of through the
// matrix descriptor and its pointer tables (two more dependent memory round trips).
struct alignas(16) GemmOperands {
    const void* A;
    const void* B;
    void* C;
    const void* PA;  // bf16 planes of A and B (null: none)
    const void* PB;
    int32_t m, n, K, pad;
};

// Device task record.
struct DevTask {
    int32_t kind;
    int32_t prec;
    int32_t mat;
    int32_t n_items;
    int32_t i, j, k;
    int32_t bucket;
    int32_t crit;  // on a longest path of the DAG: runs with no other item started on its CU
    int32_t accum; // GEMM/SYRK: add the product into C under the sub-tile lock (accumulate mode)
    int32_t edge_off, edge_cnt;  // its out-edges in DevGraph::edges
    int32_t kspan; // GEMM/SYRK: steps k .. k + kspan - 1 in one task (fused updates of one tile), at most KSPAN_MAX
    int32_t sub;   // GEMM/SYRK: rows and columns of an item, GEMM_BM or GEMM_BS; TRSM: GEMM_BS = items that keep X in LDS
};

// An out-edge of the graph with all that releasing its target takes: the task that completes reads it in one access
// instead of the target's id, record and queue bounds in turn.
struct alignas(16) DevEdge {
    int32_t succ;     // target task
    int32_t n_items;  // its work items
    int32_t bucket;   // its queue
    int32_t base;     // first slot of that queue in q_items
    int32_t cap;      // slots of that queue
    int32_t pad[3];
};

// Work items per task of tiles with elem_bytes-byte elements; host and device must agree.
// (sub: as DevTask::sub).
__host__ __device__ inline int items_of(int kind, int bi, int bj, int elem_bytes, int sub = GEMM_BM) {
    if (kind == K_POTRF) return 1;
    if (kind == K_TRSM) {
        const int rows = trsm_rows(elem_bytes, sub == GEMM_BS);
        return (bi + rows - 1) / rows;
    }
    const int tr = (bi + sub - 1) / sub;
    if (kind == K_SYRK) return tr * (tr + 1) / 2;
    if (kind == K_GEMM) return tr * ((bj + sub - 1) / sub);
    return 1;
}

}  // namespace ttad
