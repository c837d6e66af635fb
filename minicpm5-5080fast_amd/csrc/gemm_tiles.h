// gemm_tiles.h - the tile GEMM of the prefill projections (gemm_tiles.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kv_common.h"
#include "minicpm_runtime.h"

namespace mckv {

// y[M][N] = bf16(x[M][K] . w[N][K]^T), or with swiglu (w [2N][K]: gate rows,
// then up rows) y = bf16(silu(bf16 g) * bf16 u), or (part != nullptr, y
// unused) the fp32 sums of each K split in part[split][M][N]. Rows are
// contiguous, pointers 16-byte aligned.
// With rope (the qkv projection, N = kRow, y the qkv rows): the q heads are
// rotated into y, the rotated k and the v heads go to their tokens' pages, and
// the k / v columns of y, not written, hold each row's cos / sin pairs
// (mc_kv_rope_table).
struct RopeAppend {
    const uint32_t* base_pos = nullptr;    // row m is position *base_pos + row0 + m
    const uint32_t* page_table = nullptr;  // nullptr: no rope
    uint16_t* pool = nullptr;
    DevLayout ly{};
    uint32_t layer = 0u, row0 = 0u;
};
struct GemmTiles {
    const uint16_t* x;
    const uint16_t* w;
    uint16_t* y;
    float* part;
    uint32_t M, N, K;
    bool swiglu;
    RopeAppend rope{};
};
// How one projection runs: rows 0..rows0 - 1 on tile shape shape0 (an index
// into the table of gemm_tiles.hip), the rest (rows0 < M) on shape1 in a
// second launch; splits > 1 only with rows0 == M. splits = 0: no plan.
struct GemmPlan {
    uint32_t rows0 = 0u, shape0 = 0u, shape1 = 0u, splits = 0u;
};
// What a tile does with its sums.
enum class TileEnd : uint32_t { kPlain, kSwiglu, kRope };
// Plan of least estimated time, min_splits <= splits <= max_splits (1 but for
// kPlain); *us its estimate when non-null. N a multiple of 64, K of 128.
GemmPlan gemm_tiles_plan(uint32_t M, uint32_t N, uint32_t K, TileEnd end, uint32_t min_splits,
                         uint32_t max_splits, float* us = nullptr);
bool gemm_tiles_fits(uint32_t shape, uint32_t K, TileEnd end, uint32_t splits);
mc_status_t gemm_tiles(const GemmTiles& g, const GemmPlan& p, hipStream_t st);

}  // namespace mckv
