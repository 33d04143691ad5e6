// kd_mm_kernel.h - launch arguments shared by the host glue (kd_mm_host.cpp)
// and the gfx950 matrix-product kernels (kd_mm_kernel.hip).  Internal to
// libkd_fa.so.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace kdfa {

// Largest workgroup tile of the product: 256 rows of x (tokens) by 256 rows
// of w (outputs), 32 k per stage.
constexpr int kMmBM = 256;
constexpr int kMmBN = 256;
constexpr int kMmBK = 32;

struct MmArgs {
    const char *w;       // BF16 rows [N][K], row stride w_nb1 bytes
    const char *x;       // F32 or BF16 rows [M][K], row stride x_nb1 bytes
    const float *bias;   // F32 [N] or nullptr
    char *dst;           // F32 rows [M][N], row stride d_nb1 bytes
    int64_t w_nb1, x_nb1, d_nb1;
    int32_t M, N, K;
    // the tiles, and the output tiles per column of their order (not used by
    // mm_skinny)
    int32_t tiles_m, tiles_n, n_blocks, cols;
};

// Enqueue the product (x F32 when x_f32, else BF16) with tiles of 256 outputs
// x 256 (tile 88) or 128 tokens (84).
hipError_t launch_mm(const MmArgs &a, int tile, bool x_f32, hipStream_t stream);

// Enqueue the few-token kernels (kd_mm_ksplit.hip): mm_skinny (M <= 16), and
// mm_ksplit with tiles of 32 * (tile / 10) outputs x 32 * (tile % 10) tokens
// (tile 11, 21, 22, 23, 42, 43 or 44).
constexpr int kMmSkinnyRows = 16;
constexpr int64_t kMmMaxBlocks = 1 << 23;   // workgroups of 256 threads in one launch, with room to spare
hipError_t launch_mm_skinny(const MmArgs &a, bool x_f32, hipStream_t stream);
hipError_t launch_mm_ksplit(const MmArgs &a, int tile, bool x_f32, hipStream_t stream);

struct DqArgs {
    const char *w;       // weight rows [N], row stride w_nb1 bytes
    int64_t w_nb1;
    int32_t type;        // KD_MM_TYPE_*
    int32_t N, K;
    char *out;           // BF16 rows [N][K], back to back
};

// Enqueue the expansion of a weight to BF16 rows.
hipError_t launch_dequant(const DqArgs &a, hipStream_t stream);

}  // namespace kdfa
