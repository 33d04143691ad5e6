// kd_mm_host.cpp - C ABI of the linear-layer product (include/kd_mm.h):
// validation of the GGML_OP_MUL_MAT node as ops::linear builds it
// (src/core/ops.hpp:27-43), the weight expansion and the product launch.
// Nothing here allocates device memory, synchronises or keeps pointers past
// the call.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "../../include/kd_mm.h"
#include "kd_fa_kernel.h"
#include "kd_mm_kernel.h"

namespace {

constexpr int64_t kI32Max = 0x7fffffff;
constexpr uint64_t kU32Max = 0xffffffffull;

bool is_16b(uint64_t x) { return (x & 15u) == 0; }
bool is_16b(const void *p) { return is_16b(reinterpret_cast<uintptr_t>(p)); }

// bytes of one 32-element block of a weight row
int64_t block_bytes(int type) {
    switch (type) {
    case KD_MM_TYPE_Q8_0: return 34;
    case KD_MM_TYPE_Q4_0: return 18;
    case KD_MM_TYPE_F16:
    case KD_MM_TYPE_BF16: return 64;
    case KD_MM_TYPE_F32: return 128;
    default: return 0;
    }
}

// Weight tensor [K, N]: a known type, K a multiple of 32, rows of at least
// K/32 blocks; quantized rows 2-byte aligned, float rows 16-byte aligned.
int check_w(const kd_fa_tensor &w) {
    if (!w.data) return KD_FA_ERR_NULL;
    const int64_t bb = block_bytes(w.type);
    if (bb == 0) return KD_FA_ERR_TYPE;
    const int64_t K = w.ne[0], N = w.ne[1];
    if (K <= 0 || N < 0 || w.ne[2] != 1 || w.ne[3] != 1) return KD_FA_ERR_SHAPE;
    if (K % 32 != 0 || K > kI32Max || N > kI32Max) return KD_FA_ERR_SHAPE;
    const bool quant = w.type == KD_MM_TYPE_Q8_0 || w.type == KD_MM_TYPE_Q4_0;
    const uint64_t row = (uint64_t)(K / 32) * (uint64_t)bb;
    if (quant) {
        if (w.nb[0] != (size_t)bb) return KD_FA_ERR_LAYOUT;
        if ((w.nb[1] & 1u) || (reinterpret_cast<uintptr_t>(w.data) & 1u)) return KD_FA_ERR_LAYOUT;
    } else {
        if (w.nb[0] != (size_t)(bb / 32)) return KD_FA_ERR_LAYOUT;
        if (!is_16b(w.nb[1]) || !is_16b(w.data)) return KD_FA_ERR_LAYOUT;
    }
    if (w.nb[1] < row) return KD_FA_ERR_LAYOUT;
    return KD_FA_OK;
}

// rows of a [ne0, ne1, ne2, ne3] view flattened as ops::linear's reshape
// (contiguous beyond the rows); 0 on a layout it cannot flatten
int64_t flat_rows(const kd_fa_tensor &t) {
    if (t.ne[1] < 0 || t.ne[2] < 1 || t.ne[3] < 1) return -1;
    if (t.ne[2] > 1 && t.nb[2] != t.nb[1] * (size_t)t.ne[1]) return -1;
    if (t.ne[3] > 1 && t.nb[3] != t.nb[2] * (size_t)t.ne[2]) return -1;
    return t.ne[1] * t.ne[2] * t.ne[3];
}

int validate(const kd_mm_desc *d) {
    if (!d) return KD_FA_ERR_NULL;
    int st = check_w(d->w);
    if (st != KD_FA_OK) return st;
    const kd_fa_tensor &x = d->x, &o = d->dst, &b = d->bias;
    if (!x.data || !o.data) return KD_FA_ERR_NULL;
    if (x.type != KD_MM_TYPE_F32 && x.type != KD_MM_TYPE_BF16) return KD_FA_ERR_TYPE;
    if (o.type != KD_MM_TYPE_F32) return KD_FA_ERR_TYPE;
    if (b.data && b.type != KD_MM_TYPE_F32) return KD_FA_ERR_TYPE;
    const int64_t K = d->w.ne[0], N = d->w.ne[1];
    if (x.ne[0] != K || o.ne[0] != N) return KD_FA_ERR_SHAPE;
    const int64_t M = flat_rows(x);
    if (M < 0 || flat_rows(o) != M) return KD_FA_ERR_LAYOUT;
    if (o.ne[1] != x.ne[1] || o.ne[2] != x.ne[2] || o.ne[3] != x.ne[3]) return KD_FA_ERR_SHAPE;
    if (M > kI32Max) return KD_FA_ERR_SHAPE;
    if (N % 4 != 0) return KD_FA_ERR_SHAPE;
    if (b.data && (b.ne[0] != N || b.ne[1] != 1 || b.ne[2] != 1 || b.ne[3] != 1)) return KD_FA_ERR_SHAPE;
    // rows 16-byte aligned, elements contiguous
    const size_t xe = x.type == KD_MM_TYPE_F32 ? 4 : 2;
    if (x.nb[0] != xe || o.nb[0] != 4) return KD_FA_ERR_LAYOUT;
    if (!is_16b(x.data) || !is_16b(x.nb[1]) || !is_16b(o.data) || !is_16b(o.nb[1])) return KD_FA_ERR_LAYOUT;
    if (b.data && (!is_16b(b.data) || b.nb[0] != 4)) return KD_FA_ERR_LAYOUT;
    // a 256-row tile is addressed with 32-bit offsets from its first row
    if ((uint64_t)x.nb[1] * kdfa::kMmBM > kU32Max) return KD_FA_ERR_LAYOUT;
    if ((uint64_t)K * 2 * kdfa::kMmBN > kU32Max) return KD_FA_ERR_LAYOUT;
    if (d->w.type == KD_MM_TYPE_BF16 && (uint64_t)d->w.nb[1] * kdfa::kMmBN > kU32Max) return KD_FA_ERR_LAYOUT;
    return KD_FA_OK;
}

// w BF16 with 16-byte aligned rows is multiplied as stored
bool w_direct(const kd_fa_tensor &w) {
    return w.type == KD_MM_TYPE_BF16 && is_16b(w.data) && is_16b(w.nb[1]);
}

size_t ws_bytes(const kd_mm_desc *d) {
    return w_direct(d->w) ? 0 : (size_t)d->w.ne[0] * (size_t)d->w.ne[1] * 2;
}

// The tile of a call (32 * (tile / 10) outputs x 32 * (tile % 10) tokens) of
// more than kMmSkinnyRows tokens: the one whose rounds of workgroups (256 at
// once, one per CU) take least time.  A round's time with every CU at it, F32
// x, is `fixed` (first loads, sums and stores) + `us` * K / 4096.  Small tiles
// move more bytes per product, large ones leave CUs idle.  (Without the fixed
// part calls of few k and many tiles took too small a tile: 5,000 x 4096 x 32
// 36 us against 28.)  The large tiles' fixed part is mostly stores, in
// proportion to the outputs there are (60,000 tokens, K = 32, one round: 8.3
// us with 4 outputs, 11.0 with 64, 16 with 256; taken as 12 for any, 60,000 x
// 4 x 32 ran in 32 x 32 tiles, 11.4 us).  And the rounds take no less than x
// from HBM (5.6 TB/s): then rounds cost their fixed parts only, and the fewest
// do best (60,000 x 64 x 512, F32 x, 27.0 us in one round of 256 x 256, 28.9
// in four of 64 x 64).  F32 x and BF16 x take the same tile, so that F32 x has
// the bits of its rounding: the table is F32 x's, the stream BF16 x's (with
// F32 x's 61,442 x 64 x 4096 would gain 3% at F32 x and lose 19% at BF16).
// BF16 x's times are 0.4-1.1 of the table's: over 225 shapes (17 to 63,488 tokens, 4 to
// 16,384 outputs, K 32 to 16,384) the tile taken is in the mean 1.8% (F32 x)
// and 0.9% (BF16) slower than the fastest of the nine, at worst 27%.
int choose_tile(int64_t M, int64_t N, int64_t K) {
    constexpr struct { int tile, n, m; double fixed, us; } kTiles[] = {
        {88, 256, 256, 12.0, 110.0}, {84, 256, 128, 7.0, 69.0}, {44, 128, 128, 6.0, 37.0},
        {43, 128, 96, 5.0, 31.0},    {42, 128, 64, 4.0, 23.5},  {23, 64, 96, 3.5, 23.5},
        {22, 64, 64, 2.5, 16.5},     {21, 64, 32, 1.7, 10.8},   {11, 32, 32, 1.2, 7.8}};
    const double stream = (double)M * (double)K * 2.0 / 5.6e6;   // us
    int best = 88;
    double least = 1e300;
    for (const auto &t : kTiles) {
        const int64_t tiles = ((N + t.n - 1) / t.n) * ((M + t.m - 1) / t.m);
        if (t.tile != 88 && tiles > kdfa::kMmMaxBlocks) continue;
        const double stores = t.n == 256 ? 0.45 + 0.55 * (double)std::min<int64_t>(N, t.n) / t.n : 1.0;
        const double rounds = (double)((tiles + 255) / 256);
        const double cost = rounds * t.fixed * stores + std::max(rounds * t.us * (double)K / 4096.0, stream);
        if (cost < least) { least = cost; best = t.tile; }
    }
    return best;
}

hipError_t dequant(const kd_fa_tensor &w, void *out, hipStream_t s) {
    kdfa::DqArgs a;
    a.w = static_cast<const char *>(w.data);
    a.w_nb1 = (int64_t)w.nb[1];
    a.type = w.type;
    a.K = (int32_t)w.ne[0];
    a.N = (int32_t)w.ne[1];
    a.out = static_cast<char *>(out);
    return kdfa::launch_dequant(a, s);
}

}  // namespace

extern "C" {

int kd_mm_supports(const kd_mm_desc *desc, int *reason) {
    const int st = validate(desc);
    if (reason) *reason = st;
    return st == KD_FA_OK ? 1 : 0;
}

size_t kd_mm_workspace_size(const kd_mm_desc *desc) {
    if (validate(desc) != KD_FA_OK) return 0;
    return ws_bytes(desc);
}

int kd_mm_dequant(const kd_fa_tensor *w, void *out, size_t out_bytes, void *stream) {
    if (!w || !out) return KD_FA_ERR_NULL;
    const int st = check_w(*w);
    if (st != KD_FA_OK) return st;
    if (!is_16b(out) || out_bytes < (size_t)w->ne[0] * (size_t)w->ne[1] * 2) return KD_FA_ERR_LAYOUT;
    if (w->ne[1] == 0) return KD_FA_OK;
    const int dv = kdfa::device_gfx950();
    if (dv != KD_FA_OK) return dv;
    return dequant(*w, out, static_cast<hipStream_t>(stream)) == hipSuccess ? KD_FA_OK : KD_FA_ERR_LAUNCH;
}

int kd_mm_run(const kd_mm_desc *desc, void *workspace, size_t workspace_bytes, void *stream) {
    int st = validate(desc);
    if (st != KD_FA_OK) return st;
    const size_t need = ws_bytes(desc);
    if (need) {
        if (!workspace) return KD_FA_ERR_NULL;
        if (!is_16b(workspace) || workspace_bytes < need) return KD_FA_ERR_LAYOUT;
    }
    const int64_t K = desc->w.ne[0], N = desc->w.ne[1], M = flat_rows(desc->x);
    if (M == 0 || N == 0) return KD_FA_OK;
    st = kdfa::device_gfx950();
    if (st != KD_FA_OK) return st;
    hipStream_t hs = static_cast<hipStream_t>(stream);

    kdfa::MmArgs a;
    if (need) {
        if (dequant(desc->w, workspace, hs) != hipSuccess) return KD_FA_ERR_LAUNCH;
        a.w = static_cast<const char *>(workspace);
        a.w_nb1 = K * 2;
    } else {
        a.w = static_cast<const char *>(desc->w.data);
        a.w_nb1 = (int64_t)desc->w.nb[1];
    }
    a.x = static_cast<const char *>(desc->x.data);
    a.x_nb1 = (int64_t)desc->x.nb[1];
    a.bias = static_cast<const float *>(desc->bias.data);
    a.dst = static_cast<char *>(desc->dst.data);
    a.d_nb1 = (int64_t)desc->dst.nb[1];
    a.M = (int32_t)M;
    a.N = (int32_t)N;
    a.K = (int32_t)K;
    a.tiles_m = a.tiles_n = a.n_blocks = a.cols = 0;
    const bool x_f32 = desc->x.type == KD_MM_TYPE_F32;
    hipError_t e;
    if (M <= kdfa::kMmSkinnyRows && N <= 32 * kdfa::kMmMaxBlocks) {
        e = kdfa::launch_mm_skinny(a, x_f32, hs);
    } else {
        // (counted in 64 bits: M and N may be within a tile of 2^31)
        const int tile = choose_tile(M, N, K);
        const int64_t tiles_n = (N + 32 * (tile / 10) - 1) / (32 * (tile / 10));
        const int64_t tiles_m = (M + 32 * (tile % 10) - 1) / (32 * (tile % 10));
        if (tiles_n * tiles_m > kI32Max) return KD_FA_ERR_SHAPE;
        a.tiles_n = (int32_t)tiles_n;
        a.tiles_m = (int32_t)tiles_m;
        a.n_blocks = (int32_t)(tiles_n * tiles_m);
        const bool big = tile == 88 || tile == 84;
        // columns of 4 output tiles (of 1, 2, 16: 3-8% slower at 63,488 x
        // 4096 x 4096), or with the large tiles all of up to 8
        a.cols = big && tiles_n <= 8 ? a.tiles_n : 4;
        e = big ? kdfa::launch_mm(a, tile, x_f32, hs) : kdfa::launch_mm_ksplit(a, tile, x_f32, hs);
    }
    return e == hipSuccess ? KD_FA_OK : KD_FA_ERR_LAUNCH;
}

}  // extern "C"
