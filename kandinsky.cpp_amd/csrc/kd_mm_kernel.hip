// kd_mm_kernel.hip - gfx950 kernels of the CrossDiT linear layers
// (ops::linear, src/core/ops.hpp:27-43: ggml_mul_mat(w, x) + bias):
//
//   dequant_kernel  expands Q4_0 / Q8_0 / F16 / F32 weight rows to BF16 in
//                   the F32 arithmetic of ggml's dequantize_row_q4_0 / _q8_0
//   mm_bf16         dst[m][n] = sum_k w[n][k] x[m][k] (+ bias[n]) on
//                   v_mfma_f32_16x16x32_bf16, F32 accumulation
//
// The product computes D^T = W X^T: A = W (outputs on M), B = X^T (tokens
// on N), so that each lane ends with 4 consecutive outputs of one token --
// 16-byte pieces of a dst row.  Both operands are k-contiguous rows, which
// is exactly the MFMA operand form (A: lane l holds row l%16, k 8*(l/16)..
// +7; B: column l%16, the same k) -- no transposes anywhere.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/kd_mm.h"
#include "kd_fa_device.h"
#include "kd_mm_kernel.h"

namespace kdfa {

// ---------------------------------------------------------------------------
// dequant_kernel: weight rows -> BF16 rows (F32 value, then round to
// nearest even).  Q8_0 block: F16 d, 32 x int8 q; value = q * d.  Q4_0
// block: F16 d, 16 bytes whose low nibble is element j and high nibble
// element j + 16; value = (nibble - 8) * d (convert_to_gguf.py:121-123 and
// ggml's dequantize_row_q4_0 use this layout).
//
// Bound by HBM.  A thread makes 8 elements, one 16-byte store, so that a
// wave's stores are whole lines (a block per thread wrote 64 bytes apart),
// from one 8-byte load of the quants (2-byte aligned, as the blocks are) and
// d; four such chunks, 256 apart, are loaded before the first is stored.
// Flat: the rows lie back to back, so that a chunk's block is its index / 4
// without a division.  16384 x 4096: Q4_0
// 54.7 -> 32.4 us (5.3 TB/s read and written), Q8_0 59.2 -> 36.9; 4096 x 4096
// Q8_0 15.6 -> 8.7.
// ---------------------------------------------------------------------------
constexpr int kDqChunks = 4;   // chunks of 8 elements per thread and round

template <int TYPE> struct DqSrc;   // 8 elements as loaded
template <> struct DqSrc<KD_MM_TYPE_Q8_0> { uint16_t d; uint32_t q[2]; };
template <> struct DqSrc<KD_MM_TYPE_Q4_0> { uint16_t d; uint32_t q[2]; };
template <> struct DqSrc<KD_MM_TYPE_F16> { f16x8 h; };
template <> struct DqSrc<KD_MM_TYPE_BF16> { u32x4 w; };
template <> struct DqSrc<KD_MM_TYPE_F32> { f32x4 u, v; };

// chunk c (0-3) of the block at p
template <int TYPE>
static __device__ __forceinline__ DqSrc<TYPE> dq_load(const char *p, int c) {
    DqSrc<TYPE> s;
    if constexpr (TYPE == KD_MM_TYPE_Q8_0 || TYPE == KD_MM_TYPE_Q4_0) {
        s.d = *reinterpret_cast<const uint16_t *>(p);
        __builtin_memcpy(s.q, __builtin_assume_aligned(p + 2 + 8 * (TYPE == KD_MM_TYPE_Q8_0 ? c : c & 1), 2), 8);
    } else if constexpr (TYPE == KD_MM_TYPE_F16) {
        s.h = *reinterpret_cast<const f16x8 *>(p + 16 * c);
    } else if constexpr (TYPE == KD_MM_TYPE_BF16) {
        s.w = ld16(p + 16 * c);
    } else {
        s.u = *reinterpret_cast<const f32x4 *>(p + 32 * c);
        s.v = *reinterpret_cast<const f32x4 *>(p + 32 * c + 16);
    }
    return s;
}

template <int TYPE>
static __device__ __forceinline__ u32x4 dq_round(const DqSrc<TYPE> &s, int c) {
    float v[8];
    if constexpr (TYPE == KD_MM_TYPE_Q8_0) {
        const float d = (float)__builtin_bit_cast(_Float16, s.d);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = (float)(int8_t)(s.q[e >> 2] >> (8 * (e & 3))) * d;
    } else if constexpr (TYPE == KD_MM_TYPE_Q4_0) {
        const float d = (float)__builtin_bit_cast(_Float16, s.d);
        const int sh = c >= 2 ? 4 : 0;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = (float)((int)((s.q[e >> 2] >> (8 * (e & 3) + sh)) & 15) - 8) * d;
    } else if constexpr (TYPE == KD_MM_TYPE_F16) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = (float)s.h[e];
    } else if constexpr (TYPE == KD_MM_TYPE_BF16) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[2 * e] = Elem<__bf16>::lo(s.w[e]);
            v[2 * e + 1] = Elem<__bf16>::hi(s.w[e]);
        }
    } else {
        v[0] = s.u.x; v[1] = s.u.y; v[2] = s.u.z; v[3] = s.u.w;
        v[4] = s.v.x; v[5] = s.v.y; v[6] = s.v.z; v[7] = s.v.w;
    }
    u32x4 w;
#pragma unroll
    for (int e = 0; e < 4; ++e) w[e] = Elem<__bf16>::pack2(v[2 * e], v[2 * e + 1]);
    return w;
}

template <int TYPE, bool FLAT>
__global__ __launch_bounds__(256) void dequant_kernel(DqArgs a) {
    constexpr int kBlock = TYPE == KD_MM_TYPE_Q8_0 ? 34 : TYPE == KD_MM_TYPE_Q4_0 ? 18 : TYPE == KD_MM_TYPE_F32 ? 128 : 64;
    const int nbk = a.K / 32;
    const int64_t n_chunks = (int64_t)a.N * nbk * 4;
    const int64_t round = (int64_t)gridDim.x * (256 * kDqChunks);
    const int c = threadIdx.x & 3;
    for (int64_t i0 = (int64_t)blockIdx.x * (256 * kDqChunks) + threadIdx.x; i0 < n_chunks; i0 += round) {
        DqSrc<TYPE> s[kDqChunks];
#pragma unroll
        for (int u = 0; u < kDqChunks; ++u) {
            // past the end, the last block again (not stored)
            const int64_t i = i0 + 256 * u < n_chunks ? i0 + 256 * u : n_chunks - 4 + c;
            const int64_t blk = i >> 2;
            const char *p;
            if constexpr (FLAT)
                p = a.w + blk * kBlock;
            else
                p = a.w + (blk / nbk) * a.w_nb1 + (blk % nbk) * kBlock;
            s[u] = dq_load<TYPE>(p, c);
        }
#pragma unroll
        for (int u = 0; u < kDqChunks; ++u) {
            const int64_t i = i0 + 256 * u;
            if (i < n_chunks) *reinterpret_cast<u32x4 *>(a.out + i * 16) = dq_round<TYPE>(s[u], c);
        }
    }
}

template <int TYPE>
static void launch_dequant_t(const DqArgs &a, int64_t row, hipStream_t s) {
    const int64_t want = ((int64_t)a.N * (a.K / 8) + 256 * kDqChunks - 1) / (256 * kDqChunks);
    const dim3 grid((unsigned)(want < 65536 ? want : 65536));
    if (a.w_nb1 == row)
        hipLaunchKernelGGL((dequant_kernel<TYPE, true>), grid, dim3(256), 0, s, a);
    else
        hipLaunchKernelGGL((dequant_kernel<TYPE, false>), grid, dim3(256), 0, s, a);
}

hipError_t launch_dequant(const DqArgs &a, hipStream_t s) {
    const int64_t nbk = a.K / 32;
    switch (a.type) {
    case KD_MM_TYPE_Q8_0: launch_dequant_t<KD_MM_TYPE_Q8_0>(a, nbk * 34, s); break;
    case KD_MM_TYPE_Q4_0: launch_dequant_t<KD_MM_TYPE_Q4_0>(a, nbk * 18, s); break;
    case KD_MM_TYPE_F16: launch_dequant_t<KD_MM_TYPE_F16>(a, nbk * 64, s); break;
    case KD_MM_TYPE_BF16: launch_dequant_t<KD_MM_TYPE_BF16>(a, nbk * 64, s); break;
    case KD_MM_TYPE_F32: launch_dequant_t<KD_MM_TYPE_F32>(a, nbk * 128, s); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// mm_bf16: one workgroup = 4 waves (one per SIMD, 512 registers each) = a
// 256 (outputs) x 64 MB (tokens) tile of dst; wave w holds the 128 x 32 MB
// quarter (w & 1, w >> 1) as 8 x 2 MB accumulator blocks of 16 x 16 (256
// AGPRs at MB = 4).
//
// The products are v_mfma_f32_16x16x32_bf16: at full chip the power limit
// sets the rate, and on random operands 16 x 16 x 32 sustains 1,995 TFLOP/s
// against 1,700 for 32 x 32 x 16 (register operands only; on zeros 2,440 and
// 2,480).
//
// K advances 32 per stage.  With BF16 X, W (256 rows x 64 bytes) and X come
// by DMA (global_load_lds_dwordx4), kS - 1 stages ahead.  F32 X is loaded
// into registers two stages ahead of its rounding to BF16 and its way into
// one of two LDS buffers, so that it costs the LDS the same as BF16 X: read
// from LDS as F32, X alone kept it busy for 768 of a stage's 1,024 matrix
// cycles.  That leaves LDS for W in double stages of 64 k, whole 128-byte
// lines of its rows: a line asked for in two halves a stage apart crosses
// from the L2 twice (from every CU, rows of 64 bytes arrive at 65 KB per
// microsecond and CU, of 128 at 128; 16,000 x 4096 x 16384 2.11 -> 1.85 ms).
// In LDS 16-byte chunk c of row r lies at c ^ ((r >> 2) & 3) (of a 128-byte
// row, at c ^ ((r >> 1) & 7)), which spreads the 16 rows of an operand read
// over the 64 banks.  The 64-byte rows still conflict (F32 x, 63,488 tokens:
// 7.5% of the cycles: the 16-byte reads are served for lanes 0-3, 12-15,
// 20-27 together, not for 16 in a row); a swizzle without conflicts did not
// change the time.
//
// Per stage a wave reads 8 W and 2 MB X fragments and issues 16 MB MFMAs in
// two halves (all W against half of X); the fragment reads of what follows,
// the DMAs of a later stage and X's loads, roundings and LDS writes are
// spread over them one by one (the reads in one burst behind the barrier:
// 10% more at BF16 x); the one barrier, between the halves, publishes the
// next stage.  The loop has no conditions; the last steps, apart, issue as
// many operations, all of one chunk where there is no stage left (bringing
// the last stage again cost 2-6% at K = 64, 1-4% at 4096).
//
// 63,488 x 4096 x 4096: F32 x 2.30 -> 1.99 ms, BF16 x 1.89 -> 1.69 ms
// against 32 x 32 x 16 products with F32 X read from LDS; 4,000 tokens, F32
// x, 149 -> 120 us.  The large calls run at the power limit (with every load
// taken out the products alone took 75% of the time).
// Rows past M or N read clamped (repeated) rows and are not stored.  The
// output goes through LDS so that its stores are whole 128-byte lines.
// ---------------------------------------------------------------------------
constexpr int kMmWaves = 4;
constexpr int kMmWTile = kMmBN * kMmBK * 2;   // 16 KiB

template <bool XF32, int MB>
__global__ __launch_bounds__(64 * kMmWaves) __attribute__((amdgpu_waves_per_eu(1, 1)))
void mm_bf16(MmArgs a) {
    typedef Elem<__bf16> E;
    typedef E::vec8 vec8;
    constexpr int BM = 64 * MB;
    constexpr int kXTile = BM * 64;                        // BF16 X rows of a stage
    constexpr int kS = MB == 4 ? 5 : 6;                    // BF16 X: stages of W and X in LDS
    constexpr int kWRing = 4;                              // F32 X: double stages of W (128-byte rows)
    constexpr int kXC = 2 * MB;                            // F32 X: 16-byte loads of a thread per stage
    constexpr int kXD = XF32 ? 0 : MB;                     // BF16 X: DMAs of a wave per stage
    constexpr int kVm = 4 + (XF32 ? kXC : kXD);            // vector memory operations of a wave per stage
    constexpr int kX0 = XF32 ? kWRing * 2 * kMmWTile : kS * kMmWTile;   // the X buffers behind W's
    constexpr int kUse = kX0 + (XF32 ? 2 : kS) * kXTile;
    constexpr int kEpi = kMmWaves * 8192 * MB;             // two blocks of 32 outputs per wave
    __shared__ __attribute__((aligned(1024))) char lds[kUse > kEpi ? kUse : kEpi];
    lds_t *const sbase = LDS_PTR(char, lds);

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15;
    const int q4 = lane >> 4;

    // tile: XCD-contiguous runs of tiles, dealt in columns of `cols` output
    // tiles (token tiles one after another within a column): the 32
    // workgroups an XCD runs at once then share 4 W tiles and 8 X tiles in
    // its L2
    const int pid = blockIdx.x;
    const int per = a.n_blocks >> 3;
    const int lid = pid < per * 8 ? (pid & 7) * per + (pid >> 3) : pid;
    const int col = lid / (a.tiles_m * a.cols), rem = lid - col * (a.tiles_m * a.cols);
    const int width = min(a.cols, a.tiles_n - col * a.cols);
    const int mt = rem / width;
    const int n0 = (col * a.cols + rem - mt * width) * kMmBN;
    const int m0 = mt * BM;

    // DMA lane offsets, relative to the tile's first row
    constexpr int kWD = XF32 ? 8 : 4;                      // W's DMAs of a wave per (double) stage
    uint32_t w_off[kWD], xd_off[XF32 ? 1 : MB], x_off[kXC];
    const int dr = lane >> 2, dc = (lane & 3) ^ ((lane >> 4) & 3);   // chunk dc of row 16 i + dr
    const int wc = (lane & 7) ^ ((4 * wave + (lane >> 4)) & 7);      // chunk wc of row 8 i + lane / 8 (double stages)
#pragma unroll
    for (int j = 0; j < kWD; ++j) {
        const int r = XF32 ? 8 * (wave + kMmWaves * j) + (lane >> 3) : 16 * (wave + kMmWaves * j) + dr;
        w_off[j] = (uint32_t)min(r, a.N - 1 - n0) * (uint32_t)a.w_nb1 + (uint32_t)((XF32 ? wc : dc) << 4);
    }
    if constexpr (XF32) {
        // load j of a thread: 4 F32 of row 8 (wave + 4 j) + lane / 8, to
        // x_wr + 2048 j of an X buffer
#pragma unroll
        for (int j = 0; j < kXC; ++j) {
            const int r = 8 * (wave + kMmWaves * j) + (lane >> 3);
            x_off[j] = (uint32_t)min(r, a.M - 1 - m0) * (uint32_t)a.x_nb1 + (uint32_t)((lane & 7) << 4);
        }
    } else {
#pragma unroll
        for (int j = 0; j < MB; ++j)
            xd_off[j] = (uint32_t)min(16 * (wave + kMmWaves * j) + dr, a.M - 1 - m0) * (uint32_t)a.x_nb1 + (uint32_t)(dc << 4);
    }
    const int xr = 8 * wave + (lane >> 3);
    const uint32_t x_wr =
        (uint32_t)(kX0 + xr * 64 + ((((lane & 7) >> 1) ^ ((xr >> 2) & 3)) << 4) + ((lane & 1) << 3));
    const char *const wtile = a.w + (int64_t)n0 * a.w_nb1;
    const char *const xtile = a.x + (int64_t)m0 * a.x_nb1;
    const int nk = a.K / kMmBK;
    // What a DMA or load of a stage past the last one brings, where one may
    // be (end): the tile's first chunk for every lane (not used), so that the
    // operations in flight stay as many, but not the traffic.
    // DMA j of stage kt (W's four, then BF16 X's) into buffer buf
    auto dma_j = [&](int kt, int buf, int j, auto end_c) __attribute__((always_inline)) {
        const bool past = decltype(end_c)::value && kt >= nk;
        const int64_t k64 = past ? 0 : (int64_t)kt * 64;
        if (j < 4)
            dma16(wtile + k64, past ? 0 : w_off[j], sbase + buf * kMmWTile + (wave + kMmWaves * j) * 1024);
        else if constexpr (!XF32)
            dma16(xtile + k64, past ? 0 : xd_off[j - 4], sbase + kX0 + buf * kXTile + (wave + kMmWaves * (j - 4)) * 1024);
    };
    const int nws = (nk + 1) >> 1;
    // DMA j (of 8) of double stage ws into ring buffer wb; past K, in a last
    // double stage with one half, the first half's chunks again
    auto dma_w2 = [&](int ws, int wb, int j, auto end_c) __attribute__((always_inline)) {
        const bool past = decltype(end_c)::value && ws >= nws;
        const uint32_t back = (nk & 1) && ws == nws - 1 && wc >= 4 ? 64u : 0u;
        dma16(wtile + (past ? 0 : (int64_t)ws * 128), past ? 0 : w_off[j] - back,
              sbase + wb * 32768 + (wave + kMmWaves * j) * 1024);
    };
    f32x4 xs[2][kXC];
    auto load_x = [&](int kt, int j, f32x4 &v, auto end_c) __attribute__((always_inline)) {
        const bool past = decltype(end_c)::value && kt >= nk;
        v = *reinterpret_cast<const f32x4 *>(xtile + (past ? 0 : (int64_t)kt * 128) + (past ? 0 : x_off[j]));
    };
    auto write_x = [&](int buf, int j, const f32x4 &v) __attribute__((always_inline)) {
        *reinterpret_cast<__attribute__((address_space(3))) u32x2 *>(sbase + x_wr + j * 2048 + buf * kXTile) =
            (u32x2){E::pack2(v.x, v.y), E::pack2(v.z, v.w)};
    };

    // fragments: lane l holds row l % 16, k 8 * (l / 16) .. +7 of the stage
    const int wn = wave & 1;
    const int wm = wave >> 1;
    const uint32_t f_rd = (uint32_t)(l16 * 64 + ((q4 ^ ((l16 >> 2) & 3)) << 4));
    const uint32_t a_rd = f_rd + 128 * wn * 64;
    const uint32_t b_rd = f_rd + kX0 + 32 * MB * wm * 64;
    f32x4 acc[8][2 * MB];
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 2 * MB; ++j) acc[i][j] = (f32x4){};
    vec8 fa[2][8], fb[2][MB];
    typedef const __attribute__((address_space(3))) vec8 lds_v8;
    const uint32_t a2_rd = (uint32_t)((128 * wn + l16) * 128 + ((q4 ^ ((l16 >> 1) & 7)) << 4));
    auto read_a = [&](int buf, auto p_c, int i) __attribute__((always_inline)) {
        constexpr int p = decltype(p_c)::value;
        if constexpr (XF32)   // buf: the ring buffer of the double stage; the second half's chunks are the first's ^ 4
            fa[p][i] = *reinterpret_cast<lds_v8 *>(sbase + buf * 32768 + (a2_rd ^ (p << 6)) + i * 2048);
        else
            fa[p][i] = *reinterpret_cast<lds_v8 *>(sbase + buf * kMmWTile + a_rd + i * 1024);
    };
    auto read_b = [&](int buf, auto h_c, int j) __attribute__((always_inline)) {
        constexpr int h = decltype(h_c)::value;
        fb[h][j] = *reinterpret_cast<lds_v8 *>(sbase + buf * kXTile + b_rd + (h * MB + j) * 1024);
    };
    // the products of W set p with half h of X; after product i, between(i)
    auto products = [&](auto p_c, auto h_c, auto between) __attribute__((always_inline)) {
        constexpr int p = decltype(p_c)::value, h = decltype(h_c)::value;
#pragma unroll
        for (int j = 0; j < MB; ++j)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][h * MB + j]) : "v"(fa[p][i]), "v"(fb[h][j]));
                __builtin_amdgcn_sched_barrier(0);
                between(8 * j + i);
                __builtin_amdgcn_sched_barrier(0);
            }
    };

    // The vector memory work of a stage interval (between two barriers), in
    // two halves.  The first, while a step's second products run: stage dk's
    // F32 X rounded from registers (set and buffer dk & 1 = xp) into LDS and
    // the registers loaded for stage dk + 2, or the first DMAs of BF16 stage
    // dk + kS - 2 into its buffer dbuf.  The second, while the next step's
    // first products run: half of a double stage of W, or the rest of those
    // DMAs.  (F32 x, 63,488 tokens: X and W mixed in both halves 2.20 ms
    // against 2.06.)
    constexpr int kWork0 = XF32 ? kXC : 2 + MB / 2, kWork1 = XF32 ? 4 : 2 + MB / 2;
    auto work0 = [&](int slot, int dk, int dbuf, auto xp_c, auto end_c) __attribute__((always_inline)) {
        constexpr int xp = decltype(xp_c)::value;
        if constexpr (XF32) {
            write_x(xp, slot, xs[xp][slot]);
            load_x(dk + 2, slot, xs[xp][slot], end_c);
        } else {
            dma_j(dk + kS - 2, dbuf, slot, end_c);
        }
    };
    auto work1 = [&](int slot, int dk, int dbuf, auto end_c) __attribute__((always_inline)) {
        if constexpr (XF32)
            dma_w2(((dk - 1) >> 1) + kWRing - 1, dbuf, 4 * ((dk - 1) & 1) + slot, end_c);
        else
            dma_j(dk + kS - 2, dbuf, kWork0 + slot, end_c);
    };
    // (as many stages as there are)
    if constexpr (XF32) {
#pragma unroll
        for (int s = 0; s < kWRing - 1; ++s)
            if (s < nws) {
#pragma unroll
                for (int j = 0; j < 8; ++j) dma_w2(s, s, j, BC<false>());
            }
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
            for (int j = 0; j < kXC; ++j) load_x(p, j, xs[p][j], BC<true>());
    } else {
#pragma unroll
        for (int s = 0; s < kS - 1; ++s)
            if (s < nk) {
#pragma unroll
                for (int j = 0; j < 4 + kXD; ++j) dma_j(s, s, j, BC<false>());
            }
    }
    // every stage issued so far has landed: the loop's first waits count on it
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if constexpr (XF32) {
#pragma unroll
        for (int j = 0; j < kXC; ++j) {
            write_x(0, j, xs[0][j]);
            load_x(2, j, xs[0][j], BC<true>());
        }
    }
#pragma unroll
    for (int slot = 0; slot < kWork0; ++slot) work0(slot, 1, kS - 1, IC<1>(), BC<true>());   // (F32 X: no buffer)
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 8; ++i) read_a(0, IC<0>(), i);
#pragma unroll
    for (int j = 0; j < MB; ++j) read_b(0, IC<0>(), j);
    // Step kt (p = kt & 1: W set, F32 X's buffer; buf = kt % kS, or the
    // double stage's ring buffer, (kt / 2) % kWRing).  Stage kt + 1 is
    // published in the middle, when every wave's reads of stage kt have
    // returned: what follows may overwrite its buffers.
    int buf = 0;
    auto step = [&](int kt, auto p_c, auto end_c) __attribute__((always_inline)) {
        constexpr int p = decltype(p_c)::value;
        constexpr int kRing = XF32 ? kWRing : kS;
        const int cur = buf, prev = buf == 0 ? kRing - 1 : buf - 1;
        __builtin_amdgcn_sched_barrier(0);
        products(p_c, IC<0>(), [&](int i) __attribute__((always_inline)) {
            if (i % 2 == 0 && i / 2 < MB) read_b(XF32 ? p : cur, IC<1>(), i / 2);
#pragma unroll
            for (int slot = 0; slot < kWork1; ++slot)
                if (1 + slot * (8 * MB) / kWork1 == i) work1(slot, kt + 1, prev, end_c);
        });
        if (!XF32 || p == 1) buf = buf == kRing - 1 ? 0 : buf + 1;
        // stage kt + 1 (W's double stage kt / 2 + 1) was issued kS - 2 (2
        // kWRing - 4) whole intervals ago; loads and DMAs complete in issue
        // order
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"((XF32 ? 2 * (kWRing - 2) : kS - 2) * kVm) : "memory");
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
        products(p_c, IC<1>(), [&](int i) __attribute__((always_inline)) {
            constexpr int kGap = MB == 4 ? 2 : 1;   // products between fragment reads
            if (i % kGap == 0) {
                const int r = i / kGap;
                if (r < 8)
                    read_a(buf, IC<1 - p>(), r);
                else if (r < 8 + MB)
                    read_b(XF32 ? 1 - p : buf, IC<0>(), r - 8);
            }
#pragma unroll
            for (int slot = 0; slot < kWork0; ++slot)
                if (1 + slot * (8 * MB) / kWork0 == i) work0(slot, kt + 2, cur, p_c, end_c);
        });
    };
    static_assert((XF32 ? 2 * (kWRing - 2) : kS - 2) * kVm <= 63, "vmcnt range");
    // the loop's steps issue stages that there are; the rest ask
    int kt = 0;
    for (; XF32 ? kt / 2 + kWRing - 1 < nws : kt + kS + 1 < nk; kt += 2) {
        step(kt, IC<0>(), BC<false>());
        step(kt + 1, IC<1>(), BC<false>());
    }
    for (; kt + 1 < nk; kt += 2) {
        step(kt, IC<0>(), BC<true>());
        step(kt + 1, IC<1>(), BC<true>());
    }
    if (kt < nk) step(kt, IC<0>(), BC<true>());
    // (the products are asm: the wait states between the last and a read of
    // its accumulators are ours to give, and the accumulators pass through
    // what follows the wait, so that no read of them can stand before it)
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_nop 15" ::: "memory");
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 2 * MB; ++j) asm volatile("; accumulator complete" : "+a"(acc[i][j]));
    __syncthreads();

    // ---- epilogue: dst[m][n .. n+3] = acc (+ bias) ----------------------------
    // Through LDS, one 32-output block (128 bytes of each of the wave's 32 MB
    // token rows) at a time: the lanes leave their 16-byte pieces in the
    // wave's own region (chunk index XOR (row >> 1) & 7: no bank conflicts),
    // then lane L reads chunk L % 8 of row 8j + L / 8, so that every store
    // instruction writes eight whole 128-byte lines of dst, as streaming
    // (nontemporal) stores: dst is not read again here (1%).  A wave touches
    // only its own region (its LDS operations complete in order).
    lds_t *const sO = sbase + wave * 8192 * MB;
    const int rr = lane >> 3;
    const int rc = lane & 7;
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) {
        lds_t *const so = sO + (nb & 1) * 4096 * MB;
#pragma unroll
        for (int j = 0; j < 2 * MB; ++j) {
            const int row = 16 * j + l16;
#pragma unroll
            for (int i = 0; i < 2; ++i)
                *reinterpret_cast<__attribute__((address_space(3))) f32x4 *>(
                    so + row * 128 + (((4 * i + q4) ^ ((row >> 1) & 7)) << 4)) = acc[2 * nb + i][j];
        }
        const int n = n0 + 128 * wn + 32 * nb + 4 * rc;
        f32x4 bias = {0.f, 0.f, 0.f, 0.f};
        if (a.bias && n < a.N) bias = *reinterpret_cast<const f32x4 *>(a.bias + n);
#pragma unroll
        for (int j = 0; j < 4 * MB; ++j) {
            const int row = 8 * j + rr;
            f32x4 v = *reinterpret_cast<const __attribute__((address_space(3))) f32x4 *>(
                so + row * 128 + ((rc ^ ((row >> 1) & 7)) << 4));
            const int m = m0 + 32 * MB * wm + row;
            if (m < a.M && n < a.N) {
                v.x += bias.x; v.y += bias.y; v.z += bias.z; v.w += bias.w;
                __builtin_nontemporal_store(v, reinterpret_cast<f32x4 *>(a.dst + (int64_t)m * a.d_nb1 + (int64_t)n * 4));
            }
        }
    }
}

template <int MB>
static void launch_mm_t(const MmArgs &a, bool x_f32, hipStream_t s) {
    if (x_f32)
        hipLaunchKernelGGL((mm_bf16<true, MB>), dim3(a.n_blocks), dim3(64 * kMmWaves), 0, s, a);
    else
        hipLaunchKernelGGL((mm_bf16<false, MB>), dim3(a.n_blocks), dim3(64 * kMmWaves), 0, s, a);
}

hipError_t launch_mm(const MmArgs &a, int tile, bool x_f32, hipStream_t s) {
    if (tile == 88)
        launch_mm_t<4>(a, x_f32, s);
    else
        launch_mm_t<2>(a, x_f32, s);
    return hipGetLastError();
}

}  // namespace kdfa
