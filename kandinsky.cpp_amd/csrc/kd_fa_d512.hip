// kd_fa_d512.hip - the D = 512 attention of the 2-D VAE's attention block
// (src/models/vae.hpp:60-101 -> ops::attention, one head, D = channels).
//
// Built with VGPR-form MFMAs (-mllvm -amdgpu-mfma-vgpr-form, see the
// Makefile): O is rescaled by the vector unit every tile, and with the
// accumulators in AGPRs the compiler would copy all of O through VGPRs on
// every tile.  Internal to libkd_fa.so.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kd_fa_device.h"

namespace kdfa {

// fa_fwd_d512: the attention of the 2-D VAE's attention block
// (src/models/vae.hpp:60-101 -> ops::attention with one head, D = channels =
// 512), no mask, no RoPE.
//
// A workgroup is 4 waves (one per CU: 119-141 KB of LDS) and covers R blocks
// of 32 query rows of one (b, h); wave w owns the 128 columns 128w .. 128w+127
// of D for both products, so that its O (32R rows x 128) and Q (32R rows x
// 128) stay in registers.  Per 32-key tile:
//   S_w^T = K_w Q_w^T over the wave's 128 columns (8 MFMA per row block), K_w
//           staged by DMA in the wave's own LDS region (loaded straight into
//           the operands, a lane's neighbours in other rows, K came at 38 KB
//           per microsecond and CU against 130 by whole row pieces);
//   the four partial scores meet in LDS; wave w runs the online softmax of
//           rows 8Rw .. 8Rw+8R-1 (exact running max, exp2 domain) and writes
//           the weights P (rounded to the operand type), the rescale factor
//           and, at the end, the row sum to LDS for all waves;
//   O_w^T = alpha * O_w^T + V_w^T P^T (8 MFMA per row block), V_w staged the
//           same way (two buffers) and read transposed with
//           ds_read_b64_tr_b16, each fragment once for all R blocks.
// Two barriers per tile.  Keys past Lk (last tile) come as zeros and get
// weight 0.  Every K and V byte a workgroup streams serves 32R query rows.
// R = 1 and R = 2 give bitwise equal results: the same products, the same
// sums of the partial scores, and the row sums combined in the same tree (4
// keys per leaf).
// With a key split (a.n_split > 1, short query sets with a workspace), a
// workgroup runs only its range of key tiles and leaves the unnormalised O,
// running max and row sum of its rows for d512_combine.
// LDS is the busiest unit by count: at R = 2 a tile moves 212 KB through it
// (1,650 of its about 2,900 cycles; the products take 1,024).  No unit is at
// its limit: at 4,096 tokens the matrix cores are busy 24% of the time, 15%
// of the waves' time waits for an LDS instruction (conflicts: 3.7%), and the
// rest is the chain of a step with one wave per SIMD.  F16 K / V: 4,096 tokens
// with the key split 96.8 -> 72.6 us, 8,192 311 -> 203, 16,384 924 -> 706; with
// the products in sequence with the exchange and the DMAs in one burst
// before the barrier 16,384 tokens took 880.
constexpr int kD5 = 512;                     // D, four 128-column slices
constexpr int kD5Keys = 32;                    // keys per tile
constexpr int kD5SStride = kD5Keys + 4;        // floats per row of a partial-score block (pad)
constexpr int kD5PStride = kD5Keys + 8;        // 16-bit weights per row of P (pad)
constexpr int kD5Tile = kD5Keys * 256;         // one wave's K or V tile: 32 keys x 128 columns

static_assert(kD5 == 4 * 128, "one 128-column slice per wave");

// the value of lane l ^ X within each row's lanes (X = 1, 2, 4: quad_perm
// for the first two, row_half_mirror for the third, whose mirrored lane
// holds the same as lane l ^ 4 once the quads agree)
template <int X>
static __device__ __forceinline__ float row_xor(float v) {
    const int i = __builtin_bit_cast(int, v);
    constexpr int kCtrl = X == 1 ? 0xB1 : X == 2 ? 0x4E : 0x141;
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(i, i, kCtrl, 0xF, 0xF, true));
}

template <typename T, int R>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
void fa_fwd_d512(Args a) {
    typedef Elem<T> E;
    typedef typename E::vec8 vec8;
    constexpr int kRows = 32 * R;                  // query rows per workgroup
    constexpr int kLanesPerRow = 8 / R;            // softmax lanes per row
    constexpr int kKeysPerLane = 4 * R;
    __shared__ __attribute__((aligned(16))) float sS[4][kRows][kD5SStride];
    __shared__ __attribute__((aligned(16))) uint16_t sP[kRows][kD5PStride];
    __shared__ float sAlpha[kRows];
    __shared__ float sL[kRows];
    __shared__ __attribute__((aligned(1024))) char sV[4][2][kD5Tile];
    __shared__ __attribute__((aligned(1024))) char sK[4][kD5Tile];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31;
    const int hi = lane >> 5;
    // key split (a.n_split > 1): the grid holds n_split copies of the
    // unsplit grid, copy s taking keys [s * split_keys, (s + 1) * split_keys)
    const int split = a.n_split > 1 ? (int)blockIdx.x / a.n_blocks : 0;
    const int blk = (int)blockIdx.x - split * a.n_blocks;
    const int qt = blk % a.n_qt;
    const int bh = blk / a.n_qt;
    const int h = bh % a.H;
    const int b = bh / a.H;
    const int Lk = a.Lk;
    const int k_end = a.n_split > 1 ? min((split + 1) * a.split_keys, Lk) : Lk;
    const int t_begin = a.n_split > 1 ? split * a.split_keys / kD5Keys : 0;
    const int n_tiles = (k_end + kD5Keys - 1) / kD5Keys;   // one past the range's last tile
    const int col0 = 128 * wave;                  // this wave's columns of D

    // Q fragments of the wave's columns (B operands of S_w^T = K_w Q_w^T)
    vec8 qf[R][8];
#pragma unroll
    for (int rb = 0; rb < R; ++rb) {
        const int q_row = qt * kRows + 32 * rb + l32;
        const int q_ld = q_row < a.Lq ? q_row : a.Lq - 1;
        const char *qp = a.q + (int64_t)q_ld * a.q_nb1 + (int64_t)h * a.q_nb2 + (int64_t)b * a.q_nb3;
        const int esz = a.q_type == KD_FA_TYPE_F32 ? 4 : 2;
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) {
            float x[8];
            load8_f32(qp + (col0 + ks * 16 + hi * 8) * esz, a.q_type, x);
            u32x4 w;
            for (int j = 0; j < 4; ++j) w[j] = E::pack2(x[2 * j], x[2 * j + 1]);
            if (a.scale_log2 < 0.0f) w ^= (u32x4){0x80008000u, 0x80008000u, 0x80008000u, 0x80008000u};
            qf[rb][ks] = __builtin_bit_cast(vec8, w);
        }
    }
    const float c2 = __builtin_fabsf(a.scale_log2);

    const char *kbase = a.k + (int64_t)(h / a.rk2) * a.k_nb2 + (int64_t)(b / a.rk3) * a.k_nb3 + col0 * 2;
    const char *vbase = a.v + (int64_t)(h / a.rv2) * a.v_nb2 + (int64_t)(b / a.rv3) * a.v_nb3 + col0 * 2;
    // V tile of this wave: LDS row r (key t*32 + r) holds the wave's 128
    // columns, 16-byte chunk c at c ^ v_swz(r); 8 DMA rounds of 4 rows
    // K tile: the same rows, chunk c at c ^ (r & 15)
    const int dma_row = lane >> 4, dma_pc = lane & 15;
    uint32_t k_off[kD5Keys / 4], v_off[kD5Keys / 4];
#pragma unroll
    for (int j = 0; j < kD5Keys / 4; ++j) {
        const int r = 4 * j + dma_row;
        k_off[j] = (uint32_t)r * (uint32_t)a.k_nb1 + ((dma_pc ^ (r & 15)) << 4);
        v_off[j] = (uint32_t)r * (uint32_t)a.v_nb1 + ((dma_pc ^ v_swz(r)) << 4);
    }
    // a tile's resource: from its first row to the end of its last key's
    // 256 bytes; rows past that come as zeros
    auto tile_rsrc = [&](const char *base, int64_t nb1, int t) __attribute__((always_inline)) {
        const uint64_t p = (uint64_t)(base + (int64_t)t * kD5Keys * nb1);
        const uint32_t rows = (uint32_t)min(kD5Keys, Lk - t * kD5Keys);
        return (u32x4){(uint32_t)p, (uint32_t)(p >> 32) & 0xffffu, (rows - 1) * (uint32_t)nb1 + 256, 0x00020000u};
    };
    auto dma = [&](u32x4 rsrc, uint32_t off, lds_t *dst) __attribute__((always_inline)) {
        const uint32_t m0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)dst);
        asm volatile("buffer_load_dwordx4 %0, %1, 0 offen lds" :: "v"(off), "s"(rsrc), "{m0}"(m0));
    };
    lds_t *const ks_ = LDS_PTR(char, sK[wave]);
    // DMA j (of 8) of a tile: rows 4 j .. 4 j + 3
    auto dma_k = [&](u32x4 rsrc, int j) __attribute__((always_inline)) { dma(rsrc, k_off[j], ks_ + j * 1024); };
    auto dma_v = [&](u32x4 rsrc, int buf, int j) __attribute__((always_inline)) {
        dma(rsrc, v_off[j], LDS_PTR(char, sV[wave][buf]) + j * 1024);
    };
    // K fragment of k-step i: key (tile row) l32, columns 16 i + 8 hi .. +7
    auto read_k = [&](vec8 kf[8]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
            kf[i] = *reinterpret_cast<const __attribute__((address_space(3))) vec8 *>(
                ks_ + l32 * 256 + (((2 * i + hi) ^ (l32 & 15)) << 4));
    };
    const int v_sub = (lane & 15) >> 2;
    const int v_c_lo = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
    uint32_t v_rd[4];
#pragma unroll
    for (int dblk = 0; dblk < 4; ++dblk)
        v_rd[dblk] = 2048 * hi + 256 * v_sub + (((4 * dblk + v_c_lo) ^ v_swz(v_sub)) << 4) + 8 * (lane & 1);

    f32x16 o[R][4];
#pragma unroll
    for (int rb = 0; rb < R; ++rb)
#pragma unroll
        for (int i = 0; i < 4; ++i) o[rb][i] = (f32x16){};
    // softmax state of row 8R*wave + lane / (8/R) (the lanes of a row agree);
    // the lane's keys are 4R consecutive ones
    const int srow = 8 * R * wave + lane / kLanesPerRow;
    const int skey = kKeysPerLane * (lane % kLanesPerRow);
    float m_run = -INFINITY, l_run = 0.0f;

    // Step t writes the partial scores of tile t, runs the products of V(t-1)
    // while they meet, and those of K(t+1) between the steps of tile t's
    // softmax: a wave alone on its SIMD has nothing else to run under the
    // exchange.  Its DMAs, K(t+2) among the first products and V(t+1) among
    // the second, take the CU's load path about as long as the products the
    // matrix cores; at the next step's start at most V's 8 may be in flight.
    // K's one buffer is free once its fragments are in registers, V's two
    // alternate; both are the wave's own (no barrier).
    f32x16 s[R];
    vec8 kf[8];
    auto partial = [&](int rb, int i) __attribute__((always_inline)) {
        s[rb] = i == 0 ? E::mfma(kf[0], qf[rb][0], (f32x16){}) : E::mfma(kf[i], qf[rb][i], s[rb]);
    };
    // K's fragments are in registers: what follows may overwrite its buffer.
    // The DMAs are asm, so that nothing else makes the compiler keep them
    // behind those reads; it adds a wait only where one may be in flight
    auto hold_k = [&]() __attribute__((always_inline)) {
        asm volatile("; K fragments held" ::"v"(kf[0]), "v"(kf[1]), "v"(kf[2]), "v"(kf[3]), "v"(kf[4]), "v"(kf[5]),
                     "v"(kf[6]), "v"(kf[7]) : "memory");
    };
    auto keep_q = [&]() __attribute__((always_inline)) {
        // the Q fragments (read by the matrix unit only) live in AGPRs, so
        // that O, S and the K fragments have the VGPRs to themselves
#pragma unroll
        for (int rb = 0; rb < R; ++rb)
#pragma unroll
            for (int i = 0; i < 8; ++i) asm volatile("" : "+a"(qf[rb][i]));
    };
    if (n_tiles > t_begin) {
        // the first tile's V right behind its K: one round trip for both
        const u32x4 k0 = tile_rsrc(kbase, a.k_nb1, t_begin);
#pragma unroll
        for (int j = 0; j < 8; ++j) dma_k(k0, j);
        const u32x4 v0 = tile_rsrc(vbase, a.v_nb1, t_begin);
#pragma unroll
        for (int j = 0; j < 8; ++j) dma_v(v0, t_begin & 1, j);
        asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
        read_k(kf);
        keep_q();
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
            for (int rb = 0; rb < R; ++rb) partial(rb, i);
        if (t_begin + 1 < n_tiles) {
            hold_k();
            const u32x4 k1 = tile_rsrc(kbase, a.k_nb1, t_begin + 1);
#pragma unroll
            for (int j = 0; j < 8; ++j) dma_k(k1, j);
            // (the youngest: step t_begin's wait would not cover it)
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
    }
    // O_w^T = alpha * O_w^T + V_w^T P^T of tile t
    auto pv = [&](int t, auto between) __attribute__((always_inline)) {
        const lds_t *vs_ = LDS_PTR(char, sV[wave][t & 1]);
        vec8 va[2][4], pb[2][R];
#pragma unroll
        for (int kst = 0; kst < 2; ++kst) {
#pragma unroll
            for (int rb = 0; rb < R; ++rb)
                pb[kst][rb] = *reinterpret_cast<const vec8 *>(&sP[32 * rb + l32][16 * kst + 8 * hi]);
#pragma unroll
            for (int dblk = 0; dblk < 4; ++dblk) {
                const lds_t *vp = vs_ + v_rd[dblk] + 4096 * kst;
                const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)(vp));
                const s16x4 hi4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)(vp + 1024));
                va[kst][dblk] = __builtin_bit_cast(vec8, __builtin_shufflevector(lo, hi4, 0, 1, 2, 3, 4, 5, 6, 7));
            }
        }
#pragma unroll
        for (int rb = 0; rb < R; ++rb) {
            const float al = sAlpha[32 * rb + l32];
            if (__builtin_amdgcn_ballot_w64(al != 1.0f) != 0) {
#pragma unroll
                for (int dblk = 0; dblk < 4; ++dblk)
#pragma unroll
                    for (int i = 0; i < 16; ++i) o[rb][dblk][i] *= al;
            }
        }
#pragma unroll
        for (int kst = 0; kst < 2; ++kst)
#pragma unroll
            for (int dblk = 0; dblk < 4; ++dblk)
#pragma unroll
                for (int rb = 0; rb < R; ++rb) {
                    o[rb][dblk] = E::mfma(va[kst][dblk], pb[kst][rb], o[rb][dblk]);
                    __builtin_amdgcn_sched_barrier(0);
                    if (rb == R - 1) between(4 * kst + dblk);
                    __builtin_amdgcn_sched_barrier(0);
                }
    };
    // The last step leaves the next tile's part out (its reads, products and
    // DMAs took a range of one tile 0.6 us; the short ranges of a split are
    // little else: 128 tokens 13.0 -> 12.1 us, 256 15.8 -> 15.1)
    auto step = [&](int t, auto last_c) __attribute__((always_inline)) {
        constexpr bool last = decltype(last_c)::value;
        // ---- this wave's partial scores of tile t; element i of lane l: key
        // 8*(i/4) + 4*hi + i%4, query l32
#pragma unroll
        for (int rb = 0; rb < R; ++rb)
#pragma unroll
            for (int g = 0; g < 4; ++g)
                *reinterpret_cast<f32x4 *>(&sS[wave][32 * rb + l32][8 * g + 4 * hi]) =
                    (f32x4){s[rb][4 * g], s[rb][4 * g + 1], s[rb][4 * g + 2], s[rb][4 * g + 3]};
        asm volatile("s_waitcnt vmcnt(8)" ::: "memory");   // K(t+1) and V(t-1) have landed
        if (!last) read_k(kf);
        // K(t+2)'s DMAs (past the last tile, that one again) between the
        // products of V(t-1), whose operands are read after K(t+1)'s
        // fragments: no wait of their own for those (an LDS wait for them
        // here, ahead of V's reads, would show)
        const u32x4 k2 = tile_rsrc(kbase, a.k_nb1, min(t + 2, n_tiles - 1));
        if (t > t_begin) {
            pv(t - 1, [&](int j) __attribute__((always_inline)) {
                if (last) return;
                if (j == 0) hold_k();
                dma_k(k2, j);
            });
        } else if (!last) {
            hold_k();
#pragma unroll
            for (int j = 0; j < 8; ++j) dma_k(k2, j);
        }
        const u32x4 v1 = tile_rsrc(vbase, a.v_nb1, min(t + 1, n_tiles - 1));
        __syncthreads();
        // ---- softmax of the wave's rows (4R keys per lane)
        f32x4 x[R][4];
#pragma unroll
        for (int c = 0; c < R; ++c)
#pragma unroll
            for (int w = 0; w < 4; ++w) x[c][w] = *reinterpret_cast<const f32x4 *>(&sS[w][srow][skey + 4 * c]);
        keep_q();
        constexpr int kM = 8 * R;
        auto mm = [&](auto from_c, auto to_c) __attribute__((always_inline)) {
            if constexpr (last) return;
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = decltype(from_c)::value; i < decltype(to_c)::value; ++i) {
                partial(i % R, i / R);
                __builtin_amdgcn_sched_barrier(0);
                if (i % R == R - 1) dma_v(v1, (t + 1) & 1, i / R);   // V(t-1) is read
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        mm(IC<0>(), IC<kM / 4>());   // while the partial scores arrive
        float sc[kKeysPerLane];
#pragma unroll
        for (int c = 0; c < R; ++c) {
            const f32x4 sum = ((x[c][0] + x[c][1]) + x[c][2]) + x[c][3];
#pragma unroll
            for (int e = 0; e < 4; ++e) sc[4 * c + e] = sum[e] * c2;
        }
        if (t * kD5Keys + kD5Keys > k_end) {
#pragma unroll
            for (int e = 0; e < kKeysPerLane; ++e)
                if (t * kD5Keys + skey + e >= k_end) sc[e] = -INFINITY;
        }
        float mx = sc[0];
#pragma unroll
        for (int e = 1; e < kKeysPerLane; ++e) mx = __builtin_fmaxf(mx, sc[e]);
        mx = __builtin_fmaxf(mx, row_xor<1>(mx));
        mx = __builtin_fmaxf(mx, row_xor<2>(mx));
        if constexpr (R == 1) mx = __builtin_fmaxf(mx, row_xor<4>(mx));
        const float m_new = __builtin_fmaxf(m_run, mx);
        mm(IC<kM / 4>(), IC<kM / 2>());
        const float alpha = m_new == m_run ? 1.0f : __builtin_amdgcn_exp2f(m_run - m_new);
        m_run = m_new;
        const float mu = m_new == -INFINITY ? 0.0f : m_new;
        float p[kKeysPerLane];
#pragma unroll
        for (int e = 0; e < kKeysPerLane; ++e) p[e] = __builtin_amdgcn_exp2f(sc[e] - mu);
        mm(IC<kM / 2>(), IC<3 * kM / 4>());
#pragma unroll
        for (int c = 0; c < R; ++c) {
            const u32x2 w = {E::pack2(p[4 * c], p[4 * c + 1]), E::pack2(p[4 * c + 2], p[4 * c + 3])};
            *reinterpret_cast<u32x2 *>(&sP[srow][skey + 4 * c]) = w;
        }
        if (lane % kLanesPerRow == 0) sAlpha[srow] = alpha;
        mm(IC<3 * kM / 4>(), IC<kM>());
        // row sum: 4-key leaves (p0 + p1) + (p2 + p3) combined pairwise,
        // the pairs within the lane first, then across lanes
        float ps = (p[0] + p[1]) + (p[2] + p[3]);
        if constexpr (R == 2) ps = ps + ((p[4] + p[5]) + (p[6] + p[7]));
        ps += row_xor<1>(ps);
        ps += row_xor<2>(ps);
        if constexpr (R == 1) ps += row_xor<4>(ps);
        l_run = l_run * alpha + ps;
        __syncthreads();
    };
    for (int t = t_begin; t + 1 < n_tiles; ++t) step(t, BC<false>());
    if (n_tiles > t_begin) {
        step(n_tiles - 1, BC<true>());
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        pv(n_tiles - 1, [](int) {});
    }
    if (a.n_split > 1) {
        // this range's unnormalised O (times exactly 1), running max and row
        // sum, for launch_d512_combine
        const int64_t rows = (int64_t)a.B * a.Lq * a.H;
        Args pa = a;
        pa.o = reinterpret_cast<char *>(a.part + (int64_t)split * rows * kD5);
        pa.o_type = KD_FA_TYPE_F32;
        pa.o_nb1 = kD5 * 4;
        pa.o_nb2 = (int64_t)a.H * kD5 * 4;
        pa.o_nb3 = (int64_t)a.Lq * a.H * kD5 * 4;
#pragma unroll
        for (int rb = 0; rb < R; ++rb) store_o_row_l(pa, qt * kRows + 32 * rb + l32, h, b, hi, o[rb], 1.0f, col0);
        const int q_row = qt * kRows + srow;
        if (lane % kLanesPerRow == 0 && q_row < a.Lq) {   // the softmax lanes of the wave's rows
            float *ml = a.part + (int64_t)a.n_split * rows * kD5 +
                        2 * ((int64_t)split * rows + ((int64_t)b * a.Lq + q_row) * a.H + h);
            ml[0] = m_run;
            ml[1] = l_run;
        }
        return;
    }
    if (lane % kLanesPerRow == 0) sL[srow] = l_run;
    __syncthreads();
#pragma unroll
    for (int rb = 0; rb < R; ++rb)
        store_o_row_l(a, qt * kRows + 32 * rb + l32, h, b, hi, o[rb], sL[32 * rb + l32], col0);
}

// d512_combine: dst row r = sum_s w_s O_s / sum_s w_s l_s with
// w_s = 2^(m_s - max_s m_s) over the key ranges of a split call (running
// maxima in the exp2 domain, as the kernel keeps them); 128 threads per row,
// four columns each, F32 arithmetic, then the store_o_row_l rounding.
__global__ __launch_bounds__(256) void d512_combine(Args a) {
    const int64_t rows = (int64_t)a.B * a.Lq * a.H;
    const int64_t r = (int64_t)blockIdx.x * 2 + (threadIdx.x >> 7);
    if (r >= rows) return;
    const int c = (int)(threadIdx.x & 127) * 4;
    const int S = a.n_split;
    const float *ml = a.part + (int64_t)S * rows * kD5;
    float M = -INFINITY;
    for (int s = 0; s < S; ++s) M = __builtin_fmaxf(M, ml[2 * ((int64_t)s * rows + r)]);
    float L = 0.0f;
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int s = 0; s < S; ++s) {
        const float m = ml[2 * ((int64_t)s * rows + r)];
        const float w = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m - M);
        L += w * ml[2 * ((int64_t)s * rows + r) + 1];
        const f32x4 v = *reinterpret_cast<const f32x4 *>(a.part + ((int64_t)s * rows + r) * kD5 + c);
        acc.x += w * v.x; acc.y += w * v.y; acc.z += w * v.z; acc.w += w * v.w;
    }
    const float inv = L == 0.0f ? 0.0f : 1.0f / L;
    const f32x4 v = {acc.x * inv, acc.y * inv, acc.z * inv, acc.w * inv};
    const int h = (int)(r % a.H);
    const int i = (int)((r / a.H) % a.Lq);
    const int b = (int)(r / ((int64_t)a.H * a.Lq));
    char *op = a.o + (int64_t)b * a.o_nb3 + (int64_t)i * a.o_nb2 + (int64_t)h * a.o_nb1;
    if (a.o_type == KD_FA_TYPE_F32) {
        *reinterpret_cast<f32x4 *>(op + c * 4) = v;
    } else if (a.o_type == KD_FA_TYPE_BF16) {
        *reinterpret_cast<u32x2 *>(op + c * 2) = (u32x2){Elem<__bf16>::pack2(v.x, v.y), Elem<__bf16>::pack2(v.z, v.w)};
    } else {
        *reinterpret_cast<u32x2 *>(op + c * 2) =
            (u32x2){Elem<_Float16>::pack2(v.x, v.y), Elem<_Float16>::pack2(v.z, v.w)};
    }
}

template <typename T, int R>
static hipError_t launch_d512_t(const Args &a, hipStream_t s) {
    const int64_t grid = (int64_t)a.n_blocks * (a.n_split > 1 ? a.n_split : 1);
    hipLaunchKernelGGL((fa_fwd_d512<T, R>), dim3((unsigned)grid), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_d512_combine(const Args &a, hipStream_t s) {
    const int64_t rows = (int64_t)a.B * a.Lq * a.H;
    hipLaunchKernelGGL(d512_combine, dim3((unsigned)((rows + 1) / 2)), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_d512(const Args &a, int kv_type, int rows, hipStream_t stream) {
    if (rows == 64)
        return kv_type == KD_FA_TYPE_BF16 ? launch_d512_t<__bf16, 2>(a, stream) : launch_d512_t<_Float16, 2>(a, stream);
    return kv_type == KD_FA_TYPE_BF16 ? launch_d512_t<__bf16, 1>(a, stream) : launch_d512_t<_Float16, 1>(a, stream);
}

}  // namespace kdfa
