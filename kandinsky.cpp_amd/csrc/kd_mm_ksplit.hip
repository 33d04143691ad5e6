// kd_mm_ksplit.hip - the linear-layer product for calls of few tokens, whose
// 256 x 256 tiles (mm_bf16) would leave most CUs idle:
//
//   mm_skinny  up to 16 tokens: the weight rows streamed once, each wave its
//              own share of k through its own LDS ring, no barrier in the loop
//   mm_ksplit  tiles of 32 NB outputs x 32 MB tokens, the four waves of a
//              workgroup splitting every 64-k stage
//
// In both a wave computes the whole tile over its part of k and the four
// partial sums meet in LDS at the end, in wave order (the same bits on every
// call).  Operands and arithmetic are mm_bf16's: W rows on the MFMA's M
// side, X rows rounded to BF16 on its N side, F32 accumulation.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/kd_mm.h"
#include "kd_fa_device.h"
#include "kd_mm_kernel.h"

namespace kdfa {

typedef const __attribute__((address_space(3))) f32x4 lds_f32x4;

// Wait until at most `later` (0 to kMax) stages of kPer DMAs are in flight
// and every LDS read of this wave has returned.
template <int kPer, int kMax>
static __device__ __forceinline__ void wait_stages(int later) {
    static_assert(kMax * kPer <= 63, "vmcnt range");
    if constexpr (kMax > 0) {
        if (later < kMax) return wait_stages<kPer, kMax - 1>(later);
    }
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"(kMax * kPer) : "memory");
}

// Eight F32 of an X row as one BF16 fragment.
static __device__ __forceinline__ bf16x8 round8(f32x4 u, f32x4 v) {
    typedef Elem<__bf16> E;
    const u32x4 w = {E::pack2(u.x, u.y), E::pack2(u.z, u.w), E::pack2(v.x, v.y), E::pack2(v.z, v.w)};
    return __builtin_bit_cast(bf16x8, w);
}

// LDS rows of one stage hold 64 k: 128 bytes of BF16 (16-byte chunk c of row
// r at c ^ ((r >> 1) & 7)) or 256 bytes of F32 (at c ^ (r & 15)), which
// spreads the rows of an operand read over the banks (conflicts: 0.5% of
// mm_skinny's cycles, 1.3-1.9% of mm_ksplit's).
static __device__ __forceinline__ int swz16(int r) { return (r >> 1) & 7; }
static __device__ __forceinline__ int swz32(int r) { return r & 15; }

// ---------------------------------------------------------------------------
// mm_skinny: 32 NB outputs x up to XR tokens (8 or 16; M <= XR), bound by
// the stream of W from HBM.  A wave takes stages wave, wave + 4, ... of 64 k
// (whole 128-byte lines of W) and keeps S - 1 of them in flight by itself,
// 64-80 KB of W per CU; rows of X past M repeat the last one.  2 x 16384 x
// 4096, BF16 W, F32 x: 118.5 -> 29.5 us (26.6 in the kernel, W fetched once
// at 5.0 TB/s; mm_bf16 ran 64 workgroups); 2 x 4096 x 4096 116 -> 11.9, 2 x 4096 x 16384 437 -> 33.5,
// 16 x 4096 x 16384 458 -> 43.
// ---------------------------------------------------------------------------
template <int NB, int XR, int S, bool XF32>
__global__ __launch_bounds__(256) void mm_skinny(MmArgs a) {
    constexpr int kXRow = XF32 ? 256 : 128;
    constexpr int kW = NB * 4096;                 // W bytes of a stage: 32 NB rows x 64 k
    constexpr int kStage = kW + XR * kXRow;
    constexpr int kWD = kW / 1024;                // DMAs of a stage
    constexpr int kXD = XR * kXRow / 1024;
    constexpr int kPer = kWD + kXD;
    static_assert(XR * kXRow % 1024 == 0 && S >= 2, "whole DMAs");
    __shared__ __attribute__((aligned(1024))) char lds[4 * S * kStage];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31;
    const int hi = lane >> 5;
    const int n0 = blockIdx.x * (32 * NB);
    lds_t *const ring = LDS_PTR(char, lds) + wave * S * kStage;

    uint32_t w_off[kWD], x_off[kXD];
    auto w_chunk = [&](int j) { return (lane & 7) ^ swz16(8 * j + (lane >> 3)); };
    auto x_chunk = [&](int j) {
        return XF32 ? ((lane & 15) ^ swz32(4 * j + (lane >> 4))) : ((lane & 7) ^ swz16(8 * j + (lane >> 3)));
    };
#pragma unroll
    for (int j = 0; j < kWD; ++j) {
        const int r = 8 * j + (lane >> 3);
        w_off[j] = (uint32_t)min(r, a.N - 1 - n0) * (uint32_t)a.w_nb1 + (uint32_t)(w_chunk(j) << 4);
    }
#pragma unroll
    for (int j = 0; j < kXD; ++j) {
        const int r = XF32 ? 4 * j + (lane >> 4) : 8 * j + (lane >> 3);
        x_off[j] = (uint32_t)min(r, a.M - 1) * (uint32_t)a.x_nb1 + (uint32_t)(x_chunk(j) << 4);
    }
    const char *const wtile = a.w + (int64_t)n0 * a.w_nb1;
    const int nk = (a.K + 63) >> 6;
    const int n_st = (nk - wave + 3) >> 2;        // this wave's stages: wave, wave + 4, ...
    const bool half = (a.K & 32) != 0;            // the last stage holds 32 k
    auto issue = [&](int i, int buf) __attribute__((always_inline)) {
        const int kt = wave + 4 * i;
        lds_t *s = ring + buf * kStage;
        const bool tail = half && kt == nk - 1;   // the chunks past K: the first half's again, not used
#pragma unroll
        for (int j = 0; j < kWD; ++j)
            dma16(wtile + (int64_t)kt * 128, w_off[j] - (tail && w_chunk(j) >= 4 ? 64u : 0u), s + j * 1024);
#pragma unroll
        for (int j = 0; j < kXD; ++j)
            dma16(a.x + (int64_t)kt * kXRow, x_off[j] - (tail && x_chunk(j) >= kXRow / 32 ? kXRow / 2 : 0u),
                  s + kW + j * 1024);
    };

    f32x16 acc[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[nb] = (f32x16){};
#pragma unroll
    for (int i = 0; i < S - 1; ++i)
        if (i < n_st) issue(i, i);
    const int xr = l32 % XR;
    int buf = 0;
    for (int i = 0; i < n_st; ++i) {
        wait_stages<kPer, S - 2>(min(S - 2, n_st - 1 - i));
        // into the buffer of stage i - 1, whose reads have returned
        if (i + S - 1 < n_st) issue(i + S - 1, buf == 0 ? S - 1 : buf - 1);
        const lds_t *s = ring + buf * kStage;
        buf = buf == S - 1 ? 0 : buf + 1;
        const int steps = half && wave + 4 * i == nk - 1 ? 2 : 4;
        bf16x8 fw[4][NB], fx[4];
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
                fw[ks][nb] = *reinterpret_cast<const __attribute__((address_space(3))) bf16x8 *>(
                    s + (32 * nb + l32) * 128 + (((2 * ks + hi) ^ swz16(l32)) << 4));
            const lds_t *xp = s + kW + xr * kXRow;
            if constexpr (XF32)
                fx[ks] = round8(*reinterpret_cast<lds_f32x4 *>(xp + (((4 * ks + 2 * hi) ^ swz32(xr)) << 4)),
                                *reinterpret_cast<lds_f32x4 *>(xp + (((4 * ks + 2 * hi + 1) ^ swz32(xr)) << 4)));
            else
                fx[ks] = *reinterpret_cast<const __attribute__((address_space(3))) bf16x8 *>(
                    xp + (((2 * ks + hi) ^ swz16(xr)) << 4));
        }
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
            if (ks < steps) {
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) acc[nb] = Elem<__bf16>::mfma(fw[ks][nb], fx[ks], acc[nb]);
            }
    }

    // ---- the four partial sums, 32 outputs (128 bytes) of 32 tokens at a time
    lds_t *const sp = LDS_PTR(char, lds);
    __syncthreads();
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int g = 0; g < 4; ++g)
            *reinterpret_cast<__attribute__((address_space(3))) f32x4 *>(
                sp + (wave * NB + nb) * 4096 + l32 * 128 + (((2 * g + hi) ^ swz16(l32)) << 4)) =
                (f32x4){acc[nb][4 * g], acc[nb][4 * g + 1], acc[nb][4 * g + 2], acc[nb][4 * g + 3]};
    __syncthreads();
    const int m = tid >> 3, c = tid & 7;
    if (m >= a.M) return;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        const int n = n0 + 32 * nb + 4 * c;
        if (n >= a.N) break;
        const lds_t *q = sp + nb * 4096 + m * 128 + ((c ^ swz16(m)) << 4);
        f32x4 v = *reinterpret_cast<lds_f32x4 *>(q);
#pragma unroll
        for (int w = 1; w < 4; ++w) v += *reinterpret_cast<lds_f32x4 *>(q + w * NB * 4096);
        if (a.bias) v += *reinterpret_cast<const f32x4 *>(a.bias + n);
        __builtin_nontemporal_store(v, reinterpret_cast<f32x4 *>(a.dst + (int64_t)m * a.d_nb1 + (int64_t)n * 4));
    }
}

// ---------------------------------------------------------------------------
// mm_ksplit: 32 NB outputs x 32 MB tokens per workgroup.  Splitting k over
// the waves lets each read every W and X row of the tile once per 16 k: half
// the LDS reads of a 2 x 2 grid of waves, which would bind at these sizes.
// What takes most is the stages' way into LDS (64 B/clk per CU, F32 x twice
// the bytes of BF16): 16 of the kernel's 29 us at 300 tokens, 39 of 70 at
// 1,280, at the 134 KB per microsecond and CU that a probe reached; the matrix
// cores are busy 21 and 31% of the time, and 6 and 10% of the waves' time
// waits for an LDS instruction.  F32 x, N = K = 4096: 64 tokens 127 -> 15.8
// us (1 x 1 blocks), 300 131 -> 28.0 (2 x 3), 600 130 -> 37.8 (4 x 3), 1,280
// 131 -> 75, 2,000 131 -> 95 (4 x 4), weights from HBM on every call.
// ---------------------------------------------------------------------------
template <int NB, int MB, bool XF32>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
void mm_ksplit(MmArgs a) {
    constexpr int kXRow = XF32 ? 256 : 128;
    constexpr int kW = NB * 4096;
    constexpr int kStage = kW + MB * 32 * kXRow;
    constexpr int kXD = XF32 ? 2 * MB : MB;       // a wave's DMAs of a stage: NB of W, kXD of X
    constexpr int kPer = NB + kXD;
    constexpr int kFit = 163840 / kStage;
    constexpr int S = kFit < 5 ? kFit : 5;
    constexpr int kEpi = MB * 16384;              // the four waves' 32 outputs of every token
    constexpr int kLds = S * kStage > 2 * kEpi ? S * kStage : 2 * kEpi;
    static_assert(S >= 2 && 2 * kEpi <= 163840, "two stages, and two blocks of sums, at least");
    __shared__ __attribute__((aligned(1024))) char lds[kLds];
    lds_t *const sbase = LDS_PTR(char, lds);

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31;
    const int hi = lane >> 5;

    // tile: XCD-contiguous runs, dealt in columns of `cols` output tiles,
    // the token tiles of a column one after another
    const int pid = blockIdx.x;
    const int per = a.n_blocks >> 3;
    const int lid = pid < per * 8 ? (pid & 7) * per + (pid >> 3) : pid;
    const int col = lid / (a.tiles_m * a.cols), rem = lid - col * (a.tiles_m * a.cols);
    const int width = min(a.cols, a.tiles_n - col * a.cols);
    const int mt = rem / width;
    const int n0 = (col * a.cols + rem - mt * width) * (32 * NB);
    const int m0 = mt * (32 * MB);

    // DMA j of a wave: W rows 8 (wave + 4 j) .. +7; X rows 4 (wave + 4 j) ..
    // +3 (F32) or 8 (wave + 4 j) .. +7: the chunk a lane brings is the same
    // for every j
    uint32_t w_off[NB], x_off[kXD];
    const int wc = (lane & 7) ^ swz16(8 * wave + (lane >> 3));
    const int xc = XF32 ? ((lane & 15) ^ swz32(4 * wave + (lane >> 4))) : wc;
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        const int r = 8 * (wave + 4 * j) + (lane >> 3);
        w_off[j] = (uint32_t)min(r, a.N - 1 - n0) * (uint32_t)a.w_nb1 + (uint32_t)(wc << 4);
    }
#pragma unroll
    for (int j = 0; j < kXD; ++j) {
        const int r = XF32 ? 4 * (wave + 4 * j) + (lane >> 4) : 8 * (wave + 4 * j) + (lane >> 3);
        x_off[j] = (uint32_t)min(r, a.M - 1 - m0) * (uint32_t)a.x_nb1 + (uint32_t)(xc << 4);
    }
    const char *const wtile = a.w + (int64_t)n0 * a.w_nb1;
    const char *const xtile = a.x + (int64_t)m0 * a.x_nb1;
    const int nk = (a.K + 63) >> 6;
    const bool half = (a.K & 32) != 0;            // the last stage holds 32 k
    // tail: the half-filled last stage, whose chunks past K bring the first
    // half's again (not used)
    auto dma_j = [&](int kt, int buf, int j, bool tail) __attribute__((always_inline)) {
        lds_t *s = sbase + buf * kStage;
        if (j < NB)
            dma16(wtile + (int64_t)kt * 128, w_off[j] - (tail && wc >= 4 ? 64u : 0u), s + (wave + 4 * j) * 1024);
        else
            dma16(xtile + (int64_t)kt * kXRow, x_off[j - NB] - (tail && xc >= kXRow / 32 ? kXRow / 2 : 0u),
                  s + kW + (wave + 4 * (j - NB)) * 1024);
    };

    f32x16 acc[NB][MB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) acc[nb][mb] = (f32x16){};

    // fragments of this wave's 16 k of a stage, two sets: those of stage
    // kt + 1 are read before the products of stage kt
    const uint32_t w_rd = l32 * 128 + (((2 * wave + hi) ^ swz16(l32)) << 4);
    const uint32_t x_rd0 = kW + l32 * kXRow + (XF32 ? (((4 * wave + 2 * hi) ^ swz32(l32)) << 4)
                                                    : (((2 * wave + hi) ^ swz16(l32)) << 4));
    const uint32_t x_rd1 = kW + l32 * kXRow + (((4 * wave + 2 * hi + 1) ^ swz32(l32)) << 4);
    bf16x8 fw[2][NB];
    f32x4 xu[2][MB], xv[2][MB];
    auto read = [&](int buf, auto set_c) __attribute__((always_inline)) {
        constexpr int set = decltype(set_c)::value;
        const lds_t *s = sbase + buf * kStage;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
            fw[set][nb] = *reinterpret_cast<const __attribute__((address_space(3))) bf16x8 *>(s + w_rd + nb * 4096);
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
            xu[set][mb] = *reinterpret_cast<lds_f32x4 *>(s + x_rd0 + mb * 32 * kXRow);
            if constexpr (XF32) xv[set][mb] = *reinterpret_cast<lds_f32x4 *>(s + x_rd1 + mb * 32 * kXRow);
        }
    };
    // the products of a stage whose fragments are in `set`, with the DMAs of
    // stage dkt into buffer dbuf spread over them
    auto products = [&](auto set_c, bool dma, int dkt, int dbuf, bool tail) __attribute__((always_inline)) {
        constexpr int set = decltype(set_c)::value;
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
            const bf16x8 b = XF32 ? round8(xu[set][mb], xv[set][mb]) : __builtin_bit_cast(bf16x8, xu[set][mb]);
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                acc[nb][mb] = Elem<__bf16>::mfma(fw[set][nb], b, acc[nb][mb]);
                __builtin_amdgcn_sched_barrier(0);
                if (dma) {
#pragma unroll
                    for (int j = 0; j < kPer; ++j)
                        if (j * (NB * MB) / kPer == mb * NB + nb) dma_j(dkt, dbuf, j, tail);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    // Step kt: publish stage kt + 1 -- after the barrier every wave's reads
    // of stage kt have returned -- read its fragments, then the products of
    // stage kt while stage kt + S goes into stage kt's buffer.  The steps of
    // the main loop are free of conditions (a read under a branch makes the
    // compiler wait for the reads just issued); the last S + 1 or so are not.
    auto step = [&](int kt, int &buf, auto set_c) __attribute__((always_inline)) {
        const int cur = buf;
        buf = buf == S - 1 ? 0 : buf + 1;
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"((S - 2) * kPer) : "memory");
        __syncthreads();
        read(buf, IC<1 - decltype(set_c)::value>());
        __builtin_amdgcn_sched_barrier(0);
        products(set_c, true, kt + S, cur, false);
    };
    auto last_step = [&](int kt, int &buf, auto set_c) __attribute__((always_inline)) {
        const int cur = buf;
        buf = buf == S - 1 ? 0 : buf + 1;
        if (kt + 1 < nk) {
            wait_stages<kPer, S - 2>(min(S - 2, nk - 2 - kt));
            __syncthreads();
            read(buf, IC<1 - decltype(set_c)::value>());
        }
        __builtin_amdgcn_sched_barrier(0);
        // with half a stage left, waves 2 and 3 have none of it
        if (wave < 2 || !half || kt + 1 < nk) products(set_c, kt + S < nk, kt + S, cur, half && kt + S == nk - 1);
    };

#pragma unroll
    for (int i = 0; i < S; ++i)
        if (i < nk) {
#pragma unroll
            for (int j = 0; j < kPer; ++j) dma_j(i, i, j, half && i == nk - 1);
        }
    wait_stages<kPer, S - 1>(min(S, nk) - 1);
    __syncthreads();
    read(0, IC<0>());
    int buf = 0, kt = 0;
    for (; kt + S + 2 < nk; kt += 2) {   // stages kt + S and kt + S + 1 are whole ones
        step(kt, buf, IC<0>());
        step(kt + 1, buf, IC<1>());
    }
    for (; kt < nk; kt += 2) {
        last_step(kt, buf, IC<0>());
        if (kt + 1 < nk) last_step(kt + 1, buf, IC<1>());
    }

    // ---- the four partial sums, 32 outputs (128 bytes of every token row) at
    // a time: each wave leaves its own, then sums a quarter of the rows in
    // wave order and stores whole 128-byte lines
    const int rr = lane >> 3, rc = lane & 7;
    __syncthreads();
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        lds_t *const so = sbase + (nb & 1) * kEpi;
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
            for (int g = 0; g < 4; ++g)
                *reinterpret_cast<__attribute__((address_space(3))) f32x4 *>(
                    so + wave * (MB * 4096) + (32 * mb + l32) * 128 + (((2 * g + hi) ^ swz16(l32)) << 4)) =
                    (f32x4){acc[nb][mb][4 * g], acc[nb][mb][4 * g + 1], acc[nb][mb][4 * g + 2], acc[nb][mb][4 * g + 3]};
        __syncthreads();
        const int n = n0 + 32 * nb + 4 * rc;
        f32x4 bias = {0.f, 0.f, 0.f, 0.f};
        if (a.bias && n < a.N) bias = *reinterpret_cast<const f32x4 *>(a.bias + n);
#pragma unroll
        for (int j = 0; j < MB; ++j) {
            const int row = 8 * (wave + 4 * j) + rr;
            const lds_t *q = so + row * 128 + ((rc ^ swz16(row)) << 4);
            f32x4 v = *reinterpret_cast<lds_f32x4 *>(q);
#pragma unroll
            for (int w = 1; w < 4; ++w) v += *reinterpret_cast<lds_f32x4 *>(q + w * (MB * 4096));
            v += bias;
            if (m0 + row < a.M && n < a.N)
                __builtin_nontemporal_store(
                    v, reinterpret_cast<f32x4 *>(a.dst + (int64_t)(m0 + row) * a.d_nb1 + (int64_t)n * 4));
        }
    }
}

template <int NB, int XR, int S>
static void launch_skinny_t(const MmArgs &a, bool x_f32, hipStream_t s) {
    const dim3 grid((unsigned)((a.N + 32 * NB - 1) / (32 * NB)));
    if (x_f32)
        hipLaunchKernelGGL((mm_skinny<NB, XR, S, true>), grid, dim3(256), 0, s, a);
    else
        hipLaunchKernelGGL((mm_skinny<NB, XR, S, false>), grid, dim3(256), 0, s, a);
}

// 64 outputs per workgroup where that still gives every CU one (16384
// outputs, 2 tokens: 29.4 us against 33.8 with 32), else 32 (4096 outputs:
// 11.9 against 15.1).  S as LDS allows: with 32 outputs and up to 8 tokens
// three stages, two workgroups per CU.
hipError_t launch_mm_skinny(const MmArgs &a, bool x_f32, hipStream_t s) {
    const bool wide = (a.N + 63) / 64 >= 256;
    if (a.M <= 8)
        wide ? launch_skinny_t<2, 8, 4>(a, x_f32, s) : launch_skinny_t<1, 8, 3>(a, x_f32, s);
    else
        wide ? launch_skinny_t<2, 16, 3>(a, x_f32, s) : launch_skinny_t<1, 16, 5>(a, x_f32, s);
    return hipGetLastError();
}

template <int NB, int MB>
static void launch_ksplit_t(const MmArgs &a, bool x_f32, hipStream_t s) {
    if (x_f32)
        hipLaunchKernelGGL((mm_ksplit<NB, MB, true>), dim3(a.n_blocks), dim3(256), 0, s, a);
    else
        hipLaunchKernelGGL((mm_ksplit<NB, MB, false>), dim3(a.n_blocks), dim3(256), 0, s, a);
}

hipError_t launch_mm_ksplit(const MmArgs &a, int tile, bool x_f32, hipStream_t s) {
    switch (tile) {
    case 11: launch_ksplit_t<1, 1>(a, x_f32, s); break;
    case 21: launch_ksplit_t<2, 1>(a, x_f32, s); break;
    case 22: launch_ksplit_t<2, 2>(a, x_f32, s); break;
    case 23: launch_ksplit_t<2, 3>(a, x_f32, s); break;
    case 42: launch_ksplit_t<4, 2>(a, x_f32, s); break;
    case 43: launch_ksplit_t<4, 3>(a, x_f32, s); break;
    case 44: launch_ksplit_t<4, 4>(a, x_f32, s); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace kdfa
