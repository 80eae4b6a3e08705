// head_tile.hip -- the LM heads (bf16 and int8 weights) for 2 and more token
// rows on the f32 matrix cores, with the one-token head's sums bit for bit.
//
// Reference: crates/lb-ternary/src/bf16.rs:14-105 (bf16_gemv, looped over the
// rows by ops.rs:199-218), q8head.rs:34-57.
//
// The one-token head gives lane l of a wavefront the row's 8-element chunks
// l, l + 64, ...: a chain of fused multiply-adds in element order, then the
// 64 chains combine by an xor butterfly over 32, 16, 8, 4, 2, 1.
// v_mfma_f32_16x16x1_4b does one fused multiply-add of four such chains for
// 16 token rows x 16 weight rows (block b of an accumulator is one chain;
// each step correctly rounded, checked on this part against fmaf), so a
// chain of them is the lane's chain.  With l = 8 q + 2 b + a, accumulator
// (q, a) holds the chains of blocks b = 0..3; the butterfly's pairs are then
// q ^ 4, q ^ 2, q ^ 1 (whole accumulators), b ^ 2, b ^ 1 (blocks) and a.
#include <hip/hip_runtime.h>

#include "lbt_device.h"
#include "lbt_internal.h"

namespace lbt {

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kTok = 16;       // token rows per workgroup
constexpr int kVoc = 16;       // weight rows per wavefront and tile
constexpr int kNT = 512;       // two wavefronts per SIMD, wavefront q the chains 8 q ..
constexpr int kMaxNch = 5;     // chunks per chain (columns up to 2560: 80 registers of a token row)

__device__ __forceinline__ f32x16 outer4(float a, float b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_16x16x1f32(a, b, c, 0, 0, 0);
}

}  // namespace

// Eight wavefronts, one tile of 16 weight rows at a time for 16 token rows:
// wavefront q has the chains 8 q .. 8 q + 7.  Its part of the token rows
// (80 registers at 2560 columns) stays in registers, so the matrix
// instructions take both operands from there; of each weight row it reads
// 128 contiguous bytes (bf16) out of every 1024, and the eight wavefronts
// together whole rows.  Weight chunks are reloaded for the tile after the
// next as soon as they are used (20 KB in flight a wavefront, 160 KB a CU).
// The accumulators meet in LDS (64 KB a tile, two tiles' worth, one barrier
// a tile); a lane then adds one (token, row) sum's chains of one a.
// Workgroup i takes token group i / ntw of row part i % ntw: with ntw a
// multiple of 8 the groups of a part run on one XCD and share its L2's copy
// of the weights.
//
// Bound by the f32 multiply-adds (68 us per 16 rows and 128256 x 2560, used or
// not) with the widening after them (the two take turns on a SIMD), and up to
// 16 rows of bf16 by HBM beside them (657 MB, 100 us).  128256 x 2560: 16
// rows 210 -> 160 us (lmhead_batch_kernel with the next weights in flight ->
// this), 24 rows 360 -> 256, 64 rows 700 -> 460; int8 weights 16 rows 190 ->
// 135, 64 rows 710 -> 494.  Measured beside it: the token rows in LDS and a
// whole 16 x 16 tile a wavefront (16 rows 160, 64 rows 555; with 64-byte
// pieces of a row a load 200), and the exchange's reads and barrier right
// after its writes (64 rows 520).
template <int NCH, bool FULL, bool Q8>
__global__ __launch_bounds__(kNT) void lmhead_tile_kernel(const void* W, const float* rscale, int rows, int cols,
                                                          const float* xn, int m, int part_tiles, float* logits,
                                                          unsigned long long* key) {
    constexpr int NV = Q8 ? 1 : 2;  // 16-byte loads of a lane's two chunks
    extern __shared__ __align__(16) float part_s[];  // [2][q][a][16 registers][64 lanes]
    const int ngroups = (m + kTok - 1) / kTok, ntw = (int)gridDim.x / ngroups;
    const int grp = (int)blockIdx.x / ntw, part = (int)blockIdx.x % ntw;
    const int t0 = grp * kTok, nt = m - t0 < kTok ? m - t0 : kTok;
    const int tid = (int)threadIdx.x, lane = tid & 63, n = lane & 15, b = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nchunks = cols >> 3, c0 = 8 * w + 2 * b;  // this lane's chunks: c0 + a + 64 i
    const int ntiles = (rows + kVoc - 1) / kVoc;
    const int tile_end = (part + 1) * part_tiles < ntiles ? (part + 1) * part_tiles : ntiles;

    u32x4 wb[2][NCH][NV];
    auto load = [&](int tile, int i, u32x4 (&d)[NV]) {
        int r = tile * kVoc + n;
        r = r < rows ? r : rows - 1;  // past the end: a valid row (not stored)
        const char* p = (const char*)W + (size_t)r * cols * (Q8 ? 1 : 2);
        const bool all = FULL || i + 1 < NCH;  // only a last chunk can be past the row's end
        const int c = c0 + 64 * i;
        if constexpr (Q8) {
            if (FULL) {
                d[0] = __builtin_nontemporal_load((const LBT_GLOBAL u32x4*)(p + 8 * c));
            } else if (all) {  // rows are multiples of 8 bytes: two 8-byte loads
                d[0].xy = __builtin_nontemporal_load((const LBT_GLOBAL u32x2*)(p + 8 * c));
                d[0].zw = __builtin_nontemporal_load((const LBT_GLOBAL u32x2*)(p + 8 * c + 8));
            } else {
                d[0] = u32x4{0, 0, 0, 0};
                if (c < nchunks) d[0].xy = __builtin_nontemporal_load((const LBT_GLOBAL u32x2*)(p + 8 * c));
                if (c + 1 < nchunks) d[0].zw = __builtin_nontemporal_load((const LBT_GLOBAL u32x2*)(p + 8 * c + 8));
            }
        } else {
#pragma unroll
            for (int a = 0; a < 2; a++) {
                if (!all) d[a] = u32x4{0, 0, 0, 0};
                if (all || c + a < nchunks)
                    d[a] = __builtin_nontemporal_load((const LBT_GLOBAL u32x4*)(p + 16 * (c + a)));
            }
        }
    };
    int tile = part * part_tiles;
    if (tile >= tile_end) return;  // (the whole workgroup)
#pragma unroll
    for (int k = 0; k < 2; k++)
#pragma unroll
        for (int i = 0; i < NCH; i++) load(tile + k, i, wb[k][i]);

    // this lane's token row; columns past the end are -0: its product with a
    // zero weight leaves every sum as it is
    float xv[NCH][2][8];
#pragma unroll
    for (int i = 0; i < NCH; i++)
#pragma unroll
        for (int a = 0; a < 2; a++) {
            const int c = c0 + a + 64 * i;
            const float* p = xn + (size_t)(t0 + (n < nt ? n : 0)) * cols + 8 * c;
            const bool in = FULL || i + 1 < NCH || c < nchunks;
            if (((uintptr_t)xn & 15) == 0) {  // uniform
                const f32x4 pad = {-0.0f, -0.0f, -0.0f, -0.0f};
                const f32x4 lo = in ? gload((const f32x4*)p) : pad, hi = in ? gload((const f32x4*)p + 1) : pad;
#pragma unroll
                for (int e = 0; e < 4; e++) xv[i][a][e] = lo[e], xv[i][a][4 + e] = hi[e];
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++) xv[i][a][e] = in ? gload(p + e) : -0.0f;
            }
        }

    // this lane's output after the exchange: registers 4 blk + oi of lane ol
    const int oi = w >> 1, ol = (w & 1) * 32 + (lane & 31), oa = lane >> 5;
    const int otok = 4 * (ol >> 4) + oi, ovoc = ol & 15;
    unsigned long long best = 0ull;

    // the chains of this lane's output, read ahead of the next tile's work and added after it
    float pv[4][8];
    auto fetch = [&](const float* buf) {
        __syncthreads();
        const float* pr = buf + (oa * 16 + oi) * 64 + ol;
#pragma unroll
        for (int k = 0; k < 4; k++)
#pragma unroll
            for (int q = 0; q < 8; q++) pv[k][q] = pr[(q * 32 + 4 * k) * 64];
        __builtin_amdgcn_sched_barrier(0);
    };
    // the wavefront's chains of a tile; the slots reload for the tile after the next
    auto chains = [&](int tile, u32x4 (&d)[NCH][NV], f32x16 (&c)[2], const float* prev) {
#pragma unroll
        for (int i = 0; i < NCH; i++) {
            if (i == NCH / 2 && prev) fetch(prev);  // the previous tile's sums: the barrier falls amid this tile's work
#pragma unroll
            for (int v = 0; v < NV; v++) pin(d[i][v]);
#pragma unroll
            for (int a = 0; a < 2; a++) {
                float wf[8];
                if constexpr (Q8) {
                    // byte ^ 0x80 is the weight + 128; as the low byte of 2^23's
                    // mantissa it is 2^23 + 128 + weight, the subtraction exact
#pragma unroll
                    for (int e = 0; e < 8; e++)
                        wf[e] = __uint_as_float(__builtin_amdgcn_perm(0x4b000000u,
                                                                      d[i][0][2 * a + (e >> 2)] ^ 0x80808080u,
                                                                      0x07040400u + (e & 3))) -
                                8388736.0f;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        wf[2 * e] = __uint_as_float(d[i][a][e] << 16);
                        wf[2 * e + 1] = __uint_as_float(d[i][a][e] & 0xffff0000u);
                    }
                }
#pragma unroll
                for (int e = 0; e < 8; e++) c[a] = outer4(xv[i][a][e], wf[e], i == 0 && e == 0 ? f32x16{} : c[a]);
            }
            __builtin_amdgcn_sched_barrier(0);
            load(tile + 2, i, d[i]);
        }
    };
    auto publish = [&](const f32x16 (&c)[2], float* buf) {
        float* pw = buf + (size_t)w * 2 * 16 * 64 + lane;
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int r = 0; r < 16; r++) pw[(a * 16 + r) * 64] = c[a][r];
    };
    auto finish = [&](int tile) {
        float blk[4];
#pragma unroll
        for (int k = 0; k < 4; k++)
            blk[k] = ((pv[k][0] + pv[k][4]) + (pv[k][2] + pv[k][6])) + ((pv[k][1] + pv[k][5]) + (pv[k][3] + pv[k][7]));
        float sum = xor_add<32>((blk[0] + blk[2]) + (blk[1] + blk[3]));
        const int row = tile * kVoc + ovoc;
        if (oa == 0 && otok < nt && row < rows) {
            if constexpr (Q8) sum = gload(rscale + row) * sum;
            if (logits) gstore(logits + (size_t)(t0 + otok) * rows + row, sum);
            const unsigned long long k = argmax_key(sum, (uint32_t)row);
            best = k > best ? k : best;
        }
    };
    // one barrier a tile: a buffer is written again two tiles later, past the
    // barrier that follows its readers' adds
    float* const buf0 = part_s;
    float* const buf1 = part_s + 8 * 2 * 16 * 64;
    f32x16 c[2];
    chains(tile, wb[0], c, nullptr);
    publish(c, buf0);
    for (; tile + 2 < tile_end; tile += 2) {
        chains(tile + 1, wb[1], c, buf0);
        finish(tile);
        publish(c, buf1);
        chains(tile + 2, wb[0], c, buf1);
        finish(tile + 1);
        publish(c, buf0);
    }
    const float* last = buf0;
    if (tile + 1 < tile_end) {
        chains(tile + 1, wb[1], c, buf0);
        finish(tile);
        publish(c, buf1);
        tile++;
        last = buf1;
    }
    fetch(last);
    finish(tile);
#pragma unroll
    for (int k = 0; k < 2; k++)
#pragma unroll
        for (int i = 0; i < NCH; i++)
#pragma unroll
            for (int v = 0; v < NV; v++) keep(wb[k][i][v]);
    if (!key) return;
    // one atomic per (workgroup, token): lanes 16 apart hold different tokens
    unsigned long long k = best;
#pragma unroll
    for (int d = 8; d >= 1; d >>= 1) {
        const unsigned long long o = __shfl_xor(k, d);
        k = o > k ? o : k;
    }
    if (oa == 0 && ovoc == 0 && otok < nt && k) atomicMax(&key[t0 + otok], k);
}

namespace {

template <int NCH, bool FULL, bool Q8>
int launch(lbt_ctx* ctx, const void* w, const float* rscale, int rows, int cols, const float* xn, int m,
           float* logits, unsigned long long* key) {
    constexpr size_t lds = (size_t)2 * 8 * 2 * 16 * 64 * 4;
    // on every call: per device, and without state of ours
    LBT_HIP(ctx, hipFuncSetAttribute((const void*)lmhead_tile_kernel<NCH, FULL, Q8>,
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    const int ngroups = (m + kTok - 1) / kTok, ntiles = (rows + kVoc - 1) / kVoc;
    int parts = ctx->cus / ngroups;
    if (parts < 1) parts = 1;
    const int part_tiles = (ntiles + parts - 1) / parts;
    parts = (ntiles + part_tiles - 1) / part_tiles;
    hipEvent_t e0, e1;
    prof_pair(ctx, &e0, &e1);
    hipExtLaunchKernelGGL((lmhead_tile_kernel<NCH, FULL, Q8>), dim3(parts * ngroups), dim3(kNT), lds, ctx->stream, e0,
                          e1, 0, w, rscale, rows, cols, xn, m, part_tiles, logits, key);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return hip_err(ctx, e, "lmhead_tile_kernel launch");
    prof_commit(ctx, e0, e1, kProfHead, (double)rows * cols * (Q8 ? 1.0 : 2.0));
    return LBT_OK;
}

}  // namespace

int launch_head_tile(lbt_ctx* ctx, const void* w, const float* rscale, int rows, int cols, const float* xn, int m,
                     float* logits, unsigned long long* key) {
    const int nch = (cols / 8 + 63) / 64;
    if (cols % 8 || cols <= 0 || rows <= 0 || m < 1 || nch > kMaxNch) return 1;
    const bool full = cols % 512 == 0;
    // Up to 8 rows lmhead_batch_kernel's 8-row groups waste nothing: it stays
    // where columns past a chain's last chunk would have to be masked (1000
    // columns x 32000 rows, 6 rows of int8: 22.3 against 25.8 us), and so it does
    // with fewer than two tiles a CU (2560 x 4000: 11 against 17 us at 6 rows, 15
    // to 17 against 19 at 16).
    const long tiles = (long)((rows + kVoc - 1) / kVoc) * ((m + kTok - 1) / kTok);
    if ((m <= 8 && !full) || tiles <= 2L * ctx->cus) return 1;
#define LBT_HEAD_TILE(N)                                                                                \
    case N:                                                                                             \
        if (rscale)                                                                                     \
            return full ? launch<N, true, true>(ctx, w, rscale, rows, cols, xn, m, logits, key)         \
                        : launch<N, false, true>(ctx, w, rscale, rows, cols, xn, m, logits, key);       \
        return full ? launch<N, true, false>(ctx, w, nullptr, rows, cols, xn, m, logits, key)           \
                    : launch<N, false, false>(ctx, w, nullptr, rows, cols, xn, m, logits, key);
    switch (nch) {
        LBT_HEAD_TILE(1)
        LBT_HEAD_TILE(2)
        LBT_HEAD_TILE(3)
        LBT_HEAD_TILE(4)
        LBT_HEAD_TILE(5)
    }
#undef LBT_HEAD_TILE
    return 1;
}

}  // namespace lbt
