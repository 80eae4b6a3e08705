// head_tile.hip -- the LM heads (bf16 and int8 weights) for 2 and more token
// rows on the f32 matrix cores, with the one-token head's sums bit for bit.
//
// Reference: crates/lb-ternary/src/bf16.rs:14-105 (bf16_gemv, looped over the
// rows by ops.rs:199-218), q8head.rs:34-57.
//
// The one-token head gives lane l of a wavefront the row's 8-element chunks
// l, l + 64, ...: a chain of fused multiply-adds in element order, then the
// 64 chains combine by an xor butterfly over 32, 16, 8, 4, 2, 1.
// v_mfma_f32_4x4x1_16b does one fused multiply-add of sixteen such chains for
// 4 token rows x 4 weight rows (block k of an accumulator is one chain; each
// step correctly rounded, denormals kept, checked on this part against fmaf),
// so a chain of them is the lane's chain.  With l = 16 g + k, accumulator g
// holds the chains of blocks k = 0..15; the butterfly's pairs are then g ^ 2,
// g ^ 1 (accumulators) and lanes 32, 16, 8, 4 apart (lane 4 k + j), by
// recursive halving of a wavefront's sums.
#include <hip/hip_runtime.h>

#include "lbt_device.h"
#include "lbt_internal.h"

#include <type_traits>

namespace lbt {

namespace {

constexpr int kMaxNch = 5;  // chunks per chain: columns up to 2560 (16 rows of f32 fill the LDS)

}  // namespace

// 4 TG token rows in LDS (16-byte granule x of row t at x ^ ((t & 1) + 4 (t &
// 2)), so four rows' reads of four chunks fall on distinct banks), a
// wavefront takes tiles of 4 RG weight rows: a load is 256 contiguous bytes
// (bf16) of each of 4 rows, RING steps ahead of the matrix instructions (64 to
// 160 KB in flight a CU).  Up to 8 rows two workgroups of four wavefronts a
// CU, above one of eight (16 rows fill its LDS; RG = 2 there and RING = 2 at
// 12 rows of bf16 keep the sums in registers).  Workgroup i takes token group i / ntw of row part i % ntw: with
// ntw a multiple of 8 the groups of a part run on one XCD and share its L2's
// copy of the weights.
//
// Up to 8 rows of bf16 weights bound by HBM (128256 x 2560, 657 MB: 101 to
// 107 us, 6.4 TB/s; lmhead_batch_kernel 143), beyond and for int8 weights by
// the f32 multiply-adds (68 us per 16 rows, used or not, 51 per 12) with the widening
// after them: matrix and vector instructions take turns on a SIMD.  bf16, 16
// rows 199 -> 132 us, 24 rows 372 -> 215, 64 rows 756 -> 488; int8, 6 rows 129 ->
// 88, 16 rows 189 -> 132, 24 rows 359 -> 206.  Measured beside it: 16 x 16 x 1 instructions (four
// chains), with the token rows in LDS and a whole tile a wavefront (16 rows of
// bf16 160 us, with 64-byte pieces of a row a load 200), and with the chains
// split over eight wavefronts, token rows in registers and an exchange of the
// sums through LDS (150; 64 rows 477).  FULL (columns a multiple of 512, no
// bounds test on a load) is worth 1 to 3%, at 16 rows of 512 columns 9%, and up to 28%
// at 12 rows, where the test's registers add to what spills (128256 x 2560 bf16:
// 128 against 155 us).
template <int NCH, bool FULL, bool Q8, int TG, int RG, int NT>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(2))) void lmhead_tile_kernel(
    const void* W, const float* rscale, int rows, int cols, const float* xn, int m, int part_tiles, float* logits,
    unsigned long long* key) {
    constexpr int G = NCH * 128;  // 16-byte granules per token row
    constexpr int STEPS = 4 * NCH, RING = RG == 2 ? 2 * NCH : TG == 3 && !Q8 ? 2 : 4, NW = NT / 64;  // | STEPS
    constexpr int RT = 4 * RG;  // weight rows per wavefront and tile
    using Chunk = typename std::conditional<Q8, u32x2, u32x4>::type;
    extern __shared__ __align__(16) float xs[];  // [4 TG][4 G]
    const int tid = (int)threadIdx.x, lane = tid & 63, j = lane & 3, k = lane >> 2;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nchunks = cols >> 3, ntiles = (rows + RT - 1) / RT;
    const int ngroups = (m + 4 * TG - 1) / (4 * TG), ntw = (int)gridDim.x / ngroups;
    const int t0 = (int)blockIdx.x / ntw * (4 * TG), part = (int)blockIdx.x % ntw;
    const int nt = m - t0 < 4 * TG ? m - t0 : 4 * TG;
    xn += (size_t)t0 * cols;
    const int tile_end = (part + 1) * part_tiles < ntiles ? (part + 1) * part_tiles : ntiles;
    constexpr int kG[4] = {0, 2, 1, 3};

    // step s: chunks 16 g + k + 64 i of 16 rows, g = kG[s / NCH], i = s % NCH
    Chunk wb[RING][RG];
    auto load = [&](int tile, int s, Chunk (&d)[RG]) {
        const int i = s % NCH, c = 16 * kG[s / NCH] + k + 64 * i;
#pragma unroll
        for (int rg = 0; rg < RG; rg++) {
            int r = tile * RT + 4 * rg + j;
            r = r < rows ? r : rows - 1;  // past the end: a valid row (not stored)
            const Chunk* p = (const Chunk*)((const char*)W + (size_t)r * cols * (Q8 ? 1 : 2)) + c;
            d[rg] = Chunk{};
            if (FULL || i + 1 < NCH || c < nchunks)  // only a last chunk can be past the row's end
                d[rg] = __builtin_nontemporal_load((const LBT_GLOBAL Chunk*)p);
        }
    };
    int tile = part * part_tiles + w;
    const int first = tile < tile_end ? tile : 0;
#pragma unroll
    for (int s = 0; s < RING; s++) load(first, s, wb[s]);

    // token rows; columns past the end are -0: a product of it with a zero
    // weight leaves every sum as it is
    auto swz = [](int t) { return (t & 1) + 4 * (t & 2); };
    // every row starts aligned if the first does (cols is a multiple of 8); 2432
    // columns, 8500 rows, 16 tokens: 32 us, value by value 50
    if (((uintptr_t)xn & 15) == 0) {
        for (int i = tid; i < 4 * TG * G; i += NT) {
            const int t = i / G, g = i % G;
            f32x4 v = {-0.0f, -0.0f, -0.0f, -0.0f};
            if (t < nt && (FULL || 4 * g < cols)) v = gload((const f32x4*)(xn + (size_t)t * cols) + g);
            *(f32x4*)(xs + 4 * (t * G + (g ^ swz(t)))) = v;
        }
    } else {
        for (int i = tid; i < 4 * TG * G * 4; i += NT) {
            const int t = i / (4 * G), e = i % (4 * G);
            float v = -0.0f;
            if (t < nt && e < cols) v = gload(xn + (size_t)t * cols + e);
            xs[4 * (t * G + ((e >> 2) ^ swz(t))) + (e & 3)] = v;
        }
    }
    __syncthreads();
    const float* xa[TG][2];  // this lane's token row (j of each group), halves of chunk k
#pragma unroll
    for (int tg = 0; tg < TG; tg++)
#pragma unroll
        for (int h = 0; h < 2; h++) xa[tg][h] = xs + 4 * ((4 * tg + j) * G + ((2 * k + h) ^ swz(j)));

    // this lane's outputs after the halving: sums NS k .. of the 4 RG TG of a
    // weight row j, sum index (token group * RG + row group) * 4 + token
    constexpr int NS = TG * RG / 4;
    const int i0 = NS * k;
    auto orow = [&](int z) { return 4 * (((i0 + z) >> 2) % RG) + j; };
    auto otok = [&](int z) { return 4 * (((i0 + z) >> 2) / RG) + ((i0 + z) & 3); };
    unsigned long long best[NS] = {};

    for (; tile < tile_end; tile += NW) {
        f32x4 c[TG][RG], a[TG][RG], t[TG][RG];  // current g; g 0 (+ 2); g 1
        const int next = tile + NW < tile_end ? tile + NW : tile;
#pragma unroll
        for (int s = 0; s < STEPS; s++) {
            Chunk (&cur)[RG] = wb[s % RING];
            const int i = s % NCH, gs = s / NCH;
#pragma unroll
            for (int rg = 0; rg < RG; rg++) pin(cur[rg]);
            float xv[TG][8];
#pragma unroll
            for (int tg = 0; tg < TG; tg++)
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const f32x4 v = *(const f32x4*)(xa[tg][h] + 4 * (32 * kG[gs] + 128 * i));
#pragma unroll
                    for (int e = 0; e < 4; e++) xv[tg][4 * h + e] = v[e];
                }
#pragma unroll
            for (int rg = 0; rg < RG; rg++) {
                float wf[8];
                if constexpr (Q8) {
#pragma unroll
                    for (int e = 0; e < 8; e++)
                        wf[e] = __uint_as_float(__builtin_amdgcn_perm(0x4b000000u, cur[rg][e >> 2] ^ 0x80808080u,
                                                                      0x07040400u + (e & 3))) -
                                8388736.0f;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        wf[2 * e] = __uint_as_float(cur[rg][e] << 16);
                        wf[2 * e + 1] = __uint_as_float(cur[rg][e] & 0xffff0000u);
                    }
                }
#pragma unroll
                for (int e = 0; e < 8; e++)
#pragma unroll
                    for (int tg = 0; tg < TG; tg++)
                        c[tg][rg] = __builtin_amdgcn_mfma_f32_4x4x1f32(
                            xv[tg][e], wf[e], i == 0 && e == 0 ? f32x4{0.0f, 0.0f, 0.0f, 0.0f} : c[tg][rg], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            load(s + RING < STEPS ? tile : next, (s + RING) % STEPS, cur);
            if (i == NCH - 1) {
#pragma unroll
                for (int tg = 0; tg < TG; tg++)
#pragma unroll
                    for (int rg = 0; rg < RG; rg++) {
                        if (gs == 0) a[tg][rg] = c[tg][rg];
                        else if (gs == 1) a[tg][rg] = a[tg][rg] + c[tg][rg];
                        else if (gs == 2) t[tg][rg] = c[tg][rg];
                        else a[tg][rg] = a[tg][rg] + (t[tg][rg] + c[tg][rg]);
                        if (gs != 2) pin(a[tg][rg]);
                    }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        float v[TG * RG * 4], o[NS];
#pragma unroll
        for (int tg = 0; tg < TG; tg++)
#pragma unroll
            for (int rg = 0; rg < RG; rg++)
#pragma unroll
                for (int e = 0; e < 4; e++) v[(tg * RG + rg) * 4 + e] = a[tg][rg][e];
        {
            float h1[TG * RG * 2], h2[TG * RG], h3[TG * RG / 2];
            halve<32>(v, h1);
            halve<16>(h1, h2);
            halve<8>(h2, h3);
            halve<4>(h3, o);
        }
#pragma unroll
        for (int z = 0; z < NS; z++) {
            const int row = tile * RT + orow(z);
            if (row >= rows || otok(z) >= nt) continue;
            const float sum = Q8 ? gload(rscale + row) * o[z] : o[z];
            if (logits) gstore(logits + (size_t)(t0 + otok(z)) * rows + row, sum);
            const unsigned long long kz = argmax_key(sum, (uint32_t)row);
            best[z] = kz > best[z] ? kz : best[z];
        }
    }
#pragma unroll
    for (int s = 0; s < RING; s++)
#pragma unroll
        for (int rg = 0; rg < RG; rg++) keep(wb[s][rg]);
    if (!key) return;
    // one atomic per (workgroup, token): the lanes' keys meet in LDS once
    // every wavefront is done with the token rows
    __syncthreads();
    unsigned long long* wbest = (unsigned long long*)xs;  // [4 TG][NW][KW]
    constexpr int KW = RT;  // keys per wavefront and token
#pragma unroll
    for (int z = 0; z < NS; z++) wbest[otok(z) * (NW * KW) + w * KW + orow(z)] = best[z];
    __syncthreads();
    if (tid < nt) {
        unsigned long long b = 0ull;
        for (int i = 0; i < NW * KW; i++) b = wbest[tid * (NW * KW) + i] > b ? wbest[tid * (NW * KW) + i] : b;
        if (b) atomicMax(&key[t0 + tid], b);
    }
}

namespace {

template <int NCH, bool FULL, bool Q8, int TG, int RG, int NT>
int launch_tile(lbt_ctx* ctx, const void* w, const float* rscale, int rows, int cols, const float* xn, int m,
                float* logits, unsigned long long* key) {
    constexpr size_t lds = (size_t)4 * TG * NCH * 128 * 16;
    // on every call: per device, and without state of ours
    LBT_HIP(ctx, hipFuncSetAttribute((const void*)lmhead_tile_kernel<NCH, FULL, Q8, TG, RG, NT>,
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    const int ngroups = (m + 4 * TG - 1) / (4 * TG), ntiles = (rows + 4 * RG - 1) / (4 * RG);
    int parts = (NT == kThreads ? 2 : 1) * ctx->cus / ngroups;
    if (parts < 1) parts = 1;
    const int part_tiles = (ntiles + parts - 1) / parts;
    parts = (ntiles + part_tiles - 1) / part_tiles;
    hipEvent_t e0, e1;
    prof_pair(ctx, &e0, &e1);
    hipExtLaunchKernelGGL((lmhead_tile_kernel<NCH, FULL, Q8, TG, RG, NT>), dim3(parts * ngroups), dim3(NT), lds,
                          ctx->stream, e0, e1, 0, w, rscale, rows, cols, xn, m, part_tiles, logits, key);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return hip_err(ctx, e, "lmhead_tile_kernel launch");
    prof_commit(ctx, e0, e1, kProfHead, (double)rows * cols * (Q8 ? 1.0 : 2.0));
    return LBT_OK;
}
template <int NCH, bool FULL, bool Q8>
int launch_tg(lbt_ctx* ctx, const void* w, const float* rscale, int rows, int cols, const float* xn, int m,
              float* logits, unsigned long long* key) {
    if (m <= 4) return launch_tile<NCH, FULL, Q8, 1, 4, kThreads>(ctx, w, rscale, rows, cols, xn, m, logits, key);
    if (m <= 8) return launch_tile<NCH, FULL, Q8, 2, 4, kThreads>(ctx, w, rscale, rows, cols, xn, m, logits, key);
    // 12 token rows a workgroup where that takes no more groups than 16 (9 to
    // 12, 17 to 24, 33 to 36 rows): 128256 x 2560, 24 rows bf16 245 -> 215 us,
    // int8 248 -> 206; 9 rows 135 -> 122 and 130 -> 107
    if ((m + 11) / 12 == (m + 15) / 16)
        return launch_tile<NCH, FULL, Q8, 3, 4, 512>(ctx, w, rscale, rows, cols, xn, m, logits, key);
    return launch_tile<NCH, FULL, Q8, 4, 2, 512>(ctx, w, rscale, rows, cols, xn, m, logits, key);
}

}  // namespace

int launch_head_tile(lbt_ctx* ctx, const void* w, const float* rscale, int rows, int cols, const float* xn, int m,
                     float* logits, unsigned long long* key) {
    const int nch = (cols / 8 + 63) / 64;
    if (cols % 8 || cols <= 0 || rows <= 0 || m < 1 || nch > kMaxNch) return 1;
    const bool full = cols % 512 == 0;
    if (!head_tiled(rows, m, ctx->cus)) return 1;
#define LBT_HEAD_TILE(N)                                                                             \
    case N:                                                                                          \
        if (rscale)                                                                                  \
            return full ? launch_tg<N, true, true>(ctx, w, rscale, rows, cols, xn, m, logits, key)   \
                        : launch_tg<N, false, true>(ctx, w, rscale, rows, cols, xn, m, logits, key); \
        return full ? launch_tg<N, true, false>(ctx, w, nullptr, rows, cols, xn, m, logits, key)     \
                    : launch_tg<N, false, false>(ctx, w, nullptr, rows, cols, xn, m, logits, key);
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
