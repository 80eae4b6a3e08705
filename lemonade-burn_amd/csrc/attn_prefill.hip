// attn_prefill.hip -- attention splits of a prefill's rows on the f32 matrix
// cores, with the partials of attention_split_ku (attn_common.h) bit for bit
// but for the sign of a zero (below).
//
// Reference: crates/lb-model/src/model.rs:349-357 (GQA attention of a prompt).
//
// v_mfma_f32_16x16x1_4b computes four independent 16 x 16 outer products,
// D[b][i][j] = fma(A[b][i], B[b][j], C[b][i][j]): one correctly rounded fused
// multiply-add per element and instruction, denormals kept, checked on this
// part against fmaf over random operands of all magnitudes.  A chain of them is therefore
// the chain of fused multiply-adds that the fixed float order asks of one
// lane, at 1024 per instruction instead of 64 (the matrix pipe does 32 a
// clock and SIMD, the vector pipe 16, and no operand is moved or widened more
// than once for 16 rows).
#include <hip/hip_runtime.h>

#include "attn_common.h"
#include "lbt_device.h"
#include "lbt_internal.h"

namespace lbt {

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kTileRows = 16;  // query rows per wavefront
constexpr int kHd = 128;       // head dim
constexpr int kTileLds = 256;  // longest split in keys (64 KiB of scores per workgroup)

__device__ __forceinline__ f32x16 outer4(float a, float b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_16x16x1f32(a, b, c, 0, 0, 0);
}

// The four rows a lane holds of a 16 x 16 result, blocks 0..3 of an outer4
// accumulator added as the butterfly over two lane bits adds them.
__device__ __forceinline__ f32x4 blk(const f32x16& v, int b) {
    return f32x4{v[4 * b], v[4 * b + 1], v[4 * b + 2], v[4 * b + 3]};
}

// Lane l's value with that of lane l ^ 8, ^ 4, ^ 2, ^ 1 of its 16 lanes, in
// turn: xor_sum_down<8> / the max of the 16 lanes.  After the step of 8,
// lanes l and l ^ 8 agree, so a rotation by 4 reads what l ^ 4 holds; each
// step is one instruction (DPP operand).
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float row16_sum(float v) {
    v = v + dpp<0x128>(v);
    v = v + dpp<0x124>(v);
    v = v + dpp<0x4E>(v);
    return v + dpp<0xB1>(v);
}
__device__ __forceinline__ float row16_max(float v) {
    v = fmaxf(v, dpp<0x128>(v));
    v = fmaxf(v, dpp<0x124>(v));
    v = fmaxf(v, dpp<0x4E>(v));
    return fmaxf(v, dpp<0xB1>(v));
}

// lbt_expf for x <= 0 or NaN (a score less the row's max): the same value
// without the branches that such x never takes.
__device__ __forceinline__ float exp_le0(float x) {
    const float n = __builtin_rintf(x * 1.44269504088896341f);
    float r = __builtin_fmaf(-n, 0.693145751953125f, x);
    r = __builtin_fmaf(-n, 1.42860682030941723212e-6f, r);
    float p = 1.98412698412698e-4f;
    p = __builtin_fmaf(p, r, 1.38888888888889e-3f);
    p = __builtin_fmaf(p, r, 8.33333333333333e-3f);
    p = __builtin_fmaf(p, r, 4.16666666666667e-2f);
    p = __builtin_fmaf(p, r, 1.66666666666667e-1f);
    p = __builtin_fmaf(p, r, 0.5f);
    p = __builtin_fmaf(p, r, 1.0f);
    p = __builtin_fmaf(p, r, 1.0f);
    return x < -87.0f ? 0.0f : __builtin_amdgcn_ldexpf(p, (int)n);  // exact: the result is normal
}

}  // namespace

// One wavefront per (query head, 16 rows, key split), four per workgroup.
//
// Rows: tile j holds the rows with 16 j + 1 .. 16 j + 16 visible keys.  They
// have the same keys per split, max(64, j + 1), and the same number of splits
// (16 j + 1 .. 16 j + 16 lie between two multiples of 64; past 1024 keys
// every row has 16 splits), so a split is one rectangle of 16 rows x up to
// `ks` keys whose last tile of keys may be masked per row.
//
// Scores of 16 keys: lane (n = lane & 15, b = lane >> 4) holds row n's q and
// key n's k in chunks 4 i + b of 8 dims, so block b of accumulator i is chunk
// lane 4 i + b of attention_split_ku: 8 instructions per accumulator run the
// 8 dims in order, then the chunks combine 8, 4 (accumulators), 2, 1 (blocks)
// apart.  The result has key n and rows 4 b .. 4 b + 3 on lane (n, b).
// Exponentials: the sum over keys u, u + 32, u + 16 ... of one virtual
// wavefront (64 keys) is the butterfly's, four key tiles first, then lanes.
// PV: block b of the accumulator of virtual wavefront v is key group
// 4 v + b, one instruction per 16 keys and 16 dims, groups and virtual
// wavefronts combined as there; lane (n, b) loads dims 64 half + 4 n .. + 3
// of its key, so the four dims of a lane are 8 contiguous bytes of V and 16
// of the output.
//
// A key that a row does not see has p = 0 there: fma(0, v, acc) = acc, but for
// an acc of -0 (every product so far below the denormals), which may become
// +0.  A partial can so differ from attention_split_ku's in the sign of a
// zero; the o projection's input is rounded to integers, which have none.
// That needs v finite: a non-finite V value among the tile's
// partly masked keys makes the wavefront redo PV row by row, each with the
// keys past its own read as zeros.
//
// Bound by instruction issue: the f32 matrix instructions (2 x 1024 fused
// multiply-adds x 16 per 16 x 16 scores, 32 clocks per 1024) and the vector
// ones (widening, tree adds, exponentials: about half as long) take turns on
// a SIMD, they do not overlap (measured: 4 outer4 55 ns, with 32 adds 97 ns).
// Three wavefronts a SIMD; four (128 registers) spill.  2048-token prefill of
// the 2B shape, per layer (the products alone would take 150 us): one
// wavefront per (row, KV head, split) 590 us -> 315 us; 1024 tokens 163 -> 89,
// 4096 tokens 2010 -> 1190.
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(3))) void attention_tile_kernel(
    const float* q, int nh, int gh, int pos0, int m, const uint16_t* kc, const uint16_t* vc, int cap, float scaling,
    float* o, float* ml, int scw) {
    extern __shared__ __align__(16) float sc_all[];  // [4][scw], one wavefront's [key][16 rows]
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int h = (int)blockIdx.x * 4 + w, s = (int)blockIdx.z;
    if (h >= nh) return;  // the last workgroup's spare wavefronts
    const int j = pos0 / kTileRows + (int)blockIdx.y;
    const int vis_hi = kTileRows * j + kTileRows;  // visible keys of the tile's last row
    const int ks = attn_split_keys(vis_hi);
    if (s >= (vis_hi + ks - 1) / ks) return;
    const int k0 = s * ks;
    const int cmax = vis_hi - k0 < ks ? vis_hi - k0 : ks;              // keys of the rectangle
    const int avail = pos0 + m - k0 < cmax ? pos0 + m - k0 : cmax;     // of them in the cache
    const int cnt0 = vis_hi - (kTileRows - 1) - k0 < ks ? vis_hi - (kTileRows - 1) - k0 : ks;  // keys of row 0
    const int nkt = (cmax + 15) / 16;
    float* sc = sc_all + w * scw;
    const int lane = (int)threadIdx.x & 63, n = lane & 15, b = lane >> 4;
    const int H = nh * kHd;
    const size_t kvoff = ((size_t)(h / gh) * cap + k0) * kHd;
    const int trow = kTileRows * j - pos0;  // the forward's row of tile row 0 (may be negative)

    // ---- scores
    const __amdgpu_buffer_rsrc_t kr = buf_rsrc(kc + kvoff, (uint32_t)avail * kHd * 2u);
    const uint32_t koff = (uint32_t)(n * kHd + 8 * b) * 2u;
    u32x4 kb[4];
    auto k_load = [&](int kt) {
#pragma unroll
        for (int i = 0; i < 4; i++)
            kb[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                  kr, koff + 64u * i, (uint32_t)kt * 16u * kHd * 2u, 0));
    };
    k_load(0);
    float qf[4][8];
    {
        int t = trow + n;
        t = t < 0 ? 0 : (t < m ? t : m - 1);  // rows outside the forward: computed, not stored
        const float* qr = q + (size_t)t * H + h * kHd + 8 * b;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const f32x4 a = gload((const f32x4*)(qr + 32 * i)), c = gload((const f32x4*)(qr + 32 * i + 4));
#pragma unroll
            for (int e = 0; e < 4; e++) qf[i][e] = a[e], qf[i][4 + e] = c[e];
        }
    }
    // score rows of 16: key's rows 4 r .. 4 r + 3 sit at 4 (r ^ (key / 4 & 3)),
    // so 16 lanes' 16-byte accesses of one row group fall on distinct banks
    float* const sw = sc + n * 16 + 4 * (b ^ (n >> 2 & 3));  // key n of a tile, rows 4 b ..
    // visible keys of rows 4 b + i in this split
    int cnt[4];
    float mx[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int c = vis_hi - (kTileRows - 1) + 4 * b + i - k0;
        cnt[i] = c < ks ? c : ks;
        mx[i] = -__builtin_inff();
    }
#pragma unroll 1
    for (int kt = 0; kt < nkt; kt++) {
        float kf[4][8];
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                kf[i][2 * e] = bf16_to_f32((uint16_t)(kb[i][e] & 0xffffu));
                kf[i][2 * e + 1] = bf16_to_f32((uint16_t)(kb[i][e] >> 16));
            }
        if (kt + 1 < nkt) k_load(kt + 1);
        f32x16 c02, c13;
        auto chain = [&](int i) {
            f32x16 c = {};
#pragma unroll
            for (int e = 0; e < 8; e++) c = outer4(qf[i][e], kf[i][e], c);
            __builtin_amdgcn_sched_barrier(0);  // one chain at a time: 16 registers each
            return c;
        };
        c02 = chain(0);
        c02 = c02 + chain(2);
        c13 = chain(1);
        c13 = c13 + chain(3);
        c02 = c02 + c13;
        const f32x4 sum = (blk(c02, 0) + blk(c02, 2)) + (blk(c02, 1) + blk(c02, 3));
        const f32x4 sv = sum * scaling;
        const int key = 16 * kt + n;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            float x = sv[i];
            if (16 * kt + 16 > cnt0) x = key < cnt[i] ? x : -__builtin_inff();  // uniform: a partly masked tile
            mx[i] = fmaxf(mx[i], x);
        }
        *(f32x4*)(sw + 256 * kt) = sv;
    }
#pragma unroll
    for (int i = 0; i < 4; i++) mx[i] = row16_max(mx[i]);

    // ---- exponentials (each lane its own scores) and their sums
    // (l_0 + l_1) + (l_2 + l_3) over the virtual wavefronts of 64 keys; key
    // tiles past the last one in its virtual wavefront get p = 0, and a
    // virtual wavefront without keys would add 0
    float l[4], lp[4];
#pragma unroll
    for (int i = 0; i < 4; i++) l[i] = lp[i] = 0.0f;
#pragma unroll 1
    for (int v = 0; 4 * v < nkt; v++) {
        f32x4 e[4];
#pragma unroll
        for (int t = 0; t < 4; t++) {
            f32x4* sp = (f32x4*)(sw + 256 * (4 * v + t));
            const f32x4 sv = *sp;
#pragma unroll
            for (int i = 0; i < 4; i++) e[t][i] = exp_le0(sv[i] - mx[i]);
            if (64 * v + 16 * t + 16 > cnt0) {  // uniform: a partly masked tile
                const int key = 16 * (4 * v + t) + n;
#pragma unroll
                for (int i = 0; i < 4; i++) e[t][i] = key < cnt[i] ? e[t][i] : 0.0f;
            }
            *sp = e[t];
        }
        const f32x4 es = (e[0] + e[2]) + (e[1] + e[3]);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float lv = row16_sum(es[i]);
            if (v & 1) l[i] = l[i] + (lp[i] + lv), lp[i] = 0.0f;
            else lp[i] = lv;
        }
    }
#pragma unroll
    for (int i = 0; i < 4; i++) l[i] = l[i] + lp[i];
    if (n == 0) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int t = trow + 4 * b + i;
            if (t >= 0 && t < m)
                gstore((f32x2*)(ml + (((size_t)t * kAttnSplits + s) * nh + h) * 2),
                       f32x2{mx[i], l[i]});
        }
    }
    asm volatile("" ::: "memory");  // the exponential stores before the PV reads (LDS is in order per wavefront)

    // ---- PV
    const uint16_t* V = vc + kvoff;
    bool redo = false;                               // a non-finite V among the partly masked keys
    if (cnt0 < avail) {
        const __amdgpu_buffer_rsrc_t vr = buf_rsrc(V, (uint32_t)avail * kHd * 2u);
        uint32_t bad = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const u32x4 x = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                          vr, koff + 64u * i, (uint32_t)cnt0 * kHd * 2u, 0));
#pragma unroll
            for (int e = 0; e < 4; e++) {
                bad |= (uint32_t)((x[e] & 0x7f80u) == 0x7f80u);
                bad |= (uint32_t)((x[e] & 0x7f800000u) == 0x7f800000u);
            }
        }
        redo = __builtin_amdgcn_ballot_w64(bad != 0) != 0;
    }
    const int passes = redo ? kTileRows : 1;
#pragma unroll 1
    for (int pass = 0; pass < passes; pass++) {
        int vkeys = avail;
        if (redo) {
            const int c = cnt0 + pass < ks ? cnt0 + pass : ks;
            vkeys = c < avail ? c : avail;
        }
        const __amdgpu_buffer_rsrc_t vr = buf_rsrc(V, (uint32_t)vkeys * kHd * 2u);
        const uint32_t voff = (uint32_t)(b * kHd + 4 * n) * 2u;
        u32x2 vb[4];
        // keys 16 (u + i) + 4 v + b, dims 64 half + 4 n .. (hv = 4 half + v; past the last: not used)
        auto v_load = [&](int hv, int u) {
            const uint32_t so = (uint32_t)((4 * (hv & 3) + 16 * u) * kHd * 2 + 128 * (hv >> 2));
#pragma unroll
            for (int i = 0; i < 4; i++)
                vb[i] = __builtin_bit_cast(
                    u32x2, __builtin_amdgcn_raw_buffer_load_b64(vr, voff + (uint32_t)i * 16u * kHd * 2u, so, 0));
        };
        v_load(0, 0);
#pragma unroll 1
        for (int half = 0; half < 2; half++) {
            f32x4 first[4], even[4];  // sums of virtual wavefronts 0 + 1, and 2 (+ 3)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                f32x16 acc[4];
                // 64 keys of the virtual wavefront's groups: 16 (u + i) + 4 v + b
                auto batch = [&](int u, bool start) {
                    float vf[4][4], a[4];
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        a[i] = sc[(16 * (u + i) + 4 * v + b) * 16 + (n ^ 4 * v)];
#pragma unroll
                        for (int d = 0; d < 2; d++) {
                            vf[i][2 * d] = bf16_to_f32((uint16_t)(vb[i][d] & 0xffffu));
                            vf[i][2 * d + 1] = bf16_to_f32((uint16_t)(vb[i][d] >> 16));
                        }
                    }
                    const bool more = u + 4 < nkt;
                    v_load(4 * half + v + (more ? 0 : 1), more ? u + 4 : 0);
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        if (i > 0 && u + i >= nkt) break;  // uniform
#pragma unroll
                        for (int d = 0; d < 4; d++)
                            acc[d] = outer4(a[i], vf[i][d], start && i == 0 ? f32x16{} : acc[d]);
                    }
                };
                batch(0, true);
#pragma unroll 1
                for (int u = 4; u < nkt; u += 4) batch(u, false);
#pragma unroll
                for (int d = 0; d < 4; d++) {
                    f32x4 r = (blk(acc[d], 0) + blk(acc[d], 1)) + (blk(acc[d], 2) + blk(acc[d], 3));
                    pin(r);  // here, not where the sum is used: the accumulators are free again
                    if (v == 0) first[d] = r;
                    else if (v == 1) first[d] = first[d] + r;
                    else if (v == 2) even[d] = r;
                    else first[d] = first[d] + (even[d] + r);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int t = trow + 4 * b + i;
                if (t >= 0 && t < m && (!redo || 4 * b + i == pass))
                    gstore((f32x4*)(o + ((size_t)t * kAttnSplits + s) * H + h * kHd + 64 * half + 4 * n),
                           f32x4{first[0][i], first[1][i], first[2][i], first[3][i]});
            }
        }
    }
}

int launch_attention_tile(lbt_ctx* ctx, const float* q, int m, int nh, int kvh, int hd, const RowPos& rp,
                          const uint16_t* kc, const uint16_t* vc, int cap, float scaling, float* o, float* ml) {
    const int ks = attn_split_keys(rp.vis_max);
    if (hd != kHd || m < 2 || rp.tok_pos || rp.pos_dev || ks > kTileLds) return 1;
    if (ctx->tune.attn_tile < 0 && !attn_tiles_pay(m, rp.pos0, nh, kvh, attn_splits(rp.vis_max), ks)) return 1;
    const int ntiles = (rp.pos0 + m - 1) / kTileRows - rp.pos0 / kTileRows + 1;
    const int scw = (ks + 63) / 64 * 64 * kTileRows;
    hipEvent_t e0, e1;
    prof_pair(ctx, &e0, &e1);
    hipExtLaunchKernelGGL(attention_tile_kernel, dim3((nh + 3) / 4, ntiles, attn_splits(rp.vis_max)),
                          dim3(kThreads), (size_t)4 * scw * sizeof(float), ctx->stream, e0, e1, 0, q, nh, nh / kvh,
                          rp.pos0, m, kc, vc, cap, scaling, o, ml, scw);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return hip_err(ctx, e, "attention_tile_kernel launch");
    prof_commit(ctx, e0, e1, kProfAttn, 2.0 * kvh * (double)rp.vis_max * hd * 2.0 * m);
    return LBT_OK;
}

}  // namespace lbt
