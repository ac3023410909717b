// Batched prefill for gfx950: M prompt positions through one layer at a time.
//
// The reference has no batched path: its prompt phase is the per-token loop
// (model::generate runs P forwards, src/model/mod.rs:57-125; each forward is
// Qwen3::forward, src/model/qwen3.rs:139-191).  This file computes the same
// forward for M positions at once, with the linear layers as Q4_0
// dequant-GEMMs on the matrix cores (q4_gemm.hip) and causal attention as MFMA
// tiles.
//
// Attention must match the f32 per-token path, so no operand is rounded below
// what the reference computes with: K and V are f16 in the cache and enter f16
// MFMAs exactly; q and the softmax weights p are split into f16 hi + lo (22
// significant bits).  The MFMAs accumulate in f32.
//
// MFMA v_mfma_f32_16x16x32_f16 (attention): lane l holds A[l % 16][8 (l / 16)
// + j] and B[8 (l / 16) + j][l % 16] (j = 0..7) and receives
// D[4 (l / 16) + r][l % 16] (r = 0..3); any k order shared by A and B is
// valid.

#include <cmath>

#include "cw_internal.hpp"

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kT = 256;  // threads per workgroup (4 waves)

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off);
    return v;
}

// ---------------------------------------------------------------------------
// Per position: per-head QK RMSNorm (qwen3.rs:154-155) and NeoX RoPE
// (rope.wgsl:18-35) on the raw q|k|v rows of the QKV GEMM, q out as f32
// [M][n_heads][hd], k and v written into the cache rows start..start+M-1
// (cache.rs:21-24).  Workgroup (position, y) takes four heads of the
// position, one per wave.
// With S > 0 the rows are the QKV GEMM's S split-K partials, summed here in
// order (gemm_reduce_kernel's sum) instead of read from qkv.
template <typename KVT>
__global__ __launch_bounds__(kT) void qk_rope_kv_kernel(const float *__restrict__ qkv,
                                                        const float *__restrict__ qn,
                                                        const float *__restrict__ kn, float eps,
                                                        const float *__restrict__ cos_t,
                                                        const float *__restrict__ sin_t,
                                                        int n_heads, int n_kv, int start,
                                                        float *__restrict__ q_out,
                                                        KVT *__restrict__ kc,
                                                        KVT *__restrict__ vc,
                                                        const float *__restrict__ part, int S,
                                                        size_t MN) {
    constexpr int HD = 128, HALF = 64;
    const int i = blockIdx.x, pos = start + i;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int q_dim = n_heads * HD, kv_dim = n_kv * HD;
    const size_t row_off = (size_t)i * (q_dim + 2 * kv_dim);
    const float *row = (S > 0 ? part : qkv) + row_off;
    auto val = [&](const float *p) {  // p: an element of row (of partial 0)
        float v = *p;
        for (int s2 = 1; s2 < S; ++s2) v += p[(size_t)s2 * MN];
        return v;
    };
    const float c = cos_t[(size_t)pos * HALF + lane], s = sin_t[(size_t)pos * HALF + lane];
    // one head per wave: workgroup y takes heads 4 y .. 4 y + 3 of the row
    for (int h = blockIdx.y * (kT / 64) + wave; h < n_heads + n_kv; h += gridDim.y * (kT / 64)) {
        const bool isq = h < n_heads;
        const float *src = isq ? row + (size_t)h * HD : row + q_dim + (size_t)(h - n_heads) * HD;
        const float *g = isq ? qn : kn;
        const float lo = val(src + lane), hi = val(src + lane + HALF);
        const float ss = wave_sum(lo * lo + hi * hi);
        const float inv = 1.0f / sqrtf(ss / (float)HD + eps);
        const float l0 = (lo * inv) * g[lane], h0 = (hi * inv) * g[lane + HALF];
        const float r0 = l0 * c - h0 * s, r1 = h0 * c + l0 * s;
        if (isq) {
            float *dst = q_out + ((size_t)i * n_heads + h) * HD;
            dst[lane] = r0;
            dst[lane + HALF] = r1;
        } else {
            const int g2 = h - n_heads;
            KVT *kd = kc + (size_t)pos * kv_dim + (size_t)g2 * HD;
            kd[lane] = (KVT)r0;
            kd[lane + HALF] = (KVT)r1;
            const float *vs = row + q_dim + kv_dim + (size_t)g2 * HD;
            KVT *vd = vc + (size_t)pos * kv_dim + (size_t)g2 * HD;
            vd[lane] = (KVT)val(vs + lane);
            vd[lane + HALF] = (KVT)val(vs + lane + HALF);
        }
    }
}

// ---------------------------------------------------------------------------
// Causal attention (attention.wgsl:23-96 for each query position) on f16
// caches, flash style: workgroup = one query head x 64 positions, in two
// groups of four waves (one wave per 16 positions) that take alternate
// 64-key tiles, so the longest workgroup runs half as many tile steps.  Per
// tile: K and V rows staged in LDS as they are stored (16-byte writes);
// S = q K^T by MFMA (q split into f16 hi/lo), online max / sum per row,
// P (f16 hi/lo) through LDS into A layout, O += P V by MFMA with the V
// operand read by LDS transpose loads.  At the end the second group's
// (max, sum, o) per row merges into the first's through LDS.
constexpr int kAttQ = 64;   // positions per workgroup
constexpr int kAttK = 64;   // keys per tile
constexpr int kKRow = 128 + 8;  // K and V tile row stride (f16), padded

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

// B operand of v_mfma_f32_16x16x32_f16 (lane l: B[8 (l / 16) + j][l % 16],
// j = 0..7) from a row-major LDS tile, B[k][n] = tile[k0 + k][n0 + n].
// ds_read_b64_tr_b16: within each 16-lane group, lane i receives element
// i % 4 of the 8 bytes addressed by lane 4 j + i / 4, for j = 0..3.  So lane
// m of group g addresses row k0 + 8 g + m / 4 (+ 4 for the second read),
// columns n0 + 4 (m % 4) .. + 3, and lane i gets column n0 + i of rows
// k0 + 8 g + j.
__device__ __forceinline__ f16x8 lds_b_tr(const _Float16 *tile, int row_stride, int k0, int n0,
                                          int lane) {
    const int g = lane >> 4, m = lane & 15;
    const _Float16 *p = tile + (size_t)(k0 + 8 * g + (m >> 2)) * row_stride + n0 + 4 * (m & 3);
    const s16x4 r0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)p);
    const s16x4 r1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(p + 4 * row_stride));
    const uint2 a = __builtin_bit_cast(uint2, r0), b = __builtin_bit_cast(uint2, r1);
    return __builtin_bit_cast(f16x8, make_uint4(a.x, a.y, b.x, b.y));
}

__device__ __forceinline__ uint32_t pack_f16x2(float a, float b) {
    const uint32_t lo = __builtin_bit_cast(uint16_t, (_Float16)a);
    const uint32_t hi = __builtin_bit_cast(uint16_t, (_Float16)b);
    return lo | (hi << 16);
}

constexpr int kAttThreads = 2 * kT;  // two groups of four waves

__global__ __launch_bounds__(kAttThreads) void attn_prefill_kernel(
    const float *__restrict__ q, const _Float16 *__restrict__ kc, const _Float16 *__restrict__ vc,
    int M, int n_heads, int n_kv, int start, float scale, float *__restrict__ out) {
    constexpr int HD = 128;
    constexpr int TILE = kAttK * kKRow;  // f16 elements of one K (or V) tile
    // [group][K | V]; after the loop, group 1's (o, m, l) for the merge
    __shared__ __attribute__((aligned(16))) _Float16 KV[2][2][TILE];
    __shared__ float Ps[8][16 * kAttK];
    const int h = blockIdx.x, q0 = blockIdx.y * kAttQ;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = wave >> 2, gw = wave & 3, gtid = tid & (kT - 1);
    const int li = lane & 15, lg = lane >> 4;
    const int g = h / (n_heads / n_kv);
    const int kv_dim = n_kv * HD;
    const int wq = q0 + gw * 16;  // this wave's first position (row of q)
    _Float16 *Ks = KV[grp][0], *Vs = KV[grp][1];

    // q operands: row li of the wave's 16, dims 8 lg + 32 ks .. +8, hi and lo
    f16x8 qa[4][2];
    {
        const int qi = min(wq + li, M - 1);
        const float *qr = q + ((size_t)qi * n_heads + h) * HD;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            const float4 v0 = *reinterpret_cast<const float4 *>(qr + 32 * ks + 8 * lg);
            const float4 v1 = *reinterpret_cast<const float4 *>(qr + 32 * ks + 8 * lg + 4);
            const float v[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
            uint32_t ph[4], pl[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const _Float16 a0 = (_Float16)v[2 * j], a1 = (_Float16)v[2 * j + 1];
                ph[j] = (uint32_t)__builtin_bit_cast(uint16_t, a0) |
                        ((uint32_t)__builtin_bit_cast(uint16_t, a1) << 16);
                pl[j] = pack_f16x2(v[2 * j] - (float)a0, v[2 * j + 1] - (float)a1);
            }
            qa[ks][0] = __builtin_bit_cast(f16x8, make_uint4(ph[0], ph[1], ph[2], ph[3]));
            qa[ks][1] = __builtin_bit_cast(f16x8, make_uint4(pl[0], pl[1], pl[2], pl[3]));
        }
    }

    // rows of this lane in the C layout: 4 lg + r of the wave's 16
    float mrow[4], lrow[4];
    f32x4 o[8];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        mrow[r] = -INFINITY;
        lrow[r] = 0.0f;
    }
#pragma unroll
    for (int ni = 0; ni < 8; ++ni) o[ni] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int last_pos = start + min(q0 + kAttQ, M) - 1;  // last key any row needs
    const int n_tiles = last_pos / kAttK + 1;
    const int n_steps = (n_tiles + 1) / 2;  // group grp takes tiles grp, grp + 2, ...
    // K and V rows of key tile t, 64 keys x 128 dims, 16 B per load (4 each
    // per thread of the group); the group's next tile's loads are in flight
    // during this tile's MFMAs (past the last tile a clamped re-load, unused)
    u32x4 kn[4], vn[4];
    auto tile_load = [&](int t) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int f = gtid + u * kT;  // 0..1023
            const int key = f >> 4, c8 = (f & 15) * 8;
            const int p = min(t * kAttK + key, last_pos);
            kn[u] = *reinterpret_cast<const u32x4 *>(kc + (size_t)p * kv_dim + g * HD + c8);
            vn[u] = *reinterpret_cast<const u32x4 *>(vc + (size_t)p * kv_dim + g * HD + c8);
        }
    };
    tile_load(min(grp, n_tiles - 1));
    for (int st = 0; st < n_steps; ++st) {
        const int t = 2 * st + grp;
        const bool active = t < n_tiles;  // (uniform over the group)
        const int k0 = t * kAttK;
        __syncthreads();  // previous step's LDS reads are done
        // stage K and V rows
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int f = gtid + u * kT;
            const int key = f >> 4, c8 = (f & 15) * 8;
            *reinterpret_cast<u32x4 *>(&Ks[key * kKRow + c8]) = kn[u];
            *reinterpret_cast<u32x4 *>(&Vs[key * kKRow + c8]) = vn[u];
        }
        tile_load(min(t + 2, n_tiles - 1));
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        if (!active) continue;

        // S (16 rows x 64 keys): 4 key tiles of 16, K = 128 dims in 4 steps
        f32x4 sc[4];
#pragma unroll
        for (int ni = 0; ni < 4; ++ni) {
            f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
                const f16x8 kb = *reinterpret_cast<const f16x8 *>(
                    &Ks[(ni * 16 + li) * kKRow + 32 * ks + 8 * lg]);
                acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(qa[ks][0], kb, acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(qa[ks][1], kb, acc, 0, 0, 0);
            }
            sc[ni] = acc;
        }
        // mask (causal, and rows past M), scale, online softmax per row
        float pm[4][4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row_pos = start + wq + 4 * lg + r;
            float mx = -INFINITY;
#pragma unroll
            for (int ni = 0; ni < 4; ++ni) {
                const int key = k0 + ni * 16 + li;
                const float v = key <= row_pos ? sc[ni][r] * scale : -INFINITY;
                pm[ni][r] = v;
                mx = fmaxf(mx, v);
            }
            // max over the 16 lanes that share this row (same lg)
#pragma unroll
            for (int off = 8; off >= 1; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
            const float mnew = fmaxf(mrow[r], mx);
            // a row with no key yet keeps mnew = -inf: guard the rescale
            const float alpha = mnew == -INFINITY ? 1.0f : expf(mrow[r] - mnew);
            float ls = 0.0f;
#pragma unroll
            for (int ni = 0; ni < 4; ++ni) {
                const float p = pm[ni][r] == -INFINITY ? 0.0f : expf(pm[ni][r] - mnew);
                pm[ni][r] = p;
                ls += p;
            }
#pragma unroll
            for (int off = 8; off >= 1; off >>= 1) ls += __shfl_xor(ls, off);
            lrow[r] = lrow[r] * alpha + ls;
            mrow[r] = mnew;
#pragma unroll
            for (int ni = 0; ni < 8; ++ni) o[ni][r] *= alpha;
        }
        // P to LDS (row-major 16 x 64), back in A layout as f16 hi/lo
        float *P = Ps[wave];
#pragma unroll
        for (int ni = 0; ni < 4; ++ni)
#pragma unroll
            for (int r = 0; r < 4; ++r) P[(4 * lg + r) * kAttK + ni * 16 + li] = pm[ni][r];
        // (a wave's LDS accesses complete in order: its reads below see these writes)
        f16x8 pa[2][2];
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            const float *pr = P + li * kAttK + 32 * kk + 8 * lg;
            uint32_t ph[4], pl[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float v0 = pr[2 * j], v1 = pr[2 * j + 1];
                const _Float16 a0 = (_Float16)v0, a1 = (_Float16)v1;
                ph[j] = (uint32_t)__builtin_bit_cast(uint16_t, a0) |
                        ((uint32_t)__builtin_bit_cast(uint16_t, a1) << 16);
                pl[j] = pack_f16x2(v0 - (float)a0, v1 - (float)a1);
            }
            pa[kk][0] = __builtin_bit_cast(f16x8, make_uint4(ph[0], ph[1], ph[2], ph[3]));
            pa[kk][1] = __builtin_bit_cast(f16x8, make_uint4(pl[0], pl[1], pl[2], pl[3]));
        }
        // O (16 rows x 128 dims) += P (16 x 64 keys) V (64 keys x 128 dims)
#pragma unroll
        for (int ni = 0; ni < 8; ++ni) {
#pragma unroll
            for (int kk = 0; kk < 2; ++kk) {
                const f16x8 vb = lds_b_tr(Vs, kKRow, 32 * kk, ni * 16, lane);
                o[ni] = __builtin_amdgcn_mfma_f32_16x16x32_f16(pa[kk][0], vb, o[ni], 0, 0, 0);
                o[ni] = __builtin_amdgcn_mfma_f32_16x16x32_f16(pa[kk][1], vb, o[ni], 0, 0, 0);
            }
        }
    }

    // merge: group 1's (o, m, l) of each row through LDS into group 0's
    // (rescaled to the common max), then normalise and store.  Lane holds
    // rows 4 lg + r, dims ni * 16 + li.
    __syncthreads();  // every group is done with its K / V tile
    float *mo = reinterpret_cast<float *>(&KV[0][0][0]);  // [4 waves][16 rows][128]
    float *mml = mo + 4 * 16 * HD;                        // [4 waves][16 rows][2]
    if (grp == 1) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = 4 * lg + r;
#pragma unroll
            for (int ni = 0; ni < 8; ++ni) mo[(gw * 16 + row) * HD + ni * 16 + li] = o[ni][r];
            if (li == 0) {
                mml[(gw * 16 + row) * 2] = mrow[r];
                mml[(gw * 16 + row) * 2 + 1] = lrow[r];
            }
        }
    }
    __syncthreads();
    if (grp == 0) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = 4 * lg + r;
            const int qi = wq + row;
            const float m1 = mml[(gw * 16 + row) * 2], l1 = mml[(gw * 16 + row) * 2 + 1];
            const float mm = fmaxf(mrow[r], m1);
            const float f0 = mrow[r] == -INFINITY ? 0.0f : expf(mrow[r] - mm);
            const float f1 = m1 == -INFINITY ? 0.0f : expf(m1 - mm);
            const float inv = 1.0f / (lrow[r] * f0 + l1 * f1);
            if (qi < M) {
                float *dst = out + (size_t)qi * n_heads * HD + (size_t)h * HD;
#pragma unroll
                for (int ni = 0; ni < 8; ++ni)
                    dst[ni * 16 + li] =
                        (o[ni][r] * f0 + mo[(gw * 16 + row) * HD + ni * 16 + li] * f1) * inv;
            }
        }
    }
}

// Embedding rows of n tokens (Qwen3::embed, qwen3.rs:128-133): one workgroup
// per position.
__global__ __launch_bounds__(kT) void embed_rows_kernel(const float *__restrict__ table, int dim,
                                                        const uint32_t *__restrict__ tok,
                                                        float *__restrict__ out) {
    const size_t src = (size_t)tok[blockIdx.x] * dim, dst = (size_t)blockIdx.x * dim;
    for (int i = threadIdx.x; i < dim; i += kT) out[dst + i] = table[src + i];
}

}  // namespace

namespace cwi {

int launch_embed_rows(cw_ctx *ctx, const float *table, int dim, const uint32_t *tok_dev, int n,
                      float *out) {
    return launch(ctx, "prefill_embed", embed_rows_kernel, dim3(n), dim3(kT), 0, table, dim,
                  tok_dev, out);
}

int launch_qk_rope_kv(cw_ctx *ctx, const float *qkv, const float *qn, const float *kn, float eps,
                      const float *cos_t, const float *sin_t, int M, int n_heads, int n_kv,
                      int start, int kv_dtype, float *q_out, void *kc, void *vc, const float *part,
                      int splits) {
    const size_t mn = (size_t)M * (n_heads + 2 * n_kv) * 128;
    const int S = part ? splits : 0;
    const dim3 grid(M, (n_heads + n_kv + kT / 64 - 1) / (kT / 64));
    if (kv_dtype == CW_F16)
        return launch(ctx, "prefill_qk_rope_kv", qk_rope_kv_kernel<_Float16>, grid, dim3(kT), 0,
                      qkv, qn, kn, eps, cos_t, sin_t, n_heads, n_kv, start, q_out, (_Float16 *)kc,
                      (_Float16 *)vc, part, S, mn);
    return launch(ctx, "prefill_qk_rope_kv", qk_rope_kv_kernel<float>, grid, dim3(kT), 0, qkv,
                  qn, kn, eps, cos_t, sin_t, n_heads, n_kv, start, q_out, (float *)kc, (float *)vc,
                  part, S, mn);
}

int launch_attn_prefill(cw_ctx *ctx, const float *q, const void *kc, const void *vc, int M,
                        int n_heads, int n_kv, int start, float *out) {
    const float scale = 1.0f / sqrtf(128.0f);
    return launch(ctx, "prefill_attention", attn_prefill_kernel,
                  dim3(n_heads, (M + kAttQ - 1) / kAttQ), dim3(kAttThreads), 0, q,
                  (const _Float16 *)kc, (const _Float16 *)vc, M, n_heads, n_kv, start, scale, out);
}

}  // namespace cwi
