// Batched prefill for gfx950: M prompt positions through one layer at a time.
//
// The reference has no batched path: its prompt phase is the per-token loop
// (model::generate runs P forwards, src/model/mod.rs:57-125; each forward is
// Qwen3::forward, src/model/qwen3.rs:139-191).  This file computes the same
// forward for M positions at once, with the linear layers as Q4_0
// dequant-GEMMs on the matrix cores (q4_gemm.hip) and causal attention as MFMA
// tiles.
//
// Attention must match the f32 per-token path, so q and the softmax weights go
// through the matrix cores as two f16 or as f32 (details at the kernel).

#include <cmath>

#include "prompt_device.hpp"

namespace {

using namespace cwi;

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
    // elements p[lane] and p[lane + 64] of row (of partial 0)
    auto val = [&](const float *p) {
        return sum_parts(max(S, 1), [&](int s2) {
            const float *q = p + (size_t)s2 * MN + lane;
            return make_float2(q[0], q[HALF]);
        });
    };
    const float c = cos_t[(size_t)pos * HALF + lane], s = sin_t[(size_t)pos * HALF + lane];
    // one head per wave: workgroup y takes heads 4 y .. 4 y + 3 of the row
    for (int h = blockIdx.y * (kT / 64) + wave; h < n_heads + n_kv; h += gridDim.y * (kT / 64)) {
        const bool isq = h < n_heads;
        const float *src = isq ? row + (size_t)h * HD : row + q_dim + (size_t)(h - n_heads) * HD;
        const float *g = isq ? qn : kn;
        const float2 x = val(src);
        const float lo = x.x, hi = x.y;
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
            const float2 v = val(vs);
            vd[lane] = (KVT)v.x;
            vd[lane + HALF] = (KVT)v.y;
        }
    }
}

// ---------------------------------------------------------------------------
// Causal attention of M positions (attention.wgsl:23-96 for each) over the
// cache, flash style.  A workgroup takes one kv head and four waves of query
// rows: a wave is one query head and QT tiles of 16 positions; the waves are
// up to four heads of the kv head, then further positions, so that every K / V
// tile in LDS serves all of them.  It walks key tiles of KT positions, two
// tiles in LDS (the next one's global -> LDS DMAs in flight), with online
// max / sum per row.
//
// Transposed products keep the softmax in registers: S^T = K q^T leaves lane
// (g = l / 16, i = l % 16) the keys 4 g + r of query i, which is the B operand
// of O^T = V^T P^T when the MFMA's k slots are taken in that order (any order
// shared by A and B is valid).  So P never goes through LDS, and a row's
// scale is one value per lane.
//  * f16 cache: v_mfma_f32_16x16x32_f16, K and V as stored, q and P split into
//    f16 hi + lo: 22 significant bits of what is at least 2^-3 (hi is 2^-3 or
//    more, lo's last place is 2^-24), steps of 2^-24 below.  P is scaled by
//    2^15, so weights down to 2^-18 of the largest keep 22 bits (unscaled, one
//    12 nats below it kept seven: logits 2-4e-3 off behind such a key); q is
//    RMS-normalised times a gain, as the decode kernel splits it.  V^T by LDS
//    transpose loads.
//  * f32 cache: v_mfma_f32_16x16x4_f32 (lane l: A[l % 16][l / 16],
//    B[l / 16][l % 16]), every operand f32.
//
// Key chunks: a workgroup takes `ct` key tiles of its rows' range, so that few
// rows against many keys, and the long rows of a causal prompt, still spread
// over the chip.  With more than one chunk it leaves (max, sum, o) partials,
// which the pass that reads the rows merges (q4_gemm.hip).
//
// Bound by the softmax's vector work and waits beside short MFMA runs (512
// positions: matrix cores busy 7 %, waves waiting 39 % of their time), so the
// layout aims at fewer K / V reads and LDS trips.  One head per workgroup with P
// through LDS took, per layer of 32 heads over 8: 24 positions behind 700
// 29.2 us, 512 from 0 23.5, 3000 from 0 401; this form 10, 20 and 171, and the
// merge 4.6, 8.7 and 28.
template <typename KVT, int QT_>
struct AP {
    static constexpr int QT = QT_, HD = 128, ES = (int)sizeof(KVT);
    static constexpr int KT = 128 / ES;        // keys per tile: 16 KB of K
    static constexpr int ROWB = HD * ES;       // bytes of a cache row slice
    static constexpr int CPR = ROWB / 16;      // 16-byte chunks per row
    static constexpr int TILE = KT * ROWB;     // bytes of one K (or V) tile
    static constexpr int UNITS = TILE / 1024;  // 64-lane DMAs of one tile
    static constexpr int ST = KT / 16;         // score tiles of 16 keys
    // weights carry 2^UP (which cancels in o / sum), so that small ones keep
    // their bits as f16: the largest is 2^15, and f16 ends at 2^16 and 2^-24
    static constexpr float UP = ES == 2 ? 15.0f : 0.0f;
};

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
__device__ __forceinline__ f16x8 pack_f16x8(const float (&v)[8]) {
    uint32_t p[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
        p[j] = (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)v[2 * j]) |
               (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)v[2 * j + 1]) << 16;
    return __builtin_bit_cast(f16x8, make_uint4(p[0], p[1], p[2], p[3]));
}

// v = hi + lo in f16
__device__ __forceinline__ void split_f16x8(float (&v)[8], f16x8 &hi, f16x8 &lo) {
    hi = pack_f16x8(v);
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] -= (float)hi[j];
    lo = pack_f16x8(v);
}

template <typename KVT, int QT, bool PART>
__global__ __launch_bounds__(kT, 2) void attn_prefill_kernel(cwi::AttnPrefillArgs a) {
    using C = AP<KVT, QT>;
    constexpr int HD = C::HD, KT = C::KT, ST = C::ST;
    constexpr bool F16 = C::ES == 2;
    __shared__ __attribute__((aligned(1024))) unsigned char lds[2][2 * C::TILE];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, lg = lane >> 4;
    const int hpk = a.n_heads / a.n_kv, hw = hpk < 4 ? hpk : 4;  // heads per workgroup
    const int h = blockIdx.x * hw + wave % hw, g = h / hpk;
    // the longest rows first
    const int qt = gridDim.y - 1 - blockIdx.y;
    const int pt = QT * 16 * (4 / hw);  // positions per workgroup
    const int q0 = qt * pt, wq = q0 + wave / hw * (QT * 16);
    const int last_pos = a.start + min(q0 + pt, a.M) - 1;  // last key any row needs
    const int t0 = blockIdx.z * a.ct, t1 = min(t0 + a.ct, last_pos / KT + 1);
    if (t0 >= t1) return;
    // the last key of this wave's rows (none: rows past M)
    const int w_last = wq < a.M ? a.start + min(wq + QT * 16, a.M) - 1 : -1;

    const size_t row_b = (size_t)a.n_kv * C::ROWB;
    const char *const kc = static_cast<const char *>(a.kc) + (size_t)g * C::ROWB;
    const char *const vc = static_cast<const char *>(a.vc) + (size_t)g * C::ROWB;
    // Tile t's DMAs: chunk c of row r goes to slot c ^ (r % 16) of its row, so
    // that both kinds of fragment reads spread over all banks; rows past the
    // last key re-read it.
    auto load_tile = [&](int t, unsigned char *buf) {
        const size_t base = (size_t)t * KT * row_b;
#pragma unroll
        for (int p = 0; p < C::UNITS / 4; ++p) {
            const int u = wave + p * 4;
            const int r = u * (64 / C::CPR) + lane / C::CPR;
            const int c = (lane % C::CPR) ^ (r & 15);
            const uint32_t off = (uint32_t)min(r, last_pos - t * KT) * (uint32_t)row_b + c * 16;
            dma16(kc + base, off, buf + u * 1024);
            dma16(vc + base, off, buf + C::TILE + u * 1024);
        }
    };
    load_tile(t0, lds[0]);

    // q operands of this lane's queries (B: query li, dims in the k order of
    // the K fragments)
    f16x8 qh[F16 ? QT : 1][4], ql[F16 ? QT : 1][4];
    f32x4 qf[F16 ? 1 : QT][8];
#pragma unroll
    for (int i = 0; i < QT; ++i) {
        const float *qr = a.q + ((size_t)min(wq + i * 16 + li, a.M - 1) * a.n_heads + h) * HD;
        if constexpr (F16) {
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
                const float4 v0 = *reinterpret_cast<const float4 *>(qr + 32 * ks + 8 * lg);
                const float4 v1 = *reinterpret_cast<const float4 *>(qr + 32 * ks + 8 * lg + 4);
                float v[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
                split_f16x8(v, qh[i][ks], ql[i][ks]);
            }
        } else {
#pragma unroll
            for (int u = 0; u < 8; ++u)
                qf[i][u] = *reinterpret_cast<const f32x4 *>(qr + 16 * u + 4 * lg);
        }
    }

    f32x4 o[QT][8];  // O^T: dims 16 d + 4 lg + r of query li
    float mrow[QT], lsum[QT];  // running max (times log2 e); this lane's part of the sum
#pragma unroll
    for (int i = 0; i < QT; ++i) {
        mrow[i] = -INFINITY;
        lsum[i] = 0.0f;
#pragma unroll
        for (int d = 0; d < 8; ++d) o[i][d] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    // fragment addresses within a tile; other k steps (dims) by xor, other
    // rows by a constant
    const int ka = li * C::ROWB + ((lg ^ li) << 4);
    const int va = F16 ? (4 * lg + (li >> 2)) * C::ROWB +
                             ((((li & 3) >> 1) ^ (4 * lg + (li >> 2))) << 4) + (li & 1) * 8
                       : 0;

    for (int t = t0; t < t1; ++t) {
        unsigned char *const buf = lds[(t - t0) & 1];
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's part of tile t has landed
        __builtin_amdgcn_sched_barrier(0);
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
        __builtin_amdgcn_s_barrier();        // tile t published; the other buffer is free
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        if (t + 1 < t1) load_tile(t + 1, lds[(t - t0 + 1) & 1]);
        const int k0 = t * KT;
        if (k0 > w_last) continue;  // (wave-uniform) every key is past this wave's rows
        const unsigned char *const Ks = buf, *const Vs = buf + C::TILE;

        f32x4 s[QT][ST];
#pragma unroll
        for (int kt = 0; kt < ST; ++kt) {
#pragma unroll
            for (int i = 0; i < QT; ++i) s[i][kt] = f32x4{0.f, 0.f, 0.f, 0.f};
            if constexpr (F16) {
#pragma unroll
                for (int ks = 0; ks < 4; ++ks) {
                    const f16x8 kf = *reinterpret_cast<const f16x8 *>(
                        Ks + ((ka ^ (ks << 6)) + kt * 16 * C::ROWB));
#pragma unroll
                    for (int i = 0; i < QT; ++i)
                        s[i][kt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, qh[i][ks], s[i][kt],
                                                                          0, 0, 0);
#pragma unroll
                    for (int i = 0; i < QT; ++i)
                        s[i][kt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, ql[i][ks], s[i][kt],
                                                                          0, 0, 0);
                }
            } else {
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const f32x4 kf = *reinterpret_cast<const f32x4 *>(
                        Ks + ((ka ^ (u << 6)) + kt * 16 * C::ROWB));
#pragma unroll
                    for (int r = 0; r < 4; ++r)
#pragma unroll
                        for (int i = 0; i < QT; ++i)
                            s[i][kt] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[r], qf[i][u][r],
                                                                            s[i][kt], 0, 0, 0);
                }
            }
        }
        // online softmax of each query; keys past its position only in tiles
        // that reach beyond the wave's first row
        float alpha[QT];
        bool grew = false;
#pragma unroll
        for (int i = 0; i < QT; ++i) {
            const int lim = a.start + wq + i * 16 + li - k0 - 4 * lg;  // last key: 16 kt + r
            if (k0 + KT - 1 > a.start + wq + i * 16) {
#pragma unroll
                for (int kt = 0; kt < ST; ++kt)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        s[i][kt][r] = kt * 16 + r <= lim ? s[i][kt][r] : -INFINITY;
            }
            float mx = s[i][0][0];
#pragma unroll
            for (int kt = 0; kt < ST; ++kt)
#pragma unroll
                for (int r = 0; r < 4; ++r) mx = fmaxf(mx, s[i][kt][r]);
            mx = fmaxf(mx, __shfl_xor(mx, 16));
            mx = fmaxf(mx, __shfl_xor(mx, 32));
            const float mnew = fmaxf(mrow[i], mx * a.scale);
            // p = 2^(s scale log2(e) - max + UP); a query with no key yet keeps
            // max -inf: its terms are 2^-inf = 0
            const float ref = mnew == -INFINITY ? 0.0f : mnew;
            alpha[i] = __builtin_amdgcn_exp2f(mrow[i] - ref);
            grew |= mnew > mrow[i];
            mrow[i] = mnew;
            float ls = 0.0f;
#pragma unroll
            for (int kt = 0; kt < ST; ++kt)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float p =
                        __builtin_amdgcn_exp2f(__builtin_fmaf(s[i][kt][r], a.scale, C::UP - ref));
                    s[i][kt][r] = p;
                    ls += p;
                }
            lsum[i] = lsum[i] * alpha[i] + ls;
        }
        if (__any(grew)) {
#pragma unroll
            for (int i = 0; i < QT; ++i)
#pragma unroll
                for (int d = 0; d < 8; ++d)
#pragma unroll
                    for (int r = 0; r < 4; ++r) o[i][d][r] *= alpha[i];
        }
        if constexpr (F16) {
#pragma unroll
            for (int kk = 0; kk < ST / 2; ++kk) {
                f16x8 ph[QT], pl[QT];
#pragma unroll
                for (int i = 0; i < QT; ++i) {
                    float v[8];
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        v[r] = s[i][2 * kk][r];
                        v[4 + r] = s[i][2 * kk + 1][r];
                    }
                    split_f16x8(v, ph[i], pl[i]);
                }
#pragma unroll
                for (int d = 0; d < 8; ++d) {
                    // ds_read_b64_tr_b16: within each 16-lane group, lane i
                    // receives element i % 4 of the 8 bytes addressed by lane
                    // 4 j + i / 4, for j = 0..3: dim 16 d + i of keys 4 lg + j
                    const unsigned char *p = Vs + ((va ^ (d << 5)) + kk * 32 * C::ROWB);
                    const uint2 r0 = __builtin_bit_cast(
                        uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)p));
                    const uint2 r1 = __builtin_bit_cast(
                        uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                   (lds_s16x4 *)(p + 16 * C::ROWB)));
                    const f16x8 vf =
                        __builtin_bit_cast(f16x8, make_uint4(r0.x, r0.y, r1.x, r1.y));
#pragma unroll
                    for (int i = 0; i < QT; ++i)
                        o[i][d] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, ph[i], o[i][d], 0, 0, 0);
#pragma unroll
                    for (int i = 0; i < QT; ++i)
                        o[i][d] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, pl[i], o[i][d], 0, 0, 0);
                }
            }
        } else {
#pragma unroll
            for (int kt = 0; kt < ST; ++kt)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int row = 4 * lg + r;
                    const int vb = row * C::ROWB + (((li >> 2) ^ row) << 4) + (li & 3) * 4;
#pragma unroll
                    for (int d = 0; d < 8; ++d) {
                        const float vf = *reinterpret_cast<const float *>(
                            Vs + ((vb ^ (d << 6)) + kt * 16 * C::ROWB));
#pragma unroll
                        for (int i = 0; i < QT; ++i)
                            o[i][d] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf, s[i][kt][r], o[i][d],
                                                                           0, 0, 0);
                    }
                }
        }
    }

#pragma unroll
    for (int i = 0; i < QT; ++i) {
        float l = lsum[i];
        l += __shfl_xor(l, 16);
        l += __shfl_xor(l, 32);
        const int qi = wq + i * 16 + li;
        if (qi >= a.M) continue;
        const size_t row = (size_t)qi * a.n_heads + h;
        const size_t prow = (size_t)blockIdx.z * a.M * a.n_heads + row;
        float *dst = PART ? a.part + prow * HD : a.out + row * HD;
        const float f = PART ? 1.0f : 1.0f / l;
#pragma unroll
        for (int d = 0; d < 8; ++d)
            *reinterpret_cast<float4 *>(dst + 16 * d + 4 * lg) =
                make_float4(o[i][d][0] * f, o[i][d][1] * f, o[i][d][2] * f, o[i][d][3] * f);
        if (PART && lg == 0)
            *reinterpret_cast<float2 *>(a.ml + prow * 2) = make_float2(mrow[i], l);
    }
}

}  // namespace

namespace cwi {

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

// Positions per workgroup of one query tile, and the tiles of keys per
// workgroup: the share of all (query tile, key tile) steps that two
// workgroups per CU take, so no workgroup runs longer than that.  `rows`: the
// most (chunk, position) partials there is room for.
AttnPrefillPlan attn_prefill_plan(const cw_ctx *ctx, int kv_dtype, int M, int n_heads, int n_kv,
                                  int start, size_t rows) {
    const int hpk = n_heads / n_kv, hw = std::min(hpk, 4);
    AttnPrefillPlan p{};
    // two query tiles per wave read each K / V fragment once for both; one
    // when the rows fill no more, and for f32, whose MFMAs outweigh the reads
    // (and whose second tile would not fit the registers)
    p.qt = M <= 16 * (4 / hw) || kv_dtype != CW_F16 ? 1 : 2;
    p.pt = p.qt * 16 * (4 / hw);
    p.kt = kv_dtype == CW_F16 ? AP<_Float16, 1>::KT : AP<float, 1>::KT;
    p.groups = n_heads / hw;
    p.q_tiles = (M + p.pt - 1) / p.pt;
    long steps = 0;
    for (int t = 0; t < p.q_tiles; ++t)
        steps += (start + std::min((t + 1) * p.pt, M) - 1) / p.kt + 1;
    const int tiles = (start + M - 1) / p.kt + 1;
    const long slots = 2L * ctx->n_cu;
    p.ct = (int)((steps * p.groups + slots - 1) / slots);
    p.chunks = (tiles + p.ct - 1) / p.ct;
    if ((size_t)p.chunks * M > rows) {
        p.chunks = (int)std::max<size_t>(1, rows / M);
        p.ct = (tiles + p.chunks - 1) / p.chunks;
        p.chunks = (tiles + p.ct - 1) / p.ct;
    }
    return p;
}

size_t attn_prefill_rows(const cw_ctx *ctx, int M, int n_heads, int n_kv) {
    // chunks <= 2 slots / (groups q_tiles) + 1 (a causal row range is at least
    // half of the longest), and q_tiles >= M / pt
    const int hw = std::min(n_heads / n_kv, 4), groups = n_heads / hw;
    return (size_t)M + (size_t)4 * ctx->n_cu * 32 * (4 / hw) / groups + 1;
}

int launch_attn_prefill(cw_ctx *ctx, const AttnPrefillPlan &p, AttnPrefillArgs a, int kv_dtype) {
    // p = 2^(s scale log2(e) - max)
    a.scale = (float)(1.4426950408889634 / sqrt(128.0));
    a.ct = p.ct;
    const dim3 grid(p.groups, p.q_tiles, p.chunks);
    auto go = [&](auto fn) { return launch(ctx, "prefill_attention", fn, grid, dim3(kT), 0, a); };
    const bool part = p.chunks > 1;
    if (kv_dtype == CW_F16) {
        if (p.qt == 1)
            return part ? go(attn_prefill_kernel<_Float16, 1, true>)
                        : go(attn_prefill_kernel<_Float16, 1, false>);
        return part ? go(attn_prefill_kernel<_Float16, 2, true>)
                    : go(attn_prefill_kernel<_Float16, 2, false>);
    }
    return part ? go(attn_prefill_kernel<float, 1, true>)
                : go(attn_prefill_kernel<float, 1, false>);
}

}  // namespace cwi
