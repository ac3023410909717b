// Q4_0 dequant-GEMM for gfx950: y[M][N] = x[M][K] . W[N][K]^T for several
// activation rows at once (W split GGUF Q4_0), with the passes that prepare
// its operand and add its K splits.
//
// The reference has no batched path: its prompt phase is the per-token loop
// (src/model/mod.rs:57-125) over q4::gemv (src/kernels/q4.rs:9-30,
// q4.wgsl:25-82).  Every row here equals that GEMV with the rounding of an
// f32 computation.
//
// Operands, all exact:
//  * x: per row m a power of two 2^e brings max|x| into [2^10, 2^11), then
//    x 2^-e = x_hi + x_lo with x_hi = f16(.) and x_lo = f16(remainder): 22
//    significant bits.
//  * W: a nibble q masked out of its packed word and put under 0x6400 is the
//    f16 1024 + q (low nibbles) or 1024 + 16 q (high nibbles); one packed
//    subtraction leaves q - 8 or 16 (q - 8), exact.  A word of 8 weights is a
//    B fragment in nine instructions.  The elements under low nibbles carry 16
//    times their x (below 2^15), so every product has the factor 16.  (The
//    masked nibble alone is q as an f16 subnormal, with no or and no
//    subtraction, but the matrix cores align products by their nominal
//    exponents: 1.6e-5 relative error in y where this form has 1.0-1.4e-7.)
// Per block b: t = sum over its 32 k of (x_hi + x_lo) (q - 8), two MFMAs into
// a fresh f32 accumulator, then acc += d_b t, one f32 FMA per output element
// and block; every kChain blocks acc is added to a second sum and starts again
// (the kernel's comment); y = 2^(e - 4) of that sum.
//
// MFMA v_mfma_f32_16x16x32_f16: lane l holds A[l % 16][8 (l / 16) + j] and
// B[8 (l / 16) + j][l % 16] (j = 0..7) and receives D[4 (l / 16) + r][l % 16]
// (r = 0..3); any k order shared by A and B is valid.  Its 32 k are one Q4
// block: lane group g = l / 16 takes bytes 4 g .. 4 g + 3 of the block, whose
// masks yield the elements in the order kept by the x image (chunk order
// below).

#include <cmath>

#include "prompt_device.hpp"

namespace {

using namespace cwi;

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr float kUnscale = 0.0625f;  // the products' factor 16
constexpr int kChain = 16;           // blocks per chain of f32 sums (a multiple of every stage)

// ---------------------------------------------------------------------------
// The x image: per 16 rows and block 1 KB of x_hi, then 1 KB of x_lo, each as
// the MFMA's lanes take it: lane 16 g + r has the 16-byte chunk
//   e0 e2 f0 f2 e1 e3 f1 f3   (e_i = 16 x[4 g + i], f_i = x[16 + 4 g + i])
// of row r, the order in which the masks of a packed word yield the weights.  So
// a fragment is 1 KB of consecutive bytes, in memory as in LDS, and one DMA (as
// 128 bytes per row and block, whose DMAs touch 16 places: 512 rows of 4096 ->
// 6144 73.7 instead of 63.9 us).
// rowscale[row] = 2^e.
//
// One workgroup per row, or per (row, segment of the columns) with a row scale
// for each: where the consumer splits K by the same segments, few long rows
// still give every CU a workgroup (the SwiGLU pass of 24 rows of 12288: 15.6
// us as 24 workgroups, 5.0 so).  RMSNorm needs whole rows.  A thread takes whole
// chunks (8 elements), CH of them in registers.  Sources of a row: SRC_ROWS, x itself; SRC_PART, the sum in
// order of S split-K partials (+ resid), also written to y; SRC_SWIGLU,
// silu(g) u of the summed partials of the gate and the up product; SRC_EMBED,
// a token's embedding row (Qwen3::embed, qwen3.rs:128-133), also written to y;
// SRC_ATTN, the attention chunks of a position merged.  NORM: RMSNorm first
// (norm.wgsl:20-42).
enum SplitSrc { SRC_ROWS, SRC_PART, SRC_SWIGLU, SRC_EMBED, SRC_ATTN };

struct SplitArgs {
    const float *x;       // [M][K], the partials [S][M][K] ([S][2][M][K]), the table
    int S;
    size_t MK;            // elements of one [M][K] matrix
    const float *resid;   // SRC_PART, optional: [M][K]
    float *y;             // SRC_PART, SRC_EMBED: [M][K]
    const uint32_t *tok;  // SRC_EMBED
    const float *ml;      // SRC_ATTN: (max log2 e, sum) [S][M][K / 128]
    int start, pt, span;  // SRC_ATTN: first position, positions that share their
                          // chunks, positions per chunk
    int M;                // rows
    const float *norm_w;  // NORM: gain [K]
    float eps;
    int K;
    int seg, segs;  // chunks per segment, segments
    uint16_t *img;
    float *rowscale;
    cwi::ScalePad pad;  // copied by the workgroups past the segments
};

__device__ __forceinline__ float4 sum4(const float *p, int S, size_t stride) {
    return sum_parts(S, [&](int s) {
        return *reinterpret_cast<const float4 *>(p + (size_t)s * stride);
    });
}

__device__ __forceinline__ float silu_mul(float g, float u) { return g / (1.0f + expf(-g)) * u; }

// Scales whose rows are not whole groups of eight blocks (or whose address is
// not a multiple of 16), copied to rows that are: the GEMM loads them a group
// (16 bytes) at a time.  A part of the pass that makes the x image, as
// workgroups of their own (a launch of its own before: 4 rows of 288 -> 512 14.0
// us in all, 8.8-10.4 so).
__device__ __forceinline__ void copy_scales(const cwi::ScalePad &p, size_t at, size_t step) {
    const int ns = (p.nb + 7) / 8 * 8;
    const size_t total = (size_t)p.N * ns;
    for (int m = 0; m < p.mats; ++m)
        for (size_t i = at; i < total; i += step) {
            const size_t n = i / ns;
            const int b = (int)(i - n * ns);
            p.dst[m * total + i] = p.src[m][n * p.nb + min(b, p.nb - 1)];
        }
}

// With R = 4 a workgroup takes four rows, neighbouring lanes the same chunk of
// each, so a store covers 64 bytes of an image line instead of 16 (3000 rows of
// 12288: 58 us; 80 with one row, 141 with one row and in plain row order).
// PAD: the launch has workgroups that copy scales (a variant, since the test in
// front of the loads costs the others 0.2 us).
template <bool NORM, int SRC, int CH, int R, bool PAD>
__global__ __launch_bounds__(R == 1 ? 512 : 1024) void split_image_kernel(SplitArgs a) {
    __shared__ float red[2][R == 1 ? 8 : 16][R];
    if constexpr (PAD) {
        if ((int)blockIdx.y >= a.segs) {
            const size_t wg = (size_t)(blockIdx.y - a.segs) * gridDim.x + blockIdx.x;
            copy_scales(a.pad, wg * blockDim.x + threadIdx.x,
                        (size_t)(gridDim.y - a.segs) * gridDim.x * blockDim.x);
            return;
        }
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // this thread's row of the workgroup's, and its place among that row's threads
    const int ri = threadIdx.x % R, tid = threadIdx.x / R, nt = blockDim.x / R;
    // the segment's chunks [c0, nch)
    const int c0 = blockIdx.y * a.seg, nch = min(a.K >> 3, c0 + a.seg);
    // workgroups go round-robin over the 8 XCDs: within 128 rows each XCD takes
    // the 16 that share their image lines, which then meet in its L2
    const int at = blockIdx.x * R, in = (at & 127) / R;
    const int row0 = (at | 127) < a.M ? (at & ~127) + (in & 7) * 16 + (in >> 3) * R : at;
    const bool mine = row0 + ri < a.M;  // (rows past the last read it again)
    const int row = min(row0 + ri, a.M - 1);
    const size_t base = (size_t)row * a.K;
    // elements 4 g .. of the block and 16 + 4 g .. for chunk c
    auto load8 = [&](int c, float4 &ve, float4 &vf) {
        const size_t col = (size_t)(c >> 2) * 32 + 4 * (c & 3), o = base + col;
        if constexpr (SRC == SRC_ROWS || SRC == SRC_EMBED) {
            const float *p = a.x + (SRC == SRC_EMBED ? (size_t)a.tok[row] * a.K + col : o);
            ve = *reinterpret_cast<const float4 *>(p);
            vf = *reinterpret_cast<const float4 *>(p + 16);
        } else if constexpr (SRC == SRC_SWIGLU) {
            float4 v[2];
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const float4 g = sum4(a.x + o + 16 * k, a.S, 2 * a.MK);
                const float4 u = sum4(a.x + a.MK + o + 16 * k, a.S, 2 * a.MK);
                v[k] = make_float4(silu_mul(g.x, u.x), silu_mul(g.y, u.y), silu_mul(g.z, u.z),
                                   silu_mul(g.w, u.w));
            }
            ve = v[0];
            vf = v[1];
        } else if constexpr (SRC == SRC_ATTN) {
            // the chunks that reach the last key of this position's tile
            const int last = a.start + min((row / a.pt + 1) * a.pt, a.M) - 1;
            const int n = last / a.span + 1;
            const size_t heads = a.K / 128, step = (size_t)a.M * heads;
            const float2 *ml = reinterpret_cast<const float2 *>(a.ml) + row * heads +
                               col / 128;
            float m = -INFINITY, l = 0.0f;
#pragma unroll 4
            for (int i = 0; i < n; ++i) m = fmaxf(m, ml[i * step].x);
            ve = vf = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 4
            for (int i = 0; i < n; ++i) {
                const float2 p = ml[i * step];
                const float f = __builtin_amdgcn_exp2f(p.x - m);
                const float4 e = *reinterpret_cast<const float4 *>(a.x + i * a.MK + o);
                const float4 h = *reinterpret_cast<const float4 *>(a.x + i * a.MK + o + 16);
                l = __builtin_fmaf(f, p.y, l);
                ve.x = __builtin_fmaf(f, e.x, ve.x);
                ve.y = __builtin_fmaf(f, e.y, ve.y);
                ve.z = __builtin_fmaf(f, e.z, ve.z);
                ve.w = __builtin_fmaf(f, e.w, ve.w);
                vf.x = __builtin_fmaf(f, h.x, vf.x);
                vf.y = __builtin_fmaf(f, h.y, vf.y);
                vf.z = __builtin_fmaf(f, h.z, vf.z);
                vf.w = __builtin_fmaf(f, h.w, vf.w);
            }
            const float r = 1.0f / l;
            ve = make_float4(ve.x * r, ve.y * r, ve.z * r, ve.w * r);
            vf = make_float4(vf.x * r, vf.y * r, vf.z * r, vf.w * r);
        } else {
            float4 v[2];
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                v[k] = sum4(a.x + o + 16 * k, a.S, a.MK);
                if (a.resid) {
                    const float4 r = *reinterpret_cast<const float4 *>(a.resid + o + 16 * k);
                    v[k] = make_float4(r.x + v[k].x, r.y + v[k].y, r.z + v[k].z, r.w + v[k].w);
                }
            }
            ve = v[0];
            vf = v[1];
        }
    };
    float ss = 0.0f, mx = 0.0f;
    auto scan = [&](int c, float4 ve, float4 vf) {
        const int o = (c >> 2) * 32 + 4 * (c & 3);
        if constexpr (SRC == SRC_PART || SRC == SRC_EMBED) {
            if (mine) {
                *reinterpret_cast<float4 *>(a.y + base + o) = ve;
                *reinterpret_cast<float4 *>(a.y + base + o + 16) = vf;
            }
        }
        const float v[8] = {ve.x, ve.y, ve.z, ve.w, vf.x, vf.y, vf.z, vf.w};
        if constexpr (NORM) {
            // 1/rms > 0 is a common factor of the row: max|(x/rms) w| =
            // max|x w| / rms
            const float4 ge = *reinterpret_cast<const float4 *>(a.norm_w + o);
            const float4 gf = *reinterpret_cast<const float4 *>(a.norm_w + o + 16);
            const float g[8] = {ge.x, ge.y, ge.z, ge.w, gf.x, gf.y, gf.z, gf.w};
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                ss += v[k] * v[k];
                mx = fmaxf(mx, fabsf(v[k] * g[k]));
            }
        } else {
#pragma unroll
            for (int k = 0; k < 8; ++k) mx = fmaxf(mx, fabsf(v[k]));
        }
    };
    // the first CH chunks of a thread stay in registers; a longer row's rest
    // is read again for the second pass
    float4 ve[CH], vf[CH];
#pragma unroll
    for (int j = 0; j < CH; ++j) load8(min(c0 + tid + j * nt, nch - 1), ve[j], vf[j]);
#pragma unroll
    for (int j = 0; j < CH; ++j)
        if (c0 + tid + j * nt < nch) scan(c0 + tid + j * nt, ve[j], vf[j]);
    for (int c = c0 + tid + CH * nt; c < nch; c += nt) {
        float4 e, f;
        load8(c, e, f);
        scan(c, e, f);
    }
#pragma unroll
    for (int off = 32; off >= R; off >>= 1) {
        if constexpr (NORM) ss += __shfl_xor(ss, off);
        mx = fmaxf(mx, __shfl_xor(mx, off));
    }
    if (lane < R) {
        red[0][wave][ri] = ss;
        red[1][wave][ri] = mx;
    }
    __syncthreads();
    ss = red[0][0][ri];
    mx = red[1][0][ri];
    for (int w = 1; w < (int)blockDim.x / 64; ++w) {
        ss += red[0][w][ri];
        mx = fmaxf(mx, red[1][w][ri]);
    }
    if (!mine) return;
    const float inv = NORM ? 1.0f / sqrtf(ss / (float)a.K + a.eps) : 1.0f;
    mx *= inv;
    const int e = mx > 0.0f ? max(ilogbf(mx) - 10, -126) : 0;
    const float sc = ldexpf(1.0f, -e);
    if (tid == 0) a.rowscale[blockIdx.y * a.M + row] = ldexpf(1.0f, e);
    auto emit = [&](int c, float4 ve, float4 vf) {
        const int b = c >> 2, g = c & 3;
        float v[8] = {ve.x, ve.y, ve.z, ve.w, vf.x, vf.y, vf.z, vf.w};
        if constexpr (NORM) {
            const int o = b * 32 + 4 * g;
            const float4 ge = *reinterpret_cast<const float4 *>(a.norm_w + o);
            const float4 gf = *reinterpret_cast<const float4 *>(a.norm_w + o + 16);
            const float gw[8] = {ge.x, ge.y, ge.z, ge.w, gf.x, gf.y, gf.z, gf.w};
#pragma unroll
            for (int k = 0; k < 8; ++k) v[k] = (v[k] * inv) * gw[k];
        }
        uint32_t hb[8], lb[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const float t = v[k] * sc * (k < 4 ? 16.0f : 1.0f);  // exact: powers of two
            const _Float16 h = (_Float16)t;
            hb[k] = __builtin_bit_cast(uint16_t, h);
            lb[k] = __builtin_bit_cast(uint16_t, (_Float16)(t - (float)h));
        }
        uint16_t *p = a.img + (((size_t)(row >> 4) * (a.K >> 5) + b) << 10) + 128 * g + 8 * (row & 15);
        *reinterpret_cast<uint4 *>(p) = make_uint4(hb[0] | hb[2] << 16, hb[4] | hb[6] << 16,
                                                   hb[1] | hb[3] << 16, hb[5] | hb[7] << 16);
        *reinterpret_cast<uint4 *>(p + 512) = make_uint4(lb[0] | lb[2] << 16, lb[4] | lb[6] << 16,
                                                        lb[1] | lb[3] << 16, lb[5] | lb[7] << 16);
    };
#pragma unroll
    for (int j = 0; j < CH; ++j)
        if (c0 + tid + j * nt < nch) emit(c0 + tid + j * nt, ve[j], vf[j]);
    for (int c = c0 + tid + CH * nt; c < nch; c += nt) {
        float4 e, f;
        if constexpr (SRC == SRC_PART) {  // this thread's own stores
            const size_t o = base + (size_t)(c >> 2) * 32 + 4 * (c & 3);
            e = *reinterpret_cast<const float4 *>(a.y + o);
            f = *reinterpret_cast<const float4 *>(a.y + o + 16);
        } else {
            load8(c, e, f);
        }
        emit(c, e, f);
    }
}

// y = [resid +] the sum in order of S partials of n elements.
__global__ __launch_bounds__(kT) void gemm_reduce_kernel(const float *__restrict__ part, int S,
                                                         size_t n, const float *resid, float *y) {
    const size_t i = ((size_t)blockIdx.x * kT + threadIdx.x) * 4;
    if (i >= n) return;
    const bool vec = n % 4 == 0 && ((reinterpret_cast<uintptr_t>(y) |
                                     reinterpret_cast<uintptr_t>(resid)) & 15) == 0;
    if (vec) {
        float4 v = sum4(part + i, S, n);
        if (resid) {
            const float4 r = *reinterpret_cast<const float4 *>(resid + i);
            v.x = r.x + v.x;
            v.y = r.y + v.y;
            v.z = r.z + v.z;
            v.w = r.w + v.w;
        }
        *reinterpret_cast<float4 *>(y + i) = v;
        return;
    }
    for (size_t e = i; e < n && e < i + 4; ++e) {
        float v = part[e];
        for (int s = 1; s < S; ++s) v += part[(size_t)s * n + e];
        y[e] = resid ? resid[e] + v : v;
    }
}

// ---------------------------------------------------------------------------
// The GEMM.  WM x WN waves, each RT x CT MFMA tiles of 16 x 16: a workgroup
// tile of BM rows of x by BN rows of W.  A K stage is SB Q4 blocks; its x
// lines, quants and scales go from global memory straight into LDS
// (global_load_lds, no registers), NBUF stages deep: stage st + NBUF - 1 is
// requested when stage st is computed, with one barrier per stage.
template <int RT_, int CT_, int WM_, int WN_, int SB_, int NBUF_>
struct GT {
    static constexpr int RT = RT_, CT = CT_, WM = WM_, WN = WN_, SB = SB_, NBUF = NBUF_;
    static constexpr int BM = 16 * RT * WM, BN = 16 * CT * WN;
    static constexpr int WAVES = WM * WN, THREADS = 64 * WAVES;
    // one stage in LDS: x [row tile][block][hi | lo][lane] x 16 B, quants
    // [column][slot] x 16 B; beside the stages, the scales of two groups of
    // eight blocks, [column] x 16 B each (those of the stages in flight)
    static constexpr int OQ = BM * SB * 128, BUF = OQ + BN * SB * 16;
    static constexpr int GROUPS = 2;
    static constexpr int OD = NBUF * BUF, LDS = OD + GROUPS * BN * 16;
    // 64-lane DMAs: of one stage by kind (a wave issues PX + PQ of them), and
    // of one group's scales (PD each by the first DW waves)
    static constexpr int NX = BM / 16 * SB * 2, NQ = BN * SB / 64, ND = BN / 64;
    static constexpr int PX = NX / WAVES, PQ = NQ / WAVES, PENDING = PX + PQ;
    static constexpr int DW = ND < WAVES ? ND : WAVES, PD = ND / DW;
    static_assert(NX % WAVES == 0 && NQ % WAVES == 0 && ND % DW == 0 && BN % 64 == 0,
                  "every wave issues whole DMAs");
    static_assert(8 % SB == 0 && kChain % 8 == 0, "groups and chains are whole stages");
    static_assert(BM <= 64 && WM == 1, "a lane holds a row's scale");
    static_assert(NBUF <= 3 && NBUF * SB <= 12, "one new group among the stages in flight");
    static_assert(LDS <= 160 * 1024, "LDS");
    static_assert((NBUF - 1) * PENDING + PD < 64, "wait count");
};

// the same as dma16 from an address per lane
__device__ __forceinline__ void dma16v(const void *src, unsigned char *lds_dst) {
    asm volatile("global_load_lds_dwordx4 %0, off"
                 :
                 : "v"(src), "{m0}"(lds_off(lds_dst))
                 : "memory");
}

// all but the newest N of this wave's loads have completed
template <int N>
__device__ __forceinline__ void wait_vm() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
    __builtin_amdgcn_sched_barrier(0);
}

// Workgroup barrier on LDS data only: __syncthreads would also wait for
// every DMA in flight
__device__ __forceinline__ void lds_barrier() {
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// Quants of W column `col` sit in LDS slots in the order block ^ swz(col), so
// that the 16 columns a wave reads a word of spread over all banks.
template <int SB>
__device__ __forceinline__ int swz(int col) {
    return (col / (8 / SB)) & (SB - 1);
}

// Tile t of MT x NT x S -> (m tile, n tile, split): consecutive workgroups go
// round-robin over the 8 XCDs, so when the count divides evenly each XCD
// works on one x row range, which stays in its L2 across its N tiles.
__device__ __forceinline__ void tile_of(int w, int total, int NT, int MT, int *mt, int *nt,
                                        int *sp) {
    int t = w;
    if ((total & 7) == 0) t = (w & 7) * (total >> 3) + (w >> 3);
    *nt = t % NT;
    const int r = t / NT;
    *mt = r % MT;
    *sp = r / MT;
}

__device__ __forceinline__ f32x4 mfma16(f16x8 a, f16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// 4 quant bytes -> the B fragment of their 8 weights
__device__ __forceinline__ f16x8 nibbles(uint32_t w) {
    const f16x2 o1 = {(_Float16)1032.0f, (_Float16)1032.0f};
    const f16x2 o16 = {(_Float16)1152.0f, (_Float16)1152.0f};
    const uint32_t h = w >> 8;
    // one v_and_or_b32: the compiler, which would need two literals for it,
    // takes an and and an or
    auto sub = [](uint32_t v, uint32_t mask, f16x2 o) {
        uint32_t r;
        asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(v), "s"(mask), "v"(0x64006400u));
        return __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2, r) - o);
    };
    return __builtin_bit_cast(f16x8, (u32x4){sub(w, 0x000F000Fu, o1), sub(w, 0x00F000F0u, o16),
                                             sub(h, 0x000F000Fu, o1), sub(h, 0x00F000F0u, o16)});
}

// The row of y's columns that W tile column c belongs to, from the tile's
// first, and its matrix.  SwiGLU: BN / 2 gate rows, then the same BN / 2 up
// rows; with one column tile per wave, eight of each in every column tile, so
// that a wave still holds both.
template <bool SWI, class G>
__device__ __forceinline__ int w_row(int c, bool *up) {
    if constexpr (!SWI) {
        *up = false;
        return c;
    } else if constexpr (G::CT % 2 == 0) {
        *up = c >= G::BN / 2;
        return *up ? c - G::BN / 2 : c;
    } else {
        *up = (c & 8) != 0;
        return (c >> 4) * 8 + (c & 7);
    }
}

// OUT: 0 = the epilogue EPI into y, 1 = f32 partials of split sp into part.
// SwiGLU: a wave holds matching columns of both matrices, so silu(g) u is
// formed in registers.
//
// Sums: a chain of n additions has an error of about sqrt(n) roundings, so
// chains end after kChain blocks, whatever the plan's K splits.  Error against
// 64 bits (2-norm) with 2 to 3000 rows: 4096 -> 6144 1.1-1.2e-7 (one chain of
// 128 blocks 2.1e-7, four of 32 1.3e-7), 12288 -> 4096 1.2-1.4e-7 (one of 384
// 3.6e-7), 1024 -> 3072 0.9-1.0e-7; q4_gemv.hip's f32 products have 1.7-2.2e-7.
// (x_lo's MFMA before x_hi's: 1.5e-7 for 12288.)  The second sums and the
// additions cost 64-row tiles 0-1 % (512 rows of 4096 -> 6144 70.4 -> 70.6 us;
// 3000-token prompts 1-2 %).
//
// Bound, at 512 rows, by the chain of dequantization, MFMAs and scale FMAs,
// which the operands' DMAs overlap only in part (matrix cores busy 29-42 %; 4096
// -> 6144 with row-major x: 73.7 us, 53 without DMA, 90 with DMA alone); at few
// rows by the launch, the first loads and W at about 2.3 TB/s.  Four waves side
// by side along N dequantize every weight once; tiles of 16 and 32 rows keep
// few rows from paying for padding.  128 x 128 tiles with row-major x took, with the passes around them,
// 43.1 us for 16 rows of 4096 -> 12288 (here 16.5, this kernel 40.3 -> 11.5),
// 52.2 for 100 of 12288 -> 4096 (here 41.5), 86.5 for 512 of 4096 -> 6144 (here
// 70.5).
template <int EPI, int OUT, class G, int OCC>
__global__ __launch_bounds__(G::THREADS) __attribute__((amdgpu_waves_per_eu(OCC, OCC)))
void q4_gemm_kernel(cwi::GemmArgs a, int MT, int NT, int S, int per) {
    constexpr bool SWI = EPI == cwi::EPI_SWIGLU;
    constexpr int RT = G::RT, CT = G::CT, SB = G::SB, BM = G::BM, BN = G::BN;
    __shared__ __attribute__((aligned(1024))) unsigned char lds[G::LDS];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int li = lane & 15, lg = lane >> 4;
    int mt, nt, sp;
    tile_of(blockIdx.x, MT * NT * S, NT, MT, &mt, &nt, &sp);
    constexpr int NB = SWI ? BN / 2 : BN;  // columns of y per tile
    const int m0 = mt * BM, n0 = nt * NB;
    const int wm = wave / G::WN, wn = wave % G::WN;
    const int nb = a.K >> 5, ns = a.s_stride;
    const int kb0 = min(nb, sp * per), kb1 = min(nb, kb0 + per);
    const int n_st = (kb1 - kb0 + SB - 1) / SB;

    // ---- the DMAs: sources from the stage's first block, which the stage
    // adds as one uniform offset (the address arithmetic of a stage is then a
    // handful of scalar adds; xo is uniform, a lane adds only its 16 bytes).
    // Rows past N re-read the last.
    const int q_row = lane / SB, q_slot = lane % SB;
    const char *const img = reinterpret_cast<const char *>(a.img) + (size_t)m0 * nb * 128;
    uint32_t xo[G::PX], qo[G::PQ];
    const uint8_t *qb[G::PQ];  // (SwiGLU: the matrix of each DMA)
    const uint16_t *ds[G::PD];
#pragma unroll
    for (int p = 0; p < G::PX; ++p) {
        const int u = wave + p * G::WAVES;
        const int t = u / (2 * SB), b = u / 2 % SB, half = u & 1;
        xo[p] = ((uint32_t)t * nb + b) * 2048 + half * 1024;
    }
#pragma unroll
    for (int p = 0; p < G::PQ; ++p) {
        const int c0 = (wave + p * G::WAVES) * (64 / SB);
        bool up;
        const int r = min(n0 + w_row<SWI, G>(c0 + q_row, &up), a.N - 1) - n0;
        qo[p] = ((uint32_t)r * nb + (q_slot ^ swz<SB>(c0 + q_row))) * 16;
        if constexpr (!(SWI && CT % 2)) (void)w_row<SWI, G>(c0, &up);  // (one matrix per DMA)
        qb[p] = (up ? a.qB : a.qA) + (size_t)n0 * nb * 16;
    }
#pragma unroll
    for (int p = 0; p < G::PD; ++p) {
        bool up;
        const int r = min(n0 + w_row<SWI, G>((wave + p * G::DW) * 64 + lane, &up), a.N - 1);
        ds[p] = (up ? a.sB : a.sA) + (size_t)r * ns;
    }
    auto issue = [&](int st, unsigned char *buf) {
        const int kb = kb0 + st * SB;
        // blocks past the row's end (its last stage only) re-read its last
        const int over = kb + SB - nb;
#pragma unroll
        for (int p = 0; p < G::PX; ++p) {
            const int u = wave + p * G::WAVES, b = u / 2 % SB;
            const uint32_t back = over > 0 ? max(b - (SB - 1 - over), 0) * 2048u : 0u;
            dma16(img + (size_t)kb * 2048 + (xo[p] - back), lane * 16, buf + u * 1024);
        }
#pragma unroll
        for (int p = 0; p < G::PQ; ++p) {
            const int u = wave + p * G::WAVES;
            uint32_t o = qo[p];
            if (over > 0) {
                const int b = q_slot ^ swz<SB>(u * (64 / SB) + q_row);
                o -= max(b - (SB - 1 - over), 0) * 16;
            }
            if constexpr (SWI && CT % 2) dma16v(qb[p] + (size_t)kb * 16 + o, buf + G::OQ + u * 1024);
            else dma16(qb[p] + (size_t)kb * 16, o, buf + G::OQ + u * 1024);
        }
        if (kb % 8 == 0 && wave < G::DW) {  // the scales of a new group
#pragma unroll
            for (int p = 0; p < G::PD; ++p)
                dma16v(ds[p] + kb, lds + G::OD + (kb / 8 % G::GROUPS) * (BN * 16) +
                                       (wave + p * G::DW) * 1024);
        }
    };

    // ---- LDS read offsets of this lane
    int cq[CT], cd[CT];
#pragma unroll
    for (int j = 0; j < CT; ++j) {
        int col = (wn * CT + j) * 16 + li;
        if constexpr (SWI && CT % 2 == 0)
            col = (j >= CT / 2 ? BN / 2 : 0) + (wn * (CT / 2) + j % (CT / 2)) * 16 + li;
        cq[j] = G::OQ + (col * SB + swz<SB>(col)) * 16 + 4 * lg;
        cd[j] = G::OD + col * 16;
    }
    const int xr = wm * RT * SB * 2048 + lane * 16;

    f32x4 acc[RT][CT], sum[RT][CT], t[2][RT];
    float dp = 0.0f;
#pragma unroll
    for (int i = 0; i < RT; ++i) {
        t[0][i] = t[1][i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < CT; ++j) acc[i][j] = sum[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    static_assert(SB * CT % 2 == 0, "steps alternate between two sets of sums, tile CT - 1 last in the second");

#pragma unroll
    for (int s = 0; s < G::NBUF - 1; ++s)
        if (s < n_st) issue(s, lds + s * G::BUF);
    // the tile's row scales, one row per lane, asked for before the loop (at
    // its end their latency would stand alone; rowscale is padded to whole row
    // tiles); the epilogue fetches those of its rows from the other lanes
    const float rs = a.rowscale[(a.seg_blocks ? (size_t)sp * a.M : 0) + m0 + lane % BM];
    // the chain of the last kChain blocks ends; a 64-row tile folds ahead of
    // a stage, where its registers suffice without a spill, a smaller one
    // after it (16 rows of 4096 -> 12288 16.5 us, 16.9 folding ahead)
    auto fold = [&] {
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int j = 0; j < CT; ++j) {
                sum[i][j] += acc[i][j];
                acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
    };
    int cur = 0;
    for (int st = 0; st < n_st; ++st) {
        if (RT >= 4 && st != 0 && st % (kChain / SB) == 0) fold();
        // stage st has landed: what may still fly are the NBUF - 2 stages
        // after it, with the scales of the groups that they begin
        constexpr int AHEAD = G::NBUF - 2;
        if (AHEAD == 0 || st + AHEAD >= n_st) {
            wait_vm<0>();
        } else if ((kb0 + (st + 1) * SB) % 8 == 0 && wave < G::DW) {
            wait_vm<AHEAD * G::PENDING + G::PD>();
        } else {
            wait_vm<AHEAD * G::PENDING>();
        }
        lds_barrier();  // stage st published; stage st - 1's buffer is free
        if (st + G::NBUF - 1 < n_st) {
            int nx = cur + G::NBUF - 1;
            nx = nx >= G::NBUF ? nx - G::NBUF : nx;
            issue(st + G::NBUF - 1, lds + nx * G::BUF);
        }
        const unsigned char *const L = lds + cur * G::BUF;
        const int kb = kb0 + st * SB;
        uint32_t d[CT][SB / 2];  // the stage's scales, two blocks a word
#pragma unroll
        for (int j = 0; j < CT; ++j)
#pragma unroll
            for (int b = 0; b < SB / 2; ++b)
                d[j][b] = *reinterpret_cast<const uint32_t *>(
                    lds + cd[j] + (kb / 8 % G::GROUPS) * (BN * 16) + (kb & 7) * 2 + b * 4);
        // The stage as SB x CT steps.  A step runs the MFMAs of one column
        // tile of one block; beside them go the scale FMAs of the step before
        // and the dequantization of the step after, so the vector ALU works
        // while the matrix core does, and the LDS reads of the next block.
        f16x8 ah[2][RT], al[2][RT], bq[2];
        uint32_t w[2][CT];
        auto read_block = [&](int b) {
#pragma unroll
            for (int j = 0; j < CT; ++j)
                w[b & 1][j] = *reinterpret_cast<const uint32_t *>(L + (cq[j] ^ (b * 16)));
#pragma unroll
            for (int i = 0; i < RT; ++i) {
                const unsigned char *p = L + xr + (i * SB + b) * 2048;
                ah[b & 1][i] = *reinterpret_cast<const f16x8 *>(p);
                al[b & 1][i] = *reinterpret_cast<const f16x8 *>(p + 1024);
            }
        };
        read_block(0);
        bq[0] = nibbles(w[0][0]);
#pragma unroll
        for (int k = 0; k < SB * CT; ++k) {
            const int b = k / CT, j = k % CT, jp = (j + CT - 1) % CT, c = k & 1;
            if (j == 0 && b + 1 < SB) read_block(b + 1);
#pragma unroll
            for (int i = 0; i < RT; ++i)
                t[c][i] = mfma16(ah[b & 1][i], bq[c], f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
            for (int i = 0; i < RT; ++i) t[c][i] = mfma16(al[b & 1][i], bq[c], t[c][i]);
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    acc[i][jp][r] = __builtin_fmaf(dp, t[c ^ 1][i][r], acc[i][jp][r]);
            if (k + 1 < SB * CT) bq[c ^ 1] = nibbles(w[(k + 1) / CT & 1][(k + 1) % CT]);
            // (past the split's last block the scale is 0: the DMAs re-read
            // blocks in range there)
            const f16x2 dh = __builtin_bit_cast(f16x2, d[j][b >> 1]);
            dp = kb + b < kb1 ? (float)dh[b & 1] : 0.0f;
            if constexpr (RT * CT >= 8) {
#pragma unroll
                for (int g = 0; g < 2 * RT; ++g) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
                }
            }
        }
        cur = cur + 1 == G::NBUF ? 0 : cur + 1;
        if (RT < 4 && (st + 1) % (kChain / SB) == 0) fold();
    }
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            acc[i][CT - 1][r] = __builtin_fmaf(dp, t[1][i][r], acc[i][CT - 1][r]);
    fold();

    constexpr int JN = SWI ? (CT + 1) / 2 : CT;
#pragma unroll
    for (int i = 0; i < RT; ++i) {
        // the residuals of a row tile in flight together (past the matrix they
        // re-read its last row or column)
        float res[4][JN];
        if constexpr (EPI == cwi::EPI_ADD && OUT == 0) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int j = 0; j < JN; ++j)
                    res[r][j] = a.resid[(size_t)min(m0 + (wm * RT + i) * 16 + 4 * lg + r, a.M - 1) *
                                            a.N +
                                        min(n0 + (wn * JN + j) * 16 + li, a.N - 1)];
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int mi = (wm * RT + i) * 16 + 4 * lg + r, m = m0 + mi;
            const float sc = kUnscale * __shfl(rs, mi);
#pragma unroll
            for (int j = 0; j < JN; ++j) {
                int n = n0 + (wn * JN + j) * 16 + li;
                bool mine = true;
                const float v = sum[i][j][r] * sc;
                float up = 0.0f;
                if constexpr (SWI && CT % 2) {  // lanes li < 8: gate, li + 8: up
                    n = n0 + wn * 8 + (li & 7);
                    up = __shfl_xor(v, 8);
                    mine = li < 8;
                } else if constexpr (SWI) {
                    up = sum[i][j + CT / 2][r] * sc;
                }
                if (mine && m < a.M && n < a.N) {
                    const size_t o = (size_t)m * a.N + n;
                    if constexpr (OUT == 1 && SWI) {  // [split][gate | up][M][N]
                        float *p = a.part + (size_t)(2 * sp) * a.M * a.N + o;
                        p[0] = v;
                        p[(size_t)a.M * a.N] = up;
                    } else if constexpr (OUT == 1) {
                        a.part[(size_t)sp * a.M * a.N + o] = v;
                    } else if constexpr (EPI == cwi::EPI_STORE) {
                        a.y[o] = v;
                    } else if constexpr (EPI == cwi::EPI_ADD) {
                        a.y[o] = res[r][j] + v;
                    } else {
                        a.y[o] = silu_mul(v, up);
                    }
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Tiles and K splits.  Every tile size has a cost in microseconds, a fit to
// 1,800 timed launches (M 4..2048 over eight Qwen3 projection shapes; 5-7 %
// scatter): launch + blocks * (round * rounds + share * load) + mb * W +
// part * partials, where a workgroup runs `blocks` K blocks, load is the
// workgroups of the busiest CU, rounds is load over the occ workgroups that
// a CU holds, and W and the partials are in MB.  The plan with the least cost
// is within 1.3 % of the best of the timed ones on average (23 % at most; timed
// before sums went in chains, which cost 64-row tiles up to 2 %).  The
// fit of a tile of less than 64 rows holds for one or two row tiles, which is
// all it is used for: more of them read W again for too few rows (512 rows of
// 4096 -> 6144 as 32 x 128 tiles: 83.7 us, as 64 x 128 in two splits 67.9).
// Each of those launches was repeated on the same W, which the 256 MB
// last-level cache then holds: mb is that cache's rate, not HBM's.  First calls
// on new operands take longer at every size (16 rows of 4096 -> 12288: 29 us
// with the passes around it, 16.5 repeated), and their plans may not be the
// best there.
struct Tile {
    int bm, bn, occ;
    float launch, round, share, mb, part;
};
typedef GT<1, 1, 1, 4, 4, 3> G16x64;
typedef GT<1, 2, 1, 4, 4, 2> G16x128;
typedef GT<2, 1, 1, 4, 4, 2> G32x64;
typedef GT<2, 2, 1, 4, 4, 2> G32x128;
typedef GT<4, 2, 1, 4, 2, 2> G64x128;
typedef GT<4, 4, 1, 4, 2, 2> G64x256;
constexpr Tile kTiles[] = {
    {G16x64::BM, G16x64::BN, 4, 2.6f, 0.053f, 0.063f, 0.047f, 0.55f},
    {G16x128::BM, G16x128::BN, 4, 3.1f, 0.088f, 0.066f, 0.084f, 0.41f},
    {G32x64::BM, G32x64::BN, 3, 2.7f, 0.066f, 0.077f, 0.046f, 0.50f},
    {G32x128::BM, G32x128::BN, 3, 3.8f, 0.083f, 0.124f, 0.038f, 0.46f},
    {G64x128::BM, G64x128::BN, 3, 5.8f, 0.169f, 0.190f, 0.027f, 0.24f},
    {G64x256::BM, G64x256::BN, 2, 8.4f, 0.210f, 0.344f, 0.029f, 0.28f},
};
constexpr int kTileCount = sizeof(kTiles) / sizeof(kTiles[0]);
constexpr int kRowPad = 64;        // the x image has whole row tiles of any size
constexpr float kReduceMB = 0.16f; // the pass that sums the partials, per MB

struct GemmPlan {
    int tile, S, MT, NT, per;
};

// columns of the W tile: both matrices' of SwiGLU
int w_cols(cwi::Epi epi, int N) { return epi == cwi::EPI_SWIGLU ? 2 * N : N; }

GemmPlan gemm_plan(const cw_ctx *ctx, cwi::Epi epi, int M, int N, int K, size_t part_floats) {
    const int nb = K / 32, cols = w_cols(epi, N);
    const double w_mb = (double)cols * nb * 18e-6;
    GemmPlan best{};
    double best_cost = 1e30;
    for (int t = 0; t < kTileCount; ++t) {
        const Tile &T = kTiles[t];
        if (T.bm < kRowPad && M > 2 * T.bm) continue;
        const int MT = (M + T.bm - 1) / T.bm, NT = (cols + T.bn - 1) / T.bn;
        for (int S : {1, 2, 3, 4, 6, 8, 12, cwi::kMaxSplits}) {
            const int per = ((nb + S - 1) / S + 7) / 8 * 8;  // whole scale groups
            if (S > 1 && ((nb + per - 1) / per != S ||
                          (size_t)S * M * cols > part_floats))
                continue;
            const double wgs = (double)MT * NT * S, load = ceil(wgs / ctx->n_cu);
            const double rounds = ceil(load / T.occ);
            const double p_mb = S > 1 ? (double)S * M * cols * 4e-6 : 0.0;
            const double cost = T.launch + std::min(per, nb) * (T.round * rounds + T.share * load) +
                                T.mb * w_mb + (T.part + kReduceMB) * p_mb;
            if (cost < best_cost) {
                best_cost = cost;
                best = GemmPlan{t, S, MT, NT, per};
            }
        }
    }
    return best;
}

template <int EPI, int OUT>
int launch_tiles(cw_ctx *ctx, const char *label, const cwi::GemmArgs &a, const GemmPlan &p) {
    const dim3 grid((unsigned)p.MT * p.NT * p.S);
    auto go = [&](auto fn, int threads) {
        return cwi::launch(ctx, label, fn, grid, dim3(threads), 0, a, p.MT, p.NT, p.S, p.per);
    };
    switch (p.tile) {
        case 0: return go(q4_gemm_kernel<EPI, OUT, G16x64, 2>, G16x64::THREADS);
        case 1: return go(q4_gemm_kernel<EPI, OUT, G16x128, 3>, G16x128::THREADS);
        case 2: return go(q4_gemm_kernel<EPI, OUT, G32x64, 2>, G32x64::THREADS);
        case 3: return go(q4_gemm_kernel<EPI, OUT, G32x128, 2>, G32x128::THREADS);
        case 4: return go(q4_gemm_kernel<EPI, OUT, G64x128, 3>, G64x128::THREADS);
        default: return go(q4_gemm_kernel<EPI, OUT, G64x256, 2>, G64x256::THREADS);
    }
}

bool scales_in_groups(int K, const void *s) {
    return K % 256 == 0 && (reinterpret_cast<uintptr_t>(s) & 15) == 0;
}

template <bool NORM, int SRC>
int launch_split_image(cw_ctx *ctx, const char *label, SplitArgs a, int rows, int seg_blocks = 0) {
    // whole waves, no more than the row (segment) has chunks for; up to 12,288
    // elements stay in registers between the two passes
    a.seg = seg_blocks ? seg_blocks * 4 : a.K / 8;
    const int nt = std::min(512, (a.seg + 63) / 64 * 64);
    const int segs = (a.K / 8 + a.seg - 1) / a.seg;
    a.M = rows;
    a.segs = segs;
    // gx workgroups per segment, then those that copy scales (four of them a
    // thread, 4,096 workgroups at most)
    auto go = [&](auto plain, auto padded, int gx, int threads) {
        if (a.pad.mats == 0)
            return cwi::launch(ctx, label, plain, dim3(gx, segs), dim3(threads), 0, a);
        const size_t total = (size_t)a.pad.N * ((a.pad.nb + 7) / 8 * 8);
        const int wgs = (int)std::min<size_t>((total + 4 * threads - 1) / (4 * threads), 4096);
        return cwi::launch(ctx, label, padded, dim3(gx, segs + (wgs + gx - 1) / gx), dim3(threads),
                           0, a);
    };
    // four rows a workgroup where that still gives every CU one, for plain rows
    // with long segments.  Timed both ways for 64 to 3000 rows of 1024 to 16384
    // in the segments of their plans: with 384 chunks and more a segment four
    // rows take 0.66-1.03 of the time of single rows (512 rows of 12288 in four
    // segments 9.5 against 13.0 us, 3000 in one 60 against 74), with 256 and a
    // whole row 0.86-1.04, with 256 and several segments 0.80-1.08 (with 1,024
    // rows 0.86-0.98), with 192 and fewer 1.0-2.1 once the chip is full (512
    // rows of 4096 in eight of 64: 12.4 against 7.9).  (Merging the attention
    // chunks of 512 rows so took 16 us, 8.4 by single rows.)
    if constexpr (SRC == SRC_ROWS) {
        if ((rows >= 4 * ctx->n_cu && a.seg >= 256) ||
            (rows * segs >= 4 * ctx->n_cu && a.seg > 256)) {
            return a.seg <= 512 ? go(split_image_kernel<NORM, SRC, 2, 4, false>,
                                     split_image_kernel<NORM, SRC, 2, 4, true>, (rows + 3) / 4,
                                     1024)
                                : go(split_image_kernel<NORM, SRC, 6, 4, false>,
                                     split_image_kernel<NORM, SRC, 6, 4, true>, (rows + 3) / 4,
                                     1024);
        }
    }
    return a.seg <= nt ? go(split_image_kernel<NORM, SRC, 1, 1, false>,
                            split_image_kernel<NORM, SRC, 1, 1, true>, rows, nt)
                       : go(split_image_kernel<NORM, SRC, 3, 1, false>,
                            split_image_kernel<NORM, SRC, 3, 1, true>, rows, nt);
}

}  // namespace

namespace cwi {

size_t gemm_img_elems(int M, int K) {
    return (size_t)((M + kRowPad - 1) / kRowPad) * kRowPad * K * 2;
}

size_t gemm_rowscale_floats(int M) { return (size_t)M * kMaxSplits + kRowPad; }

size_t gemm_spad_elems(int N, int K, const void *scales) {
    return scales_in_groups(K, scales) ? 0 : (size_t)N * ((K / 32 + 7) / 8 * 8);
}

size_t gemm_part_floats(const cw_ctx *ctx, Epi epi, int M, int N, int K) {
    const GemmPlan p = gemm_plan(ctx, epi, M, N, K, SIZE_MAX);
    return p.S > 1 ? (size_t)p.S * M * w_cols(epi, N) : 0;
}

int gemm_seg_blocks(const cw_ctx *ctx, Epi epi, int M, int N, int K, size_t part_floats) {
    return gemm_plan(ctx, epi, M, N, K, part_floats).per;
}

ScalePad gemm_scale_pad(Epi epi, const uint16_t *sA, const uint16_t *sB, int N, int K,
                        uint16_t *dst) {
    const bool two = epi == EPI_SWIGLU;
    if (scales_in_groups(K, sA) && (!two || scales_in_groups(K, sB))) return ScalePad{};
    return ScalePad{two ? 2 : 1, N, K / 32, {sA, sB}, dst};
}

int launch_split_rows(cw_ctx *ctx, const float *x, const float *norm_w, float eps, int rows, int K,
                      uint16_t *img, float *rowscale, int seg_blocks, const ScalePad &pad) {
    SplitArgs a{};
    a.pad = pad;
    a.x = x;
    a.norm_w = norm_w;
    a.eps = eps;
    a.K = K;
    a.img = img;
    a.rowscale = rowscale;
    return norm_w ? launch_split_image<true, SRC_ROWS>(ctx, "prefill_split_rmsnorm", a, rows)
                  : launch_split_image<false, SRC_ROWS>(ctx, "prefill_split", a, rows, seg_blocks);
}

int launch_embed_split(cw_ctx *ctx, const float *table, const uint32_t *tok_dev,
                       const float *norm_w, float eps, int rows, int K, float *y, uint16_t *img,
                       float *rowscale, const ScalePad &pad) {
    SplitArgs a{};
    a.pad = pad;
    a.x = table;
    a.tok = tok_dev;
    a.y = y;
    a.norm_w = norm_w;
    a.eps = eps;
    a.K = K;
    a.img = img;
    a.rowscale = rowscale;
    return launch_split_image<true, SRC_EMBED>(ctx, "prefill_embed_split", a, rows);
}

int launch_attn_split(cw_ctx *ctx, const AttnPrefillPlan &p, const AttnPrefillArgs &t,
                      int seg_blocks, uint16_t *img, float *rowscale, const ScalePad &pad) {
    const int K = t.n_heads * 128;
    if (p.chunks == 1)
        return launch_split_rows(ctx, t.out, nullptr, 0.0f, t.M, K, img, rowscale, seg_blocks,
                                 pad);
    SplitArgs a{};
    a.pad = pad;
    a.x = t.part;
    a.MK = (size_t)t.M * K;
    a.ml = t.ml;
    a.start = t.start;
    a.pt = p.pt;
    a.span = p.ct * p.kt;
    a.K = K;
    a.img = img;
    a.rowscale = rowscale;
    return launch_split_image<false, SRC_ATTN>(ctx, "prefill_attention_merge", a, t.M,
                                               seg_blocks);
}

int launch_q4_gemm(cw_ctx *ctx, Epi epi, GemmArgs a, int *splits) {
    const GemmPlan p = gemm_plan(ctx, epi, a.M, a.N, a.K, a.part ? a.part_floats : 0);
    const int nb = a.K / 32;
    a.s_stride = nb;
    if (gemm_scale_pad(epi, a.sA, a.sB, a.N, a.K, a.s_pad).mats) {
        a.s_stride = (nb + 7) / 8 * 8;
        a.sA = a.s_pad;
        a.sB = a.s_pad + (size_t)a.N * a.s_stride;
    }
    *splits = p.S > 1 ? p.S : 0;
    switch (epi) {
        case EPI_SWIGLU:
            return p.S > 1 ? launch_tiles<EPI_SWIGLU, 1>(ctx, "q4_gemm_swiglu_splitk", a, p)
                           : launch_tiles<EPI_SWIGLU, 0>(ctx, "q4_gemm_swiglu", a, p);
        case EPI_ADD:
            if (p.S == 1) return launch_tiles<EPI_ADD, 0>(ctx, "q4_gemm_add", a, p);
            return launch_tiles<EPI_STORE, 1>(ctx, "q4_gemm_add_splitk", a, p);
        default:
            return p.S > 1 ? launch_tiles<EPI_STORE, 1>(ctx, "q4_gemm_splitk", a, p)
                           : launch_tiles<EPI_STORE, 0>(ctx, "q4_gemm", a, p);
    }
}

int launch_gemm_reduce(cw_ctx *ctx, const GemmArgs &a, int splits) {
    const size_t n = (size_t)a.M * a.N;
    return launch(ctx, "q4_gemm_reduce", gemm_reduce_kernel, dim3((unsigned)((n + 4 * kT - 1) / (4 * kT))),
                  dim3(kT), 0, (const float *)a.part, splits, n, a.resid, a.y);
}

int launch_reduce_split(cw_ctx *ctx, Epi epi, const GemmArgs &g, int splits, const float *norm_w,
                        float eps, int seg_blocks, uint16_t *img, float *rowscale,
                        const ScalePad &pad) {
    SplitArgs a{};
    a.pad = pad;
    a.x = splits ? g.part : g.y;
    a.S = splits;
    a.MK = (size_t)g.M * g.N;
    a.resid = g.resid;
    a.y = g.y;
    a.norm_w = norm_w;
    a.eps = eps;
    a.K = g.N;
    a.img = img;
    a.rowscale = rowscale;
    if (!splits)
        return launch_split_rows(ctx, g.y, norm_w, eps, g.M, g.N, img, rowscale, seg_blocks, pad);
    if (epi == EPI_SWIGLU)
        return launch_split_image<false, SRC_SWIGLU>(ctx, "q4_gemm_reduce_swiglu", a, g.M,
                                                     seg_blocks);
    return launch_split_image<true, SRC_PART>(ctx, "q4_gemm_reduce_split", a, g.M);
}

}  // namespace cwi

using namespace cwi;

extern "C" int cw_q4_gemm(cw_ctx *ctx, const float *x, int m, const uint16_t *scales,
                          const uint8_t *quants, int in_f, int out_f, float *y) {
    CW_CHECK_ARG(ctx && x && scales && quants && y, "cw_q4_gemm: null argument");
    CW_CHECK_ARG(m > 0 && m <= 65536, "cw_q4_gemm: m=%d outside [1, 65536]", m);
    CW_CHECK_ARG(in_f > 0 && in_f % 32 == 0, "cw_q4_gemm: in_f=%d must be a positive multiple of 32",
                 in_f);
    CW_CHECK_ARG(out_f > 0, "cw_q4_gemm: out_f=%d must be positive", out_f);
    CW_CHECK_ARG(((uintptr_t)quants & 15) == 0 && ((uintptr_t)scales & 1) == 0,
                 "cw_q4_gemm: quants must be 16-byte and scales 2-byte aligned");
    // image, row scales, padded scales, partials (each 16-byte aligned)
    const size_t part = gemm_part_floats(ctx, EPI_STORE, m, out_f, in_f);
    const size_t rs_off = gemm_img_elems(m, in_f) * 2;
    const size_t sp_off = rs_off + ((gemm_rowscale_floats(m) * 4 + 15) & ~size_t(15));
    const size_t part_off = sp_off + ((gemm_spad_elems(out_f, in_f, scales) * 2 + 15) & ~size_t(15));
    void *scratch = nullptr;
    CW_TRY(ctx_scratch(ctx, part_off + part * 4, &scratch));
    char *const base = static_cast<char *>(scratch);
    GemmArgs a{};
    uint16_t *img = reinterpret_cast<uint16_t *>(base);
    float *rs = reinterpret_cast<float *>(base + rs_off);
    a.seg_blocks = part ? gemm_seg_blocks(ctx, EPI_STORE, m, out_f, in_f, part) : 0;
    a.s_pad = reinterpret_cast<uint16_t *>(base + sp_off);
    CW_TRY(launch_split_rows(ctx, x, nullptr, 0.0f, m, in_f, img, rs, a.seg_blocks,
                             gemm_scale_pad(EPI_STORE, scales, nullptr, out_f, in_f, a.s_pad)));
    a.img = img;
    a.rowscale = rs;
    a.sA = scales;
    a.qA = quants;
    a.y = y;
    a.M = m;
    a.N = out_f;
    a.K = in_f;
    if (part) {
        a.part = reinterpret_cast<float *>(base + part_off);
        a.part_floats = part;
    }
    int splits = 0;
    CW_TRY(launch_q4_gemm(ctx, EPI_STORE, a, &splits));
    return splits ? launch_gemm_reduce(ctx, a, splits) : CW_OK;
}
