// k_gemm.hip -- batched Q4_0 x fp32 GEMM for prefill on gfx950 MFMA.
//
// Y[t][m] = sum_k W[m][k] * X[t][k], the per-token GEMV of reference
// src/models/model.c:1120-1561 (every prefill projection loops
// q_gemv_q4_f32_avx2 over the tokens) done as one dense contraction.
//
// Exactness plan (fp32-level accuracy on fp16 matrix cores):
//  * W: the nibble of a Q4_0 element minus 8 is an integer in [-8, 7],
//    exact in fp16.  The block scale s is NOT folded into the operand; each
//    32-element block is one K=32 MFMA step whose fp32 result D is scaled by
//    s in fp32 (inner += s * D), so W enters the matrix core exactly.
//  * X: each token row is scaled by a power of two 2^e (max |x| in
//    [2^14, 2^15)) and split into two fp16 parts: hi = rn(x') and
//    lo = rn(x' - hi) (the subtraction is exact in fp32).  The two parts hold
//    22 significant bits of every element whose lo is an fp16 normal
//    (|x'| >= 2^-3: within 2^17 of the row maximum); smaller elements keep
//    hi's 11 bits plus what the subnormal lo holds (steps of 2^-24).  Two
//    MFMAs per block (hi, lo) against the same weight operand accumulate
//    into one D; the products (q-8)*hi and (q-8)*lo are exact.
//  * Accumulation: a block's D feeds an inner fp32 sum over kInner blocks,
//    which is added to an outer sum (two-level summation): max error
//    relative to sum_k |W x| stays at or below the reference AVX2 order's
//    (four 8-lane accumulators over N/32 blocks) at Llama-3 shapes.
//  * Output: y = outer * 2^-e (exact); a token row with a non-finite input
//    gives NaN outputs (the GEMV kernel's convention).
//
// Tiling: past 64 tokens k_gemm_q4_p (below), 256 (or 192) rows x 128 tokens
// a workgroup, its workgroups ordered so that each XCD keeps one token tile of
// X resident in its L2 and streams the weight rows; 33 to 64 tokens k_gemm_q4,
// 256 rows x 64 tokens.  K advances in steps of 2 blocks staged in LDS; the
// weights stay raw nibble blocks + scales there and are dequantized per lane
// right before the MFMA.  Up to 32 tokens k_gemm_q4_s, 64 (or 32) rows,
// everything straight to registers.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "qh_kernels.hpp"
#include "qh_lds.hpp"
#include "qh_vec.hpp"

namespace qh {

typedef _Float16 h2v __attribute__((ext_vector_type(2)));
typedef _Float16 h8v __attribute__((ext_vector_type(8)));
typedef float f4v __attribute__((ext_vector_type(4)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));

constexpr int kBufFlagsG = 0x00020000;  // raw buffer resource word 3 (gfx9 family)
constexpr int kKB = 2;                  // Q4_0 blocks per K-step
constexpr int kInner = 16;              // blocks per inner sum

// In-group order of the 8 elements a lane feeds to the MFMA: the nibble
// unpack below yields (e0,e4), (e1,e5), (e2,e6), (e3,e7) as half pairs, so
// position p holds element perm8(p) = {0,4,1,5,2,6,3,7}[p].
__device__ __forceinline__ constexpr int perm8(int p) { return (p >> 1) + 4 * (p & 1); }

// ---------------------------------------------------------------------------
// X preparation: one workgroup per (padded) token row.
// xh/xl: [T_pad][N_pad] fp16 (hi, lo), permuted within groups of 8, or block
// by block ([N_pad/32][blk_rows][32]) when blk_rows is set; columns >= N and
// rows >= T are zero.  meta[t] = (2^-e, non-finite flag).
// The row fed to the matrix cores is one of
//   x                      (plain),
//   (x * r) * norm_w       (RMSNorm, r = rms_scale of the row: the decode
//                           prologue's factor, reference rmsnorm.c:33-89),
//   silu(x) * u            (the SwiGLU product, reference silu.c:75-82 then
//                           mul_fp32.c; x is the gate row, u the up row).
// ---------------------------------------------------------------------------
struct GemmXIn {
    const float* x;
    const float* u;       // SwiGLU mode when non-null
    const float* norm_w;  // RMSNorm mode when non-null
    float eps;
    // Reduction mode when part is non-null: row t is
    // (sum_s part[s][t]) * pmeta[t].x + res[t] (NaN where pmeta[t].y is set),
    // the order of k_gemm_reduce and gemm_store, and is also written to x.
    const float* part;
    uint32_t split;
    const float2* pmeta;
    const float* res;
};

constexpr uint32_t kXpMaxGroups = 16;  // 8-element groups per thread: rows of up to 32768 elements

template <uint32_t kXpGroups>
__global__ __launch_bounds__(256) void k_gemm_xprep(const GemmXIn in, uint32_t T, uint32_t N, uint32_t N_pad,
                                                    uint32_t blk_rows, _Float16* __restrict__ xh,
                                                    _Float16* __restrict__ xl, float2* meta) {  // meta may be the producer's pmeta
    __shared__ float red[4];
    __shared__ int red_f[4];
    const uint32_t t = blockIdx.x;
    const bool valid = t < T;  // uniform over the workgroup
    const uint32_t ng = N_pad / 8, nv = valid ? N / 8 : 0u;  // groups of the padded row / holding data
    const float4* x4 = reinterpret_cast<const float4*>(in.x + (size_t)t * N);
    const float4* u4 = in.u ? reinterpret_cast<const float4*>(in.u + (size_t)t * N) : nullptr;
    // The thread's groups g = tid + 256*i, read once (two 16-byte loads each).
    float v[kXpGroups][8];
    float ss = 0.0f;
    // reduction mode: the producer's scale and flag of this row (read before
    // the barriers that precede this kernel's own meta store)
    const float2 pm = (in.part && valid) ? in.pmeta[t] : make_float2(1.0f, 0.0f);
    const size_t pstride = (size_t)T * N / 4;  // float4s per partial plane
#pragma unroll
    for (uint32_t i = 0; i < kXpGroups; ++i) {
        const uint32_t g = threadIdx.x + 256u * i;
        float4 a = make_float4(0.0f, 0.0f, 0.0f, 0.0f), b = a;
        if (g < nv) {
            if (in.part) {
                const float4* p4 = reinterpret_cast<const float4*>(in.part + (size_t)t * N);
                a = p4[2 * g];
                b = p4[2 * g + 1];
                uint32_t sp = 1;
                // 4 partials' loads in flight at a time; the sum stays
                // sequential in split order
                for (; sp + 4 <= in.split; sp += 4) {
                    float4 c[4], d[4];
#pragma unroll
                    for (uint32_t u = 0; u < 4; ++u) {
                        c[u] = p4[(sp + u) * pstride + 2 * g];
                        d[u] = p4[(sp + u) * pstride + 2 * g + 1];
                    }
#pragma unroll
                    for (uint32_t u = 0; u < 4; ++u) {
                        a.x += c[u].x; a.y += c[u].y; a.z += c[u].z; a.w += c[u].w;
                        b.x += d[u].x; b.y += d[u].y; b.z += d[u].z; b.w += d[u].w;
                    }
                }
                for (; sp < in.split; ++sp) {
                    const float4 c = p4[sp * pstride + 2 * g], d = p4[sp * pstride + 2 * g + 1];
                    a.x += c.x; a.y += c.y; a.z += c.z; a.w += c.w;
                    b.x += d.x; b.y += d.y; b.z += d.z; b.w += d.w;
                }
                a.x = a.x * pm.x; a.y = a.y * pm.x; a.z = a.z * pm.x; a.w = a.w * pm.x;
                b.x = b.x * pm.x; b.y = b.y * pm.x; b.z = b.z * pm.x; b.w = b.w * pm.x;
                if (in.res) {
                    const float4* r4 = reinterpret_cast<const float4*>(in.res + (size_t)t * N);
                    const float4 c = r4[2 * g], d = r4[2 * g + 1];
                    a.x = c.x + a.x; a.y = c.y + a.y; a.z = c.z + a.z; a.w = c.w + a.w;
                    b.x = d.x + b.x; b.y = d.y + b.y; b.z = d.z + b.z; b.w = d.w + b.w;
                }
                if (pm.y != 0.0f) {
                    const float q = __builtin_nanf("");
                    a = make_float4(q, q, q, q);
                    b = a;
                }
                float4* o4 = reinterpret_cast<float4*>(const_cast<float*>(in.x) + (size_t)t * N);
                o4[2 * g] = a;
                o4[2 * g + 1] = b;
            } else {
                a = x4[2 * g];
                b = x4[2 * g + 1];
            }
        }
        v[i][0] = a.x; v[i][1] = a.y; v[i][2] = a.z; v[i][3] = a.w;
        v[i][4] = b.x; v[i][5] = b.y; v[i][6] = b.z; v[i][7] = b.w;
        if (in.norm_w) {
#pragma unroll
            for (int e = 0; e < 8; ++e) ss = ss + v[i][e] * v[i][e];
        }
        if (u4 && g < nv) {
            const float4 c = u4[2 * g], d = u4[2 * g + 1];
            const float uu[8] = {c.x, c.y, c.z, c.w, d.x, d.y, d.z, d.w};
#pragma unroll
            for (int e = 0; e < 8; ++e) v[i][e] = silu_approx(v[i][e]) * uu[e];
        }
    }
    if (in.norm_w) {
        // r = newton(rsq(sum/N + eps)), the RMSNorm factor of reference
        // rmsnorm.c:62-71 (the sum in this kernel's fixed order)
        const float sum = block_sum<256>(ss, red);
        const float av = sum / (float)N + in.eps;
        const float r0 = __builtin_amdgcn_rsqf(av);
        const float r = (r0 * (3.0f - av * (r0 * r0))) * 0.5f;
        const float4* w4 = reinterpret_cast<const float4*>(in.norm_w);
#pragma unroll
        for (uint32_t i = 0; i < kXpGroups; ++i) {
            const uint32_t g = threadIdx.x + 256u * i;
            if (g < nv) {
                const float4 c = w4[2 * g], d = w4[2 * g + 1];
                const float ww[8] = {c.x, c.y, c.z, c.w, d.x, d.y, d.z, d.w};
#pragma unroll
                for (int e = 0; e < 8; ++e) v[i][e] = (v[i][e] * r) * ww[e];
            }
        }
    }
    float m = 0.0f;
    int nf = 0;
#pragma unroll
    for (uint32_t i = 0; i < kXpGroups; ++i)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            nf |= !__builtin_isfinite(v[i][e]);
            m = fmaxf(m, fabsf(v[i][e]));
        }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        m = fmaxf(m, __shfl_xor(m, off));
        nf |= __shfl_xor(nf, off);
    }
    if ((threadIdx.x & 63) == 0) {
        red[threadIdx.x >> 6] = m;
        red_f[threadIdx.x >> 6] = nf;
    }
    __syncthreads();
    m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    nf = red_f[0] | red_f[1] | red_f[2] | red_f[3];
    int e = 0;
    if (!nf && m > 0.0f) {
        int E;
        frexpf(m, &E);  // m = f * 2^E, f in [0.5, 1)
        e = 15 - E;     // m * 2^e in [2^14, 2^15)
    }
    // [row][N_pad], or [block][blk_rows][32] for k_gemm_q4_s
    const size_t at = (size_t)t * (blk_rows ? 32u : N_pad);
    _Float16* hr = xh + at;
    _Float16* lr = xl + at;
#pragma unroll
    for (uint32_t i = 0; i < kXpGroups; ++i) {
        const uint32_t g = threadIdx.x + 256u * i;
        if (g < ng) {
            h8v hv, lv;
#pragma unroll
            for (int p = 0; p < 8; ++p) {
                const float w = nf ? 0.0f : ldexpf(v[i][perm8(p)], e);
                const _Float16 h = (_Float16)w;
                hv[p] = h;
                lv[p] = (_Float16)(w - (float)h);  // the exact difference, rounded
            }
            const size_t o = blk_rows ? (size_t)(g >> 2) * blk_rows * 32u + (g & 3u) * 8u : (size_t)g * 8u;
            *reinterpret_cast<h8v*>(hr + o) = hv;
            *reinterpret_cast<h8v*>(lr + o) = lv;
        }
    }
    if (threadIdx.x == 0) meta[t] = make_float2(ldexpf(1.0f, -e), nf ? 1.0f : 0.0f);
}

// ---------------------------------------------------------------------------
// Main kernel
// ---------------------------------------------------------------------------
constexpr int kGemmMaxSeg = 3;

struct GemmArgs {
    const uint8_t* w[kGemmMaxSeg];
    float* y[kGemmMaxSeg];
    const float* res[kGemmMaxSeg];  // optional residual rows added to y (same layout)
    uint32_t M[kGemmMaxSeg];        // weight rows (output columns) of the segment
    uint32_t ld[kGemmMaxSeg];       // row length of y and res (the whole matrix's rows)
    uint32_t mt_end[kGemmMaxSeg];   // cumulative m-tile counts per segment
    uint32_t nseg;
    uint32_t nblk;        // blocks per weight row
    uint32_t T;
    uint32_t N_pad;       // staged X row length (halfs)
    uint32_t n_tt;        // token tiles
    uint32_t split;       // K splits (partials when > 1)
    uint32_t blk_per_split;
    uint32_t xcd_map;     // 1: XCD-aware tile order
    const _Float16* xh;
    const _Float16* xl;   // the low part
    const float2* meta;
    float* part;          // [split][T][M_total-slot] partials (split > 1)
    uint32_t part_ld;     // partial row length (sum of segment M)
    uint32_t part_off[kGemmMaxSeg];  // column offset of each segment in a partial row
};

// Segment of m-tile index mt / of partial-row column c.
__device__ __forceinline__ uint32_t seg_of_tile(const GemmArgs& a, uint32_t mt) {
    return (a.nseg > 1 && mt >= a.mt_end[0] ? 1u : 0u) + (a.nseg > 2 && mt >= a.mt_end[1] ? 1u : 0u);
}
__device__ __forceinline__ uint32_t seg_of_col(const GemmArgs& a, uint32_t c) {
    return (a.nseg > 1 && c >= a.part_off[1] ? 1u : 0u) + (a.nseg > 2 && c >= a.part_off[2] ? 1u : 0u);
}

// Final value of Y[t][m] in segment sg from the fp32 sum v of the scaled
// operands: v * 2^-e, plus the residual when given; NaN for a non-finite row.
__device__ __forceinline__ void gemm_store(const GemmArgs& a, uint32_t sg, uint32_t t, uint32_t m, float v) {
    const float2 mt = a.meta[t];
    const size_t i = (size_t)t * a.ld[sg] + m;
    float y = v * mt.x;
    if (a.res[sg]) y = a.res[sg][i] + y;
    a.y[sg][i] = mt.y != 0.0f ? __builtin_nanf("") : y;
}

// gemm_store of rows m .. m+3 (those below the segment's M), with 16-byte
// accesses where the row length is a multiple of 4.  They are 4-byte aligned:
// so is Y, and a second launch's piece of a segment can start at any row.
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));

__device__ __forceinline__ void gemm_store4(const GemmArgs& a, uint32_t sg, uint32_t t, uint32_t m, f4v v) {
    const uint32_t M = a.M[sg];
    if ((a.ld[sg] & 3u) != 0 || m + 3 >= M) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (m + r < M) gemm_store(a, sg, t, m + r, v[r]);
        return;
    }
    const float2 mt = a.meta[t];
    const size_t i = (size_t)t * a.ld[sg] + m;
    f4v y = v * mt.x;
    if (a.res[sg]) y = *reinterpret_cast<const f4u*>(a.res[sg] + i) + y;
    if (mt.y != 0.0f) y = f4v{__builtin_nanf(""), __builtin_nanf(""), __builtin_nanf(""), __builtin_nanf("")};
    *reinterpret_cast<f4u*>(a.y[sg] + i) = y;
}

// (a & mask) | c in one instruction (the compiler splits it in two when both
// constants are literals).
__device__ __forceinline__ uint32_t and_or(uint32_t a, uint32_t mask, uint32_t c) {
    uint32_t r;
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "s"(mask), "v"(c));
    return r;
}

// 8 nibbles of one dword -> 8 fp16 (q - 8), in the perm8 order: half pairs
// (n_c, n_{c+4}) for c = 0..3.  A nibble OR'ed under the fp16 bit pattern of
// 1024 gives 1024 + n (bits 0-3) or 1024 + 16 n (bits 4-7); the first is
// shifted by -1032, the second scaled by 1/16 and shifted by -72 (every step
// exact in fp16).  Nibbles 2, 3, 6, 7 take the same two forms after a shift
// by 8.
__device__ __forceinline__ h8v unpack8(uint32_t w) {
    const uint32_t w8 = w >> 8;
    const h2v lo_shift = {(_Float16)-1032.0f, (_Float16)-1032.0f};
    const h2v hi_scale = {(_Float16)0.0625f, (_Float16)0.0625f};
    const h2v hi_shift = {(_Float16)-72.0f, (_Float16)-72.0f};
    const h2v p0 = __builtin_bit_cast(h2v, and_or(w, 0x000F000Fu, 0x64006400u)) + lo_shift;
    const h2v p1 = __builtin_elementwise_fma(__builtin_bit_cast(h2v, and_or(w, 0x00F000F0u, 0x64006400u)), hi_scale, hi_shift);
    const h2v p2 = __builtin_bit_cast(h2v, and_or(w8, 0x000F000Fu, 0x64006400u)) + lo_shift;
    const h2v p3 = __builtin_elementwise_fma(__builtin_bit_cast(h2v, and_or(w8, 0x00F000F0u, 0x64006400u)), hi_scale, hi_shift);
    return h8v{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
}

// The kernel of 33 to 64 tokens (one 64-token tile).  X hi/lo rows (padded: conflict-free 16-byte
// reads) and the weight blocks go through registers into double-buffered LDS,
// one barrier per K-step; global loads run ahead of the LDS stages, X one step
// (L2 hits), the weight blocks two (HBM latency).
// MI: 16-row weight subtiles per wave, JT: 16-token subtiles per wave (a
// wave's tile is 16*MI x 16*JT).
constexpr int kGemmWM = 4;  // waves, one below the other

__global__ __launch_bounds__(64 * kGemmWM) void k_gemm_q4(const GemmArgs a) {
    constexpr int MI = 4, JT = 4, KB = kKB;
    constexpr int NT = 64 * kGemmWM;
    constexpr int WR = 16 * MI;  // weight rows per wave
    constexpr int BM = WR * kGemmWM;
    constexpr int BT = 16 * JT;
    constexpr int XCK = 4 * KB;                       // 16-byte X chunks per staged row and part
    constexpr int XROW = 32 * KB + 8;                 // LDS halfs per staged X row (8 pad)
    constexpr int XCH = 2 * XCK * BT / NT;            // 16-byte X chunks per thread per K-step
    constexpr int WBL = BM * KB / NT;                 // weight blocks per thread per K-step
    static_assert(XCH * NT == 2 * XCK * BT && WBL * NT == BM * KB, "tile/thread mismatch");
    static_assert(KB == 2, "K-step of 2 blocks");
    static_assert(kInner % KB == 0, "inner sums end on K-step boundaries");
    // A row's blocks sit in its KB slots rotated by the row, so that the
    // per-lane 16-byte reads of 8 consecutive rows cover all 32 banks.
    constexpr int kSwz = 2;

    __shared__ __attribute__((aligned(16))) _Float16 lx[2][2][BT][XROW];
    __shared__ __attribute__((aligned(16))) uint32_t lw[2][BM][KB][4];
    __shared__ __attribute__((aligned(16))) float ls[2][KB][BM];

    // ---- tile of this workgroup: an (m-tile, split) pair ----
    const uint32_t mm = blockIdx.x;
    if (mm >= a.mt_end[a.nseg - 1] * a.split) return;
    const uint32_t mtile = mm / a.split, sp = mm % a.split;
    const uint32_t sg = seg_of_tile(a, mtile);
    const uint32_t m0 = (mtile - (sg ? a.mt_end[sg - 1] : 0u)) * BM;
    const uint32_t M = a.M[sg];
    const uint32_t row_bytes = a.nblk * 20u;
    const uint32_t b_begin = sp * a.blk_per_split;
    const uint32_t b_end = min(a.nblk, b_begin + a.blk_per_split);
    const uint32_t nsteps = b_end > b_begin ? (b_end - b_begin + KB - 1) / KB : 0u;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wm = __builtin_amdgcn_readfirstlane(tid >> 6);

    const __amdgpu_buffer_rsrc_t wrs =
        __builtin_amdgcn_make_buffer_rsrc((void*)a.w[sg], 0, (int)(M * row_bytes), kBufFlagsG);

    // ---- global -> register staging ----
    // X of step k is loaded one step ahead (it is served by L2); the weight
    // blocks of step k two steps ahead, into register set k & 1, so that
    // their HBM latency has two steps of compute to hide behind.  Within a
    // step the X loads are issued first: the wait before the LDS store then
    // leaves the newest weight loads in flight.
    u4v gx[XCH];
    u4v gq[2][WBL];
    float gs[2][WBL];
    // The thread's X chunks (row t, 8 halfs at column 8*ch of the step)
    // as pointers fixed for the whole loop.
    const _Float16* xsrc[XCH];
#pragma unroll
    for (int c = 0; c < XCH; ++c) {
        const uint32_t idx = (uint32_t)(tid + NT * c);
        const uint32_t part = idx / (XCK * BT);
        const uint32_t rem = idx % (XCK * BT);
        const uint32_t t = rem / XCK, ch = rem % XCK;
        xsrc[c] = (part ? a.xl : a.xh) + (size_t)t * a.N_pad + 8u * ch;
    }
    auto load_x = [&](uint32_t step) {
        // < N_pad - (32 KB - 1): splits start on multiples of KB blocks and
        // N_pad is a multiple of 128
        const uint32_t k0 = (b_begin + step * KB) * 32u;
#pragma unroll
        for (int c = 0; c < XCH; ++c) gx[c] = *reinterpret_cast<const u4v*>(xsrc[c] + k0);
    };
    auto load_w = [&](uint32_t step, auto setc) {
        constexpr int set = decltype(setc)::value;
        const uint32_t b0 = b_begin + step * KB;
#pragma unroll
        for (int j = 0; j < WBL; ++j) {
            const uint32_t idx = (uint32_t)(tid + NT * j);
            const uint32_t r = idx / KB, kb = idx % KB;
            const uint32_t b = b0 + kb;
            // rows >= M read zeros
            const uint32_t off = (m0 + r) * row_bytes + b * 20u;
            // Blocks past the split's end are masked at the LDS store (a
            // select here would wait for the load right away).
            gq[set][j] = __builtin_amdgcn_raw_buffer_load_b128(wrs, off, 0, 0);
            gs[set][j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(wrs, off + 16u, 0, 0));
        }
    };
    // LDS buffer `buf` (also the weight register set) <- the staged step.
    auto store_step = [&](uint32_t step, auto bufc) {
        constexpr int buf = decltype(bufc)::value;
        const uint32_t b0 = b_begin + step * KB;
#pragma unroll
        for (int c = 0; c < XCH; ++c) {
            const uint32_t idx = (uint32_t)(tid + NT * c);
            const uint32_t part = idx / (XCK * BT);
            const uint32_t rem = idx % (XCK * BT);
            const uint32_t t = rem / XCK, ch = rem % XCK;
            *reinterpret_cast<u4v*>(&lx[buf][part][t][8u * ch]) = gx[c];
        }
#pragma unroll
        for (int j = 0; j < WBL; ++j) {
            const uint32_t idx = (uint32_t)(tid + NT * j);
            const uint32_t r = idx / KB, kb = idx % KB;
            // A zero scale removes a masked block: its products are finite.
            *reinterpret_cast<u4v*>(&lw[buf][r][kb ^ ((r >> kSwz) & (KB - 1u))][0]) = gq[buf][j];
            ls[buf][kb][r] = b0 + kb < b_end ? gs[buf][j] : 0.0f;
        }
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;

    f4v inner[MI][JT], outer[MI][JT];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < JT; ++j) {
            inner[i][j] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
            outer[i][j] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
        }

    const int lr = lane & 15, lq = lane >> 4;
    if (nsteps > 0) {
        load_x(0);
        load_w(0, I0{});
        if (nsteps > 1) load_w(1, I1{});
        store_step(0, I0{});
    }
    __syncthreads();
    uint32_t nb_in = 0;  // blocks in the current inner sum
    // One K-step from LDS buffer `buf` (= step & 1).
    auto step_body = [&](uint32_t step, auto bufc) {
        constexpr int buf = decltype(bufc)::value;
        using Next = std::integral_constant<int, buf ^ 1>;
        // Issued unconditionally (the last steps reload step nsteps - 1, which
        // is never stored): a load issued on one path only would make the wait
        // before the LDS store cover the newest weight loads as well.
        load_x(min(step + 1, nsteps - 1));
        load_w(min(step + 2, nsteps - 1), bufc);  // set buf held step's weights, now in LDS
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
            // The weight fragment is the MFMA's A operand (D rows = weight
            // rows, D columns = tokens): register r of lane l holds weight row
            // 4*(l/16) + r of the subtile for token l%16, so each lane has 4
            // consecutive outputs of one token row, and their 4 scales.
            h8v B[MI];
            f4v s[MI];
#pragma unroll
            for (int i = 0; i < MI; ++i) {
                const int r = WR * wm + 16 * i + lr;
                B[i] = unpack8(lw[buf][r][kb ^ ((r >> kSwz) & (KB - 1))][lq]);
                s[i] = *reinterpret_cast<const f4v*>(&ls[buf][kb][WR * wm + 16 * i + 4 * lq]);
            }
            // One token subtile at a time: its hi and lo parts, then the MI
            // weight subtiles.
#pragma unroll
            for (int j = 0; j < JT; ++j) {
                const int t = 16 * j + lr;
                const h8v Ah = *reinterpret_cast<const h8v*>(&lx[buf][0][t][32 * kb + 8 * lq]);
                const h8v Al = *reinterpret_cast<const h8v*>(&lx[buf][1][t][32 * kb + 8 * lq]);
#pragma unroll
                for (int i = 0; i < MI; ++i) {
                    f4v d = __builtin_amdgcn_mfma_f32_16x16x32_f16(B[i], Ah, f4v{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
                    d = __builtin_amdgcn_mfma_f32_16x16x32_f16(B[i], Al, d, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 4; ++r) inner[i][j][r] = fmaf(s[i][r], d[r], inner[i][j][r]);
                }
            }
        }
        nb_in += KB;
        if (nb_in >= kInner) {
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < JT; ++j) {
                    outer[i][j] += inner[i][j];
                    inner[i][j] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
                }
            nb_in = 0;
        }
        if (step + 1 < nsteps) store_step(step + 1, Next{});
        __syncthreads();
    };
    for (uint32_t step = 0; step < nsteps; step += 2) {
        step_body(step, I0{});
        if (step + 1 < nsteps) step_body(step + 1, I1{});
    }

    // ---- epilogue: lane holds weight rows m .. m+3 of token t ----
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        const uint32_t m = m0 + WR * wm + 16 * i + 4 * lq;
#pragma unroll
        for (int j = 0; j < JT; ++j) {
            const uint32_t t = 16 * j + lr;
            const f4v v = outer[i][j] + inner[i][j];
            if (m < M && t < a.T) {
                if (a.split > 1) {
                    float* dst = a.part + ((size_t)sp * a.T + t) * a.part_ld + a.part_off[sg] + m;
                    if ((a.part_ld & 3u) == 0 && (a.part_off[sg] & 3u) == 0 && m + 3 < M) {
                        *reinterpret_cast<f4v*>(dst) = v;
                    } else {
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            if (m + r < M) dst[r] = v[r];
                    }
                } else {
                    gemm_store4(a, sg, t, m, v);
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Kernel of the 128-token tiles (prompts past 64 tokens): the same contraction
// and the same order of every sum as k_gemm_q4, with the K loop as a software
// pipeline.
//
// Bound by power: at 1999 x 4096 x 14336 the clock falls to 1.95 GHz (the
// same launch on all-zero rows runs 20 % faster at 2.3 GHz), the matrix
// cores are busy half of its cycles, and per MFMA a SIMD also issues 2 scale
// FMAs and 1.2 unpack instructions.  What shortens it is work taken out:
//  * X is the A operand and the weights the B operand: a lane holds 4 tokens
//    of one weight row, whose block scale is one register and one 4-byte LDS
//    read per subtile (four scales per lane the other way round).
//  * X and the weight blocks go from memory straight to LDS (no staging
//    registers, no LDS store instructions): X into a ring of 3 steps, filled
//    two steps ahead, the weights into a ring of 4, filled three steps ahead.
//  * A step (2 blocks) is 8 groups, one per block and 16-token subtile.  A
//    group issues the LDS reads of the next group, runs its own 2*MI MFMAs
//    and, between them, the scale FMAs of the group before and a part of the
//    next block's unpack: nothing that it issues is waited for in it.
//  * One barrier per step, between its two blocks: it publishes the next
//    step and frees the ring slots that the loads issued right behind it
//    overwrite.  The loads' counter is waited down to the newest weight
//    step, so they have one (X) or two (weights) whole steps to land.
// Against the staged kernel it replaced (k_gemm_q4's structure with 8 waves):
// 28672 x 512 x 4096 263.5 -> 244 us, 4096 x 1999 x 14336 494 -> 458 us, both
// with the row conversion; LDS bank conflicts 35 % -> 14 % of its active
// cycles.  32x32x16 MFMAs (half the instructions, 8 % fewer cycles) gave the
// cycles back in clock (466 us), two workgroups of 4 waves per CU with
// 64-token tiles likewise (+3 %).
// ---------------------------------------------------------------------------
constexpr uint32_t kPXSlot = 2 * 128 * 128;      // bytes of an X step: hi and lo, 128 rows of 64 halfs
constexpr uint32_t kPXSlots = 3, kPWSlots = 4;

template <int MI>
__global__ __launch_bounds__(512) void k_gemm_q4_p(const GemmArgs a) {
    constexpr int WR = 16 * MI, BM = 4 * WR, BT = 128;  // 4 x 2 waves of WR x 64
    constexpr uint32_t kWSlot = BM * 2 * 16, kSSlot = BM * 2 * 4;  // bytes of a weight step: nibbles, scales
    constexpr uint32_t kWBase = kPXSlots * kPXSlot, kSBase = kWBase + kPWSlots * kWSlot;
    constexpr uint32_t kLdsBytes = kSBase + kPWSlots * kSSlot;
    constexpr uint32_t kTRow = WR + 4;  // epilogue: floats per staged token row
    static_assert(8 * 16 * kTRow * 4 <= kLdsBytes, "the epilogue's staging reuses the rings");
    __shared__ __attribute__((aligned(1024))) uint8_t lds[kLdsBytes];

    // ---- tile of this workgroup ----
    const uint32_t n_mt = a.mt_end[a.nseg - 1] * a.split;  // (m-tile, split) pairs
    uint32_t mm, tt;
    {
        const uint32_t b = blockIdx.x;
        if (a.xcd_map) {
            const uint32_t xcd = b & 7u, k = b >> 3;
            tt = xcd % a.n_tt;
            mm = xcd / a.n_tt + (8u / a.n_tt) * k;
        } else {
            tt = b % a.n_tt;
            mm = b / a.n_tt;
        }
        if (mm >= n_mt) return;
    }
    const uint32_t mtile = mm / a.split, sp = mm % a.split;
    const uint32_t sg = seg_of_tile(a, mtile);
    const uint32_t m0 = (mtile - (sg ? a.mt_end[sg - 1] : 0u)) * BM;
    const uint32_t t0 = tt * BT;
    const uint32_t M = a.M[sg];
    const uint32_t row_bytes = a.nblk * 20u;
    const uint32_t b_begin = sp * a.blk_per_split;
    const uint32_t b_end = min(a.nblk, b_begin + a.blk_per_split);
    const uint32_t nsteps = b_end > b_begin ? (b_end - b_begin + 1u) / 2u : 0u;

    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t wm = wave % 4u, wt = wave / 4u;
    const uint32_t lr = lane & 15u, lq = lane >> 4;

    // ---- memory -> LDS ----
    // X: waves 0..3 load the hi part, 4..7 the lo part, 32 rows each, as 4
    // loads of 8 LDS rows of 128 bytes.  Of each 16 token rows, row r sits in
    // LDS row 2*(r%8) + r/8 and its 16-byte chunk c in place c ^ (r%8): the
    // 16 lanes that read one chunk of 16 rows then cover 64 banks.
    const uint32_t np2 = a.N_pad * 2u;  // bytes of a staged row
    const rsrc_v rx = make_rsrc((wave < 4u ? a.xh : a.xl) + (size_t)t0 * a.N_pad, BT * np2);
    uint32_t xvoff[2];
#pragma unroll
    for (uint32_t i = 0; i < 2; ++i) {
        const uint32_t s = 8u * i + (lane >> 3), r = (s >> 1) + 8u * (s & 1u);
        xvoff[i] = (32u * (wave & 3u) + r) * np2 + 16u * ((lane & 7u) ^ (r & 7u));
    }
    // Weights: lane pairs take the two blocks of a row (40 contiguous
    // bytes), in an order that turns with bit 3 of the row (64 banks again).
    // Waves 0 .. BM/32 - 1 load 32 rows each; with fewer than 8 of them the
    // others repeat the last one's load (every wave issues the same number).
    const uint32_t ww = min(wave, (uint32_t)BM / 32u - 1u);
    const uint32_t wrow = 32u * ww + (lane >> 1), wkb = (lane & 1u) ^ ((wrow >> 3) & 1u);
    const rsrc_v rw = make_rsrc(a.w[sg], M * row_bytes);
    const uint32_t wvoff = (m0 + wrow) * row_bytes + wkb * 20u;  // rows >= M lie past the end
    const uint32_t lds0 = lds_address(lds);
    auto load_x = [&](uint32_t step, uint32_t slot) {
        const uint32_t k0 = (b_begin + min(step, nsteps - 1u) * 2u) * 64u;  // bytes; columns < N_pad
        const uint32_t dst = lds0 + slot * kPXSlot + wave * 4096u;
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) lds_load16(rx, xvoff[i & 1u], k0 + (i >> 1) * 16u * np2, dst + i * 1024u);
    };
    auto load_w = [&](uint32_t step, uint32_t slot) {
        const uint32_t b0 = b_begin + min(step, nsteps - 1u) * 2u;
        // A block past the split's end reads zeros (a zero scale removes it).
        const uint32_t vo = b0 + wkb < b_end ? wvoff : 0x80000000u;
        lds_load16(rw, vo, b0 * 20u, lds0 + kWBase + slot * kWSlot + ww * 1024u);
        lds_load4(rw, vo, b0 * 20u + 16u, lds0 + kSBase + slot * kSSlot + ww * 256u);
    };

    // ---- LDS -> registers ----
    const uint32_t xr = (wt * 64u + 2u * (lr & 7u) + (lr >> 3)) * 128u + 16u * (lq ^ (lr & 7u));  // block 0; block 1: ^ 64
    const uint32_t wr = (wm * WR + lr) * 32u + (lr >> 3) * 16u + lq * 4u;                          // block 0; block 1: ^ 16
    const uint32_t sr = (wm * WR + lr) * 8u + (lr >> 3) * 4u;                                      // block 0; block 1: ^ 4

    f4v inner[MI][4], outer[MI][4];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            inner[i][j] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
            outer[i][j] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
        }

    if (nsteps > 0) {
        // constants of the nibble unpack, opaque so that (w & mask) | magic
        // stays one instruction
        uint32_t mlo = 0x000F000Fu, mhi = 0x00F000F0u, magic = 0x64006400u;
        asm("" : "+s"(mlo), "+s"(mhi), "+v"(magic));
        h8v xh[2], xl[2];        // X fragments, alternating by group
        u4v wf[2][MI];           // weight fragments (8 halfs) of the two blocks
        uint32_t raw[MI];        // nibbles of the next block
        float sc[2][MI];         // scales of the two blocks
        f4v d[2][MI];            // products, alternating by group
        auto read_x = [&](uint32_t slot, int kb, int j, int set) {
            const uint32_t at = slot * kPXSlot + (xr ^ (kb ? 64u : 0u)) + (uint32_t)j * 2048u;
            xh[set] = *reinterpret_cast<const h8v*>(lds + at);
            xl[set] = *reinterpret_cast<const h8v*>(lds + at + kPXSlot / 2);
        };
        auto read_raw = [&](uint32_t slot, int kb) {
#pragma unroll
            for (int i = 0; i < MI; ++i)
                raw[i] = *reinterpret_cast<const uint32_t*>(lds + kWBase + slot * kWSlot + (wr ^ (kb ? 16u : 0u)) + i * 512u);
        };
        auto read_scale = [&](uint32_t slot, int kb) {
#pragma unroll
            for (int i = 0; i < MI; ++i)
                sc[kb][i] = *reinterpret_cast<const float*>(lds + kSBase + slot * kSSlot + (sr ^ (kb ? 4u : 0u)) + i * 128u);
        };
        // Half pair c of subtile i's fragment: nibbles c and c + 4 (unpack8's
        // arithmetic, one pair at a time).
        auto unpack_pair = [&](int kb, int i, int c) {
            const uint32_t w = c < 2 ? raw[i] : raw[i] >> 8;
            const h2v lo_shift = {(_Float16)-1032.0f, (_Float16)-1032.0f};
            const h2v hi_scale = {(_Float16)0.0625f, (_Float16)0.0625f};
            const h2v hi_shift = {(_Float16)-72.0f, (_Float16)-72.0f};
            const h2v v = (c & 1) ? __builtin_elementwise_fma(__builtin_bit_cast(h2v, (w & mhi) | magic), hi_scale, hi_shift)
                                  : __builtin_bit_cast(h2v, (w & mlo) | magic) + lo_shift;
            wf[kb][i][c] = __builtin_bit_cast(uint32_t, v);
        };

        load_x(0, 0);
        load_w(0, 0);
        load_w(1, 1);
        load_x(1, 1);
        load_w(2, 2);
        wait_vm<6>();  // X and weights of step 0, weights of step 1
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        read_x(0, 0, 0, 0);
        read_raw(0, 0);
        read_scale(0, 0);
#pragma unroll
        for (int i = 0; i < MI; ++i) {
#pragma unroll
            for (int c = 0; c < 4; ++c) unpack_pair(0, i, c);
            sc[1][i] = 0.0f;  // the first group's "previous" products
            d[1][i] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
        }
        uint32_t xs = 0, ws = 0;  // ring slots of the step
        uint32_t nb_in = 0;       // blocks in the current inner sums
        for (uint32_t step = 0; step < nsteps; ++step) {
            const uint32_t xs1 = xs == kPXSlots - 1 ? 0u : xs + 1u, xs2 = xs1 == kPXSlots - 1 ? 0u : xs1 + 1u;
            const uint32_t ws1 = (ws + 1u) & 3u, ws3 = (ws + 3u) & 3u;
            auto group = [&](auto gc) {
                constexpr int g = decltype(gc)::value;
                constexpr int kb = g >> 2, j = g & 3, cur = g & 1, prv = cur ^ 1;
                constexpr int pj = (g + 7) & 3, pkb = ((g + 7) & 7) >> 2;  // the previous group's
                if constexpr (g == 4) {
                    wait_vm<2>();  // X and weights of the next step
                    __builtin_amdgcn_s_barrier();
                    asm volatile("" ::: "memory");
                    load_x(step + 2, xs2);
                    load_w(step + 3, ws3);
                }
                __builtin_amdgcn_sched_barrier(0);
                // next group's X, next block's weights
                if constexpr (g < 7)
                    read_x(xs, (g + 1) >> 2, (g + 1) & 3, prv);
                else
                    read_x(xs1, 0, 0, prv);
                if constexpr (j == 0) read_raw(kb ? ws1 : ws, kb ^ 1);
                if constexpr (j == 1) read_scale(kb ? ws1 : ws, kb ^ 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int q = 0; q < 2 * MI; ++q) {
                    // one MFMA (all hi parts, then all lo parts)
                    const int i = q % MI;
                    if (q < MI)
                        d[cur][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh[cur], __builtin_bit_cast(h8v, wf[kb][i]), f4v{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
                    else
                        d[cur][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl[cur], __builtin_bit_cast(h8v, wf[kb][i]), d[cur][i], 0, 0, 0);
                    // two of the previous group's products
                    const int pi = q >> 1, r0 = 2 * (q & 1);
                    inner[pi][pj][r0] = fmaf(sc[pkb][pi], d[prv][pi][r0], inner[pi][pj][r0]);
                    inner[pi][pj][r0 + 1] = fmaf(sc[pkb][pi], d[prv][pi][r0 + 1], inner[pi][pj][r0 + 1]);
                    // a part of the next block's unpack
                    if (j > 0) {
                        const int t = (j - 1) * 2 * MI + q, p0 = t * 2 / 3, p1 = (t + 1) * 2 / 3;
#pragma unroll
                        for (int pp = p0; pp < p1; ++pp) unpack_pair(kb ^ 1, pp >> 2, pp & 3);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
                if constexpr (g == 0) {
                    // (the sums of 16 blocks end with the previous step's last group)
                    nb_in += 2;
                    if (nb_in > kInner) {
#pragma unroll
                        for (int i = 0; i < MI; ++i)
#pragma unroll
                            for (int q = 0; q < 4; ++q) {
                                outer[i][q] += inner[i][q];
                                inner[i][q] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
                            }
                        nb_in = 2;
                    }
                }
            };
            group(std::integral_constant<int, 0>{});
            group(std::integral_constant<int, 1>{});
            group(std::integral_constant<int, 2>{});
            group(std::integral_constant<int, 3>{});
            group(std::integral_constant<int, 4>{});
            group(std::integral_constant<int, 5>{});
            group(std::integral_constant<int, 6>{});
            group(std::integral_constant<int, 7>{});
            xs = xs1;
            ws = ws1;
        }
        // the last group's products
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) inner[i][3][r] = fmaf(sc[1][i], d[1][i][r], inner[i][3][r]);
    }

    // ---- epilogue ----
    // Lane holds tokens 4*lq .. +3 of weight row lr of each subtile; through
    // LDS (a part of its own per wave) it gets 4 consecutive weight rows of a
    // token, so that 16 lanes store 256 contiguous bytes.
    wait_vm<0>();  // no load may still write the rings
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    float* tr = reinterpret_cast<float*>(lds) + wave * 16u * kTRow;
    constexpr uint32_t kF4 = WR / 4;  // float4s per token row
#pragma unroll
    for (int j = 0; j < 4; ++j) {
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            const f4v v = outer[i][j] + inner[i][j];
#pragma unroll
            for (int r = 0; r < 4; ++r) tr[(4 * lq + r) * kTRow + 16 * i + lr] = v[r];
        }
#pragma unroll
        for (uint32_t u = 0; u < kF4 / 4; ++u) {
            const uint32_t q = u * 64u + lane, tok = q / kF4, c = q % kF4;
            const f4v v = *reinterpret_cast<const f4v*>(tr + tok * kTRow + 4 * c);
            const uint32_t t = t0 + 64u * wt + 16u * j + tok, m = m0 + wm * WR + 4u * c;
            if (m < M && t < a.T) {
                if (a.split > 1) {
                    float* dst = a.part + ((size_t)sp * a.T + t) * a.part_ld + a.part_off[sg] + m;
                    if ((a.part_ld & 3u) == 0 && (a.part_off[sg] & 3u) == 0 && m + 3 < M) {
                        *reinterpret_cast<f4v*>(dst) = v;
                    } else {
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            if (m + r < M) dst[r] = v[r];
                    }
                } else {
                    gemm_store4(a, sg, t, m, v);
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Kernel of up to 32 tokens (JT = 1 or 2 tiles of 16): bound by the weights'
// bytes, which go from memory straight to registers.
//
// A workgroup takes 64 or 32 rows, its 8 waves split the K range (each a run of
// whole groups of 4*J blocks) and meet in LDS at the end, in a fixed tree, so
// one launch fills the chip without partial sums in memory (a second split,
// over workgroups, only where the rows are few).  Lane (r, g) of a 16-row
// subtile loads the 20*J contiguous bytes of row r's blocks J*g .. J*g + J-1
// of the group, so a row's 80*J bytes are taken at once (J = 4, 320 bytes,
// where the row's blocks are a multiple of 16; with J = 1 a 128-byte line
// was fetched again on the next group, and 28672 x 16 x 4096 took 27 us).
// Lane-group swaps then give every lane the MFMA's dword of four blocks at a
// time and spread their scales.  X (staged block by block,
// [block][token][32]) is the A operand, one contiguous KB per part and
// block, read through the caches two blocks ahead.  Blocks add up in sums of
// at most 16, those in the wave's total.
// With the row conversion, us (in brackets 256-row tiles through LDS with
// partial sums in memory, which ran before): 28672 x 16 x 4096 27.7 in 64-row
// tiles, 29.8 in 32-row ones [34.6]; 28672 x 32 x 4096 33.9 and 47.3 [46.1];
// 4096 x 16 x 14336 20.8 and 22.9 [26.0]; 6144 x 16 x 4096 15.3 and 12.1
// [18.4]; 4096 x 16 x 4096 15.2 and 11.7 [18.1].  The 64-row tiles read X
// half as often (it passes the caches at 3.2 times the weights' bytes in
// 32-row tiles of 16 tokens) and want enough rows for one workgroup per CU.
// ---------------------------------------------------------------------------
constexpr int kShortWaves = 8;

// The 4x4 transpose between register index and 16-lane group.
__device__ __forceinline__ void swap_groups(uint32_t& r0, uint32_t& r1, uint32_t& r2, uint32_t& r3) {
    auto a = __builtin_amdgcn_permlane32_swap(r0, r2, false, false);
    auto b = __builtin_amdgcn_permlane32_swap(r1, r3, false, false);
    auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
    auto d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
    r0 = c[0];
    r1 = c[1];
    r2 = d[0];
    r3 = d[1];
}

template <int JT, int J, int RT>
__global__ __launch_bounds__(64 * kShortWaves, RT == 2 && (JT == 1 || J < 4) ? 4 : 2) void k_gemm_q4_s(const GemmArgs a) {
    constexpr int kShortRows = 16 * RT;
    constexpr uint32_t kTok = 16 * JT, kRow = kShortRows + 4;  // staged tokens; floats per LDS row
    constexpr uint32_t kGrp = 4 * J;                           // blocks per group
    static_assert(J == 1 || J == 2 || J == 4, "blocks per lane");
    static_assert(kInner % kGrp == 0, "inner sums end on group boundaries");
    __shared__ __attribute__((aligned(16))) float red[kShortWaves][kTok][kRow];
    const uint32_t mtile = blockIdx.x / a.split, sp = blockIdx.x % a.split;
    const uint32_t sg = seg_of_tile(a, mtile);
    const uint32_t m0 = (mtile - (sg ? a.mt_end[sg - 1] : 0u)) * kShortRows;
    const uint32_t M = a.M[sg], row_bytes = a.nblk * 20u;
    const uint32_t b_begin = sp * a.blk_per_split, b_end = min(a.nblk, b_begin + a.blk_per_split);
    const uint32_t lane = threadIdx.x & 63u, lr = lane & 15u, lq = lane >> 4;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    // whole groups (J > 1: b_end - b_begin is a multiple of kGrp)
    const uint32_t groups = b_end > b_begin ? (b_end - b_begin + kGrp - 1u) / kGrp : 0u;
    const uint32_t g0 = groups * wave / kShortWaves, g1 = groups * (wave + 1u) / kShortWaves;

    const __amdgpu_buffer_rsrc_t wrs =
        __builtin_amdgcn_make_buffer_rsrc((void*)a.w[sg], 0, (int)(M * row_bytes), kBufFlagsG);
    uint32_t voff[RT];  // rows >= M lie past the end and read zeros
#pragma unroll
    for (int i = 0; i < RT; ++i) voff[i] = (m0 + 16u * i + lr) * row_bytes;
    const _Float16* xh = a.xh + lr * 32u + lq * 8u;
    const _Float16* xl = a.xl + lr * 32u + lq * 8u;

    uint32_t q[RT][5 * J];  // the lane's blocks: 4 nibble dwords and the scale each
    auto load_w = [&](uint32_t g) {
        const uint32_t b = b_begin + kGrp * g + J * lq;
        // J = 1: a block past the range reads zeros (a zero scale removes it)
        const uint32_t bo = (J > 1 || b < b_end) ? b * 20u : 0x80000000u;
#pragma unroll
        for (int i = 0; i < RT; ++i) {
#pragma unroll
            for (int c = 0; c < 5 * J / 4; ++c) {
                const u4v v = __builtin_amdgcn_raw_buffer_load_b128(wrs, voff[i] + bo + 16u * c, 0, 0);
#pragma unroll
                for (int e = 0; e < 4; ++e) q[i][4 * c + e] = v[e];
            }
#pragma unroll
            for (int c = 5 * J / 4 * 4; c < 5 * J; ++c)
                q[i][c] = __builtin_amdgcn_raw_buffer_load_b32(wrs, voff[i] + bo + 4u * c, 0, 0);
        }
    };
    h8v vh[2][JT], vl[2][JT];  // X of two blocks by turns
    auto load_x = [&](uint32_t blk, int set) {
        const size_t xo = (size_t)(b_begin + blk) * (kTok * 32u);
#pragma unroll
        for (int j = 0; j < JT; ++j) {
            vh[set][j] = *reinterpret_cast<const h8v*>(xh + xo + j * 512u);
            vl[set][j] = *reinterpret_cast<const h8v*>(xl + xo + j * 512u);
        }
    };
    f4v inner[RT][JT], outer[RT][JT];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < JT; ++j) {
            inner[i][j] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
            outer[i][j] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
        }
    uint32_t nb_in = 0;
    // Blocks of a group in the order the swaps give them: step n = 4*k + r
    // is block J*r + k (block k of lane group r).
    auto block_of = [](int n) { return (uint32_t)(J * (n & 3) + (n >> 2)); };
    const uint32_t x_last = (b_end - b_begin + 3u) & ~3u;  // staged blocks of the range (whole 4s)
    auto x_blk = [&](uint32_t g, int n) { return min(kGrp * g + block_of(n), x_last - 1u); };
    for (uint32_t g = g0; g < g1; ++g) {
        load_w(g);
        load_x(x_blk(g, 0), 0);
        load_x(x_blk(g, 1), 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < J; ++k) {
            float s[RT][4];
#pragma unroll
            for (int i = 0; i < RT; ++i) {
                swap_groups(q[i][5 * k], q[i][5 * k + 1], q[i][5 * k + 2], q[i][5 * k + 3]);
                const uint32_t v = q[i][5 * k + 4];
                const auto h = __builtin_amdgcn_permlane32_swap(v, v, false, false);
                const auto e = __builtin_amdgcn_permlane16_swap(h[0], h[0], false, false);
                const auto f = __builtin_amdgcn_permlane16_swap(h[1], h[1], false, false);
                s[i][0] = __uint_as_float(e[0]);
                s[i][1] = __uint_as_float(e[1]);
                s[i][2] = __uint_as_float(f[0]);
                s[i][3] = __uint_as_float(f[1]);
            }
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const int n = 4 * k + b, set = n & 1;
                h8v wf[RT];
#pragma unroll
                for (int i = 0; i < RT; ++i) wf[i] = unpack8(q[i][5 * k + b]);
#pragma unroll
                for (int j = 0; j < JT; ++j) {
                    f4v d[RT];
#pragma unroll
                    for (int i = 0; i < RT; ++i)
                        d[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vh[set][j], wf[i], f4v{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
                    for (int i = 0; i < RT; ++i) d[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vl[set][j], wf[i], d[i], 0, 0, 0);
#pragma unroll
                    for (int i = 0; i < RT; ++i)
#pragma unroll
                        for (int r = 0; r < 4; ++r) inner[i][j][r] = fmaf(s[i][b], d[i][r], inner[i][j][r]);
                }
                if (n + 2 < 4 * J) load_x(x_blk(g, n + 2), set);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        nb_in += kGrp;
        if (nb_in >= kInner) {
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
                for (int j = 0; j < JT; ++j) {
                    outer[i][j] += inner[i][j];
                    inner[i][j] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
                }
            nb_in = 0;
        }
    }
    // Register r of lane (lr, lq) holds token 4*lq + r of weight row lr.
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < JT; ++j) {
            const f4v v = outer[i][j] + inner[i][j];
#pragma unroll
            for (uint32_t r = 0; r < 4; ++r) red[wave][16u * j + 4u * lq + r][16 * i + lr] = v[r];
        }
    __syncthreads();
    for (uint32_t o = threadIdx.x; o < kTok * (kShortRows / 4); o += 64 * kShortWaves) {
        const uint32_t t = o / (kShortRows / 4), c = 4u * (o % (kShortRows / 4)), m = m0 + c;
        f4v p[kShortWaves];
#pragma unroll
        for (int k = 0; k < kShortWaves; ++k) p[k] = *reinterpret_cast<const f4v*>(&red[k][t][c]);
        const f4v v = ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
        if (t < a.T && m < M) {
            if (a.split > 1) {
                float* dst = a.part + ((size_t)sp * a.T + t) * a.part_ld + a.part_off[sg] + m;
                if ((a.part_ld & 3u) == 0 && (a.part_off[sg] & 3u) == 0 && m + 3 < M) {
                    *reinterpret_cast<f4v*>(dst) = v;
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (m + r < M) dst[r] = v[r];
                }
            } else {
                gemm_store4(a, sg, t, m, v);
            }
        }
    }
}

// Fixed-order sum of the K-split partials, scaled by 2^-e of the token.
__global__ __launch_bounds__(256) void k_gemm_reduce(const GemmArgs a) {
    const uint32_t ld = a.part_ld;
    const size_t n = (size_t)a.T * ld;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
        const uint32_t t = (uint32_t)(i / ld), c = (uint32_t)(i % ld);
        float v = a.part[i];
        uint32_t sp = 1;
        // 8 partials' loads in flight at a time; the sum stays sequential
        for (; sp + 8 <= a.split; sp += 8) {
            float w[8];
#pragma unroll
            for (uint32_t u = 0; u < 8; ++u) w[u] = a.part[(size_t)(sp + u) * n + i];
#pragma unroll
            for (uint32_t u = 0; u < 8; ++u) v += w[u];
        }
        for (; sp < a.split; ++sp) v += a.part[(size_t)sp * n + i];
        const uint32_t sg = seg_of_col(a, c);
        gemm_store(a, sg, t, c - a.part_off[sg], v);
    }
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
// Up to 32 tokens: workgroups that a launch aims at, and the blocks of a
// group (whole groups only: 16 or 8 where they divide the row and every wave
// gets one; 11000 x 20 x 1024 11.1 us with groups of 4, 14.8 with 16).
constexpr uint32_t kShortWgs = 192;
static uint32_t short_kb(uint32_t nblk) {
    return nblk % 16u == 0 && nblk >= 16u * kShortWaves ? 16u : nblk % 8u == 0 && nblk >= 8u * kShortWaves ? 8u : 4u;
}
constexpr uint32_t kGemmBT = 128;  // token rows per tile of k_gemm_q4_p

static uint32_t gemm_tpad(uint32_t T) { return (T + kGemmBT - 1) / kGemmBT * kGemmBT; }
static uint32_t gemm_npad(uint32_t N) { return (N + 127u) & ~127u; }  // whole K-steps of up to 4 blocks

// Launch plan of a GEMM over weight matrices of Ms[0..nseg) rows (each tiled
// on its own), T tokens and nblk blocks per row: the tile height (256 or 192
// rows), the K split (partials plus a reduction pass when > 1; each split
// keeps at least 32 blocks, and at most max_split), and, for whole-K
// launches, a cut: rows from `cut` on (counted over the matrices laid end to
// end) run in 192-row tiles in a second launch.  The cost model: a launch takes
// rounds x (20 us + K-steps x 1.93 us for 256-row tiles, 1.41 us for 192-row
// tiles), a round being up to 256 workgroups (one per CU); a reduction about 1
// us plus its traffic at 5 TB/s.  Its constants rank plans, they do not predict
// a launch: one round alone takes 12 us + 2.07 a step and 10.6 + 1.70 (512 and
// 2048 tokens, 16 to 64 steps; past those the clock falls), but plans made from
// these figures differ for 1.5 % of shapes, and of 22 such ten were 2 to 6 %
// slower (914|5709|1922 x 472 x 6592 167 -> 178 us) and two 1 % faster.
// From 33 to 128 tokens (one 128-token tile) the plan instead takes the
// smaller token tile of 64 or 128 holding them and the smallest K split (a
// power of two, each split keeping kInner blocks) that gives at least 224
// workgroups (448 for the 64-token tile, of which several fit a CU):
// measured on the Llama-3 shapes, within a few us of the best tile and split,
// 1.2-3.4x faster than 128-token tiles at K split <= 8.  Up to 32 tokens:
// k_gemm_q4_s.
struct GemmPlan {
    uint32_t bm;     // tile height of the (first) launch (up to 32 tokens: 64 or 32)
    uint32_t split;
    uint32_t cut;    // the total row count: one launch
    uint32_t bt;     // token tile: 128 (k_gemm_q4_p), 64 (k_gemm_q4), 32 or 16 (k_gemm_q4_s)
};

static uint32_t gemm_rounds(uint32_t wgs) { return (wgs + 255u) / 256u; }

static GemmPlan gemm_plan(const uint32_t* Ms, int nseg, uint32_t T, uint32_t nblk, uint32_t max_split) {
    const uint32_t n_tt = gemm_tpad(T) / kGemmBT;
    uint32_t mtot = 0;
    for (int i = 0; i < nseg; ++i) mtot += Ms[i];
    auto steps_of = [&](uint32_t sp) { return ((nblk + sp - 1) / sp + kKB - 1) / kKB; };
    // m-tiles of rows [r0, r1) of the matrices laid end to end
    auto tiles = [&](uint32_t r0, uint32_t r1, uint32_t bm) {
        uint32_t base = 0, n = 0;
        for (int i = 0; i < nseg; ++i) {
            const uint32_t lo = std::max(r0, base), hi = std::min(r1, base + Ms[i]);
            if (lo < hi) n += (hi - lo + bm - 1) / bm;
            base += Ms[i];
        }
        return n;
    };
    if (T <= kGemmBT) {
        if (T <= 32u) {
            // k_gemm_q4_s: its waves split K inside a workgroup; a second
            // split over workgroups only while the launch would leave CUs
            // idle and every wave keeps work.  64-row tiles where they then
            // still give workgroups enough: half the CUs with whole 320-byte
            // groups (9000 x 24 x 5120, 141 tiles: 27.3 us against 34.9 in
            // 32-row tiles; 6144 x 32 x 4096, 96 tiles: 18.5 against 15.6),
            // all of them with shorter ones (28672 x 24 x 4128, 448 tiles:
            // 39.1 against 44.5; 11000 x 12 x 8448, 172 tiles: 35.0 against
            // 30.2).
            const uint32_t bt = T <= 16u ? 16u : 32u, kb = short_kb(nblk);
            auto split_of = [&](uint32_t wgs, uint32_t min_blk) {
                uint32_t sp = 1;
                while (2 * sp <= max_split && wgs * sp < kShortWgs && nblk >= 2 * sp * min_blk) sp *= 2;
                return sp;
            };
            const uint32_t wgs64 = tiles(0, mtot, 64u), sp64 = split_of(wgs64, 6u * kb);
            if (wgs64 * sp64 >= (kb == 16u ? 128u : 256u)) return GemmPlan{64u, sp64, mtot, bt};
            return GemmPlan{32u, split_of(tiles(0, mtot, 32u), kShortWaves * kb), mtot, bt};
        }
        const uint32_t bt = T <= 64u ? 64u : 128u;
        const uint32_t wgs = tiles(0, mtot, 256u) * ((T + bt - 1) / bt);
        uint32_t sp = 1;
        // (each split keeps a whole inner sum of kInner blocks: with shorter
        // splits the sequential sum of the partials can exceed the AVX2
        // order's error at N = 4096)
        // (the small tiles fit two or more workgroups per CU: 448 of them
        // still run in one round)
        const uint32_t target = bt == 128u ? 224u : 448u;
        while (2 * sp <= max_split && wgs * sp < target && nblk >= 2 * sp * kInner) sp *= 2;
        return GemmPlan{256u, sp, mtot, bt};
    }
    max_split = std::min(max_split, 8u);
    auto launch_us = [&](uint32_t wgs, uint32_t bm, uint32_t steps) {
        return gemm_rounds(wgs) * (20.0 + steps * (bm == 256u ? 1.93 : 1.41));
    };
    GemmPlan best{256u, 1u, mtot, kGemmBT};
    double best_c = 1e30;
    for (uint32_t bm : {256u, 192u}) {
        for (uint32_t sp = 1; sp <= max_split; sp *= 2u) {
            if (sp > 1 && nblk / sp < 32u) break;
            double c = launch_us(tiles(0, mtot, bm) * n_tt * sp, bm, steps_of(sp));
            if (sp > 1) c += 1.0 + (double)(sp + 1) * T * mtot * 4.0 / 5e6;
            if (c < best_c) {
                best_c = c;
                best = GemmPlan{bm, sp, mtot, kGemmBT};
            }
        }
    }
    for (uint32_t r = 256u; r < mtot; r += 256u) {
        const double c = launch_us(tiles(0, r, 256u) * n_tt, 256u, steps_of(1)) +
                         launch_us(tiles(r, mtot, 192u) * n_tt, 192u, steps_of(1));
        if (c < best_c) {
            best_c = c;
            best = GemmPlan{256u, 1u, r, kGemmBT};
        }
    }
    return best;
}

// The K split a workspace is sized for: the plan of M_total rows as one
// matrix (a launch over several matrices takes at most this split).
static uint32_t gemm_ws_split(uint32_t M_total, uint32_t T, uint32_t nblk) {
    return gemm_plan(&M_total, 1, T, nblk, 32u).split;
}

static size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

size_t gemm_workspace_bytes(uint32_t N, uint32_t T, uint32_t M_total) {
    const size_t tp = gemm_tpad(T), np = gemm_npad(N);
    const uint32_t sp = gemm_ws_split(M_total, T, N / 32u);
    size_t b = 2 * align256(tp * np * 2) + align256(tp * 8);
    if (sp > 1) b += align256((size_t)sp * T * M_total * 4);
    return b;
}

// Arguments for rows [r0, r1) of the segments laid end to end, in m-tiles of
// `bm` rows (a range may cut segments: its pieces point into them).
static void gemm_rows_args(GemmArgs& a, const GemmSegs& sg, uint32_t r0, uint32_t r1, uint32_t bm,
                           uint32_t row_bytes) {
    uint32_t base = 0, mt = 0, n = 0;
    for (int i = 0; i < sg.n; ++i) {
        const uint32_t lo = std::max(r0, base), hi = std::min(r1, base + sg.M[i]);
        if (lo < hi) {
            const uint32_t off = lo - base;
            a.w[n] = sg.w[i] + (size_t)off * row_bytes;
            a.y[n] = sg.y[i] + off;
            a.res[n] = sg.res[i] ? sg.res[i] + off : nullptr;
            a.M[n] = hi - lo;
            a.ld[n] = sg.M[i];
            mt += (hi - lo + bm - 1) / bm;
            a.mt_end[n] = mt;
            ++n;
        }
        base += sg.M[i];
    }
    a.nseg = n;
}

// k_gemm_q4_s with groups of kb = 4*J blocks and tiles of 16*RT rows.
template <int JT, int RT>
static void launch_short(uint32_t kb, uint32_t grid, hipStream_t s, const GemmArgs& g) {
    const dim3 wg(64 * kShortWaves);
    if (kb == 16u)
        hipLaunchKernelGGL((k_gemm_q4_s<JT, 4, RT>), dim3(grid), wg, 0, s, g);
    else if (kb == 8u)
        hipLaunchKernelGGL((k_gemm_q4_s<JT, 2, RT>), dim3(grid), wg, 0, s, g);
    else
        hipLaunchKernelGGL((k_gemm_q4_s<JT, 1, RT>), dim3(grid), wg, 0, s, g);
}

hipError_t launch_gemm_ex(const GemmSegs& sg, const GemmRows& in, void* ws, hipStream_t s, GemmDeferred* defer_out) {
    const uint32_t N = in.N, T = in.T;
    const int nseg = sg.n;
    if (defer_out) defer_out->valid = false;
    const GemmDeferred* from = (in.from && in.from->valid) ? in.from : nullptr;
    if (nseg < 1 || nseg > kGemmMaxSeg || T == 0 || N == 0 || N % 32 != 0 || !(in.x || from))
        return hipErrorInvalidValue;
    if (gemm_npad(N) > 8u * 256u * kXpMaxGroups) return hipErrorInvalidValue;  // the row conversion's register tile
    if (in.norm_w && in.u) return hipErrorInvalidValue;
    const uint32_t tp = gemm_tpad(T), np = gemm_npad(N);
    const uint32_t row_bytes = (N / 32u) * 20u;
    uint8_t* p = static_cast<uint8_t*>(ws);
    const size_t plane = align256((size_t)tp * np * 2);
    GemmArgs a{};
    a.xh = reinterpret_cast<_Float16*>(p);
    a.xl = reinterpret_cast<_Float16*>(p + plane);
    a.meta = reinterpret_cast<float2*>(p + 2 * plane);
    float* part = reinterpret_cast<float*>(p + 2 * plane + align256((size_t)tp * 8));
    uint32_t mtot = 0;
    for (int i = 0; i < nseg; ++i) {
        // Weight offsets are 32-bit buffer offsets.
        if (sg.M[i] == 0 || (uint64_t)sg.M[i] * row_bytes >= (1ull << 31)) return hipErrorInvalidValue;
        a.part_off[i] = mtot;
        mtot += sg.M[i];
    }
    const GemmPlan plan = gemm_plan(sg.M, nseg, T, N / 32u, gemm_ws_split(mtot, T, N / 32u));
    a.nblk = N / 32;
    a.T = T;
    a.N_pad = np;
    a.n_tt = (T + plan.bt - 1) / plan.bt;
    a.split = plan.split;
    const bool is_short = plan.bt <= 32u;                   // k_gemm_q4_s
    const uint32_t kb = is_short ? short_kb(a.nblk) : (uint32_t)kKB;  // the kernel's K-step (short: its groups)
    a.blk_per_split = ((a.nblk + a.split - 1) / a.split + kb - 1) / kb * kb;
    a.part = part;
    a.part_ld = mtot;
    // The XCD-aware order needs the token-tile count to divide the 8 XCDs.
    a.xcd_map = (8u % a.n_tt == 0 && !is_short) ? 1u : 0u;
    GemmXIn xin{in.x, in.u, in.norm_w, in.eps, nullptr, 0u, nullptr, nullptr};
    if (from) {
        // The producer's partials lie beyond its own staged rows and scales;
        // in a shared workspace this launch's rows and scales must end at or
        // before those (a staged row no longer than the producer's).
        if (!from->y || from->T != T || from->M != N || (from->ws == ws && np > from->n_pad))
            return hipErrorInvalidValue;
        xin.x = from->y;
        xin.part = from->part;
        xin.split = from->split;
        xin.pmeta = from->meta;
        xin.res = from->res;
    }
    // the smallest register tile holding the row: groups of 8 per thread
    const uint32_t per = (np / 8 + 255) / 256;
    auto xprep = per <= 2 ? k_gemm_xprep<2> : per <= 4 ? k_gemm_xprep<4> : per <= 8 ? k_gemm_xprep<8>
                                                                             : k_gemm_xprep<16>;
    // the rows the token tiles read (zeros past T): all tp rows for the
    // 128-token tile, fewer for the small ones
    const uint32_t rows = std::min(tp, a.n_tt * plan.bt);
    hipLaunchKernelGGL(xprep, dim3(rows), dim3(256), 0, s, xin, T, N, np, is_short ? plan.bt : 0u,
                       const_cast<_Float16*>(a.xh), const_cast<_Float16*>(a.xl), const_cast<float2*>(a.meta));
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    // rows [r0, r1) in tiles of bm rows
    auto launch = [&](uint32_t r0, uint32_t r1, uint32_t bm) -> hipError_t {
        GemmArgs g = a;
        gemm_rows_args(g, sg, r0, r1, bm, row_bytes);
        const uint32_t pairs = g.mt_end[g.nseg - 1] * g.split * g.n_tt;
        const uint32_t grid = g.xcd_map ? (pairs + 7u) / 8u * 8u : pairs;
        if (plan.bt == 16u)
            plan.bm == 64u ? launch_short<1, 4>(kb, grid, s, g) : launch_short<1, 2>(kb, grid, s, g);
        else if (plan.bt == 32u)
            plan.bm == 64u ? launch_short<2, 4>(kb, grid, s, g) : launch_short<2, 2>(kb, grid, s, g);
        else if (plan.bt == 64u)
            hipLaunchKernelGGL(k_gemm_q4, dim3(grid), dim3(64 * kGemmWM), 0, s, g);
        else if (bm == 256u)
            hipLaunchKernelGGL(k_gemm_q4_p<4>, dim3(grid), dim3(512), 0, s, g);
        else
            hipLaunchKernelGGL(k_gemm_q4_p<3>, dim3(grid), dim3(512), 0, s, g);
        return hipGetLastError();
    };
    if (plan.cut < mtot) {
        e = launch(0, plan.cut, 256u);
        if (e != hipSuccess) return e;
        return launch(plan.cut, mtot, 192u);
    }
    e = launch(0, mtot, plan.bm);
    if (e != hipSuccess || a.split == 1) return e;
    bool no_res = true;
    for (int i = 0; i < nseg; ++i) no_res = no_res && sg.res[i] == nullptr;
    if (defer_out && (nseg == 1 || no_res) && (mtot & 3u) == 0) {
        // the next GEMM's row conversion sums the partials
        defer_out->valid = true;
        defer_out->part = part;
        defer_out->split = a.split;
        defer_out->T = T;
        defer_out->M = mtot;
        defer_out->meta = a.meta;
        defer_out->res = sg.res[0];
        defer_out->y = nseg == 1 ? sg.y[0] : nullptr;  // several matrices: the consumer knows the layout
        defer_out->ws = ws;
        defer_out->n_pad = np;
        return hipSuccess;
    }
    // the reduction reads the partials by column of the whole row set
    gemm_rows_args(a, sg, 0, mtot, plan.bm, row_bytes);
    const size_t n = (size_t)T * mtot;
    const uint32_t rg = (uint32_t)std::min<size_t>((n + 255) / 256, 4096);
    hipLaunchKernelGGL(k_gemm_reduce, dim3(rg), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_gemm(const uint8_t* const* w, float* const* y, const uint32_t* M, int nseg, uint32_t N,
                       const float* X, uint32_t T, void* ws, hipStream_t s) {
    if (nseg < 1 || nseg > kGemmMaxSeg) return hipErrorInvalidValue;
    GemmSegs sg{};
    sg.n = nseg;
    for (int i = 0; i < nseg; ++i) {
        sg.w[i] = w[i];
        sg.y[i] = y[i];
        sg.M[i] = M[i];
    }
    GemmRows in{};
    in.x = X;
    in.T = T;
    in.N = N;
    return launch_gemm_ex(sg, in, ws, s);
}

}  // namespace qh
