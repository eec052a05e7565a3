// gemm_w8a32.hip -- fp32 activations times packed E4M3 weights (W8A32) on the
// bf16 matrix cores, at fp32 accuracy.
//
// Every E4M3 weight is a bf16 value, and every finite fp32 activation is the
// sum of three: hi, its upper 16 bits; mid, the upper 16 bits of x - hi; and
// lo, what is left (24 bits in three pieces of 8; both differences are
// exact).  A piece times a weight, 8 bits by 4, is exact in the matrix unit,
// which accumulates in fp32, so hi, mid and lo through three
// v_mfma_f32_16x16x32_bf16 give sum_k x_k w_k with fewer roundings than an fma
// chain over k has (one per 32 products; error against 64 bits at 128 x 11008
// x 4096 1.5e-7 of the norm, 3.3e-7 with the fma chains).  Three of them take
// 48 cycles of a SIMD for 8192 multiply-adds; v_fma_f32 takes 512.  The
// activations are split times 2^16, so that bf16's smallest value, 2^-133,
// holds the last bit of every one, subnormals among them, and the sums are
// scaled back.
//
// What is left is to feed them.  A workgroup owns 16*MB rows and P 64-column
// panels and splits K in KS parts, one wavefront to a panel and part, that
// sum their tiles through LDS at the end.  The weights go straight to
// registers, each byte to one wavefront; the activations pass through LDS,
// split once per workgroup (6.5 VALU operations each, beside 12 MFMAs per 16
// of them per panel), 64 k a step.  The K split, and with it the order of a
// row's sum, depends on M and N.
//
// An activation that is inf, NaN or from 2^112 on leaves NaN in mid and lo.
// The wavefronts test their sums for NaN and infinities once, at the end, and
// if there is one the workgroup runs twice again: over the activations below
// 2^-64 as before, and, adding to those sums, over the others without the
// factor and with mid = lo = 0 where they are not finite: then inf * w is the
// fma chain's, and what is small keeps its bits beside it.
#include <algorithm>

#include "lcml_internal.hpp"

namespace lcml {
namespace {

constexpr uint32_t kOOB = 0x80000000u;  // buffer offset past every extent: loads return zeros
constexpr int kRsrcFlags = 0x00020000;  // raw buffer resource word 3

typedef float v4f __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));
typedef uint32_t u2 __attribute__((ext_vector_type(2)));

// four activations -> three times four bf16
struct Split {
    u2 hi, mid, lo;
};

// the upper halves of a (low 16 bits of the result) and b
__device__ inline uint32_t upper2(float a, float b) {
    return __builtin_amdgcn_perm(f32_bits(b), f32_bits(a), 0x07060302u);
}

// Which activations a run over K takes, and how.  bf16 ends at 2^-133, fp32 at
// 2^-149: times 2^16 no bit of an activation is lost.
enum Run {
    kAll,    // every one, times 2^16 (NaN in the lower pieces where that is not finite)
    kSmall,  // those below 2^-64, times 2^16
    kRest,   // the others as they are, inf and NaN among them
};
constexpr float kUp = 0x1p16f, kDown = 0x1p-16f, kSmallMax = 0x1p-64f;

template <Run RUN>
__device__ inline Split split4(f4 x) {
    float h[4], m[4], l[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const bool small = fabsf(x[i]) < kSmallMax;
        const float v = RUN == kAll ? x[i] * kUp : RUN == kSmall ? (small ? x[i] * kUp : 0.0f) : small ? 0.0f : x[i];
        h[i] = bits_f32(f32_bits(v) & 0xffff0000u);
        const float r = v - h[i];
        m[i] = bits_f32(f32_bits(r) & 0xffff0000u);
        l[i] = r - m[i];
        if constexpr (RUN == kRest)
            if (!(fabsf(v) <= 3.4028235e38f)) {
                h[i] = v != v ? bits_f32(0x7fc00000u) : v;  // a NaN's upper half may be an infinity's
                m[i] = l[i] = 0.0f;
            }
    }
    return {u2{upper2(h[0], h[1]), upper2(h[2], h[3])}, u2{upper2(m[0], m[1]), upper2(m[2], m[3])},
            u2{upper2(l[0], l[1]), upper2(l[2], l[3])}};
}

// The wavefronts are KS parts of K times P panels.  The wavefronts of a K
// part bring its activations together, 16*MB rows of 64 k per step, split
// them and lay the three pieces in LDS, rows of 64 bf16 in PITCH bytes (a
// fragment's 16 rows in distinct 16-byte bank slots); straight to registers,
// an MFMA operand's lanes lie in 16 rows and each 16-byte load takes 64 cache
// line lookups, which bounded the kernel at 68 us on 128 x 11008 x 4096.
// Step by step: activations two steps ahead in registers, pieces one step
// ahead in the other LDS buffer, weights one step ahead in registers (three
// ahead measured the same).  Lane l
// holds row (of A) or column (of a 16-column block of B) l % 16 and
// k = (l / 16)*16 + 0..15 of a step, eight per MFMA: one 16-byte chunk of the
// packed weights.
// VEC: 16-byte loads of the activations (a 16-byte aligned, lda and K
// multiples of 4), else 4-byte ones.  All loads are buffer loads with out of
// range lanes past the extent, so none sits under a branch and the waits
// count.  The leading scalar arguments arrive in SGPRs
// (-amdgpu-kernarg-preload-count).
template <int MB, int P, int KS, bool VEC>
__global__ __launch_bounds__(P *KS * 64, P == 2 && VEC ? 4 : 1) void k_gemm_w8a32(const uint8_t *bp, const float *a, int lda, int M, int K,
                                                            int kc, int npanels, int rg, Epilogue e) {
    constexpr int ROWS = 16 * MB, PITCH = 144, PIECE = ROWS * PITCH, BUF = 3 * PIECE;
    constexpr int XL = (ROWS * 16 + 64 * P - 1) / (64 * P);  // float4s of a step per thread
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int part = wave / P, pt = tid - part * (64 * P);
    // workgroup -> (panels, row group): the row groups of a panel on one XCD
    int t = (int)blockIdx.x;
    if (rg > 1) {
        const int nwg = (int)gridDim.x, q = nwg >> 3, r = nwg & 7, x = t & 7;
        t = x * q + (x < r ? x : r) + (t >> 3);
    }
    const int cgrp = rg > 1 ? t / rg : t, row0 = rg > 1 ? (t - cgrp * rg) * ROWS : 0;
    const int panel = cgrp * P + wave % P;
    const int ns = kc / 4;  // steps of 64 k, split over the parts; every part runs `steps`
    const int s_begin = (int)((uint32_t)(ns * part) / KS), s_end = (int)((uint32_t)(ns * (part + 1)) / KS);
    const int steps = (ns + KS - 1) / KS;

    const __amdgpu_buffer_rsrc_t br = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(bp + (size_t)panel * (size_t)kc * 1024), 0, panel < npanels ? kc * 1024 : 0, kRsrcFlags);
    const uint32_t b_lane = (uint32_t)(lane & 15) * 16u + (uint32_t)(lane >> 4) * 1024u;
    const int rows = min(ROWS, M - row0);  // this row group's activations
    const __amdgpu_buffer_rsrc_t ar = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(a + (int64_t)row0 * lda), 0, ((rows - 1) * lda + K) * 4, kRsrcFlags);
    uint8_t *const buf = smem + part * 2 * BUF;

    v4f acc[MB][4], low[MB][4];  // the sums of the upper pieces, and of the two lower ones
    f4 x[XL];
    u4 w[2][4];
    // float4 pt + 64*P*u of the step: row (pt + 64 P u)/16, k 4*(pt % 16)
    auto load_x = [&](int s) {
#pragma unroll
        for (int u = 0; u < XL; ++u) {
            const int r = (pt >> 4) + 4 * P * u, k = s * 64 + 4 * (pt & 15);
            const bool ok = s < s_end && r < rows;  // (rows <= ROWS)
            const uint32_t o = (uint32_t)(r * lda + k) * 4u;
            if constexpr (VEC) {
                x[u] = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(ar, (int)(ok && k < K ? o : kOOB), 0, 0));
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    x[u][i] = __builtin_bit_cast(
                        float, __builtin_amdgcn_raw_buffer_load_b32(ar, (int)(ok && k + i < K ? o + 4u * i : kOOB), 0, 0));
            }
        }
    };
    auto load_w = [&](u4 (&w)[4], int s) {
        const uint32_t o = s < s_end ? b_lane + (uint32_t)s * 4096u : kOOB;
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] = __builtin_amdgcn_raw_buffer_load_b128(br, (int)(o + j * 256), 0, 0);
    };
    auto put_x = [&](int b, auto which) {
#pragma unroll
        for (int u = 0; u < XL; ++u) {
            if (ROWS * 16 % (64 * P) != 0 && (pt >> 4) + 4 * P * u >= ROWS) continue;
            uint8_t *to = buf + b * BUF + ((pt >> 4) + 4 * P * u) * PITCH + (pt & 15) * 8;
            const Split s = split4<decltype(which)::value>(x[u]);
            *reinterpret_cast<u2 *>(to) = s.hi;
            *reinterpret_cast<u2 *>(to + PIECE) = s.mid;
            *reinterpret_cast<u2 *>(to + 2 * PIECE) = s.lo;
        }
    };
    auto compute = [&](const u4 (&w)[4], int b) {
        const uint8_t *pa = buf + b * BUF + (lane & 15) * PITCH + (lane >> 4) * 32;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            bf16x8 b16[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) b16[j] = q ? e4m3x8_to_bf16(w[j].z, w[j].w) : e4m3x8_to_bf16(w[j].x, w[j].y);
            // a piece at a time over all tiles: an MFMA's accumulator is the
            // one of 4*MB before it.  The lower pieces' sums are kept apart:
            // in one accumulator every step would round the large sum three
            // times instead of once.
#pragma unroll
            for (int p = 2; p >= 0; --p) {
                bf16x8 a16[MB];
#pragma unroll
                for (int mb = 0; mb < MB; ++mb)
                    a16[mb] = *reinterpret_cast<const bf16x8 *>(pa + p * PIECE + mb * 16 * PITCH + q * 16);
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int mb = 0; mb < MB; ++mb)
                    {
                        v4f &to = p ? low[mb][j] : acc[mb][j];
                        to = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a16[mb], b16[j], to, 0, 0, 0);
                    }
            }
        }
    };
    auto run = [&](auto which) {
        constexpr Run RUN = decltype(which)::value;
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (RUN != kRest) acc[mb][j] = v4f{0.f, 0.f, 0.f, 0.f};  // kRest adds to kSmall's sums
                low[mb][j] = v4f{0.f, 0.f, 0.f, 0.f};
            }
        load_x(s_begin);
        load_w(w[0], s_begin);
        put_x(0, which);
        load_x(s_begin + 1);
        __syncthreads();
        for (int i0 = 0; i0 < steps; i0 += 2) {
#pragma unroll
            for (int d = 0; d < 2; ++d) {
                const int i = i0 + d;
                if (i >= steps) break;
                load_w(w[1 - d], s_begin + i + 1);
                put_x(1 - d, which);
                load_x(s_begin + i + 2);
                __builtin_amdgcn_sched_barrier(0);
                compute(w[d], d);
                __syncthreads();
            }
        }
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                acc[mb][j] += low[mb][j];
                if (RUN != kRest) acc[mb][j] *= kDown;
            }
    };
    run(std::integral_constant<Run, kAll>{});
    float nan = 0.0f;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) nan = fmaf(acc[mb][j][r], 0.0f, nan);
    // (an infinite sum, 0 * inf, counts too: the factor may have made it)
    if (__builtin_expect(__syncthreads_or(nan != nan), 0)) {
        run(std::integral_constant<Run, kSmall>{});
        run(std::integral_constant<Run, kRest>{});
    }

    // the parts' sums through LDS, [wave][block][register][lane]: register r
    // of lane l of block j is row (l/16)*4 + r, column l%16
    float(*red)[4][4][64] = reinterpret_cast<float(*)[4][4][64]>(smem);
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        if (mb) __syncthreads();  // the previous block's sums are read
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) red[wave][j][r][lane] = acc[mb][j][r];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 16 / KS; ++i) {
            const int o = tid + i * P * KS * 64, l = o & 63, r = (o >> 6) & 3, j = (o >> 8) & 3, pw = o >> 10;
            const int64_t row = row0 + mb * 16 + (l >> 4) * 4 + r, col = (int64_t)(cgrp * P + pw) * 64 + j * 16 + (l & 15);
            if (row >= e.M || col >= e.N) continue;
            float v = 0.0f;
#pragma unroll
            for (int k = 0; k < KS; ++k) v += red[k * P + pw][j][r][l];
            epi_store(e, row, col, epi_value(e, epi_scale(e, 1.0f, col), row, col, v));
        }
    }
}

// The shapes: 16 rows x 1 panel with K in 8 parts, 16 x 2 in 4, 32 x 3 in 4.
// A round of up to 256 workgroups (one per CU) takes 12.5, 15.5 and 34 us at
// K = 4096, all in proportion to K, so the larger shapes win where the work
// fills their rounds: N = 11008 at M = 16: 15 us (19, 30 with the other two),
// M = 64: 28 us (40, 33), M = 128: 35 us (73, 47), M = 512: 141 us (274, 161).
// Wider still (32 x 4 in 2): 48 us at M = 128, the same at M = 512.
enum Shape { k16x1, k16x2, k32x3 };
Shape w8a32_shape(int64_t M, int64_t panels) {
    auto rounds = [&](int64_t rows, int64_t p) {
        return (double)(((M + rows - 1) / rows * ((panels + p - 1) / p) + 255) / 256);
    };
    const double c1 = 12.5 * rounds(16, 1), c2 = 15.5 * rounds(16, 2), c3 = 34.0 * rounds(32, 3);
    return c3 <= c2 && c3 <= c1 ? k32x3 : c2 < c1 ? k16x2 : k16x1;
}

bool w8a32_vec(const float *a, int64_t lda, int64_t K) {
    return (reinterpret_cast<uintptr_t>(a) & 15) == 0 && lda % 4 == 0 && K % 4 == 0;
}

}  // namespace

// Against the vector-ALU kernel, which starts a workgroup per row and panel
// (per two or four rows from 512 and 1024 of them) and needs no barriers, in
// us (vector ALU / matrix cores):
//   * up to 512 workgroups it stays, whatever K: N = 212, K = 6722, M = 56
//     11.0 / 30.9; N = 982, K = 4333, M = 30 11.3 / 21.3; N = 1495, K = 4501,
//     M = 12 10.8 / 18.2.  Few rows of many panels read the weights rather than
//     share them: N = 11008, K = 4096, M = 1 8.2 / 15, 2 17.3 / 15.1; N = 2888,
//     K = 4628, M = 8 16.2 / 13.6; N = 2882, K = 3550, M = 9 12.8 / 13.5;
//   * up to 1024 with little work: N = 1007, K = 730 (4-byte loads), M = 61
//     6.9 / 7.8; N = 150, K = 764 (16-byte loads), M = 339 8.2 / 5.9; N = 21, K =
//     2655, M = 812 18.2 / 15.4; N = 256, K = 784, M = 200 8.7 / 5.9;
//   * up to 2048 with next to none: N = 2500, K = 16, M = 39 4.5 / 5.0; N = 152,
//     K = 60, M = 391 7.6 / 4.9.
bool w8a32_mfma_wins(int64_t M, int64_t N, int64_t K, const float *a, int64_t lda) {
    const int64_t panels = pad_to(N, kPanelCols) / 64;
    const double w = (double)panels * (double)M, wk = w * (double)K;
    if (w <= 512 && !(M <= 8 && w > 256 && wk > 1.1e6)) return false;
    if (w <= 1024 && wk <= (w8a32_vec(a, lda, K) ? 3e5 : 7.5e5)) return false;
    if (w <= 2048 && wk <= 3e4) return false;
    // a row group's activations, a panel, and the grid at 16 rows per
    // workgroup of 512: a launch of 2^32 work items or more runs with that
    // number modulo 2^32 and reports no error
    return (32 * lda + K) * 4 < ((int64_t)1 << 31) && pad_to(K, kPackK) * 64 < ((int64_t)1 << 31) &&
           M < ((int64_t)1 << 31) - 64 && panels * ((M + 15) / 16) < ((int64_t)1 << 23);
}

hipError_t launch_gemm_w8a32(int64_t M, int64_t N, int64_t K, const float *a, int64_t lda, const uint8_t *bp,
                             const Epilogue &e, hipStream_t s) {
    const int64_t panels = pad_to(N, kPanelCols) / 64, Kp = pad_to(K, kPackK);
    const bool vec = w8a32_vec(a, lda, K);
    auto go = [&](auto mbv, auto pv, auto ksv, auto v) -> hipError_t {
        constexpr int MB = decltype(mbv)::value, P = decltype(pv)::value, KS = decltype(ksv)::value;
        constexpr bool V = decltype(v)::value;
        constexpr int kLds = std::max(KS * 2 * 3 * 16 * MB * 144, KS * P * 4 * 4 * 64 * 4);
        const int64_t rg = (M + 16 * MB - 1) / (16 * MB), cgrps = (panels + P - 1) / P;
        static std::atomic<uint64_t> lds_set{0};
        if (hipError_t err = ensure_dynamic_lds(reinterpret_cast<const void *>(k_gemm_w8a32<MB, P, KS, V>), kLds, lds_set);
            err != hipSuccess)
            return err;
        hipLaunchKernelGGL((k_gemm_w8a32<MB, P, KS, V>), dim3((unsigned)(cgrps * rg)), dim3(P * KS * 64), kLds, s, bp, a,
                           (int)lda, (int)M, (int)K, (int)(Kp / 16), (int)panels, (int)rg, e);
        return hipGetLastError();
    };
    auto by_vec = [&](auto mbv, auto pv, auto ksv) {
        return vec ? go(mbv, pv, ksv, std::true_type{}) : go(mbv, pv, ksv, std::false_type{});
    };
    using N1 = std::integral_constant<int, 1>;
    using N2 = std::integral_constant<int, 2>;
    using N3 = std::integral_constant<int, 3>;
    using N4 = std::integral_constant<int, 4>;
    using N8 = std::integral_constant<int, 8>;
    switch (w8a32_shape(M, panels)) {
    case k16x1: return by_vec(N1{}, N1{}, N8{});
    case k16x2: return by_vec(N1{}, N2{}, N4{});
    default: return by_vec(N2{}, N3{}, N4{});
    }
}

}  // namespace lcml
