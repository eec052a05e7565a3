// gemm_rows.hip -- medium-M FP8 GEMM (17 to a few hundred rows) behind a
// dynamic quantisation that lays the activations out for it.
//
// A workgroup takes 32 to 96 rows and 16 to 64 columns; its 8 wavefronts split
// K, read weights and activations straight into registers as in the small-M
// kernel, and sum their partial tiles through LDS.  What made that slow from row-major activations is
// the load: an MFMA operand's lanes lie in 16 rows, and every 16-byte load of
// them takes 64 cache-line lookups.  So the quantiser writes the activations
// in blocks of 16 rows, 16-byte k-chunk by chunk, the rows of a chunk side by
// side (the last block with as many rows as there are, so that M x K codes
// take M*K bytes): then an operand's load is four runs of 256 bytes.
// The products are E4M3 widened exactly to bf16, v_mfma_f32_16x16x32_bf16, with
// the K split and order of the small-M kernel, so the sums equal its sums.
//
// With the quantiser, against the small-M kernel or the 128x128 tiles on
// row-major codes (us): N = K = 4096: M = 32 14.8 -> 10.4, 64 15.1 -> 12.3, 256
// 22.2 -> 19.4; N = 4096, K = 11008: M = 32 28.3 -> 18.2, 100 32.6 -> 27.7, 256
// 46.4 -> 37.7, 512 82.3 -> 64.5; N = 12288, K = 4096: M = 64 23.9 -> 20.0, 100
// 31.7 -> 28.1, 256 43.1 -> 43.4.
#include <algorithm>

#include "lcml_internal.hpp"

namespace lcml {
namespace {

constexpr uint32_t kOOB = 0x80000000u;  // buffer offset past every extent: loads return zeros
constexpr int kRsrcFlags = 0x00020000;  // raw buffer resource word 3
constexpr int kWaves = 8;
constexpr int kThreads = 256;

typedef float v4f __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));

// The encode half of a dynamic quantisation into 16-row blocks (K % 16 == 0, x
// 16-byte aligned): a thread encodes one 16-byte chunk of a row, a
// wavefront 4 chunks of 16 rows (reads of 256, writes of 256 contiguous bytes).
// The loads are issued before the partial maxima are reduced.
__global__ __launch_bounds__(kThreads) void k_quantize_rows(const float *__restrict__ x, uint8_t *__restrict__ y, int M,
                                                            int K, const uint32_t *__restrict__ part, int npart,
                                                            float *__restrict__ scale_out) {
    __shared__ float red[kThreads / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int kc = K / 16, quads = (kc + 3) / 4;
    const int64_t unit = (int64_t)blockIdx.x * (kThreads / 64) + wave;  // (row block, four chunks)
    const int blk = (int)(unit / quads), c = (int)(unit - (int64_t)blk * quads) * 4 + (lane >> 4);
    const int rb = min(16, M - blk * 16), r = lane & 15;
    const bool ok = r < rb && c < kc;
    f4 v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
        v[i] = ok ? reinterpret_cast<const f4 *>(x)[(((int64_t)blk * 16 + r) * K + c * 16) / 4 + i] : f4{0.f, 0.f, 0.f, 0.f};
    const float s = scale_from_partials<kThreads>(part, npart, red);
    if (scale_out && blockIdx.x == 0 && threadIdx.x == 0) *scale_out = s;
    const Recip d = make_recip(s);
    u4 code;
#pragma unroll
    for (int i = 0; i < 4; ++i) code[i] = quantize4(v[i].x, v[i].y, v[i].z, v[i].w, d);
    if (ok) reinterpret_cast<u4 *>(y)[(int64_t)blk * kc * 16 + (int64_t)c * rb + r] = code;
}

// The leading scalar arguments arrive in SGPRs (-amdgpu-kernarg-preload-count).
// All loads are buffer loads with out of range lanes past the extent, so none
// sits under a branch and the waits count.
template <int MB, int NB>
__global__ __launch_bounds__(kWaves * 64) void k_gemm_rows(const uint8_t *bp, const uint8_t *a, int M, int K, int kc,
                                                           int nkb, int rg, Epilogue e) {
    static_assert(NB == 1 || NB == 2 || NB == 4, "16-column blocks of one panel");
    __shared__ float red[kWaves][NB][4][64];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // workgroup -> (columns, row group): the row groups of a panel on one XCD
    int t = (int)blockIdx.x;
    if (rg > 1) {
        const int nwg = (int)gridDim.x, q = nwg >> 3, r = nwg & 7, x = t & 7;
        t = x * q + (x < r ? x : r) + (t >> 3);
    }
    const int cgrp = rg > 1 ? t / rg : t, rblk0 = rg > 1 ? (t - cgrp * rg) * MB : 0, blk0 = cgrp * NB;
    const int kb_begin = (int)((uint32_t)(nkb * wave) / kWaves), kb_end = (int)((uint32_t)(nkb * (wave + 1)) / kWaves);

    const __amdgpu_buffer_rsrc_t br = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(bp + (size_t)(blk0 >> 2) * (size_t)kc * 1024), 0, kc * 1024, kRsrcFlags);
    const uint32_t b_lane =
        (uint32_t)(lane & 15) * 16u + (uint32_t)(lane >> 4) * 2048u + (NB < 4 ? (uint32_t)(blk0 & 3) * 256u : 0u);
    // the row blocks' codes: chunk c of row r of a block of rb rows at
    // (c * rb + r) * 16 from the block's start
    const __amdgpu_buffer_rsrc_t ar = __builtin_amdgcn_make_buffer_rsrc((void *)a, 0, M * K, kRsrcFlags);
    const int arow = lane & 15, achunk = (lane >> 4) * 2, kchunks = K / 16;
    const int rlast = (M + 15) / 16 - 1, rb_last = M - rlast * 16;

    v4f acc[MB][NB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[mb][j] = v4f{0.f, 0.f, 0.f, 0.f};
    // half a 128-k block: one 16-byte chunk per lane and tile, two MFMAs' worth
    struct Frag {
        u4 b[NB], a[MB];
    };
    auto load = [&](Frag &f, int kb, int h) {
        const bool in = kb < kb_end;
        const uint32_t o = in ? b_lane + (uint32_t)kb * 8192u : kOOB;
#pragma unroll
        for (int j = 0; j < NB; ++j)
            f.b[j] = __builtin_amdgcn_raw_buffer_load_b128(br, (int)(o + j * 256 + h * 1024), 0, 2);
        __builtin_amdgcn_sched_barrier(0);
        const int c = kb * 8 + achunk + h;
        const bool cok = in && c < kchunks;
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
            const int blk = rblk0 + mb, rb = blk < rlast ? 16 : blk == rlast ? rb_last : 0;
            const uint32_t ao = (uint32_t)blk * 16u * (uint32_t)K + (uint32_t)(c * rb + arow) * 16u;
            f.a[mb] = __builtin_amdgcn_raw_buffer_load_b128(ar, (int)(cok && arow < rb ? ao : kOOB), 0, 0);
        }
    };
    auto compute = [&](const Frag &f) {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            bf16x8 b16[NB];
#pragma unroll
            for (int j = 0; j < NB; ++j) b16[j] = q ? e4m3x8_to_bf16(f.b[j].z, f.b[j].w) : e4m3x8_to_bf16(f.b[j].x, f.b[j].y);
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) {
                const bf16x8 a16 = q ? e4m3x8_to_bf16(f.a[mb].z, f.a[mb].w) : e4m3x8_to_bf16(f.a[mb].x, f.a[mb].y);
#pragma unroll
                for (int j = 0; j < NB; ++j)
                    acc[mb][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a16, b16[j], acc[mb][j], 0, 0, 0);
            }
        }
    };
    // each half is loaded a block ahead of its use (past the end: zeros, no
    // memory traffic)
    Frag f0, f1;
    load(f0, kb_begin, 0);
    load(f1, kb_begin, 1);
    for (int kb = kb_begin; kb < kb_end; ++kb) {
        __builtin_amdgcn_sched_barrier(0);
        compute(f0);
        __builtin_amdgcn_sched_barrier(0);
        load(f0, kb + 1, 0);
        __builtin_amdgcn_sched_barrier(0);
        compute(f1);
        __builtin_amdgcn_sched_barrier(0);
        load(f1, kb + 1, 1);
    }

    // register r of lane l of block j: row (l/16)*4 + r, column l%16
    const float a_s = e.a_scale ? e.a_scale[0] : 1.0f;
    constexpr int OUT = (NB * 256 + kWaves * 64 - 1) / (kWaves * 64);
    float bsc[OUT];
#pragma unroll
    for (int i = 0; i < OUT; ++i) {
        const int o = tid + i * kWaves * 64;
        const int64_t col = (int64_t)(blk0 + (o >> 8)) * 16 + (o & 15);
        bsc[i] = o < NB * 256 && col < e.N ? epi_scale(e, a_s, col) : 0.0f;
    }
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        if ((rblk0 + mb) * 16 >= M) break;
        if (mb) __syncthreads();  // the previous block's sums are read
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) red[wave][j][r][lane] = acc[mb][j][r];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < OUT; ++i) {
            const int o = tid + i * kWaves * 64, l = o & 63, r = (o >> 6) & 3, j = o >> 8;
            const int64_t row = (int64_t)(rblk0 + mb) * 16 + (l >> 4) * 4 + r, col = (int64_t)(blk0 + j) * 16 + (l & 15);
            if (o >= NB * 256 || row >= M || col >= e.N) continue;
            float v = 0.0f;
#pragma unroll
            for (int w = 0; w < kWaves; ++w) v += red[w][j][r][l];
            epi_store(e, row, col, epi_value(e, bsc[i], row, col, v));
        }
    }
}

// A workgroup's rows (16*mb) and columns (16*nb), by the modelled time.  At
// K = 4096, all but the first 3 us in proportion to K, W workgroups took on 256
// CUs (us, without the quantiser; N = 4096 and 12288, M = 17 .. 512):
//   32 x 16: 3.0 per W/256 (5.9 at 256, 25 at 2048); 32 x 32: 4.5 (7.8 at 256,
//   28 at 1536); 64 x 32: 6.5, at least 7 (10.8 at 256, 29 at 1024), and 32 x
//   64 the same; 64 x 64, one per CU: 12 a round (15 at 256, 26 at 384, 39 at
//   768); 96 x 64, one per CU: 17.3 a round (20 at 256, 55 at 768);
// two 32 x 32 or wider share a CU, so past 256 of them whole rounds count (N = 1024,
// K = 8192, M = 384, 384 of 32 x 32: 28.0 us row-major and 29.9, by 64 x 32 27.1);
// 128 x 64 spills, 128 x 32 and 96 x 32 were slower than 64 x 32.  The weights
// take N*K bytes at 4.3 TB/s at least.
struct RowsShape {
    int mb, nb;
    double us;
};
RowsShape rows_shape(int64_t M, int64_t N, int64_t K) {
    const double kf = (double)K / 4096.0;
    const int64_t rblocks = (M + 15) / 16, cblocks = (N + 15) / 16;
    const double memory = (double)N * (double)K / 4.3e6;
    RowsShape best{0, 0, 0.0};
    auto offer = [&](int mb, int nb, double slope, bool rounds, double least) {
        double w = (double)((rblocks + mb - 1) / mb * ((cblocks + nb - 1) / nb)) / 256.0;
        if (rounds || (mb * nb >= 4 && w > 1.0)) w = (double)(int64_t)(w + 0.998);  // whole rounds
        const double us = 3.0 + std::max({slope * w * kf, least * kf, memory});
        if (!best.mb || us < best.us) best = {mb, nb, us};
    };
    if (rblocks > 4) offer(6, 4, 17.3, true, 0);
    if (rblocks > 2) {
        offer(4, 4, 12.0, true, 0);
        offer(4, 2, 6.5, false, 7.0);
    }
    offer(2, 4, 6.6, false, 7.0);
    offer(2, 2, 4.5, false, 4.0);
    offer(2, 1, 3.0, false, 2.9);
    return best;
}

}  // namespace

double gemm_rows_us(int64_t M, int64_t N, int64_t K) {
    const bool fits = M > 16 && M * K < ((int64_t)1 << 31) && pad_to(K, kPackK) * 64 < ((int64_t)1 << 31) &&
                      N < ((int64_t)1 << 30);
    return fits ? rows_shape(M, N, K).us : 1e30;
}

hipError_t launch_quantize_rows(const float *x, uint8_t *y, int64_t M, int64_t K, const uint32_t *part, int npart,
                                float *scale_out, hipStream_t s) {
    const int64_t units = (M + 15) / 16 * ((K / 16 + 3) / 4), per = kThreads / 64;
    hipLaunchKernelGGL(k_quantize_rows, dim3((unsigned)((units + per - 1) / per)), dim3(kThreads), 0, s, x, y, (int)M,
                       (int)K, part, npart, scale_out);
    return hipGetLastError();
}

hipError_t launch_gemm_rows(int64_t M, int64_t N, int64_t K, const uint8_t *a, const uint8_t *bp, const Epilogue &e,
                            hipStream_t s) {
    const RowsShape sh = rows_shape(M, N, K);
    const int64_t Kp = pad_to(K, kPackK), rg = ((M + 15) / 16 + sh.mb - 1) / sh.mb;
    const unsigned grid = (unsigned)(((N + 15) / 16 + sh.nb - 1) / sh.nb * rg);
    auto go = [&](auto mbv, auto nbv) {
        hipLaunchKernelGGL((k_gemm_rows<decltype(mbv)::value, decltype(nbv)::value>), dim3(grid), dim3(kWaves * 64), 0, s,
                           bp, a, (int)M, (int)K, (int)(Kp / 16), (int)(Kp / 128), (int)rg, e);
    };
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    using I4 = std::integral_constant<int, 4>;
    using I6 = std::integral_constant<int, 6>;
    if (sh.mb == 6)
        go(I6{}, I4{});
    else if (sh.mb == 4)
        sh.nb == 4 ? go(I4{}, I4{}) : go(I4{}, I2{});
    else
        sh.nb == 4 ? go(I2{}, I4{}) : sh.nb == 2 ? go(I2{}, I2{}) : go(I2{}, I1{});
    return hipGetLastError();
}

}  // namespace lcml
