// gemm_f32.hip -- plain fp32 Gemm, fp32 convolution and elementwise
// activations, used by the operator layer for graphs that are not (or cannot
// be) fused into the FP8 path.
//
// Gemm and convolution keep the reference's arithmetic: every output is one
// sequential fma chain from 0 (over k, src/onnx/operators/gemm.cpp:155-162;
// over kh, kw, then the group's input channels, conv.cpp:143-192), then
// alpha, beta*C or the bias, then the activation.  Both run on
// v_mfma_f32_16x16x4_f32: on gfx950 it applies its four products to the
// accumulator one after another, each with one rounding, so that a sequence
// of them over k is that chain bit for bit (equal on 512000 random outputs
// for each of four exponent ranges, subnormals among them), at twice the
// rate of v_fma_f32 and without a register operand per product and lane.
#include <algorithm>
#include <cmath>

#include "lcml_internal.hpp"

namespace lcml {
namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f2 __attribute__((ext_vector_type(2)));

constexpr uint32_t kOOB = 0x80000000u;  // buffer offset past every extent: loads return zeros
constexpr int kRsrcFlags = 0x00020000;  // raw buffer resource word 3
// A launch of 2^32 work items in one dimension or more runs with that number
// modulo 2^32 and reports no error: workgroups of 256 that a grid may have.
constexpr int64_t kGridMax = ((int64_t)1 << 24) - 1;

__device__ inline float buf_f32(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0));
}

// ------------------------------------------------------------------- Gemm --
// Workgroup tile TB x TB outputs (64, 32 or 16), 256 threads.  Two
// wavefronts bring A and two bring B, a thread 16 values of a K chunk of
// 2048 / TB: two chunks are on their way in registers and two lie in LDS,
// because with few tiles (16 x 1000 outputs: 63 of them) the time is the
// latency of the loads and of the chain itself.  The wavefronts' 16x16
// blocks: 2x2 each at TB = 64, one each at 32, and one of wavefront 0 alone
// at 16.
// LDS holds k = 16 g + 4 j + q of row r at float ((g*4 + q)*TB + r)*4 + j (+
// PAD per g): lane (r, q) of an MFMA reads its operand of four steps as one
// 16-byte word, 16 lanes 256 contiguous bytes; a thread's 16 values are four
// such words after a 4x4 transpose in registers.
// 16 x 1000 x 2048: 17 us against 337 us with one v_fma chain per thread
// (its chain alone takes 9 us); 512 x 2048 x 2048: 66 us against 355 us.
// One rule for the loads: every lane loads, out of range ones at an offset
// past the buffer's end, so that no load sits under a branch and the waits
// count.  VEC: 16-byte loads (both operands' pointers, pitches and contiguous
// extents multiples of 16 bytes); else 4-byte ones.
template <int TB, bool A_KC, bool B_KC, bool VEC>
__global__ __launch_bounds__(256) void k_sgemm(int M, int N, int K, const float *__restrict__ A, int lda,
                                               const float *__restrict__ B, int ldb, int tiles_n, Epilogue e) {
    constexpr int BK = 2048 / TB, G = BK / 16;
    constexpr int PAD = 16 / G * 4;              // floats per 16-k group: its writers fall on distinct banks
    constexpr int GS = 16 * TB + PAD;            // floats of a 16-k group
    constexpr int WB = TB == 64 ? 2 : 1;         // 16-wide blocks of a wavefront in each direction
    __shared__ __attribute__((aligned(16))) float lds[2][2][G * GS];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tm = (int)blockIdx.x / tiles_n;
    const int m0 = tm * TB, n0 = ((int)blockIdx.x - tm * tiles_n) * TB;

    // ---- this thread's 16 values of a chunk -------------------------------
    const bool is_b = wave >= 2;
    const int t = tid & 127;
    const float *src = is_b ? B + (B_KC ? (int64_t)n0 * ldb : n0) : A + (A_KC ? (int64_t)m0 * lda : m0);
    const int ld = is_b ? ldb : lda, rows = min(TB, is_b ? N - n0 : M - m0);
    auto patch = [&](auto kcontig, int k0, f4 (&v)[4]) {
        const int kk = K - k0;  // k left, may be <= 0
        if constexpr (decltype(kcontig)::value) {
            // row r, k = 16 g .. + 15
            const int g = t % G, r = t / G;
            const __amdgpu_buffer_rsrc_t rs =
                __builtin_amdgcn_make_buffer_rsrc((void *)(src + k0), 0, ((rows - 1) * ld + max(kk, 0)) * 4, kRsrcFlags);
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const int k = 16 * g + 4 * c;
                const uint32_t o = (uint32_t)(r * ld + k) * 4u;
                if constexpr (VEC) {
                    v[c] = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)(r < rows && k < kk ? o : kOOB), 0, 0));
                } else {
#pragma unroll
                    for (int x = 0; x < 4; ++x) v[c][x] = buf_f32(rs, r < rows && k + x < kk ? o + 4 * x : kOOB);
                }
            }
        } else {
            // rows r .. r + 3 at k = 16 g + q + {0, 4, 8, 12}
            const int r = t % (TB / 4) * 4, gq = t / (TB / 4);
            const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
                (void *)(src + (int64_t)k0 * ld), 0, kk > 0 ? ((min(kk, BK) - 1) * ld + rows) * 4 : 0, kRsrcFlags);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int k = (gq >> 2) * 16 + 4 * j + (gq & 3);
                const uint32_t o = (uint32_t)(k * ld + r) * 4u;
                if constexpr (VEC) {
                    v[j] = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)(r < rows && k < kk ? o : kOOB), 0, 0));
                } else {
#pragma unroll
                    for (int x = 0; x < 4; ++x) v[j][x] = buf_f32(rs, r + x < rows && k < kk ? o + 4 * x : kOOB);
                }
            }
        }
    };
    auto put = [&](auto kcontig, float *to, const f4 (&v)[4]) {
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            const f4 w = {v[0][x], v[1][x], v[2][x], v[3][x]};
            if constexpr (decltype(kcontig)::value) {  // x: k's remainder q of row r
                const int g = t % G, r = t / G;
                *reinterpret_cast<f4 *>(to + g * GS + (x * TB + r) * 4) = w;
            } else {  // x: row r + x
                const int r = t % (TB / 4) * 4, gq = t / (TB / 4);
                *reinterpret_cast<f4 *>(to + (gq >> 2) * GS + ((gq & 3) * TB + r + x) * 4) = w;
            }
        }
    };
    using AK = std::integral_constant<bool, A_KC>;
    using BKC = std::integral_constant<bool, B_KC>;
    // (a branch on the wavefront's role; with equal layouts both sides are one)
    auto load = [&](int k0, f4 (&v)[4]) {
        if constexpr (A_KC == B_KC)
            patch(AK{}, k0, v);
        else if (is_b)
            patch(BKC{}, k0, v);
        else
            patch(AK{}, k0, v);
    };
    auto store = [&](int buf, const f4 (&v)[4]) {
        float *to = lds[buf][is_b ? 1 : 0];
        if constexpr (A_KC == B_KC)
            put(AK{}, to, v);
        else if (is_b)
            put(BKC{}, to, v);
        else
            put(AK{}, to, v);
    };

    // ---- this wavefront's blocks ------------------------------------------
    const bool works = TB > 16 || wave == 0;
    const int wr = TB > 16 ? (wave >> 1) * (TB / 2) : 0, wc = TB > 16 ? (wave & 1) * (TB / 2) : 0;
    f4 acc[WB][WB] = {};
    auto compute = [&](int buf) {
        const float *pa = lds[buf][0] + ((lane >> 4) * TB + wr + (lane & 15)) * 4;
        const float *pb = lds[buf][1] + ((lane >> 4) * TB + wc + (lane & 15)) * 4;
#pragma unroll 2
        for (int g = 0; g < G; ++g) {
            f4 fa[WB], fb[WB];
#pragma unroll
            for (int i = 0; i < WB; ++i) {
                fa[i] = *reinterpret_cast<const f4 *>(pa + g * GS + i * 64);
                fb[i] = *reinterpret_cast<const f4 *>(pb + g * GS + i * 64);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int i = 0; i < WB; ++i)
#pragma unroll
                    for (int h = 0; h < WB; ++h)
                        acc[i][h] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[i][j], fb[h][j], acc[i][h], 0, 0, 0);
        }
    };
    f4 va[4], vb[4];
    load(0, va);
    load(BK, vb);
    store(0, va);
    load(2 * BK, va);
    __syncthreads();
    // chunk c is computed from LDS buffer c % 2 while c + 1 moves from its
    // registers to the other buffer and c + 3 takes its place there
    for (int k0 = 0; k0 < K; k0 += 2 * BK) {
        store(1, vb);
        load(k0 + 3 * BK, vb);
        if (works) compute(0);
        __syncthreads();
        if (k0 + BK >= K) break;
        store(0, va);
        load(k0 + 4 * BK, va);
        if (works) compute(1);
        __syncthreads();
    }
    if (!works) return;
#pragma unroll
    for (int i = 0; i < WB; ++i)
#pragma unroll
        for (int h = 0; h < WB; ++h)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t m = m0 + wr + i * 16 + (lane >> 4) * 4 + r, n = n0 + wc + h * 16 + (lane & 15);
                if (m < M && n < N) epi_store(e, m, n, epi_value(e, 1.0f, m, n, acc[i][h][r]));
            }
}

// The general Gemm: any pitch and extent, and few k.  64x64 output tile per 256-thread
// workgroup, 4x4 outputs per thread, one fma chain each, K staged through
// LDS 16 at a time.
constexpr int TM = 64, TN = 64, TK = 16;

__global__ __launch_bounds__(256) void k_sgemm_any(int64_t M, int64_t N, int64_t K, const float *__restrict__ A,
                                                   int64_t lda, int transA, const float *__restrict__ B, int64_t ldb,
                                                   int transB, Epilogue e) {
    __shared__ float sa[TK][TM + 1];
    __shared__ float sb[TK][TN + 1];
    const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
    const int64_t m0 = (int64_t)blockIdx.y * TM, n0 = (int64_t)blockIdx.x * TN;
    float acc[4][4] = {};
    for (int64_t k0 = 0; k0 < K; k0 += TK) {
        for (int i = threadIdx.x; i < TK * TM; i += 256) {
            const int kk = i / TM, mm = i % TM;
            const int64_t m = m0 + mm, k = k0 + kk;
            sa[kk][mm] = (m < M && k < K) ? (transA ? A[k * lda + m] : A[m * lda + k]) : 0.0f;
        }
        for (int i = threadIdx.x; i < TK * TN; i += 256) {
            const int kk = i / TN, nn = i % TN;
            const int64_t n = n0 + nn, k = k0 + kk;
            sb[kk][nn] = (n < N && k < K) ? (transB ? B[n * ldb + k] : B[k * ldb + n]) : 0.0f;
        }
        __syncthreads();
        const int kmax = (int)((K - k0) < TK ? (K - k0) : TK);
        for (int kk = 0; kk < kmax; ++kk)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(sa[kk][ty * 4 + i], sb[kk][tx * 4 + j], acc[i][j]);
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int64_t m = m0 + ty * 4 + i;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int64_t n = n0 + tx * 4 + j;
            if (n < N) epi_store(e, m, n, epi_value(e, 1.0f, m, n, acc[i][j]));
        }
    }
}

__global__ __launch_bounds__(256) void k_activation(const float *__restrict__ x, float *__restrict__ y, int64_t n,
                                                    int act) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256)
        y[i] = apply_act(x[i], act);
}

// Direct fp32 NCHW convolution, one thread per output element, one fma
// chain per output in the reference Conv's reduction order (kh, kw, then the
// group's input channels; conv.cpp:143-192, whose 4-wide partial sums differ
// from this chain only in fp32 rounding), begin pads only (conv.cpp:121),
// dilation, groups, bias, activation.  For few output channels per group
// or small planes (the matrix kernels would multiply mostly padding) and for
// geometries past their 16- and 32-bit offsets or their grid.
__global__ __launch_bounds__(256) void k_conv2d_f32(const float *__restrict__ x, const float *__restrict__ w,
                                                    const float *__restrict__ bias, float *__restrict__ y, int C,
                                                    int H, int W, int Cout, int KH, int KW, int sh, int sw, int ph,
                                                    int pw, int dh, int dw, int group, int OH, int OW, int act,
                                                    int64_t total) {
    const int64_t i = ((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * 256 + threadIdx.x;
    if (i >= total) return;
    const int ow = (int)(i % OW);
    const int oh = (int)((i / OW) % OH);
    const int co = (int)((i / ((int64_t)OW * OH)) % Cout);
    const int64_t n = i / ((int64_t)OW * OH * Cout);
    const int cg = C / group, mg = Cout / group, g = co / mg;
    const float *xn = x + (n * C + (int64_t)g * cg) * H * W;
    const float *wc = w + (int64_t)co * cg * KH * KW;
    float sum = 0.0f;
    for (int kh = 0; kh < KH; ++kh) {
        const int ih = oh * sh + kh * dh - ph;
        if ((unsigned)ih >= (unsigned)H) continue;
        for (int kw = 0; kw < KW; ++kw) {
            const int iw = ow * sw + kw * dw - pw;
            if ((unsigned)iw >= (unsigned)W) continue;
            for (int c = 0; c < cg; ++c)
                sum = fmaf(xn[((int64_t)c * H + ih) * W + iw], wc[((int64_t)c * KH + kh) * KW + kw], sum);
        }
    }
    if (bias) sum += bias[co];
    y[i] = apply_act(sum, act);
}

// ------------------------------------------------------------ convolution --
// NCHW fp32 convolution as an implicit GEMM on the fp32 matrix instruction:
// rows = output channels of one group, columns = output pixels of one image,
// k = (kh, kw, c) in the reference's order, so that each output is its fma
// chain (taps in the padding, which the reference skips, add products with
// zero).  256 threads; a workgroup computes CB*16 channels of 64*PB pixels,
// a wavefront 16*PB of the pixels.
//   * The weights of KT k's are staged in LDS as the chain's operands, the
//     word of four steps (j) of channel ch at (g*4 + q)*WS + ch*4 + j for
//     k = 16 g + 4 j + q, beside a table of each k's input offset and tap.
//   * The pixels' values are read straight from global memory: a lane holds
//     pixels PB*(lane%16) .. + PB-1 and one k of four, its address is the
//     pixel's corner plus the table's offset, and a tap outside the image
//     gets an offset past the buffer's end (the hardware returns 0).  Each
//     value feeds CB MFMAs of 32 cycles, so its ~10 address instructions hide
//     behind them; an image row is read from L1/L2 once per tap.
//   * The next 16 k's values are on their way while the current ones multiply.
// 64 channels of 5x5x20 on four 100x100 images: 68 us against 299 us with one
// thread per output; 8 channels of 3x3x3 on 16 images of 224x224: 34 us
// against 99 us.
// Weights that are not finite: their product with a padding zero would be
// NaN where the reference skips the tap, so a workgroup that stages one runs
// that part of k lane by lane with the taps tested (BAD).
constexpr int KT = 160;
// floats of the 16*CB channels' words of one (g, q): the padding spreads the
// writers over the banks
template <int CB>
constexpr int kWS = CB * 64 + 4;
// Channels of a group from which on the matrix kernels are the faster ones (32
// groups of 3x3x1 on 16 images of 56x56: four channels each, 47 us against
// 57 us; three, 47 us against 44 us)
constexpr int kConvMinChannels = 4;

struct ConvF32 {
    const float *x, *w, *bias;
    float *y;
    int C, H, W, Cout, KH, KW, sh, sw, ph, pw, dh, dw, group, OH, OW, act;
    int tiles_p, tiles, tiles_c, tiles_x;  // pixel tiles of an image and of all, channel tiles of a group, tiles across an image (patch kernel)
};

// The weights of k = kt .. kt + kn-1 (kn <= KT) of a tile's NC = 16*CB
// channels (the first nch exist) into wl, for all 256 threads of a workgroup;
// true when this thread met one that is not finite.  wr: the channels'
// weights [channel][c][taps], K = cg * taps of them each.  Lanes run along k
// (a channel's weights lie within a few cache lines; lanes along the channels
// read a line each and took as long as the MFMAs), wavefronts along the
// channels.
template <int CB>
__device__ __forceinline__ bool stage_weights(float *wl, __amdgpu_buffer_rsrc_t wr, int nch, int kt, int kn, int cg,
                                              int taps, int K) {
    constexpr int NC = CB * 16, WS = kWS<CB>, KQ = (KT + 63) / 64;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), k16 = (kn + 15) / 16 * 16;
    bool bad = false;
    uint32_t wo[KQ];  // this lane's k's: byte offset in a channel's weights
    int lo[KQ];       // and word in LDS
#pragma unroll
    for (int u = 0; u < KQ; ++u) {
        const int k = lane + 64 * u, tp = (kt + k) / cg, c = kt + k - tp * cg;
        wo[u] = k < kn ? (uint32_t)(c * taps + tp) * 4u : kOOB;
        lo[u] = k < k16 ? ((k >> 4) * 4 + (k & 3)) * WS + ((k >> 2) & 3) : -1;
    }
    constexpr int CU = NC / 4 < 8 ? NC / 4 : 8;  // channels loaded together
    // 64 k at a time as many as there are (with the empty ones too 64 channels of
    // 3x3x3 on 16 images of 56x56 take 19.7 us instead of 17.6)
    auto channels = [&](auto nq) {
        constexpr int Q = decltype(nq)::value;
        for (int ch = wave; ch < NC; ch += 4 * CU) {
            float v[CU][Q];
#pragma unroll
            for (int i = 0; i < CU; ++i)
#pragma unroll
                for (int u = 0; u < Q; ++u)  // kOOB plus a channel's offset stays out of range
                    v[i][u] = buf_f32(wr, ch + 4 * i < nch ? wo[u] + (uint32_t)((ch + 4 * i) * K) * 4u : kOOB);
#pragma unroll
            for (int i = 0; i < CU; ++i)
#pragma unroll
                for (int u = 0; u < Q; ++u) {
                    bad |= !(fabsf(v[i][u]) <= 3.4028235e38f);
                    if (lo[u] >= 0) wl[lo[u] + (ch + 4 * i) * 4] = v[i][u];
                }
        }
    };
    if (k16 <= 64)
        channels(std::integral_constant<int, 1>{});
    else if (k16 <= 128)
        channels(std::integral_constant<int, 2>{});
    else
        channels(std::integral_constant<int, KQ>{});
    return bad;
}

// bias and activation of one lane's outputs (channels c*16 + chl + r of a
// tile, PB pixels each), stored through put(channel, values)
template <int CB, int PB, class Put>
__device__ __forceinline__ void conv_epilogue(const f4 (&acc)[PB][CB], const float (&bs)[CB][4], bool has_bias, int act,
                                              int chl, int nch, Put put) {
    auto out = [&](auto a) {
#pragma unroll
        for (int c = 0; c < CB; ++c)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int ch = c * 16 + chl + r;
                if (ch >= nch) continue;
                float o[PB];
#pragma unroll
                for (int i = 0; i < PB; ++i)
                    o[i] = apply_act(has_bias ? acc[i][c][r] + bs[c][r] : acc[i][c][r],
                                     decltype(a)::value < 0 ? act : decltype(a)::value);
                put(ch, o);
            }
    };
    // the usual activations without a test per value; the GELU forms share a copy
    if (act == ACT_NONE)
        out(std::integral_constant<int, ACT_NONE>{});
    else if (act == ACT_RELU)
        out(std::integral_constant<int, ACT_RELU>{});
    else
        out(std::integral_constant<int, -1>{});
}

template <int CB, int PB>
__global__ __launch_bounds__(256) void k_conv2d_f32_mfma(ConvF32 a) {
    constexpr int NC = CB * 16, WS = kWS<CB>;
    __shared__ __attribute__((aligned(16))) float wl[KT / 4 * WS];
    __shared__ int2 tab[KT];  // {input offset, kh*dh in the upper half, kw*dw in the lower}
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // workgroup -> (image, pixel tile, group, channel tile), channels innermost
    const int ct = (int)blockIdx.x % a.tiles_c, grp = (int)blockIdx.x / a.tiles_c % a.group;
    const int tile = (int)blockIdx.x / (a.tiles_c * a.group), n = tile / a.tiles_p, pt = tile - n * a.tiles_p;
    const int cg = a.C / a.group, mg = a.Cout / a.group, K = a.KH * a.KW * cg;
    const int HW = a.H * a.W, OHW = a.OH * a.OW;
    const int ch0 = ct * NC;  // first channel within the group
    const int nch = min(NC, mg - ch0);
    // [channel][c][kh][kw] of this tile's channels, and their bias
    const __amdgpu_buffer_rsrc_t wr =
        __builtin_amdgcn_make_buffer_rsrc((void *)(a.w + (int64_t)(grp * mg + ch0) * K), 0, nch * K * 4, kRsrcFlags);
    const __amdgpu_buffer_rsrc_t br = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(a.bias + grp * mg + ch0), 0, a.bias ? nch * 4 : 0, kRsrcFlags);

    float bs[CB][4];
    const int chl = (lane >> 4) * 4;  // this lane's channels within a block: chl + r
#pragma unroll
    for (int c = 0; c < CB; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r) bs[c][r] = buf_f32(br, (uint32_t)(c * 16 + chl + r) * 4u);

    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(a.x + ((int64_t)n * a.C + (int64_t)grp * cg) * HW), 0, cg * HW * 4, kRsrcFlags);
    // this lane's pixels
    const int p0 = (pt * 4 + wave) * 16 * PB + PB * (lane & 15);
    int ih0[PB], iw0[PB];
    uint32_t base[PB];  // modulo 2^32, as the table's offsets: corners and taps may lie outside the image
#pragma unroll
    for (int i = 0; i < PB; ++i) {
        const int p = p0 + i < OHW ? p0 + i : OHW - 1;
        const int oh = p / a.OW, ow = p - oh * a.OW;
        ih0[i] = oh * a.sh - a.ph;
        iw0[i] = ow * a.sw - a.pw;
        base[i] = (uint32_t)ih0[i] * (uint32_t)a.W + (uint32_t)iw0[i];
    }
    auto tap = [&](int i, int2 t) {  // pixel i's value under a table entry
        const int ih = ih0[i] + (t.y >> 16), iw = iw0[i] + (int)(int16_t)t.y;
        const bool ok = (uint32_t)ih < (uint32_t)a.H && (uint32_t)iw < (uint32_t)a.W;
        return buf_f32(xr, ok ? (base[i] + (uint32_t)t.x) * 4u : kOOB);
    };

    f4 acc[PB][CB] = {};
    for (int kt = 0; kt < K; kt += KT) {
        const int kn = min(KT, K - kt), ng = (kn + 15) / 16;
        if (kt) __syncthreads();  // the previous part is consumed
        for (int k = tid; k < KT; k += 256) {
            int2 t = {0, (int)0x80008000u};  // past K: a row above every image
            if (k < kn) {
                const int tp = (kt + k) / cg, c = kt + k - tp * cg, kh = tp / a.KW, kw = tp - kh * a.KW;
                t.x = (int)((uint32_t)c * (uint32_t)HW + (uint32_t)(kh * a.dh) * (uint32_t)a.W + (uint32_t)(kw * a.dw));
                t.y = (int)((uint32_t)(kh * a.dh) << 16 | (uint32_t)(kw * a.dw));
            }
            tab[k] = t;
        }
        const bool bad = stage_weights<CB>(wl, wr, nch, kt, kn, cg, a.KH * a.KW, K);
        if (__syncthreads_or(bad)) {
            for (int k = 0; k < kn; ++k) {
                const int2 t = tab[k];
#pragma unroll
                for (int i = 0; i < PB; ++i) {
                    const float xv = tap(i, t);
                    const int ih = ih0[i] + (t.y >> 16), iw = iw0[i] + (int)(int16_t)t.y;
                    if ((uint32_t)ih < (uint32_t)a.H && (uint32_t)iw < (uint32_t)a.W)
#pragma unroll
                        for (int c = 0; c < CB; ++c)
#pragma unroll
                            for (int r = 0; r < 4; ++r) {
                                const int ch = c * 16 + (lane >> 4) * 4 + r;
                                const float wv = wl[((k >> 4) * 4 + (k & 3)) * WS + ch * 4 + ((k >> 2) & 3)];
                                acc[i][c][r] = fmaf(xv, wv, acc[i][c][r]);
                            }
                }
            }
            continue;
        }
        const int q = lane >> 4;
        float xv[4][PB];
        auto gather = [&](int g, float (&v)[4][PB]) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int2 t = tab[g * 16 + 4 * j + q];
#pragma unroll
                for (int i = 0; i < PB; ++i) v[j][i] = tap(i, t);
            }
        };
        gather(0, xv);
        for (int g = 0; g < ng; ++g) {
            float xn[4][PB];
            gather(g + 1 < ng ? g + 1 : g, xn);
            f4 wf[CB];
#pragma unroll
            for (int c = 0; c < CB; ++c)
                wf[c] = *reinterpret_cast<const f4 *>(wl + (g * 4 + q) * WS + (c * 16 + (lane & 15)) * 4);
            const int steps = (kn - g * 16 + 3) / 4;  // of four k: fewer than four in the last group
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (j >= steps) break;
#pragma unroll
                for (int i = 0; i < PB; ++i)
#pragma unroll
                    for (int c = 0; c < CB; ++c)
                        acc[i][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[c][j], xv[j][i], acc[i][c], 0, 0, 0);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int i = 0; i < PB; ++i) xv[j][i] = xn[j][i];
        }
    }
    // lane: pixels p0 .. + PB-1 of channels c*16 + (lane/16)*4 + r
    float *yn = a.y + ((int64_t)n * a.Cout + (int64_t)grp * mg + ch0) * OHW + p0;
    const bool pair = PB == 2 && (OHW & 1) == 0 && (reinterpret_cast<uintptr_t>(a.y) & 7) == 0;
    conv_epilogue<CB, PB>(acc, bs, a.bias != nullptr, a.act, chl, nch, [&](int ch, const float (&o)[PB]) {
        float *p = yn + (int64_t)ch * OHW;
        if (pair) {
            if (p0 < OHW) *reinterpret_cast<f2 *>(p) = f2{o[0], o[PB - 1]};
        } else {
#pragma unroll
            for (int i = 0; i < PB; ++i)
                if (p0 + i < OHW) p[i] = o[i];
        }
    });
}

// The same chain with the input staged too, for K of one part (at most KT) and
// more than 16 channels: a workgroup walks tiles of 16 output columns x 4*PB
// rows of one image (a wavefront PB rows, a lane one column), and the input
// under a tile (all channels of the group, zeros in the padding) lies in LDS,
// so that a pixel's value costs one LDS read and one addition instead of a
// bounds test and a load, and the weights are staged once per workgroup.  The
// LDS reads of the next 16 k's are issued before the MFMAs of the current
// ones; three workgroups per CU
// (at most 168 VGPRs) keep the matrix units busy while others stage: with two,
// the tile's loads and stores left them idle half the time.  Stem of a
// ResNet (64 channels of 7x7x3, stride 2, 16 images of 224x224): 55 us against
// 76 us with the values gathered, 72 us with two workgroups per CU, 1010 us
// one thread per output; 24 us at the full MFMA rate.
template <int CB, int PB>
__global__ __launch_bounds__(256, 3) void k_conv2d_f32_patch(ConvF32 a) {
    static_assert(CB > 1, "16 channels or fewer: the gather kernel");
    constexpr int NC = CB * 16, WS = kWS<CB>;
    extern __shared__ __attribute__((aligned(16))) float smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ct = (int)blockIdx.x % a.tiles_c, grp = (int)blockIdx.x / a.tiles_c % a.group;
    const int first = (int)blockIdx.x / (a.tiles_c * a.group), step = (int)gridDim.x / (a.tiles_c * a.group);
    const int cg = a.C / a.group, mg = a.Cout / a.group, taps = a.KH * a.KW, K = taps * cg;
    const int HW = a.H * a.W, OHW = a.OH * a.OW, KP = (K + 15) / 16 * 16;
    const int PH = (4 * PB - 1) * a.sh + (a.KH - 1) * a.dh + 1, PW = 15 * a.sw + (a.KW - 1) * a.dw + 1;
    float *wl = smem, *bias_l = smem + KP / 4 * WS + KP, *patch = bias_l + NC;
    int *tab = reinterpret_cast<int *>(smem + KP / 4 * WS);  // k's offset in the patch, at (k/16)*16 + (k%4)*4 + (k/4)%4
    const int ch0 = ct * NC, nch = min(NC, mg - ch0), chl = (lane >> 4) * 4, q = lane >> 4;
    const __amdgpu_buffer_rsrc_t wr =
        __builtin_amdgcn_make_buffer_rsrc((void *)(a.w + (int64_t)(grp * mg + ch0) * K), 0, nch * K * 4, kRsrcFlags);
    const __amdgpu_buffer_rsrc_t br = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(a.bias + grp * mg + ch0), 0, a.bias ? nch * 4 : 0, kRsrcFlags);
    // this lane's pixels in the patch: row i of the wavefront's PB
    const int pr = wave * PB, pb0 = pr * a.sh * PW + (lane & 15) * a.sw, pbs = a.sh * PW;

    // The patch by rows (channel, input row), a wavefront every fourth, lanes
    // along a row, 16 rows on their way.
    constexpr int RU = 16;
    const int nrow = cg * PH;
    struct Tile {
        int n, ih0, iw0, oh0, ow0;
    };
    auto place = [&](int tile) {
        Tile r;
        r.n = tile / a.tiles_p;
        const int t2 = tile - r.n * a.tiles_p, ty = t2 / a.tiles_x;
        r.oh0 = ty * 4 * PB;
        r.ow0 = (t2 - ty * a.tiles_x) * 16;
        r.ih0 = r.oh0 * a.sh - a.ph;
        r.iw0 = r.ow0 * a.sw - a.pw;
        return r;
    };
    auto load_rows = [&](const Tile &tl, int row0, int col, float (&v)[RU]) {
        const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(a.x + ((int64_t)tl.n * a.C + (int64_t)grp * cg) * HW), 0, cg * HW * 4, kRsrcFlags);
        const int iw = tl.iw0 + col;
        const bool cok = col < PW && (uint32_t)iw < (uint32_t)a.W;
        int c = row0 / PH, r = row0 - c * PH;
#pragma unroll
        for (int u = 0; u < RU; ++u) {
            const int ih = tl.ih0 + r;
            const bool ok = cok && c < cg && (uint32_t)ih < (uint32_t)a.H;
            v[u] = buf_f32(xr, ok ? (uint32_t)((c * a.H + ih) * a.W + iw) * 4u : kOOB);
            r += 4;
            if (r >= PH) { r -= PH; ++c; }  // PH >= 4
        }
    };
    auto store_rows = [&](int row0, int col, const float (&v)[RU]) {
#pragma unroll
        for (int u = 0; u < RU; ++u)
            if (col < PW && row0 + 4 * u < nrow) patch[(row0 + 4 * u) * PW + col] = v[u];
    };
    bool bad = false;
    for (int tile = first; tile < a.tiles; tile += step) {
        const Tile tl = place(tile);
        const int oh0 = tl.oh0, ow0 = tl.ow0, ih0 = tl.ih0, iw0 = tl.iw0, n = tl.n;
        if (tile != first) __syncthreads();  // the previous tile's patch is consumed
        for (int c0 = 0; c0 < PW; c0 += 64)
            for (int r0 = wave; r0 < nrow; r0 += 4 * RU) {
                float v[RU];
                load_rows(tl, r0, c0 + lane, v);
                store_rows(r0, c0 + lane, v);
            }
        if (tile == first && tid < NC) bias_l[tid] = buf_f32(br, (uint32_t)tid * 4u);
        if (tile == first) {  // the weights and the table, for all tiles
            for (int k = tid; k < KP; k += 256) {
                int t = 0;  // past K: any value, masked below
                if (k < K) {
                    const int tp = k / cg, c = k - tp * cg, kh = tp / a.KW, kw = tp - kh * a.KW;
                    t = (c * PH + kh * a.dh) * PW + kw * a.dw;
                }
                tab[(k & ~15) + (k & 3) * 4 + ((k >> 2) & 3)] = t;
            }
            bad = __syncthreads_or(stage_weights<CB>(wl, wr, nch, 0, K, cg, taps, K));
        } else {
            __syncthreads();
        }
        f4 acc[PB][CB] = {};
        if (__builtin_expect(bad, 0)) {
            for (int k = 0; k < K; ++k) {
                const int tp = k / cg, kh = tp / a.KW, kw = tp - kh * a.KW;
                const int t = tab[(k & ~15) + (k & 3) * 4 + ((k >> 2) & 3)], iw = iw0 + (lane & 15) * a.sw + kw * a.dw;
#pragma unroll
                for (int i = 0; i < PB; ++i) {
                    const int ih = ih0 + (pr + i) * a.sh + kh * a.dh;
                    const float xv = patch[pb0 + i * pbs + t];
                    if ((uint32_t)ih < (uint32_t)a.H && (uint32_t)iw < (uint32_t)a.W)
#pragma unroll
                        for (int c = 0; c < CB; ++c)
#pragma unroll
                            for (int r = 0; r < 4; ++r)
                                acc[i][c][r] =
                                    fmaf(xv, wl[((k >> 4) * 4 + (k & 3)) * WS + (c * 16 + chl + r) * 4 + ((k >> 2) & 3)],
                                         acc[i][c][r]);
                }
            }
        } else {
            struct Frag {
                float x[PB][4];
                f4 w[CB];
            };
            typedef int i4 __attribute__((ext_vector_type(4)));
            auto offs = [&](int g) { return *reinterpret_cast<const i4 *>(tab + g * 16 + q * 4); };
            auto fetch = [&](Frag &f, int g, i4 t) {
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int i = 0; i < PB; ++i) f.x[i][j] = patch[pb0 + i * pbs + t[j]];
#pragma unroll
                for (int c = 0; c < CB; ++c)
                    f.w[c] = *reinterpret_cast<const f4 *>(wl + (g * 4 + q) * WS + (c * 16 + (lane & 15)) * 4);
            };
            auto mma = [&](const Frag &f, int j) {
#pragma unroll
                for (int c = 0; c < CB; ++c)
#pragma unroll
                    for (int i = 0; i < PB; ++i)
                        acc[i][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(f.w[c][j], f.x[i][j], acc[i][c], 0, 0, 0);
            };
            const int gl = KP / 16 - 1;  // the last group, which may be partial
            Frag f0, f1;
            fetch(f0, 0, offs(0));
            i4 t = offs(min(1, gl));
            auto whole = [&](const Frag &cur, Frag &nxt, int g) {
                fetch(nxt, g + 1, t);
                t = offs(min(g + 2, gl));
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int j = 0; j < 4; ++j) mma(cur, j);
                __builtin_amdgcn_sched_barrier(0);
            };
            int g = 0;
            for (; g + 2 <= gl; g += 2) {
                whole(f0, f1, g);
                whole(f1, f0, g + 1);
            }
            if (g < gl) {
                whole(f0, f1, g);
                f0 = f1;
            }
            // k past K: its weights are zero, and its value has to be finite
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (gl * 16 + 4 * j >= K) break;
#pragma unroll
                for (int i = 0; i < PB; ++i) f0.x[i][j] = gl * 16 + 4 * j + q < K ? f0.x[i][j] : 0.0f;
                mma(f0, j);
            }
        }
        float bs[CB][4];
#pragma unroll
        for (int c = 0; c < CB; ++c)
#pragma unroll
            for (int r = 0; r < 4; ++r) bs[c][r] = bias_l[c * 16 + chl + r];
        const int ow = ow0 + (lane & 15);
        float *yn = a.y + ((int64_t)n * a.Cout + (int64_t)grp * mg + ch0) * OHW + (int64_t)(oh0 + pr) * a.OW + ow;
        conv_epilogue<CB, PB>(acc, bs, a.bias != nullptr, a.act, chl, nch, [&](int ch, const float (&o)[PB]) {
            float *p = yn + (int64_t)ch * OHW;
#pragma unroll
            for (int i = 0; i < PB; ++i)
                if (ow < a.OW && oh0 + pr + i < a.OH) p[(int64_t)i * a.OW] = o[i];
        });
    }
}

// How many taps of one axis lie inside the image: the mean over its outputs
// and how many do for any of them.
struct LiveTaps {
    double mean;
    int any;
};
LiveTaps live_taps(int taps, int dil, int pad, int stride, int in, int out) {
    LiveTaps l{0.0, 0};
    for (int k = 0; k < taps; ++k) {
        const int64_t at = (int64_t)k * dil - pad;  // input of output 0
        const int64_t lo = at >= 0 ? 0 : (-at + stride - 1) / stride;
        const int64_t hi = at >= in ? -1 : std::min<int64_t>(out - 1, (in - 1 - at) / stride);
        if (hi < lo) continue;
        l.mean += (double)(hi - lo + 1) / out;
        ++l.any;
    }
    return l;
}

// Modelled times (us) of the three kernels, for the choice between the direct
// one, which starts at once, wastes no lane on a plane's edge and skips the
// taps in the padding, and the matrix kernels, whose workgroups compute 64 *
// pb pixels of one image whatever its size.  Fitted to 1083 geometries (planes
// of 1 to 112^2 pixels, 1 to 128 input and 4 to 256 output channels of a
// group, 1 to 65536 images), the choice is the faster kernel or within 5 % of
// it on 1030 of them, at most 27 % behind the direct and 65 % behind a matrix
// kernel.  8 channels of 1x1x8 on 65536 single pixels: 6.7 us direct, 209 us
// matrix; 64 of 3x3x64 on 2048 planes of 4x4: 348 and 253 us.
//
// The direct kernel: a chain of `live` products at cache latency, or all
// chains at a rate that grows with the plane, since the lanes along a small
// one read different channels' weights.
double conv_direct_us(int64_t total, int64_t OHW, double live, bool one_tap) {
    const double rate = 0.38e6 + 2.0e6 * std::min(1.0, (double)(OHW - 1) / 18.0);
    return 2.2 + std::max(live * (one_tap ? 0.1 : 0.115), (double)total * live / rate) + (double)total / 2.27e5;
}
// The matrix kernels: what the first workgroup takes apart from its chains,
// and per 256 workgroups; then the chains over K, in rounds of `resident`
// workgroups per CU, and of the patch kernel (three per CU) the patch's
// loads, in batches of 16 rows of 64 columns by each wavefront.
double conv_matrix_us(bool patch, int64_t K, int64_t batches, int64_t workgroups, int cb, int pb) {
    struct Fit {
        double start, per_256, per_k, resident, per_batch;
    };
    constexpr Fit gather_fit[2][3] = {{{3.6, 0.45, 0.031, 2.0, 0}, {3.4, 0.46, 0.0434, 1.2, 0}, {3.65, 1.1, 0.065, 1.07, 0}},
                                      {{3.5, 0.74, 0.059, 3.7, 0}, {5.2, 0.54, 0.083, 3.1, 0}, {15.8, 1.04, 0.0714, 1.34, 0}}};
    constexpr Fit patch_fit[2][2] = {{{4.0, 1.4, 0.0144, 3.0, 2.27}, {5.1, 1.9, 0.0243, 3.0, 2.2}},
                                     {{7.3, 0.76, 0.037, 3.0, 2.5}, {7.75, 2.2, 0.071, 3.0, 3.0}}};
    const Fit &f = patch ? patch_fit[pb - 1][cb == 2 ? 0 : 1] : gather_fit[pb - 1][cb == 1 ? 0 : cb == 2 ? 1 : 2];
    const double w = (double)workgroups / 256.0;
    return f.start + f.per_256 * w + std::max(1.0, w / f.resident) * ((double)K * f.per_k + (double)batches * f.per_batch);
}

}  // namespace

hipError_t launch_conv2d_f32(const float *x, const float *w, const float *bias, float *y, int64_t Nb, int C, int H,
                             int W, int Cout, int KH, int KW, int sh, int sw, int ph, int pw, int dh, int dw,
                             int group, int OH, int OW, int act, hipStream_t s, const char **kernel) {
    *kernel = "conv2d_f32_direct";
    const int64_t total = Nb * Cout * OH * OW;
    if (total == 0) return hipSuccess;
    const int mg = Cout / group;
    const int64_t cg = C / group, OHW = (int64_t)OH * OW, K = cg * KH * KW;
    const int cb = mg <= 16 ? 1 : mg <= 32 ? 2 : 4;
    const int64_t tiles_c = (mg + 16 * cb - 1) / (16 * cb);
    // 32-bit element offsets of an image's group, of its outputs and of a
    // tile's weights; tap offsets and corners in 15 bits, so that the gather
    // kernel's entry for k past K (-32768 rows) is outside whatever the corner
    const bool fits = cg * H * W < ((int64_t)1 << 29) && OHW < ((int64_t)1 << 30) && K < ((int64_t)1 << 22) &&
                      Nb * OHW < ((int64_t)1 << 34) && group * tiles_c < ((int64_t)1 << 30) &&
                      (int64_t)(KH - 1) * dh < 32768 && (int64_t)(KW - 1) * dw < 32768 &&
                      (int64_t)(OH - 1) * sh < 32768 && (int64_t)(OW - 1) * sw < 32768 && ph < 32768 && pw < 32768;
    if (fits && mg >= kConvMinChannels) {
        ConvF32 a = {x, w, bias, y, C, H, W, Cout, KH, KW, sh, sw, ph, pw, dh, dw, group, OH, OW, act, 0, 0, 0, 0};
        a.tiles_c = (int)tiles_c;
        // workgroups of 64-pixel tiles at most per CU: those that LDS holds
        auto walk = [&](int64_t lds) { return std::max<int64_t>(1, 256 * (160 * 1024 / lds) / (group * tiles_c)); };
        auto tiling = [&](bool patch, int pb) {
            a.tiles_x = (OW + 15) / 16;
            a.tiles_p = (int)(patch ? (int64_t)a.tiles_x * ((OH + 4 * pb - 1) / (4 * pb)) : (OHW + 64 * pb - 1) / (64 * pb));
            a.tiles = (int)(Nb * a.tiles_p);
            return Nb * (int64_t)a.tiles_p;
        };
        // The patch kernel for K of one part (in several, its weights are
        // staged for every tile: 75 us against 68 us on 5x5x20), more than 16
        // channels (with 16 or fewer the gathers hide as well and need no
        // staging: 34 us against 51 us on 8 channels of 3x3x3) and a patch
        // that leaves room for two workgroups per CU.  Two pixels per lane
        // where that still gives every CU two workgroups.
        auto patch_lds = [&](int pb) {
            const int64_t kp = (std::min<int64_t>(K, KT) + 15) / 16 * 16;
            const int64_t prows = (int64_t)(4 * pb - 1) * sh + (int64_t)(KH - 1) * dh + 1;
            const int64_t pcols = (int64_t)15 * sw + (int64_t)(KW - 1) * dw + 1;
            return (kp / 4 * (cb * 64 + 4) + kp + cb * 16 + cg * prows * pcols) * 4;
        };
        constexpr int64_t kLdsMax = 80 * 1024 - 512;
        int pb = tiling(true, 2) * group * tiles_c >= 512 ? 2 : 1;
        if (patch_lds(pb) > kLdsMax) pb = 1;
        const bool patch = cb > 1 && K <= KT && patch_lds(pb) <= kLdsMax;
        if (!patch) pb = tiling(false, 2) * group * tiles_c >= 512 ? 2 : 1;
        const int64_t workgroups = tiling(patch, pb) * group * tiles_c;
        const LiveTaps lh = live_taps(KH, dh, ph, sh, H, OH), lw = live_taps(KW, dw, pw, sw, W, OW);
        // (lanes of a wavefront wait for each other's taps: between the mean and the union)
        const double k_live = (double)cg * std::sqrt(lh.mean * lw.mean * lh.any * lw.any);
        const int64_t batches = (cg * ((4 * pb - 1) * (int64_t)sh + (KH - 1) * (int64_t)dh + 1) + 63) / 64 *
                                ((15 * (int64_t)sw + (KW - 1) * (int64_t)dw + 64) / 64);
        if (workgroups <= kGridMax && conv_matrix_us(patch, K, batches, workgroups, cb, pb) <=
                                          conv_direct_us(total, OHW, k_live, KH * KW == 1)) {
            *kernel = patch ? "conv2d_f32_patch" : "conv2d_f32_mfma";
            const int64_t lds = patch ? patch_lds(pb) : 0;
            const int64_t grid = group * tiles_c * (patch ? std::min<int64_t>(a.tiles, walk(lds)) : a.tiles);
            auto go = [&](auto cbv, auto pbv) -> hipError_t {
                constexpr int CB = decltype(cbv)::value, PB = decltype(pbv)::value;
                if constexpr (CB > 1) {
                    if (patch) {
                        static std::atomic<uint64_t> lds_set{0};
                        if (hipError_t err = ensure_dynamic_lds(
                                reinterpret_cast<const void *>(k_conv2d_f32_patch<CB, PB>), (int)kLdsMax, lds_set);
                            err != hipSuccess)
                            return err;
                        hipLaunchKernelGGL((k_conv2d_f32_patch<CB, PB>), dim3((unsigned)grid), dim3(256), (unsigned)lds,
                                           s, a);
                        return hipGetLastError();
                    }
                }
                hipLaunchKernelGGL((k_conv2d_f32_mfma<CB, PB>), dim3((unsigned)grid), dim3(256), 0, s, a);
                return hipGetLastError();
            };
            using One = std::integral_constant<int, 1>;
            using Two = std::integral_constant<int, 2>;
            auto by_pb = [&](auto cbv) { return pb == 2 ? go(cbv, Two{}) : go(cbv, One{}); };
            return cb == 1 ? by_pb(One{}) : cb == 2 ? by_pb(Two{}) : by_pb(std::integral_constant<int, 4>{});
        }
    }
    // (a loop over the outputs cost the small planes 10 %)
    const int64_t wgs = (total + 255) / 256, gx = std::min(wgs, kGridMax);
    hipLaunchKernelGGL(k_conv2d_f32, dim3((unsigned)gx, (unsigned)((wgs + gx - 1) / gx)), dim3(256), 0, s, x, w, bias, y, C, H, W,
                       Cout, KH, KW, sh, sw, ph, pw, dh, dw, group, OH, OW, act, total);
    return hipGetLastError();
}

namespace {

template <int TB>
void launch_sgemm_tile(int M, int N, int K, const float *A, int lda, bool a_kc, const float *B, int ldb, bool b_kc,
                       bool vec, const Epilogue &e, hipStream_t s) {
    const int tiles_n = (N + TB - 1) / TB;
    const dim3 grid((unsigned)(((M + TB - 1) / TB) * tiles_n));
    auto go = [&](auto ak, auto bk, auto v) {
        hipLaunchKernelGGL((k_sgemm<TB, decltype(ak)::value, decltype(bk)::value, decltype(v)::value>), grid, dim3(256),
                           0, s, M, N, K, A, lda, B, ldb, tiles_n, e);
    };
    auto by_vec = [&](auto ak, auto bk) { vec ? go(ak, bk, std::true_type{}) : go(ak, bk, std::false_type{}); };
    auto by_b = [&](auto ak) { b_kc ? by_vec(ak, std::true_type{}) : by_vec(ak, std::false_type{}); };
    a_kc ? by_b(std::true_type{}) : by_b(std::false_type{});
}

}  // namespace

hipError_t launch_sgemm(int64_t M, int64_t N, int64_t K, const float *A, int64_t lda, int transA, const float *B,
                        int64_t ldb, int transB, const Epilogue &e, hipStream_t s, const char **kernel) {
    *kernel = "lcml_fp8_sgemm_any";
    auto tiles = [&](int64_t t) { return ((M + t - 1) / t) * ((N + t - 1) / t); };
    // The tile, in units of one 16x16 block's chain (32 cycles per four
    // k): a workgroup of 64x64 runs four per SIMD, one of 32x32 one, but
    // no less than the chain's latency (40 cycles).
    const int64_t t64 = tiles(64), t32 = tiles(32), t16 = tiles(16);
    const double c64 = 4.0 * (double)((t64 + 255) / 256), c32 = std::max(1.25, 1.5 * (double)((t32 + 255) / 256));
    const int tb = t16 <= 256 ? 16 : c32 < c64 ? 32 : 64;
    // Few k: the tiles' chunks of 32 to 128 are mostly padding, and three of
    // them are loaded ahead.  M x N x K = 697 x 978 x 1: 4.8 us in general, 5.9
    // by tiles; 59 x 1 x 1: 3.2 and 4.2; 762 x 73 x 6: 4.9 and 4.3, 254 x 33 x 7
    // 4.9 and 4.3.  With many outputs up to K = 10: 3719 x 2932 x 7 23.0 and 27.9,
    // 2812 x 426 x 9 6.5 and 8.9; 3136 x 1455 x 13 15.1 and 14.1.
    const bool few_k = K <= 6 || (K <= 10 && M * N >= ((int64_t)1 << 19));
    // a tile's loads stay within 32-bit buffer extents: 128 rows of pitch
    constexpr int64_t kPitchMax = (int64_t)1 << 22;
    if (!few_k && lda < kPitchMax && ldb < kPitchMax && M < ((int64_t)1 << 30) && N < ((int64_t)1 << 30) &&
        K < ((int64_t)1 << 30) && tiles(tb) <= kGridMax) {
        *kernel = "lcml_fp8_sgemm";
        // 16-byte loads: pointer, pitch and the extent they run along (K, or
        // the operand's rows) whole vectors
        auto whole = [](const float *p, int64_t ld, int64_t extent) {
            return (reinterpret_cast<uintptr_t>(p) & 15) == 0 && ld % 4 == 0 && extent % 4 == 0;
        };
        const bool vec = whole(A, lda, transA ? M : K) && whole(B, ldb, transB ? K : N);
#define LCML_SGEMM(TB)                                                                                            \
    launch_sgemm_tile<TB>((int)M, (int)N, (int)K, A, (int)lda, !transA, B, (int)ldb, transB != 0, vec, e, s)
        if (tb == 16)
            LCML_SGEMM(16);
        else if (tb == 32)
            LCML_SGEMM(32);
        else
            LCML_SGEMM(64);
#undef LCML_SGEMM
        return hipGetLastError();
    }
    dim3 grid((unsigned)((N + TN - 1) / TN), (unsigned)((M + TM - 1) / TM));
    hipLaunchKernelGGL(k_sgemm_any, grid, dim3(256), 0, s, M, N, K, A, lda, transA, B, ldb, transB, e);
    return hipGetLastError();
}

hipError_t launch_activation(const float *x, float *y, int64_t n, int act, hipStream_t s) {
    int64_t g = (n + 255) / 256;
    g = g < 1 ? 1 : (g > 4096 ? 4096 : g);
    hipLaunchKernelGGL(k_activation, dim3((unsigned)g), dim3(256), 0, s, x, y, n, act);
    return hipGetLastError();
}

}  // namespace lcml
