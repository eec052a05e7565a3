// pack.hip -- load-time weight packing into 64-column panels of 16-byte
// k-chunks (the operand-chunk order of the gfx950 FP8 MFMAs) and its inverse.
//
// Packed byte (k, n) of a logical [K, N] weight:
//   ((n / 64) * (Kp / 16) + k / 16) * 1024 + (n % 64) * 16 + k % 16,
// Kp = K rounded up to 128, N rounded up to 64, padding zero.
// One thread owns one 16-byte unit of the packed array, so the packed side
// is written (read) as one contiguous 1 KB run per wavefront.
#include "lcml_internal.hpp"

namespace lcml {
namespace {

typedef uint32_t u4 __attribute__((ext_vector_type(4)));

__global__ __launch_bounds__(256) void k_pack(const uint8_t *__restrict__ w, int64_t K, int64_t N,
                                              int w_is_nk, int64_t KC, int64_t units,
                                              uint8_t *__restrict__ packed) {
    int64_t u = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (u >= units) return;
    int64_t col = u & 63, c = (u >> 6) % KC, panel = (u >> 6) / KC;
    int64_t n = panel * 64 + col, k0 = c * 16;
    u4 out;
    if (w_is_nk && n < N && k0 + 16 <= K) {
        // the unit lies contiguous in row n, at any byte: the five aligned
        // words that cover it, shifted into place (16 single bytes took 89 us
        // on [11008, 4096], 23 us so).  The words hold bytes of w only or of
        // the word that its first or last byte lies in.
        const uintptr_t at = reinterpret_cast<uintptr_t>(w + n * K + k0), off = at & 3;
        const uint32_t *p = reinterpret_cast<const uint32_t *>(at - off);
        const uint32_t w0 = p[0], w1 = p[1], w2 = p[2], w3 = p[3], w4 = off ? p[4] : 0u;
        out.x = __builtin_amdgcn_alignbyte(w1, w0, (uint32_t)off);
        out.y = __builtin_amdgcn_alignbyte(w2, w1, (uint32_t)off);
        out.z = __builtin_amdgcn_alignbyte(w3, w2, (uint32_t)off);
        out.w = __builtin_amdgcn_alignbyte(w4, w3, (uint32_t)off);
    } else {
        uint8_t b[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            int64_t k = k0 + j;
            bool ok = n < N && k < K;
            b[j] = ok ? (w_is_nk ? w[n * K + k] : w[k * N + n]) : (uint8_t)0;
        }
        out.x = b[0] | (b[1] << 8) | (b[2] << 16) | ((uint32_t)b[3] << 24);
        out.y = b[4] | (b[5] << 8) | (b[6] << 16) | ((uint32_t)b[7] << 24);
        out.z = b[8] | (b[9] << 8) | (b[10] << 16) | ((uint32_t)b[11] << 24);
        out.w = b[12] | (b[13] << 8) | (b[14] << 16) | ((uint32_t)b[15] << 24);
    }
    *reinterpret_cast<u4 *>(packed + u * 16) = out;
}

__global__ __launch_bounds__(256) void k_unpack(const uint8_t *__restrict__ packed, int64_t K,
                                                int64_t N, int w_is_nk, int64_t KC, int64_t units,
                                                uint8_t *__restrict__ w) {
    int64_t u = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (u >= units) return;
    int64_t col = u & 63, c = (u >> 6) % KC, panel = (u >> 6) / KC;
    int64_t n = panel * 64 + col, k0 = c * 16;
    if (n >= N) return;
    u4 in = *reinterpret_cast<const u4 *>(packed + u * 16);
    uint32_t words[4] = {in.x, in.y, in.z, in.w};
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        int64_t k = k0 + j;
        if (k < K) {
            uint8_t v = (uint8_t)(words[j >> 2] >> (8 * (j & 3)));
            if (w_is_nk) w[n * K + k] = v;
            else w[k * N + n] = v;
        }
    }
}

}  // namespace

hipError_t launch_pack_weight(const uint8_t *w, int64_t K, int64_t N, int w_is_nk,
                              uint8_t *packed, hipStream_t s) {
    int64_t Kp = pad_to(K, kPackK), Np = pad_to(N, kPanelCols);
    int64_t units = Np * Kp / 16;
    hipLaunchKernelGGL(k_pack, dim3((unsigned)((units + 255) / 256)), dim3(256), 0, s, w, K, N,
                       w_is_nk, Kp / 16, units, packed);
    return hipGetLastError();
}

hipError_t launch_unpack_weight(const uint8_t *packed, int64_t K, int64_t N, int w_is_nk,
                                uint8_t *w, hipStream_t s) {
    int64_t Kp = pad_to(K, kPackK), Np = pad_to(N, kPanelCols);
    int64_t units = Np * Kp / 16;
    hipLaunchKernelGGL(k_unpack, dim3((unsigned)((units + 255) / 256)), dim3(256), 0, s, packed, K,
                       N, w_is_nk, Kp / 16, units, w);
    return hipGetLastError();
}

}  // namespace lcml
