// The passes around the matrix product of QuantizedLinear's backward (python/forge/nn/linear.py:
// 115-132): the FP16 weight it goes through, and the bias gradient.
#include "common.h"
#include "forge_amd.h"

#include <algorithm>
#include <climits>

namespace forge_amd {

// out (K, N) fp16 = transpose of half(w (N, K)) * w_scale[n] (one rounding: an INT8 times an FP16
// is exact in FP32). Transposed, because the library product that follows runs 7 % faster with both
// operands contiguous along the sum (2048 x 4096 x 4096 76.6 -> 71.6 us). Bound: memory, w read and
// out written once; 64 x 64 tiles through LDS keep both sides in whole 64- and 128-byte runs.
// torch's conversion and product over the same weights took 28 + 14 us at 4096 x 4096, this 13.
template <bool VEC>
__global__ __launch_bounds__(256) void dequantize_weight_t_kernel(const int8_t* __restrict__ w,
                                                                  const uint16_t* __restrict__ w_scale,
                                                                  uint16_t* __restrict__ out, int N, int K,
                                                                  unsigned tiles_k, unsigned tiles)
{
    constexpr int kT = 64, kPitch = kT + 4;
    __shared__ __align__(16) int8_t tile[kT * kPitch];
    const int t = threadIdx.x;
    // 64 x 64 tiles numbered along K first over both grid dimensions, which alone end at 65535 rows of tiles
    const unsigned id = blockIdx.y * gridDim.x + blockIdx.x;
    if (id >= tiles) return;
    const int n0 = static_cast<int>(id / tiles_k) * kT, k0 = static_cast<int>(id % tiles_k) * kT;
    {
        const int r = t >> 2, c = 16 * (t & 3);        // 16 bytes of row n0 + r
        const int n = n0 + r, k = k0 + c;
        uint32_t v[4] = {0u, 0u, 0u, 0u};
        if (n < N) {
            const int8_t* src = w + static_cast<size_t>(n) * K + k;
            if (VEC && k + 16 <= K) {
                const uint4 q = *reinterpret_cast<const uint4*>(src);
                v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
            } else {
#pragma unroll
                for (int b = 0; b < 16; b++)
                    if (k + b < K) v[b >> 2] |= static_cast<uint32_t>(static_cast<uint8_t>(src[b])) << (8 * (b & 3));
            }
        }
#pragma unroll
        for (int d = 0; d < 4; d++) *reinterpret_cast<uint32_t*>(tile + r * kPitch + c + 4 * d) = v[d];
    }
    __syncthreads();
    // thread: 8 weight rows of 2 columns k; 8 adjacent threads write one column's 128 bytes
    const int nb = 8 * (t & 7), n = n0 + nb;
    float s[8];
#pragma unroll
    for (int j = 0; j < 8; j++) s[j] = h2f(w_scale[min(n + j, N - 1)]);
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const int kc = (t >> 3) + 32 * h, k = k0 + kc;
        if (k >= K) continue;
        uint16_t o[8];
#pragma unroll
        for (int j = 0; j < 8; j++) o[j] = f2h(static_cast<float>(tile[(nb + j) * kPitch + kc]) * s[j]);
        uint16_t* dst = out + static_cast<size_t>(k) * N + n;
        if (n + 8 <= N) {
            typedef uint32_t u4 __attribute__((ext_vector_type(4), aligned(2)));
            *reinterpret_cast<u4*>(dst) = u4{o[0] | static_cast<uint32_t>(o[1]) << 16, o[2] | static_cast<uint32_t>(o[3]) << 16,
                                             o[4] | static_cast<uint32_t>(o[5]) << 16, o[6] | static_cast<uint32_t>(o[7]) << 16};
        } else {
#pragma unroll
            for (int j = 0; j < 8; j++)
                if (n + j < N) dst[j] = o[j];
        }
    }
}

// Column sums of g (M, N) fp16 in FP32, over the rows of part blockIdx.y, to partial (parts, N).
// A thread sums 8 columns (16-byte loads at element alignment; the last group moved back to end
// with the row, so that it sums some columns once more, to the same value) of every 4th row, four
// loads in flight. 2048 x 4096, kernel times: 8.0 us and 3.5 for the second kernel, torch's
// column sum 14.6 and the 4.6 us fill that goes with it.
__global__ __launch_bounds__(256) void column_sum_kernel(const uint16_t* __restrict__ g, float* __restrict__ partial,
                                                         int M, int N, int rows)
{
    __shared__ float part[3][64][9];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int grp = blockIdx.x * 64 + lane;
    const bool ok = 8 * grp < N;
    const int c = min(8 * grp, N - 8);
    const int r0 = blockIdx.y * rows, r1 = min(M, r0 + rows);
    float acc[8];
#pragma unroll
    for (int j = 0; j < 8; j++) acc[j] = 0.0f;
    if (ok) {
        typedef uint32_t u4 __attribute__((ext_vector_type(4), aligned(2)));
        for (int r = r0 + wave; r < r1; r += 16) {
            u4 v[4];
#pragma unroll
            for (int u = 0; u < 4; u++)
                v[u] = *reinterpret_cast<const u4*>(g + static_cast<size_t>(min(r + 4 * u, r1 - 1)) * N + c);
#pragma unroll
            for (int u = 0; u < 4; u++) {
                if (r + 4 * u >= r1) break;
#pragma unroll
                for (int d = 0; d < 4; d++) {
                    acc[2 * d] += h2f(static_cast<uint16_t>(v[u][d] & 0xFFFFu));
                    acc[2 * d + 1] += h2f(static_cast<uint16_t>(v[u][d] >> 16));
                }
            }
        }
    }
    if (wave > 0) {
#pragma unroll
        for (int j = 0; j < 8; j++) part[wave - 1][lane][j] = acc[j];
    }
    __syncthreads();
    if (wave == 0 && ok) {
#pragma unroll
        for (int j = 0; j < 8; j++)
            partial[static_cast<size_t>(blockIdx.y) * N + c + j] = (acc[j] + part[0][lane][j]) + (part[1][lane][j] + part[2][lane][j]);
    }
}

__global__ __launch_bounds__(256) void column_sum_finish_kernel(const float* __restrict__ partial, uint16_t* __restrict__ out,
                                                                int N, int parts)
{
    const int n = blockIdx.x * 256 + threadIdx.x;
    if (n >= N) return;
    float s = 0.0f;
    for (int p = 0; p < parts; p += 8) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = p + u < parts ? partial[static_cast<size_t>(p + u) * N + n] : 0.0f;
#pragma unroll
        for (int u = 0; u < 8; u++) s += v[u];
    }
    out[n] = f2h(s);
}

}  // namespace forge_amd

using namespace forge_amd;

extern "C" int forge_int8_linear_backward_prep(const int8_t* w, const uint16_t* w_scale, uint16_t* w16t,
                                               const uint16_t* grad, float* partial, uint16_t* grad_bias, int M, int K,
                                               int N, void* stream)
{
    // No columns of the weight (K = 0): nothing to convert. No rows of the gradient (M = 0): its sums are 0.
    if (M < 0 || N <= 0 || K < 0) return FORGE_OK;
    if (!w_scale || (K > 0 && (!w || !w16t)) || (grad_bias && (!partial || N < 8 || (M > 0 && !grad)))) return FORGE_EINVAL;
    hipStream_t s = as_stream(stream);
    int st = FORGE_OK;
    if (K > 0) {
        const long long tiles_k = divup(K, 64), tiles = tiles_k * divup(N, 64);
        if (tiles > INT_MAX) return FORGE_EINVAL;
        const unsigned gx = static_cast<unsigned>(std::min<long long>(tiles, 1 << 16));
        const dim3 grid(gx, static_cast<unsigned>(divupll(tiles, gx)));
        const unsigned tk = static_cast<unsigned>(tiles_k), nt = static_cast<unsigned>(tiles);
        if (K % 16 == 0 && aligned(w, 16))
            dequantize_weight_t_kernel<true><<<grid, 256, 0, s>>>(w, w_scale, w16t, N, K, tk, nt);
        else
            dequantize_weight_t_kernel<false><<<grid, 256, 0, s>>>(w, w_scale, w16t, N, K, tk, nt);
        if ((st = launch_status()) != FORGE_OK) return st;
    }
    if (!grad_bias) return FORGE_OK;
    // 16 rows a pass of a workgroup's four waves; FORGE_COLUMN_SUM_PARTS parts at most
    const int rows = std::max(16, divup(divup(M, FORGE_COLUMN_SUM_PARTS), 16) * 16), parts = divup(M, rows);
    if (parts > 0)
        column_sum_kernel<<<dim3(static_cast<unsigned>(divup(N, 512)), static_cast<unsigned>(parts)), 256, 0, s>>>(
            grad, partial, M, N, rows);
    if ((st = launch_status()) != FORGE_OK) return st;
    column_sum_finish_kernel<<<static_cast<unsigned>(divup(N, 256)), 256, 0, s>>>(partial, grad_bias, N, parts);
    return launch_status();
}
