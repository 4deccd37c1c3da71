// Dense INT8 GEMM for gfx950: C = A (M,K) x B (N,K)^T with exact INT32 accumulation on the matrix
// cores, and the fused dequant + bias epilogue to FP16. This file chooses the engine and holds the
// register-staged one (v_mfma_i32_32x32x32_i8; the ring-fed tiles use v_mfma_i32_16x16x64_i8).
//
// Reference: src/gemm/int8_dense.cu:26-232 (wmma 16x16x16, 128x64 / 128x128 tiles,
// unpipelined global->smem loads) and src/gemm/int8_gemm.cu:12-46 (dispatch). The
// epilogue arithmetic follows int8_dense.cu:171-174:
//     Y[m,n] = half(fma((float)acc, act_scale[m] * w_scale[n], bias[n]))
// 16-byte aligned operands with K % 16 == 0, and conv gathers with C % 16 == 0, run on the
// ring-fed tiles (gemm_ring.hip); other shapes, and operands of 2 GiB and more, on the
// register-staged engine (mfma_tile.h).
// Tiles are mapped XCD-aware. Skinny M (decode) goes to gemm_skinny.
#include "common.h"
#include "mfma_tile.h"
#include "gemm_dense.h"
#include "forge/gemm/int8_dense.h"
#include "forge/gemm/int8_gemm.h"
#include "forge/gemm/int8_dp4a.h"

#include <algorithm>
#include <type_traits>

namespace forge_amd {

// LDS bytes a tile needs: its K loop or the epilogue staging, whichever is larger.
template <class Tile, int BM, int BN, bool DEQUANT>
constexpr int tile_lds_bytes() {
    constexpr int epi = epilogue_lds_bytes<BM, BN, DEQUANT>();
    return Tile::kLdsBytes > epi ? Tile::kLdsBytes : epi;
}

// Register-staged engine: any operand type (row-major, conv gather, byte gathers).
template <int BM, int BN, bool EVEN_K, bool DEQUANT, class OpA, class OpB>
__global__ __launch_bounds__(kGemmThreads) void gemm_nt_kernel(
    OpA opa, OpB opb, GemmEpilogue ep, int tiles_m, int tiles_n, int K)
{
    extern __shared__ __align__(16) int8_t lds[];
    int tm, tn;
    tile_coords(blockIdx.x, tiles_m, tiles_n, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN;
    NtTile<BM, BN> t;
    t.template run<EVEN_K>(opa, opb, m0, n0, K, lds);
    store_tile<BM, BN, DEQUANT>(t.acc, ep, m0, n0, lds);
}

// Raises a kernel's dynamic-LDS limit once (host-side attribute; safe under graph capture).
template <class Kern>
static int allow_lds(Kern kern, int bytes) {
    if (bytes <= 65536) return FORGE_OK;
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    return e == hipSuccess ? FORGE_OK : static_cast<int>(e);
}

template <int BM, int BN, bool EVEN_K, bool DEQUANT, class OpA, class OpB>
static int launch_tile(const OpA& opa, const OpB& opb, const GemmEpilogue& ep, int M, int N, int K,
                       hipStream_t s)
{
    constexpr int lds = tile_lds_bytes<NtTile<BM, BN>, BM, BN, DEQUANT>();
    const int tiles_m = divup(M, BM), tiles_n = divup(N, BN);
    const long long total = static_cast<long long>(tiles_m) * tiles_n;
    if (total > 0x7FFFFFFFLL) return FORGE_EINVAL;
    auto kern = gemm_nt_kernel<BM, BN, EVEN_K, DEQUANT, OpA, OpB>;
    static const int attr = allow_lds(kern, lds);
    if (attr != FORGE_OK) return attr;
    gemm_nt_kernel<BM, BN, EVEN_K, DEQUANT, OpA, OpB>
        <<<static_cast<unsigned>(total), kGemmThreads, lds, s>>>(opa, opb, ep, tiles_m, tiles_n, K);
    return launch_status();
}

// Tile choice: the largest tile whose grid still covers the chip's CUs; smaller tiles
// trade MFMA efficiency (operand reuse) for parallelism.
enum class TileCfg { k256, k128, k64 };

static TileCfg pick_tile(int M, int N, int cu) {
    const long long t256 = static_cast<long long>(divup(M, 256)) * divup(N, 256);
    const long long t128 = static_cast<long long>(divup(M, 128)) * divup(N, 128);
    // A side of 128 or less would leave half of a 256 tile (two of its four waves) idle.
    if (t256 * 2 >= cu && M > 128 && N > 128) return TileCfg::k256;
    if (t128 * 2 >= cu) return TileCfg::k128;
    return TileCfg::k64;
}

static int cu_count(int* st) {
    const DeviceInfo& d = device_info(st);
    return d.cu_count;
}

// MAX256: whether the 256 x 256 tile may be used (the byte-gather operands of odd shapes
// would spill registers at that size).
template <bool EVEN_K, bool DEQUANT, bool MAX256 = true, class OpA, class OpB>
static int dispatch_tiles(const OpA& opa, const OpB& opb, const GemmEpilogue& ep, int M, int N, int K,
                          hipStream_t s)
{
    int st = FORGE_OK;
    const int cu = cu_count(&st);
    if (st != FORGE_OK) return st;
    TileCfg t = pick_tile(M, N, cu);
    note_route(t == TileCfg::k256 && MAX256 ? "regstaged256" : t == TileCfg::k64 ? "regstaged64" : "regstaged128");
    if constexpr (MAX256) {
        if (t == TileCfg::k256) return launch_tile<256, 256, EVEN_K, DEQUANT>(opa, opb, ep, M, N, K, s);
    } else {
        if (t == TileCfg::k256) t = TileCfg::k128;
    }
    if (t == TileCfg::k128) return launch_tile<128, 128, EVEN_K, DEQUANT>(opa, opb, ep, M, N, K, s);
    return launch_tile<64, 64, EVEN_K, DEQUANT>(opa, opb, ep, M, N, K, s);
}

template <bool DEQUANT, class OpA, class OpB>
static int dispatch_k(const OpA& opa, const OpB& opb, const GemmEpilogue& ep, int M, int N, int K,
                      bool even_k, hipStream_t s)
{
    if (even_k) return dispatch_tiles<true, DEQUANT>(opa, opb, ep, M, N, K, s);
    return dispatch_tiles<false, DEQUANT>(opa, opb, ep, M, N, K, s);
}

int launch_conv_gemm(const ConvGeom& g, const int8_t* w, const GemmEpilogue& ep, int Co, bool vec,
                     hipStream_t s)
{
    const int M = g.rows, K = g.K;
    if (vec) {
        int r = launch_conv_window(g, w, ep, Co, s);
        if (r == -1) r = launch_ring_conv(g, w, ep, s);
        if (r != -1) return r;
    }
    if (vec) {
        ConvOperand a;
        static_cast<ConvGeom&>(a) = g;
        RowMajorOperand b{w, Co, K};
        const bool even = K % kBK == 0;
        return ep.c16 ? dispatch_k<true>(a, b, ep, M, Co, K, even, s)
                      : dispatch_k<false>(a, b, ep, M, Co, K, even, s);
    }
    ConvBytes a;
    static_cast<ConvGeom&>(a) = g;
    if (K < 16) {
        RowMajorShort b{w, Co, K};
        return ep.c16 ? dispatch_tiles<false, true, false>(a, b, ep, M, Co, K, s)
                      : dispatch_tiles<false, false, false>(a, b, ep, M, Co, K, s);
    }
    RowMajorBytes b{w, Co, K};
    return ep.c16 ? dispatch_tiles<false, true, false>(a, b, ep, M, Co, K, s)
                  : dispatch_tiles<false, false, false>(a, b, ep, M, Co, K, s);
}

// Whether 16-byte row stores of the output are possible.
static int out_vec(const void* out, int N, int esz) {
    return aligned(out, 16) && (static_cast<long long>(N) * esz) % 16 == 0 ? 1 : 0;
}

int gemm_dense(const int8_t* A, const int8_t* B, const float* act_scale, const uint16_t* w_scale,
               const uint16_t* bias, uint16_t* out16, int32_t* out32, int M, int K, int N,
               hipStream_t s)
{
    const bool vec = (K % 16 == 0) && aligned(A, 16) && aligned(B, 16);
    GemmEpilogue ep{out32, out16, act_scale, w_scale, bias, M, N,
                    out16 ? out_vec(out16, N, 2) : out_vec(out32, N, 4)};
    if (vec && decode_supported(M, K)) {
        note_route("decode");
        return launch_decode(B, nullptr, A, ep, K, false, s);
    }
    if (M <= kSkinnyMaxM && vec) {
        note_route("skinny");
        return launch_gemm_skinny(A, B, ep, M, K, N, s);
    }
    if (vec && M <= kSkinnyTbMaxM) {
        // 16 < M <= 64, narrow N, deep K: the tile engine has too few tiles (M = 64, K = 6144,
        // N = 1536: 29.4 us on 64 x 64 tiles, 11.6 us on token blocks with K split in two).
        int st = FORGE_OK;
        const DeviceInfo& di = device_info(&st);
        if (st != FORGE_OK) return st;
        if (dense_tb_supported(M, K, N, di.cu_count)) {
            note_route("token-block");
            return launch_dense_tb(B, A, ep, K, di.cu_count, s);
        }
    }
    return gemm_tiles(A, B, ep, M, K, N, s);
}

int gemm_tiles(const int8_t* A, const int8_t* B, const GemmEpilogue& ep, int M, int K, int N, hipStream_t s)
{
    const bool vec = (K % 16 == 0) && aligned(A, 16) && aligned(B, 16);
    const bool out16 = ep.c16 != nullptr;
    if (vec) {
        const int r = launch_ring_gemm(A, B, ep, K, s);
        if (r != -1) return r;
        RowMajorOperand a{A, M, K}, b{B, N, K};
        const bool even = K % kBK == 0;
        return out16 ? dispatch_k<true>(a, b, ep, M, N, K, even, s) : dispatch_k<false>(a, b, ep, M, N, K, even, s);
    }
    if (K < 16) {
        RowMajorShort a{A, M, K}, b{B, N, K};
        return out16 ? dispatch_tiles<false, true, false>(a, b, ep, M, N, K, s)
                     : dispatch_tiles<false, false, false>(a, b, ep, M, N, K, s);
    }
    RowMajorBytes a{A, M, K}, b{B, N, K};
    return out16 ? dispatch_tiles<false, true, false>(a, b, ep, M, N, K, s)
                 : dispatch_tiles<false, false, false>(a, b, ep, M, N, K, s);
}

}  // namespace forge_amd

using namespace forge_amd;

extern "C" int forge_int8_gemm_dequant(const int8_t* A, const int8_t* B, const float* act_scale,
                                       const uint16_t* w_scale, const uint16_t* bias, uint16_t* out,
                                       int M, int K, int N, void* stream)
{
    if (M <= 0 || K <= 0 || N <= 0) return FORGE_OK;
    if (!A || !B || !act_scale || !w_scale || !out) return FORGE_EINVAL;
    return gemm_dense(A, B, act_scale, w_scale, bias, out, nullptr, M, K, N, as_stream(stream));
}

extern "C" int forge_int8_gemm(const int8_t* A, const int8_t* B, const float* act_scale,
                               const uint16_t* w_scale, const uint16_t* bias, uint16_t* out,
                               int M, int K, int N, void* stream)
{
    return forge_int8_gemm_dequant(A, B, act_scale, w_scale, bias, out, M, K, N, stream);
}

extern "C" int forge_int8_gemm_s32(const int8_t* A, const int8_t* B, int32_t* C,
                                   int M, int K, int N, void* stream)
{
    if (M <= 0 || K <= 0 || N <= 0) return FORGE_OK;
    if (!A || !B || !C) return FORGE_EINVAL;
    return gemm_dense(A, B, nullptr, nullptr, nullptr, nullptr, C, M, K, N, as_stream(stream));
}

extern "C" int forge_int8_linear(const uint16_t* x, const int8_t* w, const uint16_t* w_scale,
                                 const uint16_t* bias, uint16_t* out, int M, int K, int N,
                                 int8_t* scratch_q, float* scratch_scale, void* stream)
{
    if (M <= 0 || K <= 0 || N <= 0) return FORGE_OK;
    if (!x || !w || !w_scale || !out || !scratch_q || !scratch_scale) return FORGE_EINVAL;
    hipStream_t s = as_stream(stream);
    // Decode shapes: one kernel, the quantize fused into the decode GEMM's prologue (each
    // workgroup quantizes the few token rows itself while its first weight stages stream in).
    if (decode_fq_supported(M, K, false) && aligned(x, 16) && aligned(w, 16) && aligned(scratch_q, 8)) {
        note_route("decode+quantize");
        return launch_decode_fq(x, w, nullptr, w_scale, bias, out, scratch_q, scratch_scale, M, K, N, false, s);
    }
    int st = launch_quantize(x, scratch_q, scratch_scale, M, K, s);
    if (st != FORGE_OK) return st;
    return gemm_dense(scratch_q, w, scratch_scale, w_scale, bias, out, nullptr, M, K, N, s);
}
