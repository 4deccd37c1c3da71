// Dense INT8 GEMMs and NHWC conv gathers on the ring-fed tiles of ring_tile.h, and the choice of
// the tile.
#include "common.h"
#include "gemm_dense.h"
#include "ring_tile.h"

#include <cstdio>

namespace forge_amd {

namespace {

// ---- tile shapes --------------------------------------------------------------------------
// The cost of a call, in us, by the tiles on its busiest CU: a tile costs stages * a + b, and of
// the tiles that share a CU (`per_cu`, what the LDS holds) a full round costs stages * a + b
// together, a round of one stages * a1 + b1, of two stages * a2 + b2. The constants are
// non-negative least-squares fits of every shape's time on 100 GEMMs (M 19-8192, K 128-6144,
// N 64-11008) on MI355X, launch overhead taken as 2 us. On those shapes the pick costs 1 % over
// the fastest of 21 shapes tried (11 % at worst), and the shapes beyond these twelve gain
// nothing: 64 x 96, 96 x 96, 128 x 64, 64 x 256 and 4-wave forms of the larger ones.
struct RingShape {
    int bm, bn, per_cu;
    float a, b, a1, b1, a2, b2;
};
enum { k64x64, k64x128, k64x192, k128x128, k128x128deep, k192x128, k128x192, k128x256, k192x192, k192x256, k256x192,
       k256x256, kRingShapes };
constexpr RingShape kShapes[kRingShapes] = {
    {64, 64, 3, 0.596f, 1.72f, 0.255f, 1.07f, 0.402f, 1.31f},
    {64, 128, 1, 0.326f, 1.64f},
    {64, 192, 1, 0.415f, 1.97f},
    {128, 128, 2, 0.893f, 3.00f, 0.600f, 1.30f},
    {128, 128, 1, 0.453f, 2.30f},
    {192, 128, 1, 0.572f, 2.61f},
    {128, 192, 1, 0.566f, 3.00f},
    {128, 256, 1, 0.717f, 3.24f},
    {192, 192, 1, 0.732f, 4.35f},
    {192, 256, 1, 1.046f, 3.82f},
    {256, 192, 1, 1.060f, 3.91f},
    {256, 256, 1, 1.204f, 4.60f},
};
using T64x64 = RingTile<64, 64, 2, 2, 3>;
using T64x128 = RingTile<64, 128, 2, 4, 4>;
using T64x192 = RingTile<64, 192, 2, 4, 3>;
using T128x128 = RingTile<128, 128, 2, 4, 2>;
using T128x128deep = RingTile<128, 128, 2, 4, 4>;
using T192x128 = RingTile<192, 128, 4, 2, 3>;
using T128x192 = RingTile<128, 192, 2, 4, 3>;
using T128x256 = RingTile<128, 256, 2, 4, 3>;
using T192x192 = RingTile<192, 192, 4, 2, 3>;
using T192x256 = RingTile<192, 256, 4, 2, 2>;
using T256x192 = RingTile<256, 192, 4, 2, 2>;
using T256x256 = RingTile<256, 256, 4, 2, 2>;

float ring_cost(const RingShape& t, int M, int N, int stages, int cu) {
    const long long tiles = static_cast<long long>(divup(M, t.bm)) * divup(N, t.bn);
    const long long w = (tiles + cu - 1) / cu, full = w / t.per_cu;
    float us = static_cast<float>(full) * (stages * t.a + t.b);
    if (w % t.per_cu == 1 && t.per_cu > 1) us += stages * t.a1 + t.b1;
    if (w % t.per_cu == 2) us += stages * t.a2 + t.b2;
    return us;
}

int ring_pick(int M, int N, int K, int cu, unsigned allowed, float* cost) {
    const int stages = divup(K, kBK);
    int best = -1;
    for (int i = 0; i < kRingShapes; i++) {
        if (!(allowed >> i & 1u)) continue;
        const float c = ring_cost(kShapes[i], M, N, stages, cu);
        if (best < 0 || c < *cost) {
            best = i;
            *cost = c;
        }
    }
    return best;
}

}  // namespace

// ---- kernels ------------------------------------------------------------------------------

template <class T, bool DEQUANT, bool UP, class OpA, class OpB>
__device__ __forceinline__ void ring_tile_at(const OpA& opa, const OpB& opb, const GemmEpilogue& ep,
                                             int K, int m0, int n0, int8_t* lds)
{
    T t;
    // XCD x starts x / 8 into K (the INT32 sums do not depend on the order): the XCDs, which read
    // the same weights, then ask memory for different lines at any time. Weights not in the MALL,
    // 1024 x 6144 x 1536: 22.9 -> 19.6 us, 1500 x 2880 x 2880 23.6 -> 21.9; in the MALL level.
    const int rot = (blockIdx.x % 8) * ((K + kBK - 1) / kBK) / 8;
    t.run(opa, opb, K, m0, n0, rot, lds);
    const int wave = threadIdx.x / kWave;
    ring_store<T, DEQUANT, UP>(t, ep, m0 + (wave / T::kWN) * (T::kBM / T::kWM), n0 + (wave % T::kWN) * (T::kBN / T::kWN),
                               lds + wave * ring_epilogue_wave_bytes<T, DEQUANT>());
}

// tile_coords, with the tile columns of each group of tile rows (an XCD's share, in large grids)
// started at its own eighth of them, for the same reason: with 32 tile rows every XCD otherwise walks
// the same columns in step (8192 x 4096 x 11008, weights not in the MALL: 337 -> 301 us with
// both shifts, 295 against 298 us in the MALL).
__device__ __forceinline__ void ring_coords(int bid, int tiles_m, int tiles_n, int& tm, int& tn)
{
    tile_coords(bid, tiles_m, tiles_n, tm, tn);
    tn += (tm / kGroupM % 8) * tiles_n / 8;
    tn = tn < tiles_n ? tn : tn - tiles_n;
}

template <class T, bool DEQUANT, bool UP, class OpA, class OpB>
__global__ __launch_bounds__(T::kThreads) void gemm_ring_kernel(OpA opa, OpB opb, GemmEpilogue ep,
                                                                int tiles_m, int tiles_n, int K)
{
    extern __shared__ __align__(16) int8_t lds[];
    int tm, tn;
    ring_coords(blockIdx.x, tiles_m, tiles_n, tm, tn);
    ring_tile_at<T, DEQUANT, UP>(opa, opb, ep, K, tm * T::kBM, tn * T::kBN, lds);
}

// Whole waves of 256 x 256 tiles over the first nb1 tile columns (workgroups [0, n1)), then the
// remaining columns as one wave of 192-row tiles, in one launch: workgroups start in index order,
// so a CU takes its 192-row tile as soon as its last 256-row tile ends.
template <bool DEQUANT>
__global__ __launch_bounds__(T256x256::kThreads) void gemm_ring_tail_kernel(RingRowMajor opa, RingRowMajor opb,
                                                                            GemmEpilogue ep, int n1, int nb1,
                                                                            int tiles_m, int tiles_m2, int tiles_n,
                                                                            int K)
{
    extern __shared__ __align__(16) int8_t lds[];
    int tm, tn;
    const int bid = static_cast<int>(blockIdx.x);
    if (bid < n1) {
        ring_coords(bid, tiles_m, nb1, tm, tn);
        ring_tile_at<T256x256, DEQUANT, false>(opa, opb, ep, K, tm * 256, tn * 256, lds);
    } else {
        ring_coords(bid - n1, tiles_m2, tiles_n - nb1, tm, tn);
        ring_tile_at<T192x256, DEQUANT, false>(opa, opb, ep, K, tm * 192, (nb1 + tn) * 256, lds);
    }
}

// Raises a kernel's dynamic-LDS limit once (host-side attribute; safe under graph capture).
template <class Kern>
static int ring_allow_lds(Kern kern, int lds) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    return e == hipSuccess ? FORGE_OK : static_cast<int>(e);
}

template <class T, bool DEQUANT, bool UP, class OpA, class OpB>
static int launch_ring_tile(const OpA& opa, const OpB& opb, const GemmEpilogue& ep, int K,
                            hipStream_t s)
{
    constexpr int lds = ring_lds_bytes<T, DEQUANT>();
    static_assert(lds <= 160 * 1024, "LDS of one CU");
    const int tiles_m = divup(ep.M, T::kBM), tiles_n = divup(ep.N, T::kBN);
    const long long total = static_cast<long long>(tiles_m) * tiles_n;
    if (total > 0x7FFFFFFFLL) return FORGE_EINVAL;
    auto kern = gemm_ring_kernel<T, DEQUANT, UP, OpA, OpB>;
    static const int attr = ring_allow_lds(kern, lds);
    if (attr != FORGE_OK) return attr;
    kern<<<static_cast<unsigned>(total), T::kThreads, lds, s>>>(opa, opb, ep, tiles_m, tiles_n, K);
    return launch_status();
}

// The column tail split: more than one wave of 256 x 256 tiles but not whole waves, row tiles
// that divide the CUs (so the first columns make whole waves), and a remainder that is one wave of
// 192-row tiles. n1 = 0 where it does not apply.
struct RingTail {
    int n1, nb1, tiles_m, tiles_m2, tiles_n;
};
static RingTail ring_tail(int M, int N, int cu)
{
    RingTail t{0, 0, divup(M, 256), divup(M, 192), divup(N, 256)};
    const long long tiles = static_cast<long long>(t.tiles_m) * t.tiles_n;
    if (tiles <= cu || tiles % cu == 0 || cu % t.tiles_m != 0 || M < 192 || tiles > 0x7FFFFFFFLL) return t;
    t.nb1 = static_cast<int>(tiles / cu * cu / t.tiles_m);
    if (t.nb1 >= t.tiles_n || static_cast<long long>(t.tiles_n - t.nb1) * t.tiles_m2 > cu) return t;
    t.n1 = t.nb1 * t.tiles_m;
    return t;
}

template <bool DEQUANT>
static int launch_ring_tail(const RingRowMajor& opa, const RingRowMajor& opb, const GemmEpilogue& ep, int K,
                            const RingTail& t, hipStream_t s)
{
    constexpr int l1 = ring_lds_bytes<T256x256, DEQUANT>(), l2 = ring_lds_bytes<T192x256, DEQUANT>();
    constexpr int lds = l1 > l2 ? l1 : l2;
    const long long total = t.n1 + static_cast<long long>(t.tiles_n - t.nb1) * t.tiles_m2;
    auto kern = gemm_ring_tail_kernel<DEQUANT>;
    static const int attr = ring_allow_lds(kern, lds);
    if (attr != FORGE_OK) return attr;
    kern<<<static_cast<unsigned>(total), T256x256::kThreads, lds, s>>>(opa, opb, ep, t.n1, t.nb1, t.tiles_m, t.tiles_m2,
                                                                      t.tiles_n, K);
    return launch_status();
}

static void note_shape(int shape)
{
    char name[24];
    snprintf(name, sizeof name, "dma%dx%d%s", kShapes[shape].bm, kShapes[shape].bn, shape == k128x128deep ? " 4-slot" : "");
    note_route(name);
}

// Every shape but 256 x 256.
template <bool DEQUANT, class OpA, class OpB>
static int launch_ring_shape(int shape, const OpA& opa, const OpB& opb, const GemmEpilogue& ep, int K,
                             hipStream_t s)
{
    switch (shape) {
        case k64x64: return launch_ring_tile<T64x64, DEQUANT, false>(opa, opb, ep, K, s);
        case k64x128: return launch_ring_tile<T64x128, DEQUANT, false>(opa, opb, ep, K, s);
        case k64x192: return launch_ring_tile<T64x192, DEQUANT, false>(opa, opb, ep, K, s);
        case k128x128: return launch_ring_tile<T128x128, DEQUANT, false>(opa, opb, ep, K, s);
        case k128x128deep: return launch_ring_tile<T128x128deep, DEQUANT, false>(opa, opb, ep, K, s);
        case k192x128: return launch_ring_tile<T192x128, DEQUANT, false>(opa, opb, ep, K, s);
        case k128x192: return launch_ring_tile<T128x192, DEQUANT, false>(opa, opb, ep, K, s);
        case k128x256: return launch_ring_tile<T128x256, DEQUANT, false>(opa, opb, ep, K, s);
        case k192x192: return launch_ring_tile<T192x192, DEQUANT, false>(opa, opb, ep, K, s);
        case k192x256: return launch_ring_tile<T192x256, DEQUANT, false>(opa, opb, ep, K, s);
        case k256x192: return launch_ring_tile<T256x192, DEQUANT, false>(opa, opb, ep, K, s);
        default: return FORGE_EINVAL;
    }
}

static int launch_ring(const RingRowMajor& opa, const int8_t* B, const GemmEpilogue& ep, int K, hipStream_t s)
{
    int st = FORGE_OK;
    const int cu = device_info(&st).cu_count;
    if (st != FORGE_OK) return st;
    const RingRowMajor opb{B, ep.N, K};
    float cost = 0.0f;
    const int shape = ring_pick(ep.M, ep.N, K, cu, (1u << kRingShapes) - 1, &cost);
    const RingTail t = ring_tail(ep.M, ep.N, cu);
    if (t.n1 > 0) {
        // The sum of the two costs overstates the split (the first 192-row tiles run while the last
        // 256-row ones still store), so it is taken up to 1.2 of the best single shape's. Measured
        // (us, split / best single shape): 4096 x 4096 x 11008 149 / 153, 4096 x 6144 x 6144
        // 128 / 130, 8192 x 1280 x 5120 60.0 / 61.6; beyond the line 1024 x 4096 x 18000
        // (1.27) 88 / 79, 2048 x 2048 x 9000 (1.23) 53 / 46.
        const int stages = divup(K, kBK);
        const float tail = static_cast<float>(t.n1 / cu) * (stages * kShapes[k256x256].a + kShapes[k256x256].b) +
                           stages * kShapes[k192x256].a + kShapes[k192x256].b;
        if (tail <= 1.2f * cost) {
            note_route("dma256x256+tail192");
            return ep.c16 ? launch_ring_tail<true>(opa, opb, ep, K, t, s) : launch_ring_tail<false>(opa, opb, ep, K, t, s);
        }
    }
    note_shape(shape);
    if (shape == k256x256)
        return ep.c16 ? launch_ring_tile<T256x256, true, false>(opa, opb, ep, K, s)
                      : launch_ring_tile<T256x256, false, false>(opa, opb, ep, K, s);
    return ep.c16 ? launch_ring_shape<true>(shape, opa, opb, ep, K, s)
                  : launch_ring_shape<false>(shape, opa, opb, ep, K, s);
}

int launch_ring_gemm(const int8_t* A, const int8_t* B, const GemmEpilogue& ep, int K, hipStream_t s)
{
    // both operands as buffer resources with 32-bit offsets
    if (static_cast<long long>(ep.M) * K >= (1LL << 31) || static_cast<long long>(ep.N) * K >= (1LL << 31)) return -1;
    const RingRowMajor opa{A, ep.M, K};
    if (ep.up_w == 0) return launch_ring(opa, B, ep, K, s);
    // the upsample scatter: the three square shapes
    int st = FORGE_OK;
    const int cu = device_info(&st).cu_count;
    if (st != FORGE_OK) return st;
    const RingRowMajor opb{B, ep.N, K};
    float cost = 0.0f;
    const int shape = ring_pick(ep.M, ep.N, K, cu, 1u << k64x64 | 1u << k128x128 | 1u << k256x256, &cost);
    note_route(shape == k64x64 ? "dma64x64 scatter" : shape == k128x128 ? "dma128x128 scatter" : "dma256x256 scatter");
    if (shape == k64x64) return launch_ring_tile<T64x64, true, true>(opa, opb, ep, K, s);
    if (shape == k128x128) return launch_ring_tile<T128x128, true, true>(opa, opb, ep, K, s);
    return launch_ring_tile<T256x256, true, true>(opa, opb, ep, K, s);
}

int launch_ring_conv(const ConvGeom& g, const int8_t* w, const GemmEpilogue& ep, hipStream_t s)
{
    const int K = g.K;
    const long long img = static_cast<long long>(g.rows / (g.Ho * g.Wo)) * g.H * g.W * g.C;
    // one buffer resource per operand, and udiv_magic's range for the chunk, tap and pixel divisions
    const long long k_end = static_cast<long long>(K) + 8 * kBK;
    if (img >= (1LL << 31) || static_cast<long long>(ep.N) * K >= (1LL << 31) || K > (1 << 30) ||
        k_end * g.C >= (1LL << 32) || (k_end / g.C + 1) * g.kW >= (1LL << 32) ||
        static_cast<long long>(g.rows) * (g.Ho > g.Wo ? g.Ho : g.Wo) >= (1LL << 32))
        return -1;
    RingConv a;
    static_cast<ConvGeom&>(a) = g;
    a.x_bytes = static_cast<uint32_t>(img);
    a.mg_c = udiv_multiplier(g.C);
    a.mg_kw = udiv_multiplier(g.kW);
    a.mg_wo = udiv_multiplier(g.Wo);
    a.mg_ho = udiv_multiplier(g.Ho);
    int st = FORGE_OK;
    const int cu = device_info(&st).cu_count;
    if (st != FORGE_OK) return st;
    const RingRowMajor opb{w, ep.N, K};
    const int kH = K / (g.C * g.kW);
    const long long lead = (static_cast<long long>(g.padH) * g.W + g.padW) * g.C;
    if (g.C % kBK == 0 && kH <= 16 && g.kW <= 16 && img + 2 * lead < (1LL << 31)) {
        RingConvTap b;
        static_cast<ConvGeom&>(b) = g;
        b.lead = static_cast<uint32_t>(lead);
        b.range = static_cast<uint32_t>(img + 2 * lead);
        b.kH = kH;
        b.cps = g.C / kBK;
        b.mg_cps = udiv_multiplier(b.cps);
        b.mg_kw = a.mg_kw;
        b.mg_wo = a.mg_wo;
        b.mg_ho = a.mg_ho;
        // 256 x 256 from 8 stages on: with fewer, its epilogue, which nothing overlaps, is most of a tile
        // (INT32 outputs, us, 256 x 256 / the next pick: 256 -> 512 1x1 on 25 maps of 36 x 59 29 / 23).
        float cost = 0.0f;
        const int shape = ring_pick(ep.M, ep.N, K, cu, (1u << (K >= 8 * kBK ? kRingShapes : k256x256)) - 1, &cost);
        note_shape(shape);
        const RingRowMajorEven even{opb};
        if (shape == k256x256)
            return ep.c16 ? launch_ring_tile<T256x256, true, false>(b, even, ep, K, s)
                          : launch_ring_tile<T256x256, false, false>(b, even, ep, K, s);
        return ep.c16 ? launch_ring_shape<true>(shape, b, even, ep, K, s) : launch_ring_shape<false>(shape, b, even, ep, K, s);
    }
    // This gather's lane state does not fit beside the 256 x 256 tile's registers (172 bytes of
    // spills per lane), so these calls go without that shape.
    float cost = 0.0f;
    const int shape = ring_pick(ep.M, ep.N, K, cu, (1u << k256x256) - 1, &cost);
    note_shape(shape);
    return ep.c16 ? launch_ring_shape<true>(shape, a, opb, ep, K, s) : launch_ring_shape<false>(shape, a, opb, ep, K, s);
}

}  // namespace forge_amd
