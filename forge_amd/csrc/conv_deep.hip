// NCHW FP16 conv2d for deep layers (more weights than one CU's LDS), for gfx950.
//
// The reference's int8_conv2d_forward (src/nn/int8_conv2d.cu:126-223) gathers the im2col matrix,
// quantizes its rows, multiplies and transposes, per image. The one-launch kernels of conv.hip keep
// the whole patch depth of a tile and all weights in LDS; layers beyond that (128 -> 128 channels
// 3x3 is 147 KB of weights) ran the per-image pipeline, whose K-times inflated FP16 matrix alone
// is 75 MB per image at 135 x 240. Here two launches cover every image, with the same bits:
//   1. conv_deep_prep_kernel: per input position the maximum magnitude over its channels (FP16
//      bits; NaN skipped, as the reference quantizer's fmaxf does), and the weights permuted to
//      MFMA fragment order, both into the caller's workspace.
//   2. conv_deep_kernel: a tile of 32 output pixels per wave (Wt columns x R rows of one image) and
//      up to 128 output channels per workgroup. K runs in the order (32-channel chunk, tap,
//      channel): the INT32 sums are exact in any order. The chunk's input window sits channel-last
//      in LDS ([row][column][32 channels], double-buffered: the next chunk's 16-byte loads are in
//      registers while this one computes), so a lane's 16 taps of a K step are 32 contiguous
//      bytes; quantized with the pixel's own scale (16 v_fma_mix_f32 + 16 byte-insert adds) they
//      are the lane's fragment of v_mfma_i32_32x32x32_i8, fed to every 32-channel block. Weights
//      stream through two LDS slots of up to 9 taps by linear DMA. One barrier per slot.
// What bounds it: per K step and wave 36 VALU of quantization (144 cycles) beside NCB MFMAs of 32
// cycles, so a workgroup takes as many output channels per quantization as the registers hold;
// weights cost (tiles x weight bytes) through the DMA, so tiles are as tall as the waves and the LDS
// allow. 128 -> 128 3x3 on two 135 x 240 images: 267 -> 31.8 us (prep 6, window and scales and
// epilogue 10, K loop 15: half of what the two pipes' issue alone would take); 256 -> 256 on one
// 280 -> 49 us, 64 -> 64 5x5 at 90 x 160 89 -> 22 us.
#include "common.h"
#include "gemm_dense.h"
#include "mfma_tile.h"

#include <algorithm>
#include <climits>
#include <cstdio>

namespace forge_amd {

namespace {

constexpr int kDeepC = 32;        // channels per window chunk: one K step per tap
constexpr int kDeepTaps = 9;      // taps per weight slot
constexpr int kDeepPos = 80;      // LDS bytes per window position: 64 + 16 (conflict-free 16-byte reads)
// Workgroup sizes by window loads per lane and chunk: one leaves registers for three waves per
// SIMD, two or four (strided windows) for two.
constexpr int deep_max_waves(int items) { return items == 1 ? 12 : 8; }

struct ConvDeepArgs {
    const uint16_t* x;
    const int8_t* wf;             // weights in fragment order (workspace)
    const uint16_t* amax;         // (images, H, W) channel maxima (workspace)
    const uint16_t* w_scale;
    const uint16_t* bias;
    uint16_t* y;
    int C, H, W, Co, kH, kW, padH, padW, sH, sW, dH, dW, Ho, Wo;
    int nc, ntg, taps;            // 32-channel chunks; tap groups per chunk; taps
    int R, Wt, npix;              // tile rows / columns / pixels
    int nload;                    // window loads of a chunk (4 channels x 8 columns each)
    int G, IWr;                   // 8-column groups; row pitch (positions)
    int win_bytes, slot_bytes;    // one window buffer, one weight slot
    int tiles_h, tiles_w, tiles;  // tiles per image
    uint32_t mg_wt, mg_g, mg_tiles, mg_tw;
    uint32_t x_bytes, y_bytes;    // one image of x / of y
};

}  // namespace

// Fragment (block b of 32 output channels, chunk cc, tap): lane l's 16 bytes are output channel
// 32 b + l % 32, channels 32 cc + 16 (l / 32) .. + 15, zeros past C and C_out; fragments of one
// (group of NCB blocks, chunk) are contiguous, taps before blocks.
__global__ __launch_bounds__(256) void conv_deep_prep_kernel(const uint16_t* __restrict__ x, uint16_t* __restrict__ amax,
                                                             const int8_t* __restrict__ w, int8_t* __restrict__ wf, int C,
                                                             int HW, int groups, int images, int max_blocks, int Co,
                                                             int taps, int nc, int ncb, long long nfrag)
{
    const int t = threadIdx.x;
    if (static_cast<int>(blockIdx.x) < max_blocks) {
        // 32 groups of 8 positions x 8 channel slices
        __shared__ uint4 part[8][32];
        const int gi = static_cast<int>(blockIdx.x) * 32 + (t & 31), slice = t >> 5;
        const bool ok = gi < groups * images;
        // HW % 8 != 0: an image's last group is moved back to end with it (HW >= 8) and finds some maxima
        // once more, the same. (Gathered value by value it was a chain of C / 8 loads: the whole pass took
        // 44 us instead of 7.5 at 512 channels of 34 x 11, whose call then took 85 us, 46 now.)
        const int img = ok ? gi / groups : 0, p0 = ok ? min(8 * (gi - img * groups), HW - 8) : 0;
        const uint16_t* xi = x + static_cast<size_t>(img) * C * HW + p0;
        typedef uint32_t u4u __attribute__((ext_vector_type(4), aligned(2)));
        uint32_t m[4] = {0u, 0u, 0u, 0u};
        auto fold = [&](const uint32_t (&v)[4]) {
#pragma unroll
            for (int d = 0; d < 4; d++) {
                uint32_t b = v[d] & 0x7FFF7FFFu;
                // a NaN (above the infinity's bits) counts as 0
                if ((b & 0xFFFFu) > kHalfInfBits) b &= 0xFFFF0000u;
                if ((b >> 16) > kHalfInfBits) b &= 0x0000FFFFu;
                m[d] = pk_max_u16(m[d], b);
            }
        };
        if (ok) {
            constexpr int kB = 8;
            for (int c0 = slice; c0 < C; c0 += 8 * kB) {
                u4u v[kB];
#pragma unroll
                for (int q = 0; q < kB; q++)   // past the last channel: it again (a maximum does not change)
                    v[q] = *reinterpret_cast<const u4u*>(xi + static_cast<size_t>(min(c0 + 8 * q, C - 1)) * HW);
#pragma unroll
                for (int q = 0; q < kB; q++) {
                    const uint32_t u[4] = {v[q][0], v[q][1], v[q][2], v[q][3]};
                    fold(u);
                }
            }
        }
        part[slice][t & 31] = make_uint4(m[0], m[1], m[2], m[3]);
        __syncthreads();
        if (slice == 0 && ok) {
#pragma unroll
            for (int s = 1; s < 8; s++) {
                const uint4 o = part[s][t];
                m[0] = pk_max_u16(m[0], o.x);
                m[1] = pk_max_u16(m[1], o.y);
                m[2] = pk_max_u16(m[2], o.z);
                m[3] = pk_max_u16(m[3], o.w);
            }
            uint16_t* dst = amax + static_cast<size_t>(img) * HW + p0;
            *reinterpret_cast<u4u*>(dst) = u4u{m[0], m[1], m[2], m[3]};
        }
        return;
    }
    const long long f = (static_cast<long long>(blockIdx.x) - max_blocks) * 256 + t;
    if (f >= nfrag) return;
    const int lane = static_cast<int>(f & 63);
    long long r = f >> 6;                       // ((group * nc + cc) * taps + tap) * ncb + cb
    const int cb = static_cast<int>(r % ncb);
    r /= ncb;
    const int tap = static_cast<int>(r % taps);
    r /= taps;
    const int cc = static_cast<int>(r % nc), grp = static_cast<int>(r / nc);
    const int co = 32 * (grp * ncb + cb) + (lane & 31), c0 = 32 * cc + 16 * (lane >> 5);
    const int8_t* src = w + (static_cast<size_t>(co < Co ? co : 0) * C) * taps + tap;
    uint32_t o[4] = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int b = 0; b < 16; b++) {
        const int c = c0 + b;
        const uint32_t v = co < Co && c < C ? static_cast<uint8_t>(src[static_cast<size_t>(c) * taps]) : 0u;
        o[b >> 2] |= v << (8 * (b & 3));
    }
    *reinterpret_cast<uint4*>(wf + 16 * f) = make_uint4(o[0], o[1], o[2], o[3]);
}

// ALIGNED: W % 8 == 0 and a 16-byte aligned input, so an 8-column group lies wholly inside or
// outside the image. Otherwise loads are 16 bytes at 2-byte alignment, and the group holding the
// row's end loads the row's last 8 columns and shifts them into place (W >= 8).
template <int NCB, bool ALIGNED, int kItems, bool T9>
__global__ __launch_bounds__(64 * deep_max_waves(kItems)) void conv_deep_kernel(ConvDeepArgs a)
{
    extern __shared__ __align__(16) int8_t lds[];
    int8_t* win = lds;                             // two window buffers
    int8_t* wsl = lds + 2 * a.win_bytes;           // two weight slots
    const int t = threadIdx.x, lane = t & (kWave - 1);
    const int nthr = blockDim.x;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int l31 = lane & 31, hi = lane >> 5;
    const int HW = a.H * a.W;
    const int grp_co = blockIdx.y;

    const int tile = xcd_contiguous(blockIdx.x, gridDim.x);
    const int img = udiv_magic(tile, a.mg_tiles), rem = tile - img * a.tiles;
    const int th = udiv_magic(rem, a.mg_tw), tw = rem - th * a.tiles_w;
    const int ho0 = th * a.R, wo0 = tw * a.Wt;
    const int hb = ho0 * a.sH - a.padH, wb = wo0 * a.sW - a.padW;
    const int a0 = wb & ~7, s0 = wb - a0;          // window position 0 is the 8-aligned column a0

    // window loads: item i = ((row * G + group) * 8 + c4): channels 4 c4 .. + 3 of the chunk, columns
    // a0 + 8 group .. + 7 of window row `row`; items t (and t + nthr) of a chunk
    const __amdgpu_buffer_rsrc_t rx = buf_rsrc(a.x + static_cast<size_t>(img) * a.C * HW, a.x_bytes);
    uint32_t goff[kItems];
    int loff[kItems], c4x4 = 4 * (t & 7);
    bool edge[kItems];
#pragma unroll
    for (int q = 0; q < kItems; q++) {
        const int i = t + q * nthr;
        const int rg = i >> 3, row = udiv_magic(rg, a.mg_g), g = rg - row * a.G;
        const int h = hb + row, col = a0 + 8 * g;
        const bool ok = (i < a.nload) & (static_cast<unsigned>(h) < static_cast<unsigned>(a.H)) & (col >= 0) & (col < a.W);
        edge[q] = !ALIGNED && ok && col + 8 > a.W;
        goff[q] = ok ? 2u * static_cast<uint32_t>(c4x4 * HW + h * a.W + (edge[q] ? a.W - 8 : col)) : 0x80000000u;
        loff[q] = i < a.nload ? (row * a.IWr + 8 * g) * kDeepPos + 2 * c4x4 : -1;
    }
    const int es = 8 - (a.W & 7);                  // edge groups shift down by this many columns
    v4i pv[kItems][4];
    auto load_win = [&](int cc) {
#pragma unroll
        for (int q = 0; q < kItems; q++)
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const bool cok = 32 * cc + c4x4 + u < a.C && goff[q] != 0x80000000u;
                pv[q][u] = __builtin_amdgcn_raw_buffer_load_b128(
                    rx, cok ? goff[q] + 2u * static_cast<uint32_t>((32 * cc + u) * HW) : 0x80000000u, 0, 0);
            }
    };
    auto store_win = [&](int8_t* buf) {
#pragma unroll
        for (int q = 0; q < kItems; q++) {
            if (loff[q] < 0) continue;
            if (!ALIGNED && edge[q]) {
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    uint64_t lo = static_cast<uint32_t>(pv[q][u][0]) | static_cast<uint64_t>(static_cast<uint32_t>(pv[q][u][1])) << 32;
                    uint64_t h2 = static_cast<uint32_t>(pv[q][u][2]) | static_cast<uint64_t>(static_cast<uint32_t>(pv[q][u][3])) << 32;
                    const int sh = 16 * es;         // 16 .. 112
                    if (sh >= 64) {
                        lo = h2 >> (sh - 64);
                        h2 = 0;
                    } else {
                        lo = (lo >> sh) | (h2 << (64 - sh));
                        h2 >>= sh;
                    }
                    pv[q][u] = v4i{static_cast<int>(lo), static_cast<int>(lo >> 32), static_cast<int>(h2), static_cast<int>(h2 >> 32)};
                }
            }
            int8_t* dst = buf + loff[q];
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const int d = j >> 1;
                const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;
                uint2 o;
                o.x = __builtin_amdgcn_perm(static_cast<uint32_t>(pv[q][1][d]), static_cast<uint32_t>(pv[q][0][d]), sel);
                o.y = __builtin_amdgcn_perm(static_cast<uint32_t>(pv[q][3][d]), static_cast<uint32_t>(pv[q][2][d]), sel);
                *reinterpret_cast<uint2*>(dst + j * kDeepPos) = o;
            }
        }
    };
    // weights of phase ph = (cc, tap group): contiguous fragments, 1 KB DMA instructions over the waves
    const int nwave = nthr >> 6;
    const uint32_t wgroup = static_cast<uint32_t>(a.nc) * a.taps * NCB * 1024u;
    const __amdgpu_buffer_rsrc_t rw = buf_rsrc(a.wf + static_cast<size_t>(grp_co) * wgroup, wgroup);
    auto load_w = [&](int cc, int tg, int slot) {
        const int n = min(kDeepTaps, a.taps - tg * kDeepTaps) * NCB;
        const uint32_t src = static_cast<uint32_t>((cc * a.taps + tg * kDeepTaps) * NCB) * 1024u;
        int8_t* dst = wsl + slot * a.slot_bytes;
        for (int i = wave; i < n; i += nwave) dma16_buf(rw, 16u * lane, src + i * 1024u, dst + i * 1024);
    };

    load_w(0, 0, 0);
    load_win(0);
    float* s_ws = reinterpret_cast<float*>(wsl + 2 * a.slot_bytes);
    float* s_b = s_ws + 32 * NCB;
    const int cob = 32 * NCB * grp_co;
    if (t < 32 * NCB) {
        const int co = min(cob + t, a.Co - 1);
        s_ws[t] = h2f(a.w_scale[co]);
        s_b[t] = a.bias ? h2f(a.bias[co]) : -0.0f;   // fma(acc, s, -0) is acc * s rounded once
    }

    // the wave's 32 pixels and their scales: the maximum over the pixel's window positions (taps
    // outside the image are zeros)
    const int p0 = 32 * wave + l31, p = p0 < a.npix ? p0 : a.npix - 1;
    const int pr = udiv_magic(p, a.mg_wt), pc = p - pr * a.Wt;
    uint32_t mu = 0u;
    {
        const uint16_t* am = a.amax + static_cast<size_t>(img) * HW;
        const int h0 = hb + pr * a.sH, w0 = wb + pc * a.sW;
        int kh = 0, kw = 0;
        for (int tp = 0; tp < a.taps; tp += kDeepTaps) {   // nine loads in flight
            uint32_t v[kDeepTaps];
#pragma unroll
            for (int u = 0; u < kDeepTaps; u++) {
                const int h = h0 + kh * a.dH, w = w0 + kw * a.dW;
                const bool ok = (tp + u < a.taps) & (static_cast<unsigned>(h) < static_cast<unsigned>(a.H)) &
                                (static_cast<unsigned>(w) < static_cast<unsigned>(a.W));
                const uint32_t m = am[ok ? h * a.W + w : 0];
                v[u] = ok ? m : 0u;
                if (++kw == a.kW) {
                    kw = 0;
                    kh++;
                }
            }
#pragma unroll
            for (int u = 0; u < kDeepTaps; u++) mu = max(mu, v[u]);
        }
    }
    const float scale = row_scale(h2f(static_cast<uint16_t>(mu)));
    const float inv = 1.0f / scale;
    const int pix = (pr * a.sH * a.IWr + s0 + pc * a.sW) * kDeepPos + 32 * hi;

    v16i acc[NCB];
#pragma unroll
    for (int cb = 0; cb < NCB; cb++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[cb][e] = 0;

    store_win(win);
    wait_vm_lgkm0();
    lds_barrier();

    int slot = 0;
    for (int cc = 0; cc < a.nc; cc++) {
        const int8_t* wbuf = win + (cc & 1) * a.win_bytes + pix;
        const bool more = cc + 1 < a.nc;
        int kh = 0, kw = 0;
        for (int tg = 0; tg < a.ntg; tg++) {
            const bool last = tg + 1 == a.ntg;
            if (!last) load_w(cc, tg + 1, slot ^ 1);
            else if (more) load_w(cc + 1, 0, slot ^ 1);
            if (tg == 0 && more) load_win(cc + 1);
            const int ntap = min(kDeepTaps, a.taps - tg * kDeepTaps);
            const int8_t* ws = wsl + slot * a.slot_bytes + lane * 16;
            // a tap: its fragment quantized from 32 bytes of the window, fed to every block
            // (LDS reads as vector types: through a struct such as uint4 the compiler takes them to
            // alias the DMA's LDS writes, and waits for every load in flight before each)
            struct Tap {
                v4i h0, h1;
            };
            auto window = [&]() {              // the current tap's values; steps to the next tap
                const int8_t* src = wbuf + (kh * a.dH * a.IWr + kw * a.dW) * kDeepPos;
                if (++kw == a.kW) {
                    kw = 0;
                    kh++;
                }
                return Tap{*reinterpret_cast<const v4i*>(src), *reinterpret_cast<const v4i*>(src + 16)};
            };
            auto multiply = [&](const Tap& v, int i) {
                v4i wc[NCB];
#pragma unroll
                for (int cb = 0; cb < NCB; cb++) wc[cb] = *reinterpret_cast<const v4i*>(ws + (i * NCB + cb) * 1024);
                const int hw[8] = {v.h0[0], v.h0[1], v.h0[2], v.h0[3], v.h1[0], v.h1[1], v.h1[2], v.h1[3]};
                float pq[16];
#pragma unroll
                for (int d = 0; d < 8; d++) {
                    pq[2 * d] = fma_mix_lo(static_cast<uint32_t>(hw[d]), inv);
                    pq[2 * d + 1] = fma_mix_hi(static_cast<uint32_t>(hw[d]), inv);
                }
                const v4i fb = __builtin_bit_cast(v4i, pack16_rint_sdwa(pq));
#pragma unroll
                for (int cb = 0; cb < NCB; cb++) acc[cb] = __builtin_amdgcn_mfma_i32_32x32x32_i8(wc[cb], fb, acc[cb], 0, 0, 0);
            };
            if constexpr (T9) {
                // unrolled: the next tap's reads are in flight while one is quantized
                Tap cur = window();
#pragma unroll
                for (int i = 0; i < kDeepTaps; i++) {
                    Tap nxt;
                    if (i + 1 < kDeepTaps) nxt = window();
                    multiply(cur, i);
                    cur = nxt;
                }
            } else {
                for (int i = 0; i < ntap; i++) multiply(window(), i);
            }
            if (last && more) store_win(win + ((cc + 1) & 1) * a.win_bytes);
            if (!last || more) {
                wait_vm_lgkm0();                   // the next phase's weights, and this wave's window writes
                lds_barrier();
            }
            slot ^= 1;
        }
    }

    // the GEMM's epilogue, straight to NCHW: 32 adjacent pixels per store
    const uint32_t plane2 = 2u * static_cast<uint32_t>(a.Ho * a.Wo);
    const __amdgpu_buffer_rsrc_t ry = buf_rsrc(a.y + static_cast<size_t>(img) * a.Co * (plane2 >> 1), a.y_bytes);
    const int ho = ho0 + pr, wo = wo0 + pc;
    const bool pok = p0 < a.npix && ho < a.Ho && wo < a.Wo;
    const uint32_t vo = 2u * static_cast<uint32_t>(ho * a.Wo + wo);
#pragma unroll
    for (int cb = 0; cb < NCB; cb++) {
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const float4 ws4 = *reinterpret_cast<const float4*>(s_ws + 32 * cb + 8 * g + 4 * hi);
            const float4 b4 = *reinterpret_cast<const float4*>(s_b + 32 * cb + 8 * g + 4 * hi);
            const float wsv[4] = {ws4.x, ws4.y, ws4.z, ws4.w}, bv[4] = {b4.x, b4.y, b4.z, b4.w};
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int co = cob + 32 * cb + 8 * g + 4 * hi + e;
                const uint16_t yv = f2h(__builtin_fmaf(static_cast<float>(acc[cb][4 * g + e]), scale * wsv[e], bv[e]));
                __builtin_amdgcn_raw_buffer_store_b16(yv, ry, pok && co < a.Co ? vo + static_cast<uint32_t>(co) * plane2 : 0x80000000u,
                                                      0, 0);
            }
        }
    }
}

template <int NCB, bool ALIGNED, int kItems>
static int launch_deep_kernel(const ConvDeepArgs& a, int images, int groups_co, int waves, int lds, hipStream_t s)
{
    auto kern = a.taps == kDeepTaps ? conv_deep_kernel<NCB, ALIGNED, kItems, true> : conv_deep_kernel<NCB, ALIGNED, kItems, false>;
    static const hipError_t attr[2] = {
        hipFuncSetAttribute(reinterpret_cast<const void*>(&conv_deep_kernel<NCB, ALIGNED, kItems, true>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024),
        hipFuncSetAttribute(reinterpret_cast<const void*>(&conv_deep_kernel<NCB, ALIGNED, kItems, false>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024)};
    if (attr[0] != hipSuccess) return static_cast<int>(attr[0]);
    if (attr[1] != hipSuccess) return static_cast<int>(attr[1]);
    kern<<<dim3(static_cast<unsigned>(a.tiles * images), static_cast<unsigned>(groups_co)), 64 * waves, lds, s>>>(a);
    return launch_status();
}

template <int NCB>
static int launch_deep(const ConvDeepArgs& a, bool al, int items, int images, int groups_co, int waves, int lds, hipStream_t s)
{
    if (items == 1)
        return al ? launch_deep_kernel<NCB, true, 1>(a, images, groups_co, waves, lds, s)
                  : launch_deep_kernel<NCB, false, 1>(a, images, groups_co, waves, lds, s);
    if (items == 2)
        return al ? launch_deep_kernel<NCB, true, 2>(a, images, groups_co, waves, lds, s)
                  : launch_deep_kernel<NCB, false, 2>(a, images, groups_co, waves, lds, s);
    return al ? launch_deep_kernel<NCB, true, 4>(a, images, groups_co, waves, lds, s)
              : launch_deep_kernel<NCB, false, 4>(a, images, groups_co, waves, lds, s);
}

// -1 when the shape is not one it takes (the caller's other paths run).
int launch_conv_deep(const ConvDeepShape& c, void* workspace, size_t ws_bytes, hipStream_t s)
{
    const int taps = c.kH * c.kW;
    if (taps < 2 || taps > 81 || c.W < 8) return -1;
    const long long xb = 2LL * c.C * c.H * c.W, yb = 2LL * c.Co * c.Ho * c.Wo;
    if (xb >= (1LL << 30) || yb >= (1LL << 31) || static_cast<long long>(c.Co + 128) * (c.C + 32) * taps >= (1LL << 31) || static_cast<long long>(c.H) * c.W >= (1 << 28)) return -1;
    int st = FORGE_OK;
    const int cu = device_info(&st).cu_count;
    if (st != FORGE_OK) return st;

    ConvDeepArgs a{};
    a.x = c.x;
    a.w_scale = c.w_scale;
    a.bias = c.bias;
    a.y = c.y;
    a.C = c.C; a.H = c.H; a.W = c.W; a.Co = c.Co; a.kH = c.kH; a.kW = c.kW;
    a.padH = c.padH; a.padW = c.padW; a.sH = c.sH; a.sW = c.sW; a.dH = c.dH; a.dW = c.dW;
    a.Ho = c.Ho; a.Wo = c.Wo;
    a.taps = taps;
    a.nc = divup(c.C, kDeepC);
    a.ntg = divup(taps, kDeepTaps);
    a.x_bytes = static_cast<uint32_t>(xb);
    a.y_bytes = static_cast<uint32_t>(yb);
    const int blocks = divup(c.Co, 32);
    int groups_co = 0, ncb = 0;

    // The tile: the waves, columns and rows with the least modelled time (us). A CU's tiles run in
    // rounds; a round costs ~10 us for the window, scales and epilogue, and per K step 0.1 us plus
    // 0.14 us for each wave of a SIMD (72 steps at one wave per SIMD 18 us, 36 at 2.25 waves 15 us).
    double best = -1.0;
    int waves = 0, lds = 0;
    const int ksteps = a.nc * taps;
    // output channels: up to 128 per workgroup, fewer where the windows leave no room for their weights
    for (int grp = divup(blocks, 4); grp <= blocks && best < 0; grp++) {
        groups_co = grp;
        ncb = divup(blocks, grp);
        a.slot_bytes = std::min(taps, kDeepTaps) * ncb * 1024;
        for (int nw = 4; nw <= deep_max_waves(1); nw++) {
            const int k0 = divup(c.Wo, 32 * nw);
            for (int k = k0; k < k0 + 8; k++) {        // k tiles across the image
                const int wt = divup(c.Wo, k), R = std::min(32 * nw / wt, c.Ho);
                if (wt < 8 && k > k0) break;
                if (R < 1 || wt * R <= 32 * (nw - 1)) continue;
                const long long IH = static_cast<long long>(R - 1) * c.sH + static_cast<long long>(c.kH - 1) * c.dH + 1;
                const long long IW = static_cast<long long>(wt - 1) * c.sW + static_cast<long long>(c.kW - 1) * c.dW + 1;
                const long long G = (IW + 7 + 7) / 8, nload = IH * G * 8;
                if (nload > 64LL * nw * (nw <= deep_max_waves(4) ? 4 : 1)) continue;
                const long long win = IH * (8 * G + 1) * kDeepPos, bytes = 2 * win + 2LL * a.slot_bytes + 256LL * ncb;
                if (bytes > 160 * 1024) continue;
                const int per_cu = std::max(1, std::min(static_cast<int>(160 * 1024 / bytes), 12 / nw));
                const long long tiles = static_cast<long long>(divup(c.Ho, R)) * divup(c.Wo, wt) * c.N * groups_co;
                const long long rounds = divupll(tiles, static_cast<long long>(cu) * per_cu);
                const double cost = static_cast<double>(rounds) * (10.0 + ksteps * (0.1 + 0.035 * nw * per_cu));
                if (best < 0 || cost < best) {
                    best = cost;
                    waves = nw;
                    lds = static_cast<int>(bytes);
                    a.Wt = wt;
                    a.R = R;
                    a.G = static_cast<int>(G);
                    a.nload = static_cast<int>(nload);
                    a.win_bytes = static_cast<int>(win);
                }
            }
        }
    }
    if (best < 0) return -1;
    // Few pixels of much depth: the per-image pipeline spreads its GEMM over K and columns (16 us per
    // image plus its passes over the patch matrix; 256 -> 256 at 16 x 16: 21 us, here 28).
    const double pipeline = c.N * (16.0 + 2.9e-6 * static_cast<double>(c.Ho) * c.Wo * c.C * taps);
    if (pipeline < best) return -1;
    a.npix = a.R * a.Wt;
    a.IWr = 8 * a.G + 1;
    a.tiles_h = divup(c.Ho, a.R);
    a.tiles_w = divup(c.Wo, a.Wt);
    const long long tiles = static_cast<long long>(a.tiles_h) * a.tiles_w;

    // workspace: fragments (16-byte vectors and LDS DMA, so from its first 16-byte boundary on: the caller's
    // buffer may start anywhere), then the channel maxima of as many images as fit
    const size_t skip = -reinterpret_cast<uintptr_t>(workspace) & 15;
    if (ws_bytes < skip) return -1;
    ws_bytes -= skip;
    const long long nfrag = static_cast<long long>(groups_co) * ncb * a.nc * taps * 64;
    const long long wbytes = 16 * nfrag;
    const long long HW = static_cast<long long>(c.H) * c.W;
    if (wbytes + 2 * HW > static_cast<long long>(ws_bytes)) return -1;
    long long chunk = (static_cast<long long>(ws_bytes) - wbytes) / (2 * HW);
    chunk = std::min<long long>(chunk, c.N);
    chunk = std::min<long long>(chunk, INT_MAX / (HW / 8 + 1));
    while (chunk > 1 && (tiles * chunk > 0x7FFFFFFFLL || tiles * chunk * tiles >= (1LL << 32))) chunk--;
    if (tiles * chunk * tiles >= (1LL << 32) || tiles * a.tiles_w >= (1LL << 32)) return -1;
    a.tiles = static_cast<int>(tiles);
    a.mg_wt = udiv_multiplier(a.Wt);
    a.mg_g = udiv_multiplier(a.G);
    a.mg_tiles = udiv_multiplier(a.tiles);
    a.mg_tw = udiv_multiplier(a.tiles_w);
    int8_t* wf = static_cast<int8_t*>(workspace) + skip;
    uint16_t* amax = reinterpret_cast<uint16_t*>(wf + wbytes);
    a.wf = wf;
    a.amax = amax;
    const bool al = c.W % 8 == 0 && aligned(c.x, 16);
    const int items = a.nload <= 64 * waves ? 1 : a.nload <= 128 * waves ? 2 : 4;
    char name[32];
    snprintf(name, sizeof name, "conv-nchw-deep b%d i%d%s", ncb, items, al ? " a" : "");
    note_route(name, 32 * waves);
    for (int n0 = 0; n0 < c.N; n0 += static_cast<int>(chunk)) {
        const int cnt = static_cast<int>(std::min<long long>(chunk, c.N - n0));
        a.x = c.x + static_cast<size_t>(n0) * c.C * HW;
        a.y = c.y + static_cast<size_t>(n0) * c.Co * c.Ho * c.Wo;
        const int groups = divup(static_cast<int>(HW), 8);
        const int mblocks = divup(groups * cnt, 32);
        const long long fblocks = n0 == 0 ? divupll(nfrag, 256) : 0;
        conv_deep_prep_kernel<<<static_cast<unsigned>(mblocks + fblocks), 256, 0, s>>>(
            a.x, amax, c.w, wf, c.C, static_cast<int>(HW), groups, cnt, mblocks, c.Co, taps, a.nc, ncb, nfrag);
        if ((st = launch_status()) != FORGE_OK) return st;
        switch (ncb) {
            case 1: st = launch_deep<1>(a, al, items, cnt, groups_co, waves, lds, s); break;
            case 2: st = launch_deep<2>(a, al, items, cnt, groups_co, waves, lds, s); break;
            case 3: st = launch_deep<3>(a, al, items, cnt, groups_co, waves, lds, s); break;
            default: st = launch_deep<4>(a, al, items, cnt, groups_co, waves, lds, s); break;
        }
        if (st != FORGE_OK) return st;
    }
    return FORGE_OK;
}

}  // namespace forge_amd
