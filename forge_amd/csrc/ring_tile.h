// Ring-fed INT8 MFMA tile for gfx950 (v_mfma_i32_16x16x64_i8): the engine of the dense GEMMs and
// the NHWC conv gathers.
//
// A workgroup of WM x WN waves computes a BM x BN INT32 tile of C = A (rows, K) x B (cols, K)^T,
// each wave a (BM / WM) x (BN / WN) sub-tile of 16 x 16 blocks. K streams in 128-byte stages
// through a ring of D LDS slots filled by LDS-DMA buffer loads (mfma_tile.h dma16_buf: a stage row
// is one 128-byte line in 8 swizzled chunks), D - 1 stages in flight.
//
// What bounds it: a CU takes ~62 GB/s through the LDS DMA whatever the tile, so a tile costs its
// (BM + BN) x K bytes and a call the bytes of its busiest CU (1024 x 6144 x 1536 on 64 x 128 tiles:
// 1.18 MB, 17.9 us); at 256 x 256 the MFMAs take as long as the DMA. Hence many tile shapes
// (16-row blocks allow any multiple of 16 per wave), of which the host picks the one whose tiles
// spread most evenly over the CUs (gemm_ring.hip), and 8 waves per workgroup: two per SIMD cover
// each other's barrier and LDS latency, which one does not (128 x 192 at 4096 x 6144 x 1536: 4
// waves 48 us, 8 waves 37 us). Against the engine before (256 x 256 and 128 x 128 tiles on 4 waves
// with 2 slots, register-staged 64 x 64 below): 4096^3 60 -> 55 us (2500 TOPS), 2048 x 4096 x 4096
// 46.4 -> 32.5, 1024 x 6144 x 1536 26.6 -> 17.9, 1500 x 2880 x 2880 28 -> 19.1, 8192 x 1024 x 1024
// 20.5 -> 12.5, 700 x 1040 x 1000 8.2 -> 5.8. 32 x 32 blocks (half the operand registers read
// per multiply) measured slower in all but the smallest (4096^3 59.4 against 55.7 us);
// s_setprio around the MFMAs, an L2 prefetch of later stages, and the DMAs interleaved with
// the MFMAs by scheduling groups measured level or slower.
//
// The K loop's one barrier per stage sits between the two 64-deep sub-steps of stage kt: it
// publishes stage kt + 1 (each wave has waited for its own DMAs of it) and frees stage kt's slot
// (each wave has read its fragments of it), which stage kt + D is then loaded into.
//
// K % 16 == 0, any row count: a chunk of 16 K-bytes past K reads as zeros (its offset is moved past
// the buffer's range); rows past the end are clamped (never stored); stages past the end read
// from an empty resource (zeros, no memory traffic), so the issue has no branch and the wait
// counts stay exact.
#pragma once

#include "mfma_tile.h"

#include <type_traits>

namespace forge_amd {

typedef v4i v4i_h __attribute__((aligned(2)));   // 16 bytes at an FP16 / INT32 element's alignment
typedef v4i v4i_w __attribute__((aligned(4)));

constexpr uint32_t kOutOfRange = 0x80000000u;   // past any operand (they are under 2^31 bytes)

// Ring operands: lane(r, c) once per DMA instruction and tile; at(st) the uniform position of the tile's
// first stage and step(pos, st) that of the next one, st, cyclic; dma() once per DMA instruction and
// stage. `live` is false for stages past the end.

// Row-major (rows, K) matrix. Chunks past K read as zeros: their offset is moved out of range in
// the per-lane offset, which the range check certainly covers (a scalar offset it may not).
struct RingRowMajor {
    const int8_t* p;
    int rows, K;
    struct Lane {
        uint32_t off;
        int k16;
    };
    struct Pos {
        int st;
    };
    __device__ __forceinline__ Lane lane(int r, int c) const {
        return Lane{static_cast<uint32_t>(r < rows ? r : rows - 1) * static_cast<uint32_t>(K) + 16u * c, 16 * c};
    }
    __device__ __forceinline__ Pos at(int st) const { return Pos{st}; }
    __device__ __forceinline__ void step(Pos& p, int st) const { p.st = st; }
    __device__ __forceinline__ void dma(const Lane& l, const Pos& pos, bool live, int8_t* dst) const {
        const uint32_t soff = static_cast<uint32_t>(pos.st) * kBK;
        const uint32_t bytes = static_cast<uint32_t>(rows) * static_cast<uint32_t>(K);
        const uint32_t voff = l.k16 < K - static_cast<int>(soff) ? l.off : kOutOfRange;
        dma16_buf(buf_rsrc(p, live ? bytes : 0u), voff, live ? soff : 0u, dst);
    }
};

// The same with K % 128 == 0: no chunk past K.
struct RingRowMajorEven : RingRowMajor {
    using Lane = uint32_t;
    __device__ __forceinline__ Lane lane(int r, int c) const { return RingRowMajor::lane(r, c).off; }
    __device__ __forceinline__ void dma(Lane l, const Pos& pos, bool live, int8_t* dst) const {
        const uint32_t bytes = static_cast<uint32_t>(rows) * static_cast<uint32_t>(K);
        dma16_buf(buf_rsrc(p, live ? bytes : 0u), l, live ? static_cast<uint32_t>(pos.st) * kBK : 0u, dst);
    }
};

// Implicit im2col of an NHWC image with C % 16 == 0 (K order (kh, kw, c)): a 16-byte chunk is 16
// channels of one tap, so each lane finds its chunk's tap by two magic divisions per stage; a tap
// in the padding gets an offset past the image, which reads as zeros. Needs an image under 2^31
// bytes, (K + 8 stages) C < 2^32, ((K + 8 stages) / C + 1) kW < 2^32 and rows max(Ho, Wo) < 2^32.
struct RingConv : ConvGeom {
    uint32_t x_bytes;
    uint32_t mg_c, mg_kw, mg_wo, mg_ho;   // udiv_magic multipliers of C, kW, Wo, Ho
    struct Lane {
        int img, hb, wb, k16;             // n H, the pixel's first input row and column, 16 * chunk
    };
    __device__ __forceinline__ Lane lane(int r, int c) const {
        r = r < rows ? r : rows - 1;
        const int t = udiv_magic(r, mg_wo), wo = r - t * Wo;
        const int n = udiv_magic(t, mg_ho), ho = t - n * Ho;
        return Lane{n * H, ho * strideH - padH, wo * strideW - padW, 16 * c};
    }
    using Pos = RingRowMajor::Pos;
    __device__ __forceinline__ Pos at(int st) const { return Pos{st}; }
    __device__ __forceinline__ void step(Pos& p, int st) const { p.st = st; }
    __device__ __forceinline__ void dma(const Lane& l, const Pos& pos, bool live, int8_t* dst) const {
        const int k = pos.st * kBK + l.k16;
        const int tap = udiv_magic(k, mg_c), kh = udiv_magic(tap, mg_kw);
        const int hi = l.hb + kh * dilH, wi = l.wb + (tap - kh * kW) * dilW;
        const bool ok = (k < K) & (static_cast<unsigned>(hi) < static_cast<unsigned>(H)) &
                        (static_cast<unsigned>(wi) < static_cast<unsigned>(W));
        const uint32_t off = static_cast<uint32_t>(((l.img + hi) * W + wi - tap) * C + k);
        dma16_buf(buf_rsrc(x, live ? x_bytes : 0u), ok ? off : kOutOfRange, 0, dst);
    }
};

// The same gather with C % 128 == 0 and kH, kW <= 16: a stage is 128 channels of one tap, which is
// uniform, so a lane keeps its pixel's offset and which kernel rows and columns fall inside the image,
// and a stage costs it a bit test; the position is advanced, not divided. With RingConv's two divisions
// per DMA instruction, us, RingConv / here: 256 -> 256 3x3 on 33 maps of 36 x 92 102 / 72, 2048 -> 2048 3x3
// at 92 x 70 274 / 216, over 300 shapes 10 % less; and its lane state, twice this one's, does not fit beside
// the 256 x 256 tile's accumulators. Offsets are taken from `lead` bytes before the image, where the
// first tap of the first pixel lies, so that none is negative; the resource ends 2 lead past the image,
// so that it is longer than any scalar offset (a tap outside the image is out of the lane offset's range).
struct RingConvTap : ConvGeom {
    uint32_t lead, range;                 // (padH W + padW) C; the image + 2 lead
    int kH, cps;                          // stages per tap (C / 128)
    uint32_t mg_cps, mg_kw, mg_wo, mg_ho;
    struct Lane {
        uint32_t off;                     // of pixel (n, hb, wb) + 16 * chunk
        uint32_t in;                      // bit kh: kernel row inside, bit 16 + kw: column inside
    };
    struct Pos {
        int kh, kw, ch, row;              // row: (kh dilH W + kw dilW) C
    };
    __device__ __forceinline__ Lane lane(int r, int c) const {
        r = r < rows ? r : rows - 1;
        const int t = udiv_magic(r, mg_wo), wo = r - t * Wo;
        const int n = udiv_magic(t, mg_ho), ho = t - n * Ho;
        const int hb = ho * strideH - padH, wb = wo * strideW - padW;
        uint32_t in = 0u;
        for (int kh = 0; kh < kH; kh++)
            if (static_cast<unsigned>(hb + kh * dilH) < static_cast<unsigned>(H)) in |= 1u << kh;
        for (int kw = 0; kw < kW; kw++)
            if (static_cast<unsigned>(wb + kw * dilW) < static_cast<unsigned>(W)) in |= 0x10000u << kw;
        return Lane{static_cast<uint32_t>(((n * H + hb) * W + wb) * C + 16 * c) + lead, in};
    }
    __device__ __forceinline__ Pos at(int st) const {
        const int tap = udiv_magic(st, mg_cps), kh = udiv_magic(tap, mg_kw), kw = tap - kh * kW;
        return Pos{kh, kw, st - tap * cps, (kh * dilH * W + kw * dilW) * C};
    }
    __device__ __forceinline__ void step(Pos& p, int) const {
        // selects: a branch here would cut the K loop's schedule in two
        const bool tap = p.ch + 1 == cps, row = tap && p.kw + 1 == kW;
        p.ch = tap ? 0 : p.ch + 1;
        p.kw = row ? 0 : p.kw + (tap ? 1 : 0);
        p.kh = row ? (p.kh + 1 == kH ? 0 : p.kh + 1) : p.kh;
        p.row = (p.kh * dilH * W + p.kw * dilW) * C;
    }
    __device__ __forceinline__ void dma(const Lane& l, const Pos& pos, bool live, int8_t* dst) const {
        const bool ok = (l.in >> pos.kh) & (l.in >> (16 + pos.kw)) & 1u;
        dma16_buf(buf_rsrc(x - lead, live ? range : 0u), ok ? l.off : kOutOfRange,
                  live ? static_cast<uint32_t>(pos.row + pos.ch * kBK) : 0u, dst);
    }
};

template <int BM, int BN, int WM, int WN, int D>
struct RingTile {
    static constexpr int MB = 16;                                      // rows of an MFMA block
    static constexpr int kNW = WM * WN;
    static constexpr int kThreads = kNW * kWave;
    static constexpr int kBM = BM, kBN = BN, kWM = WM, kWN = WN, kDepth = D;
    static constexpr int kTM = BM / WM / MB, kTN = BN / WN / MB;
    static constexpr int kAIns = BM / 8 / kNW, kBIns = BN / 8 / kNW;   // 1 KB DMA instructions per wave and stage
    static constexpr int kIns = kAIns + kBIns;
    static constexpr int kSub = kBK / 64;                              // MFMA sub-steps per stage
    static constexpr int kSlotBytes = (BM + BN) * kBK;
    static_assert(BM % (8 * kNW) == 0 && BN % (8 * kNW) == 0, "a stage splits evenly over the waves");
    static_assert(BM % (MB * WM) == 0 && BN % (MB * WN) == 0, "wave tiles of whole blocks");
    static_assert(D >= 2 && kIns * (D - 2) < 64, "vmcnt immediate");

    v4i acc[kTN][kTM];

    template <class OpA, class OpB>
    __device__ __forceinline__ void run(const OpA& opa, const OpB& opb, int K, int m0, int n0, int rot, int8_t* lds) {
        const int lane = threadIdx.x & (kWave - 1);
        const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
        const int wm = (wave / WN) * (BM / WM), wn = (wave % WN) * (BN / WN);
        const int lr = lane % MB, g = lane / MB;

#pragma unroll
        for (int j = 0; j < kTN; j++)
#pragma unroll
            for (int i = 0; i < kTM; i++) acc[j][i] = v4i{0, 0, 0, 0};

        // DMA instruction i (8 rows) of an operand: lane -> row 8 i + lane / 8, physical chunk
        // lane % 8 = logical chunk (lane % 8) ^ swz(row), swz(row) = (row ^ row / 8) % 8.
        typename OpA::Lane la[kAIns];
        typename OpB::Lane lb[kBIns];
#pragma unroll
        for (int q = 0; q < kAIns; q++) {
            const int r = 8 * (wave * kAIns + q) + (lane >> 3);
            la[q] = opa.lane(m0 + r, (lane & 7) ^ lds_swz8(r));
        }
#pragma unroll
        for (int q = 0; q < kBIns; q++) {
            const int r = 8 * (wave * kBIns + q) + (lane >> 3);
            lb[q] = opb.lane(n0 + r, (lane & 7) ^ lds_swz8(r));
        }
        const int nst = (K + kBK - 1) / kBK;
        typename OpA::Pos pa = opa.at(rot);          // the stages in order from rot on
        typename OpB::Pos pb = opb.at(rot);
        auto dmas = [&](bool live, int slot) {
            int8_t* s = lds + slot * kSlotBytes;
#pragma unroll
            for (int q = 0; q < kAIns; q++) opa.dma(la[q], pa, live, s + (wave * kAIns + q) * 1024);
#pragma unroll
            for (int q = 0; q < kBIns; q++) opb.dma(lb[q], pb, live, s + BM * kBK + (wave * kBIns + q) * 1024);
        };
        auto issue = [&](int st, int slot) {         // stages 1 on
            const int at = st + rot;
            opa.step(pa, at < nst ? at : at - nst);
            opb.step(pb, at < nst ? at : at - nst);
            dmas(st < nst, slot);
        };
        struct Frags {
            v4i a[kTM], b[kTN];
        };
        auto load_frags = [&](int slot, int ks, Frags& F) {
            const int8_t* As = lds + slot * kSlotBytes;
            const int8_t* Bs = As + BM * kBK;
            const int c = (kWave / MB) * ks + g;
#pragma unroll
            for (int i = 0; i < kTM; i++) F.a[i] = *reinterpret_cast<const v4i*>(As + lds_off128(wm + MB * i + lr, c));
#pragma unroll
            for (int j = 0; j < kTN; j++) F.b[j] = *reinterpret_cast<const v4i*>(Bs + lds_off128(wn + MB * j + lr, c));
        };
        auto mfmas = [&](const Frags& F) {
#pragma unroll
            for (int j = 0; j < kTN; j++)
#pragma unroll
                for (int i = 0; i < kTM; i++)
                    acc[j][i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(F.b[j], F.a[i], acc[j][i], 0, 0, 0);
        };
        constexpr int kMf = kTM * kTN, kRd = kTM + kTN;

        dmas(true, 0);
#pragma unroll
        for (int st = 1; st < D; st++) issue(st, st);
        wait_vmcnt<kIns*(D - 1) < 64 ? kIns * (D - 1) : 63>();
        lds_barrier();
        Frags F[2];
        load_frags(0, 0, F[0]);
        int slot = 0;
        for (int kt = 0; kt + 1 < nst; kt++) {
#pragma unroll
            for (int ks = 0; ks + 1 < kSub; ks++) {
                load_frags(slot, ks + 1, F[(ks + 1) & 1]);
                mfmas(F[ks & 1]);
                sched_interleave<kMf, kRd, 0>();
            }
            // stage kt + 1 landed (own DMAs) and this wave's reads of stage kt are complete
            wait_vm_lgkm<kIns*(D - 2)>();
            lds_barrier();
            const int freed = slot;
            slot = slot + 1 == D ? 0 : slot + 1;
            load_frags(slot, 0, F[0]);
            issue(kt + D, freed);                    // into stage kt's slot
            mfmas(F[1]);
        }
#pragma unroll
        for (int ks = 0; ks + 1 < kSub; ks++) {
            load_frags(slot, ks + 1, F[(ks + 1) & 1]);
            mfmas(F[ks & 1]);
        }
        mfmas(F[1]);
        // every wave is done with the ring, and no DMA is in flight, before the epilogue
        wait_vm_lgkm0();
        lds_barrier();
    }
};

// LDS bytes of a ring tile's epilogue: per wave its staging rows (FP16 the whole sub-tile, INT32
// one block of rows at a time; padded by 16 bytes: the 16 rows of a write phase fall on distinct
// banks) and the
// w_scale / bias strips of its columns.
template <class T, bool DEQUANT>
constexpr int ring_epilogue_wave_bytes() {
    return DEQUANT ? T::MB * T::kTM * (2 * T::MB * T::kTN + 16) + 2 * T::MB * T::kTN * 2 : T::MB * (4 * T::MB * T::kTN + 16);
}
template <class T, bool DEQUANT>
constexpr int ring_lds_bytes() {
    const int ring = T::kDepth * T::kSlotBytes, epi = T::kNW * ring_epilogue_wave_bytes<T, DEQUANT>();
    return ring > epi ? ring : epi;
}

// The upsample scatter of kRows staged pixels x kCols columns (rows of `pitch` bytes, column c at
// 2 c). Column pair (co, kh), kw = 0 and 1, is one 4-byte word and two adjacent outputs of row
// 2 h + kh; pbias: post_bias per column. vec_out (W % 4 == 0): groups of 4 pixels of one image row
// go out as one 16-byte store. A lane keeps one group, whose place in the image it finds once (with the
// two divisions at every word, 16 channels at 56 x 221 -> 111 took 20.4 us, 12.4 so), and walks the pairs;
// the LDS words of a batch are all read before its first store.
template <int kRows, int kCols>
__device__ __forceinline__ void ring_flush_up2x2(const int8_t* stage, int pitch, const uint16_t* pbias,
                                                 const GemmEpilogue& ep, int row0, int col0) {
    constexpr int kPairs = kCols / 2;
    const int lane = threadIdx.x & (kWave - 1);
    const int M = ep.M, N = ep.N, W = ep.up_w, HW = ep.up_hw;
    const size_t plane = 4 * static_cast<size_t>(HW), W2 = 2 * static_cast<size_t>(W);
    const bool has_bias = ep.post_bias != nullptr;
    auto walk = [&](auto pixels) {
        constexpr int kT = decltype(pixels)::value, kGroups = kRows / kT, kStep = kWave / kGroups;
        constexpr int kIters = kPairs / kStep, kB = kIters < 4 ? kIters : 4;
        static_assert(kWave % kGroups == 0 && kPairs % kStep == 0 && kIters % kB == 0, "groups and pairs split evenly");
        const int g = lane % kGroups, m = row0 + kT * g;
        if (m >= M) return;                              // kT = 4: M % 4 == 0, a group is all in or all out
        const int img = m / HW, p = m - img * HW, h = p / W, w = p - h * W;
        uint16_t* base = ep.c16 + static_cast<size_t>(img) * (N >> 2) * plane + 2 * h * W2 + 2 * w;
#pragma unroll 1
        for (int k0 = 0; k0 < kIters; k0 += kB) {
            uint32_t d[kB][kT];
#pragma unroll
            for (int b = 0; b < kB; b++) {
                const int cw = 2 * (lane / kGroups + (k0 + b) * kStep);
#pragma unroll
                for (int t = 0; t < kT; t++) d[b][t] = *reinterpret_cast<const uint32_t*>(stage + (kT * g + t) * pitch + 2 * cw);
            }
#pragma unroll
            for (int b = 0; b < kB; b++) {
                const int cw = 2 * (lane / kGroups + (k0 + b) * kStep), n = col0 + cw;
                if (n >= N) continue;
                uint16_t* o = base + (n >> 2) * plane + ((n >> 1) & 1) * W2;
                if (has_bias) {
                    const float bf = h2f(pbias[cw]);
#pragma unroll
                    for (int t = 0; t < kT; t++) d[b][t] = add_bias_pair(d[b][t], bf);
                }
                if constexpr (kT == 4) {
                    __builtin_nontemporal_store(v4i{static_cast<int>(d[b][0]), static_cast<int>(d[b][1]),
                                                    static_cast<int>(d[b][2]), static_cast<int>(d[b][3])},
                                                reinterpret_cast<v4i*>(o));
                } else {
                    o[0] = static_cast<uint16_t>(d[b][0] & 0xFFFFu);
                    o[1] = static_cast<uint16_t>(d[b][0] >> 16);
                }
            }
        }
    };
    if (ep.vec_out) walk(std::integral_constant<int, 4>{});
    else walk(std::integral_constant<int, 1>{});
}

// Writes the wave's sub-tile (first row m, first column n) through its private staging area:
// lane l of block (j, i) holds row 16 i + l % 16 and the columns 16 j + 4 (l / 16) .. + 3.
// UP: the ConvTranspose2d scatter of GemmEpilogue (FP16 only; w_scale and post_bias per 4 columns).
template <class T, bool DEQUANT, bool UP = false>
__device__ __forceinline__ void ring_store(const T& t, const GemmEpilogue& ep, int wm, int wn, int8_t* stage) {
    constexpr int kTM = T::kTM, kTN = T::kTN;
    constexpr int kEsz = DEQUANT ? 2 : 4;
    constexpr int kPer = 16 / kEsz;                    // elements per 16-byte unit
    constexpr int MB = T::MB;
    constexpr int kU = MB * kTN * kEsz / 16;           // units per staged row
    constexpr int kPitch = 16 * kU + 16;
    const int lane = threadIdx.x & (kWave - 1);
    const int lr = lane % MB, g = lane / MB;
    const int M = ep.M, N = ep.N;

    // Copies kR staged rows from row m0 on to the output as 16-byte row chunks; all LDS reads of
    // a batch are issued before its first store.
    auto flush = [&](auto rows_c, int m0) {
        constexpr int kR = decltype(rows_c)::value;
        constexpr int kUnits = kR * kU;
        constexpr int kIters = (kUnits + kWave - 1) / kWave;
        constexpr int kB = kIters < 8 ? kIters : 8;
#pragma unroll 1
        for (int it = 0; it < kIters; it += kB) {
            v4i v[kB];
#pragma unroll
            for (int b = 0; b < kB; b++) {
                const int idx = min(lane + (it + b) * kWave, kUnits - 1);
                v[b] = *reinterpret_cast<const v4i*>(stage + (idx / kU) * kPitch + (idx % kU) * 16);
            }
#pragma unroll
            for (int b = 0; b < kB; b++) {
                const int idx = lane + (it + b) * kWave;
                const int row = m0 + idx / kU, col = wn + (idx % kU) * kPer;
                if (idx >= kUnits || row >= M || col >= N) continue;
                const size_t o = static_cast<size_t>(row) * N + col;
                if (col + kPer <= N) {
                    // any alignment the element type has: gfx950 stores 16 bytes at any address, and
                    // element stores instead cost twice the whole GEMM's time at an odd N
                    if constexpr (DEQUANT) __builtin_nontemporal_store(v[b], reinterpret_cast<v4i_h*>(ep.c16 + o));
                    else __builtin_nontemporal_store(v[b], reinterpret_cast<v4i_w*>(ep.c32 + o));
                } else {
                    // the row's last columns: element stores (constant register indices)
                    const int n_ok = N - col;
#pragma unroll
                    for (int e = 0; e < kPer; e++) {
                        if (e >= n_ok) break;
                        if constexpr (DEQUANT)
                            ep.c16[o + e] = static_cast<uint16_t>(static_cast<uint32_t>(v[b][e >> 1]) >> (16 * (e & 1)));
                        else
                            ep.c32[o + e] = v[b][e];
                    }
                }
            }
        }
    };

    if constexpr (DEQUANT) {
        float as[kTM];
#pragma unroll
        for (int i = 0; i < kTM; i++) {
            const int m = wm + MB * i + lr;
            as[i] = ep.act_scale[m < M ? m : M - 1];
        }
        // without a bias the bias strip holds w_scale (in range, ignored); the scatter's holds
        // post_bias, added after the GEMM value's own rounding
        const bool has_bias = !UP && ep.bias != nullptr;
        const uint16_t* bsrc = UP ? ep.post_bias : ep.bias;
        if (!bsrc) bsrc = ep.w_scale;
        uint16_t* wsl = reinterpret_cast<uint16_t*>(stage + MB * kTM * kPitch);
        uint16_t* bl = wsl + MB * kTN;
        constexpr int kIt = (MB * kTN + kWave - 1) / kWave;
        uint16_t wv[kIt], bw[kIt];
#pragma unroll
        for (int k = 0; k < kIt; k++) {
            const int n = min(wn + lane + kWave * k, N - 1);
            wv[k] = ep.w_scale[UP ? n >> 2 : n];
            bw[k] = bsrc[UP ? n >> 2 : n];
        }
#pragma unroll
        for (int k = 0; k < kIt; k++) {
            const int c = lane + kWave * k;
            if (c < MB * kTN) {
                wsl[c] = wv[k];
                bl[c] = bw[k];
            }
        }
#pragma unroll
        for (int j = 0; j < kTN; j++) {
            const int nl = MB * j + 4 * g;
            const uint2 w2 = *reinterpret_cast<const uint2*>(wsl + nl);
            const uint2 b2 = *reinterpret_cast<const uint2*>(bl + nl);
            const uint32_t wr[4] = {w2.x & 0xFFFFu, w2.x >> 16, w2.y & 0xFFFFu, w2.y >> 16};
            const uint32_t br[4] = {b2.x & 0xFFFFu, b2.x >> 16, b2.y & 0xFFFFu, b2.y >> 16};
            float ws[4], b[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                ws[e] = h2f(static_cast<uint16_t>(wr[e]));
                b[e] = has_bias ? h2f(static_cast<uint16_t>(br[e])) : -0.0f;   // dequant4_pk: -0 without a bias
            }
#pragma unroll
            for (int i = 0; i < kTM; i++)
                *reinterpret_cast<uint2*>(stage + (MB * i + lr) * kPitch + 2 * nl) =
                    dequant4_pk(t.acc[j][i][0], t.acc[j][i][1], t.acc[j][i][2], t.acc[j][i][3], as[i], ws, b);
        }
        if constexpr (UP) ring_flush_up2x2<MB * kTM, MB * kTN>(stage, kPitch, bl, ep, wm, wn);
        else flush(std::integral_constant<int, MB * kTM>{}, wm);
    } else {
#pragma unroll
        for (int i = 0; i < kTM; i++) {
#pragma unroll
            for (int j = 0; j < kTN; j++)
                *reinterpret_cast<v4i*>(stage + lr * kPitch + 4 * (MB * j + 4 * g)) = t.acc[j][i];
            flush(std::integral_constant<int, MB>{}, wm + MB * i);
        }
    }
}

}  // namespace forge_amd
