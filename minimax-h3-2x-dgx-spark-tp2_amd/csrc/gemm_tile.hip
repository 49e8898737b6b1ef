// Kernel 2's forms of smaller tiles (gfx950): problems and last rounds that 256 x 256 tiles would run on a few CUs.
//
// One workgroup computes one tile, TW weight rows x TT token rows, with WN x WM waves of NI x NJ MFMA blocks each, and
// the launch has at most one tile per CU, so the time is that of one tile: the form taken is the smallest whose tiles
// fit.  Every output element goes through the same MFMA sequence and epilogue arithmetic as in the 256 x 256 tiles
// (v_mfma 32x32x64, weight row at A-row n % 32, token at B-column m % 32, k ascending from a zero accumulator), so the
// output is bitwise the same.
//
// What bounds it: a k-step loads (TW + TT) x 128 bytes per CU by LDS-DMA, 16 cycles per 1 KiB instruction at best (64
// bytes per cycle and CU; measured 20 with out-of-range loads, 25-30 with real ones, where L2 misses wait on the MALL
// or HBM), while its MFMAs take TW TT / 32 cycles.  The small tiles are bound by those loads and by the latency of a
// k-step (barrier, fragment reads, MFMAs), so they keep 7-8 k-steps in flight in an LDS ring and take one barrier per
// two k-steps; the large ones are bound by the fragment reads of their waves (LDS returns 95 bytes per cycle to one
// wave per SIMD, 250 to two), so they run two waves per SIMD.  Measured against the forms before (128 x 192 and 256 x
// 128 tiles of four waves), M x N x K, operands in the MALL: 64 x 5376 x 14336 71.0 -> 20.9 us, 200 x 5376 x 14336 69.6
// -> 29.2 (weights from HBM 83.8 -> 39.7), 512 x 6144 x 4096 24.6 -> 16.9, 2048 x 3072 x 3072 23.5 -> 21.4 (behind its
// quant, both 28.6 -> 28.2: within the noise), 1000 x 5376 x 14336 81.8 -> 67.5 (weights from HBM: 79, the MLP around it
// 242 -> 237), 768 x 9216 x 3072 28.9 -> 23.2.
#include "gemm_core.h"

namespace {

using namespace h3g;

// NST: k-steps of the ring.  KS: k-steps per barrier.
// SW: the tile of kernel 3, whose TW weight rows are TW / 2 gate rows and the matching up rows; a wave's first NI / 2
// blocks are gate rows, the others the up rows of the same channels.
template <int WN_, int WM_, int NI_, int NJ_, int NST_, int KS_, bool SW_ = false>
struct Tile {
    static constexpr int WN = WN_, WM = WM_, NI = NI_, NJ = NJ_, NST = NST_, KS = KS_;
    static constexpr bool SW = SW_;
    static_assert(!SW || NI % 2 == 0, "gate and up blocks in pairs");
    static_assert(NST >= 2 * KS, "ring depth");
    static constexpr int WAVES = WN * WM;
    static constexpr int TW = 32 * NI * WN;              // weight rows per tile
    static constexpr int TT = 32 * NJ * WM;              // token rows per tile
    static constexpr int TC = SW ? TW / 2 : TW;          // output channels per tile
    static constexpr int WG = TW / 8, AG = TT / 8;       // 8-row load groups of a stage
    static constexpr int WL = (WG + WAVES - 1) / WAVES, AL = (AG + WAVES - 1) / WAVES;   // per wave
    static constexpr int LOADS = WL + AL;
    static constexpr int STAGE = (TW + TT) * ROWB;
    static constexpr int A_OFF = TW * ROWB;
    static constexpr int SA_N = (TT + 63) / 64 * 64, SB_N = (TW + 63) / 64 * 64;
    static constexpr int SCALES_OFF = NST * STAGE;
    static constexpr int JUNK_OFF = SCALES_OFF + (SA_N + SB_N) * 4;
    static constexpr bool JUNK = WG % WAVES != 0 || AG % WAVES != 0;
    static constexpr int STG_PER_WAVE = 32 * ((SW ? NI * 32 : NI * 128) + 16);   // SW: NI / 2 blocks of bf16; else of fp32
    // SW: the compact SiLU table, next to the ring where it fits, else behind the staging area once the ring is free
    static constexpr int END = (JUNK_OFF + (JUNK ? 1024 : 0) + 255) / 256 * 256;
    static constexpr bool SILU_LATE = SW && END + SILU_LDS_BYTES > 160 * 1024;
    static constexpr int SILU_OFF = SILU_LATE ? (STG_PER_WAVE * WAVES + 255) / 256 * 256 : END;
    static constexpr int LDS = SW && !SILU_LATE ? END + SILU_LDS_BYTES : END;
    static_assert(!SILU_LATE || SILU_OFF + SILU_LDS_BYTES <= NST * STAGE, "the table in the ring");
    static_assert(LDS <= 160 * 1024, "LDS of one CU");
    static_assert(STG_PER_WAVE * WAVES <= NST * STAGE, "the epilogue stages in the ring");
    static_assert(LOADS * (NST - 1) <= 63, "vmcnt range");
};

constexpr int TILE_GROUP_M = 8;                            // token-tile rows per group of the XCD-contiguous map

template <class T>
struct TileLoader {
    v4u rw, ra;
    uint32_t vw[T::WL], va[T::AL];                       // byte offsets of this lane at k = 0 (OOB: row out of range)
    uint32_t dw, da;                                     // LDS offsets of the wave's first groups within a stage
    uint32_t wbytes, abytes;
    uint32_t k0;                                         // the cursor: byte offset of the next k-step to load ...
    int left;                                            // ... and the k-steps from it on (<= 0: past the last)
    int ktail;                                           // K % BK
};

// The global weight row of row r of tile column tn, -1 past the last.
template <class T>
__device__ __forceinline__ int64_t tile_weight_row(const GemmParams& p, int tn, int r) {
    const int up = T::SW && r >= T::TW / 2;
    const int64_t n = T::SW ? (int64_t)tn * (T::TW / 2) + r - up * (T::TW / 2) : (int64_t)tn * T::TW + r;
    return n < p.N ? n + (up ? p.N : 0) : -1;
}

template <class T>
__device__ __forceinline__ void tile_loader_set(TileLoader<T>& L, const GemmParams& p, int tm, int tn, int wave,
                                                int lane) {
    L.left = (p.K + BK - 1) / BK;
    L.ktail = p.K % BK;
    L.k0 = 0;
    const int lrow = lane >> 3;
    L.rw = buffer_desc(p.w, p.w_bytes);
    L.ra = buffer_desc(p.a, p.a_bytes);
    L.wbytes = L.rw[2];
    L.abytes = L.ra[2];
    L.dw = (uint32_t)(wave * T::WL * 8 * ROWB);
    L.da = T::A_OFF + (uint32_t)(wave * T::AL * 8 * ROWB);
#pragma unroll
    for (int j = 0; j < T::WL; ++j) {
        const int g = wave * T::WL + j;
        const int64_t row = tile_weight_row<T>(p, tn, 8 * g + lrow);
        const bool ok = g < T::WG && row >= 0;
        L.vw[j] = ok ? (uint32_t)(row * p.ldw) + 16u * (uint32_t)((lane & 7) ^ swz(8 * (g & 1) + lrow)) : OOB;
    }
#pragma unroll
    for (int j = 0; j < T::AL; ++j) {
        const int g = wave * T::AL + j;
        const int64_t row = (int64_t)tm * T::TT + 8 * g + lrow;
        const bool ok = g < T::AG && row < p.M;
        L.va[j] = ok ? (uint32_t)(row * p.lda) + 16u * (uint32_t)((lane & 7) ^ swz(8 * (g & 1) + lrow)) : OOB;
    }
}

// Before the loads of the cursor's k-step.  The last k-step of a K that is no multiple of BK cuts the lanes past K off
// for good; past the last k-step the descriptors are empty (their offset too), so the loads read zeros.
template <class T>
__device__ __forceinline__ void tile_loader_edge(TileLoader<T>& L, int wave, int lane) {
    if (__builtin_expect(L.left == 1 && L.ktail != 0, 0)) {
        const int lrow = lane >> 3;
#pragma unroll
        for (int j = 0; j < T::WL; ++j)
            if (16 * ((lane & 7) ^ swz(8 * ((wave * T::WL + j) & 1) + lrow)) >= L.ktail) L.vw[j] = OOB;
#pragma unroll
        for (int j = 0; j < T::AL; ++j)
            if (16 * ((lane & 7) ^ swz(8 * ((wave * T::AL + j) & 1) + lrow)) >= L.ktail) L.va[j] = OOB;
    }
    const bool live = L.left > 0;
    L.rw[2] = live ? L.wbytes : 0;
    L.ra[2] = live ? L.abytes : 0;
    L.k0 = live ? L.k0 : 0;
}

template <class T>
__device__ __forceinline__ void tile_loader_next(TileLoader<T>& L) {
    --L.left;
    L.k0 += BK;
}

template <class T>
__device__ __forceinline__ void tile_issue(const TileLoader<T>& L, uint32_t st, uint32_t junk, int wave, int j) {
    if (j < T::WL) {
        const bool in = T::WG % T::WAVES == 0 || wave * T::WL + j < T::WG;
        dma16_at(L.rw, in ? st + L.dw + (uint32_t)(j * 8 * ROWB) : junk, L.vw[j], L.k0);
    } else {
        const int i = j - T::WL;
        const bool in = T::AG % T::WAVES == 0 || wave * T::AL + i < T::AG;
        dma16_at(L.ra, in ? st + L.da + (uint32_t)(i * 8 * ROWB) : junk, L.va[i], L.k0);
    }
}

// Fragment f of a k-step (both sub-steps): sub f / (NI + NJ), then NI weight blocks and NJ token blocks.
template <class T>
struct Frags {
    v8i a[2][T::NI], b[2][T::NJ];
};

// The tile row of weight block i of wave column wn.
template <class T>
__device__ __forceinline__ int tile_block_row(int wn, int i) {
    if (!T::SW) return (wn * T::NI + i) * 32;
    return i < T::NI / 2 ? (wn * T::NI / 2 + i) * 32 : T::TW / 2 + (wn * T::NI / 2 + i - T::NI / 2) * 32;
}

template <class T>
__device__ __forceinline__ void tile_read(Frags<T>& F, const uint8_t* stage, int wn, int wm, int lane, int f) {
    const int sub = f / (T::NI + T::NJ), r = f % (T::NI + T::NJ);
    if (r < T::NJ) F.b[sub][r] = read_frag(stage + T::A_OFF + (wm * T::NJ + r) * 32 * ROWB, lane, sub);
    else F.a[sub][r - T::NJ] = read_frag(stage + tile_block_row<T>(wn, r - T::NJ) * ROWB, lane, sub);
}

template <class T>
__device__ __forceinline__ uint32_t tile_next_slot(uint32_t s) {
    return s == (T::NST - 1) * T::STAGE ? 0 : s + T::STAGE;
}

// One k-step on the fragments F.  BAR: it publishes the next KS k-steps and frees the ring slots of the KS k-steps
// whose fragments are all read.  READ: the next k-step's fragments (ring slot rd) are read into G.  LOAD: the cursor's
// k-step is loaded into slot ld.
template <class T, bool BAR, bool READ, bool LOAD>
__device__ __forceinline__ void tile_kstep(const uint8_t* lds, uint32_t lds0, uint32_t rd, uint32_t ld,
                                           TileLoader<T>& L, int wave, int wn, int wm, int lane, v16f acc[T::NI][T::NJ],
                                           const Frags<T>& F, Frags<T>& G) {
    constexpr int NM = 2 * T::NI * T::NJ, NR = 2 * (T::NI + T::NJ);
    if (BAR) {
        wait_lgkm0();
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(T::LOADS * (T::NST - 2 * T::KS)));
        barrier_nofence();
    }
    if (LOAD) tile_loader_edge(L, wave, lane);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < NM; ++u) {
        const int sub = u / (NM / 2), t = u % (NM / 2), i = t / T::NJ, j = t % T::NJ;
        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(F.a[sub][i], F.b[sub][j], acc[i][j], 0, 0, 0, 0, 0, 0);
        if (READ) {
#pragma unroll
            for (int f = u * NR / NM; f < (u + 1) * NR / NM; ++f) tile_read<T>(G, lds + rd, wn, wm, lane, f);
        }
        if (LOAD) {
#pragma unroll
            for (int f = u * T::LOADS / NM; f < (u + 1) * T::LOADS / NM; ++f)
                tile_issue<T>(L, lds0 + ld, lds0 + T::JUNK_OFF, wave, f);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    if (LOAD) tile_loader_next(L);
}

// The 32 staged token rows from m0 on (CH 16-byte chunks each, at a stride padded by 16 bytes) to their output rows, chunk
// c of row t by lane (CH t + c) % 64 of instruction (CH t + c) / 64, so that every store writes whole row segments (the
// store path handles about one 128-byte line per cycle: the lines an instruction touches are what it costs).  Rows past M
// fall outside the output descriptor's range, columns past N get an out-of-range offset.  The stores go through the XCD's
// L2 at device scope (sc1): a launch of one round otherwise ends with all of its output dirty there.  Plain / sc1 / nt:
// 2048 x 3072 x 3072 22.1 / 21.4 / 21.6 us, 768 x 9216 x 3072 24.8 / 23.2 / 24.8, 512 x 6144 x 4096 18.5 / 18.3 / 18.3.
template <int CH, int ELEM, bool MAY_NT>
__device__ __forceinline__ void tile_store(const GemmParams& p, __amdgpu_buffer_rsrc_t yr, int col0, int m0, int lane,
                                           const uint8_t* stg) {
    constexpr int NS = 32 * CH / 64;
    static_assert((32 * CH) % 64 == 0, "whole store instructions per block row");
    const uint32_t row = (uint32_t)p.ldy * ELEM;
    wave_sync();                                         // every lane's writes before any lane's reads
    v4u v[NS];
    uint32_t off[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {                       // all reads before the first store
        const int idx = 64 * s + lane, t = idx / CH, c = idx - t * CH;
        v[s] = *reinterpret_cast<const v4u*>(stg + t * (CH * 16 + 16) + c * 16);
        const int n = col0 + c * (16 / ELEM);
        off[s] = (n < p.N) ? (uint32_t)(m0 + t) * row + (uint32_t)n * ELEM : OOB;
    }
    if (MAY_NT && p.y_nt) {
#pragma unroll
        for (int s = 0; s < NS; ++s) __builtin_amdgcn_raw_buffer_store_b128(v[s], yr, off[s], 0, 2);
    } else {
#pragma unroll
        for (int s = 0; s < NS; ++s) __builtin_amdgcn_raw_buffer_store_b128(v[s], yr, off[s], 0, 16);
    }
}

// The row maximum of token m from the two lanes that hold its channels.
__device__ __forceinline__ void tile_row_amax(const GemmParams& p, int m, uint32_t v, int lane) {
    const uint32_t o = (uint32_t)__shfl_xor((int)v, 32, 64);
    v = v > o ? v : o;
    if (lane < 32 && m < p.M && v) atomicMax(reinterpret_cast<unsigned int*>(p.row_amax) + m, v);
}

// Block (i, j) of a wave's accumulators: register 4q + r is channel col0 + 32 i + 8 q + 4 (lane >> 5) + r of token
// mrow0 + 32 j + (lane & 31); sa_l and sb_l (LDS) hold the scales of the wave's tokens and channels.  The 32 tokens of a
// block row j go through the wave's LDS area `stg`, rows of NI x 32 outputs.
template <int OUT_DT, int NI, int NJ>
__device__ __forceinline__ void tile_epilogue(const GemmParams& p, int col0, int mrow0, const float* sa_l,
                                              const float* sb_l, int lane, const v16f (&acc)[NI][NJ], uint8_t* stg) {
    constexpr int ELEM = OUT_DT == H3FP8_DT_F32 ? 4 : 2;
    constexpr int CH = NI * 2 * ELEM;                    // 16-byte chunks per staged token row
    constexpr int RS = CH * 16 + 16;                     // staged row stride (padded: rows fall on other banks)
    const int hi = lane >> 5, mj = lane & 31;
    const __amdgpu_buffer_rsrc_t yr = make_rsrc(p.y, p.y_bytes);
    const bool has_bias = p.bias != nullptr, amax = p.row_amax != nullptr;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int m = mrow0 + 32 * j + mj;
        const float sam = sa_l[32 * j + mj];
        uint32_t rmax = 0;
        wave_sync();                                     // the previous block row's reads before these writes
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (OUT_DT == H3FP8_DT_F32) {            // the raw accumulators
                    const v4f v = {acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
                    *reinterpret_cast<v4f*>(stg + mj * RS + (8 * i + 2 * q + hi) * 16) = v;
                    continue;
                }
                const int n = col0 + 32 * i + 8 * q + 4 * hi;
                const v4f sbn = *reinterpret_cast<const v4f*>(sb_l + 32 * i + 8 * q + 4 * hi);
                float v[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] = sbn[r] * acc[i][j][4 * q + r];
                if (has_bias) {                          // uniform; columns past N read column 0 (not stored)
                    const int nc = n < p.N ? n : 0;
#pragma unroll
                    for (int r = 0; r < 4; ++r) v[r] = __builtin_fmaf(sam, v[r], load_bias(p.bias, nc + r, OUT_DT));
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r) v[r] = sam * v[r];
                }
                uint32_t lo, hi2;
                if (OUT_DT) {
                    lo = fp16_rne(v[0]) | (fp16_rne(v[1]) << 16);
                    hi2 = fp16_rne(v[2]) | (fp16_rne(v[3]) << 16);
                } else {
                    lo = cvt_bf16x2(v[0], v[1]);
                    hi2 = cvt_bf16x2(v[2], v[3]);
                }
                if (amax && n < p.N)
                    rmax = OUT_DT ? max_abs_f16x2(max_abs_f16x2(rmax, lo), hi2)
                                  : max_abs_bf16x2(max_abs_bf16x2(rmax, lo), hi2);
                const v2u32 val = {lo, hi2};
                *reinterpret_cast<v2u32*>(stg + mj * RS + (4 * i + q) * 16 + 8 * hi) = val;
            }
        tile_store<CH, ELEM, OUT_DT == H3FP8_DT_F32>(p, yr, col0, mrow0 + 32 * j, lane, stg);
        if (amax) tile_row_amax(p, m, rmax, lane);
    }
}

// Kernel 3's: blocks (t, j) and (NT + t, j) are the gate and the up of channels col0 + 32 t + ...; sb_l holds the gate
// scales and, up_off entries on, the up scales.  The arithmetic and the SiLU lookup (the compact table `silu_l`, or the
// full one for a block with a gate outside its range) are those of the 256 x 256 tiles.
template <int NT, int NJ>
__device__ __forceinline__ void swiglu_epilogue(const GemmParams& p, int col0, int mrow0, const float* sa_l,
                                                const float* sb_l, int up_off, const uint16_t* silu_l, int lane,
                                                const v16f (&acc)[2 * NT][NJ], uint8_t* stg) {
    constexpr int CH = NT * 4, RS = CH * 16 + 16;
    const int hi = lane >> 5, mj = lane & 31;
    const __amdgpu_buffer_rsrc_t yr = make_rsrc(p.y, p.y_bytes);
    const bool has_bias = p.bias != nullptr, amax = p.row_amax != nullptr;
    const float zero = opaque_zero();
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int m = mrow0 + 32 * j + mj;
        const float sam = sa_l[32 * j + mj];
        uint32_t rmax = 0;
        wave_sync();                                     // the previous block row's reads before these writes
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            uint32_t key[4][4], uu[4][4], sl[4][4];
            uint64_t outside = 0;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int c = 32 * t + 8 * q + 4 * hi, f = col0 + c;
                const v4f sbg = *reinterpret_cast<const v4f*>(sb_l + c);
                const v4f sbu = *reinterpret_cast<const v4f*>(sb_l + up_off + c);
                const int fc = f < p.N ? f : 0;          // columns past F read column 0 of the bias (not stored)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float tg = sbg[r] * acc[t][j][4 * q + r], tu = sbu[r] * acc[NT + t][j][4 * q + r];
                    float gy, uy;
                    if (has_bias) {                      // uniform
                        gy = __builtin_fmaf(sam, tg, load_bias(p.bias, fc + r, 0));
                        uy = __builtin_fmaf(sam, tu, load_bias(p.bias, p.N + fc + r, 0));
                    } else {
                        gy = sam * tg;
                        uy = sam * tu;
                    }
                    uu[q][r] = cvt_bf16x2(0.0f, uy);
                    key[q][r] = ((cvt_bf16x2(gy, gy) >> 15) & 0xffffu) - H3_SILU_ROT_R0;
                    outside |= __ballot(key[q][r] >= (uint32_t)H3_SILU_ROT_LEN);
                }
            }
            if (outside == 0) {
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int r = 0; r < 4; ++r) sl[q][r] = silu_l[key[q][r]];
            } else {
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const uint32_t rk = (key[q][r] + H3_SILU_ROT_R0) & 0xffffu;
                        sl[q][r] = p.silu[(rk >> 1) | ((rk & 1u) << 15)];
                    }
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float hv[4];
#pragma unroll
                for (int r = 0; r < 4; ++r)              // -0 up -> +0 (fp8_swiglu.py:66)
                    hv[r] = bf16_to_f32(sl[q][r]) * (u2f(uu[q][r]) + zero);
                const v2u32 val = {cvt_bf16x2(hv[0], hv[1]), cvt_bf16x2(hv[2], hv[3])};
                if (amax && col0 + 32 * t + 8 * q + 4 * hi < p.N)
                    rmax = max_abs_bf16x2(max_abs_bf16x2(rmax, val[0]), val[1]);
                *reinterpret_cast<v2u32*>(stg + mj * RS + (4 * t + q) * 16 + 8 * hi) = val;
            }
        }
        tile_store<CH, 2, false>(p, yr, col0, mrow0 + 32 * j, lane, stg);
        if (amax) tile_row_amax(p, m, rmax, lane);
    }
}

// Workgroup -> tile of a launch that covers what a full-tile launch over the first `tail_first` tiles of the
// XCD-contiguous map (tile_of) has left, each 256 x 256 tile cut into CW x CT tiles.  That launch took the first
// tail_first / 8 positions of each of the 8 per-XCD ranges; the `tail_rest` positions left are listed range by range (so
// consecutive entries are consecutive positions), cut, and dealt out by the same XCD-contiguous rule: the pieces of a tile
// and neighbouring tiles run on one XCD and share its L2.  Behind them come the tiles of the token rows past the map's
// tiles_m x 256, column by column.
template <class T>
__device__ __forceinline__ void tail_tile_of(const GemmParams& p, int id, int count, int& tm, int& tn) {
    constexpr int CW = 256 / T::TW, CT = 256 / T::TT;
    const int xcd = id & 7, local = id >> 3;
    const int per = count >> 3, rem = count & 7;
    const int lid = (xcd < rem) ? xcd * (per + 1) + local : rem * (per + 1) + (xcd - rem) * per + local;
    int k = lid / (CW * CT);
    if (k >= p.tail_rest) {
        const int e = lid - p.tail_rest * (CW * CT);
        const int rows = (p.M - p.tiles_m * 256 + T::TT - 1) / T::TT;
        tm = p.tiles_m * CT + e % rows;
        tn = e / rows;
        return;
    }
    const int sub = lid - k * (CW * CT);
    const int tiles = p.tiles_m * p.tiles_n, pT = tiles >> 3, rT = tiles & 7, done = p.tail_first >> 3;
    int c = 0;
    for (; c < 7; ++c) {
        const int n_c = pT + (c < rT ? 1 : 0) - done;
        if (k < n_c) break;
        k -= n_c;
    }
    const int pos = ((c < rT) ? c * (pT + 1) : rT * (pT + 1) + (c - rT) * pT) + done + k;
    const int in_group = p.group_m * p.tiles_n;
    const int g = pos / in_group;
    const int first = g * p.group_m;
    const int gsz = min(p.tiles_m - first, p.group_m);
    const int r = pos - g * in_group;
    tm = (first + r % gsz) * CT + sub % CT;
    tn = (r / gsz) * CW + sub / CT;
}

template <int OUT_DT, class T>
__global__ void __launch_bounds__(T::WAVES * 64, 2) gemm_tile_kernel(GemmParams p) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[T::LDS];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int wn = wave % T::WN, wm = wave / T::WN;
    const uint32_t lds0 = lds_addr(lds);
    int tm, tn;
    if (p.tail_first >= 0) {                             // uniform
        tail_tile_of<T>(p, (int)blockIdx.x, (int)gridDim.x, tm, tn);
        if (tm * T::TT >= p.M || tn * T::TC >= p.N) return;      // a piece past the edge of its 256 x 256 tile's rows
    } else {
        const int tiles_m = (p.M + T::TT - 1) / T::TT;
        tile_of((int)blockIdx.x, (int)gridDim.x, tiles_m, (int)gridDim.x / tiles_m, TILE_GROUP_M, tm, tn);
    }
    TileLoader<T> L;
    tile_loader_set(L, p, tm, tn, wave, lane);
    {   // the tile's scales: 64 entries per load, dealt over the waves
        const v4u rsa = buffer_desc(p.sa, p.sa_stride ? (uint32_t)((p.M - 1) * p.sa_stride * 4 + 4) : 4u);
        const v4u rsb = buffer_desc(p.sb, p.sb_stride ? (uint32_t)((p.w_rows - 1) * p.sb_stride * 4 + 4) : 4u);
        for (int c = wave; c < (T::SA_N + T::SB_N) / 64; c += T::WAVES) {
            const uint32_t dst = lds0 + T::SCALES_OFF + (uint32_t)c * 256u;
            if (c < T::SA_N / 64) {
                const int64_t r = (int64_t)tm * T::TT + 64 * c + lane;
                dma4(rsa, dst, r < p.M ? (uint32_t)(r * p.sa_stride * 4) : OOB);
            } else {
                const int e = 64 * c - T::SA_N + lane;
                const int64_t r = e < T::TW ? tile_weight_row<T>(p, tn, e) : -1;
                dma4(rsb, dst, r >= 0 ? (uint32_t)(r * p.sb_stride * 4) : OOB);
            }
        }
    }
    auto load_silu = [&]() {                              // 256 bytes per load, dealt over the waves
        const v4u td = buffer_desc(p.silu_rot, SILU_LDS_BYTES);
        for (int c = wave; c < SILU_LDS_BYTES / 256; c += T::WAVES)
            dma4(td, lds0 + T::SILU_OFF + (uint32_t)c * 256u, (uint32_t)c * 256u + 4u * (uint32_t)lane);
    };
    if (T::SW && !T::SILU_LATE) load_silu();
#pragma unroll
    for (int s = 0; s < T::NST; ++s) {
        tile_loader_edge(L, wave, lane);
#pragma unroll
        for (int j = 0; j < T::LOADS; ++j)
            tile_issue<T>(L, lds0 + (uint32_t)s * T::STAGE, lds0 + T::JUNK_OFF, wave, j);
        tile_loader_next(L);
    }
    v16f acc[T::NI][T::NJ];
#pragma unroll
    for (int i = 0; i < T::NI; ++i)
#pragma unroll
        for (int j = 0; j < T::NJ; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(T::LOADS * (T::NST - T::KS)));
    barrier_nofence();
    Frags<T> F, G;
#pragma unroll
    for (int f = 0; f < 2 * (T::NI + T::NJ); ++f) tile_read<T>(F, lds, wn, wm, lane, f);
    // k-steps in pairs on F and G; an odd count takes one more, of zeros, which leaves every accumulator as it is (one
    // path for both, so that no accumulator is copied right behind its last MFMA)
    uint32_t ld = 0, rd = T::STAGE;
    int left = (p.K + 2 * BK - 1) / (2 * BK);
    if (T::KS == 2) {
        tile_kstep<T, false, true, false>(lds, lds0, rd, ld, L, wave, wn, wm, lane, acc, F, G);
        for (; left > 1; --left) {
            rd = tile_next_slot<T>(rd);
            tile_kstep<T, true, true, true>(lds, lds0, rd, ld, L, wave, wn, wm, lane, acc, G, F);
            rd = tile_next_slot<T>(rd), ld = tile_next_slot<T>(ld);
            tile_kstep<T, false, true, true>(lds, lds0, rd, ld, L, wave, wn, wm, lane, acc, F, G);
            ld = tile_next_slot<T>(ld);
        }
    } else {
        for (; left > 1; --left) {
            tile_kstep<T, true, true, true>(lds, lds0, rd, ld, L, wave, wn, wm, lane, acc, F, G);
            rd = tile_next_slot<T>(rd), ld = tile_next_slot<T>(ld);
            tile_kstep<T, true, true, true>(lds, lds0, rd, ld, L, wave, wn, wm, lane, acc, G, F);
            rd = tile_next_slot<T>(rd), ld = tile_next_slot<T>(ld);
        }
        tile_kstep<T, true, true, true>(lds, lds0, rd, ld, L, wave, wn, wm, lane, acc, F, G);
    }
    tile_kstep<T, false, false, false>(lds, lds0, rd, ld, L, wave, wn, wm, lane, acc, G, F);
    accumulators_ready<(T::WAVES <= 4)>(acc);
    // the reads of the last k-steps have returned before the ring is reused
    wait_lgkm0();
    // the ring becomes the epilogue's staging area once every wave's last reads have returned and the trailing
    // zero-fill loads have landed
    wait_vm0();
    barrier_nofence();
    const float* sa_l = reinterpret_cast<const float*>(lds + T::SCALES_OFF);
    if constexpr (T::SW) {
        if (T::SILU_LATE) {
            load_silu();
            wait_vm0();
            barrier_nofence();
        }
        swiglu_epilogue<T::NI / 2, T::NJ>(p, tn * T::TC + wn * T::NI * 16, tm * T::TT + wm * T::NJ * 32,
                                          sa_l + wm * T::NJ * 32, sa_l + T::SA_N + wn * T::NI * 16, T::TC,
                                          reinterpret_cast<const uint16_t*>(lds + T::SILU_OFF), lane, acc,
                                          lds + wave * T::STG_PER_WAVE);
        return;
    }
    tile_epilogue<OUT_DT, T::NI, T::NJ>(p, tn * T::TW + wn * T::NI * 32, tm * T::TT + wm * T::NJ * 32,
                                        sa_l + wm * T::NJ * 32, sa_l + T::SA_N + wn * T::NI * 32, lane, acc,
                                        lds + wave * T::STG_PER_WAVE);
}

// The forms (enum TileForm): WN x WM waves of NI x NJ blocks, ring, k-steps per barrier.  Rings and wave splits are the
// best of those measured for the tile (32 x 64 with 4 / 8 k-steps in flight, 64 x 5376 x 14336 from HBM: 30.6 / 26.6 us;
// 128 x 128 with one barrier per k-step / per two, 512 x 6144 x 4096: 17.0 / 20.2 us; 192 x 128 as 6 x 2 waves of 1 x 2 or
// 3 x 4 waves of 2 x 1 blocks: 1-3 % slower than 2 x 4 of 3 x 1; 256 x 128 with a ring of 2: 768 x 9216 x 3072 35.3 us
// against 26.9).  96 x 128, 64 x 128 and 32 x 128 tiles measured between their neighbours or equal to them.
#define H3_TILE_FORMS(X)                                                                                               \
    X(TILE_32x64, 1, 2, 1, 1, 8, 2)                                                                                    \
    X(TILE_64x64, 2, 2, 1, 1, 8, 2)                                                                                    \
    X(TILE_96x64, 3, 2, 1, 1, 7, 2)                                                                                    \
    X(TILE_128x64, 4, 1, 1, 2, 6, 2)                                                                                   \
    X(TILE_128x128, 2, 4, 2, 1, 4, 1)                                                                                  \
    X(TILE_192x128, 2, 4, 3, 1, 3, 1)                                                                                  \
    X(TILE_256x128, 4, 2, 2, 2, 3, 1)

// Kernel 3's forms: the ring of 256 x 128 leaves the compact SiLU table no room, so that form loads it at its end.
#define H3_SWIGLU_FORMS(X)                                                                                             \
    X(TILE_64x64, 1, 2, 2, 1, 7, 2, true)                                                                              \
    X(TILE_128x64, 2, 2, 2, 1, 5, 2, true)                                                                             \
    X(TILE_128x128, 2, 4, 2, 1, 4, 1, true)                                                                            \
    X(TILE_192x128, 3, 4, 2, 1, 3, 1, true)                                                                            \
    X(TILE_256x128, 4, 2, 2, 2, 3, 1, true)

constexpr bool swiglu_form(int form) { return form != TILE_32x64 && form != TILE_96x64; }

struct FormDims { int tw, tt; };
constexpr FormDims kForms[TILE_FORMS] = {
#define X(id, WN, WM, NI, NJ, NST, KS) {32 * WN * NI, 32 * WM * NJ},
    H3_TILE_FORMS(X)
#undef X
};

template <class T>
int launch_form(const GemmParams& p, int64_t tiles, int out_dt, hipStream_t st) {
    const dim3 grid((unsigned)tiles), block(T::WAVES * 64);
    if (out_dt == H3FP8_DT_F32) hipLaunchKernelGGL((gemm_tile_kernel<H3FP8_DT_F32, T>), grid, block, 0, st, p);
    else if (out_dt == H3FP8_DT_BF16) hipLaunchKernelGGL((gemm_tile_kernel<H3FP8_DT_BF16, T>), grid, block, 0, st, p);
    else hipLaunchKernelGGL((gemm_tile_kernel<H3FP8_DT_FP16, T>), grid, block, 0, st, p);
    H3_CHECK_HIP(hipGetLastError());
    return H3FP8_OK;
}

int launch_any(const GemmParams& p, int form, int64_t tiles, int out_dt, bool swiglu, hipStream_t st) {
    if (swiglu) {
        switch (form) {
#define X(id, ...)                                                                                                     \
    case id:                                                                                                           \
        hipLaunchKernelGGL((gemm_tile_kernel<H3FP8_DT_BF16, Tile<__VA_ARGS__>>), dim3((unsigned)tiles),                \
                           dim3(Tile<__VA_ARGS__>::WAVES * 64), 0, st, p);                                             \
        H3_CHECK_HIP(hipGetLastError());                                                                               \
        return H3FP8_OK;
            H3_SWIGLU_FORMS(X)
#undef X
        }
    } else {
        switch (form) {
#define X(id, ...) case id: return launch_form<Tile<__VA_ARGS__>>(p, tiles, out_dt, st);
            H3_TILE_FORMS(X)
#undef X
        }
    }
    h3host::set_error("bad tile form %d", form);
    return H3FP8_EINVAL;
}

// Tiles of a form over an M x N output.
int64_t tile_count(int form, int64_t M, int64_t N) {
    const FormDims d = kForms[form];
    return ((M + d.tt - 1) / d.tt) * ((N + d.tw - 1) / d.tw);
}

}  // namespace

namespace h3g {

int tile_form_for(int64_t M, int64_t w_rows, bool swiglu, int64_t limit) {
    int f = 0;
    while (f < TILE_FORMS && ((swiglu && !swiglu_form(f)) || tile_count(f, M, w_rows) > limit)) ++f;
    return f;
}

int launch_tiles(GemmParams p, int form, int out_dt, bool swiglu, hipStream_t st) {
    p.tail_first = -1;
    return launch_any(p, form, tile_count(form, p.M, p.w_rows), out_dt, swiglu, st);
}

int64_t tail_pieces(int form, int64_t M, int64_t w_rows, int panels, int64_t rest) {
    const FormDims d = kForms[form];
    if (256 % d.tw != 0) return INT64_MAX;
    const int64_t edge = M - (int64_t)panels * 256;
    return rest * (256 / d.tw) * (256 / d.tt) + (edge > 0 ? (edge + d.tt - 1) / d.tt * ((w_rows + d.tw - 1) / d.tw) : 0);
}

int tail_form_for(int64_t M, int64_t w_rows, bool swiglu, int panels, int64_t rest, int64_t limit) {
    int f = 0;
    while (f < TILE_FORMS && ((swiglu && !swiglu_form(f)) || tail_pieces(f, M, w_rows, panels, rest) > limit)) ++f;
    return f;
}

int launch_tile_tail(GemmParams p, int form, int first, int rest, int out_dt, bool swiglu, hipStream_t st) {
    p.tail_first = first;
    p.tail_rest = rest;
    return launch_any(p, form, tail_pieces(form, p.M, p.w_rows, p.tiles_m, rest), out_dt, swiglu, st);
}

}  // namespace h3g
