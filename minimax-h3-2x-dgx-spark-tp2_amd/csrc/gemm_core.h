// What the GEMM forms share (gfx950): the problem's parameters, the tile map, the LDS row layout and its fragment reads,
// the LDS-DMA loads and their waits, and the epilogue from the accumulators.
#pragma once

#include "h3fp8_common.h"

namespace h3g {

using namespace h3;

typedef float v16f __attribute__((ext_vector_type(16)));
typedef unsigned int v2u32 __attribute__((ext_vector_type(2)));

constexpr int BK = 128;          // k per stage: 128-byte row pieces
constexpr int ROWB = BK;         // bytes per LDS row

constexpr uint32_t OOB = 0x80000000u;         // an offset past every buffer's range: the load returns zeros

enum Epi { EPI_PLAIN = 0, EPI_AMAX = 1, EPI_SWIGLU = 2 };

struct GemmParams {
    const uint8_t* a;          // [M, K] e4m3, row stride lda
    const uint8_t* w;          // [Nw, K] e4m3, row stride ldw (Nw = N, or 2F for SwiGLU)
    const float* sa;
    const float* sb;
    const void* bias;
    void* y;                   // [M, N] (SwiGLU: [M, F])
    float* row_amax;           // EPI_AMAX / EPI_SWIGLU (may be null for SwiGLU)
    const uint16_t* silu;      // SwiGLU table
    const uint16_t* silu_rot;  // its compact rotated-key copy (loaded into LDS)
    int64_t lda, ldw, ldy;
    int64_t sa_stride, sb_stride;
    int M, N, K;               // SwiGLU: N = F (output width)
    int w_rows;                // rows of w and entries of sb (N, or 2F for SwiGLU)
    uint32_t a_bytes, w_bytes; // buffer ranges
    uint32_t y_bytes;          // output range: ((M - 1) * ldy + N) * element size; stores past it are dropped
    int tiles_m, tiles_n;
    int group_m;
    int tile_offset;           // grouped launches: first block of this problem
    int tail_first;            // tail launches: the first 256 x 256 tile (in the full tiles' order) they cover; else -1
    int tail_rest;             // ... and how many of those tiles
    int y_nt;                  // fp32 outputs: store non-temporally (the whole product is larger than the MALL)
};

// block index -> (tile_m, tile_n): XCD-contiguous ranges, then GROUP_M-row groups (column-major inside a group).
__device__ __forceinline__ void tile_of(int b, int T, int tiles_m, int tiles_n, int group_m, int& tm, int& tn) {
    const int xcd = b & 7, local = b >> 3;
    const int per = T >> 3, rem = T & 7;
    int lid = (xcd < rem) ? xcd * (per + 1) + local : rem * (per + 1) + (xcd - rem) * per + local;
    const int in_group = group_m * tiles_n;
    const int g = lid / in_group;
    const int first = g * group_m;
    const int gsz = min(tiles_m - first, group_m);
    const int r = lid - g * in_group;
    tm = first + r % gsz;
    tn = r / gsz;
}

// LDS chunk swizzle (see the header): logical 16-byte chunk c of row r is stored at chunk c ^ swz(r).
__device__ __forceinline__ int swz(int r) { return ((r >> 1) & 7) ^ ((r & 1) << 2); }

// One 32 x 64 MFMA operand of k sub-step `sub`: lane l reads row (l & 31) of the tile, logical chunks 4 sub + 2h and
// 4 sub + 2h + 1 (h = l >> 5).  Tile bases are multiples of 32 rows, so swz of the tile row equals swz of the LDS row.
__device__ __forceinline__ v8i read_frag(const uint8_t* tile, int lane, int sub) {
    const int row = lane & 31, h = lane >> 5;
    const uint8_t* p = tile + row * ROWB;
    const int s = swz(row);
    const int c0 = 4 * sub + 2 * h;
    const uint4 lo = *reinterpret_cast<const uint4*>(p + ((c0 ^ s) << 4));
    const uint4 hi = *reinterpret_cast<const uint4*>(p + (((c0 + 1) ^ s) << 4));
    v8i f;
    f[0] = (int)lo.x; f[1] = (int)lo.y; f[2] = (int)lo.z; f[3] = (int)lo.w;
    f[4] = (int)hi.x; f[5] = (int)hi.y; f[6] = (int)hi.z; f[7] = (int)hi.w;
    return f;
}

__device__ __forceinline__ float load_bias(const void* bias, int n, int out_dt) {
    uint16_t b = reinterpret_cast<const uint16_t*>(bias)[n];
    return out_dt ? fp16_to_f32(b) : bf16_to_f32(b);
}

// s_waitcnt immediate for vmcnt(n) alone (gfx9 encoding: vmcnt[3:0] in bits 3:0, vmcnt[5:4] in bits 15:14, expcnt
// and lgkmcnt left at their maxima).
constexpr int vmcnt_imm(int n) { return (n & 0xf) | ((n >> 4) << 14) | (0x7 << 4) | (0xf << 8); }

__device__ __forceinline__ void wait_vm0() { __builtin_amdgcn_s_waitcnt(vmcnt_imm(0)); }

__device__ __forceinline__ void wait_lgkm0() { __builtin_amdgcn_s_waitcnt(0xc07f); }

// Workgroup barrier without a memory-model fence: __syncthreads() would add a release fence that waits for every
// in-flight LDS-DMA load (vmcnt(0)), including the k-steps still being prefetched.  The explicit vmcnt/lgkmcnt waits
// before it carry the ordering; the "memory" clobber keeps the compiler from moving LDS accesses across it.
__device__ __forceinline__ void barrier_nofence() { asm volatile("s_barrier" ::: "memory"); }

// A buffer descriptor as four dwords (base, stride 0, num_records = byte range, gfx9 raw-buffer flags); loads at
// offsets >= num_records return zeros.
__device__ __forceinline__ v4u buffer_desc(const void* base, uint32_t bytes) {
    const uint64_t b = reinterpret_cast<uint64_t>(base);
    v4u d;
    d[0] = __builtin_amdgcn_readfirstlane((uint32_t)b);
    d[1] = __builtin_amdgcn_readfirstlane((uint32_t)(b >> 32) & 0xffffu);
    d[2] = __builtin_amdgcn_readfirstlane(bytes);
    d[3] = 0x00020000u;
    return d;
}

// 16 bytes per lane from a buffer straight into LDS at lds_base + 16 * lane (buffer_load_dwordx4 ... lds).
// Written as inline asm so that the compiler's wait-count pass does not track these loads: it cannot tell one LDS
// stage from another and would wait for every in-flight load before each LDS read.  The kernel therefore places
// every wait on these loads itself (wait_vm before the barrier that publishes a stage).  The s_nop is the wait state that
// gfx9 needs between a scalar write of M0 and an LDS-DMA load, which the compiler leaves out of inline asm.
__device__ __forceinline__ void dma16(v4u desc, uint32_t lds_base, uint32_t voff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                 :
                 : "s"(lds_base), "v"(voff), "s"(desc)
                 : "memory", "m0");
}

// The same load at a further uniform byte offset.
__device__ __forceinline__ void dma16_at(v4u desc, uint32_t lds_base, uint32_t voff, uint32_t soff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :
                 : "s"(lds_base), "v"(voff), "s"(desc), "s"(soff)
                 : "memory", "m0");
}

// ... with the non-temporal hint, for operands that stream through once.
__device__ __forceinline__ void dma16_at_nt(v4u desc, uint32_t lds_base, uint32_t voff, uint32_t soff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen nt lds"
                 :
                 : "s"(lds_base), "v"(voff), "s"(desc), "s"(soff)
                 : "memory", "m0");
}

__device__ __forceinline__ uint32_t lds_addr(const uint8_t* p) {
    typedef const __attribute__((address_space(3))) uint8_t* lds_u8;
    return __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_u8)(p));
}

// 4 bytes per lane straight into LDS at lds_base + 4 * lane (buffer_load_dword ... lds); untracked like dma16.
__device__ __forceinline__ void dma4(v4u desc, uint32_t lds_base, uint32_t voff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, 0 offen lds"
                 :
                 : "s"(lds_base), "v"(voff), "s"(desc)
                 : "memory", "m0");
}

// Orders one wave's LDS accesses across its lanes: a lane's staging writes become visible to the other lanes' reads
// that follow.  The wave's LDS accesses already complete in order, so this emits no wait; it is there for the compiler,
// which under per-lane semantics may otherwise reorder or tail-duplicate lane-divergent writes past other lanes' reads
// (the barrier is convergent: it cannot be moved into a divergent branch).
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// max(m, |lo half|, |hi half|) of a packed bf16 pair, as fp32 bit patterns (the row maximum of the fused quant).
__device__ __forceinline__ uint32_t max_abs_bf16x2(uint32_t m, uint32_t p) {
    const uint32_t lo = (p << 16) & 0x7fff0000u, hi = p & 0x7fff0000u;
    m = m > lo ? m : lo;
    return m > hi ? m : hi;
}

// The same for a packed fp16 pair: each half is widened to fp32 (exact) before its |.| bits are compared, so the row
// maximum is the fp32 value of the largest rounded fp16 output (NaN patterns exceed every finite one, as above).
__device__ __forceinline__ uint32_t max_abs_f16x2(uint32_t m, uint32_t p) {
    const uint32_t lo = f2u(fp16_to_f32(p & 0xffffu)) & 0x7fffffffu, hi = f2u(fp16_to_f32(p >> 16)) & 0x7fffffffu;
    m = m > lo ? m : lo;
    return m > hi ? m : hi;
}

// Running maxima of |x| over packed bf16 pairs, one per 16-bit half: with the sign bit cleared, bf16 magnitudes order
// as their bit patterns (NaN patterns above inf), so a pair costs one mask and one packed u16 max.  pk_max_f32 folds
// the two halves into the fp32 bit pattern of the larger, the value max_abs_bf16x2 accumulates over the same pairs.
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ u16x2 max_abs_pk(u16x2 m, uint32_t p) {
    return __builtin_elementwise_max(m, __builtin_bit_cast(u16x2, p & 0x7fff7fffu));
}
__device__ __forceinline__ uint32_t pk_max_f32(u16x2 m) {
    const uint32_t a = m[0], b = m[1];
    return (a > b ? a : b) << 16;
}

// The accumulators, readable: an instruction that reads (or copies) one needs 20 wait states behind the MFMA that wrote it
// (v_mfma 32x32x64 on 8-bit operands, 16 passes).  With a scheduling barrier behind the MFMA the compiler has placed copies
// 19 behind it, and they came out without its sum.  So the last block, whose MFMA is the last, goes through an instruction
// of 24 wait states, and every block through a statement behind that: no read or copy can come before them.  AGPR: the
// kernel keeps its accumulators in the accumulation registers, as the compiler does up to four waves per workgroup (one per
// SIMD); in the wrong file they would be copied.  It stands right behind the last k-step: further down, beside the reads of
// the scales, it changed the epilogue's schedule (16 740 x 9216 x 3072 with its producer 0.4 % longer; here 0.1 %).
template <bool AGPR, int NI, int NJ>
__device__ __forceinline__ void accumulators_ready(v16f (&acc)[NI][NJ]) {
    if constexpr (AGPR) asm volatile("s_nop 15\n\ts_nop 7" : "+a"(acc[NI - 1][NJ - 1])::"memory");
    else asm volatile("s_nop 15\n\ts_nop 7" : "+v"(acc[NI - 1][NJ - 1])::"memory");
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            if constexpr (AGPR) asm volatile("" : "+a"(acc[i][j]));
            else asm volatile("" : "+v"(acc[i][j]));
        }
}

// A +0 the compiler cannot see through, made once per epilogue: x + z turns -0 into +0 (round to nearest) and leaves
// every other value (NaN included) unchanged, and the add is not folded away.
__device__ __forceinline__ float opaque_zero() {
    float z = 0.0f;
    asm volatile("" : "+v"(z));
    return z;
}

constexpr int SILU_LDS_BYTES = H3_SILU_ROT_LEN * 2;          // the compact SiLU table (kernel 3)
static_assert(SILU_LDS_BYTES % 256 == 0, "the table loads in 256-byte pieces");

// gemm_tile.hip: the forms of smaller tiles, one per workgroup, in ascending order of their area.
enum TileForm { TILE_32x64, TILE_64x64, TILE_96x64, TILE_128x64, TILE_128x128, TILE_192x128, TILE_256x128, TILE_FORMS };

// The first form whose tiles over M tokens x w_rows weight rows number at most `limit` (TILE_FORMS: none).  swiglu: the
// tiles of kernel 3 (w_rows = 2F), which has some of the forms only.
int tile_form_for(int64_t M, int64_t w_rows, bool swiglu, int64_t limit);
// The whole problem in tiles of one form.
int launch_tiles(GemmParams p, int form, int out_dt, bool swiglu, hipStream_t st);
// The tail of a launch over the first `first` 256 x 256 tiles of the first `panels` (p.tiles_m) row panels of 256 tokens:
// the `rest` tiles that it leaves of them and the token rows past them, in tiles of one form (tail_pieces of them);
// tail_form_for: the smallest form that keeps them within `limit` (TILE_FORMS: none).
int64_t tail_pieces(int form, int64_t M, int64_t w_rows, int panels, int64_t rest);
int tail_form_for(int64_t M, int64_t w_rows, bool swiglu, int panels, int64_t rest, int64_t limit);
int launch_tile_tail(GemmParams p, int form, int first, int rest, int out_dt, bool swiglu, hipStream_t st);

}  // namespace h3g
