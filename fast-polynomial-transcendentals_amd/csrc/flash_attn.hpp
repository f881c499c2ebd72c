// flash_attn.hpp -- definitions shared by the fused attention forward
// (flash_attn.hip) and backward (flash_attn_bwd.hip): score modes, tile
// constants, operand strides and the MFMA wrapper.
#pragma once

#include <hip/hip_runtime.h>

#include "ops.hpp"
#include "score_programs.hpp"

namespace pt {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

enum AttnMode : int {
    kAttnSoftmaxNative = 0,
    kAttnSoftmaxExp2D2 = 1,
    kAttnSoftmaxExp2D3 = 2,
    kAttnSoftcapNative = 3,
    kAttnSoftcapD4 = 4,
    kAttnSigmoidNative = 5,
    kAttnSigmoidB3 = 6,
    kAttnSigmoidB3D2 = 7,
    kAttnSigmoidD3 = 8,  // 8..11: BF16 sigmoid D3..D6 on bf16(s + bias)
    kAttnSigmoidD6 = 11,
    kAttnSoftmaxExp2Pwl2 = 12,
    kAttnSoftmaxExp2Pwl2Safe = 13,     // B5 PWL2 "safe" hinge, FP32
    kAttnSoftmaxExp2Pwl2SafeF16 = 14,  // B5 PWL2 "safe" hinge, packed FP16 fraction
    // 15..21: the remaining FA4 exp2 backends (exp2_kind order 6..12)
    kAttnSoftmaxExp2Pwl1Safe = 15,
    kAttnSoftmaxExp2Pwl1SafeF16 = 16,
    kAttnSoftmaxExp2Pwl2SafeBF16 = 17,
    kAttnSoftmaxExp2D2NoClamp = 18,
    kAttnSoftmaxExp2D2SafeF16 = 19,
    kAttnSoftmaxExp2D2SafeBF16 = 20,
    kAttnSoftmaxExp2Pwl2F16 = 21,
    kAttnModes = 22,
};

constexpr bool attn_is_sigmoid(int mode) { return mode >= kAttnSigmoidNative && mode <= kAttnSigmoidD6; }
constexpr bool attn_is_plain_softmax(int mode) {
    return mode <= kAttnSoftmaxExp2D3 || mode >= kAttnSoftmaxExp2Pwl2;
}
constexpr bool attn_has_exp2_program(int mode) {
    return mode == kAttnSoftmaxExp2D2 || mode == kAttnSoftmaxExp2D3 || mode >= kAttnSoftmaxExp2Pwl2;
}

// The exp2 program of a softmax mode.
template <int MODE>
constexpr int attn_exp2_kind() {
    return MODE == kAttnSoftmaxExp2D2            ? kExp2D2
           : MODE == kAttnSoftmaxExp2D3          ? kExp2D3
           : MODE == kAttnSoftmaxExp2Pwl2        ? kExp2Pwl2
           : MODE == kAttnSoftmaxExp2Pwl2Safe    ? kExp2Pwl2Safe
           : MODE == kAttnSoftmaxExp2Pwl2SafeF16 ? kExp2Pwl2SafeF16
           : MODE >= kAttnSoftmaxExp2Pwl1Safe && MODE <= kAttnSoftmaxExp2Pwl2F16
               ? kExp2Pwl1Safe + (MODE - kAttnSoftmaxExp2Pwl1Safe)
               : kExp2Native;
}

// exp2 routing (FA4's exp2_emu_freq, any even route >= 4;
// src/sfu_repro/fa4.py:226-233).  Each lane holds 32 exponents of a 64-key
// tile; exponent slot i (kt * 16 + r of the forward's accumulators) takes the
// polynomial when bit i of the tile's routing mask is set, the rest
// v_exp_f32.  Up to 32 the pattern restarts at every tile, slot % route < 4;
// above 32 it runs on over the row's tiles, (32 tile + slot) % route < 4, so
// four of every `route` exponents of a row are routed either way.  Routes 4
// (every exponent), 6, 8, 10, 12, 16, 20, 24 and 32 are template arguments
// (the pattern folds into each register's code); kRouteRuntime takes any
// other route from the kernel arguments, with the host's mask for routes up
// to 32 and route_mask_running per tile above.
constexpr int kRouteRuntime = 2;
constexpr bool route_partial(int route) { return route > 4 || route == kRouteRuntime; }

// The mask of a route of 4..32, the same for every tile.
__host__ __device__ constexpr uint32_t route_mask_periodic(int route) {
    uint32_t m = 0;
    for (int i = 0; i < 32; ++i)
        if (i % route < 4) m |= 1u << i;
    return m;
}

// The mask of the tile-th tile of a row for a route above 32.  Slot i holds
// g = base + i with base = 32 tile mod route and base + i < 2 route, so
// g mod route < 4 for g in [0, 4) or [route, route + 4).  tile < 2^17 (the
// launchers bound S below 2^23), so 32 tile fits an int.
__host__ __device__ constexpr uint32_t route_mask_running(int route, int tile) {
    const int base = (32 * tile) % route;
    const uint32_t head = base < 4 ? (1u << (4 - base)) - 1u : 0u;
    const uint32_t next = route - base < 32 ? 0xFu << (route - base) : 0u;
    return head | next;
}

// Per-tile mask of a kRouteRuntime launch: periodic_mask is the host's
// route_mask_periodic(route) when route <= 32.
__device__ __forceinline__ uint32_t tile_route_mask(int route, uint32_t periodic_mask, int tile) {
    return route <= 32 ? periodic_mask : route_mask_running(route, tile);
}

// Host side: the periodic mask passed to the kernels (0 without routing).
constexpr uint32_t host_route_mask(int route) { return route >= 4 && route <= 32 ? route_mask_periodic(route) : 0u; }

constexpr int kAttnBlockQ = 128;  // 4 waves x 32 queries
constexpr int kAttnBlockK = 64;   // keys per staged tile
constexpr float kLog2e = 1.44269504088896340736f;
constexpr float kLn2 = 0.69314718055994530942f;

// Element strides (batch, head, sequence) of one [*, *, *, 128] operand; the
// head dimension is contiguous.
struct AttnStrides {
    int64_t b, h, s;
};

__device__ __forceinline__ f32x16_t mfma32(bf16x8_t a, bf16x8_t b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

typedef short v4i16_t __attribute__((ext_vector_type(4)));

// ds_read_b64_tr_b16 (gfx950): each lane names an 8-byte chunk (4 BF16) of
// LDS; within every group of 16 lanes, lane i receives element i % 4 of the
// chunks of lanes 4s + i / 4, s = 0..3.  With lane j of a group pointing at
// row r0 + j / 4, columns c0 + 4 (j % 4) of a row-major tile, lane i gets
// column c0 + i of rows r0 .. r0 + 3: a 4 x 16 block, transposed (layout
// measured on MI355X).
__device__ __forceinline__ v4i16_t lds_read_tr16(const uint16_t* p) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4i16_t*)(p));
}

// A launch constant held in a VGPR (opaque to the compiler, which would read
// it from an SGPR): FP32 adds, multiplies and FMAs whose operands are all
// VGPRs issue at twice the rate of ones with a scalar operand when two waves
// share a SIMD (2.5 against 4.5 cycles per wave, measured on MI355X).
__device__ __forceinline__ float vgpr(float x) {
    asm("" : "+v"(x));
    return x;
}

// x of lane l ^ 32 combined with this lane's (v_permlane32_swap_b32).
__device__ __forceinline__ float half_max(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(as_u32(x), as_u32(x), false, false);
    return __builtin_fmaxf(as_f32(r[0]), as_f32(r[1]));
}
__device__ __forceinline__ float half_sum(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(as_u32(x), as_u32(x), false, false);
    return as_f32(r[0]) + as_f32(r[1]);
}

// ---- staging straight into LDS ----------------------------------------------
//
// global_load_lds_dwordx4: each lane names 16 bytes of memory, the wave's 64
// chunks land in LDS back to back from a wave-uniform address.  No registers
// hold the data and no LDS write instructions issue (13 cycles of the LDS pipe
// per 16-byte write, measured).  The compiler does not know of the loads in
// flight: their issuer waits for them with wait_loads, and a barrier after that wait
// publishes them.
//
// Rows of HD BF16 values cannot be padded inside such a load (1 KiB, 4 or 8
// rows), so they are swizzled: the 16-byte chunk c of row r lies at chunk
// c ^ row_swizzle(r), and 32 bytes lie between groups of eight rows
// (lds_row, linear in multiples of eight rows).  LDS serves 256 bytes a cycle: 16 lanes of a row-fragment
// read (b128: one chunk of 16 consecutive rows) fall on 16 different 16-byte
// columns, and 32 lanes of a transposing read (64 bytes of four consecutive
// rows) on four different 64-byte columns.
template <int HD>
__device__ __forceinline__ constexpr int row_swizzle(int row) {
    return (HD == 128 ? (row & 3) << 2 : (row & 2) << 1) | ((row >> 2) & 1);
}
// Byte address of a row in its tile.
template <int HD>
__device__ __forceinline__ constexpr uint32_t lds_row(int row) { return (uint32_t)(row * HD * 2 + (row >> 3) * 32); }

// Moves lane 16 bytes of memory at base + offset (bytes) to LDS address lds +
// 16 * lane; lds and base wave-uniform.  The compiler does not look into the
// asm for wait states: an SGPR that a vector instruction wrote (the
// v_readfirstlane of base, or the v_readlane of a spilled one) may be read as
// an address five wait states later, M0 one after it was written.
// s_mov_b32 and s_nop 3 are five.  M0 is reserved: the compiler puts no value
// there but for an instruction that reads it, and these kernels have none
// outside the asm (a clobber of a reserved register means nothing to it).
__device__ __forceinline__ void load_to_lds(uint32_t lds, const void* base, uint32_t offset) {
    const uint64_t bits = (uint64_t)(uintptr_t)base;
    const uint64_t sbase = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(bits >> 32)) << 32) |
                           (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)bits);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(__builtin_amdgcn_readfirstlane((int)lds)), "v"(offset), "s"(sbase)
                 : "memory");
}

// The same for memory read once: it does not displace what the caches hold.
__device__ __forceinline__ void load_to_lds_once(uint32_t lds, const void* base, uint32_t offset) {
    const uint64_t bits = (uint64_t)(uintptr_t)base;
    const uint64_t sbase = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(bits >> 32)) << 32) |
                           (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)bits);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tglobal_load_lds_dwordx4 %1, %2 nt"
                 :
                 : "s"(__builtin_amdgcn_readfirstlane((int)lds)), "v"(offset), "s"(sbase)
                 : "memory");
}

// load_to_lds with an address of each lane's own, in VGPRs (no wait states but
// M0's).
__device__ __forceinline__ void load_to_lds_each(uint32_t lds, const void* lane_src) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
                 :
                 : "s"(__builtin_amdgcn_readfirstlane((int)lds)), "v"(lane_src)
                 : "memory");
}

// What rows past the end are loaded from.
static __device__ const uint32_t kZeroChunk[4] __attribute__((aligned(16))) = {0u, 0u, 0u, 0u};

// Stages rows of HD BF16 values, kLoadRows per load; wave and rows of a load as
// the kernel divides them, in whole multiples of kLoadRows.
template <int HD>
struct RowLoader {
    static constexpr int kChunks = HD / 8;               // 16-byte chunks per row
    static constexpr int kLoadRows = 64 / kChunks;       // rows that one load moves
    int lr, lc;                                          // this lane's row and chunk of a load
    int wide;                                            // a row stride beyond 32-bit lane offsets

    __device__ __forceinline__ RowLoader(int lane, int wide_) : lr(lane / kChunks), lc(lane % kChunks), wide(wide_) {}

    // Rows row0 .. row0 + kLoadRows - 1 of base to LDS address lds (their
    // lds_row in some tile, tile_row = row0's row there modulo 8).  Rows past
    // `last` are zeros: a copy of a real row that holds an infinity would meet
    // the zero probability of a masked one, and 0 * Inf is NaN.
    __device__ __forceinline__ void load(uint32_t lds, int tile_row, const uint16_t* base, int64_t stride, int row0,
                                         int last) const {
        const uint32_t col = (uint32_t)((lc ^ row_swizzle<HD>(tile_row + lr)) * 16);
        if (row0 + kLoadRows - 1 <= last && !wide) {  // wave-uniform
            load_to_lds(lds, base + row0 * stride, (uint32_t)lr * (uint32_t)(int)stride * 2 + col);
        } else {
            const unsigned char* src = reinterpret_cast<const unsigned char*>(base + (row0 + lr) * stride) + col;
            load_to_lds_each(lds, row0 + lr <= last ? src : reinterpret_cast<const unsigned char*>(kZeroChunk));
        }
    }
};

// Reads the operands of v_mfma_f32_32x32x16_bf16 (A[l%32][8(l/32)+e],
// B[8(l/32)+e][l%32]) from swizzled rows.  Lane l = (h, c32) = (l / 32, l % 32).
template <int HD>
struct TileReader {
    uint32_t row_base[HD / 32], tr_base[HD / 32];

    __device__ __forceinline__ explicit TileReader(int lane) {
        const int h = lane >> 5, c32 = lane & 31;
        // transposing reads: the lane's source chunk is row 4h + (l % 16) / 4,
        // columns 16 ((l / 16) % 2) + 4 (l % 4)
        const int tr = 4 * h + ((lane & 15) >> 2), tc = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
#pragma unroll
        for (int i = 0; i < HD / 32; ++i) {
            row_base[i] = lds_row<HD>(c32) + (uint32_t)((4 * i + h) ^ row_swizzle<HD>(c32)) * 16;
            tr_base[i] = lds_row<HD>(tr) + (uint32_t)((4 * i + tc) ^ row_swizzle<HD>(tr)) * 16 + (lane & 1) * 8;
        }
    }
    // Row c32 of the 32 rows at `rows`, columns 16 c + 8 h .. + 7 (bit 1 of the
    // chunk is the swizzle's to leave alone, so c and c + 1 share a base).
    __device__ __forceinline__ bf16x8_t row_frag(const unsigned char* rows, int c) const {
        return *reinterpret_cast<const bf16x8_t*>(rows + row_base[c >> 1] + (c & 1) * 32);
    }
    // Column 32 dt + c32 of the 16 rows at `rows` (a multiple of 16 rows in),
    // rows 4h + {0..3, 8..11}: the order in which an accumulator holds them.
    __device__ __forceinline__ bf16x8_t col_frag(const unsigned char* rows, int dt) const {
        const uint16_t* src = reinterpret_cast<const uint16_t*>(rows + tr_base[dt]);
        const u32x2_t lo = __builtin_bit_cast(u32x2_t, lds_read_tr16(src));
        const u32x2_t hi = __builtin_bit_cast(u32x2_t, lds_read_tr16(src + lds_row<HD>(8) / 2));
        return __builtin_bit_cast(bf16x8_t, (u32x4_t){lo.x, lo.y, hi.x, hi.y});
    }
};

// At most N of this wave's vector memory operations are still in flight.
template <int N>
__device__ __forceinline__ void wait_loads() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Block barrier without __syncthreads' wait for the loads in flight.  The
// wave's own LDS reads have returned: a load issued behind the barrier may
// overwrite what they read, and the products that take them need not have
// been scheduled ahead of it.
__device__ __forceinline__ void block_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

}  // namespace pt
