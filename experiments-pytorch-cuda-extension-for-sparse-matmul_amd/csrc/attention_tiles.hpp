// What the fused attention kernels share: 32-row operand tiles that go from global memory straight into LDS, the operands
// read from them, accumulators of 32 result rows, and the parts of a split group meeting in a workspace.
#pragma once

#include "bsa_device.hpp"
#include "lds_tiles.hpp"

namespace bsa {

__device__ __forceinline__ float at_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ float at_lane_xor32(float x)
{
    return __int_as_float(__builtin_amdgcn_ds_bpermute((lane_id() ^ 32) << 2, __float_as_int(x)));
}
__device__ __forceinline__ float at_finite_or_zero(float m) { return m == -__builtin_inff() ? 0.f : m; }

// ---- loads that go straight to LDS ------------------------------------------------------------------
// 16 bytes per lane from `base` + off to LDS bytes lds .. lds + 1023 (lane l: lds + 16 l).  Written as assembly so that
// the compiler, which would wait for every such load in flight before any LDS read, leaves the counting to tile_wait.
// m0 is named as clobbered: the compiler reserves it (and says so in a warning) but merges its own settings of it.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void dma16(const void *base, unsigned off, unsigned lds)
{
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(lds) : "memory", "m0");
}
// 4 bytes per lane from an address of its own
__device__ __forceinline__ void dma4_gather(const void *address, unsigned lds)
{
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" ::"v"(address), "s"(lds) : "memory", "m0");
}
#pragma clang diagnostic pop
// all but the youngest N requests of the wave have landed, and its LDS reads are done
template <int N>
__device__ __forceinline__ void tile_wait() { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory"); }
__device__ __forceinline__ unsigned lds_address(const void *p)
{
    typedef const __attribute__((address_space(3))) void *lds_ptr;
    return (unsigned)(uintptr_t)(lds_ptr)(uintptr_t)p;
}

__device__ __forceinline__ void lds_reads_done() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// Requests of one wave for whole 32-row tiles of an operand with rows of HD 16-bit values: HD / 64 panels of [32][64].
template <int HD>
struct TileRequests {
    static constexpr int N = HD / 16;        // requests per tile, a kilobyte each
    const unsigned char *base;
    unsigned off[2], lds;                    // per lane: even and odd chunks of 8 rows (they swizzle differently)
    __device__ __forceinline__ TileRequests(const half_t *operand, unsigned char *tile)
        : base((const unsigned char *)operand)
    {
        const int l = lane_id();
#pragma unroll
        for (int j = 0; j < 2; ++j) off[j] = (unsigned)((l >> 3) * (2 * HD) + 16 * panel_src_piece(l, j));
        lds = __builtin_amdgcn_readfirstlane(lds_address(tile));
    }
    // 65535 block rows of 128 values are 537 MB: the offset inside a batch entry fits 32 bits
    __device__ __forceinline__ void issue(int block) const
    {
        const unsigned at = (unsigned)block * (64u * HD);
        const unsigned o[2] = {off[0] + at, off[1] + at};
#pragma unroll
        for (int u = 0; u < HD / 64; ++u)
#pragma unroll
            for (int c = 0; c < 4; ++c) dma16(base + 128 * u + 16 * HD * c, o[c & 1], lds + 4096 * u + 1024 * c);
    }
};

// Products are 32 x 32 x 16, lane = (i = lane % 32, h = lane / 32): the first operand's index runs over the accumulator's
// rows (value v is row 8 (v / 4) + 4 h + v % 4), the second's over its column i.  The 16 x 16 x 32 shape has shorter
// chains, but two of its products take the vector ALU's issue slots of one of these: beside a chain of it another wave's
// fused multiply-adds ran at 8.4 clocks instead of 5.4 and its exponentials at 16.1 instead of 8.5.
//
// All operand addresses of a wave are eight registers and constants.  get_panel_addr(lane, s) is get_panel_addr(lane, 0)
// with 32 s exclusive-ored in; get_panel_tr_addr(lane, s, half, x0) is get_panel_tr_addr(lane, 0, 0, 0) with 16 half and
// 2 x0 exclusive-ored in, plus 2048 s + 1024 half.  Left to itself the compiler keeps an address per read: the column
// walk took 220 registers instead of 200.
struct TileReader {
    unsigned row[4], tr[2][2];               // LDS byte addresses inside the wave's first tile: [s % 4], [t % 2][half]
    __device__ __forceinline__ explicit TileReader(const unsigned char *first_tile)
    {
        const int l = lane_id();
        const unsigned base = __builtin_amdgcn_readfirstlane(lds_address(first_tile));
        const unsigned r = (unsigned)get_panel_addr(l, 0), t = (unsigned)get_panel_tr_addr(l, 0, 0, 0);
#pragma unroll
        for (int s = 0; s < 4; ++s) row[s] = base + (r ^ (32u * s));
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int half = 0; half < 2; ++half) tr[x][half] = base + ((t ^ (64u * x) ^ (16u * half)) + 1024u * half);
    }
    // index = rows, contraction = columns 16 s ..; `tile`: byte offset from the first tile
    __device__ __forceinline__ h8 rows(unsigned tile, int s) const
    {
        typedef const h8 __attribute__((address_space(3))) *lds_h8;
        return *(lds_h8)(uintptr_t)(row[s % 4] + (tile + 4096u * (s / 4)));
    }
    // index = columns 32 t .., contraction = rows 16 s ..
    __device__ __forceinline__ h8 columns(unsigned tile, int t, int s) const
    {
        typedef tr4 __attribute__((address_space(3))) *lds_tr4;
        const unsigned at = tile + 4096u * (t / 2) + 2048u * s;
        const tr4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4f16((lds_tr4)(uintptr_t)(tr[t % 2][0] + at));
        const tr4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4f16((lds_tr4)(uintptr_t)(tr[t % 2][1] + at));
        return __builtin_shufflevector(__builtin_bit_cast(h4, lo), __builtin_bit_cast(h4, hi), 0, 1, 2, 3, 4, 5, 6, 7);
    }
};
// row i, columns 16 s + 8 h .. + 7 of 32 rows of HD values (the operand that stays in registers)
template <int HD>
__device__ __forceinline__ void load_row_operands(const half_t *rows, h8 (&op)[HD / 16])
{
    const int l = lane_id();
#pragma unroll
    for (int s = 0; s < HD / 16; ++s) op[s] = as_h8(ldg16(rows + (size_t)(l & 31) * HD + 16 * s + 8 * (l >> 5)));
}

// accumulators of 32 result rows of HD columns, transposed: value v of acc[t] is column 32 t + 8 (v / 4) + 4 h + v % 4 of row i
template <int HD> using RowTile = f16v[HD / 32];
template <int HD>
__device__ __forceinline__ void clear(RowTile<HD> &acc)
{
#pragma unroll
    for (int t = 0; t < HD / 32; ++t) acc[t] = f16v{0};
}
template <int HD, class F>       // acc = f(accumulator value, its place in a parked tile)
__device__ __forceinline__ void each(RowTile<HD> &acc, F f)
{
    const int l = lane_id();
#pragma unroll
    for (int t = 0; t < HD / 32; ++t)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[t][v] = f(acc[t][v], (16 * t + v) * WAVE + l);
}

// The result rows go through 64 HD bytes of LDS, so that they leave as whole kilobytes instead of 8-byte pieces of 64
// different lines.
template <int HD, bool BF>
__device__ __forceinline__ void store_rows(const RowTile<HD> &acc, float mul, unsigned char *scratch, half_t *dst)
{
    const int l = lane_id(), row = l & 31, h = l >> 5;
    wave_lds_fence();
#pragma unroll
    for (int t = 0; t < HD / 32; ++t)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            h4 o;
#pragma unroll
            for (int j = 0; j < 4; ++j) o[j] = narrow_16<BF>(acc[t][4 * g + j] * mul);
            *reinterpret_cast<h4 *>(scratch + out_row_addr(HD, row, 4 * t + g, h)) = o;
        }
    wave_lds_fence();
#pragma unroll
    for (int j = 0; j < HD / 16; ++j) {
        const int slot = l + 64 * j, r = slot / (HD / 8), p = slot % (HD / 8);
        stg16(dst + 8 * slot, *reinterpret_cast<const uint4 *>(scratch + out_row_addr(HD, r, p, 0)));
    }
}

// the parts of a split group (split_publish in between): park, then the last to arrive sums in part order
template <int HD>
__device__ __forceinline__ void park_part(RowTile<HD> &acc, float *dst)
{
    each<HD>(acc, [&](float x, int at) {
        park_store(dst + at, x);
        return x;
    });
}
template <int HD>
__device__ __forceinline__ void sum_parts(RowTile<HD> &acc, const float *first, int stride, int parts)
{
    clear<HD>(acc);
    for (int p = 0; p < parts; ++p)
        each<HD>(acc, [&](float x, int at) { return x + park_load(first + (size_t)p * stride + at); });
}

// Workspace of a walk whose long groups are cut into parts: every part parks its accumulators and bumps the group's
// counter, the part that arrives last sums them in part order and resets the counter.
struct AtSplitWorkspace {
    int *counters;     // [batches][split_groups], zero between launches
    float *tiles;      // [batches][tile_slots][at_split_tile_floats(head dim)]
    int tile_slots, split_groups;
};
constexpr int at_split_tile_floats(int hd) { return 32 * hd + 2 * WAVE; }   // O^T, then every lane's max and sum
static inline size_t at_split_counter_bytes(int split_groups, int batches)
{
    return (((size_t)split_groups * batches * sizeof(int)) + 255) / 256 * 256;
}

}  // namespace bsa
