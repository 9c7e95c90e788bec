// Products of a block-sparse weight with many dense rows (a sparse linear layer), for gfx950, fp16 / bf16.
//
// The group walk of matmul.hip gives a wave 64 dense rows and a chunk of one group's blocks: it fetches 4 KB of dense
// operand for every 2 KB block, from rows that lie a whole matrix row apart, and nothing it fetched serves another
// group.  With a few attention heads of 64 columns that is what there is to do; a linear layer has thousands of
// dense rows and dozens of groups that read the same columns of them.  Here a workgroup owns 64 to 160 dense rows and eight
// neighbouring groups, a wave each, walks ALL of the contraction in steps of 128 and keeps the dense panels of the present and
// the next steps in LDS; a wave multiplies them by the blocks its group has there.
#include "bsa_device.hpp"
#include "lds_tiles.hpp"
#include "bsa_internal.hpp"
#include "group_walk.hpp"
#include "attention_tiles.hpp"
#include "panel_ring.hpp"
#include "../../include/bsa.h"

namespace bsa {

// Consecutive work items on one XCD (its workgroups are every eighth): neighbours share operands in its L2.
__device__ __forceinline__ int xcd_contiguous(int total)
{
    const int per_xcd = (total + 7) >> 3, w = (int)blockIdx.x;
    const int item = (w & 7) * per_xcd + (w >> 3);
    return (w >> 3) < per_xcd && item < total ? item : -1;
}

constexpr int PANEL_WAVES = 8;                  // groups of a workgroup, one wave each
constexpr int PANEL_KB = 4;                     // k-blocks of 32 per step
constexpr int PANEL_RING = 4;                   // blocks of a wave in flight
constexpr int PANEL_HELPER = PANEL_WAVES + PANEL_FETCHERS;                 // the last wave, if there is one: half of the longest group
constexpr int PANEL_THREADS = 64 * (PANEL_HELPER + 1);
constexpr int PANEL_FLAGS = 64;                 // bytes in front of the lists: panels that are there, panels that are read
constexpr int PANEL_LDS = 160 * 1024;
constexpr int PANEL_NONE = -1;
// Blocks that the set's longest chain must get shorter by, to pay for two barriers and the helper's sums through LDS.  us, a
// column of the weight full, without the helper -> with it: a quarter and a tenth of 64 x 64 blocks, 4224 rows 28.0 -> 25.1 and
// 25.8 -> 21.5, 5632 rows 39.7 -> 34.1 and 38.0 -> 30.2; 96 x 96, 8192 rows 80.7 -> 68.6; masks without one as they were (23.4 ->
// 23.5, 19.2 -> 19.2, 64.6 -> 64.5).  Two helpers, half of each of the two longest: two full columns of a set 38.7 -> 36.1 and 71.3 ->
// 62.6, everything else 1 % slower; two or five that go to the longest chains one by one: 1 us slower at one such column; half of the
// longest group to the wave of the shortest, with a second set of sums: its registers spill.
constexpr int PANEL_CUT_FROM = 8;
__host__ __device__ constexpr int panel_list_length(int kblocks) { return (kblocks + 2 * PANEL_RING + 3) / 4 * 4; }

// ---------------------------------------------------------------------------
// out[row][32 g + x] = sum over the blocks (k-block kb) of group g, sum over k of dense[row][32 kb + k] * block(x, k)
//
// dense [rows][KT] and out [rows][XT] of one batch entry, or of all of them as one matrix when the weight is shared.
//   S_KC  the stored block is [x][k] (row groups): operands straight from memory
//         otherwise [k][x] (column groups): through a wave-private LDS tile, read transposed
// Three waves request panels straight into LDS, wait for them and say so in a flag; a multiplying wave waits for the panel of
// its next block and says up to which panel it is done (panel_ring.hpp: when a buffer may be filled again).  So the waits for
// panels are the fetching waves' alone, the other waves' stay exact for the blocks, of which a wave has its next four on the way,
// and no wave waits for the fullest of the eight in every step, only for the slowest where it is a whole set of buffers ahead.
//
// What bounds it: the wave with the most blocks, about 1000 clocks a block (its panel's flag, LDS reads, ten products), then
// the panels (200 MB through the L2 -> LDS path: 18 us without the products).  us, panels through registers a step ahead and a
// barrier per step, 96 rows a workgroup -> fetching waves and a barrier per step, 160 rows -> flags -> operands of a block read
// together: 4224 rows x 2048 x 2048 at a quarter of its blocks, forward 31.3 -> 26.0 -> 24.6 -> 23.7, gradient of the dense operand
// 32.3 -> 24.5 -> 24.3 -> 22.8; 8192 x 3072 x 3072 at 0.3 107 -> 91 and 111 -> 84; every block stored, 4224 rows 56 -> 46 and 56 -> 41.
// A group that has a block in every k-block makes its wave the chain; half of it goes to another wave (PANEL_CUT_FROM).  Launches of
// two generations of workgroups in which that does not help are slower than two workgroups of eight waves a compute unit were: two such
// columns among eight, 5632 rows 31.7 -> 38.6 (input gradient 32.5 -> 34.3); half and all of 48 x 80 blocks stored, 4800 rows 35.7 ->
// 37.6 and 59.3 -> 60.4 (44 -> 30 and 69 -> 46).
// ---------------------------------------------------------------------------
template <int RT, bool S_KC, bool BF>
__global__ __launch_bounds__(PANEL_THREADS, 3) void weight_panel_kernel(
    const half_t *__restrict__ sp, const half_t *__restrict__ dn, half_t *__restrict__ out,
    const BlockDesc *__restrict__ blocks, const int *__restrict__ offsets,
    int groups, int nnz, int rows, int KT, int XT, int sp_shared, int row_tiles, int group_sets)
{
    extern __shared__ __align__(16) unsigned char lds_raw[];
    constexpr int ROWS = 32 * RT, STAGES = panel_stages(RT), PANEL_BYTES = ROWS * 256;
    const int item = xcd_contiguous(row_tiles * group_sets);
    if (item < 0) return;                                                  // whole workgroup leaves together
    const int tile = item / group_sets, set = item - tile * group_sets;
    const int batch = (int)blockIdx.y, w = wave_id(), l = lane_id();
    const int y0 = tile * ROWS, walkers = ((int)blockDim.x >> 6) - PANEL_FETCHERS;
    const int kblocks = KT / BS, steps = (kblocks + PANEL_KB - 1) / PANEL_KB;
    // Workgroups start at different steps: rows a multiple of 4 KB apart have their 256 bytes of a step in ONE of the 16
    // channels of an L2, and workgroups that walk the contraction in unison would all ask that channel.
    const int start = item % steps;

    half_t *privs = reinterpret_cast<half_t *>(lds_raw + STAGES * PANEL_BYTES);
    int *flags = reinterpret_cast<int *>(lds_raw + STAGES * PANEL_BYTES + (S_KC ? 0 : walkers * BS2 * 2));
    int *ready = flags + PANEL_READY, *done = flags + PANEL_DONE;
    static_assert(STAGES <= PANEL_DONE - PANEL_READY && 4 * (PANEL_DONE + PANEL_WAVES + 1) <= PANEL_FLAGS, "flags");
    auto load_flag = [](const int *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); };
    auto store_flag = [](int *p, int v) {
        wave_lds_fence();
        __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    };
    if (threadIdx.x < PANEL_FLAGS / 4) flags[threadIdx.x] = 0;
    lds_barrier();

    // Pairs of the set's groups, a lane each
    int begins = 0, lengths = 0;
    auto look_at_the_set = [&]() {
        const int q = set * PANEL_WAVES + l % PANEL_WAVES;
        begins = offsets[q < groups ? q : groups];
        lengths = offsets[q + 1 < groups ? q + 1 : groups];
    };
    // Where the longest group is so by PANEL_CUT_FROM blocks and more, the helper takes half of its pairs, every second one: a
    // group with a block in every k-block (a dense column of the weight) would keep a workgroup waiting for its one wave.
    int longest = 0, half = 0;
    auto pairs = [&](int from, int to) { return to <= from ? 0 : to - from < kblocks ? to - from : kblocks; };
    auto find_the_longest = [&]() {
        lengths = pairs(begins, lengths);
        if (walkers == PANEL_WAVES || __ballot(lengths >= 2 * PANEL_CUT_FROM) == 0ull) return;
        int most = 0, second = 0;
#pragma unroll
        for (int j = 0; j < PANEL_WAVES; ++j) {
            const int n = __builtin_amdgcn_readlane(lengths, j);
            second = n > most ? most : n > second ? n : second;
            longest = n > most ? j : longest;
            most = n > most ? n : most;
        }
        half = most / 2;
        if (most - (second > most - half ? second : most - half) < PANEL_CUT_FROM) half = 0;
    };

    if (w >= PANEL_WAVES && w < PANEL_HELPER) {
        // Request r covers rows 4 r .. + 3, 16 pieces each; piece p of row y goes to slot p ^ (y & 15): 16 lanes that read one
        // piece of 16 rows meet no bank twice.  Lane l fills slot l % 16 of row 4 r + l / 16.  Requests behind the last row
        // repeat the last four (the rows of a launch are whole tiles of 32), pieces behind the last k-block the first: never
        // multiplied into a stored result.
        const int f = w - PANEL_WAVES;
        const unsigned char *dnb = reinterpret_cast<const unsigned char *>(dn + (size_t)batch * rows * KT + (size_t)y0 * KT);
        const int last = (rows - y0 < ROWS ? rows - y0 : ROWS) / 4 - 1;    // request of the last four rows
        const unsigned lds0 = __builtin_amdgcn_readfirstlane(lds_address(lds_raw));
        unsigned off[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) off[c] = 2u * (unsigned)((l >> 4) * KT) + 16u * (unsigned)((l & 15) ^ (4 * c + (l >> 4)));
        const int whole = KT / (BS * PANEL_KB), pieces = 16 - (steps * 16 - KT / 8);      // the last step may have fewer pieces
        for (int s = f; s < steps; s += PANEL_FETCHERS) {
            // the panel before in this buffer, s - STAGES, is there and has been read by all
            const int *watched = flags + panel_refill_flag(l, walkers, s, STAGES);
            while (__ballot(load_flag(watched) < panel_refill_from(s, STAGES)) != 0ull) __builtin_amdgcn_s_sleep(1);
            const unsigned to = lds0 + (unsigned)(s % STAGES) * PANEL_BYTES;
            int at = s + start;
            at = at < steps ? at : at - steps;
            unsigned o[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const int piece = (l & 15) ^ (4 * c + (l >> 4));
                o[c] = at >= whole && piece >= pieces ? off[c] - 16u * piece : off[c];
            }
            const unsigned char *from = dnb + 256 * at;
#pragma unroll 1
            for (int r = 0; r < 8 * RT; r += 4) {
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    dma16(from, o[c], to + 1024u * (r + c));
                    from += r + c < last ? (size_t)8 * KT : 0;
                }
            }
            tile_wait<0>();
            if (l == 0) store_flag(ready + s % STAGES, s + 1);
        }
        look_at_the_set();
        find_the_longest();
        if (half > 0) {                          // the barriers at the end of the others
            lds_barrier();
            lds_barrier();
        }
        return;
    }

    // The group's pairs, in the order in which the steps come: block | k-block << 20, then PANEL_NONE
    const bool helper = w == PANEL_HELPER;
    const int slot = helper ? PANEL_WAVES : w;
    half_t *priv = privs + slot * BS2;
    int *list = flags + PANEL_FLAGS / 4 + slot * panel_list_length(kblocks);
    auto kblock = [&](const BlockDesc &d) { return S_KC ? d.col() : d.row(); };
    look_at_the_set();
    int g = set * PANEL_WAVES + w, begin = 0, length = 0;
    BlockDesc first = {0, -1};                                             // pair l of the group
    if (!helper) {
        begin = offsets[g < groups ? g : groups];
        length = pairs(begin, offsets[g + 1 < groups ? g + 1 : groups]);
        if (l < length) first = blocks[begin + l];
    }
    find_the_longest();
    if (helper && half > 0) {
        g = set * PANEL_WAVES + longest;
        begin = __builtin_amdgcn_readlane(begins, longest);
        length = __builtin_amdgcn_readlane(lengths, longest);
        if (l < length) first = blocks[begin + l];
    }
    const int apart = half > 0 && g == set * PANEL_WAVES + longest ? 1 : 0;                   // the wave's pairs: all, or the even or the odd ones
    const int n_own = !apart ? length : helper ? half : length - half;
    int n = n_own;
    {
        auto mine = [&](int p) { return p < length && ((p & apart) != 0) == (helper && apart); };
        int before = 0, previous = -1;                                     // pairs of steps that come around again; the lane before this one's
        bool ascending = true;
        for (int p = 0; p < length; p += WAVE) {
            const int kb = p + l >= length ? kblocks : kblock(p == 0 ? first : blocks[begin + p + l]), left = __shfl_up(kb, 1);
            ascending &= kb >= (l == 0 ? previous : left);
            before += __popcll(__ballot(mine(p + l) && kb < start * PANEL_KB));
            previous = __builtin_amdgcn_readlane(kb, WAVE - 1);
        }
        if (__ballot(!ascending) == 0ull) {
            for (int p = l; p < length; p += WAVE) {
                const BlockDesc d = p < WAVE ? first : blocks[begin + p];
                const bool inside = kblock(d) < kblocks;                   // else the walk below would wait for a step that never comes
                const int q = p >> apart;
                if (mine(p)) list[q >= before ? q - before : q + n_own - before] = inside ? (d.idx & 0xFFFFF) | kblock(d) << 20 : PANEL_NONE;
            }
        } else {                                                           // a table in another order: collected step by step
            n = 0;
            for (int s = 0; s < steps; ++s) {
                const int at = s + start < steps ? s + start : s + start - steps;
                for (int p = 0; p < length; p += WAVE) {
                    const BlockDesc d = p + l < length ? blocks[begin + p + l] : BlockDesc{0, -1};
                    const bool here = mine(p + l) && kblock(d) < kblocks && kblock(d) / PANEL_KB == at;
                    const unsigned long long all = __ballot(here);
                    if (here) list[n + __popcll(all & ((1ull << l) - 1ull))] = (d.idx & 0xFFFFF) | kblock(d) << 20;
                    n += __popcll(all);
                }
            }
        }
    }
    n = __builtin_amdgcn_readfirstlane(n);
    if (l < 2 * PANEL_RING) list[n + l] = PANEL_NONE;
    wave_lds_fence();

    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<half_t *>(sp + (sp_shared ? 0 : (size_t)batch * nnz * BS2)), 0, nnz * BS2 * 2, 0x00020000);
    // S_KC: lane (i, h) takes row perm16(i) of the block, k = 16 s + 8 h; otherwise the linear pieces l and l + 64
    const int off0 = S_KC ? 64 * perm16(l & 31) + 16 * (l >> 5) : 16 * l, off1 = off0 + (S_KC ? 32 : 1024);
    uint4 blk[PANEL_RING][2];
    int now[PANEL_RING], next[PANEL_RING];
    auto lookup = [&](int i, int (&e)[PANEL_RING]) {
        const int4 x = *reinterpret_cast<const int4 *>(list + i);          // i is a multiple of 4
        e[0] = __builtin_amdgcn_readfirstlane(x.x);
        e[1] = __builtin_amdgcn_readfirstlane(x.y);
        e[2] = __builtin_amdgcn_readfirstlane(x.z);
        e[3] = __builtin_amdgcn_readfirstlane(x.w);
    };
    // the request of an absent block carries an offset beyond the descriptor's range, which the memory pipeline answers with
    // zeros without a fetch: no load sits under a condition
    auto request_block = [&](int e, uint4 (&b)[2]) {
        const unsigned base = e >= 0 ? (unsigned)(e & 0xFFFFF) * (BS2 * 2) : 0x80000000u;
        b[0] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, base + off0, 0, 0));
        b[1] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, base + off1, 0, 0));
    };
    lookup(0, now);
#pragma unroll
    for (int j = 0; j < PANEL_RING; ++j) {
        request_block(now[j], blk[j]);
        __builtin_amdgcn_sched_barrier(0);
    }

    f16v acc[RT];
#pragma unroll
    for (int t = 0; t < RT; ++t) acc[t] = f16v{0};
    const int i = l & 31, h = l >> 5;
    int step = -1;                                                         // whose panel is there
    const unsigned char *panel = lds_raw + 256 * i;                        // row i of it
    auto walk_to = [&](int s) {
        if (s == step) return;
        if (l == 0) store_flag(done + slot, s);                             // the reads before it are in front of it in LDS order
        const int buffer = s % STAGES;
        while (__builtin_amdgcn_readfirstlane(load_flag(ready + buffer)) < s + 1) __builtin_amdgcn_s_sleep(1);
        wave_lds_fence();
        panel = lds_raw + buffer * PANEL_BYTES + 256 * i;
        step = s;
    };
    for (int p = 0; p < n; p += PANEL_RING) {
        lookup(p + PANEL_RING, next);
#pragma unroll
        for (int j = 0; j < PANEL_RING; ++j) {
            if (now[j] >= 0) {
                const int kb = now[j] >> 20;
                int s = kb / PANEL_KB - start;
                // all operands first: two at a time, as the compiler has it, the LDS shows through five times a block
                h8 sop[2], dop[2][RT];
                if (S_KC) {
                    sop[0] = as_h8(blk[j][0]);
                    sop[1] = as_h8(blk[j][1]);
                } else {
                    wave_lds_fence();
                    lds_put_ks(priv, blk[j]);
                    wave_lds_fence();
                    sop[0] = lds_get_ks<true>(priv, 0);
                    sop[1] = lds_get_ks<true>(priv, 1);
                }
                walk_to(s < 0 ? s + steps : s);
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const unsigned char *at = panel + 16 * ((4 * (kb % PANEL_KB) + 2 * u + h) ^ (i & 15));
#pragma unroll
                    for (int t = 0; t < RT; ++t) dop[u][t] = *reinterpret_cast<const h8 *>(at + 8192 * t);
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int u = 0; u < 2; ++u)
#pragma unroll
                    for (int t = 0; t < RT; ++t) acc[t] = mfma_16<BF>(sop[u], dop[u][t], acc[t]);
            }
            __builtin_amdgcn_sched_barrier(0);
            request_block(next[j], blk[j]);
            __builtin_amdgcn_sched_barrier(0);
            now[j] = next[j];
        }
    }
    if (l == 0) store_flag(done + slot, steps);
    if (half > 0) {                              // the helper's sums go back through LDS, where all panels have been read
        f4v *parts = reinterpret_cast<f4v *>(lds_raw) + l;
        lds_barrier();
        if (helper) {
#pragma unroll
            for (int t = 0; t < RT; ++t)
#pragma unroll
                for (int v = 0; v < 4; ++v) parts[WAVE * (4 * t + v)] = f4v{acc[t][4 * v], acc[t][4 * v + 1], acc[t][4 * v + 2], acc[t][4 * v + 3]};
        }
        lds_barrier();
        if (apart) {
#pragma unroll
            for (int t = 0; t < RT; ++t)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[t][v] += parts[WAVE * (4 * t + v / 4)][v % 4];
        }
    }

    if (!helper && g < groups) {
        half_t *ob = out + (size_t)batch * rows * XT + BS * g + 16 * h;
#pragma unroll
        for (int t = 0; t < RT; ++t) {
            const int y = y0 + 32 * t + i;
            uint4 lo, hi;
            pack16<BF>(acc[t], lo, hi);
            if (y < rows) {
                stg16(ob + (size_t)y * XT, lo);
                stg16(ob + (size_t)y * XT + 8, hi);
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Gradient of the weight: w[block (r, c)] = sum over tokens t of a[t][32 r + .] b[t][32 c + .]
//
// A workgroup owns 8 x 8 cells of the mask and a share of the tokens; per step of 32 tokens it fetches 256 columns
// of a and of b, a 64-column panel a wave, and the stored cells are dealt evenly to the waves.  Partial sums of the shares
// leave as fp32 and are added up in share order by weight_sum_kernel.
// Bound by what the panels take from L2, 32 KB a step and workgroup (8.7 TB/s at 64 x 64 blocks).  They go straight to LDS:
// through registers, three steps in flight took 48 of them (8 spilled), and an LDS write each.
// A quarter of 64 x 64 blocks stored, 4224 tokens, with the sum: 38.5 -> 35.1 us; 96 x 96 at 0.3, 8192 tokens: 145 -> 128;
// all of 64 x 64 stored: 74.6 -> 66.2.
// ---------------------------------------------------------------------------
constexpr int WG_EDGE = 8;                       // cells along a side
constexpr int WG_PANEL = 4096;                   // 32 tokens of 64 columns
constexpr int WG_SIDE = WG_EDGE / 2 * WG_PANEL;
constexpr int WG_STAGE = 2 * WG_SIDE;
constexpr int WG_STAGES = 4;

template <bool BF>
__global__ __launch_bounds__(512, 2) void weight_grad_kernel(
    const half_t *__restrict__ a, const half_t *__restrict__ b, float *__restrict__ parts,
    const BlockDesc *__restrict__ blocks, const int *__restrict__ offsets,
    int R, int C, int nnz, int steps_total, int shares, int sets_r, int sets_c)
{
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const int item = xcd_contiguous(shares * sets_r * sets_c);
    if (item < 0) return;
    const int share = item / (sets_r * sets_c), cell = item - share * (sets_r * sets_c);
    const int r0 = WG_EDGE * (cell / sets_c), c0 = WG_EDGE * (cell % sets_c);
    const int w = wave_id(), l = lane_id(), tid = (int)threadIdx.x;
    const int first = (int)((long long)steps_total * share / shares), last = (int)((long long)steps_total * (share + 1) / shares);
    const int M = BS * R, N = BS * C;

    // the stored cells, dealt evenly to the waves in row-major order: cells w, w + 8, ..
    int *table = reinterpret_cast<int *>(lds_raw + WG_STAGES * WG_STAGE);
    if (tid < WG_EDGE * WG_EDGE) table[tid] = -1;
    lds_barrier();
    if (r0 + w < R) {
        const int end = offsets[r0 + w + 1];
        for (int p = offsets[r0 + w] + l; p < end; p += WAVE) {
            const BlockDesc d = blocks[p];
            const int c = d.col() - c0;
            if (c >= 0 && c < WG_EDGE) table[w * WG_EDGE + c] = d.idx;
        }
    }
    lds_barrier();
    const int mine_idx = table[l];
    unsigned long long stored = __ballot(mine_idx >= 0);
    const int count = (__popcll(stored) - w + WG_EDGE - 1) / WG_EDGE;      // of this wave
    int idx[WG_EDGE], at_a[WG_EDGE], at_b[WG_EDGE];      // at_: exclusive-ored into the address of an operand's first column
    for (int j = 0; j < w && stored; ++j) stored &= stored - 1;
#pragma unroll
    for (int j = 0; j < WG_EDGE; ++j) {
        const int cell_of = stored ? __builtin_ctzll(stored) : 0;
        idx[j] = __builtin_amdgcn_readlane(mine_idx, cell_of);
        at_a[j] = (cell_of >> 4) * WG_PANEL + (cell_of >> 3 & 1) * 64;
        at_b[j] = WG_SIDE + (cell_of >> 1 & 3) * WG_PANEL + (cell_of & 1) * 64;
        for (int t = 0; t < WG_EDGE; ++t) stored &= stored ? stored - 1 : 0;
    }

    // Panel w % 4 of a (waves 0-3) or b; columns behind the last repeat the first (never stored).  A wave's offsets inside 32
    // tokens fit 32 bits.
    const unsigned lds0 = __builtin_amdgcn_readfirstlane(lds_address(lds_raw));
    const int width = w < WG_EDGE / 2 ? M : N, column0 = (w < WG_EDGE / 2 ? 32 * r0 : 32 * c0) + 64 * (w % (WG_EDGE / 2));
    const unsigned char *operand = reinterpret_cast<const unsigned char *>(w < WG_EDGE / 2 ? a : b);
    unsigned off[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        const int column = column0 + 8 * panel_src_piece(l, c);
        off[c] = 2u * ((unsigned)(l >> 3) * (unsigned)width + (unsigned)(column < width ? column : 0));
    }
    auto request = [&](int step, int stage) {
        step = step < last ? step : last - 1;
        const unsigned char *rows = operand + (size_t)step * (64 * (size_t)width);
        const unsigned to = lds0 + stage * WG_STAGE + w * WG_PANEL;
#pragma unroll
        for (int c = 0; c < 4; ++c) dma16(rows + 16 * (size_t)width * c, off[c & 1], to + 1024 * c);
    };
    f16v acc[WG_EDGE];
#pragma unroll
    for (int c = 0; c < WG_EDGE; ++c) acc[c] = f16v{0};

    const unsigned tr_lo = (unsigned)get_panel_tr_addr(l, 0, 0, 0), tr_hi = (unsigned)get_panel_tr_addr(l, 0, 1, 0);
    auto multiply = [&](int stage) {
        const unsigned base = lds0 + stage * WG_STAGE;
        auto half_of = [&](int at, h8 (&x)[2]) {
            asm volatile("" : "+s"(at));                // added where it is used: hoisted, the sums take 64 registers
            typedef tr4 __attribute__((address_space(3))) *lds_tr4;
            const unsigned lo = (tr_lo ^ (unsigned)at) + base, hi = (tr_hi ^ (unsigned)at) + base;
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const tr4 p = __builtin_amdgcn_ds_read_tr16_b64_v4f16((lds_tr4)(uintptr_t)(lo + 2048u * s));
                const tr4 q = __builtin_amdgcn_ds_read_tr16_b64_v4f16((lds_tr4)(uintptr_t)(hi + 2048u * s));
                x[s] = __builtin_shufflevector(__builtin_bit_cast(h4, p), __builtin_bit_cast(h4, q), 0, 1, 2, 3, 4, 5, 6, 7);
            }
        };
#pragma unroll
        for (int j = 0; j < WG_EDGE; j += 2) {
            if (j < count) {                       // a pair at a time; the second repeats a cell when there is none
                h8 xa[2], xb[2], ya[2], yb[2];
                half_of(at_a[j], xa);
                half_of(at_b[j], xb);
                half_of(at_a[j + 1], ya);
                half_of(at_b[j + 1], yb);
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    acc[j] = mfma_16<BF>(xb[s], xa[s], acc[j]);
                    acc[j + 1] = mfma_16<BF>(yb[s], ya[s], acc[j + 1]);
                }
            }
        }
    };
    if (first < last) {
        // Three steps in flight (the operands of a long batch come from HBM).  A wave waits for its own panel of the step, the
        // barrier for everybody's; behind it nobody reads the step before, whose buffer the next request takes.
#pragma unroll
        for (int d = 0; d < WG_STAGES - 1; ++d) request(first + d, d);
        int stage = 0;
        for (int s = first; s < last; ++s) {
            tile_wait<4 * (WG_STAGES - 2)>();
            lds_barrier();
            request(s + WG_STAGES - 1, (stage + WG_STAGES - 1) % WG_STAGES);
            multiply(stage);
            stage = (stage + 1) % WG_STAGES;
        }
        tile_wait<0>();                            // requests past the last step write to LDS that is still this workgroup's
    }
    float *dst = parts + (size_t)share * nnz * BS2 + (l & 31) * BS + 4 * (l >> 5);
#pragma unroll
    for (int c = 0; c < WG_EDGE; ++c) {
        if (c < count) {
            float *o = dst + (size_t)idx[c] * BS2;
#pragma unroll
            for (int t = 0; t < 4; ++t)
                *reinterpret_cast<float4 *>(o + 8 * t) =
                    make_float4(acc[c][4 * t], acc[c][4 * t + 1], acc[c][4 * t + 2], acc[c][4 * t + 3]);
        }
    }
}

// out[e] = sum over the shares of parts[share][e]: 8 elements a thread
template <bool BF>
__global__ __launch_bounds__(256) void weight_sum_kernel(const float *__restrict__ parts, half_t *__restrict__ out,
                                                         size_t elements, int shares)
{
    const size_t e = 8 * ((size_t)blockIdx.x * 256 + threadIdx.x);
    if (e >= elements) return;
    float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int p = 0; p < shares; ++p) {
        const float4 *src = reinterpret_cast<const float4 *>(parts + (size_t)p * elements + e);
        const float4 x = src[0], y = src[1];
        s[0] += x.x; s[1] += x.y; s[2] += x.z; s[3] += x.w;
        s[4] += y.x; s[5] += y.y; s[6] += y.z; s[7] += y.w;
    }
    h8 o;
#pragma unroll
    for (int v = 0; v < 8; ++v) o[v] = narrow_16<BF>(s[v]);
    stg16(out + e, __builtin_bit_cast(uint4, o));
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
template <int RT, bool S_KC, bool BF>
static hipError_t launch_panel(const WeightPanelArgs &p, hipStream_t st)
{
    constexpr int ROWS = 32 * RT;
    const int tiles = (p.rows + ROWS - 1) / ROWS, sets = (p.groups + PANEL_WAVES - 1) / PANEL_WAVES;
    auto lds_of = [&](int walkers) {
        return panel_stages(RT) * ROWS * 256 + PANEL_FLAGS + walkers * ((S_KC ? 0 : BS2 * 2) + (size_t)panel_list_length(p.KT / BS) * sizeof(int));
    };
    const int walkers = PANEL_WAVES + (lds_of(PANEL_WAVES + 1) <= PANEL_LDS ? 1 : 0);
    const size_t lds = lds_of(walkers);
    auto kernel = weight_panel_kernel<RT, S_KC, BF>;
    if (lds > 65536) {
        hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (err != hipSuccess) return err;
    }
    dim3 grid((unsigned)((tiles * sets + 7) / 8 * 8), (unsigned)p.batches);
    kernel<<<grid, 64 * (walkers + PANEL_FETCHERS), lds, st>>>(
        (const half_t *)p.sparse, (const half_t *)p.dense, (half_t *)p.out, (const BlockDesc *)p.blocks, p.offsets, p.groups, p.nnz,
        p.rows, p.KT, BS * p.groups, p.sparse_shared ? 1 : 0, tiles, sets);
    return hipGetLastError();
}

// Tiles of 32 rows a workgroup takes: a compute unit holds one workgroup, so the fewest generations of them, counted with
// a tile's worth of start and end.  Five leave no room for the lists of more than 700 k-blocks.
static int panel_row_tiles(const WeightPanelArgs &p)
{
    const long long sets = (p.groups + PANEL_WAVES - 1) / PANEL_WAVES;
    int best = 2;
    long long best_cost = 0;
    for (int rt = 2; rt <= (p.KT / BS <= 700 ? 5 : 4); ++rt) {
        const long long wgs = (p.rows + 32 * rt - 1) / (32 * rt) * sets * p.batches, cost = (wgs + 255) / 256 * (rt + 1);
        if (best_cost == 0 || cost < best_cost) {
            best = rt;
            best_cost = cost;
        }
    }
    return best;
}

template <bool S_KC, bool BF>
static hipError_t launch_panels(const WeightPanelArgs &p, hipStream_t st)
{
    switch (panel_row_tiles(p)) {
        case 2: return launch_panel<2, S_KC, BF>(p, st);
        case 3: return launch_panel<3, S_KC, BF>(p, st);
        case 4: return launch_panel<4, S_KC, BF>(p, st);
        default: return launch_panel<5, S_KC, BF>(p, st);
    }
}

hipError_t launch_weight_panels(int dtype, const WeightPanelArgs &p, hipStream_t st)
{
    if (dtype == BSA_BF16) return p.row_groups ? launch_panels<true, true>(p, st) : launch_panels<false, true>(p, st);
    return p.row_groups ? launch_panels<true, false>(p, st) : launch_panels<false, false>(p, st);
}

// Shares of at least eight steps: the fewest (at most eight) that leave at most a sixth of the machine idle in the last
// generation of workgroups (one per compute unit at a time: 128 KB of panels, 256 registers), else the best there is.
int weight_grad_shares(int mask_rows, int mask_cols, int tokens)
{
    const long long cells = (long long)((mask_rows + WG_EDGE - 1) / WG_EDGE) * ((mask_cols + WG_EDGE - 1) / WG_EDGE);
    const int steps = tokens / BS;
    int best = 1;
    double best_use = 0.;
    for (int s = 1; s <= (cells < 32 ? 256 / cells : 8) && (s == 1 || steps / s >= 8); ++s) {
        const long long wgs = cells * s;
        const double use = (double)wgs / (double)((wgs + 255) / 256 * 256);
        if (use > best_use + 0.01) {
            best = s;
            best_use = use;
        }
        if (use > 5. / 6.) break;
    }
    return best;
}

hipError_t launch_weight_grad(int dtype, const WeightGradArgs &p, hipStream_t st)
{
    const int sets_r = (p.mask_rows + WG_EDGE - 1) / WG_EDGE, sets_c = (p.mask_cols + WG_EDGE - 1) / WG_EDGE;
    const size_t lds = WG_STAGES * WG_STAGE + WG_EDGE * WG_EDGE * sizeof(int);
    auto kernel = dtype == BSA_BF16 ? weight_grad_kernel<true> : weight_grad_kernel<false>;
    hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (err != hipSuccess) return err;
    const unsigned grid = ((unsigned)p.shares * sets_r * sets_c + 7) / 8 * 8;
    kernel<<<grid, 64 * WG_EDGE, lds, st>>>((const half_t *)p.a, (const half_t *)p.b, p.parts, (const BlockDesc *)p.blocks,
                                            p.offsets, p.mask_rows, p.mask_cols, p.nnz, p.tokens / BS, p.shares, sets_r, sets_c);
    err = hipGetLastError();
    if (err != hipSuccess) return err;
    const size_t elements = (size_t)p.nnz * BS2;
    const unsigned wgs = (unsigned)((elements / 8 + 255) / 256);
    if (dtype == BSA_BF16) weight_sum_kernel<true><<<wgs, 256, 0, st>>>(p.parts, (half_t *)p.out, elements, p.shares);
    else weight_sum_kernel<false><<<wgs, 256, 0, st>>>(p.parts, (half_t *)p.out, elements, p.shares);
    return hipGetLastError();
}

}  // namespace bsa
