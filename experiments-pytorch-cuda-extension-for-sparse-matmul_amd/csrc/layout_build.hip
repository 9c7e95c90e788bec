// Device-side builder of the block-index tables and of the wavefront schedule.
//
// Tables: the contract is the output of SparseLayout._create_layout
// (sparse/layout.py:14-38) for a 0/1 mask, both orientations.  One workgroup
// of 16 wavefronts scans the mask twice (row-major, then column-major) with
// wave ballots + popcounts; the row-major ordinal of every cell is parked in a
// workspace so the column pass can attach it to its pairs.  Masks of more than
// 1024 cells are read once, into bits in LDS.
//
// Schedule: see bsa.h.  A serial first-fit pass over the groups (one lane)
// fixes each group's first slot and its partial-tile slots, then all lanes
// fill the wavefront slots.
#include "bsa_device.hpp"
#include "bsa_internal.hpp"
#include "../../include/bsa.h"

namespace bsa {

constexpr int LB_THREADS = 1024;
constexpr int LB_WAVES = LB_THREADS / WAVE;

// Exclusive position of this thread's flag among the flags of the workgroup,
// and the workgroup total.  `carry` is the running count of earlier tiles.
__device__ __forceinline__ int tile_scan(bool flag, int *wave_tot, int &total)
{
    unsigned long long bal = __ballot(flag);
    int lane = lane_id(), wave = (int)(threadIdx.x >> 6);
    int lane_prefix = __popcll(bal & ((1ull << lane) - 1ull));
    if (lane == 0) wave_tot[wave] = __popcll(bal);
    __syncthreads();
    int wave_prefix = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < LB_WAVES; ++w) {
        int t = wave_tot[w];
        wave_prefix += (w < wave) ? t : 0;
        tot += t;
    }
    __syncthreads();
    total = tot;
    return wave_prefix + lane_prefix;
}

// Number of set flags in front of this thread's `count`, and of the workgroup.
__device__ __forceinline__ int count_scan(int count, int *wave_tot, int &total)
{
    const int lane = lane_id(), wave = (int)(threadIdx.x >> 6);
    int sum = count;
#pragma unroll
    for (int d = 1; d < WAVE; d *= 2) {
        const int below = __shfl_up(sum, d);
        sum += lane >= d ? below : 0;
    }
    if (lane == WAVE - 1) wave_tot[wave] = sum;
    __syncthreads();
    int before = 0;
    total = 0;
#pragma unroll
    for (int w = 0; w < LB_WAVES; ++w) {
        before += w < wave ? wave_tot[w] : 0;
        total += wave_tot[w];
    }
    __syncthreads();
    return before + sum - count;
}

// Masks of more than 1024 cells whose bits fit LDS (a bit of mask and one of ordinals a cell: 512 x 1024 cells take 128 KB).
// Bound by a serial chain of barriers and dependent loads in one workgroup.  layout_build_kernel takes a scan and a round
// trip to memory for every 1024 cells and direction; here one scan covers 16384 cells, another 1024 columns, and the column
// order reads bits of LDS instead of bytes a mask row apart.  A tenth of the cells stored: 64 x 64 10.2 -> 6.4 us, 128 x 128
// 34.8 -> 11.4, 256 x 256 135 -> 35, 512 x 512 543 -> 124, 512 x 1024 1089 -> 242; up to 1024 cells the other kernel is one
// scan each way and the faster one (16 x 16: 2.7 us against 4.6).
constexpr int LB_RUN = 16;                               // neighbouring cells of a thread while the bits are collected
constexpr int LB_BIT_CELLS = 1 << 19;

__global__ __launch_bounds__(LB_THREADS) void layout_build_bits_kernel(
    const uint8_t *__restrict__ mask, int R, int C,
    int2 *__restrict__ row_blocks, int *__restrict__ row_off,
    int2 *__restrict__ col_blocks, int *__restrict__ col_off,
    int *__restrict__ nnz_out, int *__restrict__ ordinal_of)
{
    extern __shared__ unsigned bits[];                   // of the cells in row-major order, then the ordinal before every word
    __shared__ int wave_tot[LB_WAVES], counts[LB_THREADS];
    const int n = R * C, words = (n + 31) / 32, tid = (int)threadIdx.x;
    int *before = reinterpret_cast<int *>(bits + words);

    const bool aligned = (reinterpret_cast<uintptr_t>(mask) & 15) == 0;
    int carry = 0;
    for (int base = 0; base < n; base += LB_RUN * LB_THREADS) {
        const int t = base + LB_RUN * tid;
        unsigned flags = 0;
        if (aligned && t + LB_RUN <= n) {
            const uint4 v = ldg16(mask + t);
            const unsigned part[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int q = 0; q < LB_RUN; ++q) flags |= (part[q / 4] >> (8 * (q % 4)) & 0xFFu) != 0 ? 1u << q : 0u;
        } else {
            for (int q = 0; q < LB_RUN && t + q < n; ++q) flags |= mask[t + q] != 0 ? 1u << q : 0u;
        }
        int total;
        const int ord = carry + count_scan(__popc(flags), wave_tot, total);
        const unsigned pair = flags | (unsigned)__shfl_down((int)flags, 1) << 16;
        if (tid % 2 == 0 && t < n) {
            bits[t / 32] = pair;
            before[t / 32] = ord;
        }
        carry += total;
    }
    if (tid == 0) {
        row_off[R] = carry;
        col_off[C] = carry;
        nnz_out[0] = carry;
    }
    __syncthreads();
    auto stored = [&](int cell) { return (bits[cell >> 5] >> (cell & 31) & 1u) != 0; };
    auto ordinal = [&](int cell) { return before[cell >> 5] + __popc(bits[cell >> 5] & ((1u << (cell & 31)) - 1u)); };

#pragma unroll 4
    for (int t = tid; t < n; t += LB_THREADS) {
        const int r = (int)((unsigned)t / (unsigned)C), c = t - r * C, ord = ordinal(t);
        ordinal_of[t] = ord;
        if (c == 0) row_off[r] = ord;
        if (stored(t)) row_blocks[ord] = make_int2(ord, (int)(((unsigned)r << 16) + (unsigned)c));
    }

    // column order: a thread takes a run of rows of one column, the counts meet in column-major order
    const int width = C < LB_THREADS ? C : LB_THREADS, runs = LB_THREADS / width, rows = (R + runs - 1) / runs;
    const int run = tid / width, lo = run * rows;
    carry = 0;
    for (int c0 = 0; c0 < C; c0 += width) {
        const int c = c0 + tid - run * width;
        const bool mine = run < runs && c < C;
        const int hi = !mine ? lo : lo + rows < R ? lo + rows : R, slot = (tid - run * width) * runs + run;
        int count = 0;
#pragma unroll 4
        for (int r = lo; r < hi; ++r) count += stored(r * C + c) ? 1 : 0;
        counts[tid] = 0;                                 // slots of nobody, where the width is no divisor
        __syncthreads();
        if (run < runs) counts[slot] = count;
        __syncthreads();
        int total;
        const int in_front = carry + count_scan(counts[tid], wave_tot, total);
        counts[tid] = in_front;
        __syncthreads();
        if (mine) {
            int pos = counts[slot];
            if (run == 0) col_off[c] = pos;
#pragma unroll 4
            for (int r = lo; r < hi; ++r) {
                const int cell = r * C + c;
                if (stored(cell)) col_blocks[pos++] = make_int2(ordinal(cell), (int)(((unsigned)r << 16) + (unsigned)c));
            }
        }
        carry += total;
        __syncthreads();                                 // counts is written again
    }
}

// Up to 1024 cells, and masks whose bits do not fit LDS: the same order from global memory, a cell a thread and scan.
__global__ __launch_bounds__(LB_THREADS) void layout_build_kernel(
    const uint8_t *__restrict__ mask, int R, int C,
    int2 *__restrict__ row_blocks, int *__restrict__ row_off,
    int2 *__restrict__ col_blocks, int *__restrict__ col_off,
    int *__restrict__ nnz_out, int *__restrict__ ordinal_of)
{
    __shared__ int wave_tot[LB_WAVES];
    const int n = R * C;
    const int tid = (int)threadIdx.x;

    // pass 1: row-major order -> row table, ordinals
    int carry = 0;
    for (int base = 0; base < n; base += LB_THREADS) {
        int t = base + tid;
        bool nz = t < n && mask[t] != 0;
        int total;
        int ord = carry + tile_scan(nz, wave_tot, total);
        if (t < n) {
            int r = t / C, c = t - r * C;
            ordinal_of[t] = ord;
            if (c == 0) row_off[r] = ord;
            if (nz) row_blocks[ord] = make_int2(ord, (int)(((unsigned)r << 16) + (unsigned)c));
        }
        carry += total;
    }
    if (tid == 0) {
        row_off[R] = carry;
        col_off[C] = carry;
        nnz_out[0] = carry;
    }
    __syncthreads();   // ordinal_of is re-read below by other lanes of this workgroup

    // pass 2: column-major order -> column table
    carry = 0;
    for (int base = 0; base < n; base += LB_THREADS) {
        int t = base + tid;
        int c = t / R, r = t - c * R;
        int cell = r * C + c;
        bool nz = t < n && mask[cell] != 0;
        int total;
        int pos = carry + tile_scan(nz, wave_tot, total);
        if (t < n) {
            if (r == 0) col_off[c] = pos;
            if (nz) col_blocks[pos] = make_int2(ordinal_of[cell], (int)(((unsigned)r << 16) + (unsigned)c));
        }
        carry += total;
    }
}

// What a layout keeps, once its number of blocks is known: both tables at their exact size and, from the row table, the
// (row, column) and the cell number of every block.  One launch in place of two copies and seven elementwise ones.
__global__ __launch_bounds__(256) void layout_finish_kernel(
    const int2 *__restrict__ row_in, const int2 *__restrict__ col_in, int nnz, int C,
    int2 *__restrict__ row_blocks, int2 *__restrict__ col_blocks, longlong2 *__restrict__ positions,
    long long *__restrict__ cells)
{
    const int i = (int)blockIdx.x * 256 + (int)threadIdx.x;
    if (i >= nnz) return;
    const int2 d = row_in[i];
    row_blocks[i] = d;
    col_blocks[i] = col_in[i];
    const long long r = (long long)((unsigned)d.y >> 16), c = (long long)(d.y & 0xFFFF);
    positions[i] = make_longlong2(r, c);
    cells[i] = r * C + c;
}

hipError_t launch_layout_finish(const int32_t *row_in, const int32_t *col_in, int nnz, int C, int32_t *row_blocks,
                                int32_t *col_blocks, int64_t *positions, int64_t *cells, hipStream_t st)
{
    layout_finish_kernel<<<(unsigned)((nnz + 255) / 256), 256, 0, st>>>((const int2 *)row_in, (const int2 *)col_in, nnz, C,
                                                                        (int2 *)row_blocks, (int2 *)col_blocks,
                                                                        (longlong2 *)positions, (long long *)cells);
    return hipGetLastError();
}

// ---- schedule -------------------------------------------------------------
// Buffer layout (int4 units): [0, groups) per-group meta, then the wavefront slots.
//   meta[g] = (first slot of part 0, first partial-tile slot or -1, ordinal among split groups or -1, parts)

struct GroupPlan {
    int parts;      // workgroup-sized pieces the group is cut into (or row slices, see below)
    int len;
    bool sliced;    // the whole group goes to `slices` waves, each taking 32 / slices of its element rows
};

__device__ __forceinline__ GroupPlan plan_group(int len, int cap, int waves, int allow_split, int slice_max, int slices)
{
    GroupPlan p;
    p.len = len;
    p.sliced = len <= slice_max;
    if (p.sliced) {
        p.parts = slices;
        return p;
    }
    const int span = cap * waves;                       // pairs one workgroup takes at the target chunk size
    int parts = allow_split ? (len + span - 1) / span : 1;
    parts = parts < 1 ? 1 : (parts > SCHED_MAX_PARTS ? SCHED_MAX_PARTS : parts);
    p.parts = parts;
    return p;
}

// pairs [lo, hi) of piece t out of n of a range of `len`
__device__ __forceinline__ int piece_lo(int len, int t, int n) { return (int)(((long long)len * t) / n); }

__device__ __forceinline__ int waves_of_part(int part_len, int cap, int waves)
{
    int nw = (part_len + cap - 1) / cap;
    nw = nw < 1 ? 1 : nw;
    return nw > waves ? waves : nw;
}

__global__ __launch_bounds__(LB_THREADS) void schedule_build_kernel(
    const int *__restrict__ offsets, int groups, int cap, int waves, int flags, int slice_max, int slices,
    int4 *__restrict__ sched, int slot_capacity, int *__restrict__ counts_out)
{
    const int allow_split = flags & BSA_SCHED_SPLIT;
    const bool longest_first = (flags & BSA_SCHED_LONGEST_FIRST) != 0;
    __shared__ int total_slots;
    const int tid = (int)threadIdx.x;
    int4 *meta = sched;
    int4 *slots = sched + groups;
    // Serial first-fit, one pass over the groups per class.  Row-sliced groups fill whole workgroups of
    // their own (their waves need no barrier).  Split groups come before the unsplit ones: their parts
    // meet in a workspace after the walk, and workgroups are dispatched in slot order, so starting them
    // first lets that exchange run while the rest of the launch is still multiplying.
    // Without BSA_SCHED_LONGEST_FIRST: sliced, split, unsplit, each in table order.  With it, long work
    // starts first: split groups, then the unsplit ones by their longest chunk (quarters of cap), then the
    // sliced ones (all shorter than any other group) by length (quarters of the longest of them).  A wave
    // walks its chunk serially and a launch of these kernels is only one or two rounds of waves, so a long
    // chunk that starts last (the late rows of a causal mask) runs on an almost empty machine.
    // A team (the waves of one part) never straddles a workgroup boundary.
    if (tid == 0) {
        int pos = 0, tile_slots = 0, split_groups = 0;
        constexpr int LEN_CLASSES = 4;     // by length: > 3/4, > 1/2, > 1/4 of the yardstick, rest
        constexpr int CLS_SLICED = 0, CLS_SPLIT = LEN_CLASSES, CLS_UNSPLIT = LEN_CLASSES + 1;
        int longest_sliced = 0;
        if (longest_first)
            for (int g = 0; g < groups; ++g) {
                const int len = offsets[g + 1] - offsets[g];
                if (len <= slice_max && len > longest_sliced) longest_sliced = len;
            }
        auto len_class = [](int len, int yard) {
            return 4 * len > 3 * yard ? 0 : (2 * len > yard ? 1 : (4 * len > yard ? 2 : 3));
        };
        const int n_pass = longest_first ? 1 + 2 * LEN_CLASSES : 3;
        for (int pass = 0; pass < n_pass; ++pass) {
            // class handled by this pass
            const int want = longest_first ? (pass <= LEN_CLASSES ? CLS_SPLIT + pass : pass - LEN_CLASSES - 1)
                                           : (pass == 0 ? CLS_SLICED : CLS_SPLIT + pass - 1);
            // the sliced region starts (and ends) on a workgroup boundary
            if (want == CLS_SLICED || (!longest_first && want == CLS_SPLIT)) pos = (pos + waves - 1) / waves * waves;
            for (int g = 0; g < groups; ++g) {
                const GroupPlan gp = plan_group(offsets[g + 1] - offsets[g], cap, waves, allow_split, slice_max, slices);
                int cls;
                if (gp.sliced) {
                    cls = CLS_SLICED + (longest_first ? len_class(gp.len, longest_sliced) : 0);
                } else if (gp.parts > 1) {
                    cls = CLS_SPLIT;
                } else {
                    cls = CLS_UNSPLIT;
                    if (longest_first) {
                        const int nw = waves_of_part(gp.len, cap, waves);
                        cls += len_class((gp.len + nw - 1) / nw, cap);   // blocks the busiest wave of the team walks
                    }
                }
                if (cls != want) continue;
                if (gp.sliced) {
                    meta[g] = make_int4(pos, -1, -1, gp.parts);
                    pos += gp.parts;
                    continue;
                }
                int first = -1;
                for (int p = 0; p < gp.parts; ++p) {
                    int plen = piece_lo(gp.len, p + 1, gp.parts) - piece_lo(gp.len, p, gp.parts);
                    int nw = waves_of_part(plen, cap, waves);
                    int in_wg = pos % waves;
                    if (in_wg + nw > waves) pos += waves - in_wg;
                    if (p == 0) first = pos;
                    pos += nw;
                }
                const bool split = gp.parts > 1;
                meta[g] = make_int4(first, split ? tile_slots : -1, split ? split_groups : -1, gp.parts);
                if (split) { tile_slots += gp.parts; split_groups += 1; }
            }
        }
        int n_wgs = (pos + waves - 1) / waves;
        total_slots = n_wgs * waves;
        counts_out[0] = total_slots <= slot_capacity ? n_wgs : -1;   // -1: the table is too small, nothing usable
        counts_out[1] = tile_slots;
        counts_out[2] = split_groups;
        counts_out[3] = pos;
    }
    __syncthreads();
    const int n_slots = total_slots < slot_capacity ? total_slots : slot_capacity;
    for (int s = tid; s < n_slots; s += LB_THREADS) slots[s] = make_int4(-1, 0, 0, 0);
    __syncthreads();
    for (int g = tid; g < groups; g += LB_THREADS) {
        const int lo = offsets[g];
        const GroupPlan gp = plan_group(offsets[g + 1] - lo, cap, waves, allow_split, slice_max, slices);
        int pos = meta[g].x;
        if (gp.sliced) {
            for (int t = 0; t < gp.parts; ++t)
                if (pos + t < slot_capacity)
                    slots[pos + t] = make_int4(g, lo, lo + gp.len, sched_team_word((pos + t) % waves, 1, t, gp.parts));
            continue;
        }
        for (int p = 0; p < gp.parts; ++p) {
            const int pb = piece_lo(gp.len, p, gp.parts), pe = piece_lo(gp.len, p + 1, gp.parts);
            const int plen = pe - pb;
            const int nw = waves_of_part(plen, cap, waves);
            const int in_wg = pos % waves;
            if (in_wg + nw > waves) pos += waves - in_wg;
            for (int t = 0; t < nw; ++t) {
                const int b = lo + pb + piece_lo(plen, t, nw), e = lo + pb + piece_lo(plen, t + 1, nw);
                if (pos + t < slot_capacity)
                    slots[pos + t] = make_int4(g, b, e, sched_team_word(pos % waves, nw, p, gp.parts));
            }
            pos += nw;
        }
    }
}

// ---- launchers ------------------------------------------------------------

hipError_t launch_layout_build(const uint8_t *mask, int R, int C, int32_t *row_blocks,
                               int32_t *row_off, int32_t *col_blocks, int32_t *col_off,
                               int32_t *nnz_out, void *workspace, hipStream_t stream)
{
    if ((long long)R * C > LB_THREADS && (long long)R * C <= LB_BIT_CELLS) {
        const size_t lds = ((size_t)R * C + 31) / 32 * 8;
        if (lds > 32768) {
            hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void *>(layout_build_bits_kernel),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            if (err != hipSuccess) return err;
        }
        layout_build_bits_kernel<<<1, LB_THREADS, lds, stream>>>(mask, R, C, (int2 *)row_blocks, row_off, (int2 *)col_blocks,
                                                                 col_off, nnz_out, (int *)workspace);
        return hipGetLastError();
    }
    layout_build_kernel<<<1, LB_THREADS, 0, stream>>>(mask, R, C, (int2 *)row_blocks, row_off,
                                                     (int2 *)col_blocks, col_off, nnz_out,
                                                     (int *)workspace);
    return hipGetLastError();
}

hipError_t launch_schedule_build(const int32_t *offsets, int groups, int cap, int waves,
                                 int flags, int slice_max, int slices, int32_t *sched, int64_t capacity,
                                 int32_t *counts_out, hipStream_t stream)
{
    schedule_build_kernel<<<1, LB_THREADS, 0, stream>>>(offsets, groups, cap, waves, flags, slice_max, slices,
                                                       (int4 *)sched, (int)(capacity - groups),
                                                       counts_out);
    return hipGetLastError();
}

}  // namespace bsa
