// Fused block-sparse attention for gfx950: out = softmax(scale * q k^T, over the stored
// blocks of a row, causal if asked) v, without the scores ever leaving the chip, and its gradients.
//
// The reference computes this as three launches with the scores written and read twice in between
// (SDD sparse/native/sparse_smm_gpu.cu:22-95, softmax sparse_softmax.cu:113-155, DSD
// sparse_smm_gpu.cu:106-181, chained by the caller); per stored block that is 2 KB written + 2 KB
// read + 2 KB written + 2 KB read of HBM traffic that this kernel does not have.
//
// One wavefront walks a chunk of the blocks (r, c) of block row r:
//   S^T = K_c Q_r^T        32 keys x 32 queries, 4 MFMAs over head dim 64; Q_r stays in registers
//   online softmax          a lane holds ONE query column of S^T (16 keys; the other 16 sit in lane
//                           l ^ 32), so reference point, sum and the rescaling factor are per-lane scalars
//   O^T += V_c^T P^T        the probabilities go from the accumulators of the first product straight
//                           into the operand registers of the second: accumulator value v of lane
//                           half h is key 8 (v / 4) + 4 h + v % 4, and V_c is read from LDS in that
//                           order of rows.  No LDS round trip, no shuffle.
// The waves of a row (a team of the schedule) merge their (max, sum, O^T) through LDS.
//
// What bounds it.  A wave has one block in work: about 1750 clocks beside three other waves of its SIMD (LDS operands
// 500, products 200, exponentials 600, the rest scalar), so a SIMD finishes one per 440, of which the vector ALU is busy
// about 390; a wave also spends 6000 clocks before its first block (schedule slot, block columns, first tiles: three
// dependent round trips) and 3000 behind its last.  K and V go straight to LDS, each tile requested as soon as the
// operands of the one before sit in registers, and have arrived when they are wanted (45 and 80 clocks of waiting per
// block); with every request served from one address the launch takes as long.  Against tiles that pass through
// registers, a maximum per block and 8-byte result pieces (us, before -> after): 3 x 5 heads of 2976 tokens, 1053 blocks
// a head 20.1 -> 14.7; 48 heads of 8192 tokens, 2526 blocks 98 -> 82; 16 heads of 4096 tokens, 1530 blocks 23.1 -> 17.6,
// at head dim 128 41.9 -> 35.3.  Panels of four block rows sharing the tiles of a workgroup (half the L2 traffic, a
// barrier per column) took 18.7 / 84 / 21.5: the rows of a panel wait for one another.
#include <cmath>

#include "bsa_device.hpp"
#include "lds_tiles.hpp"
#include "attention_tiles.hpp"
#include "bsa_internal.hpp"
#include "../../include/bsa.h"

namespace bsa {

// per wave: the K tile and the V tile (64 HD bytes each), reused for the O^T partial of the
// team merge (HD x 32 floats: the same size), + row stats
constexpr int at_lds_per_wave(int hd) { return 128 * hd + 256; }
constexpr float AT_LAZY_SUM = 256.f;          // probabilities stay below it (fp16 holds them) until the reference point moves

// Split rows of the forward walk: a block row longer than one workgroup's share is cut into parts
// that run in different workgroups.  Every part parks (O^T, max, sum) of its 32 queries in the
// workspace and bumps the row's counter; the part that arrives last merges the parts in part order
// (so the result does not depend on arrival order), resets the counter and stores the row.  Parked
// values are published and consumed with park_store / split_publish / split_consume / park_load
// (bsa_device.hpp: release and acquire at agent scope).
size_t attention_workspace_bytes(int tile_slots, int split_groups, int batches, int head_dim)
{
    if (tile_slots <= 0 || split_groups <= 0) return 0;
    return at_split_counter_bytes(split_groups, batches) +
           (size_t)tile_slots * batches * at_split_tile_floats(head_dim) * sizeof(float);
}

// workspace of the two backward walks: [row counters | row tiles of 32 hd floats | column counters | column
// tiles of 2 x 32 hd floats (dv^T, dk^T)]
static size_t at_bwd_region_bytes(int tile_slots, int split_groups, int batches, int tile_floats)
{
    if (tile_slots <= 0 || split_groups <= 0) return 0;
    return at_split_counter_bytes(split_groups, batches) + (size_t)tile_slots * batches * tile_floats * sizeof(float);
}
size_t attention_backward_workspace_bytes(int row_tile_slots, int row_split_groups, int col_tile_slots,
                                          int col_split_groups, int batches, int head_dim)
{
    return at_bwd_region_bytes(row_tile_slots, row_split_groups, batches, 32 * head_dim) +
           at_bwd_region_bytes(col_tile_slots, col_split_groups, batches, 64 * head_dim);
}

template <int HD, bool BF>
__global__ __launch_bounds__(512, HD == 64 ? 4 : 2) void attention_fwd_f16_kernel(
    const half_t *__restrict__ q, const half_t *__restrict__ k, const half_t *__restrict__ v,
    half_t *__restrict__ out, float *__restrict__ lse, const BlockDesc *__restrict__ blocks,
    const SchedGroup *__restrict__ sched_groups, const SchedEntry *__restrict__ sched, AtSplitWorkspace ws,
    int n_swg, int batches, int rows_q, int rows_k, float scale2 /* scale * log2(e) */, int causal)
{
    extern __shared__ __align__(16) unsigned char lds_raw[];
    constexpr int KS = HD / 16, KT = HD / 32, LDS_PER_WAVE = at_lds_per_wave(HD), STAT_OFF = 128 * HD;
    int batch, swg;
    if (!map_workgroup(n_swg, batches, batch, swg)) return;
    const int w = wave_id(), l = lane_id();
    const int W = (int)(blockDim.x >> 6);
    const SchedEntry e = sched[swg * W + w];
    const bool active = e.group >= 0;
    const int r = e.group;
    const int qq = l & 31, h = l >> 5;           // query column of this lane, lane half
    const float NEG_INF = -__builtin_inff();

    unsigned char *tile_k = lds_raw + (size_t)w * LDS_PER_WAVE, *tile_v = tile_k + 64 * HD;
    const TileReader rd(tile_k);
    constexpr unsigned K_TILE = 0, V_TILE = 64 * HD;
    const TileRequests<HD> kreq(k + (size_t)batch * rows_k * HD, tile_k), vreq(v + (size_t)batch * rows_k * HD, tile_v);

    // reference point of the query (both lane halves agree), minus it (0 while nothing was seen), this half's sum;
    // unseen: some query of the wave has no reference point yet
    float m = NEG_INF, minus_m = 0.f, lsum = 0.f;
    bool unseen = true;
    RowTile<HD> oacc;
    clear<HD>(oacc);

    if (active && e.begin < e.end) {
        DescWindow win;
        h8 qop[KS];
        // Q_r waits for nothing but the schedule slot: it goes through the V tile (4 requests of whole lines; read
        // straight into operand layout every request would touch 32 lines) beside the load of the block columns.
        TileRequests<HD>(q + (size_t)batch * rows_q * HD, tile_v).issue(r);
        for (int seg = e.begin; seg < e.end; seg += WAVE) {
            const int seg_end = seg + WAVE < e.end ? seg + WAVE : e.end;
            win.fetch(blocks, seg, seg_end);
            kreq.issue(win.get(seg).col());
            if (seg == e.begin) {
                tile_wait<TileRequests<HD>::N>();
#pragma unroll
                for (int s = 0; s < KS; ++s) qop[s] = rd.rows(V_TILE, s);
                lds_reads_done();
            }
            vreq.issue(win.get(seg).col());
            for (int p = seg; p < seg_end; ++p) {
                const int c = win.get(p).col();
                const bool last = p + 1 == seg_end;
                // A stage is a single buffer: K of the next block is requested as soon as this block's operands sit in
                // registers, V likewise, so each has the other half of the block's work to arrive in.
                tile_wait<TileRequests<HD>::N>();            // everything but V
                h8 kop[KS];
#pragma unroll
                for (int s = 0; s < KS; ++s) kop[s] = rd.rows(K_TILE, s);
                lds_reads_done();
                if (!last) kreq.issue(win.get(p + 1).col());
                f16v sacc = {0};                 // keys 8 (v / 4) + 4 h + v % 4 of query qq
#pragma unroll
                for (int s = 0; s < KS; ++s) sacc = mfma_16<BF>(kop[s], qop[s], sacc);
                float mul = scale2;              // what is still to be applied to sacc in the exponent
                if (causal && c >= r) {          // -inf only once scaled, whatever the scale's sign
                    mul = 1.f;
#pragma unroll
                    for (int v = 0; v < 16; ++v)
                        sacc[v] = c > r || 8 * (v >> 2) + 4 * h + (v & 3) > qq ? NEG_INF : sacc[v] * scale2;
                }
                float psum;
                h8 pop[2];
                auto exponentials = [&]() {
                    psum = 0.f;
#pragma unroll
                    for (int v = 0; v < 16; ++v) {
                        const float pv = at_exp2(__builtin_fmaf(sacc[v], mul, minus_m));
                        psum += pv;
                        pop[v >> 3][v & 7] = narrow_16<BF>(pv);
                    }
                };
                // There is no maximum per block: the reference point of a row is the maximum of its first visible block
                // and moves only when a block's sum of exponentials exceeds AT_LAZY_SUM.
                bool move = unseen;
                if (!move) {
                    exponentials();
                    move = __builtin_amdgcn_ballot_w64(!(psum <= AT_LAZY_SUM)) != 0ull;
                }
                if (move) {
                    float bm = sacc[0] * mul;
#pragma unroll
                    for (int v = 1; v < 16; ++v) bm = fmaxf(bm, sacc[v] * mul);
                    const float m_new = fmaxf(m, fmaxf(bm, at_lane_xor32(bm)));
                    const float keep = m == NEG_INF ? 0.f : at_exp2(m - at_finite_or_zero(m_new));   // nothing accumulated so far: 0
                    m = m_new;
                    minus_m = -at_finite_or_zero(m_new);
                    lsum *= keep;
                    each<HD>(oacc, [&](float x, int) { return x * keep; });
                    unseen = __builtin_amdgcn_ballot_w64(m == NEG_INF) != 0ull;
                    exponentials();
                }
                lsum += psum;
                if (last) tile_wait<0>();
                else tile_wait<TileRequests<HD>::N>();       // everything but the next K
                h8 vop[KT][2];
#pragma unroll
                for (int t = 0; t < KT; ++t)
#pragma unroll
                    for (int s = 0; s < 2; ++s) vop[t][s] = rd.columns(V_TILE, t, s);
                lds_reads_done();
                if (!last) vreq.issue(win.get(p + 1).col());
#pragma unroll
                for (int s = 0; s < 2; ++s)
#pragma unroll
                    for (int t = 0; t < KT; ++t) oacc[t] = mfma_16<BF>(vop[t][s], pop[s], oacc[t]);
            }
        }
        lsum += at_lane_xor32(lsum);             // both halves used the same reference point
    }

    // team merge: every wave but the leader parks (max, sum) per query and O^T; the leader rescales and adds
    const int slot0 = e.first_wave(), nw = e.team_waves();
    const bool leader = active && w == slot0;
    if (active && !leader) {
        wave_lds_fence();
        each<HD>(oacc, [&](float x, int at) { return reinterpret_cast<float *>(tile_k)[at] = x; });
        if (h == 0) reinterpret_cast<float2 *>(tile_k + STAT_OFF)[qq] = make_float2(m, lsum);
    }
    __syncthreads();
    if (!leader) return;
    if (nw > 1) {
        auto stat = [&](int o) { return reinterpret_cast<const float2 *>(tile_k + o * LDS_PER_WAVE + STAT_OFF)[qq]; };
        float M = m;
        for (int o = 1; o < nw; ++o) M = fmaxf(M, stat(o).x);
        const float MM = at_finite_or_zero(M), own = at_exp2(m - MM);
        lsum *= own;
        each<HD>(oacc, [&](float x, int) { return x * own; });
        for (int o = 1; o < nw; ++o) {
            const float2 st = stat(o);
            const float f = at_exp2(st.x - MM);
            lsum += st.y * f;
            const float *src = reinterpret_cast<const float *>(tile_k + o * LDS_PER_WAVE);
            each<HD>(oacc, [&](float x, int at) { return x + src[at] * f; });
        }
        m = M;                                   // the sums are relative to the team's reference point now
    }
    if (e.parts() > 1) {
        constexpr int TILE = at_split_tile_floats(HD);
        const SchedGroup sg = sched_groups[r];
        float *tile0 = ws.tiles + ((size_t)batch * ws.tile_slots + sg.tile_slot) * TILE;
        float *mine = tile0 + (size_t)e.part() * TILE;
        park_part<HD>(oacc, mine);
        park_store(mine + 32 * HD + l, m);
        park_store(mine + 32 * HD + WAVE + l, lsum);
        int *counter = ws.counters + (size_t)batch * ws.split_groups + sg.split_index;
        const int parts = e.parts();
        if (split_publish(counter) != parts - 1) return;
        split_consume();
        m = NEG_INF;
        for (int j = 0; j < parts; ++j) m = fmaxf(m, park_load(tile0 + (size_t)j * TILE + 32 * HD + l));
        const float MM = at_finite_or_zero(m);
        lsum = 0.f;
        clear<HD>(oacc);
        for (int j = 0; j < parts; ++j) {
            const float *src = tile0 + (size_t)j * TILE;
            const float f = at_exp2(park_load(src + 32 * HD + l) - MM);
            lsum += park_load(src + 32 * HD + WAVE + l) * f;
            each<HD>(oacc, [&](float x, int at) { return x + park_load(src + at) * f; });
        }
        split_reset(counter);
    }
    // log2 of the row's sum of exponentials of the scaled scores (what the backward pass needs to rebuild the
    // probabilities); +inf for a row that sees nothing, so that they come out as zeros
    const size_t row0 = (size_t)batch * rows_q + (size_t)BS * r;
    if (lse != nullptr && h == 0) lse[row0 + qq] = lsum > 0.f ? at_finite_or_zero(m) + __builtin_amdgcn_logf(lsum) : __builtin_inff();
    store_rows<HD, BF>(oacc, lsum > 0.f ? 1.f / lsum : 0.f, tile_k, out + row0 * HD);
}

// ---------------------------------------------------------------------------
// Backward, the walk over the ROWS: dq, and (STACKS) the probabilities P and the score gradients dS of every stored
// block, from q, k, v, dO, O and the row statistics of the forward pass:
//   P  = exp2(scale2 * q k^T - lse)                         (no second softmax pass: lse is known)
//   dS = scale * P o (dO v^T - delta),  delta_q = sum_d dO_qd O_qd
//   dq^T += K_c^T dS^T
// Same walk as the forward kernel: a lane holds one query column with 16 keys, and the 16-bit dS values feed the dq product
// straight from those registers.  K_c is read from LDS twice, along d for S and along its rows for dq;
// both reads come first, so that the next K is requested before anything is multiplied.  dq alone (us, before -> after):
// 16 heads of 4096 tokens 26.8 -> 20.6, 48 of 8192 116 -> 94; at head dim 128, where two stacks were stored, 69 -> 40.
// Without STACKS nothing is stored per block and delta is left for the column walk: what sparse.attention runs.  STACKS
// serves bsa_attention_backward_scores alone, for callers that finish with products over the stored blocks.
// ---------------------------------------------------------------------------
// per wave: K and V tiles (= the dq^T part of the merge), and with STACKS the two result blocks of 2 KB
constexpr int at_bwd_lds_per_wave(int hd, bool stacks) { return 128 * hd + (stacks ? 4096 : 0); }

// Hidden scores are set to an infinity of the sign that scale2 turns into -inf, so it must not be zero: 1e-30 leaves
// every exponent of a zero scale at 0.
__device__ __forceinline__ float exponent_scale(float scale) { return scale == 0.f ? 1e-30f : scale * 1.4426950408889634f; }

template <int HD, bool BF, bool STACKS>
__global__ __launch_bounds__(512, HD == 64 ? 3 : 2) void attention_bwd_rows_kernel(
    const half_t *__restrict__ q, const half_t *__restrict__ k, const half_t *__restrict__ v,
    const half_t *__restrict__ dout, const half_t *__restrict__ out, const float *__restrict__ lse,
    half_t *__restrict__ p_out, half_t *__restrict__ ds_out, half_t *__restrict__ dq_out,
    float *__restrict__ delta_out,
    const BlockDesc *__restrict__ blocks, const SchedGroup *__restrict__ sched_groups,
    const SchedEntry *__restrict__ sched, AtSplitWorkspace ws,
    int n_swg, int batches, int rows_q, int rows_k, int nnz, float scale, float log2_scale /* of |scale| */, int causal)
{
    extern __shared__ __align__(16) unsigned char lds_raw[];
    constexpr int KS = HD / 16, KT = HD / 32, LDS_PER_WAVE = at_bwd_lds_per_wave(HD, STACKS), N = TileRequests<HD>::N;
    int batch, swg;
    if (!map_workgroup(n_swg, batches, batch, swg)) return;
    const int w = wave_id(), l = lane_id();
    const int W = (int)(blockDim.x >> 6);
    const SchedEntry e = sched[swg * W + w];
    const bool active = e.group >= 0;
    const int r = e.group;
    const int qq = l & 31, h = l >> 5;
    const float scale2 = exponent_scale(scale);
    const size_t row0 = (size_t)batch * rows_q + (size_t)BS * r;

    unsigned char *tile_k = lds_raw + (size_t)w * LDS_PER_WAVE, *tile_v = tile_k + 64 * HD, *tile_p = tile_k + 128 * HD;
    const TileReader rd(tile_k);
    constexpr unsigned K_TILE = 0, V_TILE = 64 * HD;
    const TileRequests<HD> kreq(k + (size_t)batch * rows_k * HD, tile_k), vreq(v + (size_t)batch * rows_k * HD, tile_v);

    RowTile<HD> dq;
    clear<HD>(dq);

    if (active && e.begin < e.end) {
        DescWindow win;
        h8 qop[KS], dop[KS];
        float delta = 0.f, minus_lse = 0.f;
        // Q_r and dO_r go through the tiles, as in the forward walk, while the block columns are fetched
        TileRequests<HD>(q + (size_t)batch * rows_q * HD, tile_k).issue(r);
        TileRequests<HD>(dout + (size_t)batch * rows_q * HD, tile_v).issue(r);
        for (int seg = e.begin; seg < e.end; seg += WAVE) {
            const int seg_end = seg + WAVE < e.end ? seg + WAVE : e.end;
            win.fetch(blocks, seg, seg_end);
            if (seg == e.begin) {
                h8 oop[KS];
                load_row_operands<HD>(out + row0 * HD, oop);
                // |scale| rides in the exponent (where dS alone is wanted), its sign in the store
                minus_lse = (STACKS ? 0.f : log2_scale) - lse[row0 + qq];
                tile_wait<0>();
#pragma unroll
                for (int s = 0; s < KS; ++s) {
                    qop[s] = rd.rows(K_TILE, s);
                    dop[s] = rd.rows(V_TILE, s);
                }
                lds_reads_done();
                kreq.issue(win.get(seg).col());
                vreq.issue(win.get(seg).col());
#pragma unroll
                for (int s = 0; s < KS; ++s)
#pragma unroll
                    for (int j = 0; j < 8; ++j) delta += widen_16<BF>(dop[s][j]) * widen_16<BF>(oop[s][j]);
                delta += at_lane_xor32(delta);   // the other half of the head dim sits in lane ^ 32
                if (delta_out != nullptr && w == e.first_wave() && e.part() == 0 && h == 0) delta_out[row0 + qq] = delta;
            } else {
                kreq.issue(win.get(seg).col());
                vreq.issue(win.get(seg).col());
            }
            for (int p = seg; p < seg_end; ++p) {
                const BlockDesc d = win.get(p);
                const int c = d.col();
                const bool last = p + 1 == seg_end;
                tile_wait<N>();                  // everything but V (and, in the first round, the delta store)
                h8 ktr[KT][2];
                f16v sacc = {0}, dpacc = {0};    // keys 8 (v / 4) + 4 h + v % 4 of query qq
                {
                    h8 kop[KS];
#pragma unroll
                    for (int s = 0; s < KS; ++s) kop[s] = rd.rows(K_TILE, s);
#pragma unroll
                    for (int t = 0; t < KT; ++t)
#pragma unroll
                        for (int s = 0; s < 2; ++s) ktr[t][s] = rd.columns(K_TILE, t, s);
                    lds_reads_done();
                    if (!last) kreq.issue(win.get(p + 1).col());
#pragma unroll
                    for (int s = 0; s < KS; ++s) sacc = mfma_16<BF>(kop[s], qop[s], sacc);
                }
                if (last) tile_wait<0>();
                else tile_wait<N>();             // everything but the next K
                {
                    h8 vop[KS];
#pragma unroll
                    for (int s = 0; s < KS; ++s) vop[s] = rd.rows(V_TILE, s);
                    lds_reads_done();
                    if (!last) vreq.issue(win.get(p + 1).col());
#pragma unroll
                    for (int s = 0; s < KS; ++s) dpacc = mfma_16<BF>(vop[s], dop[s], dpacc);
                }
                if (causal && c >= r) {          // a hidden score has no probability
#pragma unroll
                    for (int v = 0; v < 16; ++v)
                        if (c > r || 8 * (v >> 2) + 4 * h + (v & 3) > qq) sacc[v] = scale2 < 0.f ? __builtin_inff() : -__builtin_inff();
                }
                h8 ds[2];
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    h4 pv, dv;
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int v = 4 * g + j;
                        const float pr = at_exp2(__builtin_fmaf(sacc[v], scale2, minus_lse)), grad = dpacc[v] - delta;
                        if (STACKS) pv[j] = narrow_16<BF>(pr);
                        dv[j] = narrow_16<BF>(STACKS ? scale * pr * grad : pr * grad);
                        ds[v >> 3][v & 7] = dv[j];
                    }
                    if (STACKS) {                // rows of 64 bytes: query qq, keys 8 g + 4 h .. + 3
                        const int at = 16 * kc_slot(qq, g) + 8 * h;
                        *reinterpret_cast<h4 *>(tile_p + at) = pv;
                        *reinterpret_cast<h4 *>(tile_p + 2048 + at) = dv;
                    }
                }
                if (dq_out != nullptr) {
#pragma unroll
                    for (int s = 0; s < 2; ++s)
#pragma unroll
                        for (int t = 0; t < KT; ++t) dq[t] = mfma_16<BF>(ktr[t][s], ds[s], dq[t]);
                }
                if (STACKS) {                    // out of LDS as whole 2 KB pieces
                    wave_lds_fence();
                    uint4 raw[2];
                    lds_get_linear(reinterpret_cast<const half_t *>(tile_p), raw);
                    stg_tile32(p_out + ((size_t)batch * nnz + d.idx) * BS2, raw);
                    lds_get_linear(reinterpret_cast<const half_t *>(tile_p + 2048), raw);
                    stg_tile32(ds_out + ((size_t)batch * nnz + d.idx) * BS2, raw);
                    wave_lds_fence();
                }
            }
        }
    }
    if (dq_out == nullptr) return;               // uniform over the launch

    // team merge: every wave of a row but the leader parks its dq^T part, the leader adds and stores
    const int slot0 = e.first_wave(), nw = e.team_waves();
    const bool leader = active && w == slot0;
    if (active && !leader) {
        wave_lds_fence();
        each<HD>(dq, [&](float x, int at) { return reinterpret_cast<float *>(tile_k)[at] = x; });
    }
    __syncthreads();
    if (!leader) return;
    for (int o = 1; o < nw; ++o) {
        const float *src = reinterpret_cast<const float *>(tile_k + o * LDS_PER_WAVE);
        each<HD>(dq, [&](float x, int at) { return x + src[at]; });
    }
    if (e.parts() > 1) {                         // a row cut into parts: they add up in the workspace
        constexpr int TILE = 32 * HD;
        const SchedGroup sg = sched_groups[r];
        float *tile0 = ws.tiles + ((size_t)batch * ws.tile_slots + sg.tile_slot) * TILE;
        park_part<HD>(dq, tile0 + (size_t)e.part() * TILE);
        int *counter = ws.counters + (size_t)batch * ws.split_groups + sg.split_index;
        if (split_publish(counter) != e.parts() - 1) return;
        split_consume();
        sum_parts<HD>(dq, tile0, TILE, e.parts());
        split_reset(counter);
    }
    const float sign = !STACKS && scale < 0.f ? -1.f : 1.f;
    store_rows<HD, BF>(dq, sign, tile_k, dq_out + row0 * HD);
}

// ---------------------------------------------------------------------------
// Backward, the walk over the COLUMNS: dk and dv of block column c from the blocks (r, c) of the
// column table, with nothing but q, k, v, dO and two floats per query (lse of the forward pass,
// delta of the row walk above) read: the probabilities and the score gradients are rebuilt in
// registers a second time rather than stored by the row walk and read back (4 KB written + 4 KB
// read of HBM traffic per block that this pair of kernels does not have).
//   S  = Q_r K_c^T, dP = dO_r V_c^T    K_c and V_c stay in registers; a lane holds ONE key column, 16 queries, whose lse
//                                      and delta come into LDS with the tiles
//   dv^T += dO_r^T P,  dk^T += Q_r^T dS   the 16-bit P and dS values are the column operands straight from the
//                                      accumulators, the Q_r and dO_r tiles are read a second time along their rows
// The waves of a column add their parts through LDS.  Three waves per SIMD at head dim 64 (168 registers: V is read out of
// LDS for every block, the exponentials stay in front of the second product), two at 128 (256 registers: accumulators 128, K
// and V 64, so a tile's operands are read four at a time instead of all at once).
// us, both sides in turn on one box, two waves per SIMD (200 registers) -> three at 64: 48 heads of 8192 tokens 114.1 -> 105.8,
// the training pass 275.2 -> 266.3; one (368 registers) -> two at 128, where a wave alone had nothing to wait beside: 16 heads of
// 4096 tokens 72 -> 58 under the profiler, the training pass 137.3 -> 128.4 (left to the compiler two waves spill 53 registers and
// take nearly three times as long).  There a second stage of tiles, requested a whole block ahead, took one wave 63.1 -> 66.1 us.  At 64
// one workgroup per residency slot that walks several columns and requests the next one's tiles early took 111 -> 129 us (its
// neighbours drift apart and leave the L2's working set), forward and rows likewise.
// Delta is scaled as it is read; with scale * delta in memory the whole backward pass takes 1 % less (48.4-49.0 against 49.3-50.1
// us).  Starting the second product at delta, 184 registers, takes as long and is further from float64 (dk of fp16, causal:
// 3.1957e-4 against 3.1949e-4, at head dim 128 3.4662e-4 against 3.4642e-4).
// ---------------------------------------------------------------------------
// Q + dO tiles (= one parked accumulator set) + lse, delta; at head dim 64 also V, whose operands are read again for every
// block: kept in registers they are the 16 that stand between the walk and three waves per SIMD
constexpr bool at_bwd_col_keeps_v(int hd) { return hd == 64; }
constexpr int at_bwd_col_lds_per_wave(int hd) { return 128 * hd + 256 + (at_bwd_col_keeps_v(hd) ? 64 * hd : 0); }

template <int HD, bool BF>
__global__ __launch_bounds__(HD == 64 ? 512 : 64 * AT_COLUMN_WAVES_128, HD == 64 ? 3 : 2) void attention_bwd_dkdv_kernel(
    const half_t *__restrict__ q, const half_t *__restrict__ k, const half_t *__restrict__ v,
    const half_t *__restrict__ dout, const float *__restrict__ lse, const float *__restrict__ delta,
    half_t *__restrict__ dk_out, half_t *__restrict__ dv_out,
    const BlockDesc *__restrict__ blocks, const SchedGroup *__restrict__ sched_groups,
    const SchedEntry *__restrict__ sched, AtSplitWorkspace ws,
    int n_swg, int batches, int rows_q, int rows_k, float scale, int causal)
{
    extern __shared__ __align__(16) unsigned char lds_raw[];
    constexpr int KS = HD / 16, KT = HD / 32, LDS_PER_WAVE = at_bwd_col_lds_per_wave(HD);
    int batch, swg;
    if (!map_workgroup(n_swg, batches, batch, swg)) return;
    const int w = wave_id(), l = lane_id();
    const int W = (int)(blockDim.x >> 6);
    const SchedEntry e = sched[swg * W + w];
    const bool active = e.group >= 0;
    const int c = e.group;
    const int key = l & 31, h = l >> 5;          // key column of this lane, lane half
    const float scale2 = exponent_scale(scale);
    const size_t row0 = (size_t)batch * rows_k + (size_t)BS * c;

    unsigned char *tile_q = lds_raw + (size_t)w * LDS_PER_WAVE, *tile_do = tile_q + 64 * HD;
    const TileReader rd(tile_q);
    constexpr bool KEEPS_V = at_bwd_col_keeps_v(HD);
    constexpr unsigned Q_TILE = 0, DO_TILE = 64 * HD, V_TILE = KEEPS_V ? 128 * HD + 256 : DO_TILE;
    const float *stats = reinterpret_cast<const float *>(tile_q + 128 * HD);      // 32 lse, 32 delta of the block's queries
    const TileRequests<HD> qreq(q + (size_t)batch * rows_q * HD, tile_q), doreq(dout + (size_t)batch * rows_q * HD, tile_do);
    const float *my_stat = (l < 32 ? lse : delta) + (size_t)batch * rows_q + (l & 31);
    const unsigned stat_lds = __builtin_amdgcn_readfirstlane(lds_address(stats));

    RowTile<HD> dv, dk;
    clear<HD>(dv);
    clear<HD>(dk);

    if (active && e.begin < e.end) {
        DescWindow win;
        h8 kop[KS], vop[KS];
        // K_c and V_c go through the tiles, as Q_r does in the forward walk, while the block rows are fetched
        TileRequests<HD>(k + (size_t)batch * rows_k * HD, tile_q).issue(c);
        TileRequests<HD>(v + (size_t)batch * rows_k * HD, tile_q + V_TILE).issue(c);
        for (int seg = e.begin; seg < e.end; seg += WAVE) {
            const int seg_end = seg + WAVE < e.end ? seg + WAVE : e.end;
            win.fetch(blocks, seg, seg_end);
            auto request_q = [&](int p) {
                const int r = win.get(p).row();
                dma4_gather(my_stat + BS * r, stat_lds);
                qreq.issue(r);
            };
            // acc += rows of a tile, four operands of it in registers at a time
            auto products_of_rows = [&](unsigned tile, auto other, f16v &acc) {
#pragma unroll
                for (int s0 = 0; s0 < KS; s0 += 4) {
                    h8 op[4];
#pragma unroll
                    for (int s = 0; s < 4; ++s) op[s] = rd.rows(tile, s0 + s);
#pragma unroll
                    for (int s = 0; s < 4; ++s) acc = mfma_16<BF>(op[s], other(s0 + s), acc);
                    if (KS > 4) __builtin_amdgcn_sched_barrier(0);
                }
            };
            if (seg == e.begin) {
                tile_wait<0>();
#pragma unroll
                for (int s = 0; s < KS; ++s) {
                    kop[s] = rd.rows(Q_TILE, s);
                    if (!KEEPS_V) vop[s] = rd.rows(V_TILE, s);
                }
                lds_reads_done();
            }
            request_q(seg);
            doreq.issue(win.get(seg).row());
            for (int p = seg; p < seg_end; ++p) {
                const int r = win.get(p).row();
                const bool last = p + 1 == seg_end, masked = causal && c >= r;
                h8 pop[2], ds[2];                // queries 8 (v / 4) + 4 h + v % 4 of this lane's key
                // The probabilities need Q and lse only: dO, requested last, has the whole of them to arrive in (one wait for
                // both before: training pass of 48 heads of 8192 tokens 274.9 -> 271.8 us, bf16).
                tile_wait<TileRequests<HD>::N>();            // everything but dO
                f16v prob = {0};
                {
                    products_of_rows(Q_TILE, [&](int s) { return kop[s]; }, prob);
                    if (masked) {                // a hidden score has no probability
                        int first = key - 4 * h;
                        asm volatile("" : "+v"(first));      // its comparisons stay here: 16 masks would be kept through the walk
#pragma unroll
                        for (int v = 0; v < 16; ++v)
                            if (c > r || first > 8 * (v >> 2) + (v & 3)) prob[v] = scale2 < 0.f ? __builtin_inff() : -__builtin_inff();
                    }
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        const f4v ls = *reinterpret_cast<const f4v *>(stats + 8 * g + 4 * h);
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            const int v = 4 * g + j;
                            prob[v] = at_exp2(__builtin_fmaf(prob[v], scale2, -ls[j]));
                            if (!KEEPS_V) pop[v >> 3][v & 7] = narrow_16<BF>(prob[v]);
                        }
                    }
                }
                // The exponentials come here.  The compiler moved them behind the products below, which wait for dO, and kept
                // the 32 statistics in registers beside the scores.
                if (KEEPS_V) asm volatile("" : "+v"(prob));
                tile_wait<0>();
                {
                    f16v dpacc = {0};
                    products_of_rows(DO_TILE, [&](int s) { return KEEPS_V ? rd.rows(V_TILE, s) : vop[s]; }, dpacc);
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        const f4v dl = *reinterpret_cast<const f4v *>(stats + 32 + 8 * g + 4 * h) * scale;
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            const int v = 4 * g + j;
                            ds[v >> 3][v & 7] = narrow_16<BF>(prob[v] * __builtin_fmaf(dpacc[v], scale, -dl[j]));
                            if (KEEPS_V) pop[v >> 3][v & 7] = narrow_16<BF>(prob[v]);
                        }
                    }
                }
                // The tiles are read a second time, Q first: the requests for the next block go out as soon as each is free.
                auto products_of_columns = [&](unsigned tile, const h8 (&op)[2], RowTile<HD> &acc, auto when_read) {
#pragma unroll
                    for (int t0 = 0; t0 < KT; t0 += 2) {
                        h8 tr[2][2];
#pragma unroll
                        for (int t = 0; t < 2; ++t)
#pragma unroll
                            for (int s = 0; s < 2; ++s) tr[t][s] = rd.columns(tile, t0 + t, s);
                        lds_reads_done();
                        if (t0 + 2 == KT) when_read();
#pragma unroll
                        for (int s = 0; s < 2; ++s)
#pragma unroll
                            for (int t = 0; t < 2; ++t) acc[t0 + t] = mfma_16<BF>(tr[t][s], op[s], acc[t0 + t]);
                        if (KT > 2) __builtin_amdgcn_sched_barrier(0);
                    }
                };
                products_of_columns(Q_TILE, ds, dk, [&]() { if (!last) request_q(p + 1); });
                products_of_columns(DO_TILE, pop, dv, [&]() { if (!last) doreq.issue(win.get(p + 1).row()); });
            }
        }
    }

    // team merge, one accumulator set at a time (the staging tiles hold exactly one): every wave of a
    // column but the leader parks its part, the leader adds
    const int slot0 = e.first_wave(), nw = e.team_waves();
    const bool leader = active && w == slot0;
#pragma unroll
    for (int which = 0; which < 2; ++which) {
        RowTile<HD> &acc = which == 0 ? dv : dk;
        if (which == 1) __syncthreads();         // the leaders have read the first set
        if (active && !leader) {
            wave_lds_fence();
            each<HD>(acc, [&](float x, int at) { return reinterpret_cast<float *>(tile_q)[at] = x; });
        }
        __syncthreads();
        if (leader) {
            for (int o = 1; o < nw; ++o) {
                const float *src = reinterpret_cast<const float *>(tile_q + o * LDS_PER_WAVE);
                each<HD>(acc, [&](float x, int at) { return x + src[at]; });
            }
        }
    }
    if (!leader) return;
    if (e.parts() > 1) {                         // a column cut into parts: they add up in the workspace
        constexpr int HALF = 32 * HD, TILE = 2 * HALF;       // dv^T then dk^T
        const SchedGroup sg = sched_groups[c];
        float *tile0 = ws.tiles + ((size_t)batch * ws.tile_slots + sg.tile_slot) * TILE;
        park_part<HD>(dv, tile0 + (size_t)e.part() * TILE);
        park_part<HD>(dk, tile0 + (size_t)e.part() * TILE + HALF);
        int *counter = ws.counters + (size_t)batch * ws.split_groups + sg.split_index;
        if (split_publish(counter) != e.parts() - 1) return;
        split_consume();
        sum_parts<HD>(dv, tile0, TILE, e.parts());
        sum_parts<HD>(dk, tile0 + HALF, TILE, e.parts());
        split_reset(counter);
    }
    store_rows<HD, BF>(dv, 1.f, tile_q, dv_out + row0 * HD);
    store_rows<HD, BF>(dk, 1.f, tile_q, dk_out + row0 * HD);
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
namespace {
struct Walk {                                    // what the three kernels are launched with alike
    dim3 grid, block;
    size_t lds;
    AtSplitWorkspace ws;
    const BlockDesc *blocks;
    const SchedGroup *groups;
    const SchedEntry *slots;
    Walk(const AttentionArgs &p, int lds_per_wave)
        : grid(grid_workgroups(p.sched_wgs, p.batches)), block(64 * p.sched_waves), lds((size_t)p.sched_waves * lds_per_wave),
          blocks((const BlockDesc *)p.blocks), groups((const SchedGroup *)p.sched), slots((const SchedEntry *)p.sched + p.groups)
    {
        ws.tile_slots = p.tile_slots;
        ws.split_groups = p.split_groups;
        ws.counters = (int *)p.workspace;
        ws.tiles = (float *)((char *)p.workspace + at_split_counter_bytes(p.split_groups, p.batches));
    }
    // a launch gets 64 KB of LDS without asking
    template <class Kernel>
    hipError_t allow(Kernel kernel) const
    {
        if (lds <= 65536) return hipSuccess;
        return hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    }
};

template <int HD, bool BF>
hipError_t forward(const AttentionArgs &p, hipStream_t st)
{
    const Walk w(p, at_lds_per_wave(HD));
    const hipError_t err = w.allow(attention_fwd_f16_kernel<HD, BF>);
    if (err != hipSuccess) return err;
    attention_fwd_f16_kernel<HD, BF><<<w.grid, w.block, w.lds, st>>>(
        (const half_t *)p.q, (const half_t *)p.k, (const half_t *)p.v, (half_t *)p.out, (float *)p.lse, w.blocks, w.groups,
        w.slots, w.ws, p.sched_wgs, p.batches, 32 * p.mask_rows, 32 * p.mask_cols, p.scale * 1.4426950408889634f, p.causal ? 1 : 0);
    return hipGetLastError();
}

template <int HD, bool BF, bool STACKS>
hipError_t backward_rows(const AttentionArgs &p, hipStream_t st)
{
    const Walk w(p, at_bwd_lds_per_wave(HD, STACKS));
    const hipError_t err = w.allow(attention_bwd_rows_kernel<HD, BF, STACKS>);
    if (err != hipSuccess) return err;
    attention_bwd_rows_kernel<HD, BF, STACKS><<<w.grid, w.block, w.lds, st>>>(
        (const half_t *)p.q, (const half_t *)p.k, (const half_t *)p.v, (const half_t *)p.dout, (const half_t *)p.out,
        (const float *)p.lse, (half_t *)p.p_out, (half_t *)p.ds_out, (half_t *)p.dq_out, (float *)p.delta, w.blocks, w.groups,
        w.slots, w.ws, p.sched_wgs, p.batches, 32 * p.mask_rows, 32 * p.mask_cols, p.nnz, p.scale, log2f(fabsf(p.scale)),
        p.causal ? 1 : 0);
    return hipGetLastError();
}

template <int HD, bool BF>
hipError_t backward_columns(const AttentionArgs &p, hipStream_t st)
{
    const Walk w(p, at_bwd_col_lds_per_wave(HD));
    const hipError_t err = w.allow(attention_bwd_dkdv_kernel<HD, BF>);
    if (err != hipSuccess) return err;
    attention_bwd_dkdv_kernel<HD, BF><<<w.grid, w.block, w.lds, st>>>(
        (const half_t *)p.q, (const half_t *)p.k, (const half_t *)p.v, (const half_t *)p.dout, (const float *)p.lse,
        (const float *)p.delta, (half_t *)p.dk_out, (half_t *)p.dv_out, w.blocks, w.groups, w.slots, w.ws, p.sched_wgs,
        p.batches, 32 * p.mask_rows, 32 * p.mask_cols, p.scale, p.causal ? 1 : 0);
    return hipGetLastError();
}
}  // namespace

hipError_t launch_attention_forward(const AttentionArgs &p, hipStream_t st)
{
    if (p.head_dim == 64) return p.bf16 ? forward<64, true>(p, st) : forward<64, false>(p, st);
    return p.bf16 ? forward<128, true>(p, st) : forward<128, false>(p, st);
}

hipError_t launch_attention_backward_scores(const AttentionArgs &p, hipStream_t st)
{
    if (p.p_out != nullptr) {
        if (p.head_dim == 64) return p.bf16 ? backward_rows<64, true, true>(p, st) : backward_rows<64, false, true>(p, st);
        return p.bf16 ? backward_rows<128, true, true>(p, st) : backward_rows<128, false, true>(p, st);
    }
    if (p.head_dim == 64) return p.bf16 ? backward_rows<64, true, false>(p, st) : backward_rows<64, false, false>(p, st);
    return p.bf16 ? backward_rows<128, true, false>(p, st) : backward_rows<128, false, false>(p, st);
}

hipError_t launch_attention_backward_dkdv(const AttentionArgs &p, hipStream_t st)
{
    if (p.head_dim == 64) return p.bf16 ? backward_columns<64, true>(p, st) : backward_columns<64, false>(p, st);
    return p.bf16 ? backward_columns<128, true>(p, st) : backward_columns<128, false>(p, st);
}

}  // namespace bsa
