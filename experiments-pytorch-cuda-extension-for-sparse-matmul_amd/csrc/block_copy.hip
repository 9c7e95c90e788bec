// Dense matrix <-> stack of its stored 32x32 blocks, for gfx950.
//
// Replaces SparseLayout.to_sparse / to_dense (sparse/layout.py:40-57), which the reference writes
// as Python loops over the blocks of a CPU-side index list.  One wavefront moves one block per
// batch entry: the dense side is 32 rows of 32 elements (64 or 128 contiguous bytes each), the
// sparse side one contiguous 2 or 4 KB piece; every lane moves 16-byte pieces, and both sides are
// touched once (non-temporal).  to_dense walks every CELL of the mask and writes zeros where no
// block is stored, so the result needs no separate fill.
#include "bsa_device.hpp"
#include "bsa_internal.hpp"

namespace bsa {

constexpr int BC_WAVES = 4;

// piece p (16 bytes) of a block: row p / (2 ES), 16-byte column piece p % (2 ES)
template <int ES>
__device__ __forceinline__ size_t dense_piece_offset(int p, size_t row_bytes)
{
    return (size_t)(p / (2 * ES)) * row_bytes + 16u * (unsigned)(p % (2 * ES));
}

template <int ES>
__global__ __launch_bounds__(64 * BC_WAVES) void to_sparse_kernel(
    const unsigned char *__restrict__ dense, unsigned char *__restrict__ sparse,
    const BlockDesc *__restrict__ blocks, int nnz, int batches, int R, int C)
{
    const int idx = (int)blockIdx.x * BC_WAVES + wave_id();
    if (idx >= nnz) return;
    const int l = lane_id();
    const BlockDesc d = blocks[idx];
    const size_t row_bytes = (size_t)C * BS * ES;
    for (int b = (int)blockIdx.y; b < batches; b += (int)gridDim.y) {
        const unsigned char *src = dense + ((size_t)b * R * BS + (size_t)BS * d.row()) * row_bytes + (size_t)BS * ES * d.col();
        unsigned char *dst = sparse + ((size_t)b * nnz + d.idx) * BS2 * ES;
#pragma unroll
        for (int q = 0; q < ES; ++q) {
            const int p = l + WAVE * q;
            stg16_stream(dst + 16 * p, ldg16_stream(src + dense_piece_offset<ES>(p, row_bytes)));
        }
    }
}

// ordinal_of[cell] = number of stored blocks in front of the cell in row-major order (what
// layout_build_kernel leaves in its workspace): the block index of a stored cell.
// Bound by what it writes, mostly zeros: a wave takes as many neighbouring cells of a mask row as make 256 bytes of a
// dense row (four of fp16, two of fp32), so that a request writes whole lines; a lane keeps to one column piece, i.e. to one
// cell.  One fp16 cell a wave wrote 64-byte halves of lines: 8 matrices of 2048 x 2048, a tenth of the cells stored,
// 20.9 -> 18.5 us.
template <int ES>
__global__ __launch_bounds__(64 * BC_WAVES) void to_dense_kernel(
    const unsigned char *__restrict__ sparse, unsigned char *__restrict__ dense,
    const uint8_t *__restrict__ mask, const int *__restrict__ ordinal_of, int nnz, int batches, int R, int C)
{
    constexpr int CELLS = 8 / ES;                        // of a wave
    const int chunks = (C + CELLS - 1) / CELLS;
    const int chunk = (int)blockIdx.x * BC_WAVES + wave_id();
    if (chunk >= R * chunks) return;
    const int l = lane_id(), piece = l & 15;
    const int r = chunk / chunks, c0 = (chunk - r * chunks) * CELLS, c = c0 + piece / (2 * ES);
    if (c >= C) return;
    const bool stored = mask[(size_t)r * C + c] != 0;
    const int idx = stored ? ordinal_of[(size_t)r * C + c] : 0;
    const size_t row_bytes = (size_t)C * BS * ES;
    for (int b = (int)blockIdx.y; b < batches; b += (int)gridDim.y) {
        unsigned char *dst = dense + ((size_t)b * R * BS + (size_t)BS * r + (l >> 4)) * row_bytes + (size_t)BS * ES * c0 + 16 * piece;
        const unsigned char *src = sparse + ((size_t)b * nnz + idx) * BS2 * ES + (size_t)(l >> 4) * BS * ES + 16 * (piece % (2 * ES));
        uint4 v[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            v[q] = make_uint4(0, 0, 0, 0);
            if (stored) v[q] = ldg16_stream(src + (size_t)4 * q * BS * ES);
        }
#pragma unroll
        for (int q = 0; q < 8; ++q) stg16_stream(dst + (size_t)4 * q * row_bytes, v[q]);
    }
}

hipError_t launch_to_sparse(int elem_size, const void *dense, void *sparse, const int32_t *row_blocks,
                            int nnz, int batches, int R, int C, hipStream_t st)
{
    dim3 grid((unsigned)((nnz + BC_WAVES - 1) / BC_WAVES), (unsigned)(batches < 65535 ? batches : 65535)), block(64 * BC_WAVES);
    if (elem_size == 2)
        to_sparse_kernel<2><<<grid, block, 0, st>>>((const unsigned char *)dense, (unsigned char *)sparse,
                                                   (const BlockDesc *)row_blocks, nnz, batches, R, C);
    else
        to_sparse_kernel<4><<<grid, block, 0, st>>>((const unsigned char *)dense, (unsigned char *)sparse,
                                                   (const BlockDesc *)row_blocks, nnz, batches, R, C);
    return hipGetLastError();
}

hipError_t launch_to_dense(int elem_size, const void *sparse, void *dense, const uint8_t *mask,
                           const int32_t *ordinal_of, int nnz, int batches, int R, int C, hipStream_t st)
{
    const int cells = 8 / elem_size, chunks = R * ((C + cells - 1) / cells);
    dim3 grid((unsigned)((chunks + BC_WAVES - 1) / BC_WAVES), (unsigned)(batches < 65535 ? batches : 65535)), block(64 * BC_WAVES);
    if (elem_size == 2)
        to_dense_kernel<2><<<grid, block, 0, st>>>((const unsigned char *)sparse, (unsigned char *)dense, mask,
                                                  ordinal_of, nnz, batches, R, C);
    else
        to_dense_kernel<4><<<grid, block, 0, st>>>((const unsigned char *)sparse, (unsigned char *)dense, mask,
                                                  ordinal_of, nnz, batches, R, C);
    return hipGetLastError();
}

}  // namespace bsa
