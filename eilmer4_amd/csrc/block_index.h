// block_index.h -- where the cells of a block lie in its arrays, for blocks of any size
// that fits the memory.  Free of HIP, so that a host program can check it.
//
// An ideal-gas block takes 82 bytes a cell under the Euler scheme, 162 under pc: cell
// indices can pass 2^31, and byte offsets within a field pass 32 bits from 2^29 cells on.
#pragma once

#if defined(__HIPCC__)
#define E4_HD __host__ __device__ __forceinline__
#else
#define E4_HD inline
#endif

namespace e4 {

// Cell 0 of row (j, k): the scalar part of a cell's index for a wave that works on
// one row.  (A row has at least two cells, so the rows of a block that fits the
// memory number below 2^32, and one 32 x 32 bit product gives the cell.)
E4_HD long row_start(int ni, int nj, int j, int k)
{
    return (long)((unsigned long)((unsigned int)k * (unsigned int)nj + (unsigned int)j) * (unsigned int)ni);
}

} // namespace e4
