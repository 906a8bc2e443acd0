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

// A load from a scalar 64-bit base with an unsigned 32-bit byte offset takes no vector
// address arithmetic, and reaches 2^29 doubles.  Whether that is every cell of a block
// and every face of each of its directions (a field of one double per cell or face):
// blocks with a flow-state array and face fluxes take 482 bytes a cell and more, 259 GB
// at 2^29 cells, so larger ones can fit the memory, and kernels that use such offsets
// have another route for them.
constexpr long OFFSET32_DOUBLES = 1L << 29;
E4_HD bool offsets_reach_block(int dims, int ni, int nj, int nk)
{
    const long k = (dims == 3) ? nk : 1;
    const long fi = (ni + 1L) * nj * k, fj = ni * (nj + 1L) * k, fk = (dims == 3) ? (long)ni * nj * (k + 1) : 0;
    const long most = (fi > fj) ? ((fi > fk) ? fi : fk) : ((fj > fk) ? fj : fk);
    return most <= OFFSET32_DOUBLES;
}

} // namespace e4
