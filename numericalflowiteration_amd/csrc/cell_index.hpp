// cell_index.hpp — cell numbers of the traces that read slices or tables from
// global memory, as plain integer functions (no HIP in here: the host compiler
// takes it too).
//
// A position too large for z - N floor(z / N) to come back into one period
// (about 2^52 N; an uploaded history of absurd coefficients or a metrics grid
// that far out does that) leaves any integer as its cell on an axis that is not
// a power of two, up to the saturated ends of int.  LDS reads at such a cell
// return some number; reads of global memory have to be kept inside the slice.
#ifndef NUFI_CELL_INDEX_HPP
#define NUFI_CELL_INDEX_HPP

#include <stdint.h>

#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#define NUFI_INDEX_FN __host__ __device__ __forceinline__
#else
#define NUFI_INDEX_FN inline
#endif

namespace nufi_impl
{

// the cell floor(z) of a node counted from the window's first cell zb, in
// [0, Nz) for a position within a period of it; MASK: a power-of-two axis
template <bool MASK>
NUFI_INDEX_FN uint32_t zc_rel( int cell, int zb, int Nz )
{
    int d = int( uint32_t( cell ) - uint32_t( zb ) );
    if ( MASK ) d &= Nz - 1;
    else
    {
        d = d < 0 ? d + Nz : d;
        d = d >= Nz ? d - Nz : d;
    }
    return uint32_t( d );
}

// the cell of offset rel from zb, always one of the slice
NUFI_INDEX_FN uint32_t zc_cell( int zb, uint32_t rel, uint32_t Nz )
{
    uint32_t c = uint32_t( zb ) + rel;
    if ( c >= Nz ) c -= Nz;
    return c < Nz ? c : Nz - 1;
}

// a cell of another axis, always one of the slice
NUFI_INDEX_FN uint32_t zc_held( int i, uint32_t N )
{
    return uint32_t( i ) < N ? uint32_t( i ) : N - 1;
}

// a cell of the 1D tables, which hold cells -1 .. N
NUFI_INDEX_FN int table_cell( int i, int N )
{
    return i < -1 ? -1 : ( i > N ? N : i );
}

} // namespace nufi_impl

#endif
