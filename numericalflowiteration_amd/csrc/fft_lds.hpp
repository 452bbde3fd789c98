// fft_lds.hpp — batched Stockham FFT over LDS buffers (radix 4, with one
// radix-2 stage for odd log2 L; for an axis whose length is not a power of two
// a stage per factor 4 and per prime), shared by the field kernels and the adjoint field kernel.  All
// FIELD_BLOCK threads of the workgroup take part; every stage ends with a
// barrier.
#ifndef NUFI_FFT_LDS_HPP
#define NUFI_FFT_LDS_HPP

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace nufi_impl
{

constexpr int FIELD_BLOCK = 512;

// Products with the roundings spelled out: an FP32C run amplifies a last bit, so
// the bits must not depend on what the compiler contracts where.
__device__ __forceinline__ double2 cmul( double2 a, double2 b )
{
    return make_double2( fma( a.x, b.x, -( a.y*b.y ) ), fma( a.y, b.x, a.x*b.y ) );
}

// twiddles an axis of length L reads: exp(-2 pi i k/L) for k < L/2 (radix 2)
// or k < L (mixed radix); none for L <= 1
__host__ __device__ inline uint32_t twiddle_entries( uint32_t L, uint32_t log2L )
{
    if ( L <= 1 ) return 0;
    return log2L == 0xffffffffu ? L : L / 2;
}

// The stages of a length that is not a power of two: its factors 4, then its
// primes, 16 bits each in order, 0 after the last (none above 8 up to 5120,
// the longest line the LDS holds; one factor L past that).
struct fft_radices
{
    uint64_t lo, hi;
    __host__ __device__ uint32_t at( uint32_t i ) const
    {
        return i < 8 ? uint32_t( ( i < 4 ? lo : hi ) >> ( 16 * ( i & 3 ) ) ) & 0xffffu : 0u;
    }
};

// `direct`: the one factor L, the direct DFT
inline fft_radices make_radices( uint32_t L, bool direct = false )
{
    fft_radices r { 0, 0 };
    uint32_t f[32], n = 0, rest = L;
    for ( ; rest % 4 == 0 && rest > 1; rest /= 4 ) f[n++] = 4;
    for ( uint32_t p = 2; rest > 1; ++p )
    {
        if ( p * p > rest ) p = rest;
        for ( ; rest % p == 0 && rest > 1; rest /= p ) f[n++] = p;
    }
    if ( direct || n > 8 ) { n = 1; f[0] = L; }
    for ( uint32_t i = 0; i < n; ++i ) ( i < 4 ? r.lo : r.hi ) |= uint64_t( f[i] & 0xffffu ) << ( 16 * ( i & 3 ) );
    return r;
}

struct axis_desc
{
    uint32_t L, log2L, S;       // length, log2 (or ~0u), stride
    uint32_t nlines;
    uint32_t mode;              // 0: x lines, 1: y lines, 2: z lines
    uint32_t Nx, Ny;
    fft_radices rad;            // not a power of two: its stages
};

// x / y for x < 2^21 and an inverse of y good to a few units in the last place
__device__ __forceinline__ uint32_t div_small( uint32_t x, float inv )
{
    return uint32_t( ( float( x ) + 0.5f ) * inv );
}

__device__ __forceinline__ uint32_t line_base( const axis_desc &a, uint32_t line )
{
    if ( a.mode == 0 ) return line * a.Nx;
    if ( a.mode == 1 ) return ( line / a.Nx ) * a.Nx * a.Ny + ( line % a.Nx );
    return line;
}

// One mixed-radix stage, decimation in frequency: from lines of n = r m entries
// at stride s (n s = L), output q + s (r p + k) is
//   sum_j in[ q + s (p + m j) ] w_L^( s k (p + m j) ),   w_L = exp(-2 pi i / L).
// One output a thread: r cmuls, where a direct DFT of the line takes L (at 100
// points 14 instead of 100).  R: r where it is 2 to 5, 0 else, four terms at a time:
// one waits for its twiddle (3000 points, direct, there and back 2.61 -> 2.23 ms).
template <int R>
__device__ __forceinline__ void mixed_stage( const double2 *in, double2 *out, const axis_desc &a, const double2 *tw,
                                             bool inverse, uint32_t r_, uint32_t s )
{
    const uint32_t L = a.L, r = R > 0 ? uint32_t( R ) : r_, Lr = L / r;
    const float invL = 1.0f / float( L ), invs = 1.0f / float( s ), invr = 1.0f / float( r );
    for ( uint32_t e = threadIdx.x; e < a.nlines * L; e += FIELD_BLOCK )
    {
        const uint32_t line = a.nlines > 1 ? div_small( e, invL ) : 0u, o = e - line * L;
        const uint32_t base = line_base( a, line );
        const uint32_t t = div_small( o, invs ), q = o - t * s, p = div_small( t, invr ), k = t - p * r;
        const double2 *x = in + base + ( q + s * p ) * a.S;
        uint32_t m = s * k * p;                                 // below L, and so is the step
        const uint32_t step = Lr * k;
        double2 acc = make_double2( 0.0, 0.0 );
        auto term = [&]( double2 z, bool back, bool swapped ) __attribute__(( always_inline ))
        {
            double2 w = tw[m];
            if ( back ) w.y = -w.y;
            const double2 v = swapped ? cmul( w, z ) : cmul( z, w );
            acc.x += v.x; acc.y += v.y;
            m += step; if ( m >= L ) m -= L;
        };
        const uint32_t hop = Lr * a.S;
        if ( R > 0 )
        {
            #pragma unroll
            for ( uint32_t j = 0; j < uint32_t( R ); ++j ) term( x[ j * hop ], inverse, false );
        }
        else
            #pragma unroll 4
            for ( uint32_t j = 0; j < r; ++j, x += hop ) term( *x, inverse, !inverse );
        out[ base + o * a.S ] = acc;
    }
    __syncthreads();
}

// Transform all lines along one axis; returns the buffer holding the result.
// Inlined: called, it reads LDS by flat loads (a 256-point solve 6 us slower).
__device__ __forceinline__ double2 *fft_axis( double2 *in, double2 *out, const axis_desc &a, const double2 *tw, bool inverse )
{
    const uint32_t L = a.L;
    if ( L <= 1 ) return in;
    if ( a.log2L == 0xffffffffu )
    {
        uint32_t s = 1;
        for ( uint32_t i = 0; s < L; ++i )
        {
            const uint32_t r = a.rad.at( i );
            if ( r == 0 ) break;
            switch ( r )
            {
            case 2:  mixed_stage<2>( in, out, a, tw, inverse, r, s ); break;
            case 3:  mixed_stage<3>( in, out, a, tw, inverse, r, s ); break;
            case 4:  mixed_stage<4>( in, out, a, tw, inverse, r, s ); break;
            case 5:  mixed_stage<5>( in, out, a, tw, inverse, r, s ); break;
            default: mixed_stage<0>( in, out, a, tw, inverse, r, s );
            }
            s *= r;
            double2 *t = in; in = out; out = t;
        }
        return in;
    }
    // Stockham: one radix-2 stage when log2 L is odd, then radix-4 stages
    // (half the barriers of radix 2).  The table holds exp(-2 pi i m/L) for
    // m < L/2; m >= L/2 reads -tw[m - L/2].
    auto twid = [&]( uint32_t m )
    {
        const uint32_t hl = L >> 1;
        double2 w = m < hl ? tw[m] : make_double2( -tw[m - hl].x, -tw[m - hl].y );
        if ( inverse ) w.y = -w.y;
        return w;
    };
    uint32_t Ns = 1, log2Ns = 0;
    if ( a.log2L & 1u )
    {
        const uint32_t half = L >> 1, lh = a.log2L - 1;
        for ( uint32_t e = threadIdx.x; e < a.nlines * half; e += FIELD_BLOCK )
        {
            const uint32_t line = e >> lh, j = e & ( half - 1 );
            const uint32_t base = line_base( a, line );
            const double2 x0 = in[ base + j*a.S ], x1 = in[ base + ( j + half )*a.S ];   // Ns = 1: no twiddle
            out[ base + ( 2*j )*a.S ]     = make_double2( x0.x + x1.x, x0.y + x1.y );
            out[ base + ( 2*j + 1 )*a.S ] = make_double2( x0.x - x1.x, x0.y - x1.y );
        }
        __syncthreads();
        double2 *t = in; in = out; out = t;
        Ns = 2; log2Ns = 1;
    }
    const uint32_t quarter = L >> 2, lq = a.log2L - 2;
    for ( ; Ns < L; Ns <<= 2, log2Ns += 2 )
    {
        const uint32_t twstep = L >> ( log2Ns + 2 );       // L / (4 Ns)
        for ( uint32_t e = threadIdx.x; e < a.nlines * quarter; e += FIELD_BLOCK )
        {
            const uint32_t line = e >> lq, j = e & ( quarter - 1 );
            const uint32_t base = line_base( a, line );
            const uint32_t k = j & ( Ns - 1 );
            const double2 b0 = in[ base + j*a.S ];
            const double2 b1 = cmul( in[ base + ( j + quarter )*a.S ],     twid( k * twstep ) );
            const double2 b2 = cmul( in[ base + ( j + 2*quarter )*a.S ],   twid( 2 * k * twstep ) );
            const double2 b3 = cmul( in[ base + ( j + 3*quarter )*a.S ],   twid( 3 * k * twstep ) );
            const double2 s02 = make_double2( b0.x + b2.x, b0.y + b2.y ), d02 = make_double2( b0.x - b2.x, b0.y - b2.y );
            const double2 s13 = make_double2( b1.x + b3.x, b1.y + b3.y ), d13 = make_double2( b1.x - b3.x, b1.y - b3.y );
            // forward: -i (b1 - b3); inverse: +i (b1 - b3)
            const double2 rot = inverse ? make_double2( -d13.y, d13.x ) : make_double2( d13.y, -d13.x );
            const uint32_t o = ( ( j >> log2Ns ) << ( log2Ns + 2 ) ) + k;
            out[ base + o*a.S ]            = make_double2( s02.x + s13.x, s02.y + s13.y );
            out[ base + ( o + Ns )*a.S ]   = make_double2( d02.x + rot.x, d02.y + rot.y );
            out[ base + ( o + 2*Ns )*a.S ] = make_double2( s02.x - s13.x, s02.y - s13.y );
            out[ base + ( o + 3*Ns )*a.S ] = make_double2( d02.x - rot.x, d02.y - rot.y );
        }
        __syncthreads();
        double2 *t = in; in = out; out = t;
    }
    return in;
}

} // namespace nufi_impl

#endif
