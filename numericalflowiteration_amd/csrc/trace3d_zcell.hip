// trace3d_zcell.hip — the fast FP64 3D trace (rho and metrics): z-cell
// polynomials in LDS.
//
// The reference's node step (dim3::eval_ftilda, nufi/rho.hpp:318-367; eval_f
// with the initial half-kick, rho.hpp:369-426) evaluates grad phi from the
// 4x4x4 window of a node's cell.  FP64 VALU issue bounds it (4.7 clocks a wave
// instruction), so this kernel cuts the instructions: along z the spline of
// every (y, x) column is a cubic polynomial of the cell, whose value and slope
// together take 5 FMAs (Horner, both at once) where the two bases take 8, and
// no z basis has to be formed:
//   V_ij = a0 + t (a1 + t (a2 + t a3)),  W_ij = V_ij'(t)          (80 FMA)
//   A_j = sum_i V_ij Bx_i, X_j = sum_i V_ij Dx_i, Z_j = sum_i W_ij Bx_i  (48)
//   gx = sum_j X_j By_j, gy = sum_j A_j Dy_j, gz = sum_j Z_j By_j        (12)
// 140 FMA instead of 188, and two aligned 16-byte LDS reads a column.
//
// Polynomials of a whole slice take four times its bytes, more than the LDS
// (185 KB at 16^3).  But nodes of one z plane and one z velocity drift through
// z together (to the difference of their z kicks): a workgroup holds the nodes
// of one (z, w) and keeps the polynomials of `nzc` z-cells only, following the
// drift.  Per slice it copies the nzc + 3 coefficient planes of that window
// (direct global->LDS loads) and every thread turns columns into polynomials
// (9 VALU a cell, ~2% of the step at eight nodes a lane).  The pipeline runs
// over (pass, slice): planes of item i+2 are copied and those of item i+1
// turned into polynomials while item i is traced, one barrier an item.  The
// window of an item is predicted from where the workgroup's first node was two
// items before.  A node whose z-cell lies outside the window (strong, uneven
// z kicks) forms the same polynomials from the global history instead: slower,
// the same bits.  A workgroup that meets too many such nodes gives up and marks
// itself, and trace3d_zslice_kernel, launched behind, redoes the marked ones
// from the 4x4x4 windows of whole coefficient slices in LDS.  Which ones those
// are follows from the history alone: the workgroups have one shape, whatever
// the launch shape asked for or the slab of a call.
//
// Measured, window kernel -> this one: 16^3 x 32^3 at n = 80 107.5 -> 82 ms;
// 20x18x20 x 24^3 at n = 24 30.9 -> 16.4 ms (its window kernel had one LDS
// buffer and no compiled strides); metrics of 16^3 x 16^3 at n = 40 19.7 -> 5.8
// ms (they ran the strict layout's wave tasks).  z-cells: three instead of four
// 0.6% slower; two columns read ahead no faster; without the scheduling
// barriers 6% slower.  Fields that mix x, y and z (a product of waves
// beside separable ones, n = 60, 24^3 velocities) are traced from z-cells while
// that pays and from whole slices past it, decided per call (below): 16^3 mixing by
// 0.1 of the field 38.5 -> 32.0 ms, 0.4 47.5 -> 47.3 (by marks alone 77), 2.0 60.9 ->
// 60.7 (72); 20^3 0.1 141 -> 98, 0.2 145 -> 138 (182), 2.0 162 -> 157.
#include "device_common.hpp"
#include "internal.hpp"
#include "step3d.hpp"
#include "cell_index.hpp"

#include <stddef.h>
#include <type_traits>

namespace nufi_impl
{

using namespace nufi_dev;

namespace
{

typedef double d2_t __attribute__(( ext_vector_type( 2 ) ));
using lds_d2 = const __attribute__(( address_space( 3 ) )) d2_t *;

// the (a2, a3) pairs lie this many bytes above the (a0, a1) pairs: a constant
// the LDS reads take as an immediate
constexpr uint32_t PAIR2 = ZCELL_PAIR2;

// polynomial of 6 x the spline of a column in one cell, from its four coefficients
__device__ __forceinline__ void column_poly( double c0, double c1, double c2, double c3, double &a0, double &a1,
                                             double &a2, double &a3 )
{
    const double e = c0 + c2, d = c2 - c0;
    a0 = fma( 4.0, c1, e );
    a1 = 3.0 * d;
    a2 = fma( -6.0, c1, 3.0 * e );
    a3 = fma( 3.0, c1 - c2, c3 - c0 );
}

// a value taken under a branch as it is: without this the compiler selects
// among the addresses of a lane's nodes, which puts them in memory
__device__ __forceinline__ double held( double v )
{
    asm volatile( "" : "+v"( v ) );
    return v;
}

struct zlane
{
    uint32_t l, ix, iy, g;     // spatial point, its x and y, velocity group
    bool on, ok;               // has nodes of the grid, and of the launch's slab
};

// velocity k of the lane's group: u, v (w is the workgroup's) and whether the node is traced
__device__ __forceinline__ bool zc_velocity( const trace3_params &p, const zlane &a, uint32_t iw, uint32_t k, double &u, double &v )
{
    const uint32_t uv = p.Nu * p.Nv, i = a.g * p.zc.vg + k;
    const bool in = a.on && k < p.zc.vg && i < uv;
    const uint32_t ic = in ? i : 0u, iu = ic % p.Nu, ivv = ic / p.Nu;
    u = p.u_min + iu  * p.du + p.du / 2;           // cuda_kernel.cu:402-418
    v = p.v_min + ivv * p.dv + p.dv / 2;
    const uint64_t q = uint64_t( a.l ) * ( uint64_t( uv ) * p.Nw ) + uint64_t( iw ) * uv + ic;
    return in && a.ok && q >= p.q_begin && q < p.q_end;
}

// grad phi of one node (6x6 scaled in x, y; gz three times that of the window
// kernel, its kick constant a third): the columns come from `column(jj, ii)`,
// one ahead of the FMAs that use them
template <typename COL>
__device__ __forceinline__ void zc_gradient( COL column, double tx, double ty, double tz, double &gx, double &gy, double &gz )
{
    double c[2][4];
    column( 0, c[0] );
    __builtin_amdgcn_sched_barrier( 0 );
    double Bx[4], Dx[4], By[4], Dy[4];
    cubic_bases_x6( tx, Bx, Dx );
    cubic_bases_x6( ty, By, Dy );
    double A = 0, X = 0, Z = 0;
    #pragma unroll
    for ( int idx = 0; idx < 16; ++idx )
    {
        if ( idx + 1 < 16 ) column( idx + 1, c[ ( idx + 1 ) & 1 ] );
        __builtin_amdgcn_sched_barrier( 0 );
        const double *a = c[ idx & 1 ];
        const int ii = idx & 3, jj = idx >> 2;
        const double b = fma( a[3], tz, a[2] ), s = fma( b, tz, a[1] );
        const double W = fma( fma( a[3], tz, b ), tz, s ), V = fma( s, tz, a[0] );
        A = ii == 0 ? V * Bx[0] : fma( V, Bx[ii], A );
        X = ii == 0 ? V * Dx[0] : fma( V, Dx[ii], X );
        Z = ii == 0 ? W * Bx[0] : fma( W, Bx[ii], Z );
        if ( ii == 3 )
        {
            gx = jj == 0 ? X * By[0] : fma( X, By[jj], gx );
            gy = jj == 0 ? A * Dy[0] : fma( A, Dy[jj], gy );
            gz = jj == 0 ? Z * By[0] : fma( Z, By[jj], gz );
        }
    }
}

// The per-axis constants where they are used: read from the kernel arguments
// through a pointer the compiler cannot see through, so that it does not hold
// all of them in scalar registers for the whole kernel and spill those to
// vector lanes (18 v_readlane a node-step).
using arg_consts = const __attribute__(( address_space( 4 ) )) zcell_consts *;
__device__ __forceinline__ arg_consts zc_consts()
{
    auto a = (const __attribute__(( address_space( 4 ) )) char *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile( "" : "+s"( a ) );
    return (arg_consts)( a + offsetof( trace3_params, zc ) + offsetof( zcell_plan, k ) );
}

// workgroup -> (velocity-group block, tile, w, z); thread -> (point, group)
struct zplace
{
    zlane a;
    uint32_t iw, iz, P;
    double w0, z0;
};
__device__ __forceinline__ zplace zc_place( const trace3_params &p, uint32_t b = blockIdx.x, uint32_t thread = threadIdx.x )
{
    zplace t;
    asm volatile( "" : "+v"( thread ) );        // formed anew where it is used: nothing of it stays in registers
    const uint32_t gb = b % p.zc.ngb; b /= p.zc.ngb;
    const uint32_t tile = b % p.zc.tiles; b /= p.zc.tiles;
    t.iw = b % p.Nw; t.iz = p.zc.z_first + b / p.Nw;
    t.P = p.Nx * p.Ny;
    const uint32_t gl = thread / p.zc.tw, pt = tile * p.zc.tw + ( thread - gl * p.zc.tw );
    t.a.g = gb * p.zc.gpw + gl;
    const uint32_t pc = pt < t.P ? pt : t.P - 1;
    t.a.ix = pc % p.Nx; t.a.iy = pc / p.Nx; t.a.l = t.iz * t.P + pc;
    t.a.on = gl < p.zc.gpw && t.a.g < p.zc.ngw && pt < t.P;
    if ( !t.a.on ) t.a.g = 0;
    // points outside a launch's slab are traced all the same: which workgroups
    // are marked does not depend on how a caller cuts the nodes
    t.a.ok = t.a.on && t.a.l >= p.l_first && t.a.l < p.l_first + p.n_count;
    t.w0 = p.w_min + t.iw * p.dw + p.dw / 2; t.z0 = double( t.iz );
    return t;
}

// items of a pass (slices from the highest down) and the slice of one
template <int MODE>
__device__ __forceinline__ int zc_items( const trace3_params &p )
{
    return MODE == MODE_METRICS ? ( p.n > 0 ? int( p.n ) + 1 : 0 ) : int( p.n );
}
template <int MODE>
__device__ __forceinline__ int zc_slice( const trace3_params &p, int k )
{
    return MODE == MODE_METRICS ? int( p.n ) - k : int( p.n ) - 1 - k;
}

// f of one node at its foot, added to the lane's sums
template <int MODE, int NM>
__device__ __forceinline__ void zc_add( const trace3_params &p, const zplace &t, uint32_t k, double x, double y, double z,
                                        double u, double v, double w, csum acc[NM] )
{
    double u0, v0;
    const bool act = zc_velocity( p, t.a, t.iw, k, u0, v0 );
    const double f = act ? f0_3d( p.f0, p.x_min + x*p.dx, p.y_min + y*p.dy, p.z_min + z*p.dz, u, v, w ) : 0.0;
    if ( MODE == MODE_RHO ) acc[0] = csum_add( acc[0], csum { f, 0.0 } );
    else
    {
        // the four metric integrands (cuda_kernel.cu:453-465)
        const double wt = p.weight, v2 = u0*u0 + v0*v0 + t.w0*t.w0;
        acc[0] = csum_add( acc[0], csum { wt*f, 0.0 } );
        acc[NM > 1 ? 1 : 0] = csum_add( acc[NM > 1 ? 1 : 0], csum { wt*f*f, 0.0 } );
        acc[NM > 2 ? 2 : 0] = csum_add( acc[NM > 2 ? 2 : 0], csum { wt*v2*f/2, 0.0 } );
        acc[NM > 3 ? 3 : 0] = csum_add( acc[NM > 3 ? 3 : 0], csum { ( act && f > 0 ) ? -wt*f*log(f) : 0.0, 0.0 } );
    }
}

template <int MODE, int NM>
__device__ __forceinline__ void zc_write( const trace3_params &p, const zplace &t, const csum acc[NM] )
{
    if ( MODE == MODE_RHO )
    {
        if ( t.a.ok ) p.partials[ size_t( t.iw * p.zc.ngw + t.a.g ) * ( size_t( t.P ) * p.Nz ) + t.a.l ] = acc[0].s + acc[0].c;
        return;
    }
    #pragma unroll
    for ( int k = 0; k < NM; ++k )
    {
        const csum v = wave_csum( acc[k] );
        if ( threadIdx.x % WAVE == 0 )
            p.partials[ ( size_t( blockIdx.x ) * ( blockDim.x / WAVE ) + threadIdx.x / WAVE ) * 4 + k ] = v.s + v.c;
    }
}

// G: compile-time edge of a cubic power-of-two grid (row offsets are then
// immediates), 0 for any grid; MASK: power-of-two axes (advance_axis)
template <bool MASK, int G, int MODE>
__global__ __launch_bounds__( 512 ) __attribute__(( amdgpu_waves_per_eu( 2, 2 ) ))
void trace3d_zcell_kernel( trace3_params p )
{
    extern __shared__ __align__( 16 ) char zlds[];
    constexpr int NPT = 8;                                            // nodes a lane
    if ( p.zc.route != nullptr && p.zc.route->window != 0 )
    {
        if ( threadIdx.x == 0 ) p.zc.marks[ blockIdx.x ] = p.zc.flag_mark;
        return;
    }
    const uint32_t tid = threadIdx.x, lane = tid % WAVE, threads = blockDim.x;
    const uint32_t wave = __builtin_amdgcn_readfirstlane( tid / WAVE ), waves = threads / WAVE;
    const uint32_t nzc = p.zc.nzc, plane = G > 0 ? uint32_t( ( G + 3 ) * ( G + 3 ) ) : p.sz;
    const uint32_t sy = G > 0 ? uint32_t( G + 3 ) : p.sy, Nx = G > 0 ? uint32_t( G ) : p.Nx;
    const uint32_t rows = G > 0 ? uint32_t( G + 3 ) : p.Ny + 3, cols = rows * Nx;       // polynomials of one z-cell
    const uint32_t lds0 = uint32_t( reinterpret_cast<uintptr_t>( (__attribute__(( address_space( 3 ) )) char *)zlds ) );
    const uint32_t pp_bytes = nzc * cols * 16u, szp = p.zc.szp, c_doubles = ( nzc + 3 ) * szp;
    double *const cbuf = reinterpret_cast<double*>( zlds + PAIR2 + 2 * pp_bytes );
    double *const rep  = cbuf + 2 * c_doubles;                       // the first node's z and w after odd / even items
    volatile uint32_t *const give_up = reinterpret_cast<volatile uint32_t*>( rep + 4 );

    const int Nyi = G > 0 ? G : int( p.Ny ), Nzi = G > 0 ? G : int( p.Nz );
    const int S = zc_items<MODE>( p );
    const int passes = int( ( p.zc.vg + NPT - 1 ) / NPT );
    const int T = passes * S;
    auto slice_of = [&]( int k ) { return zc_slice<MODE>( p, k ); };

    // first z-cell of the window around z (any multiple of Nz away)
    const double zoff = 0.5 * ( double( nzc ) - 1.0 );
    auto window = [&]( double z ) __attribute__(( always_inline )) -> int
    {
        const arg_consts k3 = zc_consts();
        z -= zoff;
        z = fma( -k3->N[2], floor( z * k3->iN[2] ), z );
        const int c = int( z );
        return __builtin_amdgcn_readfirstlane( c < 0 ? 0 : ( c >= Nzi ? Nzi - 1 : c ) );
    };
    // item k of a pass from its start: so many drifts at the node velocity
    auto start_window = [&]( int k ) __attribute__(( always_inline ))
    {
        const zplace t = zc_place( p );
        return window( fma( -double( MODE == MODE_METRICS ? k : k + 1 ) * zc_consts()->cd[2], t.w0, t.z0 ) );
    };

    auto plane_of = [&]( int zb, uint32_t q ) { uint32_t r = uint32_t( zb ) + q; return r > p.Nz + 2 ? r - p.Nz : r; };
    // the nzc + 3 planes of the window, each as the 16-byte words that cover it
    auto copy_planes = [&]( double *dst, int m, int zb ) __attribute__(( always_inline ))
    {
        const double *src = p.hist + size_t( m ) * p.st;
        const uint32_t d0 = uint32_t( reinterpret_cast<uintptr_t>( (__attribute__(( address_space( 3 ) )) char *)dst ) );
        for ( uint32_t q = wave; q < nzc + 3; q += waves )               // a wave takes whole planes
        {
            const uint32_t off = plane_of( zb, q ) * plane, mis = ( uint32_t( m ) * p.st + off ) & 1u;
            const uint32_t n16 = ( plane + mis + 1 ) / 2;
            const char *g = reinterpret_cast<const char*>( src + off - mis );
            uint32_t d = d0 + q * szp * 8u;
            for ( uint32_t w = 0; w < n16; w += WAVE, d += 1024u )
                if ( w + lane < n16 ) dma_issue16( g + size_t( w + lane ) * 16, d );
        }
    };
    auto convert = [&]( uint32_t pp, const double *src, int m, int zb ) __attribute__(( always_inline ))
    {
        uint32_t at[ ZCELL_MAX + 3 ];
        #pragma unroll
        for ( uint32_t q = 0; q < ZCELL_MAX + 3; ++q )
        {
            const uint32_t qc = q < nzc + 3 ? q : nzc + 2;
            at[q] = qc * szp + ( ( uint32_t( m ) * p.st + plane_of( zb, qc ) * plane ) & 1u );
        }
        for ( uint32_t c = tid; c < cols; c += threads )
        {
            const uint32_t y = G > 0 ? c / uint32_t( G > 0 ? G : 1 ) : ( c * p.zc.inv_nx ) >> 20;    // c / Nx (c Nx < 2^20)
            const uint32_t from = c + y * ( sy - Nx );                       // y * sy + x
            double v[ ZCELL_MAX + 3 ];
            #pragma unroll
            for ( uint32_t q = 0; q < ZCELL_MAX + 3; ++q ) v[q] = src[ at[q] + from ];
            #pragma unroll
            for ( uint32_t s = 0; s < ZCELL_MAX; ++s )
                if ( s < nzc )
                {
                    double2 lo, hi;
                    column_poly( v[s], v[s+1], v[s+2], v[s+3], lo.x, lo.y, hi.x, hi.y );
                    char *d = zlds + pp + ( s * cols + c ) * 16u;
                    *reinterpret_cast<double2*>( d ) = lo;
                    *reinterpret_cast<double2*>( d + PAIR2 ) = hi;
                }
        }
    };

    double sx[NPT], sy_[NPT], sz_[NPT], vu[NPT], vv[NPT], vw[NPT];
    constexpr int NM = MODE == MODE_METRICS ? 4 : 1;
    csum acc[NM];
    #pragma unroll
    for ( int k = 0; k < NM; ++k ) acc[k] = csum { 0.0, 0.0 };

    auto start = [&]( int pass ) __attribute__(( always_inline ))
    {
        const zplace t = zc_place( p );
        #pragma unroll
        for ( int r = 0; r < NPT; ++r )
        {
            (void)zc_velocity( p, t.a, t.iw, uint32_t( pass * NPT + r ), vu[r], vv[r] );
            vw[r] = t.w0;
            sx[r] = double( t.a.ix ); sy_[r] = double( t.a.iy ); sz_[r] = t.z0;
        }
    };
    // node r of the lane, r uniform but not a constant (rolled loops, one body):
    // spelled out with constant indices, or the arrays end up in memory
    auto at_node = [&]( int r, auto &&f ) __attribute__(( always_inline ))
    {
        if ( r == 0 ) f( std::integral_constant<int, 0>() );
        if ( r == 1 ) f( std::integral_constant<int, 1>() );
        if ( r == 2 ) f( std::integral_constant<int, 2>() );
        if ( r == 3 ) f( std::integral_constant<int, 3>() );
        if ( r == 4 ) f( std::integral_constant<int, 4>() );
        if ( r == 5 ) f( std::integral_constant<int, 5>() );
        if ( r == 6 ) f( std::integral_constant<int, 6>() );
        if ( r == 7 ) f( std::integral_constant<int, 7>() );
    };
    auto finish = [&]( int pass ) __attribute__(( always_inline ))
    {
        const zplace t = zc_place( p );
        #pragma unroll 1
        for ( int r = 0; r < NPT; ++r )
        {
            double x = 0, y = 0, z = 0, u = 0, v = 0, w = 0;
            at_node( r, [&]( auto q ) __attribute__(( always_inline ))
                     { x = held( sx[q] ); y = held( sy_[q] ); z = held( sz_[q] ); u = held( vu[q] ); v = held( vv[q] ); w = held( vw[q] ); } );
            zc_add<MODE,NM>( p, t, uint32_t( pass * NPT + r ), x, y, z, u, v, w, acc );
        }
    };

    // node-steps of this wave that went to the global history.  64 scattered
    // loads make one about 13 times as dear as in the window, a step of the
    // whole-slice kernel 1.5 times: past one in 16 (and a few to begin with)
    // the workgroup is better off there, and the sooner it goes the better.
    int missed = 0;

    // one item: all nodes of the lane through slice m
    auto trace = [&]( uint32_t pp, int m, int zb, bool still ) __attribute__(( always_inline ))
    {
        const bool half = m == 0 || still;
        const arg_consts k3 = zc_consts();
        const double cdx = k3->cd[0], cdy = k3->cd[1], cdz = k3->cd[2];
        const auto kk = half ? k3->kickh : k3->kick;
        const double kx_ = kk[0], ky_ = kk[1], kz_ = kk[2];
        if ( MASK && !still && wrap3_due( m ) )
        {
            const arg_consts kw = zc_consts();
            #pragma unroll
            for ( int r = 0; r < NPT; ++r )
            {
                rewrap3( sx[r], kw->N[0], kw->iN[0] ); rewrap3( sy_[r], kw->N[1], kw->iN[1] ); rewrap3( sz_[r], kw->N[2], kw->iN[2] );
            }
        }
        // wrapped every step otherwise (MASK needs none of these)
        double Nd[3] = { 0, 0, 0 }, iN[3] = { 0, 0, 0 };
        if ( !MASK )
        {
            Nd[0] = k3->N[0]; Nd[1] = k3->N[1]; Nd[2] = k3->N[2];
            iN[0] = k3->iN[0]; iN[1] = k3->iN[1]; iN[2] = k3->iN[2];
        }
        // z first: the drift and the cell within the window, for all nodes
        uint32_t rel[NPT], worst = 0;
        #pragma unroll
        for ( int r = 0; r < NPT; ++r )
        {
            double z = still ? sz_[r] : fma( -cdz, vw[r], sz_[r] );
            if ( !MASK ) z = fma( -Nd[2], floor( z * iN[2] ), z );
            sz_[r] = z;
            rel[r] = zc_rel<MASK>( int( floor( z ) ), zb, Nzi );
            worst = worst > rel[r] ? worst : rel[r];
        }
        auto node = [&]( double &x, double &y, double z, double &u, double &v, double &w, uint32_t rl, bool local )
            __attribute__(( always_inline ))
        {
            double tx, ty;
            const int i = advance_axis<MASK>( x, u, cdx, Nd[0], iN[0], int( Nx ), tx, still );
            const int j = advance_axis<MASK>( y, v, cdy, Nd[1], iN[1], Nyi, ty, still );
            const double tz = __builtin_amdgcn_fract( z );
            double gx, gy, gz;
            if ( local )
            {
                // row j of cell rl; the four columns wrap around the row
                const uint32_t row = pp + ( __umul24( __umul24( rl, rows ) + uint32_t( j ), Nx ) ) * 16u;
                uint32_t at[4];
                #pragma unroll
                for ( uint32_t ii = 0; ii < 4; ++ii )
                {
                    const uint32_t t = uint32_t( i ) + ii;
                    if ( G > 0 ) at[ii] = ( ( t * 16u ) & ( uint32_t( G ) * 16u - 16u ) ) | row;     // rows start on their own size
                    else at[ii] = row + ( t < t - Nx ? t : t - Nx ) * 16u;                           // t < Nx: t - Nx wraps up
                }
                zc_gradient( [&]( int idx, double c[4] )
                {
                    const lds_d2 q = (lds_d2)size_t( at[ idx & 3 ] + uint32_t( idx >> 2 ) * Nx * 16u );
                    const d2_t lo = *q, hi = q[ PAIR2 / 16 ];
                    c[0] = lo.x; c[1] = lo.y; c[2] = hi.x; c[3] = hi.y;
                }, tx, ty, tz, gx, gy, gz );
            }
            else
            {
                // global memory: whatever the position, a cell of the slice
                const double *h = p.hist + size_t( m ) * p.st + size_t( zc_cell( zb, rl, p.Nz ) ) * plane +
                                  zc_held( j, uint32_t( Nyi ) ) * sy + zc_held( i, Nx );
                zc_gradient( [&]( int idx, double c[4] )
                {
                    const double *q = h + uint32_t( idx >> 2 ) * sy + uint32_t( idx & 3 );
                    column_poly( q[0], q[plane], q[2*size_t( plane )], q[3*size_t( plane )], c[0], c[1], c[2], c[3] );
                }, tx, ty, tz, gx, gy, gz );
            }
            u = fma( kx_, gx, u );
            v = fma( ky_, gy, v );
            w = fma( kz_, gz, w );
        };
        if ( __builtin_expect( __builtin_amdgcn_ballot_w64( worst >= nzc ) == 0, 1 ) )
        {
            #pragma unroll
            for ( int r = 0; r < NPT; ++r ) node( sx[r], sy_[r], sz_[r], vu[r], vv[r], vw[r], rel[r], true );
        }
        else
        {
            // some node left the window: one at a time, from the global history where any lane did
            #pragma unroll 1
            for ( int r = 0; r < NPT; ++r )
            {
                double x = 0, y = 0, z = 0, u = 0, v = 0, w = 0;
                uint32_t rl = 0;
                at_node( r, [&]( auto q ) __attribute__(( always_inline ))
                         { x = held( sx[q] ); y = held( sy_[q] ); z = held( sz_[q] ); u = held( vu[q] ); v = held( vv[q] ); w = held( vw[q] ); rl = rel[q]; } );
                if ( __builtin_amdgcn_ballot_w64( rl >= nzc ) == 0 ) node( x, y, z, u, v, w, rl, true );
                else { node( x, y, z, u, v, w, rl, false ); ++missed; }
                at_node( r, [&]( auto q ) __attribute__(( always_inline ))
                         { sx[q] = x; sy_[q] = y; vu[q] = u; vv[q] = v; vw[q] = w; } );
            }
        }
    };

    int zb0 = 0, zb1 = 0, zb2 = 0;
    if ( S > 0 )
    {
        zb0 = start_window( 0 ); zb1 = start_window( 1 % S );
        copy_planes( cbuf, slice_of( 0 ), zb0 );
        if ( T > 1 ) copy_planes( cbuf + c_doubles, slice_of( 1 % S ), zb1 );
        dma_publish();
    }
    if ( S > 0 )
    {
        convert( 0u, cbuf, slice_of( 0 ), zb0 );
        __syncthreads();
    }
    if ( tid == 0 ) *give_up = 0;                                    // read after many barriers
    int i = 0;
    for ( int pass = 0; pass < passes; ++pass )
    {
        start( pass );
        for ( int k = 0; k < S; ++k, ++i )
        {
            const uint32_t odd = uint32_t( i ) & 1u;
            const int k1 = k + 1 < S ? k + 1 : 0, k2 = k1 + 1 < S ? k1 + 1 : 0;
            if ( i + 2 < T )
            {
                // the first node's state after item i-1, three drifts on, where that item is of the same pass
                zb2 = ( k >= 1 && k + 2 < S )
                    ? window( fma( -3.0 * zc_consts()->cd[2], rep[ 2 * ( odd ^ 1u ) + 1 ], rep[ 2 * ( odd ^ 1u ) ] ) ) : start_window( k2 );
                copy_planes( cbuf + odd * c_doubles, slice_of( k2 ), zb2 );
            }
            if ( i + 1 < T ) convert( ( odd ^ 1u ) * pp_bytes, cbuf + ( odd ^ 1u ) * c_doubles, slice_of( k1 ), zb1 );
            trace( lds0 + odd * pp_bytes, slice_of( k ), zb0, MODE == MODE_METRICS && k == 0 );
            if ( tid == 0 ) { rep[ 2 * odd ] = sz_[0]; rep[ 2 * odd + 1 ] = vw[0]; }
            if ( ( i & 3 ) == 2 && lane == 0 && missed > 8 + i * NPT / 16 ) *give_up = 1;
            dma_publish();
            if ( ( i & 3 ) == 3 && *give_up != 0 )                    // set before the last barrier but one, next after another
            {
                if ( tid == 0 ) p.zc.marks[ blockIdx.x ] = 1;
                return;
            }
            zb0 = zb1; zb1 = zb2;
        }
        finish( pass );
    }
    if ( tid == 0 ) p.zc.marks[ blockIdx.x ] = 0;

    zc_write<MODE,NM>( p, zc_place( p ), acc );
}

// The workgroups trace3d_zcell_kernel marked, by the window kernel's step
// (step3_fast) from whole coefficient slices in LDS: two, or one where two do
// not fit.
template <bool MASK, int G, int MODE>
__global__ __launch_bounds__( 512 ) __attribute__(( amdgpu_waves_per_eu( 2, 2 ) ))
void trace3d_zslice_kernel( trace3_params p )
{
    extern __shared__ __align__( 16 ) double zfull[];
    if ( p.zc.marks[ blockIdx.x ] == 0 ) return;                      // uniform
    constexpr int NPT = 4, NM = MODE == MODE_METRICS ? 4 : 1;
    const uint32_t waves = blockDim.x / WAVE, st = p.st;
    const fast3_consts k3 = make_fast3( p );
    const int S = zc_items<MODE>( p ), passes = int( ( p.zc.vg + NPT - 1 ) / NPT ), T = passes * S;
    auto buffer = [&]( int i ) __attribute__(( always_inline )) { return zfull + ( ( i & 1 ) && p.dma ? st + 2u : 0u ); };
    auto copy = [&]( int i, int m ) __attribute__(( always_inline ))
    {
        const double *src = p.hist + size_t( m ) * st;
        const uint32_t mis = uint32_t( reinterpret_cast<uintptr_t>( src ) & 15u ) / 8u;
        dma_copy16( buffer( i ), src - mis, ( st + mis + 1 ) / 2, waves );
    };
    csum acc[NM];
    #pragma unroll
    for ( int k = 0; k < NM; ++k ) acc[k] = csum { 0.0, 0.0 };
    double sx[NPT], sy_[NPT], sz_[NPT], vu[NPT], vv[NPT], vw[NPT];
    if ( p.dma && T > 0 ) { copy( 0, zc_slice<MODE>( p, 0 ) ); dma_publish(); }
    int i = 0;
    for ( int pass = 0; pass < passes; ++pass )
    {
        {
            const zplace t = zc_place( p );
            #pragma unroll
            for ( int r = 0; r < NPT; ++r )
            {
                (void)zc_velocity( p, t.a, t.iw, uint32_t( pass * NPT + r ), vu[r], vv[r] );
                vw[r] = t.w0; sx[r] = double( t.a.ix ); sy_[r] = double( t.a.iy ); sz_[r] = t.z0;
            }
        }
        for ( int k = 0; k < S; ++k, ++i )
        {
            const int m = zc_slice<MODE>( p, k );
            if ( p.dma ) { if ( i + 1 < T ) copy( i + 1, zc_slice<MODE>( p, k + 1 < S ? k + 1 : 0 ) ); }
            else { __syncthreads(); copy( 0, m ); dma_publish(); }
            const double *C = buffer( i ) + ( reinterpret_cast<uintptr_t>( p.hist + size_t( m ) * st ) & 15u ) / 8u;
            const bool still = MODE == MODE_METRICS && k == 0;
            if ( MASK && !still && wrap3_due( m ) )
            {
                #pragma unroll
                for ( int r = 0; r < NPT; ++r )
                {
                    rewrap3( sx[r], k3.Nxd, k3.iNx ); rewrap3( sy_[r], k3.Nyd, k3.iNy ); rewrap3( sz_[r], k3.Nzd, k3.iNz );
                }
            }
            if ( m == 0 || still )
            {
                #pragma unroll
                for ( int r = 0; r < NPT; ++r )
                    step3_fast<MASK,GATHER_PF,G>( k3, C, true, still, sx[r], sy_[r], sz_[r], vu[r], vv[r], vw[r] );
            }
            else
            {
                #pragma unroll
                for ( int r = 0; r < NPT; ++r )
                    step3_fast<MASK,GATHER_PF,G>( k3, C, false, false, sx[r], sy_[r], sz_[r], vu[r], vv[r], vw[r] );
            }
            if ( p.dma ) dma_publish();
        }
        // one body: the inlined f0 is large
        #pragma unroll 1
        for ( int r = 0; r < NPT; ++r )
        {
            zc_add<MODE,NM>( p, zc_place( p ), uint32_t( pass * NPT + r ), sx[0], sy_[0], sz_[0], vu[0], vv[0], vw[0], acc );
            #pragma unroll
            for ( int q = 0; q + 1 < NPT; ++q )               // the next node moves to the front
            { sx[q] = sx[q+1]; sy_[q] = sy_[q+1]; sz_[q] = sz_[q+1]; vu[q] = vu[q+1]; vv[q] = vv[q+1]; vw[q] = vw[q+1]; }
        }
    }
    zc_write<MODE,NM>( p, zc_place( p ), acc );
}

// ---- which kernel traces a call -----------------------------------------------
// The z-cell kernel pays where the nodes of a workgroup keep together in z.  A
// field that mixes the axes strongly drives them apart, and then the marked
// workgroups pay for both kernels: up to twice the time of whole slices alone.
// Two launches ahead of the trace decide from the slices it will read, so that
// the result depends on the history alone and not on earlier calls or on how a
// caller cuts the nodes (6 us together where the first settles it):
//
// trace3d_spread_kernel bounds how far apart two nodes of a workgroup can get
// while their z is about the same: a slice's z kick differs over (x, y) by at
// most the spread of its coefficients' z differences (the spline's slope is a
// convex combination of them), and slice m's kick is followed by m drifts.  The bound
// knows nothing of phases and of the nodes' own motion, and is 3 to 5 times what they
// do: up to ZC_SPREAD_SURE cells (a sum of one wave per axis: 0) hardly one leaves its
// window (cost below 0.01 on every grid tried, the scouts 4% of an 11 x 13 x 9 call).
// With at most ZC_FEW workgroups, where more launches would show,
// it decides alone, at ZC_SPREAD_FEW (8^3 x 12^3 at n = 40, z-cells / whole slices:
// bound 4.2 0.76 / 1.07 ms, 4.6 0.75 / 1.07, 7.0 1.47 / 1.09, 7.7 1.40 / 1.09).
//
// It also looks at the pads of a history that nobody has looked at yet
// (nufi_rho3d_noalloc): z-cells are formed as if the slice went on periodically,
// whole slices are read with their pads.
//
// trace3d_scout_kernel runs where the bound left it open: the
// nodes of one velocity pass of up to ZC_SCOUTS workgroups, a node a lane, from
// whole slices in LDS, counting the wave-steps with a lane outside the window of
// the workgroup's first node.  They step over every second or fourth slice of a
// long history: one node a lane makes the step a bare chain of latencies (3 us).
//
// What a workgroup's misses cost: ZC_MISS_COST times the share of its steps in
// which one of its waves missed (a missed node-step is 13 times as dear, and the
// others wait for it at the barrier), at most ZC_COST_CAP, in units of its trace.
// On average whole slices are worth taking from, in 1/64: 7 at 16^3, where the
// window kernel has its strides compiled in (mixing by 0.15 of the field: cost 0.04,
// 32 ms against its 40; 0.09: 34 / 40; 0.13: 45 / 42), and for windows of two z-cells
// (24 x 20 x 12: 0.01 22 / 26, 0.44 35 / 26); 19 elsewhere (20^3: 0.12 117 / 136,
// 0.27 121 / 136, 0.40 174 / 136; 20 x 18 x 20: 0.23 26 / 30, 0.31 33 / 30).
constexpr unsigned long long ZC_FIX = 65536;                          // sums in 1/65536
constexpr double ZC_SPREAD_SURE = 2.0, ZC_SPREAD_FEW = 5.5;
constexpr uint32_t ZC_SCOUTS = 256, ZC_FEW = 2 * ZC_SCOUTS;
constexpr unsigned long long ZC_MISS_COST = 13, ZC_COST_CAP = 24;     // the cap in 1/16
constexpr unsigned long long ZC_WORTH = 19, ZC_WORTH_CLOSE = 7;
__host__ __device__ inline uint32_t zc_all( const trace3_params &p ) { return p.Nz * p.Nw * p.zc.tiles * p.zc.ngb; }   // workgroups of the grid
__host__ __device__ inline uint32_t scout_stride( uint64_t n ) { return n >= 32 ? 4u : n >= 16 ? 2u : 1u; }

__global__ __launch_bounds__( 1024 )
void trace3d_spread_kernel( trace3_params p )
{
    __shared__ double most_w[16];
    const uint32_t m = blockIdx.x, lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE, P = p.Nx * p.Ny;
    const double *const c = p.hist + size_t( m ) * p.st;
    double most = 0.0;
    bool odd = false;                                                 // not finite: no bound
    for ( uint32_t k = wave; k < p.Nz; k += 16 )
    {
        double lo = __builtin_inf(), hi = -__builtin_inf();
        #pragma unroll 4
        for ( uint32_t e = lane; e < P; e += WAVE )
        {
            const uint32_t y = e / p.Nx, at = k * p.sz + y * p.sy + ( e - y * p.Nx );
            const double d = c[ at + p.sz ] - c[at];
            odd = odd || !( d - d == 0.0 );
            lo = fmin( lo, d ); hi = fmax( hi, d );
        }
        #pragma unroll
        for ( int off = 32; off > 0; off >>= 1 )
        {
            lo = fmin( lo, __shfl_xor( lo, off ) ); hi = fmax( hi, __shfl_xor( hi, off ) );
        }
        most = fmax( most, hi - lo );
    }
    if ( __builtin_amdgcn_ballot_w64( odd ) != 0 ) most = __builtin_inf();
    bool pads = false;
    if ( p.zc.check_pads )                                            // uniform
    {
        const uint32_t sy = p.sy, rows = p.Ny + 3;
        for ( uint32_t e = threadIdx.x; e < p.st; e += 1024 )
        {
            const uint32_t row = e / sy, i = e - row * sy, k = row / rows, j = row - k * rows;
            const uint32_t from = ( k % p.Nz ) * p.sz + ( j % p.Ny ) * sy + i % p.Nx;
            pads = pads || ( from != e && __double_as_longlong( c[e] ) != __double_as_longlong( c[from] ) );
        }
    }
    pads = __syncthreads_or( pads ? 1 : 0 ) != 0;
    if ( lane == 0 ) most_w[wave] = most;
    __syncthreads();
    if ( threadIdx.x != 0 ) return;
    for ( int w = 1; w < 16; ++w ) most = fmax( most, most_w[w] );
    constexpr double CAP = 16777216.0;
    const double cells = most * p.zc.k.cd[2] * p.zc.k.cd[2] * double( m );
    zcell_route *const r = p.zc.route;
    atomicAdd( &r->spread, (unsigned long long)( ( cells < CAP ? cells : CAP ) * double( ZC_FIX ) ) );
    if ( pads ) atomicAdd( &r->odd_pads, 1u );
    __threadfence();
    if ( atomicAdd( &r->arrived[0], 1u ) != gridDim.x - 1 ) return;
    const unsigned long long all = atomicExch( &r->spread, 0ull );
    const uint32_t odd_slices = atomicExch( &r->odd_pads, 0u );
    r->arrived[0] = 0;
    r->last_spread = all; r->last_cost = 0;
    const bool few = zc_all( p ) <= ZC_FEW, open = odd_slices == 0 && zcell_decides( p.zc, p.n, p.Nz );
    r->window = odd_slices != 0 || ( open && few && double( all ) > ZC_SPREAD_FEW * double( ZC_FIX ) ) ? 1u : 0u;
    r->scout = open && !few && double( all ) > ZC_SPREAD_SURE * double( ZC_FIX ) ? 1u : 0u;
}

template <bool MASK, int G>
__global__ __launch_bounds__( 512 ) __attribute__(( amdgpu_waves_per_eu( 2, 2 ) ))
void trace3d_scout_kernel( trace3_params p )
{
    extern __shared__ __align__( 16 ) double zfull[];
    if ( p.zc.route->scout == 0 ) return;                             // uniform
    const uint32_t tid = threadIdx.x, lane = tid % WAVE, wave = tid / WAVE, waves = blockDim.x / WAVE, st = p.st;
    // scattered over the workgroups by golden-ratio steps, and over their passes
    const uint32_t all = zc_all( p );
    const uint32_t b = uint32_t( ( uint64_t( blockIdx.x * 2654435769u ) * all ) >> 32 );
    const uint32_t pass = ( blockIdx.x * 5u ) % ( ( p.zc.vg + 7 ) / 8 );
    // lane 0 of each wave is the workgroup's first node, whose window it is
    const zplace t = zc_place( p, b, lane == 0 ? 0u : tid );
    double x = double( t.a.ix ), y = double( t.a.iy ), z = t.z0, u, v, w = t.w0;
    (void)zc_velocity( p, t.a, t.iw, pass * 8 + ( lane == 0 ? 0u : ( 3 * wave ) % 8 ), u, v );
    fast3_consts k3 = make_fast3( p );
    const int n = int( p.n ), Nzi = int( p.Nz ), stride = int( scout_stride( p.n ) );
    const double ds = double( stride );
    k3.cdx *= ds; k3.cdy *= ds; k3.cdz *= ds; k3.kx *= ds; k3.ky *= ds; k3.kz *= ds;
    const double zoff = 0.5 * ( double( p.zc.nzc ) - 1.0 );
    auto buffer = [&]( int i ) __attribute__(( always_inline )) { return zfull + ( ( i & 1 ) && p.dma ? st + 2u : 0u ); };
    auto copy = [&]( int i, int m ) __attribute__(( always_inline ))
    {
        const double *src = p.hist + size_t( m ) * st;
        const uint32_t mis = uint32_t( reinterpret_cast<uintptr_t>( src ) & 15u ) / 8u;
        dma_copy16( buffer( i ), src - mis, ( st + mis + 1 ) / 2, waves );
    };
    uint32_t missed = 0;
    if ( p.dma ) { copy( 0, n - 1 ); dma_publish(); }
    for ( int i = 0, m = n - 1; m >= 0; ++i, m -= stride )
    {
        if ( p.dma ) { if ( m >= stride ) copy( i + 1, m - stride ); }
        else { __syncthreads(); copy( 0, m ); dma_publish(); }
        const double *C = buffer( i ) + ( reinterpret_cast<uintptr_t>( p.hist + size_t( m ) * st ) & 15u ) / 8u;
        if ( MASK ) { rewrap3( x, k3.Nxd, k3.iNx ); rewrap3( y, k3.Nyd, k3.iNy ); rewrap3( z, k3.Nzd, k3.iNz ); }
        step3_fast<MASK,GATHER_PF,G>( k3, C, false, false, x, y, z, u, v, w );
        double z0 = __shfl( z, 0 ) - zoff;
        z0 = fma( -k3.Nzd, floor( z0 * k3.iNz ), z0 );
        const uint32_t rel = zc_rel<MASK>( int( floor( z ) ), int( zc_held( int( z0 ), uint32_t( Nzi ) ) ), Nzi );
        missed += __builtin_amdgcn_ballot_w64( rel >= p.zc.nzc ) != 0 ? 1u : 0u;
        if ( p.dma ) dma_publish();
    }
    __syncthreads();                                                  // the slices are read
    uint32_t *const per_wave = reinterpret_cast<uint32_t*>( zfull );
    if ( lane == 0 ) per_wave[wave] = missed;
    __syncthreads();
    if ( tid != 0 ) return;
    unsigned long long out = 0;
    for ( uint32_t q = 0; q < waves; ++q ) out += per_wave[q];
    const unsigned long long steps = ( p.n + stride - 1 ) / stride, cap = ZC_COST_CAP * ZC_FIX / 16;
    unsigned long long cost = ZC_MISS_COST * ZC_FIX * out / steps;
    if ( cost > cap ) cost = cap;
    zcell_route *const r = p.zc.route;
    atomicAdd( &r->cost, cost );
    __threadfence();
    if ( atomicAdd( &r->arrived[1], 1u ) != gridDim.x - 1 ) return;
    const unsigned long long mean = atomicExch( &r->cost, 0ull ) / gridDim.x;
    r->arrived[1] = 0;
    r->last_cost = mean;
    const unsigned long long worth = G == 16 || p.zc.nzc < 3 ? ZC_WORTH_CLOSE : ZC_WORTH;
    r->window = mean > worth * ZC_FIX / 64 ? 1u : 0u;
}

template <int MODE>
const void *zslice_kernel( bool mask, bool g16 )
{
    if ( g16 )  return reinterpret_cast<const void*>( trace3d_zslice_kernel<true,16,MODE> );
    if ( mask ) return reinterpret_cast<const void*>( trace3d_zslice_kernel<true,0,MODE> );
    return reinterpret_cast<const void*>( trace3d_zslice_kernel<false,0,MODE> );
}

template <int MODE>
const void *zcell_kernel( bool mask, bool g16 )
{
    if ( g16 )  return reinterpret_cast<const void*>( trace3d_zcell_kernel<true,16,MODE> );
    if ( mask ) return reinterpret_cast<const void*>( trace3d_zcell_kernel<true,0,MODE> );
    return reinterpret_cast<const void*>( trace3d_zcell_kernel<false,0,MODE> );
}

// the z-cells whose two polynomial buffers and two plane buffers fit, 0 if not even two do
uint32_t zcell_cells( uint32_t cols, uint32_t szp, uint32_t Nz )
{
    for ( uint32_t c = std::min( ZCELL_MAX, Nz ); c >= std::min( 2u, Nz ); --c )
        if ( 2u * c * cols * 16u <= PAIR2 && zcell_lds( c, cols, szp ) <= 160u * 1024u ) return c;
    return 0;
}

} // namespace

size_t zcell_workgroups( const nufi_config &g, const zcell_plan &z, uint32_t *waves )
{
    uint32_t tw = 1, gpw = 1;
    const uint32_t P = uint32_t( g.Nx * g.Ny );
    (void)zcell_tile( P, z.ngw, &tw, &gpw );
    if ( waves ) *waves = ( tw * gpw + WAVE - 1 ) / WAVE;
    return size_t( g.Nz ) * g.Nw * ( ( P + tw - 1 ) / tw ) * ( ( z.ngw + gpw - 1 ) / gpw );
}

size_t zcell_metric_waves( const nufi_config &g, const zcell_plan &z )
{
    uint32_t waves = 0;
    const size_t n = zcell_workgroups( g, z, &waves );
    return n * waves;
}

zcell_plan plan_zcell( const nufi_config &g )
{
    zcell_plan z {};
    const uint64_t P = g.Nx * g.Ny, N = P * g.Nz, uv = g.Nu * g.Nv, plane = ( g.Nx + 3 ) * ( g.Ny + 3 );
    const uint32_t cols = uint32_t( g.Nx * ( g.Ny + 3 ) );
    if ( plane > 4096 || cols * g.Nx >= ( 1u << 20 ) || g.Nx < 3 || uv < 32 || uv >= ( 1u << 30 ) || P >= ( 1u << 24 ) || N * uv * g.Nw >= ( uint64_t( 1 ) << 62 ) ) return z;
    if ( plane * ( g.Nz + 3 ) > 20480 ) return z;                   // a whole slice has to fit the LDS: trace3d_zslice_kernel
    z.szp = uint32_t( ( plane + 3 ) & ~uint64_t( 1 ) );
    z.inv_nx = uint32_t( ( ( 1u << 20 ) + g.Nx - 1 ) / g.Nx );
    z.nzc = zcell_cells( cols, z.szp, uint32_t( g.Nz ) );
    if ( z.nzc == 0 ) return z;
    // partial sums no more than the window kernel's, or 8 MiB of them
    const uint64_t old = ( uv * g.Nw + xm3_vgroup( N, uv * g.Nw ) - 1 ) / xm3_vgroup( N, uv * g.Nw );
    const uint64_t cap = std::max<uint64_t>( uint64_t( 1 ) << 20, N * old );
    double best = 0;
    for ( uint32_t vg = 8; vg <= 256 && vg < uv + 8; vg += 8 )
    {
        const uint64_t ngw = ( uv + vg - 1 ) / vg, threads = N * g.Nw * ngw;
        if ( threads > cap ) continue;
        uint32_t tw, gpw;
        const double use = zcell_tile( uint32_t( P ), uint32_t( ngw ), &tw, &gpw ) * double( uv ) / double( ngw * vg );
        // four rounds of 512-thread workgroups on 256 CUs keep the last round's idle CUs few
        const double fill = std::min( 1.0, double( threads ) / ( 4.0 * 256 * 512 ) );
        if ( use * fill >= best * 0.999 ) { best = std::max( best, use * fill ); z.vg = vg; z.ngw = uint32_t( ngw ); }
    }
    z.ok = z.vg > 0;
    z.ppx = uint32_t( z.ngw * g.Nw );
    return z;
}

hipError_t launch_trace3d_zcell( const trace3_params &p_in, uint32_t *tasks, hipStream_t st )
{
    trace3_params p = p_in;
    const uint32_t P = p.Nx * p.Ny;
    (void)zcell_tile( P, p.zc.ngw, &p.zc.tw, &p.zc.gpw );
    p.zc.tiles = ( P + p.zc.tw - 1 ) / p.zc.tw;
    p.zc.ngb = ( p.zc.ngw + p.zc.gpw - 1 ) / p.zc.gpw;
    p.zc.z_first = p.l_first / P;
    const uint32_t nz = ( p.l_first + p.n_count - 1 ) / P - p.zc.z_first + 1;
    const double n[3] = { double( p.Nx ), double( p.Ny ), double( p.Nz ) }, dinv[3] = { p.dx_inv, p.dy_inv, p.dz_inv };
    for ( int a = 0; a < 3; ++a )
    {
        zcell_consts &k = p.zc.k;
        k.N[a] = n[a]; k.iN[a] = 1.0 / n[a]; k.cd[a] = p.dt * dinv[a];
        k.kick[a] = a == 2 ? p.kick72[a] / 3.0 : p.kick72[a];      // the z slope comes from 6 x the spline, not 2 x
        k.kickh[a] = 0.5 * k.kick[a];
    }
    const uint32_t threads = ( p.zc.tw * p.zc.gpw + WAVE - 1 ) / WAVE * WAVE;
    const uint64_t grid = uint64_t( nz ) * p.Nw * p.zc.tiles * p.zc.ngb;
    if ( grid >= ( uint64_t( 1 ) << 31 ) || p.n * ( p.zc.vg / 2 ) >= ( uint64_t( 1 ) << 30 ) ) return hipErrorInvalidValue;
    const bool mask = ( p.Nx & ( p.Nx - 1 ) ) == 0 && ( p.Ny & ( p.Ny - 1 ) ) == 0 && ( p.Nz & ( p.Nz - 1 ) ) == 0;
    const bool g16 = p.Nx == 16 && p.Ny == 16 && p.Nz == 16;
    const bool metrics = p.mode == MODE_METRICS;
    if ( p.zc.marks == nullptr ) return hipErrorInvalidValue;
    const void *k = nullptr;
    void *args[] = { &p };
    hipError_t e;
    p.dma = fast3_dma( 1, p.st ) ? 1u : 0u;
    // 16-byte words of a slice, whichever half of one it starts in
    const size_t full = p.dma ? 2 * size_t( p.st + 2 ) * sizeof(double) : size_t( ( p.st + 1 ) / 2 ) * 16u;
    auto launch = [&]( const void *f, uint32_t blocks, uint32_t block, size_t lds )
    {
        hipError_t err = lds > 0 ? hipFuncSetAttribute( f, hipFuncAttributeMaxDynamicSharedMemorySize, int( lds ) ) : hipSuccess;
        if ( err == hipSuccess ) err = hipLaunchKernel( f, dim3( blocks ), dim3( block ), args, lds, st );
        return err;
    };
    if ( zcell_routed( p.zc, p.n, p.Nz ) )
    {
        const uint32_t z_first = p.zc.z_first;
        p.zc.z_first = 0;                                  // of the whole grid, whatever slab the call traces
        e = launch( reinterpret_cast<const void*>( trace3d_spread_kernel ), uint32_t( p.n ), 1024, 0 );
        if ( e != hipSuccess ) return e;
        k = g16 ? reinterpret_cast<const void*>( trace3d_scout_kernel<true,16> )
                : mask ? reinterpret_cast<const void*>( trace3d_scout_kernel<true,0> ) : reinterpret_cast<const void*>( trace3d_scout_kernel<false,0> );
        if ( zc_all( p ) > ZC_FEW && zcell_decides( p.zc, p.n, p.Nz ) && ( e = launch( k, ZC_SCOUTS, threads, full ) ) != hipSuccess ) return e;
        p.zc.z_first = z_first;
    }
    else p.zc.route = nullptr;
    k = metrics ? zcell_kernel<MODE_METRICS>( mask, g16 ) : zcell_kernel<MODE_RHO>( mask, g16 );
    const size_t lds = zcell_lds( p.zc.nzc, p.Nx * ( p.Ny + 3 ), p.zc.szp );
    if ( ( e = launch( k, uint32_t( grid ), threads, lds ) ) != hipSuccess ) return e;
    if ( tasks ) *tasks = uint32_t( grid ) * ( threads / WAVE );
    if ( p.n == 0 || ( p.zc.nzc >= p.Nz && p.zc.route == nullptr ) ) return hipGetLastError();      // no window to leave
    k = metrics ? zslice_kernel<MODE_METRICS>( mask, g16 ) : zslice_kernel<MODE_RHO>( mask, g16 );
    if ( ( e = launch( k, uint32_t( grid ), threads, full ) ) != hipSuccess ) return e;
    return hipGetLastError();
}

} // namespace nufi_impl
