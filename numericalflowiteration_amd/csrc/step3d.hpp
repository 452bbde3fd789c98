// step3d.hpp — pieces of the fast FP64 3D step shared by the trace kernels:
// the cubic bases, one axis's drift and cell, the step's constants.
#ifndef NUFI_STEP3D_HPP
#define NUFI_STEP3D_HPP

#include "device_common.hpp"
#include "internal.hpp"

namespace nufi_impl
{

using namespace nufi_dev;

// ---- closed-form cubic B-spline bases on [0,1) ------------------------------
// values  B = ((1-t)^3, 3t^3-6t^2+4, -3t^3+3t^2+3t+1, t^3)/6
// slopes  D = (-(1-t)^2, 3t^2-4t, -3t^2+2t+1, t^2)/2
// Both kernels evaluate them times 6 (values) and 2 (slopes): integer-
// coefficient polynomials, with -(1-t)^2 and t^2 left to the contraction as a
// negation and a reuse.  The gradient from these bases is 72 times the
// gradient in reference-cell units: the FP64 kick folds 1/72 into its FP64
// constant; the FP32C kernel reads slices pre-scaled by fp32c3_scale, so its
// gradient is the kick itself.
//
// FP64 form: every constant is one the FP64 VALU takes inline (1, 2, 4, -4),
// so none occupies registers; the second value and slope come from the first
// by the symmetry B_2(t) = B_1(1-t), D_2(t) = -D_1(1-t):
//   B_1 = 3t^2 (t-2) + 4,  D_1 = 3t^2 - 4t,  3t^2 = 2t^2 + t^2.
__device__ __forceinline__ void cubic_bases_x6( double t, double B[4], double D[4] )
{
    const double a = 1.0 - t, t2 = t*t, a2 = a*a;
    const double t23 = fma( 2.0, t2, t2 ), a23 = fma( 2.0, a2, a2 );
    B[0] = a2 * a;
    B[3] = t2 * t;
    B[1] = fma( t23, t - 2.0, 4.0 );
    B[2] = fma( a23, a - 2.0, 4.0 );
    D[0] = -a2;
    D[3] = t2;
    D[1] = fma( -4.0, t, t23 );
    D[2] = fma( 4.0, a, -a23 );
}

// FP32 form.  The four slopes must sum to exactly zero as the FP32 numbers
// they are: a gradient contraction sum_i c_i D_i then carries no term in the
// level of the coefficients, only in their differences.  Rounded slopes leave
// a residual r(t) = sum_i D_i of about 2^-24 that multiplies the local level
// of phi, not its gradient; r depends on t alone, so it does not average out
// over cells or velocities, and on 3D Landau it gave 2e-6 relative energy
// error where the field passes near zero.  So (1-t)^2, t^2 and 3t^2 - 4t are
// each rounded once onto multiples of 2^-23 (an FMA that adds 1 or -1, which
// puts the result at magnitude [1,2] or a little above, then that 1 taken back
// exactly), and the third slope (a^2 - t^2) - D_1, whose partial results stay
// below 2 in magnitude, is exact.  The values need no such care (the slopes
// of the other axes cancel their level): B_2 is B_1 at 1 - t.
__device__ __forceinline__ void cubic_bases_x6( float t, float B[4], float D[4] )
{
    const float a = 1.0f - t;
    const float a2 = fmaf( a, a, 1.0f ) - 1.0f;                  // (1-t)^2 on the 2^-23 grid
    const float t2 = fmaf( t, t, 1.0f ) - 1.0f;                  // t^2 on the 2^-23 grid
    B[0] = a2 * a;
    B[3] = t2 * t;
    B[1] = fmaf( t2, fmaf( 3.0f, t, -6.0f ), 4.0f );            // 3t^3 - 6t^2 + 4
    B[2] = fmaf( a2, fmaf( 3.0f, a, -6.0f ), 4.0f );            // B_1(1-t)
    D[0] = -a2;
    D[3] = t2;
    D[1] = fmaf( t, fmaf( 3.0f, t, -4.0f ), -1.0f ) + 1.0f;     // 3t^2 - 4t on the 2^-23 grid
    D[2] = ( a2 - t2 ) - D[1];                                   // exact
}

// one axis of the fast FP64 step: drift (unless `still`), exact wrap, locate.
// MASK (power-of-two axis): no wrap here, the cell index wraps by a mask and
// the caller re-wraps the position exactly before every slice m with
// wrap3_due(m), a schedule fixed by m alone.
constexpr int WRAP3 = 16;
__device__ __forceinline__ bool wrap3_due( int64_t m ) { return ( m & ( WRAP3 - 1 ) ) == WRAP3 - 1; }

template <bool MASK>
__device__ __forceinline__ int advance_axis( double &s, double vel, double cd, double N, double invN, int Ni,
                                             double &t, bool still = false )
{
    double x = still ? s : fma( -cd, vel, s );
    if ( !MASK ) x = fma( -N, floor( x * invN ), x );
    const double k = floor( x );
    t = x - k;
    int i = int( k );
    if ( MASK ) i &= Ni - 1;
    else
    {
        i = ( i < 0 ) ? i + Ni : i;
        i = ( i >= Ni ) ? i - Ni : i;
    }
    s = x;
    return i;
}

// exact periodic re-wrap (N*floor(s/N) is an integer)
__device__ __forceinline__ void rewrap3( double &s, double N, double invN )
{
    s = fma( -N, floor( s * invN ), s );
}

struct fast3_consts
{
    double Nxd, Nyd, Nzd, iNx, iNy, iNz, cdx, cdy, cdz;
    double kx, ky, kz, kxh, kyh, kzh;     // -dt d_inv / 72 (times 72-scaled gradients), and half of it
    int Nxi, Nyi, Nzi;
    uint32_t sy, sz;
};

__device__ __forceinline__ fast3_consts make_fast3( const trace3_params &p )
{
    fast3_consts k;
    k.Nxd = p.Nx; k.Nyd = p.Ny; k.Nzd = p.Nz;
    k.iNx = 1.0 / k.Nxd; k.iNy = 1.0 / k.Nyd; k.iNz = 1.0 / k.Nzd;
    k.Nxi = int( p.Nx ); k.Nyi = int( p.Ny ); k.Nzi = int( p.Nz );
    k.cdx = p.dt * p.dx_inv; k.cdy = p.dt * p.dy_inv; k.cdz = p.dt * p.dz_inv;
    k.kx = p.kick72[0]; k.ky = p.kick72[1]; k.kz = p.kick72[2];           // kernel arguments: scalar registers
    k.kxh = p.kick72h[0]; k.kyh = p.kick72h[1]; k.kzh = p.kick72h[2];
    k.sy = p.sy; k.sz = p.sz;
    return k;
}

// Shared-basis gradient of the 4x4x4 window at c (72 times the gradient in
// reference-cell units with the bases above): per row (j,k)
//   A_jk = sum_i c_ijk Bx_i,  X_jk = sum_i c_ijk Dx_i,
// per plane k  P_k = sum_j A_jk By_j, Q_k = sum_j A_jk Dy_j, R_k = sum_j X_jk By_j,
// and g = (sum_k R_k Bz_k, sum_k Q_k Bz_k, sum_k P_k Dz_k).
//
// The window gather is software-pipelined (FP64 and FP32C kernels): the 16 rows
// (4 values each) of the 4x4x4 window are read PF rows ahead of the FMAs that
// use them, and the first PF rows before the bases are computed, so each row's
// LDS latency runs under earlier work.  The scheduling barriers keep the
// compiler from sinking the reads back next to their uses (it does so to save
// registers, and the waves a SIMD holds then cannot cover the latency).
// Measured at 512 x 4 on 3D Landau (FP64): PF = 1 is the fastest, 2 and 3 no
// faster, 4 slower.
constexpr int GATHER_PF = 1;

// The rows of a node's 4x4x4 window: row idx (j = idx & 3, k = idx >> 2) is
// the four reals from c + k*sz + j*sy.
template <typename T>
struct window_rt
{
    const T *c;
    uint32_t sy, sz;
    __device__ __forceinline__ const T *row( int idx ) const { return c + ( idx >> 2 ) * sz + ( idx & 3 ) * sy; }
};

// The same rows in the slice of a G^3 grid (strides G+3 and (G+3)^2): one LDS
// address per z plane, held in a register, and the rows of a plane at
// immediate offsets of the reads (at most 3(G+3)+3 reals, within the 255
// elements of ds_read2_b64 / ds_read2_b32 offsets for G <= 77).  Without the
// opaque register the compiler folds every row into a base address of its own.
template <int G, typename T = double>
struct window_g
{
    using lds_ptr = const __attribute__(( address_space( 3 ) )) T *;
    lds_ptr pl[4];
    __device__ __forceinline__ explicit window_g( const T *w )
    {
        pl[0] = (lds_ptr)w;
        #pragma unroll
        for ( int k = 1; k < 4; ++k )
        {
            uint32_t a = uint32_t( size_t( (lds_ptr)( w + k * ( G + 3 ) * ( G + 3 ) ) ) );
            asm volatile( "" : "+v"( a ) );
            pl[k] = (lds_ptr)size_t( a );
        }
    }
    __device__ __forceinline__ lds_ptr row( int idx ) const { return pl[ idx >> 2 ] + ( idx & 3 ) * ( G + 3 ); }
};

template <typename Win, typename T>
__device__ __forceinline__ void load_row( const Win &w, int idx, T r[4] )
{
    const auto q = w.row( idx );
    r[0] = q[0]; r[1] = q[1]; r[2] = q[2]; r[3] = q[3];
}

// the first PF rows of the window, before the bases are computed
template <int PF, typename Win, typename T>
__device__ __forceinline__ void grad_prefetch( const Win &w, T buf[PF + 1][4] )
{
    #pragma unroll
    for ( int d = 0; d < PF; ++d ) load_row( w, d, buf[d] );
    __builtin_amdgcn_sched_barrier( 0 );
}

template <int PF, typename Win, typename T>
__device__ __forceinline__ void grad_rows( const Win &w, T buf[PF + 1][4],
                                           const T Bx[4], const T Dx[4], const T By[4],
                                           const T Dy[4], const T Bz[4], const T Dz[4],
                                           T &gx, T &gy, T &gz )
{
    T P = T(0), Q = T(0), R = T(0);
    gx = T(0); gy = T(0); gz = T(0);
    #pragma unroll
    for ( int idx = 0; idx < 16; ++idx )
    {
        if ( idx + PF < 16 ) load_row( w, idx + PF, buf[ ( idx + PF ) % ( PF + 1 ) ] );
        __builtin_amdgcn_sched_barrier( 0 );
        const T *r = buf[ idx % ( PF + 1 ) ];
        const int j = idx & 3, k = idx >> 2;
        const T A = fma( r[3], Bx[3], fma( r[2], Bx[2], fma( r[1], Bx[1], r[0]*Bx[0] ) ) );
        const T X = fma( r[3], Dx[3], fma( r[2], Dx[2], fma( r[1], Dx[1], r[0]*Dx[0] ) ) );
        P = j == 0 ? A * By[0] : fma( A, By[j], P );
        Q = j == 0 ? A * Dy[0] : fma( A, Dy[j], Q );
        R = j == 0 ? X * By[0] : fma( X, By[j], R );
        if ( j == 3 )
        {
            gx = fma( R, Bz[k], gx );
            gy = fma( Q, Bz[k], gy );
            gz = fma( P, Dz[k], gz );
        }
    }
}

// one fast FP64 characteristic step of one node with slice C: drift (unless
// `still`), exact wrap, E = -grad phi from the shared-basis window, kick by hf*dt
// (`half`: hf = 1/2, the kick constants are selected per slice, not multiplied)
template <int G, typename T>
__device__ __forceinline__ typename std::enable_if<( G > 0 ), window_g<G, T>>::type
make_window( const T *w, uint32_t, uint32_t ) { return window_g<G, T>( w ); }

template <int G, typename T>
__device__ __forceinline__ typename std::enable_if<( G == 0 ), window_rt<T>>::type
make_window( const T *w, uint32_t sy, uint32_t sz ) { return window_rt<T> { w, sy, sz }; }

// G > 0: a cubic G^3 grid whose slice strides (G+3, (G+3)^2) are compile-time
// constants, so the window's row offsets are immediates of the LDS reads and
// only the window base is computed per node-step; G = 0 takes the strides from
// the kernel arguments (24-bit products: a slice stays far below 2^24 reals).
template <bool MASK = false, int PF = GATHER_PF, int G = 0>
__device__ __forceinline__ void step3_fast( const fast3_consts &k, const double *C, bool half, bool still,
                                            double &sx, double &sy_, double &sz_, double &vu, double &vv, double &vw )
{
    double tx, ty, tz;
    const int i = advance_axis<MASK>( sx,  vu, k.cdx, k.Nxd, k.iNx, k.Nxi, tx, still );
    const int j = advance_axis<MASK>( sy_, vv, k.cdy, k.Nyd, k.iNy, k.Nyi, ty, still );
    const int l = advance_axis<MASK>( sz_, vw, k.cdz, k.Nzd, k.iNz, k.Nzi, tz, still );
    constexpr uint32_t GY = G > 0 ? uint32_t( G + 3 ) : 0u, GZ = GY * GY;
    const uint32_t sy = G > 0 ? GY : k.sy, sz = G > 0 ? GZ : k.sz;
    const double *W = C + __umul24( uint32_t( l ), sz ) + __umul24( uint32_t( j ), sy ) + i;
    using Win = typename std::conditional<( G > 0 ), window_g<G>, window_rt<double>>::type;
    Win win = make_window<G>( W, sy, sz );
    double buf[PF + 1][4];
    grad_prefetch<PF>( win, buf );
    double Bx[4], Dx[4], By[4], Dy[4], Bz[4], Dz[4];
    cubic_bases_x6( tx, Bx, Dx );
    cubic_bases_x6( ty, By, Dy );
    cubic_bases_x6( tz, Bz, Dz );
    double gx, gy, gz;
    grad_rows<PF>( win, buf, Bx, Dx, By, Dy, Bz, Dz, gx, gy, gz );
    vu = fma( half ? k.kxh : k.kx, gx, vu );
    vv = fma( half ? k.kyh : k.ky, gy, vv );
    vw = fma( half ? k.kzh : k.kz, gz, vw );
}

} // namespace nufi_impl

#endif
