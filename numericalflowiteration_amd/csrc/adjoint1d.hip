// adjoint1d.hip — reverse-mode gradient of J = sum_n dt * energy_n (the time-
// integrated spectral electric energy) with respect to the parameters of the
// 1D initial condition, on the device, for the FP64 fast trace.
//
// Forward model (one time step n; the same arithmetic as trace1d.hip):
//   rho_n[i] = -du sum_u f0( foot_n(x_i, u; S_0..S_{n-1}); a )
//   S_n      = M rho_n          (Poisson + fit + periodic padding, linear)
//   e_n      = sum_k w_k |F rho_n|_k^2
// Reverse sweep, n = Nt .. 0, with lambda_m = dJ/dS_m (folded mod Nx):
//   g_n = 2 dt Re F^H( w . F rho_n ) + Re F^H( conj(m) . F lambda_n )  (= dJ/d rho_n)
//   per node: fbar = -du g_n[i]; trace forward to the foot; dJ/da += fbar df0/da;
//   then walk back through slices 0 .. n-1, undoing each Stormer-Verlet step
//   as it was taken (the states are recomputed, never stored), with the
//   polynomial p(t) = Q0 + Q1 t + Q2 t^2 of 2 dphi/dt of the forward kernel
//   (hk = h kick, h = 1, or 1/2 on slice 0):
//     forward  s_a = s_b - cd u_b,  u_a = u_b + hk p(s_a; S_m)
//     reverse  pbar = hk ubar;  sbar += pbar dp/dt;  lambda_m += pbar dp/dS_m;
//              u_b = u_a - hk p;  ubar += -cd sbar;  s_b = s_a + cd u_b
// lambda_m accumulates in LDS per workgroup (all nodes of a workgroup visit the
// same slice at the same time) and is flushed with global atomics once per
// chunk of slices; its summation order therefore varies at the rounding level.
//
// FP32C contexts differentiate the FP32-compensated trace, whose velocity w is
// in cells per step (w = cd u): the forward sweep repeats the FP32C kernel's
// steps (the shared fp32c_* helpers of step1d.hpp, so the foot points are
// those of the forward run), the reverse sweep undoes them on the same pairs
// (w_b = w_a - h q(s_a), s_b = s_a + w_b, both with TwoSum), and the adjoints
// sbar, wbar, lambda and the parameter gradients are FP64, as is the field
// adjoint.  The FP32 tables hold kick cd (Q0, Q1, Q2), so pbar = h kick cd wbar,
// sbar += h wbar dq/dt, wbar -= sbar, and the seed is wbar = fbar df0/du / cd.
#include "device_common.hpp"
#include "fft_lds.hpp"
#include "internal.hpp"
#include "step1d.hpp"

namespace nufi_impl
{

using namespace nufi_dev;

namespace
{

// d f0 / d(x, u) and d f0 / d(parameters) for the 1D families.  Parameters:
// alpha for Landau and two-stream; a_1..a_n for the multimode family.
__device__ inline void f0_grad_1d( const nufi_f0 &p, double x, double u, double &fx, double &fu,
                                   double *fa, int npar )
{
    const double e = exp( -u*u/2.0 );
    switch ( p.kind )
    {
    case NUFI_F0_LANDAU_1D:
    {
        double c, s;
        sincos( p.k*x, &s, &c );
        fx = kInvSqrt2Pi * ( -p.alpha * p.k * s ) * e;
        fu = kInvSqrt2Pi * ( 1.0 + p.alpha*c ) * e * ( -u );
        if ( npar > 0 ) fa[0] = kInvSqrt2Pi * c * e;
        break;
    }
    case NUFI_F0_TWOSTREAM_1D:
    {
        double c, s;
        sincos( p.k*x, &s, &c );
        fx = kInvSqrt2Pi * ( -p.alpha * p.k * s ) * e * u*u;
        fu = kInvSqrt2Pi * ( 1.0 + p.alpha*c ) * e * u * ( 2.0 - u*u );
        if ( npar > 0 ) fa[0] = kInvSqrt2Pi * c * e * u*u;
        break;
    }
    case NUFI_F0_MULTIMODE_1D:
    {
        double sm = 1.0, dsm = 0.0;
        #pragma unroll
        for ( int m = 1; m <= NUFI_MAX_MODES; ++m )     // static indices: no private-memory copy
        {
            if ( m > p.n_modes ) continue;
            const double km = p.k * m;
            double c, s;
            sincos( km * x, &s, &c );
            sm += p.a[m-1] * c;
            dsm -= p.a[m-1] * km * s;
            if ( m <= npar ) fa[m-1] = kInvSqrt2Pi * c * e;
        }
        fx = kInvSqrt2Pi * dsm * e;
        fu = kInvSqrt2Pi * sm * e * ( -u );
        break;
    }
    default:
        fx = fu = 0.0;
        #pragma unroll
        for ( int m = 0; m < NUFI_MAX_MODES; ++m ) if ( m < npar ) fa[m] = 0.0;
    }
}

// One node's state and its adjoint in each arithmetic: down() takes the forward
// steps of slices mlo+hi .. mlo (tables at Q, sq elements each), locate() gives
// the cell (in [-1, Nx]; POW2: in [0, Nx)) and t the forward step used at the
// present position, undo() takes a step back (h = 1, or 1/2 on slice 0) and
// returns pbar, the adjoint of the kick polynomial's value; with POW2 the
// caller re-wraps behind every slice m with poly_wrap_due(m).
template <bool POW2>
struct adjoint_fp64
{
    using table = double;
    double cd, kick, Nxd, invNx, s, u, sbar, pb;          // pb: kick times the adjoint of u
    int mask;
    uint32_t q2;

    __device__ __forceinline__ static const double *tables( const adjoint1_params &p ) { return p.qhist; }
    __device__ __forceinline__ void start( const adjoint1_params &p, uint32_t ix, uint32_t iu )
    {
        Nxd = p.Nx; invNx = 1.0 / Nxd; cd = p.dt * p.dx_inv; kick = -0.5 * p.dt * p.dx_inv;
        mask = int( p.Nx ) - 1; q2 = p.q2_off;
        s = double( ix );
        u = p.u_min + iu*p.du + p.du/2;
    }
    __device__ __forceinline__ void down( const double *Q, uint32_t sq, int mlo, int hi )
    {
        poly_down<POW2>( s, u, Q, sq, q2, mlo, hi, cd, kick, mask, Nxd, invNx );
    }
    __device__ __forceinline__ double foot_x( const adjoint1_params &p ) const { return p.x_min + s*p.dx; }
    __device__ __forceinline__ double foot_u() const { return u; }
    __device__ __forceinline__ void seed( const adjoint1_params &p, double fbar, double fx, double fu )
    {
        sbar = fbar * fx * p.dx;               // d/ds = dx d/dx
        pb = kick * ( fbar * fu );
    }
    struct cell { int i; double t, q0, q1, q2; };
    __device__ __forceinline__ cell locate( const double *Q ) const
    {
        cell c;
        const double k = floor( s );
        c.t = s - k;
        c.i = POW2 ? ( int( k ) & mask ) : int( k );
        const double2 q01 = reinterpret_cast<const double2*>( Q )[ c.i + 1 ];
        c.q0 = q01.x; c.q1 = q01.y; c.q2 = Q[ q2 + ( c.i + 1 ) ];
        return c;
    }
    __device__ __forceinline__ double undo( const cell &c, float h )
    {
        const double q = fma( c.q2, c.t, c.q1 ), dpdt = fma( c.q2, c.t, q ), pv = fma( q, c.t, c.q0 );
        const double pbar = h == 1.0f ? pb : double( h ) * pb;
        sbar = fma( pbar, dpdt, sbar );
        u = fma( h == 1.0f ? -kick : -double( h ) * kick, pv, u );
        pb = fma( -kick * cd, sbar, pb );
        s = fma( cd, u, s );
        if ( !POW2 ) wrap();
        return pbar;
    }
    __device__ __forceinline__ void wrap() { rewrap( s, Nxd, invNx ); }
};

template <bool POW2>
struct adjoint_fp32c
{
    using table = float;
    double cd, kick, sbar, ubar;               // ubar: of the velocity in cells per step
    frame1 fr;
    float sh, sl, uh, ul;
    int mask;
    uint32_t q2;

    __device__ __forceinline__ static const float *tables( const adjoint1_params &p ) { return p.qhist32; }
    __device__ __forceinline__ void start( const adjoint1_params &p, uint32_t ix, uint32_t iu )
    {
        cd = p.dt * p.dx_inv; kick = -0.5 * p.dt * p.dx_inv;
        mask = int( p.Nx ) - 1; q2 = p.q2_off;
        fr = make_frame1( p.f32_p0, p.f32_w0, p.Nx );
        fp32c_start( fr, ix, cd * ( p.u_min + iu*p.du + p.du/2 ), sh, sl, uh, ul );
    }
    __device__ __forceinline__ void down( const float *Q, uint32_t sq, int mlo, int hi )
    {
        for ( int jj = hi; jj >= 0; --jj )
        {
            const int m = mlo + jj;
            if ( POW2 && poly_wrap_due( m ) ) fp32c_rewrap( fr, sh, sl, uh, ul );
            fp32c_move( fr, sh, sl, uh, ul );
            if ( !POW2 ) fp32c_rewrap( fr, sh, sl, uh, ul );
            float t;
            const int i = fp32c_locate<POW2>( fr, sh, sl, mask, t );
            fp32c_kick( uh, ul, ( m == 0 ? 0.5f : 1.0f ) * fp32c_poly( Q + jj * sq, q2, i, t ) );
        }
    }
    __device__ __forceinline__ double foot_x( const adjoint1_params &p ) const { return p.x_min + fp32c_position( fr, sh, sl ) * p.dx; }
    __device__ __forceinline__ double foot_u() const { return fp32c_velocity( fr, uh, ul ) / cd; }
    __device__ __forceinline__ void seed( const adjoint1_params &p, double fbar, double fx, double fu )
    {
        sbar = fbar * fx * p.dx;
        ubar = fbar * fu / cd;                 // d/dw = d/du / cd
    }
    struct cell { int i; float t, q0, q1, q2; };
    __device__ __forceinline__ cell locate( const float *Q ) const
    {
        cell c;
        c.i = fp32c_locate<POW2>( fr, sh, sl, mask, c.t );
        const float2 q01 = reinterpret_cast<const float2*>( Q )[ c.i + 1 ];
        c.q0 = q01.x; c.q1 = q01.y; c.q2 = Q[ q2 + ( c.i + 1 ) ];
        return c;
    }
    __device__ __forceinline__ double undo( const cell &c, float hf )
    {
        const float q = fmaf( fmaf( c.q2, c.t, c.q1 ), c.t, c.q0 );
        const double dqdt = fma( 2.0 * double( c.q2 ), double( c.t ), double( c.q1 ) );     // of the scaled table, in FP64
        const double pbar = double( hf ) * kick * cd * ubar;
        sbar = fma( double( hf ) * ubar, dqdt, sbar );
        fp32c_kick( uh, ul, -( hf * q ) );     // undo the kick, then the drift
        ubar = ubar - sbar;
        fp32c_move<true>( fr, sh, sl, uh, ul );
        if ( !POW2 ) wrap();
        return pbar;
    }
    __device__ __forceinline__ void wrap() { fp32c_rewrap( fr, sh, sl, uh, ul ); }
};

// Sums over the wave of eight values a lane, compensated: three exchanges halve
// the values a lane holds, three more finish its one.  Lane l gets the sum of
// value (l >> 3) with its bits in the order 5, 4, 3, eight lanes each.
__device__ __forceinline__ double wave_csum8( const double f[8] )
{
    const uint32_t lane = threadIdx.x % WAVE;
    csum v[8];
    #pragma unroll
    for ( int k = 0; k < 8; ++k ) v[k] = csum { f[k], 0.0 };
    #pragma unroll
    for ( int half = 4, off = 32; half > 0; half >>= 1, off >>= 1 )
    {
        const bool up = ( lane & uint32_t( off ) ) != 0;
        #pragma unroll
        for ( int k = 0; k < half; ++k )
        {
            const csum keep = up ? v[k + half] : v[k], send = up ? v[k] : v[k + half];
            v[k] = csum_add( keep, csum { __shfl_xor( send.s, off ), __shfl_xor( send.c, off ) } );
        }
    }
    #pragma unroll
    for ( int off = 4; off > 0; off >>= 1 )
        v[0] = csum_add( v[0], csum { __shfl_xor( v[0].s, off ), __shfl_xor( v[0].c, off ) } );
    return v[0].s + v[0].c;
}

// x-major nodes (lanes over consecutive x), a whole workgroup through the same
// slices.  A node's pbar scatters into the four slice adjoints of its cell by
// LDS atomics, issued behind the next step's table read, which they would hold
// up.  With PIPE a slice's adjoints are a row of cells -1 .. Nx, entries 0 ..
// Nx+4 (one address, immediate offsets), and the tables have two buffers; tables
// too wide for two slices of that take one buffer and adjoints folded mod Nx.
//
// Bound by the serial chain of the steps (table read, polynomial, velocity,
// position; about 40 of 70 us at 256 threads), then by the global atomics (15),
// the flush's LDS passes and the LDS atomics (9 each).  128 x 512, n averaging
// 160: with velocity-major lanes, whose 64 neighbouring velocities hit the same
// cells, one table buffer with its copies waited for, 15-slice chunks and a
// runtime modulo per scattered point 103 us a launch (LDS atomics 45); this one
// 65.  The flush a row a step instead of between chunks 82 (its reads wait
// for the scatter's queue); a cell's (pbar, pbar t, pbar t^2) scattered by three
// atomics and combined at the flush 81.
template <typename NODE, bool POW2, bool PIPE>
__global__ __launch_bounds__( 1024 )
void adjoint1d_kernel( adjoint1_params p )
{
    extern __shared__ __align__( 16 ) double lds[];
    using T = typename NODE::table;
    const uint32_t threads = blockDim.x, waves = threads / WAVE, tid = threadIdx.x;
    const uint32_t sq = p.stride_q, C = p.chunk, Nx = p.Nx;
    T *const Q0 = reinterpret_cast<T*>( lds ), *const Q1 = Q0 + ( PIPE ? size_t( C ) * sq : 0 );
    double *const lam = reinterpret_cast<double*>( Q1 + size_t( C ) * sq );
    const uint32_t lw = PIPE ? Nx + 5 : Nx;                        // adjoints per slice
    const T *const hist = NODE::tables( p );

    const uint64_t nodes = uint64_t( Nx ) * p.Nu, q = uint64_t( blockIdx.x ) * threads + tid;
    const bool active = q < nodes;
    const uint64_t qn = q < nodes ? q : q % nodes;                 // lanes past the last node repeat others with weight 0
    const uint32_t iu = uint32_t( qn / Nx ), ix = uint32_t( qn - uint64_t( iu ) * Nx );
    // this wave's gradient sums, one value a lane (wave_csum8)
    const uint32_t wave = blockIdx.x * waves + tid / WAVE, l8 = tid % WAVE / 8;
    const uint32_t par = ( l8 >> 2 ) * 4 + ( ( l8 >> 1 ) & 1 ) * 2 + ( l8 & 1 );
    double *const grad = p.grad_part + size_t( wave ) * NUFI_MAX_MODES + par;
    const bool keeps = tid % 8 == 0 && wave < p.n_tasks && par < p.npar;
    const double grad0 = keeps ? *grad : 0.0, gx = p.g[ix];
    NODE nd;
    nd.start( p, ix, iu );

    // forward: slices n-1 .. 0, the steps of the trace kernel
    auto down = [&]( const T *Q, int mlo, int hi, int ) __attribute__(( always_inline )) { nd.down( Q, sq, mlo, hi ); };
    if ( PIPE ) poly_ready_pipeline( Q0, hist, sq, p.n, C, waves, down );
    else        poly_ready_direct( Q0, hist, sq, p.n, C, waves, down );

    // the reverse sweep's first tables come while the seeds are formed
    const int n = int( p.n ), Ci = int( C ), K = ( n + Ci - 1 ) / Ci;
    auto cnt_of = [&]( int k ) { return n - k * Ci < Ci ? n - k * Ci : Ci; };
    auto copy = [&]( T *dst, int k ) __attribute__(( always_inline ))
    {
        dma_copy16( dst, hist + size_t( k ) * C * sq, uint32_t( cnt_of( k ) ) * ( sq * uint32_t( sizeof( T ) ) / 16u ), waves );
    };
    __syncthreads();                                        // the forward chunks are read
    if ( K > 0 ) copy( Q0, 0 );
    for ( uint32_t e = tid; e < C * lw; e += threads ) lam[e] = 0.0;

    // seed at the foot
    {
        static_assert( NUFI_MAX_MODES == 8, "wave_csum8" );
        const double fbar = active ? -p.du * gx : 0.0;
        double fx, fu, fa[NUFI_MAX_MODES] = { 0, 0, 0, 0, 0, 0, 0, 0 };
        f0_grad_1d( p.f0, nd.foot_x( p ), nd.foot_u(), fx, fu, fa, p.npar );
        nd.seed( p, fbar, fx, fu );
        #pragma unroll
        for ( int m = 0; m < NUFI_MAX_MODES; ++m ) fa[m] *= fbar;
        const double sum = wave_csum8( fa );
        if ( keeps ) *grad = grad0 + sum;
    }

    // reverse: slices 0 .. n-1 in chunks
    auto scatter = [&]( double *L, int i, double t, double pbar ) __attribute__(( always_inline ))
    {
        // adjoints of q0 = D0 + D1, q1 = 2 (D1 - D0), q2 = D0 - 2 D1 + D2, Dl = c[i+l] - c[i+l-1] of the row from c[i]
        const double q0 = pbar, q1 = pbar * t, q2 = q1 * t;
        const double n0 = fma( 2.0, q1, -fma( q1, t, q0 ) ), d1 = fma( 2.0, q1 - q2, q0 );         // n0 = -d0
        uint32_t e = uint32_t( i + 1 );
        if ( PIPE )
        {
            atomicAdd( L + e, n0 );          atomicAdd( L + e + 1, -n0 - d1 );
            atomicAdd( L + e + 2, d1 - q2 ); atomicAdd( L + e + 3, q2 );
            return;
        }
        e = i < 0 ? Nx - 1 : uint32_t( i );                 // a ring may be shorter than the four points
        if ( e >= Nx ) e -= Nx;
        auto next = [&]() { if ( ++e == Nx ) e = 0; };
        atomicAdd( L + e, n0 );       next();
        atomicAdd( L + e, -n0 - d1 ); next();
        atomicAdd( L + e, d1 - q2 );  next();
        atomicAdd( L + e, q2 );
    };
    // the chunk's adjoints to global memory, and cleared: a wave takes whole rows.
    // PIPE: entries 0 and Nx+1 .. Nx+4 lie a period off and go by themselves.
    auto flush = [&]( uint32_t cnt, double *to ) __attribute__(( always_inline ))
    {
        const uint32_t w = __builtin_amdgcn_readfirstlane( tid / WAVE );
        for ( uint32_t jj = w; jj < cnt; jj += waves )
        {
            double *S = lam + jj * lw + ( PIPE ? 1 : 0 ), *G = to + jj * Nx;
            for ( uint32_t x = tid % WAVE; x < Nx; x += WAVE )
            {
                const double v = S[x];
                S[x] = 0.0;
                atomicAdd( G + x, v );
            }
        }
        if ( !PIPE ) return;
        for ( uint32_t e = tid; e < cnt * 5; e += threads )
        {
            const uint32_t jj = e / 5, c = e - jj * 5;
            double *S = lam + jj * lw + ( c == 4 ? 0u : Nx + 1 + c );
            const double v = *S;
            *S = 0.0;
            if ( v != 0.0 ) atomicAdd( to + jj * Nx + ( c == 4 ? Nx - 1 : c % Nx ), v );
        }
    };
    dma_publish();
    for ( int k = 0; k < K; ++k )
    {
        const int cnt = cnt_of( k ), mlo = k * Ci;
        const T *Q = ( PIPE && ( k & 1 ) ) ? Q1 : Q0;
        if ( PIPE && k + 1 < K ) copy( ( k & 1 ) ? Q0 : Q1, k + 1 );
        // the pending adjoints: of the step before, at first zeros
        double *L = lam, *now = lam, tp = 0.0, pp = 0.0;
        int ip = int( ix ), jj = 0;
        auto step = [&]( float h ) __attribute__(( always_inline ))
        {
            const auto c = nd.locate( Q );
            __builtin_amdgcn_sched_barrier( 0 );
            scatter( L, ip, tp, pp );
            __builtin_amdgcn_sched_barrier( 0 );
            pp = nd.undo( c, h );
            tp = double( c.t ); ip = c.i;
            L = now; now += lw;
            Q += sq; ++jj;
        };
        if ( mlo == 0 ) step( 0.5f );
        while ( jj < cnt )                                  // segments between re-wrap points
        {
            const int left = POLY_WRAP - ( ( mlo + jj ) & ( POLY_WRAP - 1 ) );
            const int stop = POW2 && jj + left < cnt ? jj + left : cnt;
            while ( jj < stop ) step( 1.0f );
            if ( POW2 && poly_wrap_due( mlo + jj - 1 ) ) nd.wrap();
        }
        scatter( L, ip, tp, pp );
        if ( PIPE ) dma_publish();                          // the adjoints are complete and the next tables there
        else
        {
            __syncthreads();
            if ( k + 1 < K ) copy( Q0, k + 1 );
        }
        flush( uint32_t( cnt ), p.lambda + size_t( mlo ) * Nx );
        if ( PIPE ) __syncthreads();
        else        dma_publish();
    }
}

// g = 2 dt Re F^H( w . F rho ) + Re F^H( conj(m) . F lambda )   (one workgroup).
// Latency-bound: both forward transforms go through the same stages as two
// lines, their spectra are added and one transform goes back; twiddles in LDS,
// the weights loaded at the start: 128 points 8.5 -> 4.7 us.  Lines too long for that (p.wide) are
// transformed one after the other, there and back.
__global__ __launch_bounds__( FIELD_BLOCK )
void adjoint_field_kernel( adjoint_field_params p )
{
    extern __shared__ double2 ldsa[];
    const uint32_t N = p.N;
    if ( p.wide )
    {
        double2 *A = ldsa, *B = ldsa + N;
        axis_desc ax { N, p.log2x, 1u, 1u, 0u, N, 1u, p.rx };
        for ( int pass = 0; pass < 2; ++pass )
        {
            const double *in = pass == 0 ? p.rho : p.lambda;
            for ( uint32_t i = threadIdx.x; i < N; i += FIELD_BLOCK ) A[i] = make_double2( in[i], 0.0 );
            __syncthreads();
            double2 *F = fft_axis( A, B, ax, p.tw, false );
            double2 *G = ( F == A ) ? B : A;
            for ( uint32_t k = threadIdx.x; k < N; k += FIELD_BLOCK )
            {
                if ( pass == 0 ) { const double w = 2.0 * p.dt * p.ewt[k]; F[k] = make_double2( w * F[k].x, w * F[k].y ); }
                else { const double2 m = p.mult[k]; F[k] = cmul( F[k], make_double2( m.x, -m.y ) ); }
            }
            __syncthreads();
            double2 *R = fft_axis( F, G, ax, p.tw, true );
            for ( uint32_t i = threadIdx.x; i < N; i += FIELD_BLOCK )
                p.g[i] = ( pass == 0 ) ? R[i].x : p.g[i] + R[i].x;
            __syncthreads();
        }
        return;
    }
    double2 *A = ldsa, *B = ldsa + 2*N, *tw = ldsa + 4*N;
    const uint32_t nt = twiddle_entries( N, p.log2x );
    for ( uint32_t i = threadIdx.x; i < nt; i += FIELD_BLOCK ) tw[i] = p.tw[i];
    constexpr uint32_t PRE = 2;                              // the thread's first modes; N <= 2048 has up to 4
    double2 mu[PRE];
    double ew[PRE];
    #pragma unroll
    for ( uint32_t c = 0; c < PRE; ++c )
    {
        const uint32_t k = threadIdx.x + c * FIELD_BLOCK;
        mu[c] = make_double2( 0.0, 0.0 ); ew[c] = 0.0;
        if ( k < N ) { mu[c] = p.mult[k]; ew[c] = p.ewt[k]; }
    }
    for ( uint32_t i = threadIdx.x; i < N; i += FIELD_BLOCK )
    {
        const double a = p.rho[i], b = p.lambda[i];
        A[i] = make_double2( a, 0.0 ); A[N + i] = make_double2( b, 0.0 );
    }
    __syncthreads();
    axis_desc two { N, p.log2x, 1u, 2u, 0u, N, 1u, p.rx }, one = two;
    one.nlines = 1;
    double2 *F = fft_axis( A, B, two, tw, false );
    double2 *G = ( F == A ) ? B : A;
    auto both = [&]( uint32_t k, double2 m, double e ) __attribute__(( always_inline ))
    {
        const double w = 2.0 * p.dt * e;
        const double2 f = F[k], l = cmul( F[N + k], make_double2( m.x, -m.y ) );
        F[k] = make_double2( fma( w, f.x, l.x ), fma( w, f.y, l.y ) );
    };
    #pragma unroll
    for ( uint32_t c = 0; c < PRE; ++c )
        if ( threadIdx.x + c * FIELD_BLOCK < N ) both( threadIdx.x + c * FIELD_BLOCK, mu[c], ew[c] );
    for ( uint32_t k = threadIdx.x + PRE * FIELD_BLOCK; k < N; k += FIELD_BLOCK ) both( k, p.mult[k], p.ewt[k] );
    __syncthreads();
    double2 *R = fft_axis( F, G, one, tw, true );
    for ( uint32_t i = threadIdx.x; i < N; i += FIELD_BLOCK ) p.g[i] = R[i].x;
}

__global__ __launch_bounds__( 256 )
void reduce_grad_kernel( const double *part, uint32_t n_tasks, uint32_t npar, double *grad )
{
    __shared__ double red_s[256], red_c[256];
    for ( uint32_t m = 0; m < npar; ++m )
    {
        csum acc { 0, 0 };
        for ( uint32_t g = threadIdx.x; g < n_tasks; g += 256 )
            acc = csum_add( acc, csum { part[ size_t( g ) * NUFI_MAX_MODES + m ], 0.0 } );
        red_s[threadIdx.x] = acc.s; red_c[threadIdx.x] = acc.c;
        __syncthreads();
        if ( threadIdx.x == 0 )
        {
            csum t { 0, 0 };
            for ( int i = 0; i < 256; ++i ) t = csum_add( t, csum { red_s[i], red_c[i] } );
            grad[m] = t.s + t.c;
        }
        __syncthreads();
    }
}

} // namespace

// Workgroups of 512 threads, 1024 where a CU would get two of them: one takes
// the whole LDS.  Fewer workgroups add fewer global atomics (each adds to every
// slice adjoint) and longer LDS queues: at 128 x 512, 256 threads (every CU)
// 70 us, 512 (half of them) 65, 1024 103; above 131072 nodes, gradient to T = 5 by 512 /
// 1024 threads: 133120 nodes 5.5 / 4.5 ms, 262144 7.7 / 5.7, 1048576 31.0 / 21.6 (velocity-
// major 9.3, 11.4, 41.9).  Two table buffers and padded adjoint rows where at least two slices of both fit.
void plan_adjoint1d( adjoint1_params &p, int n_cu, size_t lds_cap )
{
    const uint64_t nodes = uint64_t( p.Nx ) * p.Nu;
    p.threads = 512;
    while ( p.threads < 1024 && nodes > uint64_t( p.threads ) * uint64_t( n_cu ) ) p.threads *= 2;
    const size_t table = size_t( p.stride_q ) * ( p.qhist32 ? sizeof(float) : sizeof(double) );
    const size_t cap = std::min<size_t>( lds_cap, 160 * 1024 ), two = 2 * table + 8 * ( size_t( p.Nx ) + 5 );
    p.pipe = cap / two >= 2;
    const size_t per = p.pipe ? two : table + size_t( p.Nx ) * sizeof(double);
    p.chunk = uint32_t( std::max<size_t>( 1, std::min<size_t>( 32, cap / per ) ) );
}

size_t adjoint1d_lds_bytes( const adjoint1_params &p )
{
    const size_t table = size_t( p.stride_q ) * ( p.qhist32 ? sizeof(float) : sizeof(double) );
    return size_t( p.chunk ) * ( p.pipe ? 2 * table + 8 * ( size_t( p.Nx ) + 5 ) : table + size_t( p.Nx ) * sizeof(double) );
}

template <bool POW2, bool PIPE>
static const void *adjoint1d_entry( bool f32 )
{
    return f32 ? reinterpret_cast<const void*>( adjoint1d_kernel<adjoint_fp32c<POW2>,POW2,PIPE> )
               : reinterpret_cast<const void*>( adjoint1d_kernel<adjoint_fp64<POW2>,POW2,PIPE> );
}

hipError_t launch_adjoint1d( const adjoint1_params &p_in, hipStream_t st )
{
    adjoint1_params p = p_in;
    const uint64_t nodes = uint64_t( p.Nx ) * p.Nu, grid = ( nodes + p.threads - 1 ) / p.threads;
    if ( nodes == 0 ) return hipSuccess;
    const size_t lds = adjoint1d_lds_bytes( p );
    const bool pow2 = ( p.Nx & ( p.Nx - 1 ) ) == 0, f32 = p.qhist32 != nullptr;
    const void *k = p.pipe ? ( pow2 ? adjoint1d_entry<true,true>( f32 ) : adjoint1d_entry<false,true>( f32 ) )
                            : ( pow2 ? adjoint1d_entry<true,false>( f32 ) : adjoint1d_entry<false,false>( f32 ) );
    if ( lds > 65536 )
    {
        hipError_t e = hipFuncSetAttribute( k, hipFuncAttributeMaxDynamicSharedMemorySize, int( lds ) );
        if ( e != hipSuccess ) return e;
    }
    void *args[] = { &p };
    const hipError_t e = hipLaunchKernel( k, dim3( uint32_t( grid ) ), dim3( p.threads ), args, lds, st );
    return e != hipSuccess ? e : hipGetLastError();
}

hipError_t launch_adjoint_field( const adjoint_field_params &p_in, hipStream_t st )
{
    adjoint_field_params p = p_in;
    size_t lds = ( size_t( p.N ) * 4 + twiddle_entries( p.N, p.log2x ) ) * sizeof(double2);
    p.wide = lds > 160u * 1024u ? 1 : 0;
    if ( p.wide ) lds = size_t( p.N ) * 2 * sizeof(double2);
    if ( lds > 65536 )
    {
        hipError_t e = hipFuncSetAttribute( reinterpret_cast<const void*>( adjoint_field_kernel ),
                                            hipFuncAttributeMaxDynamicSharedMemorySize, int( lds ) );
        if ( e != hipSuccess ) return e;
    }
    hipLaunchKernelGGL( adjoint_field_kernel, dim3( 1 ), dim3( FIELD_BLOCK ), lds, st, p );
    return hipGetLastError();
}

hipError_t launch_reduce_grad( const double *part, uint32_t n_tasks, uint32_t npar, double *grad, hipStream_t st )
{
    hipLaunchKernelGGL( reduce_grad_kernel, dim3( 1 ), dim3( 256 ), 0, st, part, n_tasks, npar, grad );
    return hipGetLastError();
}

} // namespace nufi_impl
