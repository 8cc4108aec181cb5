// Diagonal operators on an ffts half spectrum (no reference counterpart as a library
// entry point; the reference applies such operators in caller functors, e.g.
// solve_poisson_3d_functor, versioned_ffts_3d_test_driver.h:128-154, and the
// spectral kernels of examples/turbulence/source/spacetime_kernels.h:66-145).
//
// Wavenumbers follow the reference drivers: k = i <= n/2 ? i : i - n on full axes
// (Nyquist positive), k = i on the halved real axis.  A radial shell filter uses
// S shells of equal width over [0, kmax], kmax = sqrt(sum_a (n_a/2)^2):
//   shell(k) = min(S - 1, floor(S * |k| / kmax)), evaluated exactly (shell_of).
#pragma once

#include "mi_complex.hpp"
#include "mi_pass.hpp"

namespace fftm_mi
{

struct spec_geom
{
    int32_t nd;        // 3 or 4
    int32_t half_axis; // logical index of the halved (real) axis
    int64_t ext[4];    // memory extents, slowest..fastest
    int32_t ax[4];     // logical axis of each memory axis
    int64_t n[4];      // full logical lengths per logical axis
    int64_t total;     // number of complex bins
    int64_t kmax2;     // sum over axes of (n_a / 2)^2
    uint64_t mg[4];    // division by ext[m] as a multiply and a shift (mg = 0: divide)
    int32_t  sh[4];
};

constexpr int SHELL_BLOCKS = 512;
constexpr int MAX_SHELLS   = 1024;

// The half spectrum as up to three slow memory axes and the fastest one (axes 0..3, slowest
// first; missing axes have extent 1), and one launch's walk over its rows.
struct spec_walk
{
    int32_t ext[4]; // extents
    int32_t n[4];   // full logical lengths; 0 marks the halved real axis and missing axes
    int32_t rows;   // rows per sweep
    int32_t s0, s1, s2; // `rows` in the mixed radix of axes 0..2
    int32_t dax;    // axis whose wavenumber is wanted (-1: none)
    int64_t total;  // bins
};

// How a grid of NT threads walks a dense half spectrum: the threads cover `rows` whole rows
// of the fastest axis per sweep, so a thread keeps its column for the whole walk and steps
// `rows` rows at a time, carrying the slower coordinates along (no division per bin).
// Consecutive threads touch consecutive bins.  Deriving every bin's coordinates by one
// multiply-and-shift division per axis, with one bin in flight per thread, the 256^3 shell
// multiply took 49 us (2.8 TB/s); walked this way it takes 29 us (4.7 TB/s) and is bound by
// the memory it moves, as is the FP64 derivative of 192 x 160 x 73 bins (14.8 -> 13.3 us).
template <typename F>
__device__ __forceinline__ void walk_rows( const spec_walk &w, F &&body )
{
    const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t r = g / (uint32_t)w.ext[3], c = g - r * (uint32_t)w.ext[3];
    if ( r >= (uint32_t)w.rows )
        return;
    int           i2 = (int)( r % (uint32_t)w.ext[2] );
    const uint32_t q = r / (uint32_t)w.ext[2];
    int           i1 = (int)( q % (uint32_t)w.ext[1] );
    int           i0 = (int)( q / (uint32_t)w.ext[1] );
    auto sq = [&]( int m, int i, int &k ) {
        k = w.n[m] == 0 || i <= w.n[m] / 2 ? i : i - w.n[m];
        return k * k;
    };
    int       kc[4] = { 0, 0, 0, 0 };
    const int k2c   = sq( 3, (int)c, kc[3] );
    const int64_t step = (int64_t)w.rows * w.ext[3];
    int64_t       at   = (int64_t)r * w.ext[3] + c;
    // U bins per trip, all loaded before the first is used
    constexpr int U = 4;
    while ( at < w.total )
    {
        int64_t o[U];
        int     k2[U], kd[U];
#pragma unroll
        for ( int u = 0; u < U; ++u )
        {
            o[u]  = at;
            k2[u] = k2c + sq( 2, i2, kc[2] ) + sq( 1, i1, kc[1] ) + sq( 0, i0, kc[0] );
            kd[u] = w.dax < 0 ? 0 : ( w.dax == 3 ? kc[3] : ( w.dax == 2 ? kc[2] : ( w.dax == 1 ? kc[1] : kc[0] ) ) );
            at += step;
            i2 += w.s2;
            i1 += w.s1;
            i0 += w.s0;
            if ( i2 >= w.ext[2] )
            {
                i2 -= w.ext[2];
                ++i1;
            }
            if ( i1 >= w.ext[1] )
            {
                i1 -= w.ext[1];
                ++i0;
            }
        }
        body( o, k2, kd );
    }
}

// out[i] = H_i * in[i], H_i = filter[i] (per bin, real)
template <typename T>
__global__ void __launch_bounds__( 256 ) k_filter_multiply( int64_t total, const cpx<T> *in, cpx<T> *out, const T *filter )
{
    constexpr int U    = 4;
    const int64_t step = (int64_t)gridDim.x * 256;
    for ( int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += U * step )
    {
        cpx<T> z[U];
        T      h[U];
#pragma unroll
        for ( int u = 0; u < U; ++u )
        {
            const int64_t j = i + u * step < total ? i + u * step : i;
            z[u]            = in[j];
            h[u]            = filter[j];
        }
#pragma unroll
        for ( int u = 0; u < U; ++u )
            if ( i + u * step < total )
                out[i + u * step] = scl( z[u], h[u] );
    }
}

// out[i] = coeffs[shell(i)] in[i].  A thread's next bin lies w.rows rows on and so, in a large
// array, many shells away: walking a table of shell bounds from the last bin's shell cost a
// dependent LDS read per shell passed (128^3 FP32: 6.8 us with 32 shells, 9.5 with 100, 51 with
// 1024; 5.5 with any number now, 256^3 27.0 -> 21.7 with 32).
template <typename T>
__global__ void __launch_bounds__( 256 )
    k_shell_multiply( const spec_walk w, int S, int64_t kmax2, const cpx<T> *in, cpx<T> *out, const T *coeffs )
{
    walk_rows( w, [&]( const int64_t( &o )[4], const int( &k2 )[4], const int( & )[4] ) {
        cpx<T> z[4];
        T      h[4];
#pragma unroll
        for ( int u = 0; u < 4; ++u )
        {
            z[u] = in[o[u] < w.total ? o[u] : o[0]];
            h[u] = coeffs[shell_of( k2[u], S, kmax2 )];
        }
#pragma unroll
        for ( int u = 0; u < 4; ++u )
            if ( o[u] < w.total )
                out[o[u]] = scl( z[u], h[u] );
    } );
}

// out[i] = H(k_i) in[i] for an analytic operator (Poisson, Gaussian, radial shells) on
// the dense half-spectrum layout
template <typename T>
__global__ void __launch_bounds__( 256 )
    k_spectral_op( const spec_walk w, const filter_params<T> f, const cpx<T> *in, cpx<T> *out )
{
    walk_rows( w, [&]( const int64_t( &o )[4], const int( &k2 )[4], const int( &kd )[4] ) {
        cpx<T> z[4];
#pragma unroll
        for ( int u = 0; u < 4; ++u )
            z[u] = in[o[u] < w.total ? o[u] : o[0]];
        with_filter_kind( f, [&]( auto op ) {
#pragma unroll
            for ( int u = 0; u < 4; ++u )
                if ( o[u] < w.total )
                    out[o[u]] = apply_h( z[u], filter_h<op()>( f, (float)k2[u], (float)kd[u] ), op() );
        } );
    } );
}

// partial[b * S + s] = sum over this block's bins in shell s of Re(conj(G_i) X_i), in FP64.
// A thread keeps its sum in a register while its bins stay in one shell and adds it to the
// block's LDS sums when the shell changes.  The shell changes at most bins where there are
// many (79 % of them at 256^3 with 32 shells, 98 % at 128^3 with 100); with few, the register
// keeps 64 lanes off a handful of addresses.  256^3 FP32 with the reduction, microseconds with
// 1 / 8 / 32 / 100 / 1024 shells: 23.7 / 24.9 / 31.5 / 25.5 / 28.0 (24.5 / 28.6 / 39.2 / 35.2 / 104
// with a walk over a table of shell bounds from the last bin's shell, 114 / 151 / 196 / 196 / 197
// with an atomic and a division per bin); 128^3 with 1024: 86 -> 12.
template <typename T>
__global__ void __launch_bounds__( 512 ) k_shell_partials( const spec_walk w, int S, int64_t kmax2, const cpx<T> *G,
                                                           const cpx<T> *X, double *partial )
{
    extern __shared__ double acc[];
    for ( int s = threadIdx.x; s < S; s += 512 )
        acc[s] = 0.0;
    __syncthreads();
    int    s   = -1;
    double sum = 0.0;
    walk_rows( w, [&]( const int64_t( &o )[4], const int( &k2 )[4], const int( & )[4] ) {
        cpx<T> a[4], b[4];
#pragma unroll
        for ( int u = 0; u < 4; ++u )
        {
            const int64_t j = o[u] < w.total ? o[u] : o[0];
            a[u]            = G[j];
            b[u]            = X[j];
        }
#pragma unroll
        for ( int u = 0; u < 4; ++u )
            if ( o[u] < w.total )
            {
                const int t = shell_of( k2[u], S, kmax2 );
                if ( t != s )
                {
                    if ( s >= 0 )
                        atomicAdd( &acc[s], sum );
                    sum = 0.0;
                    s   = t;
                }
                sum += (double)a[u].x * (double)b[u].x + (double)a[u].y * (double)b[u].y;
            }
    } );
    if ( s >= 0 )
        atomicAdd( &acc[s], sum );
    __syncthreads();
    for ( int i = threadIdx.x; i < S; i += 512 )
        partial[(int64_t)blockIdx.x * S + i] = acc[i];
}

// grad[s] = sum_b partial[b * S + s], in a fixed order: one wave per shell, 64 strided
// sums, then a butterfly over the lanes.  (One thread per shell walking all 512 partials,
// a load latency apart, took 122 us; this takes 5.)
template <typename T>
__global__ void __launch_bounds__( 256 ) k_shell_reduce( const double *partial, int nblocks, int nshells, T *grad )
{
    const int s = blockIdx.x * 4 + threadIdx.x / 64;
    const int l = threadIdx.x % 64;
    if ( s >= nshells )
        return;
    double sum = 0.0;
#pragma unroll 8
    for ( int b = l; b < nblocks; b += 64 )
        sum += partial[(int64_t)b * nshells + s];
#pragma unroll
    for ( int d = 32; d > 0; d >>= 1 )
        sum += __shfl_xor( sum, d, 64 );
    if ( l == 0 )
        grad[s] = (T)sum;
}

} // namespace fftm_mi
