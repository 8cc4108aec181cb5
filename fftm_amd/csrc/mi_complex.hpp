// Complex arithmetic and small-radix DFT butterflies for the CDNA4 FFT passes.
//
// All butterflies compute the unnormalised DFT  y[m] = sum_q x[q] e^{s 2 pi i q m / R}
// with s = -1 (forward, INV = false) or s = +1 (inverse, INV = true), matching the
// hipFFT/FFTW sign convention used by ffts (HIPFFT_FORWARD = -1, HIPFFT_BACKWARD = +1;
// source/external_wrap/hipfft_wrap.h:363-417).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace fftm_mi
{

template <typename T>
struct alignas( 2 * sizeof( T ) ) cpx
{
    T x, y;
};

template <typename T>
__device__ __forceinline__ cpx<T> mk( T a, T b )
{
    cpx<T> r;
    r.x = a;
    r.y = b;
    return r;
}

template <typename T>
__device__ __forceinline__ cpx<T> add( cpx<T> a, cpx<T> b )
{
    return mk<T>( a.x + b.x, a.y + b.y );
}

template <typename T>
__device__ __forceinline__ cpx<T> sub( cpx<T> a, cpx<T> b )
{
    return mk<T>( a.x - b.x, a.y - b.y );
}

// Fused multiply-add in the precision of T (one rounding; v_fma_f32 / v_fma_f64).
__device__ __forceinline__ float fmat( float a, float b, float c ) { return __builtin_fmaf( a, b, c ); }
__device__ __forceinline__ double fmat( double a, double b, double c ) { return __builtin_fma( a, b, c ); }

// Complex products use explicit fused multiply-adds (the library is compiled with
// -ffp-contract=off), so every kernel instantiation rounds identically whatever the
// unrolling: tile-shape variants stay bitwise equal.
template <typename T>
__device__ __forceinline__ cpx<T> mul( cpx<T> a, cpx<T> b )
{
    return mk<T>( fmat( a.x, b.x, -( a.y * b.y ) ), fmat( a.x, b.y, a.y * b.x ) );
}

// a * conj(b)
template <typename T>
__device__ __forceinline__ cpx<T> mulc( cpx<T> a, cpx<T> b )
{
    return mk<T>( fmat( a.x, b.x, a.y * b.y ), fmat( a.y, b.x, -( a.x * b.y ) ) );
}

template <typename T>
__device__ __forceinline__ cpx<T> scl( cpx<T> a, T s )
{
    return mk<T>( a.x * s, a.y * s );
}

template <typename T>
__device__ __forceinline__ cpx<T> conj( cpx<T> a )
{
    return mk<T>( a.x, -a.y );
}

// multiply by s*i  (s = -1 forward, +1 inverse)
template <bool INV, typename T>
__device__ __forceinline__ cpx<T> mul_si( cpx<T> a )
{
    return INV ? mk<T>( -a.y, a.x ) : mk<T>( a.y, -a.x );
}

// twiddle multiply: a * w (forward) or a * conj(w) (inverse), w = e^{-2 pi i k / N}
template <bool INV, typename T>
__device__ __forceinline__ cpx<T> twmul( cpx<T> a, cpx<T> w )
{
    return INV ? mulc( a, w ) : mul( a, w );
}

// ---------------------------------------------------------------------------
// Butterflies on register arrays
// ---------------------------------------------------------------------------

template <bool INV, typename T>
__device__ __forceinline__ void dft2( cpx<T> *v )
{
    const cpx<T> a = v[0], b = v[1];
    v[0]               = add( a, b );
    v[1]               = sub( a, b );
}

template <bool INV, typename T>
__device__ __forceinline__ void dft4( cpx<T> *v )
{
    const cpx<T> a = add( v[0], v[2] ), b = sub( v[0], v[2] );
    const cpx<T> c = add( v[1], v[3] ), d = mul_si<INV>( sub( v[1], v[3] ) );
    v[0]               = add( a, c );
    v[2]               = sub( a, c );
    v[1]               = add( b, d );
    v[3]               = sub( b, d );
}

// radix 8 = radix-2 DIF split followed by two radix-4 DFTs (in-place, natural order)
template <bool INV, typename T>
__device__ __forceinline__ void dft8( cpx<T> *v )
{
    const T      c = (T)0.70710678118654752440084436210484904;
    cpx<T>       a[4], b[4];
#pragma unroll
    for ( int i = 0; i < 4; ++i )
    {
        a[i] = add( v[i], v[i + 4] );
        b[i] = sub( v[i], v[i + 4] );
    }
    // b1 *= W8^{s}, b2 *= W8^{2s} = s*i, b3 *= W8^{3s}
    if ( !INV )
    {
        b[1] = mk<T>( c * ( b[1].x + b[1].y ), c * ( b[1].y - b[1].x ) );
        b[3] = mk<T>( c * ( b[3].y - b[3].x ), -c * ( b[3].x + b[3].y ) );
    }
    else
    {
        b[1] = mk<T>( c * ( b[1].x - b[1].y ), c * ( b[1].x + b[1].y ) );
        b[3] = mk<T>( -c * ( b[3].x + b[3].y ), c * ( b[3].x - b[3].y ) );
    }
    b[2] = mul_si<INV>( b[2] );
    dft4<INV>( a );
    dft4<INV>( b );
#pragma unroll
    for ( int i = 0; i < 4; ++i )
    {
        v[2 * i]     = a[i];
        v[2 * i + 1] = b[i];
    }
}

// radix 16 = 4 x 4 with internal twiddles W16^{n2 k1}
template <bool INV, typename T>
__device__ __forceinline__ void dft16( cpx<T> *v )
{
    const T c1 = (T)0.92387953251128675612818318939678829; // cos(pi/8)
    const T s1 = (T)0.38268343236508977172845998403039887; // sin(pi/8)
    const T c2 = (T)0.70710678118654752440084436210484904; // cos(pi/4)
    cpx<T>  y[4][4];
#pragma unroll
    for ( int n2 = 0; n2 < 4; ++n2 )
    {
        cpx<T> u[4] = { v[n2], v[n2 + 4], v[n2 + 8], v[n2 + 12] };
        dft4<INV>( u );
#pragma unroll
        for ( int k1 = 0; k1 < 4; ++k1 )
            y[n2][k1] = u[k1];
    }
    // W16^e for e = n2*k1 in {1,2,3,4,6,9}: (cos, -sin) of e*pi/8 for forward
    const T sg = INV ? (T)1 : (T)-1;
    const cpx<T> w1 = mk<T>( c1, sg * s1 ), w2 = mk<T>( c2, sg * c2 ), w3 = mk<T>( s1, sg * c1 );
    const cpx<T> w6 = mk<T>( -c2, sg * c2 ), w9 = mk<T>( -c1, -sg * s1 );
    y[1][1] = mul( y[1][1], w1 );
    y[1][2] = mul( y[1][2], w2 );
    y[1][3] = mul( y[1][3], w3 );
    y[2][1] = mul( y[2][1], w2 );
    y[2][2] = mul_si<INV>( y[2][2] ); // W16^4 = s*i
    y[2][3] = mul( y[2][3], w6 );
    y[3][1] = mul( y[3][1], w3 );
    y[3][2] = mul( y[3][2], w6 );
    y[3][3] = mul( y[3][3], w9 );
#pragma unroll
    for ( int k1 = 0; k1 < 4; ++k1 )
    {
        cpx<T> u[4] = { y[0][k1], y[1][k1], y[2][k1], y[3][k1] };
        dft4<INV>( u );
#pragma unroll
        for ( int k2 = 0; k2 < 4; ++k2 )
            v[k1 + 4 * k2] = u[k2];
    }
}

template <bool INV, typename T>
__device__ __forceinline__ void dft3( cpx<T> *v )
{
    const T      s  = (T)0.86602540378443864676372317075293618; // sqrt(3)/2
    const cpx<T> t1 = add( v[1], v[2] );
    const cpx<T> d  = sub( v[1], v[2] );
    const cpx<T> t2 = mk<T>( v[0].x - (T)0.5 * t1.x, v[0].y - (T)0.5 * t1.y );
    v[0]            = add( v[0], t1 );
    // (s_sign * i) * sqrt(3)/2 * d
    const cpx<T> e  = mul_si<INV>( scl( d, s ) );
    v[1]            = add( t2, e );
    v[2]            = sub( t2, e );
}

// cos and sin of 2 pi m / R, m = 1 .. (R - 1) / 2
template <int R>
struct roots_of_unity;
template <>
struct roots_of_unity<5>
{
    static constexpr double c[] = { 0.309016994374947424102293417182819058, -0.80901699437494742410229341718281905 };
    static constexpr double s[] = { 0.951056516295153572116439333379382143, 0.587785252292473129168705954639072768 };
};
template <>
struct roots_of_unity<7>
{
    static constexpr double c[] = { 0.623489801858733530525004884004239810, -0.22252093395631440428890256449679475,
                                    -0.90096886790241912623610231950744505 };
    static constexpr double s[] = { 0.781831482468029808708444526674057750, 0.974927912181823607018131682993931217,
                                    0.433883739117558120475768332848358754 };
};
template <>
struct roots_of_unity<11>
{
    static constexpr double c[] = { 0.841253532831181168861811648919367717, 0.415415013001886425529274149229623203,
                                    -0.14231483827328514044379266861636966, -0.65486073394528506405692507246629355,
                                    -0.95949297361449738989036805706632769 };
    static constexpr double s[] = { 0.540640817455597582107635954318691695, 0.909631995354518371411715383079028460,
                                    0.989821441880932732376092037776718787, 0.755749574354258283774035843972344420,
                                    0.281732556841429697711417915346616899 };
};
template <>
struct roots_of_unity<13>
{
    static constexpr double c[] = { 0.885456025653209895900375522015098878, 0.568064746731155802511807559127516624,
                                    0.120536680255323053349067687452543582, -0.35460488704253562596963789260001847,
                                    -0.74851074817110109863463059970135138, -0.97094181742605202715698227629378922 };
    static constexpr double s[] = { 0.464723172043768545656015335133104777, 0.822983865893656394579617423439381990,
                                    0.992708874098053992800751649492520179, 0.935016242685414823439784599837830729,
                                    0.663122658240795202376785492666766279, 0.239315664287557767148753726260211895 };
};

// Odd prime radix: the inputs q and R - q enter every output through their sum a_q and
// difference b_q, y[m], y[R - m] = sum_q a_q cos(2 pi q m / R) +- s i sum_q b_q sin(...).
template <int R, bool INV, typename T>
__device__ __forceinline__ void dft_prime( cpx<T> *v )
{
    using W         = roots_of_unity<R>;
    constexpr int H = ( R - 1 ) / 2;
    cpx<T>        a[H], b[H];
    const cpx<T>  x0 = v[0];
    cpx<T>        y0 = x0;
#pragma unroll
    for ( int q = 0; q < H; ++q )
    {
        a[q] = add( v[q + 1], v[R - 1 - q] );
        b[q] = sub( v[q + 1], v[R - 1 - q] );
        y0   = add( y0, a[q] );
    }
    v[0] = y0;
#pragma unroll
    for ( int m = 1; m <= H; ++m )
    {
        cpx<T> r = x0, t = mk<T>( 0, 0 );
#pragma unroll
        for ( int q = 1; q <= H; ++q )
        {
            const int e = q * m % R;
            const T   c = (T)W::c[( e <= H ? e : R - e ) - 1];
            const T   s = e <= H ? (T)W::s[e - 1] : -(T)W::s[R - e - 1];
            r           = mk<T>( fmat( c, a[q - 1].x, r.x ), fmat( c, a[q - 1].y, r.y ) );
            t           = q == 1 ? scl( b[0], s ) : mk<T>( fmat( s, b[q - 1].x, t.x ), fmat( s, b[q - 1].y, t.y ) );
        }
        t        = mul_si<INV>( t );
        v[m]     = add( r, t );
        v[R - m] = sub( r, t );
    }
}

template <int R, bool INV, typename T>
__device__ __forceinline__ void dft_fixed( cpx<T> *v );

// R = A B with coprime factors (Good 1958, Thomas 1963): input n = n1 B + n2 A mod R and
// output k = k1 mod A = k2 mod B turn the DFT into A x B with no twiddles.
template <int A, int B, bool INV, typename T>
__device__ __forceinline__ void dft_coprime( cpx<T> *v )
{
    constexpr int R = A * B;
    cpx<T>        y[A][B];
#pragma unroll
    for ( int n2 = 0; n2 < B; ++n2 )
    {
        cpx<T> u[A];
#pragma unroll
        for ( int n1 = 0; n1 < A; ++n1 )
            u[n1] = v[( n1 * B + n2 * A ) % R];
        dft_fixed<A, INV>( u );
#pragma unroll
        for ( int k1 = 0; k1 < A; ++k1 )
            y[k1][n2] = u[k1];
    }
#pragma unroll
    for ( int k1 = 0; k1 < A; ++k1 )
    {
        dft_fixed<B, INV>( y[k1] );
#pragma unroll
        for ( int k = 0; k < R; ++k )
            if ( k % A == k1 )
                v[k] = y[k1][k % B];
    }
}

// radix 9 = 3 x 3 with the twiddles W9, W9^2, W9^4
template <bool INV, typename T>
__device__ __forceinline__ void dft9( cpx<T> *v )
{
    const T      sg = INV ? (T)1 : (T)-1;
    const cpx<T> w1 = mk<T>( (T)0.766044443118978035202392650555416673, sg * (T)0.642787609686539326322643409907263432 );
    const cpx<T> w2 = mk<T>( (T)0.173648177666930348851716626769314796, sg * (T)0.984807753012208059366743024589523013 );
    const cpx<T> w4 = mk<T>( (T)-0.93969262078590838405410927732473146, sg * (T)0.342020143325668733044099614682259580 );
    cpx<T>       y[3][3];
#pragma unroll
    for ( int n2 = 0; n2 < 3; ++n2 )
    {
        cpx<T> u[3] = { v[n2], v[n2 + 3], v[n2 + 6] };
        dft3<INV>( u );
#pragma unroll
        for ( int k1 = 0; k1 < 3; ++k1 )
            y[k1][n2] = u[k1];
    }
    y[1][1] = mul( y[1][1], w1 );
    y[1][2] = mul( y[1][2], w2 );
    y[2][1] = mul( y[2][1], w2 );
    y[2][2] = mul( y[2][2], w4 );
#pragma unroll
    for ( int k1 = 0; k1 < 3; ++k1 )
    {
        dft3<INV>( y[k1] );
#pragma unroll
        for ( int k2 = 0; k2 < 3; ++k2 )
            v[k1 + 3 * k2] = y[k1][k2];
    }
}

template <int R, bool INV, typename T>
__device__ __forceinline__ void dft_fixed( cpx<T> *v )
{
    if constexpr ( R == 2 )
        dft2<INV>( v );
    else if constexpr ( R == 3 )
        dft3<INV>( v );
    else if constexpr ( R == 4 )
        dft4<INV>( v );
    else if constexpr ( R == 5 || R == 7 || R == 11 || R == 13 )
        dft_prime<R, INV>( v );
    else if constexpr ( R == 6 )
        dft_coprime<2, 3, INV>( v );
    else if constexpr ( R == 8 )
        dft8<INV>( v );
    else if constexpr ( R == 9 )
        dft9<INV>( v );
    else if constexpr ( R == 10 )
        dft_coprime<2, 5, INV>( v );
    else if constexpr ( R == 12 )
        dft_coprime<4, 3, INV>( v );
    else if constexpr ( R == 14 )
        dft_coprime<2, 7, INV>( v );
    else if constexpr ( R == 15 )
        dft_coprime<3, 5, INV>( v );
    else if constexpr ( R == 16 )
        dft16<INV>( v );
    else
        static_assert( R == 1, "no butterfly of this radix" );
}

// ---------------------------------------------------------------------------
// Workgroup -> tile mapping that keeps neighbouring tiles on one XCD.
// Workgroups are dispatched round-robin over the 8 XCDs (wg i -> XCD i % 8), so
// consecutive tiles (which share cache lines at their edges) are assigned to the
// workgroups i, i+8, i+16, ... of the same XCD and its L2.
// ---------------------------------------------------------------------------
// Chunks of CH consecutive tiles per XCD, the chunks dealt to the XCDs round-robin
// (workgroup w runs on XCD w % 8).  Workgroups past the last whole round keep their own
// index, so the mapping stays a permutation of [0, nwg).
__device__ __forceinline__ int64_t xcd_chunk( int64_t wg, int64_t nwg, int64_t ch )
{
    constexpr int64_t NX   = 8;
    const int64_t     full = nwg / ( NX * ch ) * ( NX * ch );
    if ( wg >= full )
        return wg;
    const int64_t x = wg % NX, k = wg / NX;
    return ( ( k / ch ) * NX + x ) * ch + k % ch;
}

__device__ __forceinline__ int64_t xcd_tile( int64_t wg, int64_t nwg )
{
    constexpr int64_t NX = 8;
    if ( nwg < 2 * NX )
        return wg;
    const int64_t xcd  = wg % NX;
    const int64_t k    = wg / NX;
    const int64_t base = nwg / NX, rem = nwg % NX;
    const int64_t start = xcd * base + ( xcd < rem ? xcd : rem );
    return start + k;
}

} // namespace fftm_mi
