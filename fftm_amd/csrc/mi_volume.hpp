// Volume pass: the real axis and one or more complex axes in one workgroup and one launch: a
// whole small transform, or the planes of a larger one's two inner axes, a workgroup each.
//
// Problems of a few thousand points are bound by their launches: a 12 x 10 x 8 FP64 pair
// took six kernels of 3 to 5.5 us, each nearly all latency, 28 us in all; two of these take
// 16.4, 16^3 23 instead of 27.  They are bound by one wave's chain of latencies (about 1300
// instructions for 4^3), so the loops divide by multiplying and no stage's indices are formed
// ahead of its turn.  Here the array stays in LDS
// from the first load to the last store.  Every radix stage of every axis reads one LDS
// buffer and writes the other (one barrier per stage); the first stage reads HBM, the last
// one writes HBM.  Real rows are transformed in pairs as in the pass kernel; the separation
// of a pair is folded into the reads of the first complex axis, the Hermitian extension of
// the backward transform into the reads of the real axis.
//
// Every radix to 16 of both kinds of axis is in one kernel: 72 / 124 registers FP32 forward /
// inverse, 128 / 194 FP64 (two waves per SIMD), and 108..392 scalar values kept in vector lanes.
#pragma once

#include "mi_any.hpp"

namespace fftm_mi
{

constexpr int VOL_MAX_STAGES = 3; // per axis
constexpr int vol_max_threads( int csize ) { return csize == 8 ? 1024 : 512; }
constexpr int vol_lds_limit() { return 150 * 1024; }

// What an axis's stages do at their ends: the first reads HBM or separates paired real
// lines, the last writes HBM.
enum : int
{
    VOL_READ  = 1,
    VOL_SEP   = 2,
    VOL_WRITE = 4
};

struct vol_axis
{
    int32_t  n, nst;
    int32_t  r[VOL_MAX_STAGES];
    int32_t  st, rst;      // distance in the LDS array of consecutive elements, in values and rows
    int32_t  gs;           // stride in the complex array (real axis: in the real array)
    int32_t  tw;           // offset of the axis's twiddles in the LDS table
    int32_t  ffwd, fbwd;   // VOL_* flags, forward and backward
    int32_t  lines;        // complex axes: lines along the axis
    int32_t  tst[VOL_MAX_STAGES]; // n / ( span r ) of each stage
    uint32_t mg_st, mg_lines;     // divisions by st, lines
    uint32_t mg_ns[VOL_MAX_STAGES], mg_nbf[VOL_MAX_STAGES]; // by the span, by n / r
};
// One stage of an axis: span before it, twiddle step, divisions by the span and by n / r.
struct vol_stage
{
    int32_t  ns, tst;
    uint32_t mg_ns, mg_nbf;
};

// The LDS array is [o0][o1][o2][k], k over the nh bins of the real axis (rows of the real
// array: the same with nz elements); missing outer axes have extent 1.
struct vol_geom
{
    vol_axis ax[4];            // o0, o1, o2, real
    int32_t  ext[3];
    int32_t  nz, nh, rows, pairs;
    int32_t  elems, twelems;   // LDS values: each of the two buffers, the twiddle tables
    int32_t  nt;               // threads
    // workgroups: one, or one per item of up to two batch axes (extent of the faster one and
    // the strides in the real and the complex array, faster first)
    int32_t  blocks, bd0;
    int64_t  bsr[2], bsc[2];
    uint32_t mg_nh, mg_e1, mg_e2;
    int32_t  sr[4], sc[4];     // element strides of the real and the complex array
};
template <typename T>
struct vol_params : vol_geom
{
    const void   *in;
    void         *out;
    const cpx<T> *twg[4]; // length tables
    int32_t       wmode;  // as pass_params::wmode
};

template <typename T, bool FWD>
struct vol_kernel
{
    using C = cpx<T>;

    // the workgroup's pieces of the arrays (a kernel reads one kind and writes the other)
    struct io
    {
        const C *cin;
        C       *cout;
        const T *rin;
        T       *rout;
    };

    __device__ static __forceinline__ int quot( int n, int d, uint32_t mg )
    {
        return d == 1 ? n : (int)__umulhi( (uint32_t)n, mg );
    }

    // offset of row r (all outer axes) with strides s
    __device__ static __forceinline__ int row_offset( const vol_params<T> &p, int r, const int32_t ( &s )[4] )
    {
        const int q1 = quot( r, p.ext[2], p.mg_e2 ), i2 = r - q1 * p.ext[2];
        const int i0 = quot( q1, p.ext[1], p.mg_e1 ), i1 = q1 - i0 * p.ext[1];
        return i0 * s[0] + i1 * s[1] + i2 * s[2];
    }

    // One stage of complex axis a (gr reads HBM, gw writes HBM, sep reads the paired real lines
    // and separates them).
    template <int R>
    __device__ static __forceinline__ void complex_stage( const vol_params<T> &p, const io &f, const vol_axis &a,
                                                          const vol_stage &g, const C *src, C *dst, const C *tw, bool sep,
                                                          bool gr, bool gw )
    {
        int nbf = a.n / R, gs = a.gs;
        // opaque: what follows from them is not formed for every radix ahead of the switch
        asm volatile( "" : "+s"( nbf ), "+s"( gs ) );
        const int ns = g.ns, lines = a.lines, items = lines * nbf;
        for ( int item = threadIdx.x; item < items; item += blockDim.x )
        {
            // lanes walk the lines (the inner axes are contiguous), then the butterflies
            const int j    = quot( item, lines, a.mg_lines );
            const int l    = item - j * lines;
            const int o    = quot( l, a.st, a.mg_st );
            const int base = o * a.n * a.st + ( l - o * a.st );
            const int row  = quot( base, p.nh, p.mg_nh ), k = base - row * p.nh;
            const int off = ( gr || gw ) ? row_offset( p, row, p.sc ) + k * p.sc[3] : 0;
            C             v[R];
            if ( gr )
            {
                const C *in = f.cin + off + j * gs;
#pragma unroll
                for ( int r = 0; r < R; ++r )
                    v[r] = mk<T>( in[r * nbf * gs].x, in[r * nbf * gs].y );
            }
            else if ( sep )
            {
                // A[k] = (Z[k] + conj Z[n-k]) / 2 (even rows), B[k] = (Z[k] - conj Z[n-k]) / 2i
                const T   h  = ( p.wmode == 1 && k != 0 && 2 * k != p.nz ) ? (T)1 : (T)0.5;
                const int km = k == 0 ? 0 : p.nz - k;
#pragma unroll
                for ( int r = 0; r < R; ++r )
                {
                    const int rr = row + ( j + r * nbf ) * a.rst;
                    const C   zk = src[( rr >> 1 ) * p.nz + k], zm = src[( rr >> 1 ) * p.nz + km];
                    v[r]         = rr & 1 ? mk<T>( h * ( zk.y + zm.y ), h * ( zm.x - zk.x ) )
                                          : mk<T>( h * ( zk.x + zm.x ), h * ( zk.y - zm.y ) );
                }
            }
            else
            {
#pragma unroll
                for ( int r = 0; r < R; ++r )
                    v[r] = src[base + ( j + r * nbf ) * a.st];
            }
            int d = j * R;
            if ( ns > 1 )
            {
                const int q = (int)__umulhi( (uint32_t)j, g.mg_ns );
                const int t = ( j - q * ns ) * g.tst;
                d           = q * ns * ( R - 1 ) + j;
#pragma unroll
                for ( int r = 1; r < R; ++r )
                    v[r] = twmul<!FWD>( v[r], tw[r * t] );
            }
            dft_fixed<R, !FWD>( v );
            if ( gw )
            {
                C *out = f.cout + off + d * gs;
#pragma unroll
                for ( int m = 0; m < R; ++m )
                    out[m * ns * gs] = v[m];
            }
            else
            {
#pragma unroll
                for ( int m = 0; m < R; ++m )
                    dst[base + ( d + m * ns ) * a.st] = v[m];
            }
        }
    }

    // One stage of the real axis: line q holds rows 2 q and 2 q + 1.  first: from the real
    // array (forward) or the half spectra in LDS (backward); last of the backward transform:
    // to the real array.
    template <int R>
    __device__ static __forceinline__ void real_stage( const vol_params<T> &p, const io &f, const vol_axis &a,
                                                       const vol_stage &g, const C *src, C *dst, const C *tw, bool first,
                                                       bool last )
    {
        int nbf = a.n / R, gs = a.gs;
        asm volatile( "" : "+s"( nbf ), "+s"( gs ) );
        const int ns = g.ns, items = p.pairs * nbf;
        for ( int item = threadIdx.x; item < items; item += blockDim.x )
        {
            const int  q = quot( item, nbf, g.mg_nbf ), j = item - q * nbf;
            const bool vb = 2 * q + 1 < p.rows;
            C          v[R];
            if ( first && FWD )
            {
                const T *sa = f.rin + row_offset( p, 2 * q, p.sr ) + j * gs;
                const T *sb = vb ? f.rin + row_offset( p, 2 * q + 1, p.sr ) + j * gs : sa;
#pragma unroll
                for ( int r = 0; r < R; ++r )
                    v[r] = mk<T>( sa[r * nbf * gs], sb[r * nbf * gs] );
                if ( !vb )
                {
#pragma unroll
                    for ( int r = 0; r < R; ++r )
                        v[r].y = (T)0;
                }
            }
            else if ( first )
            {
                // z = A~ + i B~ (the imaginary parts of the DC and Nyquist bins are ignored)
#pragma unroll
                for ( int r = 0; r < R; ++r )
                {
                    const int  n  = j + r * nbf;
                    const bool up = 2 * n > a.n;
                    const int  nn = up ? a.n - n : n;
                    C          za = src[2 * q * p.nh + nn];
                    C          zb = vb ? src[( 2 * q + 1 ) * p.nh + nn] : mk<T>( 0, 0 );
                    if ( n == 0 || 2 * n == a.n )
                    {
                        za.y = (T)0;
                        zb.y = (T)0;
                    }
                    else if ( p.wmode == 2 )
                    {
                        za = scl( za, (T)0.5 );
                        zb = scl( zb, (T)0.5 );
                    }
                    v[r] = up ? mk<T>( za.x + zb.y, zb.x - za.y ) : mk<T>( za.x - zb.y, za.y + zb.x );
                }
            }
            else
            {
#pragma unroll
                for ( int r = 0; r < R; ++r )
                    v[r] = src[q * p.nz + j + r * nbf];
            }
            int d = j * R;
            if ( ns > 1 )
            {
                const int o = (int)__umulhi( (uint32_t)j, g.mg_ns );
                const int t = ( j - o * ns ) * g.tst;
                d           = o * ns * ( R - 1 ) + j;
#pragma unroll
                for ( int r = 1; r < R; ++r )
                    v[r] = twmul<!FWD>( v[r], tw[r * t] );
            }
            dft_fixed<R, !FWD>( v );
            if ( last && !FWD )
            {
                T *da = f.rout + row_offset( p, 2 * q, p.sr ) + d * gs;
#pragma unroll
                for ( int m = 0; m < R; ++m )
                    da[m * ns * gs] = v[m].x;
                if ( vb )
                {
                    T *db = f.rout + row_offset( p, 2 * q + 1, p.sr ) + d * gs;
#pragma unroll
                    for ( int m = 0; m < R; ++m )
                        db[m * ns * gs] = v[m].y;
                }
            }
            else
            {
#pragma unroll
                for ( int m = 0; m < R; ++m )
                    dst[q * p.nz + d + m * ns] = v[m];
            }
        }
    }

    template <int R>
    __device__ static __forceinline__ void stage( const vol_params<T> &p, const io &f, const vol_axis &a, bool real,
                                                  const vol_stage &g, const C *src, C *dst, const C *tw, bool sep,
                                                  bool gr, bool gw )
    {
        // the markers keep the radices' register arrays apart, see any_kernel::stage_r
        if ( real )
        {
            real_stage<R>( p, f, a, g, src, dst, tw, gr, gw );
            asm volatile( "; radix %0 real" ::"n"( R ) );
        }
        else
        {
            complex_stage<R>( p, f, a, g, src, dst, tw, sep, gr, gw );
            asm volatile( "; radix %0" ::"n"( R ) );
        }
    }

    __device__ static __forceinline__ void run( const vol_params<T> &p, C *lds )
    {
        const int     item = p.blocks > 1 ? (int)ordered_tile( 0 ) : 0;
        const int     b1 = item / p.bd0, b0 = item - b1 * p.bd0;
        const int64_t oc = b0 * p.bsc[0] + b1 * p.bsc[1], orl = b0 * p.bsr[0] + b1 * p.bsr[1];
        const io      f{ static_cast<const C *>( p.in ) + oc, static_cast<C *>( p.out ) + oc,
                         static_cast<const T *>( p.in ) + orl, static_cast<T *>( p.out ) + orl };
        C  *src = lds, *dst = lds + p.elems;
        C  *tw  = lds + 2 * p.elems;
        // the twiddle tables of the axes with more than one stage
#pragma unroll
        for ( int i = 0; i < 4; ++i )
            if ( p.ax[i].nst > 1 )
                for ( int e = threadIdx.x; e < p.ax[i].n; e += blockDim.x )
                    tw[p.ax[i].tw + e] = p.twg[i][e];
        // the axes by a run-time index into the kernel's arguments where those are (p is the
        // first): through p it would copy them to scratch memory
        typedef __attribute__( ( address_space( 4 ) ) ) const vol_axis *axes;
        const axes ax = (axes)__builtin_amdgcn_kernarg_segment_ptr();
#pragma unroll 1
        for ( int s = 0; s < 4; ++s )
        {
            // forward: real axis, o2, o1, o0; backward: o0, o1, o2, real axis
            const int  i    = FWD ? 3 - s : s;
            const bool real = i == 3;
            vol_axis   a;
            a.n             = ax[i].n;
            a.nst           = ax[i].nst;
            a.st            = ax[i].st;
            a.rst           = ax[i].rst;
            a.gs            = ax[i].gs;
            a.tw            = ax[i].tw;
            a.lines         = ax[i].lines;
            a.mg_st         = ax[i].mg_st;
            a.mg_lines      = ax[i].mg_lines;
            const int flags = FWD ? ax[i].ffwd : ax[i].fbwd;
            int       ns    = 1;
#pragma unroll 1
            for ( int t = 0; t < a.nst; ++t )
            {
                const int      r   = ax[i].r[t];
                const vol_stage g{ ns, ax[i].tst[t], ax[i].mg_ns[t], ax[i].mg_nbf[t] };
                const bool     gr  = t == 0 && ( flags & VOL_READ );
                const bool     sep = t == 0 && ( flags & VOL_SEP );
                const bool     gw  = t + 1 == a.nst && ( flags & VOL_WRITE );
                const C *twl = tw + a.tw;
                switch ( r )
                {
                case 2: stage<2>( p, f, a, real, g, src, dst, twl, sep, gr, gw ); break;
                case 3: stage<3>( p, f, a, real, g, src, dst, twl, sep, gr, gw ); break;
                case 4: stage<4>( p, f, a, real, g, src, dst, twl, sep, gr, gw ); break;
                case 5: stage<5>( p, f, a, real, g, src, dst, twl, sep, gr, gw ); break;
                case 6: stage<6>( p, f, a, real, g, src, dst, twl, sep, gr, gw ); break;
                case 7: stage<7>( p, f, a, real, g, src, dst, twl, sep, gr, gw ); break;
                case 8: stage<8>( p, f, a, real, g, src, dst, twl, sep, gr, gw ); break;
                case 9: stage<9>( p, f, a, real, g, src, dst, twl, sep, gr, gw ); break;
                case 10: stage<10>( p, f, a, real, g, src, dst, twl, sep, gr, gw ); break;
                case 11: stage<11>( p, f, a, real, g, src, dst, twl, sep, gr, gw ); break;
                case 12: stage<12>( p, f, a, real, g, src, dst, twl, sep, gr, gw ); break;
                case 13: stage<13>( p, f, a, real, g, src, dst, twl, sep, gr, gw ); break;
                case 14: stage<14>( p, f, a, real, g, src, dst, twl, sep, gr, gw ); break;
                case 15: stage<15>( p, f, a, real, g, src, dst, twl, sep, gr, gw ); break;
                case 16: stage<16>( p, f, a, real, g, src, dst, twl, sep, gr, gw ); break;
                default: break; // the host plans no other radix
                }
                __syncthreads();
                ns *= r;
                C *const tmp = src;
                src          = dst;
                dst          = tmp;
            }
        }
    }
};

template <typename T, bool FWD>
__global__ void __launch_bounds__( vol_max_threads( 2 * sizeof( T ) ) ) k_volume( const vol_params<T> p )
{
    extern __shared__ __align__( 16 ) unsigned char vol_lds[];
    vol_kernel<T, FWD>::run( p, reinterpret_cast<cpx<T> *>( vol_lds ) );
}

} // namespace fftm_mi
