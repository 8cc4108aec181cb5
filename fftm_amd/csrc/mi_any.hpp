// One pass along an axis whose length has no kernel of its own: runtime N = r0 r1 ... with
// radices up to 16, the same Stockham stages, address maps and real-axis handling as the
// compile-time pass kernel (mi_pass.hpp).
//
// The host picks a schedule with as few stages as the radices allow (FP32: 250 = 10 5 5,
// 1080 = 15 12 6), a tile of `cols` lines and a workgroup in which every thread holds whole
// butterflies of at most any_values() values per stage (any_plan).  A stage is then: read
// the thread's butterflies (stage 0 from HBM, the others from LDS), twiddle, DFT in
// registers, write back to the one LDS tile (the last stage of a C2C or C2R pass straight to
// HBM).  So a line crosses LDS once per stage boundary, and every load of a tile is in
// flight at once.
//
// Lanes walk along the lines where those are contiguous in HBM and across columns
// otherwise, for the loads as for the stores.
//
// Bound by memory latency and, next to it, by the integer and twiddle work per value.
// Batches of 2^23 complex values, FP32 rows / columns: N = 250 24.9 / 27.7 us (5.4 / 4.8
// TB/s), N = 1080 27.2 / 31.8 us; FP64 250: 41.9 / 48.6 us (6.4 / 5.5 TB/s).  Its
// predecessor, one radix per thread and ping-pong LDS buffers with every line transformed
// column-fastest, took 79 / 76, 59 / 69 and 104 / 101 us.  With the tile chosen by
// any_cost, the 175 x 250 x 330 FP32 pair went from 180 (tiles of a fixed size) to 172 us.
//
// Registers: FP32 common radices 79..80, every radix 82..87, table in memory 93..96; FP64 93..97
// and 133..137.  The FP32 C2R kernels and the strided R2C one of the common radices keep 2..4 of
// theirs in scratch memory (12 bytes per lane) to stay at six waves per SIMD.
#pragma once

#include "mi_pass.hpp"

namespace fftm_mi
{

constexpr int ANY_MAX_STAGES  = 5;
constexpr int ANY_MAX_COLS    = 64; // lines per workgroup
constexpr int ANY_STAGE_LOADS = 9;  // bins that a thread has in flight while a C2R tile is staged
constexpr int any_max_threads( int csize ) { return csize == 8 ? 1024 : 512; }

// Values a thread may hold in a stage (csize: bytes of a complex value), and the whole
// butterflies of radix R that makes (one of a radix beyond it).  The FP64 kernels of lengths
// whose table stays in memory (memtw) have radix 13 and its registers anyway and hold two
// butterflies of radix 7: with one, lines from 1792 points with a factor 7 need five waves,
// which leaves a CU to one workgroup (rows of 1960 points, 2^22 values: C2C 61.1 -> 40.1 us, R2C
// 40.7 -> 26.1; 133..137 registers either way).
constexpr int any_values( int csize ) { return csize == 8 ? 16 : 10; }
constexpr int any_butterflies( int R, int csize, bool memtw )
{
    const int n = R == 7 && memtw ? 2 : any_values( csize ) / R;
    return n < 1 ? 1 : ( n > 4 ? 4 : n );
}
constexpr bool any_memtw( int64_t N, int csize ) { return N * csize > 16384; }
// The kernels that most lengths use have the common radices and read their twiddles from an
// LDS copy of the table.  A length with a factor 11 or 13 takes kernels that have every radix
// (their butterflies need more registers, which the other lengths would pay for in
// occupancy), one with too large a table kernels that read it from memory.
enum : int
{
    ANY_COMMON = 0,
    ANY_RARE   = 1,
    ANY_MEMTW  = 2
};
constexpr bool any_common_radix( int R, int csize )
{
    return R <= 10 || ( csize == 8 && R != 11 && R != 13 && R <= 16 );
}
constexpr bool any_radix( int R, int csize ) { return any_common_radix( R, csize ) || R == 11 || R == 13; }

// One length's schedule and tile (host: make_any_plan).  mg_*: n / d = mulhi( n, mg ) for
// the item counts that occur (n d < 2^32).
struct any_stage
{
    int32_t  r, ns, nbf, tst; // radix, span before the stage, butterflies per line, N / ( ns r )
    uint32_t mg_nbf, mg_ns;
};
struct any_plan
{
    int32_t   N, nst;
    int32_t   cols;  // lines per workgroup (column-fastest tiles: a power of two)
    int32_t   csh;   // log2( cols ) of column-fastest tiles
    int32_t   nt;    // threads (a multiple of cols in column-fastest tiles)
    int32_t   elems; // LDS values of the tile; the twiddle table follows
    int32_t   nh;    // N / 2 + 1
    int32_t   mode;  // ANY_COMMON, ANY_RARE or ANY_MEMTW
    uint32_t  mg_n, mg_nh, mg_cols;
    any_stage s[ANY_MAX_STAGES];
};

template <typename T, int KIND, bool INV, bool LOADB, int MODE>
struct any_kernel
{
    static constexpr bool RARE = MODE != ANY_COMMON; // every radix
    static constexpr bool TWL  = MODE != ANY_MEMTW;  // stage twiddles from an LDS copy of the table
    using C                  = cpx<T>;
    static constexpr int CPT = KIND == KIND_C2C ? 1 : 2;

    struct ctx
    {
        const pass_params<T> &p;
        const any_plan       &a;
        C                    *lds;
        C                    *tw; // LDS copy of the twiddle table
        int                   tid, nt;
        int64_t               tile;
        // column-fastest tiles: the thread's column is the same in every item
        int                   c;
        int64_t               ia, ib, oa, ob;
        bool                  va, vb;
        int64_t              *lo; // output offsets of the tile's lines (pairs), -1 past the end
    };

    __device__ static __forceinline__ int quot( int n, int d, uint32_t mg )
    {
        return d == 1 ? n : (int)__umulhi( (uint32_t)n, mg );
    }

    // line c of the tile: offsets of its column (pair) and whether they exist
    __device__ static __forceinline__ void line_offsets( const pass_params<T> &p, int64_t col, int64_t &ia, int64_t &ib,
                                                         int64_t &oa, int64_t &ob, bool &va, bool &vb )
    {
        va = col < p.ncols;
        vb = CPT == 2 && col + 1 < p.ncols;
        ib = ob = 0;
        if ( p.d0 >= p.ncols )
        {
            // one batch dimension (dense lines): no division
            ia = va ? col * p.is0 : 0;
            oa = va ? col * p.os0 : 0;
            if constexpr ( CPT == 2 )
            {
                ib = vb ? ia + p.is0 : 0;
                ob = vb ? oa + p.os0 : 0;
            }
        }
        else
        {
            col_offsets( p, va ? col : 0, ia, oa );
            if constexpr ( CPT == 2 )
                col_offsets( p, vb ? col + 1 : 0, ib, ob );
        }
    }

    // Stage s.  FIRST: from HBM (C2R: from the staged half spectra); LAST: to HBM where the
    // pass stores its lines directly.
    template <int R, bool FIRST, bool LAST>
    __device__ static __forceinline__ void stage( const ctx &x, const any_stage s )
    {
        constexpr int         NB    = any_butterflies( R, (int)sizeof( C ), MODE == ANY_MEMTW );
        const pass_params<T> &p     = x.p;
        const any_plan       &a     = x.a;
        const int             items = s.nbf * a.cols;
        const bool            out   = LAST && KIND != KIND_R2C && p.store_b == (int)LOADB;
        // distance in LDS of consecutive elements of a line, and of consecutive lines
        const int es = LOADB ? a.cols : 1, ls = LOADB ? 1 : a.N;
        C         v[NB][R];
        int       jj[NB], cc[NB];
#pragma unroll
        for ( int b = 0; b < NB; ++b )
        {
            // an item past the end repeats the last one of its column
            const int item = x.tid + b * x.nt;
            if constexpr ( LOADB )
            {
                cc[b] = x.c;
                jj[b] = item >> a.csh;
                jj[b] = jj[b] < s.nbf ? jj[b] : s.nbf - 1;
            }
            else
            {
                const int i = item < items ? item : items - 1;
                cc[b]       = quot( i, s.nbf, s.mg_nbf );
                jj[b]       = i - cc[b] * s.nbf;
            }
        }
#pragma unroll
        for ( int b = 0; b < NB; ++b )
            if ( b * x.nt < items )
            {
                const int c = cc[b], j = jj[b];
                if constexpr ( FIRST && KIND != KIND_C2R )
                {
                    // every load unconditional: a column past the end reads column 0, which
                    // exists, and is never stored
                    int64_t ia = x.ia, ib = x.ib, oa, ob;
                    bool    va = x.va, vb = x.vb;
                    if constexpr ( !LOADB )
                        line_offsets( p, ( x.tile * a.cols + c ) * CPT, ia, ib, oa, ob, va, vb );
                    const int64_t step = (int64_t)s.nbf * p.ies;
                    if constexpr ( KIND == KIND_C2C )
                    {
                        const C *src = static_cast<const C *>( p.in ) + ia + (int64_t)j * p.ies;
#pragma unroll
                        for ( int r = 0; r < R; ++r )
                            v[b][r] = mk<T>( src[r * step].x, src[r * step].y );
                    }
                    else
                    {
                        const T *sa = static_cast<const T *>( p.in ) + ia + (int64_t)j * p.ies;
                        const T *sb = static_cast<const T *>( p.in ) + ib + (int64_t)j * p.ies;
#pragma unroll
                        for ( int r = 0; r < R; ++r )
                            v[b][r] = mk<T>( sa[r * step], sb[r * step] );
                        if ( !vb )
                        {
                            // the second of a pair past the end contributes zeros
#pragma unroll
                            for ( int r = 0; r < R; ++r )
                                v[b][r].y = (T)0;
                        }
                    }
                }
                else if constexpr ( FIRST )
                {
                    // C2R: z = A~ + i B~ from the tile's staged half spectra.  Element n = j + r
                    // nbf lies below N / 2 for r < R / 2 and is the mirror image of bin N - n
                    // above; the middle r of an odd radix has both.
                    const int as = LOADB ? 2 * a.cols : 1, bs = LOADB ? 1 : a.nh;
                    const C  *at = x.lds + ( LOADB ? 2 * c : 2 * c * a.nh );
                    const T   h  = p.wmode == 2 ? (T)0.5 : (T)1;
#pragma unroll
                    for ( int r = 0; r < R; ++r )
                    {
                        const int  n   = j + r * s.nbf;
                        const bool up  = 2 * r >= R || ( 2 * r + 1 == R && 2 * n > a.N );
                        const int  nn  = up ? a.N - n : n;
                        C          za = at[nn * as], zb = at[nn * as + bs];
                        if ( p.wmode == 2 && n != 0 && 2 * n != a.N )
                        {
                            // adjoint of R2C: interior bins carry weight 1/2
                            za = scl( za, h );
                            zb = scl( zb, h );
                        }
                        // the imaginary parts of the DC and Nyquist bins are ignored
                        if ( ( r == 0 && n == 0 ) || ( ( 2 * r == R || 2 * r + 1 == R ) && 2 * n == a.N ) )
                        {
                            za.y = (T)0;
                            zb.y = (T)0;
                        }
                        v[b][r] = up ? mk<T>( za.x + zb.y, zb.x - za.y ) : mk<T>( za.x - zb.y, za.y + zb.x );
                    }
                }
                else
                {
                    const int k  = j - (int)__umulhi( (uint32_t)j, s.mg_ns ) * s.ns;
                    const C  *at = x.lds + c * ls + j * es;
                    const int st = s.nbf * es;
#pragma unroll
                    for ( int r = 0; r < R; ++r, at += st )
                        v[b][r] = *at;
                    const int ts = k * s.tst;
                    // one kind of pointer per kernel: one that may be either needs slow loads
                    const C *tw = TWL ? x.tw : p.tw;
#pragma unroll
                    for ( int r = 1; r < R; ++r )
                    {
                        tw += ts;
                        v[b][r] = twmul<INV>( v[b][r], *tw );
                    }
                }
                dft_fixed<R, INV>( v[b] );
            }
        if ( ( !FIRST || KIND == KIND_C2R ) && !out )
            __syncthreads(); // the tile is read by every thread before it is written
#pragma unroll
        for ( int b = 0; b < NB; ++b )
            if ( x.tid + b * x.nt < items )
            {
                const int c = cc[b], j = jj[b];
                if ( out )
                {
                    int64_t oa = x.oa, ob = x.ob, ia, ib;
                    bool    va = x.va, vb = x.vb;
                    if constexpr ( !LOADB )
                        line_offsets( p, ( x.tile * a.cols + c ) * CPT, ia, ib, oa, ob, va, vb );
                    // last stage: ns = nbf, so butterfly j writes elements j + m nbf
                    const int64_t step = (int64_t)s.nbf * p.oes;
                    if constexpr ( KIND == KIND_C2C )
                    {
                        C *dst = static_cast<C *>( p.out ) + oa + (int64_t)j * p.oes;
                        if ( va )
                        {
#pragma unroll
                            for ( int m = 0; m < R; ++m )
                                dst[m * step] = scl( v[b][m], p.scale );
                        }
                    }
                    else
                    {
                        T *da = static_cast<T *>( p.out ) + oa + (int64_t)j * p.oes;
                        T *db = static_cast<T *>( p.out ) + ob + (int64_t)j * p.oes;
                        if ( va )
                        {
#pragma unroll
                            for ( int m = 0; m < R; ++m )
                                da[m * step] = v[b][m].x * p.scale;
                        }
                        if ( vb )
                        {
#pragma unroll
                            for ( int m = 0; m < R; ++m )
                                db[m * step] = v[b][m].y * p.scale;
                        }
                    }
                }
                else
                {
                    // (j / ns) ns R + j mod ns
                    const int d  = FIRST ? j * R : (int)__umulhi( (uint32_t)j, s.mg_ns ) * s.ns * ( R - 1 ) + j;
                    C        *at = x.lds + c * ls + d * es;
                    const int st = s.ns * es;
#pragma unroll
                    for ( int m = 0; m < R; ++m, at += st )
                        *at = v[b][m];
                }
            }
    }

    // Stage s > 0 of the plan.  Every field of every stage is read at a constant index and
    // the right one selected: a run-time index into the kernel's arguments, or a select
    // that the compiler turns into one, would copy them to scratch memory.
    __device__ static __forceinline__ any_stage pick( const any_plan &a, int s )
    {
        any_stage o{};
#pragma unroll
        for ( int i = 1; i < ANY_MAX_STAGES; ++i )
        {
            const int f0 = __builtin_amdgcn_readfirstlane( a.s[i].r ), f1 = __builtin_amdgcn_readfirstlane( a.s[i].ns );
            const int f2 = __builtin_amdgcn_readfirstlane( a.s[i].nbf ), f3 = __builtin_amdgcn_readfirstlane( a.s[i].tst );
            const int f4 = __builtin_amdgcn_readfirstlane( (int)a.s[i].mg_nbf );
            const int f5 = __builtin_amdgcn_readfirstlane( (int)a.s[i].mg_ns );
            if ( s == i )
                o = any_stage{ f0, f1, f2, f3, (uint32_t)f4, (uint32_t)f5 };
        }
        return o;
    }

    template <int R, bool FIRST, bool LAST>
    __device__ static __forceinline__ void stage_r( const ctx &x, const any_stage &s )
    {
        if constexpr ( RARE ? any_radix( R, (int)sizeof( C ) ) : any_common_radix( R, (int)sizeof( C ) ) )
        {
            stage<R, FIRST, LAST>( x, s );
            // a different last instruction per radix: the compiler otherwise merges the
            // ends of the radices' code and with it their register arrays, into scratch
            asm volatile( "; radix %0" ::"n"( R ) );
        }
    }

    template <bool FIRST, bool LAST>
    __device__ static __forceinline__ void stage_rt( const ctx &x, const any_stage s )
    {
        switch ( s.r )
        {
        case 1:
            if constexpr ( FIRST )
                stage<1, FIRST, LAST>( x, s );
            break;
        case 2: stage_r<2, FIRST, LAST>( x, s ); break;
        case 3: stage_r<3, FIRST, LAST>( x, s ); break;
        case 4: stage_r<4, FIRST, LAST>( x, s ); break;
        case 5: stage_r<5, FIRST, LAST>( x, s ); break;
        case 6: stage_r<6, FIRST, LAST>( x, s ); break;
        case 7: stage_r<7, FIRST, LAST>( x, s ); break;
        case 8: stage_r<8, FIRST, LAST>( x, s ); break;
        case 9: stage_r<9, FIRST, LAST>( x, s ); break;
        case 10: stage_r<10, FIRST, LAST>( x, s ); break;
        case 11: stage_r<11, FIRST, LAST>( x, s ); break;
        case 12: stage_r<12, FIRST, LAST>( x, s ); break;
        case 13: stage_r<13, FIRST, LAST>( x, s ); break;
        case 14: stage_r<14, FIRST, LAST>( x, s ); break;
        case 15: stage_r<15, FIRST, LAST>( x, s ); break;
        case 16: stage_r<16, FIRST, LAST>( x, s ); break;
        default: break; // the host plans no other radix
        }
    }

    // C2R: the tile's 2 cols half spectra into LDS, every bin read once (stage 0 needs each
    // interior bin twice)
    __device__ static __forceinline__ void stage_halves( const ctx &x )
    {
        const pass_params<T> &p     = x.p;
        const any_plan       &a     = x.a;
        const int             lines = 2 * a.cols;
        const int             items = lines * a.nh;
        constexpr int         U     = ANY_STAGE_LOADS;
        if constexpr ( !LOADB )
        {
            // dense rows: the tile's half spectra are one contiguous piece of the array (a
            // whole number of 16-byte pieces, lines is even), copied with no address
            // arithmetic per bin
            const C *src = static_cast<const C *>( p.in ) + x.tile * items;
            if ( p.d0 >= p.ncols && p.ies == 1 && p.is0 == a.nh && ( x.tile + 1 ) * lines <= p.ncols &&
                 ( reinterpret_cast<uintptr_t>( p.in ) & 15 ) == 0 )
            {
                stage_copy16( src, x.lds, items * (int)sizeof( C ) / 16, x.tid, x.nt );
                stage_wait();
                return;
            }
        }
        else if ( ( x.nt & ( lines - 1 ) ) == 0 )
        {
            // a thread keeps its line: one offset for all its bins (with a division per bin the
            // C2R pass of a 8 x 7 x 66 x 9 FP64 pencil took 12.8 us, all integer work; the pair
            // 46.8 -> 41.9 us)
            const int     l = x.tid & ( lines - 1 ), dk = x.nt >> ( a.csh + 1 );
            const int64_t col = x.tile * lines + l;
            const bool    has = col < p.ncols;
            int64_t       io = has ? col * p.is0 : 0, oo;
            if ( p.d0 < p.ncols )
                col_offsets( p, has ? col : 0, io, oo );
            const C *src = static_cast<const C *>( p.in ) + io;
            for ( int k0 = x.tid >> ( a.csh + 1 ); k0 < a.nh; k0 += U * dk )
            {
                C z[U];
#pragma unroll
                for ( int u = 0; u < U; ++u )
                    z[u] = src[(int64_t)( k0 + u * dk < a.nh ? k0 + u * dk : a.nh - 1 ) * p.ies];
#pragma unroll
                for ( int u = 0; u < U; ++u )
                    if ( k0 + u * dk < a.nh )
                        x.lds[( k0 + u * dk ) * lines + l] = has ? z[u] : mk<T>( 0, 0 );
            }
            __syncthreads();
            return;
        }
        for ( int e0 = x.tid; e0 < items; e0 += U * x.nt )
        {
            C    z[U];
            bool ok[U];
#pragma unroll
            for ( int u = 0; u < U; ++u )
            {
                const int     e   = e0 + u * x.nt < items ? e0 + u * x.nt : items - 1;
                const int     l   = LOADB ? e & ( lines - 1 ) : quot( e, a.nh, a.mg_nh );
                const int     k   = LOADB ? e >> ( a.csh + 1 ) : e - l * a.nh;
                const int64_t col = x.tile * lines + l;
                ok[u]             = col < p.ncols;
                int64_t io, oo;
                if ( p.d0 >= p.ncols )
                    io = ok[u] ? col * p.is0 : 0;
                else
                    col_offsets( p, ok[u] ? col : 0, io, oo );
                z[u] = static_cast<const C *>( p.in )[io + (int64_t)k * p.ies];
            }
#pragma unroll
            for ( int u = 0; u < U; ++u )
                if ( e0 + u * x.nt < items )
                    x.lds[e0 + u * x.nt] = ok[u] ? z[u] : mk<T>( 0, 0 ); // line * nh + k, or k * lines + line
        }
        __syncthreads();
    }

    // output from the tile in LDS: the separated pair of half spectra (R2C), or the lines
    // themselves in the other thread mapping
    template <bool COLS>
    __device__ static __forceinline__ void store_tile( const ctx &x )
    {
        const pass_params<T> &p     = x.p;
        const any_plan       &a     = x.a;
        const int             len   = KIND == KIND_R2C ? a.nh : a.N;
        const int             items = a.cols * len;
        const int             es = LOADB ? a.cols : 1, ls = LOADB ? 1 : a.N;
#pragma unroll 2
        for ( int e = x.tid; e < items; e += x.nt )
        {
            int c, k;
            if ( COLS )
            {
                k = LOADB ? e >> a.csh : quot( e, a.cols, a.mg_cols );
                c = e - k * a.cols;
            }
            else
            {
                c = quot( e, len, KIND == KIND_R2C ? a.mg_nh : a.mg_n );
                k = e - c * len;
            }
            // column-fastest tiles stored column-fastest: the thread keeps its column
            const bool    own = COLS && LOADB;
            const int64_t oa = own ? x.oa : x.lo[2 * c], ob = own ? x.ob : x.lo[2 * c + 1];
            const bool    va = own ? x.va : oa >= 0, vb = own ? x.vb : ob >= 0;
            const C zk = x.lds[c * ls + k * es];
            if constexpr ( KIND == KIND_R2C )
            {
                const C zm  = x.lds[c * ls + ( k == 0 ? 0 : a.N - k ) * es];
                const T h   = ( p.wmode == 1 && k != 0 && 2 * k != a.N ) ? p.scale : (T)0.5 * p.scale;
                C      *dst = static_cast<C *>( p.out ) + (int64_t)k * p.oes;
                if ( va )
                    dst[oa] = mk<T>( h * ( zk.x + zm.x ), h * ( zk.y - zm.y ) );
                if ( vb )
                    dst[ob] = mk<T>( h * ( zk.y + zm.y ), h * ( zm.x - zk.x ) );
            }
            else
                store_line<KIND>( p, oa, ob, va, vb, k, zk );
        }
    }

    __device__ static __forceinline__ void run( const pass_params<T> &p, const any_plan &a, C *lds )
    {
        ctx x{ p, a, lds, lds + a.elems, (int)threadIdx.x, (int)blockDim.x, ordered_tile( p.vec ), 0, 0, 0, 0, 0,
               false, false, nullptr };
        // offsets for the stores from LDS: once per line, not per element
        __shared__ int64_t lo[2 * ANY_MAX_COLS];
        x.lo = lo;
        if constexpr ( LOADB )
        {
            x.c = x.tid & ( a.cols - 1 );
            line_offsets( p, ( x.tile * a.cols + x.c ) * CPT, x.ia, x.ib, x.oa, x.ob, x.va, x.vb );
        }
        if ( !( p.store_b && LOADB ) && ( KIND == KIND_R2C || p.store_b != (int)LOADB || a.nst == 1 ) )
            for ( int c = x.tid; c < a.cols; c += x.nt )
            {
                int64_t ia, ib, oa, ob;
                bool    va, vb;
                line_offsets( p, ( x.tile * a.cols + c ) * CPT, ia, ib, oa, ob, va, vb );
                lo[2 * c]     = va ? oa : -1;
                lo[2 * c + 1] = vb ? ob : -1;
            }
        if ( TWL && a.nst > 1 )
            for ( int e = x.tid; e < a.N; e += x.nt )
                x.tw[e] = p.tw[e];
        if constexpr ( KIND == KIND_C2R )
            stage_halves( x );
        stage_rt<true, false>( x, a.s[0] );
        __syncthreads();
        for ( int s = 1; s + 1 < a.nst; ++s )
        {
            stage_rt<false, false>( x, pick( a, s ) );
            __syncthreads();
        }
        if ( a.nst > 1 )
        {
            stage_rt<false, true>( x, pick( a, a.nst - 1 ) );
            if ( KIND != KIND_R2C && p.store_b == (int)LOADB )
                return;
            __syncthreads();
        }
        if ( p.store_b )
            store_tile<true>( x );
        else
            store_tile<false>( x );
    }
};

template <typename T, int KIND, bool INV, bool LOADB, int MODE>
__global__ void __launch_bounds__( any_max_threads( 2 * sizeof( T ) ) )
    __attribute__( ( amdgpu_waves_per_eu( ( sizeof( T ) == 4 ? 6 : 4 ) - ( MODE != ANY_COMMON ? 1 : 0 ) ) ) )
    k_pass_any( const pass_params<T> p, const any_plan a )
{
    extern __shared__ __align__( 16 ) unsigned char any_lds[];
    any_kernel<T, KIND, INV, LOADB, MODE>::run( p, a, reinterpret_cast<cpx<T> *>( any_lds ) );
}

} // namespace fftm_mi
