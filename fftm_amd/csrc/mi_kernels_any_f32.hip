// F32 pass kernels of lengths without a compiled kernel (runtime radix schedule).
#include "mi_launch.hpp"

namespace fftm_mi
{
namespace
{

template <int KIND, bool INV, bool LOADB>
hipError_t launch_one( const pass_params<float> &p, const any_plan &a, hipStream_t s )
{
    const int64_t per    = (int64_t)a.cols * ( KIND == KIND_C2C ? 1 : 2 );
    const int64_t ntiles = ( p.ncols + per - 1 ) / per;
    if ( ntiles <= 0 )
        return hipSuccess;
    if ( ntiles > 0x7fffffffLL )
        return hipErrorInvalidConfiguration;
    const size_t lds = sizeof( cpx<float> ) * (size_t)( a.elems + ( a.nst > 1 && a.mode != ANY_MEMTW ? a.N : 0 ) );
    const dim3   grid( (unsigned)ntiles ), block( (unsigned)a.nt );
    if ( a.mode == ANY_MEMTW )
        hipLaunchKernelGGL( ( k_pass_any<float, KIND, INV, LOADB, ANY_MEMTW> ), grid, block, lds, s, p, a );
    else if ( a.mode == ANY_RARE )
        hipLaunchKernelGGL( ( k_pass_any<float, KIND, INV, LOADB, ANY_RARE> ), grid, block, lds, s, p, a );
    else
        hipLaunchKernelGGL( ( k_pass_any<float, KIND, INV, LOADB, ANY_COMMON> ), grid, block, lds, s, p, a );
    return hipGetLastError();
}

} // namespace

hipError_t launch_any_f32( const pass_params<float> &p, const any_plan &a, int kind, bool inv, bool loadb, hipStream_t s )
{
    if ( kind == KIND_R2C )
        return loadb ? launch_one<KIND_R2C, false, true>( p, a, s ) : launch_one<KIND_R2C, false, false>( p, a, s );
    if ( kind == KIND_C2R )
        return loadb ? launch_one<KIND_C2R, true, true>( p, a, s ) : launch_one<KIND_C2R, true, false>( p, a, s );
    if ( inv )
        return loadb ? launch_one<KIND_C2C, true, true>( p, a, s ) : launch_one<KIND_C2C, true, false>( p, a, s );
    return loadb ? launch_one<KIND_C2C, false, true>( p, a, s ) : launch_one<KIND_C2C, false, false>( p, a, s );
}

} // namespace fftm_mi
