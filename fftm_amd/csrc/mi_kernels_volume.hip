// Volume-pass kernels (FP32 and FP64).
#include "mi_launch.hpp"

namespace fftm_mi
{
namespace
{

template <typename T>
hipError_t launch_volume_t( const vol_params<T> &p, bool fwd, hipStream_t s )
{
    const size_t lds = sizeof( cpx<T> ) * (size_t)( 2 * p.elems + p.twelems );
    if ( fwd )
        hipLaunchKernelGGL( ( k_volume<T, true> ), dim3( (unsigned)p.blocks ), dim3( (unsigned)p.nt ), lds, s, p );
    else
        hipLaunchKernelGGL( ( k_volume<T, false> ), dim3( (unsigned)p.blocks ), dim3( (unsigned)p.nt ), lds, s, p );
    return hipGetLastError();
}

} // namespace

hipError_t launch_volume_f32( const vol_params<float> &p, bool fwd, hipStream_t s )
{
    return launch_volume_t<float>( p, fwd, s );
}
hipError_t launch_volume_f64( const vol_params<double> &p, bool fwd, hipStream_t s )
{
    return launch_volume_t<double>( p, fwd, s );
}

} // namespace fftm_mi
