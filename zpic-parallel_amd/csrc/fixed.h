// Sums of weights (terms of about 1) in LDS in 64-bit fixed point, by integer
// atomics: on gfx950 a wave's ds_add_f32 takes about 194 cycles of its compute
// unit, whatever the addresses, its ds_add_u64 at most 16 (ds_add_f64 23), and
// a sum of integers does not depend on its order.
#pragma once

#include "common.h"

namespace zpic {

typedef unsigned long long u64;
#if defined( __HIP_DEVICE_COMPILE__ )
typedef __attribute__( ( address_space( 3 ) ) ) u64 lds_u64;
#else
typedef u64 lds_u64;
#endif

// 2^bits to the unit (the common factors of a sum are applied to its end).
// With `bits` the weights of n particles cannot overflow an element
// (FIX_HEADROOM bits are left for those of positions outside their cell), and
// a term is off by at most 2^-47 up to 2047 particles and 2^-43 at 16384.  The
// quantum is absolute: terms far below 1 lose bits (lds_sum.h holds those).
// fixed_add holds terms below 32.
constexpr int FIX_HEADROOM = 5, FIX_MAX_BITS = 46;

struct Fixed {
    double magic;   // 1.5 * 2^(52 - bits): adding it leaves value * 2^bits in the low mantissa bits
    unsigned hi;    // its upper word (the lower one is 0)
    double unit;    // 2^-bits
};
__device__ inline Fixed fixed_point( int n ) {
    const int bits = min( FIX_MAX_BITS, 62 - FIX_HEADROOM - ( 32 - __clz( n ) ) );
    Fixed f;
    f.hi = ( (unsigned) ( 1023 + 52 - bits ) << 20 ) | 0x80000u;
    f.magic = __hiloint2double( (int) f.hi, 0 );
    f.unit = __hiloint2double( ( 1023 - bits ) << 20, 0 );
    return f;
}
__device__ inline void fixed_add( lds_u64 * p, float v, const Fixed & f ) {
    u64 b = (u64) __double_as_longlong( (double) v + f.magic );
    b -= (u64) f.hi << 32;
    __hip_atomic_fetch_add( p, b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP );
}
// The sum times its terms' common factor.
__device__ inline float fixed_value( u64 sum, const Fixed & f, float factor ) {
    return (float) ( (double) (long long) sum * f.unit * (double) factor );
}

}  // namespace zpic
