// Sums of float terms in LDS, in doubles by atomic addition: on gfx950 a
// wave's ds_add_f32 takes about 194 cycles of its compute unit, whatever the
// addresses, its ds_add_f64 24 (ds_add_u64 at most 16).  Terms of any size,
// infinities and NaN are held as the float sum held them, and as the 24 bits
// of a term leave 29 of a double's 53, a sum is exact, and so does not depend
// on its order, unless its terms differ by more than about 2^29 over their
// number; where it is not exact its rounding is 2^-53 of it.  (Integers in
// fixed point, a third faster in LDS, have one absolute quantum for the whole
// tile: at 16384 particles a tile the current of particles of 1e-9 c came out
// 3e-5 off, that of 1e-13 c as zero.)
#pragma once

#include "common.h"

namespace zpic {

#if defined( __HIP_DEVICE_COMPILE__ )
typedef __attribute__( ( address_space( 3 ) ) ) double lds_f64;
#else
typedef double lds_f64;
#endif

__device__ inline void lds_add( lds_f64 * p, float v ) {
    __hip_atomic_fetch_add( p, (double) v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP );
}

}  // namespace zpic
