// Learned current denoiser (no reference counterpart): a 3-layer 5x5
// convolutional network, 3 -> 16 -> 16 -> 3 channels with ReLU between
// layers (8,835 parameters), applied to the periodic global current J
// (interior cells, [y][x][3]) in place of the binomial filter.
//
// Every convolution is an implicit GEMM on the gfx950 matrix cores
// (v_mfma_f32_16x16x32_bf16: BF16 operands, FP32 accumulation):
//
//   forward / input gradient   D[co][pixel] = W[co][k] x im2col[k][pixel]
//       16 output channels x 16 pixels per instruction, k = tap * C + ci
//       (C = 8 for the 3-channel input padded to 8, 16 otherwise), the
//       weight operand held in registers for the whole launch, the image
//       operand loaded as one 16-byte vector per lane (activations are
//       pixel-major [y][x][C] BF16, periodic wrap in the index);
//   weight gradient            D[co][col] = dZ[co][pixel] x in[pixel][col]
//       16 output channels x 16 input columns, 32 pixels of a row per
//       instruction, both operands loaded as 8 pixels of one channel (the
//       training keeps channel-major copies [C][y][x] of the activations
//       and their gradients); the five x taps are five shifts of the dZ
//       operand in registers, the five y taps the input rows around, which
//       a wave walking down a strip of columns keeps.
//
// Operand lane layouts of v_mfma_f32_16x16x32_bf16 (wave64): lane l holds
// A[row l%16][k (l/16)*8 .. +7], B[k (l/16)*8 .. +7][col l%16], and the
// result D[row (l/16)*4 + i][col l%16], i = 0..3.
//
// Parameters (FP32 master copy, the layout of the C ABI): W1[16][3][5][5],
// b1[16], W2[16][16][5][5], b2[16], W3[3][16][5][5], b3[3].  Training is
// Adam on the FP32 master copy; the BF16 operand packs are rebuilt after
// every update.
#include "common.h"

#include <algorithm>
#include <cmath>
#include <random>
#include <vector>

namespace zpic {
namespace {

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__( ( ext_vector_type( 8 ) ) );
typedef __bf16 bf16x4 __attribute__( ( ext_vector_type( 4 ) ) );
typedef unsigned u32x4 __attribute__( ( ext_vector_type( 4 ) ) );
typedef float f32x4 __attribute__( ( ext_vector_type( 4 ) ) );

constexpr int WAVE = 64;
constexpr int NPARAM = 8835;
constexpr int OFF_W1 = 0, OFF_B1 = 1200, OFF_W2 = 1216, OFF_B2 = 7616, OFF_W3 = 7632, OFF_B3 = 8832;
constexpr int KS1 = 7;   // layer 1: 25 taps x 8 channels = 200 -> 224 = 7 x 32
constexpr int KS2 = 13;  // 16-channel layers: 25 taps x 16 = 400 -> 416 = 13 x 32
constexpr int PACK_FWD1 = 0, PACK_FWD2 = 1, PACK_FWD3 = 2, PACK_BWD3 = 3, PACK_BWD2 = 4, NPACK = 5;

__host__ __device__ inline int pack_ksteps( int which ) { return which == PACK_FWD1 ? KS1 : KS2; }

// Weight-operand value of pack `which` for row (output channel) r and k.
__device__ inline float pack_value( const float * w, int which, int r, int k ) {
    if ( which == PACK_FWD1 ) {
        const int tap = k / 8, ci = k % 8;
        return ( tap < 25 && ci < 3 ) ? w[OFF_W1 + ( r * 3 + ci ) * 25 + tap] : 0.0f;
    }
    const int tap = k / 16, c = k % 16;
    if ( tap >= 25 ) return 0.0f;
    switch ( which ) {
    case PACK_FWD2: return w[OFF_W2 + ( r * 16 + c ) * 25 + tap];
    case PACK_FWD3: return r < 3 ? w[OFF_W3 + ( r * 16 + c ) * 25 + tap] : 0.0f;
    // input gradients: rows are the layer's input channels, k runs over
    // (flipped tap, output channel)
    case PACK_BWD3: return c < 3 ? w[OFF_W3 + ( c * 16 + r ) * 25 + ( 24 - tap )] : 0.0f;
    default: return w[OFF_W2 + ( c * 16 + r ) * 25 + ( 24 - tap )];
    }
}

// pack[which][ks][lane][8]: lane l holds row l%16, k = ks*32 + (l/16)*8 + j
__global__ void k_dn_pack( const float * __restrict__ w, bf16 * __restrict__ pack ) {
    const int which = blockIdx.y;
    const int ks = blockIdx.x;
    if ( ks >= pack_ksteps( which ) ) return;
    const int l = threadIdx.x;
    bf16 * dst = pack + ( (size_t) which * KS2 + ks ) * WAVE * 8 + l * 8;
    for ( int j = 0; j < 8; j++ ) dst[j] = (bf16) pack_value( w, which, l % 16, ks * 32 + ( l / 16 ) * 8 + j );
}

// One convolution of a tile of CONV_X x CONV_Y pixels per workgroup:
// D[co][p] = sum_k W[co][k] im2col[k][p] (+ bias, ReLU, mask), CIN input
// channels per pixel (8 or 16).  The tile and its 2-pixel halo are staged in
// LDS, 16 bytes (8 channels) per pixel and plane, so that the 16 pixels of an
// operand are consecutive; a wave holds the weights and takes two rows, four
// blocks of 16 pixels whose products are independent.
//   SRC  0 BF16 activations [P][CIN]; 1 FP32 [P][3] times in_scale; 2 the
//        interior of a tile-major float3 grid times in_scale
//   DST  0 BF16 [P][16] and / or channel-major [16][P]; 1 FP32 [P][3] times
//        out_scale; 2 that into the interior of a tile-major grid; 3 the
//        mean-square loss against `target` ([P][3], physical units): its
//        gradient by the network's output as BF16 [P][16] and [3][P], and
//        the sum over the workgroup
// On a 512^2 grid a 16-channel layer takes 9 us and the first 7 us, 10 and 8
// with the copies for the training (20 and 13 us when every wave loaded its
// operands, and the weights for each 16 pixels, from the caches); the matrix
// cores need 1.4 us of them, the operand reads from LDS 2.8 us, the rest is
// launch, weights and staging ahead of them.
constexpr int CONV_X = 32, CONV_Y = 8;
constexpr int HALO_X = CONV_X + 4, HALO_Y = CONV_Y + 4;

struct ConvArgs {
    const void * in;
    const bf16 * pack;
    const float * bias;
    const bf16 * mask;
    int H, W;
    float in_scale, out_scale;
    bf16 * out;          // [P][16]
    bf16 * outT;         // [16][P], DST 3: [3][P]
    bf16 * inT;          // SRC 1: the scaled input [3][P]
    float * f32;         // DST 1, and the grid of DST 2
    const float * target;
    double * partial;    // [workgroups]
    zpic_geom g;         // SRC 2, DST 2
};

// Offset (floats) of pixel (x, y) in a tile-major float3 grid.
__device__ inline size_t grid_at( const zpic_geom & g, int x, int y ) {
    const int tx = x / g.nx, ty = y / g.ny;
    return ( (size_t) ( ty * g.ntiles_x + tx ) * g.tile_vol + g.offset + ( y - ty * g.ny ) * g.ext_x + ( x - tx * g.nx ) ) * 3;
}

template <int CIN, int SRC, bool RELU, bool MASK, int DST>
__global__ void __launch_bounds__( 256 ) k_dn_conv( ConvArgs a ) {
    constexpr int KS = CIN == 16 ? KS2 : KS1, PLANES = CIN / 8;
    __shared__ bf16x8 s_in[PLANES][HALO_Y * HALO_X];
    const int H = a.H, W = a.W;
    const size_t P = (size_t) H * W;
    const int bx = W / CONV_X;
    const int x0 = blockIdx.x % bx * CONV_X, y0 = blockIdx.x / bx * CONV_Y;
    const int l = threadIdx.x % WAVE, w = threadIdx.x / WAVE;
    const int g = l / 16, r = l % 16;
    bf16x8 wa[KS];
#pragma unroll
    for ( int ks = 0; ks < KS; ks++ ) wa[ks] = *reinterpret_cast<const bf16x8 *>( a.pack + ( ks * WAVE + l ) * 8 );

    for ( int e = threadIdx.x; e < HALO_Y * HALO_X * PLANES; e += 256 ) {
        const int plane = PLANES == 2 ? e & 1 : 0, q = e / PLANES;
        const int sy = q / HALO_X, sx = q - sy * HALO_X;
        int yy = ( y0 + sy - 2 + H ) % H, xx = x0 + sx - 2;
        xx += ( xx < 0 ) ? W : ( xx >= W ? -W : 0 );
        const size_t p = (size_t) yy * W + xx;
        bf16x8 v;
        if constexpr ( SRC == 0 ) {
            v = *reinterpret_cast<const bf16x8 *>( static_cast<const bf16 *>( a.in ) + p * CIN + plane * 8 );
        } else {
            const float * f = static_cast<const float *>( a.in ) + ( SRC == 1 ? p * 3 : grid_at( a.g, xx, yy ) );
#pragma unroll
            for ( int k = 0; k < 8; k++ ) v[k] = k < 3 ? (bf16) ( f[k] * a.in_scale ) : (bf16) 0.0f;
            if ( SRC == 1 && a.inT && sx >= 2 && sx < 2 + CONV_X && sy >= 2 && sy < 2 + CONV_Y && y0 + sy - 2 < H ) {
                for ( int k = 0; k < 3; k++ ) a.inT[k * P + p] = v[k];
            }
        }
        s_in[plane][q] = v;
    }
    // the lane's place in the staged tile for each k-step's tap (two taps of
    // 16 channels, or four of 8, per k-step)
    int at[KS];
#pragma unroll
    for ( int ks = 0; ks < KS; ks++ ) {
        const int tap = min( CIN == 16 ? ks * 2 + g / 2 : ks * 4 + g, 24 );
        at[ks] = tap / 5 * HALO_X + tap % 5 + r;
    }
    const bool past = CIN == 16 ? g >= 2 : g >= 1;  // lanes whose last tap is past the 25th
    const bf16x8 * plane = s_in[PLANES == 2 ? g % 2 : 0];
    __syncthreads();

    f32x4 acc[4] = {};
    const int row0 = w * 2;
#pragma unroll
    for ( int ks = 0; ks < KS; ks++ ) {
#pragma unroll
        for ( int k = 0; k < 4; k++ ) {
            bf16x8 b = plane[at[ks] + ( row0 + k / 2 ) * HALO_X + k % 2 * 16];
            if ( ks == KS - 1 && past ) b = bf16x8{};
            acc[k] = __builtin_amdgcn_mfma_f32_16x16x32_bf16( wa[ks], b, acc[k], 0, 0, 0 );
        }
    }
    float bv[4];
#pragma unroll
    for ( int i = 0; i < 4; i++ ) bv[i] = ( a.bias && ( DST == 0 || g * 4 + i < 3 ) ) ? a.bias[g * 4 + i] : 0.0f;
    double loss = 0.0;
#pragma unroll
    for ( int k = 0; k < 4; k++ ) {
        const int y = y0 + row0 + k / 2, x = x0 + k % 2 * 16 + r;
        if ( y >= H ) continue;
        const size_t p = (size_t) y * W + x;
        float v[4];
#pragma unroll
        for ( int i = 0; i < 4; i++ ) {
            v[i] = acc[k][i] + bv[i];
            if constexpr ( RELU ) v[i] = v[i] > 0.0f ? v[i] : 0.0f;
        }
        if constexpr ( MASK ) {
            const bf16x4 m = *reinterpret_cast<const bf16x4 *>( a.mask + p * 16 + g * 4 );
#pragma unroll
            for ( int i = 0; i < 4; i++ ) v[i] = (float) m[i] > 0.0f ? v[i] : 0.0f;
        }
        if constexpr ( DST == 0 ) {
            bf16x4 o;
#pragma unroll
            for ( int i = 0; i < 4; i++ ) o[i] = (bf16) v[i];
            if ( a.out ) *reinterpret_cast<bf16x4 *>( a.out + p * 16 + g * 4 ) = o;
            if ( a.outT )
                for ( int i = 0; i < 4; i++ ) a.outT[( g * 4 + i ) * P + p] = o[i];
        } else if constexpr ( DST == 3 ) {
            bf16x4 o = {};
            if ( g == 0 ) {
                const double n = 3.0 * P;
#pragma unroll
                for ( int i = 0; i < 3; i++ ) {
                    const float d = v[i] * a.out_scale - a.target[p * 3 + i];  // physical units
                    loss += (double) d * d;
                    // out = scale * net  =>  d loss / d net = 2 d scale / n
                    o[i] = (bf16) ( 2.0 * d * a.out_scale / n );
                    a.outT[i * P + p] = o[i];
                }
            }
            *reinterpret_cast<bf16x4 *>( a.out + p * 16 + g * 4 ) = o;
        } else if ( g == 0 ) {
            float * o = a.f32 + ( DST == 1 ? p * 3 : grid_at( a.g, x, y ) );
            for ( int i = 0; i < 3; i++ ) o[i] = v[i] * a.out_scale;
        }
    }
    if constexpr ( DST == 3 ) {
        __shared__ double s_loss[4];
        for ( int o = 8; o > 0; o >>= 1 ) loss += __shfl_xor( loss, o );  // the 16 lanes of g = 0
        if ( l == 0 ) s_loss[w] = loss;
        __syncthreads();
        if ( threadIdx.x == 0 ) a.partial[blockIdx.x] = ( s_loss[0] + s_loss[1] ) + ( s_loss[2] + s_loss[3] );
    }
}

// Weight and bias gradients.  A wave takes a strip of 32 columns and WG_ROWS
// rows; the four waves of a workgroup, whose strips lie below one another,
// are summed in LDS, and the workgroup writes one partial sum.  Layers 2 and
// 3: acc[dy * 5 + dx] holds D[co][ci] of that tap, acc[25] the bias (the
// products with ones).  Layer 1: the 3 channels of the 5 rows are 15 columns
// of one operand and ones the 16th, acc[dx] holds D[co][dy * 3 + ci].  On a
// 512^2 grid the three layers take 27 us (481 us with one wave per image row
// and operands gathered element by element).
constexpr int WG_ROWS = 8;
constexpr int WG_WAVES = 4;
constexpr int WG_ACC1 = 5, WG_ACC2 = 26;
constexpr int WG_PART = WG_ACC2 * 256;  // floats of a partial sum of layers 2 and 3 (layer 1: WG_ACC1 * 256)

struct WgradArgs {
    const bf16 * in[3];   // channel-major inputs of the layers: [3][P], [16][P], [16][P]
    const bf16 * dz[3];   // channel-major gradients: [16][P], [16][P], [3][P]
    float * part[3];
    int H, W;
};

template <int LAYER>
__device__ inline void dn_wgrad( const WgradArgs & a, float * s_sum ) {
    constexpr int NACC = LAYER == 0 ? WG_ACC1 : WG_ACC2;
    const int H = a.H, W = a.W;
    const size_t P = (size_t) H * W;
    const int l = threadIdx.x % WAVE, w = threadIdx.x / WAVE;
    const int g = l / 16, r = l % 16;
    const int strips = W / 32;
    const int x = blockIdx.x % strips * 32 + g * 8;
    const int ybeg = ( blockIdx.x / strips * WG_WAVES + w ) * WG_ROWS, yend = min( H, ybeg + WG_ROWS );
    const int xl = x == 0 ? W - 2 : x - 2, xr = x + 8 == W ? 0 : x + 8;
    f32x4 acc[NACC];
#pragma unroll
    for ( int k = 0; k < NACC; k++ ) acc[k] = f32x4{ 0.f, 0.f, 0.f, 0.f };
    bf16x8 ones;
#pragma unroll
    for ( int k = 0; k < 8; k++ ) ones[k] = (bf16) 1.0f;

    const bool has_dz = LAYER != 2 || r < 3;
    const bf16 * dzc = a.dz[LAYER] + ( has_dz ? r : 0 ) * P;
    // layer 1: this lane's column is channel r % 3 of row r / 3; layers 2, 3: channel r
    const bf16 * inc = a.in[LAYER] + ( LAYER == 0 ? ( r < 15 ? r % 3 : 0 ) : r ) * P;
    auto in_row = [&]( int y ) {
        y += ( y < 0 ) ? H : ( y >= H ? -H : 0 );
        return *reinterpret_cast<const bf16x8 *>( inc + (size_t) y * W + x );
    };
    auto input = [&]( int y ) {  // layer 1: the lane's row around y; layers 2, 3: the row two below y
        if constexpr ( LAYER == 0 ) return r < 15 ? in_row( y + r / 3 - 2 ) : ones;
        else return in_row( y + 2 );
    };
    struct Dz {
        u32x4 mid;
        unsigned lo, hi;
    };
    auto dz_row = [&]( int y ) {  // columns x - 2 .. x + 9
        Dz d = {};
        if ( has_dz ) {
            const bf16 * p = dzc + (size_t) y * W;
            d.mid = *reinterpret_cast<const u32x4 *>( p + x );
            d.lo = *reinterpret_cast<const unsigned *>( p + xl );
            d.hi = *reinterpret_cast<const unsigned *>( p + xr );
        }
        return d;
    };
    if ( ybeg < yend ) {
        bf16x8 rows[5];  // input rows y - 2 .. y + 2 (layer 1: [4] alone)
        if constexpr ( LAYER != 0 ) {
#pragma unroll
            for ( int k = 0; k < 4; k++ ) rows[k + 1] = in_row( ybeg - 2 + k );
        }
        bf16x8 next_in = input( ybeg );
        Dz next_dz = dz_row( ybeg );
        for ( int y = ybeg; y < yend; y++ ) {
            if constexpr ( LAYER != 0 ) {
#pragma unroll
                for ( int k = 0; k < 4; k++ ) rows[k] = rows[k + 1];
            }
            rows[4] = next_in;
            const Dz d = next_dz;
            if ( y + 1 < yend ) {
                next_in = input( y + 1 );
                next_dz = dz_row( y + 1 );
            }
            const unsigned D[6] = { d.lo, d.mid[0], d.mid[1], d.mid[2], d.mid[3], d.hi };
            unsigned O[5];
#pragma unroll
            for ( int k = 0; k < 5; k++ ) O[k] = __builtin_amdgcn_alignbit( D[k + 1], D[k], 16 );
            // in[x] meets dz[x + 2 - dx]
#pragma unroll
            for ( int dx = 0; dx < 5; dx++ ) {
                const int s = 2 - dx;  // shift in columns
                u32x4 v;
#pragma unroll
                for ( int k = 0; k < 4; k++ ) v[k] = ( s & 1 ) ? O[k + ( s + 1 ) / 2] : D[k + 1 + s / 2];
                const bf16x8 A = __builtin_bit_cast( bf16x8, v );
                if constexpr ( LAYER == 0 ) {
                    acc[dx] = __builtin_amdgcn_mfma_f32_16x16x32_bf16( A, rows[4], acc[dx], 0, 0, 0 );
                } else {
#pragma unroll
                    for ( int dy = 0; dy < 5; dy++ )
                        acc[dy * 5 + dx] = __builtin_amdgcn_mfma_f32_16x16x32_bf16( A, rows[dy], acc[dy * 5 + dx], 0, 0, 0 );
                    if ( dx == 2 ) acc[25] = __builtin_amdgcn_mfma_f32_16x16x32_bf16( A, ones, acc[25], 0, 0, 0 );
                }
            }
        }
    }
    // the waves' sums in wave order; element k * 256 + i * 64 + lane
    for ( int v = 0; v < WG_WAVES; v++ ) {
        if ( w == v ) {
#pragma unroll
            for ( int k = 0; k < NACC; k++ )
#pragma unroll
                for ( int i = 0; i < 4; i++ ) {
                    float * q = s_sum + k * 256 + i * 64 + l;
                    *q = v == 0 ? acc[k][i] : *q + acc[k][i];
                }
        }
        __syncthreads();
    }
    float * dst = a.part[LAYER] + (size_t) blockIdx.x * NACC * 256;
    for ( int e = threadIdx.x; e < NACC * 256; e += WG_WAVES * WAVE ) dst[e] = s_sum[e];
}

__global__ void __launch_bounds__( WG_WAVES * WAVE ) k_dn_wgrad( WgradArgs a ) {
    __shared__ float s_sum[WG_PART];
    if ( blockIdx.y == 0 ) dn_wgrad<0>( a, s_sum );
    else if ( blockIdx.y == 1 ) dn_wgrad<1>( a, s_sum );
    else dn_wgrad<2>( a, s_sum );
}

// Parameter of element (acc k, i, lane) of a layer's partial sum, or -1.
// D[co = (lane / 16) * 4 + i][col = lane % 16].
__device__ inline int grad_param( int layer, int k, int i, int lane ) {
    const int co = lane / 16 * 4 + i, col = lane % 16;
    if ( layer == 0 ) {
        if ( col == 15 ) return k == 2 ? OFF_B1 + co : -1;
        return OFF_W1 + ( co * 3 + col % 3 ) * 25 + col / 3 * 5 + k;
    }
    if ( layer == 2 && co >= 3 ) return -1;
    if ( k == 25 ) return col == 0 ? ( layer == 1 ? OFF_B2 : OFF_B3 ) + co : -1;
    return ( layer == 1 ? OFF_W2 : OFF_W3 ) + ( co * 16 + col ) * 25 + k;
}

// Places of weight i in the operand packs (at most two; -1: none).
__device__ inline int pack_at( int which, int row, int k ) {
    return ( which * KS2 + k / 32 ) * WAVE * 8 + ( row + 16 * ( k % 32 / 8 ) ) * 8 + k % 8;
}
__device__ inline void param_packs( int i, int at[2] ) {
    at[0] = at[1] = -1;
    if ( i < OFF_B1 ) {
        const int co = i / 75, ci = i / 25 % 3, tap = i % 25;
        at[0] = pack_at( PACK_FWD1, co, tap * 8 + ci );
    } else if ( i >= OFF_W2 && i < OFF_B2 ) {
        const int j = i - OFF_W2, co = j / 400, ci = j / 25 % 16, tap = j % 25;
        at[0] = pack_at( PACK_FWD2, co, tap * 16 + ci );
        at[1] = pack_at( PACK_BWD2, ci, ( 24 - tap ) * 16 + co );
    } else if ( i >= OFF_W3 && i < OFF_B3 ) {
        const int j = i - OFF_W3, co = j / 400, ci = j / 25 % 16, tap = j % 25;
        at[0] = pack_at( PACK_FWD3, co, tap * 16 + ci );
        at[1] = pack_at( PACK_BWD3, ci, ( 24 - tap ) * 16 + co );
    }
}

struct AdamArgs {
    int on;
    float lr, b1, b2, eps, c1, c2;
};

// Sums the partial sums in a fixed order into the FP32 gradient, and with
// adam.on moves the parameter and its places in the packs; workgroup 0 sums
// the loss.  RED_SLICES threads share the partial sums of an element.
// (512^2: 5 us for what took 162 us as a thread per parameter over 512 rows,
// the update and the packs in launches of their own.)
constexpr int RED_SLICES = 8, RED_ELEMS = 256 / RED_SLICES;
struct ReduceArgs {
    const float * part[3];
    int nparts;
    float * grad, * w, * m, * v;
    bf16 * pack;
    const double * loss_part;
    int nloss;
    double loss_scale;
    double * loss;
    AdamArgs adam;
};
constexpr int RED_BLOCKS1 = WG_ACC1 * 256 / RED_ELEMS, RED_BLOCKS2 = WG_PART / RED_ELEMS;

__global__ void __launch_bounds__( 256 ) k_dn_reduce( ReduceArgs a ) {
    __shared__ double s[256];
    int b = blockIdx.x - 1;
    if ( b < 0 ) {
        double acc = 0.0;
        for ( int k = threadIdx.x; k < a.nloss; k += 256 ) acc += a.loss_part[k];
        s[threadIdx.x] = acc;
        __syncthreads();
        for ( int o = 128; o > 0; o >>= 1 ) {
            if ( (int) threadIdx.x < o ) s[threadIdx.x] += s[threadIdx.x + o];
            __syncthreads();
        }
        if ( threadIdx.x == 0 ) a.loss[0] = s[0] / a.loss_scale;
        return;
    }
    int layer = 0;
    if ( b >= RED_BLOCKS1 ) {
        b -= RED_BLOCKS1;
        layer = 1 + b / RED_BLOCKS2;
        b %= RED_BLOCKS2;
    }
    const int stride = layer == 0 ? WG_ACC1 * 256 : WG_PART;
    const int e = b * RED_ELEMS + threadIdx.x % RED_ELEMS, slice = threadIdx.x / RED_ELEMS;
    const int i = grad_param( layer, e / 256, e / 64 % 4, e % 64 );
    double acc = 0.0;
    if ( i >= 0 ) {
        const float * p = a.part[layer] + e;
#pragma unroll 8
        for ( int k = slice; k < a.nparts; k += RED_SLICES ) acc += p[(size_t) k * stride];
    }
    s[threadIdx.x] = acc;
    __syncthreads();
    if ( slice != 0 || i < 0 ) return;
    double sum = 0.0;
    for ( int k = 0; k < RED_SLICES; k++ ) sum += s[k * RED_ELEMS + threadIdx.x];
    const float gi = (float) sum;
    a.grad[i] = gi;
    if ( !a.adam.on ) return;
    const AdamArgs & o = a.adam;
    const float mi = o.b1 * a.m[i] + ( 1.0f - o.b1 ) * gi;
    const float vi = o.b2 * a.v[i] + ( 1.0f - o.b2 ) * gi * gi;
    a.m[i] = mi;
    a.v[i] = vi;
    const float wi = a.w[i] - o.lr * ( mi / o.c1 ) / ( sqrtf( vi / o.c2 ) + o.eps );
    a.w[i] = wi;
    int at[2];
    param_packs( i, at );
    if ( at[0] >= 0 ) a.pack[at[0]] = (bf16) wi;
    if ( at[1] >= 0 ) a.pack[at[1]] = (bf16) wi;
}

// Copies the interior of a tile-major float3 grid to FP32 [y][x][3].
__global__ void k_dn_gather( const float * __restrict__ J, zpic_geom g, float * __restrict__ f32 ) {
    const int W = g.nx * g.ntiles_x, H = g.ny * g.ntiles_y;
    const size_t P = (size_t) W * H;
    for ( size_t p = blockIdx.x * (size_t) blockDim.x + threadIdx.x; p < P; p += (size_t) gridDim.x * blockDim.x ) {
        const float * c = J + grid_at( g, p % W, p / W );
        f32[p * 3] = c[0];
        f32[p * 3 + 1] = c[1];
        f32[p * 3 + 2] = c[2];
    }
}

// Low-pass comparison for the shadow check: sum over cells of |a - b|^2 and
// |b|^2 of [P][3] arrays.
__global__ void __launch_bounds__( 256 ) k_dn_diff( const float * __restrict__ a, const float * __restrict__ b, size_t n,
                                                    double * __restrict__ partial ) {
    __shared__ double s0[256], s1[256];
    double d2 = 0.0, b2 = 0.0;
    for ( size_t i = blockIdx.x * (size_t) blockDim.x + threadIdx.x; i < n; i += (size_t) gridDim.x * blockDim.x ) {
        const double d = (double) a[i] - b[i];
        d2 += d * d;
        b2 += (double) b[i] * b[i];
    }
    s0[threadIdx.x] = d2;
    s1[threadIdx.x] = b2;
    __syncthreads();
    for ( int o = 128; o > 0; o >>= 1 ) {
        if ( (int) threadIdx.x < o ) {
            s0[threadIdx.x] += s0[threadIdx.x + o];
            s1[threadIdx.x] += s1[threadIdx.x + o];
        }
        __syncthreads();
    }
    if ( threadIdx.x == 0 ) {
        partial[2 * blockIdx.x] = s0[0];
        partial[2 * blockIdx.x + 1] = s1[0];
    }
}

constexpr int RED_BLOCKS = 256;
constexpr int LOSS_RING = 1024;  // training steps whose losses are read back together

}  // namespace
}  // namespace zpic

using namespace zpic;

struct zpic_denoiser {
    int H = 0, W = 0, max_pairs = 0, npairs = 0;
    float scale = 1.0f;
    int adam_t = 0;
    hipStream_t st = nullptr;
    float * w = nullptr;       // [NPARAM] master
    float * m = nullptr;       // Adam moments
    float * v = nullptr;
    float * grad = nullptr;    // [NPARAM]
    bf16 * pack = nullptr;     // [NPACK][KS2][64][8]
    bf16 * a1 = nullptr;       // [P][16] activations and gradients
    bf16 * a2 = nullptr;
    bf16 * dz3 = nullptr;
    bf16 * dz2 = nullptr;
    // channel-major copies for the weight gradients (with the pair store, or by the first backward pass)
    bf16 * x0T = nullptr;      // [3][P]
    bf16 * a1T = nullptr;      // [16][P]
    bf16 * a2T = nullptr;
    bf16 * dz1T = nullptr;
    bf16 * dz2T = nullptr;
    bf16 * dz3T = nullptr;     // [3][P]
    float * part[3] = { nullptr, nullptr, nullptr };  // [wgrad_groups] partial sums
    double * loss_part = nullptr;  // [conv_groups]
    double * losses = nullptr;     // [LOSS_RING]
    float * out = nullptr;     // [P][3]
    double * red = nullptr;    // [2*RED_BLOCKS]
    float * pairs_in = nullptr;   // [max_pairs][P][3]
    float * pairs_tgt = nullptr;  // [max_pairs][P][3]
    std::vector<void *> owned;
};

namespace {

template <class T>
int dn_alloc( zpic_denoiser * d, T ** p, size_t n ) {
    void * q = nullptr;
    if ( n == 0 ) { *p = nullptr; return ZPIC_OK; }
    ZPIC_HIP_TRY( hipMalloc( &q, n * sizeof( T ) ) );
    d->owned.push_back( q );
    *p = static_cast<T *>( q );
    return ZPIC_OK;
}

size_t dn_P( const zpic_denoiser * d ) { return (size_t) d->H * d->W; }

int dn_repack( zpic_denoiser * d ) {
    hipLaunchKernelGGL( k_dn_pack, dim3( KS2, NPACK ), dim3( WAVE ), 0, d->st, d->w, d->pack );
    ZPIC_LAUNCH_CHECK( "k_dn_pack" );
    return ZPIC_OK;
}

const bf16 * packp( const zpic_denoiser * d, int which ) { return d->pack + (size_t) which * KS2 * WAVE * 8; }
int conv_groups( const zpic_denoiser * d ) { return d->W / CONV_X * ( ( d->H + CONV_Y - 1 ) / CONV_Y ); }
int wgrad_groups( const zpic_denoiser * d ) {
    constexpr int rows = WG_ROWS * WG_WAVES;
    return d->W / 32 * ( ( d->H + rows - 1 ) / rows );
}

// The buffers of the backward pass.
int dn_train_buffers( zpic_denoiser * d ) {
    if ( d->losses ) return ZPIC_OK;
    const size_t P = dn_P( d ), n = wgrad_groups( d );
    if ( int rc = dn_alloc( d, &d->x0T, 3 * P ) ) return rc;
    for ( bf16 ** p : { &d->a1T, &d->a2T, &d->dz1T, &d->dz2T } )
        if ( int rc = dn_alloc( d, p, 16 * P ) ) return rc;
    if ( int rc = dn_alloc( d, &d->dz3T, 3 * P ) ) return rc;
    if ( int rc = dn_alloc( d, &d->dz3, 16 * P ) ) return rc;
    if ( int rc = dn_alloc( d, &d->dz2, 16 * P ) ) return rc;
    for ( int k = 0; k < 3; k++ )
        if ( int rc = dn_alloc( d, &d->part[k], n * ( k == 0 ? WG_ACC1 * 256 : WG_PART ) ) ) return rc;
    if ( int rc = dn_alloc( d, &d->loss_part, conv_groups( d ) ) ) return rc;
    return dn_alloc( d, &d->losses, LOSS_RING );
}

template <int CIN, int SRC, bool RELU, bool MASK, int DST>
int dn_conv( zpic_denoiser * d, ConvArgs a, int which, const float * bias ) {
    a.pack = packp( d, which );
    a.bias = bias;
    a.H = d->H;
    a.W = d->W;
    hipLaunchKernelGGL( ( k_dn_conv<CIN, SRC, RELU, MASK, DST> ), dim3( conv_groups( d ) ), dim3( 256 ), 0, d->st, a );
    ZPIC_LAUNCH_CHECK( "k_dn_conv" );
    return ZPIC_OK;
}

// The hidden layers from [P][3] physical values (g null) or the interior of a
// tile-major grid; with `train` the channel-major copies too.
int dn_hidden( zpic_denoiser * d, const float * in, const zpic_geom * g, bool train ) {
    ConvArgs a{};
    a.in = in;
    a.in_scale = 1.0f / d->scale;
    a.out = d->a1;
    if ( train ) {
        a.inT = d->x0T;
        a.outT = d->a1T;
    }
    if ( g ) a.g = *g;
    if ( int rc = g ? dn_conv<8, 2, true, false, 0>( d, a, PACK_FWD1, d->w + OFF_B1 )
                    : dn_conv<8, 1, true, false, 0>( d, a, PACK_FWD1, d->w + OFF_B1 ) )
        return rc;
    ConvArgs b{};
    b.in = d->a1;
    b.out = d->a2;
    if ( train ) b.outT = d->a2T;
    return dn_conv<16, 0, true, false, 0>( d, b, PACK_FWD2, d->w + OFF_B2 );
}

// Forward pass of [P][3] values; output d->out (physical units) = scale * net.
int dn_forward( zpic_denoiser * d, const float * in ) {
    if ( int rc = dn_hidden( d, in, nullptr, false ) ) return rc;
    ConvArgs a{};
    a.in = d->a2;
    a.f32 = d->out;
    a.out_scale = d->scale;
    return dn_conv<16, 0, false, false, 1>( d, a, PACK_FWD3, d->w + OFF_B3 );
}

// Forward and backward pass of one pair ([P][3] each, physical units): the
// loss into loss[0] (device), the gradient into d->grad, and the parameters
// moved if adam.on.
int dn_train_step( zpic_denoiser * d, const float * in, const float * target, const AdamArgs & adam, double * loss ) {
    if ( int rc = dn_hidden( d, in, nullptr, true ) ) return rc;
    ConvArgs a{};
    a.in = d->a2;
    a.out_scale = d->scale;
    a.target = target;
    a.out = d->dz3;
    a.outT = d->dz3T;
    a.partial = d->loss_part;
    if ( int rc = dn_conv<16, 0, false, false, 3>( d, a, PACK_FWD3, d->w + OFF_B3 ) ) return rc;
    // input gradients through layers 3 and 2, ReLU masks from the activations
    ConvArgs b3{};
    b3.in = d->dz3;
    b3.mask = d->a2;
    b3.out = d->dz2;
    b3.outT = d->dz2T;
    if ( int rc = dn_conv<16, 0, false, true, 0>( d, b3, PACK_BWD3, nullptr ) ) return rc;
    ConvArgs b2{};
    b2.in = d->dz2;
    b2.mask = d->a1;
    b2.outT = d->dz1T;
    if ( int rc = dn_conv<16, 0, false, true, 0>( d, b2, PACK_BWD2, nullptr ) ) return rc;
    WgradArgs wg{};
    wg.in[0] = d->x0T; wg.in[1] = d->a1T; wg.in[2] = d->a2T;
    wg.dz[0] = d->dz1T; wg.dz[1] = d->dz2T; wg.dz[2] = d->dz3T;
    ReduceArgs r{};
    for ( int k = 0; k < 3; k++ ) r.part[k] = wg.part[k] = d->part[k];
    wg.H = d->H;
    wg.W = d->W;
    const int n = wgrad_groups( d );
    hipLaunchKernelGGL( k_dn_wgrad, dim3( n, 3 ), dim3( WG_WAVES * WAVE ), 0, d->st, wg );
    ZPIC_LAUNCH_CHECK( "k_dn_wgrad" );
    r.nparts = n;
    r.grad = d->grad; r.w = d->w; r.m = d->m; r.v = d->v;
    r.pack = d->pack;
    r.loss_part = d->loss_part;
    r.nloss = conv_groups( d );
    r.loss_scale = 3.0 * dn_P( d );
    r.loss = loss;
    r.adam = adam;
    hipLaunchKernelGGL( k_dn_reduce, dim3( 1 + RED_BLOCKS1 + 2 * RED_BLOCKS2 ), dim3( 256 ), 0, d->st, r );
    ZPIC_LAUNCH_CHECK( "k_dn_reduce" );
    return ZPIC_OK;
}

int dn_check_geom( const zpic_denoiser * d, const zpic_geom * g ) {
    if ( !g || g->nx * g->ntiles_x != d->W || g->ny * g->ntiles_y != d->H )
        return set_error( ZPIC_EINVAL, "grid does not match the denoiser's size" );
    return ZPIC_OK;
}

}  // namespace

extern "C" {

zpic_denoiser * zpic_denoiser_new( int H, int W, int max_pairs ) {
    if ( H < 5 || W < 32 || W % 32 || max_pairs < 0 ) {
        set_error( ZPIC_EINVAL, "denoiser grid must be at least 5 rows and a multiple of 32 columns" );
        return nullptr;
    }
    auto * d = new zpic_denoiser();
    d->H = H;
    d->W = W;
    d->max_pairs = max_pairs;
    const size_t P = (size_t) H * W;
    int rc = ZPIC_OK;
    if ( hipStreamCreateWithFlags( &d->st, hipStreamNonBlocking ) != hipSuccess ) rc = set_error( ZPIC_EHIP, "stream" );
    if ( !rc ) rc = dn_alloc( d, &d->w, NPARAM );
    if ( !rc ) rc = dn_alloc( d, &d->m, NPARAM );
    if ( !rc ) rc = dn_alloc( d, &d->v, NPARAM );
    if ( !rc ) rc = dn_alloc( d, &d->grad, NPARAM );
    if ( !rc ) rc = dn_alloc( d, &d->pack, (size_t) NPACK * KS2 * WAVE * 8 );
    if ( !rc ) rc = dn_alloc( d, &d->a1, P * 16 );
    if ( !rc ) rc = dn_alloc( d, &d->a2, P * 16 );
    if ( !rc ) rc = dn_alloc( d, &d->out, P * 3 );
    if ( !rc ) rc = dn_alloc( d, &d->red, 2 * RED_BLOCKS );
    if ( !rc ) rc = dn_alloc( d, &d->pairs_in, (size_t) max_pairs * P * 3 );
    if ( !rc ) rc = dn_alloc( d, &d->pairs_tgt, (size_t) max_pairs * P * 3 );
    if ( !rc && max_pairs > 0 ) rc = dn_train_buffers( d );
    if ( !rc && hipMemsetAsync( d->pack, 0, sizeof( bf16 ) * NPACK * KS2 * WAVE * 8, d->st ) != hipSuccess )
        rc = set_error( ZPIC_EHIP, "hipMemsetAsync" );
    if ( !rc ) {
        // He-style initialisation, fixed seed; biases zero
        std::vector<float> h( NPARAM, 0.0f );
        std::mt19937 gen( 12345 );
        auto fill = [&]( int off, int n, int fan_in ) {
            std::normal_distribution<float> nd( 0.0f, std::sqrt( 2.0f / fan_in ) );
            for ( int i = 0; i < n; i++ ) h[off + i] = nd( gen );
        };
        fill( OFF_W1, 1200, 75 );
        fill( OFF_W2, 6400, 400 );
        fill( OFF_W3, 1200, 400 );
        rc = zpic_denoiser_set_params( d, h.data() );
    }
    if ( rc ) {
        zpic_denoiser_free( d );
        return nullptr;
    }
    return d;
}

void zpic_denoiser_free( zpic_denoiser * d ) {
    if ( !d ) return;
    if ( d->st ) (void) hipStreamSynchronize( d->st );
    for ( void * p : d->owned ) (void) hipFree( p );
    if ( d->st ) (void) hipStreamDestroy( d->st );
    delete d;
}

int zpic_denoiser_set_params( zpic_denoiser * d, const float * host ) {
    if ( !d || !host ) return set_error( ZPIC_EINVAL, "null argument" );
    ZPIC_HIP_TRY( hipMemcpyAsync( d->w, host, sizeof( float ) * NPARAM, hipMemcpyHostToDevice, d->st ) );
    ZPIC_HIP_TRY( hipMemsetAsync( d->m, 0, sizeof( float ) * NPARAM, d->st ) );
    ZPIC_HIP_TRY( hipMemsetAsync( d->v, 0, sizeof( float ) * NPARAM, d->st ) );
    d->adam_t = 0;
    if ( int rc = dn_repack( d ) ) return rc;
    ZPIC_HIP_TRY( hipStreamSynchronize( d->st ) );
    return ZPIC_OK;
}

int zpic_denoiser_get_params( zpic_denoiser * d, float * host ) {
    if ( !d || !host ) return set_error( ZPIC_EINVAL, "null argument" );
    ZPIC_HIP_TRY( hipMemcpyAsync( host, d->w, sizeof( float ) * NPARAM, hipMemcpyDeviceToHost, d->st ) );
    ZPIC_HIP_TRY( hipStreamSynchronize( d->st ) );
    return ZPIC_OK;
}

int zpic_denoiser_set_scale( zpic_denoiser * d, float scale ) {
    if ( !d || !( scale > 0.0f ) ) return set_error( ZPIC_EINVAL, "scale must be positive" );
    d->scale = scale;
    return ZPIC_OK;
}

float zpic_denoiser_get_scale( const zpic_denoiser * d ) { return d ? d->scale : 0.0f; }

int zpic_denoiser_forward_host( zpic_denoiser * d, const float * in, float * out ) {
    if ( !d || !in || !out ) return set_error( ZPIC_EINVAL, "null argument" );
    const size_t P = dn_P( d );
    float * tmp = nullptr;
    ZPIC_HIP_TRY( hipMalloc( (void **) &tmp, sizeof( float ) * P * 3 ) );
    int rc = ZPIC_OK;
    if ( hipMemcpyAsync( tmp, in, sizeof( float ) * P * 3, hipMemcpyHostToDevice, d->st ) != hipSuccess )
        rc = set_error( ZPIC_EHIP, "copy in" );
    if ( !rc ) rc = dn_forward( d, tmp );
    if ( !rc && hipMemcpyAsync( out, d->out, sizeof( float ) * P * 3, hipMemcpyDeviceToHost, d->st ) != hipSuccess )
        rc = set_error( ZPIC_EHIP, "copy out" );
    if ( !rc && hipStreamSynchronize( d->st ) != hipSuccess ) rc = set_error( ZPIC_EHIP, "sync" );
    (void) hipFree( tmp );
    return rc;
}

int zpic_denoiser_gradient_host( zpic_denoiser * d, const float * in, const float * tgt, float * grad, double * loss ) {
    if ( !d || !in || !tgt || !grad ) return set_error( ZPIC_EINVAL, "null argument" );
    const size_t P = dn_P( d );
    float * tmp = nullptr;
    ZPIC_HIP_TRY( hipMalloc( (void **) &tmp, sizeof( float ) * P * 6 ) );
    int rc = ZPIC_OK;
    if ( hipMemcpyAsync( tmp, in, sizeof( float ) * P * 3, hipMemcpyHostToDevice, d->st ) != hipSuccess ||
         hipMemcpyAsync( tmp + P * 3, tgt, sizeof( float ) * P * 3, hipMemcpyHostToDevice, d->st ) != hipSuccess )
        rc = set_error( ZPIC_EHIP, "copy in" );
    if ( !rc ) rc = dn_train_buffers( d );
    if ( !rc ) rc = dn_train_step( d, tmp, tmp + P * 3, AdamArgs{}, d->losses );
    if ( !rc && loss && hipMemcpyAsync( loss, d->losses, sizeof( double ), hipMemcpyDeviceToHost, d->st ) != hipSuccess )
        rc = set_error( ZPIC_EHIP, "copy out" );
    if ( !rc && hipMemcpyAsync( grad, d->grad, sizeof( float ) * NPARAM, hipMemcpyDeviceToHost, d->st ) != hipSuccess )
        rc = set_error( ZPIC_EHIP, "copy out" );
    if ( !rc && hipStreamSynchronize( d->st ) != hipSuccess ) rc = set_error( ZPIC_EHIP, "sync" );
    (void) hipFree( tmp );
    return rc;
}

// Stores a training pair from two tile-major J grids (device): the noisy
// input and the target.
int zpic_denoiser_add_pair( zpic_denoiser * d, const float * J_in, const float * J_target, const zpic_geom * g,
                            void * stream ) {
    if ( !d || !J_in || !J_target ) return set_error( ZPIC_EINVAL, "null argument" );
    if ( int rc = dn_check_geom( d, g ) ) return rc;
    if ( d->npairs >= d->max_pairs ) return set_error( ZPIC_ERANGE, "pair store full" );
    const size_t P = dn_P( d );
    // the grids were written on the caller's stream
    ZPIC_HIP_TRY( hipStreamSynchronize( as_stream( stream ) ) );
    float * pi = d->pairs_in + (size_t) d->npairs * P * 3;
    float * pt = d->pairs_tgt + (size_t) d->npairs * P * 3;
    hipLaunchKernelGGL( k_dn_gather, dim3( 1024 ), dim3( 256 ), 0, d->st, J_in, *g, pi );
    hipLaunchKernelGGL( k_dn_gather, dim3( 1024 ), dim3( 256 ), 0, d->st, J_target, *g, pt );
    ZPIC_LAUNCH_CHECK( "k_dn_gather" );
    ZPIC_HIP_TRY( hipStreamSynchronize( d->st ) );
    d->npairs++;
    return ZPIC_OK;
}

int zpic_denoiser_num_pairs( const zpic_denoiser * d ) { return d ? d->npairs : 0; }

int zpic_denoiser_clear_pairs( zpic_denoiser * d ) {
    if ( !d ) return set_error( ZPIC_EINVAL, "null denoiser" );
    d->npairs = 0;
    return ZPIC_OK;
}

// Root-mean-square of the stored targets (a natural scale for the network).
int zpic_denoiser_target_rms( zpic_denoiser * d, double * rms ) {
    if ( !d || !rms || d->npairs == 0 ) return set_error( ZPIC_EINVAL, "no pairs stored" );
    const size_t n = (size_t) d->npairs * dn_P( d ) * 3;
    hipLaunchKernelGGL( k_dn_diff, dim3( RED_BLOCKS ), dim3( 256 ), 0, d->st, d->pairs_tgt, d->pairs_tgt, n, d->red );
    ZPIC_LAUNCH_CHECK( "k_dn_diff" );
    std::vector<double> h( 2 * RED_BLOCKS );
    ZPIC_HIP_TRY( hipMemcpyAsync( h.data(), d->red, sizeof( double ) * 2 * RED_BLOCKS, hipMemcpyDeviceToHost, d->st ) );
    ZPIC_HIP_TRY( hipStreamSynchronize( d->st ) );
    double s = 0;
    for ( int i = 0; i < RED_BLOCKS; i++ ) s += h[2 * i + 1];
    *rms = std::sqrt( s / n );
    return ZPIC_OK;
}

// `steps` Adam steps over the first `use` stored pairs (all if use <= 0),
// pair order drawn with `seed`; loss_hist[steps] receives each step's loss
// (may be null).
int zpic_denoiser_train( zpic_denoiser * d, int steps, float lr, unsigned seed, int use, double * loss_hist ) {
    if ( !d || steps < 0 || !( lr > 0.0f ) ) return set_error( ZPIC_EINVAL, "invalid training request" );
    if ( d->npairs == 0 ) return set_error( ZPIC_ESTATE, "no training pairs stored" );
    if ( use <= 0 || use > d->npairs ) use = d->npairs;
    const size_t P = dn_P( d );
    std::mt19937 gen( seed );
    std::uniform_int_distribution<int> pick( 0, use - 1 );
    if ( int rc = dn_train_buffers( d ) ) return rc;
    // the losses stay on the device until the ring is full or the call ends
    auto read_losses = [&]( int first, int n ) -> int {
        if ( loss_hist )
            ZPIC_HIP_TRY( hipMemcpyAsync( loss_hist + first, d->losses, sizeof( double ) * n, hipMemcpyDeviceToHost, d->st ) );
        ZPIC_HIP_TRY( hipStreamSynchronize( d->st ) );
        return ZPIC_OK;
    };
    AdamArgs adam{ 1, lr, 0.9f, 0.999f, 1e-8f, 0.0f, 0.0f };
    for ( int s = 0; s < steps; s++ ) {
        const int k = pick( gen );
        d->adam_t++;
        adam.c1 = 1.0f - std::pow( adam.b1, (float) d->adam_t );
        adam.c2 = 1.0f - std::pow( adam.b2, (float) d->adam_t );
        const int at = s % LOSS_RING;
        if ( int rc = dn_train_step( d, d->pairs_in + (size_t) k * P * 3, d->pairs_tgt + (size_t) k * P * 3, adam,
                                     d->losses + at ) )
            return rc;
        if ( at == LOSS_RING - 1 )
            if ( int rc = read_losses( s - at, LOSS_RING ) ) return rc;
    }
    return read_losses( steps - steps % LOSS_RING, steps % LOSS_RING );
}

// Mean-square error of the network output (and of the unfiltered input)
// against the target of stored pair k.
int zpic_denoiser_eval_pair( zpic_denoiser * d, int k, double * mse_net, double * mse_input ) {
    if ( !d || k < 0 || k >= d->npairs ) return set_error( ZPIC_EINVAL, "bad pair index" );
    const size_t P = dn_P( d );
    const float * in = d->pairs_in + (size_t) k * P * 3;
    const float * tg = d->pairs_tgt + (size_t) k * P * 3;
    if ( int rc = dn_forward( d, in ) ) return rc;
    std::vector<double> h( 2 * RED_BLOCKS );
    auto mse = [&]( const float * a, double * out ) -> int {
        hipLaunchKernelGGL( k_dn_diff, dim3( RED_BLOCKS ), dim3( 256 ), 0, d->st, a, tg, P * 3, d->red );
        ZPIC_LAUNCH_CHECK( "k_dn_diff" );
        ZPIC_HIP_TRY( hipMemcpyAsync( h.data(), d->red, sizeof( double ) * 2 * RED_BLOCKS, hipMemcpyDeviceToHost, d->st ) );
        ZPIC_HIP_TRY( hipStreamSynchronize( d->st ) );
        double s = 0;
        for ( int i = 0; i < RED_BLOCKS; i++ ) s += h[2 * i];
        *out = s / ( 3.0 * P );
        return ZPIC_OK;
    };
    if ( mse_net )
        if ( int rc = mse( d->out, mse_net ) ) return rc;
    if ( mse_input )
        if ( int rc = mse( in, mse_input ) ) return rc;
    return ZPIC_OK;
}

// Host copies of stored pair k ([P][3] each).
int zpic_denoiser_get_pair( zpic_denoiser * d, int k, float * in, float * tgt ) {
    if ( !d || k < 0 || k >= d->npairs ) return set_error( ZPIC_EINVAL, "bad pair index" );
    const size_t P = dn_P( d );
    if ( in )
        ZPIC_HIP_TRY( hipMemcpyAsync( in, d->pairs_in + (size_t) k * P * 3, sizeof( float ) * P * 3,
                                      hipMemcpyDeviceToHost, d->st ) );
    if ( tgt )
        ZPIC_HIP_TRY( hipMemcpyAsync( tgt, d->pairs_tgt + (size_t) k * P * 3, sizeof( float ) * P * 3,
                                      hipMemcpyDeviceToHost, d->st ) );
    ZPIC_HIP_TRY( hipStreamSynchronize( d->st ) );
    return ZPIC_OK;
}

// In-place denoising of the interior of a tile-major J grid (device) issued
// on `stream`; guard cells are left to the caller (copy_to_gc).
int zpic_denoiser_apply( zpic_denoiser * d, float * J, const zpic_geom * g, void * stream ) {
    if ( !d || !J ) return set_error( ZPIC_EINVAL, "null argument" );
    if ( int rc = dn_check_geom( d, g ) ) return rc;
    hipStream_t caller = as_stream( stream );
    hipStream_t own = d->st;
    d->st = caller;  // run on the caller's stream: ordered with the step
    int rc = dn_hidden( d, J, g, false );
    if ( !rc ) {
        // J's last reader was the first layer
        ConvArgs a{};
        a.in = d->a2;
        a.f32 = J;
        a.g = *g;
        a.out_scale = d->scale;
        rc = dn_conv<16, 0, false, false, 2>( d, a, PACK_FWD3, d->w + OFF_B3 );
    }
    d->st = own;
    return rc;
}

// Relative L2 difference ||a - b|| / ||b|| of two [n] float arrays (device).
int zpic_denoiser_reldiff( zpic_denoiser * d, const float * a, const float * b, size_t n, void * stream,
                           double * out ) {
    if ( !d || !a || !b || !out ) return set_error( ZPIC_EINVAL, "null argument" );
    hipStream_t st = as_stream( stream );
    hipLaunchKernelGGL( k_dn_diff, dim3( RED_BLOCKS ), dim3( 256 ), 0, st, a, b, n, d->red );
    ZPIC_LAUNCH_CHECK( "k_dn_diff" );
    std::vector<double> h( 2 * RED_BLOCKS );
    ZPIC_HIP_TRY( hipMemcpyAsync( h.data(), d->red, sizeof( double ) * 2 * RED_BLOCKS, hipMemcpyDeviceToHost, st ) );
    ZPIC_HIP_TRY( hipStreamSynchronize( st ) );
    double s0 = 0, s1 = 0;
    for ( int i = 0; i < RED_BLOCKS; i++ ) {
        s0 += h[2 * i];
        s1 += h[2 * i + 1];
    }
    *out = s1 > 0 ? std::sqrt( s0 / s1 ) : std::sqrt( s0 );
    return ZPIC_OK;
}

int zpic_denoiser_size( const zpic_denoiser * d, int * H, int * W ) {
    if ( !d ) return set_error( ZPIC_EINVAL, "null denoiser" );
    if ( H ) *H = d->H;
    if ( W ) *W = d->W;
    return ZPIC_OK;
}

}  // extern "C"
