// Tiles taken by several workgroups in the fast-mode particle pass.
//
// A tile's particles are cut into parts of about `size` particles, at most
// PART_MAX of them, one workgroup each; a part deposits into a J region of
// its own, and k_part_merge adds the regions of a tile in part order.  Used
// where the tiles alone do not fill the device, or one crowded tile would
// hold up the rest (part_rule): with one workgroup per tile, a 128x128 Weibel
// run (64 tiles, 2 x 1M particles) took 1.18 ms a step over its first
// thousand steps, as filaments gather up to three times the mean in a tile;
// cut, and with the species side by side, it takes 0.11 ms, a 64x64 box of 8x8
// tiles and as many particles 0.11 for 1.96.  The list of parts
// follows the tiles' particle counts: the sort writes it for the next pass,
// and part_list() where the counts came about in another way.
#pragma once

#include <algorithm>

#include "zpic_amd.h"

namespace zpic {

constexpr int PART_SEG = 64;      // ints per tile of the segment table
constexpr int PART_MAX_SEG = 59;  // wave segments of one tile
constexpr int PART_MAX = 14;
constexpr unsigned PART_TARGET = 1024;  // parts beyond one per tile, at most
constexpr unsigned PART_MIN = 2048;     // particles of a part, at least

struct PartScratch {
    int on = 0;    // 0: tiles are not cut, the rest is unused
    int size = 0;  // particles of a part
    int cap = 0;   // most parts of all tiles: ntiles + part_extra
    int * seg = nullptr;    // [PART_SEG * ntiles] segment tables
    int * item = nullptr;   // [2 * cap] the parts: tile, part | parts of the tile << 8
    int * total = nullptr;  // [1] their number
    int * npt = nullptr;    // [9 * cap] direction counts of each part
    double * energy = nullptr;  // [cap]
    float * J = nullptr;        // [3 * tile_vol * cap]
};

// Up to 4096 tiles, whose counts one workgroup still scans in one launch and
// where a crowded tile or a chain of launches per species shows: a step of
// 1056x720 cells in 1485 tiles 263 -> 213 us, of 768x640 in 1920 tiles at 64
// particles per cell 1502 -> 1195, of 1024x1024 in 4096 tiles at 16 783 -> 716,
// at one 232 -> 202 us.  Beyond, the passes fill the device by themselves and
// the J regions of the parts would be written and read for every tile.
inline bool part_rule( int ntiles ) { return ntiles <= 4096; }

// Parts beyond one per tile for a buffer of max_part particles, and the
// particles of a part that keep to them, no fewer than PART_MIN: a part also
// stages its tile's fields and writes and merges a J region, which costs time
// where the device is full anyway.  Microseconds a step at PART_MIN 1024, 2048
// and 4096: 64 tiles of 2 x 16384 particles 104, 99 and 98, of one such species
// 78, 77 and 81, 16 tiles of 16384 63, 64 and 71; 64 quiet instances in one
// persistent launch 8910, 8670 and 8570 (8490 with no tile cut), after 300 steps
// 9600, 9350 and 9300 (9400).  PART_TARGET 512 instead of 1024: an evolved 512x512 run in 1024
// tiles 805 for 675; 2048: 16384 particles in each of 1024 tiles 302 for 290.
inline int part_extra( unsigned max_part ) { return (int) std::min( PART_TARGET, max_part / PART_MIN + 1 ); }
inline int part_size( unsigned max_part, int extra ) {
    return (int) std::max( PART_MIN, ( max_part / (unsigned) extra + 64 ) & ~63u );
}

// The list of parts for the tiles' particle counts np[ntiles].
int part_list( const int * np, int ntiles, const PartScratch & parts, void * stream );
// The stage and batch entry points of zpic_amd.h with such scratch (one per
// species of a batch, as its items; null: no tile is cut).  The sort's count
// also sums the tiles' push energies (fast mode) where they are given.
int push_move_deposit_parts( const zpic_particles * p, const zpic_geom * fld, const float * E, const float * B,
                             float * J, float alpha, float dt_dx, float dt_dy, float q, float qnx, float qny,
                             double * tile_energy, zpic_sort * s, int reflect, int shift_x, int set_j,
                             const PartScratch * parts, void * stream );
int tile_sort_count( zpic_particles * p, zpic_particles * tmp, zpic_sort * s, int ntiles_x, int ntiles_y, int nx, int ny,
                     int periodic_x, int periodic_y, const int * extra, const PartScratch * parts,
                     const double * tile_energy, double * energy, void * stream );
int tile_sort_copy( zpic_particles * p, zpic_particles * tmp, zpic_sort * s, int ntiles_x, int ntiles_y, int nx, int ny,
                    int periodic_x, int periodic_y, int mode, const PartScratch * parts, void * stream );
// group > 0: the n items are the species of n / group instances, `group` of
// each side by side, all in parts, and go through each stage together; J is
// written, not added to.  With n = group (one instance) J is given to the merge.
int batch_particles_new( zpic_batch_particles ** out, const zpic_batch_species * items, int n, int threads_per_tile,
                         const PartScratch * parts, int group = 0 );
// zpic_batch_particles_advance in its three parts.
int batch_particles_pass( zpic_batch_particles * plan, void * stream );
int batch_particles_merge( zpic_batch_particles * plan, float * J, void * stream );
int batch_particles_sort( zpic_batch_particles * plan, void * stream );
// dep: deposit buffers of the instances, the current formed from them in one
// stage, and with all tiles in parts the species side by side (null, or an
// entry null or the instance's J: deposited into J, stage by stage).
int batch_step_new( zpic_batch_step ** out, const zpic_batch_species * species, int nslots,
                    const zpic_batch_fields_item * fields, int n, int threads_per_tile, const PartScratch * parts,
                    const float * const * dep );

}  // namespace zpic
