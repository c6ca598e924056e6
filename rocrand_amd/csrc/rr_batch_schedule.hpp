// How a batch is launched, decided once from its own sizes: no schedule tuned later or for
// another batch changes it.
#pragma once

#include <stdint.h>

namespace rr
{

constexpr uint32_t CTR_TILE_VECS = 4096; // Philox: vecs per tile before tuning (4 wavefronts x 16 chunks of 64)
constexpr uint32_t MRG_TILE      = 256;  // MRG32k3a: engines per tile (one block)

struct batch_launch
{
    bool     single; // one launch for all groups (batch_small_kernel), else one per group
    uint32_t tile;   // Philox vecs per tile where no tuned schedule says otherwise
};

// One launch, if there are several groups to put in it.  It saves a launch per group (a graph's
// fork and join, 25 us a group) and lets the groups fill the chip together, but its kernel
// holds 3 wavefronts a SIMD and no tables in LDS, where most groups' own kernels hold 7 or 8,
// so it loses where many MRG32k3a tiles are set up for little work each.  us a plan's launch, a
// one-shot call, launch per group -> one launch:
//   6 groups, 12 streams    16 MiB 69 -> 25, 52 -> 39;  256 MiB 108 -> 86, 125 -> 98;
//                          512 MiB 163 -> 156, 200 -> 168
//   6 groups, 256 streams   16 MiB (6,900 tiles) 86 -> 33, 61 -> 52;
//                           32 MiB (13,700) 86 -> 46, 73 -> 72;  64 MiB (27,000) 86 -> 77, 95 -> 114
//   3 groups, 16 streams  1024 MiB Philox 262 -> 263, 299 -> 273;  MRG32k3a 296 -> 306, 310 -> 313
//   1 group, 4 streams      64 MiB Philox normals 32 -> 34, 41 -> 42;  512 MiB 153 -> 170, 163 -> 177;
//                          MRG32k3a normals 64 MiB 39 -> 40, 50 -> 52;  512 MiB 190 -> 204, 209 -> 223
constexpr uint64_t SINGLE_BYTES = 512ull << 20; // of output
constexpr uint64_t SINGLE_TILES = 8192;

// The Philox tiles are the smallest, from one chunk per wavefront on, of which there are not
// more than this many: a block's serial work is short and the descriptors few (one group, 4
// streams, one-shot call: 512 KiB 14.8 -> 11.3 us with the smallest, but 4 MiB in 1,024 tiles
// 23.4, in 256 tiles 14.9).
constexpr uint64_t SINGLE_FINE = SINGLE_TILES / 2, GROUP_FINE = 256;

// `bytes` = the batch's outputs, `inter_tiles` = its MRG32k3a tiles, philox_tiles(v) = its
// Philox tiles of v vecs.
template<class F>
batch_launch batch_schedule(uint64_t groups, uint64_t bytes, uint64_t inter_tiles, F philox_tiles)
{
    batch_launch l;
    l.single = groups > 1 && bytes <= SINGLE_BYTES && inter_tiles + philox_tiles(CTR_TILE_VECS) <= SINGLE_TILES;
    l.tile   = 256;
    while(l.tile < CTR_TILE_VECS && inter_tiles + philox_tiles(l.tile) > (l.single ? SINGLE_FINE : GROUP_FINE))
        l.tile *= 2;
    return l;
}

} // namespace rr
