// Index arithmetic of launches whose workgroups choose their order or their key ranges on the device: plain functions of integers, so that
// a host compiler can check them over every launch shape.
#pragma once
#include <stdint.h>

#ifdef __HIPCC__
#define NV_HD __host__ __device__ inline __attribute__((always_inline))
#else
#define NV_HD inline
#endif

namespace nv {

// Latent attention, several tokens, with ranges sized on the device: key tiles of a range of a launch with room for `slots` workgroups at a time.
NV_HD int latent_share(int64_t total_tiles, int slots, int fewest) {
    const int64_t share = (total_tiles + slots - 1) / slots, most = (int64_t)1 << 24;
    return (int)(share < fewest ? fewest : share > most ? most : share);
}
// Key tiles of a row tile whose last row sees `last_key`.  Workspace and block tables hold what the caller's longest length has room for,
// nsplit ranges of `fewest` tiles; keys beyond it, where that length was stated too small, are left out.
NV_HD int latent_tiles(int last_key, int tile_keys, int nsplit, int fewest) {
    const int tiles = last_key / tile_keys + 1, room = nsplit * fewest;
    return tiles < room ? tiles : room;
}
// Its ranges: at most nsplit, since a share is never below `fewest`.
NV_HD int latent_ranges(int tiles, int share) { return tiles <= share ? 1 : (tiles - 1) / share + 1; }

}  // namespace nv
