// CPU harness of the batches' launch rule (rocrand_amd/csrc/rr_batch_schedule.hpp) for
// tests/test_batch_schedule.py.
#include "rr_batch_schedule.hpp"

#include <cstddef>

// one launch for all groups (1) or one per group (0), and the Philox vecs per tile
extern "C" int batch_schedule_of(size_t groups, size_t bytes, size_t inter_tiles, const size_t* philox_vecs,
                                 size_t philox_streams, unsigned* tile)
{
    const rr::batch_launch l = rr::batch_schedule(groups, bytes, inter_tiles, [&](unsigned vecs) {
        size_t n = 0;
        for(size_t i = 0; i < philox_streams; i++)
            n += philox_vecs[i] / vecs + 1;
        return n;
    });
    *tile = l.tile;
    return l.single;
}
