// spt_tuning.h - what the zero fields of a tuning stand for. Plain C++ (no HIP).
#pragma once

#include "spt.h"

namespace spt {

// Idle lanes (four per ray) that make a traversal wave take new rays: 16 to 24
// measure best for every kind of ray (extension rays of a 123M-path render 8:
// 87 ms, 16: 84, 24: 83, 48: 98), so a larger spt_tuning.refill_lanes acts
// as 24.
constexpr uint32_t kRefillLanes = 20, kMaxRefillLanes = 24;

// Shading grid and refill threshold by wavefront count: one wavefront shades with 128 blocks per
// CU; with other wavefronts beside it a smaller grid measured faster (1024-spp
// mesh image, three wavefronts: 64 blocks 910 Mpaths/s, 32 893, 128 891). The
// refill threshold of one wavefront acts as kMaxRefillLanes.
inline void resolve_front_defaults(const spt_tuning& raw, spt_tuning& r, uint32_t fronts) {
    r.shade_blocks_per_cu = raw.shade_blocks_per_cu ? raw.shade_blocks_per_cu : (fronts > 1 ? 64u : 128u);
    r.refill_lanes = raw.refill_lanes ? raw.refill_lanes : (fronts > 1 ? kRefillLanes : 48u);
}

// A tuning as spt_get_tuning reports it: 3 wavefronts, with their launch
// shapes, where none are asked for.
inline spt_tuning resolve_tuning(const spt_tuning& t) {
    spt_tuning r = t;
    if (r.path_capacity == 0) r.path_capacity = 1u << 27;
    if (r.use_graph == 0) r.use_graph = 2;
    if (r.tile_pixels == 0) r.tile_pixels = 4096;
    if (r.tile_samples == 0) r.tile_samples = 16;
    if (r.check_every == 0) r.check_every = 4;
    if (r.wavefronts == 0) r.wavefronts = 3;
    resolve_front_defaults(t, r, r.wavefronts);
    return r;
}

// A tuning as a call runs it: one wavefront unless more are asked for. Its
// traversal and shading each fill the chip, and with other streams in the
// process several lose (1, 2, 3 of them: guided 800x600, 64 spp 63.9, 74.7, 72.5
// ms, 400x300, 36 spp 11.5, 11.4, 11.6; batch of 12 scenes 59.3, 64.5, 66.3).
inline spt_tuning running_tuning(const spt_tuning& t) {
    spt_tuning r = resolve_tuning(t);
    if (t.wavefronts == 0) {
        r.wavefronts = 1;
        resolve_front_defaults(t, r, 1);
    }
    return r;
}

// The tuning to keep when `t` is set and the default wavefronts have been
// reported before: the launch shapes of the report that come back with every
// field filled in, as only a report has them, are the default still, so that a
// caller who changes one other field of it keeps what ran.
inline spt_tuning returned_tuning(const spt_tuning& t) {
    const spt_tuning d = resolve_tuning(spt_tuning{});
    spt_tuning r = t;
    if (t.wavefronts == d.wavefronts && t.shade_blocks_per_cu == d.shade_blocks_per_cu &&
        t.refill_lanes == d.refill_lanes && t.path_capacity && t.use_graph && t.tile_pixels && t.tile_samples &&
        t.check_every)
        r.wavefronts = r.shade_blocks_per_cu = r.refill_lanes = 0;
    return r;
}

}  // namespace spt
