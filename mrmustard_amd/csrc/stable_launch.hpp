// Plan and launches of the tiled stable sweep (stable.hip).
#pragma once

#include "exact.hpp"
#include "host.hpp"

namespace mm {

struct StableTilePlan {
    int e[8], nt[8], h[8], ls[8];
    int cells = 0, nrow = 0, nhalo = 0, threads = 0, launches = 0;
    int64_t trows = 0;
    size_t shmem = 0;
    double us = 0.0;  // estimated time
    bool batch = false;
    bool whole() const { return launches == 1; }
};

// false when no tile fits (D > 6).
bool stable_tile_plan(const Lat &g, int64_t B, size_t ws_bytes, const DevState *ds, StableTilePlan *p);

// All launches of the sweep of B triples; nf as in StableTileArgs (unused when p.whole()).
int launch_stable_tiles(const StableTilePlan &p, const Lat &g, int64_t B, const double *A, const double *b, const double *c, double *G,
                        void *ws, int *nf, const DevState *ds, hipStream_t s);

}  // namespace mm
