// libmmhip: plan and launches of the tiled stable sweep (stable_tile_kernel).

#include "stable_launch.hpp"

#include "lds_launch.hpp"
#include "stable_tile.hpp"

namespace mm {

namespace {

__global__ void clear_flag_kernel(int *nf) { *nf = 0; }

// Fill p for tiles of at most e[j] points along axis j; false when the tile
// does not fit one workgroup or the offsets their types.
bool try_tiles(const Lat &g, int64_t B, size_t ws_bytes, const DevState *ds, const int (&e)[8], StableTilePlan *p) {
    const int D = g.D, L = D - 1;
    int64_t h0 = 1, h1 = 0, h2 = 0;  // cells zero, one and two index sums below the tile
    int64_t cells = 1, nrow = 1, trows = 1, launches = 1, steps = 1, reach = 0;
    double tiles = double(B);
    for (int j = D - 1; j >= 0; --j) {
        const int n = (g.shape[j] + e[j] - 1) / e[j];
        p->nt[j] = n;
        p->e[j] = (g.shape[j] + n - 1) / n;  // even tiles
        p->h[j] = n > 1 ? 2 : 0;
        p->ls[j] = int(cells);
        cells *= p->e[j] + p->h[j];
        const int64_t below = n > 1;
        h2 = h2 * p->e[j] + (h1 + h0) * below;
        h1 = h1 * p->e[j] + h0 * below;
        h0 *= p->e[j];
        steps += p->e[j] - 1;
        launches += n - 1;
        tiles *= n;
        reach += (p->e[j] + 2) * g.stride[j];
        if (j < L) {
            nrow *= p->e[j];
            trows *= n;
        }
        if (cells > 16384 || nrow > STABLE_TILE_ROWS || trows * B > 0x7fffffff || reach > 0x7fffffff) return false;
    }
    const int64_t lanes = nrow * stable_lanes(D);
    p->cells = int(cells);
    p->nrow = int(nrow);
    p->nhalo = int(h1 + h2);
    p->trows = trows;
    p->launches = int(launches);
    p->threads = int((lanes + MM_WAVE - 1) / MM_WAVE * MM_WAVE);
    p->shmem = size_t(cells) * 16 + size_t(p->e[L] + 1) * 16;
    if (p->threads > 1024 || int64_t(p->shmem) > ds->max_lds || trows * B * p->threads > 0xffffffffll) return false;
    if (p->whole()) return true;
    if (size_t(p->nhalo) * sizeof(StableHalo) > ws_bytes) return false;
    // A launch costs 3.5 us, a step 0.45 us and 0.01 us per wave, a halo cell
    // 4 ns, a tile of a CU 1.2 us; tiles beyond those resident at once run in
    // rounds (the middle launches have about 1.6 times the mean of tiles).
    // Fitted to (40,)^4 in tiles of 3 to 6 points, (70, 70, 60), (1000, 1000),
    // (20,)^5 and (11,)^6, which it meets to within 25 %.
    const int waves = p->threads / MM_WAVE;
    const int64_t per_cu = std::max<int64_t>(1, std::min<int64_t>(ds->max_lds / int64_t(p->shmem), 16 / waves));
    const double on_cu = tiles / double(launches) / ds->num_cu;
    const double rounds = std::max(1.0, 1.6 * on_cu / double(per_cu));
    p->us = double(launches) * (3.5 + 1.2 * on_cu + rounds * (0.004 * p->nhalo + double(steps) * (0.45 + 0.01 * waves)));
    return true;
}

}  // namespace

bool stable_tile_plan(const Lat &g, int64_t B, size_t ws_bytes, const DevState *ds, StableTilePlan *best) {
    const int D = g.D, L = D - 1;
    if (D > 6) return false;  // the box of the smallest tile, 4^7 cells, is larger than the LDS
    int e[8];
    for (int j = 0; j < D; ++j) e[j] = g.shape[j];
    if (try_tiles(g, B, ws_bytes, ds, e, best)) return true;
    static const int edges[] = {2, 3, 4, 5, 6, 8, 10, 12, 16, 24, 32, 48, 64};
    bool found = false;
    for (int edge : edges)
        for (int wide = 1; wide <= (D == 1 ? 64 : 2); wide *= 2) {  // rows of one edge or two
            for (int j = 0; j < D; ++j) e[j] = std::min(j == L ? edge * wide : edge, int(g.shape[j]));
            StableTilePlan p;
            if (!try_tiles(g, B, ws_bytes, ds, e, &p)) continue;
            if (!found || p.us < best->us) *best = p;
            found = true;
        }
    return found;
}

int launch_stable_tiles(const StableTilePlan &p, const Lat &g, int64_t B, const double *A, const double *b, const double *c, double *G,
                        void *ws, int *nf, const DevState *ds, hipStream_t s) {
    StableTileArgs a;
    memset(&a, 0, sizeof(a));
    a.g = g;
    a.A = reinterpret_cast<const double2 *>(A);
    a.b = reinterpret_cast<const double2 *>(b);
    a.c = reinterpret_cast<const double2 *>(c);
    a.G = reinterpret_cast<double2 *>(G);
    a.sq = ds->sq;
    a.rsq = ds->rsq;
    for (int j = 0; j < g.D; ++j) {
        a.e[j] = p.e[j];
        a.nt[j] = p.nt[j];
        a.h[j] = p.h[j];
        a.ls[j] = p.ls[j];
        a.em[j] = divide_magic(uint32_t(p.e[j]));
    }
    {
        // rows of one digit sum are active in the same steps: side by side, so
        // that the waves of the others skip the step
        int at[STABLE_TILE_ROWS + 1] = {0};
        auto sum_of = [&](int r) {
            int sum = 0;
            for (int j = g.D - 2; j >= 0; --j) {
                sum += r % p.e[j];
                r /= p.e[j];
            }
            return sum;
        };
        for (int r = 0; r < p.nrow; ++r) ++at[sum_of(r) + 1];
        for (int x = 1; x <= STABLE_TILE_ROWS; ++x) at[x] += at[x - 1];
        for (int r = 0; r < p.nrow; ++r) a.order[at[sum_of(r)]++] = uint16_t(r);
    }
    a.cells = p.cells;
    a.nrow = p.nrow;
    a.trows = int(p.trows);
    a.whole = p.whole();
    a.single = B == 1;
    a.nhalo = p.nhalo;
    a.halo = reinterpret_cast<const StableHalo *>(ws);
    a.nf = nf;
    if (!a.whole && B > 1) {
        hipLaunchKernelGGL(clear_flag_kernel, dim3(1), dim3(1), 0, s, nf);
        LAUNCH_CHECK("clear_flag_kernel");
    }
    for (int w = 0; w < p.launches; ++w) {
        a.w = w;
        // launch w = 0 of one triple: its first tile row alone
        const unsigned grid = unsigned(w == 0 && B == 1 ? 1 : p.trows * B);
        switch (g.D) {
#define CASE(DD)                                                                                                             \
    case DD:                                                                                                                 \
        if (w == 0) {                                                                                                        \
            raise_lds_limit(stable_tile_kernel<DD>, int(p.shmem));                                                           \
            if (!a.whole)                                                                                                    \
                hipLaunchKernelGGL((stable_halo_kernel<DD>), dim3(1), dim3(1024), 0, s, a, reinterpret_cast<StableHalo *>(ws)); \
        }                                                                                                                    \
        hipLaunchKernelGGL((stable_tile_kernel<DD>), dim3(grid), dim3(unsigned(p.threads)), p.shmem, s, a);                  \
        break;
            CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6)
#undef CASE
            default:
                return fail(MM_ERR_INVALID, "bad D");
        }
        LAUNCH_CHECK("stable_tile_kernel");
    }
    return MM_OK;
}

}  // namespace mm
