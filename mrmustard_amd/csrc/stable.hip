// libmmhip: plan and launches of the tiled stable sweep (stable_tile_kernel).

#include "stable_launch.hpp"

#include "lds_launch.hpp"
#include "stable_tile.hpp"

namespace mm {

namespace {

__global__ void clear_flag_kernel(int *nf) { *nf = 0; }

// Blocks of a tile row in a launch of B triples: from one per XCD a multiple of the
// XCDs, so that a triple stays on one.
int64_t triple_lanes(int64_t B) { return B < MM_XCDS ? B : (B + MM_XCDS - 1) / MM_XCDS * MM_XCDS; }

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
        if (cells > 16384 || nrow > STABLE_TILE_ROWS || trows * triple_lanes(B) > 0x7fffffff || reach > 0x7fffffff) return false;
    }
    const int64_t lanes = nrow * stable_lanes(D);
    p->cells = int(cells);
    p->nrow = int(nrow);
    p->nhalo = int(h1 + h2);
    p->trows = trows;
    p->launches = int(launches);
    p->threads = int((lanes + MM_WAVE - 1) / MM_WAVE * MM_WAVE);
    p->shmem = size_t(cells) * 16 + size_t(p->e[L] + 1) * 16;
    if (p->threads > 1024 || int64_t(p->shmem) > ds->max_lds || trows * triple_lanes(B) * p->threads > 0xffffffffll) return false;
    if (p->whole()) return true;
    if (size_t(p->nhalo) * sizeof(StableHalo) > ws_bytes) return false;
    // A launch costs 3.5 us, a step 0.45 us and 0.01 us per wave, a halo cell
    // 4 ns: the time of one tile.  Tiles beyond about half of one per CU and
    // launch (D = 6: any) share their CU; it gains from three of the smallest tiles
    // and of those of D >= 5 at most, where they cost 1.3 to 1.7 times their share.  A
    // block without a tile costs 0.2 ns a wave.  Meets (4,)^5 to (10,)^6, (20,)^3 to (20,)^4 and (40,)^4 in batches of 1 to
    // 2,048 to within 25 %, a few to 40 %.
    const int waves = p->threads / MM_WAVE;
    int64_t per_cu = std::max<int64_t>(1, std::min<int64_t>(ds->max_lds / int64_t(p->shmem), 16 / waves));
    if (D >= 5 || (D == 4 && waves < 4)) per_cu = std::min<int64_t>(per_cu, 3);
    const double tile = 0.004 * p->nhalo + double(steps) * (0.45 + 0.01 * waves);
    const double shared = std::max(0.0, tiles / ds->num_cu - (D <= 5 ? 0.5 * double(launches) : 0.0));
    const double idle = double(trows) * double(B) * double(launches) - tiles;
    p->batch = B >= MM_XCDS && tiles > 0.4 * ds->num_cu * double(launches);
    p->us = double(launches) * (3.5 + tile) + shared * tile / double(per_cu) * (D <= 4 ? 1.0 : (D == 5 ? 1.3 : 1.7)) + 0.2e-3 * waves * idle;
    return true;
}

template <int D, bool BATCH>
int sweep_tiles(StableTileArgs &a, const StableTilePlan &p, int64_t B, void *ws, hipStream_t s) {
    raise_lds_limit(stable_tile_kernel<D, BATCH>, int(p.shmem));
    if (!a.whole) {
        hipLaunchKernelGGL((stable_halo_kernel<D>), dim3(1), dim3(1024), 0, s, a, reinterpret_cast<StableHalo *>(ws));
        LAUNCH_CHECK("stable_halo_kernel");
    }
    // BATCH from 0.4 tiles a CU and launch: (7,)^4 in batches of 64 66 -> 57 us, but (200, 200)
    // in batches of 30 (0.27) 298 -> 310
    for (a.w = 0; a.w < p.launches; ++a.w)
        for (int64_t row = 0; row < (BATCH ? p.trows : 1); row += 65535) {  // grid y
            a.row0 = int(row);
            // launch w = 0 of one triple: its first tile row alone
            const dim3 grid = BATCH ? dim3(unsigned(triple_lanes(B)), unsigned(std::min<int64_t>(65535, p.trows - row)))
                                    : dim3(unsigned(a.w == 0 && B == 1 ? 1 : p.trows * B));
            hipLaunchKernelGGL((stable_tile_kernel<D, BATCH>), grid, dim3(unsigned(p.threads)), p.shmem, s, a);
            LAUNCH_CHECK("stable_tile_kernel");
        }
    return MM_OK;
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
    a.ntriples = int(B);
    a.single = B == 1;
    a.whole = p.whole();
    a.nhalo = p.nhalo;
    a.halo = reinterpret_cast<const StableHalo *>(ws);
    a.nf = nf;
    if (!a.whole && B > 1) {
        hipLaunchKernelGGL(clear_flag_kernel, dim3(1), dim3(1), 0, s, nf);
        LAUNCH_CHECK("clear_flag_kernel");
    }
    switch (g.D) {
#define CASE(DD) \
    case DD: return p.batch ? sweep_tiles<DD, true>(a, p, B, ws, s) : sweep_tiles<DD, false>(a, p, B, ws, s);
        CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6)
#undef CASE
        default:
            return fail(MM_ERR_INVALID, "bad D");
    }
}

}  // namespace mm
