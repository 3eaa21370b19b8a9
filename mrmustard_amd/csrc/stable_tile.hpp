// The all-pivot ("stable") recurrence of core.py:183-211 in tiles.
//
// A point needs every point one and two index sums below it, so the lattice
// has sum(shape) dependent steps however it is cut.  One launch per index sum
// pays a launch for each of them; here the box is cut into tiles of a few
// points per axis, one workgroup sweeps a tile's index sums in LDS, and the
// tiles t with sum(t) = w run together in launch w: a tile reads only tiles
// below it along some axes, which an earlier launch finished.  A launch then
// covers sum(e_j - 1) + 1 index sums at the price of an LDS step each.
//
// What bounds a step is the dependent chain of one point: LDS reads, D + 1
// complex products per pivot, a division per pivot and the final one.  So the
// D pivots of a point sit in neighbouring lanes (P lanes, a power of two),
// their terms are added in the order of the axes through DPP moves, and what
// does not change along the last axis (the products A_ij sqrt(k_j), the pivots'
// roots) stays in registers of the lanes that own the row.
// The rows are dealt to the lanes by digit sum, so that a wave without a point
// in a step skips it.  Every term, order and rounding is that of stable_point.
// Measured, one launch per index sum (or one workgroup per triple) against the
// tiles: (40,)^4 858 -> 550 us (37 launches of 4^4 tiles, 13 steps of ~0.5 us
// each), (70, 70, 60) 752 -> 344 us, (1000, 1000) 6529 -> 1970 us (31
// launches), (20,)^5 1206 -> 906 us, (50, 50) 100 -> 41 us (the whole lattice one
// tile), 1000 of (5,)^4 142 -> 43 us; but (11,)^6 912 -> 1521 us, where the halo of
// a 2^6 tile is ten times its points: the caller compares both estimates.
#pragma once

#include "common.hpp"
#include "exact.hpp"

namespace mm {

// Most rows of a tile (two lanes each at least, in a workgroup of 1024).
constexpr int STABLE_TILE_ROWS = 512;

// A cell of the box outside the tile: its place in the lattice from the tile's
// first point, in the box, and the axes along which it lies below the tile.
struct StableHalo {
    int32_t f;
    uint16_t idx, below;
};

struct StableTileArgs {
    Lat g;
    const double2 *A, *b, *c;
    double2 *G;
    const double *sq, *rsq;
    int e[8];       // points of a tile along each axis
    int nt[8];      // tiles along each axis
    int h[8];       // cells below the tile that the LDS box holds (2; 0 when the axis is one tile)
    int ls[8];      // strides of the LDS box
    uint32_t em[8];  // divide_magic of e
    const StableHalo *halo;  // the cells of the box below the tile that its points read
    int nhalo;
    int cells;      // its size
    int nrow;       // rows of a tile: the product of e over the axes but the last
    int trows;      // tile rows: the product of nt over the axes but the last
    int w;          // sum of the tile coordinates
    int whole;      // the tile is the lattice
    int single;     // one triple: the launch w = 0 sets the flag, no launch clears it
    int *nf;        // raised when a stored value is not finite (unless whole)
    uint16_t order[STABLE_TILE_ROWS];  // the rows of a tile by digit sum
    int ntriples;   // BATCH
    int row0;       // BATCH: first tile row of this launch
};

// Lanes per point.
constexpr int stable_lanes(int D) { return D <= 2 ? 2 : (D <= 4 ? 4 : 8); }

// DPP move of a complex value; every lane that is read is active.
template <int CTRL>
__device__ __forceinline__ double2 dpp_z(double2 v) {
    auto mov = [](double x) {
        return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(x), CTRL, 0xF, 0xF, true),
                                __builtin_amdgcn_mov_dpp(__double2loint(x), CTRL, 0xF, 0xF, true));
    };
    return make_double2(mov(v.x), mov(v.y));
}

// The quotients of cdiv_by without its branch: right unless quotient_rare(v).
// A non-finite v gives a non-finite quotient here, and the triple is rerun.
__device__ __forceinline__ double2 cdiv_fast(double2 v, double s, double r) {
    const double2 q = make_double2(v.x * r, v.y * r);
    return make_double2(fma(fma(-q.x, s, v.x), r, q.x), fma(fma(-q.y, s, v.y), r, q.y));
}

__device__ __forceinline__ bool quotient_rare(double2 v) {
    return (fabs(v.x) < 0x1p-960 && v.x != 0.0) || (fabs(v.y) < 0x1p-960 && v.y != 0.0);
}

// The list of halo cells, in any order (a tile's cells differ from one another).
template <int D>
__global__ __launch_bounds__(1024) void stable_halo_kernel(StableTileArgs a, StableHalo *out) {
    __shared__ int count;
    if (threadIdx.x == 0) count = 0;
    __syncthreads();
    for (int x = threadIdx.x; x < a.cells; x += blockDim.x) {
        int rem = x, under = 0;
        int64_t f = 0;
        uint32_t below = 0;
#pragma unroll
        for (int j = 0; j < D; ++j) {
            const int cj = rem / a.ls[j];
            rem -= cj * a.ls[j];
            const int u = max(0, a.h[j] - cj);
            under += u;
            below |= u ? 1u << j : 0u;
            f += (cj - a.h[j]) * a.g.stride[j];
        }
        if (under >= 1 && under <= 2) {
            const int n = atomicAdd(&count, 1);
            if (n < a.nhalo) out[n] = StableHalo{int32_t(f), uint16_t(x), uint16_t(below)};
        }
    }
}

// BATCH, eight or more triples of several tiles: the triples along x and the tile rows
// along y, so that the rows of one w spread over the XCDs and a triple's launches
// find its halo in one L2 ((5,)^5 in batches of 1,024: 3.6 -> 0.9 ms, where the tile
// rows along x left some launches with one XCD).
template <int D, bool BATCH>
__global__ __launch_bounds__(1024) void stable_tile_kernel(StableTileArgs a) {
    constexpr int P = stable_lanes(D), L = D - 1;
    extern __shared__ __align__(16) char lds[];
    __shared__ double2 red[16];
    double2 *cell = reinterpret_cast<double2 *>(lds);
    double *sqt = reinterpret_cast<double *>(cell + a.cells);  // sqrt(base[L] - 1 + x)
    double *rst = sqt + a.e[L] + 1;
    const int64_t t = BATCH ? blockIdx.x : blockIdx.x / a.trows;
    if (BATCH && t >= a.ntriples) return;
    int base[D], ext[D];
    {
        int r = BATCH ? a.row0 + int(blockIdx.y) : int(blockIdx.x - t * a.trows), w = a.w;
#pragma unroll
        for (int j = D - 2; j >= 0; --j) {
            const int tj = r % a.nt[j];
            r /= a.nt[j];
            w -= tj;
            base[j] = tj * a.e[j];
        }
        if (w < 0 || w >= a.nt[L]) return;
        base[L] = w * a.e[L];
    }
    int steps = 1;
#pragma unroll
    for (int j = 0; j < D; ++j) {
        ext[j] = min(a.e[j], a.g.shape[j] - base[j]);
        steps += ext[j] - 1;
    }
    const double2 *A = a.A + t * D * D;
    const double2 *b = a.b + t * D;
    double2 *G = a.G + t * a.g.N;

    for (int x = threadIdx.x; x <= a.e[L]; x += blockDim.x) {
        const int k = max(0, min(base[L] - 1 + x, a.g.shape[L] - 1));
        sqt[x] = a.sq[k];
        rst[x] = a.rsq[k];
    }

    // this lane: pivot i of row `row`
    const int row = a.order[min(int(threadIdx.x / P), a.nrow - 1)], lane = threadIdx.x % P, i = min(lane, L);
    const bool last = i == L;
    bool mine = int(threadIdx.x / P) < a.nrow;
    int sum0 = 0, ksum = base[L], at = a.h[L], pstep = 0, ki = 0;
    int off[D];
    double2 coef[D];
    uint32_t on = 0;
    int64_t frow = base[L];
    {
        int r = row;
#pragma unroll
        for (int j = D - 2; j >= 0; --j) {
            const int cj = r - divide(r, a.em[j]) * a.e[j];
            r = divide(r, a.em[j]);
            const int kj = base[j] + cj;
            mine = mine && cj < ext[j];
            sum0 += cj;
            ksum += kj;
            frow += kj * a.g.stride[j];
            at += (cj + a.h[j]) * a.ls[j];
            on |= kj > 0 ? 1u << j : 0u;
            const bool self = j == i;
            if (self) {
                ki = kj;
                pstep = kj > 0 ? a.ls[j] : 0;
            }
            const int kw = min(self ? max(kj - 1, 0) : kj, a.g.shape[j] - 1);
            off[j] = (self ? kj >= 2 : kj > 0) ? a.ls[j] : 0;
            coef[j] = cscale_promoted(A[i * D + j], a.sq[kw]);
        }
    }
    const double2 bi = b[i], al = A[i * D + L];
    double s = 1.0, rs = 1.0;
    if (!last && mine) {
        s = a.sq[ki];
        rs = a.rsq[ki];
    }
    const double n0 = double(max(1, __popc(on))), n1 = double(__popc(on) + 1);
    double rn0 = 1.0 / n0, rn1 = 1.0 / n1;
    asm("" : "+v"(rn0), "+v"(rn1));  // two reciprocals here, not a division in every step
    const double2 c = a.c[t];
    // the cells one and two index sums below the tile's faces
    if (!a.whole) {
        uint32_t floor = 0;  // axes with nothing below the tile
        int64_t f0 = 0;
#pragma unroll
        for (int j = 0; j < D; ++j) {
            floor |= base[j] == 0 ? 1u << j : 0u;
            f0 += base[j] * a.g.stride[j];
        }
        constexpr int FLIGHT = 4;  // loads of a thread in flight
        for (int x0 = threadIdx.x; x0 < a.nhalo; x0 += FLIGHT * blockDim.x) {
            StableHalo e[FLIGHT];
            double2 v[FLIGHT];
#pragma unroll
            for (int u = 0; u < FLIGHT; ++u) {
                const int x = x0 + u * int(blockDim.x);
                e[u] = a.halo[min(x, a.nhalo - 1)];
                if (x >= a.nhalo) e[u].below = 0xFFFF;
            }
#pragma unroll
            for (int u = 0; u < FLIGHT; ++u) {
                const int64_t f = f0 + e[u].f;
                const bool use = (e[u].below & floor) == 0 && e[u].below != 0xFFFF && f < a.g.N;
                if (use) v[u] = G[f];
                else e[u].below = 0xFFFF;
            }
#pragma unroll
            for (int u = 0; u < FLIGHT; ++u)
                if (e[u].below != 0xFFFF) cell[e[u].idx] = v[u];
        }
    }
    __syncthreads();

    for (int step = 0; step < steps; ++step) {
        const int cl = step - sum0;
        if (mine && cl >= 0 && cl < ext[L]) {
            const int kl = base[L] + cl;
            const int idx = at + cl;
            const int p = idx - (last ? (kl > 0 ? 1 : 0) : pstep);
            const double wl = sqt[last ? cl : cl + 1];
            if (last) {
                s = sqt[cl + 1];
                rs = rst[cl + 1];
            }
            // every read of the term first; a zero weight reads the pivot's own cell
            const double2 g0 = cell[p];
            double2 nb[D];
#pragma unroll
            for (int j = 0; j < L; ++j) nb[j] = cell[p - off[j]];
            nb[L] = cell[p - ((last ? kl >= 2 : kl > 0) ? 1 : 0)];
            double2 val = cmul(bi, g0);
#pragma unroll
            for (int j = 0; j < L; ++j) val = cadd(val, cmul(coef[j], nb[j]));
            val = cadd(val, cmul(cscale_promoted(al, wl), nb[L]));
            double2 term = cdiv_fast(val, s, rs);
            if (__builtin_expect(quotient_rare(val), 0)) term = cdiv_promoted(val, s);
            // the terms in the order of the axes; -0.0 in the place of a pivot
            // with k_i = 0 leaves every sum as it is
            const bool lit = last ? kl > 0 : (on >> i) & 1u;
            term = csel(lit, term, make_double2(-0.0, -0.0));
            double2 vals = make_double2(0.0, 0.0);
#define MM_TERM(I, CTRL) \
    if constexpr ((I) < D) vals = cadd(vals, dpp_z<CTRL>(term));
            if constexpr (P == 2) {
                MM_TERM(0, 0xA0)  // quad_perm [0,0,2,2]
                MM_TERM(1, 0xF5)  // quad_perm [1,1,3,3]
            } else {
                MM_TERM(0, 0x00)  // quad_perm: lane 0 of the quad, ...
                MM_TERM(1, 0x55)
                MM_TERM(2, 0xAA)
                MM_TERM(3, 0xFF)
                if constexpr (P == 8) {  // the upper quad goes on from the lower one's sum
                    vals = dpp_z<0x141>(vals);  // row_half_mirror
                    MM_TERM(4, 0x00)
                    MM_TERM(5, 0x55)
                    MM_TERM(6, 0xAA)
                    MM_TERM(7, 0xFF)
                }
            }
#undef MM_TERM
            // cdiv_py by the number of pivots: a sum that starts at +0 is never
            // -0, so its zero terms change nothing
            const double n = kl > 0 ? n1 : n0, rn = kl > 0 ? rn1 : rn0;
            double2 out = cdiv_fast(vals, n, rn);
            if (__builtin_expect(quotient_rare(vals), 0)) out = make_double2(vals.x / n, vals.y / n);
            out = csel(ksum + cl == 0, c, out);
            if (lane == (P == 8 ? 4 : 0)) cell[idx] = out;
        }
        lds_barrier();
    }

    bool bad = false;
    if (mine) {
        for (int cl = lane; cl < ext[L]; cl += P) {
            const double2 z = cell[at + cl];
            G[frow + cl] = z;
            bad = bad || !finite2(z);
        }
    }
    const bool any = __syncthreads_or(bad);
    if (a.whole) {
        // non-finite values: the reference's sequential sweep with every term
        if (any) exact_stable_forward<D>(BlockOps(red), a.g, A, b, c, G, a.sq);
    } else if (threadIdx.x == 0) {
        if (a.single && a.w == 0) *a.nf = any;
        else if (any) atomicOr(a.nf, 1);
    }
}

}  // namespace mm
