// The closed-form VJP of a lattice (gradients.py:64-80) as one Gram product
// per pair of neighbour sets, with the recompute sweep's next slab formed from
// the same loads.
//
// With k = q + 1_i in the reference's sums, every term becomes a product of
// two vectors at one point q:
//   v_j(q) = sqrt(q_j) G[q - 1_j],   u_i(q) = sqrt(q_i + 1) g[q + 1_i],
//   dA_ij = sum_q u_i v_j (j > i),  dA_ii = sum_q u_i v_i / 2,
//   db_i = sum_q u_i G[q],  dc = sum_q G[q] g[q] / c,
// so a point gathers 2 D + 2 values instead of one per sum (D (D + 3) / 2 + 2)
// and no cotangent twice.  A zero weight (q_j = 0, or q_i the last of its
// axis) reads the point itself: branch-free, all gathers issue together.
// The sums live in registers, a wave takes them over every VJP_CHAIN points
// (one sum per lane), a block adds its waves' and writes one partial row,
// vjp_finalize adds the rows of a triple in order: deterministic.
#pragma once

#include <type_traits>

#include "common.hpp"
#include "exact.hpp"
#include "global_kernels.hpp"

namespace mm {

// Largest axis whose square roots sit in LDS (LT kernels); longer ones are
// read from the device table.
constexpr int VJP_LDS_SQ = 4096;

// Points that a thread sums before the wave takes its sums: the rounding error
// of a chain of n terms grows as sqrt(n), and large lattices have hundreds of
// points per thread.  Error of the sums in eps sqrt(sum |term|^2), chains of
// all points against these: (11,)^7 kets 4.7 -> 1.3, (8,)^8 density matrices 3.4
// -> 1.3, (10,)^8 slab by slab 3.3 -> 1.2, (12,)^6 1.7 -> 1.1; the time of all of
// them is the same within 1 % (a scatter_sum is 5 to 7 % of 16 points' instructions,
// and the kernel waits for memory).
constexpr int VJP_CHAIN = 16;

struct VjpArgs {
    Geom g;
    const double2 *G;    // lattice; SLAB: level-0 slab m
    const double2 *Gdn;  // SLAB: slab m - 1 (m = 0: slab 0, weight sqrt(0))
    const double2 *gg;   // cotangent, as G
    const double2 *gup;  // SLAB: slab m + 1 of the cotangent (last m: slab m, weight 0)
    double2 *nxt;        // FWD: slab m + 1
    const double2 *A, *b;
    double2 *partial;    // nchunk rows of D (D + 1) / 2 + D + 1 sums per triple
    const double *sq, *rsq;
    double gsign;        // -1: the cotangent is read conjugated
    int m;               // SLAB: k_0
    int nchunk;          // blocks per triple and row group
    int visit;           // consecutive 256-point groups a block takes at a time
    int smax;            // LT: entries of the LDS table - 2
};

// Accumulators of one group of pivot rows [R0, R1): dA(i, j) for R0 <= i < R1
// and all j >= i, db_i for those rows, and dc with the first group.
template <int D, int R0, int R1>
struct RowGroup {
    static constexpr int NT = D * (D + 1) / 2;
    static constexpr int NA = NT + D + 1;
    static constexpr int NROWA = (R1 - R0) * D - (R1 * (R1 - 1) - R0 * (R0 - 1)) / 2;  // sum_{i=R0}^{R1-1} (D - i)
    static constexpr int NL = NROWA + (R1 - R0) + (R0 == 0 ? 1 : 0);
    static __host__ __device__ constexpr int la(int i, int j) { return (i - R0) * D - (i * (i - 1) - R0 * (R0 - 1)) / 2 + (j - i); }
    static __host__ __device__ constexpr int lb(int i) { return NROWA + (i - R0); }
    static __host__ __device__ constexpr int lc() { return NROWA + (R1 - R0); }
    // column of local sum l in the full layout (upper triangle of dA, db, dc)
    static __device__ int column(int l) {
        if (R0 == 0 && l == lc()) return NA - 1;
        if (l >= NROWA) return NT + R0 + (l - NROWA);
        int i = R0, off = 0;
        while (l - off >= D - i) {
            off += D - i;
            ++i;
        }
        return i * D - i * (i - 1) / 2 + (l - off);
    }
};

// Sums of N <= 64 values over the wave, lane l keeping the sum of value
// bit-reverse(l) (6 bits): each stage halves the values instead of summing all
// of them on every lane, 240 instructions for 60 values where wave_sum_dpp has
// 1,080.  The order is fixed.
template <int STAGE>
__device__ __forceinline__ double pair_sum(double x, double y) {
    if constexpr (STAGE < 2) {
        // lanes 32 (16) and up of x against those below of y
        auto swap = [](int u, int v) {
            if constexpr (STAGE == 0) return __builtin_amdgcn_permlane32_swap(u, v, false, false);
            else return __builtin_amdgcn_permlane16_swap(u, v, false, false);
        };
        const auto lo = swap(__double2loint(x), __double2loint(y));
        const auto hi = swap(__double2hiint(x), __double2hiint(y));
        return __hiloint2double(int(hi[0]), int(lo[0])) + __hiloint2double(int(hi[1]), int(lo[1]));
    } else {
        // row_mirror, row_half_mirror, quad_perm [2,3,0,1] and [1,0,3,2]
        constexpr int CTRL[] = {0x140, 0x141, 0x4E, 0xB1};
        const bool up = (threadIdx.x >> (5 - STAGE)) & 1;
        const double keep = up ? y : x, give = up ? x : y;
        return keep + dpp_d<CTRL[STAGE - 2], 0xF>(give);
    }
}

template <int STAGE, int N>
__device__ __forceinline__ double scatter_sum(const double (&v)[N]) {
    constexpr int H = (N + 1) / 2;
    double h[H];
#pragma unroll
    for (int i = 0; i < H; ++i) h[i] = pair_sum<STAGE>(v[2 * i], 2 * i + 1 < N ? v[2 * i + 1] : 0.0);
    if constexpr (STAGE == 5) return h[0];
    else return scatter_sum<STAGE + 1>(h);
}

// Move a thread's sums into the lane's own one of the wave (component 2 l of
// sum l, 2 l + 1 its imaginary part), and start them again from zero.
template <int D, int R0, int R1, int NL>
__device__ __forceinline__ void flush_sums(double2 (&acc)[NL], double &held) {
    using RG = RowGroup<D, R0, R1>;
    static_assert(NL == RG::NL && 2 * NL <= MM_WAVE, "accumulator count");
    double v[2 * NL];
#pragma unroll
    for (int e = 0; e < NL; ++e) {
        v[2 * e] = acc[e].x;
        v[2 * e + 1] = acc[e].y;
        acc[e] = make_double2(0.0, 0.0);
    }
#pragma unroll
    for (int i = R0; i < R1; ++i) {  // dA_ii = sum u_i v_i / 2
        v[2 * RG::la(i, i)] *= 0.5;
        v[2 * RG::la(i, i) + 1] *= 0.5;
    }
    held += scatter_sum<0>(v);
}

// Sum the waves' held sums in order and store them in, or add them to, the
// block's partial row at the group's columns.
template <int D, int R0, int R1>
__device__ __forceinline__ void block_store_group(double held, double2 *row, bool add) {
    using RG = RowGroup<D, R0, R1>;
    __shared__ double red[256];
    red[threadIdx.x] = held;
    __syncthreads();
    const int t = threadIdx.x;
    if (t < 2 * RG::NL) {
        const int lane = int(__brev(uint32_t(t)) >> 26);
        double sum = red[lane];
        for (int w = 1; w < 256 / MM_WAVE; ++w) sum += red[w * MM_WAVE + lane];
        double *out = reinterpret_cast<double *>(row + RG::column(t / 2)) + (t & 1);
        *out = add ? *out + sum : sum;
    }
}

// Row groups per D.  D <= 6: all sums in one group (28 complex sums, 112
// registers, at D = 6).  D = 7, 8 (36 and 45 sums) would leave one wave per
// SIMD: two groups, which share their loads through L1.  The first carries
// the forward role.
template <int D>
struct RowSplit {
    static constexpr int NG = D <= 6 ? 1 : 2;
    static constexpr int B1 = D <= 6 ? D : 2;
};

// Chunk `blk` of nchunk over the points of one triple (SLAB: of slab m).
// Points are taken in visits of `visit` * 256 consecutive points; the blocks
// of one XCD (blk % 8, see xcd_block) take neighbouring visits and all
// blocks advance through the lattice together, so the strided neighbours of a
// point were or will be read nearby in time.
template <int D, int R0, int R1, bool SLAB, bool FWD, bool LT, bool I32>
__device__ __forceinline__ void vjp_group(const VjpArgs &a, const double *sqt, int blk, double2 *row) {
    using RG = RowGroup<D, R0, R1>;
    constexpr int NL = RG::NL;
    constexpr int LO = SLAB ? 1 : 0;  // first axis with a digit
    const double *sq = LT ? sqt : a.sq;
    // I32: the points' byte offsets from the arrays' (uniform) addresses fit 32
    // bits.  Half of the kernel's issue slots were busy, a third of them with 64-bit
    // addresses: a slab of 10^7 points of D = 8 with the next one formed 367 -> 322 us
    // (1.9 GB read, 0.16 written: 6.4 TB/s), (12,)^6 52.5 -> 48.
    using X = std::conditional_t<I32, uint32_t, int64_t>;
    auto at = [](const double2 *p, X x) {
        if constexpr (I32) return *reinterpret_cast<const double2 *>(reinterpret_cast<const char *>(p) + x * 16u);
        else return p[x];
    };
    const X S = X(SLAB ? a.g.stride[0] : a.g.N);
    double2 acc[NL];
#pragma unroll
    for (int e = 0; e < NL; ++e) acc[e] = make_double2(0.0, 0.0);
    const int m = a.m;
    const X round = X(a.nchunk) * 256 * a.visit;
    const int place = a.nchunk % MM_XCDS == 0 ? (blk % MM_XCDS) * (a.nchunk / MM_XCDS) + blk / MM_XCDS : blk;
    // points are taken from the last one down, q = S - 1 - p: the amplitudes of
    // a state fall off with the photon numbers, and small terms go first
    X p = X(place) * 256 * a.visit;  // of thread 0
    const X hop = round - X(256) * (a.visit - 1);
    X stl[D];
    int k[D], kin[D], khop[D];
#pragma unroll
    for (int i = 0; i < D; ++i) {
        stl[i] = X(a.g.stride[i]);
        k[i] = kin[i] = khop[i] = 0;
    }
    if (p + threadIdx.x < S) {
        // a step down is one up by S less, its last carry dropped
        digits_of<D>(S - 1 - (p + threadIdx.x), a.g, LO, k);
        digits_of<D>(256 < S ? S - 256 : 0, a.g, LO, kin);
        digits_of<D>(hop < S ? S - hop : 0, a.g, LO, khop);
    }
    const double gs = a.gsign;
    const double wdn0 = a.sq[m], wup0 = m + 1 < a.g.shape[0] ? a.sq[m + 1] : 0.0;  // SLAB: axis 0
    double2 b0 = make_double2(0.0, 0.0), c00 = b0, A0[D];
    double sm = 1.0, rm = 1.0;
    if (FWD) {
        b0 = a.b[0];
        c00 = cscale_promoted(a.A[0], a.sq[m]);
        sm = a.sq[m + 1];
        rm = a.rsq[m + 1];
#pragma unroll
        for (int j = 0; j < D; ++j) A0[j] = a.A[j];
    }
    int it = 0, chain = 0;
    double held = 0.0;
    while (p < S) {
        if (p + threadIdx.x < S) {
            const X q = S - 1 - (p + threadIdx.x);
            // every load of the point first: one round trip
            const double2 G0 = at(a.G, q);
            const double2 g0 = R0 == 0 ? at(a.gg, q) : make_double2(0.0, 0.0);
            double2 v[D], u[D];
            double wd[D], wu[D];
#pragma unroll
            for (int j = 0; j < D; ++j) {
                if (j < R0) continue;
                if (SLAB && j == 0) {
                    v[0] = at(a.Gdn, q);
                    wd[0] = wdn0;
                } else {
                    v[j] = at(a.G, q - (k[j] > 0 ? stl[j] : 0));
                    wd[j] = sq[k[j]];
                }
                if (j >= R1) continue;
                if (SLAB && j == 0) {
                    u[0] = at(a.gup, q);
                    wu[0] = wup0;
                } else {
                    const bool up = k[j] + 1 < a.g.shape[j];
                    u[j] = at(a.gg, q + (up ? stl[j] : 0));
                    const double w = sq[k[j] + 1];
                    wu[j] = up ? w : 0.0;
                }
            }
            if (FWD) {
                // the recurrence of fwd_slab0_kernel for slab m + 1, same order of operations
                double2 o = cmul(b0, G0);
                if (m >= 1) o = cadd(o, cmul(c00, v[0]));
#pragma unroll
                for (int j = 1; j < D; ++j) o = cadd(o, cmul(cscale_promoted(A0[j], wd[j]), v[j]));
                if constexpr (I32) *reinterpret_cast<double2 *>(reinterpret_cast<char *>(a.nxt) + q * 16u) = cdiv_by(o, sm, rm);
                else a.nxt[q] = cdiv_by(o, sm, rm);
            }
            if (R0 == 0) acc[RG::lc()] = cfma(G0, make_double2(g0.x, gs * g0.y), acc[RG::lc()]);
#pragma unroll
            for (int j = 0; j < D; ++j) {
                if (j < R0) continue;
                v[j] = make_double2(wd[j] * v[j].x, wd[j] * v[j].y);
            }
#pragma unroll
            for (int i = R0; i < R1; ++i) {
                const double2 ui = make_double2(wu[i] * u[i].x, (wu[i] * gs) * u[i].y);
                acc[RG::lb(i)] = cfma(G0, ui, acc[RG::lb(i)]);
#pragma unroll
                for (int j = i; j < D; ++j) acc[RG::la(i, j)] = cfma(v[j], ui, acc[RG::la(i, j)]);
            }
        }
        if (++chain == VJP_CHAIN) {
            chain = 0;
            flush_sums<D, R0, R1>(acc, held);
        }
        if (++it < a.visit) {
            p += 256;
            digits_add<D>(k, kin, a.g, LO);
        } else {
            it = 0;
            p += hop;
            digits_add<D>(k, khop, a.g, LO);
        }
    }
    flush_sums<D, R0, R1>(acc, held);
    block_store_group<D, R0, R1>(held, row, SLAB && m > 0);
}

// Waves per SIMD held to what the loads of a whole point need: left to aim
// higher, the compiler moves them to their uses ((20,)^5 41 -> 73 us, 96 of (12,)^4 27 ->
// 36; held, 39 and 25.5).
template <int D, bool SLAB, bool FWD, bool LT, bool I32>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(D <= 4 ? 3 : 2, D <= 2 ? 8 : (D == 3 ? 4 : (D == 4 ? 3 : 2))))) void
vjp_kernel(VjpArgs a) {
    extern __shared__ double sqt[];
    using RS = RowSplit<D>;
    if (LT) {
        for (int t = threadIdx.x; t < a.smax + 2; t += 256) sqt[t] = a.sq[t];
        __syncthreads();
    }
    const int64_t t = blockIdx.y;
    a.G += t * a.g.N;
    a.gg += t * a.g.N;
    constexpr int NA = D * (D + 1) / 2 + D + 1;
    // the row groups of one chunk run on one XCD (block index modulo 8)
    int grp = 0, blk = blockIdx.x;
    if (RS::NG == 2) {
        if (a.nchunk % MM_XCDS == 0) {
            const int j = blk / MM_XCDS;
            grp = j % 2;
            blk = (j / 2) * MM_XCDS + blk % MM_XCDS;
        } else {
            grp = blk % 2;
            blk /= 2;
        }
    }
    double2 *row = a.partial + (t * a.nchunk + blk) * NA;
    if (grp == 0) {
        vjp_group<D, 0, RS::B1, SLAB, FWD, LT, I32>(a, sqt, blk, row);
    } else {
        if constexpr (RS::NG == 2) vjp_group<D, RS::B1, D, SLAB, false, LT, I32>(a, sqt, blk, row);
    }
}

// One block per triple.  npart partial rows of NA sums each.  Wave w sums
// columns w, w + nwaves, ...: lane l adds rows l, l + 64, ... in order, then
// the lanes combine in a fixed butterfly, so the result does not depend on
// timing.  gsign = -1: the results are conjugated.
template <int D>
__global__ __launch_bounds__(1024) void vjp_finalize(const double2 *partial, int npart, const double2 *c, double2 *dA, double2 *db,
                                                     double2 *dc, double gsign) {
    constexpr int NA = D * (D + 1) / 2 + D + 1;
    constexpr int NT = D * (D + 1) / 2;
    __shared__ double2 s[NA];
    const int64_t t = blockIdx.x;
    const double2 *p = partial + t * npart * NA;
    const int lane = threadIdx.x & (MM_WAVE - 1);
    const int nw = blockDim.x / MM_WAVE;
    for (int e = threadIdx.x / MM_WAVE; e < NA; e += nw) {
        double2 acc = make_double2(0.0, 0.0);
#pragma unroll 8
        for (int r = lane; r < npart; r += MM_WAVE) acc = cadd(acc, p[int64_t(r) * NA + e]);
        acc = wave_sum(acc);
        if (lane == 0) s[e] = acc;
    }
    __syncthreads();
    if (threadIdx.x < D * D) {
        const int i = threadIdx.x / D, j = threadIdx.x % D;
        const int lo = i < j ? i : j, hi = i < j ? j : i;
        const double2 m = s[lo * D - lo * (lo - 1) / 2 + (hi - lo)];
        const double h = i == j ? 1.0 : 0.5;
        dA[t * D * D + threadIdx.x] = make_double2(h * m.x, (h * gsign) * m.y);
    }
    if (threadIdx.x < D) db[t * D + threadIdx.x] = make_double2(s[NT + threadIdx.x].x, gsign * s[NT + threadIdx.x].y);
    if (threadIdx.x == 0) {
        const double2 q = cdiv_py(s[NA - 1], c[t]);
        dc[t] = make_double2(q.x, gsign * q.y);
    }
}

// (A, b, c) of one triple conjugated into out: the VJP with torch's
// convention, conj(sum conj(grad) dG/dtheta), is the holomorphic VJP at the
// conjugated triple with the gradient as it is, bit for bit (every operation
// of the recurrence commutes with conjugation).
__global__ void conj_triple_kernel(const double2 *A, int nA, const double2 *b, int nb, const double2 *c, double2 *out) {
    for (int t = threadIdx.x; t < nA + nb + 1; t += blockDim.x) {
        const double2 z = t < nA ? A[t] : (t < nA + nb ? b[t - nA] : c[0]);
        out[t] = make_double2(z.x, -z.y);
    }
}

}  // namespace mm
