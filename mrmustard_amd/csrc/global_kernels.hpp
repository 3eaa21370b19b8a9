// Kernels that work on G in global memory: the per-slab forward for lattices
// whose slabs do not fit in LDS, and the all-pivot ("stable") recurrence swept
// by index-sum wavefronts.
#pragma once

#include "common.hpp"
#include "exact.hpp"
#include "jobs.hpp"

namespace mm {

struct Geom {
    int32_t D;
    int32_t shape[8];
    int64_t stride[8];
    int64_t N;
};

// Mixed-radix digits of x over axes [lo, D).  Lattices below 2^31 points use
// 32-bit divisions (a 64-bit one is a long software sequence, and a thread of
// a slab launch with one point per thread would spend most of its time here).
template <int D>
__device__ __forceinline__ void digits_of(int64_t x, const Geom &g, int lo, int (&k)[D]) {
    if (g.N <= int64_t(0x7fffffff)) {
        uint32_t r = uint32_t(x);
#pragma unroll
        for (int j = 0; j < D; ++j) {
            if (j < lo) {
                k[j] = 0;
                continue;
            }
            const uint32_t sj = uint32_t(g.stride[j]);
            const uint32_t dj = r / sj;
            r -= dj * sj;
            k[j] = int(dj);
        }
        return;
    }
#pragma unroll
    for (int j = 0; j < D; ++j) {
        if (j < lo) {
            k[j] = 0;
            continue;
        }
        int64_t dj = x / g.stride[j];
        x -= dj * g.stride[j];
        k[j] = int(dj);
    }
}

// k += inc (both as digits over axes [lo, D)); returns false on overflow past axis lo.
template <int D>
__device__ __forceinline__ bool digits_add(int (&k)[D], const int (&inc)[D], const Geom &g, int lo) {
    int carry = 0;
#pragma unroll
    for (int j = D - 1; j >= 0; --j) {
        if (j < lo) break;
        int v = k[j] + inc[j] + carry;
        carry = v >= g.shape[j];
        k[j] = carry ? v - g.shape[j] : v;
    }
    return carry == 0;
}

// ------------------------------------------------------------ per-slab forward
// Slab k_d = m of the sub-lattice {k_0..k_{d-1} = 0}: every point has pivot
// axis d (core.py:88-104 with i = d) and reads only slabs m-1 and m-2.
struct SlabArgs {
    Geom g;
    const double2 *A, *b;
    double2 *G;
    const double *sq, *rsq;
    int *nf;  // raised when a stored value is not finite
    int d, m;
};

template <int D>
__global__ __launch_bounds__(256) void fwd_slab_kernel(SlabArgs a) {
    const int d = a.d, m = a.m;
    const int64_t Sd = a.g.stride[d];
    const Span sp = xcd_span(xcd_block(blockIdx.x, gridDim.x), gridDim.x, Sd);
    const int64_t q0 = sp.q0, inc = sp.inc, hi = sp.hi;
    if (q0 >= hi) return;
    int k[D], ki[D];
    digits_of<D>(q0, a.g, d + 1, k);
    digits_of<D>(inc < Sd ? inc : 0, a.g, d + 1, ki);
    const double2 bd = a.b[d];
    const double2 cdd = cscale_promoted(a.A[d * D + d], a.sq[m > 0 ? m - 1 : 0]);
    const double sm = a.sq[m], rm = a.rsq[m];
    double2 Adj[D];
#pragma unroll
    for (int j = 0; j < D; ++j) Adj[j] = (j > d) ? a.A[d * D + j] : make_double2(0.0, 0.0);
    double2 *G = a.G;
    const int64_t base = int64_t(m) * Sd;
    bool bad = false;
    for (int64_t q = q0; q < hi; q += inc) {
        const int64_t f = base + q;
        // every load of the point first (one round trip); a term with k_j = 0
        // is the zero coefficient A_dj sqrt(0) times the point's own value,
        // as the reference adds it
        double2 nbv[D];
        double wv[D];
#pragma unroll
        for (int j = 1; j < D; ++j) {
            if (j <= d) continue;
            nbv[j] = G[f - Sd - (k[j] > 0 ? a.g.stride[j] : 0)];
            wv[j] = a.sq[k[j]];
        }
        double2 v = cmul(bd, G[f - Sd]);
        if (m >= 2) v = cadd(v, cmul(cdd, G[f - 2 * Sd]));
#pragma unroll
        for (int j = 1; j < D; ++j) {
            if (j <= d) continue;
            v = cadd(v, cmul(cscale_promoted(Adj[j], wv[j]), nbv[j]));
        }
        const double2 out = cdiv_by(v, sm, rm);
        G[f] = out;
        bad = bad || !finite2(out);
        if (q + inc < hi) digits_add<D>(k, ki, a.g, d + 1);
    }
    if (__builtin_expect(bad, 0) && a.nf) atomicOr(a.nf, 1);
}

// The same for slabs of up to 2^27 points (byte offsets of 32 bits from the
// slabs' addresses) whose coefficients A_dj sqrt(k_j) fit a small LDS table,
// row j - d - 1: of 450 vector instructions per 64 points at D = 8 the general
// kernel spends two thirds on 64-bit addresses, roots and coefficients.
// Measured at D = 8: 10^7 points 154 -> 132 us, 10^6 points 23.4 -> 18.5; (12,)^5
// points of D = 6 6.9 -> 6.5.
constexpr int64_t SLAB32_POINTS = int64_t(1) << 27;
constexpr int64_t SLAB32_TABLE = 16 * 1024;

template <int D>
__global__ __launch_bounds__(256) void fwd_slab32_kernel(SlabArgs a, int smax) {
    extern __shared__ __align__(16) char lds[];
    double2 *ctab = reinterpret_cast<double2 *>(lds);
    const int d = a.d, m = a.m;
    const int64_t Sd = a.g.stride[d];
    for (int t = threadIdx.x; t < (D - 1 - d) * smax; t += 256) {
        const int j = d + 1 + t / smax, k = t % smax;
        ctab[t] = k < a.g.shape[j] ? cscale_promoted(a.A[d * D + j], a.sq[k]) : make_double2(0.0, 0.0);
    }
    __syncthreads();
    const Span sp = xcd_span(xcd_block(blockIdx.x, gridDim.x), gridDim.x, Sd);
    const int inc = int(sp.inc), hi = int(sp.hi);
    int q = int(sp.q0);
    if (q >= hi) return;
    int k[D], ki[D];
    digits_of<D>(q, a.g, d + 1, k);
    digits_of<D>(inc < Sd ? inc : 0, a.g, d + 1, ki);
    const double2 bd = a.b[d];
    const double2 cdd = cscale_promoted(a.A[d * D + d], a.sq[m > 0 ? m - 1 : 0]);
    const double sm = a.sq[m], rm = a.rsq[m];
    const char *p1 = reinterpret_cast<const char *>(a.G + int64_t(m - 1) * Sd);
    const char *p2 = reinterpret_cast<const char *>(a.G + int64_t(m >= 2 ? m - 2 : m - 1) * Sd);
    char *out = reinterpret_cast<char *>(a.G + int64_t(m) * Sd);
    auto at = [](const char *p, uint32_t x) { return *reinterpret_cast<const double2 *>(p + x); };
    bool bad = false;
    for (; q < hi; q += inc) {
        const uint32_t x = uint32_t(q) * 16u;
        // every load of the point first, zero-digit terms as in fwd_slab_kernel
        double2 nbv[D];
#pragma unroll
        for (int j = 1; j < D; ++j) {
            if (j <= d) continue;
            nbv[j] = at(p1, x - (k[j] > 0 ? uint32_t(a.g.stride[j]) * 16u : 0u));
        }
        double2 v = cmul(bd, at(p1, x));
        if (m >= 2) v = cadd(v, cmul(cdd, at(p2, x)));
#pragma unroll
        for (int j = 1; j < D; ++j) {
            if (j <= d) continue;
            v = cadd(v, cmul(ctab[(j - d - 1) * smax + k[j]], nbv[j]));
        }
        const double2 o = cdiv_by(v, sm, rm);
        *reinterpret_cast<double2 *>(out + x) = o;
        bad = bad || !finite2(o);
        if (q + inc < hi) digits_add<D>(k, ki, a.g, d + 1);
    }
    if (__builtin_expect(bad, 0) && a.nf) atomicOr(a.nf, 1);
}

// --------------------------------------------- several slabs per launch
// Slabs m0 .. m0 + T - 1 of level d in one launch, for slabs small enough
// that a launch per slab costs more than the slab's work: one block of 1024
// threads per CU, packed digits and an LDS coefficient table (32-bit index
// arithmetic; fwd_slab_kernel takes any slab size).  A point of slab m reads
// slab m - 1 at its neighbours one below along the axes j > d and both slabs
// below at itself, so a block that owns a box of the axes > d computes slab
// m0 + s (phase s) on the box and on what its later phases read: the cells at
// most T - 1 - s below it, summed over the axes.  The cells of that larger
// box keep their place for the whole launch: a phase's values go through LDS
// to the next phase (two buffers), and a cell's own values of the two slabs
// below stay in the registers of its thread.  Phase 0 loads them and the
// neighbours in slab m0 - 1.  Only owned points are written to G, each by
// the expression of fwd_slab_kernel, so G is bit for bit the same; a term
// with k_j = 0 is added as the reference adds it, a zero coefficient
// A_dj sqrt(0) times a value read at the point itself (no branch per lane).
// A box has few cells below it where a run of consecutive points of the same
// size has the whole of its outer neighbours: of the (40,)^4 density matrix
// (39 slabs of 64,000 points) a block of 250 consecutive points computes 1,850
// for two slabs.  Measured there, the whole forward: 193 ->
// 148 us (four slabs a launch, boxes of 4 x 8 x 8 points); (60,)^3 161 -> 83 us,
// (300, 80, 60) 678 -> 279 us, (500, 150, 20) 1118 -> 474 us.
constexpr int MULTI_THREADS = 1024;
constexpr int MULTI_KMAX = 2;  // cells per thread (KM): more measured slower than a launch per slab
constexpr int MULTI_CELLS = MULTI_THREADS * MULTI_KMAX;

struct SlabMultiArgs {
    Geom g;
    const double2 *A, *b;
    double2 *G;
    const double *sq, *rsq;
    int *nf;  // raised when a stored value is not finite
    int d, m0, nphase;
    int e[8], nt[8], h[8], ls[8];  // axes > d: points of a box, boxes, cells below it (0 where the box spans the axis), cell strides
    uint32_t lsm[8];        // divide_magic of ls
    int cells;
    int smax;               // row length of the coefficient table (largest shape of the axes > d)
    int kbit[8], kmask[8];  // packed digits of the axes > d
};

template <int D, int KM>
__global__ __launch_bounds__(MULTI_THREADS) void fwd_slab_multi_kernel(SlabMultiArgs a) {
    extern __shared__ __align__(16) char lds[];
    double2 *buf0 = reinterpret_cast<double2 *>(lds);
    double2 *buf1 = buf0 + (a.nphase > 1 ? a.cells : 0);
    double2 *ctab = buf1 + (a.nphase > 2 ? a.cells : 0);  // A_dj sqrt(k_j) for j > d, row j - d - 1
    const double2 zero = make_double2(0.0, 0.0);
    const int d = a.d, T = a.nphase;
    const int Sd = int(a.g.stride[d]);
    for (int t = threadIdx.x; t < (D - 1 - d) * a.smax; t += blockDim.x) {
        const int j = d + 1 + t / a.smax, k = t % a.smax;
        ctab[t] = k < a.g.shape[j] ? cscale_promoted(a.A[d * D + j], a.sq[k]) : zero;
    }
    int st[D], base[D];
    {
        int r = int(xcd_block(blockIdx.x, gridDim.x));
#pragma unroll
        for (int j = D - 1; j >= 0; --j) {
            st[j] = int(a.g.stride[j]);
            base[j] = 0;
            if (j <= d) continue;
            const int tj = r % a.nt[j];
            r /= a.nt[j];
            base[j] = tj * a.e[j];
        }
    }
    // cell x0 + r * 1024 of this thread: its point of a slab, the cells it
    // lies below the box (T: no point), its packed digits
    uint32_t kp[KM];
    int qv[KM], under[KM];
    double2 p1v[KM], p2v[KM], nb0[KM][D];
    const int64_t base0 = int64_t(a.m0) * Sd;
    const double2 *G0 = a.G + base0 - Sd;  // slab m0 - 1
#pragma unroll
    for (int r = 0; r < KM; ++r) {
        const int x = int(threadIdx.x) + r * int(blockDim.x);
        int rem = x, u = 0, q = 0;
        bool in = x < a.cells;
        kp[r] = 0;
#pragma unroll
        for (int j = 0; j < D; ++j) {
            if (j <= d) continue;
            const int cj = divide(rem, a.lsm[j]);
            rem -= cj * a.ls[j];
            const int kj = base[j] + cj - a.h[j];
            u += max(0, a.h[j] - cj);
            in = in && kj >= 0 && kj < a.g.shape[j] && cj < a.e[j] + a.h[j];
            q += kj * st[j];
            kp[r] |= uint32_t(max(kj, 0)) << a.kbit[j];
        }
        under[r] = in ? u : T;
        qv[r] = in ? q : 0;
        p1v[r] = zero;
        p2v[r] = zero;
        if (under[r] < T) {
            p1v[r] = G0[q];
            if (a.m0 >= 2) p2v[r] = G0[q - Sd];
#pragma unroll
            for (int j = 1; j < D; ++j) {
                if (j <= d) continue;
                nb0[r][j] = G0[((kp[r] >> a.kbit[j]) & uint32_t(a.kmask[j])) ? q - st[j] : q];
            }
        }
    }
    __syncthreads();  // the coefficient table
    const double2 bd = a.b[d];
    bool bad = false;
    for (int s = 0; s < T; ++s) {
        const int m = a.m0 + s;
        const double2 *prev = (s & 1) ? buf0 : buf1;
        double2 *cur = (s & 1) ? buf1 : buf0;
        const double2 cdd = cscale_promoted(a.A[d * D + d], a.sq[m > 0 ? m - 1 : 0]);
        const double sm = a.sq[m], rm = a.rsq[m];
#pragma unroll
        for (int r = 0; r < KM; ++r) {
            if (under[r] >= T - s) continue;
            const int x = int(threadIdx.x) + r * int(blockDim.x), q = qv[r];
            // k_j = 0: the point itself times the zero coefficient A_dj sqrt(0)
            double2 nb[D];
            int kj[D];
#pragma unroll
            for (int j = 1; j < D; ++j) {
                if (j <= d) continue;
                kj[j] = int((kp[r] >> a.kbit[j]) & uint32_t(a.kmask[j]));
                nb[j] = s == 0 ? nb0[r][j] : prev[kj[j] > 0 ? x - a.ls[j] : x];
            }
            double2 v = cmul(bd, p1v[r]);
            if (m >= 2) v = cadd(v, cmul(cdd, p2v[r]));
#pragma unroll
            for (int j = 1; j < D; ++j) {
                if (j <= d) continue;
                v = cadd(v, cmul(ctab[(j - d - 1) * a.smax + kj[j]], nb[j]));
            }
            const double2 out = cdiv_by(v, sm, rm);
            if (s + 1 < T) cur[x] = out;
            if (under[r] == 0) {
                a.G[int64_t(m) * Sd + q] = out;
                bad = bad || !finite2(out);
            }
            p2v[r] = p1v[r];
            p1v[r] = out;
        }
        lds_barrier();  // stores to G need no wait: no later phase reads them
    }
    if (__builtin_expect(bad, 0) && a.nf) atomicOr(a.nf, 1);
}

// Level-0 slab m with the three slabs in separate buffers (a rolling window
// that never holds the whole lattice): cur <- f(p1, p2).
struct Slab0Args {
    Geom g;
    const double2 *A, *b;
    const double2 *p1, *p2;  // slabs m-1 and m-2 (p2 unused for m = 1)
    double2 *cur;
    const double *sq, *rsq;
    int m;
};

template <int D>
__global__ __launch_bounds__(256) void fwd_slab0_kernel(Slab0Args a) {
    const int m = a.m;
    const int64_t S = a.g.stride[0];
    const Span sp = xcd_span(xcd_block(blockIdx.x, gridDim.x), gridDim.x, S);
    const int64_t q0 = sp.q0, inc = sp.inc, hi = sp.hi;
    if (q0 >= hi) return;
    int k[D], ki[D];
    digits_of<D>(q0, a.g, 1, k);
    digits_of<D>(inc < S ? inc : 0, a.g, 1, ki);
    const double2 b0 = a.b[0];
    const double2 c00 = cscale_promoted(a.A[0], a.sq[m - 1]);
    const double sm = a.sq[m], rm = a.rsq[m];
    double2 A0j[D];
#pragma unroll
    for (int j = 0; j < D; ++j) A0j[j] = (j > 0) ? a.A[j] : make_double2(0.0, 0.0);
    for (int64_t q = q0; q < hi; q += inc) {
        // every load of the point first, zero-digit terms as in fwd_slab_kernel
        double2 nbv[D];
        double wv[D];
#pragma unroll
        for (int j = 1; j < D; ++j) {
            nbv[j] = a.p1[q - (k[j] > 0 ? a.g.stride[j] : 0)];
            wv[j] = a.sq[k[j]];
        }
        double2 v = cmul(b0, a.p1[q]);
        if (m >= 2) v = cadd(v, cmul(c00, a.p2[q]));
#pragma unroll
        for (int j = 1; j < D; ++j) v = cadd(v, cmul(cscale_promoted(A0j[j], wv[j]), nbv[j]));
        a.cur[q] = cdiv_by(v, sm, rm);
        if (q + inc < hi) digits_add<D>(k, ki, a.g, 1);
    }
}

// ------------------------------------------------------------- stable sweep
// core.py:183-211.  All pivots of a point lie on the previous index-sum
// wavefront, so the lattice is swept by |k| = n.  A "row" fixes k_0..k_{D-2};
// on wavefront n row r holds exactly one point, k_{D-1} = n - |row r|, when
// that is inside the box.  The row table stores each row's digits (uint16).
struct StableArgs {
    Geom g;
    const double2 *A, *b, *c;
    double2 *G;
    const uint16_t *rows;  // nrows x 8 digits
    int64_t nrows;         // rows of the last axis: N / shape[D - 1]
    const double *sq, *rsq;
    int n;                 // wavefront (per-wavefront launch)
    int64_t tstride_a, tstride_b, tstride_g;  // batch strides (complex elements)
    int *nf;               // per-wavefront launches: raised when a stored value is not finite
};

// Digits of every row, read by the per-wavefront and block kernels (a load
// from L2 is quicker than the row's divisions on their critical path).
__global__ void row_table_kernel(Geom g, uint16_t *rows, int64_t nrows) {
    const int64_t r = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (r >= nrows) return;
    const int D = g.D;
    const int64_t slast = g.shape[D - 1];
    int64_t x = r * slast;
    uint16_t *out = rows + r * 8;
    for (int j = 0; j < 8; ++j) {
        if (j < D - 1) {
            int64_t dj = x / g.stride[j];
            x -= dj * g.stride[j];
            out[j] = uint16_t(dj);
        } else {
            out[j] = 0;
        }
    }
}

// Returns true when the stored value is not finite.  BF (branch-free): the
// compiler can issue the loads of every pivot together; a term of the
// reference whose weight is sqrt(0) (k_j = 0, or the A_ii term at k_i = 1)
// is added as the reference adds it, the zero coefficient times a value
// already computed (the pivot's own), and a pivot axis with k_i = 0 is
// evaluated on the point's own address and left out of the sum and of the
// count.  Without BF (fewer registers: the 1024-thread kernels at larger D)
// zero-weight terms and pivots are skipped, which gives the same values for
// finite G.
template <int D, bool BF>
__device__ __forceinline__ bool stable_point(const StableArgs &a, const double2 *A, const double2 *b, double2 *G, const int (&k)[D],
                                             int64_t f) {
    int num = 0;
    double2 vals = make_double2(0.0, 0.0);
    if constexpr (!BF) {
#pragma unroll
        for (int i = 0; i < D; ++i) {
            if (k[i] == 0) continue;
            ++num;
            const int64_t pivot = f - a.g.stride[i];
            double2 val = cmul(b[i], G[pivot]);
#pragma unroll
            for (int j = 0; j < D; ++j) {
                if (j >= i) break;
                if (k[j] > 0) val = cadd(val, cmul(cscale_promoted(A[i * D + j], a.sq[k[j]]), G[pivot - a.g.stride[j]]));
            }
            if (k[i] >= 2) val = cadd(val, cmul(cscale_promoted(A[i * D + i], a.sq[k[i] - 1]), G[pivot - a.g.stride[i]]));
#pragma unroll
            for (int j = i + 1; j < D; ++j)
                if (k[j] > 0) val = cadd(val, cmul(cscale_promoted(A[i * D + j], a.sq[k[j]]), G[pivot - a.g.stride[j]]));
            vals = cadd(vals, cdiv_by(val, a.sq[k[i]], a.rsq[k[i]]));
        }
        const double2 out = cdiv_py(vals, make_double2(double(num), 0.0));
        G[f] = out;
        return !finite2(out);
    }
#pragma unroll
    for (int i = 0; i < D; ++i) {
        const int64_t pivot = f - (k[i] > 0 ? a.g.stride[i] : 0);
        double2 val = cmul(b[i], G[pivot]);
#pragma unroll
        for (int j = 0; j < D; ++j) {
            if (j >= i) break;
            val = cadd(val, cmul(cscale_promoted(A[i * D + j], a.sq[k[j]]), G[pivot - (k[j] > 0 ? a.g.stride[j] : 0)]));
        }
        val = cadd(val, cmul(cscale_promoted(A[i * D + i], a.sq[k[i] > 0 ? k[i] - 1 : 0]), G[pivot - (k[i] >= 2 ? a.g.stride[i] : 0)]));
#pragma unroll
        for (int j = i + 1; j < D; ++j)
            val = cadd(val, cmul(cscale_promoted(A[i * D + j], a.sq[k[j]]), G[pivot - (k[j] > 0 ? a.g.stride[j] : 0)]));
        const double2 term = cdiv_by(val, a.sq[k[i]], a.rsq[k[i]]);
        const bool on = k[i] > 0;
        vals = make_double2(on ? vals.x + term.x : vals.x, on ? vals.y + term.y : vals.y);
        num += on ? 1 : 0;
    }
    const double2 out = cdiv_py(vals, make_double2(double(num), 0.0));
    G[f] = out;
    return !finite2(out);
}

template <int D, bool BF>
__device__ __forceinline__ bool stable_row(const StableArgs &a, const double2 *A, const double2 *b, double2 *G, int64_t r, int n) {
    const uint16_t *rd = a.rows + r * 8;
    int k[D];
    int p = 0;
#pragma unroll
    for (int j = 0; j < D - 1; ++j) {
        k[j] = rd[j];
        p += k[j];
    }
    const int kl = n - p;
    if (kl < 0 || kl >= a.g.shape[D - 1]) return false;
    k[D - 1] = kl;
    return stable_point<D, BF>(a, A, b, G, k, r * a.g.shape[D - 1] + kl);
}

// One wavefront of one triple per launch (large lattices).
template <int D>
__global__ __launch_bounds__(256) void stable_wavefront_kernel(StableArgs a) {
    const int64_t r0 = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    bool bad = false;
    for (int64_t r = r0; r < a.nrows; r += int64_t(gridDim.x) * blockDim.x) bad |= stable_row<D, true>(a, a.A, a.b, a.G, r, a.n);
    if (__builtin_expect(bad, 0) && a.nf) atomicOr(a.nf, 1);
}

// Whole sweep of one triple per workgroup (small lattices, batches).
template <int D>
__global__ __launch_bounds__(1024) void stable_block_kernel(StableArgs a) {
    const int64_t t = blockIdx.x;
    const double2 *A = a.A + t * a.tstride_a;
    const double2 *b = a.b + t * a.tstride_b;
    double2 *G = a.G + t * a.tstride_g;
    if (threadIdx.x == 0) G[0] = a.c[t];
    __syncthreads();
    int nmax = 0;
    for (int j = 0; j < D; ++j) nmax += a.g.shape[j] - 1;
    bool bad = !finite2(a.c[t]);
    for (int n = 1; n <= nmax; ++n) {
        for (int64_t r = threadIdx.x; r < a.nrows; r += blockDim.x) bad |= stable_row<D, (D <= 6)>(a, A, b, G, r, n);
        __syncthreads();
    }
    // non-finite values: the reference's sequential sweep with every term
    if (__syncthreads_or(bad)) {
        __shared__ double2 red[16];
        Lat lat;
        lat.D = D;
        for (int j = 0; j < 8; ++j) {
            lat.shape[j] = a.g.shape[j];
            lat.stride[j] = a.g.stride[j];
        }
        lat.N = a.g.N;
        exact_stable_forward<D>(BlockOps(red), lat, A, b, a.c[t], G, a.sq);
    }
}

// G[0] = c of a per-wavefront sweep; the first one of a call also clears the
// call's non-finite flag.
__global__ void set_first_kernel(double2 *G, const double2 *c, int *nf) {
    G[0] = c[0];
    if (nf) *nf = 0;
}

// ------------------------------------------------ non-finite values (exact.hpp)
// Last launch of a multi-launch vanilla path: one workgroup per triple
// reruns the triple in the reference's arithmetic when the path met a
// non-finite value (the flag of a forward, or a non-finite dL/dc of a VJP,
// whose sum of G * dL/dG every non-finite G or dL/dG value poisons).
struct FixArgs {
    Lat g;
    const double2 *A, *b, *c, *gg;
    double2 *G, *dA, *db, *dc;
    const double *sq;
    int64_t ua, ub, uc, ug;  // per-triple strides (complex elements)
    const int *nf;           // forward: the path's flag, or NULL
    int fwd, vjp, stable;
    double gsign;            // -1: VJP of the conjugated cotangent, results conjugated
};

__global__ __launch_bounds__(1024) void exact_fixup_kernel(FixArgs a) {
    __shared__ double2 red[16];
    __shared__ int s_bad;
    const int64_t t = blockIdx.x;
    if (threadIdx.x == 0) {
        bool bad = a.nf && __hip_atomic_load(a.nf, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
        if (a.vjp) bad = bad || !finite2(a.dc[t * a.uc]);
        s_bad = bad;
    }
    __syncthreads();
    if (!s_bad) return;
    if (a.fwd && a.stable) {
        // one flag for all triples of the call: rerun those with a non-finite value
        // (1,024 of (7,)^4 with one such triple 40 -> 4.8 ms)
        bool bad = false;
        for (int64_t p = threadIdx.x; p < a.g.N; p += blockDim.x) bad = bad || !finite2(a.G[t * a.ug + p]);
        if (!__syncthreads_or(bad)) return;
    }
    const BlockOps ops(red);
    const double2 c = a.c[t * a.uc];
    if (a.fwd && a.stable) {
        switch (a.g.D) {
#define CASE(DD) \
    case DD: exact_stable_forward<DD>(ops, a.g, a.A + t * a.ua, a.b + t * a.ub, c, a.G + t * a.ug, a.sq); break;
            CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) CASE(8)
#undef CASE
        }
    } else if (a.fwd) exact_forward(ops, a.g, 0, a.A + t * a.ua, a.b + t * a.ub, c, a.G + t * a.ug, a.sq);
    if (a.vjp) exact_vjp(ops, a.g, a.G + t * a.ug, a.gg + t * a.ug, c, a.dA + t * a.ua, a.db + t * a.ub, a.dc + t * a.uc, a.sq, a.gsign);
}

__global__ void zero_ints_kernel(int *p, int n) {
    if (int(threadIdx.x) < n) p[threadIdx.x] = 0;
}

}  // namespace mm
