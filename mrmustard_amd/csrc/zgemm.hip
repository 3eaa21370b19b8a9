// libmmhip: C ABI of the FP64 matrix-core complex product (zgemm_mfma_kernel).

#include "host.hpp"
#include "zgemm.hpp"

using namespace mm;

namespace {

// Tile rows of zgemm_strip_kernel (16 RT rows each), or 0 for the 64 x 128
// tiles of zgemm_mfma_kernel, which win by 2 to 5 % only where they fill
// whole rounds of the chip (two workgroups per CU) with little padding:
// 2048^3 1066 against 1121 us, but 1600^3 (325 tiles for 512 places) 829
// against 640 us.  RT: all rows in one tile row (B read once) when the strips
// alone keep every SIMD busy (100 x 10^6 x 100: 1584 us, 2024 with two tile
// rows), else at most 4 for more workgroups (81 x 6561 x 81: 15.3 against 23.9 us).
int strip_rt(int64_t M, int64_t N, int64_t batch, int num_cu) {
    const int64_t big = ((M + 63) / 64) * ((N + ZG_BN - 1) / ZG_BN) * batch;
    const int64_t rounds = (big + 2 * num_cu - 1) / (2 * num_cu);
    if (M >= 512 && N >= 512 && double(M) * double(N) * double(batch) >= 0.9 * double(rounds) * 2.0 * num_cu * 64 * ZG_BN) return 0;
    const int64_t mt = (M + 15) / 16;
    if (mt <= 8 && (N * batch + 63) / 64 >= 4 * int64_t(num_cu)) return int(mt);
    const int64_t gy = (mt + 3) / 4;
    return int((mt + gy - 1) / gy);
}

// HIP takes launches of fewer than 2^32 threads along x: 2^24 - 1 workgroups of 256.
constexpr int64_t MAX_GX = (int64_t(1) << 24) - 1;

// How a batch of products is cut into launches: `step` products of `cols`
// columns each; merged: the columns of all of them as one product (cols = N).
struct ZgemmPlan {
    int rt = 0;
    int64_t step = 0, cols = 0;
    bool merged = false;
};

// false when one product has more columns or rows than a launch of
// zgemm_mfma_kernel takes.
bool zgemm_plan(int64_t M, int64_t N, int64_t batch, bool shared_a, int num_cu, ZgemmPlan *p) {
    if (N > MAX_GX * ZG_BN || (M + 63) / 64 > 65535) return false;
    p->rt = strip_rt(M, N, batch, num_cu);
    p->step = std::min<int64_t>(batch, 65535);  // grid z
    p->cols = N;
    if (p->rt) {
        const int64_t most = MAX_GX * 64;  // columns of a launch of zgemm_strip_kernel
        p->merged = shared_a && batch > 1 && N <= most / 2;
        if (p->merged) p->step = std::min<int64_t>(batch, most / N);
        else p->cols = std::min<int64_t>(N, most);
    }
    return true;
}

// nz products of N columns each, or (cols > N) one with the columns of all.
template <int RT>
void launch_strip(const ZgemmArgs &a, int64_t nz, int64_t cols, hipStream_t s) {
    const dim3 grid(unsigned((cols + 63) / 64), unsigned((a.M + 16 * RT - 1) / (16 * RT)), unsigned(nz));
    if constexpr (RT <= 4) {
        // the whole of K in one chunk: no second round trip to memory
        if (a.K <= 16) {
            hipLaunchKernelGGL((zgemm_strip_kernel<RT, 16>), grid, dim3(256), 0, s, a, cols);
            return;
        }
    }
    hipLaunchKernelGGL((zgemm_strip_kernel<RT, ZG_BK>), grid, dim3(256), 0, s, a, cols);
}

}  // namespace

extern "C" {

int mm_zgemm_batched(const double *A, int64_t lda, int64_t sA, const double *B, int64_t ldb, int64_t sB, double *C, int64_t ldc,
                     int64_t sC, int64_t M, int64_t N, int64_t K, int64_t batch, void *stream) {
    if (M < 0 || N < 0 || K < 0 || batch < 0) return fail(MM_ERR_INVALID, "negative matrix size or batch");
    if (M == 0 || N == 0 || batch == 0) return MM_OK;
    if (!A || !B || !C) return fail(MM_ERR_INVALID, "NULL matrix pointer");
    if (lda < K || ldb < N || ldc < N) return fail(MM_ERR_INVALID, "leading dimension smaller than the row length");
    if (sA < 0 || sB < 0 || sC < 0) return fail(MM_ERR_INVALID, "negative batch stride");
    if (batch > 1 && sC < (M - 1) * ldc + N) return fail(MM_ERR_INVALID, "the products of a batch overlap in C");
    int num_cu = 1;
    const int rc = compute_units(&num_cu);
    if (rc) return rc;
    ZgemmPlan p;
    // products that share A are merged into one with all their columns
    if (!zgemm_plan(M, N, batch, sA == 0, num_cu, &p)) return fail(MM_ERR_UNSUPPORTED, "matrix too large for one launch");
    ZgemmArgs a;
    a.M = M;
    a.K = K;
    a.lda = lda;
    a.ldb = ldb;
    a.ldc = ldc;
    a.sA = sA;
    a.sB = sB;
    a.sC = sC;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    for (int64_t b0 = 0; b0 < batch; b0 += p.step)
        for (int64_t n0 = 0; n0 < N; n0 += p.cols) {
            const int64_t nz = std::min<int64_t>(p.step, batch - b0);
            a.N = std::min<int64_t>(p.cols, N - n0);
            a.A = reinterpret_cast<const double2 *>(A) + b0 * sA;
            a.B = reinterpret_cast<const double2 *>(B) + b0 * sB + n0;
            a.C = reinterpret_cast<double2 *>(C) + b0 * sC + n0;
            switch (p.rt) {
                case 0: {
                    const dim3 grid(unsigned((N + ZG_BN - 1) / ZG_BN), unsigned((M + 63) / 64), unsigned(nz));
                    hipLaunchKernelGGL(zgemm_mfma_kernel, grid, dim3(256), 0, s, a);
                    LAUNCH_CHECK("zgemm_mfma_kernel");
                    break;
                }
#define CASE(RT)                                                                    \
    case RT:                                                                        \
        launch_strip<RT>(a, p.merged ? 1 : nz, p.merged ? N * nz : a.N, s);         \
        LAUNCH_CHECK("zgemm_strip_kernel");                                         \
        break;
                    CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) CASE(8)
#undef CASE
            }
        }
    return MM_OK;
}

int mm_zgemm(const double *A, int64_t lda, const double *B, int64_t ldb, double *C, int64_t ldc, int64_t M, int64_t N, int64_t K,
             void *stream) {
    return mm_zgemm_batched(A, lda, 0, B, ldb, 0, C, ldc, 0, M, N, K, 1, stream);
}

int mm_zgemm_plan(int64_t M, int64_t N, int64_t batch, int shared_a, int num_cu, int64_t *out) {
    if (!out) return fail(MM_ERR_INVALID, "NULL pointer");
    if (M < 1 || N < 1 || batch < 1 || num_cu < 1) return fail(MM_ERR_INVALID, "sizes must be positive");
    ZgemmPlan p;
    if (!zgemm_plan(M, N, batch, shared_a != 0, num_cu, &p)) return fail(MM_ERR_UNSUPPORTED, "matrix too large for one launch");
    out[0] = p.rt;
    out[1] = p.step;
    out[2] = p.cols;
    out[3] = p.merged;
    return MM_OK;
}

}  // extern "C"
