// k_mrhs.hip -- products of a matrix with a block of up to 16 right-hand sides
// (FP64 vectors, FP32 or FP64 matrix), on the FP64 matrix cores
// (v_mfma_f64_16x16x4: exact FP32-to-FP64 operands, FP64 sums).
//
// D = a b with a[m][k] = the right-hand sides (m) and b[k][n] = the matrix.
// Lane (q, k) = (lane % 16, lane / 16) of a wave supplies a[q][k], b[k][q] and
// receives in register e the element D[4e + k][q].
// Rows of the matrix are the outputs: a lane loads rows 4q .. 4q+3 of
// one column, 16 bytes, so 16 lanes read a 256-byte column segment, and
// its element i is the operand of the product whose n stands for row
// 4n + i: no transpose and no LDS.
// The right-hand sides are read as operands straight from L2.  Per 8 KB of an
// FP32 matrix a wave issues 32 products of 64 cycles, 9.8 TB/s over 1024 SIMDs:
// above what HBM delivers.  With 16 right-hand sides (A X, FP32 A) n = 8192
// takes 62 us (4.3 TB/s), where two passes of 8 over half the symmetric matrix
// with FP64 FMAs from LDS took 244.
#include "mpc_internal.hpp"
#include <algorithm>

namespace {

typedef double v4d __attribute__((ext_vector_type(4)));
typedef double d2 __attribute__((ext_vector_type(2), aligned(8)));
constexpr int MR = 64;          // output rows of a workgroup
constexpr int MU = 4;           // columns of a group per lane (8: two waves per SIMD
                                // instead of three, 5-15 % slower)
constexpr int MG = MPC_MM_GROUP_N;      // columns of a group
static_assert(MG == 4 * MU, "group");

// part[(s nj + j) m + r] = sum_{c in chunk s} A[r][c] X[j][c] for the 64 rows of
// blockIdx.x, chunk s = blockIdx.y of cw columns (a multiple of MG).  Wave w
// takes the chunk's column groups w, w + 4, ..; the four waves' sums are added
// in wave order through LDS.
template <typename T>
__global__ __launch_bounds__(256) void mm_n_kernel(const T* __restrict__ A, int64_t lda, int64_t m,
                                                  int64_t kc, int64_t cw, const double* __restrict__ X,
                                                  int64_t ldx, int nj, double* __restrict__ part) {
    typedef T vec4 __attribute__((ext_vector_type(4), aligned(sizeof(T))));
    __shared__ double red[4][MPC_MM_NJ][MR];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int q = lane & 15, k = lane >> 4;
    const int64_t r0 = (int64_t)blockIdx.x * MR, cs = (int64_t)blockIdx.y * cw;
    const int64_t ce = cs + cw < kc ? cs + cw : kc;
    const double* __restrict__ Xj = X + (int64_t)(q < nj ? q : nj - 1) * ldx;
    const int64_t r = r0 + 4 * q;
    const bool rfull = r0 + MR <= m;
    vec4 v[MU];
    double x[MU];
    auto load = [&](int64_t c0) {
        const int64_t c = c0 + MU * k;            // this lane's columns
        if (rfull && c0 + MG <= kc) {
#pragma unroll
            for (int s = 0; s < MU; ++s) v[s] = *reinterpret_cast<const vec4*>(A + r + (c + s) * lda);
#pragma unroll
            for (int s = 0; s < MU; s += 2) {
                const d2 y = *reinterpret_cast<const d2*>(Xj + c + s);
                x[s] = y[0];
                x[s + 1] = y[1];
            }
        } else {                                 // clamped addresses, zeros outside
#pragma unroll
            for (int s = 0; s < MU; ++s) {
                const int64_t cc = c + s < kc ? c + s : kc - 1;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const T y = A[(r + i < m ? r + i : m - 1) + cc * lda];
                    v[s][i] = (r + i < m && c + s < kc) ? y : T(0);
                }
                const double y = Xj[cc];
                x[s] = c + s < kc ? y : 0.0;
            }
        }
    };
    v4d acc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = v4d{};
    int64_t c0 = cs + MG * wave;
    if (c0 < ce) load(c0);
    for (; c0 < ce; c0 += 4 * MG) {
        vec4 w[MU];
        double y[MU];
#pragma unroll
        for (int s = 0; s < MU; ++s) {
            w[s] = v[s];
            y[s] = x[s];
        }
        if (c0 + 4 * MG < ce) load(c0 + 4 * MG);     // in flight during the products
#pragma unroll
        for (int s = 0; s < MU; ++s)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                acc[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(y[s], (double)w[s][i], acc[i], 0, 0, 0);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < 4; ++i) red[wave][4 * e + k][4 * q + i] = acc[i][e];
    __syncthreads();
    if (r0 + lane < m) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int j = wave + 4 * u;
            if (j < nj)
                part[((int64_t)blockIdx.y * nj + j) * m + r0 + lane] =
                    ((red[0][j][lane] + red[1][j][lane]) + red[2][j][lane]) + red[3][j][lane];
        }
    }
}

// Y[j][r] = (B ? B[j][r] : 0) + a sum_s part[(s nj + j) m + r], chunks in order;
// thread = row, 8 loads in flight (clamped chunk, zero weight past the end)
__global__ __launch_bounds__(256) void mm_sum_kernel(int64_t m, int S,
                                                    const double* __restrict__ part,
                                                    const double* __restrict__ B, int64_t ldb,
                                                    double a, double* __restrict__ Y, int64_t ldy) {
    const int64_t r0 = (int64_t)blockIdx.x * 256 + threadIdx.x, r = r0 < m ? r0 : m - 1;
    const int j = blockIdx.y, nj = gridDim.y;
    double sum = 0.0;
    for (int s = 0; s < S; s += 8) {
        double v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u)
            v[u] = part[((int64_t)(s + u < S ? s + u : S - 1) * nj + j) * m + r];
#pragma unroll
        for (int u = 0; u < 8; ++u) sum += s + u < S ? v[u] : 0.0;
    }
    if (r0 < m) Y[j * ldy + r] = B ? fma(a, sum, B[j * ldb + r]) : a * sum;
}

inline int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }
// columns of a chunk when kc columns are split S ways (whole groups)
inline int64_t chunk(int64_t kc, int64_t S) { return cdiv(cdiv(kc, S), MG) * MG; }

template <typename T>
int launch_mm_n(hipStream_t st, const T* A, int64_t lda, int64_t m, int64_t kc,
                const double* X, int64_t ldx, int nj, double* part, int64_t S) {
    if (nj < 1 || nj > MPC_MM_NJ || S < 1) {
        mpc_set_error("mm_n: %d right-hand sides, %lld chunks", nj, (long long)S);
        return MPC_ERR_ARG;
    }
    const int64_t cw = chunk(kc, S);
    const dim3 g((unsigned)cdiv(m, MR), (unsigned)cdiv(kc, cw)), b(256);
    hipLaunchKernelGGL(mm_n_kernel<T>, g, b, 0, st, A, lda, m, kc, cw, X, ldx, nj, part);
    MPC_LAUNCH_CHECK();
    return 0;
}

}  // namespace

// Enough chunks for about 2048 workgroups, each wave of which has a column
// group.  768 run at once, so fewer leave a last wave nearly empty (16
// columns: n = 6000 67 us with 1024 workgroups, 53 with 2048, 54 with 4096;
// n = 8192 60, 62, 68), and every chunk costs a partial sum per output.
int64_t mpc_mm_splits(int64_t rows, int64_t kc) {
    const int64_t want = cdiv(2048, cdiv(rows, MR)), most = cdiv(kc, 4 * MG);
    return std::max<int64_t>(1, std::min(want, most));
}

int mpc_launch_mm_n(hipStream_t st, const float* A, int64_t lda, int64_t m, int64_t kc,
                    const double* X, int64_t ldx, int nj, double* part, int64_t S) {
    return launch_mm_n<float>(st, A, lda, m, kc, X, ldx, nj, part, S);
}
int mpc_launch_mm_n(hipStream_t st, const double* A, int64_t lda, int64_t m, int64_t kc,
                    const double* X, int64_t ldx, int nj, double* part, int64_t S) {
    return launch_mm_n<double>(st, A, lda, m, kc, X, ldx, nj, part, S);
}

int mpc_launch_mm_sum(hipStream_t st, int64_t m, int nj, int64_t kc, int64_t S,
                      const double* part, const double* B, int64_t ldb, double a, double* Y, int64_t ldy) {
    hipLaunchKernelGGL(mm_sum_kernel, dim3((unsigned)cdiv(m, 256), (unsigned)nj), dim3(256), 0, st, m,
                       (int)cdiv(kc, chunk(kc, S)), part, B, ldb, a, Y, ldy);
    MPC_LAUNCH_CHECK();
    return 0;
}
