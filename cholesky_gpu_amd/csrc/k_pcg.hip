// k_pcg.hip -- bandwidth-bound kernels of the PCG loop.
//
// Replaces, from precond_CG (mixed_cholesky.cu:145-217): cublasDgemv (A p),
// cusolverDnDpotrs (z = L^-T L^-1 r, on an FP64 copy of L made by
// convertFloattoDouble), and the cublasDdot/Daxpy/Dscal/Dcopy calls that
// return scalars to the host.  Here A and L stay FP32 in HBM (A may also be an
// FP64 operator, for solves that must match FP64 exactly) and are read once
// per product; vectors, accumulation, inner products and the alpha/beta
// scalars are FP64 and never leave the device.  Every reduction has a fixed
// order (two-stage, partials then an ordered sum), so results are bitwise
// reproducible run to run.
#include "mpc_internal.hpp"
#include <algorithm>

namespace {

constexpr int RB = 256;          // rows per workgroup

// ---------------------------------------------------------------- SYMV
// y = A x for symmetric A reading only the upper triangle (i <= j) of the
// column-major FP32 (or FP64) matrix: half the HBM traffic of a full GEMV.
// One workgroup per E x E super-tile (I <= J, E = 64 S) of S x S tiles of
// 64, walked tile by tile through LDS (the next tile's loads are in flight
// while the current one is summed).  Waves 0-1 form row sums (A_IJ x_J: lane
// = row, wave = half of the tile's columns), waves 2-3 column sums
// (A_IJ^T x_I: lane = column, wave = half of the rows), accumulated in
// registers over the super-tile, so each super-tile writes one partial per
// row of I and one per row of J:
//   P[K][L][j][r]:  L >= K row-sum partial of super-tile (K, L); L < K
//                   column-sum partial of super-tile (L, K)
// (a diagonal super-tile writes its row and column sums as one partial), and
// symv_reduce adds P[K][0..nst) in order (deterministic).  The partials take
// nst^2 E NJ doubles, NJ <= 4 right-hand sides per pass (at n = 16384, S = 4,
// one right-hand side: 1/64 of the bytes read from A).  More than four
// right-hand sides go through the matrix cores in passes of 16 that read every
// element of the triangle twice (k_mrhs.hip): the FMAs here read x from LDS per
// element and right-hand side and so cost more than the bytes (n = 8192: 48 us
// for 4, where 16 take 62 there; n = 6000: 34 and 42).
constexpr int SY_T = 64;
constexpr int SY_JMAX = 4;
// 16-byte loads of columns that are aligned to their elements only (an odd
// leading dimension): global loads need no more than 4-byte alignment
template <typename T> struct vec16 { typedef float type __attribute__((ext_vector_type(4), aligned(4))); };
template <> struct vec16<double> { typedef double type __attribute__((ext_vector_type(2), aligned(8))); };

template <typename T, int NJ, int S>
__global__ __launch_bounds__(256) void symv_super_kernel(const T* __restrict__ A, int64_t lda,
                                                        int64_t n, int nst, int j0, int nj,
                                                        const double* __restrict__ X, int64_t ldx,
                                                        double* __restrict__ P) {
    constexpr int ST = SY_T, E = SY_T * S;
    using V16 = typename vec16<T>::type;
    constexpr int VE = 16 / (int)sizeof(T);        // elements per 16-byte load
    constexpr int RV = ST / VE;                     // loads per tile column
    constexpr int CPP = 256 / RV;                   // columns per pass
    constexpr int NP = ST / CPP;                    // passes
    static_assert(S * NJ * 64 <= ST * (ST + 1) * (int)sizeof(T) / 8, "column buffer fits As");
    __shared__ T As[ST * (ST + 1)];
    __shared__ double xr[NJ][E], xc[NJ][E];
    __shared__ double hb[NJ][64];
    // super-tile index -> (I, J), I <= J, row-major over the upper triangle
    const int64_t t = blockIdx.x;
    int64_t I = (int64_t)((2.0 * nst + 1.0 - sqrt((2.0 * nst + 1.0) * (2.0 * nst + 1.0) - 8.0 * t)) * 0.5);
    auto start = [&](int64_t i) { return i * nst - i * (i - 1) / 2; };
    while (I > 0 && start(I) > t) --I;
    while (start(I + 1) <= t) ++I;
    const int64_t J = I + (t - start(I));
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t R0 = I * E, C0 = J * E;
    const bool diag = I == J;
    const int na = (int)((n - R0 + ST - 1) / ST < S ? (n - R0 + ST - 1) / ST : S);
    const int nbb = (int)((n - C0 + ST - 1) / ST < S ? (n - C0 + ST - 1) / ST : S);
    // x of the rows (xr) and of the columns (xc); a diagonal super-tile reads
    // both from xr and keeps its row partials in xc
    for (int idx = tid; idx < NJ * E; idx += 256) {
        const int j = idx / E, k = idx % E;
        const int jj = j < nj ? j : nj - 1;
        const double vr = X[(int64_t)(j0 + jj) * ldx + (R0 + k < n ? R0 + k : n - 1)];
        xr[j][k] = (j < nj && R0 + k < n) ? vr : 0.0;
        const double vc = X[(int64_t)(j0 + jj) * ldx + (C0 + k < n ? C0 + k : n - 1)];
        xc[j][k] = (!diag && j < nj && C0 + k < n) ? vc : 0.0;
    }
    const double* xcol = diag ? &xr[0][0] : &xc[0][0];
    const int q = tid % RV, cq = tid / RV;
    V16 v[NP];
    auto load_tile = [&](int a, int b) {
        const int64_t r0 = R0 + a * ST, c0 = C0 + b * ST;
        if (r0 + ST <= n && c0 + ST <= n) {
#pragma unroll
            for (int p = 0; p < NP; ++p)
                v[p] = *reinterpret_cast<const V16*>(A + r0 + VE * q + (c0 + p * CPP + cq) * lda);
        } else {
#pragma unroll
            for (int p = 0; p < NP; ++p) {
                T* e = reinterpret_cast<T*>(&v[p]);
                const int64_t gc = c0 + p * CPP + cq;
#pragma unroll
                for (int u = 0; u < VE; ++u) {
                    const int64_t gr = r0 + VE * q + u;
                    const T x = A[(gr < n ? gr : n - 1) + (gc < n ? gc : n - 1) * lda];
                    e[u] = (gr < n && gc < n) ? x : T(0);
                }
            }
        }
    };
    auto store_tile = [&](bool dtile) {
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            const int c = p * CPP + cq;
            const T* e = reinterpret_cast<const T*>(&v[p]);
#pragma unroll
            for (int u = 0; u < VE; ++u) {
                const int r = VE * q + u;
                As[c * (ST + 1) + r] = (!dtile || r <= c) ? e[u] : T(0);
            }
        }
    };
    const bool rowrole = wave < 2;
    const int half = wave & 1;
    double cacc[S][NJ];
#pragma unroll
    for (int b = 0; b < S; ++b)
#pragma unroll
        for (int j = 0; j < NJ; ++j) cacc[b][j] = 0.0;
    if (na > 0) load_tile(0, 0);
    for (int a = 0; a < na; ++a) {
        const int b0 = diag ? a : 0;
        double racc[NJ];
#pragma unroll
        for (int j = 0; j < NJ; ++j) racc[j] = 0.0;
#pragma unroll
        for (int b = 0; b < S; ++b) {
            if (b < b0 || b >= nbb) continue;
            const bool dtile = diag && a == b;
            __syncthreads();                          // the previous tile is summed
            store_tile(dtile);
            {                                         // the next tile's loads
                int an = a, bn = b + 1;
                if (bn >= nbb) { an = a + 1; bn = diag ? an : 0; }
                if (an < na) load_tile(an, bn);
            }
            __syncthreads();
            if (rowrole) {
                const int r = lane;
                double s[NJ];
#pragma unroll
                for (int j = 0; j < NJ; ++j) s[j] = 0.0;
#pragma unroll 8
                for (int cc = 0; cc < 32; ++cc) {
                    const int c = half * 32 + cc;
                    const double av = (double)As[c * (ST + 1) + r];
#pragma unroll
                    for (int j = 0; j < NJ; ++j) s[j] = fma(av, xcol[j * E + b * ST + c], s[j]);
                }
#pragma unroll
                for (int j = 0; j < NJ; ++j) racc[j] += s[j];
            } else {
                const int c = lane;
                double s[NJ];
#pragma unroll
                for (int j = 0; j < NJ; ++j) s[j] = 0.0;
                if (dtile) {                          // strict lower mirror only
#pragma unroll 8
                    for (int rr = 0; rr < 32; ++rr) {
                        const int r = half * 32 + rr;
                        const double av = r < c ? (double)As[c * (ST + 1) + r] : 0.0;
#pragma unroll
                        for (int j = 0; j < NJ; ++j) s[j] = fma(av, xr[j][a * ST + r], s[j]);
                    }
                } else {
#pragma unroll 8
                    for (int rr = 0; rr < 32; ++rr) {
                        const int r = half * 32 + rr;
                        const double av = (double)As[c * (ST + 1) + r];
#pragma unroll
                        for (int j = 0; j < NJ; ++j) s[j] = fma(av, xr[j][a * ST + r], s[j]);
                    }
                }
#pragma unroll
                for (int j = 0; j < NJ; ++j) cacc[b][j] += s[j];
            }
        }
        // row partials of tile-row a: the two column halves added in order
        if (rowrole && half == 1) {
#pragma unroll
            for (int j = 0; j < NJ; ++j) hb[j][lane] = racc[j];
        }
        __syncthreads();
        if (rowrole && half == 0) {
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const double tot = racc[j] + hb[j][lane];
                if (diag) xc[j][a * ST + lane] = tot;
                else if (j < nj) P[((I * nst + J) * NJ + j) * E + a * ST + lane] = tot;
            }
        }
    }
    // column partials: the two row halves added in order (through As), plus
    // the row partials of a diagonal super-tile
    __syncthreads();
    double* cb = reinterpret_cast<double*>(As);
    if (!rowrole && half == 1) {
#pragma unroll
        for (int b = 0; b < S; ++b)
#pragma unroll
            for (int j = 0; j < NJ; ++j) cb[(b * NJ + j) * 64 + lane] = cacc[b][j];
    }
    __syncthreads();
    if (!rowrole && half == 0) {
#pragma unroll
        for (int b = 0; b < S; ++b) {
            if (b >= nbb) continue;
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                if (j >= nj) continue;
                double tot = cacc[b][j] + cb[(b * NJ + j) * 64 + lane];
                if (diag) tot = xc[j][b * ST + lane] + tot;
                P[((J * nst + I) * NJ + j) * E + b * ST + lane] = tot;
            }
        }
    }
}

// 64 rows per workgroup (lane = row).  Wave w sums the partials of
// super-tiles [w q, (w+1) q), q = ceil(nst / 4), in batches of 16
// independent loads (clamped index, zero weight past the end) in order; the
// four quarter sums are then added in order.
__global__ __launch_bounds__(256) void symv_reduce_kernel(int64_t n, int E, int nst, int NJ, int j0,
                                                         const double* __restrict__ P,
                                                         double* __restrict__ Y, int64_t ldy) {
    __shared__ double red[4][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int64_t row0 = (int64_t)blockIdx.x * 64 + lane;
    const int64_t row = row0 < n ? row0 : n - 1;
    const int j = blockIdx.y;
    const int64_t K = row / E, r = row % E;
    const int q = (nst + 3) / 4, l0 = w * q, l1 = l0 + q < nst ? l0 + q : nst;
    double s = 0.0;
    for (int L0 = l0; L0 < l1; L0 += 16) {
        double v[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const int64_t L = L0 + u < l1 ? L0 + u : l1 - 1;
            v[u] = P[((K * nst + L) * NJ + j) * E + r];
        }
#pragma unroll
        for (int u = 0; u < 16; ++u) s += L0 + u < l1 ? v[u] : 0.0;
    }
    red[w][lane] = s;
    __syncthreads();
    if (w == 0 && row0 < n)
        Y[(int64_t)(j0 + j) * ldy + row0] = ((red[0][lane] + red[1][lane]) + red[2][lane]) + red[3][lane];
}

// ---------------------------------------------------------------- dots and updates
// Sum of a workgroup's NW waves, in thread 0
template <int NW>
__device__ __forceinline__ double wg_sum(double v) {
    __shared__ double red[NW];
    v = mpc_sum64(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double s = 0.0;
    if (threadIdx.x == 0) {
#pragma unroll
        for (int w = 0; w < NW; ++w) s += red[w];
    }
    return s;
}

// sum of a[r] b[r] over r = r0 + thread, + nthr, ..: E of them, clamped loads all
// in flight (rows from n on weigh nothing)
template <int E>
__device__ __forceinline__ double dot_rows(int64_t r0, int nthr, int64_t n, const double* __restrict__ a,
                                           const double* __restrict__ b) {
    double x[E], y[E], s = 0.0;
#pragma unroll
    for (int q = 0; q < E; ++q) {
        const int64_t r = r0 + (int64_t)q * nthr + threadIdx.x, rc = r < n ? r : n - 1;
        x[q] = a[rc];
        y[q] = b[rc];
    }
#pragma unroll
    for (int q = 0; q < E; ++q) s = r0 + (int64_t)q * nthr + threadIdx.x < n ? fma(x[q], y[q], s) : s;
    return s;
}

// Dots of column j = blockIdx.x of a and b (blockIdx.y = 1: b2), a workgroup for
// each.  Up to kDotOne rows the second launch for a split sum takes longer than
// the split saves (n = 500 / 2048 / 8192 / 16384: 3.9 / 3.9 / 4.6 / 6.9 us, split
// 5.2 / 6.0 / 8.1 / 10.0).
constexpr int64_t kDotOne = 16384;
__global__ __launch_bounds__(1024) void dot_kernel(int64_t n, const double* __restrict__ a, int64_t lda_,
                                                  const double* __restrict__ b0, int64_t ldb0,
                                                  const double* __restrict__ b2, int64_t ldb2,
                                                  double* __restrict__ out0, double* __restrict__ out2) {
    const int j = blockIdx.x;
    const double* __restrict__ b = blockIdx.y ? b2 + j * ldb2 : b0 + j * ldb0;
    double s = 0.0;
    for (int64_t r0 = 0; r0 < n; r0 += 8 * 1024) s += dot_rows<8>(r0, 1024, n, a + j * lda_, b);
    s = wg_sum<16>(s);
    if (threadIdx.x == 0) (blockIdx.y ? out2 : out0)[j] = s;
}

// blockIdx.z selects the second operand: 0 -> b, 1 -> b2 (two dots with the
// same first operand in one launch); partials of z at part + z nrhs nparts
__global__ __launch_bounds__(RB) void dot_partial_kernel(int64_t n, const double* __restrict__ a,
                                                        int64_t lda_, const double* __restrict__ b0,
                                                        int64_t ldb0, const double* __restrict__ b2,
                                                        int64_t ldb2, double* __restrict__ part) {
    const int j = blockIdx.y;
    const double* __restrict__ b = blockIdx.z ? b2 + j * ldb2 : b0 + j * ldb0;
    const double s = wg_sum<RB / 64>(dot_rows<8>((int64_t)blockIdx.x * RB * 8, RB, n, a + j * lda_, b));
    if (threadIdx.x == 0)
        part[((int64_t)blockIdx.z * gridDim.y + j) * gridDim.x + blockIdx.x] = s;
}

// blockIdx.y selects the dot: 0 -> out, 1 -> out2
__global__ __launch_bounds__(RB) void dot_final_kernel(int nparts, const double* __restrict__ part,
                                                      double* __restrict__ out0,
                                                      double* __restrict__ out2) {
    const int j = blockIdx.x;
    part += ((int64_t)blockIdx.y * gridDim.x + j) * nparts;
    double s = 0.0;
    for (int q = threadIdx.x; q < nparts; q += RB) s += part[q];
    s = wg_sum<RB / 64>(s);
    if (threadIdx.x == 0) (blockIdx.y ? out2 : out0)[j] = s;
}

__global__ __launch_bounds__(RB) void update_xr_kernel(int64_t n, double* __restrict__ X,
                                                      int64_t ldx, double* __restrict__ R,
                                                      int64_t ldr, const double* __restrict__ P,
                                                      int64_t ldp, const double* __restrict__ Q,
                                                      int64_t ldq, const double* __restrict__ rz,
                                                      const double* __restrict__ pq,
                                                      const int* __restrict__ active) {
    const int j = blockIdx.y;
    if (active && !active[j]) return;
    const int64_t r = (int64_t)blockIdx.x * RB + threadIdx.x;
    if (r >= n) return;
    const double alpha = rz[j] / pq[j];
    X[j * ldx + r] = fma(alpha, P[j * ldp + r], X[j * ldx + r]);
    R[j * ldr + r] = fma(-alpha, Q[j * ldq + r], R[j * ldr + r]);
}

__global__ __launch_bounds__(RB) void update_p_kernel(int64_t n, double* __restrict__ P, int64_t ldp,
                                                     const double* __restrict__ Z, int64_t ldz,
                                                     const double* __restrict__ rz_new,
                                                     const double* __restrict__ rz_old,
                                                     const int* __restrict__ active) {
    const int j = blockIdx.y;
    if (active && !active[j]) return;
    const int64_t r = (int64_t)blockIdx.x * RB + threadIdx.x;
    if (r >= n) return;
    const double beta = rz_new[j] / rz_old[j];
    P[j * ldp + r] = fma(beta, P[j * ldp + r], Z[j * ldz + r]);
}

// End of one PCG iteration, per right-hand side j that is still active:
// record column 0's CG coefficients (Lanczos estimate), rz <- rz_new, count
// the iteration, and test convergence (stop_rule 0: sqrt(rr)/||b||, the
// recursive residual, confirmed later on the true residual; 1: the reference
// rule sqrt(|r.z|)/||b||).  A column that meets tol becomes a candidate and is
// frozen (active = 0) so later iterations leave it untouched.
__global__ __launch_bounds__(256) void pcg_status_kernel(int nrhs, double* __restrict__ rz,
                                                        const double* __restrict__ rz_new,
                                                        const double* __restrict__ pq,
                                                        const double* __restrict__ rr,
                                                        const double* __restrict__ bb, double tol,
                                                        int stop_rule, int* __restrict__ active,
                                                        int* __restrict__ cand,
                                                        int* __restrict__ iters,
                                                        double* __restrict__ relres,
                                                        double* __restrict__ ahist,
                                                        double* __restrict__ bhist, int hmax) {
    const int j = blockIdx.x * 256 + threadIdx.x;
    if (j >= nrhs || !active[j]) return;
    const int k = iters[j];
    if (j == 0 && k < hmax) {
        ahist[k] = rz[0] / pq[0];
        bhist[k] = rz_new[0] / rz[0];
    }
    rz[j] = rz_new[j];
    iters[j] = k + 1;
    double nb = sqrt(bb[j]);
    if (nb == 0.0) nb = 1.0;
    const double res = stop_rule == 1 ? sqrt(fabs(rz_new[j])) / nb : sqrt(rr[j]) / nb;
    relres[j] = res;
    if (res <= tol) {
        cand[j] = 1;
        active[j] = 0;
    }
}

__global__ __launch_bounds__(RB) void axpby_kernel(int64_t n, double a, const double* __restrict__ X,
                                                  int64_t ldx, double b, double* __restrict__ Y,
                                                  int64_t ldy) {
    const int j = blockIdx.y;
    const int64_t r = (int64_t)blockIdx.x * RB + threadIdx.x;
    if (r >= n) return;
    Y[j * ldy + r] = (a == 0.0 && b == 0.0) ? 0.0 : a * X[j * ldx + r] + b * Y[j * ldy + r];
}

__global__ __launch_bounds__(RB) void copy2d_kernel(int64_t n, const double* __restrict__ X,
                                                   int64_t ldx, double* __restrict__ Y, int64_t ldy) {
    const int j = blockIdx.y;
    const int64_t r = (int64_t)blockIdx.x * RB + threadIdx.x;
    if (r < n) Y[j * ldy + r] = X[j * ldx + r];
}

// The lower triangle of a matrix (and what shares a 16-byte piece or a group of
// 8 columns with it): a factor reads and writes nothing else.  Four rows and
// eight columns per thread, all loads in flight; n = 8192 139 us as a copy of the
// whole matrix, 4 bytes at a time.
constexpr int CPC = 8;
typedef float v4cp __attribute__((ext_vector_type(4), aligned(4)));
__global__ __launch_bounds__(RB) void copy_lower_kernel(int64_t rows, int64_t cols,
                                                       const float* __restrict__ A, int64_t lda,
                                                       float* __restrict__ B, int64_t ldb) {
    const int64_t r = 4 * ((int64_t)blockIdx.x * RB + threadIdx.x), c0 = (int64_t)blockIdx.y * CPC;
    if (r >= rows || r + 3 < c0) return;
    if (r + 4 <= rows) {
        v4cp v[CPC];
#pragma unroll
        for (int u = 0; u < CPC; ++u) {
            const int64_t c = c0 + u < cols ? c0 + u : cols - 1;
            v[u] = *reinterpret_cast<const v4cp*>(A + r + c * lda);
        }
#pragma unroll
        for (int u = 0; u < CPC; ++u)
            if (c0 + u < cols) *reinterpret_cast<v4cp*>(B + r + (c0 + u) * ldb) = v[u];
    } else {
        for (int64_t c = c0; c < c0 + CPC && c < cols; ++c)
            for (int64_t q = r; q < rows; ++q) B[q + c * ldb] = A[q + c * lda];
    }
}

// ---------------------------------------------------------------- block PCG
// s x s products and updates of the block recurrence (s <= MPC_BLOCK_PCG_MAX
// right-hand sides, n x s blocks column-major).
constexpr int BS = MPC_BLOCK_PCG_MAX;   // largest block
constexpr int GROWS = 256;        // rows of a gram workgroup at a time, 64 per wave
constexpr int GWG = 32;           // most gram workgroups (the last one adds their sums)
typedef double v4d __attribute__((ext_vector_type(4)));
typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));

int64_t gram_rows(int64_t n) {    // rows of a workgroup
    const int64_t per = (n + GWG * GROWS - 1) / (GWG * GROWS);
    return per * GROWS;
}

// G = X^T Y on the FP64 matrix cores (v_mfma_f64_16x16x4): lane (q, k) of a wave
// holds 16 rows 16k .. 16k+15 of column q of both blocks (whole lines), product
// t multiplies the rows 16k + t, and register e of the lane is G[4e + k][q].
// Workgroup c takes rows [c chunk, (c+1) chunk), its waves' sums are added in
// wave order and the last workgroup to finish adds the workgroups' in order.
// (One thread per entry of G over 2048 rows took 74 us at n = 6000.)
__global__ __launch_bounds__(256, 2) void gram_kernel(int64_t n, int s, int64_t chunk,
                                                     const double* __restrict__ X, int64_t ldx,
                                                     const double* __restrict__ Y, int64_t ldy,
                                                     double* __restrict__ part,
                                                     double* __restrict__ G, int* __restrict__ tick) {
    __shared__ double red[4][BS * BS];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int q = lane & 15, k = lane >> 4, qc = q < s ? q : s - 1;
    const int s2 = s * s;
    const int64_t r0 = (int64_t)blockIdx.x * chunk, r1 = r0 + chunk < n ? r0 + chunk : n;
    const double* Xq = X + qc * ldx;
    const double* Yq = Y + qc * ldy;
    v4d acc = {};
    for (int64_t rw = r0 + 64 * wave; rw < r1; rw += GROWS) {
        const int64_t r = rw + 16 * k;
        double x[16], y[16];
        if (rw + 64 <= n) {
#pragma unroll
            for (int t = 0; t < 16; t += 2) {
                const d2u u = *reinterpret_cast<const d2u*>(Xq + r + t);
                const d2u v = *reinterpret_cast<const d2u*>(Yq + r + t);
                x[t] = u[0]; x[t + 1] = u[1];
                y[t] = v[0]; y[t + 1] = v[1];
            }
        } else {
#pragma unroll
            for (int t = 0; t < 16; ++t) {
                const int64_t rc = r + t < n ? r + t : n - 1;
                const double u = Xq[rc], v = Yq[rc];
                x[t] = r + t < n ? u : 0.0;
                y[t] = r + t < n ? v : 0.0;
            }
        }
#pragma unroll
        for (int t = 0; t < 16; ++t)
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(x[t], y[t], acc, 0, 0, 0);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) red[wave][(4 * e + k) + BS * q] = acc[e];
    __syncthreads();
    const int a = tid % s, b = tid / s;
    if (tid < s2) {
        const int i = a + BS * b;
        part[(int64_t)blockIdx.x * s2 + tid] = ((red[0][i] + red[1][i]) + red[2][i]) + red[3][i];
    }
    if (!mpc_last_arrival(tick, (int)gridDim.x)) return;
    if (tid < s2) {
        double v[GWG], t = 0.0;
#pragma unroll
        for (int c = 0; c < GWG; ++c)
            v[c] = part[(int64_t)(c < (int)gridDim.x ? c : 0) * s2 + tid];
#pragma unroll
        for (int c = 0; c < GWG; ++c) t += c < (int)gridDim.x ? v[c] : 0.0;
        G[tid] = t;
    }
}

// Xo = G^-1 H for s x s G (its lower triangle, SPD) and H, through the
// Cholesky factor of G.  One wave, a row of G per lane in registers: column j's
// entries are broadcast to the lanes below by lane reads; then lane c solves
// column c.  A pivot not above kSpdRelPivot times its diagonal entry (G singular
// to working precision, e.g. dependent columns), or not finite, sets *flag
// and gives Xo = 0, so the updates that use Xo leave their blocks unchanged.
// (One thread for the factor: 45 us at s = 16.)
constexpr double kSpdRelPivot = 1e-13;
__global__ __launch_bounds__(64) void spd_solve_kernel(int s, const double* __restrict__ Gm,
                                                      const double* __restrict__ H,
                                                      double* __restrict__ Xo,
                                                      int* __restrict__ flag) {
    __shared__ double C[BS][BS];                 // C[k][i] = L(i, k)
    const int tid = threadIdx.x, r = tid < s ? tid : s - 1;
    double c[BS], x[BS];
#pragma unroll
    for (int k = 0; k < BS; ++k) {
        const int kc = k < s ? k : s - 1;
        c[k] = Gm[r + kc * s];
        x[k] = H[kc + r * s];
    }
    bool bad = false;
#pragma unroll
    for (int j = 0; j < BS; ++j) {
        if (j < s && !bad) {                     // (uniform)
            const double d = mpc_lane_value(c[j], j), g = Gm[j + j * s];
            if (!(d > kSpdRelPivot * g) || !(d < INFINITY)) {
                bad = true;
            } else {
                const double l = sqrt(d);
                c[j] = tid == j ? l : c[j] / l;  // lanes above j hold nothing of use
#pragma unroll
                for (int k = j + 1; k < BS; ++k)
                    if (k < s) c[k] = fma(-c[j], mpc_lane_value(c[j], k), c[k]);
            }
        }
        if (tid < BS) C[j][tid] = c[j];
    }
    if (bad && tid == 0) flag[0] = 1;
    __syncthreads();
    if (tid >= s) return;
    if (!bad) {
#pragma unroll
        for (int i = 0; i < BS; ++i) {                 // L y = h
            if (i < s) {
#pragma unroll
                for (int k = 0; k < i; ++k) x[i] = fma(-C[k][i], x[k], x[i]);
                x[i] /= C[i][i];
            }
        }
#pragma unroll
        for (int i = BS - 1; i >= 0; --i) {            // L^T x = y
            if (i < s) {
#pragma unroll
                for (int k = i + 1; k < BS; ++k)
                    if (k < s) x[i] = fma(-C[i][k], x[k], x[i]);
                x[i] /= C[i][i];
            }
        }
    }
#pragma unroll
    for (int i = 0; i < BS; ++i)
        if (i < s) Xo[i + tid * s] = bad ? 0.0 : x[i];
}

// Y[r][j] = (Z ? Z[r][j] : Y[r][j]) + a sum_k M[r][k] Cm[k][j], one thread
// per row; the row of M is read before any write, so Y may be M.  All loads of
// a row are in flight at once, and a workgroup is one wave, so that a few
// thousand rows reach many CUs (n = 6000, s = 16: 17.3 us with 256 rows a
// workgroup and a base column at a time).
__global__ __launch_bounds__(64) void block_axpy_kernel(int64_t n, int s, const double* M,
                                                       int64_t ldm, const double* __restrict__ Cm,
                                                       double a, const double* Z, int64_t ldz,
                                                       double* Y, int64_t ldy) {
    __shared__ double cs[BS * BS];
    const int64_t r0 = (int64_t)blockIdx.x * 64 + threadIdx.x, r = r0 < n ? r0 : n - 1;
    const double* B = Z ? Z : Y;
    const int64_t ldb = Z ? ldz : ldy;
    double m[BS], y[BS];
#pragma unroll
    for (int k = 0; k < BS; ++k) {
        const int kc = k < s ? k : s - 1;
        m[k] = M[kc * ldm + r];
        y[k] = B[kc * ldb + r];
    }
    for (int idx = threadIdx.x; idx < s * s; idx += 64) cs[idx] = Cm[idx];
    __syncthreads();
    if (r0 >= n) return;
#pragma unroll
    for (int j = 0; j < BS; ++j) {
        if (j < s) {
            double v = 0.0;
#pragma unroll
            for (int k = 0; k < BS; ++k)
                if (k < s) v = fma(m[k], cs[k + j * s], v);
            Y[j * ldy + r] = fma(a, v, y[j]);
        }
    }
}

inline unsigned blocks_for(int64_t n) { return (unsigned)((n + RB - 1) / RB); }

}  // namespace

// right-hand sides of the next pass: at most SY_JMAX (padded to 1, 2 or 4) with
// the kernel above, at most MPC_MM_NJ on the matrix cores
static int symv_pass_rhs(int nrhs) {
    return nrhs > SY_JMAX ? std::min(nrhs, MPC_MM_NJ) : nrhs <= 1 ? 1 : nrhs <= 2 ? 2 : SY_JMAX;
}
// Tiles per super-tile side: small matrices need the workgroups (n = 777, one
// right-hand side: 8.7 / 10.5 / 20 us with 1 / 2 / 4; n = 3001: 11.8 / 13.9 /
// 25), large ones the fewer partial sums (n = 6000: 25.6 / 25.1 / 27.7, 12000:
// 72 / 55 / 62, 16384: 145 / 132 / 121, 36864: 671 / 580 / 540).
static int symv_tiles(int64_t n) { return n >= 14336 ? 4 : n >= 4608 ? 2 : 1; }
// Workgroups of the product on the matrix cores (16 columns: n = 3000 16.5 /
// 19.7 / 21.4 / 23.5 us with 512 / 1024 / 1536 / 2048, 8192 61 / 62 / 67 / 66, 8684
// 85 / 78 / 78 / 80, 12000 164 / 134 / 128 / 136, 16384 222 / 223 / 230 / 225)
static int64_t symv_splits(int64_t n) { return mpc_mm_splits(n, n, n <= 4096 ? 512 : 1024); }

int64_t mpc_symv_partial_doubles(int64_t n, int nrhs) {
    const int64_t E = SY_T * symv_tiles(n), nst = (n + E - 1) / E;
    const int64_t sym = nst * nst * E * (nrhs > 2 ? SY_JMAX : nrhs);
    return nrhs > SY_JMAX ? std::max(sym, symv_splits(n) * n * std::min(nrhs, MPC_MM_NJ)) : sym;
}

template <typename T, int S>
static void launch_symv_pass(hipStream_t st, const T* A, int64_t lda, int64_t n, int NJ, int j0,
                             int nj, const double* X, int64_t ldx, double* Y, int64_t ldy,
                             double* part) {
    const int64_t E = SY_T * S, nst = (n + E - 1) / E;
    const dim3 g((unsigned)(nst * (nst + 1) / 2)), b(256);
    switch (NJ) {
    case 1: hipLaunchKernelGGL((symv_super_kernel<T, 1, S>), g, b, 0, st, A, lda, n, (int)nst, j0, nj, X, ldx, part); break;
    case 2: hipLaunchKernelGGL((symv_super_kernel<T, 2, S>), g, b, 0, st, A, lda, n, (int)nst, j0, nj, X, ldx, part); break;
    default: hipLaunchKernelGGL((symv_super_kernel<T, SY_JMAX, S>), g, b, 0, st, A, lda, n, (int)nst, j0, nj, X, ldx, part); break;
    }
    hipLaunchKernelGGL(symv_reduce_kernel, dim3((unsigned)((n + 63) / 64), (unsigned)nj), dim3(256), 0,
                       st, n, (int)E, (int)nst, NJ, j0, part, Y, ldy);
}

template <typename T>
static int launch_symv_t(hipStream_t st, const T* A, int64_t lda, int64_t n, int nrhs,
                         const double* X, int64_t ldx, double* Y, int64_t ldy, double* part) {
    for (int j0 = 0; j0 < nrhs;) {
        const int NJ = symv_pass_rhs(nrhs - j0), nj = std::min(nrhs - j0, NJ);
        if (NJ > SY_JMAX) {
            const int64_t S = symv_splits(n);
            int rc = mpc_launch_mm_n(st, A, lda, n, n, 3, X + j0 * ldx, ldx, nj, part, S);
            if (!rc) rc = mpc_launch_mm_sum(st, n, nj, n, S, 0, MPC_MM_GROUP_N, part, nullptr, 0, 1.0, Y + j0 * ldy, ldy);
            if (rc) return rc;
        } else {
            switch (symv_tiles(n)) {
            case 1: launch_symv_pass<T, 1>(st, A, lda, n, NJ, j0, nj, X, ldx, Y, ldy, part); break;
            case 2: launch_symv_pass<T, 2>(st, A, lda, n, NJ, j0, nj, X, ldx, Y, ldy, part); break;
            default: launch_symv_pass<T, 4>(st, A, lda, n, NJ, j0, nj, X, ldx, Y, ldy, part); break;
            }
            MPC_LAUNCH_CHECK();
        }
        j0 += nj;
    }
    return 0;
}

int mpc_launch_symv(hipStream_t st, const float* A, int64_t lda, int64_t n, int nrhs,
                    const double* X, int64_t ldx, double* Y, int64_t ldy, double* part) {
    return launch_symv_t<float>(st, A, lda, n, nrhs, X, ldx, Y, ldy, part);
}

int mpc_launch_symv64(hipStream_t st, const double* A, int64_t lda, int64_t n, int nrhs,
                      const double* X, int64_t ldx, double* Y, int64_t ldy, double* part) {
    return launch_symv_t<double>(st, A, lda, n, nrhs, X, ldx, Y, ldy, part);
}

// ndot dots of a with b and (2) c, to out_b and out_c
static int launch_dots(hipStream_t st, int64_t n, int nrhs, const double* a, int64_t lda_,
                       const double* b, int64_t ldb, double* out_b, const double* c, int64_t ldc,
                       double* out_c, unsigned ndot, double* part) {
    if (n <= kDotOne) {
        hipLaunchKernelGGL(dot_kernel, dim3((unsigned)nrhs, ndot), dim3(1024), 0, st, n, a, lda_, b, ldb, c,
                           ldc, out_b, out_c);
        MPC_LAUNCH_CHECK();
        return 0;
    }
    const unsigned nparts = (unsigned)((n + RB * 8 - 1) / (RB * 8));
    hipLaunchKernelGGL(dot_partial_kernel, dim3(nparts, (unsigned)nrhs, ndot), dim3(RB), 0, st, n, a,
                       lda_, b, ldb, c, ldc, part);
    MPC_LAUNCH_CHECK();
    hipLaunchKernelGGL(dot_final_kernel, dim3((unsigned)nrhs, ndot), dim3(RB), 0, st, (int)nparts, part,
                       out_b, out_c);
    MPC_LAUNCH_CHECK();
    return 0;
}

int mpc_launch_dot(hipStream_t st, int64_t n, int nrhs, const double* a, int64_t lda_,
                   const double* b, int64_t ldb, double* out, double* part) {
    return launch_dots(st, n, nrhs, a, lda_, b, ldb, out, b, ldb, out, 1, part);
}

int mpc_launch_dot2(hipStream_t st, int64_t n, int nrhs, const double* a, int64_t lda_,
                    const double* b, int64_t ldb, double* out_b, const double* c, int64_t ldc,
                    double* out_c, double* part) {
    return launch_dots(st, n, nrhs, a, lda_, b, ldb, out_b, c, ldc, out_c, 2, part);
}

int mpc_launch_pcg_update_xr(hipStream_t st, int64_t n, int nrhs, double* X, int64_t ldx,
                             double* R, int64_t ldr, const double* P, int64_t ldp,
                             const double* Q, int64_t ldq, const double* rz, const double* pq,
                             const int* active) {
    hipLaunchKernelGGL(update_xr_kernel, dim3(blocks_for(n), (unsigned)nrhs), dim3(RB), 0, st, n, X,
                       ldx, R, ldr, P, ldp, Q, ldq, rz, pq, active);
    MPC_LAUNCH_CHECK();
    return 0;
}

int mpc_launch_pcg_update_p(hipStream_t st, int64_t n, int nrhs, double* P, int64_t ldp,
                            const double* Z, int64_t ldz, const double* rz_new,
                            const double* rz_old, const int* active) {
    hipLaunchKernelGGL(update_p_kernel, dim3(blocks_for(n), (unsigned)nrhs), dim3(RB), 0, st, n, P,
                       ldp, Z, ldz, rz_new, rz_old, active);
    MPC_LAUNCH_CHECK();
    return 0;
}

int mpc_launch_pcg_status(hipStream_t st, int nrhs, double* rz, const double* rz_new,
                          const double* pq, const double* rr, const double* bb, double tol,
                          int stop_rule, int* active, int* cand, int* iters, double* relres,
                          double* ahist, double* bhist, int hmax) {
    hipLaunchKernelGGL(pcg_status_kernel, dim3((unsigned)((nrhs + 255) / 256)), dim3(256), 0, st,
                       nrhs, rz, rz_new, pq, rr, bb, tol, stop_rule, active, cand, iters, relres,
                       ahist, bhist, hmax);
    MPC_LAUNCH_CHECK();
    return 0;
}

int mpc_launch_axpby(hipStream_t st, int64_t n, int nrhs, double a, const double* X, int64_t ldx,
                     double b, double* Y, int64_t ldy) {
    hipLaunchKernelGGL(axpby_kernel, dim3(blocks_for(n), (unsigned)nrhs), dim3(RB), 0, st, n, a, X,
                       ldx, b, Y, ldy);
    MPC_LAUNCH_CHECK();
    return 0;
}

int mpc_launch_copy2d(hipStream_t st, int64_t n, int nrhs, const double* X, int64_t ldx,
                      double* Y, int64_t ldy) {
    hipLaunchKernelGGL(copy2d_kernel, dim3(blocks_for(n), (unsigned)nrhs), dim3(RB), 0, st, n, X,
                       ldx, Y, ldy);
    MPC_LAUNCH_CHECK();
    return 0;
}

int mpc_launch_copy_lower(hipStream_t st, int64_t rows, int64_t cols, const float* A, int64_t lda,
                          float* B, int64_t ldb) {
    const dim3 g((unsigned)((rows + 4 * RB - 1) / (4 * RB)), (unsigned)((cols + CPC - 1) / CPC));
    hipLaunchKernelGGL(copy_lower_kernel, g, dim3(RB), 0, st, rows, cols, A, lda, B, ldb);
    MPC_LAUNCH_CHECK();
    return 0;
}

int64_t mpc_gram_partial_doubles(int64_t n, int s) {
    (void)n;
    return GWG * (int64_t)s * s;
}

int mpc_launch_gram(hipStream_t st, int64_t n, int s, const double* X, int64_t ldx,
                    const double* Y, int64_t ldy, double* part, double* G, int* tick) {
    if (s < 1 || s > BS) {
        mpc_set_error("gram: block of %d columns (1..%d)", s, BS);
        return MPC_ERR_ARG;
    }
    const int64_t chunk = gram_rows(n);
    hipLaunchKernelGGL(gram_kernel, dim3((unsigned)((n + chunk - 1) / chunk)), dim3(256), 0, st, n, s,
                       chunk, X, ldx, Y, ldy, part, G, tick);
    MPC_LAUNCH_CHECK();
    return 0;
}

int mpc_launch_spd_solve(hipStream_t st, int s, const double* G, const double* H, double* X,
                         int* flag) {
    hipLaunchKernelGGL(spd_solve_kernel, dim3(1), dim3(64), 0, st, s, G, H, X, flag);
    MPC_LAUNCH_CHECK();
    return 0;
}

int mpc_launch_block_axpy(hipStream_t st, int64_t n, int s, const double* M, int64_t ldm,
                          const double* Cm, double a, const double* Z, int64_t ldz, double* Y,
                          int64_t ldy) {
    hipLaunchKernelGGL(block_axpy_kernel, dim3((unsigned)((n + 63) / 64)), dim3(64), 0, st, n, s, M, ldm, Cm,
                       a, Z, ldz, Y, ldy);
    MPC_LAUNCH_CHECK();
    return 0;
}
