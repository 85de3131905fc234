// k_mrhs.hip -- products of a matrix with blocks of up to 16 right-hand sides
// (FP64 vectors, FP32 or FP64 matrix), on the FP64 matrix cores
// (v_mfma_f64_16x16x4: exact FP32-to-FP64 operands, FP64 sums).
//
// D = a b with a[m][k] = the right-hand sides (m) and b[k][n] = the matrix.
// Lane (q, k) = (lane % 16, lane / 16) of a wave supplies a[q][k], b[k][q] and
// receives in register e the element D[4e + k][q].
//   mm_n (rows of the matrix are the outputs): a lane loads rows 4q .. 4q+3 of
//     one column, 16 bytes, so 16 lanes read a 256-byte column segment, and
//     its element i is the operand of the product whose n stands for row
//     4n + i: no transpose and no LDS.
//     Symmetric A (mode 3) is read from its upper triangle only, as the kernels
//     for fewer right-hand sides do: left of the diagonal the product's columns
//     are rows there, so a lane takes rows 4k .. 4k+3 of columns 4q .. 4q+3
//     (FP32: through LDS) and names the 16 values the other way round.
//   mm_t (columns are the outputs): lane (q, k) loads rows 4k .. 4k+3 of
//     column q; element i is the operand with k <-> row 4k + i.
// The right-hand sides are read as operands straight from L2.  Per 8 KB of an
// FP32 matrix a wave issues 32 products of 64 cycles, 9.8 TB/s over 1024 SIMDs:
// above what HBM delivers.  With 16 right-hand sides (A X, symmetric FP32 A)
// n = 8192 takes 62 us, each element read twice (4.3 TB/s; 57 where both
// triangles are read directly), where two passes of 8 that read the elements
// once, with FP64 FMAs from LDS, took 244.
#include "mpc_internal.hpp"
#include <algorithm>

namespace {

typedef double v4d __attribute__((ext_vector_type(4)));
typedef double d2 __attribute__((ext_vector_type(2), aligned(8)));
constexpr int MR = 64;          // output rows of a workgroup (mm_n)
constexpr int MU = 4;           // columns of a group per lane (8: two waves per SIMD
                                // instead of three, 5-15 % slower)
constexpr int MG = MPC_MM_GROUP_N;      // columns of a group
static_assert(MG == 4 * MU, "group");
constexpr int MFL = 8;          // groups per partial sum of a wave
constexpr int MTC = 32;         // output columns of a workgroup (mm_t)
constexpr int MTG = MPC_MM_GROUP_T;     // rows of a group (mm_t)

// which column chunks [s cw, (s+1) cw) have work for row block r0 (mode 1:
// lower triangle, columns up to the row; 2: upper, columns from the row on)
__device__ __forceinline__ void split_range(int mode, int64_t r0, int64_t rows, int64_t cw, int S,
                                            int& s0, int& s1) {
    s0 = mode == 2 ? (int)(r0 / cw) : 0;
    const int64_t last = mode == 1 ? (r0 + rows - 1) / cw + 1 : S;
    s1 = last < S ? (int)last : S;
}

// part[(s nj + j) m + r] = sum_{c in chunk s} A[r][c] X[j][c] for the 64 rows of
// blockIdx.x, chunk s = blockIdx.y of cw columns (a multiple of MG).  Wave w
// takes the chunk's column groups w, w + 4, ..; the four waves' sums are added
// in wave order through LDS.  blockIdx.z: 16 of the right-hand sides.
//
// A last row block that is not full (m >= 64) moves up to end at row m and
// stores only its own rows: with predicated 4-byte loads its workgroups ran
// several times as long as the others (16 right-hand sides, mode 0: n = 12000
// 185 us, moved up 112; n = 8684 108 and 72).
template <typename T, int MODE>
__global__ __launch_bounds__(256) void mm_n_kernel(const T* __restrict__ A, int64_t lda, int64_t m,
                                                  int64_t kc, int64_t cw, const double* __restrict__ X,
                                                  int64_t ldx, int nj, double* __restrict__ part) {
    typedef T vec4 __attribute__((ext_vector_type(4), aligned(sizeof(T))));
    __shared__ __align__(16) double red[4][MPC_MM_NJ][MR];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int q = lane & 15, k = lane >> 4;
    const int64_t rb = (int64_t)blockIdx.x * MR, cs = (int64_t)blockIdx.y * cw;
    const int64_t r0 = m >= MR && rb + MR > m ? m - MR : rb;
    int64_t ce = cs + cw < kc ? cs + cw : kc;
    if (MODE == 1 && ce > r0 + MR) ce = r0 + MR < kc ? r0 + MR : kc;
    int64_t cb = cs;
    if (MODE == 2 && cb < r0) cb = r0 & ~(int64_t)(MG - 1);
    if (cb >= ce) return;                        // (the sum skips this chunk)
    const int j0 = blockIdx.z * MPC_MM_NJ;
    const double* __restrict__ Xj = X + (int64_t)(j0 + q < nj ? j0 + q : nj - 1) * ldx;
    const int64_t r = r0 + 4 * q;
    const bool rfull = r0 + MR <= m;
    vec4 v[MU];
    double x[MU];
    auto load = [&](int64_t c0) {
        const int64_t c = c0 + MU * k;            // this lane's columns
        if (rfull && c0 + MG <= kc) {
            if (MODE == 3 && c0 < r0 + MR - 1) {      // not above the diagonal as a whole
                vec4 t[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) t[i] = *reinterpret_cast<const vec4*>(A + c + (r + i) * lda);
                const bool mirror = c0 + MG <= r0 + 1;    // below it
#pragma unroll
                for (int s = 0; s < MU; ++s) {
                    if (!mirror) v[s] = *reinterpret_cast<const vec4*>(A + r + (c + s) * lda);
#pragma unroll
                    for (int i = 0; i < 4; ++i) v[s][i] = mirror || c + s < r + i ? t[i][s] : v[s][i];
                }
            } else {
#pragma unroll
                for (int s = 0; s < MU; ++s) v[s] = *reinterpret_cast<const vec4*>(A + r + (c + s) * lda);
            }
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
                    const int64_t rc = r + i < m ? r + i : m - 1;
                    const bool up = MODE != 3 || rc <= cc;
                    const T y = A[(up ? rc : cc) + (up ? cc : rc) * lda];
                    v[s][i] = (r + i < m && c + s < kc) ? y : T(0);
                }
                const double y = Xj[cc];
                x[s] = c + s < kc ? y : 0.0;
            }
        }
        if (MODE == 1 && c0 + MG > r0) {         // zeros above the diagonal
#pragma unroll
            for (int s = 0; s < MU; ++s)
#pragma unroll
                for (int i = 0; i < 4; ++i) v[s][i] = c + s <= r + i ? v[s][i] : T(0);
        }
        if (MODE == 2 && c0 < r0 + MR) {         // zeros below the diagonal
#pragma unroll
            for (int s = 0; s < MU; ++s)
#pragma unroll
                for (int i = 0; i < 4; ++i) v[s][i] = c + s >= r + i ? v[s][i] : T(0);
        }
    };
    // Sums of MFL groups (128 terms) are added up apart: one running sum over a
    // wave's part of the chunk (2048 terms of the longest) loses accuracy with its
    // length, which the residual of a solve at cond 1e8 shows (n = 65536).
    v4d acc[4], tot[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = tot[i] = v4d{};
    int64_t c0 = cb + MG * wave;
    int g = 1;
    if constexpr (MODE == 3 && sizeof(T) == 4) {
        // Left of the diagonal a wave's 16 columns of the product are 64-byte
        // pieces of 64 columns of A.  Loaded as such they cost a third more than
        // 256-byte ones (n = 16384, both triangles read directly 200 us, this way
        // 266; FP64, 128 bytes: no difference).  So the workgroup loads 64 x 64
        // elements at a time in 256-byte pieces, wave w columns 16 w + .., and the
        // waves read theirs from LDS (224 us): column x's 4-row piece y lies at
        // 16-byte slot y ^ (x / 4), which is free of conflicts both ways.
        typedef T lds4 __attribute__((ext_vector_type(4)));
        lds4* const buf = reinterpret_cast<lds4*>(&red[0][0][0]);
        const int64_t steps = rfull && r0 + 1 > cb ? ((ce < r0 + 1 ? ce : r0 + 1) - cb) / (4 * MG) : 0;
        const T* src = A + cb + 4 * q + (r0 + 16 * wave + k) * lda;
        lds4 st[4], w[4];
        double y[MU];
        auto fetch = [&](int64_t t) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                st[i] = *reinterpret_cast<const vec4*>(src + 4 * MG * t + (int64_t)(4 * i) * lda);
#pragma unroll
            for (int s = 0; s < MU; s += 2) {
                const d2 z = *reinterpret_cast<const d2*>(Xj + c0 + 4 * MG * t + MU * k + s);
                x[s] = z[0];
                x[s + 1] = z[1];
            }
        };
        if (steps > 0) fetch(0);
        for (int64_t t = 0; t < steps; ++t) {
            lds4* const b = buf + 1024 * (t & 1);
#pragma unroll
            for (int i = 0; i < 4; ++i) b[16 * (16 * wave + 4 * i + k) + (q ^ (4 * wave + i))] = st[i];
#pragma unroll
            for (int s = 0; s < MU; ++s) y[s] = x[s];
            mpc_lds_barrier();                   // (the other buffer is read to the end)
            if (t + 1 < steps) fetch(t + 1);
#pragma unroll
            for (int i = 0; i < 4; ++i) w[i] = b[16 * (4 * q + i) + ((4 * wave + k) ^ q)];
#pragma unroll
            for (int s = 0; s < MU; ++s)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    acc[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(y[s], (double)w[i][s], acc[i], 0, 0, 0);
            if (g++ % MFL == 0) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    tot[i] += acc[i];
                    acc[i] = v4d{};
                }
            }
        }
        c0 += 4 * MG * steps;
        __syncthreads();                         // red is written below
    }
    if (c0 < ce) load(c0);
    for (; c0 < ce; c0 += 4 * MG, ++g) {
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
        if (g % MFL == 0) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                tot[i] += acc[i];
                acc[i] = v4d{};
            }
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] += tot[i];
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < 4; ++i) red[wave][4 * e + k][4 * q + i] = acc[i][e];
    __syncthreads();
    if (r0 + lane < m && r0 + lane >= rb) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int j = wave + 4 * u;
            if (j0 + j < nj)
                part[((int64_t)blockIdx.y * nj + j0 + j) * m + r0 + lane] =
                    ((red[0][j][lane] + red[1][j][lane]) + red[2][j][lane]) + red[3][j][lane];
        }
    }
}

// part[(s nj + j) nc + c] = sum_{r in chunk s} A[r][c] X[j][r] for the 32
// columns of blockIdx.x, chunk s = blockIdx.y of rw rows (a multiple of MTG).
// Wave w takes the chunk's row groups w, w + 4, .. (blockIdx.z as above), each sum in one piece: this
// product is part of a preconditioner with FP32 entries, never of a residual.
__global__ __launch_bounds__(256) void mm_t_kernel(const float* __restrict__ A, int64_t lda,
                                                  int64_t m, int64_t nc, int64_t rw,
                                                  const double* __restrict__ X, int64_t ldx, int nj,
                                                  double* __restrict__ part) {
    typedef float vec4 __attribute__((ext_vector_type(4), aligned(4)));
    __shared__ double red[4][MPC_MM_NJ][MTC];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int q = lane & 15, k = lane >> 4;
    const int64_t c0 = (int64_t)blockIdx.x * MTC, rs = (int64_t)blockIdx.y * rw;
    const int64_t re = rs + rw < m ? rs + rw : m;
    const int j0 = blockIdx.z * MPC_MM_NJ;
    const double* __restrict__ Xj = X + (int64_t)(j0 + q < nj ? j0 + q : nj - 1) * ldx;
    const float* __restrict__ col[2];
#pragma unroll
    for (int g = 0; g < 2; ++g) {
        const int64_t c = c0 + 16 * g + q;
        col[g] = A + (c < nc ? c : nc - 1) * lda;    // (sums of a column past the end are dropped)
    }
    vec4 v[2][4];
    double x[16];
    auto load = [&](int64_t r0) {
        const int64_t r = r0 + 4 * k;
        if (r0 + MTG <= m) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
#pragma unroll
                for (int g = 0; g < 2; ++g) v[g][u] = *reinterpret_cast<const vec4*>(col[g] + r + 16 * u);
#pragma unroll
                for (int i = 0; i < 4; i += 2) {
                    const d2 y = *reinterpret_cast<const d2*>(Xj + r + 16 * u + i);
                    x[4 * u + i] = y[0];
                    x[4 * u + i + 1] = y[1];
                }
            }
        } else {
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int64_t rr = r + 16 * u + i, rc = rr < m ? rr : m - 1;
#pragma unroll
                    for (int g = 0; g < 2; ++g) {
                        const float y = col[g][rc];
                        v[g][u][i] = rr < m ? y : 0.f;
                    }
                    const double y = Xj[rc];
                    x[4 * u + i] = rr < m ? y : 0.0;
                }
        }
    };
    v4d acc[2][2];
#pragma unroll
    for (int g = 0; g < 2; ++g) acc[g][0] = acc[g][1] = v4d{};
    int64_t r0 = rs + MTG * wave;
    if (r0 < re) load(r0);
    for (; r0 < re; r0 += 4 * MTG) {
        vec4 w[2][4];
        double y[16];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
#pragma unroll
            for (int g = 0; g < 2; ++g) w[g][u] = v[g][u];
#pragma unroll
            for (int i = 0; i < 4; ++i) y[4 * u + i] = x[4 * u + i];
        }
        if (r0 + 4 * MTG < re) load(r0 + 4 * MTG);
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int g = 0; g < 2; ++g)
                    acc[g][i & 1] = __builtin_amdgcn_mfma_f64_16x16x4f64(y[4 * u + i], (double)w[g][u][i],
                                                                         acc[g][i & 1], 0, 0, 0);
    }
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int e = 0; e < 4; ++e) red[wave][4 * e + k][16 * g + q] = acc[g][0][e] + acc[g][1][e];
    __syncthreads();
    const int c = tid & 31;
    if (c0 + c < nc) {
#pragma unroll
        for (int j = tid >> 5; j < MPC_MM_NJ; j += 8)
            if (j0 + j < nj)
                part[((int64_t)blockIdx.y * nj + j0 + j) * nc + c0 + c] =
                    ((red[0][j][c] + red[1][j][c]) + red[2][j][c]) + red[3][j][c];
    }
}

// Y[j][r] = (B ? B[j][r] : 0) + a sum_s part[(s nj + j) m + r], chunks in order;
// thread = row, 8 loads in flight (clamped chunk, zero weight past the end)
__global__ __launch_bounds__(256) void mm_sum_kernel(int64_t m, int S, int mode, int64_t cw,
                                                    const double* __restrict__ part,
                                                    const double* __restrict__ B, int64_t ldb,
                                                    double a, double* __restrict__ Y, int64_t ldy) {
    const int64_t r0 = (int64_t)blockIdx.x * 256 + threadIdx.x, r = r0 < m ? r0 : m - 1;
    const int j = blockIdx.y, nj = gridDim.y;
    int s0 = 0, s1 = S;
    if (mode) split_range(mode, r & ~(int64_t)(MR - 1), MR, cw, S, s0, s1);
    double sum = 0.0;
    for (int s = s0; s < s1; s += 8) {
        double v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u)
            v[u] = part[((int64_t)(s + u < s1 ? s + u : s1 - 1) * nj + j) * m + r];
#pragma unroll
        for (int u = 0; u < 8; ++u) sum += s + u < s1 ? v[u] : 0.0;
    }
    if (r0 < m) Y[j * ldy + r] = B ? fma(a, sum, B[j * ldb + r]) : a * sum;
}

inline int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }
// columns of a chunk when kc columns are split S ways (whole groups)
inline int64_t chunk(int64_t kc, int64_t S, int64_t unit) { return cdiv(cdiv(kc, S), unit) * unit; }

template <typename T>
int launch_mm_n(hipStream_t st, const T* A, int64_t lda, int64_t m, int64_t kc, int mode,
                const double* X, int64_t ldx, int nj, double* part, int64_t S) {
    if (nj < 1 || S < 1) {
        mpc_set_error("mm_n: %d right-hand sides, %lld chunks", nj, (long long)S);
        return MPC_ERR_ARG;
    }
    const int64_t cw = chunk(kc, S, MG);
    const dim3 g((unsigned)cdiv(m, MR), (unsigned)cdiv(kc, cw), (unsigned)cdiv(nj, MPC_MM_NJ)), b(256);
    if (mode == 1) hipLaunchKernelGGL((mm_n_kernel<T, 1>), g, b, 0, st, A, lda, m, kc, cw, X, ldx, nj, part);
    else if (mode == 2) hipLaunchKernelGGL((mm_n_kernel<T, 2>), g, b, 0, st, A, lda, m, kc, cw, X, ldx, nj, part);
    else if (mode == 3) hipLaunchKernelGGL((mm_n_kernel<T, 3>), g, b, 0, st, A, lda, m, kc, cw, X, ldx, nj, part);
    else hipLaunchKernelGGL((mm_n_kernel<T, 0>), g, b, 0, st, A, lda, m, kc, cw, X, ldx, nj, part);
    MPC_LAUNCH_CHECK();
    return 0;
}

}  // namespace

// Enough chunks for about wgs workgroups, each wave of which has a column
// group, at most 8192 columns a chunk (see MFL).  Every chunk costs a partial
// sum per output.
int64_t mpc_mm_splits(int64_t rows, int64_t kc, int64_t wgs) {
    const int64_t want = std::max(wgs / cdiv(rows, MR), cdiv(kc, 8192)), most = cdiv(kc, 4 * MG);
    return std::max<int64_t>(1, std::min(want, most));
}

// One workgroup a CU, each wave of which has a row group (2048 columns, 16
// right-hand sides, 2048 / 4096 / 6144 rows: 8.3 / 12.6 / 16.8 us; two a CU 8.3 /
// 16 / 23; 3328 workgroups, half of whose waves had no row group, 24 / 41 / 46)
int64_t mpc_mm_splits_t(int64_t cols, int64_t kc) {
    const int64_t want = std::max(256 / cdiv(cols, MTC), cdiv(kc, 8192)), most = cdiv(kc, 4 * MTG);
    return std::max<int64_t>(1, std::min(want, most));
}

int mpc_launch_mm_n(hipStream_t st, const float* A, int64_t lda, int64_t m, int64_t kc, int mode,
                    const double* X, int64_t ldx, int nj, double* part, int64_t S) {
    return launch_mm_n<float>(st, A, lda, m, kc, mode, X, ldx, nj, part, S);
}
int mpc_launch_mm_n(hipStream_t st, const double* A, int64_t lda, int64_t m, int64_t kc, int mode,
                    const double* X, int64_t ldx, int nj, double* part, int64_t S) {
    return launch_mm_n<double>(st, A, lda, m, kc, mode, X, ldx, nj, part, S);
}

int mpc_launch_mm_t(hipStream_t st, const float* A, int64_t lda, int64_t m, int64_t nc,
                    const double* X, int64_t ldx, int nj, double* part, int64_t S) {
    if (nj < 1 || S < 1) {
        mpc_set_error("mm_t: %d right-hand sides, %lld chunks", nj, (long long)S);
        return MPC_ERR_ARG;
    }
    const int64_t rw = chunk(m, S, MTG);
    hipLaunchKernelGGL(mm_t_kernel,
                       dim3((unsigned)cdiv(nc, MTC), (unsigned)cdiv(m, rw), (unsigned)cdiv(nj, MPC_MM_NJ)), dim3(256), 0, st,
                       A, lda, m, nc, rw, X, ldx, nj, part);
    MPC_LAUNCH_CHECK();
    return 0;
}

int mpc_launch_mm_sum(hipStream_t st, int64_t m, int nj, int64_t kc, int64_t S, int mode, int unit,
                      const double* part, const double* B, int64_t ldb, double a, double* Y, int64_t ldy) {
    const int64_t cw = chunk(kc, S, unit);
    hipLaunchKernelGGL(mm_sum_kernel, dim3((unsigned)cdiv(m, 256), (unsigned)nj), dim3(256), 0, st, m,
                       (int)cdiv(kc, cw), mode, cw, part, B, ldb, a, Y, ldy);
    MPC_LAUNCH_CHECK();
    return 0;
}
