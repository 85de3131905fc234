// k_gp.hip -- fused gradient contraction of the GP loss.
//
// No counterpart in the reference (its RBF.cu is an empty stub); the GP
// workload is defined by the differentiable-solve configuration.  For
//   loss = 1/2 b^T A^-1 b + 1/2 logdet A,
//   A_ij = variance * exp(-1/2 sum_c ((x_ic - x_jc) / ls_c)^2) + noise [i == j],
// every parameter theta has dloss/dtheta = sum_ij M_ij dA_ij/dtheta with
//   M = -1/2 alpha alpha^T + (w / 2) sum_p A^-1 z_p z_p^T = U V^T,
//   U = [-alpha/2, w/2 A^-1 z_1, ...],  V = [alpha, z_1, ...],
// (alpha = A^-1 b; w = 1/P for Rademacher probes, 1 for unit probes, which
// make the trace exact).  dA/dtheta is symmetric, so only the lower triangle
// is visited with the symmetrised weight m_ij = (U V^T)_ij + (U V^T)_ji.
// The kernel entries are recomputed in FP64 from the FP32 points instead of
// being stored; per entry:
//   dA_ij/dls_c     = K_ij (x_ic - x_jc)^2 / ls_c^3   (isotropic: summed over c)
//   dA_ij/dvariance = K_ij / variance
//   dA_ij/dnoise    = [i == j]
// Each workgroup writes its partial sums to a fixed slot; a second kernel adds
// the slots in order, so the result is bitwise reproducible.
#include "mpc_internal.hpp"

namespace {

constexpr int GT = 64;        // tile edge
typedef double v4d __attribute__((ext_vector_type(4)));

// One 64 x 64 tile of the lower triangle per workgroup, a 32 x 32 quarter per
// wave.  m comes from the FP64 matrix cores (v_mfma_f64_16x16x4, operands
// straight from L2: lane (q, k) of a product holds row q, solve column k, and
// receives in register e the element (4e + k, q)); the 16 elements of a lane
// then share the loops over the dimensions.  Bound by the FP64 vector
// operations of the kernel entries (exp and two passes over the dimensions).
__global__ __launch_bounds__(256, 2) void gp_grad_tile_kernel(
    const float* __restrict__ X, int64_t n, int d, int64_t ldx, const double* __restrict__ inv_ls,
    int n_ls, double variance, const double* __restrict__ U, const double* __restrict__ V,
    int64_t ldu, int R, double* __restrict__ part) {
    __shared__ double xi[MPC_GP_MAXD][GT], xj[MPC_GP_MAXD][GT];
    __shared__ double red[4][MPC_GP_MAXD + 2];
    // lower tile (I >= J): t = I (I + 1) / 2 + J
    const int64_t t = blockIdx.x;
    int64_t I = (int64_t)((sqrt(8.0 * (double)t + 1.0) - 1.0) * 0.5);
    while (I * (I + 1) / 2 > t) --I;
    while ((I + 1) * (I + 2) / 2 <= t) ++I;
    const int64_t J = t - I * (I + 1) / 2;
    const int64_t i0 = I * GT, j0 = J * GT;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int q = lane & 15, k = lane >> 4;
    const int bi = 32 * (wave & 1), bj = 32 * (wave >> 1);       // this wave's quarter

    for (int idx = tid; idx < d * GT; idx += 256) {
        const int c = idx / GT, p = idx % GT;
        const double s = inv_ls[n_ls == 1 ? 0 : c];
        const int64_t ri = i0 + p < n ? i0 + p : n - 1, rj = j0 + p < n ? j0 + p : n - 1;
        const double a = (double)X[ri * ldx + c] * s, b = (double)X[rj * ldx + c] * s;
        xi[c][p] = i0 + p < n ? a : 0.0;
        xj[c][p] = j0 + p < n ? b : 0.0;
    }
    // m = (U V^T)_ij + (U V^T)_ji
    v4d m[2][2] = {};
    int64_t gi[2], gj[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int64_t i = i0 + bi + 16 * u + q, j = j0 + bj + 16 * u + q;
        gi[u] = i < n ? i : n - 1;           // (rows past the end are dropped below)
        gj[u] = j < n ? j : n - 1;
    }
    double ui[2], vi[2], uj[2], vj[2];
    auto load = [&](int r0) {
        const int r = r0 + k;
        const int64_t o = (int64_t)(r < R ? r : R - 1) * ldu;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const double a = U[o + gi[u]], b = V[o + gi[u]], c = U[o + gj[u]], e = V[o + gj[u]];
            ui[u] = r < R ? a : 0.0;
            vi[u] = r < R ? b : 0.0;
            uj[u] = r < R ? c : 0.0;
            vj[u] = r < R ? e : 0.0;
        }
    };
    load(0);
    for (int r0 = 0; r0 < R; r0 += 4) {
        double a[2], b[2], c[2], e[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            a[u] = ui[u];
            b[u] = vi[u];
            c[u] = uj[u];
            e[u] = vj[u];
        }
        if (r0 + 4 < R) load(r0 + 4);
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int v = 0; v < 2; ++v) {
                m[u][v] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u], e[v], m[u][v], 0, 0, 0);
                m[u][v] = __builtin_amdgcn_mfma_f64_16x16x4f64(b[u], c[v], m[u][v], 0, 0, 0);
            }
    }
    __syncthreads();
    // element x = 8u + 4v + e of this lane: (pi(u, e), pj(v))
    auto pi = [&](int u, int e) { return bi + 16 * u + 4 * e + k; };
    auto pj = [&](int v) { return bj + 16 * v + q; };
    double s2[16] = {};
    for (int c = 0; c < d; ++c) {
        double y[2];
#pragma unroll
        for (int v = 0; v < 2; ++v) y[v] = xj[c][pj(v)];
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const double x = xi[c][pi(u, e)];
#pragma unroll
                for (int v = 0; v < 2; ++v) {
                    const double df = x - y[v];
                    s2[8 * u + 4 * v + e] = fma(df, df, s2[8 * u + 4 * v + e]);
                }
            }
    }
    // the lower triangle's weights; m counts the diagonal twice
    double wk[16], gvar = 0.0, gnoise = 0.0, giso = 0.0;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int v = 0; v < 2; ++v)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int x = 8 * u + 4 * v + e;
                const int64_t i = i0 + pi(u, e), j = j0 + pj(v);
                double w = i < n && j <= i ? m[u][v][e] : 0.0;
                if (i == j) {
                    w *= 0.5;
                    gnoise += w;
                }
                wk[x] = w * (variance * exp(-0.5 * s2[x]));
                gvar += wk[x];
                giso = fma(wk[x], s2[x], giso);
            }
    const int nout = (n_ls == 1 ? 1 : d) + 2;
    auto out = [&](int c, double v) {
        v = mpc_sum64(v);
        if (lane == 0) red[wave][c] = v;
    };
    if (n_ls == 1) {
        out(0, giso);                        // times 1/ls on the host
    } else {
        for (int c = 0; c < d; ++c) {
            double y[2], g = 0.0;
#pragma unroll
            for (int v = 0; v < 2; ++v) y[v] = xj[c][pj(v)];
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const double x = xi[c][pi(u, e)];
#pragma unroll
                    for (int v = 0; v < 2; ++v) {
                        const double df = x - y[v];
                        g = fma(wk[8 * u + 4 * v + e], df * df, g);
                    }
                }
            out(c, g);
        }
    }
    out(nout - 2, gvar);
    out(nout - 1, gnoise);
    __syncthreads();
    if (tid < nout) part[t * nout + tid] = ((red[0][tid] + red[1][tid]) + red[2][tid]) + red[3][tid];
}

// out[q] = sum over tiles of part[t][q], tiles added in a fixed order
__global__ __launch_bounds__(256) void gp_grad_reduce_kernel(const double* __restrict__ part,
                                                            int64_t ntile, int nout,
                                                            double* __restrict__ out) {
    __shared__ double s[256];
    const int q = blockIdx.x, tid = threadIdx.x;
    double a = 0.0;
    for (int64_t t = tid; t < ntile; t += 256) a += part[t * nout + q];
    s[tid] = a;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (tid < w) s[tid] += s[tid + w];
        __syncthreads();
    }
    if (tid == 0) out[q] = s[0];
}

// out = sum_i log L_ii (fixed order: strided per thread, then a tree)
__global__ __launch_bounds__(256) void logdiag_kernel(const float* __restrict__ L, int64_t ldl,
                                                     int64_t n, double* __restrict__ out) {
    __shared__ double s[256];
    const int tid = threadIdx.x;
    double a = 0.0;
    for (int64_t i = tid; i < n; i += 256) a += log((double)L[i + i * ldl]);
    s[tid] = a;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (tid < w) s[tid] += s[tid + w];
        __syncthreads();
    }
    if (tid == 0) *out = s[0];
}

}  // namespace

int mpc_launch_logdiag(hipStream_t st, const float* L, int64_t ldl, int64_t n, double* out) {
    hipLaunchKernelGGL(logdiag_kernel, dim3(1), dim3(256), 0, st, L, ldl, n, out);
    MPC_LAUNCH_CHECK();
    return 0;
}

int64_t mpc_gp_partial_doubles(int64_t n, int nout) {
    const int64_t nt = (n + GT - 1) / GT;
    return nt * (nt + 1) / 2 * nout;
}

int mpc_launch_gp_grad(hipStream_t st, const float* X, int64_t n, int d, int64_t ldx,
                       const double* inv_ls, int n_ls, double variance, const double* U,
                       const double* V, int64_t ldu, int R, double* part, double* out) {
    if (d > MPC_GP_MAXD || d < 1 || (n_ls != 1 && n_ls != d)) {
        mpc_set_error("gp gradient: d must be 1..%d and n_ls 1 or d", MPC_GP_MAXD);
        return MPC_ERR_ARG;
    }
    const int64_t nt = (n + GT - 1) / GT;
    const int64_t ntile = nt * (nt + 1) / 2;
    const int nout = (n_ls == 1 ? 1 : d) + 2;
    hipLaunchKernelGGL(gp_grad_tile_kernel, dim3((unsigned)ntile), dim3(256), 0, st, X, n, d, ldx,
                       inv_ls, n_ls, variance, U, V, ldu, R, part);
    hipLaunchKernelGGL(gp_grad_reduce_kernel, dim3((unsigned)nout), dim3(256), 0, st, part, ntile,
                       nout, out);
    MPC_LAUNCH_CHECK();
    return 0;
}
