// k_tri.hip -- triangular solves of the PCG preconditioner, z = L^-T L^-1 r.
//
// Replaces the two FP64 cusolverDnDpotrs sweeps per PCG iteration
// (mixed_cholesky.cu:147,166,204; potrs on an FP64 copy of L made by
// convertFloattoDouble, :141).  Here L stays FP32 and is read once per sweep
// for all right-hand sides; vectors are FP64.
//
// A row-by-row substitution over n = 16384 rows is a dependency chain; the
// sweep is instead blocked with big diagonal blocks of Bo rows (mpc_block_bo:
// the power of two from n up, at most 2048) whose inverses Winv_I = L_II^{-1}
// are formed once per factor:
//   forward   for I:   y_I = Winv_I w_I ;  w_{>I} -= L_{>I,I} y_I
//   backward  for I:   x_I = Winv_I^T w_I; w_{<I} -= L_{I,<I}^T x_I
// so a sweep is 2 * n / Bo bandwidth-bound kernels with no serial work
// inside.  Winv_I is built by recursive doubling from the 32x32 inverses the
// POTRF kernel leaves behind:
//   [A 0; B C]^{-1} = [A^-1 0; -C^-1 B A^-1  C^-1]
// with a batched GEMM on the matrix cores that skips the zero triangles of
// A^-1 and C^-1.  The temporary B A^-1 lives in the unused upper triangle of
// the Winv block.
#include "mpc_internal.hpp"
#include <algorithm>

namespace {

// ---------------------------------------------------------------- block inverses
// The products of the build are FP32 operands, for up to 8192 rows (and in the
// 128-row blocks of any) with FP64 sums (v_mfma_f64_16x16x4), rounded to FP32
// once when stored: the rounding errors of FP32 sums grow with the block (z of a
// 2048-point RBF factor is then off by 1.5e-7 with Bo = 256 and 7e-7 with Bo =
// 2048; with FP64 sums 7e-8 for every Bo).  Larger matrices, whose blocks had
// 2048 rows and FP32 sums all along, keep them (see gemm_kernel): z of an FP32
// factor at cond 1e6 is off by 1.2e-7 at n = 8192, 1.7e-7 at 8200 and 1.9e-7 at
// 16384.  D = a b: lane (q, k) = (lane % 16, lane / 16) supplies a[q][k] and
// b[k][q]; its register e is D[4e + k][q].
typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

// The 128 x 128 diagonal blocks of the inverse (both W and W^T): the 32 x 32
// inverses and the two doubling levels above them, in LDS.  One workgroup per
// block, wave w = one 16 x 16 quadrant of every 32 x 32 product.  Rows and
// columns beyond n are the identity's.  The products run from short loops
// (20 us; 24 as straight-line code, each line of which is fetched once).
constexpr int LF = 128;
constexpr int LFD = LF + 1;
__global__ __launch_bounds__(256) void winv_leaf_kernel(const float* __restrict__ L, int64_t ldl,
                                                       const float* __restrict__ dinv, int64_t n,
                                                       int Bo, float* __restrict__ W,
                                                       float* __restrict__ WT, int64_t b0) {
    // column-major: the 32 x 32 inverses on the diagonal, L below them until
    // the inverse takes its place, temporaries above
    __shared__ float Ws[LF * LFD];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t r0 = (b0 + blockIdx.x) * LF;
    {
        const int r = tid & (LF - 1), h = tid >> 7;
        const int64_t gr = r0 + r < n ? r0 + r : n - 1;
        const float* Lr = L + gr;
        const float* dr = dinv + (gr >> 5) * 1024 + (gr & 31);
#pragma unroll 1
        for (int c0 = h; c0 < LF; c0 += 64) {
            float v[32];
#pragma unroll
            for (int u = 0; u < 32; ++u) {
                const int c = c0 + 2 * u;
                const int64_t gc = r0 + c < n ? r0 + c : n - 1;
                v[u] = (r >> 5) == (c >> 5) ? dr[(gc & 31) * 32] : Lr[gc * ldl];
            }
#pragma unroll
            for (int u = 0; u < 32; ++u) {
                const int c = c0 + 2 * u;
                Ws[r + c * LFD] = (r0 + r < n && r0 + c < n) ? v[u] : (r == c ? 1.f : 0.f);
            }
        }
    }
    __syncthreads();
    const int q = lane & 15, k = lane >> 4, qr = 16 * (wave & 1), qc = 16 * (wave >> 1);
    // block (r, c) = sgn sum_s A(ar, ac + 32 s) B(br + 32 s, bc), s < ns; lane
    // (q, k)'s register e: row qr + q, column qc + 4e + k (a = B^T, b = A^T)
    auto product = [&](int ns, int ar, int ac, int br, int bc, int r, int c, double sgn) {
        v4d acc = v4d{};
#pragma unroll 1
        for (int s = 0; s < ns; ++s) {
            float x[8], y[8];
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                x[t] = Ws[ar + qr + q + (ac + 32 * s + 8 * k + t) * LFD];
                y[t] = Ws[br + 32 * s + 8 * k + t + (bc + qc + q) * LFD];
            }
#pragma unroll
            for (int t = 0; t < 8; ++t)
                acc = __builtin_amdgcn_mfma_f64_16x16x4f64((double)y[t], (double)x[t], acc, 0, 0, 0);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) Ws[r + qr + q + (c + qc + 4 * e + k) * LFD] = (float)(sgn * acc[e]);
    };
    // level 32, pairs at p = 0 and 64: T = L21 A^-1 above the diagonal, then
    // -C^-1 T below it; level 64 the same in 32 x 32 blocks (i, j) of the
    // 64 x 64 products, whose zero blocks are left out
#pragma unroll 1
    for (int p = 0; p < LF; p += 64) product(1, p + 32, p, p, p, p, p + 32, 1.0);
    __syncthreads();
#pragma unroll 1
    for (int p = 0; p < LF; p += 64) product(1, p + 32, p + 32, p, p + 32, p + 32, p, -1.0);
    __syncthreads();
#pragma unroll 1
    for (int o = 0; o < 4; ++o) {
        const int i = 32 * (o & 1), j = 32 * (o >> 1);
        product(2 - (o >> 1), 64 + i, j, j, j, i, 64 + j, 1.0);
    }
    __syncthreads();
#pragma unroll 1
    for (int o = 0; o < 4; ++o) {
        const int i = 32 * (o & 1), j = 32 * (o >> 1);
        product(1 + (o & 1), 64 + i, 64, 0, 64 + j, 64 + i, j, -1.0);
    }
    __syncthreads();
    const int64_t I = r0 / Bo, p = r0 - I * Bo;       // (Bo is a multiple of LF: inside W_I)
    float* Wi = W + I * (int64_t)Bo * Bo + p + p * Bo;
    float* Ti = WT + I * (int64_t)Bo * Bo + p + p * Bo;
    const int r = tid & (LF - 1);
#pragma unroll 4
    for (int c = tid >> 7; c < LF; c += 2) {
        const float v = r >= c ? Ws[r + c * LFD] : Ws[c + r * LFD];
        (r >= c ? Wi : Ti)[r + (uint32_t)c * (uint32_t)Bo] = v;
        if (r == c) Ti[r + (uint32_t)c * (uint32_t)Bo] = v;
    }
}

// One doubling product for pair q of big block I (batch blockIdx.z = I nq + q):
//   C[m][n] = alpha sum_k A[m][k] B[k][n]    (column-major, ld per operand)
// a_lower: A[m][k] = 0 for k > m; b_lower: B[k][n] = 0 for k < n (applied per
// element while staging, the other triangles hold temporaries, and per tile to
// the K range).  CT (optional): C^T as well.
struct gemm_batch {
    const float* A; const float* B; float* C; float* CT;
    int64_t lda, ldb, ldc;
    int64_t sA, sB, sC;          // stride between pairs q (elements)
    int64_t tA, tB, tC;          // stride between big blocks I
    int nq;
    int m, n, k;
    float alpha;
    int a_lower, b_lower;
};

// 32 x 64 tiles, wave w = a 16 x 32 quadrant; 64 K per stage, the next stage's
// loads in flight during the products (16 steps of two products of 76 cycles).
// Stages inside the operands' triangles and edges move 16 bytes per load and
// LDS store: with a masked 4-byte element each, the staging cost more than the
// products (K = 1024: 50-60 us).  The LDS strides put the 64 lanes of an
// operand read on 64 banks.  Tiles with the longest K range come first.
constexpr int GM = 32, GN = 64, GK = 64;
constexpr int GAS = GM + 16, GBS = GK + 4;
// T = float (v_mfma_f32_16x16x4: FP32 sums, half the time per product; register
// e is D[4k + e][q]) for matrices of more than 8192 rows, whose blocks are
// built beside the factor and compete with it.
template <typename T>
__global__ __launch_bounds__(256) void gemm_kernel(gemm_batch g) {
    typedef T v4 __attribute__((ext_vector_type(4)));
    typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
    typedef float f4 __attribute__((ext_vector_type(4)));
    __shared__ __align__(16) float As[GK * GAS];   // As[k][m]
    __shared__ __align__(16) float Bs[GN * GBS];   // Bs[n][k]
    const int64_t q_ = blockIdx.z % g.nq, I = blockIdx.z / g.nq;
    const float* A = g.A + q_ * g.sA + I * g.tA;
    const float* B = g.B + q_ * g.sB + I * g.tB;
    const int bm = g.a_lower ? gridDim.x - 1 - blockIdx.x : blockIdx.x;
    const int m0 = bm * GM, n0 = blockIdx.y * GN;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int q = lane & 15, k = lane >> 4, wm = 16 * (wave & 1), wn = 32 * (wave >> 1);
    int klo = 0, khi = g.k;
    if (g.a_lower && m0 + GM < khi) khi = m0 + GM;
    if (g.b_lower) klo = n0;
    v4 acc[2] = {v4{}, v4{}};
    // a thread's vectors of a stage: A rows 4 am .. +3 of columns ak + 32 u, B
    // rows 4 bk .. +3 of columns bn + 16 u
    const int am = 4 * (tid & 7), ak = tid >> 3, bk = 4 * (tid & 15), bn = tid >> 4;
    const float* Ap = A + m0 + am + (int64_t)ak * g.lda;
    const float* Bp = B + bk + (int64_t)(n0 + bn) * g.ldb;
    const bool aedge = m0 + GM > g.m, bedge = n0 + GN > g.n;
    f4 xa[2], xb[4];
    auto gload = [&](int k0) {
        if (!aedge && k0 + GK <= khi && (!g.a_lower || k0 + GK <= m0 + 1)) {
#pragma unroll
            for (int u = 0; u < 2; ++u) xa[u] = *reinterpret_cast<const f4u*>(Ap + (int64_t)(k0 + 32 * u) * g.lda);
        } else {
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int gm = m0 + am + i, gk = k0 + ak + 32 * u;
                    const float x = A[(gm < g.m ? gm : g.m - 1) + (int64_t)(gk < khi ? gk : khi - 1) * g.lda];
                    xa[u][i] = (gm < g.m && gk < khi && (!g.a_lower || gk <= gm)) ? x : 0.f;
                }
        }
        if (!bedge && k0 + GK <= khi && (!g.b_lower || k0 + 1 >= n0 + GN)) {
#pragma unroll
            for (int u = 0; u < 4; ++u) xb[u] = *reinterpret_cast<const f4u*>(Bp + k0 + (int64_t)(16 * u) * g.ldb);
        } else {
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int gk = k0 + bk + i, gn = n0 + bn + 16 * u;
                    const float x = B[(gk < khi ? gk : khi - 1) + (int64_t)(gn < g.n ? gn : g.n - 1) * g.ldb];
                    xb[u][i] = (gk < khi && gn < g.n && (!g.b_lower || gk >= gn)) ? x : 0.f;
                }
        }
    };
    if (klo < khi) gload(klo);
    for (int k0 = klo; k0 < khi; k0 += GK) {
#pragma unroll
        for (int u = 0; u < 2; ++u) *reinterpret_cast<f4*>(As + (ak + 32 * u) * GAS + am) = xa[u];
#pragma unroll
        for (int u = 0; u < 4; ++u) *reinterpret_cast<f4*>(Bs + (bn + 16 * u) * GBS + bk) = xb[u];
        __syncthreads();
        if (k0 + GK < khi) gload(k0 + GK);
#pragma unroll
        for (int u = 0; u < 16; u += 8) {
            float x[8], y[2][8];
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                x[t] = As[(4 * (u + t) + k) * GAS + wm + q];
                y[0][t] = Bs[(wn + q) * GBS + 4 * (u + t) + k];
                y[1][t] = Bs[(wn + 16 + q) * GBS + 4 * (u + t) + k];
            }
#pragma unroll
            for (int t = 0; t < 8; ++t)
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    if constexpr (sizeof(T) == 8)
                        acc[b] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)y[b][t], (double)x[t], acc[b], 0, 0, 0);
                    else
                        acc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(y[b][t], x[t], acc[b], 0, 0, 0);
                }
        }
        __syncthreads();
    }
    // lane (q, k)'s register e of acc[b]: row wm + q, column wn + 16 b + 4e + k
    // (FP32: 4k + e)
    float* C = g.C + q_ * g.sC + I * g.tC;
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int m = m0 + wm + q, n = n0 + (sizeof(T) == 8 ? 4 * e + k : 4 * k + e) + wn + 16 * b, nn = n - n0;
            const float v = (float)((T)g.alpha * acc[b][e]);
            if (m < g.m && n < g.n) C[m + (int64_t)n * g.ldc] = v;
            if (g.CT) Bs[nn * GBS + wm + q] = v;
        }
    if (!g.CT) return;
    __syncthreads();
    float* CT = g.CT + q_ * g.sC + I * g.tC;
    for (int idx = tid; idx < GM * GN; idx += 256) {
        const int nn = idx & (GN - 1), mm = idx / GN;
        if (m0 + mm < g.m && n0 + nn < g.n) CT[n0 + nn + (int64_t)(m0 + mm) * g.ldc] = Bs[nn * GBS + mm];
    }
}

// ---------------------------------------------------------------- TRSV kernels
// Both sweeps are left-looking: the update a big block receives from the
// blocks solved before it is one GEMV over all of them, then the block's
// inverse is applied.  Where the columns of a matrix are the outputs (backward,
// and both inverses: W and its transpose are stored) a wave owns whole columns,
// so nothing is left to add up afterwards.  The forward GEMV, whose outputs are
// rows, is split into many workgroups with partial sums in a fixed order.
constexpr int NR = 4;       // right-hand sides per pass
// forward: columns per split (4 waves x FW_CPW).  At n = 16384 (Bo = 2048)
// 128 beat 64, 256 and 512: more workgroups with fewer loads in flight each.
constexpr int FW_CW = 128;
constexpr int FW_CPW = FW_CW / 4;
constexpr int BW_CPW = 8;   // backward by partial sums: columns per wave (32 per workgroup)
constexpr int BW_RW = 512;  // and rows per split (BW_RPL per lane)
constexpr int BW_RPL = BW_RW / 64;
constexpr int TD = 2048;    // most columns of a big block
constexpr int BW_CH = 1024; // backward: rows at a time

// Forward, big block I = rows [p0, p0 + bI):
//   part[(s nrhs + j) bI + i] = sum_{c in split s} L[p0 + i][c] Y[c][j],  c < p0
// 64 rows per workgroup (lane = row: each column load is a 256-byte
// segment), split s = FW_CW columns, wave w its FW_CPW of them, all loads of
// a lane in flight before the first product; the split's Y values are staged
// in LDS and read back by all lanes at once.
__global__ __launch_bounds__(256) void fwd_gemv_partial_kernel(
    const float* __restrict__ L, int64_t ldl, int64_t p0, int bI, const double* __restrict__ Y,
    int64_t ldy, int nrhs, double* __restrict__ part) {
    __shared__ double red[4][NR][64];
    __shared__ double ys[NR][FW_CW];        // the split's Y values, read back broadcast
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int i = blockIdx.x * 64 + lane;
    const int ic = i < bI ? i : bI - 1;
    const int sp = blockIdx.y;
    const int64_t cs = (int64_t)sp * FW_CW;
    const float* Lr = L + (p0 + ic);
    float l[FW_CPW];
#pragma unroll
    for (int u = 0; u < FW_CPW; ++u) {
        const int64_t c = cs + wave * FW_CPW + u;
        const float x = Lr[(c < p0 ? c : p0 - 1) * ldl];     // clamped, then masked
        l[u] = c < p0 ? x : 0.f;
    }
#pragma unroll
    for (int q = 0; q < NR * FW_CW / 256; ++q) {
        const int idx = tid + 256 * q, j = idx / FW_CW, cc = idx % FW_CW;
        const int64_t c = cs + cc;
        const int jj = j < nrhs ? j : nrhs - 1;
        const double v = Y[(int64_t)jj * ldy + (c < p0 ? c : p0 - 1)];
        ys[j][cc] = (j < nrhs && c < p0) ? v : 0.0;
    }
    __syncthreads();
    double acc[NR];
#pragma unroll
    for (int j = 0; j < NR; ++j) {
        double a0 = 0.0, a1 = 0.0;
        if (j < nrhs) {
#pragma unroll
            for (int u = 0; u < FW_CPW; u += 2) {
                a0 = fma((double)l[u], ys[j][wave * FW_CPW + u], a0);
                a1 = fma((double)l[u + 1], ys[j][wave * FW_CPW + u + 1], a1);
            }
        }
        acc[j] = a0 + a1;
    }
#pragma unroll
    for (int j = 0; j < NR; ++j) red[wave][j][lane] = acc[j];
    __syncthreads();
    if (wave == 0 && i < bI) {
#pragma unroll
        for (int j = 0; j < NR; ++j)
            if (j < nrhs)
                part[((int64_t)sp * nrhs + j) * bI + i] =
                    ((red[0][j][lane] + red[1][j][lane]) + red[2][j][lane]) + red[3][j][lane];
    }
}

// Backward with 3 or 4 right-hand sides, big block I = columns [p0, p0 + bI),
// rows below it [p1, n):
//   part[(s nrhs + j) bI + c] = sum_{r in split s} L[r][p0 + c] X[r][j]
// 32 columns per workgroup (8 per wave), split s = BW_RW rows; lane k of a
// wave holds rows lane + 64k, k < BW_RPL, of each of its columns (coalesced
// 256-byte loads, 8 BW_RPL in flight), then the 64 lane sums of a column are added through
// LDS: lane t sums 8 of column t/8's, three shuffle steps finish it.
__global__ __launch_bounds__(256) void bwd_gemv_partial_kernel(
    const float* __restrict__ L, int64_t ldl, int64_t p0, int bI, int64_t n,
    const double* __restrict__ X, int64_t ldx, int nrhs, double* __restrict__ part) {
    __shared__ double buf[4][BW_CPW][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t p1 = p0 + bI;
    const int sp = blockIdx.y;
    const int64_t rs = p1 + (int64_t)sp * BW_RW;
    const int c0 = blockIdx.x * (4 * BW_CPW) + wave * BW_CPW;
    float l[BW_CPW][BW_RPL];
#pragma unroll
    for (int cc = 0; cc < BW_CPW; ++cc) {
        const int c = c0 + cc < bI ? c0 + cc : bI - 1;
        const float* col = L + (p0 + c) * ldl;
#pragma unroll
        for (int k = 0; k < BW_RPL; ++k) {
            const int64_t r = rs + lane + 64 * k;
            l[cc][k] = col[r < n ? r : n - 1];
        }
    }
#pragma unroll
    for (int j = 0; j < NR; ++j) {
        if (j < nrhs) {
            const double* x = X + (int64_t)j * ldx;
            double xv[BW_RPL];
#pragma unroll
            for (int k = 0; k < BW_RPL; ++k) {
                const int64_t r = rs + lane + 64 * k;
                const double v = x[r < n ? r : n - 1];
                xv[k] = r < n ? v : 0.0;                     // rows beyond n weigh nothing
            }
#pragma unroll
            for (int cc = 0; cc < BW_CPW; ++cc) {
                double a = 0.0;
#pragma unroll
                for (int k = 0; k < BW_RPL; ++k) a = fma((double)l[cc][k], xv[k], a);
                buf[wave][cc][lane] = a;
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            const int col = lane >> 3, q = lane & 7;
            double v = 0.0;
#pragma unroll
            for (int t = 0; t < 8; ++t) v += buf[wave][col][8 * q + t];
            v += __shfl_xor(v, 1);
            v += __shfl_xor(v, 2);
            v += __shfl_xor(v, 4);
            if (q == 0 && c0 + col < bI)
                part[((int64_t)sp * nrhs + j) * bI + c0 + col] = v;
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();                 // buf is rewritten next
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
    }
}

typedef float v4u __attribute__((ext_vector_type(4), aligned(4)));     // 16-byte load, any column start
typedef double d2 __attribute__((ext_vector_type(2)));

// Where 256 values that lane l reads as 4l .. 4l+3 lie in LDS: 4l and 4l+1 of
// all lanes in a row, then 4l+2 and 4l+3 (two 16-byte reads without conflicts)
__device__ __forceinline__ int dot_slot(int x) { return (x & 2) * 64 + (x >> 2) * 2 + (x & 1); }

// Backward, big block I = columns [p0, p0 + bI), rows below it [p1, n):
//   v[j bI + c] = V[j ldv + c] - sum_{r >= p1} L[r][p0 + c] X[j][r]
// A column per wave, BW_CH rows at a time: lane l reads rows 4l .. 4l+3 of
// every 256 (16 bytes), the next rows' loads in flight during the products; the
// workgroup shares the rows' X values through LDS.  Bound by memory (n = 16384,
// one right-hand side: 14.9 us on average for 59 MB); two columns a wave are
// too few workgroups (20.7), 2048 rows at a time the same for long columns and
// slower for short ones (n = 8684: 9.3 / 10.8).  Two right-hand sides take 17.0;
// with four the X values are the larger part (28 us, n = 60000 89, where the
// partial sums above and their addition take 67).
template <int NJ>
__global__ __launch_bounds__(256, 2) void bwd_dot_kernel(const float* __restrict__ L, int64_t ldl,
                                                        int64_t p0, int bI, int64_t n,
                                                        const double* __restrict__ X, int64_t ldx,
                                                        int nj, const double* __restrict__ V,
                                                        int64_t ldv, double* __restrict__ v) {
    constexpr int NK = BW_CH / 256;
    __shared__ __align__(16) double xs[NJ][BW_CH];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int c = blockIdx.x * 4 + wave;
    const float* col = L + (p0 + (c < bI ? c : bI - 1)) * ldl;
    v4f l[NK];
    double x[NJ][NK];
    auto load = [&](int64_t rs) {
        if (rs + BW_CH <= n) {
#pragma unroll
            for (int k = 0; k < NK; ++k)
                l[k] = *reinterpret_cast<const v4u*>(col + rs + 256 * k + 4 * lane);
        } else {
            // the last rows: loads that end at row n at the latest (n > Bo >= 4
            // where there are rows below a block), moved into place
#pragma unroll
            for (int k = 0; k < NK; ++k) {
                const int64_t r = rs + 256 * k + 4 * lane, rc = r < n - 4 ? r : n - 4, off = r - rc;
                const v4f y = *reinterpret_cast<const v4u*>(col + rc);
                l[k][0] = off == 0 ? y[0] : off == 1 ? y[1] : off == 2 ? y[2] : off == 3 ? y[3] : 0.f;
                l[k][1] = off == 0 ? y[1] : off == 1 ? y[2] : off == 2 ? y[3] : 0.f;
                l[k][2] = off == 0 ? y[2] : off == 1 ? y[3] : 0.f;
                l[k][3] = off == 0 ? y[3] : 0.f;
            }
        }
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int k = 0; k < NK; ++k) {
                const int64_t r = rs + 256 * k + tid;
                const double y = X[(int64_t)(j < nj ? j : nj - 1) * ldx + (r < n ? r : n - 1)];
                x[j][k] = r < n ? y : 0.0;
            }
    };
    double acc[NJ] = {};
    int64_t rs = p0 + bI;
    load(rs);
    for (; rs < n; rs += BW_CH) {
        v4f w[NK];
#pragma unroll
        for (int k = 0; k < NK; ++k) w[k] = l[k];
        __syncthreads();                         // the last rows' values are read
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int k = 0; k < NK; ++k) xs[j][256 * k + dot_slot(tid)] = x[j][k];
        __syncthreads();
        if (rs + BW_CH < n) load(rs + BW_CH);
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int k = 0; k < NK; ++k)
#pragma unroll
                for (int i = 0; i < 4; i += 2) {
                    const d2 y = *reinterpret_cast<const d2*>(&xs[j][256 * k + 64 * i + 2 * lane]);
                    acc[j] = fma((double)w[k][i], y[0], acc[j]);
                    acc[j] = fma((double)w[k][i + 1], y[1], acc[j]);
                }
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const double sum = mpc_sum64(acc[j]);
        if (lane == 0 && j < nj && c < bI) v[(int64_t)j * bI + c] = V[(int64_t)j * ldv + c] - sum;
    }
}

// v[j bI + i] = V[j ldv + i] - sum_s part[(s nj + j) bI + i] (a GEMV's partial
// sums); wave w of a workgroup adds s = w, w + 4, .. of 64 rows
__global__ __launch_bounds__(256) void gemv_sum_kernel(const double* __restrict__ part, int bI, int S,
                                                     const double* __restrict__ V, int64_t ldv,
                                                     double* __restrict__ v) {
    __shared__ double red[4][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int i0 = blockIdx.x * 64 + lane, i = i0 < bI ? i0 : bI - 1;
    const int j = blockIdx.y, nj = gridDim.y;
    double sum = 0.0;
    for (int s0 = w; s0 < S; s0 += 64) {
        double x[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const int s = s0 + 4 * u < S ? s0 + 4 * u : S - 1;
            x[u] = part[((int64_t)s * nj + j) * bI + i];
        }
#pragma unroll
        for (int u = 0; u < 16; ++u) sum += s0 + 4 * u < S ? x[u] : 0.0;
    }
    red[w][lane] = sum;
    __syncthreads();
    if (w == 0 && i0 < bI)
        v[(int64_t)j * bI + i0] = V[(int64_t)j * ldv + i0] -
                                  (((red[0][lane] + red[1][lane]) + red[2][lane]) + red[3][lane]);
}

// A big block's inverse applied: out[r] = sum_c Mt[c + r ld] v[c] over c <= r
// (forward, Mt = Winv^T) or c >= r (backward, Mt = Winv), r, c < bI.  A wave
// owns an output: its column of Mt (16-byte loads, all in flight at once, a
// 256-row piece outside the triangle replaced by its neighbour) times v from
// LDS.  bI = 2048, one right-hand side 5.3 us, four 7.0 (two outputs a wave 6.0
// and 7.6; 64 x 64 tiles over rows of M and a launch to add them up 10 and 15).
// blockIdx.y: NJ of the right-hand sides.
template <bool UPPER, int NJ>
__global__ __launch_bounds__(256, 2) void tri_dot_kernel(const float* __restrict__ Mt, int ld, int bI,
                                                        const double* __restrict__ V, int64_t ldv,
                                                        int nj, double* __restrict__ out, int64_t ldo) {
    constexpr int NK = TD / 256;
    __shared__ __align__(16) double vs[NJ][TD];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r = blockIdx.x * 4 + wave;
    const int kd = r >> 8;                       // the diagonal's 256-row piece
    const int klo = UPPER ? kd : 0, khi = UPPER ? (bI - 1) >> 8 : kd;
    v4f m[NK];
    const float* col = Mt + (int64_t)(r < bI ? r : bI - 1) * ld;
    V += (int64_t)blockIdx.y * NJ * ldv;
    out += (int64_t)blockIdx.y * NJ * ldo;
    nj -= blockIdx.y * NJ;
#pragma unroll
    for (int k = 0; k < NK; ++k) {
        const int c = 256 * (k < klo ? klo : k > khi ? khi : k) + 4 * lane;
        m[k] = *reinterpret_cast<const v4f*>(col + (c < ld ? c : ld - 4));
    }
    for (int c = 256 * klo + tid; c < 256 * (khi + 1); c += 256)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
            vs[j][(c & ~255) + dot_slot(tid)] = V[(int64_t)(j < nj ? j : nj - 1) * ldv + (c < bI ? c : bI - 1)];
    __syncthreads();
    double acc[NJ] = {};
#pragma unroll
    for (int k = 0; k < NK; ++k) {
        if (k < klo || k > khi) continue;
#pragma unroll
        for (int i = 0; i < 4; i += 2) {
            double w[2];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int c = 256 * k + 4 * lane + i + u;
                w[u] = (UPPER ? c >= r && c < bI : c <= r) ? (double)m[k][i + u] : 0.0;
            }
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const d2 y = *reinterpret_cast<const d2*>(&vs[j][256 * k + 64 * i + 2 * lane]);
                acc[j] = fma(w[1], y[1], fma(w[0], y[0], acc[j]));
            }
        }
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const double sum = mpc_sum64(acc[j]);
        if (lane == 0 && j < nj && r < bI) out[(int64_t)j * ldo + r] = sum;
    }
}

inline unsigned cdiv(int64_t a, int64_t b) { return (unsigned)((a + b - 1) / b); }

int launch_gemm(hipStream_t st, const gemm_batch& g, int nbatch, bool f64) {
    const dim3 grid(cdiv(g.m, GM), cdiv(g.n, GN), (unsigned)nbatch);
    if (f64) hipLaunchKernelGGL(gemm_kernel<double>, grid, dim3(256), 0, st, g);
    else hipLaunchKernelGGL(gemm_kernel<float>, grid, dim3(256), 0, st, g);
    MPC_LAUNCH_CHECK();
    return 0;
}

}  // namespace

// Winv_I = L_II^{-1} for a big block (Bo x Bo, column-major, ld Bo, block I at
// W + I*Bo*Bo) and WT_I = Winv_I^T come from L and its 32x32 diagonal inverses,
// 128 x 128 blocks first, then by doubling: for the pairs q0 .. q0 + nq - 1 of
// blocks of h rows (the second of them with hc <= h rows) of nblk big blocks
//   T = B A^-1 (kept in the upper part at (p, p + h)), X21 = -C^-1 T at (p + h, p).
static int double_first(hipStream_t st, const float* L, int64_t ldl, int Bo, float* W, int h, int64_t I0,
                        int nblk, int q0, int nq, int hc, bool f64) {
    const int64_t base = I0 * Bo;
    const int64_t p = 2 * (int64_t)h * q0;
    float* Wi = W + I0 * (int64_t)Bo * Bo;
    gemm_batch g;
    g.A = L + (base + p + h) + (base + p) * ldl;  g.lda = ldl;
    g.B = Wi + p + p * (int64_t)Bo;              g.ldb = Bo;
    g.C = Wi + p + (p + h) * (int64_t)Bo;        g.ldc = Bo;
    g.CT = nullptr;
    g.sA = 2 * (int64_t)h * (1 + ldl);
    g.sB = g.sC = 2 * (int64_t)h * (1 + Bo);
    g.tA = (int64_t)Bo * (1 + ldl);
    g.tB = g.tC = (int64_t)Bo * Bo;
    g.nq = nq;
    g.m = hc; g.n = h; g.k = h; g.alpha = 1.f; g.a_lower = 0; g.b_lower = 1;
    return launch_gemm(st, g, nq * nblk, f64);
}
static int double_second(hipStream_t st, int Bo, float* W, float* WT, int h, int64_t I0, int nblk, int q0,
                         int nq, int hc, bool f64) {
    const int64_t p = 2 * (int64_t)h * q0, bs = (int64_t)Bo * Bo;
    float* Wi = W + I0 * bs;
    gemm_batch g;
    g.A = Wi + (p + h) + (p + h) * (int64_t)Bo;  g.lda = Bo;
    g.B = Wi + p + (p + h) * (int64_t)Bo;        g.ldb = Bo;
    g.C = Wi + (p + h) + p * (int64_t)Bo;        g.ldc = Bo;
    g.CT = WT + I0 * bs + p + (p + h) * (int64_t)Bo;
    g.sA = g.sB = g.sC = 2 * (int64_t)h * (1 + Bo);
    g.tA = g.tB = g.tC = bs;
    g.nq = nq;
    g.m = hc; g.n = h; g.k = hc; g.alpha = -1.f; g.a_lower = 1; g.b_lower = 0;
    return launch_gemm(st, g, nq * nblk, f64);
}

static int leaves(hipStream_t st, const float* L, int64_t ldl, int64_t n, int Bo, const float* dinv,
                  float* W, float* WT, int64_t b0, int64_t b1) {
    if (b1 > b0)
        hipLaunchKernelGGL(winv_leaf_kernel, dim3((unsigned)(b1 - b0)), dim3(256), 0, st, L, ldl, dinv, n,
                           Bo, W, WT, b0);
    MPC_LAUNCH_CHECK();
    return 0;
}

int mpc_build_block_inverse_stage(hipStream_t st, const float* L, int64_t ldl, int64_t n, int Bo,
                                  const float* dinv, float* W, float* WT, int64_t I, int64_t from,
                                  int64_t to) {
    const int64_t rows = std::min<int64_t>(Bo, n - I * Bo);
    if (Bo % LF || Bo < LF || from % LF || from < 0 || to > rows || (to < rows && to % LF)) {
        mpc_set_error("block inverse: rows %lld to %lld of %lld, block %d", (long long)from, (long long)to,
                      (long long)rows, Bo);
        return MPC_ERR_ARG;
    }
    const bool f64 = n <= 8192;
    int rc = leaves(st, L, ldl, n, Bo, dinv, W, WT, I * (Bo / LF) + from / LF, I * (Bo / LF) + cdiv(to, LF));
    if (rc) return rc;
    for (int h = LF; h < Bo; h *= 2) {
        // pairs whose first (second) half ends in (from, to]: q with
        // from < 2 h q + h <= to, and from < min(2 h q + 2 h, rows) <= to
        int f0 = -1, f1 = 0, s0 = -1, s1 = 0;
        for (int q = 0; 2 * (int64_t)h * q + h < rows; ++q) {
            const int64_t a = 2 * (int64_t)h * q + h, c = std::min<int64_t>(a + h, rows);
            if (a > from && a <= to) { if (f0 < 0) f0 = q; f1 = q + 1; }
            if (c > from && c <= to) { if (s0 < 0) s0 = q; s1 = q + 1; }
        }
        // (the last pair of the block on its own where its second half is short)
        auto each = [&](int q0, int q1, auto&& run) -> int {
            if (q0 < 0) return 0;
            const int64_t lastc = rows - (2 * (int64_t)h * (q1 - 1) + h);
            const int full = lastc >= h ? q1 : q1 - 1;
            int r = 0;
            if (full > q0) r = run(q0, full - q0, h);
            if (!r && full < q1) r = run(full, 1, (int)lastc);
            return r;
        };
        if ((rc = each(f0, f1, [&](int q, int nq, int hc) {
                 return double_first(st, L, ldl, Bo, W, h, I, 1, q, nq, hc, f64);
             })))
            return rc;
        if ((rc = each(s0, s1, [&](int q, int nq, int hc) {
                 return double_second(st, Bo, W, WT, h, I, 1, q, nq, hc, f64);
             })))
            return rc;
    }
    return 0;
}

// Big blocks [I0, I1) only (each depends on L_II and the 32x32 inverses of
// its diagonal alone, so blocks can be built as soon as they are factored).
// Full big blocks are batched per level.
int mpc_build_block_inverses_range(hipStream_t st, const float* L, int64_t ldl, int64_t n, int Bo,
                                   const float* dinv, float* W, float* WT, int64_t I0,
                                   int64_t I1) {
    if (Bo % LF || Bo < LF) {
        mpc_set_error("block inverse: Bo must be a multiple of %d", LF);
        return MPC_ERR_ARG;
    }
    const int64_t nI = (n + Bo - 1) / Bo, f1 = std::min(I1, n / Bo);     // full blocks: [I0, f1)
    const bool f64 = n <= 8192;
    int rc;
    if (f1 > I0) {
        if ((rc = leaves(st, L, ldl, n, Bo, dinv, W, WT, I0 * (Bo / LF), f1 * (Bo / LF)))) return rc;
        for (int h = LF; h < Bo; h *= 2) {
            const int pairs = Bo / (2 * h);
            if ((rc = double_first(st, L, ldl, Bo, W, h, I0, (int)(f1 - I0), 0, pairs, h, f64)) ||
                (rc = double_second(st, Bo, W, WT, h, I0, (int)(f1 - I0), 0, pairs, h, f64)))
                return rc;
        }
    }
    if (nI > n / Bo && n / Bo >= I0 && n / Bo < I1)                      // ragged last big block
        return mpc_build_block_inverse_stage(st, L, ldl, n, Bo, dinv, W, WT, n / Bo, 0, n % Bo);
    return 0;
}

int mpc_build_block_inverses(hipStream_t st, const float* L, int64_t ldl, int64_t n, int Bo,
                             const float* dinv, float* W, float* WT) {
    return mpc_build_block_inverses_range(st, L, ldl, n, Bo, dinv, W, WT, 0, (n + Bo - 1) / Bo);
}

static int tri_dot(hipStream_t st, const float* Mt, int Bo, int bI, bool upper, const double* V,
                   int64_t ldv, int nj, double* out, int64_t ldo) {
    const dim3 g(cdiv(bI, 4), cdiv(nj, NR)), b(256);
#define MPC_TRI_DOT(U, J) \
    hipLaunchKernelGGL((tri_dot_kernel<U, J>), g, b, 0, st, Mt, Bo, bI, V, ldv, nj, out, ldo)
    if (upper) {
        if (nj == 1) MPC_TRI_DOT(true, 1);
        else if (nj == 2) MPC_TRI_DOT(true, 2);
        else MPC_TRI_DOT(true, 4);
    } else {
        if (nj == 1) MPC_TRI_DOT(false, 1);
        else if (nj == 2) MPC_TRI_DOT(false, 2);
        else MPC_TRI_DOT(false, 4);
    }
#undef MPC_TRI_DOT
    MPC_LAUNCH_CHECK();
    return 0;
}

static int bwd_gemv(hipStream_t st, const float* L, int64_t ldl, int64_t p0, int bI, int64_t n,
                   const double* X, int64_t ldx, int nj, const double* V, int64_t ldv, double* v,
                    double* part) {
    const dim3 g(cdiv(bI, 4)), b(256);
    if (nj > 2) {
        const unsigned S = cdiv(n - p0 - bI, BW_RW);
        hipLaunchKernelGGL(bwd_gemv_partial_kernel, dim3(cdiv(bI, 4 * BW_CPW), S), b, 0, st, L, ldl, p0,
                           bI, n, X, ldx, nj, part);
        hipLaunchKernelGGL(gemv_sum_kernel, dim3(cdiv(bI, 64), (unsigned)nj), b, 0, st, part, bI, (int)S,
                           V, ldv, v);
    } else if (nj == 2) {
        hipLaunchKernelGGL(bwd_dot_kernel<2>, g, b, 0, st, L, ldl, p0, bI, n, X, ldx, nj, V, ldv, v);
    } else {
        hipLaunchKernelGGL(bwd_dot_kernel<1>, g, b, 0, st, L, ldl, p0, bI, n, X, ldx, nj, V, ldv, v);
    }
    MPC_LAUNCH_CHECK();
    return 0;
}

// Right-hand sides of the next pass over the factor: at most NR in the GEMV
// kernels above, on the matrix cores as many as kPass keeps the partial sums
// small for (40 MB at most).  A pass for every MPC_MM_NJ of them repeats a stage's
// launches and leaves the chip idle between them (applications with 33 columns, us,
// in passes of 16 and in one: n = 128 65 and 37, 2049 163 and 99, 6200 426 and 303,
// 16000 1313 and 1059).
constexpr int kPass = 64;
// Up to kDotRows rows (one block, no product beside it) the triangles of any number
// of right-hand sides go by column dots, two launches instead of four: n = 65, 16
// columns, 30 us and 40; 200, 64 columns 34 and 39; 300 39 and 40; 1000 68 and 52.
constexpr int64_t kDotRows = 256;
static int sweep_pass(int nrhs) { return std::min(nrhs, kPass); }

// Chunks of the products with a big block's rows: two workgroups a CU (2048
// rows, 16 right-hand sides: the triangle 7.2 us, 9.7 with three or four; 2048 /
// 4096 / 6144 columns beside it 8 / 11.5 / 15 us, with eight 10.6 / 22 / 22)
static int64_t mm_splits(int64_t bI, int64_t kc) { return mpc_mm_splits(bI, kc, 512); }

// chunks of a product with at most Bo output rows, in units of Bo partial sums:
// the chunks of bI < Bo rows take at most bI rounded up to a row block times
// 512 / blocks or one a column group, no more than those of Bo rows
static int64_t mm_chunks(int Bo, int64_t kc) {
    return std::max(mm_splits(Bo, kc), mpc_mm_splits_t(Bo, kc)) + 1;
}

// scratch of a pass: GEMV kernels: v, then the off-diagonal product's partial
// sums (over fewer than n columns, or n rows); matrix cores: the triangular product's partial sums, v,
// the off-diagonal one's
int64_t mpc_block_prec_partial_doubles(int64_t n, int Bo, int nrhs) {
    const int64_t gemv = (1 + (n + FW_CW - 1) / FW_CW) * Bo * std::min(nrhs, NR);
    if (nrhs <= NR) return gemv;
    return std::max(gemv, (mm_chunks(Bo, n) + mm_chunks(Bo, Bo) + 1) * Bo * sweep_pass(nrhs));
}

// One stage on the matrix cores: v = R_I - (sum of the S chunks of the off-
// diagonal product in gpart), out_I = M v with the triangular M (mode 1 lower,
// 2 upper).
static int mm_stage(hipStream_t st, const float* M, int Bo, int bI, int mode, const double* V,
                    int64_t ld, int nj, const double* gpart, int64_t kc, int64_t S, int unit,
                    double* v, double* tpart, double* out) {
    int rc;
    if (kc > 0) {
        if ((rc = mpc_launch_mm_sum(st, bI, nj, kc, S, 0, unit, gpart, V, ld, -1.0, v, bI))) return rc;
        V = v;
    }
    const int64_t St = mm_splits(bI, bI);
    if ((rc = mpc_launch_mm_n(st, M, Bo, bI, bI, mode, V, kc > 0 ? bI : ld, nj, tpart, St))) return rc;
    return mpc_launch_mm_sum(st, bI, nj, bI, St, mode, MPC_MM_GROUP_N, tpart, nullptr, 0, 1.0, out, ld);
}

// z = L^{-T} L^{-1} r for nrhs columns: R (in), Y (forward result), Z (out).
// late_ev (optional): the stream waits for it before the first use of big
// block I_late's inverse (which may still be in the making).
int mpc_apply_block_prec(hipStream_t st, const float* L, int64_t ldl, int64_t n, int Bo,
                         const float* Winv, const float* WinvT, const double* R, double* Y,
                         double* Z, int64_t ld, int nrhs, double* part, hipEvent_t late_ev,
                         int64_t I_late) {
    const int64_t nI = (n + Bo - 1) / Bo;
    int rc;
    for (int j0 = 0, nj; j0 < nrhs; j0 += nj, R += nj * ld, Y += nj * ld, Z += nj * ld) {
        nj = sweep_pass(nrhs - j0);
        const bool mm = nj > NR && n > kDotRows;
        double* v = part + (mm ? mm_chunks(Bo, Bo) * Bo * nj : 0);
        double* gpart = v + (int64_t)Bo * nj;
        for (int64_t I = 0; I < nI; ++I) {
            const int64_t p0 = I * Bo;
            const int bI = (int)(n - p0 < Bo ? n - p0 : Bo);
            const int64_t S = mm ? mm_splits(bI, p0) : cdiv(p0, FW_CW);
            if (p0 > 0 && mm) {
                if ((rc = mpc_launch_mm_n(st, L + p0, ldl, bI, p0, 0, Y, ld, nj, gpart, S))) return rc;
            } else if (p0 > 0) {
                hipLaunchKernelGGL(fwd_gemv_partial_kernel, dim3(cdiv(bI, 64), (unsigned)S), dim3(256), 0,
                                   st, L, ldl, p0, bI, Y, ld, nj, gpart);
                hipLaunchKernelGGL(gemv_sum_kernel, dim3(cdiv(bI, 64), (unsigned)nj), dim3(256), 0, st,
                                   gpart, bI, (int)S, R + p0, ld, v);
            }
            if (late_ev && j0 == 0 && I == I_late && hipStreamWaitEvent(st, late_ev, 0) != hipSuccess) {
                mpc_set_error("apply_block_prec: stream wait failed");
                return MPC_ERR_HIP;
            }
            const int64_t wI = I * (int64_t)Bo * Bo;
            rc = mm ? mm_stage(st, Winv + wI, Bo, bI, 1, R + p0, ld, nj, gpart, p0, S, MPC_MM_GROUP_N, v, part, Y + p0)
                    : tri_dot(st, WinvT + wI, Bo, bI, false, p0 ? v : R, p0 ? bI : ld, nj, Y + p0, ld);
            if (rc) return rc;
        }
        for (int64_t I = nI - 1; I >= 0; --I) {
            const int64_t p0 = I * Bo;
            const int bI = (int)(n - p0 < Bo ? n - p0 : Bo);
            const int64_t p1 = p0 + bI, wI = I * (int64_t)Bo * Bo;
            const bool off = p1 < n;
            if (mm) {
                const int64_t S = mpc_mm_splits_t(bI, n - p1);
                if (off && (rc = mpc_launch_mm_t(st, L + p1 + p0 * ldl, ldl, n - p1, bI, Z + p1, ld, nj, gpart, S)))
                    return rc;
                rc = mm_stage(st, WinvT + wI, Bo, bI, 2, Y + p0, ld, nj, gpart, n - p1, S, MPC_MM_GROUP_T, v, part, Z + p0);
            } else {
                if (off && (rc = bwd_gemv(st, L, ldl, p0, bI, n, Z, ld, nj, Y + p0, ld, v, gpart))) return rc;
                rc = tri_dot(st, Winv + wI, Bo, bI, true, off ? v : Y + p0, off ? bI : ld, nj, Z + p0, ld);
            }
            if (rc) return rc;
        }
    }
    MPC_LAUNCH_CHECK();
    return 0;
}
