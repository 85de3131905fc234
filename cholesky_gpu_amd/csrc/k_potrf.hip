// k_potrf.hip -- FP32 Cholesky of one diagonal block (bs <= 256) in a single
// workgroup, plus the inverses of its 32x32 diagonal sub-blocks.
//
// Replaces the cusolverDnSpotrf call of switching_chol.cuh:86-95 (CPU form:
// micro_cholesky, micro_chol.hpp:14-44).  One wave per 32-row block row, whose
// 32x32 tiles stay in registers from the first load to the last store; the
// waves work through the columns four at a time ("panels") and hand panels to
// each other through LDS:
//   - the wave of block row kb, its diagonal tile up to date, factors that
//     tile (factor_tile: a 4x4 Cholesky on broadcast scalars, the four columns
//     of every row by substitution, the rank-4 update of the rest by MFMA
//     32x32x2 f32) and runs the same row operations on the identity, which
//     leaves the inverse; each panel is published as it is done;
//   - the waves below follow panel by panel: they substitute their own rows of
//     block column kb with the published 4x4 factor and update that tile and
//     their diagonal tile, so that wave kb+1 can go on with block column kb+1
//     about one panel after wave kb has finished;
//   - their other tiles get block column kb as one rank-32 update when the
//     rows they need are published.
// There is no workgroup barrier after the start: a wave waits for a count of
// panels of one other wave, always of a smaller block row, so every wait ends.
// Every published panel has an LDS slot of its own (no slot is written twice).
//
// Bound: the chain of bs/4 panels, each about 110 dependent or nearly
// dependent instructions of one wave; the matrix cores carry the updates
// beside it.  Alone 13 us at bs = 128 and 37 at 256; with the tiles in LDS, a
// column at a time and a barrier per sub-block it took 35 and 70 (n = 3001 solve
// 2704 -> 2231 us, n = 16384 E4M3 14897 -> 13752).
// Outputs: L in place (lower; the strict upper triangle of A is untouched),
// dinv (column-major 32x32 inverse per sub-block), the running minimum pivot
// squared and, on a non-positive pivot, the 1-based failing column.
#include "mpc_internal.hpp"
#include <climits>

namespace {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v2f __attribute__((ext_vector_type(2)));

__host__ __device__ constexpr int sidx(int bi, int bj) { return bi * (bi + 1) / 2 + bj; }

// column (or row) of accumulator register i in lane half h (32x32 MFMA output)
__device__ __forceinline__ int sig(int i, int h) { return 8 * (i >> 2) + 4 * h + (i & 3); }

__device__ __forceinline__ float rdlane(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// MFMA operand of two columns x, y that are valid in lane half hp (lane n of
// that half: row n): half 0 of the result holds x, half 1 holds y
__device__ __forceinline__ float pair_op(float x, float y, int hp) {
    const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false,
                                                    false);
    return __uint_as_float(hp ? p[1] : p[0]);
}

// 1 / sqrt(p) from the hardware estimate and one Newton step (about 1 ulp): a
// short dependent chain, where a correctly rounded square root and reciprocal
// take four times the instructions.  A pivot that is not positive counts as 1
// (the caller records it).
__device__ __forceinline__ float rsqrt_pivot(float p) {
    const float r = __builtin_amdgcn_rsqf(p);
    const float hr = 0.5f * p * r;
    const float q = fmaf(fmaf(-hr, r, 0.5f), r, r);
    return p > 0.f ? q : 1.f;
}

__device__ __forceinline__ v16f mfma2(float a, float b, v16f c) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// The length of a 32x32 product, spent without an instruction at issue: a
// product issued while the last one still runs holds up the vector
// instructions of the other wave of the SIMD, which may be the chain
__device__ __forceinline__ void idle_pass() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_nop 11");
    __builtin_amdgcn_sched_barrier(0);
}

// smallest value of each 16 lanes, in all of them (rotations within the 16)
template <class F>
__device__ __forceinline__ uint32_t reduce16(uint32_t v, F f) {
    v = f(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x128, 0xf, 0xf, true));
    v = f(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x124, 0xf, 0xf, true));
    v = f(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x122, 0xf, 0xf, true));
    return f(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x121, 0xf, 0xf, true));
}

template <int NB>
struct shared_panels {
    // operands of the published panels: tile slot, panel, lane.  Slots: the
    // tiles (ib, kb) of block rows 0 .. NB-2, then the last diagonal tile (no
    // other wave reads the rest of the last row).
    v2f op[sidx(NB - 1, 0) + 1][8][64];
    v4f mic[NB][8][3];
    int prog[NB];               // panels published by a block row so far
    int done[NB];               // its summary below is written
    uint32_t pmin[NB];
    int fail[NB];               // 2 * first failing column + (pivot is NaN), or INT_MAX
    float f2[NB];
};

template <int NB>
__device__ __forceinline__ int diag_slot(int kb) {
    return kb < NB - 1 ? sidx(kb, kb) : sidx(NB - 1, 0);
}

__device__ __forceinline__ void wait_for(const int* count, int need, bool busy) {
    while (__hip_atomic_load(count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) < need)
        if (!busy) __builtin_amdgcn_s_sleep(1);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

__device__ __forceinline__ void publish(int* count, int value) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __hip_atomic_store(count, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Panel p of block column kb on the tile t (rows held negated, lane n: row n):
// t's four columns by substitution; own = their operand
template <int NB>
__device__ __forceinline__ void follow(const shared_panels<NB>& S, int kb, int p, v16f& t,
                                       v2f& own, v2f& lop) {
    const int hp = p & 1, i0 = 4 * (p >> 1);
    const int lane = threadIdx.x & 63, h = lane >> 5;
    const v4f* mp = S.mic[kb][p];
    const v4f q0 = mp[0], q1 = mp[1], q2 = mp[2];     // r0..r3, m10 m20 m30 m21, m31 m32
    if (p < 7) lop = S.op[diag_slot<NB>(kb)][p][lane];
    const float x0 = -t[i0] * q0[0];
    const float x1 = -fmaf(x0, q1[0], t[i0 + 1]) * q0[1];
    const float x2 = -fmaf(x1, q1[3], fmaf(x0, q1[1], t[i0 + 2])) * q0[2];
    const float x3 = -fmaf(x2, q2[1], fmaf(x1, q2[0], fmaf(x0, q1[2], t[i0 + 3]))) * q0[3];
    t[i0] = (h == hp) ? x0 : t[i0];
    t[i0 + 1] = (h == hp) ? x1 : t[i0 + 1];
    t[i0 + 2] = (h == hp) ? x2 : t[i0 + 2];
    t[i0 + 3] = (h == hp) ? x3 : t[i0 + 3];
    own = v2f{pair_op(x0, x1, hp), pair_op(x2, x3, hp)};
}

template <int NB>
__global__ __launch_bounds__(NB * 64, NB == 4 ? 4 : 2) void potrf_kernel(
    float* __restrict__ A, int64_t lda, int bs, int col0, float* __restrict__ dinv,
    mpc_small* __restrict__ sm, int ntiles_next, uint32_t* __restrict__ st_amax,
    uint32_t* __restrict__ st_maxrs, int mu_slot, int want_f2) {
    __shared__ __align__(16) shared_panels<NB> S;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // waves w and w + 4 share a SIMD: a long block row beside a short one
    const int row = wave < 4 ? wave : 11 - wave;
    const int nsb = (bs + 31) >> 5;
    const int n = lane & 31, h = lane >> 5;
    const int r = 32 * row + n;
    const bool last = row == nsb - 1;

    // Tiles of this block row, negated: lane (n, h) register i holds
    // -A(row n, column sig(i, h)).  Rows beyond bs (a store there is dropped,
    // a load gives 0) stand for the identity; entries above the diagonal
    // start as 0 and reach no other entry.  Addresses: one lane offset per
    // tile, the columns' in scalars.
    const __amdgpu_buffer_rsrc_t rsrc =
        __builtin_amdgcn_make_buffer_rsrc(A, 0, 0x7fffffff, 0x00020000);
    const uint32_t ld4 = 4u * (uint32_t)lda, none = 0x80000000u;
    const uint32_t vrow = r < bs ? 4u * (uint32_t)r + 4u * (uint32_t)h * ld4 : none;
    auto voff = [&](int cb, int i) -> uint32_t {
        return cb < row || sig(i, h) <= n ? vrow : none;
    };
    auto soff = [&](int cb, int i) -> uint32_t { return (uint32_t)(32 * cb + sig(i, 0)) * ld4; };
    auto load_tile = [&](int cb) -> v16f {
        v16f t;
#pragma unroll
        for (int i = 0; i < 16; ++i)
            t[i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rsrc, voff(cb, i),
                                                                        soff(cb, i), 0));
        return t;
    };
    auto store_tile = [&](int cb, const v16f& t) {
#pragma unroll
        for (int i = 0; i < 16; ++i)
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(t[i]), rsrc, voff(cb, i),
                                                  soff(cb, i), 0);
    };

    v16f cur, diag, rest[NB - 2];
    if (row < nsb) {
        diag = load_tile(row);
        if (row > 0) cur = load_tile(0);
#pragma unroll
        for (int j = 0; j < NB - 2; ++j)
            if (j + 1 < row) rest[j] = load_tile(j + 1);
    }
    const uint32_t mu_before = sm->mu_bits;
    if (sm->info != 0) return;                       // an earlier step failed
    for (int t = tid; t < ntiles_next; t += NB * 64) {
        st_amax[t] = 0u;
        st_maxrs[t] = 0u;
    }
    if (tid < NB) S.prog[tid] = S.done[tid] = 0;
    mpc_lds_barrier();
    if (row >= nsb) return;
#pragma unroll
    for (int i = 0; i < 16; ++i) diag[i] = (r >= bs && sig(i, h) == n) ? -1.f : -diag[i];
    cur = -cur;
#pragma unroll
    for (int j = 0; j < NB - 2; ++j)
        if (j + 1 < row) rest[j] = -rest[j];

    float f2 = 0.f;                  // this lane's part of ||L_jj||_F^2
    auto add_f2 = [&](int cb, const v16f& t) {
#pragma unroll
        for (int i = 0; i < 16; ++i)
            f2 = (r < bs && (cb < row || sig(i, h) <= n)) ? fmaf(t[i], t[i], f2) : f2;
    };
    for (int kb = 0; kb < row; ++kb) {
        const bool next = kb + 1 == row;             // the chain goes on here
        if (next) __builtin_amdgcn_s_setprio(2);
        // ---- block column kb, a panel behind its owner
        v2f own[8];
#pragma unroll
        for (int p = 0; p < 8; ++p) {
            v2f lop;
            wait_for(&S.prog[kb], 8 * kb + p + 1, next);
            follow<NB>(S, kb, p, cur, own[p], lop);
            diag = mfma2(own[p][0], own[p][0], diag);
            if (p < 7) cur = mfma2(lop[0], own[p][0], cur);
            diag = mfma2(own[p][1], own[p][1], diag);
            if (p < 7) cur = mfma2(lop[1], own[p][1], cur);
            if (row < NB - 1) S.op[sidx(row, kb)][p][lane] = own[p];
        }
        publish(&S.prog[row], 8 * kb + 8);
        if (next) break;                             // cur goes back after the chain
        store_tile(kb, cur);
        if (want_f2) add_f2(kb, cur);
        // ---- the tiles between: rank 32 at once, the next block columns
        // first; two at a time, as a product waits longer for the one before
        // it on the same tile than for the matrix core
#pragma unroll
        for (int j = 0; j < NB - 2; j += 2) {
            const int j0 = kb + 1 + j;
            if (j0 >= row) break;
            wait_for(&S.prog[j0], 8 * kb + 8, false);
            const v2f* q0 = &S.op[sidx(j0, kb)][0][lane];
            v2f o0[8], o1[8];
            if (j0 + 1 < row) {
                wait_for(&S.prog[j0 + 1], 8 * kb + 8, false);
                const v2f* q1 = &S.op[sidx(j0 + 1, kb)][0][lane];
#pragma unroll
                for (int p = 0; p < 8; ++p) {
                    o0[p] = q0[64 * p];
                    o1[p] = q1[64 * p];
                }
#pragma unroll
                for (int p = 0; p < 8; ++p)
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        idle_pass();
                        rest[j] = mfma2(o0[p][t], own[p][t], rest[j]);
                        idle_pass();
                        rest[j + 1] = mfma2(o1[p][t], own[p][t], rest[j + 1]);
                    }
            } else {
#pragma unroll
                for (int p = 0; p < 8; ++p) o0[p] = q0[64 * p];
#pragma unroll
                for (int p = 0; p < 8; ++p)
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        idle_pass();
                        rest[j] = mfma2(o0[p][t], own[p][t], rest[j]);
                    }
            }
        }
        cur = rest[0];
#pragma unroll
        for (int j = 0; j + 1 < NB - 2; ++j) rest[j] = rest[j + 1];
    }

    // ---- factor the diagonal tile
    __builtin_amdgcn_s_setprio(3);
    float pv = 1.f;                  // lane n: the pivot of column n as met
    const int slot = diag_slot<NB>(row);
#pragma unroll
    for (int p = 0; p < 8; ++p) {
        const int hp = p & 1, i0 = 4 * (p >> 1), l0 = 4 * p + 32 * hp;
        float s[4][4];               // the panel's diagonal block, broadcast (negated)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int q = j; q < 4; ++q) s[q][j] = rdlane(diag[i0 + j], l0 + q);
        const float d0 = -s[0][0], r0 = rsqrt_pivot(d0);
        const float m10 = -s[1][0] * r0, m20 = -s[2][0] * r0, m30 = -s[3][0] * r0;
        const float d1 = -fmaf(m10, m10, s[1][1]), r1 = rsqrt_pivot(d1);
        const float m21 = -fmaf(m20, m10, s[2][1]) * r1, m31 = -fmaf(m30, m10, s[3][1]) * r1;
        const float x0 = -diag[i0] * r0;
        const float x1 = -fmaf(x0, m10, diag[i0 + 1]) * r1;
        const float u2 = fmaf(x1, m21, fmaf(x0, m20, diag[i0 + 2]));
        const float u3 = fmaf(x1, m31, fmaf(x0, m30, diag[i0 + 3]));
        diag[i0] = (h == hp) ? x0 : diag[i0];
        diag[i0 + 1] = (h == hp) ? x1 : diag[i0 + 1];
        // Rows of the panel and above take no part in the update (their
        // entries are final).  A product issued while another runs waits for
        // it, and this wave with it: the first goes out between the second
        // and the third pivot.
        v2f a = {0.f, 0.f};
        if (p < 7) {
            a[0] = pair_op(x0, x1, hp);
            a[0] = n >= 4 * p + 4 ? a[0] : 0.f;
            __builtin_amdgcn_sched_barrier(0);
            diag = mfma2(a[0], a[0], diag);
            __builtin_amdgcn_sched_barrier(0);
        }
        const float d2 = -fmaf(m21, m21, fmaf(m20, m20, s[2][2])), r2 = rsqrt_pivot(d2);
        const float m32 = -fmaf(m31, m21, fmaf(m30, m20, s[3][2])) * r2;
        const float d3 = -fmaf(m32, m32, fmaf(m31, m31, fmaf(m30, m30, s[3][3])));
        const float r3 = rsqrt_pivot(d3);
        const float x2 = -u2 * r2, x3 = -fmaf(x2, m32, u3) * r3;
        diag[i0 + 2] = (h == hp) ? x2 : diag[i0 + 2];
        diag[i0 + 3] = (h == hp) ? x3 : diag[i0 + 3];
        if (p < 7) {
            a[1] = pair_op(x2, x3, hp);
            a[1] = n >= 4 * p + 4 ? a[1] : 0.f;
            __builtin_amdgcn_sched_barrier(0);
            diag = mfma2(a[1], a[1], diag);
            __builtin_amdgcn_sched_barrier(0);
        }
        // (every lane writes the same 4x4 factor)
        S.mic[row][p][0] = v4f{r0, r1, r2, r3};
        S.mic[row][p][1] = v4f{m10, m20, m30, m21};
        S.mic[row][p][2] = v4f{m31, m32, 0.f, 0.f};
        if (p < 7) S.op[slot][p][lane] = a;
        pv = n == 4 * p ? d0 : pv;
        pv = n == 4 * p + 1 ? d1 : pv;
        pv = n == 4 * p + 2 ? d2 : pv;
        pv = n == 4 * p + 3 ? d3 : pv;
        publish(&S.prog[row], 8 * row + p + 1);
    }
    __builtin_amdgcn_s_setprio(0);
    if (row > 0) store_tile(row - 1, cur);
    store_tile(row, diag);

    // ---- summary of this block row: smallest L_rr^2, first bad pivot, sum of
    // squares.  Lane n forms L_nn as the panel did; the bits of positive
    // floats order as the floats do (a NaN, which only a bad pivot gives,
    // counts for nothing).
    const float lnn = pv * rsqrt_pivot(pv), lnn2 = lnn * lnn;
    const uint32_t inf = 0x7f800000u;
    auto umin = [](uint32_t x, uint32_t y) { return x < y ? x : y; };
    uint32_t pm = (r < bs && lnn2 == lnn2) ? __float_as_uint(lnn2) : inf;
    pm = reduce16(pm, umin);
    pm = umin((uint32_t)__builtin_amdgcn_readlane((int)pm, 0),
              (uint32_t)__builtin_amdgcn_readlane((int)pm, 16));
    const uint64_t badm = __builtin_amdgcn_ballot_w64(!(pv > 0.f)) & 0xffffffffull;
    const uint64_t nanm = __builtin_amdgcn_ballot_w64(!(pv == pv)) & 0xffffffffull;
    const int bad = badm ? 32 * row + __builtin_ctzll(badm) : bs;
    int fail = bad < bs ? 2 * bad + (int)((nanm >> (bad & 31)) & 1u) : INT_MAX;
    if (want_f2) {
        if (row > 0) add_f2(row - 1, cur);
        add_f2(row, diag);
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) f2 += __shfl_xor(f2, o);
    }
    if (!last) {
        if (lane == 0) {
            S.pmin[row] = pm;
            S.fail[row] = fail;
            S.f2[row] = f2;
        }
        publish(&S.done[row], 1);
    } else {
        // lane b: block row b
        const int b = lane < row ? lane : row;
        if (row > 0) {
            const int bw = b < row ? b : row - 1;
            while (__builtin_amdgcn_ballot_w64(
                __hip_atomic_load(&S.done[bw], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) == 0)) {
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
            pm = b < row ? S.pmin[bw] : pm;
            fail = b < row ? S.fail[bw] : fail;
        }
        pm = reduce16(pm, umin);
        fail = (int)reduce16((uint32_t)fail, umin);
        if (lane == 0) {
            if (fail != INT_MAX) {
                sm->info = col0 + (fail >> 1) + 1;
                if (fail & 1) atomicOr(&sm->nan_flag, 1);    // the failing pivot is NaN
            } else {
                const uint32_t mu = umin(mu_before, pm);
                sm->mu_bits = mu;                    // one POTRF at a time writes it
                sm->mu_step[mu_slot] = mu;
            }
            sm->schur_max[mu_slot] = 0u;     // the step's TRSM folds its ratios in
            if (want_f2) {
                float t = 0.f;
                for (int q = 0; q < row; ++q) t += S.f2[q];
                sm->diag_f2[mu_slot] = t + f2;
            }
        }
    }
    if (row != 0) return;

    // ---- the inverses, by the wave that is free first: X L^T = I solved a
    // panel behind each owner, as the tiles below the diagonal are; lane n
    // ends with column n of the inverse
    for (int kb = 0; kb < nsb; ++kb) {
        v16f x;
#pragma unroll
        for (int i = 0; i < 16; ++i) x[i] = sig(i, h) == n ? -1.f : 0.f;
#pragma unroll
        for (int p = 0; p < 8; ++p) {
            v2f own, lop;
            wait_for(&S.prog[kb], 8 * kb + p + 1, false);
            follow<NB>(S, kb, p, x, own, lop);
            if (p < 7) {
                x = mfma2(lop[0], own[0], x);
                idle_pass();
                x = mfma2(lop[1], own[1], x);
            }
        }
        float* gd = dinv + (int64_t)((col0 >> 5) + kb) * 1024 + n * 32 + 4 * h;
#pragma unroll
        for (int v = 0; v < 4; ++v)
            *reinterpret_cast<v4f*>(gd + 8 * v) =
                v4f{x[4 * v], x[4 * v + 1], x[4 * v + 2], x[4 * v + 3]};
    }
}

}  // namespace

int mpc_launch_potrf(hipStream_t st, float* A, int64_t lda, int bs, int col0, float* dinv,
                     mpc_small* sm, int ntiles_next, uint32_t* stats_amax, uint32_t* stats_maxrs,
                     int mu_slot, int want_f2) {
    if (bs <= 0 || bs > 256) {
        mpc_set_error("potrf: block size %d outside 1..256", bs);
        return MPC_ERR_ARG;
    }
    if (lda > (1 << 21)) {
        mpc_set_error("potrf: leading dimension %lld above 2^21", (long long)lda);
        return MPC_ERR_ARG;
    }
    if (ntiles_next > 1024) {
        mpc_set_error("potrf: %d panel tiles exceed 1024", ntiles_next);
        return MPC_ERR_ARG;
    }
    if (mu_slot != 0 && mu_slot != 1) {
        mpc_set_error("potrf: mu slot %d", mu_slot);
        return MPC_ERR_ARG;
    }
    // up to four block rows: four waves and 30 KB of LDS, which fit on a CU
    // beside workgroups of the concurrent trailing update; more rows need
    // eight waves and 122 KB
    if (bs <= 128)
        hipLaunchKernelGGL(potrf_kernel<4>, dim3(1), dim3(256), 0, st, A, lda, bs, col0, dinv, sm,
                           ntiles_next, stats_amax, stats_maxrs, mu_slot, want_f2 ? 1 : 0);
    else
        hipLaunchKernelGGL(potrf_kernel<8>, dim3(1), dim3(512), 0, st, A, lda, bs, col0, dinv, sm,
                           ntiles_next, stats_amax, stats_maxrs, mu_slot, want_f2 ? 1 : 0);
    MPC_LAUNCH_CHECK();
    return 0;
}
