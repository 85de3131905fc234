// k_syrk.hip -- trailing-update SYRK, C(lower) -= Q Q^T, FP32 accumulation.
//
// Replaces the cuBLASLt launches of switching_chol.cuh:145-219
// (LtMxfp8Matmul fp8_utils.cuh:136-227, LtHSgemm_fp16in_fp32out :304-412,
// LtSgemm :231-302) and the WMMA SYRK of syrk_gemm.cuh:14-124, with the
// operand/target fix of fp8_chol.cuh:125-152 (C = A22, m = s) and only the
// lower triangle computed.
//
// Q is the quantised panel: row-major, k-contiguous payload plus one E8M0
// scale byte per row per 32 columns.  Each precision tile of Q (tile_rows
// rows) has its own storage format; an output tile pair is computed in the
// higher-precision class of its two operand tiles:
//   FP8 class  v_mfma_scale_f32_32x32x64_f8f6f4 (E4M3/E5M2 per operand, the
//              E8M0 scales applied by the matrix core: MX per 32, or the tile
//              scale replicated per 32)
//   16-bit     v_mfma_f32_32x32x16_bf16 / _f16 (FP8 operands converted exactly)
//   FP32       v_mfma_f32_32x32x2f32 for FP32 x FP32 and FP32 x FP16 pairs;
//              FP32 x FP8/BF16 pairs as three exact bf16 products per chunk
//              (the FP32 operand split as hi + mid + lo)
//
// Launch: one workgroup (4 waves) per 128x128 lower tile of C, wave (wr, wc)
// owns a 64x64 quadrant as 2x2 MFMA blocks, with the operands staged through
// LDS (one kernel per class and pair of formats); 64x64 tiles of 1x1 blocks,
// every class in one kernel, for the look-ahead's block column.  The MFMA
// "row" index runs along C's columns and the "column" index along C's rows, so
// each accumulator register maps to 32 consecutive rows of the column-major C
// (128 B per half-wave).  Block ids are remapped so consecutive tiles share an
// XCD.  At m = 16128 an E4M3 update takes 213 us with K = 64 (C's traffic at 4.9
// TB/s), 231 with 256, 253 with 512, 321 with 1024 (830 TFLOP/s); with operands
// loaded by every wave for itself 222, 234, 297 and 488.  BF16 K = 512: 464 (667
// before); FP16 437 (674).
#include "mpc_internal.hpp"
#include "mpc_formats.hpp"
#include <type_traits>

namespace {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef float v2f __attribute__((ext_vector_type(2)));

__device__ __forceinline__ int pair_class(int p, int q) {
    if (p == MPC_PREC_FP32 || q == MPC_PREC_FP32) return MPC_PREC_FP32;
    if (p == MPC_PREC_BF16 || q == MPC_PREC_BF16) return MPC_PREC_BF16;
    if (p == MPC_PREC_FP16 || q == MPC_PREC_FP16) return MPC_PREC_FP16;
    return MPC_PREC_E4M3;   // both 8-bit
}

// Position of a tile pair's launch in mpc_launch_syrk_panels' per-class
// sequence (E4M3 element pairs 00, 01, 10, 11; BF16; FP16; FP32 against
// FP32, against an FP8/BF16 format, against FP16).
__device__ __forceinline__ int launch_rank_of(int cls, int fa, int fb) {
    if (cls == MPC_PREC_E4M3) return 2 * fa + fb;
    if (cls == MPC_PREC_BF16) return 4;
    if (cls == MPC_PREC_FP16) return 5;
    return fa == 1 ? 6 : (fa == 2 ? 7 : 8);      // FP32: fa is the partner kind
}
__device__ __forceinline__ bool is_e4m3_elem(int p) {
    return p == MPC_PREC_E4M3 || p == MPC_PREC_MXE4M3;
}
__device__ __forceinline__ int launch_rank(int prow, int pcol) {
    const int cls = pair_class(prow, pcol);
    if (cls == MPC_PREC_E4M3)
        return launch_rank_of(cls, is_e4m3_elem(pcol) ? 0 : 1, is_e4m3_elem(prow) ? 0 : 1);
    if (cls == MPC_PREC_FP32) {
        const bool f32pair = prow == MPC_PREC_FP32 && pcol == MPC_PREC_FP32;
        const bool f16 = prow == MPC_PREC_FP16 || pcol == MPC_PREC_FP16;
        return launch_rank_of(cls, f32pair ? 1 : (f16 ? 0 : 2), 0);
    }
    return launch_rank_of(cls, 0, 0);
}

struct operand_src {
    const uint8_t* payload;
    const uint8_t* scales;
    int64_t row_stride;
    int kb;          // k / 32
    int prec;        // storage format of this operand tile
};

// 8 consecutive k values of one row as floats (stored format -> f32, exact)
__device__ __forceinline__ void load8_f32(const operand_src& o, int64_t row, int k0, float* f) {
    const uint8_t* p = o.payload + row * o.row_stride;
    if (o.prec == MPC_PREC_FP32) {
        float4 a = *reinterpret_cast<const float4*>(p + 4 * k0);
        float4 b = *reinterpret_cast<const float4*>(p + 4 * k0 + 16);
        f[0] = a.x; f[1] = a.y; f[2] = a.z; f[3] = a.w;
        f[4] = b.x; f[5] = b.y; f[6] = b.z; f[7] = b.w;
    } else if (o.prec == MPC_PREC_BF16 || o.prec == MPC_PREC_FP16) {
        uint4 a = *reinterpret_cast<const uint4*>(p + 2 * k0);
        uint32_t w[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (o.prec == MPC_PREC_BF16) {
                f[2 * i] = __uint_as_float(w[i] << 16);
                f[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
            } else {
                f[2 * i] = (float)__builtin_bit_cast(_Float16, (unsigned short)(w[i] & 0xffffu));
                f[2 * i + 1] = (float)__builtin_bit_cast(_Float16, (unsigned short)(w[i] >> 16));
            }
        }
    } else {
        uint2 a = *reinterpret_cast<const uint2*>(o.payload + mpc_f8_offset(row, k0, o.row_stride));
        float sc = mpc_dev_exp2i((int)o.scales[row * o.kb + (k0 >> 5)] - 127);
        v2f t0, t1, t2, t3;
        if (mpc_dev_is_e4m3(o.prec)) {
            t0 = __builtin_amdgcn_cvt_pk_f32_fp8((int)a.x, false);
            t1 = __builtin_amdgcn_cvt_pk_f32_fp8((int)a.x, true);
            t2 = __builtin_amdgcn_cvt_pk_f32_fp8((int)a.y, false);
            t3 = __builtin_amdgcn_cvt_pk_f32_fp8((int)a.y, true);
        } else {
            t0 = __builtin_amdgcn_cvt_pk_f32_bf8((int)a.x, false);
            t1 = __builtin_amdgcn_cvt_pk_f32_bf8((int)a.x, true);
            t2 = __builtin_amdgcn_cvt_pk_f32_bf8((int)a.y, false);
            t3 = __builtin_amdgcn_cvt_pk_f32_bf8((int)a.y, true);
        }
        f[0] = t0.x * sc; f[1] = t0.y * sc; f[2] = t1.x * sc; f[3] = t1.y * sc;
        f[4] = t2.x * sc; f[5] = t2.y * sc; f[6] = t3.x * sc; f[7] = t3.y * sc;
    }
}

__device__ __forceinline__ v8bf load8_bf16(const operand_src& o, int64_t row, int k0) {
    if (o.prec == MPC_PREC_BF16) {
        uint4 a = *reinterpret_cast<const uint4*>(o.payload + row * o.row_stride + 2 * k0);
        return __builtin_bit_cast(v8bf, a);
    }
    float f[8];
    load8_f32(o, row, k0, f);      // FP8 * 2^e is exact in bf16 range
    uint4 w;
    w.x = (__float_as_uint(f[0]) >> 16) | (__float_as_uint(f[1]) & 0xffff0000u);
    w.y = (__float_as_uint(f[2]) >> 16) | (__float_as_uint(f[3]) & 0xffff0000u);
    w.z = (__float_as_uint(f[4]) >> 16) | (__float_as_uint(f[5]) & 0xffff0000u);
    w.w = (__float_as_uint(f[6]) >> 16) | (__float_as_uint(f[7]) & 0xffff0000u);
    return __builtin_bit_cast(v8bf, w);
}

__device__ __forceinline__ v8h load8_f16(const operand_src& o, int64_t row, int k0) {
    uint4 a = *reinterpret_cast<const uint4*>(o.payload + row * o.row_stride + 2 * k0);
    return __builtin_bit_cast(v8h, a);
}

// x = hi + mid + lo exactly, each term a bf16 (8 significant bits, taken by
// truncation): the remainders x - hi and (x - hi) - mid are exact in FP32 and
// the last one has at most 8 significant bits.  Eight values, packed as the
// 16-bit matrix-core operand.
__device__ __forceinline__ void split3_bf16(const float* f, v8bf& hi, v8bf& mid, v8bf& lo) {
    uint32_t uh[8], um[8], ul[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        uh[e] = __float_as_uint(f[e]) & 0xffff0000u;
        const float r1 = f[e] - __uint_as_float(uh[e]);
        um[e] = __float_as_uint(r1) & 0xffff0000u;
        const float r2 = r1 - __uint_as_float(um[e]);
        ul[e] = __float_as_uint(r2) & 0xffff0000u;
    }
    uint4 wh, wm, wl;
    wh.x = (uh[0] >> 16) | uh[1]; wh.y = (uh[2] >> 16) | uh[3]; wh.z = (uh[4] >> 16) | uh[5]; wh.w = (uh[6] >> 16) | uh[7];
    wm.x = (um[0] >> 16) | um[1]; wm.y = (um[2] >> 16) | um[3]; wm.z = (um[4] >> 16) | um[5]; wm.w = (um[6] >> 16) | um[7];
    wl.x = (ul[0] >> 16) | ul[1]; wl.y = (ul[2] >> 16) | ul[3]; wl.z = (ul[4] >> 16) | ul[5]; wl.w = (ul[6] >> 16) | ul[7];
    hi = __builtin_bit_cast(v8bf, wh);
    mid = __builtin_bit_cast(v8bf, wm);
    lo = __builtin_bit_cast(v8bf, wl);
}

struct tile_ctx {
    float* C;
    const float* Cs;            // where C's old values are read (C, or a source copy)
    int64_t ldc, m;
    int64_t rowbase, colbase;   // first C row / col of this wave's quadrant
    bool diag;                  // this quadrant straddles the diagonal (rowbase == colbase)
};

// Each wave owns a (32 QA) x (32 QA) quadrant of C as QA x QA MFMA blocks.
// Element (a, b, i) of the wave's quadrant sits at wave base + byte offset
//   ((32a + n) + (32b + 8(i/4) + 4h + i%4) * ldc) * 4,
// which stays below 2^31 for ldc <= 2^23; only the base pointer is 64-bit.
// The product Q Q^T is accumulated from zero and subtracted from C once, as a
// BLAS GEMM with beta = 1 does: seeding the accumulator with -C instead would
// round every one of the k FMA steps at the scale of |C| rather than of the
// partial sum, about sqrt(k) times the error for a trailing update.
//
// C's old values are loaded (load_c) before the K loop, so their HBM latency
// overlaps the operand loads and the products; store_c subtracts and
// stores.  C is streamed: its loads and stores carry the non-temporal cache
// policy (CPOL), so the lines of C, touched once per update, do not evict
// the panel rows that the other tiles of the XCD re-read from L2.
constexpr int kCpolStream = 2;     // nt: non-temporal (streaming) policy bit

template <int QA>
struct c_frag {
    float v[QA][QA][16];
};

// Buffer addressing: the wave's base in the resource (scalar), the column
// offset (32b + 8(i/4) + i%4) * ldc * 4 as the scalar soffset and the lane's
// (32a + n + 4h ldc) * 4 as the one 32-bit VGPR per a.  With global
// addressing every load would keep its own 64-bit VGPR address alive until
// the matching store.
template <int QA>
__device__ __forceinline__ void load_c(const tile_ctx& t, c_frag<QA>& c, int lane = threadIdx.x & 63) {
    constexpr int QE = 32 * QA;
    const int h = lane >> 5, n = lane & 31;
    const __amdgpu_buffer_rsrc_t rsl = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(t.Cs) + t.rowbase + t.colbase * t.ldc, 0, 0x7fffffff, 0x00020000);
    const int ld4 = (int)t.ldc * 4;
    const int rlim = (int)(t.m - t.rowbase), clim = (int)(t.m - t.colbase);
    // Loads are unconditional (a per-lane conditional load becomes a branch
    // with its own wait): interior quadrants read every element (the
    // diagonal quadrant's upper part is a valid address, masked at the
    // store); edge quadrants read from a clamped row and column.
    const bool interior = rlim >= QE && clim >= QE;
    if (interior) {
#pragma unroll
        for (int a = 0; a < QA; ++a) {
            const int loff = ((32 * a + n) + 4 * h * (int)t.ldc) * 4;
#pragma unroll
            for (int b = 0; b < QA; ++b)
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    c.v[a][b][i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                        rsl, loff, (32 * b + 8 * (i >> 2) + (i & 3)) * ld4, kCpolStream));
        }
    } else {
#pragma unroll
        for (int a = 0; a < QA; ++a)
#pragma unroll
            for (int b = 0; b < QA; ++b)
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int r = 32 * a + n, cc0 = 32 * b + 8 * (i >> 2) + 4 * h + (i & 3);
                    const int rc = r < rlim ? r : rlim - 1, cc = cc0 < clim ? cc0 : clim - 1;
                    c.v[a][b][i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                        rsl, rc * 4 + cc * ld4, 0, kCpolStream));
                }
    }
}

template <int QA>
__device__ __forceinline__ void store_c(const tile_ctx& t, const c_frag<QA>& c,
                                        const v16f acc[QA][QA], int lane = threadIdx.x & 63) {
    const int h = lane >> 5, n = lane & 31;
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc(t.C + t.rowbase + t.colbase * t.ldc, 0, 0x7fffffff,
                                          0x00020000);
    const int ld4 = (int)t.ldc * 4;
    const int rlim = (int)(t.m - t.rowbase), clim = (int)(t.m - t.colbase);
#pragma unroll
    for (int a = 0; a < QA; ++a) {
        const int loff = ((32 * a + n) + 4 * h * (int)t.ldc) * 4;
#pragma unroll
        for (int b = 0; b < QA; ++b)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int r = 32 * a + n, cc = 32 * b + 8 * (i >> 2) + 4 * h + (i & 3);
                const bool ok = r < rlim && cc < clim && (!t.diag || r >= cc);
                if (ok)
                    __builtin_amdgcn_raw_buffer_store_b32(
                        __float_as_uint(c.v[a][b][i] - acc[a][b][i]), rs, loff,
                        (32 * b + 8 * (i >> 2) + (i & 3)) * ld4, kCpolStream);
            }
    }
}

// operand rows of the wave: column side (ra) and row side (rb), clamped to m
template <int QA>
__device__ __forceinline__ void operand_rows(const tile_ctx& t, int64_t ra[QA], int64_t rb[QA]) {
    const int n = threadIdx.x & 31;
#pragma unroll
    for (int q = 0; q < QA; ++q) {
        ra[q] = t.colbase + 32 * q + n;
        if (ra[q] >= t.m) ra[q] = t.m - 1;
        rb[q] = t.rowbase + 32 * q + n;
        if (rb[q] >= t.m) rb[q] = t.m - 1;
    }
}

// FP8 class: A operand = column-side rows, B operand = row-side rows.
template <int QA, int FA, int FB>
__device__ __forceinline__ void mm_fp8(const operand_src& oc, const operand_src& orow,
                                       const tile_ctx& t, int k, v16f acc[QA][QA]) {
    const int h = (threadIdx.x & 63) >> 5;
    int64_t ra[QA], rb[QA];
    operand_rows<QA>(t, ra, rb);
    // Operand layout of the 8-bit 32x32x64 matrix-core op (measured on gfx950):
    // the scale of lane half h (E8M0 block h of the 64-wide K chunk) multiplies
    // bytes 0-15 of BOTH lane halves when h = 0 and bytes 16-31 of both when
    // h = 1.  So lane half h carries K [kc + 16h, +16) in bytes 0-15 and
    // K [kc + 32 + 16h, +16) in bytes 16-31; K block h then spans exactly the
    // 32 elements the hardware scales with lane half h's scale byte.
    // the 32-row operand blocks of the wave (the lane's own 32 bytes of a
    // chunk: mpc_f8_offset's layout)
    const int64_t lane32 = (int64_t)(threadIdx.x & 63) * 32;
    const uint8_t* ba[QA];
    const uint8_t* bb[QA];
#pragma unroll
    for (int q = 0; q < QA; ++q) {
        ba[q] = oc.payload + (t.colbase + 32 * q) * oc.row_stride + lane32;
        bb[q] = orow.payload + (t.rowbase + 32 * q) * orow.row_stride + lane32;
    }
    for (int kc = 0; kc < k; kc += 64) {
        const int koff = kc + 32 * h;          // scale block of this lane half
        const int64_t co = (int64_t)(kc >> 6) * 2048;
        v8i A[QA], B[QA];
        int sa[QA], sb[QA];
#pragma unroll
        for (int q = 0; q < QA; ++q) {
            const uint8_t* pa = ba[q] + co;
            const uint8_t* pb = bb[q] + co;
            uint4 a0 = *reinterpret_cast<const uint4*>(pa), a1 = *reinterpret_cast<const uint4*>(pa + 16);
            uint4 b0 = *reinterpret_cast<const uint4*>(pb), b1 = *reinterpret_cast<const uint4*>(pb + 16);
            A[q] = v8i{(int)a0.x, (int)a0.y, (int)a0.z, (int)a0.w, (int)a1.x, (int)a1.y, (int)a1.z, (int)a1.w};
            B[q] = v8i{(int)b0.x, (int)b0.y, (int)b0.z, (int)b0.w, (int)b1.x, (int)b1.y, (int)b1.z, (int)b1.w};
            sa[q] = oc.scales[ra[q] * oc.kb + (koff >> 5)];
            sb[q] = orow.scales[rb[q] * orow.kb + (koff >> 5)];
        }
#pragma unroll
        for (int a = 0; a < QA; ++a)
#pragma unroll
            for (int b = 0; b < QA; ++b)
                acc[a][b] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(A[b], B[a], acc[a][b], FA, FB, 0,
                                                                           sa[b], 0, sb[a]);
    }
}

template <int QA, bool BF>
__device__ __forceinline__ void mm_16(const operand_src& oc, const operand_src& orow,
                                      const tile_ctx& t, int k, v16f acc[QA][QA]) {
    const int h = (threadIdx.x & 63) >> 5;
    int64_t ra[QA], rb[QA];
    operand_rows<QA>(t, ra, rb);
    for (int kc = 0; kc < k; kc += 16) {
        const int k0 = kc + 8 * h;
        if constexpr (BF) {
            v8bf A[QA], B[QA];
#pragma unroll
            for (int q = 0; q < QA; ++q) { A[q] = load8_bf16(oc, ra[q], k0); B[q] = load8_bf16(orow, rb[q], k0); }
#pragma unroll
            for (int a = 0; a < QA; ++a)
#pragma unroll
                for (int b = 0; b < QA; ++b)
                    acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A[b], B[a], acc[a][b], 0, 0, 0);
        } else {
            v8h A[QA], B[QA];
#pragma unroll
            for (int q = 0; q < QA; ++q) { A[q] = load8_f16(oc, ra[q], k0); B[q] = load8_f16(orow, rb[q], k0); }
#pragma unroll
            for (int a = 0; a < QA; ++a)
#pragma unroll
                for (int b = 0; b < QA; ++b)
                    acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[b], B[a], acc[a][b], 0, 0, 0);
        }
    }
}

// SPLIT: FP32 against FP8/BF16 as bf16 products (else no such pair occurs)
template <int QA, bool SPLIT>
__device__ __forceinline__ void mm_f32(const operand_src& oc, const operand_src& orow,
                                       const tile_ctx& t, int k, v16f acc[QA][QA]) {
    const int h = (threadIdx.x & 63) >> 5;
    int64_t ra[QA], rb[QA];
    operand_rows<QA>(t, ra, rb);
    // FP32 against a format exact in bf16 (FP8 with its scale, or BF16): the
    // FP32 operand as hi + mid + lo (exact), three bf16 products per 16-wide
    // chunk; the products are exact and the sums FP32, as in the FP32
    // matrix-core op, at a sixth of its cost per k
    if (SPLIT && (oc.prec == MPC_PREC_FP32) != (orow.prec == MPC_PREC_FP32) &&
        oc.prec != MPC_PREC_FP16 && orow.prec != MPC_PREC_FP16) {
        const bool col32 = oc.prec == MPC_PREC_FP32;
        for (int kc = 0; kc < k; kc += 16) {
            const int k0 = kc + 8 * h;
            v8bf F[QA][3], Lw[QA];
#pragma unroll
            for (int q = 0; q < QA; ++q) {
                float f[8];
                load8_f32(col32 ? oc : orow, col32 ? ra[q] : rb[q], k0, f);
                split3_bf16(f, F[q][0], F[q][1], F[q][2]);
                Lw[q] = load8_bf16(col32 ? orow : oc, col32 ? rb[q] : ra[q], k0);
            }
#pragma unroll
            for (int s3 = 0; s3 < 3; ++s3)
#pragma unroll
                for (int a = 0; a < QA; ++a)
#pragma unroll
                    for (int b = 0; b < QA; ++b)
                        acc[a][b] = col32
                            ? __builtin_amdgcn_mfma_f32_32x32x16_bf16(F[b][s3], Lw[a], acc[a][b], 0, 0, 0)
                            : __builtin_amdgcn_mfma_f32_32x32x16_bf16(Lw[b], F[a][s3], acc[a][b], 0, 0, 0);
        }
        return;
    }
    // k permutation: half h takes the 8-element groups k = 16c + 8h .. +8
    for (int kc = 0; kc < k; kc += 16) {
        const int k0 = kc + 8 * h;
        float A[QA][8], B[QA][8];
#pragma unroll
        for (int q = 0; q < QA; ++q) { load8_f32(oc, ra[q], k0, A[q]); load8_f32(orow, rb[q], k0, B[q]); }
#pragma unroll
        for (int e = 0; e < 8; ++e)
#pragma unroll
            for (int a = 0; a < QA; ++a)
#pragma unroll
                for (int b = 0; b < QA; ++b)
                    acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x2f32(A[b][e], B[a][e], acc[a][b], 0, 0, 0);
    }
}

// Work lists of a launch sequence (int32): 16 counters indexed by launch
// rank (launch_rank_of), then one list of tile pair ids per rank at
// 16 + rank * cap.  The first launch of a sequence runs over every tile pair
// and appends each pair to the lists of the later launches that have work on
// it; those launches then run over their lists only, instead of a full grid
// of workgroups of which most would find nothing of their class.
struct syrk_lists {
    int* base;       // nullptr: every launch runs over the full grid
    int  cap;        // tile pairs per list
    int  mode;       // 0 full grid, 1 full grid + build the later lists, 2 from the list
};
constexpr int kListHead = 16;

// The tile pairs of a launch: the lower triangle of tile columns
// [tcol0, tcol0 + ...) (column-major), or, when rect_ncol > 0, the rectangle
// of tile rows [rect_tr0, mt) and tile columns [tcol0, tcol0 + rect_ncol)
// (row-major; every pair strictly below the diagonal).
struct syrk_shape {
    int64_t mt, tcol0, tcol1, rect_tr0, rect_ncol;
};

// Launch sequence, first launch: the pair goes to the lists of the later
// launches (ranks above `rank`) that have work on it.
__device__ __forceinline__ void note_pair(const syrk_lists& L, const mpc_syrk_panels& P, int tile_rows,
                                          int64_t trow, int64_t tcol, int64_t pid, int rank) {
    if (threadIdx.x != 0) return;
    unsigned need = 0;
    for (int q = 0; q < P.np; ++q) {
        const int slot = (P.p0 + q) % P.slots;
        const uint8_t* prec = P.prec + slot * 1024 + (P.rows0 - (int64_t)q * P.nb) / tile_rows;
        need |= 1u << launch_rank(prec[trow], prec[tcol]);
    }
    need &= ~((2u << rank) - 1u);
    for (int r = 0; r < kListHead; ++r)
        if ((need >> r) & 1u) {
            const int slot = atomicAdd(&L.base[r], 1);
            L.base[kListHead + (int64_t)r * L.cap + slot] = (int)pid;
        }
}

// tile pair pid of the launch -> tile row ti, tile column tj
template <int TILE>
__device__ __forceinline__ void tile_of(const syrk_shape& G, int64_t pid, int64_t& ti, int64_t& tj) {
    if (G.rect_ncol > 0) {
        ti = G.rect_tr0 + pid / G.rect_ncol;
        tj = G.tcol0 + pid % G.rect_ncol;
    } else {
        // The lower triangle from tile column tcol0 in super-blocks of SB x SB
        // tiles (2048 rows and columns): super-columns in order, in each the
        // diagonal super-block and then the super-blocks below it, each
        // column-major.  Consecutive pair ids go to one XCD, whose L2 then
        // keeps the panel rows of the few super-blocks it works on (a plain
        // column-major order streams the whole panel past every tile column).
        // start(c) = c*mt - c*(c-1)/2 counts the pairs left of tile column c.
        constexpr int64_t SB = 2048 / TILE;
        const int64_t mt = G.mt;
        auto start = [&](int64_t c) { return c * mt - c * (c - 1) / 2; };
        const int64_t gid = pid + start(G.tcol0);
        const double tw = 2.0 * (double)mt + 1.0;
        int64_t tc = (int64_t)((tw - sqrt(tw * tw - 8.0 * (double)gid)) * 0.5);
        if (tc < 0) tc = 0;
        while (tc > 0 && start(tc) > gid) --tc;
        while (start(tc + 1) <= gid) ++tc;
        // the super-column holding tile column tc: columns [c0, c1)
        const int64_t c0 = G.tcol0 + ((tc - G.tcol0) / SB) * SB;
        const int64_t c1 = c0 + SB < G.tcol1 ? c0 + SB : G.tcol1;
        const int64_t rb = c0 + SB < mt ? c0 + SB : mt;       // rows of its diagonal block
        const int64_t loc = gid - start(c0);
        // pairs in the diagonal block: sum over tj in [c0, c1) of (rb - tj)
        const int64_t w = c1 - c0;
        const int64_t D = w * rb - (c0 + c1 - 1) * w / 2;
        if (loc < D) {
            // column-major over the triangle: column c0 + u holds the rows
            // [c0 + u, rb), M - u of them (M = rb - c0); dstart(u) = u M - u(u-1)/2
            const int64_t M = rb - c0;
            auto dstart = [&](int64_t u) { return u * M - u * (u - 1) / 2; };
            const double tw2 = 2.0 * (double)M + 1.0;
            int64_t u = (int64_t)((tw2 - sqrt(fmax(tw2 * tw2 - 8.0 * (double)loc, 0.0))) * 0.5);
            if (u < 0) u = 0;
            if (u > w - 1) u = w - 1;
            while (u > 0 && dstart(u) > loc) --u;
            while (u + 1 < w && dstart(u + 1) <= loc) ++u;
            tj = c0 + u;
            ti = tj + (loc - dstart(u));
        } else {
            // rows [rb, mt) as SB-row super-blocks, each column-major (the
            // tiles of one column, consecutive in memory, on one XCD together)
            const int64_t l2 = loc - D;
            const int64_t sbi = l2 / (SB * w), inner = l2 - sbi * SB * w;
            const int64_t rbase = rb + sbi * SB;
            const int64_t rows = mt - rbase < SB ? mt - rbase : SB;
            tj = c0 + inner / rows;
            ti = rbase + inner % rows;
        }
    }
}

template <int QA, bool F32H>
__device__ __forceinline__ void syrk_tile(float* __restrict__ C, int64_t m, int64_t ldc, int k,
                                          const mpc_syrk_panels& P, int64_t row_stride,
                                          int tile_rows, const syrk_shape& G, int64_t pid,
                                          const syrk_lists& L, float* sums);

// The products of the P.np panels are summed in the accumulators (K = np*k)
// and subtracted from C once.  F32H: only the pairs of FP32 and FP16 tiles (a
// later launch of a sequence whose others are the staged kernels below), and
// a tile without one exits without touching C; a tile mixing classes across
// panels is updated once per class launch.  Otherwise every panel, the class
// chosen per workgroup and panel.
// LISTED: a later launch of a sequence, over its work list (L.mode 2);
// otherwise one workgroup per tile pair (L.mode 0, or 1 to build the lists)
template <int QA, bool F32H, bool LISTED>
__global__ __launch_bounds__(256, 2) void syrk_kernel(float* __restrict__ C, int64_t m, int64_t ldc,
                                                   int k, const mpc_syrk_panels P,
                                                   int64_t row_stride, int tile_rows,
                                                   const mpc_small* __restrict__ sm, int64_t npair,
                                                   int64_t per_xcd, const syrk_shape G,
                                                   const syrk_lists L) {
    __shared__ float sums[QA == 1 ? 16 * 256 : 1];
    if (sm && sm->info != 0) return;
    if constexpr (LISTED) {
        const int rank = launch_rank_of(MPC_PREC_FP32, 0, 0);
        const int count = L.base[rank];
        const int* list = L.base + kListHead + (int64_t)rank * L.cap;
        for (int it = blockIdx.x; it < count; it += gridDim.x)
            syrk_tile<QA, F32H>(C, m, ldc, k, P, row_stride, tile_rows, G, list[it], L, sums);
        return;
    }
    // XCD-aware remap: hardware places block b on XCD b % 8
    const int64_t b = blockIdx.x;
    const int64_t pid = (b & 7) * per_xcd + (b >> 3);
    if (pid >= npair) return;
    syrk_tile<QA, F32H>(C, m, ldc, k, P, row_stride, tile_rows, G, pid, L, sums);
}

template <int QA, bool F32H>
__device__ __forceinline__ void syrk_tile(float* __restrict__ C, int64_t m, int64_t ldc, int k,
                                          const mpc_syrk_panels& P, int64_t row_stride,
                                          int tile_rows, const syrk_shape& G, int64_t pid,
                                          const syrk_lists& L, float* sums) {
    constexpr int TILE = 64 * QA;
    int64_t ti, tj;
    tile_of<TILE>(G, pid, ti, tj);
    const int64_t trow = (ti * TILE) / tile_rows, tcol = (tj * TILE) / tile_rows;
    const int rank = launch_rank_of(MPC_PREC_FP32, 0, 0);
    if (F32H && L.mode == 1) note_pair(L, P, tile_rows, trow, tcol, pid, rank);

    const int wave = threadIdx.x >> 6, wr = wave >> 1, wc = wave & 1;
    const bool diag = ti == tj;
    if (diag && wr == 0 && wc == 1) return;   // strictly upper quadrant

    tile_ctx t;
    t.C = C;
    t.Cs = C;
    t.ldc = ldc;
    t.m = m;
    t.rowbase = ti * TILE + 32 * QA * wr;
    t.colbase = tj * TILE + 32 * QA * wc;
    t.diag = diag && wr == wc;     // only the diagonal quadrants need the r >= c mask
    if (t.rowbase >= m || t.colbase >= m) return;

    v16f acc[QA][QA];
#pragma unroll
    for (int a = 0; a < QA; ++a)
#pragma unroll
        for (int b2 = 0; b2 < QA; ++b2) acc[a][b2] = v16f{};
    if (P.csrc) {
        // C's old values come from csrc in the first launch, in the host's
        // launch order, whose class covers one of this tile's panels
        int lo = 99;
        for (int q = 0; q < P.np; ++q) {
            const int slot = (P.p0 + q) % P.slots;
            const uint8_t* prec = P.prec + slot * 1024 + (P.rows0 - (int64_t)q * P.nb) / tile_rows;
            const int r = launch_rank(prec[trow], prec[tcol]);
            lo = r < lo ? r : lo;
        }
        if (!F32H || lo == rank) t.Cs = P.csrc;
    }
    // the panels this launch applies to the tile (bit q: panel q)
    auto operands = [&](int q, operand_src& orow, operand_src& ocol) {
        const int slot = (P.p0 + q) % P.slots;
        const int64_t roff = P.rows0 - (int64_t)q * P.nb;   // C row 0 within this panel
        const uint8_t* prec = P.prec + slot * 1024 + roff / tile_rows;
        orow.prec = prec[trow];
        ocol.prec = prec[tcol];
        orow.payload = ocol.payload = P.payload + slot * P.pstride + roff * row_stride;
        orow.scales = ocol.scales = P.scales + slot * P.sstride + roff * (k >> 5);
        orow.row_stride = ocol.row_stride = row_stride;
        orow.kb = ocol.kb = k >> 5;
    };
    unsigned use = 0;
    for (int q = 0; q < P.np; ++q) {
        operand_src orow, ocol;
        operands(q, orow, ocol);
        if (!F32H || launch_rank(orow.prec, ocol.prec) == rank) use |= 1u << q;
    }
    if (!use) return;              // no panel of this launch's class on this tile
    // C's old values in flight during the products (64-row tiles only: at
    // 128-row tiles the K loop's operand buffers need those registers)
    constexpr bool kPrefetchC = QA == 1;
    c_frag<QA> cv;
    if constexpr (kPrefetchC) load_c<QA>(t, cv);
    // Each panel's sum apart (see kSumPanels below); the sum of the panels so far
    // waits in LDS, as three workgroups per CU have no 16 registers to spare.
    for (int q = 0; q < P.np; ++q) {
        if (!((use >> q) & 1u)) continue;
        if constexpr (QA == 1) {
            if (q > 0) {
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    float* s = sums + 256 * i + threadIdx.x;
                    *s = q > 1 ? *s + acc[0][0][i] : acc[0][0][i];
                }
                acc[0][0] = v16f{};
            }
        }
        operand_src orow, ocol;
        operands(q, orow, ocol);
        if constexpr (F32H) {
            mm_f32<QA, false>(ocol, orow, t, k, acc);
        } else {
            const int c = pair_class(orow.prec, ocol.prec);
            const int fa = mpc_dev_is_e4m3(ocol.prec) ? 0 : 1, fb = mpc_dev_is_e4m3(orow.prec) ? 0 : 1;
            if (c == MPC_PREC_E4M3) {
                if (fa == 0 && fb == 0) mm_fp8<QA, 0, 0>(ocol, orow, t, k, acc);
                else if (fa == 0) mm_fp8<QA, 0, 1>(ocol, orow, t, k, acc);
                else if (fb == 0) mm_fp8<QA, 1, 0>(ocol, orow, t, k, acc);
                else mm_fp8<QA, 1, 1>(ocol, orow, t, k, acc);
            } else if (c == MPC_PREC_BF16) {
                mm_16<QA, true>(ocol, orow, t, k, acc);
            } else if (c == MPC_PREC_FP16) {
                mm_16<QA, false>(ocol, orow, t, k, acc);
            } else {
                mm_f32<QA, true>(ocol, orow, t, k, acc);
            }
        }
    }
    if constexpr (QA == 1) {
        if (P.np > 1) {
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[0][0][i] += sums[256 * i + threadIdx.x];
        }
    }
    if constexpr (!kPrefetchC) load_c<QA>(t, cv);
    store_c<QA>(t, cv, acc);
}


// ---------------------------------------------------------------- FP32 x FP32
// The pairs of two FP32 tiles, with v_mfma_f32_32x32x2f32 in the K order of
// mm_f32 (bit for bit the same sums).  The operands of 128 columns and 128
// rows of C are staged through LDS, 16 K at a time in two buffers: four lanes
// load a row's 64 bytes, where the matrix op's own layout (a lane per row)
// reads 64 rows' separate lines per load, which bound the kernel (m = 16128,
// K = 256: 832 us = 80 TFLOP/s of the 157 peak).  In LDS a block of 32 rows is in operand
// order, two groups of 16-byte elements (k 8h .. +3 and 8h + 4 .. +7 of lane
// half h), so a wave's operand is one 1 KB read.
// The rounding errors of an FP32 sum grow with the length of its chain of
// additions, systematically where the products vary slowly, and are all the error
// there is here (in the other kernels the operands' rounding is larger by orders
// of magnitude).  So a chain covers P.sum panels:
//   kSumGroups: C takes each chain's result (20 more registers: n = 32768 FP32
//     factor 113.0 -> 114.8 ms, so it has an instance of its own);
//   kSumPanels (P.sum = 1): the panels' results are added in registers and C takes
//     the sum once.  212 registers, two workgroups a CU, for updates of up to 4096
//     rows, which have no more.  FP32 factor of a matrix with cond 1e6, n = 4000,
//     nb = 128, groups of 2: ||L - exact|| 1.4e-5, 1.7e-5 with one chain and with C
//     taking every panel's (n = 4096, nb = 256: 2.6e-5, 7.7e-5 and 2.9e-5), at 1425
//     us, 1402 and 1395.
typedef float v4f __attribute__((ext_vector_type(4)));
constexpr int FSK = 16;                       // K of a chunk
constexpr int FSB = 8 * 2 * 1024;             // bytes of a buffer: 8 blocks of 2 groups
constexpr int kSumAll = 0, kSumGroups = 1, kSumPanels = 2;

template <int SUMS>
__device__ __forceinline__ void syrk_f32_tile(float* __restrict__ C, int64_t m, int64_t ldc, int k,
                                              const mpc_syrk_panels& P, int64_t row_stride,
                                              int tile_rows, const syrk_shape& G, int64_t pid,
                                              const syrk_lists& L, char* lds) {
    constexpr int TILE = MPC_SYRK_TILE;
    int64_t ti, tj;
    tile_of<TILE>(G, pid, ti, tj);
    const int64_t trow = (ti * TILE) / tile_rows, tcol = (tj * TILE) / tile_rows;
    const int rank = launch_rank_of(MPC_PREC_FP32, 1, 0);
    if (L.mode == 1) note_pair(L, P, tile_rows, trow, tcol, pid, rank);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wr = wave >> 1, wc = wave & 1;

    unsigned todo = 0;                       // the panels of this launch
    int lo = 99;                             // first launch with work on the tile
    for (int q = 0; q < P.np; ++q) {
        const int slot = (P.p0 + q) % P.slots;
        const uint8_t* prec = P.prec + slot * 1024 + (P.rows0 - (int64_t)q * P.nb) / tile_rows;
        const int r = launch_rank(prec[trow], prec[tcol]);
        lo = r < lo ? r : lo;
        if (r == rank) todo |= 1u << q;
    }
    if (!todo) return;

    tile_ctx t;
    t.C = C;
    t.Cs = P.csrc && lo == rank ? P.csrc : C;
    t.ldc = ldc;
    t.m = m;
    t.rowbase = ti * TILE + 64 * wr;
    t.colbase = tj * TILE + 64 * wc;
    t.diag = ti == tj && wr == wc;
    // (waves without a quadrant stage and meet the barriers all the same)
    const bool live = !(ti == tj && wr == 0 && wc == 1) && t.rowbase < m && t.colbase < m;

    // staging: thread (r4, l4) moves k 4 l4 .. +3 of operand rows r4 + 64 u (u < 2:
    // the columns of C, else its rows; past m the last row again)
    const int l4 = tid & 3, r4 = tid >> 2;
    char* const sd = lds + ((r4 >> 5) * 2 + (l4 & 1)) * 1024 + (l4 >> 1) * 512 + (r4 & 31) * 16;
    v4f st[4];
    const float* src[4];
    auto panel = [&](int q) {
        const int slot = (P.p0 + q) % P.slots;
        const int64_t roff = P.rows0 - (int64_t)q * P.nb;    // C row 0 within this panel
        const uint8_t* pay = P.payload + slot * P.pstride + roff * row_stride + 16 * l4;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            int64_t row = (u < 2 ? tj : ti) * TILE + 64 * (u & 1) + r4;
            if (row >= m) row = m - 1;
            src[u] = reinterpret_cast<const float*>(pay + row * row_stride);
        }
    };
    unsigned use = 0;                        // of the sum in the making
    int q = 0, kc = 0;
    bool more = true;
    auto load = [&]() {                      // the next chunk into st
#pragma unroll
        for (int u = 0; u < 4; ++u) st[u] = *reinterpret_cast<const v4f*>(src[u] + kc);
        kc += FSK;
        if (kc >= k) {
            use &= ~(1u << q);
            kc = 0;
            more = use != 0;
            if (more) {
                q = __builtin_ctz(use);
                panel(q);
            }
        }
    };
    auto store = [&](int buf) {
#pragma unroll
        for (int u = 0; u < 4; ++u) *reinterpret_cast<v4f*>(sd + buf * FSB + u * 4096) = st[u];
    };
    const char* const opa = lds + (2 * wc) * 2048 + lane * 16;
    const char* const opb = lds + (4 + 2 * wr) * 2048 + lane * 16;
    constexpr bool kGroups = SUMS == kSumGroups;
    v16f tot[2][2];                          // kSumPanels: the panels before the current one
    if constexpr (SUMS == kSumPanels) {
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b) tot[a][b] = v16f{};
    }
    unsigned group = (1u << (kGroups ? P.sum : MPC_SYRK_MAXP)) - 1;
    do {
        use = todo & group;
        group <<= P.sum;
        if (kGroups && !use) continue;
        todo &= ~use;
        v16f acc[2][2];
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b) acc[a][b] = v16f{};
        q = __builtin_ctz(use);
        kc = 0;
        more = true;
        panel(q);
        load();
        store(0);
        bool staged = true;                  // a chunk is in the current buffer
        bool held = more;                    // a chunk is in st
        if (more) load();
        int left = k;                        // of the panel being multiplied
        for (int buf = 0; staged; buf ^= 1) {
            mpc_lds_barrier();
            if (live) {
                v4f A[2][2], B[2][2];
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int g = 0; g < 2; ++g) {
                        A[b][g] = *reinterpret_cast<const v4f*>(opa + buf * FSB + b * 2048 + g * 1024);
                        B[b][g] = *reinterpret_cast<const v4f*>(opb + buf * FSB + b * 2048 + g * 1024);
                    }
#pragma unroll
                for (int e = 0; e < 8; ++e)
#pragma unroll
                    for (int a = 0; a < 2; ++a)
#pragma unroll
                        for (int b = 0; b < 2; ++b) {
                            const float av = A[b][e >> 2][e & 3];
                            const float bv = B[a][e >> 2][e & 3];
                            acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x2f32(av, bv, acc[a][b], 0, 0, 0);
                        }
            }
            staged = held;
            if constexpr (SUMS == kSumPanels) {
                left -= FSK;
                if (left == 0 && held) {
                    left = k;
#pragma unroll
                    for (int a = 0; a < 2; ++a)
#pragma unroll
                        for (int b = 0; b < 2; ++b) {
                            tot[a][b] += acc[a][b];
                            acc[a][b] = v16f{};
                        }
                }
            }
            if (held) {
                store(buf ^ 1);              // (last read before this chunk's barrier)
                held = more;
                if (more) load();
            }
        }
        if (live) {
            if constexpr (SUMS == kSumPanels) {
#pragma unroll
                for (int a = 0; a < 2; ++a)
#pragma unroll
                    for (int b = 0; b < 2; ++b) acc[a][b] += tot[a][b];
            }
            int l = lane;                    // (C's offsets and masks are worked out here: kept
            if (kGroups) asm volatile("" : "+v"(l));     // over the loop they take 50 registers)
            c_frag<2> cv;
            load_c<2>(t, cv, l);
            store_c<2>(t, cv, acc, l);
        }
        t.Cs = C;
        if (kGroups && todo) mpc_lds_barrier();          // the buffers are rewritten
    } while (kGroups && todo);
}

// ---------------------------------------------------------------- FP32 x FP8 / BF16
// The pairs of an FP32 tile and an FP8 or BF16 one, as the three exact bf16
// products of mm_f32 (bit for bit the same sums).  Staged as above, but as bf16
// planes made once per workgroup: three of the FP32 side's 128 rows (hi, mid,
// lo by truncation), one of the other side's (its values are exact in bf16).
// In LDS a plane's 32-row block is 1 KB in operand order (16 bytes = k 8h .. +7
// of a lane).  Split by every wave for itself from row-per-lane loads, these
// pairs took longer than FP32 x FP32 ones.
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {      // the leading 16 bits of each
    return (__float_as_uint(a) >> 16) | (__float_as_uint(b) & 0xffff0000u);
}
constexpr int SPB = 16 * 1024;                // bytes of a buffer: (3 + 1) planes of 4 blocks

__device__ __forceinline__ void syrk_split_tile(float* __restrict__ C, int64_t m, int64_t ldc, int k,
                                                const mpc_syrk_panels& P, int64_t row_stride,
                                                int tile_rows, const syrk_shape& G, int64_t pid,
                                                const syrk_lists& L, char* lds) {
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    constexpr int TILE = MPC_SYRK_TILE;
    int64_t ti, tj;
    tile_of<TILE>(G, pid, ti, tj);
    const int64_t trow = (ti * TILE) / tile_rows, tcol = (tj * TILE) / tile_rows;
    const int rank = launch_rank_of(MPC_PREC_FP32, 2, 0);
    if (L.mode == 1) note_pair(L, P, tile_rows, trow, tcol, pid, rank);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wr = wave >> 1, wc = wave & 1;

    unsigned use = 0;                        // the panels of this launch
    int lo = 99;                             // first launch with work on the tile
    for (int q = 0; q < P.np; ++q) {
        const int slot = (P.p0 + q) % P.slots;
        const uint8_t* prec = P.prec + slot * 1024 + (P.rows0 - (int64_t)q * P.nb) / tile_rows;
        const int r = launch_rank(prec[trow], prec[tcol]);
        lo = r < lo ? r : lo;
        if (r == rank) use |= 1u << q;
    }
    if (!use) return;

    tile_ctx t;
    t.C = C;
    t.Cs = P.csrc && lo == rank ? P.csrc : C;
    t.ldc = ldc;
    t.m = m;
    t.rowbase = ti * TILE + 64 * wr;
    t.colbase = tj * TILE + 64 * wc;
    t.diag = ti == tj && wr == wc;
    const bool live = !(ti == tj && wr == 0 && wc == 1) && t.rowbase < m && t.colbase < m;

    // staging: thread (r4, l4) moves k 4 l4 .. +3 of rows r4 and r4 + 64 of each
    // side (past m the last row again)
    const int l4 = tid & 3, r4 = tid >> 2;
    char* const sd = lds + (r4 >> 5) * 1024 + (l4 >> 1) * 512 + (r4 & 31) * 16 + (l4 & 1) * 8;
    v4f sf[2];                               // the FP32 side
    uint32_t sl[2][2];                       // the other: FP8 bytes and scale, or four BF16
    const uint8_t *pay = nullptr, *sc = nullptr;
    bool col32 = false;                      // of the panel being loaded
    int plow = 0, slow = 0;                  // the other side's format: loaded panel, staged chunk
    bool scol32 = false;
    int64_t rf[2], rl[2];                    // rows of the two sides within the panel
    auto panel = [&](int q) {
        const int slot = (P.p0 + q) % P.slots;
        const int64_t roff = P.rows0 - (int64_t)q * P.nb;    // C row 0 within this panel
        const uint8_t* prec = P.prec + slot * 1024 + roff / tile_rows;
        pay = P.payload + slot * P.pstride;
        sc = P.scales + slot * P.sstride;
        col32 = prec[tcol] == MPC_PREC_FP32;
        plow = col32 ? prec[trow] : prec[tcol];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int64_t c = tj * TILE + 64 * u + r4, r = ti * TILE + 64 * u + r4;
            const int64_t cc = roff + (c < m ? c : m - 1), rc = roff + (r < m ? r : m - 1);
            rf[u] = col32 ? cc : rc;
            rl[u] = col32 ? rc : cc;
        }
    };
    int q = __builtin_ctz(use), kc = 0;
    bool more = true;
    auto load = [&]() {                      // the next chunk into sf, sl
        const int kk = kc + 4 * l4;
        scol32 = col32;
        slow = plow;
#pragma unroll
        for (int u = 0; u < 2; ++u) sf[u] = *reinterpret_cast<const v4f*>(pay + rf[u] * row_stride + 4 * kk);
        if (plow == MPC_PREC_BF16) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const u32x2 v = *reinterpret_cast<const u32x2*>(pay + rl[u] * row_stride + 2 * kk);
                sl[u][0] = v[0];
                sl[u][1] = v[1];
            }
        } else {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                sl[u][0] = *reinterpret_cast<const uint32_t*>(pay + mpc_f8_offset(rl[u], kk, row_stride));
                sl[u][1] = sc[rl[u] * (k >> 5) + (kk >> 5)];
            }
        }
        kc += FSK;
        if (kc >= k) {
            use &= ~(1u << q);
            kc = 0;
            more = use != 0;
            if (more) {
                q = __builtin_ctz(use);
                panel(q);
            }
        }
    };
    auto store = [&](int buf) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            char* d = sd + buf * SPB + u * 2048;
            v4f f = sf[u];
#pragma unroll
            for (int p = 0; p < 3; ++p) {
                *reinterpret_cast<u32x2*>(d + p * 4096) = u32x2{pack_bf16(f[0], f[1]), pack_bf16(f[2], f[3])};
#pragma unroll
                for (int e = 0; e < 4; ++e) f[e] -= __uint_as_float(__float_as_uint(f[e]) & 0xffff0000u);
            }
            u32x2 w = {sl[u][0], sl[u][1]};
            if (slow != MPC_PREC_BF16) {
                const float s = mpc_dev_exp2i((int)sl[u][1] - 127);
                v2f a, b;
                if (mpc_dev_is_e4m3(slow)) {
                    a = __builtin_amdgcn_cvt_pk_f32_fp8((int)sl[u][0], false);
                    b = __builtin_amdgcn_cvt_pk_f32_fp8((int)sl[u][0], true);
                } else {
                    a = __builtin_amdgcn_cvt_pk_f32_bf8((int)sl[u][0], false);
                    b = __builtin_amdgcn_cvt_pk_f32_bf8((int)sl[u][0], true);
                }
                w = u32x2{pack_bf16(a.x * s, a.y * s), pack_bf16(b.x * s, b.y * s)};
            }
            *reinterpret_cast<u32x2*>(d + 3 * 4096) = w;
        }
    };
    v16f acc[2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) acc[a][b] = v16f{};
    panel(q);
    load();
    store(0);
    bool col = scol32;                       // of the chunk in the current buffer
    bool staged = true;                      // a chunk is in the current buffer
    bool held = more;                        // a chunk is in sf, sl
    if (more) load();
    for (int buf = 0; staged; buf ^= 1) {
        mpc_lds_barrier();
        if (live) {
            const char* o = lds + buf * SPB + lane * 16;
            v8bf F[2][3], W[2];
#pragma unroll
            for (int b = 0; b < 2; ++b) {
#pragma unroll
                for (int p = 0; p < 3; ++p)
                    F[b][p] = *reinterpret_cast<const v8bf*>(o + p * 4096 + (2 * (col ? wc : wr) + b) * 1024);
                W[b] = *reinterpret_cast<const v8bf*>(o + 3 * 4096 + (2 * (col ? wr : wc) + b) * 1024);
            }
#pragma unroll
            for (int p = 0; p < 3; ++p)
#pragma unroll
                for (int a = 0; a < 2; ++a)
#pragma unroll
                    for (int b = 0; b < 2; ++b)
                        acc[a][b] = col ? __builtin_amdgcn_mfma_f32_32x32x16_bf16(F[b][p], W[a], acc[a][b], 0, 0, 0)
                                        : __builtin_amdgcn_mfma_f32_32x32x16_bf16(W[b], F[a][p], acc[a][b], 0, 0, 0);
        }
        staged = held;
        if (held) {
            col = scol32;
            store(buf ^ 1);                  // (last read before this chunk's barrier)
            held = more;
            if (more) load();
        }
    }
    if (!live) return;
    c_frag<2> cv;
    load_c<2>(t, cv);
    store_c<2>(t, cv, acc);
}

// ---------------------------------------------------------------- FP8 x FP8
// The pairs of two 8-bit tiles with element formats FA (columns) and FB (rows),
// v_mfma_scale_f32_32x32x64_f8f6f4 in the K order of mm_fp8 (bit for bit the
// same sums).  The payload is in operand order already; staging it means that
// a workgroup reads each operand once instead of twice, and that three chunks
// of 64 K are in flight: two in registers, one in the LDS buffer being filled.
// A block of 32 rows is 2 KB per chunk, the lanes' first 16 bytes and then
// their second, so that every read is 1 KB in lane order.  The chunk's two
// scale bytes of a row go through LDS as well.
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
constexpr int F8B = 8 * 2048 + 512;           // bytes of a buffer: 8 blocks, 256 rows' scales

template <int FA, int FB>
__device__ __forceinline__ void syrk_f8_tile(float* __restrict__ C, int64_t m, int64_t ldc, int k,
                                             const mpc_syrk_panels& P, int64_t row_stride,
                                             int tile_rows, const syrk_shape& G, int64_t pid,
                                             const syrk_lists& L, char* lds) {
    constexpr int TILE = MPC_SYRK_TILE;
    int64_t ti, tj;
    tile_of<TILE>(G, pid, ti, tj);
    const int64_t trow = (ti * TILE) / tile_rows, tcol = (tj * TILE) / tile_rows;
    const int rank = launch_rank_of(MPC_PREC_E4M3, FA, FB);
    if (L.mode == 1) note_pair(L, P, tile_rows, trow, tcol, pid, rank);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wr = wave >> 1, wc = wave & 1;

    unsigned use = 0;                        // the panels of this launch
    int lo = 99;                             // first launch with work on the tile
    for (int q = 0; q < P.np; ++q) {
        const int slot = (P.p0 + q) % P.slots;
        const uint8_t* prec = P.prec + slot * 1024 + (P.rows0 - (int64_t)q * P.nb) / tile_rows;
        const int r = launch_rank(prec[trow], prec[tcol]);
        lo = r < lo ? r : lo;
        if (r == rank) use |= 1u << q;
    }
    if (!use) return;

    tile_ctx t;
    t.C = C;
    t.Cs = P.csrc && lo == rank ? P.csrc : C;
    t.ldc = ldc;
    t.m = m;
    t.rowbase = ti * TILE + 64 * wr;
    t.colbase = tj * TILE + 64 * wc;
    t.diag = ti == tj && wr == wc;
    const bool live = !(ti == tj && wr == 0 && wc == 1) && t.rowbase < m && t.colbase < m;

    // staging: wave w moves blocks 2w and 2w + 1 (blocks 0..3 the columns of C,
    // 4..7 its rows; past m the last one again), lane l 32 bytes of each; thread
    // t the scales of operand row t
    const int64_t bmax = (m - 1) & ~(int64_t)31;
    int64_t blk[2], srow;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int b = 2 * wave + u;
        const int64_t r = (b < 4 ? tj : ti) * TILE + 32 * (b & 3);
        blk[u] = r < bmax ? r : bmax;
    }
    srow = (tid < 128 ? tj : ti) * TILE + (tid & 127);
    if (srow >= m) srow = m - 1;
    v4u st[2][2][2];                       // [set][block][half]
    uint32_t ss[2];
    const uint8_t *pb[2] = {}, *ps = nullptr;
    auto panel = [&](int q) {
        const int slot = (P.p0 + q) % P.slots;
        const int64_t roff = P.rows0 - (int64_t)q * P.nb;    // C row 0 within this panel
        const uint8_t* pay = P.payload + slot * P.pstride;
#pragma unroll
        for (int u = 0; u < 2; ++u) pb[u] = pay + (roff + blk[u]) * row_stride + lane * 32;
        ps = P.scales + slot * P.sstride + (roff + srow) * (k >> 5);
    };
    int q = __builtin_ctz(use), kc = 0;
    int left = 0;                            // chunks not loaded yet
    for (unsigned v = use; v; v &= v - 1) left += k >> 6;
    auto load = [&](v4u (&v)[2][2], uint32_t& s) {         // the next chunk
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int g = 0; g < 2; ++g)
                v[u][g] = *reinterpret_cast<const v4u*>(pb[u] + (int64_t)(kc >> 6) * 2048 + 16 * g);
        s = *reinterpret_cast<const uint16_t*>(ps + (kc >> 5));
        --left;
        kc += 64;
        if (kc >= k) {
            use &= ~(1u << q);
            kc = 0;
            if (use) {
                q = __builtin_ctz(use);
                panel(q);
            }
        }
    };
    auto store = [&](const v4u (&v)[2][2], uint32_t s, int buf) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int g = 0; g < 2; ++g)
                *reinterpret_cast<v4u*>(lds + buf * F8B + (2 * wave + u) * 2048 + g * 1024 + lane * 16) = v[u][g];
        *reinterpret_cast<uint16_t*>(lds + buf * F8B + 8 * 2048 + 2 * tid) = (uint16_t)s;
    };
    v16f acc[2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) acc[a][b] = v16f{};
    auto operand = [&](const char* o) {
        const v4u x = *reinterpret_cast<const v4u*>(o), y = *reinterpret_cast<const v4u*>(o + 1024);
        return v8i{(int)x[0], (int)x[1], (int)x[2], (int)x[3], (int)y[0], (int)y[1], (int)y[2], (int)y[3]};
    };
    auto multiply = [&](int buf) {
        const char* o = lds + buf * F8B;
        const char* s = o + 8 * 2048 + 2 * (lane & 31) + (lane >> 5);
        v8i A[2], B[2];
        int sa[2], sb[2];
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            A[b] = operand(o + (2 * wc + b) * 2048 + lane * 16);
            B[b] = operand(o + (4 + 2 * wr + b) * 2048 + lane * 16);
            sa[b] = *reinterpret_cast<const uint8_t*>(s + 64 * (2 * wc + b));
            sb[b] = *reinterpret_cast<const uint8_t*>(s + 64 * (4 + 2 * wr + b));
        }
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b)
                acc[a][b] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
                    A[b], B[a], acc[a][b], FA, FB, 0, sa[b], 0, sb[a]);
    };
    panel(q);
    int todo = left;                         // chunks not multiplied yet
    load(st[0], ss[0]);
    if (left) load(st[1], ss[1]);
    store(st[0], ss[0], 0);
    if (left) load(st[0], ss[0]);
    // chunk c is in buffer c & 1, c + 1 in set (c + 1) & 1, c + 2 in set c & 1
    for (;;) {
        mpc_lds_barrier();
        if (todo > 1) {
            store(st[1], ss[1], 1);
            if (left) load(st[1], ss[1]);
        }
        if (live) multiply(0);
        if (--todo == 0) break;
        mpc_lds_barrier();
        if (todo > 1) {
            store(st[0], ss[0], 0);
            if (left) load(st[0], ss[0]);
        }
        if (live) multiply(1);
        if (--todo == 0) break;
    }
    if (!live) return;
    c_frag<2> cv;
    load_c<2>(t, cv);
    store_c<2>(t, cv, acc);
}

// ---------------------------------------------------------------- 16-bit classes
// The pairs of the BF16 class (at least one BF16 tile, the other BF16, FP8 or, in
// mpc_syrk only, FP16, whose values lose their last three bits; CLS BF16) and of
// two FP16 tiles (CLS FP16), in the K order of mm_16 (bit for bit the same sums),
// staged like the bf16 planes above with one plane a side.
constexpr int S16B = 8 * 1024;                // bytes of a buffer

template <int CLS>
__device__ __forceinline__ void syrk_16_tile(float* __restrict__ C, int64_t m, int64_t ldc, int k,
                                             const mpc_syrk_panels& P, int64_t row_stride,
                                             int tile_rows, const syrk_shape& G, int64_t pid,
                                             const syrk_lists& L, char* lds) {
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    constexpr int TILE = MPC_SYRK_TILE;
    int64_t ti, tj;
    tile_of<TILE>(G, pid, ti, tj);
    const int64_t trow = (ti * TILE) / tile_rows, tcol = (tj * TILE) / tile_rows;
    const int rank = launch_rank_of(CLS, 0, 0);
    if (L.mode == 1) note_pair(L, P, tile_rows, trow, tcol, pid, rank);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wr = wave >> 1, wc = wave & 1;

    unsigned use = 0;                        // the panels of this launch
    int lo = 99;                             // first launch with work on the tile
    for (int q = 0; q < P.np; ++q) {
        const int slot = (P.p0 + q) % P.slots;
        const uint8_t* prec = P.prec + slot * 1024 + (P.rows0 - (int64_t)q * P.nb) / tile_rows;
        const int r = launch_rank(prec[trow], prec[tcol]);
        lo = r < lo ? r : lo;
        if (r == rank) use |= 1u << q;
    }
    if (!use) return;

    tile_ctx t;
    t.C = C;
    t.Cs = P.csrc && lo == rank ? P.csrc : C;
    t.ldc = ldc;
    t.m = m;
    t.rowbase = ti * TILE + 64 * wr;
    t.colbase = tj * TILE + 64 * wc;
    t.diag = ti == tj && wr == wc;
    const bool live = !(ti == tj && wr == 0 && wc == 1) && t.rowbase < m && t.colbase < m;

    // staging: thread (r4, l4) moves k 4 l4 .. +3 of operand rows r4 + 64 u (u < 2:
    // the columns of C, else its rows; past m the last row again)
    const int l4 = tid & 3, r4 = tid >> 2;
    char* const sd = lds + (r4 >> 5) * 1024 + (l4 >> 1) * 512 + (r4 & 31) * 16 + (l4 & 1) * 8;
    uint32_t st[4][2];                       // four 16-bit values, or FP8 bytes and scale
    const uint8_t *pay = nullptr, *sc = nullptr;
    int pf[2] = {0, 0}, sf[2] = {0, 0};      // formats of the sides: loaded panel, staged chunk
    int64_t row[4];
    auto panel = [&](int q) {
        const int slot = (P.p0 + q) % P.slots;
        const int64_t roff = P.rows0 - (int64_t)q * P.nb;    // C row 0 within this panel
        const uint8_t* prec = P.prec + slot * 1024 + roff / tile_rows;
        pay = P.payload + slot * P.pstride;
        sc = P.scales + slot * P.sstride;
        pf[0] = prec[tcol];
        pf[1] = prec[trow];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int64_t r = (u < 2 ? tj : ti) * TILE + 64 * (u & 1) + r4;
            row[u] = roff + (r < m ? r : m - 1);
        }
    };
    int q = __builtin_ctz(use), kc = 0;
    bool more = true;
    auto load = [&]() {                      // the next chunk into st
        const int kk = kc + 4 * l4;
#pragma unroll
        for (int side = 0; side < 2; ++side) {
            sf[side] = pf[side];
            if (CLS == MPC_PREC_FP16 || pf[side] == MPC_PREC_BF16 || pf[side] == MPC_PREC_FP16) {
#pragma unroll
                for (int u = 2 * side; u < 2 * side + 2; ++u) {
                    const u32x2 v = *reinterpret_cast<const u32x2*>(pay + row[u] * row_stride + 2 * kk);
                    st[u][0] = v[0];
                    st[u][1] = v[1];
                }
            } else {
#pragma unroll
                for (int u = 2 * side; u < 2 * side + 2; ++u) {
                    st[u][0] = *reinterpret_cast<const uint32_t*>(pay + mpc_f8_offset(row[u], kk, row_stride));
                    st[u][1] = sc[row[u] * (k >> 5) + (kk >> 5)];
                }
            }
        }
        kc += FSK;
        if (kc >= k) {
            use &= ~(1u << q);
            kc = 0;
            more = use != 0;
            if (more) {
                q = __builtin_ctz(use);
                panel(q);
            }
        }
    };
    auto store = [&](int buf) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            u32x2 w = {st[u][0], st[u][1]};
            if (CLS != MPC_PREC_FP16 && sf[u >> 1] == MPC_PREC_FP16) {
                float f[4];
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    f[e] = (float)__builtin_bit_cast(_Float16, (unsigned short)(st[u][e >> 1] >> (16 * (e & 1))));
                w = u32x2{pack_bf16(f[0], f[1]), pack_bf16(f[2], f[3])};
            } else if (CLS != MPC_PREC_FP16 && sf[u >> 1] != MPC_PREC_BF16) {
                const float s = mpc_dev_exp2i((int)st[u][1] - 127);
                v2f a, b;
                if (mpc_dev_is_e4m3(sf[u >> 1])) {
                    a = __builtin_amdgcn_cvt_pk_f32_fp8((int)st[u][0], false);
                    b = __builtin_amdgcn_cvt_pk_f32_fp8((int)st[u][0], true);
                } else {
                    a = __builtin_amdgcn_cvt_pk_f32_bf8((int)st[u][0], false);
                    b = __builtin_amdgcn_cvt_pk_f32_bf8((int)st[u][0], true);
                }
                w = u32x2{pack_bf16(a.x * s, a.y * s), pack_bf16(b.x * s, b.y * s)};
            }
            *reinterpret_cast<u32x2*>(sd + buf * S16B + u * 2048) = w;
        }
    };
    v16f acc[2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) acc[a][b] = v16f{};
    panel(q);
    load();
    store(0);
    bool staged = true;                      // a chunk is in the current buffer
    bool held = more;                        // a chunk is in st
    if (more) load();
    for (int buf = 0; staged; buf ^= 1) {
        mpc_lds_barrier();
        if (live) {
            const char* o = lds + buf * S16B + lane * 16;
            v4u A[2], B[2];
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                A[b] = *reinterpret_cast<const v4u*>(o + (2 * wc + b) * 1024);
                B[b] = *reinterpret_cast<const v4u*>(o + (4 + 2 * wr + b) * 1024);
            }
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    if constexpr (CLS == MPC_PREC_FP16)
                        acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                            __builtin_bit_cast(v8h, A[b]), __builtin_bit_cast(v8h, B[a]), acc[a][b], 0, 0, 0);
                    else
                        acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                            __builtin_bit_cast(v8bf, A[b]), __builtin_bit_cast(v8bf, B[a]), acc[a][b], 0, 0, 0);
                }
        }
        staged = held;
        if (held) {
            store(buf ^ 1);                  // (last read before this chunk's barrier)
            held = more;
            if (more) load();
        }
    }
    if (!live) return;
    c_frag<2> cv;
    load_c<2>(t, cv);
    store_c<2>(t, cv, acc);
}

// The staged kernels by launch rank: 0-3 FP8 element pairs, 4 BF16, 5 FP16,
// 6 FP32 x FP32, 7 FP32 x FP8 / BF16; kF32Groups, kF32Panels: 6 with other sums.
constexpr int kF32Groups = 9, kF32Panels = 10;
template <int RANK, bool LISTED>
__global__ __launch_bounds__(256, 2) void syrk_staged_kernel(float* __restrict__ C, int64_t m, int64_t ldc,
                                                          int k, const mpc_syrk_panels P,
                                                          int64_t row_stride, int tile_rows,
                                                          const mpc_small* __restrict__ sm, int64_t npair,
                                                          int64_t per_xcd, const syrk_shape G,
                                                          const syrk_lists L) {
    constexpr int kBuf = RANK < 4 ? F8B : RANK < 6 ? S16B : RANK == 7 ? SPB : FSB;
    __shared__ __align__(16) char lds[2 * kBuf];
    if (sm && sm->info != 0) return;
    auto tile = [&](int64_t pid) {
        if constexpr (RANK < 4)
            syrk_f8_tile<RANK / 2, RANK % 2>(C, m, ldc, k, P, row_stride, tile_rows, G, pid, L, lds);
        else if constexpr (RANK < 6)
            syrk_16_tile<RANK == 4 ? MPC_PREC_BF16 : MPC_PREC_FP16>(C, m, ldc, k, P, row_stride, tile_rows,
                                                                    G, pid, L, lds);
        else if constexpr (RANK == 6 || RANK == kF32Groups || RANK == kF32Panels)
            syrk_f32_tile<RANK == 6 ? kSumAll : RANK == kF32Groups ? kSumGroups : kSumPanels>(
                C, m, ldc, k, P, row_stride, tile_rows, G, pid, L, lds);
        else
            syrk_split_tile(C, m, ldc, k, P, row_stride, tile_rows, G, pid, L, lds);
    };
    if constexpr (LISTED) {
        constexpr int rank = RANK > 7 ? 6 : RANK;
        const int count = L.base[rank];
        const int* list = L.base + kListHead + (int64_t)rank * L.cap;
        for (int it = blockIdx.x; it < count; it += gridDim.x) {
            tile(list[it]);
            mpc_lds_barrier();               // the buffers are rewritten
        }
        return;
    }
    const int64_t b = blockIdx.x;
    const int64_t pid = (b & 7) * per_xcd + (b >> 3);
    if (pid < npair) tile(pid);
}

}  // namespace

static int syrk_check(int64_t ldc, int k, int tile_rows) {
    if (ldc > (int64_t(1) << 22)) {       // 32-bit buffer offsets of a 128-column tile
        mpc_set_error("syrk: ldc %lld exceeds 2^22", (long long)ldc);
        return MPC_ERR_ARG;
    }
    if (k % 64 || tile_rows % MPC_SYRK_TILE) {
        mpc_set_error("syrk: k (%d) must be a multiple of 64 and tile_rows (%d) of 128", k,
                      tile_rows);
        return MPC_ERR_ARG;
    }
    return 0;
}

// launch geometry over tile columns [tcol0, tcol1) of the lower triangle
struct syrk_grid {
    int64_t mt, npair, per_xcd, tcol0;
    syrk_shape shape;
    dim3 grid;
};
// trow0 > 0: the rectangle of tile rows [trow0, mt) x tile columns [tcol0,
// tcol1) (trow0 >= tcol1: strictly below the diagonal)
static bool syrk_geometry(int64_t m, int tile, int64_t tcol0, int64_t tcol1, syrk_grid& g,
                          int64_t trow0 = 0) {
    g.mt = (m + tile - 1) / tile;
    if (tcol1 < 0 || tcol1 > g.mt) tcol1 = g.mt;
    if (tcol0 >= tcol1) return false;
    if (trow0 > 0) {
        if (trow0 >= g.mt) return false;
        g.npair = (g.mt - trow0) * (tcol1 - tcol0);
        g.shape = syrk_shape{g.mt, tcol0, tcol1, trow0, tcol1 - tcol0};
    } else {
        auto start = [&](int64_t c) { return c * g.mt - c * (c - 1) / 2; };
        g.npair = start(tcol1) - start(tcol0);
        g.shape = syrk_shape{g.mt, tcol0, tcol1, 0, 0};
    }
    g.per_xcd = (g.npair + 7) / 8;
    g.tcol0 = tcol0;
    g.grid = dim3((unsigned)(g.per_xcd * 8));
    return true;
}

// MPC_SYRK_LAUNCH(KERNEL, template arguments but LISTED)
#define MPC_SYRK_LAUNCH(KERNEL, ...)                                                           \
    do {                                                                                       \
        const syrk_lists L_ = next_lists();                                                    \
        if (L_.mode == 2)                                                                      \
            hipLaunchKernelGGL((KERNEL<__VA_ARGS__, true>), list_grid, dim3(256), 0, st, C, m, \
                               ldc, k, P, row_stride, tile_rows, sm, g.npair, g.per_xcd,       \
                               g.shape, L_);                                                   \
        else                                                                                   \
            hipLaunchKernelGGL((KERNEL<__VA_ARGS__, false>), g.grid, dim3(256), 0, st, C, m,   \
                               ldc, k, P, row_stride, tile_rows, sm, g.npair, g.per_xcd,       \
                               g.shape, L_);                                                   \
    } while (0)

// C(lower) -= Q Q^T restricted to the tile columns [tcol0, tcol1) of C, one
// panel.  mixed = 0: tiles of MPC_SYRK_TILE, one launch per compute class
// present in class_mask (and per FP8 element-format pair in fp8_mask; bit 0
// E4M3 elements, bit 1 E5M2).  mixed = 1: 64-row tiles in ONE launch in which
// each workgroup takes its own pair's class (the block column on the
// critical path of the look-ahead: a launch per class would serialise, and a
// 128-row tile per workgroup leaves most of the chip idle there).
int mpc_launch_syrk_classes(hipStream_t st, float* C, int64_t m, int64_t ldc, int k,
                            const uint8_t* payload, int64_t row_stride, const uint8_t* scales,
                            int tile_rows, const uint8_t* prec_of_tile, const mpc_small* sm,
                            unsigned class_mask, unsigned fp8_mask, int64_t tcol0, int64_t tcol1,
                            int mixed, int* lists, int64_t trow0) {
    if (mixed != 0 && mixed != 1) {
        mpc_set_error("syrk: mixed must be 0 or 1 (got %d)", mixed);
        return MPC_ERR_ARG;
    }
    mpc_syrk_panels P{};
    P.payload = payload;
    P.scales = scales;
    P.prec = prec_of_tile;
    P.slots = 1;
    P.np = 1;
    P.nb = tile_rows;
    return mpc_launch_syrk_panels(st, C, m, ldc, k, P, row_stride, tile_rows, sm, tcol0, tcol1,
                                  mixed ? 1 : 2, class_mask, fp8_mask, lists, trow0);
}

__global__ void clear_list_heads_kernel(int* __restrict__ heads) {
    if (threadIdx.x < kListHead) heads[threadIdx.x] = 0;
}

int64_t mpc_syrk_list_ints(int64_t m, int tile) {
    const int64_t mt = (m + tile - 1) / tile;
    return kListHead + 9 * (mt * (mt + 1) / 2);
}

int mpc_launch_syrk_panels(hipStream_t st, float* C, int64_t m, int64_t ldc, int k,
                           const mpc_syrk_panels& P, int64_t row_stride, int tile_rows,
                           const mpc_small* sm, int64_t tcol0, int64_t tcol1, int qa,
                           unsigned class_mask, unsigned fp8_mask, int* lists, int64_t trow0) {
    if (m <= 0) return 0;
    if ((qa != 1 && qa != 2) || P.np < 1 || P.np > MPC_SYRK_MAXP || P.slots < 1 ||
        P.rows0 - (int64_t)(P.np - 1) * P.nb < 0 || P.rows0 % tile_rows || P.nb % tile_rows) {
        mpc_set_error("syrk: bad panel set (qa %d, np %d of at most %d, rows0 %lld, nb %d)", qa,
                      P.np, MPC_SYRK_MAXP, (long long)P.rows0, P.nb);
        return MPC_ERR_ARG;
    }
    int rc = syrk_check(ldc, k, tile_rows);
    if (rc) return rc;
    syrk_grid g;
    if (trow0 > 0 && tcol1 >= 0 && trow0 < tcol1) {
        mpc_set_error("syrk: rectangle rows from tile %lld overlap its columns up to %lld",
                      (long long)trow0, (long long)tcol1);
        return MPC_ERR_ARG;
    }
    if (!syrk_geometry(m, 64 * qa, tcol0, tcol1, g, trow0)) return 0;
    syrk_lists none{nullptr, 0, 0};
    if (qa == 1) {
        // latency-bound: as many resident workgroups as possible.  The K loop
        // unrolled for k = 256 took 240 VGPRs (two workgroups per CU, two
        // rounds of workgroups at the first steps); the runtime-k loop takes
        // 152 (three per CU) and made the solve 0.3 ms faster.
        hipLaunchKernelGGL((syrk_kernel<1, false, false>), g.grid, dim3(256), 0, st, C, m, ldc, k, P,
                           row_stride, tile_rows, sm, g.npair, g.per_xcd, g.shape, none);
        MPC_LAUNCH_CHECK();
        return 0;
    }
    // one launch per compute class (and FP8 element pair) in the masks, in
    // launch-rank order; with lists, the first one builds the others' lists
    const bool e4 = (class_mask & (1u << MPC_PREC_E4M3)) && (fp8_mask & 1u);
    const bool e5 = (class_mask & (1u << MPC_PREC_E4M3)) && (fp8_mask & 2u);
    const bool f32 = class_mask & (1u << MPC_PREC_FP32);
    const bool f32s = f32 && (class_mask & ((1u << MPC_PREC_E4M3) | (1u << MPC_PREC_BF16)));
    const bool f32h = f32 && (class_mask & (1u << MPC_PREC_FP16));
    const int nlaunch = (int)e4 + 2 * (int)(e4 && e5) + (int)e5 +
                        (int)(bool)(class_mask & (1u << MPC_PREC_BF16)) +
                        (int)(bool)(class_mask & (1u << MPC_PREC_FP16)) + (int)f32 + (int)f32s +
                        (int)f32h;
    const bool use_lists = lists && nlaunch > 1;
    int launched = 0;
    if (use_lists) hipLaunchKernelGGL(clear_list_heads_kernel, dim3(1), dim3(64), 0, st, lists);
    // later launches: a grid that strides over the list (at most the tile count)
    const dim3 list_grid((unsigned)std::min<int64_t>(g.per_xcd * 8, 2048));
    auto next_lists = [&]() {
        syrk_lists L{use_lists ? lists : nullptr, (int)g.npair,
                     use_lists ? (launched == 0 ? 1 : 2) : 0};
        ++launched;
        return L;
    };
    if (e4) MPC_SYRK_LAUNCH(syrk_staged_kernel, 0);
    if (e4 && e5) {
        MPC_SYRK_LAUNCH(syrk_staged_kernel, 1);
        MPC_SYRK_LAUNCH(syrk_staged_kernel, 2);
    }
    if (e5) MPC_SYRK_LAUNCH(syrk_staged_kernel, 3);
    if (class_mask & (1u << MPC_PREC_BF16)) MPC_SYRK_LAUNCH(syrk_staged_kernel, 4);
    if (class_mask & (1u << MPC_PREC_FP16)) MPC_SYRK_LAUNCH(syrk_staged_kernel, 5);
    if (f32 && P.sum == 1 && P.np > 1) MPC_SYRK_LAUNCH(syrk_staged_kernel, kF32Panels);
    else if (f32 && P.sum > 0 && P.np > P.sum) MPC_SYRK_LAUNCH(syrk_staged_kernel, kF32Groups);
    else if (f32) MPC_SYRK_LAUNCH(syrk_staged_kernel, 6);        // FP32 x FP32
    if (f32s) MPC_SYRK_LAUNCH(syrk_staged_kernel, 7);            // FP32 x FP8 / BF16 (split)
    if (f32h) MPC_SYRK_LAUNCH(syrk_kernel, 2, true);             // FP32 x FP16
    MPC_LAUNCH_CHECK();
    return 0;
}
#undef MPC_SYRK_LAUNCH

int mpc_launch_syrk(hipStream_t st, float* C, int64_t m, int64_t ldc, int k,
                    const uint8_t* payload, int64_t row_stride, const uint8_t* scales,
                    int tile_rows, const uint8_t* prec_of_tile, const mpc_small* sm) {
    const unsigned all = (1u << MPC_PREC_E4M3) | (1u << MPC_PREC_BF16) | (1u << MPC_PREC_FP16) |
                         (1u << MPC_PREC_FP32);
    return mpc_launch_syrk_classes(st, C, m, ldc, k, payload, row_stride, scales, tile_rows,
                                   prec_of_tile, sm, all, 3u, 0, -1, 0);
}
