// Rows A2 (up to 8 tokens) and the generic fallback of A3/A4: affine quantized
// GEMV. One or two tokens at 4 bits: qmv_dot2_kernel. Up to 8 tokens, 16-bit T:
// qms_kernel. fp32, and shapes neither takes: qmv_kernel.
#include <math.h>

#include "mi_qmm_common.h"

namespace mi {
namespace {

// ---------------------------------------------------------------------------
// GEMV / generic path

template <typename T, int VPC>
__device__ __forceinline__ void load_x(const T *xp, float (&xf)[VPC]) {
    if constexpr (sizeof(T) == 4) {
#pragma unroll
        for (int i = 0; i < VPC; i += 4) {
            const uint4 r = ld16(xp + i);
            xf[i] = __uint_as_float(r.x);
            xf[i + 1] = __uint_as_float(r.y);
            xf[i + 2] = __uint_as_float(r.z);
            xf[i + 3] = __uint_as_float(r.w);
        }
    } else {
#pragma unroll
        for (int i = 0; i < VPC; i += 8) {
            float f[8];
            unpack8<T>(ld16(xp + i), f);
#pragma unroll
            for (int j = 0; j < 8; ++j) xf[i + j] = f[j];
        }
    }
}

// a b + c d with the rounding written out: left to contraction, the compiler
// fuses one product or the other, and an epilogue's fp32 sums may differ from the
// plain projection's in their last bit.
__device__ __forceinline__ float fma_mul(float a, float b, float c, float d) {
#pragma clang fp contract(off)
    return __builtin_fmaf(a, b, c * d);
}

template <typename T, int BITS, int MR, int EPI>
__global__ __launch_bounds__(256) void qmv_kernel(QParams p) {
    constexpr int P = epi_parts(EPI);
    constexpr int VPW = 32 / BITS;
    constexpr int VPC = 4 * VPW;
    const int lane = threadIdx.x & 63;
    const int j = lane & 15;
    int64_t nb = (int64_t)blockIdx.x * 16;
    const Bound bd = bind<EPI>(p, nb);
    const int64_t n = nb + (threadIdx.x >> 6) * 4 + (lane >> 4);
    const int64_t m0 = (int64_t)blockIdx.y * MR;
    const int64_t K = p.K, cpr = K / VPC, G = K >> p.gs_log2;
    const int mr = (int)((p.M - m0) < MR ? (p.M - m0) : MR);
    const T *x = (const T *)p.x + m0 * K;

    float acc[P][MR];
#pragma unroll
    for (int q = 0; q < P; ++q)
#pragma unroll
        for (int m = 0; m < MR; ++m) acc[q][m] = 0.0f;

    // out-of-range rows/tokens read clamped, valid addresses (no branch around
    // loads); their sums are never stored
    const int64_t nrow = n < bd.Nout ? n : bd.Nout - 1;
    const uint32_t *wr[P];
    const T *sr[P];
    const T *br[P];
#pragma unroll
    for (int q = 0; q < P; ++q) {
        const int64_t row = bd.noff(q) + nrow;
        wr[q] = bd.w(q) + row * (K / VPW);
        sr[q] = (const T *)bd.s(q) + row * G;
        br[q] = (const T *)bd.b(q) + row * G;
    }
#pragma unroll 2
    for (int64_t c = j; c < cpr; c += 16) {
        const int64_t k0 = c * VPC;
        float qf[P][VPC];
        float sc[P], bi[P];
#pragma unroll
        for (int q = 0; q < P; ++q) {
            const uint4 wv = ld16_nt(wr[q] + c * 4);
            const uint32_t words[4] = {wv.x, wv.y, wv.z, wv.w};
#pragma unroll
            for (int i = 0; i < VPC; ++i)
                qf[q][i] =
                    (float)((words[i / VPW] >> ((i % VPW) * BITS)) & ((1u << BITS) - 1u));
            sc[q] = (float)sr[q][k0 >> p.gs_log2];
            bi[q] = (float)br[q][k0 >> p.gs_log2];
        }
#pragma unroll
        for (int m = 0; m < MR; ++m) {
            float xf[VPC];
            load_x<T, VPC>(x + (m < mr ? m : mr - 1) * K + k0, xf);
            float dx = 0.0f;
#pragma unroll
            for (int i = 0; i < VPC; ++i) dx += xf[i];
#pragma unroll
            for (int q = 0; q < P; ++q) {
                float dq = 0.0f;
#pragma unroll
                for (int i = 0; i < VPC; ++i) dq = __builtin_fmaf(xf[i], qf[q][i], dq);
                // every instance rounds this as fma(bi, dx, sc dq): left to
                // contraction, all but the split(3) ones at 4 bits do. (Written
                // out everywhere, the compiler sinks the weight loads to their
                // use: 8-bit dual, one token, 7656 x 1792 8.2 -> 17.4 us.)
                if constexpr (P == 3 && BITS == 4)
                    acc[q][m] += fma_mul(bi[q], dx, sc[q], dq);
                else
                    acc[q][m] += sc[q] * dq + bi[q] * dx;
            }
        }
    }
#pragma unroll
    for (int q = 0; q < P; ++q)
#pragma unroll
        for (int m = 0; m < MR; ++m) {
            acc[q][m] = row16_sum(acc[q][m]);  // the row's 16 lanes
        }
    if (j == 0 && n < bd.Nout) {
#pragma unroll
        for (int m = 0; m < MR; ++m) {
            if (m < mr) {
                float a[P];
#pragma unroll
                for (int q = 0; q < P; ++q) a[q] = acc[q][m];
                epi1<T, EPI>(p, bd, m0 + m, n, a);
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Decode GEMV (one token; two up to K = 4096, four up to K = 512; 4-bit, bf16/fp16): the nibbles never go through a
// float conversion. (w >> 4j) & 0x000F000F | MAGIC packs nibbles j and j+4 of a
// word as the two 16-bit floats MAG + q exactly (bf16: 0x4300 = 128, ulp 1 up
// to 256; fp16: 0x6400 = 1024, ulp 1), so one v_and_or makes a pair and
// v_dot2_f32_{bf16,f16} multiplies it with the x pair (x[k], x[k+4]):
//   sum_k x_k (MAG + q_k) = D  ->  s*sum(x q) + b*sum(x) = s*D + (b - MAG*s)*sum(x).
// x is staged once per workgroup in LDS already permuted into those pairs,
// with per-32-value chunk sums. Weight chunks are loaded 8 per lane before use.

template <typename T> struct Magic;
template <> struct Magic<bf16> {
    static constexpr uint32_t pair = 0x43004300u;
    static constexpr float value = 128.0f;
    static __device__ __forceinline__ float dot2(uint32_t a, uint32_t b, float c) {
        typedef __bf16 v2 __attribute__((ext_vector_type(2)));
        return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(v2, a), __builtin_bit_cast(v2, b),
                                               c, false);
    }
};
template <> struct Magic<f16> {
    static constexpr uint32_t pair = 0x64006400u;
    static constexpr float value = 1024.0f;
    static __device__ __forceinline__ float dot2(uint32_t a, uint32_t b, float c) {
        typedef _Float16 v2 __attribute__((ext_vector_type(2)));
        return __builtin_amdgcn_fdot2(__builtin_bit_cast(v2, a), __builtin_bit_cast(v2, b), c,
                                      false);
    }
};

// ((w >> 4j) & 0x000F000F) | Mg::pair -- the magic pair of nibbles j and
// j + 4 of w -- in fewer instructions: the even and odd nibbles as bytes
// (lo, hi) once per word, then one byte permute per pair that interleaves two
// of those bytes with the magic exponent byte. Same bits.
template <typename T>
__device__ __forceinline__ uint32_t magic_pair(uint32_t w, int j) {
    constexpr uint32_t e = (Magic<T>::pair >> 8) & 0xFFu;  // the exponent byte (0x43 / 0x64)
    const uint32_t lo = w & 0x0F0F0F0Fu, hi = (w >> 4) & 0x0F0F0F0Fu;
    // v_perm_b32 bytes: 0..3 from the second operand, 4..7 from the first
    const uint32_t sel = (j & 2) ? 0x04030401u : 0x04020400u;
    return __builtin_amdgcn_perm(e * 0x01010101u, (j & 1) ? hi : lo, sel);
}

constexpr int QV_BATCH = 8;  // 16-byte weight chunks in flight per lane

inline int64_t qmv_dot2_lds_bytes(int mr, int64_t K) { return mr * K * 2 + mr * (K / 32) * 4; }

// A workgroup of blockDim.x / 64 waves owns 64 / LPR output rows per wave (LPR
// lanes a row, below): 4 waves, or for single-output epilogues without PF up
// to 16 (WIDE), sized by the host so the grid spreads the rows evenly over the
// CUs. Wider workgroups are not used for the others: batches of two or three
// weight rows take more than the 128 registers a lane may hold in a 16-wave
// workgroup, and under PF the staging barriers wait for the x loads of every
// wave, which queue behind the weight stream (one 10-wave workgroup per CU at
// N = 9728 waited 2.3 us for x against 1.5 us with 4 waves: 6.1 against 5.6
// us a launch).
// PF (4 waves at 16 lanes a row; also wide workgroups of a row a wave): the x
// loads, then the first weight batch, are issued before x is staged, so the
// weight stream runs under the staging and its two barriers (x first: vmcnt
// retires in issue order, so waiting for x then leaves the weights in
// flight). Each thread holds at most two x chunks (K / 8 <= 2 blockDim.x). It
// costs the batch registers through the staging, which pays when the grid
// fits the chip in one round and not at N = 151936.
constexpr bool qmv_dot2_wide_ok(int epi) { return epi_parts(epi) == 1 && epi != EPI_GROUP3; }

// LPR: lanes per output row, 16 (4 rows a wave) or 64 (a row a wave, for long
// K: a K = 9728 row is 19 chunks a lane at 16 lanes, loaded in three batches
// one after another, and about 5 at 64, one batch).
template <typename T, int MR, int EPI, bool PF = false, bool WIDE = false, int LPR = 16>
__global__ __launch_bounds__(WIDE ? 1024 : 256) void qmv_dot2_kernel(QParams p) {
    static_assert(!WIDE || qmv_dot2_wide_ok(EPI), "wide workgroups: single output");
    static_assert(LPR == 16 || LPR == 64, "4 rows or one a wave");
    static_assert(!PF || MR == 1, "PF: one token");
    static_assert(!PF || !WIDE || LPR == 64, "PF in wide workgroups: a row a wave");
    constexpr int RPW = 64 / LPR;  // rows a wave
    constexpr int P = epi_parts(EPI);
    typedef Magic<T> Mg;
    extern __shared__ uint4 xs_pairs[];  // [MR][K/8] pair blocks, then [MR][K/32] sums
    const int64_t K = p.K, words = K / 8, cpr = K / 32, G = K >> p.gs_log2;
    float *xsum = (float *)(xs_pairs + MR * words);
    const int lane = threadIdx.x & 63, j = lane & (LPR - 1);
    const int bs = WIDE ? (int)blockDim.x : 256;  // threads
    int64_t nb = (int64_t)blockIdx.x * ((bs >> 6) * RPW);
    const Bound bd = bind<EPI>(p, nb);
    const int64_t n = nb + (threadIdx.x >> 6) * RPW + lane / LPR;
    const int64_t nrow = n < bd.Nout ? n : bd.Nout - 1;
    const int64_t m0 = (int64_t)blockIdx.y * MR;
    const int mr = (int)((p.M - m0) < MR ? (p.M - m0) : MR);

    const uint32_t *wr[P];
    const T *sr[P];
    const T *br[P];
#pragma unroll
    for (int q = 0; q < P; ++q) {
        const int64_t row = bd.noff(q) + nrow;
        wr[q] = bd.w(q) + row * (K / 8);
        sr[q] = (const T *)bd.s(q) + row * G;
        br[q] = (const T *)bd.b(q) + row * G;
    }

    uint4 wv[P][QV_BATCH];
    T sv[P][QV_BATCH], bv[P][QV_BATCH];
    auto load_batch = [&](int64_t base) {
#pragma unroll
        for (int i = 0; i < QV_BATCH; ++i) {
            const int64_t c = base + LPR * i;
            const int64_t cc = c < cpr ? c : cpr - 1;
            const int64_t g = (cc * 32) >> p.gs_log2;
#pragma unroll
            for (int q = 0; q < P; ++q) {
                wv[q][i] = ld16_nt(wr[q] + 4 * cc);
                sv[q][i] = sr[q][g];
                bv[q][i] = br[q][g];
            }
        }
    };

    // stage x rows as pairs (e[i], e[i+4]) of each 8-value block
    const T *x = (const T *)p.x + m0 * K;
    auto pairs = [](const uint4 d) {
        return make_uint4(__builtin_amdgcn_perm(d.z, d.x, 0x05040100u),
                          __builtin_amdgcn_perm(d.z, d.x, 0x07060302u),
                          __builtin_amdgcn_perm(d.w, d.y, 0x05040100u),
                          __builtin_amdgcn_perm(d.w, d.y, 0x07060302u));
    };
    const int nw = (int)words;  // 32-bit index math: MR * K < 2^31
    if constexpr (PF) {
        // Every thread issues both loads (a clamped, valid chunk when past the
        // end) so the issue order, and with it the waits, is the same in all
        // waves: x, then the weights (K / 8 <= 2 bs)
        uint4 d[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            int idx = (int)threadIdx.x + bs * t;
            idx = idx < MR * nw ? idx : MR * nw - 1;
            const int m = MR == 1 ? 0 : idx / nw, w = idx - m * nw;
            d[t] = ld16(x + (int64_t)(m < mr ? m : mr - 1) * K + 8 * w);
        }
        __builtin_amdgcn_sched_barrier(0);  // keep the x loads ahead of the weights'
        load_batch(j);
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int64_t idx = threadIdx.x + bs * t;
            if (idx < MR * words) xs_pairs[idx] = pairs(d[t]);
        }
    } else {
        for (int idx = threadIdx.x; idx < MR * nw; idx += bs) {
            const int m = MR == 1 ? 0 : idx / nw, w = idx - m * nw;
            xs_pairs[idx] = pairs(ld16(x + (int64_t)(m < mr ? m : mr - 1) * K + 8 * w));
        }
    }
    __syncthreads();
    const int ncpr = (int)cpr;
    for (int idx = threadIdx.x; idx < MR * ncpr; idx += bs) {
        const int m = MR == 1 ? 0 : idx / ncpr, c = idx - m * ncpr;
        float s = 0.0f;
#pragma unroll
        for (int wi = 0; wi < 4; ++wi) {
            const uint4 v = xs_pairs[m * words + 4 * c + wi];
            float f[8];
            unpack8<T>(v, f);
#pragma unroll
            for (int i = 0; i < 8; ++i) s += f[i];
        }
        xsum[idx] = s;
    }
    __syncthreads();

    float acc[P][MR];
#pragma unroll
    for (int q = 0; q < P; ++q)
#pragma unroll
        for (int m = 0; m < MR; ++m) acc[q][m] = 0.0f;

    for (int64_t base = j; base < cpr; base += LPR * QV_BATCH) {
        // (Without PF the compiler sinks each chunk's loads to its use behind
        // the `c >= cpr` exit, so a lane fetches its chunks one after another;
        // at 58 registers eight waves per SIMD keep the loads in flight.)
        if (!PF || base != j) load_batch(base);
#pragma unroll
        for (int i = 0; i < QV_BATCH; ++i) {
            const int64_t c = base + LPR * i;
            if (c >= cpr) break;
#pragma unroll
            for (int q = 0; q < P; ++q) {
                const uint32_t wd[4] = {wv[q][i].x, wv[q][i].y, wv[q][i].z, wv[q][i].w};
                uint32_t qp[4][4];
#pragma unroll
                for (int wi = 0; wi < 4; ++wi)
#pragma unroll
                    for (int jj = 0; jj < 4; ++jj)
                        qp[wi][jj] = magic_pair<T>(wd[wi], jj);
                const float s = (float)sv[q][i];
                const float bb = __builtin_fmaf(-Mg::value, s, (float)bv[q][i]);
#pragma unroll
                for (int m = 0; m < MR; ++m) {
                    float d = 0.0f;
#pragma unroll
                    for (int wi = 0; wi < 4; ++wi) {
                        const uint4 xp = xs_pairs[m * words + 4 * c + wi];
                        d = Mg::dot2(qp[wi][0], xp.x, d);
                        d = Mg::dot2(qp[wi][1], xp.y, d);
                        d = Mg::dot2(qp[wi][2], xp.z, d);
                        d = Mg::dot2(qp[wi][3], xp.w, d);
                    }
                    acc[q][m] += fma_mul(s, d, bb, xsum[m * cpr + c]);
                }
            }
        }
    }
#pragma unroll
    for (int q = 0; q < P; ++q)
#pragma unroll
        for (int m = 0; m < MR; ++m) {
            acc[q][m] = row16_sum(acc[q][m]);  // the row's 16 lanes
            if constexpr (LPR == 64) {  // then the wave's four 16-lane sums
                const int v = __builtin_bit_cast(int, acc[q][m]);
                const float r0 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(v, 0));
                const float r1 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(v, 16));
                const float r2 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(v, 32));
                const float r3 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(v, 48));
                acc[q][m] = (r0 + r1) + (r2 + r3);
            }
        }
    if (j == 0 && n < bd.Nout) {
#pragma unroll
        for (int m = 0; m < MR; ++m) {
            if (m < mr) {
                float a[P];
#pragma unroll
                for (int q = 0; q < P; ++q) a[q] = acc[q][m];
                epi1<T, EPI>(p, bd, m0 + m, n, a);
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Few-token GEMM (M <= 8, 16-bit T, both widths): the factored per-group sum on
// the matrix cores. The codes enter v_mfma_f32_16x16x32 exactly, as the integers
// they are, and x as it is, so a group's D = sum x q and X = sum x (a product
// with ones) are fp32 sums of exact products, and the row adds s D + b X per
// group, up to 16 tokens at the cost of one. (Codes with an offset, as the dot2
// GEMV takes them, are cheaper to make and cost the sums three to ten bits: the
// offset's share has to cancel again.)
//
// A workgroup owns 16 output features (per part) and its waves split K in
// contiguous runs; the partial sums meet in LDS. Operands: A = x (row = token
// lane % 16), B = weights (column = feature lane % 16), both with one quarter of
// each group's k for each lane / 16. Weights are loaded GB units ahead (a ring
// of registers), the first GB before x is staged; x rows and the 16 rows' scales
// and biases come through LDS by DMA. K split and group order depend on (K, bits,
// group size) alone, so every epilogue adds alike.
//
// PAIR (a lane's share of one group is 4 or 8 bytes, and the group count is
// even): a unit is two groups. A lane then loads two quarters of one group, 8 or
// 16 bytes, and a v_permlane32_swap hands each half to its group: 64-byte pieces
// of a row per load, not 32 (N = 9728, K = 2560, 4 bits, 8 tokens: 10.1 -> 7.7
// us). Whole 128-byte lines per load (8 rows of 8 lanes, transposed by more
// swaps) lost: the registers it held left one workgroup a CU (12.4 us).
// Otherwise a unit is one group, a quarter a lane.
//
// A unit's scales and biases are read together: two 2-byte LDS reads a part and
// group had bound the narrow groups (dual 9728 x 2048, 4 tokens, group 32 21.2 ->
// 10.7 us; x 4096, group 64 20.7 -> 16.6).
//
// Bound: HBM, one memory round trip after the launch.
template <typename T> __device__ __forceinline__ f32x4 mma16(uint4 a, uint4 b, f32x4 c) {
    typedef typename Vec<T>::x8 V8;
    if constexpr (__is_same(T, bf16))
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(V8, a),
                                                       __builtin_bit_cast(V8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(V8, a),
                                                      __builtin_bit_cast(V8, b), c, 0, 0, 0);
}

// Eight codes as T, in order: the nibbles of w0 (4 bits) or the bytes of w0 and w1.
// 4 bits: a byte below 16 read as an fp8 (E4M3) number is itself 2^-9, through its
// subnormals and its first binade, so the scaled conversion to a pair of T is two
// codes an instruction (through fp32, a code an instruction, the 8848 x 9728 dual
// at 4 tokens took 44.5 us, not 36.4).
// 8 bits, bf16: an integer below 256 has at most 8 significant bits, so its fp32
// value's high half is it. fp16: q 2^-24, the subnormal whose bits q is (the
// caller scales by code_scale, exact).
template <typename T, int BITS>
__device__ __forceinline__ uint4 code_frag(uint32_t w0, uint32_t w1) {
    if constexpr (BITS == 4) {
        const uint32_t even = w0 & 0x0F0F0F0Fu, odd = (w0 >> 4) & 0x0F0F0F0Fu;
        const uint32_t lo = __builtin_amdgcn_perm(odd, even, 0x05010400u);  // codes 0 .. 3
        const uint32_t hi = __builtin_amdgcn_perm(odd, even, 0x07030602u);  // codes 4 .. 7
        if constexpr (__is_same(T, bf16))
            return make_uint4(
                __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 512.0f, false)),
                __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 512.0f, true)),
                __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 512.0f, false)),
                __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 512.0f, true)));
        else
            return make_uint4(
                __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(lo, 512.0f, false)),
                __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(lo, 512.0f, true)),
                __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(hi, 512.0f, false)),
                __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(hi, 512.0f, true)));
    } else if constexpr (__is_same(T, bf16)) {
        auto pair = [](uint32_t w, int sh) {
            return __builtin_amdgcn_perm(__float_as_uint((float)((w >> (sh + 8)) & 255u)),
                                         __float_as_uint((float)((w >> sh) & 255u)), 0x07060302u);
        };
        return make_uint4(pair(w0, 0), pair(w0, 16), pair(w1, 0), pair(w1, 16));
    } else {
        auto pair = [](uint32_t w, uint32_t sel) { return __builtin_amdgcn_perm(0u, w, sel); };
        return make_uint4(pair(w0, 0x04010400u), pair(w0, 0x04030402u), pair(w1, 0x04010400u),
                          pair(w1, 0x04030402u));
    }
}
template <typename T, int BITS> constexpr float code_scale() {
    return BITS == 8 && __is_same(T, f16) ? 16777216.0f : 1.0f;
}

template <int BITS, int P, int GSL, bool PAIR> struct QmsShape {
    static constexpr int STEPS = 1 << (GSL - 5);              // MFMAs per group
    static constexpr int WPL = STEPS * (BITS == 4 ? 1 : 2);   // words per lane and group
    static constexpr int U = PAIR ? 2 : 1;                    // groups per unit
    static constexpr int UW = WPL * U;                        // words per lane and unit
    static constexpr int FIT = (P == 3 ? 24 : 48) / (UW * P);
    // units in flight: 8 groups, 6 where a second part at group 32 takes the
    // registers (8: 3 to 5 % slower at K = 4096)
    static constexpr int CAP = GSL == 5 && BITS == 4 && P == 2 ? 3 : 8 / U;
    static constexpr int GB = FIT > CAP ? CAP : (FIT < 1 ? 1 : FIT);
};
template <int BITS, int GSL> constexpr bool qms_pairs() {
    return QmsShape<BITS, 1, GSL, false>::WPL <= 2;
}

// Waits until at most n (1 .. N) units' loads, PER each, are in flight.
template <int PER, int N> __device__ __forceinline__ void wait_units(int n) {
    if (n == N) wait_vmcnt<PER * N>();
    if constexpr (N > 1) wait_units<PER, N - 1>(n);
}

// Dynamic LDS: x rows (a 16-byte pad a row, so the rows' reads of one chunk
// spread over the banks), the scale and bias rows; the partial sums reuse it.
// spread: beside them (the waves finish runs while others still read).
struct QmsLds {
    int pitch, sb, red, total;  // bytes: of an x row; of one scale or bias array
};
__host__ __device__ inline QmsLds qms_lds(int rows, int64_t K, int64_t G, int parts, int runs,
                                          bool spread = false) {
    const int pitch = (int)(2 * K) + 16, sb = (int)(16 * G * 2);
    const int stage = rows * pitch + 2 * parts * sb, red = runs * parts * 1024;
    if (spread) return {pitch, sb, stage, stage + red};
    return {pitch, sb, 0, stage > red ? stage : red};
}
// Runs of K, whose sums are added in order: a function of K alone, about 8 groups
// of 64 a run at the projection widths. A wave takes one; or two in turn where 16
// waves, of which a CU holds one workgroup, would leave the last round of
// workgroups nearly empty (see launch_qms).
inline int qms_runs(int64_t K) { return K > 4096 ? 16 : 8; }

// bind() of an epilogue known at run time (EPI_GROUP3 among the single-part ones).
template <int P> __device__ __forceinline__ Bound bind_of(const QParams &p, int epi, int64_t &nb) {
    if constexpr (P > 1) {
        return bind<EPI_STORE>(p, nb);
    } else {
        const bool grp = epi == EPI_GROUP3;
        const int64_t e0 = grp ? p.pn[0] : p.Nout, e1 = grp ? p.pn[0] + p.pn[1] : p.Nout;
        const bool p0 = nb < e0, p1 = !p0 && nb < e1;
        nb -= p0 ? 0 : (p1 ? e0 : e1);
        Bound q = {};
        q.w0 = p0 ? p.w[0] : (p1 ? p.w[1] : p.w[2]);
        q.s0 = p0 ? p.s[0] : (p1 ? p.s[1] : p.s[2]);
        q.b0 = p0 ? p.b[0] : (p1 ? p.b[1] : p.b[2]);
        q.o0 = grp ? 0 : p.noff[0];
        q.y0 = !grp ? p.y0 : (p0 ? p.py[0] : (p1 ? p.py[1] : p.py[2]));
        q.Nout = !grp ? p.Nout : (p0 ? p.pn[0] : (p1 ? p.pn[1] : p.pn[2]));
        return q;
    }
}

template <typename T, int BITS, int P, int GSL, bool PAIR>
__global__ __launch_bounds__(1024) void qms_kernel(QParams p, int epi, int mr, int nw, int runs,
                                                   int run, int longer, int sb_dma) {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef QmsShape<BITS, P, GSL, PAIR> Sh;
    typedef __attribute__((address_space(3))) void *lds_ptr;
    constexpr int STEPS = Sh::STEPS, WPL = Sh::WPL, U = Sh::U, UW = Sh::UW, GB = Sh::GB;
    constexpr int VPW = 32 / BITS;
    extern __shared__ __attribute__((aligned(16))) char qlds[];
    const int lane = threadIdx.x & 63, nl = lane & 15, kb = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int64_t nb = (int64_t)blockIdx.x * 16;
    const Bound bd = bind_of<P>(p, epi, nb);
    const int64_t m0 = (int64_t)blockIdx.y * mr;
    const int rows = (int)(p.M - m0 < mr ? p.M - m0 : mr);
    const int64_t K = p.K;
    const int G = (int)(K >> GSL);
    const QmsLds L = qms_lds(rows, K, G, P, runs, runs > nw);
    char *sbl = qlds + rows * L.pitch;  // [part][scale, bias][16][G]

    // x rows, then the scale and bias rows, 16 bytes a lane; the instructions
    // are dealt to the waves. (sb_dma 0: scale or bias rows off a 16-byte
    // boundary, or whose last tile ends off one, come a value a thread.)
    {
        const __amdgpu_buffer_rsrc_t xr =
            buffer_rsrc((const T *)p.x + m0 * K, (uint32_t)(rows * K * (int64_t)sizeof(T)));
        const int cpr = (int)(K / 8), ipr = (cpr + 63) >> 6;
        int row = 0, i = wave;
        while (i >= ipr) i -= ipr, ++row;  // (wave-uniform)
        while (row < rows) {
            const int c = 64 * i + lane;
            if (c < cpr)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (lds_ptr)(qlds + row * L.pitch + i * 1024),
                                                         16, 16 * c, (int)(row * K * 2), 0, 0);
            i += nw;
            while (i >= ipr) i -= ipr, ++row;
        }
        const int chunks = 2 * G, ips = (chunks + 63) >> 6;
        const int64_t left = (bd.Nout - nb) * G * 2;  // the part's rows from nb on
        const uint32_t bytes = (uint32_t)(left < L.sb ? left : L.sb);
        auto sb_rows = [&](int a) {
            return (const T *)((a & 1) ? bd.b(a >> 1) : bd.s(a >> 1)) + (bd.noff(a >> 1) + nb) * G;
        };
        if (sb_dma) {
#pragma unroll
            for (int a = 0; a < 2 * P; ++a) {
                const __amdgpu_buffer_rsrc_t sr = buffer_rsrc(sb_rows(a), bytes);
                for (int j = wave; j < ips; j += nw) {
                    const int c = 64 * j + lane;
                    if (c < chunks)
                        __builtin_amdgcn_raw_ptr_buffer_load_lds(
                            sr, (lds_ptr)(sbl + a * L.sb + j * 1024), 16, 16 * c, 0, 0, 0);
                }
            }
        } else {
            for (int a = 0; a < 2 * P; ++a)
                for (int i = threadIdx.x; i < (int)(bytes / sizeof(T)); i += 64 * nw)
                    ((T *)(sbl + a * L.sb))[i] = sb_rows(a)[i];
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");  // before the barrier below
        }
    }
    __builtin_amdgcn_sched_barrier(0);

    // this wave's (first) run: its units (run + 1 for the first `longer` runs, run
    // for the rest), and the first GB of them (rows past N read a clamped, valid
    // address)
    int u0 = wave * run + (wave < longer ? wave : longer);
    int u1 = u0 + run + (wave < longer ? 1 : 0);
    const int64_t n = nb + nl;
    const int64_t nrow = n < bd.Nout ? n : bd.Nout - 1;
    const uint32_t *wr[P];
#pragma unroll
    for (int q = 0; q < P; ++q) wr[q] = bd.w(q) + (bd.noff(q) + nrow) * (K / VPW) + kb * UW;
    uint32_t w[GB][P][UW];
    auto load = [&](int i, int u) {
#pragma unroll
        for (int q = 0; q < P; ++q) {
            const uint32_t *src = wr[q] + u * (4 * UW);
            if constexpr (UW == 1) {
                w[i][q][0] = *src;
            } else if constexpr (UW == 2) {
                const uint2 v = ld8(src);
                w[i][q][0] = v.x, w[i][q][1] = v.y;
            } else {
#pragma unroll
                for (int j = 0; j < UW; j += 4) {
                    const uint4 v = ld16(src + j);
                    w[i][q][j] = v.x, w[i][q][j + 1] = v.y;
                    w[i][q][j + 2] = v.z, w[i][q][j + 3] = v.w;
                }
            }
        }
    };
    const int ahead = u1 - u0 < GB ? u1 - u0 : GB;  // units requested now
#pragma unroll
    for (int i = 0; i < GB; ++i)
        if (i < ahead) load(i, u0 + i);  // (wave-uniform)
    // x, the scales and biases have landed (they were issued first); the
    // weights stay in flight
    constexpr int PER = P * (UW > 4 ? UW / 4 : 1);  // loads per unit
    static_assert(GB * PER < 64, "vmcnt is a 6-bit count");
    __builtin_amdgcn_sched_barrier(0);
    if (ahead == 0) wait_vmcnt<0>();
    wait_units<PER, GB>(ahead);
    asm volatile("" ::: "memory");  // (no LDS read moves up)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);

    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    f32x4 acc[P];
#pragma unroll
    for (int q = 0; q < P; ++q) acc[q] = zero;
    constexpr uint32_t one = __is_same(T, bf16) ? 0x3F803F80u : 0x3C003C00u;
    const uint4 ones = make_uint4(one, one, one, one);
    // the lane's k quarter (PAIR: after the swap, lanes kb hold quarters 0, 2, 1, 3)
    const int kq = PAIR ? (kb >> 1) | ((kb & 1) << 1) : kb;
    // (a token past the last reads the last row: its sums are not stored)
    const char *xrow = qlds + (nl < rows ? nl : rows - 1) * L.pitch + kq * (1 << (GSL - 1));
    const char *srow = sbl + nl * G * 2;
    auto body = [&](const char *__restrict__ xp, const char *__restrict__ sp)
                    __attribute__((always_inline)) {
    for (int base = u0; base < u1; base += GB) {
#pragma unroll
        for (int i = 0; i < GB; ++i) {
            const int u = base + i;
            if (u >= u1) break;  // wave-uniform
            if constexpr (PAIR) {
                typedef unsigned U2 __attribute__((ext_vector_type(2)));
#pragma unroll
                for (int q = 0; q < P; ++q)
#pragma unroll
                    for (int j = 0; j < WPL; ++j) {
                        const U2 r = __builtin_amdgcn_permlane32_swap(w[i][q][j], w[i][q][WPL + j],
                                                                      false, false);
                        w[i][q][j] = r[0], w[i][q][WPL + j] = r[1];
                    }
            }
            // the unit's scales and biases (PAIR: both groups' in one read)
            T sc[P][U], bi[P][U];
#pragma unroll
            for (int q = 0; q < P; ++q) {
                const char *ps = sp + (2 * q) * L.sb + 2 * U * u, *pb = ps + L.sb;
                if constexpr (PAIR) {
                    typedef T T2 __attribute__((ext_vector_type(2)));
                    const T2 s2 = *(const T2 *)ps, b2 = *(const T2 *)pb;
                    sc[q][0] = s2.x, sc[q][1] = s2.y, bi[q][0] = b2.x, bi[q][1] = b2.y;
                } else {
                    sc[q][0] = *(const T *)ps, bi[q][0] = *(const T *)pb;
                }
            }
#pragma unroll
            for (int v = 0; v < U; ++v) {
                const int g = U * u + v;
                uint4 a[STEPS];
#pragma unroll
                for (int st = 0; st < STEPS; ++st)
                    a[st] = *(const uint4 *)(xp + (g << (GSL + 1)) + 16 * st);
                f32x4 X = zero, D[P];
#pragma unroll
                for (int q = 0; q < P; ++q) D[q] = zero;
#pragma unroll
                for (int st = 0; st < STEPS; ++st) {
                    X = mma16<T>(a[st], ones, X);
#pragma unroll
                    for (int q = 0; q < P; ++q) {
                        const uint32_t *wq = w[i][q] + v * WPL;
                        D[q] = mma16<T>(a[st], BITS == 4 ? code_frag<T, BITS>(wq[st], 0u)
                                                     : code_frag<T, BITS>(wq[2 * st], wq[2 * st + 1]),
                                        D[q]);
                    }
                }
#pragma unroll
                for (int q = 0; q < P; ++q) {
                    const float s = (float)sc[q][v] * code_scale<T, BITS>(), b = (float)bi[q][v];
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        acc[q][e] = __builtin_fmaf(s, D[q][e], __builtin_fmaf(b, X[e], acc[q][e]));
                }
            }
            if (u + GB < u1) load(i, u + GB);
        }
    }
    };
    // the runs' sums, in order: token 4 kb + e of feature nl is element e of lane
    // (kb, nl); wave e < 4 adds and stores element e
    float *red = (float *)(qlds + L.red);
    for (int vw = wave;;) {  // (wave-uniform)
        body(xrow, srow);
        if (runs == nw) __syncthreads();  // (the sums take the staged rows' place)
#pragma unroll
        for (int q = 0; q < P; ++q) {
            *(float4 *)(red + ((vw * P + q) * 64 + lane) * 4) =
                make_float4(acc[q][0], acc[q][1], acc[q][2], acc[q][3]);
            acc[q] = zero;
        }
        vw += nw;
        if (vw >= runs) break;
        u0 = vw * run + (vw < longer ? vw : longer);
        u1 = u0 + run + (vw < longer ? 1 : 0);
#pragma unroll
        for (int i = 0; i < GB; ++i)
            if (i < u1 - u0) load(i, u0 + i);
    }
    __syncthreads();
    if (wave >= 4) return;
    float v[P];
#pragma unroll
    for (int q = 0; q < P; ++q) {
        v[q] = red[(q * 64 + lane) * 4 + wave];
        for (int s = 1; s < runs; ++s) v[q] += red[((s * P + q) * 64 + lane) * 4 + wave];
    }
    const int t = 4 * kb + wave;
    if (t >= rows || n >= bd.Nout) return;
    if constexpr (P == 1) {
        if (epi == EPI_RESID)
            epi1<T, EPI_RESID>(p, bd, m0 + t, n, v);
        else
            epi1<T, EPI_STORE>(p, bd, m0 + t, n, v);
    } else if constexpr (P == 2) {
        if (epi == EPI_SWIGLU)
            epi1<T, EPI_SWIGLU>(p, bd, m0 + t, n, v);
        else
            epi1<T, EPI_DUAL>(p, bd, m0 + t, n, v);
    } else {
        epi1<T, EPI_SPLIT3>(p, bd, m0 + t, n, v);
    }
#endif
}

// ---------------------------------------------------------------------------
// dispatch

template <typename T, int BITS, int EPI>
int launch_qmv(const QParams &p, hipStream_t st) {
    const dim3 grid((unsigned)ceil_div(p.Nout, 16), (unsigned)ceil_div(p.M, QMV_MR));
    if (p.M == 1)
        qmv_kernel<T, BITS, 1, EPI><<<grid, 256, 0, st>>>(p);
    else if (p.M <= 2)
        qmv_kernel<T, BITS, 2, EPI><<<grid, 256, 0, st>>>(p);
    else if (p.M <= 4)
        qmv_kernel<T, BITS, 4, EPI><<<grid, 256, 0, st>>>(p);
    else
        qmv_kernel<T, BITS, QMV_MR, EPI><<<grid, 256, 0, st>>>(p);
    return launch_status("quantized matmul (qmv)");
}

template <typename T, int EPI>
int launch_qmv_dot2(const QParams &p, int mr, hipStream_t st) {
    // weights requested under the x staging when the 4-wave grid is at most
    // four workgroups per CU (measured: N = 9728 gains, N = 151936 loses),
    // for single-output epilogues: holding two or three weight rows' batches
    // through the staging takes 226-256 registers, one or two waves a SIMD
    // (the gate/up dual at M = 1, N = 9728: 10.9 us with PF, 8.6 without)
    const int64_t gy = ceil_div(p.M, mr);
    const bool pf = epi_parts(EPI) == 1 && mr == 1 && ceil_div(p.Nout, 16) * gy <= 1024 &&
                    p.K / 8 <= 512;
    // A row a wave (LPR 64) over long rows (K > 4096, more than 8 chunks a lane
    // at 16 lanes a row), whatever the epilogue: it is another order of sums. The
    // dual gains to 4096 features (1 token, x 8192 15.1 -> 8.6 us) and pays past
    // them (14336 x 5120 17.7 -> 20.0).
    // Waves per workgroup
    // without PF: as many as spread the rows evenly over the CUs in one round
    // of workgroups (N = 9728 at 4 rows a wave: 10 waves, 244 workgroups, at
    // most 40 rows a CU, where 16-row workgroups put 48 on some CUs and 32 on
    // the others: M = 2 7.5 -> 7.2 us); 4 when the rows
    // take more than one round of 16-wave workgroups, for the grouped q/k/v
    // epilogue, whose workgroups each lie inside one part, and for the
    // several-output ones.
    constexpr bool wide_ok = qmv_dot2_wide_ok(EPI);
    const bool row_wave = p.K / 32 > 128;  // (pf: K <= 4096)
    const int rpw = row_wave ? 1 : 4;
    int waves = 4;
    if constexpr (wide_ok) {
        const int64_t wv = ceil_div(p.Nout, rpw * (int64_t)device_cus());
        if (!pf && wv <= 16) waves = wv < 4 ? 4 : (int)wv;
    }
    const int bs = 64 * waves;
    const dim3 grid((unsigned)ceil_div(p.Nout, rpw * waves), (unsigned)gy);
    const size_t lds = (size_t)qmv_dot2_lds_bytes(mr, p.K);
    if (pf) {
        qmv_dot2_kernel<T, 1, EPI, true><<<grid, bs, lds, st>>>(p);
    } else if (!row_wave && waves == 4) {
        if (mr == 1)
            qmv_dot2_kernel<T, 1, EPI><<<grid, bs, lds, st>>>(p);
        else if (mr == 2)
            qmv_dot2_kernel<T, 2, EPI><<<grid, bs, lds, st>>>(p);
        else
            qmv_dot2_kernel<T, 4, EPI><<<grid, bs, lds, st>>>(p);
    } else if (waves == 4) {
        // a row a wave (one token: see launch_typed) takes PF too while x fits two
        // chunks a thread (Qwen3's down_proj at decode, 10-wave workgroups: 6.7 ->
        // 5.6 us), single output
        if (wide_ok && p.K / 8 <= 2 * bs)
            qmv_dot2_kernel<T, 1, EPI, wide_ok, false, 64><<<grid, bs, lds, st>>>(p);
        else
            qmv_dot2_kernel<T, 1, EPI, false, false, 64><<<grid, bs, lds, st>>>(p);
    } else if constexpr (wide_ok) {
        if (row_wave && p.K / 8 <= 2 * bs)
            qmv_dot2_kernel<T, 1, EPI, true, true, 64><<<grid, bs, lds, st>>>(p);
        else if (row_wave)
            qmv_dot2_kernel<T, 1, EPI, false, true, 64><<<grid, bs, lds, st>>>(p);
        else if (mr == 1)
            qmv_dot2_kernel<T, 1, EPI, false, true><<<grid, bs, lds, st>>>(p);
        else if (mr == 2)
            qmv_dot2_kernel<T, 2, EPI, false, true><<<grid, bs, lds, st>>>(p);
        else
            qmv_dot2_kernel<T, 4, EPI, false, true><<<grid, bs, lds, st>>>(p);
    }
    return launch_status("quantized matmul (dot2 qmv)");
}

// Whether qms_kernel takes a call's (M, K, group size): up to 8 tokens, 32-bit
// offsets, and one x row in the LDS beside the scales and biases of three parts,
// whatever the epilogue has, so that every epilogue of one shape takes it (and
// adds in its order) or none does.
inline bool qms_takes(int64_t M, int64_t K, int gs_log2) {
    return M <= QMV_MR && K < ((int64_t)1 << 24) &&
           qms_lds(1, K, K >> gs_log2, 3, qms_runs(K)).total <= LDS_PER_CU;
}
// Token rows per workgroup: all of them, halved while x does not fit the LDS.
inline int qms_rows(const QParams &p, int parts) {
    int mr = (int)p.M;
    while (mr > 1 && qms_lds(mr, p.K, p.K >> p.gs_log2, parts, qms_runs(p.K)).total > LDS_PER_CU)
        mr = (mr + 1) / 2;
    return mr;
}

// Whether 16-byte DMA takes the scale and bias rows of every tile.
inline bool qms_sb_dma(const QParams &p, int epi) {
    const int64_t G = p.K >> p.gs_log2;
    for (int i = 0; i < 3; ++i) {
        const int64_t rows = epi == EPI_GROUP3 ? p.pn[i] : p.Nout;
        if (!aligned(p.s[i], 16) || !aligned(p.b[i], 16) || (p.noff[i] * G) % 8 || (rows * G) % 8)
            return false;
    }
    return true;
}

template <typename T, int BITS, int P, int GSL>
void launch_qms_gs(const QParams &p, int epi, int mr, int nw, dim3 grid, size_t lds,
                   hipStream_t st) {
    const int G = (int)(p.K >> GSL), runs = qms_runs(p.K), dma = qms_sb_dma(p, epi);
    if constexpr (qms_pairs<BITS, GSL>()) {
        if (G % 2 == 0) {
            qms_kernel<T, BITS, P, GSL, true><<<grid, 64 * nw, lds, st>>>(
                p, epi, mr, nw, runs, G / 2 / runs, G / 2 % runs, dma);
            return;
        }
    }
    qms_kernel<T, BITS, P, GSL, false><<<grid, 64 * nw, lds, st>>>(p, epi, mr, nw, runs, G / runs,
                                                                   G % runs, dma);
}

template <typename T, int BITS, int P>
int launch_qms(const QParams &p, int epi, int mr, hipStream_t st) {
    const dim3 grid((unsigned)ceil_div(p.Nout, 16), (unsigned)ceil_div(p.M, mr));
    const int64_t G = p.K >> p.gs_log2;
    int nw = qms_runs(p.K);
    size_t lds = (size_t)qms_lds(mr, p.K, G, P, nw).total;
    // Eight waves of two runs past one 16-wave workgroup a CU, while two such
    // workgroups fit its LDS. Same sums. 8-bit, one token, 12000 x 8192 29.8 -> 21.4
    // us, 5040 x 5120 10.5 -> 8.7; 4-bit, 3 tokens, 12000 x 5120 14.3 -> 9.5.
    if (nw == 16 && (int64_t)grid.x * grid.y > device_cus()) {
        const int spread = qms_lds(mr, p.K, G, P, nw, true).total;
        if (2 * spread <= LDS_PER_CU) nw = 8, lds = (size_t)spread;
    }
    if (p.gs_log2 == 5)
        launch_qms_gs<T, BITS, P, 5>(p, epi, mr, nw, grid, lds, st);
    else if (p.gs_log2 == 6)
        launch_qms_gs<T, BITS, P, 6>(p, epi, mr, nw, grid, lds, st);
    else
        launch_qms_gs<T, BITS, P, 7>(p, epi, mr, nw, grid, lds, st);
    return launch_status("quantized matmul (few-token mfma)");
}

template <typename T, int EPI>
int launch_typed(const QParams &p, int bits, hipStream_t st) {
    if constexpr (sizeof(T) == 2) {
        // The few-token kernel from three tokens (4-bit) or two (8-bit), and for
        // rows past K = 4096 from two or one; a function of M, K, the width and the
        // group size, so every epilogue at one shape adds alike. Measured (us, N x
        // K; the GEMVs / it): 4-bit, 9728 x 2560, M = 2 7.2 / 6.5, M = 4 9.8 / 6.3,
        // M = 8 34 / 6.7; the dual of it M = 2 10.0 / 11.5, M = 4 13.3 / 10.2; 2560 x
        // 9728, M = 2 7.9 / 7.1, M = 4 27 / 7.5, M = 6 50 / 8.0. 8-bit, 2048 x 8192,
        // M = 1 11.4 / 10.1, M = 6 58 / 11.1, but 12000 x 5120, M = 1 12.4 / 13.7; the
        // 8192 x 2048 dual M = 1 9.4 / 10.4, M = 2 13.9 / 8.9, M = 6 24 / 9.0; lm_head
        // (151936 x 2560) M = 1 71 / 77, M = 8 445 / 92.
        // Short rows stay with the GEMVs, which have less to set up: 8-bit M = 2,
        // 8192 x 768 3.6 / 4.2, 892 x 1024 4.8 / 4.4, M = 3, 944 x 256 2.7 / 3.2, x 768
        // 4.2 / 3.4; 4-bit M = 3, 2048 x 512 3.1 / 3.3, x 768 3.7 / 3.6.
        constexpr int P = epi_parts(EPI);
        const int64_t M = p.M;
        const bool few = bits == 4 ? M > 4 || (M > 1 && p.K > (M > 2 ? 512 : 4096))
                                   : p.K > (M == 1 ? 4096 : M == 2 ? 768 : 256);
        if (few && qms_takes(M, p.K, p.gs_log2)) {
            const int rows = qms_rows(p, P);
            return bits == 4 ? launch_qms<T, 4, P>(p, EPI, rows, st)
                             : launch_qms<T, 8, P>(p, EPI, rows, st);
        }
        const int mr = M > 2 ? 4 : (int)M;
        if (bits == 4 && (M == 1 || (M <= 4 && p.K <= 4096)) &&
            qmv_dot2_lds_bytes(mr, p.K) <= 65536)
            return launch_qmv_dot2<T, EPI>(p, mr, st);
    }
    return bits == 4 ? launch_qmv<T, 4, EPI>(p, st) : launch_qmv<T, 8, EPI>(p, st);
}

template <int EPI> int run(const QParams &p, int bits, int dtype, hipStream_t st) {
    switch (dtype) {
    case MI_BF16: return launch_typed<bf16, EPI>(p, bits, st);
    case MI_F16: return launch_typed<f16, EPI>(p, bits, st);
    default: return launch_typed<float, EPI>(p, bits, st);
    }
}

}  // namespace

// Compute units of the current device (cached per device).
int device_cus() {
    static int cache[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    if (cache[dev] == 0) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
            n <= 0)
            n = 256;
        cache[dev] = n;
    }
    return cache[dev];
}

int gemv_launch(const QParams &p, int epi, int bits, int dtype, hipStream_t st) {
    switch (epi) {
    case EPI_STORE: return run<EPI_STORE>(p, bits, dtype, st);
    case EPI_RESID: return run<EPI_RESID>(p, bits, dtype, st);
    case EPI_SPLIT3: return run<EPI_SPLIT3>(p, bits, dtype, st);
    case EPI_DUAL: return run<EPI_DUAL>(p, bits, dtype, st);
    case EPI_SWIGLU: return run<EPI_SWIGLU>(p, bits, dtype, st);
    default: return run<EPI_GROUP3>(p, bits, dtype, st);
    }
}

}  // namespace mi
