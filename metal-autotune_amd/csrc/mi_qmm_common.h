// What the quantized-matmul kernels share: the launch parameters, the
// epilogues of the region cuts, buffer resources and waits.
#pragma once

#include "mi_common.h"

namespace mi {

enum Epi { EPI_STORE = 0, EPI_RESID = 1, EPI_SPLIT3 = 2, EPI_DUAL = 3, EPI_SWIGLU = 4,
           EPI_GROUP3 = 5, EPI_HEADNR = 6 };

struct QParams {
    const void *x;             // T [M, K]
    const uint32_t *w[3];      // packed weights per part
    const void *s[3];          // scales per part
    const void *b[3];          // biases per part
    int64_t noff[3];           // row offset of each part inside its weight
    const void *resid;         // T [M, Nout] (EPI_RESID)
    void *y0;                  // T [M, Nout]
    void *y1;                  // T [M, Nout] (EPI_SPLIT3, EPI_DUAL)
    int64_t M, Nout, K;
    int64_t pn[3];             // EPI_GROUP3: N of each part (Nout = their sum)
    void *py[3];               // EPI_GROUP3: output of each part, T [M, pn[i]]
    int gs;
    int gs_log2;               // log2(gs): group sizes are powers of two
    int wk;                    // K-split waves (qmm_mfma_kernel)
    int sbp;                   // qmm_mfma_kernel: groups per row of a wave's scale/bias table
    int n4;                    // qmm_mfma_mixed_kernel: feature tiles taken as 128-token tiles
    int sbninst;               // qmm_mfma_kernel: DMA instructions per scale/bias table array
    unsigned sbmagic;          // ceil(2^20 / (sbp / 2)): v / (sbp / 2) as (v * sbmagic) >> 20
    int ks;                    // K parts (kpart_count): each is split over the wk waves
    int kslice;                // k values a scale/bias table covers (a wave chunk, or all of K)
    int kint;                  // interleaved K split (kint_of): wave w takes stages w, w + wk, ...
    float *part;               // non-null: write K part blockIdx.z's sums, fp32 [ks, M, Nout]
    // EPI_HEADNR (the parts are q, k, v; py[] = q_out [B, Hq, L, D], k_cache,
    // v_cache [B, Hkv, cap, D]; D = 128)
    const void *nw[2];         // q_norm, k_norm: T [D]
    int64_t L;                 // tokens per sequence (M = B L)
    int64_t cap, pos0;         // cache rows per head; first row written
    int64_t offset;            // RoPE position of a sequence's token 0
    float eps, log2base, rscale;
};

constexpr int QMV_MR = 8;  // rows per GEMV block (and the GEMV/MFMA switch)
constexpr int LDS_PER_CU = 160 * 1024;

int device_cus();  // compute units of the current device (mi_gemv.hip)
// The GEMV kernels (few rows, fp32, shapes off the MFMA step): mi_gemv.hip.
int gemv_launch(const QParams &p, int epi, int bits, int dtype, hipStream_t st);

namespace {

// weight rows each output element combines (EPI_GROUP3 selects one weight per tile)
constexpr int epi_parts(int e) {
    return e == EPI_SPLIT3 ? 3 : ((e == EPI_DUAL || e == EPI_SWIGLU) ? 2 : 1);
}


template <typename T> __device__ __forceinline__ float swiglu1(float g, float u) {
    const float gt = (float)cvt<T>(g);
    const float sig = (float)cvt<T>(1.0f / (1.0f + __expf(-gt)));
    const float act = (float)cvt<T>(gt * sig);
    return act * (float)cvt<T>(u);
}

// The arrays one workgroup reads and writes, held as scalar fields with
// select accessors: the kernels never modify the QParams argument (a modified
// copy whose arrays are indexed in loops ends up in scratch memory).
struct Bound {
    const uint32_t *w0, *w1, *w2;
    const void *s0, *s1, *s2;
    const void *b0, *b1, *b2;
    int64_t o0, o1, o2;  // row offset of each part inside its weight
    void *y0;            // this workgroup's output
    int64_t Nout;        // its width
    int gp;              // EPI_GROUP3 / EPI_HEADNR: the part it lies in
    __device__ const uint32_t *w(int i) const { return i == 0 ? w0 : (i == 1 ? w1 : w2); }
    __device__ const void *s(int i) const { return i == 0 ? s0 : (i == 1 ? s1 : s2); }
    __device__ const void *b(int i) const { return i == 0 ? b0 : (i == 1 ? b1 : b2); }
    __device__ int64_t noff(int i) const { return i == 0 ? o0 : (i == 1 ? o1 : o2); }
};

// Binds a workgroup whose first output feature is nb. EPI_GROUP3: the three
// weights and outputs are concatenated along N and the host guarantees every
// part's N is a multiple of each tile width, so the whole tile lies in one
// part: bind that part as part 0 and make nb relative to it.
template <int EPI>
__device__ __forceinline__ Bound bind(const QParams &p, int64_t &nb) {
    Bound q = {p.w[0], p.w[1], p.w[2], p.s[0], p.s[1], p.s[2], p.b[0], p.b[1], p.b[2],
               p.noff[0], p.noff[1], p.noff[2], p.y0, p.Nout, 0};
    if constexpr (EPI == EPI_GROUP3 || EPI == EPI_HEADNR) {
        const int64_t e0 = p.pn[0], e1 = p.pn[0] + p.pn[1];
        const bool p0 = nb < e0, p1 = !p0 && nb < e1;
        nb -= p0 ? 0 : (p1 ? e0 : e1);
        q.w0 = p0 ? p.w[0] : (p1 ? p.w[1] : p.w[2]);
        q.s0 = p0 ? p.s[0] : (p1 ? p.s[1] : p.s[2]);
        q.b0 = p0 ? p.b[0] : (p1 ? p.b[1] : p.b[2]);
        q.y0 = p0 ? p.py[0] : (p1 ? p.py[1] : p.py[2]);
        q.Nout = p0 ? p.pn[0] : (p1 ? p.pn[1] : p.pn[2]);
        q.gp = p0 ? 0 : (p1 ? 1 : 2);
    }
    return q;
}

// Epilogue for one output element (m, n) of the output sub-space.
template <typename T, int EPI>
__device__ __forceinline__ void epi1(const QParams &p, const Bound &bd, int64_t m, int64_t n,
                                     const float *acc) {
    T *y0 = (T *)bd.y0;
    const int64_t o = m * bd.Nout + n;
    if constexpr (EPI == EPI_STORE || EPI == EPI_GROUP3 || EPI == EPI_HEADNR) {
        y0[o] = cvt<T>(acc[0]);
    } else if constexpr (EPI == EPI_RESID) {
        y0[o] = cvt<T>(pin32<T>((float)((const T *)p.resid)[o] + (float)cvt<T>(acc[0])));
    } else if constexpr (EPI == EPI_SPLIT3) {
        // split(3): parts 0, 1, 2 are B, C, x; outputs C and T(B * x)
        y0[o] = cvt<T>(acc[1]);
        ((T *)p.y1)[o] = cvt<T>((float)cvt<T>(acc[0]) * (float)cvt<T>(acc[2]));
    } else if constexpr (EPI == EPI_DUAL) {
        y0[o] = cvt<T>(acc[0]);
        ((T *)p.y1)[o] = cvt<T>(acc[1]);
    } else {
        y0[o] = cvt<T>(swiglu1<T>(acc[0], acc[1]));
    }
}

// Whether epi4 takes its vector path at (m, n): in range, four whole features.
__device__ __forceinline__ bool epi4_vec(const QParams &p, const Bound &bd, int64_t m, int64_t n) {
    return m < p.M && n + 4 <= bd.Nout && !(bd.Nout & 3);
}

// EPI_RESID: the residual's four values at (m, n) for epi4's vector path,
// loaded ahead so a wave's loads are all in flight before its first store
// (each epi4 loading its own had waited for every load in turn); zeros where
// the vector path does not run (the element path loads its own).
template <typename T>
__device__ __forceinline__ uint2 resid4(const QParams &p, const Bound &bd, int64_t m, int64_t n) {
    return epi4_vec(p, bd, m, n) ? ld8((const T *)p.resid + m * bd.Nout + n) : make_uint2(0u, 0u);
}

// Epilogue for 4 consecutive output features n..n+3 of token m; acc[part][e].
// rpre: EPI_RESID's residual from resid4 (null: loaded here).
template <typename T, int EPI, int P>
__device__ __forceinline__ void epi4(const QParams &p, const Bound &bd, int64_t m, int64_t n,
                                     const float (&acc)[P][4], const uint2 *rpre = nullptr) {
    if (m >= p.M || n >= bd.Nout) return;
    if (n + 4 > bd.Nout || (bd.Nout & 3)) {  // ragged tail: element stores
        for (int e = 0; e < 4 && n + e < bd.Nout; ++e) {
            float a[P];
#pragma unroll
            for (int q = 0; q < P; ++q) a[q] = acc[q][e];
            epi1<T, EPI>(p, bd, m, n + e, a);
        }
        return;
    }
    const int64_t o = m * bd.Nout + n;
    float v[4];
    if constexpr (EPI == EPI_STORE || EPI == EPI_GROUP3 || EPI == EPI_HEADNR) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = acc[0][e];
    } else if constexpr (EPI == EPI_RESID) {
        const uint2 rr = rpre ? *rpre : ld8((const T *)p.resid + o);
        typedef typename Vec<T>::x4 V4;
        const V4 rv = __builtin_bit_cast(V4, rr);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = pin32<T>((float)rv[e] + (float)cvt<T>(acc[0][e]));
    } else if constexpr (EPI == EPI_SPLIT3) {
        float bx[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[e] = acc[1][e];
            bx[e] = (float)cvt<T>(acc[0][e]) * (float)cvt<T>(acc[2][e]);
        }
        st8((T *)p.y1 + o, pack4<T>(bx));
    } else if constexpr (EPI == EPI_DUAL) {
        float u[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[e] = acc[0][e];
            u[e] = acc[1][e];
        }
        st8((T *)p.y1 + o, pack4<T>(u));
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = swiglu1<T>(acc[0][e], acc[1][e]);
    }
    st8((T *)bd.y0 + o, pack4<T>(v));
}

// A raw buffer resource over [base, base + bytes): 32-bit offsets, and reads
// past the end return zero instead of touching memory.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_rsrc(const void *base, uint32_t bytes) {
    // dword 3: 32-bit data format (gfx9 raw buffer access)
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, (int)bytes,
                                             0x00020000);
}

// s_waitcnt with vmcnt = N and no wait on the other counters (gfx9 encoding:
// vmcnt[3:0] at bits 3:0 and vmcnt[5:4] at bits 15:14, expcnt 7, lgkmcnt 15).
template <int N> __device__ __forceinline__ void wait_vmcnt() {
    static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit count");
    __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}

// s_waitcnt lgkmcnt(0) with no wait on vmcnt (63) or expcnt (7)
__device__ __forceinline__ void wait_lgkmcnt0() {
    __builtin_amdgcn_s_waitcnt(15 | (7 << 4) | (0 << 8) | (3 << 14));
}

}  // namespace
}  // namespace mi
