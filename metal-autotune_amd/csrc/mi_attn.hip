// Row A7: causal GQA scaled-dot-product attention (mx.fast.scaled_dot_product_attention
// with mask='causal' or none), flash-style over 32-key tiles.
//
// The arithmetic of one query row is fixed: its key tiles of 32 (from key 0)
// are dealt to four streams by tile index (stream w: tiles w, w + 4, ...);
// each stream runs its own online softmax from scratch; the streams' states
// are then folded as (0 + 1) + (2 + 3). Two kernels carry it out, bit for bit
// alike (same tile-update and merge functions, no floating-point contraction
// in them), whatever their work split:
//   attn_prefill_kernel  many query rows. A workgroup is two units (a unit: one
//                        q head's 32-row block; the units of one kv head are
//                        its q heads' blocks) of four waves, a wave a stream;
//                        the units share each stage of four key tiles in LDS.
//   attn_wave_kernel     few query rows. A workgroup is one unit, or (at most
//                        DEC_MAX_LQ rows: decode) the rows of all q heads of
//                        one kv head as the columns of one tile, so K and V
//                        are read once per kv head. A wave a stream, each with
//                        LDS of its own: no barrier before the fold.
// Past DEC_SPLIT_MIN_LK keys a decode call's key tiles are also cut into
// contiguous splits, one workgroup each, whose states attn_combine_kernel folds
// in split order (with a caller's workspace; without one a single workgroup
// runs all of them): the one case where a row's last bits depend on the call's
// shape.
// Per wave and tile:
//   S^T[key][q] = K . Q^T   32x32x16 MFMA, A = K rows, B = Q^T held in
//                           registers for the whole kernel;
//   lane (q = lane%32, half) then holds 16 of the 32 keys of its query row, so
//   the row max/sum needs one exchange between the wave's halves;
//   O^T[d][q] += V^T . P^T  A = V^T, read by transposing LDS loads from the
//                           V tile staged key-major as it sits in memory,
//                           B = P^T straight from the S^T registers
//                           (bf16/fp16): the k order inside each MFMA is
//                           permuted to match the S^T register layout, for
//                           both operands.
// K and V tiles go from memory to LDS by direct DMA (buffer_load ... lds), the
// 16-byte chunks of a row XOR-swizzled so the fragment reads hit distinct
// banks. Online softmax in the log2 domain, fp32 running max/sum, one division
// at the end. Causal masking is bottom-right aligned (query i sees keys
// j <= i + Lk - Lq) and key tiles past the last visible key are skipped.
// A row's result depends only on its global position and the keys, so a
// chunked prefill whose chunks start at multiples of 32 reproduces the whole
// prefill bit for bit, and a decode call the last prefill row; except that split
// calls (at most DEC_MAX_LQ rows over more than DEC_SPLIT_MIN_LK keys, with a
// workspace), a short last chunk among them, agree within rounding.
//
// What bounds it: at long prompts the softmax VALU, some 60 instructions and 16
// v_exp (a quarter-rate unit) for the 16 MFMAs of a tile at D = 128, 8 at D = 64
// (143 VALU a tile counted with everything in), and its waves' turns (two a SIMD at D = 128); for decode one memory round
// trip and the launches. Measured on MI355X in a graph, 32 q / 8 kv heads (in
// brackets: a form that masked and rescaled every score with 360 VALU a tile,
// staged tiles through registers, and ran decode on one workgroup per q head):
// 2048 tokens D = 128 61 us (85), D = 64 30 (60); 501 behind 777, D = 128, 19
// (54); 128 tokens 5.6 (6.5); decode over 129 keys 5.2 (7.6), 1001 9.6 (18.8),
// 8191 11.5 us, 2.9 TB/s of K and V (115).
#include <math.h>

#include "mi_common.h"

namespace mi {
namespace {

template <typename T> struct AMfma;
template <> struct AMfma<bf16> {
    static __device__ __forceinline__ f32x16 mma(bf16x8 a, bf16x8 b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    }
};
template <> struct AMfma<f16> {
    static __device__ __forceinline__ f32x16 mma(f16x8 a, f16x8 b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
    }
};

constexpr int ATT_KT = 32;       // keys per tile
constexpr int ATT_STREAMS = 4;   // key-tile streams per query row
constexpr int DEC_MAX_LQ = 8;    // query rows of a decode call (the GEMV row limit)
constexpr int64_t DEC_SPLIT_MIN_LK = 1024;  // keys past which decode calls are split

// Online-softmax state of one wave: O^T tiles (lane = query column r, half
// h2), the row's reference maximum m (log2 units) and this lane's half of the
// row sum l.
template <int D> struct AttnState {
    f32x16 o[D / 32];
    float m, l;
};

template <int D> __device__ __forceinline__ void attn_init(AttnState<D> &st) {
#pragma unroll
    for (int t = 0; t < D / 32; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) st.o[t][i] = 0.0f;
    st.m = -INFINITY;
    st.l = 0.0f;
}

// The larger of a lane's value and that of the lane 32 away, in both. (The pair's
// members are copied out first: a bit cast of a vector's subscript reads its first
// element, whatever the subscript.)
__device__ __forceinline__ float max_halves(float v) {
    typedef unsigned U2 __attribute__((ext_vector_type(2)));
    const unsigned u = __builtin_bit_cast(unsigned, v);
    const U2 r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    const unsigned lo = r[0], hi = r[1];
    return fmaxf(__builtin_bit_cast(float, lo), __builtin_bit_cast(float, hi));
}

// Scores of keys from `vis` on (of the tile's 32) set to -inf.
__device__ __forceinline__ void attn_mask(f32x16 &s, int vis, int h2) {
#pragma unroll
    for (int i = 0; i < 16; ++i)
        s[i] = 8 * (i / 4) + 4 * h2 + (i % 4) < vis ? s[i] : -INFINITY;
}

// Scores to probabilities of one key tile: s[i] = S^T (key 8*(i/4) + 4*h2 +
// i%4 of the tile, the lane's query row; -inf where the row does not see the
// key), pk gets 2^(s scale - m) in pairs of T, in register order. The row sum
// adds the fp32 values, in four chains (rounded to T first, the denominator
// would carry T's error of a probability, up to 2^-8 in bf16). scale > 0 (a
// negative scale was moved into Q's sign).
template <typename T, int D>
__device__ __forceinline__ void attn_softmax(AttnState<D> &st, const f32x16 &s, uint32_t (&pk)[8],
                                             float scale) {
#pragma clang fp contract(off)
    float mt = fmaxf(s[0], s[1]);
#pragma unroll
    for (int i = 2; i < 16; i += 2) mt = fmaxf(fmaxf(mt, s[i]), s[i + 1]);
    mt = max_halves(mt) * scale;
    // Lazy rescale: the exponents are taken against a running reference m
    // that moves only when a row's maximum passes it by more than 8 (log2
    // units). p then stays below 2^8, where fp32 sums and the bf16/fp16 P
    // operand keep their relative precision, and the accumulator rescales run
    // only on those (wave-uniform) steps.
    const bool grow = mt > st.m + 8.0f;
    if (__builtin_amdgcn_ballot_w64(grow) != 0) {
        const float m_new = grow ? mt : st.m;
        const float corr = st.m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(st.m - m_new);
        st.l *= corr;
#pragma unroll
        for (int t = 0; t < D / 32; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) st.o[t][i] *= corr;
        st.m = m_new;
    }
    // (a row that has seen no key yet: every score is -inf, and p is 0)
    const float nm = st.m == -INFINITY ? 0.0f : -st.m;
    float sum[4];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[2 * i], scale, nm));
        const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[2 * i + 1], scale, nm));
        pk[i] = pk2<T>(p0, p1);
        float &a = sum[2 * (i & 1)], &b = sum[2 * (i & 1) + 1];
        a = i < 2 ? p0 : a + p0;
        b = i < 2 ? p1 : b + p1;
    }
    st.l += (sum[0] + sum[1]) + (sum[2] + sum[3]);
}

// Swizzles of a staged tile: 16-byte chunk c of key row r sits at chunk
// position c ^ swz(r). K: the 32 rows' ds_read_b128 of one chunk spread over
// the banks. V: the four rows one transposing read covers (64 bytes of each)
// take four distinct 64-byte windows.
template <int D> __device__ __forceinline__ int swz_k(int r) {
    return D == 128 ? (r & 15) : ((r >> 1) & 7);
}
template <int D> __device__ __forceinline__ int swz_v(int r) {
    return D == 128 ? (r & 3) << 2 : ((r >> 1) & 1) << 2;
}

template <int D> struct Tile {
    static constexpr int BYTES = ATT_KT * D * 2;      // a K or V tile in LDS
    static constexpr int CPR = D / 8;                 // 16-byte chunks per row
    static constexpr int RPI = 64 / CPR;              // rows per DMA instruction
    static constexpr int NI = ATT_KT / RPI;           // DMA instructions per tile
};

typedef __attribute__((address_space(3))) void *lds_ptr;

// Division of a block or unit index by a launch constant: a multiply by
// ceil(2^32 / d), exact for n d < 2^32 (the host checks the largest n; else m =
// 0 and the quotient is computed), where a division costs a workgroup tens of
// dependent scalar instructions before its first load.
struct Div {
    unsigned d, m;
    __device__ __forceinline__ unsigned of(unsigned n) const {
        if (d == 1) return n;
        return m ? __umulhi(n, m) : n / d;
    }
};
inline Div make_div(int64_t d, int64_t n_max) {
    const bool exact = d > 1 && n_max * d < ((int64_t)1 << 32);
    return {(unsigned)d, exact ? (unsigned)((((uint64_t)1 << 32) + d - 1) / d) : 0u};
}

#if defined(__HIP_DEVICE_COMPILE__)
// A raw buffer resource over [base, base + bytes): reads past the end return
// zero instead of touching memory.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t att_rsrc(const void *base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, (int)bytes,
                                             0x00020000);
}

// DMA instructions [i0, i0 + n) of key tile kt of one kv head's K or V (base:
// its row 0) into the tile's LDS. Rows past Lk, whole tiles too, arrive as
// zeros without a memory access (the resource ends at row Lk).
template <typename T, int D, bool ISV>
__device__ __forceinline__ void dma_tile(const T *base, int64_t kt, int64_t Lk, char *dst, int i0,
                                         int n, int lane) {
    typedef Tile<D> Tl;
    const int64_t left = Lk - kt * ATT_KT;
    const int rows = left < 0 ? 0 : (left < ATT_KT ? (int)left : ATT_KT);
    const __amdgpu_buffer_rsrc_t rs =
        att_rsrc(base + (rows ? kt * ATT_KT * D : 0), (uint32_t)(rows * D * 2));
#pragma unroll
    for (int i = 0; i < n; ++i) {
        const int row = (i0 + i) * Tl::RPI + lane / Tl::CPR, pos = lane % Tl::CPR;
        const int c = pos ^ (ISV ? swz_v<D>(row) : swz_k<D>(row));
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr)(dst + (i0 + i) * 1024), 16,
                                                 (row * D + 8 * c) * 2, 0, 0, 0);
    }
}
#endif

// s_waitcnt with vmcnt = N and no wait on the other counters.
template <int N> __device__ __forceinline__ void att_wait_vmcnt() {
    static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit count");
    __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}
// s_waitcnt lgkmcnt(0) alone.
__device__ __forceinline__ void att_wait_lds() {
    __builtin_amdgcn_s_waitcnt(15 | (7 << 4) | (0 << 8) | (3 << 14));
}

// K fragments of the lane: row r, head-dim chunk 16 s + 8 h2 of MFMA step s.
template <int D>
__device__ __forceinline__ void read_k(const char *ks, uint4 (&kf)[D / 16], int r, int h2) {
    const int a = r * (D * 2) + ((h2 ^ swz_k<D>(r)) << 4);
#pragma unroll
    for (int s = 0; s < D / 16; ++s) kf[s] = *(const uint4 *)(ks + (a ^ (s << 5)));
}

template <typename T, int D>
__device__ __forceinline__ f32x16 attn_scores(const uint4 (&kf)[D / 16], const uint4 (&qf)[D / 16]) {
    typedef typename Vec<T>::x8 V8;
    f32x16 s;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.0f;
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks)
        s = AMfma<T>::mma(__builtin_bit_cast(V8, kf[ks]), __builtin_bit_cast(V8, qf[ks]), s);
    return s;
}

// Four 16-bit values by ds_read_b64_tr_b16. Within each 16-lane group, with
// lane s addressing four consecutive values E[s][0..3], lane 4a + b receives
// (E[a][b], E[a + 4][b], E[a + 8][b], E[a + 12][b]) (probed on gfx950: LDS
// filled with each value's index, lanes addressing rows of 4 and of 16).
template <typename T>
__device__ __forceinline__ typename Vec<T>::x4 lds_read_tr4(const char *p) {
    typedef short S4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) S4 *LP;
    return __builtin_bit_cast(typename Vec<T>::x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((LP)p));
}

// O^T += V^T . P^T over one tile, in two steps: read_v fetches the A fragments
// (before the softmax, whose arithmetic then covers the LDS latency: read at
// their MFMAs, each pair of reads was waited for in turn), attn_pv runs the
// MFMAs. The fragment of lane (r, h2), MFMA k2 of head-dim tile t, is
// V^T[32 t + r][keys 16 k2 + 4 h2 + (0..3), then the same + 8]. Lane s of
// 16-lane group G addresses key row 16 k2 + 4 (G / 2) + s / 4 at column 32 t +
// 16 (G % 2) + 4 (s % 4); by the rule above lane 4a + b of the group (r = 16
// (G % 2) + 4a + b) then receives column 32 t + r of the key rows 16 k2 + 4 h2
// + 0..3.
template <typename T, int D> struct VFrag {
    typename Vec<T>::x4 v[D / 32][2][2];
};
template <typename T, int D>
__device__ __forceinline__ void read_v(const char *vs, VFrag<T, D> &f, int lane) {
    const int s = lane & 15, g = lane >> 4;
    const int row = 4 * (g >> 1) + (s >> 2);  // + 16 k2 (+ 8): the same swizzle
    const int low = ((2 * (g & 1) + ((s & 3) >> 1)) << 4) + 8 * (s & 1);
    const int a0 = row * (D * 2) + low, z = swz_v<D>(row) << 4;
#pragma unroll
    for (int t = 0; t < D / 32; ++t) {
        const char *vr = vs + a0 + ((t << 6) ^ z);
#pragma unroll
        for (int k2 = 0; k2 < 2; ++k2) {
            f.v[t][k2][0] = lds_read_tr4<T>(vr + (16 * k2) * (D * 2));
            f.v[t][k2][1] = lds_read_tr4<T>(vr + (16 * k2 + 8) * (D * 2));
        }
    }
}
template <typename T, int D>
__device__ __forceinline__ void attn_pv(AttnState<D> &st, const uint32_t (&pk)[8],
                                        const VFrag<T, D> &f) {
    typedef typename Vec<T>::x8 V8;
    const V8 pb[2] = {__builtin_bit_cast(V8, (uint4){pk[0], pk[1], pk[2], pk[3]}),
                      __builtin_bit_cast(V8, (uint4){pk[4], pk[5], pk[6], pk[7]})};
#pragma unroll
    for (int k2 = 0; k2 < 2; ++k2)
#pragma unroll
        for (int t = 0; t < D / 32; ++t) {
            V8 a;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                a[e] = f.v[t][k2][0][e];
                a[4 + e] = f.v[t][k2][1][e];
            }
            st.o[t] = AMfma<T>::mma(a, pb[k2], st.o[t]);
        }
}

// Folding a later state (mw, lw, o_w) into an earlier (m, l, o):
// m' = max(m, mw); o' = o c0 + o_w cw and l' = l c0 + lw cw with
// c0 = 2^(m - m'), cw = 2^(mw - m'); a state that saw no visible key of the
// row (m = -inf) has coefficient 0.
struct MergeCoef {
    float c0, cw, m_new;
};
__device__ __forceinline__ MergeCoef merge_coef(float m, float mw) {
#pragma clang fp contract(off)
    const float m_new = fmaxf(m, mw);
    return {m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m - m_new),
            mw == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mw - m_new), m_new};
}
__device__ __forceinline__ float merge_one(float o, float ow, const MergeCoef &c) {
#pragma clang fp contract(off)
    return __builtin_fmaf(o, c.c0, ow * c.cw);
}

// 1 / the row's sum (both halves), 0 for a row that saw no key.
__device__ __forceinline__ float row_inv(float l) {
#pragma clang fp contract(off)
    const float l_tot = l + __shfl_xor(l, 32, 64);
    return l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
}

// Key tiles visible to a q block (causal: up to its last row).
__device__ __forceinline__ int attn_ntiles(int64_t q0, int64_t off, int64_t Lk, int causal) {
    int64_t kend = Lk;
    if (causal) {
        const int64_t last = q0 + 31 + off + 1;
        kend = last < Lk ? last : Lk;
    }
    return kend > 0 ? (int)ceil_div(kend, ATT_KT) : 0;
}

// The Q fragments of a row.
template <int D>
__device__ __forceinline__ void read_q(const void *row, int h2, uint4 (&qf)[D / 16]) {
    const char *qp = (const char *)row + 16 * h2;
#pragma unroll
    for (int s = 0; s < D / 16; ++s) qf[s] = ld16(qp + 32 * s);
}
// The sign of a negative scale moved into them (exact), once: called where they
// have landed, so that the loads in flight behind them are not waited for.
template <int D> __device__ __forceinline__ void flip_q(uint4 (&qf)[D / 16], uint32_t &flip) {
    if (flip == 0) return;  // (uniform)
#pragma unroll
    for (int s = 0; s < D / 16; ++s)
        qf[s].x ^= flip, qf[s].y ^= flip, qf[s].z ^= flip, qf[s].w ^= flip;
    flip = 0;
}

// A wave's state in LDS for the last fold: float4 [D / 32 * 4][64] (registers
// 4j .. 4j + 3 of tile t at t * 4 + j), then float2 (l, m) [64].
template <int D> struct Part {
    static constexpr int WORDS = D / 32 * 4 * 64 + 32;  // 16-byte words
    static constexpr int BYTES = WORDS * 16;
};
template <int D>
__device__ __forceinline__ void part_put(float4 *pp, const AttnState<D> &st, int t, int lane) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
        pp[(t * 4 + j) * 64 + lane] = make_float4(st.o[t][4 * j], st.o[t][4 * j + 1],
                                                  st.o[t][4 * j + 2], st.o[t][4 * j + 3]);
}
template <int D> __device__ __forceinline__ float2 *part_lm(float4 *pp) {
    return (float2 *)(pp + D / 32 * 4 * 64);
}
struct Fold {  // one O^T tile of a state
    float4 o[4];
    float l, m;
};
__device__ __forceinline__ void fold(Fold &a, const Fold &b) {
    const MergeCoef c = merge_coef(a.m, b.m);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        a.o[j].x = merge_one(a.o[j].x, b.o[j].x, c);
        a.o[j].y = merge_one(a.o[j].y, b.o[j].y, c);
        a.o[j].z = merge_one(a.o[j].z, b.o[j].z, c);
        a.o[j].w = merge_one(a.o[j].w, b.o[j].w, c);
    }
    a.l = merge_one(a.l, b.l, c);
    a.m = c.m_new;
}
template <int D>
__device__ __forceinline__ Fold part_get(float4 *pp, int t, int lane) {
    Fold f;
#pragma unroll
    for (int j = 0; j < 4; ++j) f.o[j] = pp[(t * 4 + j) * 64 + lane];
    const float2 lm = part_lm<D>(pp)[lane];
    f.l = lm.x;
    f.m = lm.y;
    return f;
}

// O^T tile t of the four streams' states at part, folded (0 + 1) + (2 + 3).
template <int D> __device__ __forceinline__ Fold fold_streams(float4 *part, int t, int lane) {
    Fold f = part_get<D>(part, t, lane);
    fold(f, part_get<D>(part + Part<D>::WORDS, t, lane));
    Fold g = part_get<D>(part + 2 * Part<D>::WORDS, t, lane);
    fold(g, part_get<D>(part + 3 * Part<D>::WORDS, t, lane));
    fold(f, g);
    return f;
}
template <typename T>
__device__ __forceinline__ void store_fold(const Fold &f, float inv, T *orow, int t, int h2) {
#pragma clang fp contract(off)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float e[4] = {f.o[j].x * inv, f.o[j].y * inv, f.o[j].z * inv, f.o[j].w * inv};
        st8(orow + 32 * t + 8 * j + 4 * h2, pack4<T>(e));
    }
}

// ---------------------------------------------------------------------------
// attn_prefill_kernel

// LDS: two stages (a key tile of K, then of V, per stream), reused for the fold.
template <int D, int HW> struct PrefillLds {
    static constexpr int STAGE = 2 * ATT_STREAMS * Tile<D>::BYTES;
    static constexpr int FOLD = HW * ATT_STREAMS * Part<D>::BYTES;
    static constexpr int BYTES = 2 * STAGE > FOLD ? 2 * STAGE : FOLD;
};
// (64-value heads fit four waves a SIMD, two workgroups of eight a CU)
template <int D> constexpr int prefill_waves_per_eu() { return D == 64 ? 4 : 2; }

template <typename T, int D, int HW>
__global__ __launch_bounds__(256 * HW)
__attribute__((amdgpu_waves_per_eu(prefill_waves_per_eu<D>()))) void attn_prefill_kernel(
    const T *__restrict__ q, const T *__restrict__ k, const T *__restrict__ v,
    T *__restrict__ out, int64_t H, int64_t Lq, int64_t Lk, int64_t cap, float scale,
    uint32_t flip, int causal, int out_layout, Div nbk, Div HK, Div rep, unsigned units,
    unsigned nub) {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef Tile<D> Tl;
    typedef PrefillLds<D, HW> L;
    constexpr int SW = ATT_STREAMS;
    constexpr int NI = Tl::NI / HW;  // DMA instructions of a tile a wave issues
    static_assert(Tl::NI % HW == 0, "a tile's DMA splits over the units' waves");
    __shared__ __attribute__((aligned(1024))) char lds[L::BYTES];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int hw = wave / SW, ws = wave % SW;  // unit slot, stream
    const int h2 = lane >> 5, r = lane & 31;
    // Blocks: kv heads fastest (consecutive blocks go to the XCDs in turn, so
    // with 8 kv heads each XCD's L2 holds one head's K and V), the units with
    // the most key tiles first (the grid then drains evenly). nbk = B HK.
    const unsigned bid = blockIdx.x, bq = nbk.of(bid), bk = bid - bq * nbk.d, ub = nub - 1 - bq;
    const unsigned bb = HK.d == nbk.d ? 0u : HK.of(bk);
    const int64_t b = bb, hk = bk - bb * HK.d;
    const unsigned u = ub * HW + hw;
    const bool active = u < units;
    const unsigned uc = active ? u : units - 1, uq = rep.of(uc);
    const int64_t hq = hk * rep.d + (uc - uq * rep.d), q0 = (int64_t)uq * 32;
    const int64_t off = Lk - Lq, qrow = q0 + r;
    const bool qok = active && qrow < Lq;
    const int nt = active ? attn_ntiles(q0, off, Lk, causal) : 0;
    // the workgroup's last unit has the most tiles
    const unsigned ul = ub * HW + HW - 1 < units ? ub * HW + HW - 1 : units - 1;
    const int total = (attn_ntiles((int64_t)rep.of(ul) * 32, off, Lk, causal) + SW - 1) / SW;
    const T *kb = k + (int64_t)bk * cap * D;
    const T *vb = v + (int64_t)bk * cap * D;

    // Stage i holds key tiles 4 i .. 4 i + 3; the waves of one stream share
    // its tile's DMA.
    auto issue = [&](int i, char *dst) {
        const int kt = SW * i + ws;
        dma_tile<T, D, false>(kb, kt, Lk, dst + ws * Tl::BYTES, hw * NI, NI, lane);
        dma_tile<T, D, true>(vb, kt, Lk, dst + (SW + ws) * Tl::BYTES, hw * NI, NI, lane);
    };
    AttnState<D> st;
    attn_init(st);
    uint4 qf[D / 16];
    // tiles before nfull: every row of the block sees all 32 keys
    const int64_t seen = causal && q0 + off + 1 < Lk ? q0 + off + 1 : Lk;
    const int nfull = (int)(seen / ATT_KT);
    const int64_t end = causal && qrow + off + 1 < Lk ? qrow + off + 1 : Lk;
    // One stage: cb is read, the next stage's DMAs land in nb. (restrict:
    // the waits the compiler adds before LDS reads then leave those DMAs in
    // flight.)
    auto step = [&](const char *__restrict__ cb, char *__restrict__ nb, int i)
                    __attribute__((always_inline)) {
        // every wave's DMAs of stage i have landed, and every wave is done with
        // the buffer the next ones go to
        att_wait_vmcnt<0>();
        __syncthreads();
        flip_q<D>(qf, flip);
        if (i + 1 < total) issue(i + 1, nb);
        const int kt = SW * i + ws;
        if (kt < nt) {  // wave-uniform
            uint4 kf[D / 16];
            read_k<D>(cb + ws * Tl::BYTES, kf, r, h2);
            VFrag<T, D> vf;
            read_v<T, D>(cb + (SW + ws) * Tl::BYTES, vf, lane);
            __builtin_amdgcn_sched_barrier(0);  // (not sunk to the PV MFMAs)
            f32x16 s = attn_scores<T, D>(kf, qf);
            if (kt >= nfull) attn_mask(s, (int)(end - (int64_t)kt * ATT_KT), h2);
            uint32_t p[8];
            attn_softmax<T, D>(st, s, p, scale);
            attn_pv<T, D>(st, p, vf);
        }
    };
    char *buf0 = lds, *buf1 = lds + L::STAGE;
    if (total > 0) issue(0, buf0);
    // (a row past the last reads the first: its results are not stored)
    read_q<D>(q + ((b * H + hq) * Lq + (qok ? qrow : 0)) * D, h2, qf);
    for (int i = 0; i < total; i += 2) {  // workgroup-uniform
        step(buf0, buf1, i);
        if (i + 1 < total) step(buf1, buf0, i + 1);
    }

    // The fold, (0 + 1) + (2 + 3): the states pass through LDS, and wave t of
    // a unit folds and stores its O^T tile t.
    __syncthreads();  // every wave is done with the stages
    float4 *part = (float4 *)lds + (size_t)(hw * SW) * Part<D>::WORDS;
    float4 *mine = part + (size_t)ws * Part<D>::WORDS;
#pragma unroll
    for (int t = 0; t < D / 32; ++t) part_put<D>(mine, st, t, lane);
    part_lm<D>(mine)[lane] = make_float2(st.l, st.m);
    __syncthreads();
    if (ws >= D / 32) return;
    const Fold f = fold_streams<D>(part, ws, lane);
    const float inv = row_inv(f.l);
    T *orow = out_layout ? out + ((b * Lq + qrow) * H + hq) * D
                         : out + ((b * H + hq) * Lq + qrow) * D;
    if (qok) store_fold<T>(f, inv, orow, ws, h2);
#endif
}

// ---------------------------------------------------------------------------
// attn_wave_kernel: four waves, a stream each; a wave owns its tiles' LDS: no
// barrier until the fold. One K and one V slot a wave; each is refilled with
// the wave's next tile as soon as its reads are in registers, so K's next tile
// flies under the softmax and the PV MFMAs, V's under the next scores.
// PACK (decode): grid (column block, split). Column c of block cb is row idx =
// 32 cb + c of the kv head's rep Lq query rows (q head idx / Lq, query row idx
// % Lq: contiguous in q). Otherwise the grid is attn_prefill_kernel's with one
// unit a workgroup.
constexpr int DEC_WAVES = ATT_STREAMS;
template <int D> struct DecodeLds {
    static constexpr int SLOTS = DEC_WAVES * 2 * Tile<D>::BYTES;
    static constexpr int FOLD = DEC_WAVES * Part<D>::BYTES;
    static constexpr int BYTES = SLOTS > FOLD ? SLOTS : FOLD;
};

template <typename T, int D, bool PACK>
__global__ __launch_bounds__(64 * DEC_WAVES) void attn_wave_kernel(
    const T *__restrict__ q, const T *__restrict__ k, const T *__restrict__ v,
    T *__restrict__ out, float *__restrict__ part_o, float2 *__restrict__ part_lm_out, int64_t H,
    int64_t Lq, int64_t Lk, int64_t cap, float scale, uint32_t flip, int causal, int out_layout,
    Div ncb, Div nbk, Div HK, Div rep, int cols, int tps) {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef Tile<D> Tl;
    __shared__ __attribute__((aligned(1024))) char lds[DecodeLds<D>::BYTES];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int h2 = lane >> 5, r = lane & 31;
    const unsigned bid = blockIdx.x, split = PACK ? blockIdx.y : 0u;
    // causal: query row i sees keys j <= i + off
    const int64_t off = Lk - Lq;
    unsigned bk, bb;
    int idx = 0, ntiles;
    int64_t hq, hk, qrow, full_end;
    bool ok;
    if constexpr (PACK) {
        bk = ncb.of(bid);
        bb = HK.d == nbk.d ? 0u : HK.of(bk);
        hk = bk - bb * HK.d;
        idx = (int)(bid - bk * ncb.d) * 32 + r;
        ok = idx < cols;
        const int hrow = Lq == 1 ? idx : (int)((unsigned)idx / (unsigned)Lq);
        qrow = idx - hrow * (int)Lq;
        hq = hk * rep.d + hrow;
        full_end = causal ? off + 1 : Lk;  // every row sees the keys before it
        ntiles = (int)ceil_div(Lk, ATT_KT);
    } else {
        // the units with the most key tiles first; nbk blocks a unit
        const unsigned bq = nbk.of(bid), u = (unsigned)cols - 1 - bq;  // cols: units
        bk = bid - bq * nbk.d;
        bb = HK.d == nbk.d ? 0u : HK.of(bk);
        hk = bk - bb * HK.d;
        const unsigned uq = rep.of(u);
        hq = hk * rep.d + (u - uq * rep.d);
        const int64_t q0 = (int64_t)uq * 32;
        qrow = q0 + r;
        ok = qrow < Lq;
        full_end = causal && q0 + off + 1 < Lk ? q0 + off + 1 : Lk;
        ntiles = attn_ntiles(q0, off, Lk, causal);
    }
    const int64_t b = bb, end = causal && qrow + off + 1 < Lk ? qrow + off + 1 : Lk;
    const T *kb = k + (int64_t)bk * cap * D;
    const T *vb = v + (int64_t)bk * cap * D;
    const int t0 = (int)split * tps, t1 = !PACK || t0 + tps > ntiles ? ntiles : t0 + tps;

    char *kslot = lds + wave * 2 * Tl::BYTES, *vslot = kslot + Tl::BYTES;
    const int first = t0 + wave;  // tps is a multiple of four: stream = wave
    AttnState<D> st;
    attn_init(st);
    uint4 qf[D / 16];
    auto run = [&](char *__restrict__ ks, char *__restrict__ vs) __attribute__((always_inline)) {
        // (a column without a row reads the first: its results are not stored)
        read_q<D>(q + ((b * H + (ok ? hq : 0)) * Lq + (ok ? qrow : 0)) * D, h2, qf);
        if (first < t1) {
            dma_tile<T, D, false>(kb, first, Lk, ks, 0, Tl::NI, lane);
            dma_tile<T, D, true>(vb, first, Lk, vs, 0, Tl::NI, lane);
        }
        for (int kt = first; kt < t1; kt += DEC_WAVES) {  // wave-uniform
            const bool more = kt + DEC_WAVES < t1;
            // K (and, the first time, q) has landed once only V's loads, issued
            // after it, are in flight
            att_wait_vmcnt<Tl::NI>();
            flip_q<D>(qf, flip);
            uint4 kf[D / 16];
            read_k<D>(ks, kf, r, h2);
#pragma unroll
            for (int s = 0; s < D / 16; ++s) launder(kf[s]);  // the reads have returned
            __builtin_amdgcn_sched_barrier(0);
            if (more) dma_tile<T, D, false>(kb, kt + DEC_WAVES, Lk, ks, 0, Tl::NI, lane);
            f32x16 s = attn_scores<T, D>(kf, qf);
            const int64_t k0 = (int64_t)kt * ATT_KT;
            if (k0 + ATT_KT > full_end) attn_mask(s, (int)(end - k0), h2);
            uint32_t p[8];
            attn_softmax<T, D>(st, s, p, scale);
            if (more)
                att_wait_vmcnt<Tl::NI>();
            else
                att_wait_vmcnt<0>();
            VFrag<T, D> vf;
            read_v<T, D>(vs, vf, lane);
            attn_pv<T, D>(st, p, vf);
            __builtin_amdgcn_sched_barrier(0);
            att_wait_lds();  // V's reads have returned
            if (more) dma_tile<T, D, true>(vb, kt + DEC_WAVES, Lk, vs, 0, Tl::NI, lane);
        }
    };
    run(kslot, vslot);

    // fold (0 + 1) + (2 + 3), as in the prefill kernel: wave t folds O^T tile t
    __syncthreads();
    float4 *part = (float4 *)lds;
    float4 *mine = part + (size_t)wave * Part<D>::WORDS;
    if (ok) {
#pragma unroll
        for (int t = 0; t < D / 32; ++t) part_put<D>(mine, st, t, lane);
        part_lm<D>(mine)[lane] = make_float2(st.l, st.m);
    }
    __syncthreads();
    if (wave >= D / 32) return;
    const int t = wave;
    const Fold f = fold_streams<D>(part, t, lane);  // (lanes without a column: unused)
    if (PACK && part_o) {  // one split's state, for attn_combine_kernel
        const int64_t rows = (int64_t)ncb.of(gridDim.x) * cols;
        const int64_t row = (int64_t)bk * cols + idx;
        const float l_tot = f.l + __shfl_xor(f.l, 32, 64);
        if (!ok) return;
        float *o = part_o + ((int64_t)split * rows + row) * D + 32 * t + 4 * h2;
#pragma unroll
        for (int j = 0; j < 4; ++j) *(float4 *)(o + 8 * j) = f.o[j];
        if (t == 0 && h2 == 0) part_lm_out[(int64_t)split * rows + row] = make_float2(l_tot, f.m);
        return;
    }
    const float inv = row_inv(f.l);
    if (!ok) return;
    T *orow = out_layout ? out + ((b * Lq + qrow) * H + hq) * D
                         : out + ((b * H + hq) * Lq + qrow) * D;
    store_fold<T>(f, inv, orow, t, h2);
#endif
}

// One query row (b, q head, query row) per workgroup: out = sum_s w_s O_s /
// sum_s w_s l_s with w_s = 2^(m_s - max m), s over the splits. The weights
// first (a lane a split), then 256 / (D / 4) thread groups take every so manyth
// split, in order, and the groups are added in order.
constexpr int DEC_MAX_SPLITS = 512;
template <typename T, int D>
__global__ __launch_bounds__(256) void attn_combine_kernel(const float *__restrict__ part_o,
                                                           const float2 *__restrict__ part_lm_in,
                                                           T *__restrict__ out, int64_t H,
                                                           int64_t Lq, int nsplit,
                                                           int out_layout) {
#pragma clang fp contract(off)
    constexpr int LANES = D / 4, GROUPS = 256 / LANES, IN_FLIGHT = 8;
    __shared__ float wt[DEC_MAX_SPLITS];
    __shared__ float4 acc[GROUPS][LANES];
    __shared__ float lw[4];
    const int64_t rows = gridDim.x, row = blockIdx.x;
    const int c = threadIdx.x % LANES, g = threadIdx.x / LANES;
    // this thread's first partial sums, requested before the weights are known
    const float *po = part_o + row * D + 4 * c;
    float4 v[IN_FLIGHT];
#pragma unroll
    for (int i = 0; i < IN_FLIGHT; ++i) {
        const int s = g + GROUPS * i;
        v[i] = *(const float4 *)(po + (s < nsplit ? s : 0) * rows * D);
    }
    float m = -INFINITY;
    for (int s = threadIdx.x & 63; s < nsplit; s += 64) m = fmaxf(m, part_lm_in[s * rows + row].y);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
    float l = 0.0f;
    for (int s = threadIdx.x; s < nsplit; s += 256) {
        const float2 lm = part_lm_in[s * rows + row];
        const float w = lm.y == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(lm.y - m);
        wt[s] = w;
        l = __builtin_fmaf(w, lm.x, l);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) l += __shfl_xor(l, o, 64);
    if ((threadIdx.x & 63) == 0) lw[threadIdx.x >> 6] = l;
    __syncthreads();
    float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int s0 = g; s0 < nsplit; s0 += GROUPS * IN_FLIGHT) {
        if (s0 != g) {
#pragma unroll
            for (int i = 0; i < IN_FLIGHT; ++i) {
                const int s = s0 + GROUPS * i;
                v[i] = *(const float4 *)(po + (s < nsplit ? s : 0) * rows * D);
            }
        }
#pragma unroll
        for (int i = 0; i < IN_FLIGHT; ++i) {
            const int s = s0 + GROUPS * i;
            if (s < nsplit) {
                const float w = wt[s];
                o.x = __builtin_fmaf(w, v[i].x, o.x);
                o.y = __builtin_fmaf(w, v[i].y, o.y);
                o.z = __builtin_fmaf(w, v[i].z, o.z);
                o.w = __builtin_fmaf(w, v[i].w, o.w);
            }
        }
    }
    acc[g][c] = o;
    __syncthreads();
    if (g) return;
#pragma unroll
    for (int i = 1; i < GROUPS; ++i) {
        const float4 a = acc[i][c];
        o.x += a.x;
        o.y += a.y;
        o.z += a.z;
        o.w += a.w;
    }
    l = ((lw[0] + lw[1]) + lw[2]) + lw[3];
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
    const int64_t bh = row / Lq, lq = row % Lq, b = bh / H, h = bh % H;
    T *orow = out_layout ? out + ((b * Lq + lq) * H + h) * D : out + row * D;
    const float e[4] = {o.x * inv, o.y * inv, o.z * inv, o.w * inv};
    st8(orow + 4 * c, pack4<T>(e));
}

// ---------------------------------------------------------------------------
// dispatch

struct AttnArgs {
    const void *q, *k, *v;
    void *out;
    int64_t B, H, HK, Lq, Lk, cap;
    float scale;    // > 0, log2 units
    uint32_t flip;  // sign bits of a negative scale, for Q
    int causal, out_layout;
};

// Splits of a decode call and key tiles per split (a multiple of four: the
// streams keep their tiles). One workgroup per split and column block; past
// DEC_SPLIT_MIN_LK keys as many as put two workgroups on every CU (256), each
// wave at least one tile. Up to that line one workgroup a kv head, so that a
// decode row keeps the bits of the prefill's there (by time alone the line would
// lie lower: 1001 keys unsplit take 9.6 us, 1025 split 8.1).
struct DecSplit {
    int ncb, nsplit, tps;
};
inline DecSplit decode_split(int64_t B, int64_t H, int64_t HK, int64_t Lq, int64_t Lk) {
    const int ncb = (int)ceil_div(H / HK * Lq, 32);
    const int64_t quads = ceil_div(ceil_div(Lk, ATT_KT), ATT_STREAMS);
    int64_t n = 1;
    if (Lk > DEC_SPLIT_MIN_LK) {
        n = DEC_MAX_SPLITS / (B * HK * ncb);
        n = n < 1 ? 1 : (n > quads ? quads : n);
    }
    const int64_t tps = ceil_div(quads, n) * ATT_STREAMS;
    return {ncb, (int)ceil_div(quads * ATT_STREAMS, tps), (int)tps};
}

template <typename T, int D>
int launch_decode(const AttnArgs &a, float *ws, hipStream_t st) {
    DecSplit d = decode_split(a.B, a.H, a.HK, a.Lq, a.Lk);
    if (!ws) {
        d.tps = (int)(ceil_div(ceil_div(a.Lk, ATT_KT), ATT_STREAMS) * ATT_STREAMS);
        d.nsplit = 1;
    }
    const int64_t rows = a.B * a.H * a.Lq, nbk = a.B * a.HK, rep = a.H / a.HK;
    float *po = d.nsplit > 1 ? ws : nullptr;
    float2 *plm = d.nsplit > 1 ? (float2 *)(ws + d.nsplit * rows * D) : nullptr;
    const dim3 grid((unsigned)(nbk * d.ncb), (unsigned)d.nsplit);
    attn_wave_kernel<T, D, true><<<grid, 64 * DEC_WAVES, 0, st>>>(
        (const T *)a.q, (const T *)a.k, (const T *)a.v, (T *)a.out, po, plm, a.H, a.Lq, a.Lk,
        a.cap, a.scale, a.flip, a.causal, a.out_layout, make_div(d.ncb, nbk * d.ncb),
        make_div(nbk, nbk), make_div(a.HK, nbk), make_div(rep, rep), (int)(rep * a.Lq), d.tps);
    if (d.nsplit > 1)
        attn_combine_kernel<T, D><<<(unsigned)rows, 256, 0, st>>>(po, plm, (T *)a.out, a.H, a.Lq,
                                                                  d.nsplit, a.out_layout);
    return launch_status("sdpa (decode)");
}

// Two units (q heads' 32-row blocks) share each staged K/V tile where that leaves
// a workgroup for most CUs and the rows are long (half the K/V traffic, two waves a
// SIMD); else one unit a workgroup, of which a CU holds two and whose waves wait
// for no barrier (64 tokens 5.05 us against 6.2 for one unit through the shared
// stages, 16 behind 4080 26.6 against 35). Short rows fill few of the stages: 205
// tokens, 64/8 heads of 64 5.2 / 6.4; 265 tokens, 64/8 of 128 10.1 / 14.4; 16 x 289
// tokens 114 / 150. Past 256 keys only while K and V of all heads (a unit reads
// its own copy) stay in the caches: 8 x 436 tokens, 64/32 heads of 128 (57 MB) 226
// / 161. Same results.
template <typename T, int D>
int launch_attn_d(const AttnArgs &a, float *ws, hipStream_t st) {
    if (a.Lq <= DEC_MAX_LQ) return launch_decode<T, D>(a, ws, st);
    const int64_t rep = a.H / a.HK, units = rep * ceil_div(a.Lq, 32), nbk = a.B * a.HK;
    const int64_t nub = ceil_div(units, 2);
    const bool short_rows =
        a.Lk <= 256 || (a.Lk <= 640 && nbk * a.Lk * D * 4 <= ((int64_t)40 << 20));
    if (nbk * nub >= 192 && !short_rows)
        attn_prefill_kernel<T, D, 2><<<(unsigned)(nbk * nub), 512, 0, st>>>(
            (const T *)a.q, (const T *)a.k, (const T *)a.v, (T *)a.out, a.H, a.Lq, a.Lk, a.cap,
            a.scale, a.flip, a.causal, a.out_layout, make_div(nbk, nbk * nub),
            make_div(a.HK, nbk), make_div(rep, units), (unsigned)units, (unsigned)nub);
    else
        attn_wave_kernel<T, D, false><<<(unsigned)(nbk * units), 64 * DEC_WAVES, 0, st>>>(
            (const T *)a.q, (const T *)a.k, (const T *)a.v, (T *)a.out, nullptr, nullptr, a.H,
            a.Lq, a.Lk, a.cap, a.scale, a.flip, a.causal, a.out_layout, make_div(1, 1),
            make_div(nbk, nbk * units), make_div(a.HK, nbk), make_div(rep, units), (int)units, 0);
    return launch_status("sdpa");
}

int run_sdpa(const void *q, const void *k, const void *v, void *out, int64_t B, int64_t H,
             int64_t HK, int64_t Lq, int64_t Lk, int64_t D, int64_t kv_cap, float scale,
             int causal, int out_layout, int dtype, void *ws, int64_t ws_bytes, void *stream) {
    if (dtype != MI_BF16 && dtype != MI_F16)
        return fail(MI_ERR_UNSUPPORTED, "sdpa covers bf16 and fp16 (dtype code %d)", dtype);
    if (D != 64 && D != 128) return fail(MI_ERR_UNSUPPORTED, "sdpa head dim %lld", (long long)D);
    if (B < 0 || H <= 0 || HK <= 0 || H % HK || Lq < 0 || Lk <= 0 || kv_cap < Lk)
        return fail(MI_ERR_ARG, "sdpa shape B=%lld H=%lld HK=%lld Lq=%lld Lk=%lld cap=%lld",
                    (long long)B, (long long)H, (long long)HK, (long long)Lq, (long long)Lk,
                    (long long)kv_cap);
    if (causal && Lq > Lk) return fail(MI_ERR_ARG, "causal sdpa needs Lq <= Lk");
    if (B * Lq && (!q || !k || !v || !out)) return fail(MI_ERR_ARG, "null pointer");
    if (!aligned(q, 16) || !aligned(k, 16) || !aligned(v, 16) || !aligned(out, 8))
        return fail(MI_ERR_ARG, "q/k/v must be 16-byte aligned, out 8-byte aligned");
    if (B * Lq == 0) return MI_OK;
    const int64_t need = mi_sdpa_workspace_bytes(B, H, HK, Lq, Lk, D);
    float *w = need > 0 && ws && ws_bytes >= need && aligned(ws, 16) ? (float *)ws : nullptr;
    const float sl = scale * 1.4426950408889634f;
    // (a scale of 0 as the smallest normal: masked scores stay -inf; NaN stays
    // NaN)
    const float mag = fabsf(sl) < 1.17549435e-38f ? 1.17549435e-38f : fabsf(sl);
    const AttnArgs a = {q, k, v, out, B, H, HK, Lq, Lk, kv_cap, mag,
                        sl < 0.0f ? 0x80008000u : 0u, causal, out_layout};
    hipStream_t st = as_stream(stream);
    if (dtype == MI_BF16)
        return D == 128 ? launch_attn_d<bf16, 128>(a, w, st) : launch_attn_d<bf16, 64>(a, w, st);
    return D == 128 ? launch_attn_d<f16, 128>(a, w, st) : launch_attn_d<f16, 64>(a, w, st);
}

}  // namespace
}  // namespace mi

using namespace mi;

extern "C" int64_t mi_sdpa_workspace_bytes(int64_t B, int64_t H, int64_t HK, int64_t Lq,
                                           int64_t Lk, int64_t D) {
    if (B <= 0 || H <= 0 || HK <= 0 || H % HK || Lq <= 0 || Lq > DEC_MAX_LQ || Lk <= 0 ||
        (D != 64 && D != 128))
        return 0;
    const DecSplit d = decode_split(B, H, HK, Lq, Lk);
    return d.nsplit > 1 ? d.nsplit * B * H * Lq * (D + 2) * (int64_t)sizeof(float) : 0;
}

extern "C" int mi_sdpa(const void *q, const void *k, const void *v, void *out, int64_t B,
                       int64_t H, int64_t HK, int64_t Lq, int64_t Lk, int64_t D, int64_t kv_cap,
                       float scale, int causal, int out_layout, int dtype, void *stream) {
    return run_sdpa(q, k, v, out, B, H, HK, Lq, Lk, D, kv_cap, scale, causal, out_layout, dtype,
                    nullptr, 0, stream);
}

extern "C" int mi_sdpa_ws(const void *q, const void *k, const void *v, void *out, int64_t B,
                          int64_t H, int64_t HK, int64_t Lq, int64_t Lk, int64_t D,
                          int64_t kv_cap, float scale, int causal, int out_layout, int dtype,
                          void *workspace, int64_t workspace_bytes, void *stream) {
    return run_sdpa(q, k, v, out, B, H, HK, Lq, Lk, D, kv_cap, scale, causal, out_layout, dtype,
                    workspace, workspace_bytes, stream);
}
