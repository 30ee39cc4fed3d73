// gla_prefill.hip -- batched causal prefill attention on MFMA (gfx950).
//
// Math: for every query row, flash_attn_1d_ext over [window_start, pos]
// (src/transformer/forward.rs:927-958, src/tensor/flash.rs:46-124).
//
// Tiling. A workgroup (4 waves) owns a block of query rows of one sequence
// and HPW q-heads that share one KV head; every wave owns 16*NT queries of one
// head. K/V tiles of KT=32 positions are staged in LDS once per workgroup and
// read by all waves (GQA reuse). Per wave and tile:
//   S^T[key][query] = K . Q^T      MFMA, Q^T held in VGPRs
//   online softmax per query column (log2 domain)
//   O^T[d][query]  += V^T . P^T    P^T is packed from the lane's S^T
//                                  accumulators: V's pieces hold the keys in
//                                  that order, so no value changes its lane.
#include <math.h>

#include <algorithm>
#include <type_traits>

#include "gla_internal.h"

namespace gla {

namespace {

constexpr int KT = 32;  // keys per tile
constexpr float kLog2e = 1.4426950408889634f;

typedef float floatx4 __attribute__((ext_vector_type(4)));

struct PrefillParams {
    KvLayout kv;
    PageMap pm;
    const int32_t *q_start;
    const int32_t *pos_offset;
    const float *q;
    float *out;
    int n_heads;
    int n_kv_heads;
    int group;
    int hpw;           // q-heads per workgroup
    int n_qblocks;     // grid.x
    int max_q_len;     // per-sequence query counts are clamped to it
    float q_mul;       // scale*log2(e), or scale with a soft-cap
    float softcap;     // > 0: cap * tanh(s / cap)
    int sliding_window;
};

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// max of two floats as IEEE-754 maximum (a NaN operand gives NaN): gfx950
// has v_maximum3_f32, which needs no NaN-quieting max per operand the way
// fmaxf does after a row swap or a select. Not inline asm: the compiler
// inserts the wait states an MFMA result needs before a VALU read only for
// instructions it emits itself, and these maxima read MFMA results directly.
__device__ __forceinline__ float max2f(float a, float b) { return __builtin_elementwise_maximum(a, b); }

// max / sum over the four 16-lane rows (lane ^ 16, lane ^ 32) with the gfx950
// row swaps: VALU only, no LDS round trip.
__device__ __forceinline__ float max_rows4(float x) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = max2f(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const auto c = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return max2f(__uint_as_float(c[0]), __uint_as_float(c[1]));
}
__device__ __forceinline__ float sum_rows4(float x) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    const auto c = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(c[0]) + __uint_as_float(c[1]);
}

// max / min of unsigned words over the wave, in every lane: DPP rotations within
// each 16-lane row, then the row swaps.
template <bool MAX>
__device__ __forceinline__ uint32_t wave_extreme(uint32_t x) {
    const auto pick = [](uint32_t a, uint32_t b) { return MAX ? max(a, b) : min(a, b); };
    x = pick(x, __builtin_amdgcn_update_dpp(0, x, 0x121, 0xf, 0xf, true));  // row_ror 1, 2, 4, 8
    x = pick(x, __builtin_amdgcn_update_dpp(0, x, 0x122, 0xf, 0xf, true));
    x = pick(x, __builtin_amdgcn_update_dpp(0, x, 0x124, 0xf, 0xf, true));
    x = pick(x, __builtin_amdgcn_update_dpp(0, x, 0x128, 0xf, 0xf, true));
    const auto a = __builtin_amdgcn_permlane16_swap(x, x, false, false);
    x = pick(a[0], a[1]);
    const auto c = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    return pick(c[0], c[1]);
}
__device__ __forceinline__ uint32_t umax_rows4(uint32_t x) {
    const auto a = __builtin_amdgcn_permlane16_swap(x, x, false, false);
    x = max(a[0], a[1]);
    const auto c = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    return max(c[0], c[1]);
}

// cap * tanh(x / cap) * log2(e), without the long division sequences: x / cap
// by the reciprocal of cap and one correction, 1 / (1 + t) by v_rcp_f32 and one
// Newton step (each then within an ulp).
struct SoftCap {
    float cap, inv, out;
    __device__ __forceinline__ explicit SoftCap(float c) : cap(c), inv(1.0f / c), out(c * kLog2e) {}
    __device__ __forceinline__ float operator()(float x) const {
        const float q = x * inv;
        // past 16 tanh is 1, and an infinite score has no remainder
        const float y = fabsf(q) < 16.0f ? fmaf(fmaf(-cap, q, x), inv, q) : q;
        const float t = fast_exp2(-2.0f * kLog2e * fabsf(y));
        const float d = 1.0f + t;
        float r = __builtin_amdgcn_rcpf(d);
        r = fmaf(fmaf(-d, r, 1.0f), r, r);
        return copysignf((1.0f - t) * r * out, x);
    }
};

// Soft-cap and causal/window mask of one query column of a 32-key score tile
// (sacc[mt][i]: key kbase + 16*mt + i), in place, log2 domain. The
// soft-cap is a template argument and the mask one wave-uniform branch per
// tile with selects inside: written per score, both conditions became a
// branch around every score.
template <bool CAP>
__device__ __forceinline__ void cap_and_mask(floatx4 (&s)[2], float softcap, bool interior, int kbase, int qpos,
                                             int qlo, int klo, int khi) {
    if constexpr (CAP) {
        const SoftCap f(softcap);
#pragma unroll
        for (int mt = 0; mt < 2; mt++)
#pragma unroll
            for (int i = 0; i < 4; i++) s[mt][i] = f(s[mt][i]);
    }
    if (!interior) {
        const int lo = max(qlo, klo), hi = min(qpos, khi);
#pragma unroll
        for (int mt = 0; mt < 2; mt++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int kp = kbase + mt * 16 + i;
                s[mt][i] = (kp >= lo && kp <= hi) ? s[mt][i] : -INFINITY;
            }
    }
}

__device__ __forceinline__ int window_lo(int pos, int w) {
    if (w <= 0) return 0;
    int s = pos - w + 1;
    return s > 0 ? s : 0;
}

// ---------------------------------------------------------------------------
// bf16-input variant: Q, K, V and the probabilities are rounded to bf16 and
// both products run on v_mfma_f32_16x16x32_bf16 with fp32 accumulation; the
// softmax stays fp32. Same workgroup shape, masks and online softmax as the
// fp32 kernel. K is staged row-major and V transposed (Vt[d][key]) in LDS
// as bf16, so every MFMA operand a lane needs is one 8- or 16-byte read.
//   S^T[key][q] = K . Q^T   A = K (16 keys x 32 d), B = Q^T from registers
//   O^T[d][q]  += V^T . P^T A = Vt (16 d x 32 keys), B = P^T packed from the
//                           S^T accumulators: k-slots 0..3 of lane group g
//                           are keys 4g+r of the first 16-key half and 4..7
//                           the same keys of the second half, which is what
//                           the lane's two accumulators hold.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

template <int D>
constexpr int kKRowH = D + 8;  // K row in LDS (bf16): 16 bytes of padding
constexpr int kVtRowH = KT + 8;  // Vt row in LDS (bf16): 32 keys + 16 bytes

// The 4 keys x 4 dims block of K and of V that one thread stages, as f32.
struct Block44 {
    float4 k[4];  // k[i] = K[key 4*kq + i][4*dq .. 4*dq+3]
    float4 v[4];  // v[i] = V[key 4*kq + i][4*dq .. 4*dq+3]
};

template <int D, bool Q8>
__device__ __forceinline__ void fetch_block44(const PrefillParams &p, int b, int kvh, int key0, int d0, int klo,
                                              int khi, Block44 &o) {
    const int64_t head_off = (int64_t)kvh * p.kv.head_stride;
    // key0 is a multiple of 4, so the 4 keys share one page; a block past
    // khi (zeroed below) looks up khi's page, so the page-table read stays
    // inside the sequence's row
    const int64_t pid = map_page(p.pm, b, min(key0, max(khi, 0)) >> 4);
    if constexpr (Q8) {
        const int64_t hb = pid * p.kv.page_stride + head_off;
        const int slot0 = key0 & 15;
        const int blk = d0 >> 5;
        const uint16_t *vsp = reinterpret_cast<const uint16_t *>(p.kv.vs + hb);
        const uint16_t *ksp = reinterpret_cast<const uint16_t *>(p.kv.ks + hb);
        // V: 4 consecutive slots of one d are 4 consecutive bytes (q8v_off)
        float vq[4][4];  // [d][key]
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint32_t w = *reinterpret_cast<const uint32_t *>(p.kv.v + hb + q8v_off(slot0, d0 + j, D));
#pragma unroll
            for (int i = 0; i < 4; i++) vq[j][i] = (float)((int)((w >> (8 * i)) & 0xff) - 128);
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int kp = key0 + i;
            const bool ok = kp >= klo && kp <= khi;
            // K: 4 consecutive d of one slot are 4 consecutive bytes (q8k_off)
            const uint32_t w = *reinterpret_cast<const uint32_t *>(p.kv.k + hb + q8k_off(slot0 + i, d0, D));
            const float ksc = ok ? __half2float(__ushort_as_half(ksp[q8ks_off(slot0 + i, blk, D)])) : 0.0f;
            const float vsc = ok ? __half2float(__ushort_as_half(vsp[(slot0 + i) * (D / 32) + blk])) : 0.0f;
            o.k[i] = make_float4((float)((int)(w & 0xff) - 128) * ksc, (float)((int)((w >> 8) & 0xff) - 128) * ksc,
                                 (float)((int)((w >> 16) & 0xff) - 128) * ksc,
                                 (float)((int)((w >> 24) & 0xff) - 128) * ksc);
            o.v[i] = make_float4(vq[0][i] * vsc, vq[1][i] * vsc, vq[2][i] * vsc, vq[3][i] * vsc);
        }
    } else {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int kp = key0 + i;
            if (kp >= klo && kp <= khi) {
                const int64_t base =
                    pid * p.kv.page_stride + head_off + (int64_t)((kp & 15)) * p.kv.row_stride + (int64_t)d0 * 4;
                o.k[i] = *reinterpret_cast<const float4 *>(p.kv.k + base);
                o.v[i] = *reinterpret_cast<const float4 *>(p.kv.v + base);
            } else {
                o.k[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                o.v[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            }
        }
    }
}

__device__ __forceinline__ bf16x4 to_bf16x4(float a, float b, float c, float d) {
    return bf16x4{(__bf16)a, (__bf16)b, (__bf16)c, (__bf16)d};
}

template <int D>
__device__ __forceinline__ void store_block44(const Block44 &o, int kq, int dq, __bf16 *Kh, __bf16 *Vt) {
#pragma unroll
    for (int i = 0; i < 4; i++)
        *reinterpret_cast<bf16x4 *>(Kh + (4 * kq + i) * kKRowH<D> + 4 * dq) =
            to_bf16x4(o.k[i].x, o.k[i].y, o.k[i].z, o.k[i].w);
    *reinterpret_cast<bf16x4 *>(Vt + (4 * dq + 0) * kVtRowH + 4 * kq) =
        to_bf16x4(o.v[0].x, o.v[1].x, o.v[2].x, o.v[3].x);
    *reinterpret_cast<bf16x4 *>(Vt + (4 * dq + 1) * kVtRowH + 4 * kq) =
        to_bf16x4(o.v[0].y, o.v[1].y, o.v[2].y, o.v[3].y);
    *reinterpret_cast<bf16x4 *>(Vt + (4 * dq + 2) * kVtRowH + 4 * kq) =
        to_bf16x4(o.v[0].z, o.v[1].z, o.v[2].z, o.v[3].z);
    *reinterpret_cast<bf16x4 *>(Vt + (4 * dq + 3) * kVtRowH + 4 * kq) =
        to_bf16x4(o.v[0].w, o.v[1].w, o.v[2].w, o.v[3].w);
}

template <int D, int NTHR>
struct TileBlocks {
    static constexpr int UNITS = (KT / 4) * (D / 4);
    static constexpr int PER_THREAD = (UNITS + NTHR - 1) / NTHR;
    Block44 blk[PER_THREAD];
};

template <int D, int NTHR, bool Q8>
__device__ __forceinline__ void fetch_tile_bf16(const PrefillParams &p, int b, int kvh, int k0, int klo, int khi,
                                                TileBlocks<D, NTHR> &t) {
#pragma unroll
    for (int j = 0; j < TileBlocks<D, NTHR>::PER_THREAD; j++) {
        const int u = threadIdx.x + j * NTHR;
        if (u >= TileBlocks<D, NTHR>::UNITS) break;
        const int kq = u / (D / 4);
        const int dq = u - kq * (D / 4);
        fetch_block44<D, Q8>(p, b, kvh, k0 + 4 * kq, 4 * dq, klo, khi, t.blk[j]);
    }
}

template <int D, int NTHR>
__device__ __forceinline__ void store_tile_bf16(const TileBlocks<D, NTHR> &t, __bf16 *Kh, __bf16 *Vt) {
#pragma unroll
    for (int j = 0; j < TileBlocks<D, NTHR>::PER_THREAD; j++) {
        const int u = threadIdx.x + j * NTHR;
        if (u >= TileBlocks<D, NTHR>::UNITS) break;
        const int kq = u / (D / 4);
        const int dq = u - kq * (D / 4);
        store_block44<D>(t.blk[j], kq, dq, Kh, Vt);
    }
}

// Waves per workgroup of the bf16 kernel (32 queries each): 8 share each
// staged K/V tile (d = 256: 4, whose registers need the 512-VGPR budget of
// one wave per SIMD).
template <int D>
constexpr int kBf16Waves = D == 256 ? 4 : 8;

// bf16 softmax: how far (log2 units) a score may pass the row's running
// maximum before the maximum, and with it O, is rescaled.
constexpr float kLazyMax = 8.0f;
// The bf16 kernels' reference maximum before a query's first attended key:
// finite, so the first attended tile is an ordinary move of the reference
// (its factor 2^(-1e30 - max) = 0 scales the still-zero O and sums) and the
// per-tile logic needs no "no key yet" case; a masked score (-inf) still
// gives p = 0, and a query that attends no key keeps l = 0 (output 0).
constexpr float kMInit = -1e30f;

// S^T accumulators of a tile before S = K.Q^T: zero (the first MFMA takes an
// inline 0), so the scores arrive absolute and p = 2^(s - m) takes one
// subtraction per score.
template <int NT>
__device__ __forceinline__ void bf16_score_init(floatx4 (&sacc)[2][NT]) {
#pragma unroll
    for (int nt = 0; nt < NT; nt++)
#pragma unroll
        for (int mt = 0; mt < 2; mt++) sacc[mt][nt] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
}

// max of three floats as one v_maximum3_f32 (as max2f)
__device__ __forceinline__ float max3f(float a, float b, float c) { return max2f(max2f(a, b), c); }

// Online softmax of one 32-key tile of the bf16 kernels (both share it):
// soft-cap and (MASK) the causal/window mask, the lazy maximum (the reference
// moves only when a score passes it by more than 8 log2 units, so p stays at
// most 256, exact range for bf16 and f32, and the rescale of O is rare), p =
// 2^(s - m) rounded to bf16 for both MFMAs, and the factor rs[nt] that O and
// the row sums take before this tile is added (bf16_rescale). Each lane first
// takes the maximum of its own 8 scores of a query; only when one of them
// passes its reference by more than the margin (in some lane of the wave: a
// wave-uniform branch) does the tile take the row maxima across the query's
// 4 lanes. A row whose maximum passes has that maximum in one of its lanes,
// so the rare path makes the decisions that taking every row maximum would.
template <int NT, bool CAP, bool MASK>
__device__ __forceinline__ void bf16_softmax_p(const floatx4 (&sacc)[2][NT], float (&m)[NT], float (&rs)[NT],
                                               bf16x8 (&pb)[NT], float softcap, int kbase, const int (&qpos)[NT],
                                               const int (&qlo)[NT], int klo, int khi) {
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
        floatx4 col[2] = {sacc[0][nt], sacc[1][nt]};
        cap_and_mask<CAP>(col, softcap, !MASK, kbase, qpos[nt], qlo[nt], klo, khi);
        float mx = max3f(max3f(col[0][0], col[0][1], col[0][2]), max3f(col[0][3], col[1][0], col[1][1]),
                         max2f(col[1][2], col[1][3]));
        const float m_old = m[nt];
        rs[nt] = 1.0f;
        if (__ballot(mx - m_old > kLazyMax)) {
            mx = max_rows4(mx);
            // (selects: the conditions differ from lane to lane)
            const bool up = mx - m_old > kLazyMax;
            m[nt] = up ? mx : m_old;
            rs[nt] = up ? fast_exp2(m_old - mx) : 1.0f;
        }
        float pr[2][4];
#pragma unroll
        for (int mt = 0; mt < 2; mt++)
#pragma unroll
            for (int i = 0; i < 4; i++) pr[mt][i] = fast_exp2(col[mt][i] - m[nt]);
        pb[nt] = bf16x8{(__bf16)pr[0][0], (__bf16)pr[0][1], (__bf16)pr[0][2], (__bf16)pr[0][3],
                        (__bf16)pr[1][0], (__bf16)pr[1][1], (__bf16)pr[1][2], (__bf16)pr[1][3]};
    }
}

// O and the row sums take the factor of a moved reference (rare: a wave-uniform
// branch per query tile).
template <int NT, int DT>
__device__ __forceinline__ void bf16_rescale(const float (&rs)[NT], floatx4 (&lacc)[NT], floatx4 (&o)[DT][NT]) {
#pragma unroll
    for (int nt = 0; nt < NT; nt++)
        if (__ballot(rs[nt] != 1.0f)) {
#pragma unroll
            for (int t = 0; t < DT; t++) o[t][nt] *= rs[nt];
            lacc[nt] *= rs[nt];
        }
}

// The softmax of a tile inside every query's causal and window bounds, both
// query tiles decided by one wave-uniform branch: the row maxima are taken,
// and references moved, only when some lane's own maximum passes its
// reference by more than the margin; for a query tile none of whose lanes
// passes, the rare path moves nothing and scales nothing, so the decisions
// are bf16_softmax_p's.
template <int NT, int DT, bool CAP>
__device__ __forceinline__ void bf16_softmax_interior(floatx4 (&sacc)[2][NT], float (&m)[NT],
                                                      floatx4 (&lacc)[NT], floatx4 (&o)[DT][NT],
                                                      bf16x8 (&pb)[NT], float softcap) {
    float mx[NT];
    bool pass = false;
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
        if constexpr (CAP) {
            floatx4 col[2] = {sacc[0][nt], sacc[1][nt]};
            cap_and_mask<CAP>(col, softcap, true, 0, 0, 0, 0, 0);
            sacc[0][nt] = col[0];
            sacc[1][nt] = col[1];
        }
        mx[nt] = max3f(max3f(sacc[0][nt][0], sacc[0][nt][1], sacc[0][nt][2]),
                       max3f(sacc[0][nt][3], sacc[1][nt][0], sacc[1][nt][1]), max2f(sacc[1][nt][2], sacc[1][nt][3]));
        pass = pass || mx[nt] - m[nt] > kLazyMax;
    }
    if (__ballot(pass)) {
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
            const float mr = max_rows4(mx[nt]);
            // (selects: the conditions differ from lane to lane)
            const float m_old = m[nt];
            const bool up = mr - m_old > kLazyMax;
            m[nt] = up ? mr : m_old;
            const float rs = up ? fast_exp2(m_old - mr) : 1.0f;
            if (__ballot(rs != 1.0f)) {
#pragma unroll
                for (int t = 0; t < DT; t++) o[t][nt] *= rs;
                lacc[nt] *= rs;
            }
        }
    }
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
        float pr[2][4];
#pragma unroll
        for (int mt = 0; mt < 2; mt++)
#pragma unroll
            for (int i = 0; i < 4; i++) pr[mt][i] = fast_exp2(sacc[mt][nt][i] - m[nt]);
        pb[nt] = bf16x8{(__bf16)pr[0][0], (__bf16)pr[0][1], (__bf16)pr[0][2], (__bf16)pr[0][3],
                        (__bf16)pr[1][0], (__bf16)pr[1][1], (__bf16)pr[1][2], (__bf16)pr[1][3]};
    }
}

// The whole softmax of a tile whose mask need is known at run time.
template <int NT, int DT, bool CAP>
__device__ __forceinline__ void bf16_softmax(floatx4 (&sacc)[2][NT], float (&m)[NT],
                                             floatx4 (&lacc)[NT], floatx4 (&o)[DT][NT], bf16x8 (&pb)[NT],
                                             float softcap, bool interior, int kbase, const int (&qpos)[NT],
                                             const int (&qlo)[NT], int klo, int khi) {
    float rs[NT];
    if (interior)
        bf16_softmax_p<NT, CAP, false>(sacc, m, rs, pb, softcap, kbase, qpos, qlo, klo, khi);
    else
        bf16_softmax_p<NT, CAP, true>(sacc, m, rs, pb, softcap, kbase, qpos, qlo, klo, khi);
    bf16_rescale<NT, DT>(rs, lacc, o);
}

// Row sums of the tile's bf16 probabilities, from one MFMA against an
// all-ones operand: every element of a lane accumulates its query's sum.
template <int NT>
__device__ __forceinline__ void bf16_row_sums(floatx4 (&lacc)[NT], const bf16x8 (&pb)[NT]) {
    const bf16x8 ones = bf16x8{(__bf16)1.0f, (__bf16)1.0f, (__bf16)1.0f, (__bf16)1.0f,
                               (__bf16)1.0f, (__bf16)1.0f, (__bf16)1.0f, (__bf16)1.0f};
#pragma unroll
    for (int nt = 0; nt < NT; nt++) lacc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, pb[nt], lacc[nt], 0, 0, 0);
}

template <int D, bool Q8, bool CAP>
__global__ __launch_bounds__(kBf16Waves<D> * 64) void prefill_bf16_kernel(const PrefillParams p) {
    constexpr int NW = kBf16Waves<D>, NT = 2, NTHR = NW * 64;
    constexpr int QW = 16 * NT;
    constexpr int KS = D / 32;  // k-steps of S (32 dims each)
    constexpr int DT = D / 16;  // d tiles of O
    __shared__ __attribute__((aligned(16))) __bf16 Kh[2][KT * kKRowH<D>];
    __shared__ __attribute__((aligned(16))) __bf16 Vt[2][D * kVtRowH];

    // grid (sequence x KV head x head group, query block): every unit's
    // longest (last) query block is dispatched before any shorter one, so the
    // grid ends on short workgroups
    const int n_hgrp = p.group / p.hpw;
    const int unit = blockIdx.x;
    const int b = unit / (p.n_kv_heads * n_hgrp);
    const int kvh = (unit - b * p.n_kv_heads * n_hgrp) / n_hgrp;
    const int hgrp = unit - (b * p.n_kv_heads + kvh) * n_hgrp;
    const int qblk = p.n_qblocks - 1 - (int)blockIdx.y;
    const int waves_per_head = NW / p.hpw;
    const int qwg = QW * waves_per_head;

    const int row0 = p.q_start[b];
    const int q_len = min(max(p.q_start[b + 1] - row0, 0), p.max_q_len);
    const int pos0 = p.pos_offset[b];
    const int qb0 = qblk * qwg;
    if (qb0 >= q_len) return;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int lrow = lane & 15;
    const int lgrp = lane >> 4;
    const int head = kvh * p.group + hgrp * p.hpw + (wave % p.hpw);
    const int wq0 = qb0 + (wave / p.hpw) * QW;

    const int q_last = min(q_len, qb0 + qwg) - 1;
    const int khi = min(pos0 + q_last, p.pm.pos_limit - 1);
    const int klo = window_lo(pos0 + qb0, p.sliding_window);

    // Q^T operand: qb[nt][ks] = Q[query nt*16 + lrow][d = ks*32 + lgrp*8 + 0..7] as bf16
    bf16x8 qb[NT][KS];
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
        const int lq = wq0 + nt * 16 + lrow;
        const bool ok = lq < q_len;
        const float *qp = p.q + ((int64_t)(row0 + (ok ? lq : 0)) * p.n_heads + head) * D;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const float4 a = *reinterpret_cast<const float4 *>(qp + ks * 32 + lgrp * 8);
            const float4 c = *reinterpret_cast<const float4 *>(qp + ks * 32 + lgrp * 8 + 4);
            const float mul = ok ? p.q_mul : 0.0f;
            qb[nt][ks] = bf16x8{(__bf16)(a.x * mul), (__bf16)(a.y * mul), (__bf16)(a.z * mul), (__bf16)(a.w * mul),
                                (__bf16)(c.x * mul), (__bf16)(c.y * mul), (__bf16)(c.z * mul), (__bf16)(c.w * mul)};
        }
    }

    floatx4 o[DT][NT];
    floatx4 lacc[NT];
    float m[NT];  // the query's reference maximum (log2 domain)
    int qpos[NT], qlo[NT];
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
#pragma unroll
        for (int t = 0; t < DT; t++) o[t][nt] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
        lacc[nt] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
        m[nt] = kMInit;
        const int lq = wq0 + nt * 16 + lrow;
        qpos[nt] = lq < q_len ? pos0 + lq : -1;
        qlo[nt] = window_lo(pos0 + lq, p.sliding_window);
    }
    // keys this wave's queries attend: [wlo, whi]
    const int whi = min(khi, pos0 + wq0 + QW - 1);
    const int wlo = max(klo, window_lo(pos0 + wq0, p.sliding_window));

    if (khi >= klo) {
        const int kfirst = (klo / KT) * KT;
        TileBlocks<D, NTHR> tb;
        fetch_tile_bf16<D, NTHR, Q8>(p, b, kvh, kfirst, klo, khi, tb);
        store_tile_bf16<D, NTHR>(tb, Kh[0], Vt[0]);
        __syncthreads();
        int buf = 0;
        for (int k0 = kfirst; k0 <= khi; k0 += KT, buf ^= 1) {
            const bool more = k0 + KT <= khi;
            if (more) fetch_tile_bf16<D, NTHR, Q8>(p, b, kvh, k0 + KT, klo, khi, tb);
            const __bf16 *kh = Kh[buf];
            const __bf16 *vt = Vt[buf];
            // a tile wholly past this wave's last query or before its window adds nothing
            if (k0 <= whi && k0 + KT - 1 >= wlo) {
            // S^T = K . Q^T
            floatx4 sacc[2][NT];
            bf16_score_init<NT>(sacc);
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {
                bf16x8 a[2];
#pragma unroll
                for (int mt = 0; mt < 2; mt++)
                    a[mt] = *reinterpret_cast<const bf16x8 *>(kh + (mt * 16 + lrow) * kKRowH<D> + ks * 32 + lgrp * 8);
#pragma unroll
                for (int mt = 0; mt < 2; mt++)
#pragma unroll
                    for (int nt = 0; nt < NT; nt++)
                        sacc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[mt], qb[nt][ks], sacc[mt][nt], 0, 0, 0);
            }

            const bool interior = k0 >= klo && k0 + KT - 1 <= min(khi, pos0 + wq0) &&
                                  (p.sliding_window <= 0 || k0 >= window_lo(pos0 + wq0 + QW - 1, p.sliding_window));
            bf16x8 pb[NT];
            bf16_softmax<NT, DT, CAP>(sacc, m, lacc, o, pb, p.softcap, interior, k0 + 4 * lgrp, qpos, qlo, klo,
                                      khi);

            // O^T += V^T . P^T, and the row sums
            bf16_row_sums<NT>(lacc, pb);
#pragma unroll
            for (int t = 0; t < DT; t++) {
                const __bf16 *vr = vt + (16 * t + lrow) * kVtRowH;
                const bf16x4 lo = *reinterpret_cast<const bf16x4 *>(vr + 4 * lgrp);
                const bf16x4 hi = *reinterpret_cast<const bf16x4 *>(vr + 16 + 4 * lgrp);
                const bf16x8 a = bf16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
#pragma unroll
                for (int nt = 0; nt < NT; nt++)
                    o[t][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, pb[nt], o[t][nt], 0, 0, 0);
            }
            }

            if (more) store_tile_bf16<D, NTHR>(tb, Kh[buf ^ 1], Vt[buf ^ 1]);
            __syncthreads();
        }
    }

    // normalise and store: lane holds O^T[d = 16t + 4*lgrp + r][query lrow]
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
        const float lt = lacc[nt][0];
        const int lq = wq0 + nt * 16 + lrow;
        if (lq >= q_len) continue;
        const float inv = lt > 0.0f ? 1.0f / lt : 0.0f;
        float *op = p.out + ((int64_t)(row0 + lq) * p.n_heads + head) * D;
#pragma unroll
        for (int t = 0; t < DT; t++) {
            const floatx4 v = o[t][nt] * inv;
            *reinterpret_cast<float4 *>(op + 16 * t + 4 * lgrp) = make_float4(v[0], v[1], v[2], v[3]);
        }
    }
}

// ---------------------------------------------------------------------------
// Staged bf16 path: a pre-pass converts each (sequence, KV head, 32-key tile)
// the prefill reads to bf16 once, in the exact LDS image the MFMA operand
// reads want, and the main kernel copies tile images into an LDS ring with
// direct global->LDS loads (no registers, no conversion, kRingTiles - 1 tiles
// ahead).
// The image of a tile is 128*D bytes, 16-byte pieces:
//   K: piece ((mt*(D/8) + c)*16 + r) = K[key mt*16 + r][dims 8c .. 8c+7]
//   V: piece ((t*4 + g)*16 + r)      = V[keys 4g..4g+3, 16+4g..16+4g+3][dim 16t + r]
// so the 16 lanes of each read pass (r = 0..15) take 16 consecutive pieces
// of one 256-byte line: no LDS bank conflicts, and the whole image is one
// contiguous copy. Keys outside the sequence's window union [window_lo(pos0),
// last query] are zero, as the in-kernel staging zeroes them.
// Tile images in a workgroup's ring: three (48 KB at d = 128) lets three
// workgroups share a CU, so one's prologue, epilogue and barrier waits meet
// the others' matrix work; d = 256 keeps four (one workgroup per CU).
template <int D>
constexpr int kRingTiles = D == 256 ? 4 : 3;

template <int D>
constexpr int kTileImage = 128 * D;

// Waves per workgroup of the staged kernel (32 queries each): one per SIMD;
// a CU holds several workgroups.
template <int D>
constexpr int kBf16sWaves = 4;
// Kilobyte copies per wave of the staged kernel's tile ring (every wave copies).
template <int D>
constexpr int kCopiesPerWave = D == 64 ? 2 : (D == 128 ? 4 : 8);
// Waves per SIMD the staged kernel's registers are sized for: d = 64: 4
// (<= 128 VGPRs), d = 128: 3 (<= 168; the soft-capped variant spills one
// register), d = 256: 1.
template <int D>
constexpr int kBf16sOccupancy = D == 64 ? 4 : (D == 128 ? 3 : 1);

template <int D, bool CAP, int NT>
__global__ __launch_bounds__(kBf16sWaves<D> * 64, kBf16sOccupancy<D>) void prefill_bf16s_kernel(const PrefillParams p,
                                                                          const uint8_t *img, int n_tiles) {
    constexpr int NW = kBf16sWaves<D>;
    constexpr int QW = 16 * NT;
    constexpr int KS = D / 32;
    constexpr int DT = D / 16;
    constexpr int NC = kTileImage<D> / 1024;  // 1 KB copies per tile, dealt to the waves in turn
    constexpr int RT = kRingTiles<D>;
    __shared__ __attribute__((aligned(16))) uint8_t ring[RT][kTileImage<D>];

    const int n_hgrp = p.group / p.hpw;
    const int unit = blockIdx.x;
    const int b = unit / (p.n_kv_heads * n_hgrp);
    const int kvh = (unit - b * p.n_kv_heads * n_hgrp) / n_hgrp;
    const int hgrp = unit - (b * p.n_kv_heads + kvh) * n_hgrp;
    const int qblk = p.n_qblocks - 1 - (int)blockIdx.y;
    const int waves_per_head = NW / p.hpw;
    const int qwg = QW * waves_per_head;

    const int row0 = p.q_start[b];
    const int q_len = min(max(p.q_start[b + 1] - row0, 0), p.max_q_len);
    const int pos0 = p.pos_offset[b];
    const int qb0 = qblk * qwg;
    if (qb0 >= q_len) return;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lrow = lane & 15;
    const int lgrp = lane >> 4;
    const int head = kvh * p.group + hgrp * p.hpw + (wave % p.hpw);
    const int wq0 = qb0 + (wave / p.hpw) * QW;

    // The keys are those of whole blocks of 32 rows, also where a wave takes 16:
    // 0 times an infinity or a NaN of V is not 0, so which masked keys a row's tiles
    // hold must not depend on NT
    const int q_last = min(q_len, (qb0 + qwg + 31) & ~31) - 1;
    const int khi = min(pos0 + q_last, p.pm.pos_limit - 1);
    const int klo = window_lo(pos0 + (qb0 & ~31), p.sliding_window);

    bf16x8 qb[NT][KS];
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
        const int lq = wq0 + nt * 16 + lrow;
        const bool ok = lq < q_len;
        const float *qp = p.q + ((int64_t)(row0 + (ok ? lq : 0)) * p.n_heads + head) * D;
        // q rows are read once per call and the output rows written once:
        // non-temporal accesses (measured: the f32 output stream otherwise
        // slows the q reads of the workgroups starting beside it)
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const floatx4 a = __builtin_nontemporal_load(reinterpret_cast<const floatx4 *>(qp + ks * 32 + lgrp * 8));
            const floatx4 c = __builtin_nontemporal_load(reinterpret_cast<const floatx4 *>(qp + ks * 32 + lgrp * 8 + 4));
            const float mul = ok ? p.q_mul : 0.0f;
            qb[nt][ks] = bf16x8{(__bf16)(a.x * mul), (__bf16)(a.y * mul), (__bf16)(a.z * mul), (__bf16)(a.w * mul),
                                (__bf16)(c.x * mul), (__bf16)(c.y * mul), (__bf16)(c.z * mul), (__bf16)(c.w * mul)};
        }
    }

    floatx4 o[DT][NT];
    floatx4 lacc[NT];
    float m[NT];
    int qpos[NT], qlo[NT];
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
#pragma unroll
        for (int t = 0; t < DT; t++) o[t][nt] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
        lacc[nt] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
        m[nt] = kMInit;
        const int lq = wq0 + nt * 16 + lrow;
        qpos[nt] = lq < q_len ? pos0 + lq : -1;
        qlo[nt] = window_lo(pos0 + lq, p.sliding_window);
    }
    // keys that the wave's block of 32 rows attends: [wlo, whi]
    const int whi = min(khi, pos0 + (wq0 | 31));
    const int wlo = max(klo, window_lo(pos0 + (wq0 & ~31), p.sliding_window));

    if (khi >= klo) {
        const int tfirst = klo / KT;
        const int n = khi / KT - tfirst + 1;
        const uint8_t *unit_img = img + ((int64_t)b * p.n_kv_heads + kvh) * n_tiles * kTileImage<D>;
        const uint32_t ring_lds = __builtin_amdgcn_readfirstlane(
            (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void *)&ring[0][0]);
        // A tile's NC kilobyte copies go to the first NC / CPW waves, CPW each,
        // so every wave that copies has the same count in flight and one
        // wait count (chosen by the tiles left) serves every wave.
        constexpr int CPW = kCopiesPerWave<D>;
        static_assert(NC % CPW == 0 && NC / CPW <= NW, "copies cover the tile");
        auto issue = [&](int i) {
            if (wave < NC / CPW) {
                const uint8_t *src = unit_img + (int64_t)(tfirst + i) * kTileImage<D>;
                const uint32_t dst = ring_lds + (uint32_t)((i % RT) * kTileImage<D>);
#pragma unroll
                for (int c = 0; c < CPW; c++) {
                    const int piece = wave * CPW + c;
                    lds_copy16(src, (uint32_t)(piece * 1024 + lane * 16), dst + piece * 1024);
                }
            }
        };
#pragma unroll
        for (int i = 0; i < RT - 1; i++)
            if (i < n) issue(i);
        static_assert(RT == 3 || RT == 4, "the waits below assume one or two tiles in flight behind the current one");
        // this wave's copies of tile i have landed (later tiles may be in
        // flight), and every wave's have; every wave is also done with tile
        // i - 1, whose buffer the next copy reuses
        auto arrive = [&](int i) {
            const int ahead = n - 1 - i;
            if (RT == 4 && ahead >= 2)
                wait_vm<(RT - 2) * CPW>();
            else if (ahead >= 1)
                wait_vm<CPW>();
            else
                wait_vm<0>();
            __syncthreads();
            if (i + RT - 1 < n) issue(i + RT - 1);
        };
        // S^T = K . Q^T of tile i
        auto scores = [&](const uint8_t *kimg, floatx4 (&sacc)[2][NT]) {
            bf16_score_init<NT>(sacc);
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {
                bf16x8 a[2];
#pragma unroll
                for (int mt = 0; mt < 2; mt++)
                    a[mt] = *reinterpret_cast<const bf16x8 *>(kimg + ((mt * (D / 8) + ks * 4 + lgrp) * 16 + lrow) * 16);
#pragma unroll
                for (int mt = 0; mt < 2; mt++)
#pragma unroll
                    for (int nt = 0; nt < NT; nt++)
                        sacc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[mt], qb[nt][ks], sacc[mt][nt], 0, 0, 0);
            }
        };
        // O^T += V^T . P^T, and the row sums
        auto accumulate = [&](const uint8_t *vimg, const bf16x8 (&pb)[NT]) {
            bf16_row_sums<NT>(lacc, pb);
#pragma unroll
            for (int t = 0; t < DT; t++) {
                const bf16x8 a = *reinterpret_cast<const bf16x8 *>(vimg + ((t * 4 + lgrp) * 16 + lrow) * 16);
#pragma unroll
                for (int nt = 0; nt < NT; nt++)
                    o[t][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, pb[nt], o[t][nt], 0, 0, 0);
            }
        };
        // The leading tiles inside the causal and window bounds of every query
        // of the workgroup, when its waves share one query block (one q-head
        // each): no mask, no skip test and one lazy-maximum branch per tile.
        int n_int = 0;
        if (p.hpw == NW) {
            const int k_first = tfirst * KT;
            const bool lead = k_first >= klo &&
                              (p.sliding_window <= 0 || k_first >= window_lo(pos0 + wq0 + QW - 1, p.sliding_window));
            if (lead) n_int = max(0, min(n, (min(khi, pos0 + wq0) + 1) / KT - tfirst));
        }
        int i = 0;
        for (; i < n_int; i++) {
            arrive(i);
            const uint8_t *kimg = ring[i % RT];
            floatx4 sacc[2][NT];
            scores(kimg, sacc);
            bf16x8 pb[NT];
            bf16_softmax_interior<NT, DT, CAP>(sacc, m, lacc, o, pb, p.softcap);
            accumulate(kimg + 64 * D, pb);
        }
        for (; i < n; i++) {
            arrive(i);
            const int k0 = (tfirst + i) * KT;
            // a tile wholly past this wave's last query (the causal diagonal of
            // the workgroup's later waves) or before its window adds nothing
            if (k0 > whi || k0 + KT - 1 < wlo) continue;
            const uint8_t *kimg = ring[i % RT];
            floatx4 sacc[2][NT];
            scores(kimg, sacc);
            const bool interior = k0 >= klo && k0 + KT - 1 <= min(khi, pos0 + wq0) &&
                                  (p.sliding_window <= 0 || k0 >= window_lo(pos0 + wq0 + QW - 1, p.sliding_window));
            bf16x8 pb[NT];
            bf16_softmax<NT, DT, CAP>(sacc, m, lacc, o, pb, p.softcap, interior, k0 + 4 * lgrp, qpos, qlo, klo,
                                      khi);
            accumulate(kimg + 64 * D, pb);
        }
    }

    // Output rows through LDS (the ring is free once every wave is done with
    // it): a lane holds 4 dims of one query, so direct stores would write
    // half lines; read back row-major, each store instruction writes whole
    // D-float rows. Each wave stages its 16 queries of one nt at a time in
    // its own region (rows padded by 4 floats against bank conflicts); a
    // wave's LDS operations run in order, so it needs no barrier of its own.
    constexpr int SROW = D + 4;
    static_assert(NW * 16 * SROW * 4 <= kRingTiles<D> * kTileImage<D>, "output staging fits the ring");
    __syncthreads();
    float *stage = reinterpret_cast<float *>(&ring[0][0]) + wave * 16 * SROW;
    constexpr int LPR = D / 4;    // lanes per row (16 bytes each)
    constexpr int RPI = 64 / LPR;  // rows per store instruction
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
        const float lt = lacc[nt][0];
        const float inv = lt > 0.0f ? 1.0f / lt : 0.0f;
#pragma unroll
        for (int t = 0; t < DT; t++)
            *reinterpret_cast<floatx4 *>(stage + lrow * SROW + 16 * t + 4 * lgrp) = o[t][nt] * inv;
#pragma unroll
        for (int k = 0; k < 16 / RPI; k++) {
            const int r = k * RPI + lane / LPR;
            const int c = (lane % LPR) * 4;
            const floatx4 v = *reinterpret_cast<const floatx4 *>(stage + r * SROW + c);
            const int lq = wq0 + nt * 16 + r;
            if (lq < q_len)
                __builtin_nontemporal_store(v, reinterpret_cast<floatx4 *>(p.out + ((int64_t)(row0 + lq) * p.n_heads + head) * D + c));
        }
    }
}

// ---------------------------------------------------------------------------
// fp32 prefill on the f16 matrix cores. Every f32 operand is two f16 pieces
// after a power-of-two scaling, hi = f16(x) and lo = f16((x - hi) * 2^11): 22
// bits of x wherever hi is a normal f16, which is 29 binades below 2^15. A
// product is three MFMAs, hi.hi and, 2^-11 below, hi.lo + lo.hi; the dropped
// lo.lo is 2^-24 of it. Products of f16 pieces are exact in the f32
// accumulators, and a 32-wide MFMA rounds once where the 4-wide f32 one rounds
// eight times, so the error against 64 bits is smaller: 4 prompts of 2,048 at
// 32/8 heads, d = 128, 2.0e-7 relative (f32 MFMAs: 4.4e-7). Three f16 MFMAs do
// the work of a 16x16x32 tile in 48 cycles, the f32 ones in 256: the same four
// prompts take 400 us, of them 23 the staging (f32 MFMAs: 1,083 us). What bounds
// it is the chain S -> softmax -> O at two waves per SIMD: matrix and vector
// cycles add up.
//
// Scaling. A row's result follows from the row and the keys it attends alone,
// bit for bit, whatever rows, chunks and sequences share its call: every scale
// belongs to one key or to one row. A key's K and V each take a power of two
// from their own largest value, one for eight binades (kClass), and a query row
// one from its own. K's and the query's are undone on the scores. V's is carried
// by the probability: O accumulates p * 2^(E - R) times the scaled V, E the key's
// exponent and R the row's: the largest E it has attended, moved (with O) when
// one passes it by more than 2^2. So the products' operand is largest where the
// contribution p * V is, and it is the small contributions that reach the end of
// f16's range. Tiles whose keys share the exponents of the first that has the same
// for all and hold nothing odd, as with most data, are taken by a loop that holds
// the scales as constants; the others key by key. Both give the same bits.
//
// What the pieces cannot hold is named per key ("odd"): infinities and NaN, K
// with a run of 8 dims below 2^-20 of its largest value, V's values below kSmall
// (scaled). The scores of an odd key, or of a query row that is odd in the same
// way, come from the f32 MFMA. Odd V values are zero in the image; the small
// ones' products are added by the f32 MFMA, the others' for the rows that attend
// them. us per call of 4 x 2,048 rows, 32/8 heads, d = 128: 400 where nothing
// differs, 410 with a NaN in V, 430 with a small value, 500 where every tile's keys differ, 1,400 with every
// 16th dim of V at 2^-34 of the others, 2,200 with eight dims of every key at 2^-30
// (f32 MFMAs for everything: 1,080).
typedef _Float16 half8p __attribute__((ext_vector_type(8)));

// instruction groups for the scheduler: MFMAs, LDS reads
constexpr int kSchedMfma = 0x8, kSchedLds = 0x100;
constexpr float kMLowest = -3.402823466e38f;  // a row's maximum before its first key
constexpr float kLazyF32 = 4.0f;  // the lazy maximum's margin: p = 2^(s - m) stays below 2^4, whatever m's ulp
constexpr int kLazyExp = 2;       // R's: p * 2^(E - R) stays below 2^6
constexpr int kScaleP = 9;        // and in f16 below 2^15
constexpr int kTop = 15;          // scaled K, V and q stay below 2^15
constexpr int kNoExp = -300;      // R before a row's first key
constexpr float kSmall = 0x1p-16f;  // scaled V values below it are odd

// A tile's image: K hi, K lo, V hi, V lo, each 64*D bytes in the piece order
// of the bf16 image.
template <int D>
constexpr int kSplitImage = 256 * D;
// What the attention needs to know of a tile.
struct TileHead {
    int32_t exps;           // the keys' exponents (key_exps); kMixed: they differ
    uint32_t odd_k;         // odd keys, a bit each: of K,
    uint32_t bad_v, small_v;  // of V by an infinity or a NaN, by a small value
};
struct TileMeta {
    TileHead head;
    int32_t exps[KT];  // by key, where it is in range
    uint32_t pad[28];  // 256 bytes: four for each lane of a wave
};
static_assert(sizeof(TileMeta) == 256, "one 4-byte copy per lane");
constexpr int32_t kMixed = -1;
// The exponents of a key's K and V in one number.
__device__ __forceinline__ int32_t key_exps(int k, int v) { return (k + 1024) << 12 | (v + 1024); }
__device__ __forceinline__ int k_exp_of(int32_t exps) { return (exps >> 12) - 1024; }
__device__ __forceinline__ int v_exp_of(int32_t exps) { return (exps & 0xfff) - 1024; }

// The pieces of 8 values times mul.
__device__ __forceinline__ void split8(const float (&x)[8], float mul, half8p &hi, half8p &lo) {
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const float t = x[j] * mul;
        const _Float16 h = (_Float16)t;
        hi[j] = h;
        lo[j] = (_Float16)fmaf((float)h, -2048.0f, t * 2048.0f);
    }
}

// The exponent e of a positive value m, from its bits: m is in [2^(e-1), 2^e). At
// least -100 (smaller values keep fewer bits).
__device__ __forceinline__ int exponent_of(uint32_t bits) { return max((int)(bits >> 23) - 126, -100); }
// A key's: e rounded up to 5 more than a multiple of 8, so that the largest
// values of [1/8, 32) share one. (A key of zeros has that of 1.)
constexpr int kClass = 8;
__device__ __forceinline__ int class_of(uint32_t bits) {
    return bits ? (exponent_of(bits) + kClass * 16 - 6 + kClass) / kClass * kClass - kClass * 16 + 5 : 5;
}
__device__ __forceinline__ float pow2f(int e) { return __uint_as_float((uint32_t)(e + 127) << 23); }

// max of |x| over 8 values, as bits (an infinity or a NaN is the largest)
__device__ __forceinline__ uint32_t top_bits(const float (&x)[8]) {
    uint32_t t = 0;
#pragma unroll
    for (int j = 0; j < 8; j++) t = max(t, __float_as_uint(x[j]) & 0x7fffffffu);
    return t;
}
constexpr uint32_t kInfBits = 0x7f800000u;
// Whether a run of 8 values, the largest `run`, is too small beside `top`.
__device__ __forceinline__ bool run_is_odd(uint32_t run, uint32_t top) { return run != 0 && run + (20u << 23) < top; }

// max over the lanes that share lane % N (N = 2, 4 or 8)
template <int N>
__device__ __forceinline__ uint32_t umax_stride(uint32_t x) {
    if constexpr (N <= 2) x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, x, 0x122, 0xf, 0xf, true));  // row_ror 2, 4, 8
    if constexpr (N <= 4) x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, x, 0x124, 0xf, 0xf, true));
    x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, x, 0x128, 0xf, 0xf, true));
    return umax_rows4(x);
}
// max over N neighbouring lanes (N = 8, 16 or 32)
template <int N>
__device__ __forceinline__ uint32_t umax_group(uint32_t x) {
    x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, x, 0xB1, 0xf, 0xf, true));   // quad_perm [1 0 3 2]
    x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, x, 0x4E, 0xf, 0xf, true));   // quad_perm [2 3 0 1]
    x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, x, 0x141, 0xf, 0xf, true));  // row_half_mirror
    if constexpr (N >= 16) x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, x, 0x128, 0xf, 0xf, true));  // row_ror 8
    if constexpr (N >= 32) {
        const auto a = __builtin_amdgcn_permlane16_swap(x, x, false, false);
        x = max(a[0], a[1]);
    }
    return x;
}

// Four values of a cached K row from d on (page and head offset in hb).
template <int D, bool Q8>
__device__ __forceinline__ floatx4 k_values4(const PrefillParams &p, int64_t hb, int slot, int d) {
    if constexpr (Q8) {
        const uint16_t sc = reinterpret_cast<const uint16_t *>(p.kv.ks + hb)[q8ks_off(slot, d >> 5, D)];
        const uint32_t w = *reinterpret_cast<const uint32_t *>(p.kv.k + hb + q8k_off(slot, d, D));
        floatx4 x;
#pragma unroll
        for (int j = 0; j < 4; j++) x[j] = (float)((int)((w >> (8 * j)) & 0xff) - 128) * __half2float(__ushort_as_half(sc));
        return x;
    } else {
        return *reinterpret_cast<const floatx4 *>(p.kv.k + hb + (int64_t)slot * p.kv.row_stride + 4 * (int64_t)d);
    }
}

// V of a cached row at the dims 16*t + d0 + r, d0 + r < 16. (The
// addresses are opaque so that nothing of them is kept in registers over the
// tiles that need none.)
template <int D, bool Q8>
struct LaneV {
    const uint8_t *v;
    const uint16_t *scale;
    __device__ __forceinline__ LaneV(const PrefillParams &p, int64_t hb, int slot, int d0) {
        if constexpr (Q8) {
            v = p.kv.v + hb + q8v_off(slot, d0, D);
            scale = reinterpret_cast<const uint16_t *>(p.kv.vs + hb) + slot * (D / 32);
            asm volatile("" : "+v"(scale));
        } else {
            v = p.kv.v + hb + (int64_t)slot * p.kv.row_stride + 4 * d0;
            scale = nullptr;
        }
        asm volatile("" : "+v"(v));
    }
    __device__ __forceinline__ float operator()(int t, int r) const {
        if constexpr (Q8) {
            return (float)((int)v[(t >> 2) * 1024 + r * 16 + (t & 3) * 4] - 128) * __half2float(__ushort_as_half(scale[t >> 1]));
        } else {
            return reinterpret_cast<const float *>(v)[16 * t + r];
        }
    }
};

// Whether the image holds V value v of a key with scale 2^(kTop - e) as zero.
__device__ __forceinline__ bool v_is_bad(float v) { return !(fabsf(v) < INFINITY); }
__device__ __forceinline__ bool v_is_small(float v, float scale) {
    const float t = fabsf(v) * scale;
    return t < kSmall && t > 0.0f;
}

// One 32-key tile of a (sequence, KV head) pair on its way from the cache to
// its pieces, by 256 threads: fetch() issues the loads, convert() finds the
// keys' exponents and hands out the pieces.
// K piece i is 8 consecutive dims of one key, V piece i 8 keys of one dim.
template <int D>
__device__ __forceinline__ int k_piece_key(int i) { return i / (D / 8 * 16) * 16 + (i & 15); }
template <int D>
__device__ __forceinline__ int k_piece_dim(int i) { return (i % (D / 8 * 16) >> 4) * 8; }
__device__ __forceinline__ int v_piece_key(int i, int j) { return (j >> 2) * 16 + 4 * ((i >> 4) & 3) + (j & 3); }
__device__ __forceinline__ int v_piece_dim(int i) { return 16 * (i >> 6) + (i & 15); }

// What convert() needs in LDS; odd[] is zero between tiles.
template <int D, bool Q8>
struct SplitAux {
    int k_exp[KT], v_exp[KT];
    uint32_t odd[3];  // TileHead's masks
    uint32_t pad[1];
    TileMeta meta;
    float v[Q8 ? 1 : KT][Q8 ? 4 : D + 4];  // scaled rows of V, read back along the keys
};

template <int D, bool Q8>
struct SplitTile {
    static constexpr int NK = 4 * D / 256;  // 16-byte pieces of K (and of V) per thread
    static constexpr int KPW = 512 / D;     // f32: whole K rows per wave and round, the low bits of the lane
    // f32: the rows' own 16-byte loads; Q8_0: quants and scales
    floatx4 ka[Q8 ? 1 : NK][2], va[Q8 ? 1 : NK][2];
    uint2 kw[Q8 ? NK : 1];
    uint32_t vw[Q8 ? NK : 1][2];
    uint16_t ks[Q8 ? NK : 1], vs[Q8 ? NK : 1][8];
    uint16_t row_scale[Q8 ? D / 32 : 1];  // threads 0..63: all scales of one key's K (0..31) or V

    static __device__ __forceinline__ int k_row(int r) {  // f32: the key of the thread's piece r
        return ((int)(threadIdx.x >> 6) + 4 * r) * KPW + (int)(threadIdx.x & (KPW - 1));
    }
    static __device__ __forceinline__ int k_col(int) { return (int)(threadIdx.x & 63) / KPW; }  // its dims / 8

    // keys outside [klo, khi] are zero (khi >= 0, and the tile meets the range)
    __device__ __forceinline__ void fetch(const PrefillParams &p, int b, int kvh, int k0, int klo, int khi) {
        const int64_t head_off = (int64_t)kvh * p.kv.head_stride;
        const int64_t hb0 = map_page(p.pm, b, min(k0, khi) >> 4) * p.kv.page_stride + head_off;
        const int64_t hb1 = map_page(p.pm, b, min(k0 + 16, khi) >> 4) * p.kv.page_stride + head_off;
        if constexpr (Q8) {
            if (threadIdx.x < 64) {
                const int key = threadIdx.x & 31;
                const int64_t hb = key < 16 ? hb0 : hb1;
#pragma unroll
                for (int blk = 0; blk < D / 32; blk++)
                    row_scale[blk] = threadIdx.x < 32
                                         ? reinterpret_cast<const uint16_t *>(p.kv.ks + hb)[q8ks_off(key & 15, blk, D)]
                                         : reinterpret_cast<const uint16_t *>(p.kv.vs + hb)[(key & 15) * (D / 32) + blk];
            }
#pragma unroll
            for (int r = 0; r < NK; r++) {
                const int i = threadIdx.x + 256 * r;
                const int key = k_piece_key<D>(i), d = k_piece_dim<D>(i);
                const int64_t hb = key < 16 ? hb0 : hb1;
                kw[r] = *reinterpret_cast<const uint2 *>(p.kv.k + hb + q8k_off(key & 15, d, D));
                ks[r] = reinterpret_cast<const uint16_t *>(p.kv.ks + hb)[q8ks_off(key & 15, d >> 5, D)];
                const int vd = v_piece_dim(i), g4 = 4 * ((i >> 4) & 3);
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const int64_t vb = h ? hb1 : hb0;
                    vw[r][h] = *reinterpret_cast<const uint32_t *>(p.kv.v + vb + q8v_off(g4, vd, D));
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        vs[r][4 * h + j] =
                            reinterpret_cast<const uint16_t *>(p.kv.vs + vb)[(g4 + j) * (D / 32) + (vd >> 5)];
                }
            }
        } else {
#pragma unroll
            for (int r = 0; r < NK; r++) {
                const int u = threadIdx.x + 256 * r;
                const int key = u / (D / 8);
                const int kp = k0 + key;
                va[r][0] = va[r][1] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
                if (kp >= klo && kp <= khi) {
                    const float *vr = reinterpret_cast<const float *>(p.kv.v + (key < 16 ? hb0 : hb1) +
                                                                      (int64_t)(kp & 15) * p.kv.row_stride) +
                                      8 * (u - key * (D / 8));
                    va[r][0] = *reinterpret_cast<const floatx4 *>(vr);
                    va[r][1] = *reinterpret_cast<const floatx4 *>(vr + 4);
                }
            }
#pragma unroll
            for (int r = 0; r < NK; r++) {
                const int key = k_row(r);
                const int kp = k0 + key;
                ka[r][0] = ka[r][1] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
                if (kp >= klo && kp <= khi) {
                    const float *kr = reinterpret_cast<const float *>(p.kv.k + (key < 16 ? hb0 : hb1) +
                                                                      (int64_t)(kp & 15) * p.kv.row_stride) +
                                      8 * k_col(r);
                    ka[r][0] = *reinterpret_cast<const floatx4 *>(kr);
                    ka[r][1] = *reinterpret_cast<const floatx4 *>(kr + 4);
                }
            }
        }
    }

    // Q8_0: the thread's pieces in f32 (keys outside [klo, khi] zero).
    __device__ __forceinline__ void dequantize(int k0, int klo, int khi, float (&kf)[NK][8], float (&vf)[NK][8]) const {
#pragma unroll
        for (int r = 0; r < NK; r++) {
            const int i = threadIdx.x + 256 * r;
            const int kp = k0 + k_piece_key<D>(i);
            const bool ok = kp >= klo && kp <= khi;
            const float ksc = __half2float(__ushort_as_half(ks[r]));
#pragma unroll
            for (int j = 0; j < 8; j++) {  // stored quants are x + 128
                const uint32_t w = j < 4 ? kw[r].x : kw[r].y;
                kf[r][j] = ok ? (float)((int)((w >> (8 * (j & 3))) & 0xff) - 128) * ksc : 0.0f;
                const int vp = k0 + v_piece_key(i, j);
                const float vsc = __half2float(__ushort_as_half(vs[r][j]));
                vf[r][j] = vp >= klo && vp <= khi
                               ? (float)((int)((vw[r][j >> 2] >> (8 * (j & 3))) & 0xff) - 128) * vsc
                               : 0.0f;
            }
        }
    }

    // put_k(i, hi, lo) and put_v(i, hi, lo) take piece i of each image. No
    // thread may still be reading aux; after the next barrier aux.meta may be read.
    template <typename PutK, typename PutV>
    __device__ __forceinline__ void convert(SplitAux<D, Q8> &aux, int k0, int klo, int khi, PutK put_k, PutV put_v) const {
        half8p hi, lo;
        if constexpr (Q8) {
            // exponents from a key's scales: a value is at most 128 of them,
            // at least 1 where it is not zero
            if (threadIdx.x < 64) {
                const int key = threadIdx.x & 31;
                const int kp = k0 + key;
                uint32_t top = 0, low = 0xffffffffu;
                bool bad = false;
#pragma unroll
                for (int blk = 0; blk < D / 32; blk++) {
                    const float x = fabsf(__half2float(__ushort_as_half(row_scale[blk])));
                    const uint32_t bits = __float_as_uint(x);
                    const bool finite = bits < kInfBits;
                    bad = bad || !finite;
                    if (finite && bits) {
                        top = max(top, bits);
                        low = min(low, bits);
                    }
                }
                const bool in = kp >= klo && kp <= khi;
                const int e = class_of(in && top ? top + (7u << 23) : 0);
                const bool small = top && (threadIdx.x < 32 ? low + (13u << 23) < top
                                                            : __uint_as_float(low) * pow2f(kTop - e) < kSmall);
                (threadIdx.x < 32 ? aux.k_exp : aux.v_exp)[key] = e;
                if (in && threadIdx.x < 32 && (bad || small)) atomicOr(&aux.odd[0], 1u << key);
                if (in && threadIdx.x >= 32 && bad) atomicOr(&aux.odd[1], 1u << key);
                if (in && threadIdx.x >= 32 && small) atomicOr(&aux.odd[2], 1u << key);
            }
            float kf[NK][8], vf[NK][8];
            dequantize(k0, klo, khi, kf, vf);
            __syncthreads();
#pragma unroll
            for (int r = 0; r < NK; r++) {
                const int i = threadIdx.x + 256 * r;
                split8(kf[r], pow2f(kTop - aux.k_exp[k_piece_key<D>(i)]), hi, lo);
                put_k(i, hi, lo);
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const float sc = pow2f(kTop - aux.v_exp[v_piece_key(i, j)]);
                    if ((aux.odd[1] | aux.odd[2]) && (v_is_bad(vf[r][j]) || v_is_small(vf[r][j], sc))) vf[r][j] = 0.0f;
                    vf[r][j] *= sc;
                }
                split8(vf[r], 1.0f, hi, lo);
                put_v(i, hi, lo);
            }
        } else {
#pragma unroll
            for (int r = 0; r < NK; r++) {
                const int u = threadIdx.x + 256 * r;
                const int key = u / (D / 8);
                float x[8];
                uint32_t low = 0xffffffffu;  // of the non-zero values' bits, less 1
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    x[j] = va[r][j >> 2][j & 3];
                    low = min(low, (__float_as_uint(x[j]) & 0x7fffffffu) - 1u);
                }
                uint32_t top = umax_group<D / 8>(top_bits(x));
                if (__ballot(top >= kInfBits)) {  // of the finite values
                    top = 0;
#pragma unroll
                    for (int j = 0; j < 8; j++) {
                        const uint32_t bits = __float_as_uint(x[j]) & 0x7fffffffu;
                        top = max(top, bits < kInfBits ? bits : 0);
                    }
                    top = umax_group<D / 8>(top);
                }
                const int e = class_of(top);
                const float sc = pow2f(kTop - e);
                if (top_bits(x) > top || __uint_as_float(low + 1u) * sc < kSmall) {
                    bool bad = false, small = false;
#pragma unroll
                    for (int j = 0; j < 8; j++) {
                        const bool b = v_is_bad(x[j]), l = v_is_small(x[j], sc);
                        bad = bad || b;
                        small = small || l;
                        x[j] = b || l ? 0.0f : x[j];
                    }
                    if (bad) atomicOr(&aux.odd[1], 1u << key);
                    if (small) atomicOr(&aux.odd[2], 1u << key);
                }
#pragma unroll
                for (int j = 0; j < 8; j++) x[j] *= sc;
                const int c = u - key * (D / 8);
                if (c == 0) aux.v_exp[key] = e;
                floatx4 *dst = reinterpret_cast<floatx4 *>(&aux.v[key][8 * c]);
                dst[0] = floatx4{x[0], x[1], x[2], x[3]};
                dst[1] = floatx4{x[4], x[5], x[6], x[7]};
            }
#pragma unroll
            for (int r = 0; r < NK; r++) {
                const int key = k_row(r), c = k_col(r);
                float x[8];
#pragma unroll
                for (int j = 0; j < 8; j++) x[j] = ka[r][j >> 2][j & 3];
                const uint32_t run = top_bits(x);
                const uint32_t top = umax_stride<KPW>(run);
                const int e = class_of(top < kInfBits ? top : 0);
                if (top >= kInfBits || run_is_odd(run, top)) atomicOr(&aux.odd[0], 1u << key);
                if (c == 0) aux.k_exp[key] = e;
                split8(x, pow2f(kTop - e), hi, lo);
                put_k(((key >> 4) * (D / 8) + c) * 16 + (key & 15), hi, lo);
            }
            __syncthreads();
#pragma unroll
            for (int r = 0; r < NK; r++) {
                const int i = threadIdx.x + 256 * r;
                float x[8];
#pragma unroll
                for (int j = 0; j < 8; j++) x[j] = aux.v[v_piece_key(i, j)][v_piece_dim(i)];
                split8(x, 1.0f, hi, lo);
                put_v(i, hi, lo);
            }
        }
        if (threadIdx.x < 64) {
            const int key = threadIdx.x & 31;
            const int32_t exps = key_exps(aux.k_exp[key], aux.v_exp[key]);
            const uint32_t odd_k = aux.odd[0], bad_v = aux.odd[1], small_v = aux.odd[2];
            const int kp = k0 + key;
            const bool in = kp >= klo && kp <= khi;
            const uint32_t keys = (uint32_t)__ballot(in);
            const int32_t first = __builtin_amdgcn_readlane(exps, __builtin_ctz(keys));  // (a tile has a key in range)
            const bool same = !__ballot(in && exps != first);
            if (threadIdx.x < 32) aux.meta.exps[key] = exps;
            if (threadIdx.x == 0) {
                aux.meta.head = TileHead{same ? first : kMixed, odd_k, bad_v, small_v};
                aux.odd[0] = aux.odd[1] = aux.odd[2] = 0;
            }
        }
    }
};

// The tiles that some query of sequence b attends.
struct SeqTiles {
    int lo, hi;        // the keys: [lo, hi], hi < 0 if there are none
    int first, count;  // their tiles
    __device__ __forceinline__ SeqTiles(const PrefillParams &p, int b) {
        const int q_len = min(max(p.q_start[b + 1] - p.q_start[b], 0), p.max_q_len);
        const int pos0 = p.pos_offset[b];
        lo = window_lo(pos0, p.sliding_window);
        hi = q_len > 0 ? min(pos0 + q_len - 1, p.pm.pos_limit - 1) : -1;
        first = lo / KT;
        count = hi >= lo ? hi / KT - first + 1 : 0;
    }
};

// Where the tile images of a (sequence, KV head) pair are. `start` null: every
// pair has `stride` places. Else the attended tiles of all pairs are numbered one
// after the other, start[b] being the first of sequence b's, and taken in rounds:
// a pair belongs to the round in whose `span` numbers its first tile falls, and
// may run past them by up to `over`. A longer pair, or one past the last round,
// has none.
struct Images {
    uint8_t *img;
    TileMeta *meta;
    const int64_t *start;
    int stride, span, over, round, rounds;
    __device__ __forceinline__ bool here(int b, int kvh, int count) const {
        if (!start) return true;
        const int64_t at = start[b] + (int64_t)kvh * count - (int64_t)round * span;
        return at >= 0 && at < span && count <= over;
    }
    __device__ __forceinline__ bool nowhere(int b, int kvh, int count) const {
        return !start || start[b] + (int64_t)kvh * count >= (int64_t)rounds * span || count > over;
    }
    __device__ __forceinline__ int64_t first(int b, int kvh, int n_kv_heads, int count) const {
        return start ? start[b] + (int64_t)kvh * count - (int64_t)round * span
                     : ((int64_t)b * n_kv_heads + kvh) * stride;
    }
};

// start[b] of every sequence. One workgroup; a call that has a place for every
// tile its storage could have it attend does without.
__global__ __launch_bounds__(1024) void image_start_kernel(const PrefillParams p, int n_seqs, int64_t *start) {
    __shared__ int64_t sum[1024];
    int64_t before = 0;
    for (int b0 = 0; b0 < n_seqs; b0 += 1024) {
        const int b = b0 + threadIdx.x;
        const int64_t mine = b < n_seqs ? (int64_t)SeqTiles(p, b).count * p.n_kv_heads : 0;
        sum[threadIdx.x] = mine;
        for (int d = 1; d < 1024; d *= 2) {
            __syncthreads();
            const int64_t x = (int)threadIdx.x >= d ? sum[threadIdx.x - d] : 0;
            __syncthreads();
            sum[threadIdx.x] += x;
        }
        __syncthreads();
        if (b < n_seqs) start[b] = before + sum[threadIdx.x] - mine;
        before += sum[1023];
        __syncthreads();
    }
}

// Grid (sequence, slice): the workgroups of a sequence take its (KV head, tile)
// pairs in turn, as many as it has. 256 threads.
template <int D, bool Q8>
__global__ __launch_bounds__(256) void stage_split_kernel(const PrefillParams p, const Images im) {
    const int b = blockIdx.x;
    const SeqTiles seq(p, b);
    __shared__ __attribute__((aligned(16))) SplitAux<D, Q8> aux;
    if (threadIdx.x < 3) aux.odd[threadIdx.x] = 0;
    for (int item = blockIdx.y; item < seq.count * p.n_kv_heads; item += gridDim.y) {
        const int kvh = item / seq.count;
        const int t = item - kvh * seq.count;
        if (!im.here(b, kvh, seq.count)) continue;
        const int k0 = (seq.first + t) * KT;
        SplitTile<D, Q8> tile;
        tile.fetch(p, b, kvh, k0, seq.lo, seq.hi);
        __syncthreads();  // aux is free
        const int64_t at = im.first(b, kvh, p.n_kv_heads, seq.count) + t;
        uint8_t *dst = im.img + at * kSplitImage<D>;
        const auto put = [](uint8_t *to) {
            return [to](int i, const half8p &hi, const half8p &lo) {
                *reinterpret_cast<half8p *>(to + i * 16) = hi;
                *reinterpret_cast<half8p *>(to + 64 * D + i * 16) = lo;
            };
        };
        tile.convert(aux, k0, seq.lo, seq.hi, put(dst), put(dst + 128 * D));
        __syncthreads();
        constexpr int WORDS = sizeof(TileMeta) / 4;
        if (threadIdx.x < WORDS)
            reinterpret_cast<uint32_t *>(im.meta + at)[threadIdx.x] = reinterpret_cast<const uint32_t *>(&aux.meta)[threadIdx.x];
    }
}

// The staging launch of the bf16 path.
template <int D, bool Q8>
__global__ __launch_bounds__(256) void stage_bf16_kernel(const PrefillParams p, uint8_t *img, int n_tiles) {
    const int t = blockIdx.x;
    const int kvh = blockIdx.y;
    const int b = blockIdx.z;
    const int row0 = p.q_start[b];
    const int q_len = min(max(p.q_start[b + 1] - row0, 0), p.max_q_len);
    if (q_len == 0) return;
    const int pos0 = p.pos_offset[b];
    const int khi = min(pos0 + q_len - 1, p.pm.pos_limit - 1);
    const int klo = window_lo(pos0, p.sliding_window);
    const int k0 = t * KT;
    if (khi < klo || k0 > khi || k0 + KT - 1 < klo) return;  // a tile no query of the sequence reads

    uint8_t *dst = img + (((int64_t)b * p.n_kv_heads + kvh) * n_tiles + t) * kTileImage<D>;
    constexpr int NP = 4 * D;  // pieces of K (and of V) per tile
    if constexpr (!Q8) {
        // f32 cache: a K piece is 8 consecutive dims of one key, read and
        // converted straight from the row; V pieces run across keys, so V
        // goes through LDS as bf16 rows. The tile's 32 keys lie in two pages.
        __shared__ __attribute__((aligned(16))) __bf16 Vh[KT][D + 8];
        const int64_t head_off = (int64_t)kvh * p.kv.head_stride;
        const int64_t pid0 = map_page(p.pm, b, min(k0, khi) >> 4);
        const int64_t pid1 = map_page(p.pm, b, min(k0 + 16, khi) >> 4);
        // every load of the thread is issued before any store (the stores to
        // the image could alias the cache for the compiler)
        constexpr int NV = KT * (D / 8) / 256;  // V (key, 8 dims) runs per thread
        constexpr int NK = NP / 256;            // K pieces per thread
        float4 va[NV][2], ka[NK][2];
#pragma unroll
        for (int r = 0; r < NV; r++) {
            const int u = threadIdx.x + 256 * r;
            const int key = u / (D / 8);
            const int kp = k0 + key;
            va[r][0] = va[r][1] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (kp >= klo && kp <= khi) {
                const float *vr = reinterpret_cast<const float *>(
                    p.kv.v + (key < 16 ? pid0 : pid1) * p.kv.page_stride + head_off +
                    (int64_t)(kp & 15) * p.kv.row_stride) + 8 * (u - key * (D / 8));
                va[r][0] = *reinterpret_cast<const float4 *>(vr);
                va[r][1] = *reinterpret_cast<const float4 *>(vr + 4);
            }
        }
#pragma unroll
        for (int r = 0; r < NK; r++) {
            const int i = threadIdx.x + 256 * r;
            const int mt = i / (D / 8 * 16);
            const int rem = i - mt * (D / 8 * 16);
            const int key = mt * 16 + (rem & 15);
            const int kp = k0 + key;
            ka[r][0] = ka[r][1] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (kp >= klo && kp <= khi) {
                const float *kr = reinterpret_cast<const float *>(
                    p.kv.k + (key < 16 ? pid0 : pid1) * p.kv.page_stride + head_off +
                    (int64_t)(kp & 15) * p.kv.row_stride) + 8 * (rem >> 4);
                ka[r][0] = *reinterpret_cast<const float4 *>(kr);
                ka[r][1] = *reinterpret_cast<const float4 *>(kr + 4);
            }
        }
#pragma unroll
        for (int r = 0; r < NV; r++) {
            const int u = threadIdx.x + 256 * r;
            const int key = u / (D / 8);
            const float4 x = va[r][0], y = va[r][1];
            *reinterpret_cast<bf16x8 *>(&Vh[key][8 * (u - key * (D / 8))]) =
                bf16x8{(__bf16)x.x, (__bf16)x.y, (__bf16)x.z, (__bf16)x.w,
                       (__bf16)y.x, (__bf16)y.y, (__bf16)y.z, (__bf16)y.w};
        }
        // K pieces, straight to the image
#pragma unroll
        for (int r = 0; r < NK; r++) {
            const float4 x = ka[r][0], y = ka[r][1];
            *reinterpret_cast<bf16x8 *>(dst + (int64_t)(threadIdx.x + 256 * r) * 16) =
                bf16x8{(__bf16)x.x, (__bf16)x.y, (__bf16)x.z, (__bf16)x.w,
                       (__bf16)y.x, (__bf16)y.y, (__bf16)y.z, (__bf16)y.w};
        }
        __syncthreads();
        for (int i = threadIdx.x; i < NP; i += 256) {
            const int tt = i >> 6;
            const int g = (i >> 4) & 3;
            const int d = 16 * tt + (i & 15);
            const bf16x8 h = bf16x8{Vh[4 * g][d], Vh[4 * g + 1][d], Vh[4 * g + 2][d], Vh[4 * g + 3][d],
                                    Vh[16 + 4 * g][d], Vh[17 + 4 * g][d], Vh[18 + 4 * g][d], Vh[19 + 4 * g][d]};
            *reinterpret_cast<bf16x8 *>(dst + 64 * D + (int64_t)i * 16) = h;
        }
        return;
    }
    // Q8_0: the pieces of a thread straight from the quants (8 dims of a key
    // are 8 bytes, 4 keys of a dim are 4), not through f32 rows in LDS: 300
    // Gemma-2 rows after 2,000 cached positions 101.2 -> 97.0 us per call
    SplitTile<D, true> tile;
    tile.fetch(p, b, kvh, k0, klo, khi);
    float kf[SplitTile<D, true>::NK][8], vf[SplitTile<D, true>::NK][8];
    tile.dequantize(k0, klo, khi, kf, vf);
#pragma unroll
    for (int r = 0; r < SplitTile<D, true>::NK; r++) {
        bf16x8 kh, vh;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            kh[j] = (__bf16)kf[r][j];
            vh[j] = (__bf16)vf[r][j];
        }
        const int64_t at = (int64_t)(threadIdx.x + 256 * r) * 16;
        *reinterpret_cast<bf16x8 *>(dst + at) = kh;
        *reinterpret_cast<bf16x8 *>(dst + 64 * D + at) = vh;
    }
}

// Waves per SIMD the kernel's registers are sized for; LDS holds two tiles of
// a workgroup: d = 64 32 KB, d = 128 64 KB, d = 256 128 KB. A workgroup that
// converts its own tiles holds one image and the conversion's buffers, and the
// next tile's loads in registers (not at d = 256, whose registers are full).
template <int D, bool STAGED, int NT>
constexpr int kSplitOccupancy = !STAGED ? (D == 64 ? 2 : 1) : (D == 64 ? 4 - NT : (D == 128 ? 2 : 1));

template <int D, bool Q8, bool CAP, bool STAGED, int NT>
__global__ __launch_bounds__(256, (kSplitOccupancy<D, STAGED, NT>)) void prefill_split_kernel(const PrefillParams p,
                                                                                                const Images im) {
    constexpr int NW = 4;
    constexpr int QW = 16 * NT;
    constexpr int KS = D / 32;
    constexpr int DT = D / 16;
    constexpr int IMG = kSplitImage<D>;
    constexpr int CPW = IMG / 1024 / NW;  // kilobyte copies per wave and tile
    constexpr int AUX = IMG + (int)sizeof(SplitAux<D, Q8>);
    constexpr int SROW = D + 4;  // an output row in LDS
    constexpr int METAS = 2 * IMG;  // staged: where the two tiles' TileMeta are
    constexpr int LDS = std::max(STAGED ? METAS + 2 * (int)sizeof(TileMeta) : AUX, NW * 16 * SROW * 4);
    __shared__ __attribute__((aligned(16))) uint8_t lds[LDS];

    const int n_hgrp = p.group / p.hpw;
    const int pair = (int)blockIdx.x / n_hgrp;
    const int b = pair / p.n_kv_heads;
    const int kvh = pair - b * p.n_kv_heads;
    const int hgrp = (int)blockIdx.x - pair * n_hgrp;
    const int qblk = p.n_qblocks - 1 - (int)(blockIdx.z * gridDim.y + blockIdx.y);
    const int waves_per_head = NW / p.hpw;
    const int qwg = QW * waves_per_head;

    const int row0 = p.q_start[b];
    const int q_len = min(max(p.q_start[b + 1] - row0, 0), p.max_q_len);
    const int pos0 = p.pos_offset[b];
    const int qb0 = qblk * qwg;
    if (qblk < 0 || qb0 >= q_len) return;
    const SeqTiles seq(p, b);
    if (STAGED ? !im.here(b, kvh, seq.count) : !im.nowhere(b, kvh, seq.count)) return;  // another launch's

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lrow = lane & 15;
    const int lgrp = lane >> 4;
    const int head = kvh * p.group + hgrp * p.hpw + (wave % p.hpw);
    const int wq0 = qb0 + (wave / p.hpw) * QW;

    const int q_last = min(q_len, qb0 + qwg) - 1;
    const int khi = min(pos0 + q_last, p.pm.pos_limit - 1);
    const int klo = window_lo(pos0 + qb0, p.sliding_window);
    const int tfirst = klo / KT;
    const int n = khi >= klo ? khi / KT - tfirst + 1 : 0;
    // the keys that some query of the sequence attends; others are zero in the images
    const int ulo = seq.lo, uhi = seq.hi;
    const int64_t first = STAGED ? im.first(b, kvh, p.n_kv_heads, seq.count) + tfirst - seq.first : 0;
    const TileMeta *unit_meta = im.meta + first;
    const uint8_t *unit_img = im.img + first * IMG;
    const uint32_t ring = __builtin_amdgcn_readfirstlane(
        (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void *)&lds[0]);
    auto issue = [&](int i) {
        const uint8_t *src = unit_img + (int64_t)i * IMG;
        const uint32_t dst = ring + (uint32_t)((i & 1) * IMG);
#pragma unroll
        for (int c = 0; c < CPW; c++) {
            const int piece = wave * CPW + c;
            lds_copy16(src + piece * 1024, (uint32_t)(lane * 16), dst + piece * 1024);
        }
    };

    const auto issue_meta = [&](int i) __attribute__((always_inline)) {
        if (wave == 0)
            lds_copy4(reinterpret_cast<const uint8_t *>(unit_meta + i), (uint32_t)(lane * 4),
                      ring + METAS + (uint32_t)((i & 1) * sizeof(TileMeta)));
    };

    if (STAGED && n > 0) issue(0);
    // the exponents of the first tile whose keys share them (a prompt's first keys
    // often differ from the rest)
    int32_t exps = kMixed;
    for (int i = 0; STAGED && i < n && exps == kMixed; i += 64) {
        const int32_t mine = unit_meta[min(i + lane, n - 1)].head.exps;
        const uint64_t found = __ballot(mine != kMixed);
        if (found) exps = __builtin_amdgcn_readlane(mine, __builtin_ctzll(found));
    }

    // Q^T operand: pieces of Q[query nt*16 + lrow][d = ks*32 + lgrp*8 + 0..7]
    // times the query's own power of two
    half8p qh[NT][KS], ql[NT][KS];
    float qinv[NT];
    bool qodd[NT];  // the lane's query row holds what the pieces cannot
    bool any_odd = false;  // some row of the wave does
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
        const int lq = wq0 + nt * 16 + lrow;
        const bool ok = lq < q_len;
        const float *qp = p.q + ((int64_t)(row0 + (ok ? lq : 0)) * p.n_heads + head) * D;
        float x[KS][8];
        uint32_t run[KS], top = 0;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const floatx4 a = __builtin_nontemporal_load(reinterpret_cast<const floatx4 *>(qp + ks * 32 + lgrp * 8));
            const floatx4 c = __builtin_nontemporal_load(reinterpret_cast<const floatx4 *>(qp + ks * 32 + lgrp * 8 + 4));
#pragma unroll
            for (int j = 0; j < 8; j++) x[ks][j] = ok ? (j < 4 ? a[j & 3] : c[j & 3]) * p.q_mul : 0.0f;
        }
#pragma unroll
        for (int ks = 0; ks < KS; ks++) top = max(top, run[ks] = top_bits(x[ks]));
        top = umax_rows4(top);
        const int e = top && top < kInfBits ? exponent_of(top) : kTop;
        uint32_t bad = top >= kInfBits;
        qinv[nt] = pow2f(e - kTop);
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            bad |= run_is_odd(run[ks], top);
            split8(x[ks], pow2f(kTop - e), qh[nt][ks], ql[nt][ks]);
        }
        qodd[nt] = umax_rows4(bad);
        any_odd = any_odd || __ballot(qodd[nt]);
    }
    const bool plain = !__syncthreads_or(any_odd) && (!STAGED || exps != kMixed);

    floatx4 o[DT][NT];
    float m[NT], lpart[NT];
    int rexp[NT];  // R: O is in units of 2^(rexp - kTop - kScaleP)
    float weight[NT];  // 2^(E - R + kScaleP) of `exps`
    int qpos[NT], qlo[NT];
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
#pragma unroll
        for (int t = 0; t < DT; t++) o[t][nt] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
        lpart[nt] = 0.0f;
        rexp[nt] = kNoExp;
        weight[nt] = (float)(1 << kScaleP);
        m[nt] = kMLowest;  // finite: the first attended key is an ordinary move of the reference
        const int lq = wq0 + nt * 16 + lrow;
        qpos[nt] = lq < q_len ? pos0 + lq : -1;
        qlo[nt] = window_lo(pos0 + lq, p.sliding_window);
    }
    // keys this wave's queries attend: [wlo, whi]
    const int whi = min(khi, pos0 + wq0 + QW - 1);
    const int wlo = max(klo, window_lo(pos0 + wq0, p.sliding_window));

    // The rare path reads the arguments again: held for it over the tiles that
    // need none, they and what follows from them crowd the other registers.
    const auto arguments = [&]() __attribute__((always_inline)) {
        const PrefillParams *a = (const PrefillParams *)__builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+s"(a));
        return a;
    };
    const auto head_page = [&](const PrefillParams *a, int k) __attribute__((always_inline)) {
        return map_page(a->pm, b, min(k, uhi) >> 4) * a->kv.page_stride + (int64_t)kvh * a->kv.head_stride;
    };
    // The f32 scores of a tile in place of the pieces' for odd keys and rows.
    const auto odd_scores = [&](floatx4 (&s)[2][NT], int k0, uint32_t keys) __attribute__((always_inline)) {
        const PrefillParams *a = arguments();
        const int64_t hb[2] = {head_page(a, k0), head_page(a, k0 + 16)};
        const float *qp[NT];
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
            const int lq = min(wq0 + nt * 16 + lrow, q_len - 1);  // (a row past the end has no result)
            qp[nt] = a->q + ((int64_t)(row0 + lq) * a->n_heads + head) * D + lgrp * (D / 4);
        }
        floatx4 e[2][NT];
#pragma unroll
        for (int mt = 0; mt < 2; mt++)
#pragma unroll
            for (int nt = 0; nt < NT; nt++) e[mt][nt] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 2
        for (int d = 0; d < D / 4; d += 4) {  // lane group g multiplies the dims g * D/4 ..
            floatx4 kd[2], qd[NT];
#pragma unroll
            for (int mt = 0; mt < 2; mt++) {
                const int kp = k0 + 16 * mt + lrow;
                kd[mt] = k_values4<D, Q8>(*a, hb[mt], lrow, lgrp * (D / 4) + d);
                if (kp < ulo || kp > uhi) kd[mt] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
            }
#pragma unroll
            for (int nt = 0; nt < NT; nt++) qd[nt] = *reinterpret_cast<const floatx4 *>(qp[nt] + d) * a->q_mul;
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int mt = 0; mt < 2; mt++)
#pragma unroll
                    for (int nt = 0; nt < NT; nt++)
                        e[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x4f32(kd[mt][j], qd[nt][j], e[mt][nt], 0, 0, 0);
        }
#pragma unroll
        for (int mt = 0; mt < 2; mt++)
#pragma unroll
            for (int nt = 0; nt < NT; nt++)
#pragma unroll
                for (int r = 0; r < 4; r++)
                    if (qodd[nt] || (keys >> (16 * mt + 4 * lgrp + r) & 1)) s[mt][nt][r] = e[mt][nt][r];
    };
    // The products of V's small values with the probabilities pv (element 4*mt + r
    // of a lane: key 16*mt + 4*lgrp + r) on the f32 MFMA: its step (mt, r) takes
    // those four keys.
    const auto small_values = [&](const float (&pv)[NT][8], int k0, uint32_t keys, const TileMeta *meta) __attribute__((always_inline)) {
        const PrefillParams *a = arguments();
        const int64_t hb[2] = {head_page(a, k0), head_page(a, k0 + 16)};
        float unit[NT];
#pragma unroll
        for (int nt = 0; nt < NT; nt++)  // (a row that has attended no key has only zeros to multiply)
            unit[nt] = rexp[nt] == kNoExp ? 0.0f : ldexpf(1.0f, kTop + kScaleP - rexp[nt]);
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int key = (j >> 2) * 16 + 4 * lgrp + (j & 3);
            const bool has = keys >> key & 1;
            const float scale = pow2f(kTop - v_exp_of(meta->exps[key]));
            const LaneV<D, Q8> v(*a, hb[j >> 2], key & 15, lrow);
            float x[DT];
#pragma unroll
            for (int t = 0; t < DT; t++) x[t] = v(t, 0);
#pragma unroll
            for (int t = 0; t < DT; t++) x[t] = has && v_is_small(x[t], scale) ? x[t] : 0.0f;
#pragma unroll
            for (int t = 0; t < DT; t++)
#pragma unroll
                for (int nt = 0; nt < NT; nt++)
                    o[t][nt] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[t], pv[nt][j] * unit[nt], o[t][nt], 0, 0, 0);
        }
    };
    // The products of V's infinities and NaN with the probabilities, for the
    // queries that attend them.
    const auto bad_values = [&](const float (&pv)[NT][8], int k0, uint32_t keys) __attribute__((always_inline)) {
        for (; keys; keys &= keys - 1) {
            const int key = __builtin_ctz(keys), reg = 4 * (key >> 4) + (key & 3);
            const int kp = k0 + key;
            const PrefillParams *a = arguments();
            const LaneV<D, Q8> v(*a, head_page(a, k0 + (key & 16)), key & 15, 4 * lgrp);
            float x[DT][4];
#pragma unroll
            for (int t = 0; t < DT; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) x[t][r] = v(t, r);
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                float mine = pv[nt][0];
#pragma unroll
                for (int j = 1; j < 8; j++) mine = reg == j ? pv[nt][j] : mine;
                const float pk = __shfl(mine, ((key >> 2) & 3) * 16 + lrow);
                const bool attends = kp >= qlo[nt] && kp <= qpos[nt];
#pragma unroll
                for (int t = 0; t < DT; t++)
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        o[t][nt][r] = attends && v_is_bad(x[t][r]) ? fmaf(pk, x[t][r], o[t][nt][r]) : o[t][nt][r];
            }
        }
    };

    // Tile i. `same`: its keys' exponents are those of `exps`, and nothing is odd;
    // otherwise they are in `meta`.
    const auto attend = [&](auto same, int i, const uint8_t *kimg, const TileMeta *meta) __attribute__((always_inline)) {
        const int k0 = (tfirst + i) * KT;
        if (k0 > whi || k0 + KT - 1 < wlo) return;  // no query of this wave attends it

        // S^T = K . Q^T: the hi products and the cross terms apart, added at
        // the end (the small terms are not rounded at the large ones' unit)
        floatx4 s[2][NT], x[2][NT];
#pragma unroll
        for (int mt = 0; mt < 2; mt++)
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                s[mt][nt] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
                x[mt][nt] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
            }
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            half8p ah[2], al[2];
#pragma unroll
            for (int mt = 0; mt < 2; mt++) {
                const uint8_t *src = kimg + ((mt * (D / 8) + ks * 4 + lgrp) * 16 + lrow) * 16;
                ah[mt] = *reinterpret_cast<const half8p *>(src);
                al[mt] = *reinterpret_cast<const half8p *>(src + 64 * D);
            }
#pragma unroll
            for (int mt = 0; mt < 2; mt++)
#pragma unroll
                for (int nt = 0; nt < NT; nt++)
                    s[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[mt], qh[nt][ks], s[mt][nt], 0, 0, 0);
#pragma unroll
            for (int mt = 0; mt < 2; mt++)
#pragma unroll
                for (int nt = 0; nt < NT; nt++)
                    x[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[mt], ql[nt][ks], x[mt][nt], 0, 0, 0);
#pragma unroll
            for (int mt = 0; mt < 2; mt++)
#pragma unroll
                for (int nt = 0; nt < NT; nt++)
                    x[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al[mt], qh[nt][ks], x[mt][nt], 0, 0, 0);
        }

        // operands of the next d step in flight while one is multiplied
        __builtin_amdgcn_sched_group_barrier(kSchedLds, 8, 0);
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            __builtin_amdgcn_sched_group_barrier(kSchedMfma, 6 * NT, 0);
            if (ks + 2 < KS) __builtin_amdgcn_sched_group_barrier(kSchedLds, 4, 0);
        }

        // softmax: as the bf16 kernels' (a lazy maximum), in f32; c undoes the scales
        const bool interior = k0 >= klo && k0 + KT - 1 <= min(khi, pos0 + wq0) &&
                              (p.sliding_window <= 0 || k0 >= window_lo(pos0 + wq0 + QW - 1, p.sliding_window));
#pragma unroll
        for (int mt = 0; mt < 2; mt++)
#pragma unroll
            for (int nt = 0; nt < NT; nt++)
#pragma unroll
                for (int r = 0; r < 4; r++) s[mt][nt][r] = fmaf(x[mt][nt][r], 0x1p-11f, s[mt][nt][r]);
        float c[NT];  // undoes the scales (powers of two, so where it is done changes no bit)
        int32_t key[8];
#pragma unroll
        for (int nt = 0; nt < NT; nt++) c[nt] = same ? pow2f(k_exp_of(exps) - kTop) * qinv[nt] : 1.0f;
        if constexpr (!same) {
#pragma unroll
            for (int j = 0; j < 8; j++) key[j] = meta->exps[(j >> 2) * 16 + 4 * lgrp + (j & 3)];
#pragma unroll
            for (int mt = 0; mt < 2; mt++)
#pragma unroll
                for (int nt = 0; nt < NT; nt++)
#pragma unroll
                    for (int r = 0; r < 4; r++) s[mt][nt][r] *= pow2f(k_exp_of(key[4 * mt + r]) - kTop) * qinv[nt];
            const uint32_t odd_k = __builtin_amdgcn_readfirstlane(meta->head.odd_k);
            if (odd_k || any_odd) odd_scores(s, k0, odd_k);
        }
        float pv[NT][8];
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
            floatx4 col[2] = {s[0][nt], s[1][nt]};
            if constexpr (CAP) {
                col[0] *= c[nt];
                col[1] *= c[nt];
                c[nt] = 1.0f;
            }
            cap_and_mask<CAP>(col, p.softcap, interior, k0 + 4 * lgrp, qpos[nt], qlo[nt], klo, khi);
            float mx = max3f(max3f(col[0][0], col[0][1], col[0][2]), max3f(col[0][3], col[1][0], col[1][1]),
                             max2f(col[1][2], col[1][3])) * c[nt];
            if (__ballot(mx - m[nt] > kLazyF32)) {
                mx = max_rows4(mx);
                const bool up = mx - m[nt] > kLazyF32;
                const float rs = up ? fast_exp2(m[nt] - mx) : 1.0f;
                m[nt] = up ? mx : m[nt];
#pragma unroll
                for (int t = 0; t < DT; t++) o[t][nt] *= rs;
                lpart[nt] *= rs;
            }
            float ls = 0.0f;
#pragma unroll
            for (int j = 0; j < 8; j++) {
                pv[nt][j] = fast_exp2(fmaf(col[j >> 2][j & 3], c[nt], -m[nt]));
                ls += pv[nt][j];
            }
            lpart[nt] += ls;
        }

        // O^T += V^T . P^T, the probabilities times 2^(E - R)
        half8p ph[NT], pl[NT];
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
            float x[8];
            if constexpr (same) {
#pragma unroll
                for (int j = 0; j < 8; j++) x[j] = pv[nt][j] * weight[nt];
            } else {
                const int lo = max(qlo[nt], klo), hi = min(qpos[nt], khi);
                int top = kNoExp;  // of the keys that the row attends
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const int kp = k0 + (j >> 2) * 16 + 4 * lgrp + (j & 3);
                    top = kp >= lo && kp <= hi ? max(top, v_exp_of(key[j])) : top;
                }
                top = (int)umax_rows4((uint32_t)(top - kNoExp)) + kNoExp;
                if (__ballot(top > rexp[nt] + kLazyExp)) {
                    const bool up = top > rexp[nt] + kLazyExp;
                    // (before its first key a row's O is zero)
                    const float f = up && rexp[nt] != kNoExp ? ldexpf(1.0f, rexp[nt] - top) : 1.0f;
                    rexp[nt] = up ? top : rexp[nt];
#pragma unroll
                    for (int t = 0; t < DT; t++) o[t][nt] *= f;
                }
#pragma unroll
                for (int j = 0; j < 8; j++)
                    x[j] = pv[nt][j] * ldexpf(1.0f, min(v_exp_of(key[j]) - rexp[nt], kLazyExp) + kScaleP);
            }
            split8(x, 1.0f, ph[nt], pl[nt]);
        }
        const uint8_t *vimg = kimg + 128 * D;
        const auto add_cross = [](floatx4 &to, const floatx4 &x) __attribute__((always_inline)) {
#pragma unroll
            for (int r = 0; r < 4; r++) to[r] = fmaf(x[r], 0x1p-11f, to[r]);
        };
        floatx4 cross[NT];
#pragma unroll
        for (int t = 0; t < DT; t++) {
            const uint8_t *src = vimg + ((t * 4 + lgrp) * 16 + lrow) * 16;
            const half8p ah = *reinterpret_cast<const half8p *>(src);
            const half8p al = *reinterpret_cast<const half8p *>(src + 64 * D);
            floatx4 now[NT];
#pragma unroll
            for (int nt = 0; nt < NT; nt++)
                now[nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al, ph[nt], floatx4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
            for (int nt = 0; nt < NT; nt++)
                o[t][nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, ph[nt], o[t][nt], 0, 0, 0);
#pragma unroll
            for (int nt = 0; nt < NT; nt++) now[nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, pl[nt], now[nt], 0, 0, 0);
            // the cross terms of the d tile before, whose products are done by now
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                if (t > 0) add_cross(o[t - 1][nt], cross[nt]);
                cross[nt] = now[nt];
            }
        }
#pragma unroll
        for (int nt = 0; nt < NT; nt++) add_cross(o[DT - 1][nt], cross[nt]);
        __builtin_amdgcn_sched_group_barrier(kSchedLds, 4, 1);
#pragma unroll
        for (int t = 0; t < DT; t++) {
            __builtin_amdgcn_sched_group_barrier(kSchedMfma, 3 * NT, 1);
            if (t + 2 < DT) __builtin_amdgcn_sched_group_barrier(kSchedLds, 2, 1);
        }
        if constexpr (!same) {
            const uint32_t small_v = __builtin_amdgcn_readfirstlane(meta->head.small_v);
            if (small_v) small_values(pv, k0, small_v, meta);
            const uint32_t bad_v = __builtin_amdgcn_readfirstlane(meta->head.bad_v);
            if (bad_v) bad_values(pv, k0, bad_v);
        }
    };

    if constexpr (STAGED) {
        // this wave's copies of tile i have landed, then every wave's; every wave
        // is also done with tile i - 1, whose buffer the next copy takes
        const auto arrive = [&](int i) __attribute__((always_inline)) {
            wait_vm<0>();
            __syncthreads();
            if (i + 1 < n) issue(i + 1);
        };
        // the first tile from `i` on whose keys have other exponents than `exps` or
        // hold something odd
        const auto next_special = [&](int i) __attribute__((always_inline)) {
            if (!plain) return i;
            for (; i < n; i += 64) {
                const TileHead h = unit_meta[min(i + lane, n - 1)].head;
                const uint64_t found = __ballot(h.exps != exps || (h.odd_k | h.bad_v | h.small_v));
                if (found) return min(n, i + __builtin_ctzll(found));
            }
            return n;
        };
        const TileMeta *metas = reinterpret_cast<const TileMeta *>(lds + METAS);
        int stop = n > 0 ? next_special(0) : 0;
        if (stop == n) {  // (the usual case in a loop of its own, whose registers nothing else shares)
#pragma unroll
            for (int nt = 0; nt < NT; nt++) rexp[nt] = v_exp_of(exps);
            for (int i = 0; i < n; i++) {
                arrive(i);
                attend(std::true_type{}, i, lds + (i & 1) * IMG, nullptr);
            }
            stop = -1;
        }
        for (int i = 0; stop >= 0 && i < n; stop = i < n ? next_special(i) : 0) {
            if (i < stop) {
                // R as the first of these tiles would have it, for the rows that
                // attend it; a row that has attended nothing may take it early
#pragma unroll
                for (int nt = 0; nt < NT; nt++) {
                    const int e = v_exp_of(exps);
                    const bool up = e > rexp[nt] + kLazyExp &&
                                    (rexp[nt] == kNoExp || qpos[nt] >= (tfirst + i) * KT);
                    if (__ballot(up && rexp[nt] != kNoExp)) {
                        const float f = up && rexp[nt] != kNoExp ? ldexpf(1.0f, rexp[nt] - e) : 1.0f;
#pragma unroll
                        for (int t = 0; t < DT; t++) o[t][nt] *= f;
                    }
                    rexp[nt] = up ? e : rexp[nt];
                    weight[nt] = ldexpf(1.0f, min(e - rexp[nt], kLazyExp) + kScaleP);
                }
                for (; i < stop; i++) {
                    arrive(i);
                    attend(std::true_type{}, i, lds + (i & 1) * IMG, nullptr);
                }
            }
            if (i < n) {
                // (a row that has attended a key has moved its maximum)
#pragma unroll
                for (int nt = 0; nt < NT; nt++) rexp[nt] = m[nt] != kMLowest ? rexp[nt] : kNoExp;
                issue_meta(i);
                arrive(i);
                attend(std::false_type{}, i, lds + (i & 1) * IMG, metas + (i & 1));
                i++;
            }
        }
    } else if (n > 0) {
        SplitAux<D, Q8> &aux = *reinterpret_cast<SplitAux<D, Q8> *>(lds + IMG);
        constexpr bool AHEAD = D < 256;
        SplitTile<D, Q8> tile;
        tile.fetch(p, b, kvh, tfirst * KT, ulo, uhi);
        if (tid < 3) aux.odd[tid] = 0;
        __syncthreads();
        const auto put = [&](int base) {
            uint8_t *to = lds + base;
            return [to](int j, const half8p &hi, const half8p &lo) {
                *reinterpret_cast<half8p *>(to + j * 16) = hi;
                *reinterpret_cast<half8p *>(to + 64 * D + j * 16) = lo;
            };
        };
        // tile i, ready for every wave
        const auto arrive = [&](int i) __attribute__((always_inline)) {
            const int k0 = (tfirst + i) * KT;
            if (i > 0) __syncthreads();  // its place is free
            if (!AHEAD && i > 0) tile.fetch(p, b, kvh, k0, ulo, uhi);
            tile.convert(aux, k0, ulo, uhi, put(0), put(128 * D));
            __syncthreads();
            if (AHEAD && i + 1 < n) tile.fetch(p, b, kvh, k0 + KT, ulo, uhi);
        };
        int i = 0;
        bool here = false;  // tile i is ready
        for (; i < n && plain; i++) {
            arrive(i);
            if (i == 0) exps = __builtin_amdgcn_readfirstlane(aux.meta.head.exps);
            here = exps == kMixed || __builtin_amdgcn_readfirstlane(aux.meta.head.exps) != exps ||
                   __builtin_amdgcn_readfirstlane(aux.meta.head.odd_k | aux.meta.head.bad_v | aux.meta.head.small_v);
            if (here) break;
            attend(std::true_type{}, i, lds, nullptr);
        }
        // (a row that has attended a key has moved its maximum)
#pragma unroll
        for (int nt = 0; nt < NT; nt++)
            if (i > 0 && m[nt] != kMLowest) rexp[nt] = v_exp_of(exps);
        for (; i < n; i++, here = false) {
            if (!here) arrive(i);
            attend(std::false_type{}, i, lds, &aux.meta);
        }
    }

    // Output rows through LDS, as the staged bf16 kernel writes them
    __syncthreads();
    float *stage = reinterpret_cast<float *>(lds) + wave * 16 * SROW;
    constexpr int LPR = D / 4;    // lanes per row (16 bytes each)
    constexpr int RPI = 64 / LPR;  // rows per store instruction
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
        const float lt = sum_rows4(lpart[nt]);
        const float inv = lt > 0.0f ? 1.0f / lt : 0.0f;
        const int unit_exp = rexp[nt] == kNoExp ? 0 : rexp[nt] - kTop - kScaleP;
#pragma unroll
        for (int t = 0; t < DT; t++) {
            floatx4 x;
#pragma unroll
            for (int r = 0; r < 4; r++) x[r] = ldexpf(o[t][nt][r] * inv, unit_exp);
            *reinterpret_cast<floatx4 *>(stage + lrow * SROW + 16 * t + 4 * lgrp) = x;
        }
#pragma unroll
        for (int k = 0; k < 16 / RPI; k++) {
            const int r = k * RPI + lane / LPR;
            const int c = (lane % LPR) * 4;
            const floatx4 v = *reinterpret_cast<const floatx4 *>(stage + r * SROW + c);
            const int lq = wq0 + nt * 16 + r;
            if (lq < q_len)
                __builtin_nontemporal_store(v, reinterpret_cast<floatx4 *>(p.out + ((int64_t)(row0 + lq) * p.n_heads + head) * D + c));
        }
    }
}

// Query blocks of a call whose waves (four to a workgroup) take nt 16-query
// tiles each.
int wg_blocks(const PrefillParams &prm, int nt) {
    const int rows = 16 * nt * (4 / prm.hpw);
    return (prm.max_q_len + rows - 1) / rows;
}
// 16-query tiles per wave of a staged kernel: two share every operand read, one
// gives twice the workgroups (the same bits), which is worth more until they
// fill the chip: at up to 1.5 workgroups per CU. us per call, two tiles / one,
// 32/8 heads, d = 128: 400 rows (104 workgroups of two tiles) f32 32.5 / 25.0,
// bf16 18.6 / 14.4; 1,500 rows (376) 97.9 / 78.4, 47.5 / 39.6; 2 x 1,000 rows
// (512) 76.6 / 72.7, 39.4 / 40.9; 217 rows after 3,800 cached, Q8_0, bf16 104.7 /
// 76.5; six Gemma-2 prompts (528, half of them empty) f32 96.2 / 104.9.
int wave_tiles(const gla_ctx *ctx, const PrefillParams &prm, int n_units) {
    return 2 * (int64_t)n_units * wg_blocks(prm, 2) <= 3 * (int64_t)ctx->n_cu ? 1 : 2;
}

template <int D, bool CAP>
void launch_bf16s(gla_ctx *ctx, PrefillParams prm, int n_units, const uint8_t *img, int n_tiles) {
    const int nt = wave_tiles(ctx, prm, n_units);
    prm.n_qblocks = wg_blocks(prm, nt);
    const dim3 grid(n_units, prm.n_qblocks), block(kBf16sWaves<D> * 64);
    if (nt == 1)
        hipLaunchKernelGGL((prefill_bf16s_kernel<D, CAP, 1>), grid, block, 0, ctx->stream, prm, img, n_tiles);
    else
        hipLaunchKernelGGL((prefill_bf16s_kernel<D, CAP, 2>), grid, block, 0, ctx->stream, prm, img, n_tiles);
}

template <int D, bool Q8>
int launch_bf16_staged(gla_ctx *ctx, const PrefillParams &prm, int n_units, int n_seqs, uint8_t *img, int n_tiles) {
    hipLaunchKernelGGL((stage_bf16_kernel<D, Q8>), dim3(n_tiles, prm.n_kv_heads, n_seqs), dim3(256), 0, ctx->stream,
                       prm, img, n_tiles);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(GLA_ERR_KERNEL, "stage_bf16_kernel launch: %s", hipGetErrorString(e));
    if (prm.softcap > 0.0f)
        launch_bf16s<D, true>(ctx, prm, n_units, img, n_tiles);
    else
        launch_bf16s<D, false>(ctx, prm, n_units, img, n_tiles);
    e = hipGetLastError();
    if (e != hipSuccess) return set_error(GLA_ERR_KERNEL, "prefill_bf16s_kernel launch: %s", hipGetErrorString(e));
    return GLA_OK;
}

template <int D, bool Q8>
int launch_bf16(gla_ctx *ctx, const PrefillParams &prm, dim3 grid) {
    if (prm.softcap > 0.0f)
        hipLaunchKernelGGL((prefill_bf16_kernel<D, Q8, true>), grid, dim3(kBf16Waves<D> * 64), 0, ctx->stream, prm);
    else
        hipLaunchKernelGGL((prefill_bf16_kernel<D, Q8, false>), grid, dim3(kBf16Waves<D> * 64), 0, ctx->stream, prm);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(GLA_ERR_KERNEL, "prefill_bf16_kernel launch: %s", hipGetErrorString(e));
    return GLA_OK;
}

// Bytes of tile images that an fp32 prefill may hold in scratch, and up to which
// it keeps a place for every tile that the storage could have it attend. Above
// that the device numbers the tiles that it does attend, and the host, which
// knows the storage's length but not the contexts, launches the rounds that the
// longest ones would need, up to kRounds; an empty one costs some 5 us. 64 prompts of 200
// rows in a storage of 32,768 positions 234 us, of 200 positions 194.
constexpr size_t kSplitScratch = (size_t)1 << 30, kSplitDirect = (size_t)256 << 20;
constexpr int kRounds = 4;
// Query rows of a call's longest sequence, and tiles of its storage, up to which
// workgroups convert their own tiles: the second launch costs such a call more than
// the repeated conversion. One sequence, us per call, unstaged / staged: from
// position 0, d = 128 20 rows 9.2 / 11.5, 60 rows 12.4 / 13.6, 90 rows 15.5 / 14.5;
// d = 64 20 rows 7.1 / 9.4, 50 rows 9.3 / 10.8; d = 256 20 rows 13.4 / 15.2, 40 rows
// 18.8 / 17.3; after 300 cached positions, d = 128, 20 rows 36 / 22, after 4,000
// 387 / 151.
template <int D>
constexpr int kUnstagedRows = D == 256 ? 32 : 64;
constexpr int kUnstagedTiles = 3;

template <int D, bool Q8, bool CAP, bool STAGED, int NT>
int launch_split_as(gla_ctx *ctx, PrefillParams prm, int n_units, const Images &im) {
    prm.n_qblocks = wg_blocks(prm, NT);
    const int y = std::min(prm.n_qblocks, 65535);
    hipLaunchKernelGGL((prefill_split_kernel<D, Q8, CAP, STAGED, NT>), dim3(n_units, y, (prm.n_qblocks - 1) / y + 1),
                       dim3(256), 0, ctx->stream, prm, im);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(GLA_ERR_KERNEL, "prefill_split_kernel launch: %s", hipGetErrorString(e));
    return GLA_OK;
}

// fp32 prefill: the images of the tiles that its sequences attend, then the
// attention. A call of few rows over a small storage has each workgroup convert
// its own tiles instead (the same bits), and so have the pairs that no round
// takes and a call whose scratch cannot be had (it would have to grow during a
// capture, or the device is full): 4 x 2,048 rows 944 us, 997 rows 105 us.
template <int D, bool Q8, bool CAP>
int launch_split(gla_ctx *ctx, const PrefillParams &prm, int n_seqs, int n_hgrp, int n_tiles) {
    const int n_pairs = n_seqs * prm.n_kv_heads, n_units = n_pairs * n_hgrp;
    // tiles that one sequence can attend
    if (prm.sliding_window > 0)
        n_tiles = (int)std::min<int64_t>(n_tiles, ((int64_t)prm.max_q_len + prm.sliding_window - 2) / KT + 2);
    constexpr size_t per = kSplitImage<D> + sizeof(TileMeta);
    const bool few = prm.max_q_len <= kUnstagedRows<D> && n_tiles <= kUnstagedTiles;
    Images im{};
    im.rounds = 1;
    bool all_placed = true;
    if (!few && n_tiles > 0) {
        const size_t all = (size_t)n_pairs * n_tiles;
        const bool direct = all * per <= kSplitDirect;
        const size_t places = std::min(all, kSplitScratch / per);
        const size_t start_bytes = direct ? 0 : (size_t)n_seqs * sizeof(int64_t);
        void *scr = nullptr;
        if (ensure_scratch(ctx, places * per + start_bytes, &scr) == GLA_OK) {
            im.img = (uint8_t *)scr;
            im.meta = reinterpret_cast<TileMeta *>(im.img + places * kSplitImage<D>);
            im.stride = n_tiles;
            if (!direct) {
                int64_t *start = reinterpret_cast<int64_t *>(im.meta + places);
                im.start = start;
                // (all of them in one round, or a quarter of the places for the last pair's overrun)
                im.over = (int)(places == all ? (size_t)n_tiles : places / 4);
                im.span = (int)(places == all ? all : places - im.over);
                const size_t rounds = (all - 1) / im.span + 1;
                im.rounds = (int)std::min<size_t>(rounds, kRounds);
                all_placed = rounds <= kRounds && n_tiles <= im.over;
                hipLaunchKernelGGL(image_start_kernel, dim3(1), dim3(1024), 0, ctx->stream, prm, n_seqs, start);
                const hipError_t e = hipGetLastError();
                if (e != hipSuccess) return set_error(GLA_ERR_KERNEL, "image_start_kernel launch: %s", hipGetErrorString(e));
            }
        } else {
            clear_error();
            (void)hipGetLastError();
        }
    }
    if (!im.img) return launch_split_as<D, Q8, CAP, false, 1>(ctx, prm, n_units, im);
    // one tile a workgroup, up to some eight workgroups per CU
    const int64_t items = (int64_t)n_tiles * prm.n_kv_heads;
    const int slices = (int)std::min<int64_t>({items, std::max(64, 8 * ctx->n_cu / n_seqs), 65535});
    for (; im.round < im.rounds; im.round++) {
        hipLaunchKernelGGL((stage_split_kernel<D, Q8>), dim3(n_seqs, slices), dim3(256), 0, ctx->stream, prm, im);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return set_error(GLA_ERR_KERNEL, "stage_split_kernel launch: %s", hipGetErrorString(e));
        const int rc = wave_tiles(ctx, prm, n_units) == 1 ? launch_split_as<D, Q8, CAP, true, 1>(ctx, prm, n_units, im)
                                                          : launch_split_as<D, Q8, CAP, true, 2>(ctx, prm, n_units, im);
        if (rc != GLA_OK) return rc;
    }
    return all_placed ? GLA_OK : launch_split_as<D, Q8, CAP, false, 1>(ctx, prm, n_units, im);
}

template <int D>
int launch_f32(gla_ctx *ctx, bool q8, const PrefillParams &prm, int n_seqs, int n_hgrp, int n_tiles) {
    const bool cap = prm.softcap > 0.0f;
    if (q8)
        return cap ? launch_split<D, true, true>(ctx, prm, n_seqs, n_hgrp, n_tiles)
                   : launch_split<D, true, false>(ctx, prm, n_seqs, n_hgrp, n_tiles);
    return cap ? launch_split<D, false, true>(ctx, prm, n_seqs, n_hgrp, n_tiles)
               : launch_split<D, false, false>(ctx, prm, n_seqs, n_hgrp, n_tiles);
}

}  // namespace

int launch_prefill(gla_ctx *ctx, const PrefillLaunch &a) {
    const int D = a.head_dim;
    const int group = a.n_heads / a.n_kv_heads;
    const int hpw = (group % 4 == 0) ? 4 : ((group % 2 == 0) ? 2 : 1);
    if (D != 64 && D != 128 && D != 256) return set_error(GLA_ERR_INVALID, "unsupported head_dim %d", D);
    constexpr int NT = 2;  // 32 queries per wave
    int NW = 4;
    // bf16: the staged path keeps the bf16 tile images of every (sequence, KV
    // head) in scratch, up to 1 GiB, and its staging grid has one z row per
    // sequence (at most 65,535); beyond either each workgroup converts its own
    // tiles (prefill_bf16_kernel, the same bits)
    const int n_tiles = (a.pm.pos_limit + KT - 1) / KT;
    const size_t img_bytes = (size_t)a.n_seqs * a.n_kv_heads * (size_t)n_tiles * (size_t)(128 * D);
    const bool staged = a.precision == GLA_PREC_BF16 && getenv("GLA_BF16_UNSTAGED") == nullptr && n_tiles > 0 &&
                        img_bytes <= ((size_t)1 << 30) && a.n_seqs <= 65535;
    if (a.precision == GLA_PREC_BF16) {
        if (staged)
            NW = D == 64 ? kBf16sWaves<64> : (D == 128 ? kBf16sWaves<128> : kBf16sWaves<256>);
        else
            NW = D == 256 ? kBf16Waves<256> : kBf16Waves<128>;
    }
    const int qwg = 16 * NT * (NW / hpw);
    PrefillParams prm;
    prm.kv = a.kv;
    prm.pm = a.pm;
    prm.q_start = a.q_start;
    prm.pos_offset = a.pos_offset;
    prm.q = a.q;
    prm.out = a.out;
    prm.n_heads = a.n_heads;
    prm.n_kv_heads = a.n_kv_heads;
    prm.group = group;
    prm.hpw = hpw;
    prm.n_qblocks = (a.max_q_len + qwg - 1) / qwg;
    prm.max_q_len = a.max_q_len;
    const bool cap = a.softcap > 0.0f;
    prm.q_mul = cap ? a.scale : a.scale * kLog2e;
    prm.softcap = cap ? a.softcap : 0.0f;
    prm.sliding_window = a.sliding_window;
    if (prm.n_qblocks > 65535) return set_error(GLA_ERR_INVALID, "prefill: %d query blocks > 65535", prm.n_qblocks);
    dim3 grid(a.n_seqs * a.n_kv_heads * (group / hpw), prm.n_qblocks, 1);
    if (a.precision == GLA_PREC_BF16) {
        if (staged) {
            void *scr = nullptr;
            int rc = ensure_scratch(ctx, img_bytes, &scr);
            if (rc != GLA_OK) return rc;
            uint8_t *img = (uint8_t *)scr;
            switch (D) {
            case 64:
                return a.q8 ? launch_bf16_staged<64, true>(ctx, prm, grid.x, a.n_seqs, img, n_tiles)
                            : launch_bf16_staged<64, false>(ctx, prm, grid.x, a.n_seqs, img, n_tiles);
            case 128:
                return a.q8 ? launch_bf16_staged<128, true>(ctx, prm, grid.x, a.n_seqs, img, n_tiles)
                            : launch_bf16_staged<128, false>(ctx, prm, grid.x, a.n_seqs, img, n_tiles);
            default:
                return a.q8 ? launch_bf16_staged<256, true>(ctx, prm, grid.x, a.n_seqs, img, n_tiles)
                            : launch_bf16_staged<256, false>(ctx, prm, grid.x, a.n_seqs, img, n_tiles);
            }
        }
        switch (D) {
        case 64:
            return a.q8 ? launch_bf16<64, true>(ctx, prm, grid) : launch_bf16<64, false>(ctx, prm, grid);
        case 128:
            return a.q8 ? launch_bf16<128, true>(ctx, prm, grid) : launch_bf16<128, false>(ctx, prm, grid);
        default:
            return a.q8 ? launch_bf16<256, true>(ctx, prm, grid) : launch_bf16<256, false>(ctx, prm, grid);
        }
    }
    const int n_hgrp = group / hpw;
    switch (D) {
    case 64:
        return launch_f32<64>(ctx, a.q8, prm, a.n_seqs, n_hgrp, n_tiles);
    case 128:
        return launch_f32<128>(ctx, a.q8, prm, a.n_seqs, n_hgrp, n_tiles);
    default:
        return launch_f32<256>(ctx, a.q8, prm, a.n_seqs, n_hgrp, n_tiles);
    }
}

}  // namespace gla
