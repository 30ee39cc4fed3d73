// gla_prefill.hip -- batched causal prefill attention on MFMA (gfx950).
//
// Math: for every query row, flash_attn_1d_ext over [window_start, pos]
// (src/transformer/forward.rs:927-958, src/tensor/flash.rs:46-124).
//
// Tiling. A workgroup (4 waves) owns a block of query rows of one sequence
// and HPW q-heads that share one KV head; every wave owns 16*NT queries of one
// head. K/V tiles of KT=32 positions are staged in LDS once per workgroup and
// read by all waves (GQA reuse). Per wave and tile, in the f32 body (the f16
// pieces and bf16 take 32-wide MFMAs in the same scheme, below):
//   S^T[key][query] = K . Q^T      v_mfma_f32_16x16x4_f32, Q^T held in VGPRs
//   online softmax per query column (log2 domain)
//   O^T[d][query]  += V^T . P^T    P^T is the S^T accumulator itself: the
//                                  k-step i of a 16-key tile takes keys
//                                  {4j + i}, j = lane / 16, which is exactly
//                                  what accumulator register i holds.
// Permuting the reduction index this way costs nothing and avoids any
// register shuffle between the two products.
#include <math.h>

#include <algorithm>

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
// (sacc[mt][i]: key k0 + 16*mt + 4*lgrp + i), in place, log2 domain. The
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

// One tile's K/V as f32 in registers: thread u of the workgroup holds 16
// consecutive elements (unit u / (D/16) is the key, unit % (D/16) the
// 16-element column block) of K and of V; keys outside [klo, khi] are zero.
template <int D, int NTHR>
struct TileRegs {
    static constexpr int UNITS = KT * D / 16;
    static constexpr int PER_THREAD = (UNITS + NTHR - 1) / NTHR;
    float4 k[PER_THREAD][4];
    float4 v[PER_THREAD][4];
};

template <int D, int NTHR, bool Q8>
__device__ __forceinline__ void fetch_tile(const PrefillParams &p, int b, int kvh, int k0, int klo, int khi,
                                           TileRegs<D, NTHR> &t) {
    const int64_t head_off = (int64_t)kvh * p.kv.head_stride;
#pragma unroll
    for (int j = 0; j < TileRegs<D, NTHR>::PER_THREAD; j++) {
        const int u = threadIdx.x + j * NTHR;
        const int key = u / (D / 16);
        const int c16 = u - key * (D / 16);
        const int kp = k0 + key;
        float kf[16], vf[16];
        if (u < TileRegs<D, NTHR>::UNITS && kp >= klo && kp <= khi) {
            const int64_t pid = map_page(p.pm, b, kp >> 4);
            const int slot = kp & 15;
            if constexpr (Q8) {
                // quants in the decode kernel's MFMA operand order (gla_internal.h)
                const int64_t hb = pid * p.kv.page_stride + head_off;
                const uint2 ka = *reinterpret_cast<const uint2 *>(p.kv.k + hb + q8k_off(slot, c16 * 16, D));
                const uint2 kb = *reinterpret_cast<const uint2 *>(p.kv.k + hb + q8k_off(slot, c16 * 16 + 8, D));
                const uint4 kq = make_uint4(ka.x, ka.y, kb.x, kb.y);
                uint32_t vw4[4] = {0u, 0u, 0u, 0u};
#pragma unroll
                for (int e = 0; e < 16; e++)
                    vw4[e >> 2] |= (uint32_t)p.kv.v[hb + q8v_off(slot, c16 * 16 + e, D)] << ((e & 3) * 8);
                const int blk = (c16 * 16) >> 5;
                const uint16_t *ksp = reinterpret_cast<const uint16_t *>(p.kv.ks + hb) + q8ks_off(slot, blk, D);
                const uint16_t *vsp = reinterpret_cast<const uint16_t *>(p.kv.vs + hb) + slot * (D / 32) + blk;
                const float ksc = __half2float(__ushort_as_half(*ksp));
                const float vsc = __half2float(__ushort_as_half(*vsp));
                const uint32_t kw[4] = {kq.x, kq.y, kq.z, kq.w};
#pragma unroll
                for (int e = 0; e < 16; e++) {  // stored quants are x + 128
                    kf[e] = (float)((int)((kw[e >> 2] >> ((e & 3) * 8)) & 0xff) - 128) * ksc;
                    vf[e] = (float)((int)((vw4[e >> 2] >> ((e & 3) * 8)) & 0xff) - 128) * vsc;
                }
            } else {
                const int64_t base = pid * p.kv.page_stride + head_off + (int64_t)slot * p.kv.row_stride;
                // chunk q of the lane: floats 4*c16 + q*D/4 of the row, so
                // each load and each LDS store instruction covers whole
                // 128-byte runs of a row (16 consecutive floats per lane
                // made the LDS stores conflict)
                const float4 *kp4 = reinterpret_cast<const float4 *>(p.kv.k + base) + c16;
                const float4 *vp4 = reinterpret_cast<const float4 *>(p.kv.v + base) + c16;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    t.k[j][q] = kp4[q * (D / 16)];
                    t.v[j][q] = vp4[q * (D / 16)];
                }
                continue;
            }
#pragma unroll
            for (int q = 0; q < 4; q++) {
                t.k[j][q] = make_float4(kf[4 * q], kf[4 * q + 1], kf[4 * q + 2], kf[4 * q + 3]);
                t.v[j][q] = make_float4(vf[4 * q], vf[4 * q + 1], vf[4 * q + 2], vf[4 * q + 3]);
            }
        } else {
#pragma unroll
            for (int q = 0; q < 4; q++) {
                t.k[j][q] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                t.v[j][q] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            }
        }
    }
}

// K and V rows in LDS: D floats + 4 of padding, so the 16 rows a 16-lane
// group reads with 16-byte loads start in distinct bank groups.
template <int D>
constexpr int kRow = D + 4;

template <int D, int NTHR, bool Q8>
__device__ __forceinline__ void store_tile(const TileRegs<D, NTHR> &t, float *Ks, float *Vs) {
#pragma unroll
    for (int j = 0; j < TileRegs<D, NTHR>::PER_THREAD; j++) {
        const int u = threadIdx.x + j * NTHR;
        if (u >= TileRegs<D, NTHR>::UNITS) break;
        const int key = u / (D / 16);
        const int c16 = u - key * (D / 16);
        // chunk q: floats 16*c16 + 4*q of the row (Q8) or 4*c16 + q*D/4 (f32)
        float4 *kd = reinterpret_cast<float4 *>(Ks + key * kRow<D> + (Q8 ? c16 * 16 : c16 * 4));
        float4 *vd = reinterpret_cast<float4 *>(Vs + key * kRow<D> + (Q8 ? c16 * 16 : c16 * 4));
#pragma unroll
        for (int q = 0; q < 4; q++) {
            kd[Q8 ? q : q * (D / 16)] = t.k[j][q];
            vd[Q8 ? q : q * (D / 16)] = t.v[j][q];
        }
    }
}

// Workgroup: NW waves; a wave owns 16*NT queries of one q-head, the HPW
// heads of the workgroup share one KV head (NW / HPW waves per head). K/V tiles of KT keys are
// double-buffered in LDS: the next tile is fetched into registers while the
// current one is multiplied, then stored to the other buffer, with one
// barrier per tile.
// Reduction order. Lane group g (lanes 16g..16g+15) covers the head
// dimensions [g*D/4, (g+1)*D/4): k-step s of S^T = K.Q^T multiplies d =
// g*D/4 + s, so a lane reads its K operands four at a time from one row.
// O^T row R of d-tile t is d = R*DT + t, so the V^T operands a lane needs
// for one key are DT consecutive floats, and a lane's outputs for a query
// are the 4*DT consecutive floats [4g*DT, 4(g+1)*DT).
template <int D>
constexpr int kF32Lds = 4 * KT * kRow<D> * 4;  // two K and two V tiles

template <int D, int NT, int NW, bool Q8, bool CAP>
__device__ __forceinline__ void prefill_f32_body(const PrefillParams &p, uint8_t *lds, int unit, int qb0) {
    constexpr int NTHR = NW * 64;
    constexpr int QW = 16 * NT;  // queries per wave
    constexpr int KS = D / 4;    // k-steps of S = K Q^T
    constexpr int DT = D / 16;   // d tiles of O
    float *Kb = reinterpret_cast<float *>(lds);
    float *Vb = Kb + 2 * KT * kRow<D>;

    const int n_hgrp = p.group / p.hpw;
    const int b = unit / (p.n_kv_heads * n_hgrp);
    const int kvh = (unit - b * p.n_kv_heads * n_hgrp) / n_hgrp;
    const int hgrp = unit - (b * p.n_kv_heads + kvh) * n_hgrp;
    const int waves_per_head = NW / p.hpw;
    const int qwg = QW * waves_per_head;

    const int row0 = p.q_start[b];
    const int q_len = min(max(p.q_start[b + 1] - row0, 0), p.max_q_len);
    const int pos0 = p.pos_offset[b];
    if (qb0 >= q_len) return;  // qb0: first local query

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int lrow = lane & 15;
    const int lgrp = lane >> 4;
    const int head = kvh * p.group + hgrp * p.hpw + (wave % p.hpw);
    const int wq0 = qb0 + (wave / p.hpw) * QW;  // first local query of this wave

    // key range of the workgroup
    const int q_last = min(q_len, qb0 + qwg) - 1;
    const int khi = min(pos0 + q_last, p.pm.pos_limit - 1);
    const int klo = window_lo(pos0 + qb0, p.sliding_window);

    // Q^T fragments: qf[nt][s] = Q[query nt*16 + lrow][d = lgrp*KS + s]
    float qf[NT][KS];
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
        const int lq = wq0 + nt * 16 + lrow;
        const bool ok = lq < q_len;
        const float4 *qp = reinterpret_cast<const float4 *>(
            p.q + ((int64_t)(row0 + (ok ? lq : 0)) * p.n_heads + head) * D + lgrp * KS);
#pragma unroll
        for (int s4 = 0; s4 < KS / 4; s4++) {
            const float4 v = qp[s4];
            qf[nt][4 * s4 + 0] = ok ? v.x * p.q_mul : 0.0f;
            qf[nt][4 * s4 + 1] = ok ? v.y * p.q_mul : 0.0f;
            qf[nt][4 * s4 + 2] = ok ? v.z * p.q_mul : 0.0f;
            qf[nt][4 * s4 + 3] = ok ? v.w * p.q_mul : 0.0f;
        }
    }

    floatx4 o[DT][NT];
#pragma unroll
    for (int t = 0; t < DT; t++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++) o[t][nt] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    float m[NT], lpart[NT];
    int qpos[NT], qlo[NT];
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
        m[nt] = -INFINITY;
        lpart[nt] = 0.0f;
        const int lq = wq0 + nt * 16 + lrow;
        qpos[nt] = lq < q_len ? pos0 + lq : -1;  // -1: padding query, every key masked
        qlo[nt] = window_lo(pos0 + lq, p.sliding_window);
    }

    if (khi >= klo) {
        const int kfirst = (klo / KT) * KT;
        TileRegs<D, NTHR> tr;
        fetch_tile<D, NTHR, Q8>(p, b, kvh, kfirst, klo, khi, tr);
        store_tile<D, NTHR, Q8>(tr, Kb, Vb);
        __syncthreads();
        int buf = 0;
        for (int k0 = kfirst; k0 <= khi; k0 += KT, buf ^= 1) {
            const bool more = k0 + KT <= khi;
            if (more) fetch_tile<D, NTHR, Q8>(p, b, kvh, k0 + KT, klo, khi, tr);
            const float *ks = Kb + buf * KT * kRow<D>;
            const float *vs = Vb + buf * KT * kRow<D>;

            // S^T = K . Q^T
            floatx4 sacc[2][NT];
#pragma unroll
            for (int mt = 0; mt < 2; mt++)
#pragma unroll
                for (int nt = 0; nt < NT; nt++) sacc[mt][nt] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int s4 = 0; s4 < KS / 4; s4++) {
                float av[2][4];
#pragma unroll
                for (int mt = 0; mt < 2; mt++) {
                    const float4 a = *reinterpret_cast<const float4 *>(ks + (mt * 16 + lrow) * kRow<D> + lgrp * KS +
                                                                       4 * s4);
                    av[mt][0] = a.x;
                    av[mt][1] = a.y;
                    av[mt][2] = a.z;
                    av[mt][3] = a.w;
                }
                // the 2*NT accumulators in turn: a dependent MFMA every 2*NT issues
#pragma unroll
                for (int e = 0; e < 4; e++)
#pragma unroll
                    for (int mt = 0; mt < 2; mt++)
#pragma unroll
                        for (int nt = 0; nt < NT; nt++)
                            sacc[mt][nt] =
                                __builtin_amdgcn_mfma_f32_16x16x4f32(av[mt][e], qf[nt][4 * s4 + e], sacc[mt][nt], 0, 0, 0);
            }

            // online softmax over this tile, per query column. Only tiles that
            // cross the diagonal, a window edge or the key range need the mask.
            const bool interior = k0 >= klo && k0 + KT - 1 <= min(khi, pos0 + wq0) &&
                                  (p.sliding_window <= 0 || k0 >= window_lo(pos0 + wq0 + QW - 1, p.sliding_window));
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                floatx4 col[2] = {sacc[0][nt], sacc[1][nt]};
                cap_and_mask<CAP>(col, p.softcap, interior, k0 + 4 * lgrp, qpos[nt], qlo[nt], klo, khi);
                sacc[0][nt] = col[0];
                sacc[1][nt] = col[1];
                float mx = -INFINITY;
#pragma unroll
                for (int mt = 0; mt < 2; mt++)
#pragma unroll
                    for (int i = 0; i < 4; i++) mx = fmaxf(mx, sacc[mt][nt][i]);
                mx = max_rows4(mx);
                const float m_new = fmaxf(m[nt], mx);
                if (m_new == -INFINITY) {
#pragma unroll
                    for (int mt = 0; mt < 2; mt++)
#pragma unroll
                        for (int i = 0; i < 4; i++) sacc[mt][nt][i] = 0.0f;
                    continue;
                }
                const float rs = fast_exp2(m[nt] - m_new);
                m[nt] = m_new;
                float ls = 0.0f;
#pragma unroll
                for (int mt = 0; mt < 2; mt++)
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const float pv = fast_exp2(sacc[mt][nt][i] - m_new);
                        sacc[mt][nt][i] = pv;
                        ls += pv;
                    }
                lpart[nt] = lpart[nt] * rs + ls;
                if (__ballot(rs != 1.0f)) {  // the running max moved for some query
#pragma unroll
                    for (int t = 0; t < DT; t++) o[t][nt] *= rs;
                }
            }

            // O^T += V^T . P^T
#pragma unroll
            for (int mt = 0; mt < 2; mt++) {
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float *vrow = vs + (mt * 16 + 4 * lgrp + i) * kRow<D> + lrow * DT;
                    float av[DT];
#pragma unroll
                    for (int t4 = 0; t4 < DT / 4; t4++) {
                        const float4 a = reinterpret_cast<const float4 *>(vrow)[t4];
                        av[4 * t4] = a.x;
                        av[4 * t4 + 1] = a.y;
                        av[4 * t4 + 2] = a.z;
                        av[4 * t4 + 3] = a.w;
                    }
#pragma unroll
                    for (int t = 0; t < DT; t++)
#pragma unroll
                        for (int nt = 0; nt < NT; nt++)
                            o[t][nt] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[t], sacc[mt][nt][i], o[t][nt], 0, 0, 0);
                }
            }

            if (more) store_tile<D, NTHR, Q8>(tr, Kb + (buf ^ 1) * KT * kRow<D>, Vb + (buf ^ 1) * KT * kRow<D>);
            __syncthreads();
        }
    }

    // normalise and store: lane holds O^T[d = (4*lgrp + r)*DT + t][query lrow]
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
        float lt = lpart[nt];
        lt = sum_rows4(lt);
        const int lq = wq0 + nt * 16 + lrow;
        if (lq >= q_len) continue;
        const float inv = lt > 0.0f ? 1.0f / lt : 0.0f;
        float *op = p.out + ((int64_t)(row0 + lq) * p.n_heads + head) * D + 4 * lgrp * DT;
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int t4 = 0; t4 < DT / 4; t4++)
                *reinterpret_cast<float4 *>(op + r * DT + 4 * t4) =
                    make_float4(o[4 * t4][nt][r] * inv, o[4 * t4 + 1][nt][r] * inv, o[4 * t4 + 2][nt][r] * inv,
                                o[4 * t4 + 3][nt][r] * inv);
    }
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

// 16 bytes per lane from sbase + voff into LDS at m0 + 16*lane (m0 restored).
// Default (cached) loads: each tile image is read by every query block of
// its unit. The s_nop is the wait state an LDS-DMA load needs after an SALU
// write of M0, which the compiler cannot insert into inline assembly.
__device__ __forceinline__ void lds_copy16(const uint8_t *sbase, uint32_t voff, uint32_t m0) {
    uint32_t save;
    asm volatile(
        "s_mov_b32 %0, m0\n\t"
        "s_mov_b32 m0, %3\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dwordx4 %1, %2\n\t"
        "s_mov_b32 m0, %0"
        : "=&s"(save)
        : "v"(voff), "s"(sbase), "s"(m0)
        : "memory");
}

template <int N>
__device__ __forceinline__ void wait_vm() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
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

    const int q_last = min(q_len, qb0 + qwg) - 1;
    const int khi = min(pos0 + q_last, p.pm.pos_limit - 1);
    const int klo = window_lo(pos0 + qb0, p.sliding_window);

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
    // keys this wave's queries attend: [wlo, whi]
    const int whi = min(khi, pos0 + wq0 + QW - 1);
    const int wlo = max(klo, window_lo(pos0 + wq0, p.sliding_window));

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
// (hi = f16(x), lo = f16(x - hi): 22 bits) after a power-of-two scaling, and a
// product is three MFMAs, hi.hi + hi.lo + lo.hi; the dropped lo.lo is 2^-24 of
// the product. Products of f16 pieces are exact in the f32 accumulators, and a
// 32-wide MFMA rounds once where the 4-wide f32 one rounds eight times, so the
// error against 64 bits does not grow: 4 prompts of 2,048 at 32/8 heads, d =
// 128, have a relative error of 2.7e-7 (f32 MFMAs: 4.4e-7). Three f16 MFMAs do
// the work of a 16x16x32 tile in 48 cycles, the f32 ones in 256: the same four
// prompts take 375 us, of them 23 the staging (f32 MFMAs: 1,083 us), 367
// TFLOP/s. What bounds it is the chain S -> softmax -> O at two waves per SIMD:
// a tile takes a workgroup 2.2 us and its MFMAs 0.65 us of each wave's SIMD.
//
// Scaling. K takes one power of two per 32-key tile, undone on the scores (with
// the query's own); V one per tile as well, which is the unit O is accumulated
// in: when it changes, O is moved to the new unit (an exact product). The
// exponents are rounded up to multiples of 4, so tiles of like magnitude share
// a unit. p = 2^(s - m) is held below 2^14 (kSplitP).
//
// What the pieces cannot carry at f32 precision goes through the f32 body
// above, decided per workgroup: a tile that holds an infinity or a NaN, whose
// largest value lies outside [2^-45, 2^45] (K) or [2^-20, 2^20] (V), or whose
// values differ too much in magnitude (kSplitRange), and a query row with a
// non-finite value or a maximum outside [2^-45, 2^45]. A value x of a tile whose
// largest is M has an error of at most max(2^-23 |x|, 2^-35 M).
typedef _Float16 half8p __attribute__((ext_vector_type(8)));

constexpr int kSplitP = 6;            // p is scaled by 2^6: with the lazy maximum's 2^8 it stays below 2^14
// How much smaller than a tile's largest value that of 8 dims of a key (K) or
// of 8 keys of a dim (V) may be: 2^12; in a tile that is not full 2^20, since
// there a V run may hold one key, whose value is small by chance.
constexpr float kSplitRange = 0x1p12f, kSplitRangePart = 0x1p20f;

// A tile's image: K hi, K lo, V hi, V lo, each 64*D bytes in the piece order
// of the bf16 image.
template <int D>
constexpr int kSplitImage = 256 * D;
// What the attention needs to know of a tile: the factor that undoes K's
// scale (NaN: the tile takes the f32 body), and V's scale (0: V is all zero).
struct TileMeta {
    float k_inv, v_scale;
};

__device__ __forceinline__ void split8(const float (&x)[8], float mul, half8p &hi, half8p &lo) {
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const float t = x[j] * mul;
        const _Float16 h = (_Float16)t;
        hi[j] = h;
        lo[j] = (_Float16)(t - (float)h);
    }
}

// 2^(14 - e) for the exponent e of m (m in [2^(e-1), 2^e)), e rounded up to a
// multiple of STEP: m times it lies in [2^(14-STEP), 2^14).
template <int STEP>
__device__ __forceinline__ int split_exponent(float m) {
    int e = (int)((__float_as_uint(m) >> 23) & 0xff) - 126;
    e = (e + STEP - 1) & ~(STEP - 1);
    return 14 - e;
}
__device__ __forceinline__ float pow2f(int e) { return __uint_as_float((uint32_t)(e + 127) << 23); }

// One 32-key tile of a (sequence, KV head) pair on its way from the cache to
// its pieces, by 256 threads: fetch() issues the loads, convert() finds the
// tile's scales and hands out the pieces.
// K piece i is 8 consecutive dims of one key, V piece i 8 keys of one dim.
template <int D>
__device__ __forceinline__ int k_piece_key(int i) { return i / (D / 8 * 16) * 16 + (i & 15); }
template <int D>
__device__ __forceinline__ int k_piece_dim(int i) { return (i % (D / 8 * 16) >> 4) * 8; }
__device__ __forceinline__ int v_piece_key(int i, int j) { return (j >> 2) * 16 + 4 * ((i >> 4) & 3) + (j & 3); }
__device__ __forceinline__ int v_piece_dim(int i) { return 16 * (i >> 6) + (i & 15); }

// What convert() needs in LDS.
template <int D, bool Q8>
struct SplitAux {
    uint4 ext[4];  // per wave, as bits: largest |K|, smallest non-zero run maximum of K; the same of V
    TileMeta meta;
    uint32_t pad[2];
    float v[Q8 ? 1 : KT][Q8 ? 4 : D + 4];  // f32 rows of V, read back along the keys
};

template <int D, bool Q8>
struct SplitTile {
    static constexpr int NK = 4 * D / 256;  // 16-byte pieces of K (and of V) per thread
    // f32: the rows' own 16-byte loads; Q8_0: quants and scales
    floatx4 ka[Q8 ? 1 : NK][2], va[Q8 ? 1 : NK][2];
    uint2 kw[Q8 ? NK : 1];
    uint32_t vw[Q8 ? NK : 1][2];
    uint16_t ks[Q8 ? NK : 1], vs[Q8 ? NK : 1][8];

    // keys outside [klo, khi] are zero (khi >= 0, and the tile meets the range)
    __device__ __forceinline__ void fetch(const PrefillParams &p, int b, int kvh, int k0, int klo, int khi) {
        const int64_t head_off = (int64_t)kvh * p.kv.head_stride;
        const int64_t hb0 = map_page(p.pm, b, min(k0, khi) >> 4) * p.kv.page_stride + head_off;
        const int64_t hb1 = map_page(p.pm, b, min(k0 + 16, khi) >> 4) * p.kv.page_stride + head_off;
        if constexpr (Q8) {
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
                const int i = threadIdx.x + 256 * r;
                const int key = k_piece_key<D>(i);
                const int kp = k0 + key;
                ka[r][0] = ka[r][1] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
                if (kp >= klo && kp <= khi) {
                    const float *kr = reinterpret_cast<const float *>(p.kv.k + (key < 16 ? hb0 : hb1) +
                                                                      (int64_t)(kp & 15) * p.kv.row_stride) +
                                      k_piece_dim<D>(i);
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

    // put(i, k_hi, k_lo, v_hi, v_lo) takes piece i of each image, unless the
    // pieces cannot carry the tile (aux.meta.k_inv is NaN). No thread may
    // still be reading aux; after the next barrier aux.meta may be read.
    template <typename Put>
    __device__ __forceinline__ void convert(SplitAux<D, Q8> &aux, int k0, int klo, int khi, Put put) const {
        float kf[NK][8], vf[NK][8];
        if constexpr (!Q8) {
#pragma unroll
            for (int r = 0; r < NK; r++) {
                const int u = threadIdx.x + 256 * r;
                const int key = u / (D / 8);
                floatx4 *dst = reinterpret_cast<floatx4 *>(&aux.v[key][8 * (u - key * (D / 8))]);
                dst[0] = va[r][0];
                dst[1] = va[r][1];
            }
            __syncthreads();
        }
        if constexpr (Q8) {
            dequantize(k0, klo, khi, kf, vf);
        } else {
#pragma unroll
            for (int r = 0; r < NK; r++) {
                const int i = threadIdx.x + 256 * r;
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    kf[r][j] = ka[r][j >> 2][j & 3];
                    vf[r][j] = aux.v[v_piece_key(i, j)][v_piece_dim(i)];
                }
            }
        }
        // magnitudes, as the bits of |x| (an infinity or a NaN is the largest)
        uint32_t ktop = 0, klow = 0xffffffffu, vtop = 0, vlow = 0xffffffffu;
#pragma unroll
        for (int r = 0; r < NK; r++) {
            uint32_t km = 0, vm = 0;
#pragma unroll
            for (int j = 0; j < 8; j++) {
                km = max(km, __float_as_uint(kf[r][j]) & 0x7fffffffu);
                vm = max(vm, __float_as_uint(vf[r][j]) & 0x7fffffffu);
            }
            ktop = max(ktop, km);
            klow = min(klow, km ? km : 0xffffffffu);
            vtop = max(vtop, vm);
            vlow = min(vlow, vm ? vm : 0xffffffffu);
        }
        const uint4 mine = make_uint4(wave_extreme<true>(ktop), wave_extreme<false>(klow), wave_extreme<true>(vtop),
                                      wave_extreme<false>(vlow));
        if ((threadIdx.x & 63) == 0) aux.ext[threadIdx.x >> 6] = mine;
        __syncthreads();
#pragma unroll
        for (int w = 0; w < 4; w++) {
            const uint4 x = aux.ext[w];
            ktop = max(w ? ktop : 0, x.x);
            klow = min(w ? klow : 0xffffffffu, x.y);
            vtop = max(w ? vtop : 0, x.z);
            vlow = min(w ? vlow : 0xffffffffu, x.w);
        }
        const float kmax = __uint_as_float(ktop), vmax = __uint_as_float(vtop);
        const float range = k0 >= klo && k0 + KT - 1 <= khi ? kSplitRange : kSplitRangePart;
        bool plain = ktop < 0x7f800000u && vtop < 0x7f800000u;
        int ke = 0, ve = 0;
        if (plain && ktop) {
            plain = kmax >= 0x1p-45f && kmax <= 0x1p45f && __uint_as_float(klow) * range >= kmax;
            ke = split_exponent<4>(kmax);
        }
        if (plain && vtop) {
            plain = vmax >= 0x1p-20f && vmax <= 0x1p20f && __uint_as_float(vlow) * range >= vmax;
            ve = split_exponent<4>(vmax);
        }
        if (threadIdx.x == 0)
            aux.meta = TileMeta{plain ? pow2f(-ke) : __uint_as_float(0x7fc00000u), vtop ? pow2f(ve) : 0.0f};
        if (!plain) return;
        const float kmul = pow2f(ke), vmul = pow2f(ve);
#pragma unroll
        for (int r = 0; r < NK; r++) {
            half8p kh, kl, vh, vl;
            split8(kf[r], kmul, kh, kl);
            split8(vf[r], vmul, vh, vl);
            put(threadIdx.x + 256 * r, kh, kl, vh, vl);
        }
    }
};

// Grid (tile, (sequence, KV head) pair), 256 threads.
template <int D, bool Q8>
__global__ __launch_bounds__(256) void stage_split_kernel(const PrefillParams p, uint8_t *img, TileMeta *meta,
                                                          int n_tiles, int pair0) {
    const int t = blockIdx.x;
    const int pair = pair0 + blockIdx.y;
    const int b = pair / p.n_kv_heads;
    const int kvh = pair - b * p.n_kv_heads;
    const int row0 = p.q_start[b];
    const int q_len = min(max(p.q_start[b + 1] - row0, 0), p.max_q_len);
    if (q_len == 0) return;
    const int pos0 = p.pos_offset[b];
    const int khi = min(pos0 + q_len - 1, p.pm.pos_limit - 1);
    const int klo = window_lo(pos0, p.sliding_window);
    const int k0 = t * KT;
    if (khi < klo || k0 > khi || k0 + KT - 1 < klo) return;  // a tile no query of the sequence reads

    __shared__ __attribute__((aligned(16))) SplitAux<D, Q8> aux;
    SplitTile<D, Q8> tile;
    tile.fetch(p, b, kvh, k0, klo, khi);
    const int64_t at = (int64_t)blockIdx.y * n_tiles + t;
    uint8_t *dst = img + at * kSplitImage<D>;
    tile.convert(aux, k0, klo, khi, [&](int i, const half8p &kh, const half8p &kl, const half8p &vh, const half8p &vl) {
        *reinterpret_cast<half8p *>(dst + (int64_t)i * 16) = kh;
        *reinterpret_cast<half8p *>(dst + 64 * D + (int64_t)i * 16) = kl;
        *reinterpret_cast<half8p *>(dst + 128 * D + (int64_t)i * 16) = vh;
        *reinterpret_cast<half8p *>(dst + 192 * D + (int64_t)i * 16) = vl;
    });
    if (threadIdx.x == 0) meta[at] = aux.meta;
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
// a workgroup (or the f32 body's buffers): d = 64 35 KB, d = 128 68 KB,
// d = 256 133 KB. A workgroup that converts its own tiles holds one image and
// the conversion's buffers, and the next tile's loads in registers (not at
// d = 256, whose registers are full).
template <int D, bool STAGED>
constexpr int kSplitOccupancy = !STAGED ? (D == 64 ? 2 : 1) : (D == 64 ? 3 : (D == 128 ? 2 : 1));

template <int D, bool Q8, bool CAP, bool STAGED, int NT>
__global__ __launch_bounds__(256, (kSplitOccupancy<D, STAGED>)) void prefill_split_kernel(const PrefillParams p,
                                                                                const uint8_t *img,
                                                                                const TileMeta *meta, int n_tiles,
                                                                                int pair0) {
    constexpr int NW = 4;
    constexpr int QW = 16 * NT;
    constexpr int KS = D / 32;
    constexpr int DT = D / 16;
    constexpr int IMG = kSplitImage<D>;
    constexpr int CPW = IMG / 1024 / NW;  // kilobyte copies per wave and tile
    constexpr int AUX = IMG + (int)sizeof(SplitAux<D, Q8>);
    constexpr int LDS = std::max(kF32Lds<D>, STAGED ? 2 * IMG : AUX);
    __shared__ __attribute__((aligned(16))) uint8_t lds[LDS];

    const int n_hgrp = p.group / p.hpw;
    const int unit = pair0 * n_hgrp + (int)blockIdx.x;
    const int pair = unit / n_hgrp;
    const int b = pair / p.n_kv_heads;
    const int kvh = pair - b * p.n_kv_heads;
    const int hgrp = unit - pair * n_hgrp;
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

    const int q_last = min(q_len, qb0 + qwg) - 1;
    const int khi = min(pos0 + q_last, p.pm.pos_limit - 1);
    const int klo = window_lo(pos0 + qb0, p.sliding_window);
    const int tfirst = klo / KT;
    const int n = khi >= klo ? khi / KT - tfirst + 1 : 0;
    const TileMeta *unit_meta = meta + (int64_t)(pair - pair0) * n_tiles + tfirst;
    const uint8_t *unit_img = img + ((int64_t)(pair - pair0) * n_tiles + tfirst) * IMG;
    const uint32_t ring = __builtin_amdgcn_readfirstlane(
        (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void *)&lds[0]);
    auto issue = [&](int i) {
        const uint8_t *src = unit_img + (int64_t)i * IMG;
        const uint32_t dst = ring + (uint32_t)((i & 1) * IMG);
#pragma unroll
        for (int c = 0; c < CPW; c++) {
            const int piece = wave * CPW + c;
            lds_copy16(src, (uint32_t)(piece * 1024 + lane * 16), dst + piece * 1024);
        }
    };

    if (STAGED && n > 0) issue(0);
    // tiles and queries that the pieces cannot carry
    bool odd = false;
    for (int i = tid; STAGED && i < n; i += 256) odd = odd || unit_meta[i].k_inv != unit_meta[i].k_inv;

    // Q^T operand: pieces of Q[query nt*16 + lrow][d = ks*32 + lgrp*8 + 0..7]
    // times the query's own power of two
    half8p qh[NT][KS], ql[NT][KS];
    float qinv[NT];
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
        const int lq = wq0 + nt * 16 + lrow;
        const bool ok = lq < q_len;
        const float *qp = p.q + ((int64_t)(row0 + (ok ? lq : 0)) * p.n_heads + head) * D;
        float x[KS][8];
        uint32_t mx = 0;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const floatx4 a = __builtin_nontemporal_load(reinterpret_cast<const floatx4 *>(qp + ks * 32 + lgrp * 8));
            const floatx4 c = __builtin_nontemporal_load(reinterpret_cast<const floatx4 *>(qp + ks * 32 + lgrp * 8 + 4));
#pragma unroll
            for (int j = 0; j < 8; j++) x[ks][j] = ok ? (j < 4 ? a[j & 3] : c[j & 3]) * p.q_mul : 0.0f;
        }
#pragma unroll
        for (int ks = 0; ks < KS; ks++)
#pragma unroll
            for (int j = 0; j < 8; j++) mx = max(mx, __float_as_uint(x[ks][j]) & 0x7fffffffu);
        mx = umax_rows4(mx);
        const float top = __uint_as_float(mx);
        const bool fits = mx == 0 || (top >= 0x1p-45f && top <= 0x1p45f);  // false for an infinity or a NaN
        odd = odd || !fits;
        const int e = mx && fits ? split_exponent<1>(top) : 0;
        qinv[nt] = pow2f(-e);
#pragma unroll
        for (int ks = 0; ks < KS; ks++) split8(x[ks], pow2f(e), qh[nt][ks], ql[nt][ks]);
    }
    if (STAGED) wait_vm<0>();  // the first tile has landed, so the f32 body may use its place
    const auto in_f32 = [&]() {
        constexpr int FT = D == 256 ? 1 : NT;  // d = 256: half a wave's queries at a time, more would spill
        for (int q = qb0; q < qb0 + qwg; q += 16 * FT * waves_per_head) {
            __syncthreads();  // the LDS is free
            prefill_f32_body<D, FT, NW, Q8, CAP>(p, lds, unit, q);
        }
    };
    bool f32 = __syncthreads_or(odd);
    if (STAGED && f32) {
        in_f32();
        return;
    }

    floatx4 o[DT][NT];
    float m[NT], lpart[NT];
    int qpos[NT], qlo[NT];
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
#pragma unroll
        for (int t = 0; t < DT; t++) o[t][nt] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
        lpart[nt] = 0.0f;
        m[nt] = kMInit;
        const int lq = wq0 + nt * 16 + lrow;
        qpos[nt] = lq < q_len ? pos0 + lq : -1;
        qlo[nt] = window_lo(pos0 + lq, p.sliding_window);
    }
    // keys this wave's queries attend: [wlo, whi]
    const int whi = min(khi, pos0 + wq0 + QW - 1);
    const int wlo = max(klo, window_lo(pos0 + wq0, p.sliding_window));
    float unit_v = 0.0f;  // O's unit: the scale of the last tile's V (0: none yet)

    auto attend = [&](int i, const uint8_t *kimg, const TileMeta &cur) {
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

        // softmax: as the bf16 kernels' (a lazy maximum), in f32; c undoes the scales
        const bool interior = k0 >= klo && k0 + KT - 1 <= min(khi, pos0 + wq0) &&
                              (p.sliding_window <= 0 || k0 >= window_lo(pos0 + wq0 + QW - 1, p.sliding_window));
        half8p ph[NT], pl[NT];
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
            float c = cur.k_inv * qinv[nt];
            floatx4 col[2] = {s[0][nt] + x[0][nt], s[1][nt] + x[1][nt]};
            if constexpr (CAP) {
                col[0] *= c;
                col[1] *= c;
                c = 1.0f;
            }
            cap_and_mask<CAP>(col, p.softcap, interior, k0 + 4 * lgrp, qpos[nt], qlo[nt], klo, khi);
            float mx = max3f(max3f(col[0][0], col[0][1], col[0][2]), max3f(col[0][3], col[1][0], col[1][1]),
                             max2f(col[1][2], col[1][3])) * c;
            if (__ballot(mx - m[nt] > kLazyMax)) {
                mx = max_rows4(mx);
                const bool up = mx - m[nt] > kLazyMax;
                const float rs = up ? fast_exp2(m[nt] - mx) : 1.0f;
                m[nt] = up ? mx : m[nt];
#pragma unroll
                for (int t = 0; t < DT; t++) o[t][nt] *= rs;
                lpart[nt] *= rs;
            }
            const float sub = (float)kSplitP - m[nt];
            float ls = 0.0f;
#pragma unroll
            for (int mt = 0; mt < 2; mt++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const float pv = fast_exp2(fmaf(col[mt][r], c, sub));
                    ls += pv;
                    const _Float16 h = (_Float16)pv;
                    ph[nt][4 * mt + r] = h;
                    pl[nt][4 * mt + r] = (_Float16)(pv - (float)h);
                }
            lpart[nt] += ls;
        }

        // O^T += V^T . P^T in V's unit
        if (cur.v_scale == 0.0f) return;
        if (cur.v_scale != unit_v) {
            const float f = unit_v == 0.0f ? 1.0f : cur.v_scale / unit_v;
#pragma unroll
            for (int t = 0; t < DT; t++)
#pragma unroll
                for (int nt = 0; nt < NT; nt++) o[t][nt] *= f;
            unit_v = cur.v_scale;
        }
        const uint8_t *vimg = kimg + 128 * D;
#pragma unroll
        for (int t = 0; t < DT; t++) {
            const uint8_t *src = vimg + ((t * 4 + lgrp) * 16 + lrow) * 16;
            const half8p ah = *reinterpret_cast<const half8p *>(src);
            const half8p al = *reinterpret_cast<const half8p *>(src + 64 * D);
#pragma unroll
            for (int nt = 0; nt < NT; nt++)
                o[t][nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al, ph[nt], o[t][nt], 0, 0, 0);
#pragma unroll
            for (int nt = 0; nt < NT; nt++)
                o[t][nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, pl[nt], o[t][nt], 0, 0, 0);
#pragma unroll
            for (int nt = 0; nt < NT; nt++)
                o[t][nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, ph[nt], o[t][nt], 0, 0, 0);
        }
    };

    if constexpr (STAGED) {
        TileMeta tm = n > 0 ? unit_meta[0] : TileMeta{1.0f, 0.0f};
        for (int i = 0; i < n; i++) {
            // this wave's copies of tile i have landed, then every wave's; every
            // wave is also done with tile i - 1, whose buffer the next copy takes
            wait_vm<0>();
            __syncthreads();
            if (i + 1 < n) issue(i + 1);
            const TileMeta cur = tm;
            tm = unit_meta[min(i + 1, n - 1)];
            attend(i, lds + (i & 1) * IMG, cur);
        }
    } else if (n > 0 && !f32) {
        SplitAux<D, Q8> &aux = *reinterpret_cast<SplitAux<D, Q8> *>(lds + IMG);
        // the keys that a staged tile would hold: what any query of the sequence attends
        const int ulo = window_lo(pos0, p.sliding_window);
        const int uhi = min(pos0 + q_len - 1, p.pm.pos_limit - 1);
        constexpr bool AHEAD = D < 256;
        SplitTile<D, Q8> tile;
        tile.fetch(p, b, kvh, tfirst * KT, ulo, uhi);
        for (int i = 0; i < n; i++) {
            const int k0 = (tfirst + i) * KT;
            if (!AHEAD && i > 0) tile.fetch(p, b, kvh, k0, ulo, uhi);
            tile.convert(aux, k0, ulo, uhi, [&](int j, const half8p &kh, const half8p &kl, const half8p &vh, const half8p &vl) {
                *reinterpret_cast<half8p *>(lds + j * 16) = kh;
                *reinterpret_cast<half8p *>(lds + 64 * D + j * 16) = kl;
                *reinterpret_cast<half8p *>(lds + 128 * D + j * 16) = vh;
                *reinterpret_cast<half8p *>(lds + 192 * D + j * 16) = vl;
            });
            __syncthreads();
            const TileMeta cur = aux.meta;
            if (cur.k_inv != cur.k_inv) {
                f32 = true;
                break;
            }
            if (AHEAD && i + 1 < n) tile.fetch(p, b, kvh, k0 + KT, ulo, uhi);
            attend(i, lds, cur);
            __syncthreads();  // before the next tile takes its place
        }
    }

    if (!STAGED && f32) {
        in_f32();
        return;
    }

    // Output rows through LDS, as the staged bf16 kernel writes them
    constexpr int SROW = D + 4;
    static_assert(NW * 16 * SROW * 4 <= LDS, "output staging fits");
    __syncthreads();
    float *stage = reinterpret_cast<float *>(lds) + wave * 16 * SROW;
    constexpr int LPR = D / 4;    // lanes per row (16 bytes each)
    constexpr int RPI = 64 / LPR;  // rows per store instruction
    const float unscale = unit_v == 0.0f ? 1.0f : 1.0f / unit_v;
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
        const float lt = sum_rows4(lpart[nt]);
        const float inv = lt > 0.0f ? 1.0f / lt * unscale : 0.0f;
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

// Tile images an fp32 prefill may hold in scratch; a call with more (sequence,
// KV head) pairs runs in several rounds over them.
constexpr size_t kSplitScratch = (size_t)1 << 30;
// Query rows of a call's longest sequence up to which workgroups convert their
// own tiles: the second launch costs a short prompt more than the repeated
// conversion, but each row block converts the whole past again. One sequence,
// us per call, unstaged / staged: from position 0, d = 128 20 rows 7.7 / 12.0,
// 90 rows 12.6 / 16.1, 150 rows 17.8 / 19.7; d = 64 20 rows 5.6 / 9.2, 100 rows
// 11.0 / 13.5; d = 256 with the soft-cap 20 rows 11.4 / 17.3, 100 rows 27.9 /
// 30.6. After 1,000 cached positions, d = 128: 100 rows 93 / 71.
constexpr int kUnstagedRows = 96;

// fp32 prefill: the tile images of as many (sequence, KV head) pairs as the
// scratch takes, then their attention. A call of few query blocks has each
// workgroup convert its own tiles instead (the same bits), and so has one whose
// scratch cannot be had: it would have to grow during a capture, the device is
// full, or one pair's images alone pass the bound.
template <int D, bool Q8, bool CAP>
int launch_split(gla_ctx *ctx, PrefillParams prm, int n_pairs, int n_hgrp, int n_tiles) {
    const size_t per = (size_t)n_tiles * (kSplitImage<D> + sizeof(TileMeta));
    uint8_t *img = nullptr;
    int round = n_pairs;
    if (prm.max_q_len > kUnstagedRows && n_tiles > 0 && per <= kSplitScratch) {
        round = (int)std::min<size_t>({(size_t)n_pairs, kSplitScratch / per, (size_t)65535});
        void *scr = nullptr;
        if (ensure_scratch(ctx, round * per, &scr) == GLA_OK) {
            img = (uint8_t *)scr;
        } else {
            clear_error();
            (void)hipGetLastError();
            round = n_pairs;
        }
    }
    // (the few rows of an unstaged call are spread over the most waves)
    const int nt = img ? wave_tiles(ctx, prm, std::min(round, n_pairs) * n_hgrp) : 1;
    prm.n_qblocks = wg_blocks(prm, nt);
    if (prm.n_qblocks > 65535) return set_error(GLA_ERR_INVALID, "prefill: %d query blocks > 65535", prm.n_qblocks);
    if (!img) {
        hipLaunchKernelGGL((prefill_split_kernel<D, Q8, CAP, false, 1>), dim3(n_pairs * n_hgrp, prm.n_qblocks), dim3(256),
                           0, ctx->stream, prm, (const uint8_t *)nullptr, (const TileMeta *)nullptr, n_tiles, 0);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return set_error(GLA_ERR_KERNEL, "prefill_split_kernel launch: %s", hipGetErrorString(e));
        return GLA_OK;
    }
    TileMeta *meta = reinterpret_cast<TileMeta *>(img + (size_t)round * n_tiles * kSplitImage<D>);
    for (int p0 = 0; p0 < n_pairs; p0 += round) {
        const int np = std::min(round, n_pairs - p0);
        hipLaunchKernelGGL((stage_split_kernel<D, Q8>), dim3(n_tiles, np), dim3(256), 0, ctx->stream, prm, img, meta,
                           n_tiles, p0);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return set_error(GLA_ERR_KERNEL, "stage_split_kernel launch: %s", hipGetErrorString(e));
        const dim3 grid(np * n_hgrp, prm.n_qblocks);
        if (nt == 1)
            hipLaunchKernelGGL((prefill_split_kernel<D, Q8, CAP, true, 1>), grid, dim3(256), 0, ctx->stream, prm,
                               (const uint8_t *)img, (const TileMeta *)meta, n_tiles, p0);
        else
            hipLaunchKernelGGL((prefill_split_kernel<D, Q8, CAP, true, 2>), grid, dim3(256), 0, ctx->stream, prm,
                               (const uint8_t *)img, (const TileMeta *)meta, n_tiles, p0);
        e = hipGetLastError();
        if (e != hipSuccess) return set_error(GLA_ERR_KERNEL, "prefill_split_kernel launch: %s", hipGetErrorString(e));
    }
    return GLA_OK;
}

template <int D>
int launch_f32(gla_ctx *ctx, bool q8, const PrefillParams &prm, int n_pairs, int n_hgrp, int n_tiles) {
    const bool cap = prm.softcap > 0.0f;
    if (q8)
        return cap ? launch_split<D, true, true>(ctx, prm, n_pairs, n_hgrp, n_tiles)
                   : launch_split<D, true, false>(ctx, prm, n_pairs, n_hgrp, n_tiles);
    return cap ? launch_split<D, false, true>(ctx, prm, n_pairs, n_hgrp, n_tiles)
               : launch_split<D, false, false>(ctx, prm, n_pairs, n_hgrp, n_tiles);
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
    const int n_pairs = a.n_seqs * a.n_kv_heads, n_hgrp = group / hpw;
    switch (D) {
    case 64:
        return launch_f32<64>(ctx, a.q8, prm, n_pairs, n_hgrp, n_tiles);
    case 128:
        return launch_f32<128>(ctx, a.q8, prm, n_pairs, n_hgrp, n_tiles);
    default:
        return launch_f32<256>(ctx, a.q8, prm, n_pairs, n_hgrp, n_tiles);
    }
}

}  // namespace gla
