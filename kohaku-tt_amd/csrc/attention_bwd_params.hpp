// Parameters, per-sequence geometry and mask / row-statistics rules shared by the attention
// backward kernels: attention_bwd.hip (host side, row statistics, sums, head dims padded
// past 128) and attention_bwd_tile.hpp (gradient kernels for head dims padded to 128 or
// less, instantiated per padded head dim in attention_bwd_d<D>.hip).
#pragma once

#include "common.hpp"

namespace kmi {
namespace bwd {

constexpr int BWD_THREADS = 256;
constexpr float kLog2e = 1.4426950408889634f;
// A forward lse below this carries the -5e5 offset of a row with no kept key.
constexpr float kRawLse = 0.5f * kMaskedLogit;

struct BwdParams {
    const void *q, *k, *v, *o, *dout;
    const float* lse;
    void *dq, *dk, *dv;
    float* nd;  // [hq][rows_total] fp32 negated row dots -D
    // dK / dV partials [hkv][splits][keys_total][DP] fp32 (splits > 1), else null.
    float *pdk, *pdv;
    // dQ partials [hq][ksplit][rows_total][DP] fp32 (ksplit > 1), else null.
    float* pdq;
    int splits, ksplit;
    int64_t qs[3], ks[3], vs[3], os[3], dos[3], dqs[3], dks[3], dvs[3], ls[3];
    const void* mask;
    int64_t ms[4];
    int64_t mask_numel;
    int mask_mode;
    const int64_t* mask_off;
    const int32_t *cu_q, *cu_k;
    const int32_t* klen;  // dense key lengths [batch] (or null)
    int total_q, total_k;
    int batch, hq, hkv, group, seq_q, seq_k, causal;
    int d, dval;  // q / k and v / out head dims (DP: the larger, padded)
    int64_t rows_total, keys_total;
    float scale, c2;  // c2 = scale * log2(e) (attn_bwd_tile_kernel: never 0)
    // attn_bwd_tile_kernel, unmasked: the score of a key the row does not see (minus infinity
    // with c2's sign).
    float hidden;
};

// One sequence's geometry: query rows [q0, q0 + lq) and keys [k0, k0 + lk) of the packed
// (varlen) tensors, or the whole batch entry (dense); causal: row i sees keys
// j <= i + coff (top-left dense: coff = 0; bottom-right varlen: coff = lk - lq).
struct Geo {
    int q0, lq, k0, lk, coff;
    int64_t row_base, key_base;       // row / key index in [rows_total] / [keys_total]
    int64_t qb, kb, vb, ob, dob, dqb, dkb, dvb, lb;  // batch-entry element offsets (dense)
    int64_t mbase;                    // the mask element of (head 0, row 0, key 0)
    int64_t mrow;                     // mask elements per query row
    int64_t mkey;                     // mask elements per key
    int64_t mend;                     // mask elements (reads at or past it count as masked)
    bool mpacked_ok;                  // packed masks: the sequence's block lies within the mask
};

__device__ __forceinline__ Geo geo_of(const BwdParams& p, int seq) {
    Geo g;
    if (p.cu_q) {
        g.q0 = min(max(p.cu_q[seq], 0), p.total_q);
        g.lq = min(min(max(p.cu_q[seq + 1], g.q0), p.total_q) - g.q0, p.seq_q);
        g.k0 = min(max(p.cu_k[seq], 0), p.total_k);
        g.lk = min(min(max(p.cu_k[seq + 1], g.k0), p.total_k) - g.k0, p.seq_k);
        g.coff = g.lk - g.lq;
        g.row_base = g.q0;
        g.key_base = g.k0;
        g.qb = g.kb = g.vb = g.ob = g.dob = g.dqb = g.dkb = g.dvb = g.lb = 0;
    } else {
        g.q0 = 0;
        g.lq = p.seq_q;
        g.k0 = 0;
        g.lk = p.klen ? min(max(p.klen[seq], 1), p.seq_k) : p.seq_k;
        g.coff = 0;
        g.row_base = static_cast<int64_t>(seq) * p.seq_q;
        g.key_base = static_cast<int64_t>(seq) * p.seq_k;
        g.qb = seq * p.qs[0];
        g.kb = seq * p.ks[0];
        g.vb = seq * p.vs[0];
        g.ob = seq * p.os[0];
        g.dob = seq * p.dos[0];
        g.dqb = seq * p.dqs[0];
        g.dkb = seq * p.dks[0];
        g.dvb = seq * p.dvs[0];
        g.lb = seq * p.ls[0];
    }
    g.mbase = 0;
    g.mrow = 0;
    g.mkey = 0;
    g.mend = INT64_MAX;
    g.mpacked_ok = false;
    if (p.mask_mode == KMI_MASK_PACKED) {
        int64_t off = 0;
        if (p.mask_off) {
            off = p.mask_off[seq];
        } else {
            for (int s = 0; s < seq; ++s) {
                const int a0 = min(max(p.cu_q[s], 0), p.total_q), a1 = min(max(p.cu_q[s + 1], a0), p.total_q);
                const int b0 = min(max(p.cu_k[s], 0), p.total_k), b1 = min(max(p.cu_k[s + 1], b0), p.total_k);
                off += static_cast<int64_t>(a1 - a0) * (b1 - b0);
            }
        }
        g.mbase = off;
        g.mrow = g.lk;
        g.mkey = 1;
        g.mend = p.mask_numel;
        g.mpacked_ok = off + static_cast<int64_t>(g.lq) * g.lk <= p.mask_numel;
    } else if (p.mask_mode == KMI_MASK_STRIDED) {
        g.mbase = p.cu_q ? static_cast<int64_t>(g.q0) * p.ms[2] + static_cast<int64_t>(g.k0) * p.ms[3] : seq * p.ms[0];
        g.mrow = p.ms[2];
        g.mkey = p.ms[3];
    }
    return g;
}

// The mask logit of (head h, row i, key j) of a sequence (0 without a mask).
template <int MK>
__device__ __forceinline__ float mask_at(const BwdParams& p, const Geo& g, int h, int i, int j) {
    if constexpr (MK == MK_NONE) {
        return 0.f;
    } else {
        typedef typename MaskRaw<MK>::type R;
        const int64_t idx = g.mbase + h * p.ms[1] + i * g.mrow + j * g.mkey;
        if (idx >= g.mend) return kMaskedLogit;
        return mask_logit_of<MK>(static_cast<const R*>(p.mask)[idx]);
    }
}

// Row statistics of row i (i < lq): base-2 lse of the row's softmax and whether the row
// ran over its raw scores (no kept key in the forward).  Rows past the end or without
// keys get +inf (P = 0).
__device__ __forceinline__ void row_stats(float lse_nat, bool valid, float& lse2, bool& raw) {
    raw = valid && lse_nat < kRawLse;
    const float l = raw ? lse_nat - kMaskedLogit : lse_nat;
    lse2 = (valid && l != -INFINITY) ? l * kLog2e : INFINITY;
}

// The gradient launch of attention_bwd_tile.hpp: workgroups of each pass.
struct BwdGrid {
    int nq, nk;       // dQ and dK / dV workgroups
    int tiles_q;      // virtual-row tiles of a (sequence, K/V head)
    int half_q, half_k;  // 64 rows (keys) a workgroup, two wavefronts per 32, instead of 128
};

// Enqueues the gradient kernel for element type T and padded head dim DP (instantiated in
// attention_bwd_d<DP>.hip); mk: the mask kind.
template <typename T, int DP>
hipError_t launch_tile(const BwdParams& p, const BwdGrid& gr, int mk, hipStream_t s);

}  // namespace bwd
}  // namespace kmi
