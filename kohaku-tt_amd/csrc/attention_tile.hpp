// Attention forward on 32x32x16 MFMA tiles (gfx950): prefill-sized calls, dense or packed,
// causal or not, GQA, with or without a mask.  attention.hip's plan says which calls.
//
// A 256-thread workgroup owns 128 "virtual rows" of one (sequence, K/V head) (row r is query
// position r / G of query head kvh G + r % G), 32 per wavefront with their Q in registers,
// and walks the keys in tiles of KT: K and V go by LDS DMA into double buffers that the four
// wavefronts share (attn_fwd_kernel's wavefronts split the keys and each load their own).
// S^T = K Q^T leaves one query row per lane and 16 keys in registers, the B operand of
// O^T += V^T P^T as it stands; V^T is a transposed LDS read.  One row per lane also makes
// the softmax state scalar: the row's other half of the keys is in lane + 32.
//
// Unmasked calls are software-pipelined: while tile t's exponentials and PV products run,
// tile t + 1's S products run with them (its K is staged a tile earlier than its V).
// Masked calls hold a tile's mask logits beside its products, add them in one FMA once the
// products are whole and select minus infinity for masked keys (whatever their K row holds),
// skip tiles in which a wavefront keeps no key, and run a second pass over the raw scores only
// for rows that kept none.
#pragma once

#include "attention_params.hpp"
#include "mfma_tile.hpp"

namespace kmi {
namespace fwd {

constexpr float kTileLazy = 8.f;  // log2 units a row max may grow before O is rescaled
// The first tiles a wavefront works on (five with four row groups, three of each of a row's two
// wavefronts with two) set the reference point to their own maximum, also where that is lower
// (by kTileDrop at most): one weight of each is exactly 1 and so carries no rounding.
// attn_fwd_kernel has such a weight per wavefront, and its results' distance from 64-bit ones is
// kept so (relative, attn_fwd_kernel / the first tile alone / as here): 8 packed x 16/8 x 64 to
// 1024 x 128 causal 0.001932 / 0.001981 / 0.001929, 24x4396x128 0.002338 / 0.002343 / 0.002330,
// 16x2048x64 additive 0.002019 / 0.002041 / 0.001997; 1% over it is left where a call has two or
// three tiles.  Costs 1.6% of the masked call (46.2 -> 47.0 us), nothing that shows of the others.
constexpr int tile_own(int rg) { return rg == 4 ? 5 : 3; }
constexpr float kTileDrop = 3.f;
constexpr float kTileLn2 = 0.6931471805599453f;

// Row groups of a workgroup: 4 (128 rows, one wavefront per 32), or 2 (64 rows, two
// wavefronts per 32 that take one half of each key tile and merge their states at the end).
// Keys of a tile: 64, and 128 for two row groups up to head dim 64, so that a wavefront there
// still has 64 (32 past it).  64 KiB of tiles at most up to head dim 128, two workgroups per CU;
// 128 KiB past it, one.
constexpr int tile_keys(int dp, int rg) { return dp <= 64 && rg == 2 ? 128 : 64; }

// Sum of a packed pair of probabilities (as rounded for the PV product) onto acc.
template <typename T>
__device__ __forceinline__ float dot_ones(uint32_t pair, float acc);
template <>
__device__ __forceinline__ float dot_ones<bf16>(uint32_t pair, float acc) {
    typedef __bf16 v2 __attribute__((ext_vector_type(2)));
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(v2, pair), __builtin_bit_cast(v2, 0x3f803f80u), acc, false);
}
template <>
__device__ __forceinline__ float dot_ones<f16>(uint32_t pair, float acc) {
    typedef _Float16 v2 __attribute__((ext_vector_type(2)));
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(v2, pair), __builtin_bit_cast(v2, 0x3c003c00u), acc, false);
}

// The value of the other lane that holds this lane's row (lane ^ 32).
__device__ __forceinline__ float other_half(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float((threadIdx.x & 32) ? r[0] : r[1]);
}

template <typename T, int DP, int MK, int RG>
__device__ __forceinline__ void attn_tile(const AttnParams& p, unsigned char* smem, const int bh, const int xt) {
    constexpr int KP = 4 / RG;                       // wavefronts that share a row group
    constexpr int KT = tile_keys(DP, RG), NB = KT / 32 / KP;  // NB: 32-key blocks of a wavefront
    constexpr int ROWS = 32 * RG;
    constexpr bool MASKED = MK != MK_NONE;
    typedef Tile<T, DP, KT> TL;
    typedef typename TL::v8 v8;
    constexpr int DC = DP / 16, DB = DP / 32;
    constexpr int ES = static_cast<int>(sizeof(T));
    constexpr uint32_t TILE_B = TL::ELEMS * sizeof(T);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int h2 = lane >> 5, l32 = lane & 31;
    const int rg = wave % RG, kp = wave / RG;
    const int seq = fdiv(bh, p.fd_hkv), kvh = bh - seq * p.hkv;
    const int G = p.group;

    int q0 = 0, lq = p.seq_q, k0 = 0, lk = p.seq_k;
    int64_t qb = 0, kb = 0, vb = 0, ob = 0, lb = 0;
    if (p.cu_q) {
        q0 = min(max(p.cu_q[seq], 0), p.total_q);
        lq = min(min(max(p.cu_q[seq + 1], q0), p.total_q) - q0, p.seq_q);
        k0 = min(max(p.cu_k[seq], 0), p.total_k);
        lk = min(min(max(p.cu_k[seq + 1], k0), p.total_k) - k0, p.seq_k);
    } else {
        qb = seq * p.qs[0];
        kb = seq * p.ks[0];
        vb = seq * p.vs[0];
        ob = seq * p.os[0];
        lb = seq * p.ls[0];
        if (p.klen) lk = min(max(p.klen[seq], 1), p.seq_k);
    }
    const int vrows = lq * G;
    const int r0 = xt * ROWS;
    if (r0 >= vrows || lk <= 0) return;  // uniform: no barrier has run
    const int rw0 = r0 + 32 * rg;
    const int row = rw0 + l32;
    const int rr = min(row, vrows - 1);  // rows past the end repeat the last (never written)
    // (Uniform.)  A wavefront whose rows all lie past the end stages its share of the tiles and
    // keeps the barriers, nothing else.
    const bool live = rw0 < vrows;
    const int pos = fdiv(rr, p.fd_group), head = kvh * G + (rr - pos * G);
    const int coff = p.cu_q ? lk - lq : 0;

    // Q fragments (a negative scale flips their sign, so that c2 is positive; a zero one
    // becomes a c2 that finite scores vanish under and minus infinity does not).
    const float c2 = fmaxf(fabsf(p.scale_log2), 1e-30f);
    v8 qf[DC];
    {
        const T* qp = static_cast<const T*>(p.q) + qb + head * p.qs[1] + static_cast<int64_t>(q0 + pos) * p.qs[2];
        const uint32_t flip = p.scale_log2 < 0.f ? 0x80008000u : 0u;
#pragma unroll
        for (int c = 0; c < DC; ++c) {
            const int col = 16 * c + 8 * h2;
            const u32x4 x = *reinterpret_cast<const u32x4*>(qp + min(col, p.d - 8)) ^ flip;
            qf[c] = __builtin_bit_cast(v8, col < p.d ? x : u32x4{0u, 0u, 0u, 0u});
        }
    }
    // Causal: keys below lim are visible to this row; those below lim_w to every row of the
    // wavefront; none at or past kend to any row of the workgroup.
    const int lim = p.causal ? max(0, min(lk, pos + 1 + coff)) : lk;
    const int lim_w = p.causal ? min(lk, fdiv(min(rw0, vrows - 1), p.fd_group) + 1 + coff) : lk;
    const int kend = p.causal ? max(0, min(lk, fdiv(min(r0 + ROWS, vrows) - 1, p.fd_group) + 1 + coff)) : lk;
    const int nt = (kend + KT - 1) / KT;

    const uint32_t kst = static_cast<uint32_t>(p.ks[2] * ES), vst = static_cast<uint32_t>(p.vs[2] * ES);
    const typename TL::Offs okk = TL::offs(lane, kst), ovv = TL::offs(lane, vst);
    const char* const kbase = reinterpret_cast<const char*>(static_cast<const T*>(p.k) + kb + kvh * p.ks[1] +
                                                            static_cast<int64_t>(k0) * p.ks[2]);
    const char* const vbase = reinterpret_cast<const char*>(static_cast<const T*>(p.v) + vb + kvh * p.vs[1] +
                                                            static_cast<int64_t>(k0) * p.vs[2]);
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_addr(smem));
    auto request_k = [&](int t, int buf) {
        TL::request(kbase, kst, t * KT, lk, p.d * ES, okk, wave, lds0 + buf * TILE_B);
    };
    auto request_v = [&](int t, int buf) {
        TL::request(vbase, vst, t * KT, lk, p.dv * ES, ovv, wave, lds0 + (2 + buf) * TILE_B);
    };
    // All of vmcnt (the builtin, so that the compiler knows the mask loads are back too).
    auto landed = [&] {
        __builtin_amdgcn_s_waitcnt(0x0f70);
        __asm__ volatile("" ::: "memory");
        __syncthreads();
    };
    const typename TL::Addr ad = TL::addr(lane);

    f32x16 o[DB];
#pragma unroll
    for (int b = 0; b < DB; ++b) o[b] = splat16(0.f);
    // The row's reference point m (base 2), the threshold past which it moves, -m (0 while
    // m is minus infinity), and this lane's half of the row sum.
    float m = -INFINITY, thr = -INFINITY, neg_m = 0.f, lsum = 0.f;

    const int kw = 32 * NB * kp;  // the wavefront's first key within a tile
    // Scores in units of 1 / xs (base 2): the products, or (masked calls) scaled already.
    const float xs = MASKED ? 1.f : c2;
    // Minus infinity where the row does not see the key.
    auto edge = [&](f32x16 (&s)[NB], int t) {
        if (t * KT + kw + 32 * NB <= lim_w) return;
        const int rel = lim - t * KT - kw - 4 * h2;
#pragma unroll
        for (int n = 0; n < NB; ++n)
#pragma unroll
            for (int i = 0; i < 16; ++i)
                if (32 * n + 8 * (i / 4) + i % 4 >= rel) s[n][i] = -INFINITY;
    };
    auto block_max = [&](const f32x16 (&s)[NB]) {
        float mx = fmaxf(s[0][0], s[0][15]);
#pragma unroll
        for (int n = 0; n < NB; ++n)
#pragma unroll
            for (int i = n == 0 ? 1 : 0; i + 1 < 16; i += 2) mx = fmaxf(fmaxf(mx, s[n][i]), s[n][i + 1]);
        return mx;
    };
    // Moves the reference points that the tile's scores exceed by more than 2^kTileLazy (own: that
    // they do not stay below by 2^kTileDrop).
    auto rescale = [&](const f32x16 (&s)[NB], bool own) {
        const float lmax = block_max(s);
        const float at = own ? thr - (kTileLazy + kTileDrop) : thr;
        if (__builtin_amdgcn_ballot_w64(lmax * xs > at)) {
            const float mt = fmaxf(lmax, other_half(lmax)) * xs;
            const bool move = mt > at;
            const float alpha = move ? __builtin_amdgcn_exp2f(m - mt) : 1.f;  // 0 while m was -inf
            if (move) {
                m = mt;
                thr = mt + kTileLazy;
                neg_m = -mt;
            }
            lsum *= alpha;
#pragma unroll
            for (int b = 0; b < DB; ++b)
#pragma unroll
                for (int i = 0; i < 16; ++i) o[b][i] *= alpha;
        }
    };
    // The step below is laid out by hand: one MFMA, the LDS read of the operand LA products
    // on, and a share of the exponentials per group, with no instruction moving between
    // groups (left alone, the compiler issues all exponentials first and then waits for each
    // operand where it is used: 2x10x4096x64 127 us against 123).
    constexpr int NS = NB * DC, NP = NB * 2 * DB, LA = DP <= 64 ? 4 : 3;
    constexpr int PAIRS = 8 * NB;                       // pairs of scores of a lane
    constexpr int SPREAD = NB > 1 ? NS + NP / NB : NS;  // groups that share them
    auto k_frag = [&](uint32_t ra, int i) { return TL::rows(ra, i / NB, 2u * 32 * (i % NB) * TL::PITCH); };
    auto v_frag = [&](uint32_t t0, uint32_t t1, int j) {
        return TL::cols(t0, t1, (j / DB) % 2, j % DB, 2u * 32 * (j / (2 * DB)) * TL::PITCH);
    };
    auto pair = [&](const f32x16 (&s)[NB], v8 (&pb)[NB][2], int k) {
        const int n = k / 8, i = 2 * (k % 8);
        pb[n][i / 8][i % 8] = from_f32<T>(__builtin_amdgcn_exp2f(s[n][i] * xs + neg_m));
        pb[n][i / 8][i % 8 + 1] = from_f32<T>(__builtin_amdgcn_exp2f(s[n][i + 1] * xs + neg_m));
        lsum = dot_ones<T>(__builtin_bit_cast(u32x4, pb[n][i / 8])[(i % 8) / 2], lsum);
    };
    // PV of a tile from its probabilities (the pairs past `done` groups are formed here).
    auto pv = [&](const f32x16 (&s)[NB], v8 (&pb)[NB][2], v8 (&vr)[LA], uint32_t t0, uint32_t t1, int done, int spread) {
#pragma unroll
        for (int j = 0; j < NP; ++j) {
            o[j % DB] = Mfma32<T>::run(vr[j % LA], pb[j / (2 * DB)][(j / DB) % 2], o[j % DB]);
            if (j + LA < NP) vr[j % LA] = v_frag(t0, t1, j + LA);
#pragma unroll
            for (int k = 0; k < PAIRS; ++k)
                if (k * spread / PAIRS == done + j) pair(s, pb, k);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // S of a tile alone.
    auto scores = [&](f32x16 (&s)[NB], uint32_t ra) {
        v8 kr[LA];
#pragma unroll
        for (int i = 0; i < LA; ++i) kr[i] = k_frag(ra, i);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < NS; ++i) {
            s[i % NB] = Mfma32<T>::run(kr[i % LA], qf[i / NB], s[i % NB]);
            if (i + LA < NS) kr[i % LA] = k_frag(ra, i + LA);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // Softmax and PV of a tile alone, from its scores.
    auto finish = [&](f32x16 (&s)[NB], uint32_t t0, uint32_t t1, bool own) {
        rescale(s, own);
        v8 pb[NB][2], vr[LA];
#pragma unroll
        for (int j = 0; j < LA; ++j) vr[j] = v_frag(t0, t1, j);
#pragma unroll
        for (int k = 0; k < 8; ++k) pair(s, pb, k);
        __builtin_amdgcn_sched_barrier(0);
        // (NB = 2: the second block's pairs among the first's products.)
        pv(s, pb, vr, t0, t1, NP / NB, NB > 1 ? 2 * NP / NB : 0);
    };
    auto k_addr = [&](int buf) { return lds0 + buf * TILE_B + 2u * kw * TL::PITCH; };
    auto v_addr = [&](int buf) { return lds0 + (2 + buf) * TILE_B + 2u * kw * TL::PITCH; };

    bool dead = false;  // masked calls: the row kept no key (its output is over its raw scores)
    if constexpr (!MASKED) {
        // Tile t's softmax and PV with tile t + 1's S: K of tile t + 1 and V of tile t are in
        // (requested a tile ago), and every wavefront is done with K of tile t, V of tile t - 1.
        auto step = [&](f32x16 (&s)[NB], f32x16 (&sn)[NB], int t) {
            landed();
            uint32_t ra = k_addr((t + 1) & 1) + ad.row, t0 = v_addr(t & 1) + ad.tr0, t1 = v_addr(t & 1) + ad.tr1;
            __asm__ volatile("" : "+v"(ra), "+v"(t0), "+v"(t1));
            v8 kr[LA], vr[LA], pb[NB][2];
#pragma unroll
            for (int i = 0; i < LA; ++i) kr[i] = k_frag(ra, i);
            if (t + 2 < nt) request_k(t + 2, t & 1);
            request_v(t + 1, (t + 1) & 1);
            edge(s, t);
            rescale(s, t < tile_own(RG));
#pragma unroll
            for (int n = 0; n < NB; ++n) sn[n] = splat16(0.f);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < NS; ++i) {
                sn[i % NB] = Mfma32<T>::run(kr[i % LA], qf[i / NB], sn[i % NB]);
                if (i + LA < NS)
                    kr[i % LA] = k_frag(ra, i + LA);
                else
                    vr[i + LA - NS] = v_frag(t0, t1, i + LA - NS);
#pragma unroll
                for (int k = 0; k < PAIRS; ++k)
                    if (k * SPREAD / PAIRS == i) pair(s, pb, k);
                __builtin_amdgcn_sched_barrier(0);
            }
            pv(s, pb, vr, t0, t1, NS, SPREAD);
        };
        auto last = [&](f32x16 (&s)[NB], int t) {
            landed();
            edge(s, t);
            uint32_t t0 = v_addr(t & 1) + ad.tr0, t1 = v_addr(t & 1) + ad.tr1;
            __asm__ volatile("" : "+v"(t0), "+v"(t1));
            finish(s, t0, t1, t < tile_own(RG));
        };
        if (nt > 0) {
            request_k(0, 0);
            request_v(0, 0);
            if (nt > 1) request_k(1, 1);
            landed();
        }
        if (!live) {
            // The requests and barriers of the steps below (a test inside them costs their
            // registers: 44 spills at head dim 128 against 9).
            for (int t = 0; t < nt; ++t) {
                landed();
                if (t + 2 < nt) request_k(t + 2, t & 1);
                if (t + 1 < nt) request_v(t + 1, (t + 1) & 1);
            }
        } else if (nt > 0) {
            f32x16 sa[NB], sb[NB];
            uint32_t ra = k_addr(0) + ad.row;
            __asm__ volatile("" : "+v"(ra));
#pragma unroll
            for (int n = 0; n < NB; ++n) sa[n] = splat16(0.f);
            scores(sa, ra);
            int t = 0;
            for (; t + 2 < nt; t += 2) {
                step(sa, sb, t);
                step(sb, sa, t + 1);
            }
            if (t + 1 < nt) {
                step(sa, sb, t);
                last(sb, t + 1);
            } else {
                last(sa, t);
            }
        }
    } else {
        typedef typename MaskRaw<MK>::type MRaw;
        const bool packed = p.mask_mode == KMI_MASK_PACKED;
        const int64_t m_key = packed ? 1 : p.ms[3];
        const int64_t m_end = packed ? p.mask_numel : INT64_MAX;
        int64_t mrow;
        bool mvec = p.mask_vec4 != 0;  // uniform: whole tiles read four keys per load
        if (packed) {
            const int64_t off = packed_block_offset(p, seq);
            mrow = off + static_cast<int64_t>(pos) * lk;
            mvec = mvec && off + static_cast<int64_t>(lq) * lk <= m_end;
        } else {
            mrow = (p.cu_q ? static_cast<int64_t>(q0) * p.ms[2] + static_cast<int64_t>(k0) * p.ms[3] : seq * p.ms[0]) +
                   head * p.ms[1] + static_cast<int64_t>(pos) * p.ms[2];
        }
        const MRaw* const mp = static_cast<const MRaw*>(p.mask);
        // A padding mask (the keys alone decide): tiles that keep no key are not staged, once
        // some key is kept.  The flags are one byte per tile.
        constexpr int FLAGS = 2048, EPV = 16 / static_cast<int>(sizeof(MRaw));
        uint8_t* const flag = smem + 4 * TILE_B;
        bool skip = false;
        if (!packed && p.ms[1] == 0 && p.ms[2] == 0 && m_key == 1 && nt <= FLAGS && lk % EPV == 0 &&
            (reinterpret_cast<uintptr_t>(mp + mrow) & 15) == 0) {
            for (int i = threadIdx.x; i < nt; i += 256) flag[i] = 0;
            __syncthreads();
            bool keeps = false;
            for (int v = threadIdx.x; v < lk / EPV; v += 256) {
                const u32x4 raw = *reinterpret_cast<const u32x4*>(mp + mrow + static_cast<int64_t>(v) * EPV);
                MRaw e[EPV];
                __builtin_memcpy(e, &raw, 16);
                bool any = false;
#pragma unroll
                for (int j = 0; j < EPV; ++j) any = any || mask_logit_of<MK>(e[j]) > kMaskedLogit;
                keeps = keeps || any;
                if (any && v * EPV / KT < nt) flag[v * EPV / KT] = 1;
            }
            skip = __builtin_amdgcn_readfirstlane(__syncthreads_or(keeps)) != 0;
        }
        int met = 0;       // tiles the wavefront has worked on
        MRaw raw[NB][16];  // the staged tile's mask values
        auto load_mask = [&](MRaw (&x)[NB][16], int t) {
            const int key0 = t * KT + kw + 4 * h2;
            if (mvec && t * KT + KT <= lk) {
                const MRaw* src = mp + mrow + key0;
#pragma unroll
                for (int n = 0; n < NB; ++n)
#pragma unroll
                    for (int q = 0; q < 4; ++q) __builtin_memcpy(&x[n][4 * q], src + 32 * n + 8 * q, 4 * sizeof(MRaw));
            } else if (mvec && lk >= 4) {
                // The last, partial tile: four keys per load that end with the last key at most,
                // shifted into place (whatever lies past the last key is not seen).  Key by key
                // its 16 or 32 loads and their addresses cost more than a whole tile.
                const MRaw* src = mp + mrow;
#pragma unroll
                for (int n = 0; n < NB; ++n)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const int k = key0 + 32 * n + 8 * q, from = min(k, lk - 4), by = min(k - from, 3);
                        if constexpr (sizeof(MRaw) == 4) {
                            MRaw e[4];
                            __builtin_memcpy(e, src + from, sizeof(e));
                            if (by & 1) e[0] = e[1], e[1] = e[2], e[2] = e[3];
                            if (by & 2) e[0] = e[2], e[1] = e[3];
                            __builtin_memcpy(&x[n][4 * q], e, sizeof(e));
                        } else {
                            typename std::conditional<sizeof(MRaw) == 2, uint64_t, uint32_t>::type e;
                            __builtin_memcpy(&e, src + from, sizeof(e));
                            e >>= 8 * static_cast<int>(sizeof(MRaw)) * by;
                            __builtin_memcpy(&x[n][4 * q], &e, sizeof(e));
                        }
                    }
            } else {
#pragma unroll
                for (int n = 0; n < NB; ++n)
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        const int64_t at = mrow + min(key0 + 32 * n + 8 * (i / 4) + i % 4, lk - 1) * m_key;
                        x[n][i] = at < m_end ? mp[at] : MRaw{};
                    }
            }
        };
        auto next = [&](int t, bool all) {
            if (skip && !all)
                while (t < nt && __builtin_amdgcn_readfirstlane(flag[t]) == 0) ++t;
            return __builtin_amdgcn_readfirstlane(t);  // (scalar, as the staging's addresses are)
        };
        // Two passes at most: over the kept keys, and (when a row of the workgroup kept none)
        // over the raw scores of the rows that kept none.
        for (int pass = 0; pass < 2; ++pass) {
            int t = next(0, pass == 1);
            int buf = 0;
            if (t < nt) {
                request_k(t, 0);
                request_v(t, 0);
                if (pass == 0 && live) load_mask(raw, t);
            }
            while (t < nt) {
                const int tn = next(t + 1, pass == 1);
                landed();
                f32x16 s[NB], ml[NB];  // ml: the logits, kMaskedLogit or less where masked or not seen
                if (pass == 0) {
#pragma unroll
                    for (int n = 0; n < NB; ++n)
#pragma unroll
                        for (int i = 0; i < 16; ++i) ml[n][i] = mask_value_of<MK>(raw[n][i]);
                } else {
#pragma unroll
                    for (int n = 0; n < NB; ++n) ml[n] = splat16(dead ? 0.f : kMaskedLogit);
                }
                if (tn < nt) {
                    request_k(tn, buf ^ 1);
                    request_v(tn, buf ^ 1);
                    if (pass == 0 && live) load_mask(raw, tn);
                }
                edge(ml, t);
                // (Uniform.)  A tile in which no row of the wavefront keeps a key adds nothing.
                if (live && __builtin_amdgcn_ballot_w64(block_max(ml) > kMaskedLogit)) {
                    uint32_t ra = k_addr(buf) + ad.row, t0 = v_addr(buf) + ad.tr0, t1 = v_addr(buf) + ad.tr1;
                    __asm__ volatile("" : "+v"(ra), "+v"(t0), "+v"(t1));
#pragma unroll
                    for (int n = 0; n < NB; ++n) s[n] = splat16(0.f);
                    scores(s, ra);
#pragma unroll
                    for (int n = 0; n < NB; ++n)
#pragma unroll
                        for (int i = 0; i < 16; ++i) s[n][i] = masked_score(s[n][i], c2, ml[n][i]);
                    finish(s, t0, t1, met++ < tile_own(RG));
                }
                t = tn;
                buf ^= 1;
            }
            if (pass == 0) {
                float l = lsum + other_half(lsum);
                if constexpr (KP == 2) {
                    // The row's other wavefront may have met a kept key.
                    __syncthreads();  // the tiles are read
                    float* ls = reinterpret_cast<float*>(smem);
                    if (h2 == 0) ls[kp * 64 + 32 * rg + l32] = l;
                    __syncthreads();
                    l = ls[32 * rg + l32] + ls[64 + 32 * rg + l32];
                }
                dead = live && lim > 0 && l == 0.f;
                if (__builtin_amdgcn_readfirstlane(__syncthreads_or(dead)) == 0) break;
            }
        }
    }

    if constexpr (KP == 2) {
        // The second wavefront of each row group hands its state over through LDS.
        static_assert(4 * TILE_B >= RG * (DB * 4 + 1) * kWave * sizeof(f32x4), "exchange fits the tiles");
        __syncthreads();  // the last tile's reads are done
        f32x4* ex = reinterpret_cast<f32x4*>(smem) + rg * (DB * 4 + 1) * kWave;
        if (kp == 1) {
#pragma unroll
            for (int b = 0; b < DB; ++b)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    ex[(b * 4 + q) * kWave + lane] = f32x4{o[b][4 * q], o[b][4 * q + 1], o[b][4 * q + 2], o[b][4 * q + 3]};
            ex[DB * 4 * kWave + lane] = f32x4{m, lsum, 0.f, 0.f};
        }
        __syncthreads();
        if (kp == 1) return;
        const f32x4 st = ex[DB * 4 * kWave + lane];
        const float mn = fmaxf(m, st[0]);
        // (Minus infinity: that wavefront's sums are zero.)
        const float wa = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - mn);
        const float wb = st[0] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(st[0] - mn);
        m = mn;
        lsum = lsum * wa + st[1] * wb;
#pragma unroll
        for (int b = 0; b < DB; ++b)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const f32x4 x = ex[(b * 4 + q) * kWave + lane];
#pragma unroll
                for (int e = 0; e < 4; ++e) o[b][4 * q + e] = o[b][4 * q + e] * wa + x[e] * wb;
            }
    }
    // Lane (l32, h2) of block b, register 4 q + e: row rw0 + l32, dim 32 b + 8 q + 4 h2 + e.
    const float l = lsum + other_half(lsum);
    if (row >= vrows) return;
    const float inv = l > 0.f ? 1.f / l : 0.f;
    T* dst = static_cast<T*>(p.out) + ob + head * p.os[1] + static_cast<int64_t>(q0 + pos) * p.os[2];
    typedef T t4 __attribute__((ext_vector_type(4)));
#pragma unroll
    for (int b = 0; b < DB; ++b)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int d = 32 * b + 8 * q + 4 * h2;
            if (d >= p.dv) continue;
            t4 w;
#pragma unroll
            for (int e = 0; e < 4; ++e) w[e] = from_f32<T>(o[b][4 * q + e] * inv);
            *reinterpret_cast<t4*>(dst + d) = w;
        }
    if (p.lse && h2 == 0)
        p.lse[lb + head * p.ls[1] + static_cast<int64_t>(q0 + pos) * p.ls[2]] =
            l > 0.f ? (m + log2f(l)) * kTileLn2 + (dead ? kMaskedLogit : 0.f) : -INFINITY;
}

// Wavefronts per SIMD the kernel is held to.
constexpr int tile_waves(int dp) { return dp <= 128 ? 2 : 1; }

// Workgroup order: causal query tiles heaviest first, the units of a tile row next to each
// other.  xcd_map 3: unit u on XCD u % 8 with each tile row's units rotated by the row
// (ragged packed batches would otherwise meet the same few units' work row after row).
// snake: as in attn_fwd_kernel, rounds of CU-count blocks alternate direction.
template <typename T, int DP, int MK, int RG>
__global__ __launch_bounds__(NTHREADS, tile_waves(DP)) void attn_tile_kernel(const AttnParams p) {
    constexpr size_t TILES = 4 * sizeof(T) * Tile<T, DP, tile_keys(DP, RG)>::ELEMS;
    __shared__ __align__(1024) unsigned char smem[TILES + (MK != MK_NONE ? 2048 : 0)];
    int lin = blockIdx.x;
    const int units = p.batch * p.hkv;
    int bh, xi;
    if (p.xcd_map == 3) {
        const int x = lin & 7, s = lin >> 3;
        const int nxu = (units - x + 7) >> 3;
        if (nxu <= 0) return;
        const int rank = s / nxu;
        if (rank >= p.nx) return;
        bh = x + 8 * ((s - rank * nxu + rank) % nxu);
        xi = rank;
    } else {
        if (p.snake > 0) {
            const int round = fdiv(lin, p.fd_snake), at = lin - round * p.snake;
            const int in_round = min(p.snake, p.nx * units - round * p.snake);
            if (round & 1) lin = round * p.snake + (in_round - 1 - at);
        }
        xi = fdiv(lin, p.fd_units);
        bh = lin - xi * units;
    }
    attn_tile<T, DP, MK, RG>(p, smem, bh, p.causal ? p.nx - 1 - xi : xi);
}

template <typename T, int DP, int MK>
hipError_t launch_tile_mk(const AttnParams& p_in, int rg, hipStream_t stream) {
    AttnParams p = p_in;
    const int64_t units = static_cast<int64_t>(p.batch) * p.hkv;
    int64_t grid = units * p.nx;
    p.xcd_map = p.cu_q && units >= 8 ? 3 : 0;
    p.snake = 0;
    if (p.xcd_map == 3)
        grid = 8 * ceil_div(units, 8) * static_cast<int64_t>(p.nx);
    else if ((p.causal || MK != MK_NONE) && grid <= 2 * cu_count())
        p.snake = cu_count();
    p.fd_snake = fast_div(static_cast<uint32_t>(p.snake));
    const dim3 g(static_cast<unsigned>(grid));
    if constexpr (DP <= 128) {
        if (rg == 4) {
            hipLaunchKernelGGL((attn_tile_kernel<T, DP, MK, 4>), g, dim3(NTHREADS), 0, stream, p);
            return hipGetLastError();
        }
    }
    hipLaunchKernelGGL((attn_tile_kernel<T, DP, MK, 2>), g, dim3(NTHREADS), 0, stream, p);
    return hipGetLastError();
}

template <typename T, int DP>
hipError_t launch_tile(const AttnParams& p, int rg, hipStream_t stream) {
    if (p.mask_mode == KMI_MASK_NONE) return launch_tile_mk<T, DP, MK_NONE>(p, rg, stream);
    switch (p.mask_dtype) {
        case KMI_BOOL: return launch_tile_mk<T, DP, MK_BOOL>(p, rg, stream);
        case KMI_BF16: return launch_tile_mk<T, DP, MK_BF16>(p, rg, stream);
        case KMI_F16: return launch_tile_mk<T, DP, MK_F16>(p, rg, stream);
        default: return launch_tile_mk<T, DP, MK_F32>(p, rg, stream);
    }
}

}  // namespace fwd
}  // namespace kmi
