// Attention backward, the gradient kernels for head dims padded to 128 or less (gfx950).
// What they compute and the launches around them are described in attention_bwd.hip.
//
// Both passes run on v_mfma_f32_32x32x16: 256-thread workgroups stage 64-row tiles of the
// two operands the pass walks over (Q and dO for dK / dV, K and V for dQ) in LDS, double
// buffered, by buffer loads that write LDS directly, and every wavefront keeps 32 rows of
// the other side (keys or query rows) in registers as B operands:
//
//   dK / dV  S = Q K^T and dP = dO V^T of a 32-row block come out with one key per lane
//            and 16 query rows in registers, which is the B operand of dV^T += dO^T P and
//            dK^T += Q^T dS as it stands: P and dS never leave the registers.
//   dQ       S^T = K Q^T and dP^T = V dO^T: one query row per lane, 16 keys in registers,
//            the B operand of dQ^T += K^T dS^T.
//
// The A operands of the second products (dO^T, Q^T, K^T) are gfx950 transposed LDS reads
// of the same tiles.  dP accumulates from -D (the row dot), so dS = P dP has no subtraction.
//
// What bounds it: a 32x32 block of dK / dV is D / 4 MFMAs (1024 cycles of the matrix unit
// at D = 128) over about 64 VALU instructions a lane and 48 LDS reads, so with everything
// in registers the matrix unit should lead; what is left are waits at the tile barriers and
// the chain S -> P -> dV / dK within a wavefront (two wavefronts a SIMD at D = 128, three at
// 64).  Whole backward, before (16x16x32 MFMAs, P and dS through LDS, staging through
// registers) -> with this kernel, us:
//   1x24x4396x128        1388 -> 861  (428 -> 689 TFLOP/s)
//   2x10x4096x64          542 -> 371  (396 -> 579)
//   2x8/2x3062x128 causal 320 -> 161  (300 -> 597)
//   1x14/2x2048x64 causal  72 -> 51   (263 -> 373)
//   8 packed x 16/8 x 128 causal, 64 to 1024 tokens 153 -> 92 (211 -> 354)
//   2x12x2433x128, additive mask 1425 -> 480 (128 -> 380)
// What mattered on the way (1x24x4396x128): no spill in the loop (1351 with fragments
// spilled -> 984 with V in LDS and one code path per block); swizzles for 64 banks (LDS busy
// 39% -> 19% of the time); the order of the products (925 -> 861).
#pragma once

#include <cstddef>
#include <type_traits>

#include "attention_bwd_params.hpp"
#include "mfma_tile.hpp"

namespace kmi {
namespace bwd {


// A 16-byte fragment of row `row` at column `col` of an [nrows, d] operand, zeros past
// the last row or the head dim.
template <typename V, typename T>
__device__ __forceinline__ V frag16(const T* base, int64_t rs, int row, int nrows, int col, int d) {
    const int rc = min(max(row, 0), nrows - 1);
    const u32x4 x = *reinterpret_cast<const u32x4*>(base + static_cast<int64_t>(rc) * rs + min(col, d - 8));
    return __builtin_bit_cast(V, (row >= 0 && row < nrows && col < d) ? x : u32x4{0u, 0u, 0u, 0u});
}

// Four consecutive dims of an output row: fp32 partials or the gradient's own type.
template <typename T>
__device__ __forceinline__ void store4(T* dst, const f32x4 v) {
    typedef T t4 __attribute__((ext_vector_type(4)));
    t4 w;
#pragma unroll
    for (int e = 0; e < 4; ++e) w[e] = from_f32<T>(v[e]);
    *reinterpret_cast<t4*>(dst) = w;
}

// dK / dV workgroups take 32 KG keys: 64 (two wavefronts per 32 keys) at padded head dims
// up to 64 and, at 96 and 128, where 128 keys (one wavefront per 32) would leave most of the
// chip idle (HALF).  Past head dim 64 the accumulators and the K fragments leave no registers
// for V's, so V sits in LDS beside the tiles: 32-row tiles with 128 keys (two workgroups per
// CU), 64-row ones with 64 (one).
template <typename T, int DP, bool HALF>
struct DkdvShared {
    static constexpr int KG = DP <= 64 || HALF ? 2 : 4;
    static constexpr int TR = KG == 2 ? 64 : 32;
    static constexpr bool VL = DP > 64;
    typedef Tile<T, DP, TR> TL;
    T tile[2][2][TL::ELEMS];
    T v[VL ? 32 * KG * TL::PITCH : 8];
    // Base-2 lse, -D, raw flag (masked calls) of the tile's rows; a DMA instruction fills 64.
    float stats[2][3][kWave];
};

// dK / dV of 32 KG keys of one K/V head (wavefront w: key group w % KG; with KG = 2 the
// two wavefronts of a key group take one 32-row block of each tile each and add their
// sums at the end) over the split's (query head, query tile) items.
template <typename T, int DP, int MK, bool HALF>
__device__ __forceinline__ void bwd_dkdv(const BwdParams& p, unsigned char* smem, const int tile, const int split,
                                         const int bkv) {
    typedef DkdvShared<T, DP, HALF> SH;
    typedef typename SH::TL TL;
    typedef typename TL::v8 v8;
    constexpr int KG = SH::KG, TR = SH::TR, DC = DP / 16, DB = DP / 32, RB = TR / 32;
    constexpr int ES = static_cast<int>(sizeof(T));
    constexpr int RS = 4 / KG;  // wavefronts that share a key group
    constexpr bool VL = SH::VL;
    static_assert(RS <= RB, "a wavefront of a key group takes whole 32-row blocks");
    SH& sh = *reinterpret_cast<SH*>(smem);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int h2 = lane >> 5, l32 = lane & 31;
    const int kg = wave % KG, rsp = wave / KG;
    const int seq = bkv / p.hkv, kvh = bkv - seq * p.hkv;
    const Geo g = geo_of(p, seq);
    const int kt0 = tile * 32 * KG;
    // Keys written: the sequence's (varlen) or every key row of the batch entry (dense:
    // keys past a key length get zero gradients).
    const int kwrite = p.cu_q ? g.lk : p.seq_k;
    if (kt0 >= kwrite) return;  // uniform: no barrier has run
    const int kw0 = kt0 + 32 * kg;
    const int key = kw0 + l32;
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_addr(smem));
    constexpr uint32_t TILE_B = TL::ELEMS * sizeof(T);

    // Items: (query head of the group, query tile), tiles from the first that sees this key
    // tile (causal: rows i >= kt0 - coff); split s takes items s, s + splits, ....  The walk
    // steps (gi, bi) by (splits / nblk, splits % nblk) with one carry.
    const int rfirst = p.causal ? max(0, kt0 - g.coff) / TR : 0;
    const int nblk = (kt0 < g.lk && g.lq > rfirst * TR) ? (g.lq + TR - 1) / TR - rfirst : 0;
    const int items = nblk * p.group;
    const int sp_g = nblk > 0 ? p.splits / nblk : 0, sp_b = p.splits - sp_g * nblk;
    int gi = nblk > 0 ? split / nblk : 0, bi = split - gi * nblk;
    const uint32_t qst = static_cast<uint32_t>(p.qs[2] * ES), dst = static_cast<uint32_t>(p.dos[2] * ES);
    const typename TL::Offs oq = TL::offs(lane, qst), od = TL::offs(lane, dst);
    // Head 0 of the group; head gi is gi * (head stride) bytes on.
    const char* const qg = reinterpret_cast<const char*>(static_cast<const T*>(p.q) + g.qb + kvh * p.group * p.qs[1] +
                                                         static_cast<int64_t>(g.q0) * p.qs[2]);
    const char* const dg = reinterpret_cast<const char*>(static_cast<const T*>(p.dout) + g.dob +
                                                         kvh * p.group * p.dos[1] + static_cast<int64_t>(g.q0) * p.dos[2]);
    const int64_t qh = p.qs[1] * ES, dh = p.dos[1] * ES;
    const float* const sg = p.nd + static_cast<int64_t>(kvh) * p.group * p.rows_total + g.row_base;
    const float* const lg = p.lse + g.lb + kvh * p.group * p.ls[1] + static_cast<int64_t>(g.q0) * p.ls[2];
    float lse_n = 0.f;  // wavefront 0: the requested item's lse, row `lane`
    auto request = [&](int gi_, int bi_, int buf) {
        const int r0 = (rfirst + bi_) * TR;
        const uint32_t at = lds0 + buf * 2 * TILE_B;
        TL::request(qg + gi_ * qh, qst, r0, g.lq, p.d * ES, oq, wave, at);
        TL::request(dg + gi_ * dh, dst, r0, g.lq, p.dval * ES, od, wave, at + TILE_B);
        if (wave == 0) {
            dma4(dma_rsrc(sg + gi_ * p.rows_total + r0, 4u * static_cast<uint32_t>(min(TR, g.lq - r0))), 4u * lane,
                 lds0 + static_cast<uint32_t>(offsetof(SH, stats)) + static_cast<uint32_t>((buf * 3 + 1) * kWave * 4));
            lse_n = lg[gi_ * p.ls[1] + min(r0 + lane, g.lq - 1) * p.ls[2]];
        }
    };
    // Before the fragments' loads, whose values are selected from as they come: after them the
    // first tiles would start a memory round trip later (the whole backward of 8x2/30x30x80 14.4 ->
    // 13.7 us, 11x6/3x23x128 additive 17.4 -> 16.7).  Not up to head dim 64, where it costs
    // registers (three spilled without a mask; causal 2x10x4096x64 206 instead of 200).
    constexpr bool EARLY = VL;
    if constexpr (EARLY)
        if (split < items) request(gi, bi, 0);
    const typename TL::Addr ad = TL::addr(lane);
    v8 kf[DC], vf[VL ? 1 : DC];
    {
        const T* kp = static_cast<const T*>(p.k) + g.kb + kvh * p.ks[1] + static_cast<int64_t>(g.k0) * p.ks[2];
        const T* vp = static_cast<const T*>(p.v) + g.vb + kvh * p.vs[1] + static_cast<int64_t>(g.k0) * p.vs[2];
#pragma unroll
        for (int c = 0; c < DC; ++c) kf[c] = frag16<v8>(kp, p.ks[2], key, g.lk, 16 * c + 8 * h2, p.d);
        if constexpr (VL) {
            // (Published with the first item's tiles.)
            typedef Tile<T, DP, 32 * KG> TV;
            const uint32_t vst = static_cast<uint32_t>(p.vs[2] * ES);
            const typename TV::Offs ov = TV::offs(lane, vst);
            TV::request(reinterpret_cast<const char*>(vp), vst, kt0, g.lk, p.dval * ES, ov, wave,
                        lds0 + static_cast<uint32_t>(offsetof(SH, v)));
        } else {
#pragma unroll
            for (int c = 0; c < DC; ++c) vf[c] = frag16<v8>(vp, p.vs[2], key, g.lk, 16 * c + 8 * h2, p.dval);
        }
    }
    f32x16 dk[DB], dv[DB];
#pragma unroll
    for (int b = 0; b < DB; ++b) dk[b] = dv[b] = splat16(0.f);
    typedef typename MaskRaw<MK>::type MRaw;
    // S in units of 1 / xs (base 2): the products, or (masked calls) scaled already; `hidden`
    // makes P exactly 0 where the row does not see the key.
    constexpr bool MASKED = MK != MK_NONE;
    const float xs = MASKED ? 1.f : p.c2, hidden = MASKED ? -INFINITY : p.hidden;

    // One 32-row block (rows r0b ..) at LDS address qt (dO's a tile on).
    auto block = [&](uint32_t qt, const float* st, int h, int r0b) {
        // ml: the mask's logits, added once S is whole (masked_score).
        constexpr int LA = DP <= 64 ? 1 : 3;
        f32x16 s = splat16(0.f), ml, dp;
        if constexpr (MASKED) {
            const int64_t msz = static_cast<int64_t>(sizeof(MRaw));
            const int64_t b0 = g.mbase + h * p.ms[1] + r0b * g.mrow;
            const int rlast = min(31, g.lq - 1 - r0b), klast = min(kw0 + 31, g.lk - 1);
            const bool flat = g.mrow >= 0 && g.mkey >= 0 && (32 * g.mrow + g.lk * g.mkey) * msz < (int64_t{1} << 30) &&
                              b0 + rlast * g.mrow + klast * g.mkey < g.mend;
            // (Uniform.)  32-bit offsets from the block's first row; rows past the last and keys
            // past the last read those (rows in order: the clamp is a minimum of offsets).
            if (flat) {
                const auto rs = buffer_rsrc(static_cast<const MRaw*>(p.mask) + b0, 0x7fffffffu);
                auto load = [&](uint32_t off, int so) -> MRaw {
                    if constexpr (sizeof(MRaw) == 1)
                        return __builtin_amdgcn_raw_buffer_load_b8(rs, off, so, 0);
                    else if constexpr (sizeof(MRaw) == 2)
                        return __builtin_amdgcn_raw_buffer_load_b16(rs, off, so, 0);
                    else
                        return __builtin_bit_cast(MRaw, __builtin_amdgcn_raw_buffer_load_b32(rs, off, so, 0));
                };
                uint32_t step = static_cast<uint32_t>(g.mrow * msz);
                if constexpr (DP > 32) __asm__ volatile("" : "+s"(step));  // (else its multiples live across the loop)
                const uint32_t row = 4 * h2 * step;
                const uint32_t col = static_cast<uint32_t>(min(key, g.lk - 1)) * static_cast<uint32_t>(g.mkey * msz);
                MRaw raw[16];
                if (rlast == 31) {
#pragma unroll
                    for (int i = 0; i < 16; ++i)
                        raw[i] = load(row + col, (8 * (i / 4) + i % 4) * step);
                } else {
                    const uint32_t most = rlast * step;
#pragma unroll
                    for (int i = 0; i < 16; ++i)
                        raw[i] = load(min(row + (8 * (i / 4) + i % 4) * step, most) + col, 0);
                }
#pragma unroll
                for (int i = 0; i < 16; ++i) ml[i] = mask_value_of<MK>(raw[i]);
            } else {
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    ml[i] = mask_at<MK>(p, g, h, min(r0b + 8 * (i / 4) + 4 * h2 + i % 4, g.lq - 1), min(key, g.lk - 1));
            }
            // (Uniform; rows that kept no key are rare.)
            if (__builtin_amdgcn_ballot_w64(st[2 * kWave + l32] != 0.f)) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const f32x4 rw = *reinterpret_cast<const f32x4*>(st + 2 * kWave + 8 * q + 4 * h2);
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (rw[e] != 0.f) ml[4 * q + e] = 0.f;
                }
            }
        }
        // (Opaque lane addresses: the compiler would otherwise keep every sum it can hoist in
        // registers across the loop, and V's fragments too.)
        uint32_t ra = qt + ad.row, t0 = qt + ad.tr0, t1 = qt + ad.tr1;
        uint32_t va = lds0 + static_cast<uint32_t>(offsetof(SH, v)) + 2u * 32 * kg * TL::PITCH + ad.row;
        __asm__ volatile("" : "+v"(ra), "+v"(t0), "+v"(t1), "+v"(va));
        // The order below is kept by the fences: one MFMA, the LDS read of the operand LA
        // products on, and a share of the VALU work per group.  (Left alone, the compiler reads
        // each operand where it is used and bunches the exponentials: 8 packed x 16/8 x 128 121
        // us against 92, 1x24x4396x128 925 against 861.  LA as far as the registers go: 2 at
        // head dim 64 spills, 89 us against 78 on 4x16x1024x64.)
        v8 fa[LA], fb[VL ? LA : 1];
        auto neg_dots = [&](int q) {
            const f32x4 nd = *reinterpret_cast<const f32x4*>(st + kWave + 8 * q + 4 * h2);
#pragma unroll
            for (int e = 0; e < 4; ++e) dp[4 * q + e] = nd[e];
        };
        auto col = [&](int j, uint32_t imm) { return TL::cols(t0, t1, j / DB, j % DB, imm); };
#pragma unroll
        for (int c = 0; c < LA; ++c) fa[c] = TL::rows(ra, c, 0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 0; c < DC; ++c) {
            s = Mfma32<T>::run(fa[c % LA], kf[c], s);
            if (c + LA < DC) {
                fa[c % LA] = TL::rows(ra, c + LA, 0);
            } else {
                fa[c % LA] = TL::rows(ra, (c + LA) - DC, TILE_B);
                if constexpr (VL) fb[(c + LA) - DC] = TL::rows(va, (c + LA) - DC, 0);
            }
            // (Masked: dP's start follows below, in the registers that ml leaves.)
            if (!MASKED && (c >= DC - 4 || DC < 4)) {
                const int q = DC < 4 ? c : c - (DC - 4);
#pragma unroll
                for (int qq = q * (DC < 4 ? 4 / DC : 1); qq < (q + 1) * (DC < 4 ? 4 / DC : 1); ++qq) neg_dots(qq);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (MASKED) {
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] = masked_score(s[i], p.c2, ml[i]);
#pragma unroll
            for (int q = 0; q < 4; ++q) neg_dots(q);
        }
        // Blocks whose rows all see all 32 keys (uniform) need no per-element test.
        if (!(kw0 + 31 < g.lk && (!p.causal || kw0 + 31 <= r0b + g.coff))) {
            // Rows whose index (from this lane's first) is below `seen` do not see the key.
            const int seen = key >= g.lk ? 32 : (p.causal ? key - g.coff - r0b - 4 * h2 : -1);
#pragma unroll
            for (int i = 0; i < 16; ++i)
                if (8 * (i / 4) + i % 4 < seen) s[i] = hidden;
        }
        __builtin_amdgcn_sched_barrier(0);
        // dP, with P formed from S meanwhile.
        v8 pb[2], sb[2];
        f32x4 l2[2];
        auto lse4 = [&](int q) { return *reinterpret_cast<const f32x4*>(st + 8 * q + 4 * h2); };
        l2[0] = lse4(0);
        l2[1] = lse4(1);
#pragma unroll
        for (int c = 0; c < DC; ++c) {
            // (Ring slots: dO's fragment c was read into slot (DC - LA + c) % LA.)
            const int slot = (DC - LA + c) % LA;
            if constexpr (VL)
                dp = Mfma32<T>::run(fa[slot], fb[c % LA], dp);
            else
                dp = Mfma32<T>::run(fa[slot], vf[c], dp);
            if (c + LA < DC) {
                fa[slot] = TL::rows(ra, c + LA, TILE_B);
                if constexpr (VL) fb[c % LA] = TL::rows(va, c + LA, 0);
            } else {
                fa[slot] = col((c + LA) - DC, TILE_B);
            }
#pragma unroll
            for (int k = 0; k < 8; ++k)
                if (k * DC / 8 == c) {
#pragma unroll
                    for (int i = 2 * k; i < 2 * k + 2; ++i) {
                        s[i] = __builtin_amdgcn_exp2f(s[i] * xs - l2[(k / 2) % 2][i % 4]);
                        pb[i / 8][i % 8] = from_f32<T>(s[i]);
                    }
                    if (k % 2 == 1 && k / 2 + 2 < 4) l2[(k / 2) % 2] = lse4(k / 2 + 2);
                }
            __builtin_amdgcn_sched_barrier(0);
        }
        // dV^T += dO^T P while dS = P (dP - D) is formed, then dK^T += Q^T dS.
        constexpr int NP = 2 * DB;
#pragma unroll
        for (int j = 0; j < 2 * NP; ++j) {
            const int slot = (2 * DC - LA + j) % LA;
            if (j < NP)
                dv[j % DB] = Mfma32<T>::run(fa[slot], pb[j / DB], dv[j % DB]);
            else
                dk[j % DB] = Mfma32<T>::run(fa[slot], sb[(j - NP) / DB], dk[j % DB]);
            if (j + LA < NP)
                fa[slot] = col(j + LA, TILE_B);
            else if (j + LA < 2 * NP)
                fa[slot] = col(j + LA - NP, 0);
#pragma unroll
            for (int k = 0; k < 8; ++k)
                if (j < NP && k * NP / 8 == j) {
#pragma unroll
                    for (int i = 2 * k; i < 2 * k + 2; ++i) sb[i / 8][i % 8] = from_f32<T>(s[i] * dp[i]);
                }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    if constexpr (!EARLY)
        if (split < items) request(gi, bi, 0);
    int buf = 0;
    for (int it = split; it < items; it += p.splits) {
        const int h = kvh * p.group + gi, r0 = (rfirst + bi) * TR;
        gi += sp_g;
        bi += sp_b;
        if (bi >= nblk) {
            bi -= nblk;
            ++gi;
        }
        // This item's tiles were requested an item ago; past the barrier every wavefront's
        // share has landed and the other buffer's reads are done.
        __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (wave == 0) {
            float l2;
            bool raw;
            row_stats(lse_n, r0 + lane < g.lq, l2, raw);
            sh.stats[buf][0][lane] = l2;
            if constexpr (MASKED) sh.stats[buf][2][lane] = raw ? 1.f : 0.f;
        }
        __syncthreads();
        if (it + p.splits < items) request(gi, bi, buf ^ 1);
        if (kw0 < g.lk) {
#pragma unroll 1
            for (int rb = RS == 1 ? 0 : rsp; rb < RB; rb += RS) {
                const int r0b = r0 + 32 * rb;
                if (r0b >= g.lq || (p.causal && kw0 > r0b + 31 + g.coff)) continue;
                const uint32_t qt = lds0 + buf * 2 * TILE_B + 2u * 32 * rb * TL::PITCH;
                const float* st = sh.stats[buf][0] + 32 * rb;
                block(qt, st, h, r0b);
            }
        }
        buf ^= 1;
    }
    if constexpr (RS == 2) {
        // The second wavefront of each key group hands its sums over through LDS.
        static_assert(sizeof(sh.tile) >= KG * 2 * DB * 4 * kWave * sizeof(f32x4), "exchange fits the tiles");
        __syncthreads();  // the last item's tile reads are done
        f32x4* ex = reinterpret_cast<f32x4*>(smem) + kg * (2 * DB * 4 * kWave);
        if (rsp == 1) {
#pragma unroll
            for (int b = 0; b < DB; ++b)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    ex[((2 * b) * 4 + q) * kWave + lane] =
                        f32x4{dk[b][4 * q], dk[b][4 * q + 1], dk[b][4 * q + 2], dk[b][4 * q + 3]};
                    ex[((2 * b + 1) * 4 + q) * kWave + lane] =
                        f32x4{dv[b][4 * q], dv[b][4 * q + 1], dv[b][4 * q + 2], dv[b][4 * q + 3]};
                }
        }
        __syncthreads();
        if (rsp == 1) return;
#pragma unroll
        for (int b = 0; b < DB; ++b)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const f32x4 xk = ex[((2 * b) * 4 + q) * kWave + lane], xv = ex[((2 * b + 1) * 4 + q) * kWave + lane];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    dk[b][4 * q + e] += xk[e];
                    dv[b][4 * q + e] += xv[e];
                }
            }
    }
    // Lane (l32, h2) of block b, register 4 q + e: key kw0 + l32, dim 32 b + 8 q + 4 h2 + e.
    if (key >= kwrite) return;
    auto quad = [](const f32x16& v, int q, float m) {
        return f32x4{v[4 * q] * m, v[4 * q + 1] * m, v[4 * q + 2] * m, v[4 * q + 3] * m};
    };
    if (p.pdk) {
        const int64_t at = ((static_cast<int64_t>(kvh) * p.splits + split) * p.keys_total + g.key_base + key) * DP;
#pragma unroll
        for (int b = 0; b < DB; ++b)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int d = 32 * b + 8 * q + 4 * h2;
                if (d < p.d) *reinterpret_cast<f32x4*>(p.pdk + at + d) = quad(dk[b], q, p.scale);
                if (d < p.dval) *reinterpret_cast<f32x4*>(p.pdv + at + d) = quad(dv[b], q, 1.f);
            }
        return;
    }
    T* dkp = static_cast<T*>(p.dk) + g.dkb + kvh * p.dks[1] + static_cast<int64_t>(g.k0 + key) * p.dks[2];
    T* dvp = static_cast<T*>(p.dv) + g.dvb + kvh * p.dvs[1] + static_cast<int64_t>(g.k0 + key) * p.dvs[2];
#pragma unroll
    for (int b = 0; b < DB; ++b)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int d = 32 * b + 8 * q + 4 * h2;
            if (d < p.d) store4(dkp + d, quad(dk[b], q, p.scale));
            if (d < p.dval) store4(dvp + d, quad(dv[b], q, 1.f));
        }
}

// dQ of 32 RG "virtual rows" of one (sequence, K/V head): row r is query position r / G of
// query head kvh G + r % G, so a GQA group shares every K/V tile.  Wavefront w owns row
// group w % RG; with RG = 2 the two wavefronts of a row group take one 32-key block of
// each tile each and add their sums at the end.  Split `ksp` takes the 64-key tiles ksp,
// ksp + ksplit, ....
template <typename T, int DP, int MK, int RG>
__device__ __forceinline__ void bwd_dq(const BwdParams& p, unsigned char* smem, const int tile, const int ksp,
                                       const int bkv) {
    constexpr int TR = 64;
    typedef Tile<T, DP, TR> TL;
    typedef typename TL::v8 v8;
    constexpr int DC = DP / 16, DB = DP / 32;
    constexpr int KS = 4 / RG;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int h2 = lane >> 5, l32 = lane & 31;
    const int rg = wave % RG, kspw = wave / RG;
    const int seq = bkv / p.hkv, kvh = bkv - seq * p.hkv;
    const Geo g = geo_of(p, seq);
    const int G = p.group;
    const int vrows = g.lq * G;
    const int r0 = tile * 32 * RG;
    if (r0 >= vrows || g.lk <= 0) return;  // uniform: no barrier has run
    const int rw0 = r0 + 32 * rg;
    const int row = rw0 + l32;
    const int rr = min(row, vrows - 1);  // rows past the end repeat the last (never written)
    const int pos = rr / G, h = kvh * G + (rr - pos * G);

    // Causal: keys below lim are visible to this row; those below lim_w to every row of
    // the wavefront, none at or past kend_w to any.
    const int lim = p.causal ? min(g.lk, pos + 1 + g.coff) : g.lk;
    const int first = min(rw0, vrows - 1) / G, last = min(rw0 + 31, vrows - 1) / G;
    const int lim_w = p.causal ? min(g.lk, first + 1 + g.coff) : g.lk;
    const int kend_w = rw0 < vrows ? (p.causal ? min(g.lk, last + 1 + g.coff) : g.lk) : 0;
    const int kend = p.causal ? min(g.lk, max(0, min(r0 + 32 * RG, vrows) - 1) / G + 1 + g.coff) : g.lk;
    constexpr int ES = static_cast<int>(sizeof(T));
    const uint32_t kst = static_cast<uint32_t>(p.ks[2] * ES), vst = static_cast<uint32_t>(p.vs[2] * ES);
    const typename TL::Offs ok = TL::offs(lane, kst), ov = TL::offs(lane, vst);
    const char* const kbase = reinterpret_cast<const char*>(static_cast<const T*>(p.k) + g.kb + kvh * p.ks[1] +
                                                            static_cast<int64_t>(g.k0) * p.ks[2]);
    const char* const vbase = reinterpret_cast<const char*>(static_cast<const T*>(p.v) + g.vb + kvh * p.vs[1] +
                                                            static_cast<int64_t>(g.k0) * p.vs[2]);
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_addr(smem));
    constexpr uint32_t TILE_B = TL::ELEMS * sizeof(T);
    auto request = [&](int k0, int buf) {
        TL::request(kbase, kst, k0, g.lk, p.d * ES, ok, wave, lds0 + buf * 2 * TILE_B);
        TL::request(vbase, vst, k0, g.lk, p.dval * ES, ov, wave, lds0 + (buf * 2 + 1) * TILE_B);
    };
    const int kstep = p.ksplit * TR;
    int k0 = ksp * TR;
    constexpr bool EARLY = DP > 64;  // (as in bwd_dkdv)
    if constexpr (EARLY)
        if (k0 < kend) request(k0, 0);

    v8 qf[DC], of[DC];
    {
        const T* qp = static_cast<const T*>(p.q) + g.qb + h * p.qs[1] + static_cast<int64_t>(g.q0 + pos) * p.qs[2];
        const T* dp = static_cast<const T*>(p.dout) + g.dob + h * p.dos[1] + static_cast<int64_t>(g.q0 + pos) * p.dos[2];
#pragma unroll
        for (int c = 0; c < DC; ++c) {
            qf[c] = frag16<v8>(qp, 0, 0, 1, 16 * c + 8 * h2, p.d);
            of[c] = frag16<v8>(dp, 0, 0, 1, 16 * c + 8 * h2, p.dval);
        }
    }
    const float nd = p.nd[static_cast<int64_t>(h) * p.rows_total + g.row_base + pos];
    float l2;
    bool raw;
    row_stats(p.lse[g.lb + h * p.ls[1] + static_cast<int64_t>(g.q0 + pos) * p.ls[2]], true, l2, raw);
    f32x16 dq[DB];
#pragma unroll
    for (int b = 0; b < DB; ++b) dq[b] = splat16(0.f);

    const typename TL::Addr ad = TL::addr(lane);
    typedef typename MaskRaw<MK>::type MRaw;
    constexpr bool MASKED = MK != MK_NONE;
    const float xs = MASKED ? 1.f : p.c2, hidden = MASKED ? -INFINITY : p.hidden;  // (as in bwd_dkdv)
    const int64_t moff = g.mbase + h * p.ms[1] + pos * g.mrow;  // the row's mask values

    // One 32-key block (keys kb0 ..) at LDS address kt (V's a tile on).
    auto block = [&](uint32_t kt, int kb0) {
        f32x16 s = splat16(0.f), ml, dp = splat16(nd);  // (ml: as in bwd_dkdv)
        if constexpr (MASKED) {
            // Unit key stride: four consecutive keys per load.
            const bool vec = g.mkey == 1 && kb0 + 31 < g.lk && (p.mask_mode != KMI_MASK_PACKED || g.mpacked_ok);
            if (vec) {
                const MRaw* src = static_cast<const MRaw*>(p.mask) + moff + kb0 + 4 * h2;
                struct E {
                    MRaw e[4];
                } x[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) __builtin_memcpy(&x[q], src + 8 * q, sizeof(E));
#pragma unroll
                for (int i = 0; i < 16; ++i) ml[i] = mask_value_of<MK>(x[i / 4].e[i % 4]);
            } else {
                // Keys past the last read the last; a packed mask's end as in mask_at, but as a
                // clamped load and a select (a branch around each load would make it wait for the
                // one before).
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int64_t at = moff + min(kb0 + 8 * (i / 4) + 4 * h2 + i % 4, g.lk - 1) * g.mkey;
                    const float x = mask_logit_of<MK>(static_cast<const MRaw*>(p.mask)[min(at, g.mend - 1)]);
                    ml[i] = at < g.mend ? x : kMaskedLogit;
                }
            }
            if (__builtin_amdgcn_ballot_w64(raw)) {
#pragma unroll
                for (int i = 0; i < 16; ++i) ml[i] = raw ? 0.f : ml[i];
            }
        }
        uint32_t ra = kt + ad.row, t0 = kt + ad.tr0, t1 = kt + ad.tr1;
        __asm__ volatile("" : "+v"(ra), "+v"(t0), "+v"(t1));  // (as in bwd_dkdv)
        // S, dP with the exponentials, dQ: the operands in one stream, LA ahead.
        constexpr int LA = DP <= 64 ? 2 : 3, NP = 2 * DB, TOT = 2 * DC + NP;
        v8 fa[LA], sb[2];
        auto operand = [&](int i) {
            if (i < 2 * DC) return TL::rows(ra, i % DC, i < DC ? 0u : TILE_B);
            return TL::cols(t0, t1, (i - 2 * DC) / DB, (i - 2 * DC) % DB, 0);
        };
#pragma unroll
        for (int i = 0; i < LA; ++i) fa[i] = operand(i);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < DC; ++i) {
            s = Mfma32<T>::run(fa[i % LA], qf[i], s);
            fa[i % LA] = operand(i + LA);
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (MASKED) {
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] = masked_score(s[i], p.c2, ml[i]);
        }
        if (kb0 + 31 >= lim_w) {
            const int rel = lim - kb0 - 4 * h2;  // keys whose index is below rel are visible
#pragma unroll
            for (int i = 0; i < 16; ++i)
                if (8 * (i / 4) + i % 4 >= rel) s[i] = hidden;
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < DC; ++i) {
            dp = Mfma32<T>::run(fa[(DC + i) % LA], of[i], dp);
            fa[(DC + i) % LA] = operand(DC + i + LA);
#pragma unroll
            for (int k = 0; k < 8; ++k)
                if (k * DC / 8 == i) {
                    s[2 * k] = __builtin_amdgcn_exp2f(s[2 * k] * xs - l2);
                    s[2 * k + 1] = __builtin_amdgcn_exp2f(s[2 * k + 1] * xs - l2);
                }
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) sb[i / 8][i % 8] = from_f32<T>(s[i] * dp[i]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < NP; ++j) {
            const int i = 2 * DC + j;
            dq[j % DB] = Mfma32<T>::run(fa[i % LA], sb[j / DB], dq[j % DB]);
            if (i + LA < TOT) fa[i % LA] = operand(i + LA);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    if constexpr (!EARLY)
        if (k0 < kend) request(k0, 0);
    int buf = 0;
    for (; k0 < kend; k0 += kstep) {
        __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (as in bwd_dkdv)
        __syncthreads();
        if (k0 + kstep < kend) request(k0 + kstep, buf ^ 1);
#pragma unroll 1
        for (int kb = KS == 1 ? 0 : kspw; kb < 2; kb += KS)
            if (k0 + 32 * kb < kend_w) block(lds0 + buf * 2 * TILE_B + 2u * 32 * kb * TL::PITCH, k0 + 32 * kb);
        buf ^= 1;
    }
    if constexpr (KS == 2) {
        __syncthreads();  // the last tile's reads are done
        f32x4* ex = reinterpret_cast<f32x4*>(smem) + rg * (DB * 4 * kWave);
        if (kspw == 1) {
#pragma unroll
            for (int b = 0; b < DB; ++b)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    ex[(b * 4 + q) * kWave + lane] =
                        f32x4{dq[b][4 * q], dq[b][4 * q + 1], dq[b][4 * q + 2], dq[b][4 * q + 3]};
        }
        __syncthreads();
        if (kspw == 1) return;
#pragma unroll
        for (int b = 0; b < DB; ++b)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const f32x4 x = ex[(b * 4 + q) * kWave + lane];
#pragma unroll
                for (int e = 0; e < 4; ++e) dq[b][4 * q + e] += x[e];
            }
    }
    // Lane (l32, h2) of block b, register 4 q + e: row rw0 + l32, dim 32 b + 8 q + 4 h2 + e.
    if (row >= vrows) return;
    T* dst = static_cast<T*>(p.dq) + g.dqb + h * p.dqs[1] + static_cast<int64_t>(g.q0 + pos) * p.dqs[2];
    float* part = p.pdq ? p.pdq + ((static_cast<int64_t>(h) * p.ksplit + ksp) * p.rows_total + g.row_base + pos) * DP
                        : nullptr;
#pragma unroll
    for (int b = 0; b < DB; ++b)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int d = 32 * b + 8 * q + 4 * h2;
            if (d >= p.d) continue;
            const f32x4 v = f32x4{dq[b][4 * q] * p.scale, dq[b][4 * q + 1] * p.scale, dq[b][4 * q + 2] * p.scale,
                                  dq[b][4 * q + 3] * p.scale};
            if (part)
                *reinterpret_cast<f32x4*>(part + d) = v;
            else
                store4(dst + d, v);
        }
}

// Wavefronts per SIMD the kernel is held to: what its LDS leaves room for, three up to head dim
// 64 (168 registers), two past it with 128-key dK / dV workgroups (214 and 254), one with 64-key
// ones.  Unmasked kernels spill no vector registers; masked ones up to 14 (head dim 64).  The
// build fails past _build.TILE_VGPR_SPILLS.
constexpr int bwd_waves(int dp, bool half) { return dp <= 64 ? 3 : (half ? 1 : 2); }

// Both gradient passes in one launch, their workgroups interleaved in proportion (neither
// reads the other's output).  Workgroups are dealt to the eight XCDs in turn (block b runs
// on XCD b % 8), so the interleaving is done within each XCD's blocks and a pass's work
// item number keeps its residue: items with one (sequence, K/V head) fastest stay on few
// XCDs, whose L2 then holds what they walk over.  Item order: heaviest tiles first.
template <typename T, int DP, int MK, bool HALF>
__global__ __launch_bounds__(BWD_THREADS, bwd_waves(DP, HALF)) void attn_bwd_tile_kernel(const BwdParams p, const BwdGrid gr) {
    constexpr size_t DQ_BYTES = 4 * sizeof(T) * Tile<T, DP, 64>::ELEMS;
    constexpr size_t KV_BYTES = sizeof(DkdvShared<T, DP, HALF>);
    __shared__ __align__(1024) unsigned char sh[KV_BYTES > DQ_BYTES ? KV_BYTES : DQ_BYTES];
    const int x = blockIdx.x & 7, s = blockIdx.x >> 3;
    const int per_q = (gr.nq + 7) >> 3, per_k = (gr.nk + 7) >> 3, tot = per_q + per_k;
    const int q0 = static_cast<int>(static_cast<int64_t>(s) * per_q / tot);
    const int q1 = static_cast<int>(static_cast<int64_t>(s + 1) * per_q / tot);
    const int units = p.batch * p.hkv;
    if (q1 > q0) {
        const int i = 8 * q0 + x;
        if (i >= gr.nq) return;
        const int rest = i / units, unit = i - rest * units;
        const int t = rest / p.ksplit, ks = rest - t * p.ksplit;
        const int tile = p.causal ? gr.tiles_q - 1 - t : t;
        if (gr.half_q)
            bwd_dq<T, DP, MK, 2>(p, sh, tile, ks, unit);
        else
            bwd_dq<T, DP, MK, 4>(p, sh, tile, ks, unit);
    } else {
        const int i = 8 * (s - q0) + x;
        if (i >= gr.nk) return;
        const int rest = i / units, unit = i - rest * units;
        const int t = rest / p.splits, sp = rest - t * p.splits;
        bwd_dkdv<T, DP, MK, HALF>(p, sh, t, sp, unit);
    }
}

template <typename T, int DP, int MK>
hipError_t launch_tile_mk(const BwdParams& p, const BwdGrid& gr, hipStream_t s) {
    const int per = (gr.nq + 7) / 8 + (gr.nk + 7) / 8;
    const dim3 grid(static_cast<unsigned>(8 * per)), block(BWD_THREADS);
    if constexpr (DP > 64) {
        if (!gr.half_k) {
            hipLaunchKernelGGL((attn_bwd_tile_kernel<T, DP, MK, false>), grid, block, 0, s, p, gr);
            return hipGetLastError();
        }
    }
    hipLaunchKernelGGL((attn_bwd_tile_kernel<T, DP, MK, true>), grid, block, 0, s, p, gr);
    return hipGetLastError();
}

template <typename T, int DP>
hipError_t launch_tile(const BwdParams& p, const BwdGrid& gr, int mk, hipStream_t s) {
    switch (mk) {
        case MK_NONE: return launch_tile_mk<T, DP, MK_NONE>(p, gr, s);
        case MK_BOOL: return launch_tile_mk<T, DP, MK_BOOL>(p, gr, s);
        case MK_BF16: return launch_tile_mk<T, DP, MK_BF16>(p, gr, s);
        case MK_F16: return launch_tile_mk<T, DP, MK_F16>(p, gr, s);
        default: return launch_tile_mk<T, DP, MK_F32>(p, gr, s);
    }
}

}  // namespace bwd
}  // namespace kmi
