// Building blocks of the 32x32x16 MFMA attention kernels (attention_tile.hpp,
// attention_bwd_tile.hpp): the MFMA wrappers, LDS DMA and the swizzled operand tile.
#pragma once

#include <type_traits>

#include "common.hpp"

namespace kmi {

typedef float f32x16 __attribute__((ext_vector_type(16)));

template <typename T>
struct Mfma32;
template <>
struct Mfma32<bf16> {
    typedef bf16x8 v8;
    static __device__ __forceinline__ f32x16 run(v8 a, v8 b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    }
};
template <>
struct Mfma32<f16> {
    typedef f16x8 v8;
    static __device__ __forceinline__ f32x16 run(v8 a, v8 b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
    }
};

// gfx950's transposed LDS read: within each 16-lane group, output lane j, slot s receives
// element j % 4 of the 4-element chunk that source lane 4 s + j / 4 addressed.
template <typename T>
__device__ __forceinline__ u32x2 lds_tr(uint32_t at) {
    if constexpr (std::is_same<T, bf16>::value) {
        typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 x4;
        return __builtin_bit_cast(u32x2,
                                  __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) x4*)(at)));
    } else {
        typedef __attribute__((__vector_size__(4 * sizeof(__fp16)))) __fp16 x4;
        return __builtin_bit_cast(u32x2,
                                  __builtin_amdgcn_ds_read_tr16_b64_v4f16((__attribute__((address_space(3))) x4*)(at)));
    }
}

// LDS DMA: every lane's 16 (or 4) bytes at byte offset `off` of the resource (zeros past
// its range) go to LDS at dst + 16 (4) lane.  Written as asm because the compiler takes
// every transposed LDS read for a use of every load of this kind in flight and waits for
// all of them first, which would end each prefetch at the next read (C1 backward's dK / dV
// loop had one such wait per 32 rows).  The loops below wait for a tile themselves (all of
// vmcnt) before the barrier that publishes it.
//
// The compiler does not see the load inside the asm, so the asm holds the wait states itself:
// one between a write of m0 and its use, and five between a VALU write of the resource's
// registers (readfirstlane, or a reload of spilled ones, which the compiler may put right
// before the asm) and the load that reads them: the move and a nop of four.  Every load holds
// them, since nothing ties the resource to its registers from one load to the next.
__device__ __forceinline__ u32x4 dma_rsrc(const void* base, uint32_t bytes) {
    // (Uniform; readfirstlane keeps it in scalar registers where the compiler cannot tell.)
    const uint64_t a = reinterpret_cast<uint64_t>(base);
    return u32x4{static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<uint32_t>(a))),
                 static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<uint32_t>(a >> 32))) & 0xffffu,
                 static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(bytes)), 0x00020000u};
}
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
    return static_cast<uint32_t>(
        reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) char*)(static_cast<const char*>(p))));
}
__device__ __forceinline__ void dma16(u32x4 rs, uint32_t off, uint32_t dst) {
    __asm__ volatile("s_mov_b32 m0, %2\n\ts_nop 3\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds"
                     :
                     : "v"(off), "s"(rs), "s"(dst)
                     : "memory", "m0");
}
__device__ __forceinline__ void dma4(u32x4 rs, uint32_t off, uint32_t dst) {
    __asm__ volatile("s_mov_b32 m0, %2\n\ts_nop 3\n\tbuffer_load_dword %0, %1, 0 offen lds"
                     :
                     : "v"(off), "s"(rs), "s"(dst)
                     : "memory", "m0");
}

// A [TR][DP] tile in LDS: rows of NCH 16-byte chunks (a power of two; at DP = 96 and 192 the
// last quarter stays zero), chunk c of row r at c ^ swz(r).  LDS reads take 256 bytes a cycle from
// 64 banks: 16 lanes of a b128 row read (16 rows, one column) and 32 lanes of a transposed
// read (4 rows of 4 chunks, or 8 rows of 2).  With r0 .. r3 the low bits of the row, the
// swizzles below put each of those sets on distinct banks (a row of 128 or 64 bytes already
// takes its half or quarter of the banks from r0, or r0 and r1).
template <typename T, int DP, int TR>
struct Tile {
    typedef typename Mfma32<T>::v8 v8;
    static constexpr int NCH = DP <= 32 ? 4 : (DP <= 64 ? 8 : (DP <= 128 ? 16 : 32));
    static constexpr int PITCH = 8 * NCH;
    static constexpr int ELEMS = TR * PITCH;
    // DMA: one instruction fills 1 KiB (RPI rows); wavefront w fills rows RW w .. + RW - 1.
    static constexpr int RPI = kWave / NCH;
    static constexpr int RW = TR / 4 < RPI ? RPI : TR / 4;
    static constexpr int IPW = RW / RPI;
    static constexpr int NRA = NCH / 2, NTA = NCH / 4;
    static constexpr uint32_t kNoChunk = 0x80000000u;  // past every range (below 2^31 bytes)

    static __device__ __forceinline__ int swz(int r) {
        const int r1 = (r >> 1) & 1, r2 = (r >> 2) & 1, r3 = (r >> 3) & 1;
        return NCH == 4 ? 2 * r2 + r3 : (NCH == 8 ? 4 * r1 + 2 * r2 + r3 : 4 * (r & 3) + 2 * r2 + r3);
    }

    // A lane's place in a DMA instruction's RPI rows: its row's byte offset, and the chunk it
    // reads in instruction 0 (instruction i, rows RPI i .., reads chunk ^ swz(RPI i)).
    struct Offs {
        uint32_t row, chunk;
    };
    static __device__ __forceinline__ Offs offs(int lane, uint32_t stride) {
        const int r = lane / NCH;
        return Offs{static_cast<uint32_t>(r) * stride, static_cast<uint32_t>((lane % NCH) ^ swz(r))};
    }
    // Requests rows [row0 + RW wave, + RW) of an [nrows, row_bytes] operand (row stride
    // `stride` bytes, below 2^26) into the tile at LDS address dst; rows at or past nrows
    // read zeros.
    static __device__ __forceinline__ void request(const char* base, uint32_t stride, int row0, int nrows, int row_bytes,
                                                   const Offs& off, int wave, uint32_t dst) {
        if (RW * wave >= TR) return;
        const int first = row0 + RW * wave;
        const u32x4 rs = dma_rsrc(base + static_cast<int64_t>(first) * stride,
                                  rows_extent(min(RW, nrows - first), stride, static_cast<uint32_t>(row_bytes)));
        const uint32_t at = __builtin_amdgcn_readfirstlane(dst + RW * wave * PITCH * static_cast<uint32_t>(sizeof(T)));
        // (The offsets are formed per tile: held across the loop they would cost registers.)
        uint32_t x0 = swz(RW * wave);
        __asm__ volatile("" : "+s"(x0));
#pragma unroll
        for (int i = 0; i < IPW; ++i) {
            const uint32_t c = 16u * (off.chunk ^ x0 ^ swz(RPI * i));  // chunks past the row read zeros
            dma16(rs, c < static_cast<uint32_t>(row_bytes) ? off.row + static_cast<uint32_t>(i * RPI) * stride + c : kNoChunk,
                  at + i * RPI * PITCH * static_cast<uint32_t>(sizeof(T)));
        }
    }

    // Lane byte addresses of the operand reads, relative to a tile's first row; tiles start at
    // multiples of a row's bytes, so that a chunk's swizzled place is an XOR of low bits.
    struct Addr {
        uint32_t row;      // A operand: row l32, dims 8 h ..
        uint32_t tr0, tr1; // A operand transposed: dims lane % 32, rows 4 h + s and 8 + 4 h + s
    };
    static __device__ __forceinline__ Addr addr(int lane) {
        const int l32 = lane & 31, h = lane >> 5, k = lane & 15, dh = (lane >> 4) & 1;
        auto tr = [&](int r) {
            return static_cast<uint32_t>(2 * (r * PITCH + 8 * ((2 * dh + ((k & 3) >> 1)) ^ swz(r)) + 4 * (k & 1)));
        };
        return Addr{static_cast<uint32_t>(2 * (l32 * PITCH + 8 * (h ^ swz(l32)))), tr(4 * h + (k >> 2)),
                    tr(8 + 4 * h + (k >> 2))};
    }
    // Rows l32, dims 16 c + 8 h .. + 7 at LDS address ra (+ imm, a constant).
    static __device__ __forceinline__ v8 rows(uint32_t ra, int c, uint32_t imm) {
        return *(const __attribute__((address_space(3))) v8*)((ra ^ (32u * c)) + imm);
    }
    // Dims 32 b + lane % 32, rows 16 kc + {4 h + s, 8 + 4 h + s}: the k order of an
    // accumulator's registers 8 kc .. + 7 as a B operand.
    static __device__ __forceinline__ v8 cols(uint32_t t0, uint32_t t1, int kc, int b, uint32_t imm) {
        const uint32_t at = imm + 2u * 16 * kc * PITCH;
        const u32x2 lo = lds_tr<T>((t0 ^ (64u * b)) + at), hi = lds_tr<T>((t1 ^ (64u * b)) + at);
        return __builtin_bit_cast(v8, u32x4{lo[0], lo[1], hi[0], hi[1]});
    }
};

// A loaded mask element as a logit: a kept key's value, anything at or below kMaskedLogit for a
// masked key (mask_logit_of without its clamp, which only the raw-score rows of the 16x16
// kernels need).
template <int MK, typename R>
__device__ __forceinline__ float mask_value_of(R raw) {
    if constexpr (MK == MK_BF16) {
        const uint32_t mag = __builtin_bit_cast(uint16_t, raw) & 0x7fffu;
        return mag > 0x7f80u ? kMaskedLogit : static_cast<float>(__builtin_bit_cast(bf16, raw));
    } else if constexpr (MK == MK_F16) {
        const uint32_t mag = __builtin_bit_cast(uint16_t, raw) & 0x7fffu;
        return mag > 0x7c00u ? kMaskedLogit : static_cast<float>(__builtin_bit_cast(f16, raw));
    } else if constexpr (MK == MK_F32) {
        const uint32_t mag = __builtin_bit_cast(uint32_t, raw) & 0x7fffffffu;
        return mag > 0x7f800000u ? kMaskedLogit : raw;
    } else {
        return mask_logit_of<MK>(raw);
    }
}

// A masked call's scaled score (base 2) from the whole product s: a kept key's logit joins in
// one rounding; a masked key's is minus infinity whatever its product holds (a select, since
// the product may be NaN or infinite).
__device__ __forceinline__ float masked_score(float s, float c2, float logit) {
    return logit > kMaskedLogit ? logit * 1.4426950408889634f + s * c2 : -INFINITY;
}

template <typename T>
__device__ __forceinline__ f32x16 splat16(T x) {
    f32x16 v;
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = x;
    return v;
}

}  // namespace kmi
