// Decoders of the reference's 32-lane layouts: the bit reader of the batched MoE kernel and of GEMVs that keep every CU
// full (the other GEMVs, dequant and row gather have their own, lane_ring) and what both share.
#pragma once

#include "bf16n_c.h"
#include "dev_common.h"

namespace bf16n {
namespace dev {

struct hp_ptrs { const uint8_t * plane; const uint32_t * lut; const uint32_t * ubase; const uint16_t * lrel; const uint32_t * stream; };
struct huf_ptrs { const uint8_t * plane; const uint32_t * lut; const uint32_t * lane_off; const uint32_t * stream; };
struct nib_ptrs { const uint8_t * plane; const uint8_t * codes; const uint8_t * table; const uint32_t * esc_off; const uint32_t * esc; };

__device__ __forceinline__ hp_ptrs hpp(const bf16n_weight & w) {
    return {w.plane, (const uint32_t *) (w.aux + w.off_a), (const uint32_t *) (w.aux + w.off_b),
            (const uint16_t *) (w.aux + w.off_c), (const uint32_t *) (w.aux + w.off_d)};
}
__device__ __forceinline__ huf_ptrs hufp(const bf16n_weight & w) {
    return {w.plane, (const uint32_t *) (w.aux + w.off_a), (const uint32_t *) (w.aux + w.off_b),
            (const uint32_t *) (w.aux + w.off_c)};
}
__device__ __forceinline__ nib_ptrs nibp(const bf16n_weight & w, int64_t shift_rows) {
    // the up half of a merged [gate; up] matrix: every per-row array shifted by shift_rows (escape offsets are absolute)
    return {w.plane + shift_rows * w.K, w.aux + w.off_a + shift_rows * (w.K / 2), w.aux + w.off_b + shift_rows * 16,
            (const uint32_t *) (w.aux + w.off_c) + shift_rows, (const uint32_t *) (w.aux + w.off_d)};
}

// MSB-first bit buffer over one lane stream: `v` valid bits at the top of `buf`, one word of lookahead in `nxt`.
// Two table lookups (<= 24 bits) are always covered because v > 32 after every refill.  The stream buffers end with
// padding words, so the lookahead never leaves the allocation.
struct lane_bits {
    const uint32_t * sp;
    uint64_t buf;
    uint32_t nxt;
    int v;
    __device__ __forceinline__ void begin(const uint32_t * p) {
        sp = p;
        buf = ((uint64_t) sp[0] << 32) | sp[1];
        nxt = sp[2];
        sp += 3;
        v = 64;
    }
    template <int BITS>
    __device__ __forceinline__ uint32_t take(const uint32_t * lut) {
        const uint32_t ent = lut[(uint32_t) (buf >> (64 - BITS))];
        const int len = (int) (ent & 31u);
        buf <<= len;
        v -= len;
        return ent;
    }
    __device__ __forceinline__ void refill() {
        if (v <= 32) {
            buf |= (uint64_t) nxt << (32 - v);
            v += 32;
            nxt = *sp++;
        }
    }
};

// the 16 weights of one lane in one chunk as 8 BF16 pairs: wp[2j], wp[2j+1] = columns 128j + 4l + {0,1}, {2,3}
template <int FORMAT>
__device__ __forceinline__ void decode_chunk(lane_bits & bits, const uint32_t * lut, const uint4 sm, uint32_t (&wp)[8]) {
    const uint32_t smw[4] = {sm.x, sm.y, sm.z, sm.w};
    if (FORMAT == FMT_HUFPAIR) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint32_t e0 = bits.take<HP_LP>(lut);
            const uint32_t e1 = bits.take<HP_LP>(lut);
            bits.refill();
            wp[2 * j] = merge(spread_lo(smw[j]), e0);
            wp[2 * j + 1] = merge(spread_hi(smw[j]), e1);
        }
    } else { // single exponents, entry = len | exponent << 7
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint32_t a = bits.take<HUF_LMAX>(lut), b = bits.take<HUF_LMAX>(lut);
            bits.refill();
            const uint32_t c = bits.take<HUF_LMAX>(lut), d = bits.take<HUF_LMAX>(lut);
            bits.refill();
            wp[2 * j] = merge(spread_lo(smw[j]), (a & 0x7F80u) | ((b & 0x7F80u) << 16));
            wp[2 * j + 1] = merge(spread_hi(smw[j]), (c & 0x7F80u) | ((d & 0x7F80u) << 16));
        }
    }
}

// ---------------------------------------------------------------- NIBBLE (shared by the GEMV / dequant kernels and the batched kernels)

// The exponents of 8 adjacent columns from their 8 nibble codes and the row's 16-byte table: even has those of columns
// 0, 2, 4, 6 as bytes, odd those of columns 1, 3, 5, 7.  The even and the odd nibbles of the word are selectors of a byte
// permute as they stand (masked to the 8 bytes of half a table); bit 3 of a code picks between the two halves' answers
// in a third permute.  13 instructions for 8 codes.
__device__ __forceinline__ uint32_t nib_pick4(const uint4 T, uint32_t c, uint32_t c_shr1) {
    const uint32_t s = c & 0x07070707u;
    const uint32_t lo = __builtin_amdgcn_perm(T.y, T.x, s), hi = __builtin_amdgcn_perm(T.w, T.z, s);
    return __builtin_amdgcn_perm(hi, lo, (c_shr1 & 0x04040404u) | 0x03020100u);
}
__device__ __forceinline__ void nib_lookup8(const uint4 T, uint32_t codes, uint32_t & even, uint32_t & odd) {
    even = nib_pick4(T, codes, codes >> 1);
    odd = nib_pick4(T, codes >> 4, codes >> 5);
}

// a row's table with every byte rotated right by one: bit 7 of a byte is the exponent's lowest bit
__device__ __forceinline__ uint32_t nib_rotate4(uint32_t t) { return ((t >> 1) & 0x7F7F7F7Fu) | ((t << 7) & 0x80808080u); }
__device__ __forceinline__ uint4 nib_rotated(const uint4 T) {
    return make_uint4(nib_rotate4(T.x), nib_rotate4(T.y), nib_rotate4(T.z), nib_rotate4(T.w));
}

// the 16 weights of one lane in one NIBBLE chunk.  ROT: T is the row's rotated table: an exponent duplicated into both
// bytes of its half then has every bit where merge() wants it, which saves the shift of each pair; for rows of which a
// lane decodes several chunks (rotating the table costs as much as one and a half chunks save).  50 instructions (58
// without ROT) where a shift, a widening and a multiply per four codes took 84; by itself that moved no launch by more
// than 0.5 % (they wait for their loads).
template <bool ROT = false>
__device__ __forceinline__ void nib_chunk(const uint4 sm, const uint2 cd, const uint4 T, uint32_t (&wp)[8]) {
    const uint32_t smw[4] = {sm.x, sm.y, sm.z, sm.w}, cw[2] = {cd.x, cd.y};
#pragma unroll
    for (int i = 0; i < 2; i++) {
        uint32_t even, odd;
        nib_lookup8(T, cw[i], even, odd);
#pragma unroll
        for (int p = 0; p < 4; p++) { // columns 2 p and 2 p + 1 of the eight
            const uint32_t sel = ROT ? 0x04040000u + 0x01010101u * p : 0x0c040c00u + 0x00010001u * p;
            const uint32_t e = __builtin_amdgcn_perm(odd, even, sel), s = smw[2 * i + (p >> 1)];
            wp[4 * i + p] = merge(p & 1 ? spread_hi(s) : spread_lo(s), ROT ? e : e << 7);
        }
    }
}

__device__ __forceinline__ uint32_t esc_bits(uint32_t rec) { // BF16 bits of an escape record col | sm << 12 | exponent << 20
    const uint32_t smb = (rec >> 12) & 0xFFu, ex = rec >> 20;
    return ((smb & 0x80u) << 8) | (ex << 7) | (smb & 0x7Fu);
}

} // namespace dev
} // namespace bf16n
