// Kernels for the reference's 32-lane layouts: HUFPAIR row-/chunk-major, HUFFMAN and NIBBLE (GEMV, GLU-GEMV, exact
// dequant, row gather).  Buffers made by the reference encoder decode here unchanged.
//
// A wave64 carries two units (HUFPAIR / HUFFMAN) or two rows (NIBBLE): lanes 0..31 the even one, lanes 32..63 the odd
// one; each half reads its 512-byte plane chunk with one 16-byte load per lane, four chunks ahead.  Lane streams pass
// through rings in LDS (lane_ring), except in products with enough wavefronts to cover each other's misses (huf_direct).
// Dense products and exact rows of few HUFPAIR units take a block per unit instead (k_hp_split).
// These kernels take any K, R, layout, expert ids and FP32 or BF16 activations; the wave64 layout (kernels_w64.hip),
// which has twice the chains per unit, is the fast path.
#include "dev_common.h"
#include "dev_compat.h"
#include "dev_norm.h"
#include "launchers.h"

#include <algorithm>
#include <type_traits>

namespace bf16n {
namespace dev {

namespace {

constexpr int NT = 256;          // threads per block
constexpr int NIB_MM_MIN_COLS = 5; // dense NIBBLE batches of BF16 columns go through the matrix cores from this many on at the earliest
constexpr int HALVES = NT / 32;  // units (rows) per block
constexpr int LUT_PAIRS = 1 << HP_LP;

// One lane's MSB-first bit stream, read through a ring of 16 words in LDS.  What bounds these kernels is the chain of
// one unit (two dependent table lookups per two codes, all lanes of a half-wave in step), so nothing else may be waited
// for in it: 64 lanes read 64 cache lines, and with the next word loaded where it is needed nearly every pair of codes
// waited for some lane's cache miss (one column of 8192 x 2048, R = 16, a chain each: 77.7 us then, 39.6 now, about 15 of the
// difference by the ring, the rest by plane chunks ahead, small blocks, sums on the VALU and loads that the compiler knows to be
// global; 65536 x 4096: 266 and 143; dequant of the first 88 and 34).  Here a lane loads whole 16-byte blocks, one per four code pairs (96 bits at most, less than a block), LOOK blocks beyond the one it reads, and stores
// what it loaded DEEP rounds ago; the same block again while it has not moved on.  The stream buffers end with padding
// words (32 of HUFPAIR, 16 of HUFFMAN): the last lane reads at most 17 (13) words past its end.
constexpr int LR_WORDS = 16;                     // ring words per lane
constexpr int LR_BYTES = LR_WORDS * 64 * 4;      // per wavefront: word i of a lane at [i % 16][lane]
template <int FORMAT> struct lane_ring {
    static constexpr int BITS = FORMAT == FMT_HUFPAIR ? HP_LP : HUF_LMAX;
    static constexpr int DEEP = FORMAT == FMT_HUFPAIR ? 2 : 1, LOOK = DEEP + 1;
    const uint4 * src;    // the block that holds the lane's first word
    uint32_t * ring;      // this lane's column of the ring
    uint32_t w0, w1, nw;  // the next 32 bits are bits s.. of w0:w1; nw: the word after w1
    int s;                // unread bits of w0 (0: it is used up)
    uint32_t p;           // index of nw, counted from src
    uint4 f[DEEP];        // blocks in flight
    uint32_t fb[DEEP];    // their indices
    __device__ __forceinline__ void put(uint32_t b, const uint4 v) {
        uint32_t * r = ring + (b & 3) * 256;
        r[0] = v.x; r[64] = v.y; r[128] = v.z; r[192] = v.w;
    }
    __device__ __forceinline__ uint32_t word(uint32_t i) const { return ring[(i & (LR_WORDS - 1)) * 64]; }
    __device__ __forceinline__ void begin(const uint32_t * sp, uint32_t * ring_) {
        src = (const uint4 *) (sp - ((uintptr_t) sp >> 2 & 3)); // (as a number it would lose its address space)
        ring = ring_;
        uint4 b[LOOK + 1];
#pragma unroll
        for (int i = 0; i <= LOOK; i++) {
            b[i] = src[i];
        }
#pragma unroll
        for (int i = 0; i <= LOOK; i++) {
            put(i, b[i]);
        }
#pragma unroll
        for (int i = 0; i < DEEP; i++) {
            f[i] = b[LOOK];
            fb[i] = LOOK;
        }
        p = ((uint32_t) ((uintptr_t) sp & 15) >> 2) + 1;
        w0 = 0;
        w1 = word(p - 1);
        nw = word(p);
        s = 0;
    }
    __device__ __forceinline__ void round(int i) { // before every four code pairs; i: a compile-time counter
        put(fb[i % DEEP], f[i % DEEP]);
        fb[i % DEEP] = (p >> 2) + LOOK;
        f[i % DEEP] = src[fb[i % DEEP]];
    }
    __device__ __forceinline__ void two(const uint32_t * lut, uint32_t & e0, uint32_t & e1) {
        const uint32_t W = __builtin_amdgcn_alignbit(w0, w1, (uint32_t) s);
        e0 = lut[W >> (32 - BITS)];
        e1 = lut[(W << (e0 & 31u)) >> (32 - BITS)];
        s -= (int) ((e0 + e1) & 31u); // (bits 5 and 6 of an entry are zero, two codes at most 24 bits)
        const bool m = s < 0;
        s += m ? 32 : 0;
        w0 = m ? w1 : w0;
        w1 = m ? nw : w1;
        p += m ? 1 : 0;
        nw = word(p);
    }
    // the 16 weights of the lane in one chunk as 8 BF16 pairs, columns 128 j + 4 l + {0, 1}, {2, 3}; i: chunk counter
    __device__ __forceinline__ void chunk(int i, const uint32_t * lut, const uint4 sm, uint32_t (&wp)[8]) {
        const uint32_t smw[4] = {sm.x, sm.y, sm.z, sm.w};
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (FORMAT == FMT_HUFPAIR) {
                uint32_t e0, e1;
                if (j == 0) {
                    round(i);
                }
                two(lut, e0, e1);
                wp[2 * j] = merge(spread_lo(smw[j]), e0);
                wp[2 * j + 1] = merge(spread_hi(smw[j]), e1);
            } else { // single exponents, entry = len | exponent << 7
                uint32_t a, b, c, d;
                if (j % 2 == 0) {
                    round(0);
                }
                two(lut, a, b);
                two(lut, c, d);
                wp[2 * j] = merge(spread_lo(smw[j]), (a & 0x7F80u) | ((b & 0x7F80u) << 16));
                wp[2 * j + 1] = merge(spread_hi(smw[j]), (c & 0x7F80u) | ((d & 0x7F80u) << 16));
            }
        }
    }
};

// the chunks [0, n) of a half-wave's unit in stream order, four plane chunks in flight: f(chunk, weights), and before a
// chunk is decoded pre().  RING = false: the lanes read their streams and the plane where they need them (lane_bits),
// for launches with enough wavefronts to wait beside each other (huf_direct)
template <int FORMAT, bool RING = true, typename P, typename F>
__device__ __forceinline__ void for_chunks(const uint8_t * plane, const uint32_t * sp, uint32_t * ring, const uint32_t * lut, int n, int l32, P pre, F f) {
    constexpr int D = 4;
    const uint4 * pl = (const uint4 *) plane + l32;
    if constexpr (!RING) {
        lane_bits bits;
        bits.begin(sp);
        for (int o = 0; o < n; o++) {
            uint32_t wp[8];
            decode_chunk<FORMAT>(bits, lut, pl[o * 32], wp);
            pre();
            f(o, wp);
        }
        return;
    }
    uint4 sm[D];
#pragma unroll
    for (int i = 0; i < D; i++) {
        sm[i] = pl[(i < n ? i : n - 1) * 32];
    }
    lane_ring<FORMAT> bits;
    bits.begin(sp, ring);
    auto one = [&](int o, int i) {
        uint32_t wp[8];
        pre();
        bits.chunk(i, lut, sm[i], wp);
        sm[i] = pl[(o + i + D < n ? o + i + D : n - 1) * 32]; // (past the end the last chunk again, unused)
        f(o + i, wp);
    };
    int o = 0;
#pragma unroll 1
    for (; o + D <= n; o += D) { // (no exit inside: the waits for loads in flight stay exact)
#pragma unroll
        for (int i = 0; i < D; i++) {
            one(o, i);
        }
    }
#pragma unroll
    for (int i = 0; i < D - 1; i++) {
        if (o + i < n) {
            one(o, i);
        }
    }
}

template <typename TX>
__device__ __forceinline__ float x_at(const char * x, int i);
template <> __device__ __forceinline__ float x_at<float>(const char * x, int i) { return ((const float *) x)[i]; }
template <> __device__ __forceinline__ float x_at<bf16_t>(const char * x, int i) { return bf16_bits_to_f32(((const uint16_t *) x)[i]); }

template <typename TX>
__device__ __forceinline__ float4 x_four(const char * x, int i);
template <> __device__ __forceinline__ float4 x_four<float>(const char * x, int i) { return ((const float4 *) x)[i]; }
template <> __device__ __forceinline__ float4 x_four<bf16_t>(const char * x, int i) {
    const uint2 v = ((const uint2 *) x)[i];
    return make_float4(__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xFFFF0000u), __uint_as_float(v.y << 16), __uint_as_float(v.y & 0xFFFF0000u));
}

__device__ __forceinline__ float dot_chunk(const uint32_t (&wp)[8], const float4 (&x)[4]) {
    float a0 = 0.f, a1 = 0.f, a2 = 0.f, a3 = 0.f;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        a0 = fmaf(bf16_bits_to_f32(wp[2 * j] & 0xFFFFu), x[j].x, a0);
        a1 = fmaf(__uint_as_float(wp[2 * j] & 0xFFFF0000u), x[j].y, a1);
        a2 = fmaf(bf16_bits_to_f32(wp[2 * j + 1] & 0xFFFFu), x[j].z, a2);
        a3 = fmaf(__uint_as_float(wp[2 * j + 1] & 0xFFFF0000u), x[j].w, a3);
    }
    return (a0 + a1) + (a2 + a3);
}

// the activations a lane meets in a chunk, from LDS (or from where they came): as FP32, or as BF16 (several columns)
template <typename TX> struct x_lds;
template <> struct x_lds<float> {
    float4 v[4];
    __device__ __forceinline__ void load(const float * xs, int col0) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            v[j] = *(const float4 *) (xs + col0 + 128 * j);
        }
    }
    __device__ __forceinline__ float4 get(int j) const { return v[j]; }
    __device__ __forceinline__ static float store(const char * x, int i) { return ((const float *) x)[i]; }
};
template <> struct x_lds<bf16_t> {
    uint2 v[4];
    __device__ __forceinline__ void load(const uint16_t * xs, int col0) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            v[j] = *(const uint2 *) (xs + col0 + 128 * j);
        }
    }
    __device__ __forceinline__ float4 get(int j) const { return x_four<bf16_t>((const char *) v, j); }
    __device__ __forceinline__ static uint16_t store(const char * x, int i) { return ((const uint16_t *) x)[i]; }
};

// One unit of R rows: y[rr] (rr < R) of column n ends up in mine[n] of lane rr of the half-wave.  Row-major streams finish a
// row every C chunks; chunk-major streams add one partial sum per (chunk, row).  Column n's activations: xs + n * K.
template <int FORMAT, bool RING, int NC, typename XL, typename XS>
__device__ __forceinline__ void unit_dot(const uint8_t * plane, const uint32_t * lut, const uint32_t * sp, uint32_t * ring, int64_t gu, int R,
                                         int C, bool cm, const XS * xs, int l32, float (&mine)[NC]) {
    const bool upper = (threadIdx.x & 32) != 0;
    auto sum = [&](float v) { // over the half-wave, on the VALU (lanes 31 and 63 get the sums)
        const int t = __builtin_bit_cast(int, half_wave_sum_dpp(v));
        const int lo = __builtin_amdgcn_readlane(t, 31), hi = __builtin_amdgcn_readlane(t, 63);
        return __builtin_bit_cast(float, upper ? hi : lo);
    };
    float acc[NC];
#pragma unroll
    for (int n = 0; n < NC; n++) {
        mine[n] = acc[n] = 0.f;
    }
    int rr = 0, c = 0;
    XL x[NC]; // the chunk's activations, requested before its chain of lookups (8192 x 2048, one column: 3 us)
    for_chunks<FORMAT, RING>(plane + gu * R * (int64_t) C * CHUNK, sp, ring, lut, R * C, l32, [&] {
#pragma unroll
        for (int n = 0; n < NC; n++) {
            x[n].load(xs + n * C * CHUNK, c * CHUNK + 4 * l32);
        }
        __builtin_amdgcn_sched_barrier(0);
    }, [&](int, const uint32_t (&wp)[8]) {
        float d[NC];
#pragma unroll
        for (int n = 0; n < NC; n++) {
            float4 xv[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                xv[j] = x[n].get(j);
            }
            d[n] = dot_chunk(wp, xv);
        }
        if (cm) {
#pragma unroll
            for (int n = 0; n < NC; n++) {
                const float v = sum(d[n]);
                mine[n] += l32 == rr ? v : 0.f;
            }
            rr = rr + 1 < R ? rr + 1 : 0;
            c += rr == 0;
        } else {
#pragma unroll
            for (int n = 0; n < NC; n++) {
                acc[n] += d[n];
            }
            c = c + 1 < C ? c + 1 : 0;
            if (c == 0) {
#pragma unroll
                for (int n = 0; n < NC; n++) {
                    const float v = sum(acc[n]);
                    mine[n] = l32 == rr ? v : mine[n];
                    acc[n] = 0.f;
                }
                rr++;
            }
        }
    });
}

template <int FORMAT>
__device__ __forceinline__ const uint32_t * lane_stream(const bf16n_weight & w, int64_t gu, int l32) {
    if (FORMAT == FMT_HUFPAIR) {
        const hp_ptrs p = hpp(w);
        return p.stream + p.ubase[gu] + p.lrel[gu * 32 + l32];
    }
    const huf_ptrs p = hufp(w);
    return p.stream + p.lane_off[gu * 32 + l32];
}

// y = W x (GLU: y = silu(gate x) * up x) for HUFPAIR / HUFFMAN in the 32-lane layouts; one half-wave per unit,
// blockIdx.y = NC columns, which share a decode (NC > 1: dense products; columns past the last repeat it and are not stored).
// Shared memory: x [NC][K] as FP32 (several BF16 columns: as they are), then one table per matrix, then (RING) a ring per wavefront.
// What bounds it is the chain of a unit while the device has half-waves to spare, then the lookups; a column more adds 32
// instructions and four LDS reads to a chunk's 140 and sixteen (huf_columns has the times).
template <int FORMAT, typename TX, bool GLU, bool RING, int NC = 1>
__global__ void __launch_bounds__(NT) k_huf_mmv(const bf16n_weight w, const bf16n_weight w_up, const cols p, int ncols) {
    constexpr int LUT_N = FORMAT == FMT_HUFPAIR ? (1 << HP_LP) : (1 << HUF_LMAX);
    typedef typename std::conditional<NC == 1 || sizeof(TX) == 4, float, uint16_t>::type xs_t;
    typedef x_lds<typename std::conditional<NC == 1 || sizeof(TX) == 4, float, bf16_t>::type> xl_t;
    extern __shared__ __align__(16) unsigned char shm_raw[];
    const int K = (int) w.K, C = K / CHUNK, R = w.R;
    xs_t * xs = (xs_t *) shm_raw;
    uint32_t * lut = (uint32_t *) (xs + NC * K);
    uint32_t * lut_up = lut + LUT_N;
    uint32_t * ring = lut + (GLU ? 2 : 1) * LUT_N + (threadIdx.x >> 6) * (LR_BYTES / 4) + (threadIdx.x & 63);
    const int nt = (int) blockDim.x, col0 = (int) blockIdx.y * NC;
    const col_view cv = col_setup(p, col0);
    // (many loads in flight: the smallest blocks are one wavefront)
#pragma unroll 16
    for (int i = threadIdx.x; i < LUT_N; i += nt) {
        lut[i] = ((const uint32_t *) (w.aux + w.off_a))[i];
    }
    if (GLU) {
#pragma unroll 16
        for (int i = threadIdx.x; i < LUT_N; i += nt) {
            lut_up[i] = ((const uint32_t *) (w_up.aux + w_up.off_a))[i];
        }
    }
#pragma unroll
    for (int n = 0; n < NC; n++) {
        const char * x = cv.x + (col0 + n < ncols ? n : ncols - 1 - col0) * p.x_tok;
#pragma unroll 8
        for (int i = threadIdx.x; i < K; i += nt) {
            if constexpr (NC == 1) {
                xs[i] = x_at<TX>(cv.x, i);
            } else {
                xs[n * K + i] = xl_t::store(x, i);
            }
        }
    }
    __syncthreads();
    const int l32 = threadIdx.x & 31, half = threadIdx.x >> 5, halves = nt >> 5;
    const bool cm = (w.flags & FLAG_CHUNK_MAJOR) != 0;
    const int64_t units = p.nrows / R;
    for (int64_t u0 = (int64_t) blockIdx.x * halves + (half & ~1); u0 < units; u0 += (int64_t) gridDim.x * halves) {
        // (both halves of a wavefront stay together: a missing last unit is decoded twice and stored once)
        const int64_t u = u0 + (half & 1) < units ? u0 + (half & 1) : u0;
        const int64_t gu = cv.rbase / R + u;
        float v[NC];
        unit_dot<FORMAT, RING, NC, xl_t>(w.plane, lut, lane_stream<FORMAT>(w, gu, l32), ring, gu, R, C, cm, xs, l32, v);
        if constexpr (GLU) {
            float uv[NC];
            unit_dot<FORMAT, RING, NC, xl_t>(w_up.plane, lut_up, lane_stream<FORMAT>(w_up, gu, l32), ring, gu, R, C, false, xs, l32, uv);
            v[0] = uv[0] * silu(v[0]);
        }
        if (l32 < R && u == u0 + (half & 1)) {
#pragma unroll
            for (int n = 0; n < NC; n++) {
                if (NC == 1 || col0 + n < ncols) {
                    store_y(cv.y + n * p.y_tok, p.y_bf16, u * R + l32, v[n]);
                }
            }
        }
    }
}

// exact BF16 bits of unit gu, the u-th of the rows at out, by one half-wave
template <int FORMAT>
__device__ __forceinline__ void unit_rows(const bf16n_weight & w, const uint32_t * lut, uint32_t * ring, int64_t gu, int64_t u, int l32, uint16_t * __restrict__ out) {
    const int K = (int) w.K, C = K / CHUNK, R = w.R;
    const bool cm = (w.flags & FLAG_CHUNK_MAJOR) != 0;
    int rr = 0, c = 0;
    for_chunks<FORMAT>(w.plane + gu * R * (int64_t) K, lane_stream<FORMAT>(w, gu, l32), ring, lut, R * C, l32, [] {}, [&](int, const uint32_t (&wp)[8]) {
        uint16_t * dst = out + (u * R + rr) * K + c * CHUNK;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            *(uint2 *) (dst + 128 * j + 4 * l32) = make_uint2(wp[2 * j], wp[2 * j + 1]);
        }
        if (cm) {
            rr = rr + 1 < R ? rr + 1 : 0;
            c += rr == 0;
        } else {
            c = c + 1 < C ? c + 1 : 0;
            rr += c == 0;
        }
    });
}

// exact BF16 bits of rows [row0, row0 + nrows) (whole units), row-major; one half-wave per unit
template <int FORMAT>
__global__ void __launch_bounds__(NT) k_huf_dequant(const bf16n_weight w, int64_t row0, int64_t nrows, uint16_t * __restrict__ out) {
    constexpr int LUT_N = FORMAT == FMT_HUFPAIR ? (1 << HP_LP) : (1 << HUF_LMAX);
    __shared__ uint32_t lut[LUT_N];
    __shared__ uint32_t rings[NT / 64 * LR_BYTES / 4];
    const int nt = (int) blockDim.x;
#pragma unroll 16
    for (int i = threadIdx.x; i < LUT_N; i += nt) {
        lut[i] = ((const uint32_t *) (w.aux + w.off_a))[i];
    }
    __syncthreads();
    const int R = w.R, l32 = threadIdx.x & 31, half = threadIdx.x >> 5, halves = nt >> 5;
    uint32_t * ring = rings + (threadIdx.x >> 6) * (LR_BYTES / 4) + (threadIdx.x & 63);
    for (int64_t u = (int64_t) blockIdx.x * halves + half; u < nrows / R; u += (int64_t) gridDim.x * halves) {
        unit_rows<FORMAT>(w, lut, ring, row0 / R + u, u, l32, out);
    }
}

// dst[i] = row (row0 + ids[i]) as FP32 or BF16: the half-wave decodes the row's unit from its start and stores only
// the requested row (reference kernels.cuh:840-891)
template <bool BF>
__global__ void __launch_bounds__(NT) k_hp_get_rows(const bf16n_weight w, const char * __restrict__ ids, int64_t ids_s0, int64_t n,
                                                    int64_t row0, char * __restrict__ dst, int64_t dst_s1) {
    __shared__ uint32_t lut[1 << HP_LP];
    __shared__ uint32_t rings[NT / 64 * LR_BYTES / 4];
#pragma unroll 16
    for (int i = threadIdx.x; i < (1 << HP_LP); i += NT) {
        lut[i] = ((const uint32_t *) (w.aux + w.off_a))[i];
    }
    __syncthreads();
    const int K = (int) w.K, C = K / CHUNK, R = w.R;
    const int l32 = threadIdx.x & 31, half = threadIdx.x >> 5;
    uint32_t * ring = rings + (threadIdx.x >> 6) * (LR_BYTES / 4) + (threadIdx.x & 63);
    const int64_t i = (int64_t) blockIdx.x * HALVES + half;
    if (i >= n) {
        return;
    }
    const int64_t gr = row0 + *(const int32_t *) (ids + i * ids_s0);
    const int64_t gu = gr / R;
    char * o = dst + i * dst_s1;
    const int chunks = (int) (gr - gu * R + 1) * C; // of the unit, up to the end of the row
    for_chunks<FMT_HUFPAIR>(w.plane + gu * R * (int64_t) K, lane_stream<FMT_HUFPAIR>(w, gu, l32), ring, lut, chunks, l32, [] {},
                            [&](int k, const uint32_t (&wp)[8]) {
        if (k >= chunks - C) {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int col = (k - (chunks - C)) * CHUNK + 128 * j + 4 * l32;
                if (BF) {
                    *(uint2 *) (o + 2 * col) = make_uint2(wp[2 * j], wp[2 * j + 1]);
                } else {
                    *(float4 *) (o + 4 * col) = make_float4(bf16_bits_to_f32(wp[2 * j] & 0xFFFFu), __uint_as_float(wp[2 * j] & 0xFFFF0000u),
                                                            bf16_bits_to_f32(wp[2 * j + 1] & 0xFFFFu), __uint_as_float(wp[2 * j + 1] & 0xFFFF0000u));
                }
            }
        }
    });
}

// ---------------------------------------------------------------- NIBBLE

// the 16 activations one lane meets in a 512-column chunk (columns 128 j + 4 l + 0..3), as FP32
template <typename TX>
__device__ __forceinline__ void x_chunk16(const char * x, int col0, float (&xv)[16]);
template <> __device__ __forceinline__ void x_chunk16<float>(const char * x, int col0, float (&xv)[16]) {
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const float4 t = *(const float4 *) (x + 4 * (col0 + 128 * j));
        xv[4 * j] = t.x; xv[4 * j + 1] = t.y; xv[4 * j + 2] = t.z; xv[4 * j + 3] = t.w;
    }
}
template <> __device__ __forceinline__ void x_chunk16<bf16_t>(const char * x, int col0, float (&xv)[16]) {
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const uint2 t = *(const uint2 *) (x + 2 * (col0 + 128 * j));
        xv[4 * j] = __uint_as_float(t.x << 16); xv[4 * j + 1] = __uint_as_float(t.x & 0xFFFF0000u);
        xv[4 * j + 2] = __uint_as_float(t.y << 16); xv[4 * j + 3] = __uint_as_float(t.y & 0xFFFF0000u);
    }
}

// the 16 weights of one lane in (row gr, chunk c) as 8 BF16 pairs; escaped weights read as +0 here
__device__ __forceinline__ void nib_load_chunk(const nib_ptrs & w, int64_t gr, int C, int c, const uint4 T, int l32, uint32_t (&wp)[8]) {
    const int64_t K = (int64_t) C * CHUNK;
    const uint4 sm = *((const uint4 *) (w.plane + gr * K + c * CHUNK) + l32);
    const uint2 cd = *((const uint2 *) (w.codes + gr * (K / 2) + c * 256) + l32);
    nib_chunk(sm, cd, T, wp);
}

// ---------------------------------------------------------------- HUFPAIR units, a lane's stream in segments
//
// With one half-wave per unit (above) a matrix of few units is the chain of one lane: R K / 64 pair codes one after the other
// on a device that is otherwise idle (8192 x 2048, R = 16: 512 units, two per CU).  Here a block takes a unit and S threads a
// lane's stream, each a segment of its bits.  Where the first code of a segment begins is not stored, but a prefix code falls
// into step by itself after a few codes: every thread decodes from its segment's first bit and notes where the first code
// past its end begins, then again from where the thread before it ended, until no beginning changes any more.  The first
// segment's is known, so all are then exact: after two rounds nearly always, after S at worst (codes of one length never fall
// into step; of normal weights' codes 3 in 100 starts take more than 16, 1 in 1000 more than 32: the first round begins half a
// segment early, 48 codes, because one thread out of step costs its block another round).
// The number of codes in the segments before it gives a thread its place, and a last round writes the exponents to LDS in the
// order of the plane.  The products are those of unit_dot, a row per half-wave, added in the same order: the same bits.
// Codes whose lengths are nearly all multiples of one number keep a wrong phase for long: such tables are told by their lengths
// (falls_into_step), and their units go to one half-wave each in here too (split_whole).  In a run of one code, rows of zeros for
// instance, no thread falls into step: every second round the threads past the first one that still moves take their phase from
// the code that begins there, if the next three are the same and four like it stand where they would begin (14 of 16 rows of
// 4096, one unit of 64: 136 us with a round per segment, 39 so, 80 in k_huf_mmv; without the look at their own place the threads
// past the run were put out of step as well: 51, and a row of zeros here and there 34.6 for 28.7; the threads before it are exact,
// and it gains one a round, so S rounds are enough).
// Two rounds and a half of a sixteenth of the chain instead of the chain, for as many lookups per code: for launches that wait for
// the chain (hp_split_cols).  8192 x 2048, one column: 39.6 -> 24.7 us (7 more with a third round that wrote the exponents: the
// codes of the second stay in registers until their place is known).
constexpr int SPLIT_PAIRS = 32;                  // pair codes per segment at most
constexpr int SPLIT_PAD = 4;                     // words in front of and behind the staged streams
constexpr int SPLIT_KEEP = 24;                   // twice as many of a segment's codes stay in registers
constexpr int SPLIT_AHEAD = 4;                   // plane chunks of a row asked for before its streams are decoded
// words of a unit's streams at most: twelve bits a pair code, the last word of each lane begun
__host__ __device__ constexpr uint32_t split_words(int pairs) { return (uint32_t) (HP_LP * pairs + 32); }
constexpr size_t split_shm(int pairs, int threads) {
    return ((size_t) LUT_PAIRS + split_words(pairs) + 2 * SPLIT_PAD + 16 * (size_t) pairs + 2 * (size_t) threads + 32 + (size_t) threads / 32 + 1) * 4;
}

// A position in the words at st.  n: minus the bit position; its low five bits are what the funnel shift takes (the next 32
// bits are in w0:w1, w0 used up where they are zero), and a word boundary is passed where bit 5 changes (24 bits at a time
// at most).  nw: the word after w1.  Words past the staged ones are read and not used: the padding, then what follows in LDS.
struct seg_bits {
    const uint32_t * st;
    uint32_t w0, w1, nw, n;
    __device__ __forceinline__ uint32_t ahead() const { // the word after w1
        return *(const uint32_t *) ((const char *) st + 4 - (((int32_t) n >> 3) & ~3));
    }
    __device__ __forceinline__ seg_bits(const uint32_t * st_, uint32_t pos) : st(st_), n(0u - pos) {
        const uint32_t j = (pos + 31) >> 5;
        w0 = st[(int) j - 1]; // (in front of the first word: unused)
        w1 = st[j];
        nw = ahead();
    }
    // the next pair code, and the one after it if it begins before bit `nstop` (as n); returns how many.  e: the entries' sum has the
    // length of both in its low five bits; an entry of unused codes, met out of step only, was given a length when staged
    __device__ __forceinline__ bool two(const uint32_t * lut, uint32_t nstop, uint32_t & e0, uint32_t & e1) {
        const uint32_t W = __builtin_amdgcn_alignbit(w0, w1, n);
        e0 = lut[W >> (32 - HP_LP)];
        e1 = lut[(W << (e0 & 31u)) >> (32 - HP_LP)];
        const bool both = (int32_t) (n - (e0 & 31u)) > (int32_t) nstop;
        const uint32_t to = n - ((e0 + (both ? e1 : 0u)) & 31u);
        const bool m = ((to ^ n) & 32u) != 0;
        n = to;
        w0 = m ? w1 : w0;
        w1 = m ? nw : w1;
        nw = ahead();
        return both;
    }
};

// Whether a decoder that begins anywhere falls into step with this table's codes soon enough.  Its phase modulo g moves only at
// codes whose length is no multiple of g: with a share s of multiples one of 2 (1 - s) codes moves one of the two, and one in
// g - 1 moves ends in step, after (g - 1) / (2 (1 - s)) codes on average.  The share is that of 64 samples of the table, which
// stands in the order of its codes: as many of a length as its codes are met.  Codes all of one length are told by the first
// and the last: segments begin at multiples of it, all in step, and only the LDS bank at which every lane's stream then begins costs.
__device__ __forceinline__ bool falls_into_step(uint32_t entry, uint32_t inv_codes, bool equal) { // lane i: entry 64 i + 32, lanes 0 and 63: the first, the last
    const uint32_t len = entry & 31u;
    bool does = true;
#pragma unroll
    for (int g : {2, 3, 4, 5, 6, 7, 11}) { // (8 to 10 and 12 are multiples of these)
        does &= (uint32_t) __builtin_popcountll(__ballot(len != 0 && len % (uint32_t) g == 0)) <= 64 - (((uint32_t) (g - 1) * inv_codes + 255) >> 8);
    }
    const uint32_t first = __builtin_amdgcn_readlane(len, 0), last = __builtin_amdgcn_readlane(len, 63);
    return first == last ? equal : does;
}

// units: the launch's first, all of the matrix, the launch's; the device's CUs; 8192 over the codes that a wrong phase may last
struct split_units { int64_t first, all; int count, cus; uint32_t inv_codes; };

// The units of a launch by one half-wave each, two units of a column to a wavefront, in `words` words of LDS at lds: the
// activations of the block's column and a ring per wavefront (5120 words at K = 4096 with one, of 7700 at least).
template <typename TX, bool DEQ>
__device__ __forceinline__ void split_whole(const bf16n_weight & w, const cols & p, int ncols, uint16_t * __restrict__ out, const split_units & su,
                                            const uint32_t * lut, uint32_t * lds, int words) {
    const int K = (int) w.K, lane = threadIdx.x & 63, l32 = lane & 31, wave = threadIdx.x >> 6, all = blockDim.x >> 6;
    const int n = DEQ ? 1 : ncols, per_col = (su.count + 1) / 2; // wavefronts a column
    // one block of a CU while its wavefronts have a SIMD each (512 units, four columns: 41.1 us, on two blocks 46.7)
    const int blocks = per_col * n <= 4 * su.cus && (int) gridDim.x > su.cus ? su.cus : (int) gridDim.x;
    int mine = (per_col * n + blocks - 1) / blocks; // wavefronts of a block, all of one column
    while ((per_col + mine - 1) / mine * n > blocks && mine < per_col) {
        mine++;
    }
    const int col_blocks = (per_col + mine - 1) / mine, fit = (words - (DEQ ? 0 : K)) / (LR_BYTES / 4), waves = fit < all ? fit : all;
    for (int b = (int) blockIdx.x; b < col_blocks * n; b += (int) gridDim.x) { // (once but for more columns than blocks)
        const int col = b / col_blocks, j0 = b % col_blocks * mine, j1 = j0 + mine < per_col ? j0 + mine : per_col;
        float * xs = (float *) lds;
        __syncthreads();
        if constexpr (!DEQ) {
            for (int i = threadIdx.x; i < K / 4; i += (int) blockDim.x) {
                ((float4 *) xs)[i] = x_four<TX>(p.x + col * p.x_tok, i);
            }
            __syncthreads();
        }
        uint32_t * ring = lds + (DEQ ? 0 : K) + wave * (LR_BYTES / 4) + lane;
        for (int j = wave < waves ? j0 + wave : j1; j < j1; j += waves) {
            const int u = 2 * j + (lane >> 5) < su.count ? 2 * j + (lane >> 5) : 2 * j;
            if constexpr (DEQ) {
                unit_rows<FMT_HUFPAIR>(w, lut, ring, su.first + u, u, l32, out);
            } else {
                float v[1];
                unit_dot<FMT_HUFPAIR, true, 1, x_lds<float>>(w.plane, lut, lane_stream<FMT_HUFPAIR>(w, su.first + u, l32), ring, su.first + u, w.R, K / CHUNK,
                                                             (w.flags & FLAG_CHUNK_MAJOR) != 0, xs, l32, v);
                if (l32 < w.R && u == 2 * j + (lane >> 5)) { // (a missing second unit is the first again, which is stored once)
                    store_y(p.y + col * p.y_tok, p.y_bf16, (int64_t) u * w.R + l32, v[0]);
                }
            }
        }
    }
}

// DEQ: the exact BF16 bits of the rows to out, no products
template <typename TX, bool DEQ>
__global__ void __launch_bounds__(1024) k_hp_split(const bf16n_weight w, const cols p, int ncols, uint16_t * __restrict__ out, const split_units su) {
    extern __shared__ __align__(16) unsigned char shm_raw[];
    const int K = (int) w.K, C = K / CHUNK, R = w.R, pairs = R * C * 8, S = (int) blockDim.x >> 5;
    const uint32_t cap = split_words(pairs);
    uint32_t * lut = (uint32_t *) shm_raw;
    uint32_t * st = lut + LUT_PAIRS + SPLIT_PAD;
    uint16_t * ex = (uint16_t *) (st + cap + SPLIT_PAD); // [chunk][lane][8 pairs], an exponent per byte
    uint32_t * ends = (uint32_t *) (ex + 32 * pairs), * counts = ends + blockDim.x;
    uint32_t * front = counts + blockDim.x, * again = front + 32, * in_step = lut + LUT_PAIRS; // [lane], [round], in front of the streams
    const hp_ptrs q = hpp(w);
    const int tid = threadIdx.x, l32 = tid & 31, seg = tid >> 5;
    const bool cm = (w.flags & FLAG_CHUNK_MAJOR) != 0;
    // what the first unit's loads and the branch wait for is asked for ahead of the table
    const uint32_t sample = q.lut[tid % 64 == 0 ? 0 : tid % 64 == 63 ? LUT_PAIRS - 1 : tid % 64 * (LUT_PAIRS / 64) + LUT_PAIRS / 128];
    uint32_t base, end, from, to;
    auto head = [&](int u) {
        const int64_t gu = su.first + u;
        base = q.ubase[gu];
        end = gu + 1 < su.all ? q.ubase[gu + 1] : (uint32_t) ((const aux_header *) w.aux)->n_b;
        from = q.lrel[gu * 32 + l32];
        to = q.lrel[gu * 32 + (l32 < 31 ? l32 + 1 : l32)];
    };
    head((int) blockIdx.x < su.count ? (int) blockIdx.x : 0);
    for (int i = tid; i < LUT_PAIRS / 4; i += (int) blockDim.x) {
        uint4 v = ((const uint4 *) q.lut)[i];
        v.x += (v.x & 31u) == 0; v.y += (v.y & 31u) == 0; v.z += (v.z & 31u) == 0; v.w += (v.w & 31u) == 0;
        ((uint4 *) lut)[i] = v;
    }
    if (tid < 64) {
        const bool does = falls_into_step(sample, su.inv_codes, su.count <= (int) gridDim.x);
        if (tid == 0) {
            *in_step = does;
        }
    }
    for (int u = (int) blockIdx.x; u == (int) blockIdx.x || u < su.count; u += (int) gridDim.x) { // (split_whole has work for a block without a unit)
        if (u != (int) blockIdx.x) {
            head(u);
        }
        const int64_t gu = su.first + (u < su.count ? u : 0);
        const uint4 * plane = (const uint4 *) (w.plane + gu * R * (int64_t) K) + l32;
        auto chunk_at = [&](int rr, int c) { return cm ? c * R + rr : rr * C + c; }; // in stream order
        const uint32_t words = end <= base ? 0 : end - base < cap ? end - base : cap; // (none for a base past the stream's end)
        to = l32 < 31 ? to : words;
        from = from < words ? from : words;
        to = to < from ? from : to < words ? to : words;
        uint4 ahead[SPLIT_AHEAD];
#pragma unroll
        for (int i = 0; i < SPLIT_AHEAD; i++) {
            ahead[i] = plane[chunk_at(seg < R ? seg : R - 1, i < C ? i : C - 1) * 32];
        }
        for (uint32_t i0 = tid; i0 < words; i0 += 8 * blockDim.x) {
            uint32_t v[8];
#pragma unroll
            for (uint32_t k = 0; k < 8; k++) { // (asked for together; past the end the last one again, unused)
                const uint32_t i = i0 + k * blockDim.x;
                v[k] = q.stream[base + (i < words ? i : words - 1)];
            }
#pragma unroll
            for (uint32_t k = 0; k < 8; k++) {
                const uint32_t i = i0 + k * blockDim.x;
                if (i < words) {
                    st[i] = v[k];
                }
            }
        }
        if (tid <= S) {
            again[tid] = 0;
        }
        __syncthreads();
        if (__builtin_amdgcn_readfirstlane(*in_step) == 0) {
            split_whole<TX, DEQ>(w, p, ncols, out, su, lut, lut + LUT_PAIRS, (int) (again - lut) - LUT_PAIRS);
            return;
        }
        if (u >= su.count) {
            return;
        }
        const uint32_t first = 32 * from, bits = 32 * (to - from); // (12 a pair code and the last word's rest: 12.3 K at most)
        const uint32_t nstop = 0u - (first + bits * (uint32_t) (seg + 1) / (uint32_t) S);
        uint32_t start = first + bits * (uint32_t) seg / (uint32_t) S - (seg ? bits / (uint32_t) (2 * S) : 0), n = 0;
        auto pair = [](uint32_t e) { return (e >> 7 & 0xFFu) | (e >> 15 & 0xFF00u); };
        uint32_t kept[SPLIT_KEEP] = {}; // the segment's codes, two exponents of a pair each, as far as they fit
        { // round 0: only where the next segment's first code begins
            uint32_t e0, e1;
            seg_bits b(st, start);
            while ((int32_t) b.n > (int32_t) nstop) {
                b.two(lut, nstop, e0, e1);
            }
            ends[tid] = 0u - b.n;
        }
        __syncthreads();
        for (int round = 0; round <= S; round++) {
            const uint32_t exact = seg ? ends[tid - 32] : first;
            bool moved = exact != start || round == 0;
            start = exact;
            if (moved) {
                again[round] = 1;
                if (round % 2 == 0) {
                    atomicMin(&front[l32], (uint32_t) seg);
                }
            }
            if (round % 2 != 0 && seg == 0) {
                front[l32] = (uint32_t) S;
            }
            __syncthreads();
            if (again[round] == 0) {
                break;
            }
            if (round != 0 && round % 2 == 0 && front[l32] < (uint32_t) seg) {
                const uint32_t begins = ends[32 * front[l32] - 32 + l32], mine = first + bits * (uint32_t) seg / (uint32_t) S;
                uint32_t e0, e1, e2, e3;
                seg_bits b(st, begins);
                b.two(lut, 0x80000000u, e0, e1);
                b.two(lut, 0x80000000u, e2, e3);
                if (e0 == e1 && e1 == e2 && e2 == e3) { // a run
                    const uint32_t run = e0, len = run & 31u, at = mine > begins ? begins + (mine - begins + len - 1) / len * len : begins;
                    seg_bits here(st, at);
                    here.two(lut, 0x80000000u, e0, e1);
                    here.two(lut, 0x80000000u, e2, e3);
                    if (at != start && e0 == run && e1 == run && e2 == run && e3 == run) { // (it may have ended)
                        start = at;
                        moved = true;
                    }
                }
            }
            if (moved) {
                seg_bits b(st, start);
                n = 0;
#pragma unroll
                for (int k = 0; k < SPLIT_KEEP; k++) {
                    if ((int32_t) b.n > (int32_t) nstop) {
                        uint32_t e0, e1;
                        n += b.two(lut, nstop, e0, e1) ? 2 : 1;
                        kept[k] = pair(e0) | pair(e1) << 16;
                    }
                }
                while ((int32_t) b.n > (int32_t) nstop) {
                    uint32_t e0, e1;
                    n += b.two(lut, nstop, e0, e1) ? 2 : 1;
                }
                ends[tid] = 0u - b.n;
                counts[tid] = n;
            }
            __syncthreads();
        }
        uint32_t at = 0;
        for (int i = 0; i < seg; i++) {
            at += counts[32 * i + l32];
        }
        auto put = [&](uint32_t i, uint32_t e) { ex[((i >> 3) * 32 + (uint32_t) l32) * 8 + (i & 7)] = (uint16_t) e; };
        n = at + n < (uint32_t) pairs ? n : at < (uint32_t) pairs ? (uint32_t) pairs - at : 0; // (the last word's unused bits)
#pragma unroll
        for (int k = 0; k < SPLIT_KEEP; k++) {
            if (2 * k < (int) n) {
                put(at + 2 * k, kept[k]);
                if (2 * k + 1 < (int) n) {
                    put(at + 2 * k + 1, kept[k] >> 16);
                }
            }
        }
        if (n > 2 * SPLIT_KEEP || (seg == S - 1 && at + n < (uint32_t) pairs)) { // many short codes: once more, code by code
            seg_bits b(st, start);
            const uint32_t to = seg == S - 1 ? (uint32_t) pairs : at + n;
            while (at < to) {
                uint32_t e0, e1;
                const bool both = b.two(lut, 0x80000000u, e0, e1);
                put(at, pair(e0));
                if (both && at + 1 < to) {
                    put(at + 1, pair(e1));
                }
                at += 2;
            }
        }
        __syncthreads();
        for (int rr = seg; rr < R; rr += S) {
            auto weights = [&](int c, const uint4 sm, uint32_t (&wp)[8]) {
                const uint4 e = ((const uint4 *) ex)[chunk_at(rr, c) * 32 + l32];
                const uint32_t ew[4] = {e.x, e.y, e.z, e.w}, smw[4] = {sm.x, sm.y, sm.z, sm.w};
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    wp[2 * j] = merge(spread_lo(smw[j]), (ew[j] & 0xFFu) << 7 | (ew[j] & 0xFF00u) << 15);
                    wp[2 * j + 1] = merge(spread_hi(smw[j]), (ew[j] >> 9 & 0x7F80u) | (ew[j] >> 1 & 0x7F800000u));
                }
            };
            for (int col = 0; col < (DEQ ? 1 : ncols); col++) {
                float acc = 0.f;
                for (int c0 = 0; c0 < C; c0 += SPLIT_AHEAD) {
                    if (c0 != 0 || rr != seg || (col != 0 && C > SPLIT_AHEAD)) {
#pragma unroll
                        for (int i = 0; i < SPLIT_AHEAD; i++) {
                            ahead[i] = plane[chunk_at(rr, c0 + i < C ? c0 + i : C - 1) * 32];
                        }
                    }
#pragma unroll
                    for (int i = 0; i < SPLIT_AHEAD; i++) {
                        const int c = c0 + i;
                        if (c < C) {
                            uint32_t wp[8];
                            weights(c, ahead[i], wp);
                            if constexpr (DEQ) {
                                uint16_t * dst = out + ((int64_t) u * R + rr) * K + c * CHUNK;
#pragma unroll
                                for (int j = 0; j < 4; j++) {
                                    *(uint2 *) (dst + 128 * j + 4 * l32) = make_uint2(wp[2 * j], wp[2 * j + 1]);
                                }
                            } else {
                                float xv[16];
                                x_chunk16<TX>(p.x + col * p.x_tok, c * CHUNK + 4 * l32, xv);
                                float4 x[4];
#pragma unroll
                                for (int j = 0; j < 4; j++) {
                                    x[j] = make_float4(xv[4 * j], xv[4 * j + 1], xv[4 * j + 2], xv[4 * j + 3]);
                                }
                                const float d = dot_chunk(wp, x);
                                acc += cm ? half_wave_sum_dpp(d) : d; // (lane 31 has the sum)
                            }
                        }
                    }
                }
                if (!DEQ) {
                    const float v = cm ? acc : half_wave_sum_dpp(acc);
                    if (l32 == 31) {
                        store_y(p.y + col * p.y_tok, p.y_bf16, (int64_t) u * R + rr, v);
                    }
                }
            }
        }
        __syncthreads();
    }
}

// partial dot of a decoded chunk with x.  The four per-position sums are combined as in the reference
// (kernels.cuh:130-187), then over the 32 lanes on the VALU (DPP, no LDS traffic); result in lane 31 of the half-wave.
__device__ __forceinline__ float nib_dot(const uint32_t (&wp)[8], const float (&xv)[16]) {
    float a0 = 0.f, a1 = 0.f, a2 = 0.f, a3 = 0.f;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        a0 = fmaf(bf16_bits_to_f32(wp[2 * j] & 0xFFFFu), xv[4 * j], a0);
        a1 = fmaf(__uint_as_float(wp[2 * j] & 0xFFFF0000u), xv[4 * j + 1], a1);
        a2 = fmaf(bf16_bits_to_f32(wp[2 * j + 1] & 0xFFFFu), xv[4 * j + 2], a2);
        a3 = fmaf(__uint_as_float(wp[2 * j + 1] & 0xFFFF0000u), xv[4 * j + 3], a3);
    }
    return half_wave_sum_dpp((a0 + a1) + (a2 + a3));
}

// the same with BF16 activations left as the 8 pairs they arrive in: a pair of weights meets a pair of activations in
// one dot2 instruction (8 instructions where conversions and FMAs took 48)
__device__ __forceinline__ void x_pairs16(const char * x, int col0, uint32_t (&xp)[8]) {
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const uint2 t = *(const uint2 *) (x + 2 * (col0 + 128 * j));
        xp[2 * j] = t.x;
        xp[2 * j + 1] = t.y;
    }
}
__device__ __forceinline__ float nib_dot_pairs(const uint32_t (&wp)[8], const uint32_t (&xp)[8]) {
    float a01 = 0.f, a23 = 0.f;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        a01 = dot2_bf16(wp[2 * j], xp[2 * j], a01);
        a23 = dot2_bf16(wp[2 * j + 1], xp[2 * j + 1], a23);
    }
    return half_wave_sum_dpp(a01 + a23);
}

// the exact products of a row's escaped weights, summed over the half-wave (result in lane 31)
// (e0, e1: the row's range of escape records, esc_off[gr] and esc_off[gr + 1], which the caller requests together with
// the row's other loads: 3 to 8 % off the four-column launches)
template <typename TX>
__device__ __forceinline__ float nib_escapes(const nib_ptrs & w, uint32_t e0, uint32_t e1, const char * x, int l32) {
    float acc = 0.f;
    for (uint32_t i = e0 + l32; i < e1; i += 32) {
        const uint32_t rec = w.esc[i];
        acc = fmaf(bf16_bits_to_f32(esc_bits(rec)), x_at<TX>(x, (int) (rec & 0xFFFu)), acc);
    }
    return e1 > e0 ? half_wave_sum_dpp(acc) : 0.f;
}

// NIBBLE GEMV; GLU 1: rows_per_matrix = [gate (nrows); up (nrows)] of one matrix; GLU 2: separate gate / up matrices.
// These matrices are small (a few MB at most), so the launch is laid out for latency: one half-wave per (row, chunk)
// pair, every load of a pair issued at once, the C chunk sums of a row combined through LDS in chunk order.
// NC: columns per decode (dense batches: a (row, chunk) is decoded once for NC token columns, each of which gets the
// bits of its single-column launch); columns past the last repeat it and are not stored.
// RW: (row, chunk) pairs per half-wave and turn.  A launch is a few latencies of memory, so the more of its bytes are asked
// for before the first wait the better, until a block's decode is longer than what it waits for.  The barrier keeps the
// loads of all pairs ahead of the first decode: left alone the compiler waits for one pair before it asks for the next
// (a gate / up pair of 512 x 2048 for two slots: 6.8 us, 5.3 with it, 5.2 with RW = 1).  us with RW = 1 / 2 (4 is behind 2 nearly everywhere):
//   dense, one BF16 column: 2048 x 2048 3.55 / 3.35, 5120 x 2048 6.0 / 5.5, 2048 x 4096 5.3 / 5.1, 16384 x 512 5.0 / 4.7
//   FP32, three / eight columns: 5120 x 2048 10.2 / 16.8 -> 8.2 / 12.9, 2048 x 4096 9.3 / 15.8 -> 8.0 / 12.7
//   257 experts' down (2048 x 512), 1 / 4 / 12 tokens of nine slots: 6.8 / 18.1 / 47 -> 5.7 / 14.5 / 35.3; gate / up 8.8 / 24.8 / 65 -> 9.2 / 23.6 / 59
// One column and one pair: eight wavefronts to a SIMD, 64 registers; with the 65 that gate and up of FP32 take if left alone eight
// blocks do not fit a CU (512 x 2048, eight slots 8.3 us for 7.7).
template <typename TX, int GLU, int NC, int RW>
__global__ void __launch_bounds__(NT, NC == 1 && RW == 1 ? 8 : 0) k_nib_mmv(const bf16n_weight w, const bf16n_weight w_up, const cols p, const int ncols) {
    constexpr int M = GLU ? 2 : 1;
    __shared__ float part[RW][M][NC][HALVES];
    const int K = (int) w.K, C = K / CHUNK; // 1 .. 8
    col_view cv[NC];
#pragma unroll
    for (int j = 0; j < NC; j++) {
        const int col = (int) blockIdx.y * NC + j;
        cv[j] = col_setup(p, col < ncols ? col : ncols - 1);
    }
    const nib_ptrs q[2] = {nibp(w, 0), GLU == 1 ? nibp(w, p.nrows) : nibp(w_up, 0)};
    const int l32 = threadIdx.x & 31, half = threadIdx.x >> 5;
    const int rpb = HALVES / C; // rows per block and turn: C half-waves per row (C = 3, 5, 6, 7 leave some half-waves idle)
    const int lr = half / C, c = half % C;
    for (int64_t base = (int64_t) blockIdx.x * (rpb * RW); base < p.nrows; base += (int64_t) gridDim.x * (rpb * RW)) {
        uint4 sm[RW][M], T[RW][M];
        uint2 cd[RW][M], esc[RW][M];
#pragma unroll
        for (int t = 0; t < RW; t++) {
            const int64_t r = base + t * rpb + lr, gr = cv[0].rbase + (lr < rpb && r < p.nrows ? r : 0); // dense batches share the rows; with expert ids NC is 1
#pragma unroll
            for (int m = 0; m < M; m++) {
                sm[t][m] = *((const uint4 *) (q[m].plane + gr * K + c * CHUNK) + l32);
                cd[t][m] = *((const uint2 *) (q[m].codes + gr * (K / 2) + c * (CHUNK / 2)) + l32);
                T[t][m] = *(const uint4 *) (q[m].table + gr * 16);
                esc[t][m] = make_uint2(q[m].esc_off[gr], q[m].esc_off[gr + 1]);
            }
        }
        uint32_t xp[8];
        float xv[16];
        auto load_x = [&](int j) {
            if constexpr (sizeof(TX) == 2) {
                x_pairs16(cv[j].x, c * CHUNK + 4 * l32, xp);
            } else {
                x_chunk16<TX>(cv[j].x, c * CHUNK + 4 * l32, xv);
            }
        };
        if constexpr (NC == 1) {
            load_x(0);
        }
        if constexpr (RW > 1) {
            __builtin_amdgcn_sched_barrier(0);
        }
        uint32_t wp[RW][M][8];
#pragma unroll
        for (int t = 0; t < RW; t++) {
#pragma unroll
            for (int m = 0; m < M; m++) {
                nib_chunk(sm[t][m], cd[t][m], T[t][m], wp[t][m]);
            }
        }
#pragma unroll
        for (int j = 0; j < NC; j++) {
            float v[RW][M];
            if constexpr (NC > 1) {
                load_x(j);
            }
#pragma unroll
            for (int t = 0; t < RW; t++) {
#pragma unroll
                for (int m = 0; m < M; m++) {
                    if constexpr (sizeof(TX) == 2) {
                        v[t][m] = nib_dot_pairs(wp[t][m], xp);
                    } else {
                        v[t][m] = nib_dot(wp[t][m], xv);
                    }
                }
            }
            if (c == 0) {
#pragma unroll
                for (int t = 0; t < RW; t++) {
#pragma unroll
                    for (int m = 0; m < M; m++) {
                        v[t][m] += nib_escapes<TX>(q[m], esc[t][m].x, esc[t][m].y, cv[j].x, l32);
                    }
                }
            }
            if (l32 == 31) {
#pragma unroll
                for (int t = 0; t < RW; t++) {
#pragma unroll
                    for (int m = 0; m < M; m++) {
                        part[t][m][j][half] = v[t][m];
                    }
                }
            }
        }
        __syncthreads();
        const int t = l32 / NC, j = l32 % NC; // one lane per (turn, column) of the row's first half-wave
        const int64_t r = base + t * rpb + lr;
        if (c == 0 && lr < rpb && t < RW && r < p.nrows && (int) blockIdx.y * NC + j < ncols) {
            float s = part[t][0][j][half], su = part[t][M - 1][j][half];
            for (int i = 1; i < C; i++) {
                s += part[t][0][j][half + i];
                su += part[t][M - 1][j][half + i];
            }
            store_y(cv[0].y + j * p.y_tok, p.y_bf16, r, GLU ? su * silu(s) : s); // j > 0 only in dense batches
        }
        __syncthreads();
    }
}

// The router of a decode step with the glue before it: y = W bf16(norm(a + b + c)) in FP32 for a 4-bit-code matrix of
// K = 2048, one token per blockIdx.y.  Both are a few kilobytes whose time is a launch's latency; here every block forms
// the token's row itself (12 KB at most, while its weights are on their way) and takes its two rows of the matrix from
// there, and the first block stores the row.  The bits are those of k_add_rmsnorm8 and k_nib_mmv<bf16_t, 0, 1>.  256 rows,
// one token: 3.9 us against 3.7 + 3.0 and the gap between two launches (three layers of the decode step 158 -> 150 us,
// half a microsecond a layer of it by the faster selection); 16 tokens, two layers: 330 and 325, which is what runs differ by.
// More than 4096 results (rows x tokens) form the rows again in a second round of blocks: the two launches then (the
// operator layer's NORM_MMV_RESULTS has the figures).
__global__ void __launch_bounds__(NT) k_norm_nib_mmv(const bf16n_weight w, const add_norm_args p, float * __restrict__ y, int64_t y_tok) {
    constexpr int C = NORM8_N / CHUNK, RPB = HALVES / C;
    static_assert(NT == NORM8_THREADS, "a thread per eight elements of the row");
    __shared__ __align__(16) uint16_t xs[NORM8_N];
    __shared__ float wave_sq[NT / 64], part[HALVES];
    const nib_ptrs q = nibp(w, 0);
    const int tid = threadIdx.x, l32 = tid & 31, half = tid >> 5, lr = half / C, c = half % C;
    const int64_t tok = blockIdx.y, at = tok * NORM8_N + 8 * tid;
    const int64_t base = (int64_t) blockIdx.x * RPB, row = base + lr < w.rows ? base + lr : w.rows - 1;
    const uint4 va = *(const uint4 *) (p.a + at);
    const uint4 vb = p.b ? *(const uint4 *) (p.b + at) : make_uint4(0, 0, 0, 0);
    const uint4 vc = p.c ? *(const uint4 *) (p.c + at) : make_uint4(0, 0, 0, 0);
    const uint4 sm = *((const uint4 *) (q.plane + row * NORM8_N + c * CHUNK) + l32);
    const uint2 cd = *((const uint2 *) (q.codes + row * (NORM8_N / 2) + c * (CHUNK / 2)) + l32);
    const uint4 T = *(const uint4 *) (q.table + row * 16);
    const uint32_t e0 = q.esc_off[row], e1 = q.esc_off[row + 1];
    float v[8], fb[8], fc[8];
    unpack8(va, v);
    unpack8(vb, fb);
    unpack8(vc, fc);
#pragma unroll
    for (int i = 0; i < 8; i++) {
        if (p.b) {
            v[i] += fb[i];
        }
        if (p.c) {
            v[i] += fc[i];
        }
    }
    const uint4 o = norm8_row(v, p.gamma, p.eps, wave_sq);
    *(uint4 *) (xs + 8 * tid) = o;
    if (blockIdx.x == 0) {
        if (p.y_sum) {
            *(uint4 *) (p.y_sum + at) = pack8(v);
        }
        *(uint4 *) (p.y_norm + at) = o;
    }
    uint32_t wp[8], xp[8];
    nib_chunk(sm, cd, T, wp);
    __syncthreads();
    x_pairs16((const char *) xs, c * CHUNK + 4 * l32, xp);
    float s = nib_dot_pairs(wp, xp);
    if (c == 0) {
        s += nib_escapes<bf16_t>(q, e0, e1, (const char *) xs, l32);
    }
    if (l32 == 31) {
        part[half] = s;
    }
    __syncthreads();
    if (c == 0 && l32 == 0 && base + lr < w.rows) {
        float sum = part[half];
#pragma unroll
        for (int i = 1; i < C; i++) {
            sum += part[half + i];
        }
        y[tok * y_tok + base + lr] = sum;
    }
}

// Dense NIBBLE products through the matrix cores: y[t] = W x[t] for BF16 token columns, 32 per block (gridDim.y blocks
// of tokens; columns past the last repeat it and are not stored).  The 4-bit code has no decode chain, so one decode of
// the matrix serves 32 tokens at the cost of one.  A block is one group of 32 rows with K / 256 wavefronts; wavefront v
// takes half a chunk: the slots [16 (v & 1), +16) of chunk v / 2.  Lane (row r, half h) decodes two adjacent slots of
// its row per step, 16 (v & 1) + 4n + 2h and the next (n = 0..3): 32 weights, which are eight adjacent columns
// 128 j + 64 (v & 1) + 16 n + 8 h + [0, 8) in each of the chunk's four column blocks j — the A operands of four matrix
// instructions (k positions 8h + [0, 8) of instruction j) — and lane (token t, half h) supplies the same columns of its
// token's activations as B operands, one 16-byte load each: which columns an instruction's k positions stand for is
// free as long as both operands agree.  (The activations staged through LDS by loads that take a token's 128 bytes
// with eight adjacent lanes measured the same for K = 2048 and, in two turns of eight wavefronts, slower for K = 4096:
// a launch is a few serial latencies, not the rate of its loads.)  BF16 products are exact in FP32; the partial sums of
// the wavefronts are added in K order through LDS, the products of escaped weights (decoded as +0) last, and the sum
// is rounded once.
typedef __bf16 nm_bf16x8_t __attribute__((ext_vector_type(8)));
typedef float nm_f32x16_t __attribute__((ext_vector_type(16)));
typedef uint32_t nm_u32x4_t __attribute__((ext_vector_type(4)));
constexpr int NM_WAVES = 8; // per block: K / 256 half chunks in one turn each, K > 2048 in two
// Words per (wavefront, accumulator register) row of the partial sums in LDS: lane l at l + l / 32.  The threads that add
// the partial sums of one token's 32 rows read 16 registers x 2 half-waves of one lane position: 64 words apart they
// all met one bank (32-way conflicts: 7,900 conflict cycles per block, 3 of a launch's 14 us), 66 apart with the
// upper half-wave shifted by one they spread over all banks, two to a bank.
constexpr int NM_PSTRIDE = 66;
__device__ __forceinline__ int nm_part_at(int wave, int i, int lane) { return (wave * 16 + i) * NM_PSTRIDE + lane + (lane >> 5); }

// TURNS: half chunks per wavefront (wavefront v takes v TURNS + [0, TURNS)).  The loads of a wavefront are written
// ahead of their uses; with one turn the compiler issues them in batches of about nine (68 registers, three blocks per
// CU).  All 28 pinned ahead of the first use (a scheduling barrier; 148 registers) measured 2 to 6 % faster for
// 5120 x 2048 up to 32 columns, 30 % slower at 64 (one block per CU), and with two turns 5 to 7 % slower (256
// registers and spills): left to the compiler.
template <int TURNS>
__global__ void __launch_bounds__(NM_WAVES * 64) k_nib_mm(const bf16n_weight w, const cols p, const int ncols) {
    extern __shared__ __align__(16) float nm_part[]; // [wavefront][accumulator register][lane]
    const nib_ptrs q = nibp(w, 0);
    const int K = (int) w.K;
    const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5, wave = (int) (threadIdx.x >> 6), n_waves = (int) (blockDim.x >> 6);
    const int64_t g0 = (int64_t) blockIdx.x * 32;
    const int64_t row = p.row0 + (g0 + r < p.nrows ? g0 + r : p.nrows - 1);
    const int t0 = (int) blockIdx.y * 32;
    const char * x = p.x + (int64_t) (t0 + r < ncols ? t0 + r : ncols - 1) * p.x_tok;
    const uint4 T = nib_rotated(*(const uint4 *) (q.table + row * 16));
    // the sums this thread finishes at the end are (token, row) = (e / 32, e % 32) for e = thread, thread + block size:
    // one row (the block size is a multiple of 32), whose escape range is requested now
    const int64_t my_row = g0 + (threadIdx.x & 31);
    const int64_t my_gr = p.row0 + (my_row < p.nrows ? my_row : p.nrows - 1);
    const uint32_t esc0 = q.esc_off[my_gr], esc1 = q.esc_off[my_gr + 1];
    uint4 sm0[TURNS][4], sm1[TURNS][4], cdv[TURNS][4], b[TURNS][4][4];
#pragma unroll
    for (int turn = 0; turn < TURNS; turn++) {
        // a last wavefront with a half chunk too few (K / 256 odd) repeats its first
        const int hc = (wave * TURNS + turn) * 256 < K ? wave * TURNS + turn : wave * TURNS;
        const int c = hc >> 1, s0 = 16 * (hc & 1) + 2 * h; // this lane's first slot
        const uint8_t * pl = q.plane + row * K + c * CHUNK + 16 * s0;
        const uint8_t * cd = q.codes + row * (K / 2) + c * (CHUNK / 2) + 8 * s0;
        const char * xb = x + 2 * (c * CHUNK + 4 * s0);
#pragma unroll
        for (int n = 0; n < 4; n++) {
            sm0[turn][n] = *(const uint4 *) (pl + 64 * n);
            sm1[turn][n] = *(const uint4 *) (pl + 64 * n + 16);
            cdv[turn][n] = *(const uint4 *) (cd + 32 * n);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                b[turn][n][j] = *(const uint4 *) (xb + 32 * n + 256 * j);
            }
        }
    }
    nm_f32x16_t acc;
#pragma unroll
    for (int i = 0; i < 16; i++) {
        acc[i] = 0.f;
    }
#pragma unroll
    for (int turn = 0; turn < TURNS; turn++) {
        if ((wave * TURNS + turn) * 256 < K) {
#pragma unroll
            for (int n = 0; n < 4; n++) {
                uint32_t w0[8], w1[8];
                nib_chunk<true>(sm0[turn][n], make_uint2(cdv[turn][n].x, cdv[turn][n].y), T, w0);
                nib_chunk<true>(sm1[turn][n], make_uint2(cdv[turn][n].z, cdv[turn][n].w), T, w1);
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const nm_u32x4_t a = {w0[2 * j], w0[2 * j + 1], w1[2 * j], w1[2 * j + 1]};
                    const nm_u32x4_t bv = {b[turn][n][j].x, b[turn][n][j].y, b[turn][n][j].z, b[turn][n][j].w};
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(nm_bf16x8_t, a), __builtin_bit_cast(nm_bf16x8_t, bv), acc, 0, 0, 0);
                }
            }
        }
    }
#pragma unroll
    for (int i = 0; i < 16; i++) {
        nm_part[nm_part_at(wave, i, lane)] = acc[i];
    }
    __syncthreads();
    // accumulator register i of lane l: row 8 (i / 4) + 4 (l / 32) + i % 4 of the group, token l % 32.  A thread per
    // (token, row), rows adjacent in a wavefront: a token's 32 outputs are stored side by side.
    for (int e = (int) threadIdx.x; e < 1024; e += (int) blockDim.x) {
        const int tok = e >> 5, rr = e & 31;
        const int i = 4 * (rr >> 3) + (rr & 3), l = tok + 32 * ((rr >> 2) & 1);
        if (g0 + rr < p.nrows && t0 + tok < ncols) {
            float v = 0.f;
            for (int k = 0; k < n_waves; k++) {
                v += nm_part[nm_part_at(k, i, l)];
            }
            const char * xt = p.x + (int64_t) (t0 + tok) * p.x_tok;
            for (uint32_t k = esc0; k < esc1; k++) {
                const uint32_t rec = q.esc[k];
                v = fmaf(bf16_bits_to_f32(esc_bits(rec)), x_at<bf16_t>(xt, (int) (rec & 0xFFFu)), v);
            }
            store_y(p.y + (int64_t) (t0 + tok) * p.y_tok, p.y_bf16, g0 + rr, v);
        }
    }
}

// The same product for at most 16 token columns per block on 16-row groups (v_mfma_f32_16x16x32_bf16): twice the blocks
// of k_nib_mm, which matters while its groups of 32 rows leave CUs idle (2048 rows: 64 blocks on 256 CUs).  Lane
// (row r of 16, k part q of 4) decodes two adjacent slots of its row per step, 8 n + 2 q and the next: eight adjacent
// columns 128 j + 32 n + 8 q + [0, 8) in each of the chunk's four column blocks j, the A operands of four matrix
// instructions (k positions 8 q + [0, 8) of instruction j); lane (token t of 16, q) supplies the same columns of its
// token as B operands.  A wavefront takes STEPS consecutive steps of a row (a chunk is four steps); the partial sums of
// the wavefronts are added in K order through LDS (rows of 68 words: the 64 threads that add for four tokens meet every
// bank twice), the products of escaped weights last.
typedef float nm_f32x4_t __attribute__((ext_vector_type(4)));
constexpr int NM16_PSTRIDE = 68;
template <int STEPS>
__global__ void __launch_bounds__(NM_WAVES * 64) k_nib_mm16(const bf16n_weight w, const cols p, const int ncols) {
    extern __shared__ __align__(16) float nm_part[]; // [wavefront][accumulator register][lane]
    const nib_ptrs q = nibp(w, 0);
    const int K = (int) w.K;
    const int lane = threadIdx.x & 63, r = lane & 15, kq = lane >> 4, wave = (int) (threadIdx.x >> 6), n_waves = (int) (blockDim.x >> 6);
    const int64_t g0 = (int64_t) blockIdx.x * 16;
    const int64_t row = p.row0 + (g0 + r < p.nrows ? g0 + r : p.nrows - 1);
    const int t0 = (int) blockIdx.y * 16;
    const char * x = p.x + (int64_t) (t0 + r < ncols ? t0 + r : ncols - 1) * p.x_tok;
    const uint4 T = nib_rotated(*(const uint4 *) (q.table + row * 16));
    // the sums this thread finishes at the end are (token, row) = (e / 16, e % 16) for e = thread, thread + block size
    const int64_t my_row = g0 + (threadIdx.x & 15);
    const int64_t my_gr = p.row0 + (my_row < p.nrows ? my_row : p.nrows - 1);
    const uint32_t esc0 = q.esc_off[my_gr], esc1 = q.esc_off[my_gr + 1];
    const int first = wave * STEPS, c = first >> 2, s0 = 8 * (first & 3) + 2 * kq; // this lane's first slot
    const uint8_t * pl = q.plane + row * K + c * CHUNK + 16 * s0;
    const uint8_t * cd = q.codes + row * (K / 2) + c * (CHUNK / 2) + 8 * s0;
    const char * xb = x + 2 * (c * CHUNK + 4 * s0);
    uint4 sm0[STEPS], sm1[STEPS], cdv[STEPS], b[STEPS][4];
#pragma unroll
    for (int n = 0; n < STEPS; n++) {
        sm0[n] = *(const uint4 *) (pl + 128 * n);
        sm1[n] = *(const uint4 *) (pl + 128 * n + 16);
        cdv[n] = *(const uint4 *) (cd + 64 * n);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            b[n][j] = *(const uint4 *) (xb + 64 * n + 256 * j);
        }
    }
    nm_f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int n = 0; n < STEPS; n++) {
        uint32_t w0[8], w1[8];
        nib_chunk<true>(sm0[n], make_uint2(cdv[n].x, cdv[n].y), T, w0);
        nib_chunk<true>(sm1[n], make_uint2(cdv[n].z, cdv[n].w), T, w1);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const nm_u32x4_t a = {w0[2 * j], w0[2 * j + 1], w1[2 * j], w1[2 * j + 1]};
            const nm_u32x4_t bv = {b[n][j].x, b[n][j].y, b[n][j].z, b[n][j].w};
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(nm_bf16x8_t, a), __builtin_bit_cast(nm_bf16x8_t, bv), acc, 0, 0, 0);
        }
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        nm_part[(wave * 4 + i) * NM16_PSTRIDE + lane] = acc[i];
    }
    __syncthreads();
    // accumulator register i of lane l: row 4 (l / 16) + i of the group, token l % 16
    for (int e = (int) threadIdx.x; e < 256; e += (int) blockDim.x) {
        const int tok = e >> 4, rr = e & 15;
        const int i = rr & 3, l = tok + 16 * (rr >> 2);
        if (g0 + rr < p.nrows && t0 + tok < ncols) {
            float v = 0.f;
            for (int k = 0; k < n_waves; k++) {
                v += nm_part[(k * 4 + i) * NM16_PSTRIDE + l];
            }
            const char * xt = p.x + (int64_t) (t0 + tok) * p.x_tok;
            for (uint32_t k = esc0; k < esc1; k++) {
                const uint32_t rec = q.esc[k];
                v = fmaf(bf16_bits_to_f32(esc_bits(rec)), x_at<bf16_t>(xt, (int) (rec & 0xFFFu)), v);
            }
            store_y(p.y + (int64_t) (t0 + tok) * p.y_tok, p.y_bf16, g0 + rr, v);
        }
    }
}

// exact rows of a NIBBLE matrix: FP32 or BF16, to out + i * stride (bytes); row index from ids (gather) or row0 + i.
// AHEAD: chunks whose bytes are asked for together, the row's first four at most: a half-wave's row is otherwise one latency
// of memory per chunk.  The barrier keeps them so.  us, one chunk at a time / this: dequant of 2048 x 2048 6.0 / 5.2, 2048 x 4096
// 11.3 / 9.7, 3000 x 1536 5.6 / 5.3, 5120 x 2048 8.7 / 8.6 (37 MB read and written); 513 rows of 5120 x 2048 4.0 / 3.6, of 2048 x 4096 7.9 / 6.9
template <bool BF, int AHEAD>
__global__ void __launch_bounds__(NT) k_nib_rows(const bf16n_weight w, const char * __restrict__ ids, int64_t ids_s0, int64_t n,
                                                 int64_t row0, char * __restrict__ dst, int64_t dst_s1) {
    const nib_ptrs q = nibp(w, 0);
    const int K = (int) w.K, C = K / CHUNK;
    const int l32 = threadIdx.x & 31, half = threadIdx.x >> 5;
    for (int64_t i = (int64_t) blockIdx.x * HALVES + half; i < n; i += (int64_t) gridDim.x * HALVES) {
        const int64_t gr = row0 + (ids ? (int64_t) * (const int32_t *) (ids + i * ids_s0) : i);
        char * o = dst + i * dst_s1;
        const uint4 T = nib_rotated(*(const uint4 *) (q.table + gr * 16));
        const uint32_t e0 = q.esc_off[gr], e1 = q.esc_off[gr + 1];
        auto store = [&](int c, const uint4 sm, const uint2 cd) {
            uint32_t wp[8];
            nib_chunk<true>(sm, cd, T, wp);
            // the row's escapes go into the registers of the lane that holds their column: every element is stored once
            for (uint32_t e = e0; e < e1; e++) {
                const uint32_t rec = q.esc[e];
                const int rel = (int) (rec & 0xFFFu) - c * CHUNK;
                if (rel >= 0 && rel < CHUNK && ((rel & 127) >> 2) == l32) {
                    const int at = (rel >> 7) * 2 + ((rel & 3) >> 1);
                    const uint32_t b = esc_bits(rec);
#pragma unroll
                    for (int i2 = 0; i2 < 8; i2++) {
                        if (i2 == at) {
                            wp[i2] = (rel & 1) ? (wp[i2] & 0xFFFFu) | (b << 16) : (wp[i2] & 0xFFFF0000u) | b;
                        }
                    }
                }
            }
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int col = c * CHUNK + 128 * j + 4 * l32;
                if (BF) {
                    *(uint2 *) (o + 2 * col) = make_uint2(wp[2 * j], wp[2 * j + 1]);
                } else {
                    *(float4 *) (o + 4 * col) = make_float4(bf16_bits_to_f32(wp[2 * j] & 0xFFFFu), __uint_as_float(wp[2 * j] & 0xFFFF0000u),
                                                            bf16_bits_to_f32(wp[2 * j + 1] & 0xFFFFu), __uint_as_float(wp[2 * j + 1] & 0xFFFF0000u));
                }
            }
        };
        for (int c0 = 0; c0 < C; c0 += AHEAD) {
            uint4 sm[AHEAD];
            uint2 cd[AHEAD];
#pragma unroll
            for (int i = 0; i < AHEAD; i++) { // (past the end the last chunk again, unused)
                const int c = c0 + i < C ? c0 + i : C - 1;
                sm[i] = *((const uint4 *) (q.plane + gr * K + c * CHUNK) + l32);
                cd[i] = *((const uint2 *) (q.codes + gr * (K / 2) + c * 256) + l32);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < AHEAD; i++) {
                if (c0 + i < C) {
                    store(c0 + i, sm[i], cd[i]);
                }
            }
        }
    }
}

// blocks of HALVES units (rows) each, capped so that a launch of several columns stays within a few blocks per CU
int grid_for(int64_t work, int ncols, int cus, int per_block = HALVES) {
    const int64_t blocks = (work + per_block - 1) / per_block;
    const int64_t cap = (int64_t) cus * 8 / (ncols < 1 ? 1 : ncols > 4 ? 4 : ncols);
    return (int) (blocks < 1 ? 1 : blocks > cap ? cap : blocks);
}

// Wavefronts per block of the HUFPAIR / HUFFMAN kernels, two units each: four, fewer where that leaves CUs without a
// block (the units' chains set the time: alone on a CU they share its LDS with nobody).  Units of a chunk or two are done
// sooner than a smaller block stages its table: 1024 rows of 512, R = 1, one column 8.4 us with two wavefronts, 7.2 with four.
int huf_waves(int64_t units, int ncols, int cus, int chunks) {
    int waves = NT / 64;
    while (waves > 1 && chunks > 2 && (units + 2 * waves - 1) / (2 * waves) * ncols < cus) {
        waves /= 2;
    }
    return waves;
}

// LDS of a block of k_huf_mmv with several columns
size_t huf_shared(const bf16n_weight & w, int nc, bool x_bf16) {
    return (size_t) nc * w.K * (x_bf16 ? 2 : 4) + (w.format == FMT_HUFPAIR ? 4u << HP_LP : 4u << HUF_LMAX) + (size_t) (NT / 64) * LR_BYTES;
}

// What a chunk of a unit costs with nc columns to a decode, in 10 ns, by the blocks that a CU has at once (fitted to 8000 launches of
// 64 to 9000 units of one to 128 chunks, two to sixteen columns; 6 to 8 % rms): mostly the chain of lookups, a column and the second
// block beside the first a sixth to a quarter of it each.  Three and four FP32 columns have registers for three blocks.
constexpr uint16_t HUF_CHUNK[2][2][3][4] = { // [HUFFMAN, HUFPAIR][FP32, BF16][nc - 2][blocks - 1]
    {{{101, 123, 172, 199}, {111, 136, 180, 0}, {121, 149, 200, 0}}, {{104, 130, 181, 234}, {118, 146, 200, 258}, {130, 163, 225, 288}}},
    {{{64, 80, 105, 125}, {73, 90, 120, 0}, {84, 103, 131, 0}}, {{69, 88, 119, 144}, {82, 102, 142, 166}, {94, 121, 159, 197}}}};
int64_t huf_time(const bf16n_weight & w, int64_t units, int ncols, int nc, bool x_bf16, int cus) {
    const uint16_t (&t)[4] = HUF_CHUNK[w.format == FMT_HUFPAIR][x_bf16][nc - 2];
    const int64_t fit = std::min<int64_t>((int64_t) (LDS_BYTES / huf_shared(w, nc, x_bf16)), x_bf16 || nc == 2 ? 4 : 3); // blocks of a CU at once
    const int64_t blocks = (units + HALVES - 1) / HALVES * ((ncols + nc - 1) / nc), rounds = blocks / (fit * cus), last = (blocks % (fit * cus) + cus - 1) / cus;
    return rounds * t[fit - 1] + (last ? t[last - 1] : 0);
}

// Columns that share one decode in dense products.  Each column in a launch of its own units decodes the matrix again, which
// costs nothing while the device has half-waves to spare (a unit's chain is longer than what they do beside it), and everything
// beyond: from fifteen half-waves per CU on two or three columns share one (from sixteen in units of at most 32 chunks, 24 of at
// most four), from eight groups of four per CU on four.  us, each column by itself / two / three / four, BF16 and HUFPAIR but where named:
//   two columns: 16384 x 2048, R = 16 (1024 units) 41 / 49, 32768 x 2048 49 / 49, 16656 x 3584, R = 8 (2082) 70 / 53, 42264 x 3072,
//     R = 8 127 / 82, 59473 x 2560, R = 1 108 / 68
//   three: 10920 x 3072, R = 8 (1365 units, 16 half-waves per CU) 53.3 / 48.2 / 46.0, FP32 54.2 / 44.2 / 41.6
//   four: 24608 x 1024, R = 16 (1538) 58 / 35 / - / 38, 32768 x 2048 96 / 60 / - / 61, 42264 x 3072 235 / 139 / - / 98, 218800 x 512, R = 1
//     216 / 123 / - / 84
//   eight: 10336 x 3584, R = 16 (646) 137 / 99 / - / 106, 24608 x 1024 98 / 66 / - / 47, 42264 x 3072 441 / 238 / - / 173, 16384 x 3072, R = 8,
//     HUFFMAN 209 / 111 / - / 84
// Another count than these lines give where huf_time has it 6 % ahead: three, where a group of four would lack a column or more or leave a
// CU one block of FP32, and pairs where their blocks fit the CUs at once: FP32, six columns, 1365 units of 8 x 3072 97 / 74 / 48 / 53; nine,
// 848 of 1 x 3584 16.2 / 17.9 / 12.6 / 22.6, 1368 of 1 x 1536 12.4 / 12.2 / 9.4 / 15.0; BF16, nine, 5057 of 1 x 1536 31.7 / 31.2 / 27.1 / 31.2;
// HUFFMAN, four FP32, 2152 of 1 x 4096 26 / 17.6 / 26 / 24.
// Blocks of eight wavefronts instead of four: 5 to 25 % behind but for long rows of short units.
int huf_columns(const bf16n_weight & w, int64_t units, int ncols, bool x_bf16, int cus) {
    const int chunks = w.R * (int) (w.K / CHUNK);
    if (ncols == 1 || units * ncols <= (chunks <= 4 ? 24 : chunks <= 32 ? 16 : 15) * (int64_t) cus) {
        return 1;
    }
    const int line = ncols > 2 && units * ((ncols + 3) / 4) > HALVES * (int64_t) cus ? 4 : ncols == 3 ? 3 : 2;
    int best = line;
    int64_t time = huf_time(w, units, ncols, line, x_bf16, cus) * 94;
    for (int nc = 2; nc <= std::min(4, ncols); nc++) {
        const int64_t t = huf_time(w, units, ncols, nc, x_bf16, cus) * 100;
        if (nc != line && t < time) {
            best = nc;
            time = t;
        }
    }
    return best;
}

// Dense products of one column whose lanes read their streams without the rings.  A ring costs 4 KiB of LDS and thirty registers
// per wavefront, so that 16 of them (12 at K = 4096) fit a CU instead of 20 (16), and a lane that has not moved on loads its
// block again; with many wavefronts the misses of one are covered by the others.  us without against with rings:
//  * HUFPAIR in short units that the caches hold, from 64 wavefronts per CU on: 32768 x 512 11.7 against 14.2 (from memory, 32768 x 2048,
//    R = 1, 30.6 and 28.2).  The line is on the careful side: 16384 x 512 has 7.9 and 9.7.
//  * HUFFMAN, which loads a block per eight codes where HUFPAIR has one per sixteen, from 16 wavefronts per CU on unless
//    the matrix comes from memory in short units: 8192 x 512 5.6 against 6.1, 32768 x 4096, R = 4 139 and 199 (16384 x 2048, R = 4 32.3 and 24.7).
bool huf_direct(const bf16n_weight & w, int64_t units, int cus) {
    const int64_t per_cu = units / (2 * cus), weights = units * w.R * w.K; // wavefronts of the launch per CU
    const int chunks = w.R * (int) (w.K / CHUNK);
    return w.format == FMT_HUFPAIR ? chunks <= 8 && per_cu >= 64 && weights <= (16 << 20) : per_cu >= 16 && (weights <= (16 << 20) || chunks >= 32);
}

// Columns up to which a launch over `units` units takes k_hp_split (0: none): while the chain of a unit is longer than what its
// blocks take on the CUs they get.  A CU holds two blocks up to 512 pair codes a lane, one beyond.  Every column adds its products
// to a block, and where a row has more chunks than its first wavefront keeps it reads the plane again (`rows`: exact rows, which
// read it once).  Times as multiples of k_huf_mmv's, BF16 columns:
//   up to two units per CU, one / 2 / 4 / 6 / 8 columns: 8192 x 2048, R = 16 0.64 / 0.64 / 0.78 / 0.78 / 0.87, 4096 x 2048 0.46 / 0.50 /
//     0.55 / 0.58 / 0.73; 4096 x 4096, R = 8 0.58 / 0.64 / 0.86 / 0.89 / 1.02; 4096 x 3584, R = 8 0.69 / 0.72 / 0.93 / 0.95 / 1.09; 4096 x 3072,
//     R = 8 0.71 / 0.76 / 0.96 / 0.98 / 1.12; 8192 x 1024 0.84 / 0.87 / 1.07 / 1.09 / 1.22; 8192 x 4096 0.68 / 0.72 / 0.96 / 1.05 / 1.28
//   up to one, where the plane read again finds the CU idle: 1912 x 4096, R = 8, 7 / 8 FP32 columns 0.65 / 0.69, BF16 0.79 / 0.86
//   three, in two passes of two blocks: 12288 x 2048 0.82 / 0.84 / 0.95 / 0.77 / 0.82 (640 units, six: 1.05); 6144 x 4096, R = 8 0.83 / 0.94 /
//     1.14 / 1.00 / 1.09; 6144 x 3584 0.92 / 0.99; 6144 x 3072 1.00 / 1.07; or in three passes of one, a column: 12288 x 2560 1.06,
//     12288 x 3072 0.96, 12288 x 3584 0.96, 12288 x 4096 0.94
//   dequant at two units per CU 0.78 / 0.70 / 0.80 / 0.82 / 0.93 / 0.79 in the first line's order, at three 0.93, 0.93, 1.02, 1.11
int hp_split_cols(const bf16n_weight & w, int64_t units, int cus, bool rows = false) {
    const int C = (int) (w.K / CHUNK), pairs = w.R * C * 8;
    const bool kept = rows || C <= SPLIT_AHEAD;
    if (w.format != FMT_HUFPAIR || pairs < 256 || pairs > 1024 || units > 3 * (int64_t) cus) {
        return 0;
    }
    if (units > 2 * (int64_t) cus) {
        return pairs == 512 ? kept ? 8 : 2 : pairs == 448 || pairs >= 768 ? 1 : 0;
    }
    return pairs <= 512 ? std::min((pairs - 128) / 48, kept || units <= cus ? 8 : 6) : units > cus ? 4 : 8;
}
constexpr int SPLIT_DEQUANT_COLS = 3; // what the exact rows cost in its place, in columns
int split_threads(const bf16n_weight & w) {
    const int pairs = w.R * (int) (w.K / CHUNK) * 8, segs = (pairs + SPLIT_PAIRS - 1) / SPLIT_PAIRS;
    return 64 * ((segs + 1) / 2);
}
// Codes that a wrong phase may last on average before the units go to a half-wave each (falls_into_step): a round more costs
// a sixteenth of the chain on a CU that has one unit, more beside others, and beyond two the gain is small.  One column, in
// segments / by half-waves against a chain each (k_huf_mmv), at 1 / 2 / 3 units of 16 x 2048 per CU: codes of three bits
// with one in eight of four (8) 0.57 / 0.76 / 0.93, of five bits with one in eight of four and six (16) 0.72 / 0.80 / 1.17, of seven
// so (24) 0.92 / 1.27 / 1.55, 94 % of four bits (24) 0.65 to 1.10 / 0.84 to 1.13 / 1.04 to 1.87, 95 % and all but a few of six
// (50 and more) 1.21 and 1.34 / 1.33 and 1.52 / 1.96 and 2.11; by half-waves in here 0.98 to 1.07 throughout
uint32_t split_codes(int64_t units, int cus) { return units <= cus ? 30 : units <= 2 * (int64_t) cus ? 20 : 7; }
template <typename TX, bool DEQ>
void launch_hp_split(const bf16n_weight & w, const cols & p, int ncols, uint16_t * out, int cus, hipStream_t stream) {
    const int threads = split_threads(w);
    const size_t shm = split_shm(w.R * (int) (w.K / CHUNK) * 8, threads);
    const int64_t units = p.nrows / w.R, fit = (int64_t) cus * std::max<int64_t>(1, std::min<int64_t>(2048 / threads, (int64_t) (LDS_BYTES / shm)));
    const int64_t blocks = std::max(units, (units + 1) / 2 * ncols); // (split_whole: a block per two units of a column)
    if (!DEQ) { // (the note is of products)
        note_kernel("k_hp_split", tx_name<TX>(), 1, 0);
    }
    hipLaunchKernelGGL((k_hp_split<TX, DEQ>), dim3((unsigned) std::min(blocks, fit)), dim3(threads), shm, stream, w, p, ncols, out,
                       split_units{p.row0 / w.R, w.rows / w.R, (int) units, cus, 8192u / split_codes(units, cus)});
}

} // namespace

void compat_init() {
#define HUFA(F, TX, N) (void) hipFuncSetAttribute((const void *) k_huf_mmv<F, TX, false, true, N>, hipFuncAttributeMaxDynamicSharedMemorySize, (int) LDS_BYTES)
#define HUFAN(F, TX) HUFA(F, TX, 2); HUFA(F, TX, 3); HUFA(F, TX, 4)
    HUFAN(FMT_HUFPAIR, bf16_t); HUFAN(FMT_HUFPAIR, float); HUFAN(FMT_HUFFMAN, bf16_t); HUFAN(FMT_HUFFMAN, float);
#undef HUFAN
#undef HUFA
    const int shm = (int) split_shm(1024, 1024);
    (void) hipFuncSetAttribute((const void *) k_hp_split<bf16_t, false>, hipFuncAttributeMaxDynamicSharedMemorySize, shm);
    (void) hipFuncSetAttribute((const void *) k_hp_split<float, false>, hipFuncAttributeMaxDynamicSharedMemorySize, shm);
    (void) hipFuncSetAttribute((const void *) k_hp_split<bf16_t, true>, hipFuncAttributeMaxDynamicSharedMemorySize, shm);
}

// Steps per wavefront of k_nib_mm16 (a row has K / 128): the fewest for which a block has at most eight wavefronts, or
// four (fewer, longer wavefronts) when the row groups outnumber the CUs anyway; 0: K does not fit the kernel.
int nib_mm16_steps(const bf16n_weight & w, int64_t nrows, int cus) {
    if (w.format != FMT_NIBBLE || w.K % CHUNK != 0 || w.K / 128 > 4 * NM_WAVES) {
        return 0;
    }
    const int steps_all = (int) (w.K / 128);
    const int fewest = steps_all <= NM_WAVES ? 1 : steps_all <= 2 * NM_WAVES ? 2 : 4;
    return fewest == 2 && (nrows + 15) / 16 > cus ? 4 : fewest;
}
// Whether a dense batch of BF16 columns takes the 16-row matrix-core kernel (k_nib_mm16): by the CUs its row groups
// fill, from two columns (a group per CU), three (half of them) or five (a quarter) on; smaller matrices stay with the
// GEMV columns, which run side by side on idle CUs (256 x 2048: 3.2-4.6 us at 2-16 columns against 4.7-5.9; 512 x 4096:
// 4.6-9.3 against 7.4-10.0).  Beyond 16 columns every block of 16 tokens decodes the matrix again, which still wins
// while the launch is at most two blocks per CU (2048 x 4096: 10.5-10.7 us at 17-32 columns and 15.7-17.3 at 40-64
// against 16.5-19.9 in 32-row groups; 1024 x 2048: 6.5-6.8 us up to 64 against 10.7-12.8; 5120 x 2048, 640 blocks at
// 17 columns: 12.4 against 11.2, left to the 32-row groups).  The dispatch below and bf16n_gemv_max_tokens share this
// rule.
bool nib_mm16_pays(const bf16n_weight & w, int64_t nrows, int ncols, int cus) {
    const int64_t groups = (nrows + 15) / 16, token_blocks = (ncols + 15) / 16;
    const bool enough = (ncols >= 2 && groups >= cus) || (ncols >= 3 && groups * 2 >= cus) || (ncols >= 5 && groups * 4 >= cus);
    return enough && (token_blocks == 1 || groups * token_blocks <= 2 * (int64_t) cus) && nib_mm16_steps(w, nrows, cus) != 0;
}

// Whether a dense batch of `ncols` BF16 columns over `nrows` rows of a 4-bit-code matrix goes through the matrix cores
// (k_nib_mm): the row groups of 32 must give enough CUs a block, by column count.  The dispatch below and
// bf16n_gemv_max_tokens share this rule.
bool nib_mm_pays(const bf16n_weight & w, int64_t nrows, int ncols, int cus) {
    const int64_t nm_blocks = (nrows + 31) / 32;
    const bool enough = (ncols >= NIB_MM_MIN_COLS && nm_blocks * 2 >= cus) || (ncols > 8 && nm_blocks * 4 >= cus) ||
                        (ncols > 24 && nm_blocks * 8 >= cus);
    return w.format == FMT_NIBBLE && w.K % CHUNK == 0 && w.K / 256 <= 2 * NM_WAVES && enough;
}

void launch_compat_mmv(const bf16n_weight & w, const bf16n_weight * up, int glu, const cols & p, int ncols, bool x_bf16,
                       int cus, hipStream_t stream, bool matrix_cores) {
    const bf16n_weight & wu = up ? *up : w;
    // the matrix cores where the row groups of 32 give enough CUs a block: from five BF16 columns on with blocks for half
    // of the CUs, from nine with a quarter, from 25 with an eighth (5120 x 2048, 160 blocks: 11.0-13.0 us for 5-32
    // columns against 9.6 / 17.9 us for 4 / 8 GEMV columns and 20 us for dequant + GEMM; 2048 x 4096, 64 blocks: 16.7-20.7
    // us against 8.6 / 15.4 us and 24-28 us; 1024 x 2048, 32 blocks: 10.6-12.8 us against 7.8 / 9.5 / 14.9 / 25.5 us in
    // GEMV columns at 9 / 16 / 32 / 64).  Smaller matrices stay with the GEMV columns, which run side by side on idle CUs
    // (256 x 2048: 4.9-9.5 us for 9-64 columns against 10.5-12.6 us here).
    const int64_t nm_blocks = (p.nrows + 31) / 32;
    if (matrix_cores && !p.ids && glu == 0 && x_bf16 && nib_mm16_pays(w, p.nrows, ncols, cus) && ((uintptr_t) p.x & 15) == 0 &&
        p.x_tok % 16 == 0) {
        // 16-row groups (5120 x 2048: 7.7 / 8.2 / 8.8 / 10.5 us at 2 / 4 / 8 / 16 columns against 8.3 / 11.4
        // in GEMV columns and 9.7 / 10.8 in 32-row groups; 2048 x 4096: 8.0 / 8.2 / 9.0 / 10.3 us at 3 / 4 / 8 / 16
        // against 9.4 / 9.3 / 15.3 / 15.5; 1024 x 2048: 5.6 / 6.5 us at 5 / 16 against 6.8 / 9.1; 2048 x 512: 3.3 / 3.6
        // us at 2 / 16 against 3.5 / 5.5)
        const int steps = nib_mm16_steps(w, p.nrows, cus), waves = (int) (w.K / 128) / steps;
        note_kernel("k_nib_mm16", nullptr, 1, steps);
        const dim3 grid((unsigned) ((p.nrows + 15) / 16), (unsigned) ((ncols + 15) / 16));
        const size_t shm = (size_t) waves * 4 * NM16_PSTRIDE * sizeof(float);
        if (steps == 1)      hipLaunchKernelGGL(k_nib_mm16<1>, grid, dim3(waves * 64), shm, stream, w, p, ncols);
        else if (steps == 2) hipLaunchKernelGGL(k_nib_mm16<2>, grid, dim3(waves * 64), shm, stream, w, p, ncols);
        else                 hipLaunchKernelGGL(k_nib_mm16<4>, grid, dim3(waves * 64), shm, stream, w, p, ncols);
        return;
    }
    if (matrix_cores && !p.ids && glu == 0 && x_bf16 && nib_mm_pays(w, p.nrows, ncols, cus) && ((uintptr_t) p.x & 15) == 0 &&
        p.x_tok % 16 == 0) {
        const int halves = (int) (w.K / 256), turns = halves > NM_WAVES ? 2 : 1, waves = (halves + turns - 1) / turns;
        note_kernel("k_nib_mm", nullptr, 1, turns);
        const dim3 grid((unsigned) nm_blocks, (unsigned) ((ncols + 31) / 32));
        const size_t shm = (size_t) waves * 16 * NM_PSTRIDE * sizeof(float);
        if (turns == 2) {
            hipLaunchKernelGGL(k_nib_mm<2>, grid, dim3(waves * 64), shm, stream, w, p, ncols);
        } else {
            hipLaunchKernelGGL(k_nib_mm<1>, grid, dim3(waves * 64), shm, stream, w, p, ncols);
        }
        return;
    }
    if (w.format == FMT_NIBBLE) {
        const int rpb = HALVES / (int) (w.K / CHUNK);
        // dense batches: four (two) columns share one decode of the matrix once there are columns enough to keep at
        // least four groups of blocks (below that the columns run side by side on the idle CUs, which is faster)
        const int64_t blocks1 = (p.nrows + rpb - 1) / rpb;
        const bool fills = blocks1 >= 4 * (int64_t) cus; // one column's blocks keep every CU busy by themselves
        const int nc = p.ids ? 1 : fills ? (ncols >= 3 ? 4 : ncols == 2 ? 2 : 1) : ncols >= 16 ? 4 : ncols >= 8 ? 2 : 1;
        const int ngroups = (ncols + nc - 1) / nc;
        // two (row, chunk) pairs per half-wave from three blocks per CU on, gate and up (twice the loads to a pair) from
        // sixteen: 256 x 2048, eight FP32 columns (two per CU) 3.3 us with one pair, 3.6 with two, 512 x 2048, three columns 3.4 and 3.3;
        // gate / up of 512 x 2048, nine slots (nine per CU) 8.8 and 9.2, of 1024 x 1536 (eighteen) 13.0 and 11.7
        const int rw = blocks1 * ngroups >= (glu ? 16 : 3) * (int64_t) cus ? 2 : 1;
        const int64_t per = (int64_t) rpb * rw;
        const dim3 grid(grid_for((p.nrows + per - 1) / per * HALVES, ngroups, cus), ngroups);
        note_kernel("k_nib_mmv", x_bf16 ? "bf16_t" : "float", 3, glu, nc, rw);
#define NIBC(TX, G, N, R) hipLaunchKernelGGL((k_nib_mmv<TX, G, N, R>), grid, dim3(NT), 0, stream, w, wu, p, ncols)
#define NIBR(TX, G, N) do { if (rw == 2) NIBC(TX, G, N, 2); else NIBC(TX, G, N, 1); } while (0)
#define NIB(TX, G) do { if (nc == 4) NIBR(TX, G, 4); else if (nc == 2) NIBR(TX, G, 2); else NIBR(TX, G, 1); } while (0)
        if (x_bf16) { if (glu == 0) NIB(bf16_t, 0); else if (glu == 1) NIB(bf16_t, 1); else NIB(bf16_t, 2); }
        else        { if (glu == 0) NIB(float, 0);  else if (glu == 1) NIB(float, 1);  else NIB(float, 2); }
#undef NIB
#undef NIBR
#undef NIBC
        return;
    }
    const bool hp = w.format == FMT_HUFPAIR;
    const int64_t work = p.nrows / w.R;
    if (glu == 0 && !p.ids && ncols <= hp_split_cols(w, work, cus) && ((uintptr_t) p.x & 15) == 0 && (ncols == 1 || p.x_tok % 16 == 0)) {
        if (x_bf16) launch_hp_split<bf16_t, false>(w, p, ncols, nullptr, cus, stream);
        else        launch_hp_split<float, false>(w, p, ncols, nullptr, cus, stream);
        return;
    }
    const size_t shared = (size_t) w.K * 4 + (size_t) (glu ? 2 : 1) * (hp ? (4u << HP_LP) : (4u << HUF_LMAX));
    const char * instance = hp ? x_bf16 ? "3, bf16_t" : "3, float" : x_bf16 ? "2, bf16_t" : "2, float";
    const int nc = glu || p.ids ? 1 : huf_columns(w, work, ncols, x_bf16, cus);
    if (nc > 1) {
        const int waves = NT / 64, groups = (ncols + nc - 1) / nc;
        const size_t shm = huf_shared(w, nc, x_bf16);
        const int64_t blocks = std::min<int64_t>((work + 2 * waves - 1) / (2 * waves), (int64_t) cus * (int64_t) (LDS_BYTES / shm));
        const dim3 grid((unsigned) blocks, (unsigned) groups); // (a block stages its table and columns once)
        note_kernel("k_huf_mmv", instance, 3, 0, 1, nc);
#define HUFN(F, TX, N) hipLaunchKernelGGL((k_huf_mmv<F, TX, false, true, N>), grid, dim3(waves * 64), shm, stream, w, wu, p, ncols)
#define HUFNX(F, TX) do { if (nc == 4) HUFN(F, TX, 4); else if (nc == 3) HUFN(F, TX, 3); else HUFN(F, TX, 2); } while (0)
        if (hp) {
            if (x_bf16) HUFNX(FMT_HUFPAIR, bf16_t); else HUFNX(FMT_HUFPAIR, float);
        } else {
            if (x_bf16) HUFNX(FMT_HUFFMAN, bf16_t); else HUFNX(FMT_HUFFMAN, float);
        }
#undef HUFNX
#undef HUFN
        return;
    }
    const bool direct = !glu && !p.ids && ncols == 1 && huf_direct(w, work, cus);
    note_kernel("k_huf_mmv", instance, 3, glu != 0, !direct, 1);
    const int waves = direct ? NT / 64 : huf_waves(work, ncols, cus, w.R * (int) (w.K / CHUNK));
    const size_t shm = shared + (direct ? 0 : (size_t) waves * LR_BYTES);
    const dim3 grid(grid_for(work, ncols, cus, 2 * waves), ncols);
#define HUF(F, TX, G, RING) hipLaunchKernelGGL((k_huf_mmv<F, TX, G, RING>), grid, dim3(waves * 64), shm, stream, w, wu, p, ncols)
#define HUFX(F, TX) do { if (glu) HUF(F, TX, true, true); else if (direct) HUF(F, TX, false, false); else HUF(F, TX, false, true); } while (0)
    if (hp) {
        if (x_bf16) HUFX(FMT_HUFPAIR, bf16_t); else HUFX(FMT_HUFPAIR, float);
    } else {
        if (x_bf16) HUFX(FMT_HUFFMAN, bf16_t); else HUFX(FMT_HUFFMAN, float);
    }
#undef HUFX
#undef HUF
}

bool norm_nib_mmv_ok(const bf16n_weight & w, const add_norm_args & a) {
    const auto al = [](const void * q) { return ((uintptr_t) q & 15) == 0; };
    return w.format == FMT_NIBBLE && w.K == NORM8_N && a.n == NORM8_N && w.rows <= 65536 && !a.ys && al(a.a) && al(a.b) && al(a.c) && al(a.gamma) &&
           al(a.y_sum) && al(a.y_norm);
}

void launch_norm_nib_mmv(const bf16n_weight & w, const add_norm_args & a, float * y, int64_t y_tok, int n_tok, hipStream_t stream) {
    constexpr int RPB = HALVES * CHUNK / NORM8_N;
    note_kernel("k_norm_nib_mmv", nullptr, 0);
    hipLaunchKernelGGL(k_norm_nib_mmv, dim3((unsigned) ((w.rows + RPB - 1) / RPB), n_tok), dim3(NT), 0, stream, w, a, y, y_tok);
}

// (rows of one or two chunks: one at a time; 16384 x 512 measured 7.1 us so and 7.3 with four ahead, 8192 x 1024 6.6, with two 7.3, with four 6.9)
static void launch_nib_rows(const bf16n_weight & w, const char * ids, int64_t ids_s0, int64_t n, int64_t row0, char * dst, bool dst_bf16,
                            int64_t dst_s1, dim3 grid, hipStream_t stream) {
#define ROWS(BF, A) hipLaunchKernelGGL((k_nib_rows<BF, A>), grid, dim3(NT), 0, stream, w, ids, ids_s0, n, row0, dst, dst_s1)
#define ROWSA(BF) do { if (w.K <= 2 * CHUNK) ROWS(BF, 1); else ROWS(BF, 4); } while (0)
    if (dst_bf16) ROWSA(true); else ROWSA(false);
#undef ROWSA
#undef ROWS
}

void launch_compat_dequant(const bf16n_weight & w, int64_t row0, int64_t nrows, uint16_t * out, int cus, hipStream_t stream) {
    const int64_t work = w.format == FMT_NIBBLE ? nrows : nrows / w.R;
    const int waves = w.format == FMT_NIBBLE ? NT / 64 : huf_waves(work, 1, cus, w.R * (int) (w.K / CHUNK));
    const int64_t blocks = (work + 2 * waves - 1) / (2 * waves);
    const dim3 grid((unsigned) (blocks < (int64_t) cus * 16 ? blocks : (int64_t) cus * 16));
    if (w.format == FMT_NIBBLE) {
        launch_nib_rows(w, nullptr, 0, nrows, row0, (char *) out, true, (int64_t) w.K * 2, grid, stream);
    } else if (hp_split_cols(w, work, cus, true) >= SPLIT_DEQUANT_COLS) {
        cols p = {};
        p.row0 = row0;
        p.nrows = nrows;
        launch_hp_split<bf16_t, true>(w, p, 0, out, cus, stream);
    } else if (w.format == FMT_HUFPAIR) {
        hipLaunchKernelGGL((k_huf_dequant<FMT_HUFPAIR>), grid, dim3(waves * 64), 0, stream, w, row0, nrows, out);
    } else {
        hipLaunchKernelGGL((k_huf_dequant<FMT_HUFFMAN>), grid, dim3(waves * 64), 0, stream, w, row0, nrows, out);
    }
}

void launch_compat_get_rows(const bf16n_weight & w, const void * ids, int64_t ids_s0, int64_t n, void * dst, bool dst_bf16,
                            int64_t dst_s1, int64_t row0, hipStream_t stream) {
    const dim3 grid((unsigned) ((n + HALVES - 1) / HALVES));
    if (w.format == FMT_NIBBLE) {
        launch_nib_rows(w, (const char *) ids, ids_s0, n, row0, (char *) dst, dst_bf16, dst_s1, grid, stream);
    } else {
        if (dst_bf16) hipLaunchKernelGGL((k_hp_get_rows<true>), grid, dim3(NT), 0, stream, w, (const char *) ids, ids_s0, n, row0, (char *) dst, dst_s1);
        else          hipLaunchKernelGGL((k_hp_get_rows<false>), grid, dim3(NT), 0, stream, w, (const char *) ids, ids_s0, n, row0, (char *) dst, dst_s1);
    }
}

} // namespace dev
} // namespace bf16n
