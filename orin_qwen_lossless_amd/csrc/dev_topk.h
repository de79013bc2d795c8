// The router's selection for one token by one wavefront, shared by the stand-alone top-k kernels (kernels_moe.hip) and
// the routed GEMV that selects in its prologue (kernels_tile.hip).
#pragma once

#include "dev_common.h"

namespace bf16n {
namespace dev {

// softmax over the experts, k largest (ties: lower index), weights renormalised to sum 1 if asked; one wave per token.
// The logits of a token sit in registers (NQ per lane, expert = lane + 64 q).  NaN logits count as -inf, and a selection only
// ever returns an index below n_experts that was not taken before, whatever the values are: the ids feed address
// arithmetic in the kernels that follow.
// the logits of a token into registers (issued early by callers that have other loads to overlap them with)
template <int NQ>
__device__ __forceinline__ void topk_load(const float * __restrict__ lg, int n_experts, int lane, float (&val)[NQ], bool (&open)[NQ]) {
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        const int i = lane + 64 * q;
        open[q] = i < n_experts;
        val[q] = open[q] ? lg[i] : -INFINITY;
    }
}

// the selection on loaded logits; ids_row / weights_row / ids_copy may be global or LDS rows
template <int NQ>
__device__ __forceinline__ void topk_select(float (&val)[NQ], bool (&open)[NQ], int k, bool renorm, int32_t * ids_row, float * weights_row,
                                            int lane, int * ids_copy = nullptr) {
    float mx = -INFINITY;
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        const float v = val[q];
        val[q] = v != v ? -INFINITY : v;
        mx = fmaxf(mx, val[q]);
    }
    mx = lane63(wave_max_dpp(mx));
    float sum = 0.f;
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        sum += open[q] ? expf(val[q] - mx) : 0.f;
    }
    sum = lane63(wave_sum_dpp(sum));
    // A selection: one wave reduction for the maximum, then the lowest open place that holds it from the lanes' votes, on
    // the scalar unit (with a second reduction, over the indices, and each pick's weight computed where it was picked 8192
    // tokens took 15.9 us, now 11.4; the gate / up GEMV that selects in its prologue 17.7, now 17.1).  A taken expert's
    // logit becomes -inf; the open places stay apart from that for rows of -inf.
    uint64_t left[NQ];
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        left[q] = __ballot(open[q]);
    }
    float mine = 0.f; // lane j keeps the j-th pick
    int mine_id = 0;
    for (int j = 0; j < k; j++) {
        float bv = val[0];
#pragma unroll
        for (int q = 1; q < NQ; q++) {
            bv = fmaxf(bv, val[q]);
        }
        bv = lane63(wave_max_dpp(bv));
        uint32_t bi = 0; // k <= n_experts: an open place holds the maximum of the open ones
#pragma unroll
        for (int q = NQ - 1; q >= 0; q--) {
            const uint64_t at = __ballot(val[q] == bv) & left[q];
            bi = at ? 64 * q + (uint32_t) __builtin_ctzll(at) : bi;
        }
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            left[q] &= ~((bi >> 6) == (uint32_t) q ? 1ull << (bi & 63) : 0ull);
            val[q] = (uint32_t) (lane + 64 * q) == bi ? -INFINITY : val[q];
        }
        mine = lane == j ? bv : mine; // k <= 64
        mine_id = lane == j ? (int) bi : mine_id;
    }
    mine = lane < k ? expf(mine - mx) / sum : 0.f;
    float top = 0.f;
    for (int j = 0; j < k; j++) {
        top += __uint_as_float((uint32_t) __builtin_amdgcn_readlane((int) __float_as_uint(mine), j));
    }
    if (lane < k) {
        ids_row[lane] = mine_id;
        if (ids_copy) {
            ids_copy[lane] = mine_id;
        }
        weights_row[lane] = renorm ? mine / top : mine;
    }
}

template <int NQ>
__device__ __forceinline__ void topk_token(const float * __restrict__ lg, int n_experts, int k, bool renorm, int32_t * ids_row,
                                           float * weights_row, int lane, int * ids_copy = nullptr) {
    float val[NQ];
    bool open[NQ]; // a real expert that has not been taken yet
    topk_load<NQ>(lg, n_experts, lane, val, open);
    topk_select<NQ>(val, open, k, renorm, ids_row, weights_row, lane, ids_copy);
}

// what a GEMV needs to select the experts of its token itself: the router's logits and the rows to leave the result in
struct topk_args {
    const float * logits; int64_t stride; // one row of n_experts logits per token
    int n_experts, k;
    bool renorm;
    float * weights; int64_t out_stride;  // weights row of token t at weights + t * out_stride (the ids go to the launch's id rows)
};

} // namespace dev
} // namespace bf16n
