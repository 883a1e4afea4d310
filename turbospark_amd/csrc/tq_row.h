// One quantized KV row's arithmetic, as a wave does it (kvquant.hip, prompt.hip): every operation is a single rounded f32 operation in
// the reference's order, so that the indices are the reference's by bits.
#pragma once
#include "tsv_internal.h"

namespace tsv {

// crates/compute/src/wht.rs:15-29, bottom-up: stage h pairs i with i + h, (lo + hi) and (lo - hi), each
// scaled by 1/sqrt(2).  Lane l holds elements l and l + 64.
template <int EPL>
__device__ __forceinline__ void wht(float (&e)[EPL], int lane, float c) {
#pragma unroll
    for (int j = 0; j < EPL; j++) {  // the partner on the vector ALU: __shfl_xor goes through the LDS, six times one behind the other
        auto stage = [&](float other, bool upper) { e[j] = __fmul_rn(upper ? __fsub_rn(other, e[j]) : __fadd_rn(e[j], other), c); };
        stage(lane_xor<1>(e[j]), lane & 1);
        stage(lane_xor<2>(e[j]), lane & 2);
        stage(lane_xor<4>(e[j]), lane & 4);
        stage(lane_xor<8>(e[j]), lane & 8);
        const float2 r = lanes_by_16(e[j]);
        stage(lane & 16 ? r.x : r.y, lane & 16);
        const float2 h = lanes_by_32(e[j]);
        stage(lane & 32 ? h.x : h.y, lane & 32);
    }
    if (EPL == 2) {
        const float lo = e[0], hi = e[EPL - 1];
        e[0] = __fmul_rn(__fadd_rn(lo, hi), c);
        e[EPL - 1] = __fmul_rn(__fsub_rn(lo, hi), c);
    }
}

// The side's midpoints, +inf past the last: the index is the count of midpoints below the coordinate
struct TqMidpoints {
    float at[15];
    __device__ __forceinline__ explicit TqMidpoints(const TqSide& t) {
        const int n = (1 << t.bits) - 1;
#pragma unroll
        for (int i = 0; i < 15; i++) {
            const float v = uniform_memory(t.mid)[i];  // the table holds sixteen slots
            at[i] = i < n ? v : INFINITY;
        }
    }
    __device__ __forceinline__ uint32_t index(float e) const {
        uint32_t c = 0;
#pragma unroll
        for (int i = 0; i < 15; i++) c += e > at[i] ? 1u : 0u;
        return c;
    }
};

}  // namespace tsv
