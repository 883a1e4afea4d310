// Flash-decoding split-KV GQA attention for a verify pass on gfx950.
//
// Replaces the reference's per-row loop of split-KV decode dispatches
// (crates/runtime/src/families/qwen/batched_layers.rs:409-430 over
// crates/gpu/src/attention_decode.rs:1092-1363, tree variant :1153-1230); arithmetic contract
// crates/compute/src/attention.rs:53-137.  Differences by design:
//  * ALL rows of the pass (and all q heads of a GQA group) share ONE read of K and V: the
//    (row, q-head-in-group) pairs are the 16-wide N operand of the MFMA, so the KV bytes are
//    read once per layer instead of once per row;
//  * the causal / tree mask over the drafted suffix is a 16-bit ancestor set per row;
//  * S^T = K Q^T is computed with v_mfma_f32_16x16x32_f16 (K positions as the M operand), whose
//    accumulator layout (lane: row j, positions 4*kg..4*kg+3) is exactly the B-operand layout
//    of v_mfma_f32_16x16x16_f16, so O^T += V^T P^T needs no data movement; V is stored in the
//    cache pre-arranged as that MFMA's A fragments.
#include <algorithm>

#include "attn_tq_core.h"

namespace tsv {

int attn_chunks(int nkv) {
    int n = 256 / nkv;
    if (n < 1) n = 1;
    if (n > 64) n = 64;
    return n;
}

// blocks in flight per wave when a workgroup holds two row tiles: two at 128-wide heads (a third block's
// registers would spill), three at 64-wide ones
#ifndef TSV_ATTN_STAGES2_HD128
#define TSV_ATTN_STAGES2_HD128 2
#endif
#ifndef TSV_ATTN_STAGES2_HD64
#define TSV_ATTN_STAGES2_HD64 3
#endif

// Eight waves per workgroup share a chunk of the context (attn_core.h).  Grid (chunks, kv heads, 16-row blocks of a prompt pass).
// What a launch costs beside its bytes is the round trips before the first K and V are asked for: the arguments come in one batch, and nothing
// is divided on the way.
template <int HD, int RT, int STAGES>
__global__ __launch_bounds__(512) void k_attn_partial(AttnArgs a, int G, int R) {
    extern __shared__ float xch[];  // [8 slots][PER_LANE values][64 lanes]
    ask_for_arguments(a, G, R);
    const AttnArgs v = a.blocks > 1 ? attn_block_view(a, blockIdx.z) : a;
    attn_partial_body<HD, RT, STAGES>(v, G, R, blockIdx.x, blockIdx.y, 0, xch);
}

// A pass of more than two row tiles: TG tile groups side by side in one workgroup (attn_core.h), one read of the
// chunk's K / V blocks out of the L2 for all of them.  Grid (chunks, kv heads, 16-row blocks of a prompt pass).
template <int HD, int RT, int STAGES, int TG>
__global__ __launch_bounds__(64 * TG * attn_phases(TG)) void k_attn_partial_groups(AttnArgs a, int G, int R) {
    extern __shared__ float xch[];
    ask_for_arguments(a, G, R);
    const AttnArgs v = a.blocks > 1 ? attn_block_view(a, blockIdx.z) : a;
    attn_partial_body<HD, RT, STAGES, TG>(v, G, R, blockIdx.x, blockIdx.y, 0, xch);
}

// A short context (launch_hd): one workgroup per KV head and row group, which finishes its rows
template <int HD, int RT, int STAGES>
__global__ __launch_bounds__(512) void k_attn_direct(AttnArgs a, int G, int R) {
    extern __shared__ float xch[];
    ask_for_arguments(a, G, R);
    attn_partial_body<HD, RT, STAGES, 1, true>(a, G, R, 0, blockIdx.y, blockIdx.z * RT, xch);
}

// The same pass over a layer that keeps quantized rows (attn_tq_core.h)
template <int HD, int RT, int KB, int VB>
__global__ __launch_bounds__(512) void k_attn_partial_tq(AttnArgs a, int G, int R) {
    extern __shared__ float xch[];
    __shared__ uint32_t s_kpair[1 << (2 * KB)], s_vpair[1 << (2 * VB)];
    asm volatile("" ::"s"(a.tq.kq), "s"(a.tq.kn), "s"(a.tq.vq), "s"(a.tq.vn), "s"(a.tq.k_cb), "s"(a.tq.v_cb), "s"(a.by_xcd_groups.magic), "s"(a.nkv),
                 "s"(a.q16), "s"(a.part_o), "s"(a.part_ml), "s"(a.nq), "s"(a.max_ctx), "s"(a.nch), "s"(a.scale), "s"(a.vp), "s"(a.m_hint), "s"(a.base_hint),
                 "s"(a.blocks), "s"(a.xcd_groups), "s"(a.by_group.magic), "s"(a.by_chunks.magic), "s"(G), "s"(R));
    TqPairs<KB> kp(a.tq.k_cb, threadIdx.x);
    TqPairs<VB> vp(a.tq.v_cb, threadIdx.x);
    // The tables are filled ahead of everything that differs between the waves: how many blocks a wave has chooses its walk, and no barrier may stand in one.
    // (Behind the first blocks' loads all waves had to share one walk, whose loads stood under tail conditions: one, four and sixteen rows over 6001
    // positions 7.9, 8.9 and 16.2 us for 6.8, 7.7 and 14.1; 3-bit and 2-bit keys, four rows over 12000, 13.1 and 11.5 for 11.4 and 9.9.)
    kp.put(s_kpair, threadIdx.x);
    vp.put(s_vpair, threadIdx.x);
    __syncthreads();
    // blocks in flight: three, two where the three-bit fields' extra words would push the registers past 256
    constexpr int STAGES = (HD == 128 && RT == 2 && KB == 3 && VB == 3) ? 2 : 3;
    // several row groups of a verify pass are placed by die; else grid z: row groups of the pass, times the 16-row blocks of a prompt pass
    int chunk = blockIdx.x, kvh = blockIdx.y, grp = blockIdx.z, blk = 0;
    if (a.xcd_groups) {
        if (!attn_grid_place(a, blockIdx.x, chunk, kvh, grp)) return;
    } else if (a.blocks > 1) {
        const int groups = gridDim.z / a.blocks;
        blk = blockIdx.z / groups;
        grp = blockIdx.z - blk * groups;
    }
    const AttnArgs v = a.blocks > 1 ? attn_block_view(a, blk) : a;
    attn_partial_body_tq<HD, RT, STAGES, KB, VB>(v, G, R, chunk, kvh, grp * RT, xch, s_kpair, s_vpair);
}

// Merge the chunk partials (crates/gpu/src/shaders/attention.metal:122-140 semantics:
// m* = max m_c, D = sum l_c e^{m_c-m*}, O = sum O_c e^{m_c-m*}, out = O / D) and store the row
// as fp16 activation fragments (and sub-block sums) of the output projection (K index =
// q_head*hd + d).  Every wave turns the (m_c, l_c) pairs into per-chunk weights, lane c chunk c's, and hands them to all of its
// lanes through scalar registers: no LDS and no barrier (with them, arguments fetched where they were needed and lane sums through the LDS the merge
// of 32 chunks took 3.4 us in the 8B step).
// NCH > 0: the chunk count as a compile-time constant -- every thread then asks for its output
// element of all chunks before the (m, l) pairs are looked at (the two groups of loads do not
// depend on each other), and the kernel is one memory latency instead of two.  NCH == 0: any count, the first 32 chunks that
// way, then 32 more at a time.  (A loop over chunks is not unrolled here whatever a pragma asks, because it reads lanes: with
// a round trip for each of 64 chunks the merge of one row of 32 heads took 17.5 us.)
template <int NCH, bool UNROT>
__global__ __launch_bounds__(128) void k_attn_combine(AttnArgs a0, int G, int R) {
    asm volatile("" ::"s"(a0.part_o), "s"(a0.part_ml), "s"(a0.xfrag), "s"(a0.nq), "s"(a0.hd), "s"(a0.nch), "s"(a0.sinks), "s"(a0.frag16), "s"(a0.unrot),
                 "s"(a0.blocks), "s"(a0.by_group.magic), "s"(G), "s"(R));
    const AttnArgs a = a0.blocks > 1 ? attn_block_view(a0, blockIdx.z) : a0;
    const int m = blockIdx.x, qh = blockIdx.y, t = threadIdx.x, lane = t & 63;
    const int hd = a.hd, nch = NCH > 0 ? NCH : a.nch;  // (the workgroup has hd threads, 64 or 128)
    const int h = a.by_group.quotient(qh), g = qh - h * G, r = m * G + g;
    const long slot0 = (long)h * nch * R + r;
    const float* const po = a.part_o + slot0 * hd;
    const long stride = (long)R * hd;
    auto element = [&](int c) { return *(const float*)((const char*)(po + c * stride) + (uint32_t)(t * 4)); };
    // (a lane past the last chunk: the last chunk's pair, not used)
    const float2 ml = *(const float2*)(a.part_ml + (slot0 + (long)min(lane, nch - 1) * R) * 2);
    constexpr int BATCH = NCH > 0 ? NCH : 32;
    float pre[BATCH];
#pragma unroll
    for (int c = 0; c < BATCH; c++) pre[c] = element(NCH > 0 ? c : min(c, nch - 1));
    const float sink = a.sinks ? uniform_memory(a.sinks)[qh] : -INFINITY;
    const float sign = UNROT ? a.unrot[t] : 1.0f;
    const bool live = lane < nch;
    const float mc = live ? ml.x : -INFINITY, lc = live ? ml.y : 0.f;
    // the sink joins the maximum and the denominator, never the numerator
    // (crates/compute/src/attention.rs:94-105)
    const float mx = fmaxf(max_of_wave(mc), sink);
    const float w = mc > -INFINITY ? __expf(mc - mx) : 0.f;
    float den = sum_of_wave(lc * w);
    if (a.sinks) den += __expf(sink - mx);
    auto weight = [&](int c) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, w), c)); };
    float num = 0.f;
#pragma unroll
    for (int c = 0; c < BATCH; c++)
        if (NCH > 0 || c < nch) num = fmaf(weight(c), pre[c], num);
    if (NCH == 0)
        for (int c0 = BATCH; c0 < nch; c0 += BATCH) {
#pragma unroll
            for (int c = 0; c < BATCH; c++) pre[c] = element(min(c0 + c, nch - 1));
#pragma unroll
            for (int c = 0; c < BATCH; c++)
                if (c0 + c < nch) num = fmaf(weight(c0 + c), pre[c], num);
        }
    float res = num / den;
    if (UNROT) {
        // the sum was taken over rotated value rows: back through the normalized Hadamard transform
        // (crates/compute/src/wht.rs:15-29, stage h pairs d with d + h) and the value signs
        __shared__ float s_h[128];
        const float c = 0.70710678118654752440f;
        auto stage = [&](float other, bool upper) { res = (upper ? other - res : res + other) * c; };
        stage(lane_xor<1>(res), lane & 1);
        stage(lane_xor<2>(res), lane & 2);
        stage(lane_xor<4>(res), lane & 4);
        stage(lane_xor<8>(res), lane & 8);
        const float2 p = lanes_by_16(res);
        stage(lane & 16 ? p.x : p.y, lane & 16);
        const float2 q = lanes_by_32(res);
        stage(lane & 32 ? q.x : q.y, lane & 32);
        if (hd == 128) {  // the two waves' halves
            s_h[t] = res;
            __syncthreads();
            stage(s_h[t ^ 64], t & 64);
        }
        res *= sign;
    }
    const _Float16 o16 = pinned_half((_Float16)res);
    const int kk = qh * hd + t;
    ((_Float16*)a.xfrag)[a.frag16 ? frag16_index(kk, m) : frag_index(kk, m)] = o16;
    // sum of each 32-element sub-block of the output projection's input (32 neighbouring threads)
    const float sum = sum_of_32((float)o16);
    if ((t & 31) == 0) ((float*)((char*)a.xfrag + xfrag_sum_offset(a.nq * hd)))[xsum_index(kk >> 5, m)] = sum;
}

template <int HD, int RT, int STAGES>
static int launch_partial(hipStream_t s, const AttnArgs& a, int G, int R) {
    constexpr int PER_LANE = RT * (HD / 16) * 4 + 2 * RT;
    constexpr size_t lds = (size_t)8 * 64 * PER_LANE * 4;
    static OncePerDevice allowed;
    if (int rc = allow_lds((const void*)k_attn_partial<HD, RT, STAGES>, lds, allowed)) return rc;
    hipLaunchKernelGGL((k_attn_partial<HD, RT, STAGES>), dim3(a.nch, a.nkv, std::max(a.blocks, 1)), dim3(512), lds, s, a, G, R);
    TSV_HIP(hipGetLastError());
    return TSV_OK;
}

template <int HD, int RT, int STAGES>
static int launch_direct(hipStream_t s, const AttnArgs& a, int G, int R, int groups) {
    constexpr int PER_LANE = RT * (HD / 16) * 4 + 2 * RT;
    constexpr size_t lds = (size_t)8 * 64 * PER_LANE * 4;
    static OncePerDevice allowed;
    if (int rc = allow_lds((const void*)k_attn_direct<HD, RT, STAGES>, lds, allowed)) return rc;
    hipLaunchKernelGGL((k_attn_direct<HD, RT, STAGES>), dim3(1, a.nkv, groups), dim3(512), lds, s, a, G, R);
    TSV_HIP(hipGetLastError());
    return TSV_OK;
}

template <int HD, int RT, int STAGES, int TG>
static int launch_partial_groups(hipStream_t s, const AttnArgs& a, int G, int R) {
    constexpr int PER_LANE = RT * (HD / 16) * 4 + 2 * RT, NW = attn_phases(TG);
    const size_t lds = (size_t)TG * NW * 64 * PER_LANE * 4;
    static OncePerDevice allowed;
    if (int rc = allow_lds((const void*)k_attn_partial_groups<HD, RT, STAGES, TG>, lds, allowed)) return rc;
    hipLaunchKernelGGL((k_attn_partial_groups<HD, RT, STAGES, TG>), dim3(a.nch, a.nkv, std::max(a.blocks, 1)), dim3(64 * TG * NW),
                       lds, s, a, G, R);
    TSV_HIP(hipGetLastError());
    return TSV_OK;
}

template <int HD>
static int launch_combine(hipStream_t s, const AttnArgs& a, int m, int G, int R);

template <int HD, int RT, int KB, int VB>
static int launch_partial_tq(hipStream_t s, const AttnArgs& a, int G, int R, int groups) {
    constexpr int PER_LANE = RT * (HD / 16) * 4 + 2 * RT;
    const size_t lds = (size_t)8 * 64 * PER_LANE * 4;
    static OncePerDevice allowed;  // (36, 68, 72 or 136 KiB: the pair tables, 2 KiB of static LDS at most, take none of them over the line)
    if (int rc = allow_lds((const void*)k_attn_partial_tq<HD, RT, KB, VB>, lds, allowed)) return rc;
    const dim3 grid = a.xcd_groups ? dim3(attn_grid_size(a.nch * a.nkv, groups)) : dim3(a.nch, a.nkv, groups * std::max(a.blocks, 1));
    hipLaunchKernelGGL((k_attn_partial_tq<HD, RT, KB, VB>), grid, dim3(512), lds, s, a, G, R);
    TSV_HIP(hipGetLastError());
    return TSV_OK;
}
template <int HD, int RT>
static int launch_partial_tq_widths(hipStream_t s, const AttnArgs& a, int G, int R, int groups) {
    const int kb = a.tq.k_bits, vb = a.tq.v_bits;
    if (kb == 4 && vb == 4) return launch_partial_tq<HD, RT, 4, 4>(s, a, G, R, groups);
    if (kb == 3 && vb == 4) return launch_partial_tq<HD, RT, 3, 4>(s, a, G, R, groups);
    if (kb == 3 && vb == 3) return launch_partial_tq<HD, RT, 3, 3>(s, a, G, R, groups);
    if (kb == 2 && vb == 2) return launch_partial_tq<HD, RT, 2, 2>(s, a, G, R, groups);
    set_error("attention: no kernel for these KV quantization widths");
    return TSV_ERR_UNSUPPORTED;
}

template <int HD>
static int launch_hd(hipStream_t s, const AttnArgs& a0, int m, int G, int R) {
    const int trt = (R + 15) / 16;
    // more than 32 (row, q head) pairs: groups of 32, each re-reading K and V (from L2)
    const int groups = trt <= 2 ? 1 : (trt + 1) / 2;
    // about one workgroup per compute unit: the chunk count shrinks as the row groups multiply
    // (fewer, longer chunks also mean fewer partial results for the merge to read)
    AttnArgs a = a0;
    a.by_group = UniformDivisor(G);
    // A short context in one workgroup per KV head and row group, up to ATTN_DIRECT_BLOCKS / 8 blocks a wave, which finishes its rows
    // itself.  What that takes off a layer against chunks and a merge (8B shape, 1 / 5 / 16 rows, us): 2.5 / 2.9 / 5.3 at 250 positions,
    // 0.7 / 0.6 / 3.5 at 490, and with the line further out 0.0 / -0.6 / 2.4 at 620, -0.4 / -1.2 / 1.8 at 730; four KV heads with groups
    // of eight, five rows: 2.6 at 250, 0.2 at 490, -0.8 at 620.
    // A wave walks more blocks alone the longer the context is; the line lies where the first form of all, one group of two row tiles,
    // begins to lose.  The others would still gain behind it (sixteen rows), but a line by rows would make a row's bits depend
    // on its pass over a range of positions.  As it is they do where the passes' ends lie on two sides of the line, which is one of the
    // 16-position boundaries at which the chunks change.  Layers of a short window always go this way (a window's blocks: its own, the
    // pass's, one cut).  All row groups take the form of eight phases here, so that a row's sums do not depend on how many share its pass.
    const bool few = attn_short(a.kv_end) || (a.window > 0 && (a.window + TSV_MAX_ROWS + 14) / 16 + 1 <= ATTN_DIRECT_BLOCKS);
    if (a.kv_end > 0 && a.blocks <= 1 && !a.tq.k_bits && !a.frag16 && few) {
        a.nch = 1;
        a.by_chunks = UniformDivisor(1);
        return trt <= 1 ? launch_direct<HD, 1, 3>(s, a, G, R, 1)
                        : launch_direct<HD, 2, (HD == 128 ? TSV_ATTN_STAGES2_HD128 : TSV_ATTN_STAGES2_HD64)>(s, a, G, R, groups);
    }
    a.nch = std::max(std::min(a0.nch, 8), std::min(a0.nch, 256 / (a0.nkv * groups * std::max(a0.blocks, 1))));
    // Several row groups of a verify pass read the same K / V: they are placed on one die.  A workgroup fills a
    // compute unit (eight waves at two per SIMD) and a die has 32 of them: no die may be handed more than 32
    // workgroups, or its last one waits for a whole workgroup to end (26 against 18 us at 21 chunks x 4 heads x 3)
    a.xcd_groups = (groups > 1 && a0.blocks <= 1) ? groups : 0;
    if (a.xcd_groups) a.nch = std::max(std::min(a0.nch, 8), std::min(a0.nch, 8 * (32 / groups) / a0.nkv));
    a.by_chunks = UniformDivisor(a.nch);
    if (a.xcd_groups) a.by_xcd_groups = UniformDivisor(a.xcd_groups);
    int rc;
    if (a.tq.k_bits) {
        if (a.window || a.ring || !a.unrot) {
            set_error("attention: quantized rows go with full attention and a linear cache");
            return TSV_ERR_UNSUPPORTED;
        }
        rc = trt <= 1 ? launch_partial_tq_widths<HD, 1>(s, a, G, R, 1) : launch_partial_tq_widths<HD, 2>(s, a, G, R, groups);
    } else if (trt <= 1)
        rc = launch_partial<HD, 1, 3>(s, a, G, R);
    else if (trt <= 2)
        rc = launch_partial<HD, 2, (HD == 128 ? TSV_ATTN_STAGES2_HD128 : TSV_ATTN_STAGES2_HD64)>(s, a, G, R);
    else {
        // more row tiles than a wave holds: tile groups inside one workgroup, about one workgroup per compute unit
        a.xcd_groups = 0;
        a.nch = std::max(1, std::min(a0.nch, 256 / (a0.nkv * std::max(a0.blocks, 1))));
        // (64 chunks at four KV heads would fill the chip, but what the partial pass wins the merge loses reading
        // twice the partial results: 10.9 + 6.0 us against 12.9 + 4.1 us at the Qwen3-30B-A3B shape)
        if (a.nch > 32) a.nch = 32;
        a.by_chunks = UniformDivisor(a.nch);
        constexpr int ST = HD == 128 ? TSV_ATTN_STAGES2_HD128 : TSV_ATTN_STAGES2_HD64;
        if (HD == 64 && trt >= 7)
            rc = launch_partial_groups<HD, (HD == 64 ? 4 : 2), 2, 2>(s, a, G, R);
        else if (HD == 64 && trt >= 5)
            rc = launch_partial_groups<HD, (HD == 64 ? 3 : 2), 2, 2>(s, a, G, R);
        else if (trt <= 4)
            rc = launch_partial_groups<HD, 2, ST, 2>(s, a, G, R);
        else if (trt <= 6)
            rc = launch_partial_groups<HD, 2, ST, 3>(s, a, G, R);
        else
            rc = launch_partial_groups<HD, 2, ST, 4>(s, a, G, R);
    }
    if (rc) return rc;
    return launch_combine<HD>(s, a, m, G, R);
}

template <int HD>
static int launch_combine(hipStream_t s, const AttnArgs& a, int m, int G, int R) {
    static_assert(HD == 64 || HD == 128, "whole waves, one thread to a dimension");
    const dim3 cgrid(m, a.nq, std::max(a.blocks, 1)), cblock(HD);
    // the chunk count as a compile-time constant puts every partial's load in flight before the
    // first add (a counted loop waits on each in turn); the sum runs in the same order either way
    // UNROT: the variant that rotates each head's result back (quantized KV rows); the other one is unchanged code
#define TSV_COMBINE(N)                                                                         \
    case N:                                                                                    \
        if (a.unrot)                                                                           \
            hipLaunchKernelGGL((k_attn_combine<N, true>), cgrid, cblock, 0, s, a, G, R);       \
        else                                                                                   \
            hipLaunchKernelGGL((k_attn_combine<N, false>), cgrid, cblock, 0, s, a, G, R);      \
        break;
    switch (a.nch) {
        TSV_COMBINE(1) TSV_COMBINE(2) TSV_COMBINE(3) TSV_COMBINE(4) TSV_COMBINE(5) TSV_COMBINE(6) TSV_COMBINE(7) TSV_COMBINE(8)
        TSV_COMBINE(9) TSV_COMBINE(10) TSV_COMBINE(11) TSV_COMBINE(12) TSV_COMBINE(13) TSV_COMBINE(14) TSV_COMBINE(15)
        TSV_COMBINE(16) TSV_COMBINE(17) TSV_COMBINE(18) TSV_COMBINE(19) TSV_COMBINE(20) TSV_COMBINE(21) TSV_COMBINE(22)
        TSV_COMBINE(23) TSV_COMBINE(24) TSV_COMBINE(25) TSV_COMBINE(26) TSV_COMBINE(27) TSV_COMBINE(28) TSV_COMBINE(29)
        TSV_COMBINE(30) TSV_COMBINE(31) TSV_COMBINE(32)
        default:
            if (a.unrot)
                hipLaunchKernelGGL((k_attn_combine<0, true>), cgrid, cblock, 0, s, a, G, R);
            else
                hipLaunchKernelGGL((k_attn_combine<0, false>), cgrid, cblock, 0, s, a, G, R);
            break;
    }
#undef TSV_COMBINE
    TSV_HIP(hipGetLastError());
    return TSV_OK;
}

// the merge alone, over partials some other kernel left (a.nch chunks)
int launch_attention_merge(hipStream_t s, const AttnArgs& a0, int m) {
    AttnArgs a = a0;
    const int G = a.nq / a.nkv, R = m * G;
    a.by_group = UniformDivisor(G);
    return a.hd == 128 ? launch_combine<128>(s, a, m, G, R) : launch_combine<64>(s, a, m, G, R);
}

int launch_attention(hipStream_t s, const AttnArgs& a, int m) {
    const int G = a.nq / a.nkv, R = m * G;
    if (a.hd == 128) return launch_hd<128>(s, a, m, G, R);
    if (a.hd == 64) return launch_hd<64>(s, a, m, G, R);
    set_error("attention: head_dim must be 64 or 128");
    return TSV_ERR_UNSUPPORTED;
}

}  // namespace tsv
