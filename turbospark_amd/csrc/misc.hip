// Small per-row kernels of the verify pass: embedding lookup, residual-add + RMSNorm,
// q/k rotation + KV-cache store, KV row gather / read-back.
#include <type_traits>

#include "embed_row.h"
#include "tsv_internal.h"
#include "x8.h"

namespace tsv {

// ---------------------------------------------------------------- embedding lookup
// One dequantized table row per fed token (crates/runtime/src/real_forward_dispatch.rs:154),
// arithmetic of dequantize_q4_k / dequantize_q8_0.
// The last workgroup of a row (when `cs` is given) fills the row's rotation table instead:
// (cos, sin) of pos * freq, scaled, for every pair index - the same for all layers of the step.
__device__ __forceinline__ void embed_rows(const uint8_t* raw, int dtype, int hidden, float* x, long tok, int rot_pos, const float* freqs, float mscale,
                                           int half, float2* cs, int nblk) {
    const int m = blockIdx.x;
    if ((int)blockIdx.y == nblk) {
        const float pos = (float)rot_pos;
        for (int i = threadIdx.x; i < half; i += blockDim.x) {
            float sn, c;
            sincosf(pos * freqs[i], &sn, &c);
            cs[m * half + i] = float2{c * mscale, sn * mscale};
        }
        return;
    }
    // (workgroups of 256, two values to a thread)
    embed_types(dtype, [&](auto type) {
        float v[2];
        const int e0 = blockIdx.y * 256 + threadIdx.x, step = 256 * nblk;
#pragma unroll
        for (int j = 0; j < 2; j++) v[j] = embed_elem<decltype(type)::value>(raw, hidden, tok, min(e0 + j * step, hidden - 1));
#pragma unroll
        for (int j = 0; j < 2; j++)
            if (e0 + j * step < hidden) x[(long)m * hidden + e0 + j * step] = v[j];
    });
}
__global__ void k_embed(const uint8_t* __restrict__ raw, int dtype, int hidden, float* __restrict__ x,
                        const VerifyParams* __restrict__ vp, const float* __restrict__ freqs, float mscale,
                        int half, float2* __restrict__ cs, int nblk) {
    const int m = blockIdx.x;
    if (m >= vp->m) return;
    embed_rows(raw, dtype, hidden, x, vp->feed[m], vp->pos[m], freqs, mscale, half, cs, nblk);
}
// ... with the pass's parameters by value, and an acceptance's, which the first workgroup leaves in device memory
struct EmbedCall {
    VerifyParams vp;
    AcceptUpload accept;
    VerifyParams* vp_dev;
    AcceptUpload* accept_dev;  // nullable
};
__global__ void k_embed_call(const uint8_t* __restrict__ raw, int dtype, int hidden, float* __restrict__ x, EmbedCall now, const float* __restrict__ freqs,
                             float mscale, int half, float2* __restrict__ cs, int nblk) {
    static_assert(sizeof(VerifyParams) % 4 == 0 && sizeof(AcceptUpload) % 4 == 0, "copied by words");
    if (blockIdx.x == 0 && blockIdx.y == 0) {
        for (int i = threadIdx.x; i < (int)(sizeof(VerifyParams) / 4); i += blockDim.x) ((uint32_t*)now.vp_dev)[i] = ((const uint32_t*)&now.vp)[i];
        if (now.accept_dev)
            for (int i = threadIdx.x; i < (int)(sizeof(AcceptUpload) / 4); i += blockDim.x) ((uint32_t*)now.accept_dev)[i] = ((const uint32_t*)&now.accept)[i];
    }
    embed_rows(raw, dtype, hidden, x, now.vp.feed[blockIdx.x], now.vp.pos[blockIdx.x], freqs, mscale, half, cs, nblk);
}

int launch_embed(hipStream_t s, const uint8_t* raw, int dtype, int hidden, float* x,
                 const VerifyParams* vp, int m, const float* freqs, float mscale, int half, float2* cs, const PassUpload* now) {
    const int nblk = (hidden + 511) / 512;  // two elements per thread
    const dim3 grid(m, nblk + (cs ? 1 : 0));
    if (now) {
        EmbedCall call{};
        call.vp = *now->vp;
        call.vp_dev = now->vp_dev;
        if (now->accept) {
            call.accept = *now->accept;
            call.accept_dev = now->accept_dev;
        }
        hipLaunchKernelGGL(k_embed_call, grid, dim3(256), 0, s, raw, dtype, hidden, x, call, freqs, mscale, half, cs, nblk);
    } else {
        hipLaunchKernelGGL(k_embed, grid, dim3(256), 0, s, raw, dtype, hidden, x, vp, freqs, mscale, half, cs, nblk);
    }
    TSV_HIP(hipGetLastError());
    return TSV_OK;
}

// ---------------------------------------------------------------- residual add + RMSNorm
// The sum over a workgroup of 1024 threads: within each wave on the vector ALU, then the sixteen waves' in order.  `red`: 16 floats that nothing
// else uses until the next barrier.
__device__ __forceinline__ float block_sum(float v, float* red) {
    v = sum_of_wave(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    float4 r[4];
#pragma unroll
    for (int i = 0; i < 4; i++) r[i] = ((const float4*)red)[i];
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        t += r[i].x;
        t += r[i].y;
        t += r[i].z;
        t += r[i].w;
    }
    return t;
}

// x[m] += sum over split-K partials of the previous matmul (fixed order: deterministic), then
// y = x * w / sqrt(mean x^2 + eps) (crates/compute/src/rms_norm.rs:5-14) stored as the next
// matmul's fp16 activation fragments plus the sums of the rounded values over every 32-element
// sub-block (eight neighbouring threads).  One workgroup per row, four consecutive elements per
// thread so every load of a row is issued before the first one is waited on.
// What bounds it is one round trip behind the other: the arguments, the row, the sum over the workgroup.  So the partial sums' count and
// whether they are weighted are known at compile time (chosen by a branch in the kernel, nine bodies had to be jumped over, in an instruction
// cache that the launches before have filled), the bias is asked for with the row, and the sums stay out of the LDS's permutes.
struct AddNormArgs {
    float* x;
    const float* partial;
    const float* w;
    _Float16* xfrag;
    const float* weights;  // WEIGHTED: [16][8] factors
    const float* bias;     // nullable; else
    int ldp, hidden, x8_terms;
    float eps;
    NormBlocks nb;
    X8 x8;
};
template <int NS, bool WEIGHTED>
__global__ __launch_bounds__(1024) void k_addnorm(AddNormArgs a) {
    __shared__ __attribute__((aligned(16))) float red[16];
    asm volatile("" ::"s"(a.x), "s"(a.partial), "s"(a.w), "s"(a.xfrag), "s"(a.weights), "s"(a.bias), "s"(a.ldp), "s"(a.hidden), "s"(a.x8_terms), "s"(a.eps),
                 "s"(a.nb.x), "s"(a.nb.partial), "s"(a.nb.frag), "s"(a.nb.frag16), "s"(a.nb.frag2));
    const int m = blockIdx.x, blk = blockIdx.y, hidden = a.hidden, n4 = hidden >> 2;
    // a prompt pass of several 16-row blocks: block blockIdx.y has its own rows, partial sums and fragments
    float4* const xr = (float4*)(a.x + (long)blk * a.nb.x + (long)m * hidden);
    const float* const partial = a.partial + (long)blk * a.nb.partial + (long)m * a.ldp;
    _Float16* const xfrag = (_Float16*)((char*)a.xfrag + (long)blk * a.nb.frag);
    const float4* const wr = (const float4*)a.w;
    float ws[NS > 0 ? NS : 1];
    if (WEIGHTED) {  // (block b's factors follow block b - 1's)
#pragma unroll
        for (int s = 0; s < NS; s++) ws[s] = uniform_memory(a.weights)[(blk * 16 + m) * 8 + s];
    }
    auto add = [&](int i) {
        float4 v = xr[i];
        float4 p[NS > 0 ? NS : 1];
#pragma unroll
        for (int s = 0; s < NS; s++) p[s] = *(const float4*)(partial + (long)s * 16 * a.ldp + 4 * i);
        if (WEIGHTED) {
            // routed experts (families/llama/moe.rs:193-198): the slot outputs are weighted and summed
            // in rank order starting from zero, then added to the stream; product and sum rounded apart
            float4 r = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < NS; s++) {
                r.x = __fadd_rn(r.x, __fmul_rn(ws[s], p[s].x));
                r.y = __fadd_rn(r.y, __fmul_rn(ws[s], p[s].y));
                r.z = __fadd_rn(r.z, __fmul_rn(ws[s], p[s].z));
                r.w = __fadd_rn(r.w, __fmul_rn(ws[s], p[s].w));
            }
            v.x = __fadd_rn(v.x, r.x);
            v.y = __fadd_rn(v.y, r.y);
            v.z = __fadd_rn(v.z, r.z);
            v.w = __fadd_rn(v.w, r.w);
        } else {
            float4 b = {0.f, 0.f, 0.f, 0.f};
            if (a.bias) b = *(const float4*)(a.bias + 4 * i);  // the output projection's (families/gptoss/mod.rs:16)
#pragma unroll
            for (int s = 0; s < NS; s++) {
                v.x = __fadd_rn(v.x, p[s].x);
                v.y = __fadd_rn(v.y, p[s].y);
                v.z = __fadd_rn(v.z, p[s].z);
                v.w = __fadd_rn(v.w, p[s].w);
            }
            if (a.bias) {
                v.x += b.x;
                v.y += b.y;
                v.z += b.z;
                v.w += b.w;
            }
        }
        xr[i] = v;
        return v;
    };
    auto squares = [](const float4& v) { return v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w; };
    const int mine = threadIdx.x;
    float4 v_first = {0.f, 0.f, 0.f, 0.f}, g_first = v_first;
    float ss = 0.f;
    if (mine < n4) {
        // the norm weights are asked for now: they come from HBM (nothing else reads them in a step)
        // and would otherwise be waited for after the reduction
        g_first = wr[mine];
        v_first = add(mine);
        ss += squares(v_first);
        for (int i = mine + 1024; i < n4; i += 1024) ss += squares(add(i));
    }
    ss = block_sum(ss, red);
    const float inv = 1.0f / sqrtf(ss / (float)hidden + a.eps);
    float* sums = (float*)((char*)xfrag + xfrag_sum_offset(hidden));
    auto finish = [&](int i, const float4& v, const float4& g) {
        // elements 4i..4i+3 are one K step of the fragment layout, stored in the order (0, 2, 1, 3)
        typedef _Float16 half4 __attribute__((ext_vector_type(4)));
        typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
        // (the products as floats first: a product converted in the instruction that makes it is rounded once, and which ones that happens to
        // would differ from one count of partial sums to the next)
        float e[4] = {v.x * g.x * inv, v.z * g.z * inv, v.y * g.y * inv, v.w * g.w * inv};
        asm volatile("" : "+v"(e[0]), "+v"(e[1]), "+v"(e[2]), "+v"(e[3]));
        half4 h = {(_Float16)e[0], (_Float16)e[1], (_Float16)e[2], (_Float16)e[3]};
        // The sums must be those of the stored bits: the matmuls multiply them by the weights' code offsets
        // (up to 1024), so one value rounded differently on the way to the sum than on the way to the store
        // is an error a thousand times its size.  The compiler is free to convert the same product twice, by
        // different instructions; pinning the packed halves in registers leaves it one copy to read.
        u32x2_t hb = __builtin_bit_cast(u32x2_t, h);
        asm volatile("" : "+v"(hb.x), "+v"(hb.y));
        h = __builtin_bit_cast(half4, hb);
        *(half4*)(xfrag + (a.nb.frag16 ? frag16_index(4 * i, m) : frag_index(4 * i, m))) = h;
        float sum = ((float)h.x + (float)h.y) + ((float)h.z + (float)h.w);
        sum += dpp_f32<0xB1>(sum);   // over eight lanes: l ^ 1, l ^ 2, l ^ 4
        sum += dpp_f32<0x4E>(sum);
        sum += dpp_f32<0x141>(sum);
        if ((i & 7) == 0) sums[xsum_index(i >> 3, m)] = sum;
        if (a.nb.frag2) {  // the same fragments once more, in the other of the two layouts (sums included)
            _Float16* x2 = (_Float16*)((char*)a.nb.frag2 + (long)blk * a.nb.frag);
            *(half4*)(x2 + (a.nb.frag16 ? frag_index(4 * i, m) : frag16_index(4 * i, m))) = h;
            if ((i & 7) == 0) ((float*)((char*)x2 + xfrag_sum_offset(hidden)))[xsum_index(i >> 3, m)] = sum;
        }
        if (a.x8_terms) {
            // the same row as block-scaled fp8 terms, from the unrounded values; the eight threads of a
            // 32-element block are neighbours in one wave (hidden is a multiple of 32)
            float r[4] = {v.x * g.x * inv, v.z * g.z * inv, v.y * g.y * inv, v.w * g.w * inv};
            for (int t = 0; t < a.x8_terms; t++) {
                float amax = x8_amax4(r);
                amax = fmaxf(amax, __shfl_xor(amax, 1));
                amax = fmaxf(amax, __shfl_xor(amax, 2));
                amax = fmaxf(amax, __shfl_xor(amax, 4));
                const int byte = x8_scale_byte(amax);
                const uint32_t word = x8_term4(r, byte);
                *(uint32_t*)(a.x8.q + ((size_t)t * 16 + m) * a.x8.kpad + 4 * i) = word;
                if ((i & 7) == 0) a.x8.s[((size_t)t * 16 + m) * (a.x8.kpad >> 5) + (i >> 3)] = (uint8_t)byte;
            }
        }
    };
    if (mine >= n4) return;
    finish(mine, v_first, g_first);
    for (int i = mine + 1024; i < n4; i += 1024) finish(i, xr[i], wr[i]);
}

int launch_addnorm(hipStream_t s, float* x, const float* partial, int splits, int ldp, const float* w,
                   float eps, int hidden, uint4* xfrag, int m, const float* weights, const float* bias, const X8* x8,
                   int x8_terms, int blocks, const NormBlocks* nb) {
    if (splits < 0 || splits > 8) {
        set_error("residual add: at most eight partial sums");
        return TSV_ERR_UNSUPPORTED;
    }
    const AddNormArgs a{x,     partial, w,      (_Float16*)xfrag,          weights, bias, ldp,
                        hidden, x8 ? x8_terms : 0, eps, nb ? *nb : NormBlocks{}, x8 ? *x8 : X8{}};
    const dim3 grid(m, blocks);
#define TSV_ADDNORM(N)                                                                               \
    case N:                                                                                          \
        if (weights) hipLaunchKernelGGL((k_addnorm<N, true>), grid, dim3(1024), 0, s, a);            \
        else hipLaunchKernelGGL((k_addnorm<N, false>), grid, dim3(1024), 0, s, a);                   \
        break;
    switch (splits) {
        TSV_ADDNORM(0) TSV_ADDNORM(1) TSV_ADDNORM(2) TSV_ADDNORM(3) TSV_ADDNORM(4) TSV_ADDNORM(5) TSV_ADDNORM(6) TSV_ADDNORM(7) TSV_ADDNORM(8)
    }
#undef TSV_ADDNORM
    TSV_HIP(hipGetLastError());
    return TSV_OK;
}

// ---------------------------------------------------------------- the drafter head's input
// fc's input rows (docs/MTP.md:53-60, families/qwen/mtp.rs:512-590) as matmul fragments, one workgroup per row:
//   [ norm_e(e) ; norm_h(norm_t(h)) ]   e = the embedding row of the row's NEXT token (from the parameter block, or
//   for row 0 from device memory: a proposal the step before picked on the GPU), h = the residual row of the row's
//   position; every norm is x * w / sqrt(mean x^2 + eps) (crates/compute/src/rms_norm.rs:5-14).
// Also the row's rotation table (as the embedding kernel leaves it), and the row of the head's own residual
// stream `x_zero` cleared LAST -- it may be the very row h was read from (a chained step), and fc's partial sums
// are added onto it by the layer's first residual kernel.  Embedding lookup, three norms, the fragment conversion
// and the token hand-over were four launches and a copy before.
template <int J>  // values to a thread: hidden <= 1024 J
__global__ __launch_bounds__(1024) void k_mtp_input(const uint8_t* __restrict__ raw, int dtype, const VerifyParams* __restrict__ vp,
                                                    const int32_t* __restrict__ token_dev, int vocab, const float* h_rows,
                                                    const float* __restrict__ w_e, const float* __restrict__ w_t,
                                                    const float* __restrict__ w_h, float eps, int hidden,
                                                    _Float16* __restrict__ xfrag, float* x_zero,
                                                    const float* __restrict__ freqs, float mscale, int half,
                                                    float2* __restrict__ cs) {
    __shared__ __attribute__((aligned(16))) float red[3][16];
    const int m = blockIdx.x;
    asm volatile("" ::"s"(raw), "s"(dtype), "s"(vp), "s"(token_dev), "s"(vocab), "s"(h_rows), "s"(w_e), "s"(w_t), "s"(w_h), "s"(eps), "s"(hidden), "s"(xfrag),
                 "s"(x_zero), "s"(freqs), "s"(mscale), "s"(half), "s"(cs));
    const int rows = uniform_memory(vp)->m, fed = uniform_memory(vp)->feed[m], rot = uniform_memory(vp)->pos[m];
    const int drawn = uniform_memory(token_dev ? token_dev : (const int32_t*)vp)[0];
    // The row and the norms' weights are asked for before the token is waited for, and the angles come last: one workgroup is all
    // there is at a single row, and what it costs is the round trips one behind the other (11.1 -> 10.5 us under a trace; 48 tokens of the loop 16107 -> 15742)
    const float* h = h_rows + (long)m * hidden;
    // J elements per thread, kept in registers across the reductions
    const float freq = freqs[min((int)threadIdx.x, half - 1)];
    float ev[J], hv[J], ge[J], gt[J], gh[J];
#pragma unroll
    for (int j = 0; j < J; j++) {
        const int i = threadIdx.x + 1024 * j;
        if (i < hidden) {
            hv[j] = h[i];
            ge[j] = w_e[i];
            gt[j] = w_t[i];
            gh[j] = w_h[i];
        } else {
            hv[j] = ge[j] = gt[j] = gh[j] = 0.f;
        }
    }
    if (m >= rows) return;
    long tok = fed;
    if (token_dev && m == 0) tok = drawn < 0 ? 0 : drawn >= vocab ? vocab - 1 : drawn;
    embed_types(dtype, [&](auto type) {
#pragma unroll
        for (int j = 0; j < J; j++) {
            const int i = threadIdx.x + 1024 * j;
            ev[j] = embed_elem<decltype(type)::value>(raw, hidden, tok, min(i, hidden - 1));
        }
    });
    float se = 0.f, sh = 0.f;
#pragma unroll
    for (int j = 0; j < J; j++) {
        if (threadIdx.x + 1024 * j >= hidden) ev[j] = 0.f;
        se += ev[j] * ev[j];
        sh += hv[j] * hv[j];
    }
    se = block_sum(se, red[0]);
    sh = block_sum(sh, red[1]);
    const float inv_e = 1.0f / sqrtf(se / (float)hidden + eps), inv_h = 1.0f / sqrtf(sh / (float)hidden + eps);
    float st = 0.f;
#pragma unroll
    for (int j = 0; j < J; j++) {
        const int i = threadIdx.x + 1024 * j;
        hv[j] = i < hidden ? hv[j] * gt[j] * inv_h : 0.f;
        st += hv[j] * hv[j];
    }
    st = block_sum(st, red[2]);
    const float inv_t = 1.0f / sqrtf(st / (float)hidden + eps);
    float* sums = (float*)((char*)xfrag + xfrag_sum_offset(2 * hidden));
#pragma unroll
    for (int j = 0; j < J; j++) {
        const int i = threadIdx.x + 1024 * j;  // hidden is a multiple of 32: whole sub-blocks stay or leave together
        if (i >= hidden) continue;
        const _Float16 he = pinned_half((_Float16)(ev[j] * ge[j] * inv_e));
        const _Float16 hh = pinned_half((_Float16)(hv[j] * gh[j] * inv_t));
        xfrag[frag_index(i, m)] = he;
        xfrag[frag_index(hidden + i, m)] = hh;
        const float s0 = sum_of_32((float)he), s1 = sum_of_32((float)hh);
        if ((i & 31) == 0) {
            sums[xsum_index(i >> 5, m)] = s0;
            sums[xsum_index((hidden + i) >> 5, m)] = s1;
        }
        x_zero[(long)m * hidden + i] = 0.f;
    }
    if ((int)threadIdx.x < half) {  // (64 pairs at most)
        float sn, c;
        sincosf((float)rot * freq, &sn, &c);
        cs[m * half + threadIdx.x] = float2{c * mscale, sn * mscale};
    }
}

int launch_mtp_input(hipStream_t s, const uint8_t* raw, int dtype, const VerifyParams* vp, const int32_t* token_dev, int vocab,
                     const float* h_rows, const float* w_e, const float* w_t, const float* w_h, float eps, int hidden, uint4* xfrag,
                     float* x_zero, const float* freqs, float mscale, int half, float2* cs, int m) {
    if (hidden > 8192 || hidden % 32) {
        set_error("drafter head: hidden must be a multiple of 32, at most 8192");
        return TSV_ERR_UNSUPPORTED;
    }
    if (half > 1024) {
        set_error("drafter head: at most 1024 rotation pairs");
        return TSV_ERR_UNSUPPORTED;
    }
    const auto kernel = hidden <= 4096 ? k_mtp_input<4> : k_mtp_input<8>;
    hipLaunchKernelGGL(kernel, dim3(m), dim3(1024), 0, s, raw, dtype, vp, token_dev, vocab, h_rows, w_e, w_t, w_h, eps, hidden,
                       (_Float16*)xfrag, x_zero, freqs, mscale, half, cs);
    TSV_HIP(hipGetLastError());
    return TSV_OK;
}

__global__ void k_f32_to_xfrag(const float* __restrict__ x, int k, _Float16* __restrict__ xfrag) {
    const int m = blockIdx.y;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= k) return;  // k is a multiple of 32: whole sub-blocks leave together
    const _Float16 h = pinned_half((_Float16)x[(long)m * k + i]);
    xfrag[frag_index(i, m)] = h;
    float sum = (float)h;
    for (int o = 1; o < 32; o <<= 1) sum += __shfl_xor(sum, o);
    if ((i & 31) == 0) ((float*)((char*)xfrag + xfrag_sum_offset(k)))[xsum_index(i >> 5, m)] = sum;
}

int launch_f32_to_xfrag(hipStream_t s, const float* x, int k, uint4* xfrag, int m) {
    hipLaunchKernelGGL(k_f32_to_xfrag, dim3((k + 255) / 256, m), dim3(256), 0, s, x, k, (_Float16*)xfrag);
    TSV_HIP(hipGetLastError());
    return TSV_OK;
}

// ---------------------------------------------------------------- rope + KV store
// One wave per (row, head): sums the split-K partials of the fused q/k/v projection, applies
// the optional per-head RMSNorm (families/llama/state.rs:344-347) and the NeoX rotation
// (crates/compute/src/rope.rs:208-256: pairs (i, i + hd/2), angle = position * freq_i), then
// stores q as fp16 rows and K/V straight into the cache slot of that row
// (families/qwen/batched_layers.rs:84-113).  V is stored in 16-position blocks laid out as
// MFMA A-fragments: [hd/16][lane = (pos%16/4)*16 + d%16][pos%4].
__global__ __launch_bounds__(64) void k_rope_kv(RopeKvArgs a) {
    const int m = blockIdx.x, head = blockIdx.y;
    // a prompt pass of several 16-row blocks: block blockIdx.z has its own parameters, partial sums and q rows
    const VerifyParams* vp = a.vp + blockIdx.z;
    a.qkv += (long)blockIdx.z * a.qkv_block_stride;
    a.q16 += (long)blockIdx.z * 16 * a.nq * a.hd;
    asm volatile("" ::"s"(a.qkv), "s"(a.cs), "s"(a.bias), "s"(a.q_norm), "s"(a.k_norm), "s"(a.q16), "s"(a.kc), "s"(a.vc), "s"(a.vp), "s"(a.splits), "s"(a.ldq),
                 "s"(a.eps), "s"(a.nq), "s"(a.nkv), "s"(a.hd), "s"(a.max_ctx), "s"(a.paired), "s"(a.blocks), "s"(a.qkv_block_stride));
    // (how many rows the pass has and where they go: waited for at the end)
    const int rows = uniform_memory(vp)->m, base = uniform_memory(vp)->base;
    const int hd = a.hd, half = hd >> 1, i = threadIdx.x;
    const int kind = head < a.nq ? 0 : head < a.nq + a.nkv ? 1 : 2;
    const int h = kind == 0 ? head : kind == 1 ? head - a.nq : head - a.nq - a.nkv;
    const int col = head * hd;  // q heads, then k heads, then v heads: the fused projection's row order
    float x0 = 0.f, x1 = 0.f;
    // where dims i and i + half sit among the head's columns: side by side in the natural order, or -- q and k rows
    // tiled for the rotating epilogue (128-wide heads) -- dims 32 t .. 32 t + 31 in the low half of 64-row tile t and
    // their partners in its high half
    const bool paired = a.paired && kind != 2;
    const int c0 = paired ? (i >> 5) * 64 + (i & 31) : i, c1 = paired ? c0 + 32 : i + half;
    // (the head's norm weights and the pair's rotation are asked for with the partial sums)
    const float* nw = kind == 0 ? a.q_norm : kind == 1 ? a.k_norm : nullptr;
    float nw0 = 0.f, nw1 = 0.f;
    const float2 cs = a.cs[((long)blockIdx.z * 16 + m) * half + min(i, half - 1)];
    if (nw) {
        nw0 = nw[min(i, half - 1)];
        nw1 = nw[min(i, half - 1) + half];
    }
    if (i < half) {
        // compile-time split count (a uniform branch picks the variant): every partial is in flight
        // before the first add
        auto sum_splits = [&](auto S) {
            constexpr int NS = decltype(S)::value;
            float p0[NS], p1[NS];
#pragma unroll
            for (int s = 0; s < NS; s++) {
                const float* p = a.qkv + ((long)s * 16 + m) * a.ldq + col;
                p0[s] = p[c0];
                p1[s] = p[c1];
            }
#pragma unroll
            for (int s = 0; s < NS; s++) {
                x0 += p0[s];
                x1 += p1[s];
            }
        };
        switch (a.splits) {
            case 1: sum_splits(std::integral_constant<int, 1>{}); break;
            case 2: sum_splits(std::integral_constant<int, 2>{}); break;
            case 3: sum_splits(std::integral_constant<int, 3>{}); break;
            case 4: sum_splits(std::integral_constant<int, 4>{}); break;
            case 5: sum_splits(std::integral_constant<int, 5>{}); break;
            case 6: sum_splits(std::integral_constant<int, 6>{}); break;
            case 7: sum_splits(std::integral_constant<int, 7>{}); break;
            default: sum_splits(std::integral_constant<int, 8>{}); break;
        }
        if (a.bias) {  // before the rotation (families/gptoss/attn.rs:88-101)
            x0 += a.bias[col + i];
            x1 += a.bias[col + i + half];
        }
    }
    if (nw) {
        const float ss = sum_of_wave(i < half ? x0 * x0 + x1 * x1 : 0.f);
        const float inv = 1.0f / sqrtf(ss / (float)hd + a.eps);
        if (i < half) {
            x0 = x0 * nw0 * inv;
            x1 = x1 * nw1 * inv;
        }
    }
    if (i >= half || m >= rows) return;
    if (kind != 2) {
        const float r0 = x0 * cs.x - x1 * cs.y;
        const float r1 = x0 * cs.y + x1 * cs.x;
        x0 = r0;
        x1 = r1;
    }
    const _Float16 h0 = (_Float16)x0, h1 = (_Float16)x1;
    if (kind == 0) {
        _Float16* q = (_Float16*)a.q16 + ((long)m * a.nq + h) * hd;
        q[i] = h0;
        q[i + half] = h1;
    } else {
        const int pos = (base + m) % a.max_ctx;  // the cache slot of row m (a ring layer wraps at its capacity)
        if (kind == 1) {
            ((_Float16*)a.kc)[kcache_index(h, pos, i, hd, a.max_ctx)] = h0;
            ((_Float16*)a.kc)[kcache_index(h, pos, i + half, hd, a.max_ctx)] = h1;
        } else {
            ((_Float16*)a.vc)[vcache_index(h, pos, i, hd, a.max_ctx)] = h0;
            ((_Float16*)a.vc)[vcache_index(h, pos, i + half, hd, a.max_ctx)] = h1;
        }
    }
}

int launch_rope_kv(hipStream_t s, const RopeKvArgs& a, int m) {
    if (a.splits < 1 || a.splits > 8) {
        set_error("rope: one to eight partial sums");
        return TSV_ERR_UNSUPPORTED;
    }
    hipLaunchKernelGGL(k_rope_kv, dim3(m, a.nq + 2 * a.nkv, std::max(1, a.blocks)), dim3(64), 0, s, a);
    TSV_HIP(hipGetLastError());
    return TSV_OK;
}

// ---------------------------------------------------------------- KV row gather / read

// Tree compaction (families/qwen/dflash_tree.rs:106-207): rows of slots path[0..n) move to
// base..base+n.  path is strictly increasing with path[i] >= i, so walking i upward never
// overwrites a row that is still to be read.  One workgroup per (kv head, layer), sequential over i:
// every layer's cache in one launch.
__global__ void k_kv_gather(uint16_t* const* caches, const int32_t* caps, int hd, const int32_t* path, int n, int base) {
    // grid (kv heads, layers): caches[2 * layer] is the layer's K buffer, [2 * layer + 1] its V buffer,
    // caps[layer] the positions it holds (a ring layer wraps there)
    uint16_t* kc = caches[2 * blockIdx.y];
    uint16_t* vc = caches[2 * blockIdx.y + 1];
    const int max_ctx = caps[blockIdx.y];
    if (max_ctx == 0) return;  // a layer without fp16 rows (quantized KV)
    const int h = blockIdx.x, d = threadIdx.x;
    for (int i = 0; i < n; i++) {
        const int src = (base + path[i]) % max_ctx, dst = (base + i) % max_ctx;
        if (src == dst) continue;
        if (d < hd) {
            kc[kcache_index(h, dst, d, hd, max_ctx)] = kc[kcache_index(h, src, d, hd, max_ctx)];
            vc[vcache_index(h, dst, d, hd, max_ctx)] = vc[vcache_index(h, src, d, hd, max_ctx)];
        }
    }
}

int launch_kv_gather(hipStream_t s, uint16_t* const* caches_dev, const int32_t* caps_dev, int n_layers, int nkv, int hd,
                     const int32_t* path_dev, int n, int base) {
    hipLaunchKernelGGL(k_kv_gather, dim3(nkv, n_layers), dim3(128), 0, s, caches_dev, caps_dev, hd, path_dev, n, base);
    TSV_HIP(hipGetLastError());
    return TSV_OK;
}

__global__ void k_kv_read(const uint16_t* kc, const uint16_t* vc, int nkv, int hd, int max_ctx, int pos0,
                          uint16_t* k_out, uint16_t* v_out) {
    const int p = blockIdx.x, h = blockIdx.y, d = threadIdx.x;
    if (d >= hd) return;
    const long o = ((long)p * nkv + h) * hd + d;
    const int pos = (pos0 + p) % max_ctx;
    k_out[o] = kc[kcache_index(h, pos, d, hd, max_ctx)];
    v_out[o] = vc[vcache_index(h, pos, d, hd, max_ctx)];
}

__global__ void k_kv_fill(uint16_t* kc, uint16_t* vc, int nkv, int hd, int max_ctx, int pos0,
                          const uint16_t* k_in, const uint16_t* v_in) {
    const int p = blockIdx.x, h = blockIdx.y, d = threadIdx.x;
    if (d >= hd) return;
    const long o = ((long)p * nkv + h) * hd + d;
    const int pos = (pos0 + p) % max_ctx;
    kc[kcache_index(h, pos, d, hd, max_ctx)] = k_in[o];
    vc[vcache_index(h, pos, d, hd, max_ctx)] = v_in[o];
}

int launch_kv_fill(hipStream_t s, uint16_t* kc, uint16_t* vc, int nkv, int hd, int max_ctx, int pos0, int n,
                   const uint16_t* k_in, const uint16_t* v_in) {
    hipLaunchKernelGGL(k_kv_fill, dim3(n, nkv), dim3(128), 0, s, kc, vc, nkv, hd, max_ctx, pos0, k_in, v_in);
    TSV_HIP(hipGetLastError());
    return TSV_OK;
}

int launch_kv_read(hipStream_t s, const uint16_t* kc, const uint16_t* vc, int nkv, int hd, int max_ctx,
                   int pos0, int n, uint16_t* k_out, uint16_t* v_out) {
    hipLaunchKernelGGL(k_kv_read, dim3(n, nkv), dim3(128), 0, s, kc, vc, nkv, hd, max_ctx, pos0, k_out, v_out);
    TSV_HIP(hipGetLastError());
    return TSV_OK;
}

}  // namespace tsv
