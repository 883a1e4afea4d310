// What a prompt pass does between its matmuls, over all of its rows at once: embedding, residual add + RMSNorm, rotation and
// cache stores, attention (crates/runtime/src/families/llama/{prefill,attn}.rs).  The verify passes' kernels (misc.hip,
// attn.hip) take sixteen rows and read tree shapes from device memory; here rows are consecutive positions, so a row's number
// says everything about it.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "attn_tq_core.h"
#include "embed_row.h"
#include "prompt.h"
#include "prompt_place.h"
#include "tq_row.h"

namespace tsv {

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef float float16v __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float float2v __attribute__((ext_vector_type(2)));

// ---- embedding --------------------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_prompt_embed(const uint8_t* __restrict__ raw, int dtype, int hidden, float* __restrict__ x,
                                                      const int32_t* __restrict__ ids, int base, const float* __restrict__ freqs, float mscale,
                                                      int half, float2* __restrict__ cs) {
    const int row = blockIdx.x;
    const long tok = ids[row];
    // (four values to a thread, in flight together)
    embed_types(dtype, [&](auto type) {
        float v[4];
        const int e0 = blockIdx.y * 1024 + threadIdx.x;
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] = embed_elem<decltype(type)::value>(raw, hidden, tok, min(e0 + 256 * j, hidden - 1));
#pragma unroll
        for (int j = 0; j < 4; j++)
            if (e0 + 256 * j < hidden) x[(size_t)row * hidden + e0 + 256 * j] = v[j];
    });
    if (blockIdx.y) return;
    const float pos = (float)(base + row);
    for (int i = threadIdx.x; i < half; i += 256) {
        float sn, c;
        sincosf(pos * freqs[i], &sn, &c);
        cs[(size_t)row * half + i] = float2{c * mscale, sn * mscale};
    }
}

// ---- a drafter head's input ----------------------------------------------------------------------------------------------------
template <int WAVES>
__device__ __forceinline__ float sum_of_waves(float v, float* red) {
    v = sum_of_wave(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    v = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; w++) v += red[w];
    __syncthreads();
    return v;
}

// Eight values (consecutive K) of a row as activations, and the sum of its 32-value sub-block, whose other values sit in the
// three neighbouring lanes.  The halves are pinned in registers between the store and the sum: the sum has to be that of the
// stored bits (pinned_half).
__device__ __forceinline__ void put_activations(uint8_t* a, uint8_t* asum, int row, int k, int k16, const float (&v)[8], bool live,
                                                uint16_t* rows16 = nullptr) {
    half8 h = {(_Float16)v[0], (_Float16)v[2], (_Float16)v[1], (_Float16)v[3], (_Float16)v[4], (_Float16)v[6], (_Float16)v[5], (_Float16)v[7]};
    u32x4 b = __builtin_bit_cast(u32x4, h);
    asm volatile("" : "+v"(b.x), "+v"(b.y), "+v"(b.z), "+v"(b.w));
    if (live) *(u32x4*)(a + (((size_t)(row >> 5) * k16 + (k >> 4)) * 64 + ((k >> 3) & 1) * 32 + (row & 31)) * 16) = b;
    if (live && rows16) *(u32x4*)(rows16 + (size_t)row * (k16 * 16) + k) = b;
    if (asum) {
        h = __builtin_bit_cast(half8, b);
        float s = (((float)h[0] + (float)h[1]) + ((float)h[2] + (float)h[3])) + (((float)h[4] + (float)h[5]) + ((float)h[6] + (float)h[7]));
        s += lane_xor<1>(s);
        s += lane_xor<2>(s);
        if (live && (k & 31) == 0) {
            s *= PROMPT_SUM_SCALE;
            const _Float16 hi = (_Float16)s, lo = (_Float16)((s - (float)hi) * PROMPT_SUM_LEFT);
            _Float16* o = (_Float16*)(asum + ((size_t)(row >> 5) * (k16 >> 4) + (k >> 8)) * 1024) + (row & 31) * 8 + ((k >> 5) & 7);
            o[0] = hi;
            o[256] = lo;
        }
    }
}

// One workgroup per row.  The table's row is decoded value by value side by side (its bytes are) and passes through LDS to the
// lanes, which hold eight consecutive values of it and of the state, NV times.  400 rows of 4096 take 26 us, most of it the decoding's
// round trips; sixteen rows at a time (k_mtp_input) took 25 x 14.
template <int NV>
__global__ __launch_bounds__(512) void k_prompt_mtp_input(PromptMtpArgs p) {
    __shared__ float red[8];
    __shared__ __attribute__((aligned(16))) float emb[NV * 4096];
    const int row = blockIdx.x;
    const long tok = p.ids[row];
    float* const xr = p.x + (size_t)row * p.hidden;
    float hv[NV][8], ev[NV][8], se = 0.f, sh = 0.f;
    auto for_each = [&](auto f) {
#pragma unroll
        for (int i = 0; i < NV; i++) {
            const int k = i * 4096 + threadIdx.x * 8;
            f(i, k, k < p.hidden);
        }
    };
    for_each([&](int i, int k, bool live) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const float4 t = live ? *(const float4*)(xr + k + 4 * h) : float4{0.f, 0.f, 0.f, 0.f};
            hv[i][4 * h] = t.x, hv[i][4 * h + 1] = t.y, hv[i][4 * h + 2] = t.z, hv[i][4 * h + 3] = t.w;
        }
    });
    embed_types(p.dtype, [&](auto type) {
#pragma unroll
        for (int j0 = 0; j0 < NV * 8; j0 += 8) {
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; j++) v[j] = embed_elem<decltype(type)::value>(p.raw, p.hidden, tok, min((j0 + j) * 512 + (int)threadIdx.x, p.hidden - 1));
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const int e = (j0 + j) * 512 + threadIdx.x;
                emb[e] = e < p.hidden ? v[j] : 0.f;
            }
        }
    });
    const float pos = (float)(p.base + row);
    for (int i = threadIdx.x; i < p.half; i += 512) {
        float sn, c;
        sincosf(pos * p.freqs[i], &sn, &c);
        p.cs[(size_t)row * p.half + i] = float2{c * p.mscale, sn * p.mscale};
    }
    __syncthreads();
    for_each([&](int i, int k, bool) {
#pragma unroll
        for (int e = 0; e < 8; e++) {
            ev[i][e] = emb[k + e];
            se += ev[i][e] * ev[i][e];
            sh += hv[i][e] * hv[i][e];
        }
    });
    const float inv_e = 1.0f / sqrtf(sum_of_waves<8>(se, red) / (float)p.hidden + p.eps);
    const float inv_h = 1.0f / sqrtf(sum_of_waves<8>(sh, red) / (float)p.hidden + p.eps);
    float st = 0.f;
    for_each([&](int i, int k, bool live) {
#pragma unroll
        for (int e = 0; e < 8; e++) {
            hv[i][e] = live ? hv[i][e] * p.norm_t[k + e] * inv_h : 0.f;
            st += hv[i][e] * hv[i][e];
        }
    });
    const float inv_t = 1.0f / sqrtf(sum_of_waves<8>(st, red) / (float)p.hidden + p.eps);
    const int k16 = prompt_k16(2 * p.hidden);
    for_each([&](int i, int k, bool live) {
#pragma unroll
        for (int e = 0; e < 8; e++) {
            ev[i][e] = live ? ev[i][e] * p.norm_e[k + e] * inv_e : 0.f;
            hv[i][e] = live ? hv[i][e] * p.norm_h[k + e] * inv_t : 0.f;
            if (live) xr[k + e] = 0.f;
        }
        put_activations(p.a, p.asum, row, k, k16, ev[i], live);
        put_activations(p.a, p.asum, row, p.hidden + k, k16, hv[i], live);
    });
}

// The row in the registers of W waves (NV x 512 values each), 8 / W rows to a workgroup.  Bound by what one compute unit draws
// from L2 (a row is up to nine of its length: the stream and every split), so a pass has to spread over all of them: W is the
// smallest that gives every compute unit a workgroup (norm_waves).  Where rows suffice W = 1: the sixteen-byte pieces that eight
// rows' waves write side by side fill cache lines.  The partial sums are added in order, as many splits' loads in flight together as the
// registers hold, the norm's weights and the bias with them where there is room: with a loop of one split after the other, a round
// trip each, 299 rows of 4096 in eight splits took 11.8 us.
template <int NV, int W, bool ROUTED>
__global__ __launch_bounds__(512) void k_prompt_norm(PromptNormArgs p) {
    constexpr int ROOM = (ROUTED ? 8 : NV == 8 ? 16 : 12) / NV, BATCH = ROOM < 1 ? 1 : ROOM < 8 ? ROOM : 8;
    constexpr bool EARLY = NV <= 2;
    __shared__ float sums[8];
    asm volatile("" ::"s"(p.x), "s"(p.partial), "s"(p.weights), "s"(p.bias), "s"(p.w), "s"(p.a), "s"(p.asum), "s"(p.rows16), "s"(p.n), "s"(p.hidden),
                 "s"(p.splits), "s"(p.ldp), "s"(p.slots), "s"(p.eps));
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), row = blockIdx.x * (8 / W) + wave / W,
              k0 = wave % W * (NV * 512) + lane * 8;
    const bool here = row < p.n;
    if (W == 1 && !here) return;  // (with more waves to a row every wave reaches the barrier)
    float* const xr = p.x + (size_t)row * p.hidden;
    auto load8 = [&](float (&to)[8], const float* from, int i) {
        const int k = k0 + i * 512;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const float4 t = here && k < p.hidden ? *(const float4*)(from + k + 4 * h) : float4{0.f, 0.f, 0.f, 0.f};
            to[4 * h] = t.x, to[4 * h + 1] = t.y, to[4 * h + 2] = t.z, to[4 * h + 3] = t.w;
        }
    };
    float v[NV][8], g[NV][8], b[NV][8];
#pragma unroll
    for (int i = 0; i < NV; i++) load8(v[i], xr, i);
    float r[ROUTED ? NV : 1][8];
    if (ROUTED) {
#pragma unroll
        for (int i = 0; i < NV; i++)
#pragma unroll
            for (int e = 0; e < 8; e++) r[i][e] = 0.f;
    }
    auto weights = [&] {
        if (p.w) {
#pragma unroll
            for (int i = 0; i < NV; i++) load8(g[i], p.w, i);
        }
    };
    auto biases = [&] {
        if (p.bias) {
#pragma unroll
            for (int i = 0; i < NV; i++) load8(b[i], p.bias, i);
        }
    };
    if (EARLY) {
        weights();
        biases();
    }
    const float* const part = p.partial + ((size_t)(row >> 4) * p.slots * 16 + (row & 15)) * p.ldp;
    for (int s0 = 0; s0 < p.splits; s0 += BATCH) {
        float f[BATCH][NV][8], ws[BATCH];
#pragma unroll
        for (int j = 0; j < BATCH; j++)
            if (s0 + j < p.splits) {
                ws[j] = ROUTED && here ? uniform_memory(p.weights)[(size_t)row * 8 + s0 + j] : 1.0f;
#pragma unroll
                for (int i = 0; i < NV; i++) load8(f[j][i], part + (size_t)(s0 + j) * 16 * p.ldp, i);
            }
#pragma unroll
        for (int j = 0; j < BATCH; j++)
            if (s0 + j < p.splits) {
#pragma unroll
                for (int i = 0; i < NV; i++)
#pragma unroll
                    for (int e = 0; e < 8; e++) {
                        // routed experts (families/llama/moe.rs:193-198): the slots' outputs are weighted and summed in rank order
                        // from zero, then added to the stream; product and sum rounded apart
                        if (ROUTED) r[i][e] = __fadd_rn(r[i][e], __fmul_rn(ws[j], f[j][i][e]));
                        else v[i][e] = __fadd_rn(v[i][e], f[j][i][e]);
                    }
            }
    }
    if (!EARLY) biases();
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < NV; i++) {
        const int k = k0 + i * 512;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            if (ROUTED) v[i][e] = __fadd_rn(v[i][e], r[i][e]);
            if (p.bias && k < p.hidden) v[i][e] += b[i][e];
            ss += v[i][e] * v[i][e];
        }
        if (p.splits && here && k < p.hidden) {
            *(float4*)(xr + k) = float4{v[i][0], v[i][1], v[i][2], v[i][3]};
            *(float4*)(xr + k + 4) = float4{v[i][4], v[i][5], v[i][6], v[i][7]};
        }
    }
    if (!p.a) return;
    if (!EARLY) weights();
    float inv = 1.0f;
    if (p.w) {
        ss = sum_of_wave(ss);
        if (W > 1) {
            if (lane == 0) sums[wave] = ss;
            __syncthreads();
            ss = 0.f;
#pragma unroll
            for (int u = 0; u < W; u++) ss += sums[wave / W * W + u];
        }
        inv = 1.0f / sqrtf(ss / (float)p.hidden + p.eps);
    }
    const int k16 = prompt_k16(p.hidden);
#pragma unroll
    for (int i = 0; i < NV; i++) {
        const int k = k0 + i * 512;
        const bool live = here && k < p.hidden;
        float o[8];
#pragma unroll
        for (int e = 0; e < 8; e++) o[e] = p.w ? v[i][e] * g[i][e] * inv : v[i][e];
        put_activations(p.a, p.asum, row, k, k16, o, live, p.rows16);
    }
}

// The same for rows wider than a wave's registers hold: the row is read again after its sum of squares.
template <bool ROUTED>
__global__ __launch_bounds__(512) void k_prompt_norm_long(PromptNormArgs p) {
    const int lane = threadIdx.x & 63, row = blockIdx.x * 8 + (threadIdx.x >> 6);
    if (row >= p.n) return;
    float* const xr = p.x + (size_t)row * p.hidden;
    float ss = 0.f;
    for (int k = lane * 8; k < p.hidden; k += 512) {
        float v[8], r[8] = {};
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = xr[k + e];
        for (int s = 0; s < p.splits; s++) {
            const float* pr = p.partial + (((size_t)(row >> 4) * p.slots + s) * 16 + (row & 15)) * p.ldp + k;
            const float ws = ROUTED ? p.weights[(size_t)row * 8 + s] : 1.0f;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                if (ROUTED) r[e] = __fadd_rn(r[e], __fmul_rn(ws, pr[e]));
                else v[e] = __fadd_rn(v[e], pr[e]);
            }
        }
#pragma unroll
        for (int e = 0; e < 8; e++) {
            if (ROUTED) v[e] = __fadd_rn(v[e], r[e]);
            if (p.bias) v[e] += p.bias[k + e];
            ss += v[e] * v[e];
            if (p.splits) xr[k + e] = v[e];
        }
    }
    if (!p.a) return;
    ss = sum_of_wave(ss);
    const float inv = p.w ? 1.0f / sqrtf(ss / (float)p.hidden + p.eps) : 1.0f;
    const int k16 = prompt_k16(p.hidden);
    for (int k0 = 0; k0 < p.hidden; k0 += 512) {  // (whole waves: the sub-block sums cross lanes)
        const int k = k0 + lane * 8;
        const bool live = k < p.hidden;
        float o[8];
#pragma unroll
        for (int e = 0; e < 8; e++) o[e] = live ? (p.w ? xr[k + e] * p.w[k + e] * inv : xr[k + e]) : 0.f;
        put_activations(p.a, p.asum, row, k, k16, o, live, p.rows16);
    }
}

// ---- rotation + cache stores --------------------------------------------------------------------------------------------------
// One workgroup per (block of sixteen cache positions, head): a K or V block of the head is one contiguous run of the cache
// (kcache_index / vcache_index), put together in LDS and written sixteen bytes at a time.  Element by element from one wave per
// (row, head), as the verify passes do it, a pass of 2048 rows is 98 000 waves of two-byte stores.
// TQ: the layer keeps quantized rows (kvquant.hip, whose arithmetic this is on sixteen rows at once).  q is rotated with the key signs;
// a K or V row's norm and indices go straight to the stores, from the fp16 values that an fp16 cache would hold.  A block of the
// stores belongs to one workgroup, so the V groups' words, which hold a position's index beside fifteen others', need no atomics.
// Quantizing, the levels below and the norms in the attention add 53 us to a layer of 2048 rows (8B shape: 9274 us for eight layers, seven
// of them quantized, 8909 with fp16 rows); in the 64-row passes that such a prompt took before, each with a quantizer launch and an
// attention of its own, the eight layers were 36 560 us, 300 rows 6290 (now 2285).
template <int HD, bool TQ>
__global__ __launch_bounds__(256) void k_prompt_rope(PromptRopeArgs p) {
    constexpr int HALF = HD / 2, LANES = HALF, RPI = 256 / LANES;  // rows per iteration
    __shared__ __attribute__((aligned(16))) _Float16 sh[16][HD + 8];
    const int head = blockIdx.y, pb = (p.base >> 4) + blockIdx.x;
    const int kind = head < p.nq ? 0 : head < p.nq + p.nkv ? 1 : 2;
    const int h = kind == 0 ? head : kind == 1 ? head - p.nq : head - p.nq - p.nkv;
    const int i = threadIdx.x % LANES, col = head * HD;
    const bool paired = p.paired && kind != 2;
    const int c0 = paired ? (i >> 5) * 64 + (i & 31) : i, c1 = paired ? c0 + 32 : i + HALF;
    // Everything the rows need is asked for before the first addition, two splits at a time (a split after the other, and a row's rotation behind
    // its sums, were sixteen round trips for 16.6 us at 1000 rows of four splits).  Rows that the pass does not have stand in for one another.
    constexpr int ITS = 16 / RPI, BATCH = 2;
    const int turn = HD == 128 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : threadIdx.x / LANES;  // (whole waves share a row: scalar addresses)
    const float b0 = p.bias ? p.bias[col + i] : 0.f, b1 = p.bias ? p.bias[col + i + HALF] : 0.f;
    const float* nw = kind == 0 ? p.q_norm : kind == 1 ? p.k_norm : nullptr;
    const float nw0 = nw ? nw[i] : 0.f, nw1 = nw ? nw[i + HALF] : 0.f;
    const int row0 = pb * 16 + turn - p.base;
    float2 cs[ITS];
    float x0[ITS], x1[ITS];
    const float* q[ITS];
#pragma unroll
    for (int it = 0; it < ITS; it++) {
        const int row = min(max(row0 + it * RPI, 0), p.n - 1);
        if (kind != 2) cs[it] = *(const float2*)((const char*)(p.cs + (size_t)row * HALF) + (uint32_t)(i * 8));
        q[it] = p.qkv + ((size_t)(row >> 4) * p.splits * 16 + (row & 15)) * p.ldq + col;
        x0[it] = x1[it] = 0.f;
    }
    for (int s0 = 0; s0 < p.splits; s0 += BATCH) {
        float y0[BATCH][ITS], y1[BATCH][ITS];
#pragma unroll
        for (int j = 0; j < BATCH; j++)
            if (s0 + j < p.splits) {
#pragma unroll
                for (int it = 0; it < ITS; it++) {
                    const char* const at = (const char*)(q[it] + (size_t)(s0 + j) * 16 * p.ldq);
                    y0[j][it] = *(const float*)(at + (uint32_t)(c0 * 4));
                    y1[j][it] = *(const float*)(at + (uint32_t)(c1 * 4));
                }
            }
#pragma unroll
        for (int j = 0; j < BATCH; j++)
            if (s0 + j < p.splits) {
#pragma unroll
                for (int it = 0; it < ITS; it++) {
                    x0[it] += y0[j][it];
                    x1[it] += y1[j][it];
                }
            }
    }
#pragma unroll
    for (int it = 0; it < ITS; it++) {
        const int slot = it * RPI + turn, row = row0 + it * RPI;
        const bool live = row >= 0 && row < p.n;
        float a0 = live ? x0[it] : 0.f, a1 = live ? x1[it] : 0.f;
        if (p.bias && live) {  // before the rotation (families/gptoss/attn.rs:88-101)
            a0 += b0;
            a1 += b1;
        }
        if (nw) {  // RMSNorm over the head (families/llama/state.rs:344-347)
            const float ss = HD == 128 ? sum_of_wave(a0 * a0 + a1 * a1) : sum_of_32_down(a0 * a0 + a1 * a1);
            const float inv = 1.0f / sqrtf(ss / (float)HD + p.eps);
            a0 = a0 * nw0 * inv;
            a1 = a1 * nw1 * inv;
        }
        if (kind != 2 && live) {  // NeoX pairs (i, i + hd / 2) (crates/compute/src/rope.rs:208-256)
            const float r0 = a0 * cs[it].x - a1 * cs[it].y, r1 = a0 * cs[it].y + a1 * cs[it].x;
            a0 = r0;
            a1 = r1;
        }
        sh[slot][i] = (_Float16)a0;
        sh[slot][i + HALF] = (_Float16)a1;
    }
    __syncthreads();
    const int t = threadIdx.x;
    if (TQ) {
        constexpr int EPL = HD / 64;
        __shared__ float norm[16];
        __shared__ uint8_t code[16][HD];
        const int lane = t & 63, wave = t >> 6;
        const TqSide& side = kind == 2 ? p.tq_v : p.tq_k;
        if (kind != 0) {
            if (t < 16) {  // the squares in index order (the reference's sum), a row to a lane
                float ss = 0.f;
#pragma unroll
                for (int i = 0; i < HD; i += 8) {
                    const half8 r = *(const half8*)&sh[t][i];
#pragma unroll
                    for (int e = 0; e < 8; e++) ss = __fadd_rn(ss, __fmul_rn((float)r[e], (float)r[e]));
                }
                norm[t] = sqrtf(ss);
            }
            __syncthreads();
        }
        const TqMidpoints mid(side);
        for (int slot = 4 * wave; slot < 4 * wave + 4; slot++) {
            const float inv = kind != 0 ? 1.0f / fmaxf(norm[slot], 1e-6f) : 1.0f;  // (times one: the same bits)
            float e[EPL];
#pragma unroll
            for (int j = 0; j < EPL; j++) e[j] = __fmul_rn(__fmul_rn((float)sh[slot][lane + 64 * j], inv), side.signs[lane + 64 * j]);
            wht<EPL>(e, lane, p.inv_sqrt2);
#pragma unroll
            for (int j = 0; j < EPL; j++) {
                if (kind == 0) sh[slot][lane + 64 * j] = (_Float16)e[j];
                else code[slot][lane + 64 * j] = (uint8_t)mid.index(e[j]);
            }
        }
        __syncthreads();
        if (kind != 0) {
            const int r0 = pb * 16 - p.base, lo = max(0, -r0), hi = min(16, p.n - r0);  // the pass's slots of the block
            if (t >= lo && t < hi) (kind == 2 ? p.store.vn : p.store.kn)[(long)h * p.cap + pb * 16 + t] = norm[t];
            const int bits = side.bits;
            if (kind == 1) {  // a row's indices LSB first (kv_quant.rs:289-312), a word to a thread
                const int words = side.words;
                for (int id = t; id < 16 * words; id += 256) {
                    const int slot = id / words, w = id - slot * words;
                    uint32_t v = 0;
                    for (int d = 32 * w / bits; d < HD && d * bits < 32 * w + 32; d++) {
                        const int at = d * bits - 32 * w;
                        v |= at >= 0 ? (uint32_t)code[slot][d] << at : (uint32_t)code[slot][d] >> -at;
                    }
                    if (slot >= lo && slot < hi) p.store.kq[((long)h * p.cap + pb * 16 + slot) * words + w] = v;
                }
            } else if (t < HD) {  // a dimension's indices of the block's positions, a group to a thread
                const int gw = tq_v_group_words(bits);
                uint32_t* g = p.store.vq + (((long)h * (p.cap >> 4) + pb) * HD + t) * gw;
                uint64_t v = 0, mask = 0;
#pragma unroll
                for (int slot = 0; slot < 16; slot++)
                    if (slot >= lo && slot < hi) {
                        v |= (uint64_t)code[slot][t] << (slot * bits);
                        mask |= (uint64_t)((1u << bits) - 1u) << (slot * bits);
                    }
                if (lo != 0 || hi != 16) v |= (gw == 2 ? ((uint64_t)g[1] << 32) | g[0] : (uint64_t)g[0]) & ~mask;
                g[0] = (uint32_t)v;
                if (gw == 2) g[1] = (uint32_t)(v >> 32);
            }
            return;
        }
    }
    if (t >= 16 * HD / 8) return;
    if (kind == 0) {
        const int slot = t / (HD / 8), d = t % (HD / 8) * 8, row = pb * 16 + slot - p.base;
        if (row >= 0 && row < p.n) *(u32x4*)((_Float16*)p.q16 + ((size_t)row * p.nq + h) * HD + d) = *(const u32x4*)&sh[slot][d];
        return;
    }
    const long blk = ((long)h * (p.cap >> 4) + pb % (p.cap >> 4)) * (16 * HD);
    if (kind == 1) {  // piece t: dims 32 (t / 64) + 8 (t % 64 / 16) .. of position t % 16
        const int slot = t & 15, d = (t >> 6) * 32 + ((t >> 4) & 3) * 8, row = pb * 16 + slot - p.base;
        if (row >= 0 && row < p.n) *(u32x4*)((_Float16*)p.kc + blk + t * 8) = *(const u32x4*)&sh[slot][d];
        return;
    }
    // piece t: positions 4 q .. 4 q + 3 (q = t % 64 / 16) of dims d and d + 16, d = 32 (t / 64) + t % 16
    const int q4 = ((t >> 4) & 3) * 4, d = (t >> 6) * 32 + (t & 15), row = pb * 16 + q4 - p.base;
    _Float16* o = (_Float16*)p.vc + blk + t * 8;
    half8 v;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        v[e] = sh[q4 + e][d];
        v[4 + e] = sh[q4 + e][d + 16];
    }
    if (row >= 0 && row + 3 < p.n) {
        *(half8*)o = v;
    } else {
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (row + e >= 0 && row + e < p.n) {
                o[e] = v[e];
                o[4 + e] = v[4 + e];
            }
    }
}

// ---- quantized rows as attention operands -----------------------------------------------------------------------------------------
// The codebook levels of positions [0, 16 gridDim.x * DECODE) as fp16 in the layout of an fp16 cache, for the attention kernel below; the
// norms stay where they are, f32.  A layer's 4096 positions of the 8B shape are 4.5 MB of codes and 16.8 MB of levels, and every wave of
// the pass reads them instead of unpacking them: 64 waves a KV head at 512 rows.
constexpr int DECODE = 4;
template <int HD>
__global__ __launch_bounds__(256) void k_prompt_tq_levels(TqKv q, int blocks, int cap, uint16_t* __restrict__ kc, uint16_t* __restrict__ vc) {
    __shared__ uint32_t kpair[256], vpair[256];
    const int t = threadIdx.x, h = blockIdx.y, kb = q.k_bits, vb = q.v_bits, kw = HD * kb / 32, gw = tq_v_group_words(vb);
    tq_fill_pairs(kpair, q.k_cb, kb, t, 256);
    tq_fill_pairs(vpair, q.v_cb, vb, t, 256);
    __syncthreads();
    if (t >= 2 * HD) return;
    const uint32_t km = (1u << (2 * kb)) - 1u, vm = (1u << (2 * vb)) - 1u;
    for (int b = blockIdx.x * DECODE; b < min(blocks, (int)(blockIdx.x + 1) * DECODE); b++) {
        const size_t blk = ((size_t)h * (cap >> 4) + b) * (16 * HD) + t * 8;
        {  // piece t of K: eight dims of one position
            const int d = (t >> 6) * 32 + ((t >> 4) & 3) * 8, bit = d * kb, w = bit >> 5;
            const uint32_t* row = q.kq + ((size_t)h * cap + b * 16 + (t & 15)) * kw;
            const uint32_t f = (uint32_t)((((uint64_t)row[min(w + 1, kw - 1)] << 32) | row[w]) >> (bit & 31));
            *(u32x4*)(kc + blk) = u32x4{kpair[f & km], kpair[(f >> (2 * kb)) & km], kpair[(f >> (4 * kb)) & km], kpair[(f >> (6 * kb)) & km]};
        }
        u32x4 o;  // piece t of V: four positions of two dims
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const uint32_t* g = q.vq + (((size_t)h * (cap >> 4) + b) * HD + (t >> 6) * 32 + (t & 15) + 16 * e) * gw;
            const uint32_t f = (uint32_t)((((uint64_t)(gw == 2 ? g[1] : 0u) << 32) | g[0]) >> (((t >> 4) & 3) * 4 * vb));
            o[2 * e] = vpair[f & vm];
            o[2 * e + 1] = vpair[(f >> (2 * vb)) & vm];
        }
        *(u32x4*)(vc + blk) = o;
    }
}

// ---- attention ------------------------------------------------------------------------------------------------------------------
// A wave holds 32 (row, q head of the group) pairs as the columns of v_mfma_f32_32x32x16_f16 and walks the cache 32 positions at
// a time: S^T = K Q^T, weights, O^T += V^T P^T.  A lane's sixteen scores are of ONE pair, so the softmax crosses lanes once
// (lane ^ 32), and they come out as the B operand of the second product in an order of positions that V is simply read in; K and
// V are operands as the cache keeps them.  The four waves of a workgroup (128 pairs) walk the same blocks, so the L1 serves all
// but the first.  2048 rows of the 8B shape: 107 us a layer (rotation and cache stores 16 us), where the verify passes' kernels,
// 64 rows at a time, took 32 x (9.7 + 4.8 merge) us (and 32 x 4.8).
// The weights go in as two fp16 terms, 21 bits.  With one term a weight is exact only where it is its wave's largest, and here a
// wave keeps one reference for all of a row's positions, where the verify passes' kernel has one for every few blocks: 1504 rows,
// scores of 2.5 standard deviations, came out 2.72e-4 of the exact result's norm off (2.11e-4 there), now 2.066e-4, all of it the
// rounding of the fp16 output.  The second product costs 0.25 of 36.3 ms in a 2048-row pass of 32 layers.
// Rows see [0, position] (window: the last `window` positions); only blocks that straddle an edge look.
__device__ __forceinline__ float other_half_max(float v) {
    float w = v;
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\tv_max_f32 %0, %0, %1" : "+v"(v), "+v"(w));
    return v;
}
// w minus half HALF of h, exact (one instruction: the conversion rides on the fused add)
template <int HALF>
__device__ __forceinline__ float left_over(float w, uint32_t h) {
    float r;
    if (HALF == 0) asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h), "v"(w));
    else asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h), "v"(w));
    return r;
}
constexpr float LOG2E = 1.44269504088896340736f, REF_SLACK = 8.0f;

// TQ: the rows are codebook levels (k_prompt_tq_levels) and an f32 norm a position and side, q is rotated (attn_tq_core.h): a key's norm
// multiplies its score, a value's the weight before it is cut into two fp16 terms (with no slack in the reference: a weight is at
// most 1, so that a norm up to fp16's largest value passes), and the sum is rotated back in registers: six of the seven stages at
// 128 dims pair values of one lane.
template <int HD, bool PART, bool TQ>
__global__ __launch_bounds__(256, 2) void k_prompt_attn(PromptAttnArgs p) {
    constexpr int KS = HD / 16, VT = HD / 32;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int G = p.nq / p.nkv, cols = p.n * G;
    const PromptAttnPlace place = prompt_attn_place(blockIdx.x, gridDim.x, p.nkv, !PART);
    const int kvh = place.head, c_first = (place.group * 4 + wave) * 32;
    if (c_first >= cols) return;
    const int hl = lane >> 5, c = min(c_first + (lane & 31), cols - 1), row = c / G, hq = kvh * G + (c - row * G);
    const int row_lo = c_first / G, row_hi = min(c_first + 31, cols - 1) / G;
    const int pos = p.base + row;
    int b0 = p.window > 0 ? max(p.base + row_lo + 1 - p.window, 0) >> 5 : 0, b1 = (p.base + row_hi) / 32 + 1;
    if (PART) {
        const int per = (b1 - b0 + p.nch - 1) / p.nch;
        b0 += blockIdx.z * per;
        b1 = min(b1, b0 + per);
    }
    const _Float16* qp = (const _Float16*)p.q16 + ((size_t)row * p.nq + hq) * HD + 8 * hl;
    u32x4 q[KS];
#pragma unroll
    for (int t = 0; t < KS; t++) q[t] = *(const u32x4*)(qp + 16 * t);
    const uint32_t head_bytes = (uint32_t)p.cap * HD * 2;  // (bounds the reads: blocks past the cache come back as zeros)
    const __amdgpu_buffer_rsrc_t krs = __builtin_amdgcn_make_buffer_rsrc((void*)((const uint8_t*)p.kc + (size_t)kvh * head_bytes), 0, head_bytes, 0x00027000);
    const __amdgpu_buffer_rsrc_t vrs = __builtin_amdgcn_make_buffer_rsrc((void*)((const uint8_t*)p.vc + (size_t)kvh * head_bytes), 0, head_bytes, 0x00027000);
    const uint32_t koff = ((lane >> 4) & 1) * (HD * 32) + hl * 256 + (lane & 15) * 16;
    const uint32_t voff = hl * 256 + (lane & 15) * 16 + ((lane >> 4) & 1) * 8;
    float16v O[VT];
#pragma unroll
    for (int u = 0; u < VT; u++)
#pragma unroll
        for (int i = 0; i < 16; i++) O[u][i] = 0.f;
    float mrun = -INFINITY, lrun = 0.f;
    const float c2 = p.scale * LOG2E;
    const __amdgpu_buffer_rsrc_t knrs = __builtin_amdgcn_make_buffer_rsrc((void*)(p.kn + (size_t)(TQ ? kvh : 0) * p.cap), 0, TQ ? (p.base + p.n) * 4 : 0, 0x00027000);
    const __amdgpu_buffer_rsrc_t vnrs = __builtin_amdgcn_make_buffer_rsrc((void*)(p.vn + (size_t)(TQ ? kvh : 0) * p.cap), 0, TQ ? (p.base + p.n) * 4 : 0, 0x00027000);
    u32x4 kf[KS];
    // a block's norms: a lane asks for one position's, with its K, and the wave passes them round through 256 bytes of LDS (sixteen
    // registers a side for each lane's own would be 33 more than there are at 128 dims)
    __shared__ __attribute__((aligned(16))) float norms[TQ ? 4 : 1][64];
    float kn = 0.f, vn = 0.f;
    auto order = [] {  // one wave writes and reads its own LDS: program order is enough, and the compiler is kept to it
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    auto load_k = [&](int b) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < KS; t++)
            kf[t] = __builtin_amdgcn_raw_buffer_load_b128(krs, koff + (uint32_t)b * (HD * 64) + (t >> 1) * 1024 + (t & 1) * 512, 0, 0);
        if (TQ) {
            kn = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(knrs, (uint32_t)b * 128 + 4 * (lane & 31), 0, 0));
            vn = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(vnrs, (uint32_t)b * 128 + 4 * (lane & 31), 0, 0));
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // (a block's V is asked for before its scores are made, the next block's K right after: both have the softmax and a product
    // to arrive in, and one set of registers each)
    auto step = [&](int b) {
        u32x2 vf[2][VT][2];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int u = 0; u < VT; u++)
#pragma unroll
                for (int x = 0; x < 2; x++)
                    vf[t][u][x] = __builtin_amdgcn_raw_buffer_load_b64(vrs, voff + (uint32_t)(2 * b + t) * (HD * 32) + u * 1024 + x * 512, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        float16v S;
#pragma unroll
        for (int i = 0; i < 16; i++) S[i] = 0.f;
#pragma unroll
        for (int t = 0; t < KS; t++)
            S = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, kf[t]), __builtin_bit_cast(half8, q[t]), S, 0, 0, 0);
        if (TQ) {
            norms[TQ ? wave : 0][lane] = hl ? vn : kn;
            order();
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float4v f = *(const float4v*)&norms[TQ ? wave : 0][8 * i + 4 * hl];
#pragma unroll
                for (int e = 0; e < 4; e++) S[4 * i + e] *= f[e];
            }
        }
        load_k(min(b + 1, b1 - 1));
        // register i: position 32 b + 8 (i / 4) + 4 hl + i % 4
        const int p0 = 32 * b;
        if (p0 + 31 > p.base + row_lo || (p.window > 0 && p0 <= p.base + row_hi - p.window)) {  // (wave-uniform)
            const int lo = p.window > 0 ? pos - p.window : -1;
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int at = p0 + 8 * (i >> 2) + 4 * hl + (i & 3);
                S[i] = at <= pos && at > lo ? S[i] : -INFINITY;
            }
        }
        float mb = S[0];
#pragma unroll
        for (int i = 1; i < 16; i++) mb = fmaxf(mb, S[i]);
        mb = other_half_max(mb) * c2;
        // the reference follows the maximum lazily (attn_core.h): a weight never exceeds 2^REF_SLACK
        const bool grow = mb > mrun + (TQ ? 0.f : REF_SLACK);
        if (__builtin_amdgcn_ballot_w64(grow) != 0) {
            const float mnew = grow ? mb : mrun;
            const float alpha = __builtin_amdgcn_exp2f(mrun - fmaxf(mnew, -3.0e38f));
            lrun *= alpha;
#pragma unroll
            for (int u = 0; u < VT; u++)
#pragma unroll
                for (int i = 0; i < 16; i++) O[u][i] *= alpha;
            mrun = mnew;
        }
        const float nref = -fmaxf(mrun, -3.0e38f);
        u32x4 P[2], R[2];  // the weights as two fp16 terms
        float ps = 0.f;
#pragma unroll
        for (int i = 0; i < 16; i += 2) {
            const float2v f = TQ ? *(const float2v*)&norms[TQ ? wave : 0][TQ ? 32 + 8 * (i >> 2) + 4 * hl + (i & 3) : 0] : float2v{1.f, 1.f};
            float w0 = __builtin_amdgcn_exp2f(__builtin_fmaf(S[i], c2, nref)), w1 = __builtin_amdgcn_exp2f(__builtin_fmaf(S[i + 1], c2, nref));
            ps += w0;
            ps += w1;
            if (TQ) {  // the denominator takes the weight alone
                w0 *= f[0];
                w1 *= f[1];
            }
            const uint32_t h = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(w0, w1));
            P[i >> 3][(i & 7) >> 1] = h;
            R[i >> 3][(i & 7) >> 1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(left_over<0>(w0, h), left_over<1>(w1, h)));
        }
        lrun += ps;
        if (TQ) order();
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int u = 0; u < VT; u++) {
                const u32x4 va = {vf[t][u][0].x, vf[t][u][0].y, vf[t][u][1].x, vf[t][u][1].y};
                O[u] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, va), __builtin_bit_cast(half8, P[t]), O[u], 0, 0, 0);
                O[u] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, va), __builtin_bit_cast(half8, R[t]), O[u], 0, 0, 0);
            }
    };
    if (b0 < b1) {
        load_k(b0);
        for (int b = b0; b < b1; b++) step(b);
    }
    float l = lrun + __shfl_xor(lrun, 32);
    const bool live = c_first + (lane & 31) < cols;
    if (PART) {
        const size_t at = ((size_t)blockIdx.z * p.nkv + kvh) * cols + c;
        if (!live) return;
        if (hl == 0) {
            p.part_ml[at * 2] = mrun;
            p.part_ml[at * 2 + 1] = l;
        }
#pragma unroll
        for (int u = 0; u < VT; u++)
#pragma unroll
            for (int i = 0; i < 4; i++)
                *(float4*)(p.part_o + at * HD + 32 * u + 8 * i + 4 * hl) = float4{O[u][4 * i], O[u][4 * i + 1], O[u][4 * i + 2], O[u][4 * i + 3]};
        return;
    }
    float scale = 1.0f;
    if (p.sinks) {  // joins maximum and denominator only (crates/compute/src/attention.rs:94-105)
        const float sink = p.sinks[hq] * LOG2E, m = fmaxf(mrun, sink);
        scale = __builtin_amdgcn_exp2f(mrun - m);
        l = l * scale + __builtin_amdgcn_exp2f(sink - m);
    }
    scale /= l;
    const int k16 = prompt_k16(p.nq * HD);
    if (TQ) {  // back through the normalized Hadamard transform (crates/compute/src/wht.rs:15-29): dim 32 u + 8 (i / 4) + 4 hl + i % 4
        const float c = 0.70710678118654752440f;
#pragma unroll
        for (int st = 1; st < HD; st <<= 1) {
            const int ri = st == 1 ? 1 : st == 2 ? 2 : st == 8 ? 4 : st == 16 ? 8 : 0, ru = st >= 32 ? st / 32 : 0;
#pragma unroll
            for (int u = 0; u < VT; u++)
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    if (st == 4) {
                        const float other = __shfl_xor(O[u][i], 32);
                        O[u][i] = (hl ? other - O[u][i] : O[u][i] + other) * c;
                    } else if (!(i & ri) && !(u & ru)) {
                        const float a = O[u][i], b = O[u ^ ru][i ^ ri];
                        O[u][i] = (a + b) * c;
                        O[u ^ ru][i ^ ri] = (a - b) * c;
                    }
                }
        }
#pragma unroll
        for (int u = 0; u < VT; u++)
#pragma unroll
            for (int i = 0; i < 16; i++) O[u][i] *= p.unrot[32 * u + 8 * (i >> 2) + 4 * hl + (i & 3)];
    }
#pragma unroll
    for (int u = 0; u < VT; u++) {
        float sum = 0.f;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int k = hq * HD + 32 * u + 8 * i + 4 * hl;
            half4 o = {(_Float16)(O[u][4 * i] * scale), (_Float16)(O[u][4 * i + 2] * scale), (_Float16)(O[u][4 * i + 1] * scale),
                       (_Float16)(O[u][4 * i + 3] * scale)};
            u32x2 bits = __builtin_bit_cast(u32x2, o);
            asm volatile("" : "+v"(bits.x), "+v"(bits.y));
            o = __builtin_bit_cast(half4, bits);
            sum += ((float)o[0] + (float)o[1]) + ((float)o[2] + (float)o[3]);
            if (live) *(u32x2*)((_Float16*)p.a + prompt_a_index(row, k, k16)) = bits;
        }
        if (p.asum) {
            sum += __shfl_xor(sum, 32);
            if (live && hl == 0) {
                sum *= PROMPT_SUM_SCALE;
                const int k = hq * HD + 32 * u;
                const _Float16 hi = (_Float16)sum, lo = (_Float16)((sum - (float)hi) * PROMPT_SUM_LEFT);
                _Float16* o = (_Float16*)(p.asum + ((size_t)(row >> 5) * (k16 >> 4) + (k >> 8)) * 1024) + (row & 31) * 8 + ((k >> 5) & 7);
                o[0] = hi;
                o[256] = lo;
            }
        }
    }
}

// The chunks' partial results of one (row, q head) merged, one thread per eight dims; HD / 8 threads to a pair
// MOST: chunks there are at most (prompt_attn_chunks), or 2: just two, as passes of many rows have.  With room for sixteen those held registers that
// their many workgroups' occupancy was worth more than (1000 rows 9.6 us for 8.2, 4-bit rows 10.5 for 8.9); fewer rows have more chunks to wait for.
template <int HD, bool TQ, int MOST>
__global__ __launch_bounds__(256) void k_prompt_attn_merge(PromptAttnArgs p) {
    constexpr int TPP = HD / 8;
    constexpr int BATCH = MOST < 4 ? MOST : 4;  // of the values, in flight together
    auto have = [&](int ch) { return MOST == 2 || ch < p.nch; };
    const int G = p.group, cols = p.n * G;
    const int id = blockIdx.x * 256 + threadIdx.x, pair = id / TPP, d = id % TPP * 8;
    // consecutive threads: dims, then rows of one head, so that the pieces written side by side are neighbours
    const int turn = p.by_n.quotient(pair), row = pair - turn * p.n, hq = min(turn, p.nq - 1), kvh = p.by_group.quotient(hq);
    const bool live = pair < p.n * p.nq;
    const size_t c = (size_t)row * G + (hq - kvh * G), at0 = (size_t)kvh * cols + c, step = (size_t)p.nkv * cols;
    const float sink = p.sinks ? p.sinks[hq] * LOG2E : -INFINITY;
    // (chunk by chunk, each behind the one before, the merge of 299 rows was 8.2 us)
    float2 ml[MOST];
#pragma unroll
    for (int ch = 0; ch < MOST; ch++)
        if (have(ch)) ml[ch] = *(const float2*)(p.part_ml + (at0 + ch * step) * 2);
    float m = sink;
#pragma unroll
    for (int ch = 0; ch < MOST; ch++)
        if (have(ch)) m = fmaxf(m, ml[ch].x);
    float l = p.sinks ? __builtin_amdgcn_exp2f(sink - m) : 0.f, o[8] = {};
#pragma unroll
    for (int c0 = 0; c0 < MOST; c0 += BATCH) {
        if (!have(c0)) break;
        float4 a[BATCH], b[BATCH];
#pragma unroll
        for (int j = 0; j < BATCH; j++)
            if (have(c0 + j)) {
                a[j] = *(const float4*)(p.part_o + (at0 + (c0 + j) * step) * HD + d);
                b[j] = *(const float4*)(p.part_o + (at0 + (c0 + j) * step) * HD + d + 4);
            }
#pragma unroll
        for (int j = 0; j < BATCH; j++)
            if (have(c0 + j)) {
                const float w = __builtin_amdgcn_exp2f(ml[c0 + j].x - m);
                l = __builtin_fmaf(ml[c0 + j].y, w, l);
                const float f[8] = {a[j].x, a[j].y, a[j].z, a[j].w, b[j].x, b[j].y, b[j].z, b[j].w};
#pragma unroll
                for (int e = 0; e < 8; e++) o[e] = __builtin_fmaf(f[e], w, o[e]);
            }
    }
    const float inv = 1.0f / l;
    // (the products as floats first: converted in the instruction that makes it a value is rounded once, and which ones are would differ from variant to variant)
#pragma unroll
    for (int e = 0; e < 8; e++) {
        o[e] *= inv;
        asm volatile("" : "+v"(o[e]));
    }
    if (TQ) {  // back out of the rotated space: three stages inside a thread, the others over the TPP lanes of the pair
        const float c = 0.70710678118654752440f;
#pragma unroll
        for (int st = 1; st < 8; st <<= 1)
#pragma unroll
            for (int e = 0; e < 8; e++)
                if (!(e & st)) {
                    const float a = o[e], b = o[e ^ st];
                    o[e] = (a + b) * c;
                    o[e ^ st] = (a - b) * c;
                }
#pragma unroll
        for (int st = 1; st < TPP; st <<= 1)
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float other = st == 1 ? lane_xor<1>(o[e]) : st == 2 ? lane_xor<2>(o[e]) : st == 4 ? lane_xor<4>(o[e]) : lane_xor<8>(o[e]);
                o[e] = (threadIdx.x & st ? other - o[e] : o[e] + other) * c;
            }
#pragma unroll
        for (int e = 0; e < 8; e++) o[e] *= p.unrot[d + e];
    }
    put_activations(p.a, p.asum, row, hq * HD + d, prompt_k16(p.nq * HD), o, live);
}

// ---- routed experts: pairs sorted by expert -------------------------------------------------------------------------------
// One workgroup: counts, runs and tiles of all experts, then every pair's place.  (Where a pair lands inside its expert's run
// depends on the order of the atomics; no value does: a row of a product does not see its neighbours.)  Bound by round trips, not
// by bytes: a thread's choices are read once, all in flight, and the count's own atomic says where in the run each goes; the
// sums over the experts cross lanes, not barriers (8000 pairs of 128 experts 12.6 -> 9.7 us, 6000 10.5 -> 9.4).
constexpr int MAX_EXPERTS = 256;
constexpr int GROUP_SLOTS = PROMPT_ROWS * 8 / 1024;  // of a thread
__global__ __launch_bounds__(1024) void k_prompt_groups(const int32_t* __restrict__ selected, int n, int top_k, int ne, int bm, PromptRoutes r) {
    __shared__ int cnt[MAX_EXPERTS], first[MAX_EXPERTS], part[MAX_EXPERTS / 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int expert[GROUP_SLOTS], place[GROUP_SLOTS];
#pragma unroll
    for (int i = 0; i < GROUP_SLOTS; i++) {
        const int q = tid + i * 1024;  // row * 8 + slot
        expert[i] = q < n * 8 && (q & 7) < top_k ? min(max(selected[q], 0), ne - 1) : -1;
    }
    if (tid < MAX_EXPERTS) cnt[tid] = 0;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < GROUP_SLOTS; i++)
        if (expert[i] >= 0) place[i] = atomicAdd(&cnt[expert[i]], 1);
    __syncthreads();
    // sums over the experts: rows of the padded runs (16 bits: 8 of 2048 rows, 31 more for each of 256 experts), tiles above them
    static_assert(PROMPT_ROWS * 8 + MAX_EXPERTS * 31 < 1 << 16, "packed sums");
    uint32_t mine = 0, upto = 0;
    if (tid < MAX_EXPERTS) {
        mine = (uint32_t)(((cnt[tid] + 31) & ~31) | (cnt[tid] + bm - 1) / bm << 16);
        upto = mine;
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t below = __shfl_up(upto, o);
            if (lane >= o) upto += below;
        }
        if (lane == 63) part[wave] = (int)upto;
    }
    __syncthreads();
    uint32_t all = 0;
#pragma unroll
    for (int w = 0; w < MAX_EXPERTS / 64; w++) {
        if (w < wave) upto += (uint32_t)part[w];
        all += (uint32_t)part[w];
    }
    if (tid < ne) {
        const int at = (int)((upto - mine) & 0xFFFF), t0 = (int)((upto - mine) >> 16), tiles = (int)(mine >> 16);
        first[tid] = at;
        for (int t = 0; t < tiles; t++) r.tiles[t0 + t] = PromptTile{tid, at + t * bm, min(bm, cnt[tid] - t * bm), 0};
    }
    if (tid == 0) *r.n_tiles = (int)(all >> 16);
    for (int q = (int)(all & 0xFFFF) + tid * 32; q < prompt_sorted_rows(n, top_k, ne); q += 32 * 1024) r.pair[q] = -2;  // a block past the last run
    __syncthreads();
    const int e = tid >> 2;  // four threads fill an expert's last block
    if (e < ne)
        for (int q = cnt[e] + (tid & 3); q < ((cnt[e] + 31) & ~31); q += 4) r.pair[first[e] + q] = -1;
#pragma unroll
    for (int i = 0; i < GROUP_SLOTS; i++)
        if (expert[i] >= 0) r.pair[first[expert[i]] + place[i]] = tid + i * 1024;
}

// 32 sorted pairs to a workgroup, of a part of K: lane = pair, so the stores are whole lines of the operand layout; the
// sixteen-byte loads of a row's line come from the eight half waves side by side, four of a thread in flight.
// Bound by round trips: 374 workgroups of whole rows (8000 x 2048) took 16.0 us, in three parts of K 13.6; 312 (6000 x 2880) 21.5,
// in four 14.6.
__global__ __launch_bounds__(256) void k_prompt_gather(const uint16_t* __restrict__ rows, const uint8_t* __restrict__ row_sums, int k16,
                                                       const int32_t* __restrict__ pair, int n_sorted, uint8_t* __restrict__ a, uint8_t* __restrict__ asum) {
    const int p = blockIdx.x * 32 + (threadIdx.x & 31), half = threadIdx.x >> 5;
    // (both asked for together; what lies behind a block's -2 is not used)
    const int pr = pair[min(p, n_sorted - 1)], lead = uniform_memory(pair)[blockIdx.x * 32];
    if (lead == -2 || p >= n_sorted || pr < 0) return;
    const u32x4* src = (const u32x4*)(rows + (size_t)(pr >> 3) * (k16 * 16));
    u32x4* dst = (u32x4*)(a + (size_t)blockIdx.x * k16 * 1024) + (threadIdx.x & 31);
    const int end = 2 * k16;
    for (int k8 = blockIdx.y * 32 + half; k8 < end; k8 += gridDim.y * 32) {
        u32x4 v[4];
#pragma unroll
        for (int j = 0; j < 4; j++)
            if (k8 + 8 * j < end) v[j] = src[k8 + 8 * j];
#pragma unroll
        for (int j = 0; j < 4; j++)
            if (k8 + 8 * j < end) dst[(k8 + 8 * j) * 32] = v[j];
    }
    if (!asum) return;
    const int row = pr >> 3, kc = k16 >> 4;
    for (int c = blockIdx.y * 8 + half; c < 2 * kc; c += gridDim.y * 8)  // (both halves of the sums of every 256 K)
        *(u32x4*)(asum + ((size_t)blockIdx.x * 2 * kc + c) * 512 + (threadIdx.x & 31) * 16) =
            *(const u32x4*)(row_sums + ((size_t)(row >> 5) * 2 * kc + c) * 512 + (row & 31) * 16);
}

}  // namespace

int launch_prompt_embed(hipStream_t s, const uint8_t* raw, int dtype, int hidden, float* x, const int32_t* ids, int n, int base, const float* freqs,
                        float mscale, int half, float2* cs) {
    hipLaunchKernelGGL(k_prompt_embed, dim3(n, (hidden + 1023) / 1024), dim3(256), 0, s, raw, dtype, hidden, x, ids, base, freqs, mscale, half, cs);
    TSV_HIP(hipGetLastError());
    return TSV_OK;
}

int launch_prompt_mtp_input(hipStream_t s, const PromptMtpArgs& a) {
    if (a.hidden > 8192 || a.hidden % 32 || a.n < 1) {
        set_error("drafter head: hidden must be a multiple of 32, at most 8192");
        return TSV_ERR_UNSUPPORTED;
    }
    if (a.hidden <= 4096) hipLaunchKernelGGL(k_prompt_mtp_input<1>, dim3(a.n), dim3(512), 0, s, a);
    else hipLaunchKernelGGL(k_prompt_mtp_input<2>, dim3(a.n), dim3(512), 0, s, a);
    TSV_HIP(hipGetLastError());
    return TSV_OK;
}

template <int NV, int W>
static void launch_norm(hipStream_t s, const PromptNormArgs& a) {
    const dim3 grid((a.n + 8 / W - 1) / (8 / W)), block(512);
    if (a.weights) hipLaunchKernelGGL((k_prompt_norm<NV, W, true>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((k_prompt_norm<NV, W, false>), grid, block, 0, s, a);
}

// Waves to a row: as many as it takes for a workgroup per compute unit, as long as each keeps 512 values
static int norm_waves(int n, int nv) {
    int w = 1;
    while (w < 8 && w < nv && (n * w + 7) / 8 < 256) w *= 2;
    return w;
}

int launch_prompt_norm(hipStream_t s, const PromptNormArgs& a) {
    if (a.hidden % 32 || a.splits < 0 || a.splits > 8 || a.n < 1) {
        set_error("prompt pass: bad norm arguments");
        return TSV_ERR_UNSUPPORTED;
    }
    const int nv = (a.hidden + 511) / 512;
    if (nv > 8) {
        const dim3 grid((a.n + 7) / 8), block(512);
        if (a.weights) hipLaunchKernelGGL(k_prompt_norm_long<true>, grid, block, 0, s, a);
        else hipLaunchKernelGGL(k_prompt_norm_long<false>, grid, block, 0, s, a);
    } else {
        const int w = norm_waves(a.n, nv), per = (nv + w - 1) / w;
        if (w == 8) launch_norm<1, 8>(s, a);
        else if (w == 4) per == 1 ? launch_norm<1, 4>(s, a) : launch_norm<2, 4>(s, a);
        else if (w == 2) per == 1 ? launch_norm<1, 2>(s, a) : per == 2 ? launch_norm<2, 2>(s, a) : per == 3 ? launch_norm<3, 2>(s, a) : launch_norm<4, 2>(s, a);
        else nv <= 2 ? launch_norm<2, 1>(s, a) : nv <= 4 ? launch_norm<4, 1>(s, a) : nv <= 6 ? launch_norm<6, 1>(s, a) : launch_norm<8, 1>(s, a);
    }
    TSV_HIP(hipGetLastError());
    return TSV_OK;
}

int launch_prompt_groups(hipStream_t s, const int32_t* selected, int n, int top_k, int n_experts, int bm, const PromptRoutes& r) {
    if (n < 1 || n > PROMPT_ROWS || n_experts < 1 || n_experts > MAX_EXPERTS || top_k < 1 || top_k > 8) {
        set_error("moe: at most 2048 rows, 256 experts and top-k 8 in a prompt pass");
        return TSV_ERR_UNSUPPORTED;
    }
    hipLaunchKernelGGL(k_prompt_groups, dim3(1), dim3(1024), 0, s, selected, n, top_k, n_experts, bm, r);
    TSV_HIP(hipGetLastError());
    return TSV_OK;
}

int launch_prompt_gather(hipStream_t s, const uint16_t* rows, const uint8_t* row_sums, int k, const PromptRoutes& r, int n, int top_k, int n_experts,
                         uint8_t* a, uint8_t* asum) {
    const int sorted = prompt_sorted_rows(n, top_k, n_experts);
    // parts of K: four workgroups to a compute unit, as long as every thread keeps four loads
    const int blocks = (sorted + 31) / 32, parts = std::max(1, std::min((1024 + blocks - 1) / blocks, prompt_k16(k) / 16));
    hipLaunchKernelGGL(k_prompt_gather, dim3(blocks, parts), dim3(256), 0, s, rows, row_sums, prompt_k16(k), r.pair, sorted, a, asum);
    TSV_HIP(hipGetLastError());
    return TSV_OK;
}

int launch_prompt_rope(hipStream_t s, const PromptRopeArgs& a0) {
    PromptRopeArgs a = a0;
    const bool tq = a.store.k_bits != 0;
    if (a.splits < 1 || a.splits > 8 || (a.hd != 64 && a.hd != 128) || a.cap % 16 || a.n > a.cap || (tq && a.base + a.n > a.cap)) {
        set_error("prompt pass: bad rotation arguments");
        return TSV_ERR_INVALID;
    }
    a.inv_sqrt2 = 1.0f / std::sqrt(2.0f);
    const dim3 grid((a.base + a.n - 1) / 16 - a.base / 16 + 1, a.nq + 2 * a.nkv);
    if (a.hd == 128 && tq) hipLaunchKernelGGL((k_prompt_rope<128, true>), grid, dim3(256), 0, s, a);
    else if (a.hd == 128) hipLaunchKernelGGL((k_prompt_rope<128, false>), grid, dim3(256), 0, s, a);
    else if (tq) hipLaunchKernelGGL((k_prompt_rope<64, true>), grid, dim3(256), 0, s, a);
    else hipLaunchKernelGGL((k_prompt_rope<64, false>), grid, dim3(256), 0, s, a);
    TSV_HIP(hipGetLastError());
    return TSV_OK;
}

int launch_prompt_tq_levels(hipStream_t s, const TqKv& q, int positions, int nkv, int hd, int cap, uint16_t* kc, uint16_t* vc) {
    if ((hd != 64 && hd != 128) || cap % 16 || positions < 1 || positions > cap || q.k_bits < 2 || q.k_bits > 4 || q.v_bits < 2 || q.v_bits > 4) {
        set_error("prompt pass: bad arguments for quantized rows");
        return TSV_ERR_INVALID;
    }
    const int blocks = (positions + 15) / 16;
    const dim3 grid((blocks + DECODE - 1) / DECODE, nkv);
    if (hd == 128) hipLaunchKernelGGL(k_prompt_tq_levels<128>, grid, dim3(256), 0, s, q, blocks, cap, kc, vc);
    else hipLaunchKernelGGL(k_prompt_tq_levels<64>, grid, dim3(256), 0, s, q, blocks, cap, kc, vc);
    TSV_HIP(hipGetLastError());
    return TSV_OK;
}

// Chunks of the context per pair: a wave walks its positions alone, so where the pairs do not fill the chip (about two
// workgroups per compute unit) the context is cut, as long as a chunk keeps sixteen blocks of 32.
int prompt_attn_chunks(int n, int base, int nq, int nkv, int window) {
    const int wgs = (n * (nq / nkv) + 127) / 128 * nkv, blocks = (window > 0 ? std::min(base + n, window + n) : base + n) / 32 + 1;
    return std::max(1, std::min(std::min(512 / std::max(1, wgs), blocks / 16), 16));
}

template <int HD, bool TQ>
static int launch_attn(hipStream_t s, const PromptAttnArgs& a0) {
    PromptAttnArgs a = a0;
    a.group = a.nq / a.nkv;
    a.by_n = UniformDivisor(a.n);
    a.by_group = UniformDivisor(a.group);
    const int cols = a.n * (a.nq / a.nkv);
    const dim3 grid((cols + 127) / 128 * a.nkv, 1, a.nch);
    if (a.nch > 1) {
        hipLaunchKernelGGL((k_prompt_attn<HD, true, TQ>), grid, dim3(256), 0, s, a);
        const dim3 mgrid(((size_t)a.n * a.nq * (HD / 8) + 255) / 256);
        if (a.nch == 2) hipLaunchKernelGGL((k_prompt_attn_merge<HD, TQ, 2>), mgrid, dim3(256), 0, s, a);
        else hipLaunchKernelGGL((k_prompt_attn_merge<HD, TQ, 16>), mgrid, dim3(256), 0, s, a);
    } else {
        hipLaunchKernelGGL((k_prompt_attn<HD, false, TQ>), grid, dim3(256), 0, s, a);
    }
    TSV_HIP(hipGetLastError());
    return TSV_OK;
}

int launch_prompt_attention(hipStream_t s, const PromptAttnArgs& a) {
    if ((a.hd != 64 && a.hd != 128) || a.nch < 1 || a.nch > 16 || a.cap % 16 || a.base + a.n > a.cap || (int64_t)a.cap * a.hd * 2 > 0x7FFFFFFF) {
        set_error("prompt pass: bad attention arguments");
        return TSV_ERR_INVALID;
    }
    if (a.unrot) return a.hd == 128 ? launch_attn<128, true>(s, a) : launch_attn<64, true>(s, a);
    return a.hd == 128 ? launch_attn<128, false>(s, a) : launch_attn<64, false>(s, a);
}

}  // namespace tsv
