// Device-side core of the dequant-fused small-M matmul: weight-tile formats, the register stage
// of the software pipeline, and the per-tile MFMA sequences.  Shared by the dense and the expert
// matmul kernels.
#pragma once
#include <type_traits>
#include <utility>

#include "tsv_internal.h"

namespace tsv {

typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// ------------------------------------------------------------------------------- helpers
template <int... I, class Fn>
__device__ __forceinline__ void static_for_impl(std::integer_sequence<int, I...>, Fn&& f) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class Fn>
__device__ __forceinline__ void static_for(Fn&& f) {
    static_for_impl(std::make_integer_sequence<int, N>{}, f);
}

// D[i] += sum_k A_step[i][k] * B_lane[k]: A taken from block `STEP` of the a operand for all lanes
template <int STEP>
__device__ __forceinline__ float4v mfma_f16(u32x2 a, u32x2 b, float4v c) {
    return __builtin_amdgcn_mfma_f32_4x4x4f16(__builtin_bit_cast(half4, a), __builtin_bit_cast(half4, b), c, 4, STEP, 0);
}
template <int STEP>
__device__ __forceinline__ float4v mfma_f32(float a, float b, float4v c) {
    return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, c, 4, STEP, 0);
}

__device__ __forceinline__ float h2f_lo(uint32_t v) {
    return (float)__builtin_bit_cast(_Float16, (uint16_t)(v & 0xFFFF));
}
__device__ __forceinline__ float h2f_hi(uint32_t v) {
    return (float)__builtin_bit_cast(_Float16, (uint16_t)(v >> 16));
}
__device__ __forceinline__ float ubyte(uint32_t v, int i) { return (float)((v >> (8 * i)) & 0xFF); }

// (v & mask) | bits as ONE v_and_or_b32: the instruction can take a single literal / scalar
// operand, so the second constant is pinned in a vector register.
__device__ __forceinline__ uint32_t and_or(uint32_t v, uint32_t mask, uint32_t bits_vgpr) {
    return (v & mask) | bits_vgpr;
}

struct Consts {
    uint32_t k6400, k5400, k64;
};

// A tile's units are asked for in the order in which they are multiplied: loads come back in order, so the first products do not wait for
// the last unit.  (Left to itself the scheduler puts those that share an address register together.)
template <class T>
__device__ __forceinline__ void load_in_order(T& to, const T* p) {
    to = __builtin_nontemporal_load(p);
    __builtin_amdgcn_sched_barrier(0);
}

// ------------------------------------------------------------------------------- formats
// PARTS: the pieces of a tile (beside its scales) that come free one after the other while it is multiplied; 0: all at the end (load_part)
struct Q4K {
    static constexpr int NSUB = 8, NPAIR = 4, TILE_BYTES = 9216, PARTS = 4;
    static constexpr bool SUMS = true;  // the matmul needs the activations' sub-block sums
    struct Regs {
        u32x4 q[8];
        u32x4 s;
    };
    static __device__ __forceinline__ void load(Regs& r, const uint8_t* tile, int lane) {
        const u32x4* p = (const u32x4*)tile + lane;
#pragma unroll
        for (int u = 0; u < 8; u++) load_in_order(r.q[u], p + u * 64);
        r.s = __builtin_nontemporal_load(p + 512);
    }
    // float index of the sub-block sums of chunk c, and this lane's place in them before the row's own offset
    // (ActLoader::sumoff) is added: lane (b, i) reads sub-block b
    static __device__ __forceinline__ int xs_base(int c) { return c * 128; }
    static __device__ __forceinline__ int xs_lane(int lane) { return ((lane >> 2) & 7) * 4; }
};

// Q5_K (crates/compute/src/quant_gguf/q5_k.rs:47-96): the Q4_K tile followed by the fifth bits,
// [2 units][64 lanes][16 B] = the lane's 32 qh bytes.
struct Q5K {
    static constexpr int NSUB = 8, NPAIR = 4, TILE_BYTES = 11264, PARTS = 0;
    static constexpr bool SUMS = true;
    struct Regs {
        u32x4 q[8];
        u32x4 s;
        u32x4 h[2];
    };
    static __device__ __forceinline__ void load(Regs& r, const uint8_t* tile, int lane) {
        const u32x4* p = (const u32x4*)tile + lane;
#pragma unroll
        for (int u = 0; u < 8; u++) load_in_order(r.q[u], p + u * 64);
        r.s = __builtin_nontemporal_load(p + 512);
        r.h[0] = __builtin_nontemporal_load(p + 576);
        r.h[1] = __builtin_nontemporal_load(p + 640);
    }
    static __device__ __forceinline__ int xs_base(int c) { return c * 128; }
    static __device__ __forceinline__ int xs_lane(int lane) { return ((lane >> 2) & 7) * 4; }
};

struct Q80 {
    static constexpr int NSUB = 4, NPAIR = 2, TILE_BYTES = 8704, PARTS = 2;
    static constexpr bool SUMS = true;
    struct Regs {
        u32x4 q[8];
        u32x2 s;
    };
    static __device__ __forceinline__ void load(Regs& r, const uint8_t* tile, int lane) {
        const u32x4* p = (const u32x4*)tile + lane;
#pragma unroll
        for (int u = 0; u < 8; u++) load_in_order(r.q[u], p + u * 64);
        r.s = __builtin_nontemporal_load((const u32x2*)(tile + 8192) + lane);
    }
    // a 128-element chunk is half of a 256-element sum group: its four sub-blocks go to blocks 0..3
    static __device__ __forceinline__ int xs_base(int c) { return (c >> 1) * 128 + (c & 1) * 16; }
    static __device__ __forceinline__ int xs_lane(int lane) { return ((lane >> 2) & 3) * 4; }
};

// activation registers of one K chunk
// MXFP4 (ggml block_mxfp4: one e8m0 scale byte + 16 bytes of e2m1 nibbles per 32 elements;
// crates/compute/src/quant_gguf_mxfp4.rs:76-141).  A tile is 64 rows x 256 K: unit u holds the
// 32 nibbles of the lane's sub-block u, re-ordered at load time so that the four bytes of word w
// are K elements (8w, 8w+2), (8w+1, 8w+3), (8w+4, 8w+6), (8w+5, 8w+7) -- what
// v_cvt_scalef32_pk_f16_fp4 turns, byte by byte, into the fp16 pairs of two MFMA K steps in the
// activations' element order; then the eight scale bytes per lane.  e2m1 values are exact in
// fp16 and signed, so there is no code offset and no use for the activation sums.
struct MX4 {
    static constexpr int NSUB = 8, NPAIR = 4, TILE_BYTES = 8704, PARTS = 4;
    static constexpr bool SUMS = false;
    typedef Q80::Regs Regs;
    static __device__ __forceinline__ void load(Regs& r, const uint8_t* tile, int lane) { Q80::load(r, tile, lane); }
    static __device__ __forceinline__ int xs_base(int c) { return Q4K::xs_base(c); }
    static __device__ __forceinline__ int xs_lane(int lane) { return Q4K::xs_lane(lane); }
};

// bf16 matrices (crates/compute/src/quant.rs:14-39: a bf16 is the upper half of the fp32 bits).
// A tile is 64 rows x 64 K: unit u holds the lane's row at K steps 2u and 2u + 1, four values per
// step in the activations' element order (k % 4 = 0, 2, 1, 3), i.e. exactly the B operand of
// v_mfma_f32_4x4x4_16B_bf16.  The fp16 activations are split exactly into two bf16 terms
// (upper eight significant bits + remainder), so the products are those of the fp16 values.
struct BF16W {
    static constexpr int NSUB = 2, NPAIR = 1, TILE_BYTES = 8192, PARTS = 0;  // (in parts 1 % slower)
    static constexpr bool SUMS = false;
    struct Regs {
        u32x4 q[8];
    };
    static __device__ __forceinline__ void load(Regs& r, const uint8_t* tile, int lane) {
        const u32x4* p = (const u32x4*)tile + lane;
#pragma unroll
        for (int u = 0; u < 8; u++) load_in_order(r.q[u], p + u * 64);
    }
    static __device__ __forceinline__ int xs_base(int) { return 0; }
    static __device__ __forceinline__ int xs_lane(int) { return 0; }
};

// Q6_K (crates/compute/src/quant_gguf/q6_k.rs:44-88): value = d * sc_j * (level - 32), level = 4 low
// bits + 2 high bits, one signed int8 scale per 16 elements.  The level goes to the MFMA as the
// exact fp16 integer level - 32: (low nibble | 0x6400) | (high pair << 4) is 1024 + level, and one
// packed fp16 add of -1056 removes offset and bias together.
struct Q6K {
    static constexpr int NSUB = 16, NPAIR = 4, TILE_BYTES = 13568, PARTS = 4;
    static constexpr bool SUMS = false;
    struct Regs {
        u32x4 q[12];
        u32x4 s;
        uint32_t d;
    };
    static __device__ __forceinline__ void load(Regs& r, const uint8_t* tile, int lane) {
        const u32x4* p = (const u32x4*)tile + lane;
#pragma unroll
        for (int u = 0; u < 12; u++) load_in_order(r.q[u], p + u * 64);
        r.s = __builtin_nontemporal_load(p + 12 * 64);
        r.d = __builtin_nontemporal_load((const uint32_t*)(tile + 13312) + lane);
    }
    static __device__ __forceinline__ int xs_base(int) { return 0; }
    static __device__ __forceinline__ int xs_lane(int) { return 0; }
};

template <int STEP>
__device__ __forceinline__ float4v mfma_bf16(u32x2 a, u32x2 b, float4v c) {
    typedef short short4v __attribute__((ext_vector_type(4)));
    return __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(__builtin_bit_cast(short4v, a), __builtin_bit_cast(short4v, b), c, 4,
                                                  STEP, 0);
}

template <class F, int NG>
struct XRegs {
    u32x2 xa[F::NPAIR][NG];
    float xs[NG];
};

template <class F, int NG>
struct Stage {
    typename F::Regs w;
    XRegs<F, NG> x;
};

// Where a tile's bytes are read from while it is being multiplied: the registers of a stage.
template <class F>
struct RegSrc {
    const typename F::Regs& r;
    __device__ __forceinline__ u32x4 unit(int u) const { return r.q[u]; }
    __device__ __forceinline__ auto scales() const { return r.s; }
    __device__ __forceinline__ auto dval() const { return r.d; }
    __device__ __forceinline__ u32x4 high(int u) const { return r.h[u]; }
};
// The activation loads.  Which activation row feeds slot (g, i) of the MFMA A operand is a per-lane offset table: the
// identity for a dense matmul, a gather for a routed expert that sees only its own rows.
struct ActLoader {
    const u32x2* fragp;
    const float* sump;
    int rowoff[4], sumoff[4];  // offsets of row group g's row for this lane, in 8-byte units / floats
    __device__ __forceinline__ void set_row(int g, int row) {
        rowoff[g] = (row >> 2) * 64 + (row & 3);
        sumoff[g] = (row >> 2) * 32 + (row & 3);
    }
    // row `row` of a buffer made of 16-row blocks `block_bytes` apart (fragments and sums move together)
    __device__ __forceinline__ void set_row_blocked(int g, int row, size_t block_bytes) {
        set_row(g, row & 15);
        rowoff[g] += (int)((row >> 4) * (block_bytes >> 3));
        sumoff[g] += (int)((row >> 4) * (block_bytes >> 2));
    }
    __device__ __forceinline__ ActLoader(const void* xfrag, const void* xsum, int lane) {
        fragp = (const u32x2*)xfrag;
        sump = (const float*)xsum;
#pragma unroll
        for (int g = 0; g < 4; g++) set_row(g, 4 * g + (lane & 3));
    }
    // fragment `lane_at` (in 8-byte units) behind unit `at`, which is the same for a wave: its share of the address stays on the scalar unit
    __device__ __forceinline__ u32x2 frag_at(int at, int lane_at) const {
        return *(const u32x2*)((const char*)(fragp + at) + (uint32_t)(lane_at * 8));
    }
    __device__ __forceinline__ float sum_at(int at, int lane_at) const {
        return *(const float*)((const char*)(sump + at) + (uint32_t)(lane_at * 4));
    }
};

// activations of K chunk c (chunk index in the activation's own K axis)
template <class F, int NG>
__device__ __forceinline__ void load_x(XRegs<F, NG>& xr, const ActLoader& x, int c, int lane) {
#pragma unroll
    for (int p = 0; p < F::NPAIR; p++)
#pragma unroll
        for (int g = 0; g < NG; g++) xr.xa[p][g] = x.frag_at((c * F::NPAIR + p) * 256, x.rowoff[g] + (lane >> 2) * 4);
    if (F::SUMS) {
#pragma unroll
        for (int g = 0; g < NG; g++) xr.xs[g] = x.sum_at(F::xs_base(c), F::xs_lane(lane) + x.sumoff[g]);
    }
}

// The loads of one stage stay together and in program order (scheduling fences on both sides),
// so "stage s has landed" is one s_waitcnt vmcnt(n) with the same n on every path.
template <class F, int NG>
__device__ __forceinline__ void load_stage(Stage<F, NG>& st, const ActLoader& x, const uint8_t* tile_chunk, int c,
                                           int lane) {
    __builtin_amdgcn_sched_barrier(0);
    load_x(st.x, x, c, lane);
    __builtin_amdgcn_sched_barrier(0);
    F::load(st.w, tile_chunk, lane);
    __builtin_amdgcn_sched_barrier(0);
}

__device__ __forceinline__ void fma4(float4v& t, float s, const float4v& d) {
    t.x = __builtin_fmaf(s, d.x, t.x);
    t.y = __builtin_fmaf(s, d.y, t.y);
    t.z = __builtin_fmaf(s, d.z, t.z);
    t.w = __builtin_fmaf(s, d.w, t.w);
}

// One Q4_K superblock tile (64 weight rows x 256 K) against NG groups of four activation rows.
//   t  = - sum_j (d*sc_j*off_j + dmin*m_j) * sum_k X_jk       8 fp32 MFMAs per group
//   t += sum_j d*sc_j * (X_j . (off_j + q_j))                  64 fp16 MFMAs per group
// Both parts are summed per tile first so the large code offsets cancel before they reach the
// running accumulator.
// after(p): called where pair p of the sub-blocks is through (-1: the scales and the sums)
template <int NG, class Src, class After>
__device__ __forceinline__ void compute_tile_then(Q4K, const Src& w, const XRegs<Q4K, NG>& x, const Consts& k,
                                                  float4v (&acc)[NG], After&& after) {
    const u32x4 hs = w.scales();
    const float d = h2f_lo(hs.x), dmin = h2f_hi(hs.x);
    // 6-bit scale / min unpack (q4_k.rs:43-54), four sub-blocks per 32-bit word
    const uint32_t sl = hs.y & 0x3F3F3F3Fu, ml = hs.z & 0x3F3F3F3Fu;
    const uint32_t sh = (hs.w & 0x0F0F0F0Fu) | ((hs.y >> 2) & 0x30303030u);
    const uint32_t mh = ((hs.w >> 4) & 0x0F0F0F0Fu) | ((hs.z >> 2) & 0x30303030u);
    float sc[8], cf[8];
#pragma unroll
    for (int j = 0; j < 8; j++) {
        sc[j] = d * ubyte(j < 4 ? sl : sh, j & 3);
        const float mn = dmin * ubyte(j < 4 ? ml : mh, j & 3);
        // even sub-blocks carry the 1024 code offset, odd ones 64
        cf[j] = -__builtin_fmaf(sc[j], (j & 1) ? 64.0f : 1024.0f, mn);
    }
    float4v t[NG];
#pragma unroll
    for (int g = 0; g < NG; g++) t[g] = float4v{0.f, 0.f, 0.f, 0.f};
    static_for<8>([&](auto J) {
        constexpr int j = decltype(J)::value;
#pragma unroll
        for (int g = 0; g < NG; g++) t[g] = mfma_f32<j>(x.xs[g], cf[j], t[g]);
    });
    after(-1);
#pragma unroll
    for (int p = 0; p < 4; p++) {
        const u32x4 qa = w.unit(2 * p), qb = w.unit(2 * p + 1);
        float4v dlo[NG], dhi[NG];
#pragma unroll
        for (int g = 0; g < NG; g++) dlo[g] = dhi[g] = float4v{0.f, 0.f, 0.f, 0.f};
        static_for<8>([&](auto W) {
            constexpr int wi = decltype(W)::value;
            const uint32_t word = wi < 4 ? qa[wi % 4] : qb[wi % 4];
            const uint32_t v = word >> 8;
            const u32x2 blo = {and_or(word, 0x000F000Fu, k.k6400), and_or(v, 0x000F000Fu, k.k6400)};
            const u32x2 bhi = {and_or(word, 0x00F000F0u, k.k5400), and_or(v, 0x00F000F0u, k.k5400)};
#pragma unroll
            for (int g = 0; g < NG; g++) {
                dlo[g] = mfma_f16<wi>(x.xa[p][g], blo, dlo[g]);
                dhi[g] = mfma_f16<wi + 8>(x.xa[p][g], bhi, dhi[g]);
            }
        });
#pragma unroll
        for (int g = 0; g < NG; g++) {
            fma4(t[g], sc[2 * p], dlo[g]);
            fma4(t[g], sc[2 * p + 1], dhi[g]);
        }
        after(p);
    }
#pragma unroll
    for (int g = 0; g < NG; g++) acc[g] += t[g];
}
// One Q5_K superblock tile: Q4_K's sequence with the fifth bit of every code OR-ed into the fp16
// integer before the MFMA (bit 4 of 1024 + q for the low-nibble elements, bit 8 of the 1/16-ulp
// 64 + q form for the high-nibble ones).  Byte l of the lane's 32 qh bytes serves elements l of all
// eight sub-blocks: sub-block pair p reads bit 2p (low nibbles) and bit 2p + 1 (high nibbles).
template <int NG, class Src>
__device__ __forceinline__ void compute_tile(Q5K, const Src& w, const XRegs<Q5K, NG>& x, const Consts& k,
                                             float4v (&acc)[NG]) {
    const u32x4 hs = w.scales();
    const float d = h2f_lo(hs.x), dmin = h2f_hi(hs.x);
    const uint32_t sl = hs.y & 0x3F3F3F3Fu, ml = hs.z & 0x3F3F3F3Fu;
    const uint32_t sh = (hs.w & 0x0F0F0F0Fu) | ((hs.y >> 2) & 0x30303030u);
    const uint32_t mh = ((hs.w >> 4) & 0x0F0F0F0Fu) | ((hs.z >> 2) & 0x30303030u);
    float sc[8], cf[8];
#pragma unroll
    for (int j = 0; j < 8; j++) {
        sc[j] = d * ubyte(j < 4 ? sl : sh, j & 3);
        const float mn = dmin * ubyte(j < 4 ? ml : mh, j & 3);
        cf[j] = -__builtin_fmaf(sc[j], (j & 1) ? 64.0f : 1024.0f, mn);
    }
    float4v t[NG];
#pragma unroll
    for (int g = 0; g < NG; g++) t[g] = float4v{0.f, 0.f, 0.f, 0.f};
    static_for<8>([&](auto J) {
        constexpr int j = decltype(J)::value;
#pragma unroll
        for (int g = 0; g < NG; g++) t[g] = mfma_f32<j>(x.xs[g], cf[j], t[g]);
    });
    const u32x4 h0 = w.high(0), h1 = w.high(1);
    static_for<4>([&](auto P) {
        constexpr int p = decltype(P)::value;
        const u32x4 qa = w.unit(2 * p), qb = w.unit(2 * p + 1);
        float4v dlo[NG], dhi[NG];
#pragma unroll
        for (int g = 0; g < NG; g++) dlo[g] = dhi[g] = float4v{0.f, 0.f, 0.f, 0.f};
        static_for<8>([&](auto W) {
            constexpr int wi = decltype(W)::value;
            const uint32_t word = wi < 4 ? qa[wi % 4] : qb[wi % 4];
            const uint32_t hw = wi < 4 ? h0[wi % 4] : h1[wi % 4];
            const uint32_t v = word >> 8, hv = hw >> 8;
            // bit 2p of a qh byte -> bit 4 of its fp16 half; bit 2p + 1 -> bit 8
            constexpr int slo = 4 - 2 * p, shi = 7 - 2 * p;
            const uint32_t l0 = slo >= 0 ? hw << (slo >= 0 ? slo : 0) : hw >> (slo < 0 ? -slo : 0);
            const uint32_t l1 = slo >= 0 ? hv << (slo >= 0 ? slo : 0) : hv >> (slo < 0 ? -slo : 0);
            const uint32_t u0 = hw << shi, u1 = hv << shi;
            const u32x2 blo = {and_or(l0, 0x00100010u, and_or(word, 0x000F000Fu, k.k6400)),
                               and_or(l1, 0x00100010u, and_or(v, 0x000F000Fu, k.k6400))};
            const u32x2 bhi = {and_or(u0, 0x01000100u, and_or(word, 0x00F000F0u, k.k5400)),
                               and_or(u1, 0x01000100u, and_or(v, 0x00F000F0u, k.k5400))};
#pragma unroll
            for (int g = 0; g < NG; g++) {
                dlo[g] = mfma_f16<wi>(x.xa[p][g], blo, dlo[g]);
                dhi[g] = mfma_f16<wi + 8>(x.xa[p][g], bhi, dhi[g]);
            }
        });
#pragma unroll
        for (int g = 0; g < NG; g++) {
            fma4(t[g], sc[2 * p], dlo[g]);
            fma4(t[g], sc[2 * p + 1], dhi[g]);
        }
    });
#pragma unroll
    for (int g = 0; g < NG; g++) acc[g] += t[g];
}

// One Q8_0 tile (64 rows x 128 K = four 32-element blocks).  Codes go in as 1024 + (q + 128);
// the 1152 offset comes back out through the activation sums on the fp32 matrix pipe.
template <int NG, class Src, class After>
__device__ __forceinline__ void compute_tile_then(Q80, const Src& w, const XRegs<Q80, NG>& x, const Consts& k,
                                             float4v (&acc)[NG], After&& after) {
    const u32x2 hs = w.scales();
    float dj[4] = {h2f_lo(hs.x), h2f_hi(hs.x), h2f_lo(hs.y), h2f_hi(hs.y)};
    float4v t[NG];
#pragma unroll
    for (int g = 0; g < NG; g++) t[g] = float4v{0.f, 0.f, 0.f, 0.f};
    static_for<4>([&](auto J) {
        constexpr int j = decltype(J)::value;
#pragma unroll
        for (int g = 0; g < NG; g++) t[g] = mfma_f32<j>(x.xs[g], dj[j] * -1152.0f, t[g]);
    });
    after(-1);
#pragma unroll
    for (int p = 0; p < 2; p++) {
        const u32x4 qa0 = w.unit(4 * p), qa1 = w.unit(4 * p + 1), qb0 = w.unit(4 * p + 2), qb1 = w.unit(4 * p + 3);
        float4v da[NG], db[NG];
#pragma unroll
        for (int g = 0; g < NG; g++) da[g] = db[g] = float4v{0.f, 0.f, 0.f, 0.f};
        static_for<8>([&](auto W) {
            constexpr int wi = decltype(W)::value;
            // bytes -> fp16 1024 + (q + 128): interleave each byte with 0x64
            const uint32_t wa = (wi < 4 ? qa0[wi % 4] : qa1[wi % 4]) ^ 0x80808080u;
            const uint32_t wb = (wi < 4 ? qb0[wi % 4] : qb1[wi % 4]) ^ 0x80808080u;
            const u32x2 ba = {__builtin_amdgcn_perm(k.k64, wa, 0x04020400u), __builtin_amdgcn_perm(k.k64, wa, 0x04030401u)};
            const u32x2 bb = {__builtin_amdgcn_perm(k.k64, wb, 0x04020400u), __builtin_amdgcn_perm(k.k64, wb, 0x04030401u)};
#pragma unroll
            for (int g = 0; g < NG; g++) {
                da[g] = mfma_f16<wi>(x.xa[p][g], ba, da[g]);
                db[g] = mfma_f16<wi + 8>(x.xa[p][g], bb, db[g]);
            }
        });
#pragma unroll
        for (int g = 0; g < NG; g++) {
            fma4(t[g], dj[2 * p], da[g]);
            fma4(t[g], dj[2 * p + 1], db[g]);
        }
        after(p);
    }
#pragma unroll
    for (int g = 0; g < NG; g++) acc[g] += t[g];
}

// One MXFP4 tile (64 rows x 256 K = eight 32-element blocks): value = e2m1(code) * 2^(e - 127).
template <int NG, class Src, class After>
__device__ __forceinline__ void compute_tile_then(MX4, const Src& w, const XRegs<MX4, NG>& x, const Consts&,
                                             float4v (&acc)[NG], After&& after) {
    typedef _Float16 half2v __attribute__((ext_vector_type(2)));
    const u32x2 hs = w.scales();
    float sc[8];
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const uint32_t e = ((j < 4 ? hs.x : hs.y) >> (8 * (j & 3))) & 0xFFu;
        sc[j] = __uint_as_float(e ? e << 23 : 0x00400000u);  // 2^(e-127); e = 0 is the subnormal 2^-127
    }
    after(-1);
#pragma unroll
    for (int p = 0; p < 4; p++) {
        const u32x4 qa = w.unit(2 * p), qb = w.unit(2 * p + 1);
        float4v da[NG], db[NG];
#pragma unroll
        for (int g = 0; g < NG; g++) da[g] = db[g] = float4v{0.f, 0.f, 0.f, 0.f};
        static_for<4>([&](auto W) {
            constexpr int wi = decltype(W)::value;
            const uint32_t wa = qa[wi], wb = qb[wi];
            auto pair2 = [](uint32_t word, int lo) {
                const half2v h0 = lo ? __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(word, 1.0f, 2)
                                     : __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(word, 1.0f, 0);
                const half2v h1 = lo ? __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(word, 1.0f, 3)
                                     : __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(word, 1.0f, 1);
                return u32x2{__builtin_bit_cast(uint32_t, h0), __builtin_bit_cast(uint32_t, h1)};
            };
            const u32x2 a0 = pair2(wa, 0), a1 = pair2(wa, 1), b0 = pair2(wb, 0), b1 = pair2(wb, 1);
#pragma unroll
            for (int g = 0; g < NG; g++) {
                da[g] = mfma_f16<2 * wi>(x.xa[p][g], a0, da[g]);
                da[g] = mfma_f16<2 * wi + 1>(x.xa[p][g], a1, da[g]);
                db[g] = mfma_f16<8 + 2 * wi>(x.xa[p][g], b0, db[g]);
                db[g] = mfma_f16<8 + 2 * wi + 1>(x.xa[p][g], b1, db[g]);
            }
        });
#pragma unroll
        for (int g = 0; g < NG; g++) {
            fma4(acc[g], sc[2 * p], da[g]);
            fma4(acc[g], sc[2 * p + 1], db[g]);
        }
        after(p);
    }
}

// One Q6_K superblock tile (64 rows x 256 K): sixteen 16-element sub-blocks, four K steps each.
template <int NG, class Src, class After>
__device__ __forceinline__ void compute_tile_then(Q6K, const Src& w, const XRegs<Q6K, NG>& x, const Consts& k,
                                             float4v (&acc)[NG], After&& after) {
    typedef _Float16 half2v __attribute__((ext_vector_type(2)));
    const u32x4 scw = w.scales();
    const float d = h2f_lo(w.dval());
    const half2v off = {(_Float16)-1056.0f, (_Float16)-1056.0f};
    after(-1);
#pragma unroll
    for (int p = 0; p < 4; p++) {
        const u32x4 n0 = w.unit(3 * p), n1 = w.unit(3 * p + 1), hh = w.unit(3 * p + 2);
        static_for<4>([&](auto Q) {
            constexpr int q = decltype(Q)::value;
            const uint32_t H = hh[q];
            float4v t[NG];
#pragma unroll
            for (int g = 0; g < NG; g++) t[g] = float4v{0.f, 0.f, 0.f, 0.f};
            static_for<4>([&](auto SI) {
                constexpr int si = decltype(SI)::value;
                constexpr int s = 4 * q + si;
                const uint32_t nw = s < 8 ? n0[(s & 7) >> 1] : n1[(s & 7) >> 1];
                auto build = [&](int ab) {
                    const int lo_sh = (s & 1) * 8 + 4 * ab, e = 2 * si + ab;
                    const uint32_t lo = and_or(nw >> lo_sh, 0x000F000Fu, k.k6400);
                    const uint32_t hi = 2 * e >= 4 ? H >> (2 * e - 4) : H << (4 - 2 * e);
                    const uint32_t v = and_or(hi, 0x00300030u, lo);  // 1024 + level, twice
                    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2v, v) + off);
                };
                const u32x2 b = {build(0), build(1)};
#pragma unroll
                for (int g = 0; g < NG; g++) t[g] = mfma_f16<s>(x.xa[p][g], b, t[g]);
            });
            constexpr int j = 4 * q;  // sub-block 4p + q: byte (4p + q) of the scale unit
            const int sc8 = (int)(scw[p] << (24 - 8 * (j >> 2))) >> 24;
            const float sc = d * (float)sc8;
#pragma unroll
            for (int g = 0; g < NG; g++) fma4(acc[g], sc, t[g]);
        });
        after(p);
    }
}

// One bf16 tile (64 rows x 64 K).
template <int NG, class Src>
__device__ __forceinline__ void compute_tile(BF16W, const Src& w, const XRegs<BF16W, NG>& x, const Consts&,
                                             float4v (&acc)[NG]) {
    u32x2 ahi[NG], alo[NG];
#pragma unroll
    for (int g = 0; g < NG; g++) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const uint32_t word = x.xa[0][g][h];
            const float f0 = h2f_lo(word), f1 = h2f_hi(word);
            const uint32_t b0 = __float_as_uint(f0) & 0xFFFF0000u, b1 = __float_as_uint(f1) & 0xFFFF0000u;
            const uint32_t r0 = __float_as_uint(f0 - __uint_as_float(b0)), r1 = __float_as_uint(f1 - __uint_as_float(b1));
            ahi[g][h] = (b0 >> 16) | b1;
            alo[g][h] = (r0 >> 16) | (r1 & 0xFFFF0000u);
        }
    }
    static_for<16>([&](auto S) {
        constexpr int s = decltype(S)::value;
        const u32x4 u = w.unit(s >> 1);
        const u32x2 b = (s & 1) ? u32x2{u.z, u.w} : u32x2{u.x, u.y};
#pragma unroll
        for (int g = 0; g < NG; g++) {
            acc[g] = mfma_bf16<s>(ahi[g], b, acc[g]);
            acc[g] = mfma_bf16<s>(alo[g], b, acc[g]);
        }
    });
}

// a register stage
template <class F, int NG>
__device__ __forceinline__ void compute(const Stage<F, NG>& st, const Consts& k, float4v (&acc)[NG]) {
    if constexpr (F::PARTS) compute_tile_then<NG>(F{}, RegSrc<F>{st.w}, st.x, k, acc, [](int) {});
    else compute_tile<NG>(F{}, RegSrc<F>{st.w}, st.x, k, acc);
}

// Part u of a tile and of its activations: -1 the scales and the sums, else what is multiplied behind them, one after the other.  Loads come
// back in this order.
template <class F, int NG>
__device__ __forceinline__ void load_part(Stage<F, NG>& st, const ActLoader& x, const uint8_t* tile_chunk, int c, int lane, int u) {
    const u32x4* p = (const u32x4*)tile_chunk + lane;
    constexpr bool Q6 = std::is_same<F, Q6K>::value, Q4 = std::is_same<F, Q4K>::value;
    constexpr int UNITS = Q6 ? 3 : std::is_same<F, Q80>::value ? 4 : 2;  // of a part
    __builtin_amdgcn_sched_barrier(0);
    if (u < 0) {
        if constexpr (Q6) {
            st.w.s = __builtin_nontemporal_load(p + 12 * 64);
            st.w.d = __builtin_nontemporal_load((const uint32_t*)(tile_chunk + 13312) + lane);
        } else if constexpr (Q4) {
            st.w.s = __builtin_nontemporal_load(p + 512);
        } else {
            st.w.s = __builtin_nontemporal_load((const u32x2*)(tile_chunk + 8192) + lane);
        }
        if (F::SUMS) {
#pragma unroll
            for (int g = 0; g < NG; g++) st.x.xs[g] = x.sum_at(F::xs_base(c), F::xs_lane(lane) + x.sumoff[g]);
        }
    } else {
#pragma unroll
        for (int g = 0; g < NG; g++) st.x.xa[u][g] = x.frag_at((c * F::NPAIR + u) * 256, x.rowoff[g] + (lane >> 2) * 4);
#pragma unroll
        for (int i = 0; i < UNITS; i++) st.w.q[UNITS * u + i] = __builtin_nontemporal_load(p + (UNITS * u + i) * 64);
    }
    __builtin_amdgcn_sched_barrier(0);
}
template <class F, int NG>
__device__ __forceinline__ void load_tile(Stage<F, NG>& st, const ActLoader& x, const uint8_t* tile_chunk, int c, int lane) {
    if constexpr (F::PARTS) {
#pragma unroll
        for (int u = -1; u < F::PARTS; u++) load_part(st, x, tile_chunk, c, lane, u);
    } else load_stage(st, x, tile_chunk, c, lane);
}
// Multiplies a tile and asks for the next one, its parts as this one's come free: the first of them are on their way for the rest of the products,
// in the same registers.  (All of it behind the last product, five rows through 32 layers of the 8B shape in Q4_K took 1938 us for 1900, one row at a time
// through the Q4_K_M mix 3874 for 3746, six rows of eight Q8_0 layers 687 for 660, nine through routed MXFP4 layers 1018 for 993 and 768 for 752.)
template <class F, int NG>
__device__ __forceinline__ void compute_and_load(Stage<F, NG>& st, const Consts& k, float4v (&acc)[NG], const ActLoader& x, const uint8_t* tile_chunk,
                                                 int c, int lane) {
    if constexpr (F::PARTS) {
        const Stage<F, NG> now = st;
        compute_tile_then<NG>(F{}, RegSrc<F>{now.w}, now.x, k, acc, [&](int u) { load_part(st, x, tile_chunk, c, lane, u); });
    } else {
        compute(st, k, acc);
        load_stage(st, x, tile_chunk, c, lane);
    }
}

__device__ __forceinline__ float silu_f(float x) { return x / (1.0f + __expf(-x)); }

// How many rows a pass has and where they begin: asked for before a matmul's K loop, through scalar loads that its end waits for.
// (A plain load of such a value went through the vector unit, and the compiler waited for it where it stood: the first weights were asked for
// one round trip to memory later.  With the arguments in one batch, the divisions gone and the ends' sums on the vector ALU, five rows through 32 layers of
// the 8B shape in Q4_K, 128 launches, 2127 -> 2052 us; twelve routed layers 1153 -> 1131; one row through a Q4_K_M mix 1.9 %.)
struct PassRows {
    int m, base;
    static __device__ __forceinline__ PassRows ask(const VerifyParams* vp) { return {uniform_memory(vp)->m, uniform_memory(vp)->base}; }
    // keeps the loads where they were asked for, ahead of what stands before this
    __device__ __forceinline__ void asked() const { asm volatile("" ::"s"(m), "s"(base)); }
};

// All that a matmul reads of its arguments, asked for together (uniform_memory)
template <int EPI>
__device__ __forceinline__ void ask_for_arguments(const GemmArgs& a) {
    if (EPI == EPI_ROPE)
        asm volatile("" ::"s"(a.w), "s"(a.xfrag), "s"(a.xsum), "s"(a.vp), "s"(a.kchunks), "s"(a.kslice), "s"(a.splits), "s"(a.by_splits.magic), "s"(a.kparts),
                     "s"(a.per), "s"(a.rope.cs), "s"(a.rope.bias), "s"(a.rope.q16), "s"(a.rope.kc), "s"(a.rope.vc), "s"(a.rope.nq), "s"(a.rope.nkv),
                     "s"(a.rope.hd), "s"(a.rope.max_ctx));
    else
        asm volatile("" ::"s"(a.w), "s"(a.xfrag), "s"(a.xsum), "s"(a.out), "s"(a.vp), "s"(a.kchunks), "s"(a.kslice), "s"(a.splits), "s"(a.by_splits.magic),
                     "s"(a.kparts), "s"(a.per), "s"(a.ldo), "s"(a.n_valid), "s"(a.out16));
}

// The fused q/k/v projection finishing its own rows (no split-K: the sums are complete here).
// A tile of the rotated sections holds dims i (lanes 0..31) and i + hd/2 (lanes 32..63) of one
// head: the NeoX pair of a lane is lane ^ 32 (crates/compute/src/rope.rs:208-256).  Bias first,
// then the rotation (families/gptoss/attn.rs:88-118); q goes to the fp16 q buffer, K and V
// straight into the cache slot of the row (families/qwen/batched_layers.rs:84-113).
struct RopeTile {  // what a tile holds for this lane
    int kind, head, d, idim;  // 0: q, 1: k, 2: v; the dimension; the rotation pair
    __device__ __forceinline__ RopeTile(const RopeEpi& e, int tile, int lane) {
        const int hd = e.hd, half = hd >> 1, sh = hd == 128 ? 1 : 0;  // tiles per head: 1 << sh
        const int tq = e.nq << sh, tk = e.nkv << sh;
        kind = tile < tq ? 0 : tile < tq + tk ? 1 : 2;
        const int st = kind == 0 ? tile : kind == 1 ? tile - tq : tile - tq - tk;
        head = st >> sh;
        const int t = st - (head << sh);
        idim = (sh ? 32 * t : 0) + (lane & 31);  // 0 .. hd/2
        d = kind == 2 ? t * 64 + lane : (lane >= 32 ? idim + half : idim);
    }
};
// ... and what its rows 4 g .. 4 g + 3 need from memory.  (Rows that do not exist: the table has sixteen.)
struct RopePre {
    float2 cs[4];
    float bias;
    static __device__ __forceinline__ RopePre ask(const RopeEpi& e, int tile, int g, int lane) {
        const RopeTile at(e, tile, lane);
        const int half = e.hd >> 1, col = (at.kind == 0 ? 0 : at.kind == 1 ? e.nq * e.hd : (e.nq + e.nkv) * e.hd) + at.head * e.hd + at.d;
        RopePre p;
        const float b = *(e.bias ? e.bias + col : (const float*)e.cs);  // (no branch around a load)
        p.bias = e.bias ? b : 0.f;
#pragma unroll
        for (int i = 0; i < 4; i++) p.cs[i] = e.cs[(4 * g + i) * half + at.idim];
        return p;
    }
};
__device__ __forceinline__ void rope_epilogue(const RopeEpi& e, const PassRows& pass, const RopePre& pre, int tile, int g, float4v v, int lane) {
    const RopeTile at(e, tile, lane);
    const int hd = e.hd, first = pass.base % e.max_ctx;
    const bool hi = lane >= 32;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int b = 4 * g + i;
        float x = v[i] + pre.bias;
        const float2 pair = lanes_by_32(x);
        if (b >= pass.m) continue;
        if (at.kind != 2) x = hi ? pair.x * pre.cs[i].y + pair.y * pre.cs[i].x : pair.x * pre.cs[i].x - pair.y * pre.cs[i].y;
        const _Float16 h = (_Float16)x;
        if (at.kind == 0) {
            ((_Float16*)e.q16)[((long)b * e.nq + at.head) * hd + at.d] = h;
        } else {
            const int pos = first + b - (first + b >= e.max_ctx ? e.max_ctx : 0);  // the cache slot of row b (a ring layer wraps at its capacity)
            if (at.kind == 1)
                ((_Float16*)e.kc)[kcache_index(at.head, pos, at.d, hd, e.max_ctx)] = h;
            else
                ((_Float16*)e.vc)[vcache_index(at.head, pos, at.d, hd, e.max_ctx)] = h;
        }
    }
}

}  // namespace tsv
