// The matmuls of a prompt pass (crates/runtime/src/families/llama/prefill.rs): Y[row][n] = sum_k W[n][k] X[row][k] over
// hundreds of rows, straight from the quantized row tiles the verify passes read.
//
// One workgroup of four waves makes a BM x 128 tile of Y on v_mfma_f32_32x32x16_f16 (BM = 256, 128 or 64 rows; a wave
// always has 64 rows and 128, 64 or 32 columns).  The workgroup walks K in stages of 64 or 128: each stage's 128 weight rows
// are unpacked ONCE, by all four waves, into fp16 B operands in LDS (two buffers, one barrier per stage); the activations
// arrive as ready A operands (prompt.h) and go from the L2 straight to the registers of the one wave that needs them, so
// LDS carries the weights only: 4 KiB read per wave and 16-K step against 8 matrix instructions of 32 cycles.  Two workgroups
// share a compute unit where there are enough; a wave by itself keeps the matrix pipe busy too, because the next stage is
// unpacked between the products of this one (prompt_tile), a share behind each.
//
// What is multiplied are the stored values themselves, in operands that hold all of their bits:
//   Q4_K / Q5_K   sc_j * q, an integer below 2048.  The superblock's d is the unit its sums are counted in: the accumulator is
//                 multiplied by (unit before) / d when the walk enters a chunk.  At the chunk's end the unit becomes -dmin and
//                 one more matrix instruction adds the sub-block sums times the integers m_j: two multiplies per element and
//                 256 K in all, and no second accumulator
//   Q6_K          (level - 32) * 16 (sc >> 4) and (level - 32) * (sc & 15), two exact integer operands; units as above
//   Q8_0          q * d split into an fp16 and what it leaves over
//   bf16, MXFP4   the value, in fp16
// the last three times the power of two that brings the row's largest value to the top of fp16's range.  That is taken while
// every value of the row is a normal fp16 then (below, bits fall off, and before that the matrix instructions' sums grow coarser:
// they align products by the exponent fields): Q8_0 scales within 2^21 of the row's largest (smaller ones than 2^-24 there are
// not, so a row of weights below 16 always is), MXFP4 block scales within 2^25, bf16 values within 2^29.  k_row_scale looks at
// every row.  Tiles with another row of bf16 are multiplied as bf16 by activations split into two bf16 terms, at half the rate (of
// rows of 4096 normally distributed values one in about 80 000); a model with one in Q8_0 or MXFP4 takes the 16- and 64-row
// passes (prompt_supported).
//
// What bounds it, 28672 x 4096 Q4_K with the silu epilogue, operands of random bits on an MI355X.  At 2048 rows power: 523 us, 1042
// TFLOP/s with the unpack left out and the activations in the L1, 2457 if the operands are all zero (a loop of products alone:
// 1640 with random values); in a model 446 us = 1078 TFLOP/s (before 476), where a library product of 8192^3 normally distributed values
// reaches 1164.  With few rows the instructions a wave has to issue and the round trips between them: 128 rows take 47.6 us
// and 256 74.  With a stage unpacked ahead of its products, flat addresses for every load and the last registers of a load under
// way given to something else (which then waits for it) these were 564, 62 and 90, 299 rows 119 (now 109; Q5_K 131 and 115).
//
// Workgroups are numbered so that an XCD works on every eighth (block of columns, part of K) with all row blocks side by side: its
// weights come into that XCD's L2 once, and the activations are shared by the blocks in flight.  (Numbered by the column block alone a
// router of 128 experts, one block in eight parts, had all of its work on one XCD: 1000 rows of 2048 24.8 us a launch, 11.8 spread.)
#include <algorithm>
#include <type_traits>

#include "prompt.h"

namespace tsv {

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float float16v __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float half_lo(uint32_t v) { return (float)__builtin_bit_cast(_Float16, (uint16_t)(v & 0xFFFF)); }
__device__ __forceinline__ float half_hi(uint32_t v) { return (float)__builtin_bit_cast(_Float16, (uint16_t)(v >> 16)); }
__device__ __forceinline__ half2v as_h2(uint32_t v) { return __builtin_bit_cast(half2v, v); }
__device__ __forceinline__ uint32_t as_u32(half2v v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ half2v pair_of(float v) { return half2v{(_Float16)v, (_Float16)v}; }

// Loads through a buffer descriptor: lane offset in a register, the walk's offset in a scalar one, so that no vector instruction
// goes into addresses (a third of the loop's in the forms of few rows).  The descriptor's end bounds the lane offset alone: the scalar
// one has to stay inside by itself (Walk).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void* p, size_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, (uint32_t)bytes, 0x00027000);
}
__device__ __forceinline__ u32x4 load16(__amdgpu_buffer_rsrc_t b, uint32_t lane_at, uint32_t at) {
    return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(b, lane_at, at, 0));
}

// Constants that v_and_or_b32 takes from registers (the instruction has room for one literal)
struct Bits {
    uint32_t k6400, k5400;
};

// LDS of one stage: B operands [virtual 16-K step][4 column blocks of 32][64 lanes][16 B]; lane n % 32 + 32 * (k % 16 / 8).
constexpr int STEP_BYTES = 4096;
constexpr int MIN_BYTES = 4096;                    // min operands of a chunk, [4][64 lanes][16 B]
constexpr int COEF_BYTES = 128 * 8;                // the rescale factors of the tile's 128 columns: into the chunk, into its min term
constexpr int CHUNK_BYTES = MIN_BYTES + COEF_BYTES;  // two of them: a chunk's are used up to its end, the next one's written before
__device__ __forceinline__ void put_piece(uint8_t* buf, int step, int half, int t64, int lane, u32x4 v) {
    *(u32x4*)(buf + ((step * 4 + 2 * t64 + (lane >> 5)) * 64 + half * 32 + (lane & 31)) * 16) = v;
}

// The unit a row's sums are counted in, followed chunk by chunk by the lane that unpacks the row.
struct Unit {
    float u = 1.0f;
    bool first = true;
    // enters a chunk with scale d; returns what the accumulator has to be multiplied by.  d == 0 keeps the unit (the chunk's
    // integers are then cleared by the caller)
    __device__ __forceinline__ float enter(float d) {
        const float nu = d == 0.0f ? u : d;
        const float ratio = first ? 1.0f : u / nu;
        first = false;
        u = nu;
        return ratio;
    }
    __device__ __forceinline__ float enter_mins(float dmin) {
        const float nu = dmin == 0.0f ? u : -dmin;
        const float ratio = u / nu;
        u = nu;
        return ratio;
    }
};

// ---- storage types ------------------------------------------------------------------------------------------------------
// STAGE_K real K per stage, TERMS operands per weight, SPC stages per tile chunk.  A wave's share of a stage is one half of
// its K (`part`) of one 64-row tile.  It is unpacked in PIECES, so that each can stand between the products of another step:
// prepare() takes the scales (and, with the first stage of a chunk, leaves the chunk's rescale factors and min operands),
// piece() leaves a run of operands in LDS.  The bytes come in PARTS: load() asks for one, which is free for the next stage's
// once the piece last_piece(part) is through (-1: after prepare()).
template <bool Q5>
struct PromptQ45 {
    static constexpr int TILE_BYTES = Q5 ? 11264 : 9216, STAGE_K = 128, TERMS = 1, SPC = 2, PIECES = 8, PARTS = 3;
    static constexpr bool UNITS = true, MINS = true;
    struct Regs {
        u32x4 q[2], h, f[Q5 ? 2 : 1];
        half2v sc_lo, sc_hi, off_lo, off_hi;
    };
    static constexpr int last_piece(int part) { return 4 * part - 1; }
    static __device__ __forceinline__ void load(Regs& r, int what, __amdgpu_buffer_rsrc_t w, uint32_t at, int sub, int part, int lane) {
        const int u = 4 * sub + 2 * part;
        if (what == 0) {
            if (sub == 0) r.h = load16(w, lane * 16, at + 8192);  // (the chunk's second stage has it from the first; every word of it is read there: a register of a
            return;                      // load under way that nothing reads is given to something else, which then waits for the load)
        }
        r.q[what - 1] = load16(w, lane * 16, at + (u + what - 1) * 1024);
        if (Q5) r.f[Q5 ? what - 1 : 0] = load16(w, lane * 16, at + 9216 + 1024 * (what - 1));
    }
    static __device__ __forceinline__ void prepare(Regs& r, const Bits& k, Unit& unit, float, uint8_t* mins, float2* coef, int sub, int part, int t64,
                                                   int lane) {
        const float d = half_lo(r.h.x), dmin = half_hi(r.h.x);
        uint32_t sl = r.h.y & 0x3F3F3F3Fu, sh = (r.h.w & 0x0F0F0F0Fu) | ((r.h.y >> 2) & 0x30303030u);
        if (d == 0.0f) sl = sh = 0;
        if (sub == 0) {  // (the two waves of a tile's halves leave the same factors, and one term of the min operands each)
            const float into = unit.enter(d), into_mins = unit.enter_mins(dmin);
            coef[t64 * 64 + lane] = float2{into, into_mins};
            uint32_t ml = r.h.z & 0x3F3F3F3Fu, mh = ((r.h.w >> 4) & 0x0F0F0F0Fu) | ((r.h.z >> 2) & 0x30303030u);
            if (dmin == 0.0f) ml = mh = 0;
            const half2v by = pair_of(part ? 1.0f / (PROMPT_SUM_SCALE * PROMPT_SUM_LEFT) : 1.0f / PROMPT_SUM_SCALE);
            u32x4 o;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint32_t m2 = (i < 2 ? ml : mh) >> (16 * (i & 1));
                o[i] = as_u32((as_h2(k.k6400 | (m2 & 0xFF) | ((m2 & 0xFF00) << 8)) + pair_of(-1024.0f)) * by);
            }
            put_piece(mins, 0, part, t64, lane, o);
        }
        const uint32_t s2 = (sub == 0 ? sl : sh) >> (16 * part);
        r.sc_lo = as_h2(k.k6400 | (s2 & 0xFF) | ((s2 & 0xFF) << 16)) + pair_of(-1024.0f);
        r.sc_hi = as_h2(k.k6400 | ((s2 >> 8) & 0xFF) | (((s2 >> 8) & 0xFF) << 16)) + pair_of(-1024.0f);
        r.off_lo = r.sc_lo * pair_of(-1024.0f);
        r.off_hi = r.sc_hi * pair_of(-64.0f);
    }
    // 64 K of the row: sub-blocks 2 p (low nibbles) and 2 p + 1 (high), p = 2 sub + part; unit i of the pair holds elements
    // 16 i .. 16 i + 15 of both
    static __device__ __forceinline__ void piece(const Regs& r, int n, const Bits& k, float, uint8_t* buf, int sub, int part, int t64, int lane) {
        const int i = n >> 2, h = (n >> 1) & 1, high = n & 1, p = 2 * sub + part;
        u32x4 out;
#pragma unroll
        for (int w = 0; w < 2; w++) {
            const uint32_t v = r.q[i][2 * h + w];
#pragma unroll
            for (int o = 0; o < 2; o++) {
                const uint32_t x = o ? v >> 8 : v;
                uint32_t b = high ? (x & 0x00F000F0u) | k.k5400 : (x & 0x000F000Fu) | k.k6400;  // 64 + q, 1024 + q
                if (Q5) {  // the fifth bit: bit 2 p (low) / 2 p + 1 (high) of the element's byte
                    const uint32_t y = (o ? r.f[Q5 ? i : 0][2 * h + w] >> 8 : r.f[Q5 ? i : 0][2 * h + w]) >> (2 * p);
                    b |= high ? (y & 0x00020002u) << 7 : (y & 0x00010001u) << 4;
                }
                out[2 * w + o] = as_u32(__builtin_elementwise_fma(as_h2(b), high ? r.sc_hi : r.sc_lo, high ? r.off_hi : r.off_lo));
            }
        }
        put_piece(buf, 4 * part + 2 * high + i, h, t64, lane, out);
    }
};

// Q6_K: the stage is one 64-K pair; part h holds K 32 h .. 32 h + 31 = words 0..3 of unit 3 p + h and words 2 h, 2 h + 1 of
// unit 3 p + 2 (the order of the nibbles and bit pairs is k_repack_q6k's)
struct PromptQ6 {
    static constexpr int TILE_BYTES = 13568, STAGE_K = 64, TERMS = 2, SPC = 4, PIECES = 4, PARTS = 2;
    static constexpr bool UNITS = true, MINS = false;
    struct Regs {
        u32x4 n;
        u32x2 hb;
        uint32_t sc, d;
        half2v fa[2], fb[2];
    };
    static constexpr int last_piece(int part) { return part ? 3 : -1; }
    static __device__ __forceinline__ void load(Regs& r, int what, __amdgpu_buffer_rsrc_t w, uint32_t at, int sub, int part, int lane) {
        if (what == 0) {
            r.sc = __builtin_amdgcn_raw_buffer_load_b32(w, lane * 16, at + 12288 + 4 * sub, 0);
            if (sub == 0) r.d = __builtin_amdgcn_raw_buffer_load_b32(w, lane * 4, at + 13312, 0);
            return;
        }
        r.n = load16(w, lane * 16, at + (3 * sub + part) * 1024);
        r.hb = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(w, lane * 16, at + (3 * sub + 2) * 1024 + 8 * part, 0));
    }
    static __device__ __forceinline__ void prepare(Regs& r, const Bits&, Unit& unit, float, uint8_t*, float2* coef, int sub, int part, int t64, int lane) {
        const float d = half_lo(r.d);
        if (sub == 0) coef[t64 * 64 + lane] = float2{unit.enter(d), 0.0f};
        const uint32_t sc2 = d == 0.0f ? 0u : r.sc >> (16 * part);
#pragma unroll
        for (int q = 0; q < 2; q++) {  // 16 K with one scale each
            const int s8 = (int)(sc2 << (24 - 8 * q)) >> 24;
            r.fa[q] = pair_of((float)(s8 & ~15));
            r.fb[q] = pair_of((float)(s8 & 15));
        }
    }
    static __device__ __forceinline__ void piece(const Regs& r, int n, const Bits& k, float, uint8_t* buf, int, int part, int t64, int lane) {
        const int q = n >> 1, h = n & 1;
        const uint32_t H = r.hb[q];
        u32x4 a, b;
#pragma unroll
        for (int s = 0; s < 2; s++)  // 4-K steps
#pragma unroll
            for (int ab = 0; ab < 2; ab++) {
                const int e = 2 * (2 * h + s) + ab;
                const uint32_t lo = ((r.n[2 * q + h] >> (s * 8 + 4 * ab)) & 0x000F000Fu) | k.k6400;
                const uint32_t v = lo | (((H >> (2 * e)) & 0x00030003u) << 4);
                const half2v lv = as_h2(v) + pair_of(-1056.0f);
                a[s * 2 + ab] = as_u32(lv * r.fa[q]);
                b[s * 2 + ab] = as_u32(lv * r.fb[q]);
            }
        put_piece(buf, 2 * part + q, h, t64, lane, a);
        put_piece(buf, 4 + 2 * part + q, h, t64, lane, b);
    }
};

// Q8_0: 64 K = blocks 2 sub, 2 sub + 1 of the tile chunk, part = block
struct PromptQ8 {
    static constexpr int TILE_BYTES = 8704, STAGE_K = 64, TERMS = 2, SPC = 2, PIECES = 4, PARTS = 3;
    static constexpr bool UNITS = false, MINS = false;
    struct Regs {
        u32x4 q[2];
        uint32_t d;
        float f;
    };
    static constexpr int last_piece(int part) { return 2 * part - 1; }
    static __device__ __forceinline__ void load(Regs& r, int what, __amdgpu_buffer_rsrc_t w, uint32_t at, int sub, int part, int lane) {
        if (what == 0) r.d = __builtin_amdgcn_raw_buffer_load_b16(w, lane * 8, at + 8192 + 2 * (2 * sub + part), 0);
        else r.q[what - 1] = load16(w, lane * 16, at + (4 * sub + 2 * part + what - 1) * 1024);
    }
    static __device__ __forceinline__ void prepare(Regs& r, const Bits&, Unit&, float rs, uint8_t*, float2*, int, int, int, int) { r.f = half_lo(r.d) * rs; }
    static __device__ __forceinline__ void piece(const Regs& r, int n, const Bits&, float, uint8_t* buf, int, int part, int t64, int lane) {
        const int i = n >> 1, h = n & 1;
        u32x4 hi, lo;
#pragma unroll
        for (int w = 0; w < 2; w++) {
            const uint32_t v = r.q[i][2 * h + w];
            float f[4];
#pragma unroll
            for (int b = 0; b < 4; b++) f[b] = (float)((int)(v << (24 - 8 * b)) >> 24) * r.f;
#pragma unroll
            for (int o = 0; o < 2; o++) {  // (0, 2) then (1, 3)
                const half2v t = {(_Float16)f[o], (_Float16)f[o + 2]};
                hi[2 * w + o] = as_u32(t);
                lo[2 * w + o] = as_u32(half2v{(_Float16)(f[o] - (float)t.x), (_Float16)(f[o + 2] - (float)t.y)});
            }
        }
        put_piece(buf, 2 * part + i, h, t64, lane, hi);
        put_piece(buf, 4 + 2 * part + i, h, t64, lane, lo);
    }
};

// MXFP4: sub-blocks 4 sub + 2 part, + 1 of the chunk; word w of a unit is eight K in operand order
struct PromptMx {
    static constexpr int TILE_BYTES = 8704, STAGE_K = 128, TERMS = 1, SPC = 2, PIECES = 8, PARTS = 3;
    static constexpr bool UNITS = false, MINS = false;
    struct Regs {
        u32x4 q[2];
        uint32_t e;
        float f[2];
    };
    static constexpr int last_piece(int part) { return 4 * part - 1; }
    static __device__ __forceinline__ void load(Regs& r, int what, __amdgpu_buffer_rsrc_t w, uint32_t at, int sub, int part, int lane) {
        const int u = 4 * sub + 2 * part;
        if (what == 0) r.e = __builtin_amdgcn_raw_buffer_load_b16(w, lane * 8, at + 8192 + u, 0);
        else r.q[what - 1] = load16(w, lane * 16, at + (u + what - 1) * 1024);
    }
    static __device__ __forceinline__ void prepare(Regs& r, const Bits&, Unit&, float rs, uint8_t*, float2*, int, int, int, int) {
        const int shift = (int)(__float_as_uint(rs) >> 23) - 127;
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int field = (int)((r.e >> (8 * i)) & 0xFF) + shift;  // 2^(e - 127) times the row's factor
            r.f[i] = __uint_as_float((uint32_t)min(max(field, 1), 254) << 23);
        }
    }
    static __device__ __forceinline__ void piece(const Regs& r, int n, const Bits&, float, uint8_t* buf, int, int part, int t64, int lane) {
        const int i = n >> 2, w = n & 3;
        const uint32_t v = r.q[i][w];
        const float sc = r.f[i];
        const u32x4 o = {__builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(v, sc, 0)),
                         __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(v, sc, 1)),
                         __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(v, sc, 2)),
                         __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(v, sc, 3))};
        put_piece(buf, 4 * part + 2 * i + (w >> 1), w & 1, t64, lane, o);
    }
};

// bf16: a stage is one tile chunk of 64 K; part holds units 4 part .. 4 part + 3, eight K each in operand order
struct PromptBf {
    static constexpr int TILE_BYTES = 8192, STAGE_K = 64, TERMS = 1, SPC = 1, PIECES = 4, PARTS = 4;
    static constexpr bool UNITS = false, MINS = false;
    struct Regs {
        u32x4 q[4];
    };
    static constexpr int last_piece(int part) { return part; }
    static __device__ __forceinline__ void load(Regs& r, int what, __amdgpu_buffer_rsrc_t w, uint32_t at, int, int part, int lane) {
        r.q[what] = load16(w, lane * 16, at + (4 * part + what) * 1024);
    }
    static __device__ __forceinline__ void prepare(Regs&, const Bits&, Unit&, float, uint8_t*, float2*, int, int, int, int) {}
    static __device__ __forceinline__ void piece(const Regs& r, int i, const Bits&, float rs, uint8_t* buf, int, int part, int t64, int lane) {
        u32x4 o;
#pragma unroll
        for (int w = 0; w < 4; w++) {
            const uint32_t v = r.q[i][w];
            o[w] = as_u32(half2v{(_Float16)(__uint_as_float(v << 16) * rs), (_Float16)(__uint_as_float(v & 0xFFFF0000u) * rs)});
        }
        put_piece(buf, 2 * part + (i >> 1), i & 1, t64, lane, o);
    }
};

// ... and as it is stored, for tiles with a row that fp16 cannot hold
struct PromptBfStored : PromptBf {
    static __device__ __forceinline__ void piece(const Regs& r, int i, const Bits&, float, uint8_t* buf, int, int part, int t64, int lane) {
        put_piece(buf, 2 * part + (i >> 1), i & 1, t64, lane, r.q[i]);
    }
};
// what a launch over a bf16 matrix with such tiles is compiled for: each workgroup takes the form its two tiles allow
struct PromptBfEither : PromptBf {};

// Eight fp16 values as two bf16 terms, both exact: the upper eight bits and the rest
__device__ __forceinline__ void split_bf16(u32x4 v, u32x4& hi, u32x4& lo) {
#pragma unroll
    for (int w = 0; w < 4; w++) {
        const float f0 = half_lo(v[w]), f1 = half_hi(v[w]);
        const uint32_t b0 = __float_as_uint(f0) & 0xFFFF0000u, b1 = __float_as_uint(f1) & 0xFFFF0000u;
        const uint32_t r0 = __float_as_uint(f0 - __uint_as_float(b0)), r1 = __float_as_uint(f1 - __uint_as_float(b1));
        hi[w] = (b0 >> 16) | b1;
        lo[w] = (r0 >> 16) | (r1 & 0xFFFF0000u);
    }
}

__device__ __forceinline__ float silu_prompt(float x) { return x / (1.0f + __expf(-x)); }
// silu(gate) * up, or with alpha > 0 the clamped form (moe_gguf.metal:528-556)
__device__ __forceinline__ float gated(float gate, float up, float alpha, float limit) {
    if (alpha > 0.0f) {
        const float x = fminf(gate, limit), y = fminf(fmaxf(up, -limit), limit);
        return (x / (1.0f + __expf(-alpha * x))) * (y + 1.0f);
    }
    return silu_prompt(gate) * up;
}

template <class F>
constexpr int stage_bytes() {
    return F::STAGE_K / 16 * F::TERMS * STEP_BYTES;
}
template <class F>
constexpr int lds_bytes() {
    return (2 * stage_bytes<F>() < 65536 ? 65536 : 2 * stage_bytes<F>()) + 2 * CHUNK_BYTES;
}

// What a tile's walk over K asks for ahead: the weights of two stages further on, activations RING - 1 steps of 16 K.  Past the end of
// its part these are of the last chunk again, and nobody uses them (the matrix may end there, and its allocation).  The chunk is chosen once
// for all steps of a chunk: a clamp of every step took 0.3 % of a prompt of 1300 rows.
template <class F, int WN>
struct Walk {
    static constexpr int NT = 4 / WN, KS = F::STAGE_K / 16, STEPS = F::SPC * KS;  // 16-K steps of a stage, of a chunk
    static constexpr int WANT = 16 / NT, RING = STEPS < WANT ? STEPS : WANT;      // activations: steps in registers
    static __host__ __device__ __forceinline__ int chunk(int stage, int c1) { return stage / F::SPC < c1 ? stage / F::SPC : c1 - 1; }
    // step `at` of `c` or of the chunk behind it (at < 2 STEPS)
    static __host__ __device__ __forceinline__ int step(int c, int at, int c1) {
        return at < STEPS ? c * STEPS + at : (c + 1 < c1 ? c + 1 : c) * STEPS + at - STEPS;
    }
    // the furthest chunk and step asked for in part [c0, c1), as prompt_tile asks
    static void reach(int c0, int c1, int* far_chunk, int* far_step) {
        *far_chunk = std::max(chunk(c0 * F::SPC, c1), chunk(c0 * F::SPC + 1, c1));
        *far_step = step(c0, RING - 2, c1);
        for (int c = c0; c < c1; c++)
            for (int sub = 0; sub < F::SPC; sub++) {
                *far_chunk = std::max(*far_chunk, chunk(c * F::SPC + sub + 2, c1));
                for (int i = 0; i < KS; i++) *far_step = std::max(*far_step, step(c, sub * KS + i + RING - 1, c1));
            }
    }
};

// The order of a slot's instructions: what others wait for first (activations, operands), then a share of the vector instructions
// behind every product, which keeps the matrix pipe for 32 cycles and the issue port for four.
template <int NT, bool STORED>
__device__ __forceinline__ void slot_order(bool rescaled) {
    if (STORED) return;
    __builtin_amdgcn_sched_group_barrier(0x20, 4, 0);
    if (NT < 4) __builtin_amdgcn_sched_group_barrier(0x100, 2 * NT, 0);
    if (rescaled) {
#pragma unroll
        for (int i = 0; i < 2 * NT; i++) {
            __builtin_amdgcn_sched_group_barrier(0x2, 24, 0);
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < 2 * NT; i++) {
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x2, 16 / NT, 0);
        if (NT == 4 && (i & 1)) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x200, 2, 0);
}

// One tile: BM = 64 * 4 / WN rows from row0 on, of which `rows` exist.
template <class F, int WN, int EPI>
__device__ __forceinline__ void prompt_tile(const PromptGemmArgs& g, uint8_t* lds, int split, int nb, int row0, int rows, int expert) {
    using K = Walk<F, WN>;
    constexpr int NT = K::NT, BM = 64 * NT, KS = K::KS, SLOTS = KS * F::TERMS, STAGE = stage_bytes<F>(), STEPS = K::STEPS, RING = K::RING;
    constexpr int AHEAD = NT == 4 ? 1 : NT == 2 ? 2 : 3, BARRIER = SLOTS - AHEAD, SETS = NT == 4 ? 1 : 4;  // operands: slots ahead of their products
    static_assert(STEPS % RING == 0 && (SETS == 1 || SLOTS % SETS == 0), "the place of a step's registers is known at compile time");
    uint8_t* const side = lds + lds_bytes<F>() - 2 * CHUNK_BYTES;  // [chunk % 2][min operands, coefficients]
    auto mins_of = [&](int c) { return side + (c & 1) * CHUNK_BYTES; };
    auto coef_of = [&](int c) { return (float2*)(side + (c & 1) * CHUNK_BYTES + MIN_BYTES); };
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave / WN, wn = wave % WN, t64 = wave >> 1, part = wave & 1;
    const int c0 = split * g.chunks_per_split, c1 = min(c0 + g.chunks_per_split, g.kchunks);
    const int s0 = c0 * F::SPC, s1 = c1 * F::SPC;
    const int tile = expert * g.n_tiles + min(2 * nb + t64, g.n_tiles - 1);  // (an odd count: the last block's second half repeats the last tile)
    const size_t tile_bytes = (size_t)g.kchunks * F::TILE_BYTES, rbs = (size_t)g.a_k16 * 1024, sbs = (size_t)(g.a_k16 >> 4) * 1024;
    const int rb0 = (row0 >> 5) + wm * 2;
    const __amdgpu_buffer_rsrc_t wsrc = buffer_of(g.w + tile * tile_bytes, tile_bytes), asrc = buffer_of(g.a + rb0 * rbs, 2 * rbs),
                                 ssrc = buffer_of(F::MINS ? g.asum + rb0 * sbs : nullptr, 2 * sbs);
    const uint32_t a_at[2] = {(uint32_t)lane * 16, (uint32_t)(lane * 16 + rbs)}, s_at[2] = {(uint32_t)lane * 16, (uint32_t)(lane * 16 + sbs)};
    constexpr bool STORED = std::is_same<F, PromptBfStored>::value;
    const float rs = F::UNITS || STORED ? 1.0f : g.rs[tile * 64 + lane];
    Bits bits{0x64006400u, 0x54005400u};
    asm volatile("" : "+v"(bits.k6400), "+v"(bits.k5400));

    float16v acc[2][NT];
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[t][j][i] = 0.f;
    Unit unit;
    float left_in = 1.0f;  // the unit of the chunk being multiplied
    typename F::Regs w;
    u32x4 a[RING][2], b[SETS][NT], sm[2], mn[NT];
    float into[NT];
    auto load_w = [&](int what, int s, int sub) {
        F::load(w, what, wsrc, K::chunk(s, c1) * F::TILE_BYTES, sub, part, lane);
    };
    auto load_a = [&](int place, int c, int step) {
        const int at = K::step(c, step, c1) * 1024;
#pragma unroll
        for (int t = 0; t < 2; t++) a[place][t] = load16(asrc, a_at[t], at);
    };
    // operand j of a stage's slot: 16-K step slot / TERMS, term slot % TERMS
    auto load_b = [&](u32x4& to, const uint8_t* stage, int slot, int j) {
        to = *(const u32x4*)(stage + (((slot % F::TERMS * KS + slot / F::TERMS) * 4 + wn * NT + j) * 64 + lane) * 16);
    };
    auto load_into = [&](int c) {
        if (!F::UNITS) return;
#pragma unroll
        for (int j = 0; j < NT; j++) into[j] = coef_of(c)[(wn * NT + j) * 32 + (lane & 31)].x;
    };
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < F::PARTS; i++) load_w(i, s0, 0);
    __builtin_amdgcn_sched_barrier(0);
    F::prepare(w, bits, unit, rs, mins_of(c0), coef_of(c0), 0, part, t64, lane);
#pragma unroll
    for (int i = 0; i < F::PIECES; i++) F::piece(w, i, bits, rs, lds, 0, part, t64, lane);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < F::PARTS; i++) load_w(i, s0 + 1, 1 % F::SPC);
    // (the activations behind the weights, as in the loop: its first wait for weights is compiled for what either way into it leaves)
#pragma unroll
    for (int i = 0; i < RING - 1; i++) load_a(i, c0, i);
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < AHEAD; i++)
#pragma unroll
        for (int j = 0; j < NT; j++) load_b(b[i][j], lds, i, j);
    load_into(c0);
    int buf = 0;
    // A slot is one operand's products.  Around them stand, all for later: the operands of slot + AHEAD from LDS (with one or two
    // products to a slot the LDS answers later than the next one starts), activations RING - 1 steps ahead, and a share of the
    // next stage's unpacking.  The barrier stands AHEAD slots before a stage's end: everything unpacked is written by then, and
    // every wave holds the stage's last operands in registers.
    for (int s = s0; s < s1; s += F::SPC) {
#pragma unroll
        for (int sub = 0; sub < F::SPC; sub++) {
            const uint8_t* const cur = lds + buf * STAGE;
            uint8_t* const nxt = lds + (buf ^ 1) * STAGE;
            const int c = s / F::SPC, sub_next = (sub + 1) % F::SPC, c_next = (s + sub + 1) / F::SPC;
#pragma unroll
            for (int slot = 0; slot < SLOTS; slot++) {
                const int step = slot / F::TERMS, at = (sub * KS + step) % RING;
                __builtin_amdgcn_sched_barrier(0);
                if (slot == BARRIER) {
                    __syncthreads();
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (slot % F::TERMS == 0) load_a((at + RING - 1) % RING, c, sub * KS + step + RING - 1);
                if (F::MINS && sub == F::SPC - 1 && slot == 0) {
#pragma unroll
                    for (int t = 0; t < 2; t++) sm[t] = load16(ssrc, s_at[t], c * 1024);
                }
                const bool mins_next = F::MINS && sub == F::SPC - 1 && slot == SLOTS - 1;
                auto next_b = [&](u32x4& to, int j) {
                    if (slot + AHEAD < SLOTS) load_b(to, cur, slot + AHEAD, j);
                    else if (NT == 4 && mins_next) to = *(const u32x4*)(mins_of(c) + ((wn * NT + j) * 64 + lane) * 16);
                    else load_b(to, nxt, slot + AHEAD - SLOTS, j);
                };
                if (NT < 4) {
#pragma unroll
                    for (int j = 0; j < NT; j++) next_b(b[(slot + AHEAD) % SETS][j], j);
                    if (mins_next) {
#pragma unroll
                        for (int j = 0; j < NT; j++) mn[j] = *(const u32x4*)(mins_of(c) + ((wn * NT + j) * 64 + lane) * 16);
                    }
                }
                // the share of the next stage's unpacking (past the last stage: of that stage again, into the buffer that nobody
                // reads any more; the unit that the sums were left in is kept)
                if (slot == 0) {
                    if (sub_next == 0) left_in = unit.u;
                    F::prepare(w, bits, unit, rs, mins_of(c_next), coef_of(c_next), sub_next, part, t64, lane);
                }
#pragma unroll
                for (int p = 0; p < F::PIECES; p++)
                    if (p * BARRIER / F::PIECES == slot) F::piece(w, p, bits, rs, nxt, sub_next, part, t64, lane);
#pragma unroll
                for (int i = 0; i < F::PARTS; i++)
                    if ((F::last_piece(i) < 0 ? 0 : F::last_piece(i) * BARRIER / F::PIECES) == slot) load_w(i, s + sub + 2, (sub + 2) % F::SPC);
#pragma unroll
                for (int j = 0; j < NT; j++) {
                    const u32x4 bj = b[slot % SETS][j];
#pragma unroll
                    for (int t = 0; t < 2; t++) {
                        if (F::UNITS && sub == 0 && slot == 0) {
#pragma unroll
                            for (int i = 0; i < 16; i++) acc[t][j][i] *= into[j];
                        }
                        if constexpr (STORED) {
                            u32x4 hi, lo;
                            split_bf16(a[at][t], hi, lo);
                            acc[t][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, hi), __builtin_bit_cast(bf16x8, bj), acc[t][j], 0, 0, 0);
                            acc[t][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, lo), __builtin_bit_cast(bf16x8, bj), acc[t][j], 0, 0, 0);
                        } else {
                            acc[t][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, a[at][t]), __builtin_bit_cast(half8, bj), acc[t][j], 0, 0, 0);
                        }
                    }
                    if (NT == 4) next_b(b[0][j], j);
                }
                slot_order<NT, STORED>(F::UNITS && sub == 0 && slot == 0);
                if (mins_next) {
                    __builtin_amdgcn_sched_barrier(0);
                    float by[NT];
#pragma unroll
                    for (int j = 0; j < NT; j++) by[j] = coef_of(c)[(wn * NT + j) * 32 + (lane & 31)].y;
#pragma unroll
                    for (int j = 0; j < NT; j++) {
                        const u32x4 bj = NT == 4 ? b[0][j] : mn[j];
#pragma unroll
                        for (int t = 0; t < 2; t++) {
#pragma unroll
                            for (int i = 0; i < 16; i++) acc[t][j][i] *= by[j];
                            acc[t][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, sm[t]), __builtin_bit_cast(half8, bj), acc[t][j], 0, 0, 0);
                        }
                        if (NT == 4) load_b(b[0][j], nxt, 0, j);
                    }
#pragma unroll
                    for (int i = 0; i < 2 * NT; i++) {
                        __builtin_amdgcn_sched_group_barrier(0x2, 16, 0);
                        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                    }
                }
                if (sub == F::SPC - 1 && slot == SLOTS - 1) load_into(c + 1);
            }
            buf ^= 1;
        }
    }
    __syncthreads();
    // the columns' units (or the rows' power-of-two factors taken back out)
    float* const fin = (float*)side;
    if (part == 0) fin[t64 * 64 + lane] = F::UNITS ? left_in : 1.0f / rs;
    __syncthreads();
    float un[NT];
#pragma unroll
    for (int j = 0; j < NT; j++) un[j] = fin[(wn * NT + j) * 32 + (lane & 31)];
    // register i of a 32 x 32 block is row 8 (i / 4) + 4 (lane / 32) + i % 4, column lane % 32
    if (EPI == EPI_PARTIAL) {
        float* const out = (float*)g.out;
#pragma unroll
        for (int j = 0; j < NT; j++) {
            const int col = nb * 128 + (wn * NT + j) * 32 + (lane & 31);
            if (col >= g.n_valid) continue;
            const float bias = g.bias ? g.bias[(size_t)expert * g.n_valid + col] : 0.f;
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const int local = (wm * 2 + t) * 32 + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
                    if (local >= rows) continue;
                    if (g.tiles) {  // into the row's slot
                        const int pr = g.pair[row0 + local], row = pr >> 3;
                        out[((size_t)(row >> 4) * 128 + (pr & 7) * 16 + (row & 15)) * g.ldo + col] = acc[t][j][i] * un[j] + bias;
                    } else {
                        const int row = row0 + local;
                        out[(((size_t)(row >> 4) * g.splits + split) * 16 + (row & 15)) * g.ldo + col] = acc[t][j][i] * un[j];
                    }
                }
        }
        return;
    }
    // silu(gate) * up: column block 2 q of the tile is 32 gate rows, 2 q + 1 the matching up rows.  The products go through LDS
    // into the order of the next matmul's activations
    _Float16* const act = (_Float16*)lds;
    auto put_act = [&](int q, int t, int i, float gate, float up, float bg, float bu) {
        const int c = q * 32 + (lane & 31), row = (wm * 2 + t) * 32 + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
        if (g.tiles) {  // (biases before the activation, where the clamp reads them too: moe_gguf.metal:585-600)
            gate += bg;
            up += bu;
        }
        const float v = gated(gate, up, g.alpha, g.limit);
        act[((((row >> 5) * 4 + (c >> 4)) * 2 + ((c >> 3) & 1)) * 32 + (row & 31)) * 8 + (c & 4) + (((c & 1) << 1) | ((c >> 1) & 1))] = (_Float16)v;
    };
    auto bias_of = [&](const float* b, int q) {
        const int col = nb * 64 + q * 32 + (lane & 31);
        return b && col < g.n_valid ? b[(size_t)expert * g.n_valid + col] : 0.f;
    };
    if (NT >= 2) {
#pragma unroll
        for (int jq = 0; jq < NT / 2; jq++) {
            const int q = (wn * NT) / 2 + jq;
            const float bg = bias_of(g.bias, q), bu = bias_of(g.bias2, q);
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int i = 0; i < 16; i++)
                    put_act(q, t, i, acc[t][2 * jq][i] * un[2 * jq], acc[t][(2 * jq + 1) % NT][i] * un[(2 * jq + 1) % NT], bg, bu);
        }
    } else {
        // a wave holds one column block: gate and up meet in LDS (behind the activations' area), wave (q, t) finishes row block t
        float* const swap = (float*)(lds + 32768);
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int i = 0; i < 16; i++) swap[((wn * 2 + t) * 16 + i) * 64 + lane] = acc[t][0][i] * un[0];
        __syncthreads();
        const int q = wave >> 1, t = wave & 1;
        const float bg = bias_of(g.bias, q), bu = bias_of(g.bias2, q);
#pragma unroll
        for (int i = 0; i < 16; i++)
            put_act(q, t, i, swap[((2 * q * 2 + t) * 16 + i) * 64 + lane], swap[(((2 * q + 1) * 2 + t) * 16 + i) * 64 + lane], bg, bu);
    }
    __syncthreads();
    const int kvalid = g.n_valid;  // K of the next matmul
    for (int p = threadIdx.x; p < BM * 8; p += 256) {
        const int rb = p >> 8, k16 = nb * 4 + ((p >> 6) & 3);
        if (k16 * 16 < kvalid && rb * 32 < rows)  // (a 32-row block belongs to one tile)
            *(u32x4*)((uint8_t*)g.out + (((size_t)((row0 >> 5) + rb) * g.out_k16 + k16) * 64 + (p & 63)) * 16) = ((const u32x4*)lds)[p];
    }
    if (g.out_sum) {
        for (int p = threadIdx.x; p < BM * 2; p += 256) {
            const int row = p >> 1, sub = p & 1, gs = nb * 2 + sub;
            if (gs * 32 >= kvalid || (row & ~31) >= rows) continue;
            float sum = 0.f;
#pragma unroll
            for (int x = 0; x < 4; x++) {
                const half8 v = __builtin_bit_cast(half8, ((const u32x4*)lds)[((row >> 5) * 4 + 2 * sub + (x >> 1)) * 64 + (x & 1) * 32 + (row & 31)]);
#pragma unroll
                for (int e = 0; e < 8; e++) sum += (float)v[e];
            }
            sum *= PROMPT_SUM_SCALE;
            const _Float16 hi = (_Float16)sum, lo = (_Float16)((sum - (float)hi) * PROMPT_SUM_LEFT);
            _Float16* o = (_Float16*)(g.out_sum + ((size_t)((row0 >> 5) + (row >> 5)) * (g.out_k16 >> 4) + (gs >> 3)) * 1024) + (row & 31) * 8 + (gs & 7);
            o[0] = hi;
            o[256] = lo;
        }
    }
}

// Into scalar registers: a buffer descriptor made from vector registers is gone through lane by lane
__device__ __forceinline__ PromptTile uniform_tile(PromptTile t) {
    return {__builtin_amdgcn_readfirstlane(t.expert), __builtin_amdgcn_readfirstlane(t.first), __builtin_amdgcn_readfirstlane(t.cnt), 0};
}

// The grid's tiles are g.bm rows; a tile that holds fewer takes the smallest form that covers them, and these come after all
// full ones: they fill the places that the long ones leave free.  299 rows in tiles of 256 (28672 x 4096 Q4_K, 224 long tiles and
// 224 short ones) took 111 us with a column block's two tiles side by side and take 91 so; the short tiles' weights come from
// memory a second time, which is hidden.
template <class F, int EPI>
__global__ __launch_bounds__(256, 2) void k_prompt_gemm(PromptGemmArgs g) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const PromptGrid& q = g.grid;
    asm volatile("" ::"s"(q.units), "s"(q.first_short), "s"(q.full), "s"(q.by_full.magic), "s"(q.nt), "s"(q.by_nt.magic), "s"(g.w), "s"(g.a), "s"(g.asum),
                 "s"(g.rs), "s"(g.m), "s"(g.n_tiles), "s"(g.kchunks), "s"(g.chunks_per_split), "s"(g.bm), "s"(g.a_k16), "s"(g.tiles), "s"(g.tile_count), "s"(g.mt));
    int split, nb, mb;
    if (!q.place(blockIdx.x, split, nb, mb)) return;
    int row0 = mb * g.bm, rows = min(g.m - row0, g.bm), expert = 0;  // the tile's first row and how many of its rows exist
    if (g.tiles) {
        // (asked for together: what lies behind the count is in the buffer, and not used)
        const auto* const t = uniform_memory(g.tiles) + min(mb, g.mt - 1);
        const int count = *uniform_memory(g.tile_count);
        row0 = t->first;
        rows = t->cnt;
        expert = t->expert;
        asm volatile("" ::"s"(row0), "s"(rows), "s"(expert), "s"(count));
        if (mb >= count) return;
    }
    if constexpr (std::is_same<F, PromptBfEither>::value) {
        const float* const rs = g.rs + (size_t)expert * g.n_tiles * 64 + (threadIdx.x & 63);
        const bool unfit = rs[2 * nb * 64] == 0.0f || rs[min(2 * nb + 1, g.n_tiles - 1) * 64] == 0.0f;
        if (__builtin_amdgcn_ballot_w64(unfit) != 0) {  // (the same for all four waves)
            if (rows > 128) prompt_tile<PromptBfStored, 1, EPI>(g, lds, split, nb, row0, rows, expert);
            else if (rows > 64) prompt_tile<PromptBfStored, 2, EPI>(g, lds, split, nb, row0, rows, expert);
            else prompt_tile<PromptBfStored, 4, EPI>(g, lds, split, nb, row0, rows, expert);
            return;
        }
    }
    if (rows > 128) prompt_tile<F, 1, EPI>(g, lds, split, nb, row0, rows, expert);
    else if (rows > 64) prompt_tile<F, 2, EPI>(g, lds, split, nb, row0, rows, expert);
    else prompt_tile<F, 4, EPI>(g, lds, split, nb, row0, rows, expert);
}

// ---- experts with few rows, MXFP4 -----------------------------------------------------------------------------------------
// The tile of the kernel above at 64 rows is bound by the L1 and the LDS, not by the matrix pipes (each wave draws all 64 rows'
// activations, and every unpacked weight crosses the LDS for 64 rows only), and a stage ahead is too little in flight for a
// stream of weights.  Here a workgroup makes the 128 columns of TWO row tiles, its waves each a quarter of K: a lane unpacks the
// weights of its own row and one v_permlane32_swap per register turns two eight-K pieces of 64 rows into the B operands of two
// 32-column blocks, so nothing goes through LDS before the four partial sums meet there, no barrier stands in the loop, and
// operands are asked for `RING - 1` units of 32 K ahead (activations and weights alike: loads return in order, the nearer
// distance is the one that counts).  32-row blocks past the expert's last row are not multiplied.
// A workgroup's neighbours on its XCD are the other tiles of the same expert: the activations stay in that L2, weights pass once.
// Measured, gate/up and down of one layer, 1500 rows, 128 experts, top 4, 2880 x 2880: 577 + 339 us in tiles of the kernel above,
// 452 + 247 with one row tile to a workgroup (every activation drawn twice as often), 357 + 228 here (3.1 TB/s of weights); 1000
// rows, 128 experts, top 8, 768 x 2048: 144 each, 114 + 93, 93 + 96.  Of the 357, 298 are left with the weights in the cache, 331
// with the activations in the L1 and 334 without the unpack: no one thing bounds it, a workgroup's start and end are the rest.
// Rings of 3 and 4 (1 and 2 units more ahead) are 2 and 4 % slower.
// So what a start or an end waits for is asked for ahead: the tile beside the count, the row factors behind nothing but the first
// weights, pairs and biases before the sums meet.  In whole prompts down 98 -> 90 us (1000 rows) and 233 -> 226 (1500), gate/up
// 96.6 -> 95.9 and 374 -> 373.
constexpr int NARROW_ROWS = 64, NARROW_RING2 = 2, NARROW_RING1 = 4;
template <int RB, int RING>
__device__ __forceinline__ void narrow_products(__amdgpu_buffer_rsrc_t w0, __amdgpu_buffer_rsrc_t w1, __amdgpu_buffer_rsrc_t a, uint32_t rbs, int units,
                                                int unit0, const float (&rs)[2], int lane, float16v (&acc)[2][2][2]) {
    struct Piece {
        u32x4 q[2], a[2][RB];
        uint32_t e[2];
    } r[RING];
    const int last = unit0 + units - 1;
    int shift[2];
    auto load = [&](Piece& p, int u) {
        u = min(u, last);
        const uint32_t t = (u >> 3) * PromptMx::TILE_BYTES, qa = t + (u & 7) * 1024, ea = t + 8192 + (u & 7);
        __builtin_amdgcn_sched_barrier(0);
        p.q[0] = load16(w0, lane * 16, qa);
        p.q[1] = load16(w1, lane * 16, qa);
        p.e[0] = __builtin_amdgcn_raw_buffer_load_b8(w0, lane * 8, ea, 0);
        p.e[1] = __builtin_amdgcn_raw_buffer_load_b8(w1, lane * 8, ea, 0);
#pragma unroll
        for (int q = 0; q < 2; q++)
#pragma unroll
            for (int b = 0; b < RB; b++) p.a[q][b] = load16(a, lane * 16 + b * rbs, u * 2048 + q * 1024);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto multiply = [&](const Piece& p) {
#pragma unroll
        for (int q = 0; q < 2; q++)
#pragma unroll
            for (int c = 0; c < 2; c++) {
                const float sc = __uint_as_float((uint32_t)min(max((int)p.e[c] + shift[c], 1), 254) << 23);
                u32x4 b[2];
                const uint32_t lo = p.q[c][2 * q], hi = p.q[c][2 * q + 1];
                auto put = [&](int i, auto l, auto h) {
                    const auto t = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, l), __builtin_bit_cast(uint32_t, h), false, false);
                    b[0][i] = t[0];
                    b[1][i] = t[1];
                };
                put(0, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(lo, sc, 0), __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(hi, sc, 0));
                put(1, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(lo, sc, 1), __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(hi, sc, 1));
                put(2, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(lo, sc, 2), __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(hi, sc, 2));
                put(3, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(lo, sc, 3), __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(hi, sc, 3));
#pragma unroll
                for (int j = 0; j < 2; j++)
#pragma unroll
                    for (int t = 0; t < RB; t++)
                        acc[c][t][j] =
                            __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, p.a[q][t]), __builtin_bit_cast(half8, b[j]), acc[c][t][j], 0, 0, 0);
            }
    };
#pragma unroll
    for (int i = 0; i < RING - 1; i++) load(r[i], unit0 + i);
#pragma unroll
    for (int c = 0; c < 2; c++) shift[c] = (int)(__float_as_uint(rs[c]) >> 23) - 127;  // (behind the first loads: the factors are under way too)
    for (int u = unit0; u <= last; u += RING) {
#pragma unroll
        for (int i = 0; i < RING; i++) {
            load(r[(i + RING - 1) % RING], u + i + RING - 1);
            if (i == 0 || u + i <= last) multiply(r[i]);
        }
    }
}

template <int EPI>
__global__ __launch_bounds__(256, 2) void k_prompt_experts_narrow(PromptGemmArgs g) {
    __shared__ __attribute__((aligned(16))) float meet[4 * 3 * 16 * 64];  // [reader][the other waves][values][lanes]
    __shared__ float factor[128];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // XCD x takes the row tiles x, x + 8, ..., all columns of one before the next
    const int slot = blockIdx.x >> 3, mb = slot / g.nt * 8 + (blockIdx.x & 7), nb0 = slot % g.nt * 2;
    // (asked for together: what lies behind the count is in the buffer, and not used)
    const PromptTile t = uniform_tile(g.tiles[min(mb, g.mt - 1)]);
    if (mb >= *g.tile_count) return;
    const int columns = min(2, g.n_tiles - nb0);  // (an odd count: the last workgroup's second half repeats the last tile, and leaves nothing)
    float rs[2];
    const size_t tile_bytes = (size_t)g.kchunks * PromptMx::TILE_BYTES;
    const uint8_t* const w = g.w + ((size_t)t.expert * g.n_tiles + nb0) * tile_bytes;
#pragma unroll
    for (int c = 0; c < 2; c++) rs[c] = g.rs[(t.expert * g.n_tiles + nb0 + min(c, columns - 1)) * 64 + lane];
    float16v acc[2][2][2];
#pragma unroll
    for (int c = 0; c < 2; c++)
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int i = 0; i < 16; i++) acc[c][b][j][i] = 0.f;
    const size_t rbs = (size_t)g.a_k16 * 1024;
    const __amdgpu_buffer_rsrc_t w0 = buffer_of(w, tile_bytes), w1 = buffer_of(w + (columns - 1) * tile_bytes, tile_bytes),
                                 a = buffer_of(g.a + (size_t)(t.first >> 5) * rbs, (t.cnt > 32 ? 2 : 1) * rbs);
    const int units = 2 * g.kchunks;
    if (t.cnt > 32) narrow_products<2, NARROW_RING2>(w0, w1, a, rbs, units, wave * units, rs, lane, acc);
    else narrow_products<1, NARROW_RING1>(w0, w1, a, rbs, units, wave * units, rs, lane, acc);
    if (wave == 0) {
#pragma unroll
        for (int c = 0; c < 2; c++) factor[c * 64 + lane] = 1.0f / rs[c];
    }
    // where this lane's sums go and what is added to them, asked for ahead of the barriers
    int pair[8];
    float bias[2][2];
    if (EPI == EPI_PARTIAL) {
#pragma unroll
        for (int v = 0; v < 8; v++) pair[v] = g.pair[t.first + min(32 * (v >> 2) + 8 * wave + 4 * (lane >> 5) + (v & 3), t.cnt - 1)];
    }
#pragma unroll
    for (int c = 0; c < 2; c++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const float* const b = EPI == EPI_PARTIAL || !j ? g.bias : g.bias2;
            const int col = (EPI == EPI_PARTIAL ? (nb0 + c) * 64 + 32 * j : (nb0 + c) * 32) + (lane & 31);
            bias[c][j] = b && col < g.n_valid ? b[(size_t)t.expert * g.n_valid + col] : 0.f;
        }
#pragma unroll
    for (int c = 0; c < 2; c++) {
        const int nb = nb0 + c;
        if (c >= columns) break;
        if (c) __syncthreads();  // (what the first tile left in `meet` has been read)
        // wave d ends with registers 4 d .. 4 d + 3 of all four blocks: rows 8 d + 4 (lane / 32) + i of both row blocks, column lane % 32
        // of both column blocks.  Summed in the order of K.
        float mine[16];
#pragma unroll
        for (int d = 0; d < 4; d++) {
            if (wave == d) {
#pragma unroll
                for (int v = 0; v < 16; v++) mine[v] = acc[c][v >> 3][(v >> 2) & 1][4 * d + (v & 3)];
            } else {
                float* o = meet + (size_t)(d * 3 + (wave < d ? wave : wave - 1)) * 1024 + lane;
#pragma unroll
                for (int v = 0; v < 16; v++) o[v * 64] = acc[c][v >> 3][(v >> 2) & 1][4 * d + (v & 3)];
            }
        }
        __syncthreads();
        const float* in = meet + (size_t)wave * 3 * 1024 + lane;
        const float f0 = factor[c * 64 + (lane & 31)], f1 = factor[c * 64 + 32 + (lane & 31)];
        float sum[16];
#pragma unroll
        for (int v = 0; v < 16; v++) {
            float x = 0.f;
#pragma unroll
            for (int k = 0; k < 4; k++) x += k == wave ? mine[v] : in[((k < wave ? k : k == wave ? 0 : k - 1) * 16 + v) * 64];
            sum[v] = x * ((v >> 2) & 1 ? f1 : f0);
        }
        if (EPI == EPI_PARTIAL) {
            float* const out = (float*)g.out;
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const int col = nb * 64 + 32 * j + (lane & 31);
                if (col >= g.n_valid) continue;
#pragma unroll
                for (int b = 0; b < 2; b++)
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const int local = 32 * b + 8 * wave + 4 * (lane >> 5) + i;
                        if (local >= t.cnt) continue;
                        const int pr = pair[b * 4 + i], row = pr >> 3;
                        out[((size_t)(row >> 4) * 128 + (pr & 7) * 16 + (row & 15)) * g.ldo + col] = sum[b * 8 + j * 4 + i] + bias[c][j];
                    }
            }
            continue;
        }
        // 32 gate columns and the matching up columns; the products go through LDS into the order of the next matmul's activations
        __syncthreads();
        _Float16* const act = (_Float16*)meet;
        const int cc = lane & 31;
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int row = 8 * wave + 4 * (lane >> 5) + i;
                act[(((b * 2 + (cc >> 4)) * 2 + ((cc >> 3) & 1)) * 32 + row) * 8 + (cc & 4) + (((cc & 1) << 1) | ((cc >> 1) & 1))] =
                    (_Float16)gated(sum[b * 8 + i] + bias[c][0], sum[b * 8 + 4 + i] + bias[c][1], g.alpha, g.limit);
            }
        __syncthreads();
        const int p = threadIdx.x, b = p >> 7, k16 = nb * 2 + ((p >> 6) & 1);
        if (k16 * 16 < g.n_valid && b * 32 < t.cnt)
            *(u32x4*)((uint8_t*)g.out + (((size_t)((t.first >> 5) + b) * g.out_k16 + k16) * 64 + (p & 63)) * 16) = ((const u32x4*)meet)[p];
    }
}

// ---- row factors ----------------------------------------------------------------------------------------------------------
// The power of two that brings the largest magnitude of a row near the top of fp16's range: 2^7 for a Q8_0 scale (its product
// with a code stays below 2^15), 2^12 for an MXFP4 block scale (times 6), 2^15 for a bf16 value (65280 at most).  Blocks whose
// codes are all zero say nothing, whatever their scale.  0 for a row with a non-zero value (Q8_0: scale) that is below the normal
// fp16 range then, or an infinity or a NaN; `unfit` counts those.  One wave per tile.
__global__ __launch_bounds__(64) void k_row_scale(const uint8_t* __restrict__ tiles, int fmt, int kchunks, float* __restrict__ rs, int32_t* unfit) {
    const int lane = threadIdx.x, tile = blockIdx.x;
    const int tb = fmt == FMT_BF16 ? 8192 : 8704;
    const uint8_t* t = tiles + (size_t)tile * kchunks * tb;
    int e = -1000, low = 1000;  // exponents of the largest and the smallest magnitude
    bool finite = true;
    for (int c = 0; c < kchunks; c++, t += tb) {
        u32x4 q[8];
#pragma unroll
        for (int u = 0; u < 8; u++) q[u] = ((const u32x4*)t)[u * 64 + lane];
        if (fmt == FMT_Q80) {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const u32x4 any = q[2 * j] | q[2 * j + 1];
                const float d = fabsf((float)*(const _Float16*)(t + 8192 + lane * 8 + 2 * j));
                finite &= d < INFINITY;
                if (d == 0.f || !(d < INFINITY) || (any.x | any.y | any.z | any.w) == 0) continue;
                e = max(e, ilogbf(d));
                low = min(low, ilogbf(d));
            }
        } else if (fmt == FMT_MX4) {
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const int b = t[8192 + lane * 8 + j];
                finite &= b < 255;
                if (((q[j].x | q[j].y | q[j].z | q[j].w) & 0x77777777u) == 0) continue;
                e = max(e, b - 127);
                low = min(low, b - 128);  // (half a scale)
            }
        } else {
#pragma unroll
            for (int u = 0; u < 8; u++)
#pragma unroll
                for (int w = 0; w < 8; w++) {
                    const int v = (int)(q[u][w >> 1] >> (16 * (w & 1))) & 0x7FFF, exponent = v >> 7;
                    if (v == 0) continue;
                    finite &= exponent < 255;
                    const int at = exponent ? exponent - 127 : -102 - __clz(v);  // (subnormals: v * 2^-133)
                    e = max(e, at);
                    low = min(low, at);
                }
        }
    }
    const int top = fmt == FMT_Q80 ? 7 : fmt == FMT_MX4 ? 12 : 15;
    const int s = e == -1000 ? 0 : min(max(top - e, -126), 126);
    const bool fits = finite && low + s >= -14;
    rs[tile * 64 + lane] = fits ? __uint_as_float((uint32_t)(s + 127) << 23) : 0.0f;
    if (!fits) atomicAdd(unfit, 1);
}

template <class F, int EPI>
int launch_p(hipStream_t s, PromptGemmArgs& g) {
    static OncePerDevice allowed;
    if (int rc = allow_lds((const void*)k_prompt_gemm<F, EPI>, lds_bytes<F>(), allowed)) return rc;
    g.grid = PromptGrid::of(g.nt, g.splits, g.mt, !g.tiles && g.m % g.bm != 0);
    hipLaunchKernelGGL((k_prompt_gemm<F, EPI>), dim3(g.grid.blocks(g.mt)), dim3(256), lds_bytes<F>(), s, g);
    TSV_HIP(hipGetLastError());
    return TSV_OK;
}
template <class F>
int launch_f(hipStream_t s, PromptGemmArgs& g, int epi) {
    if (!g.tiles) g.mt = (g.m + g.bm - 1) / g.bm;
    return epi == EPI_SILU ? launch_p<F, EPI_SILU>(s, g) : launch_p<F, EPI_PARTIAL>(s, g);
}

// What a matmul of m rows in tiles of bm and `splits` parts of K takes, us (6 for the launch left out).  A tile of 256 / 128 / 64 rows
// x 128 columns takes 3.95 / 2.52 / 1.52 us per 256 K by itself on a compute unit, and one of two that share it half of 6.9 / 4.14 /
// 2.8 (Q4_K; 1.7 times that with two operands per weight); beside that 1.1 us a tile, and the partial sums' way through memory
// (written here, read by the norm or the rotation).  Full tiles go out first, 256 at a time, and the short ones into what these
// leave.  Fitted to 24 shapes of 90 to 1500 rows (Q4_K, Q5_K, Q6_K, Q8_0, bf16) measured in every tiling: the choice is within 2 %
// of the best one on average, 13 % at worst.  Tiles of 256 in as many parts as fill 512 places were up to 1.9 times the best: 299
// rows of 6144 x 4096 took 46 us so and 31 in (128, 2), of 4096 x 4096 31 and 21 in (128, 4), of 1024 x 4096 Q6_K 29 and 15 in
// (64, 6).
float tiling_time(const TiledW& w, int m, int bm, int splits) {
    struct Cost {
        float alone, shared;
    };
    auto cost = [](int rows) { return rows > 128 ? Cost{3.95f, 3.45f} : rows > 64 ? Cost{2.52f, 2.07f} : Cost{1.52f, 1.4f}; };
    const int per = (w.kchunks + splits - 1) / splits, nt = (w.n_tiles + 1) / 2 * splits;
    const int full = m / bm, rest = m % bm, n_long = nt * std::max(full, 1), n_short = full && rest ? nt : 0;
    const Cost l = cost(full ? bm : rest), s = cost(rest);
    const int deep = (n_long + 255) / 256;
    float t = deep % 2 ? (deep - 1) * l.shared + l.alone : deep * l.shared;
    if (n_short) t = std::max(t, (n_long * l.shared + n_short * s.shared) / 256 + 0.26f * s.shared);
    const float k256 = per * fmt_chunk_elems(w.fmt) / 256.0f * (w.fmt == FMT_Q6K || w.fmt == FMT_Q80 ? 1.7f : 1.0f);
    return k256 * t + (n_long + n_short) * (1.1f / 256) + (float)splits * m * w.n_rows * 1.7e-6f;
}
int row_block(const TiledW& w, int m, int splits) {
    int best = 256;
    for (int bm : {128, 64})
        if (bm < 2 * m && tiling_time(w, m, bm, splits) < tiling_time(w, m, best, splits)) best = bm;
    return best;
}

}  // namespace

void prompt_walk_reach(int fmt, int rows, int c0, int c1, int* far_chunk, int* far_step) {
    auto of = [&](auto f) {
        using F = decltype(f);
        if (rows > 128) Walk<F, 1>::reach(c0, c1, far_chunk, far_step);
        else if (rows > 64) Walk<F, 2>::reach(c0, c1, far_chunk, far_step);
        else Walk<F, 4>::reach(c0, c1, far_chunk, far_step);
    };
    if (fmt == FMT_Q4K) of(PromptQ45<false>{});
    else if (fmt == FMT_Q5K) of(PromptQ45<true>{});
    else if (fmt == FMT_Q6K) of(PromptQ6{});
    else if (fmt == FMT_Q80) of(PromptQ8{});
    else if (fmt == FMT_MX4) of(PromptMx{});
    else of(PromptBf{});
}

bool prompt_fmt_has_sums(int fmt) { return fmt == FMT_Q4K || fmt == FMT_Q5K; }

int make_row_scale(hipStream_t s, TiledW& w) {
    const size_t n = (size_t)w.n_tiles * TILE_ROWS;
    int32_t* const unfit = (int32_t*)(w.row_scale + n);
    int32_t count = 0;
    TSV_HIP(hipMemsetAsync(unfit, 0, 4, s));
    hipLaunchKernelGGL(k_row_scale, dim3(w.n_tiles), dim3(64), 0, s, w.tiles, w.fmt, w.kchunks, w.row_scale, unfit);
    TSV_HIP(hipGetLastError());
    TSV_HIP(hipMemcpyAsync(&count, unfit, 4, hipMemcpyDeviceToHost, s));
    TSV_HIP(hipStreamSynchronize(s));
    w.rows_unfit = count;
    return TSV_OK;
}

bool prompt_holds(const TiledW& w) { return !w.rows_unfit || w.fmt == FMT_BF16; }

int prompt_splits(const TiledW& w, int m, const TiledW* beside) {
    auto fits = [](const TiledW& t, int k) {
        const int per = (t.kchunks + k - 1) / k;
        return (t.kchunks + per - 1) / per == k;
    };
    auto time = [&](const TiledW& t, int k) { return tiling_time(t, m, row_block(t, m, k), k); };
    const int64_t sums = (int64_t)((m + 15) / 16 * 16) * (w.n_rows + (beside ? beside->n_rows : 0));
    int best = 1;
    float least = 0.f;
    for (int k = 1; k <= 8 && (k == 1 || k * sums <= PROMPT_PARTIALS); k++) {
        if (!fits(w, k) || (beside && !fits(*beside, k))) continue;
        const float t = time(w, k) + (beside ? time(*beside, k) : 0.f);
        if (k == 1 || t < least) {
            best = k;
            least = t;
        }
    }
    return best;
}

static int launch_any(hipStream_t s, const TiledW& w, PromptGemmArgs& g, int epi) {
    const int fmt = w.fmt;
    return fmt == FMT_Q4K    ? launch_f<PromptQ45<false>>(s, g, epi)
           : fmt == FMT_Q5K  ? launch_f<PromptQ45<true>>(s, g, epi)
           : fmt == FMT_Q6K  ? launch_f<PromptQ6>(s, g, epi)
           : fmt == FMT_Q80  ? launch_f<PromptQ8>(s, g, epi)
           : fmt == FMT_MX4  ? launch_f<PromptMx>(s, g, epi)
           : w.rows_unfit    ? launch_f<PromptBfEither>(s, g, epi)
                             : launch_f<PromptBf>(s, g, epi);
}

int launch_prompt_gemm(hipStream_t s, const TiledW& w, const void* a, const void* asum, void* out, void* out_sum, int m, int splits, int epi,
                       int ldo, int n_valid) {
    if (m < 1 || (epi != EPI_PARTIAL && epi != EPI_SILU) || (epi == EPI_SILU && w.n_rows % 64) || splits < 1 || splits > 8 ||
        (epi == EPI_SILU && splits != 1) || (prompt_fmt_has_sums(w.fmt) && !asum) ||
        !prompt_holds(w) ||
        (!w.row_scale && (w.fmt == FMT_Q80 || w.fmt == FMT_BF16 || w.fmt == FMT_MX4))) {
        set_error("prompt matmul: bad argument, or a weight row that spans more than fp16 operands hold");
        return TSV_ERR_INVALID;
    }
    PromptGemmArgs g{};
    g.w = w.tiles;
    g.a = (const uint8_t*)a;
    g.asum = (const uint8_t*)asum;
    g.rs = w.row_scale;
    g.out = out;
    g.out_sum = (uint8_t*)out_sum;
    g.m = m;
    g.n_tiles = w.n_tiles;
    g.kchunks = w.kchunks;
    g.chunks_per_split = (w.kchunks + splits - 1) / splits;
    g.splits = (w.kchunks + g.chunks_per_split - 1) / g.chunks_per_split;
    if (g.splits != splits) {
        set_error("prompt matmul: split count leaves an empty K slice");
        return TSV_ERR_INVALID;
    }
    g.ldo = ldo;
    g.a_k16 = prompt_k16(w.k);
    g.nt = (w.n_tiles + 1) / 2;
    g.n_valid = epi == EPI_SILU ? w.n_rows / 2 : n_valid;
    g.out_k16 = prompt_k16(w.n_rows / 2);
    g.bm = row_block(w, m, splits);
    return launch_any(s, w, g, epi);
}

int launch_prompt_experts(hipStream_t s, const TiledW& w, const void* a, const void* asum, void* out, void* out_sum, int epi, int ldo,
                          const PromptExperts& x) {
    if ((epi != EPI_PARTIAL && epi != EPI_SILU) || x.n_experts < 1 || w.n_tiles % x.n_experts || (prompt_fmt_has_sums(w.fmt) && !asum) ||
        !prompt_holds(w) ||
        (!w.row_scale && (w.fmt == FMT_Q80 || w.fmt == FMT_BF16 || w.fmt == FMT_MX4)) || (x.bm != 64 && x.bm != 128 && x.bm != 256)) {
        set_error("prompt experts: bad argument, or a weight row that spans more than fp16 operands hold");
        return TSV_ERR_INVALID;
    }
    PromptGemmArgs g{};
    g.w = w.tiles;
    g.a = (const uint8_t*)a;
    g.asum = (const uint8_t*)asum;
    g.rs = w.row_scale;
    g.out = out;
    g.out_sum = (uint8_t*)out_sum;
    g.n_tiles = w.n_tiles / x.n_experts;
    g.kchunks = g.chunks_per_split = w.kchunks;
    g.splits = 1;
    g.ldo = ldo;
    g.a_k16 = prompt_k16(w.k);
    g.nt = (g.n_tiles + 1) / 2;
    const int cols = w.n_rows / x.n_experts;
    g.n_valid = epi == EPI_SILU ? cols / 2 : cols;
    g.out_k16 = prompt_k16(cols / 2);
    g.mt = x.max_tiles;
    g.tiles = x.routes.tiles;
    g.tile_count = x.routes.n_tiles;
    g.pair = x.routes.pair;
    g.bias = x.bias;
    g.bias2 = x.bias2;
    g.alpha = epi == EPI_SILU ? x.alpha : 0.f;
    g.limit = x.limit;
    if (w.fmt == FMT_MX4 && x.bm == NARROW_ROWS && !out_sum) {
        const dim3 grid((x.max_tiles + 7) / 8 * 8 * g.nt);
        if (epi == EPI_SILU) hipLaunchKernelGGL(k_prompt_experts_narrow<EPI_SILU>, grid, dim3(256), 0, s, g);
        else hipLaunchKernelGGL(k_prompt_experts_narrow<EPI_PARTIAL>, grid, dim3(256), 0, s, g);
        TSV_HIP(hipGetLastError());
        return TSV_OK;
    }
    g.bm = x.bm;
    return launch_any(s, w, g, epi);
}

}  // namespace tsv
