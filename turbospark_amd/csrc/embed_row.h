// One element of an embedding table row, as stored (shared by the verify passes' lookup and the prompt passes').
#pragma once
#include <type_traits>

#include "tsv_internal.h"

namespace tsv {

__device__ __forceinline__ float f16_bits_to_f32(uint16_t h) {
    return (float)__builtin_bit_cast(_Float16, h);
}

// Element e of table row `tok`: the arithmetic of the reference's dequantize_* for the row's storage type.
// (The type at compile time, embed_types: behind a branch on it a thread's values are fetched one after the other.)
template <int dtype>
__device__ __forceinline__ float embed_elem(const uint8_t* __restrict__ raw, int hidden, long tok, int e) {
    float v;
    if constexpr (dtype == TSV_Q4_K) {
        const uint8_t* blk = raw + (tok * (hidden / 256) + (e >> 8)) * 144;
        const float d = f16_bits_to_f32(*(const uint16_t*)blk);
        const float dmin = f16_bits_to_f32(*(const uint16_t*)(blk + 2));
        const uint8_t* packed = blk + 4;
        const int w = e & 255, g = w >> 6, hi = (w >> 5) & 1, l = w & 31, j = 2 * g + hi;
        int sc, mn;
        if (j < 4) {
            sc = packed[j] & 63;
            mn = packed[j + 4] & 63;
        } else {
            sc = (packed[j + 4] & 0xF) | ((packed[j - 4] >> 6) << 4);
            mn = (packed[j + 4] >> 4) | ((packed[j] >> 6) << 4);
        }
        const uint8_t byte = blk[16 + 32 * g + l];
        const int q = hi ? (byte >> 4) : (byte & 0xF);
        const float dl = d * (float)sc, ml = dmin * (float)mn;
        v = __fsub_rn(__fmul_rn(dl, (float)q), ml);
    } else if constexpr (dtype == TSV_Q8_0) {
        const uint8_t* blk = raw + (tok * (hidden / 32) + (e >> 5)) * 34;
        const float d = f16_bits_to_f32(*(const uint16_t*)blk);
        v = (float)(int8_t)blk[2 + (e & 31)] * d;
    } else if constexpr (dtype == TSV_Q5_K) {  // q5_k.rs:47-96
        const uint8_t* blk = raw + (tok * (hidden / 256) + (e >> 8)) * 176;
        const float d = f16_bits_to_f32(*(const uint16_t*)blk);
        const float dmin = f16_bits_to_f32(*(const uint16_t*)(blk + 2));
        const uint8_t* packed = blk + 4;
        const int w = e & 255, g = w >> 6, hi = (w >> 5) & 1, l = w & 31, j = 2 * g + hi;
        int sc, mn;
        if (j < 4) {
            sc = packed[j] & 63;
            mn = packed[j + 4] & 63;
        } else {
            sc = (packed[j + 4] & 0xF) | ((packed[j - 4] >> 6) << 4);
            mn = (packed[j + 4] >> 4) | ((packed[j] >> 6) << 4);
        }
        const uint8_t byte = blk[48 + 32 * g + l];
        const int q = (hi ? (byte >> 4) : (byte & 0xF)) + (((blk[16 + l] >> j) & 1) << 4);
        const float dl = d * (float)sc, ml = dmin * (float)mn;
        v = __fsub_rn(__fmul_rn(dl, (float)q), ml);
    } else if constexpr (dtype == TSV_Q6_K) {  // q6_k.rs:44-88
        const uint8_t* blk = raw + (tok * (hidden / 256) + (e >> 8)) * 210;
        const int w = e & 255, h = w >> 7, k = (w >> 5) & 3, l = w & 31;
        const int lo = (blk[64 * h + l + 32 * (k & 1)] >> (4 * (k >> 1))) & 0xF;
        const int hi = (blk[128 + 32 * h + l] >> (2 * k)) & 3;
        const float d = f16_bits_to_f32((uint16_t)(blk[208] | (blk[209] << 8)));
        v = d * (float)(int8_t)blk[192 + (w >> 4)] * (float)((lo | (hi << 4)) - 32);
    } else if constexpr (dtype == TSV_F16) {
        v = f16_bits_to_f32(((const uint16_t*)raw)[tok * hidden + e]);
    } else if constexpr (dtype == TSV_BF16) {
        v = __uint_as_float((uint32_t)((const uint16_t*)raw)[tok * hidden + e] << 16);
    } else {
        v = ((const float*)raw)[tok * hidden + e];
    }
    return v;
}

// f(the row's storage type as a constant)
template <class Fn>
__device__ __forceinline__ void embed_types(int dtype, Fn&& f) {
    switch (dtype) {
        case TSV_Q4_K: f(std::integral_constant<int, TSV_Q4_K>{}); break;
        case TSV_Q8_0: f(std::integral_constant<int, TSV_Q8_0>{}); break;
        case TSV_Q5_K: f(std::integral_constant<int, TSV_Q5_K>{}); break;
        case TSV_Q6_K: f(std::integral_constant<int, TSV_Q6_K>{}); break;
        case TSV_F16: f(std::integral_constant<int, TSV_F16>{}); break;
        case TSV_BF16: f(std::integral_constant<int, TSV_BF16>{}); break;
        default: f(std::integral_constant<int, TSV_F32>{}); break;
    }
}

}  // namespace tsv
