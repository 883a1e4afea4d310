// What the prompt passes share (producer.rs:122-150, the chunked prefill runner; families/llama/prefill.rs): a pass of up to
// PROMPT_ROWS consecutive positions whose matmuls are real contractions (gemm_prompt.hip), with embedding, norms, rotation
// and attention over all of its rows at once (prompt.hip).
//
// Activations of a matmul are kept as ready A operands of v_mfma_f32_32x32x16_f16: blocks of 32 rows, each
// [K / 16][64 lanes][8 halfs], lane (row % 32) + 32 * (k % 16 / 8) holding its row's eight values of the step, in the
// order 0 2 1 3 inside every four (what the nibble unpack of the weights produces).  K is padded to whole 256s with zeros.
// Formats with a min term (Q4_K, Q5_K) need the sums of every 32 values as well; they are kept as an A operand of the same
// instruction, one per 256 K: [K / 256][64 lanes][8 halfs], lane row % 32 the eight sub-block sums / 64 rounded to fp16, lane
// 32 + row % 32 what that rounding left over, times 2048.  A sum of fp16 values is a multiple of 2^-24: below 1/2 the two terms
// are exact, above they are within 2^-23 of its size, where an fp32 is within 2^-24.  Products of 4096 values by Q4_K weights come out
// 2.8e-7 of the exact result's norm off (weights whose codes are all zero, the min terms alone: 8e-8), by the verify passes'
// kernels, which keep fp32 sums and take 1024 times them off again, 1.7e-5 (7e-6).
#pragma once
#include "tsv_internal.h"

namespace tsv {

constexpr int PROMPT_ROWS = 2048;     // most rows of one pass
constexpr int PROMPT_MIN_ROWS = 64;   // fewer go in verify-sized passes
constexpr int PROMPT_MIN_ROWS_TQ = 160;  // of a handle with quantized KV rows (prompt_pays)
constexpr float PROMPT_SUM_SCALE = 1.0f / 64.0f, PROMPT_SUM_LEFT = 2048.0f;

__host__ __device__ inline int prompt_k16(int k) { return (k + 255) / 256 * 16; }
__host__ __device__ inline int prompt_chunks(int k) { return (k + 255) / 256; }
// halfs from the start of the activations to element (row, k) of a K-wide input
__host__ __device__ inline size_t prompt_a_index(int row, int k, int k16) {
    return (((size_t)(row >> 5) * k16 + (k >> 4)) * 64 + ((k >> 3) & 1) * 32 + (row & 31)) * 8 + (k & 4) + (((k & 1) << 1) | ((k >> 1) & 1));
}
__host__ __device__ inline size_t prompt_a_bytes(int rows, int k) { return (size_t)((rows + 31) / 32) * prompt_k16(k) * 1024; }
__host__ __device__ inline size_t prompt_sum_bytes(int rows, int k) { return (size_t)((rows + 31) / 32) * prompt_chunks(k) * 1024; }

// Rows are padded to whole 256-row tiles in every activation buffer: the padding is read (its products are never stored)
inline int prompt_padded(int rows) { return (rows + 255) / 256 * 256; }

// Routed experts: the (row, slot) pairs of a pass sorted by expert, every expert's run padded to whole 32-row blocks, and the
// row tiles the expert matmuls work on, all of one expert side by side.
struct PromptTile {
    int32_t expert, first, cnt, pad;  // pairs [first, first + cnt) in sorted order
};
struct PromptRoutes {
    int32_t* pair;       // sorted position -> row * 8 + slot
    PromptTile* tiles;
    int32_t* n_tiles;    // device count
};
__host__ __device__ inline int prompt_sorted_rows(int n, int top_k, int n_experts) { return n * top_k + 31 * n_experts; }
// Rows of an expert tile; narrow: both of the expert's matrices go through k_prompt_experts_narrow, which takes tiles of 64.  Two
// layers, whole prompts, us (n rows of them to the average expert):
//   MXFP4, 128 experts of 768 x 2048    n = 18     38     62     96    128;  64 experts  192    256
//   64 rows in the narrow kernel           551    715    955   1302   1645              1254   1589
//   128 in k_prompt_gemm                   709    816   1046   1349   1742              1290   1619
//   256                                    693    821   1052   1364   1785              1274   1626
//   Q4_K, 128 experts of 768 x 2048,  64:  723    872   1191   1625   2051
//                                    128:  716    862   1156   1470   1879
//                                    256:  734    872   1151   1523   1984
// 256 is as far as a pass of 2048 rows gets with eight of 64 experts; beyond, and for other formats beyond 192, tiles of 256 save
// unpacking.  The average decides, also where the rows crowd: with one expert in every row's choice, or the same experts in all rows', 32
// tiles of 64 rows unpack a crowded expert's weights each and are still the faster ones (MXFP4, narrow against 128 / 256 rows):
//   even / one / all       32 of 2880 x 2880, four chosen, n = 256: 1922 / 1895 / 1767 against 2181 / 2166 / 1938;  n = 187: 1482 / 1522 /
//   1360 against 1628 / 1710 / 1447;  128 of 768 x 2048, eight chosen, n = 128: 1486 / 1473 / 1344 against 1599 / 1566 / 1404
inline int prompt_expert_rows(int n, int top_k, int n_experts, bool narrow) {
    const int avg = n * top_k / n_experts;
    return narrow && avg <= 256 ? 64 : !narrow && avg <= 192 ? 128 : 256;
}
inline int prompt_max_tiles(int n, int top_k, int n_experts, int bm) { return n * top_k / bm + n_experts; }
// selected: [n][8], rank order
int launch_prompt_groups(hipStream_t s, const int32_t* selected, int n, int top_k, int n_experts, int bm, const PromptRoutes& r);
// rows [n][k_pad] (fp16, four in the order 0 2 1 3) -> activations of the sorted pairs; asum (nullable): their sums too, out of
// the rows' own
int launch_prompt_gather(hipStream_t s, const uint16_t* rows, const uint8_t* row_sums, int k, const PromptRoutes& r, int n, int top_k, int n_experts,
                         uint8_t* a, uint8_t* asum);

// The order of k_prompt_gemm's workgroups: XCD x takes the units (a part of K of a column block: what shares no weights) x, x + 8, ..., all full
// row tiles of one before the next; the short tiles (a last row tile that does not fill up) come after all full ones.
struct PromptGrid {
    int units, first_short, full, nt;  // nt column blocks x parts of K; the first workgroup of the short tiles; full row tiles
    UniformDivisor by_full, by_nt;
    int blocks(int mt) const { return (units + 7) / 8 * 8 * mt; }
    static PromptGrid of(int nt, int splits, int mt, bool last_is_short) {
        const int full = last_is_short && mt > 1 ? mt - 1 : mt;
        return PromptGrid{nt * splits, (nt * splits + 7) / 8 * 8 * full, full, nt, UniformDivisor(full), UniformDivisor(nt)};
    }
    __host__ __device__ __forceinline__ bool place(int block, int& split, int& nb, int& mb) const {
        const bool is_short = block >= first_short;
        const int at = is_short ? block - first_short : block, slot = at >> 3;
        const int rank = is_short ? slot : by_full.quotient(slot), unit = rank * 8 + (at & 7);
        mb = is_short ? full : slot - rank * full;
        split = by_nt.quotient(unit);
        nb = unit - split * nt;
        return unit < units;
    }
};

struct PromptGemmArgs {
    PromptGrid grid;
    const uint8_t* w;     // row tiles (TiledW)
    const uint8_t* a;     // activations
    const uint8_t* asum;  // their sums (formats with a min term)
    const float* rs;      // power-of-two factor of every tiled row (formats without a scale per chunk), see row_scale
    void* out;            // EPI_PARTIAL: float [m / 16][splits][16][ldo]; EPI_SILU: the next matmul's activations
    uint8_t* out_sum;     // EPI_SILU, nullable: their sums
    int m, n_tiles, kchunks, chunks_per_split, splits, ldo, n_valid;
    int a_k16;            // 16-K steps per row of the activations
    int out_k16;
    int mt, nt, bm;       // tiles of the grid: row tiles of bm = 256, 128 or 64 rows, 128 columns
    // routed experts: the row tiles, expert e owning n_tiles row tiles of w from e * n_tiles on; biases [expert][columns];
    // alpha > 0: the clamped SwiGLU (moe_gguf.metal:528-556).  EPI_PARTIAL then writes float [row / 16][8 slots][16][ldo]
    const PromptTile* tiles;
    const int32_t* tile_count;
    const int32_t* pair;
    const float *bias, *bias2;
    float alpha, limit;
};
struct PromptExperts {
    PromptRoutes routes;
    int n_experts, max_tiles, bm;
    const float *bias, *bias2;
    float alpha, limit;
};

int launch_prompt_gemm(hipStream_t s, const TiledW& w, const void* a, const void* asum, void* out, void* out_sum, int m, int splits, int epi,
                       int ldo, int n_valid);
// a: the sorted pairs' activations; EPI_SILU or EPI_PARTIAL; w holds every expert's tiles one after the other
int launch_prompt_experts(hipStream_t s, const TiledW& w, const void* a, const void* asum, void* out, void* out_sum, int epi, int ldo,
                          const PromptExperts& x);
// How many parts of K a matmul of m rows goes in, or one of the same rows by w and `beside` into the same sums: at most 8, and (more
// than one) at most PROMPT_PARTIALS sums in all
constexpr int64_t PROMPT_PARTIALS = (int64_t)512 * 256 * 128;
int prompt_splits(const TiledW& w, int m, const TiledW* beside = nullptr);
// Host arithmetic: the furthest chunk of weights and 16-K step of activations that a tile of `rows` rows asks for in chunks [c0, c1)
void prompt_walk_reach(int fmt, int rows, int c0, int c1, int* far_chunk, int* far_step);
// Q8_0, bf16, MXFP4: fills w.row_scale (prompt_row_scales floats), the power-of-two factors of the matrix's rows, and w.rows_unfit;
// waits for the stream
inline size_t prompt_row_scales(const TiledW& w) { return (size_t)w.n_tiles * TILE_ROWS + 1; }
int make_row_scale(hipStream_t s, TiledW& w);
// whether the prompt matmuls have operands for all bits of the matrix
bool prompt_holds(const TiledW& w);
bool prompt_fmt_has_sums(int fmt);

// residual rows x [n][hidden] += the partial sums of the matmul before (PromptGemmArgs::out); then, with w, their RMSNorm, as
// the next matmul's activations (w NULL and a non-NULL: the rows themselves; a NULL: the residual add alone)
struct PromptNormArgs {
    float* x;
    const float* partial;   // [n / 16][splits][16][ldp]; routed: [n / 16][8 slots][16][hidden] with `weights`
    const float* weights;   // nullable: [n][8] factors of the slots
    const float* bias;      // nullable, added after the partial sums
    const float* w;
    uint8_t *a, *asum;      // asum nullable
    uint16_t* rows16;       // nullable: the same values as plain rows [n][prompt_k16 * 16], for the experts' gather
    int n, hidden, splits, ldp, slots;  // slots: distance of the partials in rows of sixteen (splits, or 8)
    float eps;
};
int launch_prompt_norm(hipStream_t s, const PromptNormArgs& a);
// embedding rows of ids[0, n), and the rotation table of positions base ..
int launch_prompt_embed(hipStream_t s, const uint8_t* raw, int dtype, int hidden, float* x, const int32_t* ids, int n, int base, const float* freqs,
                        float mscale, int half, float2* cs);

// A drafter head's input rows (k_mtp_input, misc.hip): [norm_e(embedding of ids[row]) ; norm_h(norm_t(x[row]))] as the fc matmul's
// activations (K = 2 hidden) and sums (nullable), the rotation table of positions base .., and x cleared for the sums to come
struct PromptMtpArgs {
    const uint8_t* raw;
    int dtype, hidden, n, base, half;
    float* x;
    const int32_t* ids;
    const float *norm_e, *norm_t, *norm_h, *freqs;
    float eps, mscale;
    float2* cs;
    uint8_t *a, *asum;
};
int launch_prompt_mtp_input(hipStream_t s, const PromptMtpArgs& a);

// bias, per-head norm, rotation; q as fp16 rows, K and V into the cache
struct PromptRopeArgs {
    const float* qkv;  // [n / 16][splits][16][ldq]
    int splits, ldq, n, base;
    const float2* cs;  // [n][hd / 2]
    const float *bias, *q_norm, *k_norm;
    float eps;
    uint16_t *q16, *kc, *vc;
    int nq, nkv, hd, cap;  // cap: positions of the cache, position p in slot p % cap; nq = 0: the columns are those of K and V alone
    int paired;            // as in RopeKvArgs
    // store.k_bits: the layer keeps quantized rows: K and V go there (kc and vc unused, cap: the positions it holds), q16 is rotated
    TqKv store;
    TqSide tq_k, tq_v;
    float inv_sqrt2;       // set by the launcher
};
int launch_prompt_rope(hipStream_t s, const PromptRopeArgs& a);

// codebook levels of a quantized layer's first `positions` positions (rounded up to whole blocks) as an fp16 cache of `cap` positions
int launch_prompt_tq_levels(hipStream_t s, const TqKv& q, int positions, int nkv, int hd, int cap, uint16_t* kc, uint16_t* vc);

struct PromptAttnArgs {
    const uint16_t *q16, *kc, *vc;
    // with unrot (the value side's signs): kc and vc hold codebook levels, q16 is rotated; the norms are [nkv][cap]
    const float *kn, *vn, *unrot;
    int n, base, nq, nkv, hd, cap, window;
    float scale;
    const float* sinks;
    uint8_t *a, *asum;      // the output projection's activations (K index = head * hd + d) and sums
    float *part_o, *part_ml;  // nch > 1: [nch][nkv][n * G][hd] and [nch][nkv][n * G][2]
    int nch;
    int group;                      // set by the launcher: q heads to a kv head, and its and n's reciprocals
    UniformDivisor by_n, by_group;
};
int prompt_attn_chunks(int n, int base, int nq, int nkv, int window);
int launch_prompt_attention(hipStream_t s, const PromptAttnArgs& a);

}  // namespace tsv
