// Prompt passes: the launch sequence of hundreds of consecutive rows through the decoder (crates/runtime/src/producer.rs:122-150,
// the chunked prefill runner; families/llama/prefill.rs).  A pass takes up to PROMPT_ROWS rows, so that a matmul reads its
// weights once for all of them and is bound by the matrix pipes; everything between the matmuls runs over all rows at once
// (prompt.hip).  Rows are cached before any of them attends, as in the reference's batched prefill.
#include <type_traits>

#include "ctx.h"
#include "prompt.h"

namespace tsv {

bool prompt_supported(const tsv_ctx* c) {
    if (c->mtp.on) return false;
    for (const LayerW& L : c->layers)
        if (L.cap < c->ctx_alloc || (L.n_experts && c->moe_fp4_terms) || !prompt_holds(L.qkv) || !prompt_holds(L.v_only) ||
            !prompt_holds(L.wo) || !prompt_holds(L.gate_up) || !prompt_holds(L.down) || !prompt_holds(L.router))
            return false;
    return true;
}

namespace {

// The buffers of passes of up to `rows` rows (a multiple of 256) one after the other from `at` on: sets the handle's pointers,
// or with `at` null counts only.  Returns the bytes in all.
size_t lay_out(tsv_ctx* c, int rows, uint8_t* at) {
    tsv_ctx::Prompt& w = c->prompt;
    size_t used = 0;
    auto put = [&](auto*& p, size_t bytes) {
        if (at) p = (std::remove_reference_t<decltype(p)>)(at + used);
        used += (bytes + 255) & ~(size_t)255;
    };
    const int qd = c->nq * c->hd;
    size_t width = (size_t)qd + 2 * c->nkv * c->hd;
    for (const LayerW& L : c->layers)
        width = std::max(width, (size_t)(L.n_experts ? std::max(c->hidden, L.n_experts) : c->hidden));
    // one partial sum per row and column, or what prompt_splits makes of them
    const size_t partial_floats = std::max((size_t)rows * width, std::min((size_t)8 * rows * width, (size_t)PROMPT_PARTIALS));
    put(w.x, (size_t)rows * c->hidden * 4);
    put(w.a_h, prompt_a_bytes(rows, c->hidden));
    put(w.s_h, prompt_sum_bytes(rows, c->hidden));
    put(w.a_q, prompt_a_bytes(rows, qd));
    put(w.s_q, prompt_sum_bytes(rows, qd));
    put(w.a_f, prompt_a_bytes(rows, c->ffn));
    put(w.s_f, prompt_sum_bytes(rows, c->ffn));
    put(w.partial, partial_floats * 4);
    put(w.q16, (size_t)rows * qd * 2);
    put(w.cs, (size_t)rows * (c->hd / 2) * sizeof(float2));
    put(w.ids, (size_t)rows * 4);
    put(w.part_o, (size_t)512 * 128 * c->hd * 4);
    put(w.part_ml, (size_t)512 * 128 * 2 * 4);
    for (const LayerW& L : c->layers)
        if (L.tq.k_bits) {  // one layer's rows as attention operands
            put(w.k_levels, (size_t)c->nkv * L.cap * c->hd * 2);
            put(w.v_levels, (size_t)c->nkv * L.cap * c->hd * 2);
            break;
        }
    int sorted = 0, tiles = 0;
    for (const LayerW& L : c->layers)
        if (L.n_experts) {
            sorted = std::max(sorted, prompt_padded(prompt_sorted_rows(rows, L.top_k, L.n_experts)) + 256);  // (a tile may reach past its run)
            tiles = std::max(tiles, prompt_max_tiles(rows, L.top_k, L.n_experts, 64));
        }
    if (sorted) {
        put(w.route_w, (size_t)rows * 8 * 4);
        put(w.route_sel, (size_t)rows * 8 * 4);
        put(w.pair, (size_t)sorted * 4);
        put(w.n_tiles, 4);
        put(w.tiles, (size_t)tiles * sizeof(PromptTile));
        put(w.rows16, (size_t)rows * prompt_k16(c->hidden) * 32);
        put(w.a_s, prompt_a_bytes(sorted, c->hidden));
        put(w.s_s, prompt_sum_bytes(sorted, c->hidden));
        put(w.a_e, prompt_a_bytes(sorted, c->ffn));
        put(w.s_e, prompt_sum_bytes(sorted, c->ffn));
        put(w.moe_out, (size_t)rows * 8 * c->hidden * 4);
    }
    return used;
}

int fewer(int rows) { return rows > 256 ? (rows / 2 + 255) / 256 * 256 : 0; }

}  // namespace

// One allocation with the handle, for the longest pass its context allows; where the device has no room for it, for half the
// rows, and so on down to 256.  A prompt takes as many passes as that makes (64-row ones if there was no room at all), and none
// of them allocates: an allocation in a call would stop the whole device, other handles' streams and captures with it, and takes
// longer than a short prompt's pass (a handle's first 1500 tokens over four gpt-oss layers: 8.2 ms with allocations, 4.7 without).
int prompt_open(tsv_ctx* c) {
    tsv_ctx::Prompt& w = c->prompt;
    size_t q8 = 0, all = 0;
    for (const LayerW& L : c->layers) {
        if (L.n_experts) w.full_experts = std::max(w.full_experts, (3 * L.n_experts + L.top_k - 1) / L.top_k);
        for (const TiledW* t : {&L.qkv, &L.v_only, &L.wo, &L.gate_up, &L.down}) {
            all += t->bytes;
            q8 += t->fmt == FMT_Q80 ? t->bytes : 0;
        }
    }
    w.two_terms = 2 * q8 > all;
    if (c->max_context < PROMPT_MIN_ROWS) return TSV_OK;
    for (int rows = prompt_padded(std::min(c->max_context, PROMPT_ROWS)); rows; rows = fewer(rows)) {
        const size_t bytes = lay_out(c, rows, nullptr);
        if (hipMalloc((void**)&w.arena, bytes) != hipSuccess) {
            w.arena = nullptr;
            (void)hipGetLastError();  // a refused allocation is not the next launch's error
            continue;
        }
        // Cleared once: the K padding behind a width that is not whole 256s has to stay zero, and rows past a pass's last one hold
        // finite values
        TSV_HIP(hipMemsetAsync(w.arena, 0, bytes, c->stream));
        TSV_HIP(hipStreamSynchronize(c->stream));
        lay_out(c, rows, w.arena);
        w.rows = w.most = rows;
        w.bytes = bytes;
        break;
    }
    return TSV_OK;
}

// Against three smaller passes and more a prompt pass is the faster one (81 rows of the 8B shape in Q4_K_M, six layers: 1118 us
// against 1587; gpt-oss, three layers: 1470 against 1594), against a single one it is not (64 rows: 976 against 789, 1367 against
// 962: its tiles have 128 columns, where 64 rows leave most of the chip idle).  Of two passes (65 to 80 rows, or 128 without a
// tail) the 64-row pass and the sixteen rows behind it, or the second one, win
//   for Q8_0 weights (8B shape, 65 / 80 / 128 rows at position 0: 799 / 882 / 1010 us, a prompt pass 945 / 948 / 974; with 16
//   layers of 2048 486 / 530 / 612 against 580 / 583 / 613, and the further the longer the context);
//   where routed experts have fewer than three rows on average, so that each is read for next to nothing whatever reads it
//   (gpt-oss layers, 65 / 80 rows: 1151 / 1482 us against 1403 / 1524; the 128-expert shape of eight chosen at 65 rows, four each:
//   788 against 743);
//   with quantized KV rows below PROMPT_MIN_ROWS_TQ: not the faster side, a prompt pass is from 65 rows on (8B shape, 4-bit rows, eight
//   layers, 64-row passes against a prompt pass: 65 / 96 / 128 / 159 rows at position 0 1612 / 2395 / 3615 / 3438 us against 1359 / 1425 /
//   1478 / 1741, behind 4000 positions 1741 / 2588 / 3886 / 3758 against 1678 / 1707 / 1745 / 2107; 64-wide heads, 2-bit rows, 65 / 159: 1026 /
//   2166 against 820 / 942).  The line keeps prompts of up to 150 rows of such a handle in the 64-row passes that they are known by, which
//   are held to the oracle's quantized rows at these lengths;
//   far into a context: a prompt pass's attention takes its blocks in whole 128-pair workgroups.  Q4_K, 8B shape, 65 rows: 715
//   against 695 us at 0, 750 / 765 at 4000, 780 / 846 at 8000; 80 rows: 799 / 701, 831 / 769, 861 / 856, and 564 / 588 (two
//   layers) at 32 000.
bool prompt_pays(const tsv_ctx* c, int64_t n, int64_t base, bool tail) {
    if (n < PROMPT_MIN_ROWS || (n == PROMPT_MIN_ROWS && tail)) return false;  // (see prefill_passes)
    if (!c->wide.ok) return true;
    if (c->tq_kc && n < PROMPT_MIN_ROWS_TQ) return false;
    tail |= c->mtp_head != nullptr;  // (the rows an attached head steps from)
    const int64_t blocks = n / 64 - (tail && n % 64 == 0), rest = n - 64 * blocks, smaller = blocks + (rest + 15) / 16;
    if (smaller != 2) return smaller > 2;
    return !c->prompt.two_terms && n >= c->prompt.full_experts && (n > 80 || base < 2048 * (n - 63));
}

void prompt_limit(tsv_ctx* c, size_t bytes) {
    c->prompt.most = c->prompt.rows;
    while (c->prompt.most && lay_out(c, c->prompt.most, nullptr) > bytes) c->prompt.most = fewer(c->prompt.most);
}

namespace {

int launch_prompt_pass(tsv_ctx* c, int n, int64_t base, bool finish, bool logits) {
    hipStream_t s = c->stream;
    tsv_ctx::Prompt& w = c->prompt;
    const int H = c->hidden, qkv_n = (c->nq + 2 * c->nkv) * c->hd;
    int rc = launch_prompt_embed(s, c->embed_raw, c->embed_dtype, H, w.x, w.ids, n, (int)base, c->freqs, c->rope_mscale, c->hd / 2, w.cs);
    if (rc) return rc;
    PromptNormArgs na{};
    na.x = w.x;
    na.partial = w.partial;
    na.n = n;
    na.hidden = na.ldp = H;
    na.eps = c->eps;
    na.a = w.a_h;
    auto norm = [&](const float* weight, int splits, const float* bias, const TiledW& next) {
        na.w = weight;
        na.splits = splits;
        na.slots = na.weights ? 8 : splits;
        na.bias = bias;
        na.asum = prompt_fmt_has_sums(next.fmt) ? w.s_h : nullptr;
        return launch_prompt_norm(s, na);
    };
    // router, ranking, the pairs sorted by expert, then every expert's matrices against the rows that chose it
    auto routed_ffn = [&](const LayerW& L) {
        const int rsp = prompt_splits(L.router, n);
        int rc = launch_prompt_gemm(s, L.router, w.a_h, w.s_h, w.partial, nullptr, n, rsp, EPI_PARTIAL, L.n_experts, L.n_experts);
        if (rc) return rc;
        MoeRouteArgs ra{};
        ra.logits = w.partial;
        ra.splits = rsp;
        ra.ld = L.n_experts;
        ra.n_experts = L.n_experts;
        ra.top_k = L.top_k;
        ra.m = 16;
        ra.weights = w.route_w;
        ra.selected = w.route_sel;
        ra.bias = L.router_bias;
        ra.blocks = (n + 15) / 16;
        ra.logits_block_stride = (long)rsp * 16 * L.n_experts;
        PromptExperts x{};
        x.routes = PromptRoutes{w.pair, w.tiles, w.n_tiles};
        x.n_experts = L.n_experts;
        x.bm = prompt_expert_rows(n, L.top_k, L.n_experts, L.gate_up.fmt == FMT_MX4 && L.down.fmt == FMT_MX4);
        x.max_tiles = prompt_max_tiles(n, L.top_k, L.n_experts, x.bm);
        x.bias = L.be_gate;
        x.bias2 = L.be_up;
        x.alpha = c->act_alpha;
        x.limit = c->act_limit;
        if ((rc = launch_route(s, ra)) || (rc = launch_prompt_groups(s, w.route_sel, n, L.top_k, L.n_experts, x.bm, x.routes)) ||
            (rc = launch_prompt_gather(s, w.rows16, w.s_h, H, x.routes, n, L.top_k, L.n_experts, w.a_s,
                                       prompt_fmt_has_sums(L.gate_up.fmt) ? w.s_s : nullptr)) ||
            (rc = launch_prompt_experts(s, L.gate_up, w.a_s, w.s_s, w.a_e, prompt_fmt_has_sums(L.down.fmt) ? w.s_e : nullptr, EPI_SILU, 0, x)))
            return rc;
        x.bias = L.be_down;
        x.bias2 = nullptr;
        return launch_prompt_experts(s, L.down, w.a_e, w.s_e, w.moe_out, nullptr, EPI_PARTIAL, H, x);
    };
    int sp = 0;
    for (int l = 0; l < c->n_layers; l++) {
        LayerW& L = c->layers[l];
        na.rows16 = nullptr;
        if ((rc = norm(L.attn_norm, sp, nullptr, prompt_fmt_has_sums(L.qkv.fmt) || !L.v_only.tiles ? L.qkv : L.v_only))) return rc;
        na.partial = w.partial;
        na.weights = nullptr;
        sp = prompt_splits(L.qkv, n, L.v_only.tiles ? &L.v_only : nullptr);
        if ((rc = launch_prompt_gemm(s, L.qkv, w.a_h, w.s_h, w.partial, nullptr, n, sp, EPI_PARTIAL, qkv_n, L.qkv.n_rows))) return rc;
        if (L.v_only.tiles &&
            (rc = launch_prompt_gemm(s, L.v_only, w.a_h, w.s_h, w.partial + L.qkv.n_rows, nullptr, n, sp, EPI_PARTIAL, qkv_n, L.v_only.n_rows)))
            return rc;
        PromptRopeArgs ra{};
        ra.qkv = w.partial;
        ra.splits = sp;
        ra.ldq = qkv_n;
        ra.n = n;
        ra.base = (int)base;
        ra.cs = w.cs;
        ra.bias = L.bqkv;
        ra.q_norm = L.q_norm;
        ra.k_norm = L.k_norm;
        ra.eps = c->eps;
        ra.q16 = w.q16;
        ra.kc = L.kc;
        ra.vc = L.vc;
        ra.nq = c->nq;
        ra.nkv = c->nkv;
        ra.hd = c->hd;
        ra.cap = L.cap;
        ra.paired = L.rope_fused && c->hd == 128;
        ra.store = L.tq;
        ra.tq_k = c->tq_k;
        ra.tq_v = c->tq_v;
        if ((rc = launch_prompt_rope(s, ra))) return rc;
        PromptAttnArgs aa{};
        aa.q16 = w.q16;
        aa.kc = L.kc;
        aa.vc = L.vc;
        if (L.tq.k_bits) {
            if ((rc = launch_prompt_tq_levels(s, L.tq, (int)base + n, c->nkv, c->hd, L.cap, w.k_levels, w.v_levels))) return rc;
            aa.kc = w.k_levels;
            aa.vc = w.v_levels;
            aa.kn = L.tq.kn;
            aa.vn = L.tq.vn;
            aa.unrot = c->tq_v.signs;
        }
        aa.n = n;
        aa.base = (int)base;
        aa.nq = c->nq;
        aa.nkv = c->nkv;
        aa.hd = c->hd;
        aa.cap = L.cap;
        aa.window = L.window;
        aa.scale = c->attn_scale;
        aa.sinks = L.sinks;
        aa.a = w.a_q;
        aa.asum = prompt_fmt_has_sums(L.wo.fmt) ? w.s_q : nullptr;
        aa.part_o = w.part_o;
        aa.part_ml = w.part_ml;
        aa.nch = prompt_attn_chunks(n, (int)base, c->nq, c->nkv, L.window);
        if ((rc = launch_prompt_attention(s, aa))) return rc;
        sp = prompt_splits(L.wo, n);
        if ((rc = launch_prompt_gemm(s, L.wo, w.a_q, w.s_q, w.partial, nullptr, n, sp, EPI_PARTIAL, H, H))) return rc;
        if (L.n_experts) {
            na.rows16 = w.rows16;
            if ((rc = norm(L.ffn_norm, sp, L.bo, prompt_fmt_has_sums(L.gate_up.fmt) ? L.gate_up : L.router)) || (rc = routed_ffn(L))) return rc;
            na.partial = w.moe_out;
            na.weights = w.route_w;
            sp = L.top_k;
            continue;
        }
        if ((rc = norm(L.ffn_norm, sp, L.bo, L.gate_up)) ||
            (rc = launch_prompt_gemm(s, L.gate_up, w.a_h, w.s_h, w.a_f, prompt_fmt_has_sums(L.down.fmt) ? w.s_f : nullptr, n, 1, EPI_SILU, 0, 0)))
            return rc;
        sp = prompt_splits(L.down, n);
        if ((rc = launch_prompt_gemm(s, L.down, w.a_f, w.s_f, w.partial, nullptr, n, sp, EPI_PARTIAL, H, H))) return rc;
    }
    if (!finish && !logits) return TSV_OK;
    const int m = (n - 1) % 16 + 1, t0 = n - m;
    int tail_splits = sp;
    if (finish) {  // the rows as a drafter head reads them
        na.a = nullptr;
        na.w = na.bias = nullptr;
        na.splits = sp;
        na.slots = na.weights ? 8 : sp;
        if ((rc = launch_prompt_norm(s, na))) return rc;
        tail_splits = 0;
    }
    TSV_HIP(hipMemcpyAsync(c->x, w.x + (size_t)t0 * H, (size_t)m * H * 4, hipMemcpyDeviceToDevice, s));
    const float* tail = na.weights ? w.moe_out + (size_t)t0 * 8 * H : w.partial + (size_t)(t0 / 16) * sp * 16 * H;
    if ((rc = launch_addnorm(s, c->x, tail, tail_splits, H, c->final_norm, c->eps, H, c->xf_a, m, na.weights && tail_splits ? na.weights + (size_t)t0 * 8 : nullptr)))
        return rc;
    if (!logits) return TSV_OK;
    return launch_gemm(s, c->head, c->xf_a, c->logits, c->vp_dev, m, 1, EPI_LOGITS, c->vocab, c->vocab);
}

}  // namespace

// fc's columns pass through the target's buffers, and the head's K / V columns too
int prompt_prime_open(tsv_ctx* h) {
    const tsv_ctx* t = h->mtp.target;
    const LayerW& L = h->layers[0];
    if (!t->prompt.ok || !t->prompt.rows || L.tq.k_bits || !prompt_holds(h->mtp.fc) || !prompt_holds(L.qkv) || !prompt_holds(L.v_only) || h->nq * h->hd % 64 ||
        h->hd > t->hd || 2 * h->nkv * h->hd > std::max(t->hidden, (t->nq + 2 * t->nkv) * t->hd))
        return TSV_OK;
    const size_t a = prompt_a_bytes(t->prompt.rows, 2 * h->hidden), s = prompt_fmt_has_sums(h->mtp.fc.fmt) ? prompt_sum_bytes(t->prompt.rows, 2 * h->hidden) : 0;
    uint8_t* at = nullptr;
    if (hipMalloc((void**)&at, a + s) != hipSuccess) {
        (void)hipGetLastError();  // (no room: sixteen rows at a time)
        return TSV_OK;
    }
    h->allocs.push_back(at);
    TSV_HIP(hipMemsetAsync(at, 0, a + s, h->stream));  // (rows past a pass's last one hold finite values, K padding zeros)
    h->mtp.prompt_a = at;
    h->mtp.prompt_s = s ? at + a : nullptr;
    return TSV_OK;
}

// A prompt leaves nothing in a head but its cache rows, so these are made and nothing behind them: fc, the layer's first norm, the
// K and V columns of its projection, rotation.  In the buffers of the target's pass, on its stream.
int prompt_prime(tsv_ctx* h, const int32_t* next, int n, int64_t position) {
    tsv_ctx* t = h->mtp.target;
    tsv_ctx::Prompt& w = t->prompt;
    hipStream_t s = h->stream;
    const LayerW& L = h->layers[0];
    const int H = h->hidden, q_rows = h->nq * h->hd, kv_n = 2 * h->nkv * h->hd;
    if (position != h->position || position + n > h->max_context) {
        set_error(position != h->position ? "mtp: the rows to prime do not start where the head's cache ends" : "verify: block would write past the KV capacity");
        return TSV_ERR_INVALID;
    }
    for (int i = 0; i < n; i++)
        if (next[i] < 0 || next[i] >= h->vocab) {
            set_error("verify: token id outside the vocabulary");
            return TSV_ERR_INVALID;
        }
    int rc;
    // (from the caller's pageable memory: the runtime has taken its copy when this returns)
    TSV_HIP(hipMemcpyAsync(w.ids, next, (size_t)n * 4, hipMemcpyHostToDevice, s));
    PromptMtpArgs ma{};
    ma.raw = h->embed_raw;
    ma.dtype = h->embed_dtype;
    ma.hidden = H;
    ma.n = n;
    ma.base = (int)position;
    ma.half = h->hd / 2;
    ma.x = w.x;
    ma.ids = w.ids;
    ma.norm_e = h->mtp.norm_e;
    ma.norm_t = t->final_norm;
    ma.norm_h = h->mtp.norm_h;
    ma.freqs = h->freqs;
    ma.eps = h->eps;
    ma.mscale = h->rope_mscale;
    ma.cs = w.cs;
    ma.a = h->mtp.prompt_a;
    ma.asum = h->mtp.prompt_s;
    if ((rc = launch_prompt_mtp_input(s, ma))) return rc;
    int sp = prompt_splits(h->mtp.fc, n);
    if ((rc = launch_prompt_gemm(s, h->mtp.fc, ma.a, ma.asum, w.partial, nullptr, n, sp, EPI_PARTIAL, H, H))) return rc;
    PromptNormArgs na{};
    na.x = w.x;
    na.partial = w.partial;
    na.w = L.attn_norm;
    na.a = w.a_h;
    na.asum = prompt_fmt_has_sums(L.qkv.fmt) || (L.v_only.tiles && prompt_fmt_has_sums(L.v_only.fmt)) ? w.s_h : nullptr;
    na.n = n;
    na.hidden = na.ldp = H;
    na.splits = na.slots = sp;
    na.eps = h->eps;
    if ((rc = launch_prompt_norm(s, na))) return rc;
    TiledW kv = L.qkv;  // the rows behind the q heads'
    kv.tiles += (size_t)(q_rows / TILE_ROWS) * kv.kchunks * fmt_tile_bytes(kv.fmt);
    kv.n_tiles -= q_rows / TILE_ROWS;
    kv.n_rows -= q_rows;
    if (kv.row_scale) kv.row_scale += q_rows;
    sp = prompt_splits(kv, n, L.v_only.tiles ? &L.v_only : nullptr);
    if ((rc = launch_prompt_gemm(s, kv, w.a_h, w.s_h, w.partial, nullptr, n, sp, EPI_PARTIAL, kv_n, kv.n_rows))) return rc;
    if (L.v_only.tiles && (rc = launch_prompt_gemm(s, L.v_only, w.a_h, w.s_h, w.partial + kv.n_rows, nullptr, n, sp, EPI_PARTIAL, kv_n, L.v_only.n_rows)))
        return rc;
    PromptRopeArgs ra{};
    ra.qkv = w.partial;
    ra.splits = sp;
    ra.ldq = kv_n;
    ra.n = n;
    ra.base = (int)position;
    ra.cs = w.cs;
    ra.bias = L.bqkv ? L.bqkv + q_rows : nullptr;
    ra.k_norm = L.k_norm;
    ra.eps = h->eps;
    ra.kc = L.kc;
    ra.vc = L.vc;
    ra.nkv = h->nkv;
    ra.hd = h->hd;
    ra.cap = L.kv_slots;
    ra.paired = L.rope_fused && h->hd == 128;
    if ((rc = launch_prompt_rope(s, ra))) return rc;
    h->position = position + n;
    h->high_water = std::max(h->high_water, h->position);
    h->mtp.own_valid = false;
    return TSV_OK;
}

int enqueue_prompt_pass(tsv_ctx* c, const int32_t* ids, int n, int64_t base, bool finish, bool logits) {
    if (base != c->position) {
        set_error("prefill: start position does not match the KV cursor");
        return TSV_ERR_INVALID;
    }
    if (base + n > c->max_context) {
        set_error("prefill: block would write past the KV capacity");
        return TSV_ERR_INVALID;
    }
    if (n < PROMPT_MIN_ROWS || n > c->prompt.most) {
        set_error("prefill: rows of a prompt pass");
        return TSV_ERR_INVALID;
    }
    for (int i = 0; i < n; i++)
        if (ids[i] < 0 || ids[i] >= c->vocab) {
            set_error("verify: token id outside the vocabulary");
            return TSV_ERR_INVALID;
        }
    int rc;
    // (from the caller's pageable memory: the runtime has taken its copy when this returns)
    TSV_HIP(hipMemcpyAsync(c->prompt.ids, ids, (size_t)n * 4, hipMemcpyHostToDevice, c->stream));
    const int m = (n - 1) % 16 + 1;
    VerifyParams vp;
    if (logits) {  // the last rows are left as a verify pass of their own would leave them
        if ((rc = fill_params(vp, ids + n - m, nullptr, m, base + n - m, c->vocab))) return rc;
        *c->vp_host = vp;
        if ((rc = stage_params(c, &vp, 1, c->vp_dev))) return rc;
    }
    if ((rc = launch_prompt_pass(c, n, base, finish, logits))) return rc;
    c->prompt.passes++;
    c->position = base + n;
    c->high_water = std::max(c->high_water, c->position);
    c->last_m = logits ? m : 0;
    c->last_base = base + n - m;
    if (logits) c->last_shape_known = true;
    c->x_base = base + n - m;
    c->x_rows = finish || logits ? m : 0;
    if (c->mtp_head) c->mtp_head->mtp.own_valid = false;
    return TSV_OK;
}

}  // namespace tsv
