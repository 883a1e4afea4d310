// Device-side acceptance for a speculative round: softmax statistics, greedy / rejection
// sampling acceptance, the residual or bonus draw, and the round's bookkeeping.
//
// Restates on the GPU what the reference runs on the host in f64
// (crates/runtime/src/speculative.rs:694-754,861-879; crates/selection/src/choose.rs:111-338,
// distribution.rs:61-126, derive.rs:19-45) so a round returns a few dozen bytes instead of
// m x vocab fp16 logits.
//
// Arithmetic: every probability is computed in f64 with the reference's operation sequence
//   e = exp(f64(w) - max);  p = e / sum;  weight = pow(p / top, 1/T);  prob = weight / total
// but `sum` and `total` are parallel (fixed-order, deterministic) reductions rather than one
// sequential loop, and the cumulative draw walks rank order (logit descending, index ascending)
// through a 65536-bin histogram keyed by the fp16 logit -- exp is monotone, so rank-by-exp is
// rank-by-logit -- instead of sorting the vocabulary.  Integer outputs can therefore differ
// from the host sequence only when a comparison is within ~1e-13 of flipping; every comparison's
// distance from flipping is folded into `min_margin` so a caller can see that it never was.
// Bin masses are accumulated as 2^-62 fixed point with integer atomics: order independent,
// hence bit-reproducible run to run.
//
// Repetition / presence / frequency penalties (sampled chain and tree rounds, the draft draws) are
// applied per candidate as it is read, from a per-token table of the history (see score_of);
// the kernels are compiled twice, and the variant without penalties is the code it always was.
#include <algorithm>
#include <cstring>

#include "tsv_internal.h"

namespace tsv {

namespace {

constexpr int NSEG = 64;          // index segments per vocabulary row
constexpr int MAX_DIST_ROWS = 32;  // target rows + drafter rows
constexpr int MAX_JOBS = 16;
constexpr int NSUB = 4;  // workgroups per segment in the mass / histogram pass
// A round's rank histograms: [job][p, residual][65536] bins, and behind them the sums of every 64 consecutive ones, which is what the
// draw's cumulative walk reads (8 KB instead of 512 by one workgroup: k_pick 21.0 -> 15.8 us a draw at 128 256 entries)
constexpr int RANK_GROUPS = 65536 / 64;
constexpr double FIX = 4611686018427387904.0;  // 2^62

struct RowStat {
    int32_t cut_key, cut_idx;  // last surviving candidate in rank order (truncation off: 65536, INT_MAX)
    float cut_w;               // its score (penalised rounds: a rank bin can hold several values)
};
__device__ __forceinline__ unsigned long long* rank_groups(unsigned long long* hist) { return hist + (size_t)MAX_JOBS * 2 * 65536; }
struct Cut {
    int32_t key, idx;
    float w, pad;
};

// Scratch layout inside AcceptScratch::stats (doubles):
//   [0, 4*32)                         truncation cut per distribution row (16 bytes each)
//   pmax / psum / ptot partials follow, then the residual pieces and the decisions
struct Layout {
    double* pmax;  // [rows][NSEG]
    double* psum;  // [rows][NSEG][4]
    double* ptot;            // of the reweighted values, which k_row_total leaves in the work rows
    double* segtot;  // [jobs][NSEG * NSUB] residual mass per piece of a segment
    Cut* cut;        // [rows] truncation cut
};
__host__ __device__ inline Layout layout(double* base) {
    Layout l;
    l.pmax = base + 4 * MAX_DIST_ROWS;
    l.psum = l.pmax + MAX_DIST_ROWS * NSEG;
    l.ptot = l.psum + MAX_DIST_ROWS * NSEG * 4;
    l.segtot = l.ptot + MAX_DIST_ROWS * NSEG * 4;
    l.cut = (Cut*)base;
    return l;
}

struct Job {
    int32_t mode;  // 0 none, 1 draw from p, 2 draw from residual(p, q)
    int32_t row_p, row_q;
    double u;
};

struct Decision {
    Job job;
    int32_t accepted, committed, stopped, pad;
    uint64_t draw_step;
    double margin;
};

__device__ __forceinline__ float h2f(uint16_t b) { return (float)__builtin_bit_cast(_Float16, b); }

// crates/selection/src/derive.rs:19-45
__device__ __forceinline__ uint64_t mix64(uint64_t x) {
    x += 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
}
__device__ __forceinline__ double unit_draw(uint64_t seed, uint64_t position) {
    const uint64_t v = mix64(seed ^ (position * 0x9E3779B97F4A7C15ull));
    return (double)(v >> 11) * (1.0 / 9007199254740992.0);
}

// Rank key of an fp16 logit: 0 for the largest value, ascending as the logit falls; +0 and
// -0 share a key (they have the same exp, so the reference breaks their tie by index).
__device__ __forceinline__ uint32_t rank_key(uint16_t b) {
    if (b == 0x8000u) b = 0;
    const uint32_t asc = (b & 0x8000u) ? (uint32_t)(~b & 0xFFFFu) : (uint32_t)(b | 0x8000u);
    return 0xFFFFu - asc;
}

// Where the histogram keeps rank bin `key`: the two low 6-bit fields are swapped, so the 64
// consecutive keys one thread of the cumulative walk owns are 64 words apart and neighbouring
// threads read neighbouring words.
__device__ __forceinline__ uint32_t bin_addr(uint32_t key) {
    return (key & 0xF000u) | ((key & 63u) << 6) | ((key >> 6) & 63u);
}

// (p / top)^(1/T), choose.rs:296-311.  At T = 1 the power is the identity -- the host library's pow returns its
// argument exactly there -- and the device's software pow, the most expensive operation of these kernels, is skipped
// (a branch every lane takes the same way).
__device__ __forceinline__ double temper(double x, double inv_t) { return inv_t == 1.0 ? x : pow(x, inv_t); }

// ---- penalised scores -------------------------------------------------------------------------
// crates/selection/src/penalty.rs:15-82 through choose.rs:138-154: the repetition penalty divides
// (positive) or multiplies (other) the f32 score of every distinct token of the history once; the
// presence / frequency penalties subtract presence + frequency * count for every token of the
// generated suffix.  `pen_cnt[v]` holds, for the history the round started with, bit 31 = seen and
// the low bits = occurrences in the generated suffix; target row i of a chain round adds the i
// proposals committed before it was judged (speculative.rs:694-716: each accepted proposal goes
// through the sink before the next row is shaped) -- in general the tokens on the row's root path,
// which is the same rule for a tree node -- and drafter rows add nothing (speculative.rs:636-641).
//
// A penalised score is an f32 that need not be an fp16 value.  Its rank bin is the bin of the
// largest fp16 value not above it, so bins stay ordered; inside a bin the candidates with a score
// above the bin's own value come first (score descending, index ascending: the few "side"
// candidates), then the candidates exactly on the value in index order.
__device__ __forceinline__ float penalised(const AcceptParams& ap, float w, bool seen, uint32_t gen) {
    if (ap.pen_has_rep && seen) {
        const float a = w > 0.0f ? __fdiv_rn(w, ap.pen_rep) : __fmul_rn(w, ap.pen_rep);
        w = fminf(fmaxf(a, -3.40282347e+38f), 3.40282347e+38f);
    }
    if (ap.pen_has_pf && gen != 0)
        w = __fsub_rn(w, (float)__dadd_rn(ap.pen_presence, __dmul_rn(ap.pen_frequency, (double)gen)));
    return w;
}

template <bool PEN>
__device__ __forceinline__ float score_of(const AcceptParams& ap, int row, int v, uint16_t bits) {
    float w = h2f(bits);
    if constexpr (PEN) {
        const uint32_t c = ap.pen_cnt[v];
        bool seen = (c >> 31) != 0;
        uint32_t gen = c & 0x7FFFFFFFu;
        // the tokens committed on the way to this row: its root path without the root (chain: rows 1..row)
        for (int s = row < ap.m ? row : 0; s > 0; s = ap.parent[s])
            if (ap.feed[s] == v) {
                seen = true;
                gen += 1;
            }
        w = penalised(ap, w, seen, gen);
    }
    return w;
}

// The largest fp16 value not above w (w clamped into the fp16 range first).
__device__ __forceinline__ uint16_t floor16(float w) {
    const float c = fminf(fmaxf(w, -65504.0f), 65504.0f);
    const _Float16 h = (_Float16)c;
    uint16_t b = __builtin_bit_cast(uint16_t, h);
    if ((float)h > c) {
        if ((b & 0x7FFFu) == 0)
            b = 0x8001u;  // below zero: the smallest negative value
        else if (b & 0x8000u)
            b += 1;
        else
            b -= 1;
    }
    return b;
}

template <bool PEN>
__device__ __forceinline__ uint32_t key_of(float w, uint16_t bits) {
    if constexpr (PEN) return rank_key(floor16(w));
    return rank_key(bits);
}

// Whether candidate v is inside the row's truncated candidate set: the set is a prefix of the rank order (logit descending, index
// ascending), so it is described by its last member.
template <bool PEN>
__device__ __forceinline__ bool survives_w(float w, int key, int v, const RowStat& s) {
    if constexpr (PEN)
        return key < s.cut_key || (key == s.cut_key && (w > s.cut_w || (w == s.cut_w && v <= s.cut_idx)));
    return key < s.cut_key || (key == s.cut_key && v <= s.cut_idx);
}

template <typename T>
__device__ __forceinline__ T shfl_xor_t(T v, int o) {
    static_assert(sizeof(T) == 8, "64-bit only");
    uint64_t u = __builtin_bit_cast(uint64_t, v);
    uint32_t lo = __shfl_xor((uint32_t)u, o), hi = __shfl_xor((uint32_t)(u >> 32), o);
    return __builtin_bit_cast(T, ((uint64_t)hi << 32) | lo);
}

// Deterministic block sum: xor-butterfly inside a wave, then the waves in index order.
__device__ double block_sum_f64(double v, double* red) {
    for (int o = 32; o > 0; o >>= 1) v += shfl_xor_t(v, o);
    const int wave = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[wave] = v;
    __syncthreads();
    double t = 0.0;
    for (int i = 0; i < nw; i++) t += red[i];
    return t;
}

__device__ __forceinline__ const uint16_t* row_ptr(const uint16_t* target, const uint16_t* draft, int m,
                                                   int vocab, int row) {
    return row < m ? target + (long)row * vocab : draft + (long)(row - m) * vocab;
}

// Wave-wide fold of a row's NSEG (= wave size) partials: lane s loads segment s, an xor
// butterfly combines them.  Both lanes of a pair add the same two operands, so every lane ends
// with the same bits, and every kernel that needs a row's statistics gets them this way.
__device__ __forceinline__ double wave_max_f64(double v) {
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, shfl_xor_t(v, o));
    return v;
}
__device__ __forceinline__ double wave_sum_f64(double v) {
    for (int o = 32; o > 0; o >>= 1) v += shfl_xor_t(v, o);
    return v;
}
static_assert(NSEG == 64, "one lane per segment");

// ---- statistics, three short passes over every distribution row -------------------------
template <bool PEN>
__global__ __launch_bounds__(256) void k_row_max(const uint16_t* target, const uint16_t* draft, int m,
                                                 int vocab, double* scratch, int32_t* err,
                                                 unsigned long long* hist, int jobs,
                                                 const AcceptParams* app, unsigned long long* tmass, uint32_t* tcount) {
    __shared__ double red[4];
    const int row = blockIdx.y, seg = blockIdx.x;
    {
        // the rank histograms of this round's draws start from zero: every workgroup clears a slice
        const int nwg = gridDim.x * gridDim.y, wg = blockIdx.y * gridDim.x + blockIdx.x;
        auto clear = [&](unsigned long long* at, int words) {
            const int per = (words + nwg - 1) / nwg, h0 = wg * per, h1 = min(h0 + per, words);
            for (int i = h0 + threadIdx.x; i < h1; i += 256) at[i] = 0;
        };
        clear(hist, jobs * 2 * 65536);
        clear(rank_groups(hist), jobs * 2 * RANK_GROUPS);
        // and so do the row's truncation histograms, where there will be a cut
        if (tmass) {
            const int i = seg * 256 + threadIdx.x;
            if (i < TRUNC_WORDS) tmass[row * TRUNC_WORDS + i] = 0, tcount[row * TRUNC_WORDS + i] = 0;
        }
    }
    const uint16_t* p = row_ptr(target, draft, m, vocab, row);
    const int per = (vocab + NSEG - 1) / NSEG, v0 = seg * per, v1 = min(v0 + per, vocab);
    float mx = -INFINITY;
    bool bad = false;
    bool low = false;
    for (int v = v0 + threadIdx.x; v < v1; v += 256) {
        const uint16_t b = p[v];
        bad |= (b & 0x7C00u) == 0x7C00u;
        if constexpr (PEN) {
            const float w = score_of<true>(*app, row, v, b);
            low |= !(w >= -65504.0f);
            mx = fmaxf(mx, w);
        } else {
            mx = fmaxf(mx, h2f(b));
        }
    }
    if (bad) atomicOr(err, 1);
    if (low) atomicOr(err, 4);  // a penalised score below every fp16 value: no rank bin to put it in
    double d = (double)mx;
    for (int o = 32; o > 0; o >>= 1) d = fmax(d, shfl_xor_t(d, o));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = d;
    __syncthreads();
    if (threadIdx.x == 0) {
        Layout L = layout(scratch);
        L.pmax[row * NSEG + seg] = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
        if (seg == 0) L.cut[row] = Cut{65536, 0x7FFFFFFF, 0.f, 0.f};  // no truncation until a cut is computed
    }
}

// The sum of value(v) over a segment's [v0, v1): 256 chains, chain t every 256th value from v0 + t on, folded over the 64 lanes of a wave
// and left as four numbers (fold_row adds them up).  A thread to a chain; or, SPLIT, the four folds are workgroups of their own
// (blockIdx.z) whose four waves make the values of the chains (an exp, and a pow with it, in f64 each) a quarter each.  The same bits.
// 64 segments of a single row, a draft step's, leave three quarters of the chip idle otherwise: k_row_total 10.6 -> 4.9 us at
// 128 256 entries and T = 0.8.
template <bool SPLIT, class Value>
__device__ __forceinline__ void chained_sum(int v0, int v1, double* out, Value&& value) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, fold = SPLIT ? blockIdx.z : wave;
    double acc = 0.0;
    if (SPLIT) {
        __shared__ double vals[8][64];
        for (int at = v0 + 64 * fold + lane; at - lane < v1; at += 8 * 256) {
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const int v = at + (wave + 4 * i) * 256;
                if (v < v1) vals[wave + 4 * i][lane] = value(v);
            }
            __syncthreads();
            if (wave == 0)
                for (int i = 0; i < 8 && at + i * 256 < v1; i++) acc += vals[i][lane];
            __syncthreads();
        }
    } else {
        for (int v = v0 + threadIdx.x; v < v1; v += 256) acc += value(v);
    }
    for (int o = 32; o > 0; o >>= 1) acc += shfl_xor_t(acc, o);
    if (lane == 0 && (!SPLIT || wave == 0)) out[fold] = acc;
}
// Called by whole waves: the row's sum out of its segments' four folds each, identical in every lane
__device__ __forceinline__ double fold_row(const double* folds, int row) {
    const double* f = folds + ((size_t)row * NSEG + (threadIdx.x & 63)) * 4;
    const double a = f[0], b = f[1], c = f[2], d = f[3];
    return wave_sum_f64(((a + b) + c) + d);
}

template <bool PEN, bool SPLIT>
__global__ __launch_bounds__(256) void k_row_sum(const uint16_t* target, const uint16_t* draft, int m,
                                                 int vocab, double* scratch, const AcceptParams* app) {
    const int row = blockIdx.y, seg = blockIdx.x;
    Layout L = layout(scratch);
    const double mx = wave_max_f64(L.pmax[row * NSEG + (threadIdx.x & 63)]);
    const uint16_t* p = row_ptr(target, draft, m, vocab, row);
    const int per = (vocab + NSEG - 1) / NSEG, v0 = seg * per, v1 = min(v0 + per, vocab);
    chained_sum<SPLIT>(v0, v1, L.psum + ((size_t)row * NSEG + seg) * 4, [&](int v) {
        float w;
        if constexpr (PEN)
            w = score_of<true>(*app, row, v, p[v]);
        else
            w = h2f(p[v]);
        return exp((double)w - mx);
    });
}

// Also leaves the reweighted values (zero: not a candidate) in work row slot0 + row * slot_step: whoever needs a probability
// divides one by the row's total.  (Every later kernel made them again, an exp and a pow in f64 each: k_mass_hist 13.0 -> 5.3 us; a
// tree's rows took a kernel of their own for it, 17.9 us, for 4 that this one has become slower by with 32 rows.)
template <bool PEN, bool SPLIT>
__global__ __launch_bounds__(256) void k_row_total(const uint16_t* target, const uint16_t* draft, int m,
                                                   int vocab, double* scratch, double inv_t,
                                                   const AcceptParams* app, double* work, int slot0, int slot_step) {
    const int row = blockIdx.y, seg = blockIdx.x;
    Layout L = layout(scratch);
    const double mx = wave_max_f64(L.pmax[row * NSEG + (threadIdx.x & 63)]);
    const double sum = fold_row(L.psum, row);
    const double top = 1.0 / sum;  // the arg-max candidate has e == exp(0) == 1
    const uint16_t* p = row_ptr(target, draft, m, vocab, row);
    const int per = (vocab + NSEG - 1) / NSEG, v0 = seg * per, v1 = min(v0 + per, vocab);
    RowStat cs;
    cs.cut_key = L.cut[row].key;
    cs.cut_idx = L.cut[row].idx;
    cs.cut_w = L.cut[row].w;
    double* out = work + (size_t)(slot0 + row * slot_step) * vocab;
    chained_sum<SPLIT>(v0, v1, L.ptot + ((size_t)row * NSEG + seg) * 4, [&](int v) {
        const uint16_t b = p[v];
        const float w = score_of<PEN>(*app, row, v, b);
        double t = 0.0;
        if (survives_w<PEN>(w, (int)key_of<PEN>(w, b), v, cs)) {
            const double e = exp((double)w - mx);
            if (!PEN || !app->has_min_p || !(e < app->min_p)) t = temper((e / sum) / top, inv_t);
        }
        out[v] = t;
        return t;
    });
}

// Called by whole waves: the total of `row`, identical in every lane (1 where there is no candidate: its values are zeros).
__device__ __forceinline__ double row_total(const Layout& L, int row) {
    const double t = fold_row(L.ptot, row);
    return t > 0.0 ? t : 1.0;
}

__device__ __forceinline__ void fold_margin(double& margin, double a, double b) {
    const double scale = fmax(fabs(a), fabs(b));
    if (scale == 0.0) return;  // two exact zeros (a candidate outside both truncated sets): nothing can flip
    margin = fmin(margin, fabs(a - b) / scale);
}

// TokenSink::commit restricted to what a token-id interface can see
// (crates/runtime/src/token_sink.rs:64-124): 0 continue, 1 stop token, 2 budget.
__device__ int sink_commit(const AcceptParams& ap, int32_t token, uint64_t& generated, int32_t& committed) {
    generated += 1;
    for (int i = 0; i < ap.n_stop; i++)
        if (ap.stop_tokens[i] == token) return 1;
    if (ap.max_new_tokens != 0 && generated >= ap.max_new_tokens) return 2;
    committed += 1;
    return 0;
}

// speculative.rs:694-754: the sequential walk over the proposals of a sampled chain round.
// pxs / qxs: p_i(x_i) and q_i(x_i) of every proposal, computed by the caller in parallel (one lane
// per proposal: an f64 exp + pow chain per value is long for a single thread to walk k times).
__device__ Decision decide_chain_sampled(const AcceptParams& ap, const double* pxs, const double* qxs) {
    Decision d;
    d.job.mode = 0;
    d.job.row_p = d.job.row_q = 0;
    d.job.u = 0.0;
    d.accepted = d.committed = d.stopped = d.pad = 0;
    d.margin = 1.0;
    uint64_t ds = ap.draw_step, gen = ap.generated;
    int reject = -1;
    for (int i = 0; i < ap.k; i++) {
        const int32_t x = ap.feed[i + 1];
        const double px = pxs[i], qx = qxs[i];
        const double r = unit_draw(ap.seed, ds);
        ds += 1;
        fold_margin(d.margin, r * qx, px);
        if (r * qx <= px) {
            d.accepted += 1;
            if ((d.stopped = sink_commit(ap, x, gen, d.committed))) break;
        } else {
            reject = i;
            break;
        }
    }
    if (!d.stopped) {
        d.job.u = unit_draw(ap.seed, ds);
        ds += 1;
        if (reject >= 0) {
            d.job.mode = 2;
            d.job.row_p = reject;
            d.job.row_q = ap.m + reject;
        } else {
            d.job.mode = 1;
            d.job.row_p = d.accepted;
        }
    }
    d.draw_step = ds;
    return d;
}

// ---- masses + rank histogram --------------------------------------------------------------
// kind 0: the job comes out of the chain decision (every workgroup re-derives it: a few
// dozen f64 ops).  kind 1: jobs are "draw from drafter row j at position draw_step + j".
template <bool PEN>
__global__ __launch_bounds__(256) void k_mass_hist(const uint16_t* target, const uint16_t* draft,
                                                   const AcceptParams* app, double* scratch, double* work,
                                                   unsigned long long* hist, Decision* dec_out, int kind) {
    __shared__ Decision dec;
    __shared__ double red[4];
    __shared__ double totals[MAX_DIST_ROWS];
    __shared__ double s_px[TSV_MAX_ROWS], s_qx[TSV_MAX_ROWS];
    __shared__ unsigned long long groups[2][RANK_GROUPS];
    const AcceptParams& ap = *app;
    const int seg = blockIdx.x, jobi = blockIdx.y, sub = blockIdx.z;
    Layout L = layout(scratch);
    // the reweighted values (k_row_total): of a chain round in the work rows behind its draw's two, of draft draw j beside its own
    auto weights = [&](int row) { return work + (size_t)(kind == 0 ? 2 + row : 2 * row + 1) * ap.vocab; };
    if (kind == 0 && (int)threadIdx.x < ap.k) {
        const int i = threadIdx.x;
        const int32_t x = ap.feed[i + 1];
        s_px[i] = weights(i)[x];
        s_qx[i] = weights(ap.m + i)[x];
    }
    {
        // every row's total, one wave per row at a time
        const int rows = kind == 0 ? ap.m + ap.k : ap.k;
        for (int r = threadIdx.x >> 6; r < rows; r += 4) {
            const double t = row_total(L, r);
            if ((threadIdx.x & 63) == 0) totals[r] = t;
        }
    }
    for (int i = threadIdx.x; i < RANK_GROUPS; i += 256) groups[0][i] = groups[1][i] = 0;
    __syncthreads();
    if (kind == 0 && (int)threadIdx.x < ap.k) {
        const int i = threadIdx.x;
        s_px[i] /= totals[i];
        s_qx[i] /= totals[ap.m + i];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        if (kind == 0) {
            dec = decide_chain_sampled(ap, s_px, s_qx);
        } else {
            dec.job.mode = 1;
            dec.job.row_p = ap.m + jobi;
            dec.job.row_q = 0;
            dec.job.u = unit_draw(ap.seed, ap.draw_step + jobi);
            dec.accepted = dec.committed = dec.stopped = 0;
            dec.draw_step = ap.draw_step;
            dec.margin = 1.0;
        }
        if (seg == 0 && sub == 0) dec_out[jobi] = dec;
    }
    __syncthreads();
    const Job job = dec.job;
    if (job.mode == 0) return;
    const int vocab = ap.vocab, row_q = job.mode == 2 ? job.row_q : job.row_p;
    const double total_p = totals[job.row_p], total_q = totals[row_q];
    const uint16_t* lp = row_ptr(target, draft, ap.m, vocab, job.row_p);
    const double *tp = weights(job.row_p), *tq = weights(row_q);
    double* wp = work + (long)jobi * 2 * vocab;
    double* wr = wp + vocab;
    unsigned long long* hp = hist + (long)jobi * 2 * 65536;
    unsigned long long* hr = hp + 65536;
    const int per = (vocab + NSEG - 1) / NSEG, v0 = seg * per, v1 = min(v0 + per, vocab);
    double racc = 0.0;
    for (int v = v0 + sub * 256 + threadIdx.x; v < v1; v += 256 * NSUB) {
        const uint16_t b = lp[v];
        const uint32_t rk = key_of<PEN>(score_of<PEN>(ap, job.row_p, v, b), b);
        const double pv = tp[v] / total_p;
        const uint32_t key = bin_addr(rk);
        wp[v] = pv;
        auto add = [&](unsigned long long* bins, unsigned long long* sums, double mass) {
            const unsigned long long fixed = (unsigned long long)(mass * FIX);
            if (!fixed) return;
            atomicAdd(bins + key, fixed);
            atomicAdd(sums + (rk >> 6), fixed);
        };
        add(hp, groups[0], pv);
        if (job.mode == 2) {
            const double mv = fmax(pv - tq[v] / total_q, 0.0);
            wr[v] = mv;
            racc += mv;
            add(hr, groups[1], mv);
        }
    }
    __syncthreads();
    unsigned long long* gp = rank_groups(hist) + (long)jobi * 2 * RANK_GROUPS;
    for (int i = threadIdx.x; i < 2 * RANK_GROUPS; i += 256) {
        const unsigned long long s = groups[i / RANK_GROUPS][i % RANK_GROUPS];
        if (s) atomicAdd(gp + i, s);
    }
    if (job.mode == 2) {
        racc = block_sum_f64(racc, red);
        if (threadIdx.x == 0) L.segtot[(jobi * NSEG + seg) * NSUB + sub] = racc;
    }
}

// Calls on_match(v) for every index v in [v0, v1) whose logit bits are `want` (or -0 when the
// bin is the zero bin), eight keys per 16-byte load when the row allows it.
template <class Fn>
__device__ __forceinline__ void scan_chunk(const uint16_t* lp, int v0, int v1, uint32_t want, bool zero_bin, bool vec,
                                           Fn&& on_match) {
    // sixty-four keys at a time while the range lasts: the eight loads are in flight together (the loop below, one
    // load per turn with the matches' own loads behind it, waits out a memory round trip per eight keys)
    if (vec) {
        for (; v0 + 64 <= v1; v0 += 64) {
            uint4 q[8];
#pragma unroll
            for (int i = 0; i < 8; i++) q[i] = *(const uint4*)(lp + v0 + 8 * i);
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const uint32_t w[4] = {q[i].x, q[i].y, q[i].z, q[i].w};
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const uint32_t bits = (w[j >> 1] >> (16 * (j & 1))) & 0xFFFFu;
                    if (bits == want || (zero_bin && bits == 0x8000u)) on_match(v0 + 8 * i + j);
                }
            }
        }
    }
    for (int g = v0; g < v1; g += 8) {
        uint32_t w[4];
        if (vec && g + 8 <= v1) {
            const uint4 q = *(const uint4*)(lp + g);
            w[0] = q.x;
            w[1] = q.y;
            w[2] = q.z;
            w[3] = q.w;
        } else {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint32_t lo = g + 2 * j < v1 ? lp[g + 2 * j] : (want ^ 0x4000u);
                const uint32_t hi = g + 2 * j + 1 < v1 ? lp[g + 2 * j + 1] : (want ^ 0x4000u);
                w[j] = lo | (hi << 16);
            }
        }
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const uint32_t bits = (w[j >> 1] >> (16 * (j & 1))) & 0xFFFFu;
            if (bits == want || (zero_bin && bits == 0x8000u)) on_match(g + j);
        }
    }
}

// ---- truncation of the candidate set (top-k, top-p, min-p) ---------------------------------
// choose.rs:111-228 / truncation.rs:79-236: candidates are ranked by softmax mass descending, ties
// by ascending index; top-k keeps the first k, top-p the shortest prefix whose cumulative
// `e / sum` reaches top_p, min-p those with e >= min_p * e_top.  All three keep a PREFIX of the
// rank order, so the surviving set is described by its last member (rank bin, index); it is found
// from per-row histograms (candidates, fixed-point mass) instead of a sort, and the one bin the cut falls into is resolved in index
// order.  The histograms have two levels: every group of 64 consecutive rank bins, then the bins of the groups that hold
// a cut.  A group's sums come together in LDS, and few entries fall into the second level, where a histogram of all 65536 bins was
// two atomics on memory for every entry, and 5 MB to clear and to read again (seven rows of 128 256 entries: cleared, filled and cut in 5.3 + 52.5 +
// 45.5 us; a penalised round of four rows with top-k and top-p 892 -> 838).  The sums are of integers: their order does not matter.
__device__ __forceinline__ unsigned long long mass_of(float w, double mx, double sum) { return (unsigned long long)((exp((double)w - mx) / sum) * FIX); }

template <bool PEN>
__global__ __launch_bounds__(256) void k_trunc_groups(const uint16_t* target, const uint16_t* draft, int m, int vocab,
                                                      double* scratch, unsigned long long* tmass, uint32_t* tcount,
                                                      int want_mass, const AcceptParams* app) {
    __shared__ unsigned long long mass_sum[RANK_GROUPS];
    __shared__ uint32_t count[RANK_GROUPS];
    const int row = blockIdx.y, seg = blockIdx.x, lane = threadIdx.x & 63;
    Layout L = layout(scratch);
    const double mx = wave_max_f64(L.pmax[row * NSEG + lane]);
    const double sum = fold_row(L.psum, row);
    const uint16_t* p = row_ptr(target, draft, m, vocab, row);
    const int per = (vocab + NSEG - 1) / NSEG, v0 = seg * per, v1 = min(v0 + per, vocab);
    for (int i = threadIdx.x; i < RANK_GROUPS; i += 256) mass_sum[i] = 0, count[i] = 0;
    __syncthreads();
    for (int v = v0 + threadIdx.x; v < v1; v += 256) {
        const uint16_t b = p[v];
        const float w = score_of<PEN>(*app, row, v, b);
        const uint32_t key = key_of<PEN>(w, b), group = key >> 6;
        const unsigned long long mass = want_mass ? mass_of(w, mx, sum) : 0;
        // a run of equal logits (a flat row) would serialise on one address: one lane adds for all
        const uint32_t first = __builtin_amdgcn_readfirstlane(key);
        const unsigned long long active = __ballot(1);
        if (!PEN && __ballot(key == first) == active) {  // (equal keys are equal masses only without penalties)
            if (lane == (int)__builtin_ctzll(active)) {
                const int n = __builtin_popcountll(active);
                atomicAdd(count + group, (uint32_t)n);
                if (want_mass) atomicAdd(mass_sum + group, mass * (unsigned long long)n);
            }
        } else {
            atomicAdd(count + group, 1u);
            if (want_mass && mass) atomicAdd(mass_sum + group, mass);
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < RANK_GROUPS; i += 256) {
        if (count[i]) atomicAdd(tcount + (size_t)row * TRUNC_WORDS + i, count[i]);
        if (mass_sum[i]) atomicAdd(tmass + (size_t)row * TRUNC_WORDS + i, mass_sum[i]);
    }
}

// Exclusive prefix of a 64-bit value over the 64 NW threads of a workgroup; *total gets the sum.
template <int NW>
__device__ unsigned long long block_scan_u64(unsigned long long loc, unsigned long long* wsum,
                                             unsigned long long* total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    unsigned long long inc = loc;
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t lo = __shfl_up((uint32_t)inc, o), hi = __shfl_up((uint32_t)(inc >> 32), o);
        const unsigned long long up = ((unsigned long long)hi << 32) | lo;
        if (lane >= o) inc += up;
    }
    __syncthreads();
    if (lane == 63) wsum[wave] = inc;
    __syncthreads();
    unsigned long long wbase = 0, t = 0;
    for (int i = 0; i < NW; i++) {
        if (i < wave) wbase += wsum[i];
        t += wsum[i];
    }
    *total = t;
    return wbase + inc - loc;
}

// The group in which a running sum over the groups reaches `target` (sum before < target <= sum with it), found by 64 NW threads; -1 where the sums
// end below it.  Thread t brings the sums of groups t * PER ..; *before: the sum before the group, *all: over every group.
// `wsum`, `found`, `at`: LDS.
template <int NW, int PER>
__device__ __forceinline__ int group_reaching(const unsigned long long (&v)[PER], unsigned long long target, unsigned long long* wsum, int* found,
                                              unsigned long long* at, unsigned long long* before, unsigned long long* all) {
    unsigned long long loc = 0;
#pragma unroll
    for (int i = 0; i < PER; i++) loc += v[i];
    if (threadIdx.x == 0) *found = -1;
    unsigned long long c = block_scan_u64<NW>(loc, wsum, all);
#pragma unroll
    for (int i = 0; i < PER; i++) {
        if (c < target && target <= c + v[i]) {
            *found = threadIdx.x * PER + i;
            *at = c;
        }
        c += v[i];
    }
    __syncthreads();
    *before = *at;
    return *found;
}

// The second level: candidates and mass of the bins of the groups that hold the cuts, which every workgroup looks for again.
template <bool PEN>
__global__ __launch_bounds__(256) void k_trunc_bins(const uint16_t* target, const uint16_t* draft, int m, int vocab, double* scratch,
                                                    unsigned long long* tmass, uint32_t* tcount, const AcceptParams* app) {
    __shared__ unsigned long long wsum[4], at, mass_sum[64];
    __shared__ uint32_t count[2][64];
    __shared__ int found;
    const AcceptParams& ap = *app;
    const int row = blockIdx.y, seg = blockIdx.x, lane = threadIdx.x & 63, tid = threadIdx.x;
    Layout L = layout(scratch);
    unsigned long long* const gm = tmass + (size_t)row * TRUNC_WORDS;
    uint32_t* const gc = tcount + (size_t)row * TRUNC_WORDS;
    const double mx = wave_max_f64(L.pmax[row * NSEG + lane]);
    const double sum = fold_row(L.psum, row);
    if (tid < 64) mass_sum[tid] = 0, count[0][tid] = count[1][tid] = 0;
    static_assert(RANK_GROUPS == 4 * 256, "four groups to a thread");
    unsigned long long v[4], before, all;
    int group_k = -1, group_p = -1;
    if (ap.top_k > 0) {
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = gc[4 * tid + i];
        group_k = group_reaching<4, 4>(v, (unsigned long long)ap.top_k, wsum, &found, &at, &before, &all);
        __syncthreads();
    }
    if (ap.has_top_p) {
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = gm[4 * tid + i];
        group_p = group_reaching<4, 4>(v, (unsigned long long)(ap.top_p * FIX), wsum, &found, &at, &before, &all);
    }
    if (group_k < 0 && group_p < 0) return;
    __syncthreads();
    const uint16_t* p = row_ptr(target, draft, m, vocab, row);
    const int per = (vocab + NSEG - 1) / NSEG, v0 = seg * per, v1 = min(v0 + per, vocab);
    for (int i = v0 + tid; i < v1; i += 256) {
        const uint16_t b = p[i];
        const float w = score_of<PEN>(ap, row, i, b);
        const uint32_t key = key_of<PEN>(w, b);
        const int group = (int)(key >> 6), bin = (int)(key & 63u);
        if (group == group_k) atomicAdd(&count[0][bin], 1u);
        if (group == group_p) {
            atomicAdd(&count[1][bin], 1u);
            atomicAdd(&mass_sum[bin], mass_of(w, mx, sum));
        }
    }
    __syncthreads();
    if (tid >= 64) return;
    if (count[0][tid]) atomicAdd(gc + RANK_GROUPS + tid, count[0][tid]);
    if (count[1][tid]) atomicAdd(gc + RANK_GROUPS + 64 + tid, count[1][tid]);
    if (mass_sum[tid]) atomicAdd(gm + RANK_GROUPS + 64 + tid, mass_sum[tid]);
}

// fp16 bits whose rank key is `key` (inverse of rank_key; the zero bin maps to +0)
__device__ __forceinline__ uint32_t key_bits(int key) {
    const uint32_t asc = 0xFFFFu - (uint32_t)key;
    return (asc & 0x8000u) ? (asc & 0x7FFFu) : (~asc & 0xFFFFu);
}

// Calls fn(v) for the tokens of a row's root path without the root (the ones its penalties count besides the history), from
// as many lanes, a repeated token once.
template <class Fn>
__device__ __forceinline__ void on_path_tokens(const AcceptParams& ap, int row, Fn&& fn) {
    if (row >= ap.m || threadIdx.x >= TSV_MAX_ROWS) return;
    int at = row;
    for (int i = threadIdx.x; i > 0 && at > 0; i--) at = ap.parent[at];
    if (at <= 0) return;
    const int v = ap.feed[at];
    for (int s = row; s != at; s = ap.parent[s])
        if (ap.feed[s] == v) return;
    fn(v);
}

// The candidates of rank bin `bin` that sit exactly on the bin's value, found by a workgroup of 1024 threads: the row (and with
// penalties the history's table) is read ONCE, coalesced -- neighbouring lanes take neighbouring groups of eight entries, where
// a lane reading its own contiguous chunk touches 64 cache lines per load -- and leaves one bit per entry in LDS; each thread
// then walks the bits of its own contiguous chunk of `groups` bytes, in the index order the sums are defined in.
// Penalised: an entry that no penalty touches is found by its fp16 bits like any other; the few touched ones are noted in
// registers and scored afterwards, each lane its own (scoring inside the sweep would have every wave do it for every group).
// 128 256 entries, 2000 tokens of history: k_pick 192 -> 43 us; k_trunc_cut, seven rows, 281 -> 46 us: they read
// entry by entry and walked the root path for each.
constexpr int PICK_MASK_GROUPS = 32;  // groups of eight entries per thread the match mask holds: vocabularies to 262 144
__device__ __forceinline__ int mask_groups(int vocab) { return ((vocab + 1023) / 1024 + 7) >> 3; }
// `ahead`: the first of a lane's groups, asked for before the bin was known (row_ahead).
constexpr int MASK_AHEAD = 16;
struct RowAhead {
    uint4 q[MASK_AHEAD];
};
__device__ __forceinline__ RowAhead row_ahead(const uint16_t* lp, int vocab) {
    RowAhead a;
    const int groups = mask_groups(vocab), whole = vocab >> 3;
#pragma unroll
    for (int j = 0; j < MASK_AHEAD; j++) {
        const int g = j * 1024 + threadIdx.x;
        a.q[j] = *(const uint4*)(lp + (j < groups && g < whole ? (long)g * 8 : 0));
    }
    return a;
}
template <bool PEN>
__device__ __forceinline__ void build_mask(const AcceptParams& ap, int row, const uint16_t* lp, int bin, uint8_t* mask8, const RowAhead& ahead) {
    const int tid = threadIdx.x, vocab = ap.vocab, groups = mask_groups(vocab);
    const uint32_t want = key_bits(bin);
    const bool zero_bin = want == 0;
    const float g16 = h2f((uint16_t)want);
    const int whole = vocab >> 3;  // groups of eight entries that lie wholly inside the row
    constexpr int B = MASK_AHEAD;  // loads of the row in flight per lane; a group past the last whole one reads group 0 and is discarded
    const uint8_t* const seen = PEN ? (const uint8_t*)pen_seen(ap.pen_cnt, vocab) : nullptr;  // a group's eight bits
    auto take = [&](int g0, const uint4 (&q)[B]) {
        uint32_t pen[PEN ? B : 1];
        if constexpr (PEN) {
#pragma unroll
            for (int j = 0; j < B; j++) {
                const int g = (g0 + j) * 1024 + tid;
                pen[j] = seen[g0 + j < groups && g < whole ? g : 0];
            }
        }
        uint32_t touched[PEN ? B / 4 : 1] = {};
#pragma unroll
        for (int j = 0; j < B; j++) {
            const int g = (g0 + j) * 1024 + tid;
            const uint32_t t[4] = {q[j].x, q[j].y, q[j].z, q[j].w};
            uint32_t m = 0;
#pragma unroll
            for (int h = 0; h < 8; h++) {
                const uint32_t bits = (t[h >> 1] >> (16 * (h & 1))) & 0xFFFFu;
                m |= (uint32_t)(bits == want || (zero_bin && bits == 0x8000u)) << h;
            }
            if constexpr (PEN) {
                m &= ~pen[j];
                if (g0 + j < groups && g < whole) touched[j >> 2] |= pen[j] << (8 * (j & 3));
            }
            if (g0 + j < groups) mask8[g] = g < whole ? (uint8_t)m : (uint8_t)0;
        }
        if constexpr (PEN) {
#pragma unroll
            for (int w = 0; w < B / 4; w++)
                for (uint32_t left = touched[w]; left; left &= left - 1) {
                    const int at = __ffs(left) - 1, g = (g0 + 4 * w + (at >> 3)) * 1024 + tid, v = g * 8 + (at & 7);
                    const uint32_t cnt = ap.pen_cnt[v];
                    if (penalised(ap, h2f(lp[v]), (cnt >> 31) != 0, cnt & 0x7FFFFFFFu) == g16) mask8[g] |= (uint8_t)(1u << (at & 7));
                }
        }
    };
    take(0, ahead.q);
    for (int g0 = B; g0 < groups; g0 += B) {
        uint4 q[B];
#pragma unroll
        for (int j = 0; j < B; j++) {
            const int g = (g0 + j) * 1024 + tid;
            q[j] = *(const uint4*)(lp + (g0 + j < groups && g < whole ? (long)g * 8 : 0));
        }
        take(g0, q);
    }
    if ((vocab & 7) && whole < groups * 1024 && tid == (whole & 1023)) {  // the row's last, partial group
        uint32_t m = 0;
        for (int h = 0; h < (vocab & 7); h++) {
            const int v = whole * 8 + h;
            bool on = lp[v] == want || (zero_bin && lp[v] == 0x8000u);
            if constexpr (PEN) on = score_of<true>(ap, row, v, lp[v]) == g16;
            m |= (uint32_t)on << h;
        }
        mask8[whole] = (uint8_t)m;
    }
    __syncthreads();
    if constexpr (PEN) {
        on_path_tokens(ap, row, [&](int v) {  // their penalties count more than the table says
            uint32_t* const word = (uint32_t*)mask8 + (v >> 5);
            if (score_of<true>(ap, row, v, lp[v]) == g16) atomicOr(word, 1u << (v & 31));
            else atomicAnd(word, ~(1u << (v & 31)));
        });
        __syncthreads();
    }
}
// the entries of thread tid's chunk whose bit is set, ascending
template <class Fn>
__device__ __forceinline__ void walk_mask(const uint8_t* mask8, int groups, Fn&& on_match) {
    const uint8_t* mine = mask8 + threadIdx.x * groups;
    int k = 0;
    if ((groups & 15) == 0) {  // sixteen bytes at a time, nearly all of them zero
        for (; k < groups; k += 16) {
            const uint4 q = *(const uint4*)(mine + k);
            if (!(q.x | q.y | q.z | q.w)) continue;
            const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
            for (int i = 0; i < 4; i++)
                for (uint32_t m = w[i]; m; m &= m - 1) on_match((threadIdx.x * groups + k) * 8 + 32 * i + (__ffs(m) - 1));
        }
        return;
    }
    for (; k < groups; k++)
        for (uint32_t m = mine[k]; m; m &= m - 1) on_match((threadIdx.x * groups + k) * 8 + (__ffs(m) - 1));
}

// The same candidates over [v0, v1) without a mask, for rows that are not 16-byte aligned or longer than it holds.
template <bool PEN, class Fn>
__device__ __forceinline__ void scan_on(const AcceptParams& ap, int row, const uint16_t* lp, int v0, int v1, int bin,
                                        bool vec, Fn&& on_match) {
    const uint32_t want = key_bits(bin);
    if constexpr (PEN) {
        const float g = h2f((uint16_t)want);
        for (int v = v0; v < v1; v++)
            if (score_of<true>(ap, row, v, lp[v]) == g) on_match(v);
    } else {
        scan_chunk(lp, v0, v1, want, want == 0, vec, on_match);
    }
}

// Penalised rounds, whole workgroup of 1024 threads: the candidates of `row` whose score falls
// into rank bin `bin` without being the bin's own value, ordered by score descending, index
// ascending, in sorted[0 .. n).  They precede the bin's on-value candidates in rank order.
constexpr int SIDE_CAP = 1024;
struct SideEnt {
    float w;
    int32_t v;
};
__device__ __forceinline__ int collect_side(const AcceptParams& ap, int row, const uint16_t* lp, int bin, SideEnt* raw,
                            SideEnt* sorted, int* counter, int32_t* err) {
    const int tid = threadIdx.x;
    const float g = h2f((uint16_t)key_bits(bin));
    __syncthreads();
    if (tid == 0) *counter = 0;
    __syncthreads();
    // (an untouched score is an fp16 value: on its bin's value)
    auto look = [&](int v, float w) {
        if (w != g && (int)rank_key(floor16(w)) == bin) {
            const int i = atomicAdd(counter, 1);
            if (i < SIDE_CAP) raw[i] = SideEnt{w, v};
        }
    };
    // the tokens of the history, out of its bits, each lane its own, and the tokens of the row's path once more by themselves
    auto on_path = [&](int v) {
        for (int s = row < ap.m ? row : 0; s > 0; s = ap.parent[s])
            if (ap.feed[s] == v) return true;
        return false;
    };
    auto from_table = [&](int v) {
        const uint32_t c = ap.pen_cnt[v];
        const float w = penalised(ap, h2f(lp[v]), (c >> 31) != 0, c & 0x7FFFFFFFu);
        if (!on_path(v)) look(v, w);
    };
    const uint32_t* const seen = pen_seen(ap.pen_cnt, ap.vocab);
    const int words = (ap.vocab + 31) >> 5;
    for (int w0 = 0; w0 < words; w0 += 4 * 1024) {
        uint32_t bits[4];
#pragma unroll
        for (int j = 0; j < 4; j++) bits[j] = seen[min(w0 + j * 1024 + tid, words - 1)];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int w = w0 + j * 1024 + tid;
            for (uint32_t left = w < words ? bits[j] : 0u; left; left &= left - 1) from_table(w * 32 + __ffs(left) - 1);
        }
    }
    on_path_tokens(ap, row, [&](int v) { look(v, score_of<true>(ap, row, v, lp[v])); });
    __syncthreads();
    int n = *counter;
    if (n > SIDE_CAP) {  // refused: more penalised candidates between two neighbouring fp16 values than the list holds
        if (tid == 0) atomicOr(err, 8);
        n = SIDE_CAP;
    }
    for (int i = tid; i < n; i += 1024) {
        const SideEnt me = raw[i];
        int rank = 0;
        for (int j = 0; j < n; j++) rank += raw[j].w > me.w || (raw[j].w == me.w && raw[j].v < me.v);
        sorted[rank] = me;
    }
    __syncthreads();
    return n;
}

// The bin of a group, by one whole wave: the first of its 64 bins at which the running sum from `c` on reaches `target`, in every lane (-1: none); *before: the
// sum before it.
__device__ __forceinline__ int bin_reaching(unsigned long long v, unsigned long long c, unsigned long long target, unsigned long long* before) {
    const int lane = threadIdx.x & 63;
    unsigned long long inc = v;
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t lo = __shfl_up((uint32_t)inc, o), hi = __shfl_up((uint32_t)(inc >> 32), o);
        const unsigned long long up = ((unsigned long long)hi << 32) | lo;
        if (lane >= o) inc += up;
    }
    const unsigned long long excl = c + inc - v;
    const unsigned long long hit = __ballot(excl < target && target <= excl + v);
    if (!hit) return -1;
    const int at = __builtin_ctzll(hit);
    const uint32_t lo = __shfl((uint32_t)excl, at), hi = __shfl((uint32_t)(excl >> 32), at);
    *before = ((unsigned long long)hi << 32) | lo;
    return at;
}

// One workgroup per distribution row.
template <bool PEN>
__global__ __launch_bounds__(1024) void k_trunc_cut(const uint16_t* target, const uint16_t* draft,
                                                    const AcceptParams* app, int m, double* scratch,
                                                    const unsigned long long* tmass, const uint32_t* tcount,
                                                    AcceptResult* res, int32_t* err) {
    __shared__ SideEnt s_raw[PEN ? SIDE_CAP : 1], s_sorted[PEN ? SIDE_CAP : 1];
    __shared__ __attribute__((aligned(16))) uint32_t s_mask[1024 * PICK_MASK_GROUPS / 4];  // build_mask
    __shared__ int s_nside;
    __shared__ unsigned long long wsum[16];
    __shared__ unsigned long long s_before_p, s_at;
    __shared__ int s_bin_k, s_j_k, s_bin_p, s_cnt_p, s_minp_key, s_bin, s_j, s_idx, s_found, s_held_k, s_held_p;
    __shared__ double s_margin;
    const AcceptParams& ap = *app;
    const int row = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
    const int vocab = ap.vocab;
    Layout L = layout(scratch);
    const double mx = wave_max_f64(L.pmax[row * NSEG + lane]);
    const double sum = fold_row(L.psum, row);
    const uint16_t* lp = row_ptr(target, draft, m, vocab, row);
    const uint32_t* const gc = tcount + (size_t)row * TRUNC_WORDS;
    const unsigned long long* const gm = tmass + (size_t)row * TRUNC_WORDS;
    static_assert(RANK_GROUPS == 1024, "a group to a thread");
    if (tid == 0) {
        s_bin_k = s_bin_p = s_minp_key = s_bin = -1;
        s_idx = 0x7FFFFFFF;
        s_margin = 1.0;
    }
    __syncthreads();
    unsigned long long total, total_p = 0, before;
    if (ap.top_k > 0) {
        const unsigned long long mine[1] = {gc[tid]}, K = (unsigned long long)ap.top_k;
        const int group = group_reaching<16, 1>(mine, K, wsum, &s_found, &s_at, &before, &total);
        if (group >= 0 && tid < 64) {
            const uint32_t held = gc[RANK_GROUPS + lane];
            unsigned long long c = 0;
            const int i = bin_reaching(held, before, K, &c);
            if (lane == i) {
                s_bin_k = group * 64 + i;
                s_j_k = (int)(K - c);
                s_held_k = (int)held;
            }
        }
        __syncthreads();
    }
    if (ap.has_top_p) {
        const unsigned long long mine[1] = {gm[tid]}, tgt = (unsigned long long)(ap.top_p * FIX);
        const int group = group_reaching<16, 1>(mine, tgt, wsum, &s_found, &s_at, &before, &total);
        total_p = total;
        if (group >= 0 && tid < 64) {
            const int held = (int)gc[RANK_GROUPS + 64 + lane];
            unsigned long long c = 0;
            const int i = bin_reaching(gm[RANK_GROUPS + 64 + lane], before, tgt, &c);
            if (lane == i) {
                s_bin_p = group * 64 + i;
                s_before_p = c;
                s_cnt_p = s_held_p = held;
            }
        }
    }
    if (!PEN && ap.has_min_p) {  // (penalised rounds test e >= min_p per candidate instead)
        int best = -1;
        for (int i = 0; i < 64; i++) {
            const int key = tid * 64 + i;
            const uint32_t bits = key_bits(key);
            if ((bits & 0x7C00u) == 0x7C00u) continue;  // no finite logit has this key
            if (exp((double)h2f((uint16_t)bits) - mx) >= ap.min_p) best = key;  // e_top == exp(0) == 1
        }
        if (best >= 0) atomicMax(&s_minp_key, best);
    }
    __syncthreads();
    int ns_p = 0;  // penalised rounds: the top-p bin's candidates above the bin's own value
    if constexpr (PEN) {
        if (s_bin_p >= 0) ns_p = collect_side(ap, row, lp, s_bin_p, s_raw, s_sorted, &s_nside, err);
    }
    if (tid == 0) {
        int bin = s_bin_k, j = s_bin_k >= 0 ? s_j_k : 0;
        if (s_bin_p >= 0) {
            // how many candidates of the bin it takes to reach top_p: each carries the same mass
            const double pm = exp((double)h2f((uint16_t)key_bits(s_bin_p)) - mx) / sum;
            double before = (double)s_before_p / FIX;
            long taken = 0;  // candidates above the bin's value, each with a mass of its own
            bool reached = false;
            double mg_side = 1.0;
            if constexpr (PEN) {
                for (int i = 0; i < ns_p && !reached; i++) {
                    before += exp((double)s_sorted[i].w - mx) / sum;
                    taken += 1;
                    fold_margin(mg_side, before, ap.top_p);
                    reached = before >= ap.top_p;
                }
                s_cnt_p -= ns_p;
            }
            long jp = reached || s_cnt_p <= 0 ? 0 : (long)ceil((ap.top_p - before) / pm);
            if (reached || s_cnt_p <= 0) {
                s_margin = mg_side;
                jp = taken;
                if (bin < 0 || s_bin_p < bin || (s_bin_p == bin && jp < j)) {
                    bin = s_bin_p;
                    j = (int)jp;
                }
            } else {
                jp = jp < 1 ? 1 : jp;
                while (jp > 1 && before + (double)(jp - 1) * pm >= ap.top_p) jp--;
                while (jp < s_cnt_p && before + (double)jp * pm < ap.top_p) jp++;
                jp = jp > s_cnt_p ? s_cnt_p : jp;
                double mg = 1.0;
                fold_margin(mg, before + (double)jp * pm, ap.top_p);
                if (jp > 1 || s_before_p > 0) fold_margin(mg, before + (double)(jp - 1) * pm, ap.top_p);
                s_margin = fmin(mg, mg_side);
                jp += taken;
                if (bin < 0 || s_bin_p < bin || (s_bin_p == bin && jp < j)) {
                    bin = s_bin_p;
                    j = (int)jp;
                }
            }
        }
        if (ap.has_top_p && s_bin_p < 0) {  // the cumulative mass never reached top_p: everything ranked survives
            double mg = 1.0;
            fold_margin(mg, (double)total_p / FIX, ap.top_p);
            s_margin = mg;
        }
        s_bin = bin;
        s_j = j;
    }
    __syncthreads();
    const int bin = s_bin;
    int j = s_j;
    float cut_w = bin >= 0 ? h2f((uint16_t)key_bits(bin)) : 0.f;
    if (bin >= 0 && j < (bin == s_bin_k ? s_held_k : s_held_p)) {
        bool on_value = true;
        if constexpr (PEN) {
            // the bin's candidates above its own value come first in rank order
            const int ns = bin == s_bin_p ? ns_p : collect_side(ap, row, lp, bin, s_raw, s_sorted, &s_nside, err);
            if (j <= ns) {
                if (tid == 0) s_idx = s_sorted[j - 1].v;
                cut_w = s_sorted[j - 1].w;
                on_value = false;
            } else {
                j -= ns;
            }
        }
        if (on_value) {
            // the j-th candidate on the bin's value in index order
            const int groups = mask_groups(vocab), v0 = min(tid * groups * 8, vocab), v1 = min(v0 + groups * 8, vocab);
            const bool vec = ((uintptr_t)lp & 15) == 0, masked = vec && groups <= PICK_MASK_GROUPS;
            if (masked) build_mask<PEN>(ap, row, lp, bin, (uint8_t*)s_mask, row_ahead(lp, vocab));
            auto for_matches = [&](auto&& on_match) {
                if (masked) walk_mask((const uint8_t*)s_mask, groups, on_match);
                else scan_on<PEN>(ap, row, lp, v0, v1, bin, vec, on_match);
            };
            int n = 0;
            for_matches([&](int) { n++; });
            const unsigned long long excl = block_scan_u64<16>((unsigned long long)n, wsum, &total);
            if ((int)excl < j && j <= (int)excl + n) {
                int c = (int)excl;
                for_matches([&](int v) {
                    c++;
                    if (c == j) s_idx = v;
                });
            }
        }
        __syncthreads();
    }
    if (tid == 0) {
        Cut cut{65536, 0x7FFFFFFF, 0.f, 0.f};
        if (bin >= 0) cut = Cut{bin, s_idx, cut_w, 0.f};
        if (!PEN && ap.has_min_p && s_minp_key >= 0 && s_minp_key < cut.key) cut = Cut{s_minp_key, 0x7FFFFFFF, 0.f, 0.f};
        L.cut[row] = cut;
        atomicMin((unsigned long long*)&res->min_margin, __builtin_bit_cast(unsigned long long, s_margin));
    }
}

// ---- the cumulative walk --------------------------------------------------------------------
// One workgroup per job.  Finds the rank bin in which the cumulative mass first exceeds the
// uniform (exact integer prefix over the fixed-point bins, which the round's first kernel zeroed), then
// walks that bin's candidates in index order in f64.
template <bool PEN>
__global__ __launch_bounds__(1024) void k_pick(const uint16_t* target, const uint16_t* draft,
                                               const AcceptParams* app, double* scratch, const double* work,
                                               unsigned long long* hist, const Decision* dec_in,
                                               AcceptResult* res, int32_t* tokens_out, int32_t* err,
                                               int kind, AcceptResult* host) {
    __shared__ SideEnt s_raw[PEN ? SIDE_CAP : 1], s_sorted[PEN ? SIDE_CAP : 1];
    __shared__ __attribute__((aligned(16))) uint32_t s_mask[1024 * PICK_MASK_GROUPS / 4];  // one bit per vocabulary entry: on the bin's value
    __shared__ int s_nside, s_side_last;
    __shared__ double s_side_sum;
    __shared__ unsigned long long wsum[16];
    __shared__ double dsum[16];
    __shared__ unsigned long long s_total, s_before;
    __shared__ int s_group, s_bin, s_last_bin, s_token, s_fallback;
    __shared__ double s_cum_before, s_cum_at;
    const AcceptParams& ap = *app;
    const int jobi = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // What one workgroup costs is the round trips one behind the other: the sums of both modes and the residual's pieces are asked for with the
    // decision that says which are wanted
    Layout L = layout(scratch);
    static_assert(NSEG * NSUB == 256, "four waves fold the pieces");
    const unsigned long long* const sums = rank_groups(hist) + (size_t)jobi * 2 * RANK_GROUPS + tid;
    const unsigned long long loc_p = sums[0], loc_r = sums[RANK_GROUPS];
    const double piece = L.segtot[jobi * NSEG * NSUB + (tid & 255)];
    const Decision dec = dec_in[jobi];
    const int vocab = ap.vocab;
    int token = -1;
    double margin = dec.margin;

    if (dec.job.mode != 0) {
        int mode = dec.job.mode;
        double R = 1.0;
        if (mode == 2) {
            // residual mass: the pieces' partial sums folded in a fixed order
            if (tid < 256) {
                const double part = wave_sum_f64(piece);
                if (lane == 0) dsum[wave] = part;
            }
            __syncthreads();
            R = (dsum[0] + dsum[1]) + (dsum[2] + dsum[3]);
            __syncthreads();
            if (R < 1e-12) mode = 1;  // distribution.rs:96-126: residual underflow -> plain p draw
        }
        unsigned long long* hp = hist + (long)jobi * 2 * 65536;
        unsigned long long* hsel = mode == 2 ? hp + 65536 : hp;
        const double* w = kind == 2 ? work + (long)dec.pad * vocab : work + (long)jobi * 2 * vocab + (mode == 2 ? vocab : 0);
        const uint16_t* lp = row_ptr(target, draft, ap.m, vocab, dec.job.row_p);
        const int groups = mask_groups(vocab), v0 = min(tid * groups * 8, vocab), v1 = min(v0 + groups * 8, vocab);
        const bool vec = ((uintptr_t)lp & 15) == 0, masked = vec && groups <= PICK_MASK_GROUPS;
        RowAhead ahead;  // (the row is on its way while the bin is looked for)
        if (masked) ahead = row_ahead(lp, vocab);

        // 64 consecutive rank bins per thread (see bin_addr), whose sum is there already; integer sums are exact and order
        // independent
        const unsigned long long loc = mode == 2 ? loc_r : loc_p;
        unsigned long long inc = loc;
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t lo = __shfl_up((uint32_t)inc, o), hi = __shfl_up((uint32_t)(inc >> 32), o);
            const unsigned long long up = ((unsigned long long)hi << 32) | lo;
            if (lane >= o) inc += up;
        }
        if (lane == 63) wsum[wave] = inc;
        if (tid == 0) {
            s_group = s_bin = -1;
            s_last_bin = -1;
            s_token = -1;
            s_fallback = 0;
        }
        __syncthreads();
        unsigned long long wbase = 0, total = 0;
        for (int i = 0; i < 16; i++) {
            if (i < wave) wbase += wsum[i];
            total += wsum[i];
        }
        const unsigned long long excl = wbase + inc - loc;
        // target in fixed point: u * total (the bins hold unnormalised mass in residual mode)
        const unsigned long long tgt = (unsigned long long)(dec.job.u * (double)total);
        if (loc > 0) atomicMax(&s_last_bin, tid * 64 + 63);
        if (excl <= tgt && tgt < excl + loc) {
            s_group = tid;
            s_before = excl;
        }
        if (tid == 0) s_total = total;
        __syncthreads();
        const int group = s_group;  // the group that holds the target (not written again: what comes next differs by it)
        if (group >= 0) {
            // its first bin at which the running sum passes the target: a lane to a bin, every wave for itself
            const unsigned long long mine = hsel[(group >> 6) * 4096 + (group & 63) + lane * 64], from = s_before;
            unsigned long long upto = mine;
            for (int o = 1; o < 64; o <<= 1) {
                const uint32_t lo = __shfl_up((uint32_t)upto, o), hi = __shfl_up((uint32_t)(upto >> 32), o);
                if (lane >= o) upto += ((unsigned long long)hi << 32) | lo;
            }
            const int hit = __builtin_ctzll(__ballot(tgt < from + upto));  // (the group's sum passes it)
            __syncthreads();
            if (tid == hit) {
                s_bin = group * 64 + hit;
                s_before = from + upto - mine;
            }
        } else {
            // rounding at the tail: the reference falls back to the LAST surviving candidate
            // (choose.rs:333-338).  Last occupied bin, last matching index.
            const int lb = s_last_bin;  // upper end of the last occupied 64-bin group
            if (tid * 64 + 63 == lb) {
                int bb = lb;
                while (bb > tid * 64 && hsel[bin_addr(bb)] == 0) bb--;
                s_bin = bb;
                s_before = total;
                s_fallback = 1;
            }
        }
        __syncthreads();
        const int bin = s_bin;
        const bool fallback = s_fallback != 0;
        const double norm = (double)s_total;  // fixed-point total <-> 1.0 (p mode) or R (residual)
        const double cum0 = (double)s_before / norm;  // cumulative mass before this bin
        double side_sum = 0.0;
        if constexpr (PEN) {
            // the bin's candidates above its own value come first: few, walked by one thread
            const int ns = collect_side(ap, dec.job.row_p, lp, bin, s_raw, s_sorted, &s_nside, err);
            if (tid == 0) {
                double c = cum0;
                int last = -1;
                bool found = false;
                for (int i = 0; i < ns; i++) {
                    const int v = s_sorted[i].v;
                    const double wv = mode == 2 ? w[v] / R : w[v];
                    if (mode == 2 && !(wv > 0.0)) continue;
                    if (!fallback && !found && dec.job.u < c + wv) {
                        s_token = v;
                        s_cum_before = c;
                        s_cum_at = c + wv;
                        found = true;
                    }
                    c += wv;
                    last = v;
                }
                s_side_sum = c - cum0;
                s_side_last = last;
            }
            __syncthreads();
            side_sum = s_side_sum;
        }
        // walk the bin in index order: contiguous index chunk per thread
        if (masked) build_mask<PEN>(ap, dec.job.row_p, lp, bin, (uint8_t*)s_mask, ahead);
        // on_match(v) for the candidates of this thread's chunk that sit on the bin's value, ascending
        auto for_matches = [&](auto&& on_match) {
            if (masked) walk_mask((const uint8_t*)s_mask, groups, on_match);
            else scan_on<PEN>(ap, dec.job.row_p, lp, v0, v1, bin, vec, on_match);
        };
        double lsum = 0.0;
        int lastv = -1;
        for_matches([&](int v) {
            const double wv = mode == 2 ? w[v] / R : w[v];
            if (mode != 2 || wv > 0.0) {
                lsum += wv;
                lastv = v;
            }
        });
        double incd = lsum;
        for (int o = 1; o < 64; o <<= 1) {
            uint64_t u = __builtin_bit_cast(uint64_t, incd);
            uint32_t lo = __shfl_up((uint32_t)u, o), hi = __shfl_up((uint32_t)(u >> 32), o);
            const double up = __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
            if (lane >= o) incd += up;
        }
        if (lane == 63) dsum[wave] = incd;
        __syncthreads();
        double dbase = 0.0;
        for (int i = 0; i < wave; i++) dbase += dsum[i];
        const double before = PEN ? cum0 + side_sum + (dbase + incd - lsum) : cum0 + (dbase + incd - lsum);
        if (fallback) {
            if (lastv >= 0) atomicMax(&s_token, lastv);
        } else {
            const double u = dec.job.u;
            if (lsum > 0.0 && !(u < before) && u < before + lsum) {
                double c = before;
                bool found = false;
                for_matches([&](int v) {
                    if (found) return;
                    const double wv = mode == 2 ? w[v] / R : w[v];
                    if (mode == 2 && !(wv > 0.0)) return;
                    if (u < c + wv) {
                        s_token = v;
                        s_cum_before = c;
                        s_cum_at = c + wv;
                        found = true;
                        return;
                    }
                    c += wv;
                });
            }
        }
        __syncthreads();
        token = s_token;
        if (PEN && fallback && token < 0) token = s_side_last;  // no on-value candidate: the last of the others
        if (token < 0) {
            // the f64 walk and the fixed-point bin search disagreed by a rounding: the uniform
            // sits on a bin edge.  Take the bin's first (u below) or last candidate and report
            // a zero margin.
            __syncthreads();  // (every wave has read that there is none)
            if (lastv >= 0) atomicMax(&s_token, lastv);
            __syncthreads();
            token = s_token;
            if (PEN && token < 0) token = s_side_last;
            margin = 0.0;
        } else if (!fallback) {
            margin = fmin(margin, fmin(dec.job.u - s_cum_before, s_cum_at - dec.job.u));
        }
    }

    if (tid == 0) {
        if (kind == 1) {
            tokens_out[jobi] = token;
            if (const int32_t seen = *err) atomicOr(&res->error, seen);  // (each draw's own: what another refuses may come after this one's end)
            // margins of the k draws are folded on the host side from res->min_margin
            atomicMin((unsigned long long*)&res->min_margin, __builtin_bit_cast(unsigned long long, margin));
        } else {
            const unsigned long long mine = __builtin_bit_cast(unsigned long long, margin);
            const double least = __builtin_bit_cast(double, min(atomicMin((unsigned long long*)&res->min_margin, mine), mine));
            auto put = [&](AcceptResult* to) {
                to->accepted = dec.accepted;
                to->committed = dec.committed;
                to->stopped = dec.stopped;
                to->next = dec.stopped ? -1 : token;
                to->draw_step = dec.draw_step;
                to->path_len = dec.accepted + 1;
                for (int i = 0; i <= dec.accepted; i++) to->path[i] = kind == 2 ? tokens_out[i] : i;
                to->error = *err;
            };
            put(res);
            if (host) {
                put(host);
                host->min_margin = least;
                __threadfence_system();
            }
        }
    }
}

// ---- sampled acceptance over a draft tree ---------------------------------------------------
// The reference has no multi-branch rejection sampler (speculative.rs:390-392 keeps tree rounds
// greedy); this follows the oracle's definition: at node `at`, with p the target distribution of
// row `at` and q the distribution its children were drawn from, the children are tried in slot
// order -- child x is accepted when r * q(x) <= p(x) for a fresh uniform r; a rejection replaces
// p by normalise(max(p - q, 0)) (kept as is when that mass is below 1e-12) -- and when no child
// survives the next token is drawn from the p that is left.  No stop / budget bookkeeping.
//
// The statistics leave every node's p and q as dense f64 rows (work slots 0..m-1 and m..2m-1) that are divided by their row's
// total where they are read; then the tree is walked one child test per launch.  A test is two lookups;
// only a rejection costs a pass over the vocabulary (slots 32 and 33 alternate as the residual,
// whose normalising division is applied when it is read, so a pass reads two rows and writes one).
constexpr int TREE_SCRATCH_SLOT = 2 * TSV_MAX_ROWS;  // two residual rows behind the 32 distribution rows

// The walk as a sequence of short chip-wide launches (one per child test there can be, then the
// finish): every workgroup re-derives the step's decision from the walk state (two lookups), a
// rejection's residual pass is spread over all of them, and the pass's total is folded by the next
// launch.  The state and the partial sums are double-buffered: launch k reads copy k & 1 and writes the
// other one, so a workgroup that starts late still sees what the previous launch left.
constexpr int TREE_WGS = 256;
struct TreeWalk {
    int32_t at, next_s, plen, which, done, pending, src_slot, pend_slot;
    double Z, margin;
    uint64_t ds;
    int32_t path[TSV_MAX_ROWS + 1];
    int32_t pad;
};
static_assert(sizeof(TreeWalk) % 8 == 0 && sizeof(TreeWalk) <= 32 * 8, "fits its slot of the statistics block");

// behind the decisions: two copies of the state (32 doubles each), then two sets of TREE_WGS partial sums
constexpr int DECISIONS_AT = 4 * MAX_DIST_ROWS + 9 * MAX_DIST_ROWS * NSEG + MAX_JOBS * NSEG * NSUB;
constexpr int STATS_DOUBLES = DECISIONS_AT + MAX_JOBS * 16;
constexpr int TREE_STATE_DOUBLES = 2 * 32 + 2 * TREE_WGS;
__device__ TreeWalk* tree_walk(double* scratch, int copy) { return (TreeWalk*)(scratch + STATS_DOUBLES + 32 * copy); }
__device__ double* tree_partials(double* scratch, int copy) { return scratch + STATS_DOUBLES + 64 + TREE_WGS * copy; }

// The state launch k starts from: copy k & 1 with the previous launch's residual pass resolved
// (its total decides whether the residual replaces the node's distribution: distribution.rs:96-126).
__device__ TreeWalk tree_state(const AcceptParams& ap, double* scratch, int k, double* red) {
    TreeWalk w;
    if (k == 0) {  // the walk starts at the root
        w.at = 0;
        w.next_s = 1;
        w.plen = 1;
        w.which = w.done = w.pending = w.src_slot = w.pend_slot = w.pad = 0;
        w.Z = row_total(layout(scratch), 0);
        w.margin = 1.0;
        w.ds = ap.draw_step;
        w.path[0] = 0;
        return w;
    }
    w = *tree_walk(scratch, k & 1);
    if (w.pending) {
        const double part = (int)threadIdx.x < TREE_WGS ? tree_partials(scratch, k & 1)[threadIdx.x] : 0.0;
        const double total = block_sum_f64(part, red);
        if (total >= 1e-12) {
            w.src_slot = w.pend_slot;
            w.Z = total;
            w.which ^= 1;
        }
        w.pending = 0;
    }
    return w;
}

template <bool PEN>
__global__ __launch_bounds__(256) void k_tree_step(const AcceptParams* app, double* scratch, double* work, int k) {
    __shared__ double red[4];
    const AcceptParams& ap = *app;
    const int vocab = ap.vocab, m = ap.m;
    TreeWalk w = tree_state(ap, scratch, k, red);
    TreeWalk* out = tree_walk(scratch, (k + 1) & 1);
    const bool writer = blockIdx.x == 0 && threadIdx.x == 0;
    int s = -1;
    if (!w.done)
        for (int c = w.next_s; c < m; c++)
            if (ap.parent[c] == w.at) {
                s = c;
                break;
            }
    if (s < 0) {  // nothing left to try below this node (or the walk had ended already)
        w.done = 1;
        if (writer) *out = w;
        return;
    }
    const double* src = work + (long)w.src_slot * vocab;  // the node's p; its values are src[v] / Z
    const double* q = work + (long)(m + w.at) * vocab;
    const double total_q = row_total(layout(scratch), m + w.at);
    const int32_t x = ap.feed[s];
    const double r = unit_draw(ap.seed, w.ds);
    const double px = src[x] / w.Z, qx = q[x] / total_q;
    fold_margin(w.margin, r * qx, px);
    w.ds += 1;
    w.next_s = s + 1;
    if (r * qx <= px) {
        w.path[w.plen] = s;
        w.plen += 1;
        w.at = s;
        w.src_slot = s;
        w.Z = row_total(layout(scratch), s);
        w.which = 0;
        if (writer) *out = w;
        return;
    }
    // residual max(p - q, 0) of this workgroup's slice; the next launch folds the totals
    double* dst = work + (long)(TREE_SCRATCH_SLOT + w.which) * vocab;
    const int per = (vocab + TREE_WGS - 1) / TREE_WGS, v0 = blockIdx.x * per, v1 = min(v0 + per, vocab);
    double acc = 0.0;
    for (int v = v0 + threadIdx.x; v < v1; v += 256) {
        const double mv = fmax(src[v] / w.Z - q[v] / total_q, 0.0);
        dst[v] = mv;
        acc += mv;
    }
    acc = block_sum_f64(acc, red);
    if (threadIdx.x == 0) tree_partials(scratch, (k + 1) & 1)[blockIdx.x] = acc;
    w.pending = 1;
    w.pend_slot = TREE_SCRATCH_SLOT + w.which;
    if (writer) *out = w;
}

// After the last step: the rank histogram of what is left of p at the node the walk ended on, and the
// round's decision; the draw itself is k_pick's.
template <bool PEN>
__global__ __launch_bounds__(256) void k_tree_finish(const uint16_t* target, const AcceptParams* app, double* scratch,
                                                     double* work, unsigned long long* hist, Decision* dec_out,
                                                     int32_t* path_out, int k) {
    __shared__ double red[4];
    __shared__ unsigned long long groups[RANK_GROUPS];
    for (int i = threadIdx.x; i < RANK_GROUPS; i += 256) groups[i] = 0;
    __syncthreads();
    const AcceptParams& ap = *app;
    const int vocab = ap.vocab;
    const TreeWalk w = tree_state(ap, scratch, k, red);
    Layout L = layout(scratch);
    unsigned long long* hr = hist + 65536;
    const double* src = work + (long)w.src_slot * vocab;
    const uint16_t* lpk = target + (long)w.at * vocab;
    const int per = (vocab + TREE_WGS - 1) / TREE_WGS, v0 = blockIdx.x * per, v1 = min(v0 + per, vocab);
    for (int v = v0 + threadIdx.x; v < v1; v += 256) {
        const double mv = src[v] / w.Z;
        const unsigned long long fixed = (unsigned long long)(mv * FIX);
        if (fixed) {
            const uint16_t b = lpk[v];
            const uint32_t rk = key_of<PEN>(score_of<PEN>(ap, w.at, v, b), b);
            atomicAdd(hr + bin_addr(rk), fixed);
            atomicAdd(&groups[rk >> 6], fixed);
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < RANK_GROUPS; i += 256)
        if (groups[i]) atomicAdd(rank_groups(hist) + RANK_GROUPS + i, groups[i]);
    if (blockIdx.x != 0) return;
    // the draw divides the stored values by the fold of these pieces: Z, exactly
    if (threadIdx.x < NSEG * NSUB) L.segtot[threadIdx.x] = threadIdx.x == 0 ? w.Z : 0.0;
    if (threadIdx.x == 0) {
        for (int i = 0; i < w.plen; i++) path_out[i] = w.path[i];
        Decision d;
        d.job.mode = 2;
        d.job.row_p = w.at;
        d.job.row_q = 0;
        d.job.u = unit_draw(ap.seed, w.ds);
        d.accepted = w.plen - 1;
        d.committed = w.plen - 1;
        d.stopped = 0;
        d.pad = w.src_slot;  // the work slot the draw reads
        d.draw_step = w.ds + 1;
        d.margin = w.margin;
        dec_out[0] = d;
    }
}

// ---- greedy --------------------------------------------------------------------------------
// choose.rs:277-285: first maximum.  ARGMAX_SEG workgroups per target row, each over a contiguous
// run of the vocabulary: the best (value, index) of every run goes to a partial slot, and whoever
// needs the row's arg-max folds the runs in index order (a later run wins only with a strictly
// larger value, so ties go to the lower index whatever the split).
constexpr int ARGMAX_SEG = 16;

__global__ __launch_bounds__(256) void k_argmax_part(const uint16_t* target, int vocab, float* pv, int32_t* pi, int32_t* err) {
    __shared__ float bv[4];
    __shared__ int bi[4];
    const int row = blockIdx.y, seg = blockIdx.x;
    const uint16_t* p = target + (long)row * vocab;
    const int chunk = ((vocab + ARGMAX_SEG - 1) / ARGMAX_SEG + 7) & ~7;
    const int v0 = min(seg * chunk, vocab), v1 = min(v0 + chunk, vocab);
    float best = -INFINITY;
    int idx = 0x7FFFFFFF;
    bool bad = false;
    auto take = [&](uint16_t b, int v) {
        bad |= (b & 0x7C00u) == 0x7C00u;
        const float f = h2f(b);
        if (f > best || (f == best && v < idx)) {
            best = f;
            idx = v;
        }
    };
    if ((((uintptr_t)p) & 15) == 0) {  // eight logits per 16-byte load (v0 is a multiple of 8)
        const int i0 = v0 >> 3, i1 = v1 >> 3;
        for (int i = i0 + threadIdx.x; i < i1; i += 256) {
            const uint4 q = ((const uint4*)p)[i];
            const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
            for (int j = 0; j < 8; j++) take((uint16_t)(w[j >> 1] >> (16 * (j & 1))), 8 * i + j);
        }
        for (int v = max(i1 << 3, v0) + threadIdx.x; v < v1; v += 256) take(p[v], v);
    } else {
        for (int v = v0 + threadIdx.x; v < v1; v += 256) take(p[v], v);
    }
    if (bad) atomicOr(err, 1);
    for (int o = 32; o > 0; o >>= 1) {
        const float ob = __shfl_xor(best, o);
        const int oi = __shfl_xor(idx, o);
        if (ob > best || (ob == best && oi < idx)) {
            best = ob;
            idx = oi;
        }
    }
    if ((threadIdx.x & 63) == 0) {
        bv[threadIdx.x >> 6] = best;
        bi[threadIdx.x >> 6] = idx;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int i = 1; i < 4; i++)
            if (bv[i] > best || (bv[i] == best && bi[i] < idx)) {
                best = bv[i];
                idx = bi[i];
            }
        pv[row * ARGMAX_SEG + seg] = best;
        pi[row * ARGMAX_SEG + seg] = idx;
    }
}

// the row's arg-max from its runs' partial results, read by one thread
__device__ __forceinline__ int32_t fold_argmax(const float* pv, const int32_t* pi, int row) {
    float v[ARGMAX_SEG];
    int32_t ix[ARGMAX_SEG];
#pragma unroll
    for (int s = 0; s < ARGMAX_SEG; s++) {
        v[s] = pv[row * ARGMAX_SEG + s];
        ix[s] = pi[row * ARGMAX_SEG + s];
    }
    float best = v[0];
    int32_t idx = ix[0];
#pragma unroll
    for (int s = 1; s < ARGMAX_SEG; s++)
        if (v[s] > best) {  // an empty run holds -inf and never wins
            best = v[s];
            idx = ix[s];
        }
    return idx;
}

__global__ void k_argmax_fold(const float* pv, const int32_t* pi, int rows, int32_t* out) {
    if ((int)threadIdx.x < rows) out[threadIdx.x] = fold_argmax(pv, pi, threadIdx.x);
}

// speculative.rs:736-754 (chain) and 494-550 (tree walk) at temperature 0, by one thread over the
// rows' arg-max tokens.
struct GreedyWalk {
    int32_t accepted, committed, stopped, next, path_len;
    int32_t path[TSV_MAX_ROWS + 1];
};
__device__ GreedyWalk walk_greedy(const AcceptParams& ap, const int32_t* amax) {
    GreedyWalk g;
    uint64_t gen = ap.generated;
    int32_t committed = 0, stopped = 0, next = -1;
    int at = 0, plen = 1;
    g.path[0] = 0;
    for (;;) {
        const int32_t want = amax[at];
        int hit = -1;
        if (ap.tree) {
            for (int s = 1; s < ap.m; s++)
                if (ap.parent[s] == at && ap.feed[s] == want) {
                    hit = s;
                    break;
                }
        } else if (at + 1 < ap.m && ap.feed[at + 1] == want) {
            hit = at + 1;
        }
        if (hit < 0) {
            next = want;
            break;
        }
        g.path[plen++] = hit;
        at = hit;
        if ((stopped = sink_commit(ap, want, gen, committed))) break;
    }
    g.accepted = plen - 1;
    g.committed = committed;
    g.stopped = stopped;
    g.next = stopped ? -1 : next;
    g.path_len = plen;
    return g;
}

__global__ void k_walk_greedy(const AcceptParams* app, const float* pv, const int32_t* pi, AcceptResult* res,
                              const int32_t* err, AcceptResult* host) {
    __shared__ int32_t amax[TSV_MAX_ROWS];
    const AcceptParams& ap = *app;
    if ((int)threadIdx.x < ap.m) amax[threadIdx.x] = fold_argmax(pv, pi, threadIdx.x);
    __syncthreads();
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    const GreedyWalk g = walk_greedy(ap, amax);
    auto put = [&](AcceptResult* to) {
        for (int i = 0; i < g.path_len; i++) to->path[i] = g.path[i];
        to->accepted = g.accepted;
        to->committed = g.committed;
        to->stopped = g.stopped;
        to->next = g.next;
        to->draw_step = ap.draw_step;
        to->path_len = g.path_len;
        to->min_margin = 1.0;
        to->error = *err;
    };
    put(res);
    if (host) {
        put(host);
        __threadfence_system();
    }
}

__global__ void k_clear_result(AcceptResult* res, int32_t* err) {
    if (threadIdx.x == 0) {
        *err = 0;
        res->error = 0;
        res->min_margin = 1.0;
    }
}

}  // namespace

// scratch.counters (ACCEPT_COUNTER_WORDS words): [0] error flag of an arg-max chain, [32..49) tree path, [64..) the greedy
// arg-max partials (value, then index, per row and run); decisions live after the
// statistics block; histograms and work arrays are separate allocations in AcceptScratch.
size_t accept_stats_doubles() { return STATS_DOUBLES + TREE_STATE_DOUBLES; }
size_t accept_hist_words() { return (size_t)MAX_JOBS * 2 * (65536 + RANK_GROUPS); }
int accept_work_rows() { return 2 + MAX_DIST_ROWS; }

static Decision* decisions(const AcceptScratch& sc) {
    return (Decision*)(sc.stats + DECISIONS_AT);
}

// Between the softmax sums and the reweighting totals: the truncation cut of every row.
template <bool PEN>
static void launch_trunc(hipStream_t s, const uint16_t* target, const uint16_t* draft, int m, int rows,
                         const AcceptParams* ap_dev, const AcceptParams& ap, const AcceptScratch& sc) {
    if (ap.top_k == 0 && !ap.has_top_p) {
        if (PEN || !ap.has_min_p) return;  // (penalised rounds test min-p per candidate)
    }
    unsigned long long* tm = (unsigned long long*)sc.tmass;
    if (ap.top_k != 0 || ap.has_top_p) {
        hipLaunchKernelGGL(k_trunc_groups<PEN>, dim3(NSEG, rows), dim3(256), 0, s, target, draft, m, ap.vocab, sc.stats, tm,
                           sc.tcount, ap.has_top_p, ap_dev);
        hipLaunchKernelGGL(k_trunc_bins<PEN>, dim3(NSEG, rows), dim3(256), 0, s, target, draft, m, ap.vocab, sc.stats, tm, sc.tcount, ap_dev);
    }
    hipLaunchKernelGGL(k_trunc_cut<PEN>, dim3(rows), dim3(1024), 0, s, target, draft, ap_dev, m, sc.stats, tm, sc.tcount,
                       sc.result, &sc.result->flag);
}

// The statistics of `rows` distribution rows, their truncation cuts and reweighting totals.
// Up to SPLIT_ROWS rows the sums' folds are workgroups of their own: one to four rows are a draft block's draws (a loop of 48 tokens,
// block 4, on a small decoder: 9640 -> 9300 us with this and the stored values).  Nine rows, a round of five, fill the chip without, and
// everything a wave does besides is done once (the same loop with the folds of all rows apart: 9060 -> 9380; sixteen-row trees 517 -> 530).
constexpr int SPLIT_ROWS = 4;
template <bool PEN>
static void launch_stats(hipStream_t s, const uint16_t* target, const uint16_t* draft, int m, int rows, int jobs,
                         const AcceptParams* ap_dev, const AcceptParams& ap, const AcceptScratch& sc, int slot0, int slot_step) {
    int32_t* err = &sc.result->flag;
    const double inv_t = 1.0 / ap.temperature;
    hipLaunchKernelGGL(k_row_max<PEN>, dim3(NSEG, rows), dim3(256), 0, s, target, draft, m, ap.vocab, sc.stats, err,
                       (unsigned long long*)sc.hist, jobs, ap_dev, ap.top_k != 0 || ap.has_top_p ? (unsigned long long*)sc.tmass : nullptr, sc.tcount);
    const dim3 grid(NSEG, rows, rows <= SPLIT_ROWS ? 4 : 1), block(256);
    if (grid.z > 1) hipLaunchKernelGGL((k_row_sum<PEN, true>), grid, block, 0, s, target, draft, m, ap.vocab, sc.stats, ap_dev);
    else hipLaunchKernelGGL((k_row_sum<PEN, false>), grid, block, 0, s, target, draft, m, ap.vocab, sc.stats, ap_dev);
    launch_trunc<PEN>(s, target, draft, m, rows, ap_dev, ap, sc);
    if (grid.z > 1)
        hipLaunchKernelGGL((k_row_total<PEN, true>), grid, block, 0, s, target, draft, m, ap.vocab, sc.stats, inv_t, ap_dev, sc.work, slot0, slot_step);
    else
        hipLaunchKernelGGL((k_row_total<PEN, false>), grid, block, 0, s, target, draft, m, ap.vocab, sc.stats, inv_t, ap_dev, sc.work, slot0, slot_step);
}

template <bool PEN>
static void launch_chain_sampled(hipStream_t s, const uint16_t* target, const uint16_t* draft,
                                 const AcceptParams* ap_dev, const AcceptParams& ap, const AcceptScratch& sc) {
    int32_t* err = &sc.result->flag;
    launch_stats<PEN>(s, target, draft, ap.m, ap.m + ap.k, 1, ap_dev, ap, sc, 2, 1);
    hipLaunchKernelGGL(k_mass_hist<PEN>, dim3(NSEG, 1, NSUB), dim3(256), 0, s, target, draft, ap_dev, sc.stats, sc.work,
                       (unsigned long long*)sc.hist, decisions(sc), 0);
    hipLaunchKernelGGL(k_pick<PEN>, dim3(1), dim3(1024), 0, s, target, draft, ap_dev, sc.stats, sc.work,
                       (unsigned long long*)sc.hist, decisions(sc), sc.result, (int32_t*)nullptr, err, 0, sc.host_result);
}

// The most child tests a walk can take before it stops.  At a node with children c_1 < ... < c_n (tested in slot
// order) the walk either rejects all n, or rejects j - 1, accepts c_j and goes on from there: worst(node) =
// max(n, max_j (j + worst(c_j))).  A parent's slot is below its children's, so one descending sweep fills the
// table.  Never more than m - 1 (every slot behind the root is tested at most once); 6 for the 16-node tree of a
// root with four chains, where m - 1 is 15.
int tree_walk_bound(const int32_t* parent, int m) {
    int worst[TSV_MAX_ROWS] = {0}, seen[TSV_MAX_ROWS] = {0};
    // children in descending slot order: the j of child c is known once all of its parent's children are counted
    int count[TSV_MAX_ROWS] = {0};
    for (int c = 1; c < m; c++) count[parent[c]]++;
    for (int c = m - 1; c >= 1; c--) {
        const int par = parent[c];
        const int j = count[par] - seen[par];  // c is the j-th child of its parent in ascending order
        seen[par]++;
        worst[par] = std::max(worst[par], std::max(count[par], j + worst[c]));
    }
    return std::min(worst[0], m - 1);
}

template <bool PEN>
static void launch_tree_sampled(hipStream_t s, const uint16_t* target, const uint16_t* draft, const AcceptParams* ap_dev,
                                const AcceptParams& ap, const AcceptScratch& sc) {
    int32_t* err = &sc.result->flag;
    int32_t* path = (int32_t*)sc.counters + 32;
    // statistics of the m target rows and the m rows the children were drawn from
    launch_stats<PEN>(s, target, draft, ap.m, 2 * ap.m, 1, ap_dev, ap, sc, 0, 1);
    // one child test per launch: as many launches as the longest walk through this tree can take
    const int steps = tree_walk_bound(ap.parent, ap.m);
    for (int k = 0; k < steps; k++)
        hipLaunchKernelGGL(k_tree_step<PEN>, dim3(TREE_WGS), dim3(256), 0, s, ap_dev, sc.stats, sc.work, k);
    hipLaunchKernelGGL(k_tree_finish<PEN>, dim3(TREE_WGS), dim3(256), 0, s, target, ap_dev, sc.stats, sc.work,
                       (unsigned long long*)sc.hist, decisions(sc), path, steps);
    hipLaunchKernelGGL(k_pick<PEN>, dim3(1), dim3(1024), 0, s, target, draft, ap_dev, sc.stats, sc.work,
                       (unsigned long long*)sc.hist, decisions(sc), sc.result, path, err, 2, sc.host_result);
}

template <bool PEN>
static void launch_draft_sampled(hipStream_t s, const uint16_t* draft, const AcceptParams* ap_dev,
                                 const AcceptParams& ap, const AcceptScratch& sc, int32_t* proposals_dev) {
    int32_t* err = &sc.result->flag;
    launch_stats<PEN>(s, draft, draft, 0, ap.k, ap.k, ap_dev, ap, sc, 1, 2);
    hipLaunchKernelGGL(k_mass_hist<PEN>, dim3(NSEG, ap.k, NSUB), dim3(256), 0, s, draft, draft, ap_dev, sc.stats, sc.work,
                       (unsigned long long*)sc.hist, decisions(sc), 1);
    hipLaunchKernelGGL(k_pick<PEN>, dim3(ap.k), dim3(1024), 0, s, draft, draft, ap_dev, sc.stats, sc.work,
                       (unsigned long long*)sc.hist, decisions(sc), sc.result, proposals_dev, err, 1, (AcceptResult*)nullptr);
}

int launch_accept(hipStream_t s, const uint16_t* target, const uint16_t* draft, const AcceptParams* ap_dev,
                  const AcceptParams& ap, const AcceptScratch& sc) {
    int32_t* err = &sc.result->flag;
    float* pv = (float*)sc.counters + 64;
    int32_t* pi = (int32_t*)sc.counters + 64 + TSV_MAX_ROWS * ARGMAX_SEG;
    if (!ap.sampled) {  // (the arg-max ignores penalties and truncation: choose.rs:84-88)
        hipLaunchKernelGGL(k_argmax_part, dim3(ARGMAX_SEG, ap.m), dim3(256), 0, s, target, ap.vocab, pv, pi, err);
        hipLaunchKernelGGL(k_walk_greedy, dim3(1), dim3(64), 0, s, ap_dev, pv, pi, sc.result, err, sc.host_result);
        TSV_HIP(hipGetLastError());
        return TSV_OK;
    }
    if (ap.tree) {
        if (ap.pen)
            launch_tree_sampled<true>(s, target, draft, ap_dev, ap, sc);
        else
            launch_tree_sampled<false>(s, target, draft, ap_dev, ap, sc);
        TSV_HIP(hipGetLastError());
        return TSV_OK;
    }
    if (ap.pen)
        launch_chain_sampled<true>(s, target, draft, ap_dev, ap, sc);
    else
        launch_chain_sampled<false>(s, target, draft, ap_dev, ap, sc);
    TSV_HIP(hipGetLastError());
    return TSV_OK;
}

// Draft half of a chain round: proposals[j] = q_j.draw(seed, draw_step + j) (speculative.rs:636-648),
// or the arg-max at temperature 0.  ap_dev: m = 0, k = rows, draw_step = first position.
int launch_draft_chain(hipStream_t s, const uint16_t* draft, const AcceptParams* ap_dev, const AcceptParams& ap,
                       const AcceptScratch& sc, int32_t* proposals_dev) {
    int32_t* err = &sc.result->flag;
    if (!ap.sampled) {
        float* pv = (float*)sc.counters + 64;
        int32_t* pi = (int32_t*)sc.counters + 64 + TSV_MAX_ROWS * ARGMAX_SEG;
        hipLaunchKernelGGL(k_argmax_part, dim3(ARGMAX_SEG, ap.k), dim3(256), 0, s, draft, ap.vocab, pv, pi, err);
        hipLaunchKernelGGL(k_argmax_fold, dim3(1), dim3(64), 0, s, pv, pi, ap.k, proposals_dev);
        TSV_HIP(hipGetLastError());
        return TSV_OK;
    }
    if (ap.pen)
        launch_draft_sampled<true>(s, draft, ap_dev, ap, sc, proposals_dev);
    else
        launch_draft_sampled<false>(s, draft, ap_dev, ap, sc, proposals_dev);
    TSV_HIP(hipGetLastError());
    return TSV_OK;
}

// The arg-max of `rows` logit rows (select() at temperature 0, crates/selection/src/choose.rs:61-98: the
// lowest index among equals, penalties and truncation ignored) into out[0, rows), nothing else touched but the error word, which is cleared only when
// `clear_error` says so: a chain of such calls keeps the first non-finite row's flag until the host reads it.
int launch_argmax_rows(hipStream_t s, const uint16_t* logits, int rows, int vocab, const AcceptScratch& sc, int32_t* out,
                       bool clear_error) {
    int32_t* err = (int32_t*)sc.counters;
    if (clear_error) hipLaunchKernelGGL(k_clear_result, dim3(1), dim3(64), 0, s, sc.result, err);
    float* pv = (float*)sc.counters + 64;
    int32_t* pi = (int32_t*)sc.counters + 64 + TSV_MAX_ROWS * ARGMAX_SEG;
    hipLaunchKernelGGL(k_argmax_part, dim3(ARGMAX_SEG, rows), dim3(256), 0, s, logits, vocab, pv, pi, err);
    hipLaunchKernelGGL(k_argmax_fold, dim3(1), dim3(64), 0, s, pv, pi, rows, out);
    TSV_HIP(hipGetLastError());
    return TSV_OK;
}

// The history's token statistics for a penalised round: cnt[v] bit 31 = v occurs in history[0, n),
// low bits = occurrences in history[suffix_start, n).  Token ids outside [0, vocab) are skipped
// (penalty.rs:27-33,73-78).
namespace {
__global__ void k_pen_clear(uint32_t* cnt, int words) {
    const int v = blockIdx.x * 256 + threadIdx.x;
    if (v < words) cnt[v] = 0;
}
__global__ void k_pen_count(const int32_t* history, long n, long suffix_start, int vocab, uint32_t* cnt) {
    for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long)gridDim.x * 256) {
        const int32_t t = history[i];
        if (t < 0 || t >= vocab) continue;
        atomicOr(cnt + t, 0x80000000u);
        atomicOr(pen_seen(cnt, vocab) + (t >> 5), 1u << (t & 31));
        if (i >= suffix_start) atomicAdd(cnt + t, 1u);
    }
}
}  // namespace

int launch_pen_counts(hipStream_t s, const int32_t* history_dev, long n, long suffix_start, int vocab, uint32_t* cnt) {
    const int words = pen_words(vocab);
    hipLaunchKernelGGL(k_pen_clear, dim3((words + 255) / 256), dim3(256), 0, s, cnt, words);
    if (n > 0) {
        const int blocks = (int)std::min<long>((n + 255) / 256, 256);
        hipLaunchKernelGGL(k_pen_count, dim3(blocks), dim3(256), 0, s, history_dev, n, suffix_start, vocab, cnt);
    }
    TSV_HIP(hipGetLastError());
    return TSV_OK;
}

}  // namespace tsv

// ---- greedy acceptance for callers that cannot allocate ----------------------------------------
// The greedy round of tsv_accept (arg-max per row, the walk, the stop ladder and budget) over logits
// the caller holds on the device, writing the result to device memory of the caller's, on the
// caller's stream, with no handle behind it: nothing is allocated, copied from the host or waited
// for.  The partial results of the arg-max (one value / index pair per row and vocabulary run) and
// the error flag live in a static device array; every GPU the library runs on holds its own copy
// until the process ends, and every call on a GPU shares that GPU's copy, so two calls that overlap
// on one GPU race.
static __device__ __align__(256) unsigned char scratch[4096];

namespace tsv {
namespace {

struct NoAllocScratch {
    int32_t err;
    int32_t pad[63];
    float pv[TSV_MAX_ROWS * ARGMAX_SEG];
    int32_t pi[TSV_MAX_ROWS * ARGMAX_SEG];
};
static_assert(sizeof(NoAllocScratch) <= sizeof(scratch), "the static array holds the greedy round's partial results");

// the flag must start at zero; a fill kernel rather than a memset node, so a caller may capture the call
// (on a stream of its own, with the scratch address already resolved on the device: noalloc_prepare_device)
__global__ void k_noalloc_clear(int32_t* err) {
    if (threadIdx.x == 0) *err = 0;
}

__global__ void k_walk_greedy_value(AcceptParams ap, int64_t base, const float* pv, const int32_t* pi, const int32_t* err,
                                    tsv_round_result* out) {
    __shared__ int32_t amax[TSV_MAX_ROWS];
    if ((int)threadIdx.x < ap.m) amax[threadIdx.x] = fold_argmax(pv, pi, threadIdx.x);
    __syncthreads();
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    for (int i = 0; i <= TSV_MAX_ROWS; i++) out->path[i] = 0;
    if (*err) {  // a non-finite logit (choose.rs:122-132 refuses the row): no round was judged
        out->accepted = out->committed = 0;
        out->next = -1;
        out->stopped = -1;
        out->draw_step = ap.draw_step;
        out->path_len = 0;
        out->kv_position = base;
        out->min_margin = 0.0;
        return;
    }
    const GreedyWalk g = walk_greedy(ap, amax);
    for (int i = 0; i < g.path_len; i++) out->path[i] = g.path[i];
    out->accepted = g.accepted;
    out->committed = g.committed;
    out->next = g.next;
    out->stopped = g.stopped;
    out->draw_step = ap.draw_step;
    out->path_len = g.path_len;
    out->kv_position = base + g.committed + 1;
    out->min_margin = 1.0;
}

constexpr int NOALLOC_MAX_DEVICES = 64;
// device address of `scratch` on each GPU (the array's name is only a host-side handle of the symbol)
NoAllocScratch* g_noalloc_scratch[NOALLOC_MAX_DEVICES];

int noalloc_scratch(NoAllocScratch** out) {
    int dev = -1;
    TSV_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= NOALLOC_MAX_DEVICES) {
        set_error("accept_greedy_noalloc: device ordinal outside 0..63");
        return TSV_ERR_UNSUPPORTED;
    }
    NoAllocScratch* p = __atomic_load_n(&g_noalloc_scratch[dev], __ATOMIC_ACQUIRE);
    if (!p) {
        void* sym = nullptr;
        TSV_HIP(hipGetSymbolAddress(&sym, HIP_SYMBOL(scratch)));
        if (!sym) {
            set_error("accept_greedy_noalloc: the scratch symbol has no device address");
            return TSV_ERR_DEVICE;
        }
        p = (NoAllocScratch*)sym;
        __atomic_store_n(&g_noalloc_scratch[dev], p, __ATOMIC_RELEASE);
    }
    *out = p;
    return TSV_OK;
}

}  // namespace

// Resolves the scratch array's address on the current device, so that a later tsv_accept_greedy_noalloc makes no
// runtime query (tsv_open calls this: after any handle was opened on a device the entry point can be captured).
int noalloc_prepare_device() {
    NoAllocScratch* sc = nullptr;
    return noalloc_scratch(&sc);
}
}  // namespace tsv

extern "C" int32_t tsv_accept_greedy_noalloc(void* stream, const uint16_t* logits_dev, int32_t vocab, const int32_t* feed,
                                             const int32_t* parent, int32_t m, int64_t base, const int32_t* stop_tokens,
                                             int32_t n_stop, uint64_t generated, uint64_t max_new_tokens,
                                             tsv_round_result* result_dev) {
    using namespace tsv;
    if (!logits_dev || !feed || !result_dev || (n_stop > 0 && !stop_tokens)) {
        set_error("accept_greedy_noalloc: null argument");
        return TSV_ERR_INVALID;
    }
    if (m < 1 || m > TSV_MAX_ROWS) {
        set_error("accept_greedy_noalloc: 1..16 rows (the static scratch holds the partial results of 16 rows)");
        return TSV_ERR_INVALID;
    }
    if (vocab < 1 || base < 0 || n_stop < 0 || n_stop > 16) {
        set_error("accept_greedy_noalloc: vocabulary and base must be positive / non-negative, at most 16 stop tokens");
        return TSV_ERR_INVALID;
    }
    AcceptParams ap;
    std::memset(&ap, 0, sizeof ap);
    ap.m = m;
    ap.k = m - 1;
    ap.vocab = vocab;
    ap.tree = parent != nullptr;
    ap.n_stop = n_stop;
    for (int i = 0; i < m; i++) {
        if (parent && (i == 0 ? parent[0] != -1 : (parent[i] < 0 || parent[i] >= i))) {
            set_error("accept_greedy_noalloc: parent[0] must be -1 and parent[s] in [0, s)");
            return TSV_ERR_INVALID;
        }
        ap.feed[i] = feed[i];
        ap.parent[i] = parent ? parent[i] : i - 1;
    }
    for (int i = 0; i < n_stop; i++) ap.stop_tokens[i] = stop_tokens[i];
    ap.generated = generated;
    ap.max_new_tokens = max_new_tokens;
    NoAllocScratch* sc = nullptr;
    int rc = noalloc_scratch(&sc);
    if (rc) return rc;
    hipStream_t s = (hipStream_t)stream;
    hipLaunchKernelGGL(k_noalloc_clear, dim3(1), dim3(64), 0, s, &sc->err);
    hipLaunchKernelGGL(k_argmax_part, dim3(ARGMAX_SEG, m), dim3(256), 0, s, logits_dev, vocab, sc->pv, sc->pi, &sc->err);
    hipLaunchKernelGGL(k_walk_greedy_value, dim3(1), dim3(64), 0, s, ap, base, sc->pv, sc->pi, &sc->err, result_dev);
    TSV_HIP(hipGetLastError());
    return TSV_OK;
}

// Test hook: the number of walk launches a sampled tree round of this shape gets (host arithmetic only).
extern "C" int32_t tsv_tree_walk_bound(const int32_t* parent, int32_t m) {
    using namespace tsv;
    if (!parent || m < 1 || m > TSV_MAX_ROWS || parent[0] != -1) {
        set_error("tree_walk_bound: 1..16 slots, parent[0] == -1");
        return -1;
    }
    for (int i = 1; i < m; i++)
        if (parent[i] < 0 || parent[i] >= i) {
            set_error("tree_walk_bound: parent[s] must lie in [0, s)");
            return -1;
        }
    return tree_walk_bound(parent, m);
}
