// A chain of transformer blocks on one token grid, issued by one call (gfx950).
//
// Host code: the launches of a block are a fixed sequence of this library's own entry points, but issued one by one
// from Python every launch costs 25 - 30 us of interpreter time (allocating its outputs, checking its operands,
// converting twenty arguments), more than most of them run for below a batch of some hundred pictures.  Here the
// caller hands over three buffers and a table of parameter addresses once per call, and a launch costs what
// hipLaunchKernel costs.  The kernels and their order are those that engine.block_forward issues, but for what it leaves to
// separate launches: scatter-back, sampling and LayerNorm where regions are few enough (vtdge_region_step, the same bits), the splits
// of several blocks' fp32 weights (vtdge_linear_split_set) and the packing of their reduction weights (vtdge_layernorm_patch_pack).
//
// Buffers: `ints` holds the small results a caller may read later (gate logits, offsets, lengths, and the status words
// of the chained scatter-backs), `big` the tokens between blocks, the packed queries before and after the block and
// the patch descriptors, `scratch` everything that dies inside the call.  vtdge_chain_layout says how large they are
// and where each block's results lie.
#include "common.h"
#include <unistd.h>

namespace vtdge {

// order of a block's entries in the parameter table
enum {
    P_N1W, P_N1B, P_N2W, P_N2B, P_RW, P_RB, P_SPLITS, P_QW, P_QB, P_KVW, P_KVB, P_PROJW, P_PROJB, P_FC1W, P_FC1B,
    P_FC2W, P_FC2B, P_QP, P_KVP, P_PROJP, P_FC1P, P_FC2P, P_QFW, P_QFR, P_QFP, P_KVFW, P_KVFR, P_KVFP, P_FC1FW,
    P_FC1FR, P_FC1FP, P_SRW, P_SRB, P_SRNW, P_SRNB, P_COUNT
};
static_assert(P_COUNT == VTDGE_CHAIN_PARAMS, "the parameter table's documented length");

// first `n` rows of every sample of x [B, N, C] = rows [n, C] (the class tokens), 16 bytes a lane; `words` 64-bit words at
// `clear` = 0 (the status words of the scatter-backs)
__global__ __launch_bounds__(256) void front_rows_kernel(u32x4 *__restrict__ x, const u32x4 *__restrict__ rows,
                                                         int64_t sample_vecs, int vecs, int64_t total,
                                                         unsigned long long *__restrict__ clear, int64_t words)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < total) x[i / vecs * sample_vecs + i % vecs] = rows[i % vecs];
    if (i < words) clear[i] = 0ull;
}

constexpr int LINEARS = 5;         // of a block: q, kv, proj, fc1, fc2, as in the parameter table

struct ChainPlan {
    int64_t rows, cap, regions;
    int esz, N, n_kv;              // tokens per sample, keys per sample
    bool folded;                   // norms folded into weight-stationary Linears, chained scatter-back (384-channel bf16)
    bool by_region, pack;          // compress by region; the scatter-back packs the next block's queries
    bool step;                     // vtdge_region_step joins the blocks: the scatter-back also writes what the next block's norm1 wants
    bool tail;                     // narrow bf16 rows: everything behind attention as one kernel
    bool ln_kvq, ln_fc1;           // few rows: norm1 inside the kv and q Linear, norm2 inside fc1
    bool ln_sr;                    // many rows: norm1 inside the spatial reduction
    int64_t ws_words;
    bool split[LINEARS];           // fp32 Linears on split weights
    int split_blocks;              // blocks whose weights are split in one launch, 0: none are
    int64_t split_at[LINEARS], split_sz, split0;                         // in `scratch`, of one block
    // byte offsets
    int64_t ints_total, big_total, scratch_total;
    int64_t gate0, off0, len0, ws0, gate_sz, off_sz, len_sz, ws_sz;      // in `ints`, block i at start + i * size
    int64_t tok0, comp0, q20, pat0, tok_sz, row_sz, pat_sz;              // in `big`
    int64_t srw_sz;                // a packed weight of the spatial reduction
    int64_t xln, red, srw, kv, comp_ln, q, o, q1, q1_ln, hid, rec_x[2], rec_c[2], rec2, idx[2], cnt[2], rrows[2];   // in `scratch`
};

#define VT_TRY(expr)                      \
    do {                                  \
        const int vt_rc = (expr);         \
        if (vt_rc != VTDGE_OK) return vt_rc; \
    } while (0)

static int64_t align256(int64_t v) { return (v + 255) / 256 * 256; }

// A block's Linears in the order of the parameter table: what they multiply, and whether on split weights where that is faster
struct SplitShape {
    int64_t rows;
    int N, K;
    bool wanted;
};
static SplitShape split_shape(const vtdge_chain *c, const ChainPlan &p, int linear)
{
    const bool f32 = c->dtype == VTDGE_F32;
    switch (linear) {
    case 0: return {p.cap, c->C, c->C, f32 && !p.ln_kvq};
    case 1: return {(int64_t)c->B * p.n_kv, 2 * c->C, c->C, f32 && !p.ln_kvq};
    case 2: return {p.cap, c->C, c->C, f32};
    case 3: return {p.cap, c->hidden, c->C, f32 && !p.ln_fc1};
    default: return {p.cap, c->C, c->hidden, f32};
    }
}

// Split weights are made anew by every call: it multiplies by the weights as they are when it runs, in a replayed graph and
// beside calls on other streams too.  As many blocks a launch as stay in the last-level cache until they are read.  GPU time of
// a forward at 256 px, us, without split weights / split by the call / kept from an earlier one (pictures, channels): 128, 192:
// 3367 / 3023 / 3001; 12, 384: 1730 / 1528 / 1485; 32, 384: 2880 / 2546 / 2500; 8, 768: 3162 / 2863 / 2668; 2, 768: 1804 / 1741 /
// 1685.
constexpr int64_t SPLIT_ROOM = 64 << 20;
constexpr int SPLIT_BLOCKS = 16;

static int split_block_weights(const vtdge_chain *c, const ChainPlan &p, const void *const *params, int first, char *scratch,
                               void *stream)
{
    const void *W[SPLIT_BLOCKS * LINEARS];
    int32_t N[SPLIT_BLOCKS * LINEARS], K[SPLIT_BLOCKS * LINEARS];
    int64_t at[SPLIT_BLOCKS * LINEARS];
    int count = 0;
    for (int b = 0; b < p.split_blocks && first + b < c->depth; b++)
        for (int j = 0; j < LINEARS; j++) {
            if (!p.split[j]) continue;
            const SplitShape w = split_shape(c, p, j);
            W[count] = params[(int64_t)(first + b) * P_COUNT + P_QW + 2 * j];
            N[count] = w.N;
            K[count] = w.K;
            at[count++] = b * p.split_sz + p.split_at[j];
        }
    return vtdge_linear_split_set(W, N, K, at, count, scratch + p.split0, stream);
}

static int plan_chain(const vtdge_chain *c, ChainPlan &p)
{
    VT_REQUIRE(c != nullptr, VTDGE_ERR_ARG, "chain: NULL description");
    VT_REQUIRE(c->dtype == VTDGE_F32 || c->dtype == VTDGE_BF16, VTDGE_ERR_ARG, "chain: unknown dtype %d", c->dtype);
    VT_REQUIRE(c->B > 0 && c->H > 0 && c->W > 0 && c->C > 0 && c->heads > 0 && c->hidden > 0 && c->extra >= 0 &&
                   c->S > 0 && c->S <= VTDGE_MAX_SPLITS && c->depth > 0 && c->sr > 0,
               VTDGE_ERR_ARG, "chain: bad sizes");
    VT_REQUIRE(c->H % 4 == 0 && c->W % 4 == 0, VTDGE_ERR_UNSUPPORTED, "chain: a %dx%d grid does not tile into regions of 4",
               c->H, c->W);
    VT_REQUIRE(c->C % c->heads == 0, VTDGE_ERR_ARG, "chain: %d channels do not divide into %d heads", c->C, c->heads);
    VT_REQUIRE(c->sr == 1 || (c->extra == 0 && c->H % c->sr == 0 && c->W % c->sr == 0), VTDGE_ERR_UNSUPPORTED,
               "chain: a %dx%d grid with %d extra tokens has no spatial reduction by %d", c->H, c->W, c->extra, c->sr);
    p.esz = c->dtype == VTDGE_BF16 ? 2 : 4;
    p.N = c->extra + c->H * c->W;
    p.n_kv = c->sr > 1 ? (c->H / c->sr) * (c->W / c->sr) : p.N;
    p.rows = p.cap = (int64_t)c->B * p.N;
    p.regions = (int64_t)c->B * (c->H / 4) * (c->W / 4);
    const int nvec = c->C * p.esz / 16;
    VT_REQUIRE((c->C * p.esz) % 16 == 0 && (c->hidden * p.esz) % 16 == 0, VTDGE_ERR_UNSUPPORTED,
               "chain: rows of %d / %d values are no whole 16-byte vectors", c->C, c->hidden);
    p.by_region = c->splits_124 && nvec > 32 && nvec <= 64 && c->extra <= 64 && p.regions <= 65536 && p.rows < (1 << 24);
    p.folded = p.by_region && c->dtype == VTDGE_BF16 && c->C == 384 && p.rows >= 2048 && c->sr == 1 &&
               c->hidden % 384 == 0 && c->hidden <= 3072;
    p.ln_kvq = !p.folded && c->sr == 1 && vtdge_layernorm_linear_wanted(p.rows, 2 * c->C, p.cap, c->C, c->C, c->dtype);
    p.ln_sr = c->sr > 1 && vtdge_layernorm_patch_linear_wanted(c->B, c->H, c->W, c->C, c->sr, c->dtype);
    p.tail = vtdge_block_tail_wanted(p.rows, c->C, c->hidden, c->dtype);
    p.ln_fc1 = !p.folded && !p.tail && vtdge_layernorm_linear_wanted(p.cap, c->hidden, 0, 0, c->C, c->dtype);
    p.step = c->depth > 1 && c->splits_124 && vtdge_region_step_fits(c->B, c->H, c->W, c->C, c->extra, c->dtype);
    p.pack = p.step || (p.folded && c->depth > 1 && p.regions % 4 == 0);
    p.ws_words = p.step   ? vtdge_region_step_workspace(c->B, c->H, c->W) / 8
                 : p.pack ? vtdge_decompress_router_compress_workspace(c->B, c->H, c->W, 4) / 8
                          : 0;

    int64_t at = 0;
    auto take = [&](int64_t bytes) {
        const int64_t o = at;
        at += align256(bytes);
        return o;
    };
    p.gate_sz = align256(p.regions * c->S * p.esz);
    p.off_sz = align256((c->B + 1) * 8);
    p.len_sz = align256(c->B * 8);
    p.ws_sz = p.ws_words * 8;                                   // contiguous: cleared as one range
    p.gate0 = take(p.gate_sz * c->depth);
    p.off0 = take(p.off_sz * c->depth);
    p.len0 = take(p.len_sz * c->depth);
    p.ws0 = take(p.ws_sz * (c->depth - 1));
    p.ints_total = at;
    at = 0;
    p.row_sz = p.tok_sz = align256(p.rows * c->C * p.esz);
    p.pat_sz = align256(p.cap * 32);
    p.tok0 = take(p.tok_sz * (c->depth - 1));
    p.comp0 = take(p.row_sz * c->depth);
    p.q20 = take(p.row_sz * c->depth);
    p.pat0 = take(p.pat_sz * c->depth);
    p.big_total = at;
    at = 0;
    const int64_t row = p.rows * c->C * p.esz;
    p.xln = p.folded ? 0 : take(row);
    p.red = c->sr > 1 ? take((int64_t)c->B * p.n_kv * c->C * p.esz) : 0;
    p.srw_sz = (int64_t)c->sr * c->sr * c->C * c->C * p.esz;
    p.srw = p.ln_sr ? take(c->depth * p.srw_sz) : 0;
    p.kv = take(2 * (int64_t)c->B * p.n_kv * c->C * p.esz);
    p.comp_ln = p.folded ? 0 : take(row);
    p.q = take(row);
    p.o = take(row);
    p.q1 = p.tail ? 0 : take(row);
    p.q1_ln = p.folded || p.tail ? 0 : take(row);
    p.hid = p.tail ? 0 : take(p.cap * c->hidden * p.esz);
    p.rec2 = p.folded ? take(p.rows * 32) : 0;
    for (int i = 0; i < 2; i++) {
        p.rec_x[i] = p.folded ? take(p.rows * 32) : 0;
        p.rec_c[i] = p.folded ? take(p.rows * 32) : 0;
        p.idx[i] = take(p.regions * 8);
        p.cnt[i] = take((p.regions + 15) / 16 * 16);
        p.rrows[i] = take(p.regions * 4);
    }
    p.split_sz = p.split_blocks = 0;
    for (int j = 0; j < LINEARS; j++) {
        const SplitShape w = split_shape(c, p, j);
        int64_t bytes = 0;
        if (w.wanted && vtdge_linear_split_wanted(w.rows, w.N, w.K)) VT_TRY(vtdge_linear_split_size(w.N, w.K, &bytes));
        p.split[j] = bytes > 0;
        p.split_at[j] = p.split_sz;
        p.split_sz += align256(bytes);
    }
    if (p.split_sz > 0) {
        const int64_t fit = SPLIT_ROOM / p.split_sz;
        p.split_blocks = fit < 1 ? 1 : fit > SPLIT_BLOCKS ? SPLIT_BLOCKS : (int)fit;
        if (p.split_blocks > c->depth) p.split_blocks = c->depth;
        p.split0 = take(p.split_sz * p.split_blocks);
    }
    p.scratch_total = at;
    return VTDGE_OK;
}

// A pair of events per host thread and device for the fork to the side stream and the join behind it; each is recorded
// anew before it is waited for.  They end with their thread (not in a process forked from it, where the runtime is not to be
// called any more).
struct ForkEvents {
    hipEvent_t fork[16] = {}, join[16] = {};
    const pid_t owner = getpid();
    ~ForkEvents()
    {
        if (getpid() != owner) return;
        for (int i = 0; i < 16; i++) {
            if (fork[i] != nullptr) (void)hipEventDestroy(fork[i]);
            if (join[i] != nullptr) (void)hipEventDestroy(join[i]);
        }
    }
};
static int fork_events(hipEvent_t &fork, hipEvent_t &join)
{
    static thread_local ForkEvents ev;
    int dev = 0;
    VT_REQUIRE(hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < 16, VTDGE_ERR_LAUNCH, "chain: no device");
    if (ev.fork[dev] == nullptr)
        VT_REQUIRE(hipEventCreateWithFlags(&ev.fork[dev], hipEventDisableTiming) == hipSuccess &&
                       hipEventCreateWithFlags(&ev.join[dev], hipEventDisableTiming) == hipSuccess,
                   VTDGE_ERR_LAUNCH, "chain: cannot create an event");
    fork = ev.fork[dev];
    join = ev.join[dev];
    return VTDGE_OK;
}

// The side stream of a chain: begin() lets it start behind the main stream, end() orders the main stream behind it.  Every
// way out of the chain goes through end(), a failed launch's too: the caller frees the buffers when the call returns, on the
// main stream, and a capture must not end with a stream that was forked and not joined.
struct SideStream {
    hipStream_t main, side;
    hipEvent_t fork = nullptr, join = nullptr;
    bool open = false;
    SideStream(void *m, void *s) : main((hipStream_t)m), side((hipStream_t)s) {}
    ~SideStream() { end(); }
    int begin()
    {
        if (fork == nullptr) {
            const int rc = fork_events(fork, join);
            if (rc != VTDGE_OK) return rc;
        }
        VT_REQUIRE(hipEventRecord(fork, main) == hipSuccess && hipStreamWaitEvent(side, fork, 0) == hipSuccess, VTDGE_ERR_LAUNCH,
                   "chain: cannot fork to the side stream");
        open = true;
        return VTDGE_OK;
    }
    int end()
    {
        if (!open) return VTDGE_OK;
        open = false;
        VT_REQUIRE(hipEventRecord(join, side) == hipSuccess && hipStreamWaitEvent(main, join, 0) == hipSuccess, VTDGE_ERR_LAUNCH,
                   "chain: cannot join the side stream");
        return VTDGE_OK;
    }
};

static int run_chain(const vtdge_chain *c, const ChainPlan &p, const void *const *params, const void *front, char *x0,
                     char *ints, char *big, char *scratch, char *out, void *stream, void *side)
{
    const int B = c->B, H = c->H, W = c->W, C = c->C, S = c->S, extra = c->extra, dt = c->dtype, N = p.N, esz = p.esz;
    const int d = C / c->heads;
    char *x = x0;
    int cur = 0;                 // which of the double buffers holds what the previous block left for this one
    bool routed = false, packed = false, have_counts = false;
    SideStream beside(stream, side);
    if (p.ln_sr) {
        // the weights of all blocks that use them packed at once: a launch for sixteen
        const int blocks = p.pack ? 1 : c->depth;
        for (int at = 0; at < blocks; at += 16) {
            const void *weights[16];
            int n = 0;
            for (; n < 16 && at + n < blocks; n++) weights[n] = params[(int64_t)(at + n) * P_COUNT + P_SRW];
            VT_TRY(vtdge_layernorm_patch_pack(weights, n, scratch + p.srw + at * p.srw_sz, C, c->sr, stream));
        }
    }

    for (int i = 0; i < c->depth; i++) {
        const void *const *P = params + (int64_t)i * P_COUNT;
        const void *const *Q = i + 1 < c->depth ? P + P_COUNT : nullptr;      // the next block
        char *gate = ints + p.gate0 + i * p.gate_sz;
        int64_t *offsets = (int64_t *)(ints + p.off0 + i * p.off_sz), *lengths = (int64_t *)(ints + p.len0 + i * p.len_sz);
        char *comp = big + p.comp0 + i * p.row_sz, *q2 = big + p.q20 + i * p.row_sz;
        int64_t *patches = (int64_t *)(big + p.pat0 + i * p.pat_sz);
        const int64_t *live = offsets + B;
        const int64_t *splits = (const int64_t *)P[P_SPLITS];
        int64_t *idx = (int64_t *)(scratch + p.idx[cur]), *nidx = (int64_t *)(scratch + p.idx[cur ^ 1]);
        uint8_t *cnt = (uint8_t *)(scratch + p.cnt[cur]), *ncnt = (uint8_t *)(scratch + p.cnt[cur ^ 1]);
        int32_t *rr = (int32_t *)(scratch + p.rrows[cur]), *nrr = (int32_t *)(scratch + p.rrows[cur ^ 1]);
        char *recx = scratch + p.rec_x[cur], *nrecx = scratch + p.rec_x[cur ^ 1];
        char *recc = scratch + p.rec_c[cur], *nrecc = scratch + p.rec_c[cur ^ 1];
        char *kv = scratch + p.kv, *q = scratch + p.q, *o = scratch + p.o, *q1 = scratch + p.q1, *hid = scratch + p.hid;
        char *xout = Q ? big + p.tok0 + i * p.tok_sz : out;
        char *ngate = Q ? ints + p.gate0 + (i + 1) * p.gate_sz : nullptr;
        // the copy of a weight for so many rows: bf16 packed (from 2048 rows on), fp32 split
        auto copy_for = [&](int which, int64_t rows) -> const void * {
            if (dt != VTDGE_F32) return rows >= 2048 ? P[which] : nullptr;
            const int j = which - P_QP;
            return p.split[j] ? scratch + p.split0 + i % p.split_blocks * p.split_sz + p.split_at[j] : nullptr;
        };
        auto pk = [&](int which) { return copy_for(which, p.rows); };

        if (p.folded) {
            if (i == 0) {
                VT_TRY(vtdge_router_stats(x, front, P[P_RW], P[P_RB], gate, idx, recx, c->eps1, splits, cnt,
                                          p.pack ? ints + p.ws0 : nullptr, p.pack ? p.ws_words * (c->depth - 1) : 0, B, H,
                                          W, C, extra, 4, S, dt, stream));
                routed = have_counts = true;
            }
            if (!packed)
                VT_TRY(vtdge_compress_regions(x, idx, splits, cnt, comp, recc, c->eps1, patches, p.cap, offsets, lengths,
                                              rr, B, H, W, C, extra, 4, S, dt, stream));
            VT_TRY(vtdge_linear_layernorm_pair(x, C, recx, P[P_KVFW], P[P_KVFP], P[P_KVFR], kv, 2 * C, nullptr, p.rows,
                                               2 * C, comp, C, recc, P[P_QFW], P[P_QFP], P[P_QFR], q, C, live, p.cap, C,
                                               C, dt, stream));
        } else {
            const int64_t words = p.step ? p.ws_words * (c->depth - 1) : 0;
            if (i == 0 && (front != nullptr || words > 0)) {
                const int vecs = extra * C * esz / 16;
                const int64_t total = front != nullptr ? (int64_t)B * vecs : 0;
                note_kernel(reinterpret_cast<const void *>(front_rows_kernel));
                front_rows_kernel<<<(unsigned)ceil_div(total > words ? total : words, 256), 256, 0, (hipStream_t)stream>>>(
                    (u32x4 *)x, (const u32x4 *)front, (int64_t)N * C * esz / 16, vecs, total,
                    (unsigned long long *)(ints + p.ws0), words);
                VT_TRY(check_launch("chain"));
            }
            char *comp_ln = p.ln_kvq ? nullptr : scratch + p.comp_ln, *xln = scratch + p.xln;
            if (!packed) {
                void *routing = stream;
                if (side != nullptr) {
                    // the routing chain beside the key/value chain, joined before attention
                    routing = side;
                    VT_TRY(beside.begin());
                }
                if (!routed)
                    VT_TRY(vtdge_router(x, P[P_RW], P[P_RB], gate, idx, B, H, W, C, extra, 4, S, dt, routing));
                if (p.by_region) {
                    VT_TRY(vtdge_compress_regions(x, idx, splits, have_counts ? cnt : nullptr, comp, nullptr, 0.f, patches,
                                                  p.cap, offsets, lengths, rr, B, H, W, C, extra, 4, S, dt, routing));
                    if (comp_ln != nullptr)
                        VT_TRY(vtdge_layernorm(comp, P[P_N1W], P[P_N1B], comp_ln, live, p.cap, C, c->eps1, dt, routing));
                } else {
                    VT_TRY(vtdge_index_to_patch(idx, splits, B, H / 4, W / 4, S, 4, extra, patches, p.cap, offsets, lengths,
                                                routing));
                    VT_TRY(vtdge_compress(x, patches, live, p.cap, comp, comp_ln, comp_ln ? P[P_N1W] : nullptr,
                                          comp_ln ? P[P_N1B] : nullptr, c->eps1, B, N, C, W, extra, dt, routing));
                }
            }
            if (p.split_blocks > 0 && i % p.split_blocks == 0)       // on the stream of the Linears that read them, and read the last
                VT_TRY(split_block_weights(c, p, params, i, scratch, stream));
            if (p.ln_kvq && packed) {
                // the scatter-back has left norm1 of tokens and queries
                VT_TRY(vtdge_linear_pair(scratch + p.xln, C, P[P_KVW], P[P_KVB], kv, nullptr, p.rows, 2 * C, scratch + p.comp_ln,
                                         C, P[P_QW], P[P_QB], q, live, p.cap, C, C, dt, stream));
            } else if (p.ln_kvq) {
                VT_TRY(vtdge_layernorm_linear(x, C, P[P_KVW], P[P_KVB], kv, nullptr, p.rows, 2 * C, comp, C, P[P_QW], P[P_QB],
                                              q, live, p.cap, C, P[P_N1W], P[P_N1B], c->eps1, C, VTDGE_ACT_NONE, dt,
                                              stream));
            } else {
                const bool ln_sr = p.ln_sr && !packed;
                if (!packed && !ln_sr)
                    VT_TRY(vtdge_layernorm(x, P[P_N1W], P[P_N1B], xln, nullptr, p.rows, C, c->eps1, dt, stream));
                char *src = xln;
                if (c->sr > 1) {
                    char *red = scratch + p.red;
                    if (ln_sr)
                        VT_TRY(vtdge_layernorm_patch_linear(x, P[P_N1W], P[P_N1B], c->eps1, scratch + p.srw + i * p.srw_sz,
                                                            P[P_SRB], P[P_SRNW], P[P_SRNB], c->sr_eps, xln, B, H, W, C, c->sr,
                                                            dt, stream));
                    else {
                        VT_TRY(vtdge_patch_linear(xln, P[P_SRW], P[P_SRB], red, B, H, W, C, c->sr, C, dt, stream));
                        // the normalised rows take the place of LN1(x), which nothing reads any more
                        VT_TRY(vtdge_layernorm(red, P[P_SRNW], P[P_SRNB], xln, nullptr, (int64_t)B * p.n_kv, C, c->sr_eps, dt,
                                               stream));
                    }
                }
                const int64_t kv_rows = (int64_t)B * p.n_kv;
                VT_TRY(vtdge_linear_prepacked(src, C, P[P_KVW], copy_for(P_KVP, kv_rows), P[P_KVB], nullptr, 0, kv,
                                              2 * C, nullptr, kv_rows, 2 * C, C, VTDGE_ACT_NONE, dt, stream));
                VT_TRY(beside.end());
                VT_TRY(vtdge_linear_prepacked(comp_ln, C, P[P_QW], pk(P_QP), P[P_QB], nullptr, 0, q, C, live, p.cap, C, C,
                                              VTDGE_ACT_NONE, dt, stream));
            }
        }
        VT_TRY(vtdge_sparse_attention(q, C, d, kv, kv + (int64_t)C * esz, (int64_t)p.n_kv * 2 * C, 2 * C, d, offsets, o, C,
                                      d, B, c->heads, d, p.n_kv, N, c->scale, dt, stream));
        if (p.tail) {
            VT_TRY(vtdge_block_tail(o, comp, P[P_PROJW], P[P_PROJB], P[P_N2W], P[P_N2B], c->eps2, P[P_FC1W], P[P_FC1B],
                                    P[P_FC2W], P[P_FC2B], q2, live, p.cap, C, c->hidden, dt, stream));
        } else if (p.folded) {
            VT_TRY(vtdge_linear_stats(o, C, P[P_PROJW], P[P_PROJP], P[P_PROJB], comp, C, q1, C, scratch + p.rec2, c->eps2,
                                      live, p.cap, C, C, dt, stream));
            VT_TRY(vtdge_linear_layernorm(q1, C, scratch + p.rec2, P[P_FC1FW], P[P_FC1FP], P[P_FC1FR], hid, c->hidden,
                                          live, p.cap, c->hidden, C, VTDGE_ACT_GELU, dt, stream));
        } else {
            char *q1_ln = scratch + p.q1_ln;
            VT_TRY(vtdge_linear_prepacked(o, C, P[P_PROJW], pk(P_PROJP), P[P_PROJB], comp, C, q1, C, live, p.cap, C, C,
                                          VTDGE_ACT_NONE, dt, stream));
            if (p.ln_fc1) {
                VT_TRY(vtdge_layernorm_linear(q1, C, P[P_FC1W], P[P_FC1B], hid, live, p.cap, c->hidden, nullptr, 0, nullptr,
                                              nullptr, nullptr, nullptr, 0, 0, P[P_N2W], P[P_N2B], c->eps2, C,
                                              VTDGE_ACT_GELU, dt, stream));
            } else {
                VT_TRY(vtdge_layernorm(q1, P[P_N2W], P[P_N2B], q1_ln, live, p.cap, C, c->eps2, dt, stream));
                VT_TRY(vtdge_linear_prepacked(q1_ln, C, P[P_FC1W], pk(P_FC1P), P[P_FC1B], nullptr, 0, hid, c->hidden, live,
                                              p.cap, c->hidden, C, VTDGE_ACT_GELU, dt, stream));
            }
        }
        if (!p.tail)
            VT_TRY(vtdge_linear_prepacked(hid, c->hidden, P[P_FC2W], pk(P_FC2P), P[P_FC2B], q1, C, q2, C, live, p.cap, C,
                                          c->hidden, VTDGE_ACT_NONE, dt, stream));
        if (Q == nullptr) {
            VT_TRY(vtdge_decompress(q2, comp, patches, live, p.cap, x, xout, B, N, C, W, extra, dt, stream));
            break;
        }
        // where this block's regions lie: left by compress by region (or by the scatter-back before it) with the counts
        const bool placed = (p.by_region || p.step) && have_counts;
        const int64_t *nsplits = p.by_region || p.step ? (const int64_t *)Q[P_SPLITS] : nullptr;
        if (p.step) {
            const bool normed = !p.folded;
            VT_TRY(vtdge_region_step(
                q2, comp, idx, splits, offsets, placed ? rr : nullptr, placed ? cnt : nullptr, x, xout, Q[P_RW], Q[P_RB], ngate,
                nidx, nsplits, ncnt, p.folded ? nrecx : nullptr, normed ? scratch + p.xln : nullptr,
                normed ? Q[P_N1W] : nullptr, normed ? Q[P_N1B] : nullptr, c->eps1, big + p.comp0 + (i + 1) * p.row_sz,
                p.folded ? nrecc : nullptr, normed ? scratch + p.comp_ln : nullptr,
                (int64_t *)(big + p.pat0 + (i + 1) * p.pat_sz), p.cap, (int64_t *)(ints + p.off0 + (i + 1) * p.off_sz), nrr,
                ints + p.ws0 + i * p.ws_sz, p.ws_sz, B, H, W, C, extra, S, S, dt, stream));
        } else if (p.pack)
            VT_TRY(vtdge_decompress_router_compress(
                q2, comp, idx, splits, offsets, x, xout, Q[P_RW], Q[P_RB], ngate, nidx, nrecx, c->eps1, nsplits, ncnt,
                placed ? rr : nullptr, placed ? cnt : nullptr, big + p.comp0 + (i + 1) * p.row_sz, nrecc, c->eps1,
                (int64_t *)(big + p.pat0 + (i + 1) * p.pat_sz), p.cap, (int64_t *)(ints + p.off0 + (i + 1) * p.off_sz), nrr,
                ints + p.ws0 + i * p.ws_sz, p.ws_sz, 0, B, H, W, C, extra, 4, S, S, dt, stream));
        else
            VT_TRY(vtdge_decompress_router(q2, comp, idx, splits, offsets, x, xout, Q[P_RW], Q[P_RB], ngate, nidx,
                                           p.folded ? nrecx : nullptr, c->eps1, nsplits, p.by_region ? ncnt : nullptr,
                                           placed ? rr : nullptr, placed ? cnt : nullptr, B, H, W, C, extra, 4, S, S, dt,
                                           stream));
        routed = true;
        packed = p.pack;
        have_counts = p.by_region || p.step;
        x = xout;
        cur ^= 1;
    }
    return VTDGE_OK;
}

}  // namespace vtdge

using namespace vtdge;

extern "C" int vtdge_chain_layout(const vtdge_chain *chain, int64_t *layout_host)
{
    VT_REQUIRE(layout_host != nullptr, VTDGE_ERR_ARG, "chain: NULL layout");
    ChainPlan p;
    VT_TRY(plan_chain(chain, p));
    int64_t *l = layout_host;
    l[0] = p.ints_total;
    l[1] = p.big_total;
    l[2] = p.scratch_total;
    l[3] = p.pack ? p.ws_sz : 0;
    l[4] = p.folded ? 1 : 0;
    for (int i = 0; i < chain->depth; i++) {
        int64_t *b = l + VTDGE_CHAIN_LAYOUT_HEAD + (int64_t)i * VTDGE_CHAIN_LAYOUT_BLOCK;
        b[0] = p.gate0 + i * p.gate_sz;
        b[1] = p.off0 + i * p.off_sz;
        b[2] = p.pack && i > 0 ? -1 : p.len0 + i * p.len_sz;
        b[3] = p.pack && i > 0 ? p.ws0 + (i - 1) * p.ws_sz : -1;
        b[4] = i > 0 ? p.tok0 + (i - 1) * p.tok_sz : -1;
        b[5] = p.comp0 + i * p.row_sz;
        b[6] = p.q20 + i * p.row_sz;
        b[7] = p.pat0 + i * p.pat_sz;
    }
    return VTDGE_OK;
}

extern "C" int vtdge_chain_forward(const vtdge_chain *chain, const void *const *params_host, const void *front_rows,
                                   void *x, void *ints, void *big, void *scratch, void *out, void *stream,
                                   void *side_stream)
{
    VT_REQUIRE(params_host && x && ints && big && scratch && out, VTDGE_ERR_ARG, "chain: NULL operand");
    ChainPlan p;
    VT_TRY(plan_chain(chain, p));
    VT_REQUIRE(front_rows == nullptr || chain->extra > 0, VTDGE_ERR_ARG, "chain: front rows without extra tokens");
    VT_REQUIRE((((uintptr_t)x | (uintptr_t)ints | (uintptr_t)big | (uintptr_t)scratch | (uintptr_t)out |
                 (uintptr_t)front_rows) & 15) == 0,
               VTDGE_ERR_ARG, "chain: buffers must be 16-byte aligned");
    for (int i = 0; i < chain->depth; i++) {
        const void *const *P = params_host + (int64_t)i * P_COUNT;
        bool ok = true;
        for (int k = P_N1W; k <= P_FC2B; k++) ok = ok && (P[k] != nullptr || k == P_QB || k == P_KVB || k == P_PROJB || k == P_FC1B || k == P_FC2B);
        if (p.folded) ok = ok && P[P_QFW] && P[P_QFR] && P[P_KVFW] && P[P_KVFR] && P[P_FC1FW] && P[P_FC1FR];
        if (chain->sr > 1) ok = ok && P[P_SRW] && P[P_SRB] && P[P_SRNW] && P[P_SRNB];
        VT_REQUIRE(ok, VTDGE_ERR_ARG, "chain: block %d lacks a parameter", i);
    }
    return run_chain(chain, p, params_host, front_rows, (char *)x, (char *)ints, (char *)big, (char *)scratch, (char *)out,
                     stream, p.folded || p.ln_kvq ? nullptr : side_stream);
}
