// Gradients of the sparse attention of packed queries (gfx950): dQ, dK, dV from Q, K, V and the output's gradient.
//
// The composition this stands in for (a product of queries and keys, a softmax, a product with the values, and their
// five products backward: vtpack/models/dge/deit_dge.py:86-95) keeps four score-sized tensors in HBM, [heads, L, n] each:
// 90 MB apiece at 14500 queries, 6 heads and 257 keys in bf16, against 45 MB of operands.  Here scores exist in registers
// only: they are worked out again from Q and K where a gradient needs them,
//   P = exp2(scale log2e q.k - m) / s,   dP = dO.v,   dS = P (dP - delta) scale,   delta = sum_k P dP,
//   dQ = dS K,   dV = P^T dO,   dK = dS^T Q.
// Two kernels, no atomics, so the result is the same bytes on every call: one over query tiles, which first finds m (the
// row's maximum in log2 units), s (the sum of its exponentials) and delta and leaves them for the other, over key tiles.
// m and 1 / s stay apart: added up to m + log2(s), rounded at its own size (8 to 9 with 257 keys), they would put 2e-7 into
// every P of a row and the subtraction as much again (fp32, 64 samples, 3 heads, 257 keys, unit normals: relative error of dV
// 4.2e-7 against 3.0e-7 this way; a softmax and products 2.9e-7).  In bf16, where P is rounded to 2^-9, they are added up.
// Every exponent is one fused multiply-add: the passes have to see the same e, or dS does not add up to zero.
// delta equals dO.O, but is summed from the P and dP that dS is made of: a row of dS then adds up to zero within fp32, where
// dO times an output rounded to bf16 leaves a remainder that multiplies the mean key (relative error of dQ with a common
// component of twice the spread in keys and values: 5.1e-2 from the rounded output, 3.6e-3 this way).
//
// Both are one scheme.  A wave keeps 16 rows of two operands in registers (Q and dO, or K and V) and walks the rows of
// the other two, which the workgroup's four waves share through LDS in stages of 32 by direct loads (two buffers; over the queries
// three or four, statistics among them: us, 64 samples, 3 heads, 257 keys, fp32 69.6 -> 60.7, 128, 6, bf16 46.2 -> 41.4).  With
// the walked rows as rows of v_mfma_f32_16x16 tiles and the kept ones as columns, lane (l = lane % 16, g = lane / 16) holds
// the score of walked rows 4 g + r (r < 4) with kept row l: the operand layout of the products over the walked rows, so
// nothing moves between lanes.  Those products read the walked rows transposed: in fp32 a lane takes 4 consecutive channels
// of row 4 g + r (block db of the output is then channels 4 i + db), in bf16 the LDS read itself transposes
// (ds_read_b64_tr_b16: four rows of one channel).  Rows are stored with their 16-byte chunks XOR-ed by the row against bank
// conflicts.  Every (sample, head) keeps to one XCD.
#include "common.h"

namespace vtdge {

constexpr int AB_ROWS = 32;      // walked rows per stage
constexpr int AB_WAVES = 4;      // kept tiles of 16 rows per workgroup

template <typename T> struct BackTile {
    static constexpr int ROWB = 64 * sizeof(T);               // bytes of a row (head dim 64)
    static constexpr int CPR = ROWB / 16;
    static constexpr int HALF = AB_ROWS * ROWB;               // one operand's stage
    static constexpr int NF = sizeof(T) == 4 ? 4 : 2;         // register fragments of a kept row: 16 bytes a lane each
    static __device__ __forceinline__ int slot(int row, int chunk)
    {
        return sizeof(T) == 4 ? chunk ^ (row & 15) : chunk ^ ((row >> 1) & 7);
    }
};

// the four products of a stage, by storage type
template <typename T> struct BackMath;
template <> struct BackMath<float> {
    typedef f32x4 Frag;
    // walked rows 16 blk .. (rows) times the kept rows (columns), over the channels: d = 16 j + 4 g + e in step (j, e)
    static __device__ __forceinline__ f32x4 scores(const unsigned char *S, int blk, const Frag (&x)[4], int l, int g)
    {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const f32x4 a = *reinterpret_cast<const f32x4 *>(S + (16 * blk + l) * 256 + BackTile<float>::slot(l, 4 * j + g) * 16);
#pragma unroll
            for (int e = 0; e < 4; e++) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], x[j][e], acc, 0, 0, 0);
        }
        return acc;
    }
    // of both operands, for a stage's 32 walked rows
    static __device__ __forceinline__ void both_scores(const unsigned char *S0, const unsigned char *S1, const Frag (&x)[4],
                                                       const Frag (&y)[4], f32x4 (&t)[2], f32x4 (&dp)[2], int l, int g)
    {
#pragma unroll
        for (int blk = 0; blk < 2; blk++) {
            t[blk] = scores(S0, blk, x, l, g);
            dp[blk] = scores(S1, blk, y, l, g);
        }
    }
    // out[channel][kept row] += walked rows^T p, p[blk][r] = lane's value of walked row 16 blk + 4 g + r
    static __device__ __forceinline__ void accumulate(const unsigned char *S, const f32x4 (&p)[2], f32x4 (&out)[4], int l, int g)
    {
#pragma unroll
        for (int blk = 0; blk < 2; blk++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const f32x4 a = *reinterpret_cast<const f32x4 *>(S + (16 * blk + 4 * g + r) * 256 +
                                                                 BackTile<float>::slot(4 * g + r, l) * 16);
#pragma unroll
                for (int db = 0; db < 4; db++)
                    out[db] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[db], p[blk][r], out[db], 0, 0, 0);
            }
    }
    // out[db][r] is channel 16 g + 4 r + db of kept row l
    static __device__ __forceinline__ void store(float *row, const f32x4 (&o)[4], int g)
    {
#pragma unroll
        for (int r = 0; r < 4; r++)
            *reinterpret_cast<f32x4 *>(row + 16 * g + 4 * r) = f32x4{o[0][r], o[1][r], o[2][r], o[3][r]};
    }
    static __device__ __forceinline__ void add(const float *row, f32x4 (&o)[4], int g)
    {
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const f32x4 v = *reinterpret_cast<const f32x4 *>(row + 16 * g + 4 * r);
#pragma unroll
            for (int db = 0; db < 4; db++) o[db][r] += v[db];
        }
    }
};
template <> struct BackMath<bf16_t> {
    typedef u32x4 Frag;
    static __device__ __forceinline__ f32x4 mma(const u32x4 &a, const u32x4 &b, const f32x4 &c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0,
                                                       0);
    }
    static __device__ __forceinline__ f32x4 scores(const unsigned char *S, int blk, const Frag (&x)[2], int l, int g)
    {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 2; j++)
            acc = mma(*reinterpret_cast<const u32x4 *>(S + (16 * blk + l) * 128 + BackTile<bf16_t>::slot(l, 4 * j + g) * 16),
                      x[j], acc);
        return acc;
    }
    // All of the stage's fragments are asked for before the first product: left to itself the compiler keeps registers for two
    // and waits for LDS in every step.  Us, with the masks of keys past the last in the last stage alone, before / now, dQ and dK with
    // dV (samples, heads, keys): 128, 6, 257: 48.5 / 44.5 and 45.2 / 43.6; 64, 3, 257: 18.2 / 16.2 and 15.6 / 14.8; 30, 5, 401: 27.2 / 23.5 and
    // 20.4 / 19.3; 16, 3, 1025: 46.4 / 38.7 and 35.5 / 34.0.
    static __device__ __forceinline__ void both_scores(const unsigned char *S0, const unsigned char *S1, const Frag (&x)[2],
                                                       const Frag (&y)[2], f32x4 (&t)[2], f32x4 (&dp)[2], int l, int g)
    {
        u32x4 f[2][2][2];
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int blk = 0; blk < 2; blk++) {
                const int at = (16 * blk + l) * 128 + BackTile<bf16_t>::slot(l, 4 * j + g) * 16;
                f[0][blk][j] = *reinterpret_cast<const u32x4 *>(S0 + at);
                f[1][blk][j] = *reinterpret_cast<const u32x4 *>(S1 + at);
            }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int blk = 0; blk < 2; blk++) t[blk] = dp[blk] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int blk = 0; blk < 2; blk++) {
                t[blk] = mma(f[0][blk][j], x[j], t[blk]);
                dp[blk] = mma(f[1][blk][j], y[j], dp[blk]);
            }
    }
    static __device__ __forceinline__ u32x4 pack(const f32x4 (&p)[2])
    {
        return u32x4{pack_bf16x2(p[0][0], p[0][1]), pack_bf16x2(p[0][2], p[0][3]), pack_bf16x2(p[1][0], p[1][1]),
                     pack_bf16x2(p[1][2], p[1][3])};
    }
    static __device__ __forceinline__ void accumulate(const unsigned char *S, const f32x4 (&p)[2], f32x4 (&out)[4], int l, int g)
    {
        accumulate(S, pack(p), out, l, g);
    }
    // contraction over the stage's 32 rows in the order (4 g .. 4 g + 3, 16 + 4 g .. 16 + 4 g + 3) of lane group g
    static __device__ __forceinline__ void accumulate(const unsigned char *S, const u32x4 &b, f32x4 (&out)[4], int l, int g)
    {
        // this lane as a source of the transposing reads: row 4 g + l / 4, channels 16 db + 4 (l % 4) .. + 3
        const int row = 4 * g + (l >> 2);
        const unsigned char *src = S + row * 128 + 8 * (l & 1);
        u32x2 lo[4], hi[4];
#pragma unroll
        for (int db = 0; db < 4; db++) {
            const unsigned char *at = src + BackTile<bf16_t>::slot(row, 2 * db + ((l & 3) >> 1)) * 16;
            lo[db] = lds_read_tr16(at);
            hi[db] = lds_read_tr16(at + 16 * 128);
        }
#pragma unroll
        for (int db = 0; db < 4; db++) out[db] = mma(u32x4{lo[db].x, lo[db].y, hi[db].x, hi[db].y}, b, out[db]);
    }
    // out[db][r] is channel 16 db + 4 g + r of kept row l
    static __device__ __forceinline__ void store(bf16_t *row, const f32x4 (&o)[4], int g)
    {
#pragma unroll
        for (int db = 0; db < 4; db++) {
            u32x2 w;
            w.x = pack_bf16x2(o[db][0], o[db][1]);
            w.y = pack_bf16x2(o[db][2], o[db][3]);
            *reinterpret_cast<u32x2 *>(row + 16 * db + 4 * g) = w;
        }
    }
};

// the forward pass
struct AttnTrain {
    const bf16_t *q, *k, *v;
    bf16_t *out;
    const int64_t *offsets;
    int64_t q_rs, q_hs, kv_bs, kv_ts, kv_hs, o_rs, o_hs;
    int pairs, h, n;
    float scale_log2;
};

struct AttnBack {
    const void *q, *k, *v, *dout;
    void *dq, *dk, *dv;
    float *m, *inv, *delta;                               // [h, L] each; bf16, or inv NULL: m + log2(s) in m's place; inv < 0: see BackSplit
    const int64_t *offsets;
    int64_t q_rs, q_hs, kv_bs, kv_ts, kv_hs, o_rs, o_hs, dq_rs, dq_hs, dkv_bs, dkv_ts, dkv_hs, L;
    int pairs, h, n;
    float scale, scale_log2;
    bool search;                                          // see find_chunk
    bool by_chunk;                                        // see dkv_place
};

// the stages of two operands' rows in LDS: `rows` of them from base0 / base1 with the given row pitches in bytes
template <typename T> struct Stager {
    using B = BackTile<T>;
    static constexpr int NL = 2 * B::HALF / 1024 / AB_WAVES;  // direct loads a wave and stage
    const unsigned char *base;
    uint32_t pitch, lds0;
    int rows, wid, lane;
    __device__ __forceinline__ void load(int st, int slot) const
    {
        const int r0 = st * AB_ROWS, last = rows - 1 - r0;
        const uint32_t dst = lds0 + (uint32_t)(slot * 2 * B::HALF + wid * NL * 1024);
        const void *src = uniform_ptr(base + (int64_t)r0 * pitch);
#pragma unroll
        for (int i = 0; i < NL; i++) {
            const int row = ((wid & 1) * NL + i) * (64 / B::CPR) + lane / B::CPR;
            dma16(src, (uint32_t)min(row, last) * pitch + (uint32_t)B::slot(row, lane % B::CPR) * 16u, dst + i * 1024);
        }
    }
    // at most `younger` stages of this wave's loads, PER of them each, are outstanding
    template <int PER> static __device__ __forceinline__ void wait(int younger)
    {
        if (younger >= 2) wait_vmcnt<2 * PER>();
        else if (younger == 1) wait_vmcnt<PER>();
        else wait_vmcnt<0>();
    }
};

template <typename T>
__device__ __forceinline__ void load_kept(typename BackMath<T>::Frag (&f)[BackTile<T>::NF], const T *row, bool live, int g)
{
    using Frag = typename BackMath<T>::Frag;
    const unsigned char *p = reinterpret_cast<const unsigned char *>(row) + 16 * g;
#pragma unroll
    for (int j = 0; j < BackTile<T>::NF; j++) {
        u32x4 z = {0u, 0u, 0u, 0u};
        if (live) z = *reinterpret_cast<const u32x4 *>(p + 64 * j);
        f[j] = __builtin_bit_cast(Frag, z);
    }
}

// The (sample, head) pair and the chunk of 64 of its queries that this workgroup takes: from a grid with room for the longest
// sample's chunks in every pair, as it stands, or searched for: the pairs of an XCD (8 i + xcd) lie one behind the other then with as
// many workgroups each as they have chunks, found from the samples' offsets.  The holes of the grid as it stands are dealt out by
// the dispatcher like work, and the last live workgroups start when the first have ended; the search costs a workgroup 1 to 1.5
// us, and that again for every 256 pairs of the XCD.  So it pays for the queries' gradients where there are holes, more
// workgroups than compute units and enough keys (us inside a training pass, grid as it stands / searched; samples, heads, keys): fp32 64,
// 3, 257: 63.4 / 46.3; 16, 6, 257: 42.4 / 31.0; 30, 5, 144: 25.9 / 20.5; 30, 3, 256: 73.6 / 63.7; bf16 128, 6, 257: 45.8 / 43.4; 60, 5,
// 401: 43.6 / 39.5; 30, 3, 256: 26.5 / 22.9; and costs where there are not (launches one behind the other, both kernels): bf16 1024, 8, 20: 46.9 /
// 67.0; 600, 12, 65: 134 / 162; 100, 8, 65 (inside a pass): 12.0 / 13.0; 128, 3, 257, no holes: 68.1 / 73.1; 4, 3, 257: 19.7 /
// 21.1.  For the forward pass from 4096 workgroups on: 256, 6, 257: 46.6 / 39.8; with fewer 64, 6, 257: 16.0 / 17.2; 16, 6, 257: 10.4 /
// 11.0; 64, 3, 257, no holes: 13.8 / 16.0; 2000, 4, 17: 12.7 / 35.1.
constexpr int AB_SEARCH = 1024;                           // pairs of an XCD that are looked through
// about as many chunks of 64 queries as L queries in all make: half a chunk of every pair is lost
__host__ __device__ __forceinline__ int64_t live_chunks(int64_t L, int64_t pairs, int h) { return L * h / (16 * AB_WAVES) + pairs / 2; }
// whether a grid of `chunks` for each pair has holes worth a search
__host__ __device__ __forceinline__ bool has_holes(int64_t L, int64_t pairs, int h, int64_t chunks)
{
    return live_chunks(L, pairs, h) * 100 < pairs * chunks * 88;
}
__device__ __forceinline__ bool find_chunk(bool search, const int64_t *offsets, int pairs, int h, int &pair, int &chunk, int64_t &row0,
                                           int &Lb)
{
    const int rest = blockIdx.x >> 3, xcd = blockIdx.x & 7, pairs_x = (pairs + 7) / 8;
    if (!search) {
        pair = (rest % pairs_x) * 8 + xcd;
        chunk = rest / pairs_x;
        if (pair >= pairs) return false;
        row0 = offsets[pair / h];
        Lb = (int)(offsets[pair / h + 1] - row0);
        return chunk * 16 * AB_WAVES < Lb;
    }
    __shared__ int totals[AB_SEARCH / 256][4], found[2];
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    int mine[AB_SEARCH / 256], upto[AB_SEARCH / 256];
    if (tid == 0) found[0] = -1;
#pragma unroll
    for (int k = 0; k < AB_SEARCH / 256; k++) {
        const int p = (k * 256 + tid) * 8 + xcd;
        mine[k] = 0;
        if (k * 256 < pairs_x && p < pairs) {
            const int b = p / h;
            mine[k] = (int)((offsets[b + 1] - offsets[b] + 16 * AB_WAVES - 1) / (16 * AB_WAVES));
        }
    }
#pragma unroll
    for (int k = 0; k < AB_SEARCH / 256; k++) {
        int v = mine[k];
        if (k * 256 < pairs_x) {
#pragma unroll
            for (int o = 1; o < WAVE; o <<= 1) {
                const int up = __shfl_up(v, o, WAVE);
                if (lane >= o) v += up;
            }
        }
        upto[k] = v;
        if (lane == 63) totals[k][wid] = v;
    }
    __syncthreads();
    int before = 0;
#pragma unroll
    for (int k = 0; k < AB_SEARCH / 256; k++)
#pragma unroll
        for (int w = 0; w < 4; w++) {
            if (w == wid) {
                const int first = before + upto[k] - mine[k];
                if (rest >= first && rest < first + mine[k]) {
                    found[0] = (k * 256 + tid) * 8 + xcd;
                    found[1] = rest - first;
                }
            }
            before += totals[k][w];
        }
    __syncthreads();
    pair = __builtin_amdgcn_readfirstlane(found[0]);
    chunk = __builtin_amdgcn_readfirstlane(found[1]);
    if (pair < 0) return false;
    row0 = offsets[pair / h];
    Lb = (int)(offsets[pair / h + 1] - row0);
    return true;
}

// The forward pass in bf16, from the same scores as the gradients: the inference kernels round the queries once more, times
// the scale, and take their reference score from the first 32 keys, so that a row whose first scores are all -infinity comes
// out as NaN.  Here a query's reference is its running maximum; until a finite score comes there is none and nothing is
// added.  The row sum is taken of the probabilities as rounded for the product with the values.
template <bool SEARCH> __global__ __launch_bounds__(256, 4) void attention_train_kernel(AttnTrain a)
{
    using B = BackTile<bf16_t>;
    using M = BackMath<bf16_t>;
    constexpr int DEPTH = 2;                              // stages in LDS
    __shared__ __attribute__((aligned(1024))) unsigned char smem[DEPTH * 2 * B::HALF];
    int pair, chunk, Lb;
    int64_t row0;
    const bool search = SEARCH && has_holes(a.offsets[a.pairs / a.h], a.pairs, a.h, (int)(gridDim.x >> 3) / ((a.pairs + 7) / 8));
    if (!find_chunk(search, a.offsets, a.pairs, a.h, pair, chunk, row0, Lb)) return;
    const int b = pair / a.h, head = pair - b * a.h;
    const int lane = threadIdx.x & 63, l = lane & 15, g = lane >> 4;
    const int wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int row = (chunk * AB_WAVES + wid) * 16 + l;
    const bool live = row < Lb, wave_live = (chunk * AB_WAVES + wid) * 16 < Lb;

    const int64_t kv_at = (int64_t)b * a.kv_bs + (int64_t)head * a.kv_hs;
    const Stager<bf16_t> kv{reinterpret_cast<const unsigned char *>((wid < 2 ? a.k : a.v) + kv_at), (uint32_t)(a.kv_ts * 2),
                            (uint32_t)(uintptr_t)smem, a.n, wid, lane};
    const int stages = (a.n + AB_ROWS - 1) / AB_ROWS;
    for (int st = 0; st < DEPTH - 1 && st < stages; st++) kv.load(st, st);
    typename M::Frag qf[B::NF];
    load_kept<bf16_t>(qf, a.q + (row0 + row) * a.q_rs + (int64_t)head * a.q_hs, live, g);
    f32x4 o[4];
#pragma unroll
    for (int i = 0; i < 4; i++) o[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, s = 0.f;                         // of this lane's query; s of this lane's keys
    for (int st = 0; st < stages; st++) {
        Stager<bf16_t>::wait<Stager<bf16_t>::NL>(min(stages - 1 - st, DEPTH - 2));
        block_barrier();
        if (st + DEPTH - 1 < stages) kv.load(st + DEPTH - 1, (st + DEPTH - 1) % DEPTH);
        unsigned char *Ks = smem + st % DEPTH * 2 * B::HALF, *Vs = Ks + B::HALF;
        const int left = a.n - st * AB_ROWS;
        if (left < AB_ROWS) {                             // values past the last key: nothing of them, not even 0 * infinity
            for (int i = left * B::CPR + threadIdx.x; i < AB_ROWS * B::CPR; i += 64 * AB_WAVES)
                *reinterpret_cast<u32x4 *>(Vs + i * 16) = u32x4{0u, 0u, 0u, 0u};
            lds_barrier();
        }
        if (!wave_live) continue;
        f32x4 p[2];
        float mx = m;
#pragma unroll
        for (int blk = 0; blk < 2; blk++) {
            p[blk] = M::scores(Ks, blk, qf, l, g);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                p[blk][r] = 16 * blk + 4 * g + r < left ? p[blk][r] * a.scale_log2 : -INFINITY;
                mx = fmaxf(mx, p[blk][r]);
            }
        }
        mx = fmaxf(mx, __shfl_xor(mx, 16, WAVE));
        mx = fmaxf(mx, __shfl_xor(mx, 32, WAVE));
        const float ref = mx == -INFINITY ? 0.f : mx, down = __builtin_amdgcn_exp2f(m - ref);
        m = mx;
#pragma unroll
        for (int blk = 0; blk < 2; blk++)
#pragma unroll
            for (int r = 0; r < 4; r++) p[blk][r] = __builtin_amdgcn_exp2f(p[blk][r] - ref);
        const u32x4 pb = M::pack(p);
        s = bf16_pair_sum(pb.w, bf16_pair_sum(pb.z, bf16_pair_sum(pb.y, bf16_pair_sum(pb.x, s * down))));
#pragma unroll
        for (int i = 0; i < 4; i++) o[i] *= down;
        M::accumulate(Vs, pb, o, l, g);
    }
    s += __shfl_xor(s, 16, WAVE);
    s += __shfl_xor(s, 32, WAVE);
    const float inv = 1.0f / s;
#pragma unroll
    for (int i = 0; i < 4; i++) o[i] *= inv;
    if (live) M::store(a.out + (row0 + row) * a.o_rs + (int64_t)head * a.o_hs, o, g);
}

// dQ of 64 query rows of one (sample, head), with their m, 1 / s and delta.
// HELD: stages of keys whose scores and dP stay in registers between the two walks (0: they are worked out again)
// MARKED: 1 / s is left with its sign set (see attention_dkv_split_rows)
template <typename T, int HELD, bool MARKED = false>
__device__ __forceinline__ void attention_dq_rows(const AttnBack &a, unsigned char *smem, int pair, int chunk, int64_t row0, int Lb)
{
    using B = BackTile<T>;
    using M = BackMath<T>;
    constexpr int DEPTH = 2;                              // stages in LDS
    const int b = pair / a.h, head = pair - b * a.h;
    const int lane = threadIdx.x & 63, l = lane & 15, g = lane >> 4;
    const int wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int row = (chunk * AB_WAVES + wid) * 16 + l;
    const bool live = row < Lb, wave_live = (chunk * AB_WAVES + wid) * 16 < Lb;

    const int64_t kv_at = (int64_t)b * a.kv_bs + (int64_t)head * a.kv_hs;
    const Stager<T> kv{reinterpret_cast<const unsigned char *>((const T *)(wid < 2 ? a.k : a.v) + kv_at),
                       (uint32_t)(a.kv_ts * sizeof(T)), (uint32_t)(uintptr_t)smem, a.n, wid, lane};
    // the keys are walked twice, as one sequence of stages: the second walk's first ones are on their way when the first
    // ends (of scores held it takes keys only)
    const int stages = (a.n + AB_ROWS - 1) / AB_ROWS;
    const bool twice = HELD == 0 || wid < 2;
    const int total = twice ? 2 * stages : stages;        // stages that this wave loads
    auto load = [&](int u) {
        if (u < total) kv.load(u < stages ? u : u - stages, u % DEPTH);
    };
    auto stage_at = [&](int u) { return smem + u % DEPTH * 2 * B::HALF; };
    for (int u = 0; u < DEPTH - 1; u++) load(u);

    typename M::Frag qf[B::NF], df[B::NF];
    load_kept<T>(qf, (const T *)a.q + (row0 + row) * a.q_rs + (int64_t)head * a.q_hs, live, g);
    load_kept<T>(df, (const T *)a.dout + (row0 + row) * a.o_rs + (int64_t)head * a.o_hs, live, g);
    // ---- m, s and delta of this lane's query: maximum, sum of e and sum of e dP over the lane's keys, then over the four
    // lanes that share the query
    float m = -INFINITY, s = 0.f, sd = 0.f;
    f32x4 held_t[HELD > 0 ? HELD : 1][2], held_dp[HELD > 0 ? HELD : 1][2];
    auto sums = [&](int st, f32x4 (&t)[2], f32x4 (&dp)[2]) {
        M::both_scores(stage_at(st), stage_at(st) + B::HALF, qf, df, t, dp, l, g);
        // keys past the last are left out by a mask: of the last stage alone where the code of a stage is there once
        auto add_up = [&](auto partial) {
            constexpr bool PARTIAL = decltype(partial)::value;
            float hi = -INFINITY, lo = INFINITY;          // (one of them times the scale is the largest)
#pragma unroll
            for (int blk = 0; blk < 2; blk++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const bool in = !PARTIAL || st * AB_ROWS + 16 * blk + 4 * g + r < a.n;
                    dp[blk][r] = in ? dp[blk][r] : 0.f;
                    hi = fmaxf(hi, in ? t[blk][r] : -INFINITY);
                    lo = fminf(lo, in ? t[blk][r] : INFINITY);
                }
            const float mx = fmaxf(m, a.scale_log2 < 0.f ? lo * a.scale_log2 : hi * a.scale_log2);
            // (a maximum leaves NaN out, and a lane's keys may be one that is NaN and keys past the last: those are summed too)
            const float ref = mx == -INFINITY ? 0.f : mx, down = __builtin_amdgcn_exp2f(m - ref);
            // a stage's eight keys in pairs first: fewer roundings in a row than key by key
            f32x4 e[2], ed[2];
#pragma unroll
            for (int blk = 0; blk < 2; blk++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const bool in = !PARTIAL || st * AB_ROWS + 16 * blk + 4 * g + r < a.n;
                    e[blk][r] = in ? __builtin_amdgcn_exp2f(__builtin_fmaf(t[blk][r], a.scale_log2, -ref)) : 0.f;
                    ed[blk][r] = e[blk][r] * dp[blk][r];
                }
            s = s * down + (((e[0][0] + e[0][1]) + (e[0][2] + e[0][3])) + ((e[1][0] + e[1][1]) + (e[1][2] + e[1][3])));
            sd = sd * down + (((ed[0][0] + ed[0][1]) + (ed[0][2] + ed[0][3])) + ((ed[1][0] + ed[1][1]) + (ed[1][2] + ed[1][3])));
            m = mx;
        };
        if (HELD > 0 || a.n - st * AB_ROWS < AB_ROWS) add_up(std::true_type{});
        else add_up(std::false_type{});
    };
    auto next_stage = [&](int u) {
        Stager<T>::template wait<Stager<T>::NL>(min(total - 1 - u, DEPTH - 2));
        block_barrier();
        load(u + DEPTH - 1);
    };
    if constexpr (HELD > 0) {
        static_for<HELD>([&](auto st_c) {
            constexpr int st = decltype(st_c)::value;
            if (st < stages) {
                next_stage(st);
                if (wave_live) sums(st, held_t[st], held_dp[st]);
            }
        });
    } else {
        for (int st = 0; st < stages; st++) {
            next_stage(st);
            if (wave_live) sums(st, held_t[0], held_dp[0]);
        }
    }
    float all = fmaxf(m, __shfl_xor(m, 16, WAVE));
    all = fmaxf(all, __shfl_xor(all, 32, WAVE));
    const float down = __builtin_amdgcn_exp2f(m - all);   // a lane without keys: exp2(-inf) = 0 times 0
    s *= down;
    sd *= down;
    s += __shfl_xor(s, 16, WAVE);
    sd += __shfl_xor(sd, 16, WAVE);
    s += __shfl_xor(s, 32, WAVE);
    sd += __shfl_xor(sd, 32, WAVE);
    const float inv = 1.0f / s, delta = sd / s, scale_s = a.scale * inv;
    if (live && g == 0) {
        const int64_t at = (int64_t)head * a.L + row0 + row;
        const bool apart = sizeof(T) == 4 && a.inv != nullptr;
        a.m[at] = apart ? all : all + __builtin_amdgcn_logf(s);                 // v_log_f32: base 2
        if (apart) a.inv[at] = MARKED ? __uint_as_float(__float_as_uint(inv) | 0x80000000u) : inv;
        a.delta[at] = delta;
    }

    // ---- dQ^T += K^T dS^T, dS whole before it is rounded and added up: behind the sums, scale / s would come too late for those
    // that pass the largest number without it
    f32x4 dq[4];
#pragma unroll
    for (int i = 0; i < 4; i++) dq[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto add = [&](int st, const f32x4 (&t)[2], const f32x4 (&dp)[2]) {
        f32x4 ds[2];
#pragma unroll
        for (int blk = 0; blk < 2; blk++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                ds[blk][r] = __builtin_amdgcn_exp2f(__builtin_fmaf(t[blk][r], a.scale_log2, -all)) * (dp[blk][r] - delta) * scale_s;
        if (HELD > 0 || a.n - st * AB_ROWS < AB_ROWS)
#pragma unroll
            for (int e = 0; e < 8; e++)
                if (st * AB_ROWS + 16 * (e / 4) + 4 * g + e % 4 >= a.n) ds[e / 4][e % 4] = 0.f;
        M::accumulate(stage_at(stages + st), ds, dq, l, g);
    };
    if constexpr (HELD > 0) {
        static_for<HELD>([&](auto st_c) {
            constexpr int st = decltype(st_c)::value;
            if (st < stages) {
                next_stage(stages + st);
                if (wave_live) add(st, held_t[st], held_dp[st]);
            }
        });
    } else {
        for (int st = 0; st < stages; st++) {
            next_stage(stages + st);
            if (!wave_live) continue;
            f32x4 t[2], dp[2];
            M::both_scores(stage_at(stages + st), stage_at(stages + st) + B::HALF, qf, df, t, dp, l, g);
            add(st, t, dp);
        }
    }
    if (live) M::store((T *)a.dq + (row0 + row) * a.dq_rs + (int64_t)head * a.dq_hs, dq, g);
}

template <typename T, int HELD> __global__ __launch_bounds__(256, HELD == 0 ? 4 : HELD <= 5 ? 3 : 2) void attention_dq_kernel(AttnBack a)
{
    __shared__ __attribute__((aligned(1024))) unsigned char smem[4 * BackTile<T>::HALF];
    int pair, chunk, Lb;
    int64_t row0;
    if (!find_chunk(a.search, a.offsets, a.pairs, a.h, pair, chunk, row0, Lb)) return;
    attention_dq_rows<T, HELD>(a, smem, pair, chunk, row0, Lb);
}

// The (sample, head), counted over the launch, and the 64 keys of it that a workgroup of the dK and dV kernels takes.
// bf16: the chunks of a pair one behind the other (39.1 us at 128 samples of 6 heads and 257 keys, 40.9 chunk by chunk), unless
// a small last chunk would then always fall to the same of an XCD's 32 compute units (both kernels, 600 samples of 6 heads, 65
// keys: 73.6 us, chunk by chunk 66.0; of 5 queries each 64.1 and 55.6); fp32 chunk by chunk (60.7 us at 64 of 3 on the fp32
// instructions; 63.1), on the bf16 instructions, with the longest samples first, behind one another (both kernels, 64, 3, 257: 77.5
// us, chunk by chunk 80.5; 16, 3, 1025: 235 and 257; with a small last chunk, 64, 6, 200: 102.5 and 107).
__device__ __forceinline__ void dkv_place(const AttnBack &a, int &pair, int &chunk)
{
    const int rest = blockIdx.x >> 3, pairs_x = (a.pairs + 7) / 8, chunks = (a.n + 16 * AB_WAVES - 1) / (16 * AB_WAVES);
    chunk = a.by_chunk ? rest / pairs_x : rest % chunks;
    pair = (a.by_chunk ? rest % pairs_x : rest / chunks) * 8 + (blockIdx.x & 7);
}

// dK and dV of 64 keys of one (sample, head), from DEPTH stages of queries in LDS and their m, 1 / s and delta (of 32 rows, twice)
// MARKED: of the stages alone whose 1 / s has its sign set, and added to what this wave has stored before
template <typename T, int DEPTH, bool MARKED = false>
__device__ __forceinline__ void attention_dkv_rows(const AttnBack &a, unsigned char *smem, float (*stats)[3][64], int pair, int chunk)
{
    using B = BackTile<T>;
    using M = BackMath<T>;
    const int b = pair / a.h, head = pair - b * a.h;
    const int64_t row0 = a.offsets[b];
    const int Lb = (int)(a.offsets[b + 1] - row0);
    const int lane = threadIdx.x & 63, l = lane & 15, g = lane >> 4;
    const int wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int key = (chunk * AB_WAVES + wid) * 16 + l;
    const bool live = key < a.n, wave_live = (chunk * AB_WAVES + wid) * 16 < a.n;

    const int stages = (Lb + AB_ROWS - 1) / AB_ROWS;      // none for a sample without queries: its gradients are zero
    const Stager<T> qd{wid < 2 ? reinterpret_cast<const unsigned char *>((const T *)a.q + row0 * a.q_rs + (int64_t)head * a.q_hs)
                               : reinterpret_cast<const unsigned char *>((const T *)a.dout + row0 * a.o_rs + (int64_t)head * a.o_hs),
                       (uint32_t)((wid < 2 ? a.q_rs : a.o_rs) * sizeof(T)), (uint32_t)(uintptr_t)smem, Lb, wid, lane};
    const int64_t stat = (int64_t)head * a.L + row0;
    const bool apart = sizeof(T) == 4 && a.inv != nullptr;
    const float *rm = a.m + stat, *rinv = apart ? a.inv + stat : nullptr, *delta = a.delta + stat;
    // waves 1 to 3 bring one of them each, behind their share of the rows
    const float *mine = wid == 1 ? rm : wid == 2 ? rinv : delta;
    const bool brings = wid == 1 || wid == 3 || (wid == 2 && apart);
    auto load = [&](int st) {
        const int slot = st % DEPTH;
        qd.load(st, slot);
        if (brings)
            dma4(uniform_ptr(mine + st * AB_ROWS), (uint32_t)min(lane & 31, Lb - 1 - st * AB_ROWS) * 4u,
                 (uint32_t)(uintptr_t)&stats[slot][wid - 1][0]);
    };
    for (int st = 0; st < DEPTH - 1 && st < stages; st++) load(st);
    typename M::Frag kf[B::NF], vf[B::NF];
    const int64_t kv_at = (int64_t)b * a.kv_bs + (int64_t)key * a.kv_ts + (int64_t)head * a.kv_hs;
    load_kept<T>(kf, (const T *)a.k + kv_at, live, g);
    load_kept<T>(vf, (const T *)a.v + kv_at, live, g);
    f32x4 dk[4], dv[4];
#pragma unroll
    for (int i = 0; i < 4; i++) dk[i] = dv[i] = f32x4{0.f, 0.f, 0.f, 0.f};

    for (int st = 0; st < stages; st++) {
        const int younger = min(stages - 1 - st, DEPTH - 2);
        if (brings) Stager<T>::template wait<Stager<T>::NL + 1>(younger);
        else Stager<T>::template wait<Stager<T>::NL>(younger);
        block_barrier();
        if (st + DEPTH - 1 < stages) load(st + DEPTH - 1);
        unsigned char *Qs = smem + st % DEPTH * 2 * B::HALF, *Ds = Qs + B::HALF;
        const int left = Lb - st * AB_ROWS;
        if (left < AB_ROWS) {                             // dO past the last query: nothing of it, not even 0 * infinity
            for (int i = left * B::CPR + threadIdx.x; i < AB_ROWS * B::CPR; i += 64 * AB_WAVES)
                *reinterpret_cast<u32x4 *>(Ds + i * 16) = u32x4{0u, 0u, 0u, 0u};
            lds_barrier();
        }
        if (!wave_live) continue;
        if (MARKED && __builtin_amdgcn_readfirstlane(__float_as_int(stats[st % DEPTH][1][0])) >= 0) continue;
        f32x4 ms[2], iv[2], dl[2];                        // rows past the sample's last query: probability zero
#pragma unroll
        for (int blk = 0; blk < 2; blk++) {
            const float (&of)[3][64] = stats[st % DEPTH];
            const int i = 16 * blk + 4 * g;
            ms[blk] = *reinterpret_cast<const f32x4 *>(&of[0][i]);
            iv[blk] = f32x4{1.f, 1.f, 1.f, 1.f};
            if (apart) iv[blk] = *reinterpret_cast<const f32x4 *>(&of[1][i]);
            dl[blk] = *reinterpret_cast<const f32x4 *>(&of[2][i]);
            if (left < AB_ROWS)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const bool in = i + r < left;
                    ms[blk][r] = in ? ms[blk][r] : INFINITY;
                    iv[blk][r] = in ? iv[blk][r] : 1.f;
                    dl[blk][r] = in ? dl[blk][r] : 0.f;
                }
        }
        f32x4 p[2], ds[2];
        M::both_scores(Qs, Ds, kf, vf, p, ds, l, g);
#pragma unroll
        for (int blk = 0; blk < 2; blk++) {
#pragma unroll
            for (int r = 0; r < 4; r++) {
                p[blk][r] = __builtin_amdgcn_exp2f(__builtin_fmaf(p[blk][r], a.scale_log2, -ms[blk][r])) *
                            (MARKED ? fabsf(iv[blk][r]) : iv[blk][r]);
                ds[blk][r] = p[blk][r] * (ds[blk][r] - dl[blk][r]) * a.scale;
            }
        }
        M::accumulate(Ds, p, dv, l, g);
        M::accumulate(Qs, ds, dk, l, g);
    }
    if (!live) return;
    const int64_t at = (int64_t)b * a.dkv_bs + (int64_t)key * a.dkv_ts + (int64_t)head * a.dkv_hs;
    if constexpr (MARKED) {
        M::add((const T *)a.dk + at, dk, g);
        M::add((const T *)a.dv + at, dv, g);
    }
    M::store((T *)a.dk + at, dk, g);
    M::store((T *)a.dv + at, dv, g);
}

template <typename T> __global__ __launch_bounds__(256, sizeof(T) == 4 ? 3 : 4) void attention_dkv_kernel(AttnBack a)
{
    constexpr int DEPTH = sizeof(T) == 4 ? 3 : 4;
    __shared__ __attribute__((aligned(1024))) unsigned char smem[DEPTH * 2 * BackTile<T>::HALF];
    __shared__ __attribute__((aligned(256))) float stats[DEPTH][3][64];
    int pair, chunk;                    // samples as they come; handed over with the longest first bf16 would take 36.0 us for 37.2
    dkv_place(a, pair, chunk);
    if (pair < a.pairs) attention_dkv_rows<T, DEPTH>(a, smem, stats, pair, chunk);
}

// ---------------------------------------------------------------------------------------------------------
// fp32 on the bf16 matrix instructions, as exact: every operand of the products is the sum of three bf16 values, of whose nine
// partial products the six large ones are multiplied and added in fp32 (linear_dma_split.hip).  A walked row is split once by
// its workgroup on the way into LDS (planes of bf16 rows), a kept one once in its registers, P and dS where they arise.
//
// What bounds both kernels are the vector instructions (the splits: 44 for a fragment of 8 values a lane; they hide behind the
// products only in part, two of them a matrix instruction) beside 96 (72) matrix instructions of 16 clocks a wave and stage, where the
// fp32 ones were 128 (96) of 32.  Three (two) workgroups a compute unit fill each other's waits: one buffer of parts and two barriers a
// stage (both kernels, 64 samples, 6 heads, 257 keys: two buffers and one barrier an eighth slower, rows by direct loads into a ring of
// three 6 %, two workgroups a compute unit for dK and dV 3 %).  Us, fp32 / bf16 instructions, dQ and dK with dV (samples, heads,
// keys, queries): 64, 3, 257, 7352: 43.3 / 32.5 and 61.8 / 36.3; 64, 6: 82.0 / 61.1 and 95.1 / 56.2; 128, 6, 257, 15262: 157 / 120 and 165 / 107; 16, 3,
// 1025, 7598: 190 / 125 and 186 / 98.  Relative errors against float64 (2-norm): dQ 4.2e-7 / 2.9e-7, dK 3.6e-7 / 2.2e-7, dV 3.4e-7 / 2.1e-7;
// queries 16 times as large: 3.3e-6 / 1.7e-6, 3.4e-6 / 1.7e-6, 1.3e-6 / 6.3e-7; 1000 times: 1.8e-4 / 9.1e-5, 1.8e-4 / 9.4e-5, 9.6e-6 / 4.6e-6; queries
// that point at one key each: 1.0e-2 / 7.9e-3, 8.8e-3 / 6.8e-3, 1.8e-8 / 4.2e-8 (a copy of dO, within a rounding).
//
// The values that this is not exact for take the fp32 instructions: an operand that is not zero and not in [2^-60, 2^20) in size (its
// third part, and products of parts, would reach below the smallest bf16 and fp32 numbers; infinities and NaN are out of that
// range too).  A workgroup of 64 queries that meets one takes them from the start and marks its rows by the sign of 1 / s; the key
// tiles leave the stages of such rows out and add them up by the fp32 instructions behind the others: the scores that P is made of
// are always those, to the last bit, that m and s are of.  With other scores, of another order of sums, P of a row's largest key
// would be exp2 of some last bits of the score (queries that point at one key each: dV 8.6e-6 and dK 0.51 off).  P and dS carry a factor of 2^32 into their parts and out of the results: their smallest values would
// reach below 2^-134 otherwise.  Nothing can overflow: scores and dP stay below 2^46, sums of dS over rows below 2^120.
constexpr float BS_UP = 0x1p32f, BS_DOWN = 0x1p-32f;
constexpr int BS_PLANE = AB_ROWS * 128, BS_BUF = 6 * BS_PLANE;      // bytes of a plane, and of two operands' three

struct BackSplit {
    static constexpr int PA[6] = {2, 0, 1, 1, 0, 0}, PB[6] = {0, 2, 1, 0, 1, 0};      // partial products, the small ones first
    // place of a row's 16-byte chunk: sixteen rows at one chunk (scores) and four rows at the two chunks of a block of channels
    // (the transposing reads) both lie in different banks
    static __device__ __forceinline__ int slot(int row, int chunk)
    {
        const int p = (row >> 1) & 7;
        return chunk ^ (((p << 1) | (p >> 2)) & 7);
    }
    static __device__ __forceinline__ f32x4 mma(const u32x4 &a, const u32x4 &b, const f32x4 &c) { return BackMath<bf16_t>::mma(a, b, c); }
    static __device__ __forceinline__ void split(const float (&x)[8], u32x4 (&p)[3])
    {
        float r[8];
#pragma unroll
        for (int e = 0; e < 8; e++) r[e] = x[e];
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                p[i][e] = pack_bf16x2(r[2 * e], r[2 * e + 1]);
                if (i < 2) {
                    r[2 * e] -= bf16lo(p[i][e]);
                    r[2 * e + 1] -= bf16hi(p[i][e]);
                }
            }
    }
    // whether one of the bf16 values is not zero and not in [2^-60, 2^20)
    typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
    static __device__ __forceinline__ bool outside(const u32x4 &a, const u32x4 &b)
    {
        u16x2 big = {0, 0}, small = {0xffff, 0xffff};
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const u16x2 m = __builtin_bit_cast(u16x2, (e < 4 ? a[e] : b[e - 4]) & 0x7fff7fffu);
            big = __builtin_elementwise_max(big, m);
            small = __builtin_elementwise_min(small, (u16x2)(m - (unsigned short)1));      // zero becomes the largest
        }
        constexpr unsigned short LOW = (127 - 60) << 7, HIGH = (127 + 20) << 7;
        return (big[0] > big[1] ? big[0] : big[1]) >= HIGH || (small[0] < small[1] ? small[0] : small[1]) < LOW - 1;
    }
    // a kept row's 64 channels: step t of a contraction takes d = 32 t + 8 g + (0 .. 7)
    static __device__ __forceinline__ bool load_kept(u32x4 (&f)[2][3], const float *row, bool live, int g)
    {
#pragma unroll
        for (int t = 0; t < 2; t++) {
            float x[8];
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const f32x4 v = live ? *reinterpret_cast<const f32x4 *>(row + 32 * t + 8 * g + 4 * j) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int e = 0; e < 4; e++) x[4 * j + e] = v[e];
            }
            split(x, f[t]);
        }
        return outside(f[0][0], f[1][0]);
    }
    // the three planes of 8 channels (chunk) of a walked row
    static __device__ __forceinline__ void store_row(unsigned char *planes, int row, int chunk, const float (&x)[8], u32x4 (&p)[3])
    {
        split(x, p);
#pragma unroll
        for (int i = 0; i < 3; i++) *reinterpret_cast<u32x4 *>(planes + i * BS_PLANE + row * 128 + slot(row, chunk) * 16) = p[i];
    }
    // Fragments are asked for a batch of products ahead: left to itself the compiler keeps registers for one or two and waits for LDS
    // before nearly every product.
    // scores of a stage's 32 walked rows of two operands with the kept rows.  The walk over the queries adds the same products in
    // the same order as the walk over the keys, so both have the same scores to the last bit.
    template <bool QUERIES_WALKED>
    static __device__ __forceinline__ void both_scores(const unsigned char *S0, const unsigned char *S1, const u32x4 (&x)[2][3],
                                                       const u32x4 (&y)[2][3], f32x4 (&t)[2], f32x4 (&dp)[2], int l, int g)
    {
        u32x4 f[2][3];
        auto read = [&](int k) {                          // batch k: rows 16 (k / 4) .., operand k / 2 % 2, channels 32 (k % 2) ..
            const unsigned char *at = (k & 2 ? S1 : S0) + (16 * (k >> 2) + l) * 128 + slot(l, 4 * (k & 1) + g) * 16;
#pragma unroll
            for (int i = 0; i < 3; i++) f[k & 1][i] = *reinterpret_cast<const u32x4 *>(at + i * BS_PLANE);
        };
        read(0);
        f32x4 acc[2];
        static_for<8>([&](auto k_c) {
            constexpr int k = decltype(k_c)::value;
            if constexpr (k < 7) read(k + 1);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr ((k & 1) == 0) acc[0] = acc[1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < 6; i++) {
                const u32x4 &kept = (k & 2 ? y : x)[k & 1][QUERIES_WALKED ? PA[i] : PB[i]];
                acc[i & 1] = mma(f[k & 1][QUERIES_WALKED ? PB[i] : PA[i]], kept, acc[i & 1]);
            }
            if constexpr ((k & 1) == 1) (k & 2 ? dp : t)[k >> 2] = acc[0] + acc[1];
            __builtin_amdgcn_sched_barrier(0);
        });
    }
    // out[db] += walked rows^T p; the layout of BackMath<bf16_t>::accumulate (a second set of fragments gains nothing here)
    static __device__ __forceinline__ void accumulate(const unsigned char *planes, const f32x4 (&p)[2], f32x4 (&out)[4], int l, int g)
    {
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; e++) x[e] = p[e / 4][e % 4];
        u32x4 b[3];
        split(x, b);
        const int row = 4 * g + (l >> 2);
        const unsigned char *src = planes + row * 128 + 8 * (l & 1);
#pragma unroll
        for (int db = 0; db < 4; db++) {
            u32x4 f[3];
#pragma unroll
            for (int i = 0; i < 3; i++) {
                const unsigned char *at = src + i * BS_PLANE + slot(row, 2 * db + ((l & 3) >> 1)) * 16;
                const u32x2 lo = lds_read_tr16(at), hi = lds_read_tr16(at + 16 * 128);
                f[i] = u32x4{lo.x, lo.y, hi.x, hi.y};
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 6; i++) out[db] = mma(f[PA[i]], b[PB[i]], out[db]);
        }
    }
    // out[db][r] is channel 16 db + 4 g + r of kept row l
    static __device__ __forceinline__ void store(float *row, const f32x4 (&o)[4], int g)
    {
#pragma unroll
        for (int db = 0; db < 4; db++) *reinterpret_cast<f32x4 *>(row + 16 * db + 4 * g) = o[db];
    }
};

// attention_dq_rows on split operands -> whether it could
template <int HELD>
__device__ __forceinline__ bool attention_dq_split_rows(const AttnBack &a, unsigned char *smem, int *odd_seen, int pair, int chunk,
                                                        int64_t row0, int Lb)
{
    using S = BackSplit;
    // keys past the last: a score of -infinity, below; and what is said above of overflow
    if (!(a.scale_log2 >= 0x1p-40f && a.scale_log2 <= 0x1p40f)) return false;
    const int b = pair / a.h, head = pair - b * a.h;
    const int tid = threadIdx.x, lane = tid & 63, l = lane & 15, g = lane >> 4;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int row = (chunk * AB_WAVES + wid) * 16 + l;
    const bool live = row < Lb, wave_live = (chunk * AB_WAVES + wid) * 16 < Lb;
    if (tid == 0) *odd_seen = 0;

    // the keys are walked twice, as one sequence of stages; this thread's part of one: 8 channels of a key and, on the first
    // walk (on both where nothing is held), of a value
    const int srow = tid >> 3, schunk = tid & 7;
    const int64_t kv_at = (int64_t)b * a.kv_bs + (int64_t)head * a.kv_hs + 8 * schunk;
    const int stages = (a.n + AB_ROWS - 1) / AB_ROWS;
    float rk[8], rv[8];
    auto load_stage = [&](int u) {                        // rows past the last key repeat it
        const int64_t at = kv_at + (int64_t)min((u < stages ? u : u - stages) * AB_ROWS + srow, a.n - 1) * a.kv_ts;
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const f32x4 x = *reinterpret_cast<const f32x4 *>((const float *)a.k + at + 4 * i);
#pragma unroll
            for (int e = 0; e < 4; e++) rk[4 * i + e] = x[e];
            if (HELD == 0 || u < stages) {
                const f32x4 y = *reinterpret_cast<const f32x4 *>((const float *)a.v + at + 4 * i);
#pragma unroll
                for (int e = 0; e < 4; e++) rv[4 * i + e] = y[e];
            }
        }
    };
    bool odd = false;
    const unsigned char *Ks = smem, *Vs = smem + 3 * BS_PLANE;
    // -> whether the operands are still such as the split covers
    auto next_stage = [&](int u) {
        lds_barrier();                                    // the stage before has been read (before the first: odd_seen is zero)
        const int st = u < stages ? u : u - stages;
        if (st * AB_ROWS + AB_ROWS > a.n) {               // nothing of a repeated row
            const bool past = st * AB_ROWS + srow >= a.n;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                rk[e] = past ? 0.f : rk[e];
                rv[e] = past ? 0.f : rv[e];
            }
        }
        u32x4 p[2][3];
        S::store_row(smem, srow, schunk, rk, p[0]);
        if (HELD == 0 || u < stages) S::store_row(smem + 3 * BS_PLANE, srow, schunk, rv, p[1]);
        if (u < stages) {                                 // (the second walk meets the same keys)
            odd = odd || S::outside(p[0][0], p[1][0]);
            if (odd) *odd_seen = 1;
        }
        if (u + 1 < 2 * stages) load_stage(u + 1);
        lds_barrier();                                    // stage u is whole
        return u >= stages || __builtin_amdgcn_readfirstlane(*odd_seen) == 0;
    };

    load_stage(0);
    u32x4 qf[2][3], df[2][3];
    odd = S::load_kept(qf, (const float *)a.q + (row0 + row) * a.q_rs + (int64_t)head * a.q_hs, live, g);
    odd = S::load_kept(df, (const float *)a.dout + (row0 + row) * a.o_rs + (int64_t)head * a.o_hs, live, g) || odd;
    // scores and dP of a stage; of a key past the last -infinity and (its value is zero) 0: nothing that is summed below
    auto scores = [&](int st, f32x4 (&t)[2], f32x4 (&dp)[2]) {
        S::both_scores<false>(Ks, Vs, qf, df, t, dp, l, g);
        const int left = a.n - st * AB_ROWS - 4 * g;      // keys from this lane's first one on
        if (a.n - st * AB_ROWS < AB_ROWS)
#pragma unroll
            for (int e = 0; e < 8; e++)
                if (16 * (e / 4) + e % 4 >= left) t[e / 4][e % 4] = -INFINITY;
    };
    // ---- m, s and delta as in attention_dq_rows
    float m = -INFINITY, s = 0.f, sd = 0.f;
    f32x4 held_t[HELD > 0 ? HELD : 1][2], held_dp[HELD > 0 ? HELD : 1][2];
    auto sums = [&](int st, f32x4 (&t)[2], f32x4 (&dp)[2]) {
        scores(st, t, dp);
        float mx = -INFINITY;
#pragma unroll
        for (int e = 0; e < 8; e++) mx = fmaxf(mx, t[e / 4][e % 4]);
        mx = fmaxf(m, mx * a.scale_log2);
        const float ref = mx == -INFINITY ? 0.f : mx, down = __builtin_amdgcn_exp2f(m - ref);
        f32x4 e[2], ed[2];
#pragma unroll
        for (int blk = 0; blk < 2; blk++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                e[blk][r] = __builtin_amdgcn_exp2f(__builtin_fmaf(t[blk][r], a.scale_log2, -ref));
                ed[blk][r] = e[blk][r] * dp[blk][r];
            }
        s = s * down + (((e[0][0] + e[0][1]) + (e[0][2] + e[0][3])) + ((e[1][0] + e[1][1]) + (e[1][2] + e[1][3])));
        sd = sd * down + (((ed[0][0] + ed[0][1]) + (ed[0][2] + ed[0][3])) + ((ed[1][0] + ed[1][1]) + (ed[1][2] + ed[1][3])));
        m = mx;
    };
    if constexpr (HELD > 0) {
        bool good = true;
        static_for<HELD>([&](auto st_c) {
            constexpr int st = decltype(st_c)::value;
            if (good && st < stages) {
                good = next_stage(st);
                if (good && wave_live) sums(st, held_t[st], held_dp[st]);
            }
        });
        if (!good) return false;
    } else {
        for (int st = 0; st < stages; st++) {
            if (!next_stage(st)) return false;
            if (wave_live) sums(st, held_t[0], held_dp[0]);
        }
    }
    float all = fmaxf(m, __shfl_xor(m, 16, WAVE));
    all = fmaxf(all, __shfl_xor(all, 32, WAVE));
    const float down = __builtin_amdgcn_exp2f(m - all);   // a lane without keys: exp2(-inf) = 0 times 0
    s *= down;
    sd *= down;
    s += __shfl_xor(s, 16, WAVE);
    sd += __shfl_xor(sd, 16, WAVE);
    s += __shfl_xor(s, 32, WAVE);
    sd += __shfl_xor(sd, 32, WAVE);
    const float inv = 1.0f / s, delta = sd / s, scale_s = a.scale * inv * BS_DOWN, up_delta = BS_UP * delta;
    if (live && g == 0) {
        const int64_t at = (int64_t)head * a.L + row0 + row;
        a.m[at] = all;
        a.inv[at] = inv;
        a.delta[at] = delta;
    }

    // ---- dQ^T += K^T dS^T
    f32x4 dq[4];
#pragma unroll
    for (int i = 0; i < 4; i++) dq[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto add = [&](const f32x4 (&t)[2], const f32x4 (&dp)[2]) {
        f32x4 ds[2];
#pragma unroll
        for (int blk = 0; blk < 2; blk++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                ds[blk][r] = __builtin_amdgcn_exp2f(__builtin_fmaf(t[blk][r], a.scale_log2, -all)) *
                             __builtin_fmaf(dp[blk][r], BS_UP, -up_delta);      // 2^32 (dP - delta), to the last bit
        S::accumulate(Ks, ds, dq, l, g);
    };
    if constexpr (HELD > 0) {
        static_for<HELD>([&](auto st_c) {
            constexpr int st = decltype(st_c)::value;
            if (st < stages) {
                next_stage(stages + st);
                if (wave_live) add(held_t[st], held_dp[st]);
            }
        });
    } else {
        for (int st = 0; st < stages; st++) {
            next_stage(stages + st);
            if (!wave_live) continue;
            scores(st, held_t[0], held_dp[0]);
            add(held_t[0], held_dp[0]);
        }
    }
#pragma unroll
    for (int i = 0; i < 4; i++) dq[i] *= scale_s;         // this lane's query's
    if (live) S::store((float *)a.dq + (row0 + row) * a.dq_rs + (int64_t)head * a.dq_hs, dq, g);
    return true;
}

template <int HELD> __global__ __launch_bounds__(256, HELD == 0 ? 3 : 2) void attention_dq_split_kernel(AttnBack a)
{
    static_assert(4 * BackTile<float>::HALF >= BS_BUF, "one LDS for either");
    __shared__ __attribute__((aligned(1024))) unsigned char smem[4 * BackTile<float>::HALF];
    __shared__ int odd_seen;
    int pair, chunk, Lb;
    int64_t row0;
    if (!find_chunk(a.search, a.offsets, a.pairs, a.h, pair, chunk, row0, Lb)) return;
    if (attention_dq_split_rows<HELD>(a, smem, &odd_seen, pair, chunk, row0, Lb)) return;
    __syncthreads();
    attention_dq_rows<float, 0, true>(a, smem, pair, chunk, row0, Lb);
}

// The sample in place `place` of the order by length, longest first: a lane a sample, of whose numbers (length, then the first
// of equals) each wave finds the place-th from the top bit by bit.  A workgroup's time is its sample's queries, and those
// that start last should be short (64 samples of 3 heads, 257 keys, both kernels: 85.3 -> 80.5 us).  Of more than 64 samples there
// are workgroups enough to fill the end: as they come.
__device__ __forceinline__ int longest_first(const AttnBack &a, int place)
{
    const int samples = a.pairs / a.h, t = threadIdx.x & 63;
    if (samples > WAVE || a.L >= (1 << 26)) return place;
    const uint32_t mine = t < samples ? ((uint32_t)(a.offsets[t + 1] - a.offsets[t]) << 6) + 63 - t : 0u;
    unsigned long long left = ~0ull >> (WAVE - samples);
    int k = __builtin_amdgcn_readfirstlane(place);
    for (int bit = 31; bit >= 0; bit--) {
        const unsigned long long ones = __builtin_amdgcn_ballot_w64((mine >> bit) & 1) & left;
        const int count = __builtin_popcountll(ones);
        if (k < count) left = ones;
        else {
            k -= count;
            left &= ~ones;
        }
    }
    return __builtin_ctzll(left);
}

// attention_dkv_rows on split operands, of the stages whose rows are not marked -> whether any were.  A stage is of one workgroup's rows
// of the queries' kernel, and one with an operand that the split does not cover is marked: the queries' own, or all for a key's.
__device__ __forceinline__ bool attention_dkv_split_rows(const AttnBack &a, unsigned char *smem, float (*stats)[AB_ROWS], int pair, int chunk)
{
    using S = BackSplit;
    const int b = pair / a.h, head = pair - b * a.h;
    const int64_t row0 = a.offsets[b];
    const int Lb = (int)(a.offsets[b + 1] - row0);
    const int tid = threadIdx.x, lane = tid & 63, l = lane & 15, g = lane >> 4;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int key = (chunk * AB_WAVES + wid) * 16 + l;
    const bool live = key < a.n, wave_live = (chunk * AB_WAVES + wid) * 16 < a.n;

    // this thread's part of a stage: 8 channels of a query and of its dO, and one of the 96 statistics
    const int srow = tid >> 3, schunk = tid & 7;
    const float *qp = (const float *)a.q + row0 * a.q_rs + (int64_t)head * a.q_hs + 8 * schunk;
    const float *dp_ = (const float *)a.dout + row0 * a.o_rs + (int64_t)head * a.o_hs + 8 * schunk;
    const int64_t stat = (int64_t)head * a.L + row0;
    const int which = tid >> 5;                           // 0: m, 1: 1 / s, 2: delta
    const float *mine = which == 0 ? a.m : which == 1 ? a.inv : a.delta;
    float rq[8], rd[8], rs = 0.f;
    auto load_stage = [&](int st) {                       // rows past the last query repeat it
        const int64_t r = min(st * AB_ROWS + srow, Lb - 1);
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const f32x4 x = *reinterpret_cast<const f32x4 *>(qp + r * a.q_rs + 4 * i), y = *reinterpret_cast<const f32x4 *>(dp_ + r * a.o_rs + 4 * i);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                rq[4 * i + e] = x[e];
                rd[4 * i + e] = y[e];
            }
        }
        if (which < 3) rs = mine[stat + min(st * AB_ROWS + (tid & 31), Lb - 1)];
    };
    auto store_stage = [&](int st) {
        if (st * AB_ROWS + AB_ROWS > Lb) {                // nothing of a repeated row: probability zero
            const bool past = st * AB_ROWS + srow >= Lb;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                rq[e] = past ? 0.f : rq[e];
                rd[e] = past ? 0.f : rd[e];
            }
            if (st * AB_ROWS + (tid & 31) >= Lb) rs = which == 0 ? INFINITY : which == 1 ? 1.f : 0.f;
        }
        u32x4 p[2][3];
        S::store_row(smem, srow, schunk, rq, p[0]);
        S::store_row(smem + 3 * BS_PLANE, srow, schunk, rd, p[1]);
        if (which < 3) stats[which][tid & 31] = which == 1 ? rs * BS_UP : rs;
    };

    const int stages = (Lb + AB_ROWS - 1) / AB_ROWS;      // none for a sample without queries: its gradients are zero
    if (stages > 0) load_stage(0);
    u32x4 kf[2][3], vf[2][3];
    const int64_t kv_at = (int64_t)b * a.kv_bs + (int64_t)key * a.kv_ts + (int64_t)head * a.kv_hs;
    S::load_kept(kf, (const float *)a.k + kv_at, live, g);
    S::load_kept(vf, (const float *)a.v + kv_at, live, g);
    f32x4 dk[4], dv[4];
#pragma unroll
    for (int i = 0; i < 4; i++) dk[i] = dv[i] = f32x4{0.f, 0.f, 0.f, 0.f};

    const unsigned char *Qs = smem, *Ds = smem + 3 * BS_PLANE;
    bool marked = false;
    for (int st = 0; st < stages; st++) {
        lds_barrier();                                    // the stage before has been read
        store_stage(st);
        if (st + 1 < stages) load_stage(st + 1);
        lds_barrier();                                    // stage st is whole
        if (__builtin_amdgcn_readfirstlane(__float_as_int(stats[1][0])) < 0) {
            marked = true;
            continue;
        }
        if (!wave_live) continue;
        f32x4 p[2], ds[2];
        S::both_scores<true>(Qs, Ds, kf, vf, p, ds, l, g);
#pragma unroll
        for (int blk = 0; blk < 2; blk++) {
            const int i = 16 * blk + 4 * g;
            const f32x4 ms = *reinterpret_cast<const f32x4 *>(&stats[0][i]), iv = *reinterpret_cast<const f32x4 *>(&stats[1][i]),
                        dl = *reinterpret_cast<const f32x4 *>(&stats[2][i]);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                p[blk][r] = __builtin_amdgcn_exp2f(__builtin_fmaf(p[blk][r], a.scale_log2, -ms[r])) * iv[r];
                ds[blk][r] = p[blk][r] * (ds[blk][r] - dl[r]);
            }
        }
        S::accumulate(Ds, p, dv, l, g);
        S::accumulate(Qs, ds, dk, l, g);
    }
    if (!live) return marked;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        dk[i] *= a.scale * BS_DOWN;
        dv[i] *= BS_DOWN;
    }
    const int64_t at = (int64_t)b * a.dkv_bs + (int64_t)key * a.dkv_ts + (int64_t)head * a.dkv_hs;
    S::store((float *)a.dk + at, dk, g);
    S::store((float *)a.dv + at, dv, g);
    return marked;
}

__global__ __launch_bounds__(256, 3) void attention_dkv_split_kernel(AttnBack a)
{
    constexpr int DEPTH = 2;                              // of the fp32 instructions
    static_assert(DEPTH * 2 * BackTile<float>::HALF >= BS_BUF, "one LDS for either");
    __shared__ __attribute__((aligned(1024))) unsigned char smem[DEPTH * 2 * BackTile<float>::HALF];
    __shared__ __attribute__((aligned(256))) float stats[DEPTH][3][64];
    int place, chunk;
    dkv_place(a, place, chunk);
    if (place >= a.pairs) return;
    const int pair = longest_first(a, place / a.h) * a.h + place % a.h;
    if (!attention_dkv_split_rows(a, smem, reinterpret_cast<float(*)[AB_ROWS]>(&stats[0][0][0]), pair, chunk)) return;
    __syncthreads();                                      // LDS has been read, and what the wave has stored can be
    attention_dkv_rows<float, DEPTH, true>(a, smem, stats, pair, chunk);
}

template <typename T> static int launch_backward(AttnBack a, int max_rows, hipStream_t st)
{
    const int64_t pairs_x = ceil_div(a.pairs, 8);
    const int64_t qc = ceil_div(max_rows, 16 * AB_WAVES), kc = ceil_div(a.n, 16 * AB_WAVES);
    VT_REQUIRE(pairs_x * 8 * (qc > kc ? qc : kc) < (1ll << 31), VTDGE_ERR_UNSUPPORTED,
               "sparse_attention_backward: too many workgroups for one launch");
    a.search = qc >= 2 && a.n >= 128 && pairs_x <= AB_SEARCH && a.pairs * qc > compute_units() && has_holes(a.L, a.pairs, a.h, qc);
    // fp32 on the bf16 instructions: from 161 keys on, where live workgroups are about as many as compute units.  Us, both kernels, fp32 /
    // bf16 instructions (samples, heads, keys): 64, 3, 257: 106.6 / 74.2; 64, 6, 257: 177.7 / 122.1; 128, 6, 257: 321 / 231; 16, 3, 1025: 376 /
    // 224.  With fewer, one wave a SIMD waits for its own vector instructions, of which the split has more, and gains less; out of a replayed
    // graph, by live workgroups: 12: 35.9 / 34.6, 54: 39.4 / 37.0, 109: 40.7 / 38.0, 215: 49.2 / 44.5, 431: 86.8 / 65.3; of 161 keys 70: 30.0 /
    // 29.1, 208: 36.9 / 35.6; of 1025 keys 38: 141 / 121, 89: 177 / 135, 180: 180 / 145, 357: 316 / 204.  The line is not where its
    // lead ends but where it is a fifth and more (322, 257 keys: 72.3 / 55.9); one further down would be sound too.  Both kernels or
    // neither, and with 1 / s to carry the marks: scores of another order of sums than those that m and s are of would be off where
    // they are large.
    const bool split = sizeof(T) == 4 && a.inv != nullptr && a.n > 5 * AB_ROWS && live_chunks(a.L, a.pairs, a.h) >= compute_units();
    a.by_chunk = sizeof(T) == 4 ? !split : 32 % kc == 0 && (a.n - 1) % (16 * AB_WAVES) < 8 * AB_WAVES;
    if (qc > 0) {
        // fp32: up to 288 keys the scores and dP of the first walk are kept for the second, the same bits in three products
        // instead of five.  Us, both kernels on the fp32 instructions, worked out again / kept (samples, heads, keys): 64, 3,
        // 257: 161 / 127; 128, 6, 257: 366 / 322; 64, 6, 145: 104 / 80; 64, 3, 65: 36.5 / 31.3; 8, 3, 257: 58.4 / 51.6.  bf16
        // loses more by the registers than it gains: 128, 6, 257: 86 / 101; 64, 6, 145: 30.0 / 29.4.
        auto kern = attention_dq_kernel<T, 0>;
        if constexpr (sizeof(T) == 4) {
            if (a.n <= 3 * AB_ROWS) kern = attention_dq_kernel<T, 3>;
            else if (a.n <= 5 * AB_ROWS) kern = attention_dq_kernel<T, 5>;
            else if (split) kern = a.n <= 9 * AB_ROWS ? attention_dq_split_kernel<9> : attention_dq_split_kernel<0>;
            else if (a.n <= 9 * AB_ROWS) kern = attention_dq_kernel<T, 9>;
        }
        note_kernel(reinterpret_cast<const void *>(kern));
        kern<<<dim3((unsigned)(pairs_x * 8 * qc)), dim3(64 * AB_WAVES), 0, st>>>(a);
        const int rc = check_launch("sparse_attention_backward");
        if (rc != VTDGE_OK) return rc;
    }
    auto kern = attention_dkv_kernel<T>;
    if constexpr (sizeof(T) == 4)
        if (split) kern = attention_dkv_split_kernel;
    note_kernel(reinterpret_cast<const void *>(kern));
    kern<<<dim3((unsigned)(pairs_x * 8 * kc)), dim3(64 * AB_WAVES), 0, st>>>(a);
    return check_launch("sparse_attention_backward");
}

// offsets[base + 1 ..] of `count` lengths that travel in the kernel's arguments: no copy of host memory
constexpr int OFF_MAX = 448;
struct Lengths {
    int32_t v[OFF_MAX];
};
__global__ __launch_bounds__(512) void lengths_offsets_kernel(Lengths len, int count, int64_t start, int64_t *__restrict__ out)
{
    __shared__ int64_t wave_total[8];
    const int i = threadIdx.x, lane = i & 63;
    int64_t v = i < count ? len.v[i] : 0;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int64_t up = __shfl_up(v, o, WAVE);
        if (lane >= o) v += up;
    }
    if (lane == 63) wave_total[i >> 6] = v;
    __syncthreads();
    int64_t before = start;
    for (int w = 0; w < (i >> 6); w++) before += wave_total[w];
    if (i < count) out[i + 1] = before + v;
    if (i == 0 && start == 0) out[0] = 0;
}

}  // namespace vtdge

using namespace vtdge;

extern "C" int vtdge_lengths_to_offsets(const int64_t *lengths_host, int B, int64_t *offsets, void *stream)
{
    VT_REQUIRE(offsets && (lengths_host || B == 0) && B >= 0, VTDGE_ERR_ARG, "lengths_to_offsets: NULL operand");
    int64_t start = 0;
    for (int at = 0; at == 0 || at < B; at += OFF_MAX) {
        Lengths len;
        const int count = B - at < OFF_MAX ? B - at : OFF_MAX;
        int64_t sum = 0;
        for (int i = 0; i < count; i++) {
            const int64_t v = lengths_host[at + i];
            VT_REQUIRE(v >= 0 && v < (1ll << 31), VTDGE_ERR_ARG, "lengths_to_offsets: length %lld of sample %d", (long long)v,
                       at + i);
            len.v[i] = (int32_t)v;
            sum += v;
        }
        // (`start` is zero for the first launch only, or where everything before it was empty: out[0] of a later slice
        // is then the zero that is there already)
        note_kernel(reinterpret_cast<const void *>(lengths_offsets_kernel));
        lengths_offsets_kernel<<<1, 512, 0, (hipStream_t)stream>>>(len, count, start, offsets + at);
        const int rc = check_launch("lengths_to_offsets");
        if (rc != VTDGE_OK) return rc;
        start += sum;
    }
    return VTDGE_OK;
}

extern "C" int vtdge_sparse_attention_train(const void *q, int64_t q_row_stride, int64_t q_head_stride, const void *k,
                                            const void *v, int64_t kv_batch_stride, int64_t kv_tok_stride,
                                            int64_t kv_head_stride, const int64_t *offsets, void *out, int64_t o_row_stride,
                                            int64_t o_head_stride, int B, int h, int d, int n, int max_rows_per_sample,
                                            float scale, int dtype, void *stream)
{
    VT_REQUIRE(q && k && v && offsets && out, VTDGE_ERR_ARG, "sparse_attention_train: NULL operand");
    VT_REQUIRE(B > 0 && h > 0 && n > 0 && max_rows_per_sample >= 0 && (int64_t)B * h < (1ll << 28), VTDGE_ERR_ARG,
               "sparse_attention_train: bad sizes");
    VT_REQUIRE(d == 64 && dtype == VTDGE_BF16, VTDGE_ERR_UNSUPPORTED,
               "sparse_attention_train: head_dim %d, dtype %d (only 64 and bf16 are built)", d, dtype);
    const int64_t strides[] = {q_row_stride, q_head_stride, kv_batch_stride, kv_tok_stride, kv_head_stride, o_row_stride,
                               o_head_stride};
    for (int64_t s : strides)
        VT_REQUIRE(s >= 0 && s % 8 == 0, VTDGE_ERR_UNSUPPORTED, "sparse_attention_train: strides must keep 16-byte alignment");
    VT_REQUIRE(kv_tok_stride < (1 << 23), VTDGE_ERR_UNSUPPORTED, "sparse_attention_train: row stride too large");
    VT_REQUIRE((((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)out) & 15) == 0, VTDGE_ERR_ARG,
               "sparse_attention_train: operands must be 16-byte aligned");
    const int64_t chunks = ceil_div(max_rows_per_sample, 16 * AB_WAVES), grid = ceil_div((int64_t)B * h, 8) * 8 * chunks;
    VT_REQUIRE(grid < (1ll << 31), VTDGE_ERR_UNSUPPORTED, "sparse_attention_train: too many workgroups for one launch");
    if (grid == 0) return VTDGE_OK;
    const AttnTrain a{(const bf16_t *)q, (const bf16_t *)k, (const bf16_t *)v, (bf16_t *)out, offsets, q_row_stride,
                      q_head_stride, kv_batch_stride, kv_tok_stride, kv_head_stride, o_row_stride, o_head_stride, B * h, h, n,
                      scale * 1.44269504088896340736f};
    const bool search = chunks >= 2 && n >= 128 && B * h <= 8 * AB_SEARCH && B * h * chunks >= 16 * compute_units();
    auto kern = search ? attention_train_kernel<true> : attention_train_kernel<false>;
    note_kernel(reinterpret_cast<const void *>(kern));
    kern<<<dim3((unsigned)grid), dim3(64 * AB_WAVES), 0, (hipStream_t)stream>>>(a);
    return check_launch("sparse_attention_train");
}

static int backward(const void *q, int64_t q_row_stride, int64_t q_head_stride, const void *k, const void *v,
                    int64_t kv_batch_stride, int64_t kv_tok_stride, int64_t kv_head_stride, const void *dout,
                    int64_t o_row_stride, int64_t o_head_stride, const int64_t *offsets, void *dq, int64_t dq_row_stride,
                    int64_t dq_head_stride, void *dk, void *dv, int64_t dkv_batch_stride, int64_t dkv_tok_stride,
                    int64_t dkv_head_stride, float *workspace, bool apart, int64_t L, int B, int h, int d, int n,
                    int max_rows_per_sample, float scale, int dtype, void *stream)
{
    VT_REQUIRE(k && v && offsets && dk && dv && (L == 0 || (q && dout && dq && workspace)), VTDGE_ERR_ARG,
               "sparse_attention_backward: NULL operand");
    VT_REQUIRE(dtype == VTDGE_F32 || dtype == VTDGE_BF16, VTDGE_ERR_ARG, "sparse_attention_backward: unknown dtype %d", dtype);
    VT_REQUIRE(B > 0 && h > 0 && n > 0 && L >= 0 && max_rows_per_sample >= 0 && (int64_t)B * h < (1ll << 28), VTDGE_ERR_ARG,
               "sparse_attention_backward: bad sizes");
    VT_REQUIRE(d == 64, VTDGE_ERR_UNSUPPORTED, "sparse_attention_backward: head_dim %d (only 64 is built)", d);
    const int esz = dtype == VTDGE_F32 ? 4 : 2, vec = 16 / esz;
    const int64_t strides[] = {q_row_stride,  q_head_stride, kv_batch_stride, kv_tok_stride,    kv_head_stride, o_row_stride,
                               o_head_stride, dq_row_stride, dq_head_stride,  dkv_batch_stride, dkv_tok_stride, dkv_head_stride};
    for (int64_t s : strides)
        VT_REQUIRE(s >= 0 && s % vec == 0, VTDGE_ERR_UNSUPPORTED,
                   "sparse_attention_backward: strides must keep 16-byte alignment");
    VT_REQUIRE(q_row_stride < (1 << 23) && kv_tok_stride < (1 << 23) && o_row_stride < (1 << 23), VTDGE_ERR_UNSUPPORTED,
               "sparse_attention_backward: row stride too large");
    VT_REQUIRE((((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)dout | (uintptr_t)dq | (uintptr_t)dk | (uintptr_t)dv) &
                15) == 0,
               VTDGE_ERR_ARG, "sparse_attention_backward: operands must be 16-byte aligned");
    float *last = workspace + (int64_t)h * L;
    AttnBack a{q, k, v, dout, dq, dk, dv, workspace, apart ? last : nullptr, apart ? last + (int64_t)h * L : last, offsets,
               q_row_stride, q_head_stride, kv_batch_stride, kv_tok_stride, kv_head_stride, o_row_stride, o_head_stride, dq_row_stride, dq_head_stride,
               dkv_batch_stride, dkv_tok_stride, dkv_head_stride, L, B * h, h, n, scale,
               scale * 1.44269504088896340736f};
    if (dtype == VTDGE_F32) return launch_backward<float>(a, max_rows_per_sample, (hipStream_t)stream);
    return launch_backward<bf16_t>(a, max_rows_per_sample, (hipStream_t)stream);
}

extern "C" int vtdge_sparse_attention_backward(
    const void *q, int64_t q_row_stride, int64_t q_head_stride, const void *k, const void *v, int64_t kv_batch_stride,
    int64_t kv_tok_stride, int64_t kv_head_stride, const void *out, const void *dout, int64_t o_row_stride,
    int64_t o_head_stride, const int64_t *offsets, void *dq, int64_t dq_row_stride, int64_t dq_head_stride, void *dk,
    void *dv, int64_t dkv_batch_stride, int64_t dkv_tok_stride, int64_t dkv_head_stride, float *workspace, int64_t L, int B,
    int h, int d, int n, int max_rows_per_sample, float scale, int dtype, void *stream)
{
    (void)out;
    return backward(q, q_row_stride, q_head_stride, k, v, kv_batch_stride, kv_tok_stride, kv_head_stride, dout, o_row_stride,
                    o_head_stride, offsets, dq, dq_row_stride, dq_head_stride, dk, dv, dkv_batch_stride, dkv_tok_stride,
                    dkv_head_stride, workspace, false, L, B, h, d, n, max_rows_per_sample, scale, dtype, stream);
}

extern "C" int vtdge_sparse_attention_train_backward(
    const void *q, int64_t q_row_stride, int64_t q_head_stride, const void *k, const void *v, int64_t kv_batch_stride,
    int64_t kv_tok_stride, int64_t kv_head_stride, const void *dout, int64_t o_row_stride, int64_t o_head_stride,
    const int64_t *offsets, void *dq, int64_t dq_row_stride, int64_t dq_head_stride, void *dk, void *dv,
    int64_t dkv_batch_stride, int64_t dkv_tok_stride, int64_t dkv_head_stride, float *workspace, int64_t L, int B, int h, int d,
    int n, int max_rows_per_sample, float scale, int dtype, void *stream)
{
    return backward(q, q_row_stride, q_head_stride, k, v, kv_batch_stride, kv_tok_stride, kv_head_stride, dout, o_row_stride,
                    o_head_stride, offsets, dq, dq_row_stride, dq_head_stride, dk, dv, dkv_batch_stride, dkv_tok_stride,
                    dkv_head_stride, workspace, true, L, B, h, d, n, max_rows_per_sample, scale, dtype, stream);
}
