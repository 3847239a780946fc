// Sparse attention of packed queries against each sample's full K/V, fp32 (gfx950).
//
// What bounds it: the fp32 matrix instructions (64 flops a clock and SIMD) and the vector instructions beside them,
// which do not overlap with them, so the split keeps every SIMD's matrix pipe fed and the softmax short.
//   * A workgroup is 64 query rows of one (sample, head): four waves of ONE 16-query tile each, on
//     v_mfma_f32_16x16x4_f32.  Sixteen-row tiles waste less on ragged query counts and on n = 257 keys than 32-row ones
//     (17 key blocks of 16 against 9 of 32), and in a workgroup of one or two tiles two waves share a tile and split
//     its keys, adding up through LDS at the end.
//   * K/V come in stages of 32 keys by direct loads into two LDS buffers (32 KB): four workgroups share a compute unit,
//     and a stage's loads run under the stage before it.
//   * All first chunks of the samples are dealt out before the second ones: whole workgroups first, remainders into
//     the holes.
// Measured at 64 samples x 6 heads, 26 to 199 queries (6402 rows), n = 257, d = 64: 45 us; workgroups of 8 tiles with
// a ring of 3 or 4 stages 46 us; chunks of a sample next to each other 49 us; 2 tiles a workgroup 60 us; five or six
// workgroups a compute unit 46 and 51 us.  At 128 rows for every sample 37 us, 87 TFLOP/s (8 tiles: 46 us).  At
// one mix of 1/4/16 queries a region (7277 rows, 17 to 257 a sample) 48 us; the kernel before this one, 32-query tiles
// on 128-row workgroups with K/V through registers, took 104 us.
//
// MFMA mapping: S^T = K Q^T (keys are rows, queries columns), then O^T = V^T P^T.  Lane (l = lane % 16, g = lane / 16)
// holds S^T of keys 4 g + r (r < 4) and query l, which is exactly the B operand of the second product when its step r
// contracts over keys 4 g + r: P never moves between lanes.  V stays row-major: in step r a lane needs V[4 g + r] at
// NDB values of d, one per d block, and taking d = NDB l + db for block db makes them one vector read; the output then
// has d = NDB (4 g + r) + db.  For the first product the contraction order is d = 16 j + 4 g + e for step (j, e): one
// 16-byte read of K per four instructions.  K and V rows are stored with their 16-byte chunks XOR-ed by the row, which
// keeps both kinds of read free of bank conflicts without padding (direct loads cannot pad).
#include "common.h"

namespace vtdge {

constexpr int AF_KEYS = 32;      // keys per stage
constexpr int AF_TILES = 4;      // waves = query tiles of a full workgroup
constexpr float AF_RAISE = 8.f;  // log2 units a score may exceed its query's reference by

template <int D> struct AttnF32 {
    static constexpr int ROWB = D * 4;                        // bytes of a K/V row
    static constexpr int CPR = ROWB / 16;                     // 16-byte chunks of it
    static constexpr int BUF = 2 * AF_KEYS * ROWB;            // one stage: K then V
    static constexpr int NDB = D / 16;                        // d blocks of the output
    static __device__ __forceinline__ int slot(int row, int chunk)
    {
        return D == 64 ? chunk ^ (row & 15) : chunk ^ ((row >> 1) & 7);
    }
};

// The 64 query rows `chunk` of (sample, head) `pair`, by a workgroup of four waves.
// WIDE: token strides of 2^23 values and more, or negative ones: 64-bit addresses of the direct loads
template <int D, bool WIDE>
__device__ __forceinline__ void attention_f32_rows(
    unsigned char *smem, const float *__restrict__ q, int64_t q_rs, int64_t q_hs, const float *__restrict__ k,
    const float *__restrict__ v, int64_t kv_bs, int64_t kv_ts, int64_t kv_hs, const int64_t *__restrict__ offsets,
    float *__restrict__ out, int64_t o_rs, int64_t o_hs, int pair, int chunk, int h, int n, float scale_log2)
{
    using G = AttnF32<D>;
    constexpr int NL = G::BUF / 1024 / AF_TILES;              // direct loads a wave and stage
    const int b = pair / h, head = pair - b * h;
    const int64_t row0 = offsets[b];
    const int Lb = (int)(offsets[b + 1] - row0);
    if (chunk * 16 * AF_TILES >= Lb) return;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l = lane & 15, g = lane >> 4;
    // tiles of this workgroup, and how its waves share them
    const int tiles = min(AF_TILES, (Lb - chunk * 16 * AF_TILES + 15) / 16);
    const int split = tiles <= AF_TILES / 2 ? 2 : 1;
    const int tile = wid / split, part = wid % split;
    const bool live = tile < tiles;
    const int qrow = (chunk * AF_TILES + tile) * 16 + l;
    const bool row_live = live && qrow < Lb;

    const unsigned char *kbase = reinterpret_cast<const unsigned char *>(k + (int64_t)b * kv_bs + (int64_t)head * kv_hs);
    const unsigned char *vbase = reinterpret_cast<const unsigned char *>(v + (int64_t)b * kv_bs + (int64_t)head * kv_hs);
    const int64_t rowp = kv_ts * 4;
    const uint32_t lds0 = (uint32_t)(uintptr_t)smem;
    // one stage: loads [wid NL, wid NL + NL) of its BUF / 1024, K rows first.  Rows past the last key repeat it.
    auto load_stage = [&](int st) {
        const int key0 = st * AF_KEYS, last = n - 1 - key0;
        const uint32_t dst = lds0 + (uint32_t)((st & 1) * G::BUF + wid * NL * 1024);
        const unsigned char *src = (wid < AF_TILES / 2 ? kbase : vbase) + (int64_t)key0 * rowp;
        const void *base = uniform_ptr(src);
#pragma unroll
        for (int i = 0; i < NL; i++) {
            const int row = ((wid % (AF_TILES / 2)) * NL + i) * (64 / G::CPR) + lane / G::CPR;
            const uint32_t piece = (uint32_t)G::slot(row, lane % G::CPR) * 16u;
            if constexpr (WIDE) VT_GLOBAL_TO_LDS(src + min(row, last) * rowp + piece, smem + (dst - lds0) + i * 1024);
            else dma16(base, (uint32_t)min(row, last) * (uint32_t)rowp + piece, dst + i * 1024);
        }
    };

    const int stages = (n + AF_KEYS - 1) / AF_KEYS;
    load_stage(0);
    // queries times scale * log2(e): the scores come out of the matrix pipe in log2 units
    f32x4 qf[D / 16];
    {
        const float *qp = q + (row0 + qrow) * q_rs + (int64_t)head * q_hs + 4 * g;
#pragma unroll
        for (int j = 0; j < D / 16; j++)
            qf[j] = (row_live ? *reinterpret_cast<const f32x4 *>(qp + 16 * j) : f32x4{0.f, 0.f, 0.f, 0.f}) * scale_log2;
    }
    f32x4 o[G::NDB];
#pragma unroll
    for (int i = 0; i < G::NDB; i++) o[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    // The softmax's reference m of a query: the accumulators of its scores start from -m, so a probability is one
    // exp2 of what the matrix pipe delivers.  m is the query's maximum over its first stage and is raised (and the
    // running sums rescaled) only when a score exceeds it by more than AF_RAISE; any reference cancels in the end.
    float neg_m = 0.f, l_run = 0.f;
    bool first = true;

    // LDS offsets of this lane's fragments in a stage: K row l, V rows 4 g + r, of the block this part starts with
    int koff[D / 16], voff[4];
#pragma unroll
    for (int j = 0; j < D / 16; j++) koff[j] = (part * 16 + l) * G::ROWB + G::slot(l, 4 * j + g) * 16;
#pragma unroll
    for (int r = 0; r < 4; r++)
        voff[r] = (AF_KEYS + part * 16 + 4 * g + r) * G::ROWB +
                  (D == 64 ? G::slot(4 * g + r, l) * 16 : G::slot(4 * g + r, l >> 1) * 16 + (l & 1) * 8);

    // one stage of a wave: NB blocks of 16 keys (this part's only one, or both), keys >= n masked where TAIL
    auto compute = [&](auto nbc, auto tailc, int st) {
        constexpr int NB = decltype(nbc)::value;
        constexpr bool TAIL = decltype(tailc)::value;
        const unsigned char *S = smem + (st & 1) * G::BUF;
        const int key0 = st * AF_KEYS + part * 16 + 4 * g;    // this lane's first key of block 0
        f32x4 s[NB];
#pragma unroll
        for (int i = 0; i < NB; i++) s[i] = f32x4{neg_m, neg_m, neg_m, neg_m};
#pragma unroll
        for (int j = 0; j < D / 16; j++)
#pragma unroll
            for (int i = 0; i < NB; i++) {
                const f32x4 kf = *reinterpret_cast<const f32x4 *>(S + koff[j] + i * 16 * G::ROWB);
#pragma unroll
                for (int e = 0; e < 4; e++) s[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[e], qf[j][e], s[i], 0, 0, 0);
            }
        float mx = -INFINITY;
#pragma unroll
        for (int i = 0; i < NB; i++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                if constexpr (TAIL)
                    if (key0 + 16 * i + r >= n) s[i][r] = -INFINITY;
                mx = fmaxf(mx, s[i][r]);
            }
        if (__any(first || mx > AF_RAISE)) {
            mx = fmaxf(mx, __shfl_xor(mx, 16, WAVE));
            mx = fmaxf(mx, __shfl_xor(mx, 32, WAVE));
            // a query that has met scores of -infinity only has no reference yet: its probabilities are zero, it waits
            const float d = !first ? fmaxf(mx, 0.f) : mx == -INFINITY ? 0.f : mx;
            const float alpha = first ? 1.f : __builtin_amdgcn_exp2f(-d);
            first = first && mx == -INFINITY;
            neg_m -= d;
#pragma unroll
            for (int i = 0; i < NB; i++) s[i] -= d;
            l_run *= alpha;
#pragma unroll
            for (int i = 0; i < G::NDB; i++) o[i] *= alpha;
        }
#pragma unroll
        for (int i = 0; i < NB; i++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float p = __builtin_amdgcn_exp2f(s[i][r]);
                l_run += p;
                float vf[G::NDB];
                const unsigned char *vp = S + voff[r] + i * 16 * G::ROWB;
                if constexpr (D == 64) {
                    const f32x4 t = *reinterpret_cast<const f32x4 *>(vp);
                    vf[0] = t[0]; vf[1] = t[1]; vf[2] = t[2]; vf[3] = t[3];
                } else {
                    const f32x2 t = *reinterpret_cast<const f32x2 *>(vp);
                    vf[0] = t[0]; vf[1] = t[1];
                }
                if constexpr (TAIL)                           // a repeated row: nothing of it, not even 0 * infinity
                    if (key0 + 16 * i + r >= n)
#pragma unroll
                        for (int db = 0; db < G::NDB; db++) vf[db] = 0.f;
#pragma unroll
                for (int db = 0; db < G::NDB; db++)
                    o[db] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[db], p, o[db], 0, 0, 0);
            }
    };

    for (int st = 0; st < stages; st++) {
        wait_vmcnt<0>();                                      // this wave's loads of stage st have landed
        block_barrier();                                      // stage st is whole; the buffer of st - 1 is free
        if (st + 1 < stages) load_stage(st + 1);
        if (!live) continue;
        const int left = n - st * AF_KEYS - part * 16;        // keys of this part's blocks of the stage, and beyond
        if (split == 1) {
            if (left >= 32) compute(std::integral_constant<int, 2>{}, std::false_type{}, st);
            else if (left > 16) compute(std::integral_constant<int, 2>{}, std::true_type{}, st);
            else compute(std::integral_constant<int, 1>{}, std::true_type{}, st);
        } else {
            if (left >= 16) compute(std::integral_constant<int, 1>{}, std::false_type{}, st);
            else if (left > 0) compute(std::integral_constant<int, 1>{}, std::true_type{}, st);
        }
    }
    float m_run = first ? -INFINITY : -neg_m;                 // a part without keys has no maximum

    l_run += __shfl_xor(l_run, 16, WAVE);
    l_run += __shfl_xor(l_run, 32, WAVE);
    if (split > 1) {
        // the parts of a tile meet in LDS: maximum, sum and accumulators of every part but the first
        float *sh = reinterpret_cast<float *>(smem) + wid * (4 * G::NDB + 2) * 64 + lane;
        lds_barrier();                                        // the last stage has been read
        if (part > 0) {
            sh[0] = m_run;
            sh[64] = l_run;
#pragma unroll
            for (int db = 0; db < G::NDB; db++)
#pragma unroll
                for (int r = 0; r < 4; r++) sh[(2 + 4 * db + r) * 64] = o[db][r];
        }
        lds_barrier();
        if (part > 0) return;
        for (int p = 1; p < split; p++) {
            const float *sp = sh + p * (4 * G::NDB + 2) * 64;
            const float m_new = fmaxf(m_run, sp[0]);
            const float fa = __builtin_amdgcn_exp2f(m_run - m_new), fb = __builtin_amdgcn_exp2f(sp[0] - m_new);
            m_run = m_new;
            l_run = l_run * fa + sp[64] * fb;
#pragma unroll
            for (int db = 0; db < G::NDB; db++)
#pragma unroll
                for (int r = 0; r < 4; r++) o[db][r] = o[db][r] * fa + sp[(2 + 4 * db + r) * 64] * fb;
        }
    }
    if (!row_live) return;
    const float inv = 1.0f / l_run;
    float *op = out + (row0 + qrow) * o_rs + (int64_t)head * o_hs + 4 * G::NDB * g;
    if constexpr (D == 64) {
#pragma unroll
        for (int r = 0; r < 4; r++)
            *reinterpret_cast<f32x4 *>(op + 4 * r) = f32x4{o[0][r] * inv, o[1][r] * inv, o[2][r] * inv, o[3][r] * inv};
    } else {
#pragma unroll
        for (int r = 0; r < 4; r += 2)
            *reinterpret_cast<f32x4 *>(op + 2 * r) =
                f32x4{o[0][r] * inv, o[1][r] * inv, o[0][r + 1] * inv, o[1][r + 1] * inv};
    }
}

template <int D, bool WIDE>
__global__ __launch_bounds__(64 * AF_TILES, 4) void attention_f32_kernel(
    const float *__restrict__ q, int64_t q_rs, int64_t q_hs, const float *__restrict__ k, const float *__restrict__ v,
    int64_t kv_bs, int64_t kv_ts, int64_t kv_hs, const int64_t *__restrict__ offsets, float *__restrict__ out,
    int64_t o_rs, int64_t o_hs, int pairs, int h, int n, float scale_log2)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    // the chunks of a (sample, head) pair run on one XCD, so its K/V are fetched into one L2
    const int rest = blockIdx.x >> 3, pairs_x = (pairs + 7) / 8;
    const int pair = (rest % pairs_x) * 8 + (blockIdx.x & 7), chunk = rest / pairs_x;
    if (pair >= pairs) return;
    attention_f32_rows<D, WIDE>(smem, q, q_rs, q_hs, k, v, kv_bs, kv_ts, kv_hs, offsets, out, o_rs, o_hs, pair, chunk, h, n,
                                scale_log2);
}

// ---------------------------------------------------------------------------------------------------------
// head_dim 64 on the bf16 matrix instructions, as exact: queries, keys, probabilities and values are each the sum of three bf16
// values (exactly, where the third is no smaller than bf16 goes), six of the nine partial products of two such sums are multiplied
// and added in fp32 (linear_dma_split.hip says what the other three are).  Per 32 keys and 16 queries that is 768 clocks of matrix
// instructions against 2048; against float64 the output is off by 3.7e-7 against 4.1e-7 (2-norm; 257 keys, unit normals).
// What bounds it are the vector instructions: splitting a stage of K and V (88 a wave) and the probabilities (44), the
// exponentials and 36 reads of LDS, some 300 a wave and stage beside 48 matrix instructions.
//   * 64 query rows a workgroup, 16 a wave; a stage of 32 keys goes through registers, is split and written to LDS as planes of
//     bf16 rows (24 KB), the next one on its way from memory meanwhile.  One buffer and two barriers a stage leave room for
//     four workgroups a compute unit, which fill each other's waits: 34.5 us at 128 samples, 3 heads, 257 keys, 14146 rows;
//     with two buffers (three workgroups) 39.7, 128 rows on eight waves 39.1, two tiles of queries a wave 47.9.
//   * V comes out of LDS transposed (ds_read_b64_tr_b16), so that the operand of step j holds the keys whose probabilities the
//     lane has: P never moves between lanes.
//   * A workgroup of one or two tiles takes the fp32 instructions, whose waves share a tile (20 queries of 128 samples: 17.4
//     against 20.9 us), and so does one with anything the split is not exact for: sums that are not finite, tiny or huge
//     ones, queries far from one, large values.
constexpr int AS_KEYS = 32;                          // keys per stage
constexpr int AS_PLANE = AS_KEYS * 128;              // bytes of a plane: 32 rows of 64 bf16 values
constexpr int AS_BUF = 6 * AS_PLANE;                 // one stage: three planes of K, then three of V
constexpr float AS_TINY = 0x1p-80f, AS_FAR = 0x1p60f;
// A probability below 2^-108 loses parts under the smallest bf16 number, up to 2^-134: over values below 2^20 that is less than
// 2^-34 a key of a sum that is not tiny.
constexpr float AS_LARGE = 0x1p20f;

// x[0..7] into three bf16 parts each: x = p[0] + p[1] + p[2] (nearest parts, signed remainders)
__device__ __forceinline__ void split8(const float (&x)[8], u32x4 (&p)[3])
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
__device__ __forceinline__ f32x4 mma_bf16_16(const u32x4 &a, const u32x4 &b, const f32x4 &c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// The 64 query rows `chunk` of a pair as attention_f32_rows computes them -> whether it could
__device__ __forceinline__ bool attention_f32_split_rows(
    unsigned char *smem, const float *__restrict__ q, int64_t q_rs, int64_t q_hs, const float *__restrict__ k, const float *__restrict__ v,
    int64_t kv_bs, int64_t kv_ts, int64_t kv_hs, const int64_t *__restrict__ offsets, float *__restrict__ out,
    int64_t o_rs, int64_t o_hs, int pair, int chunk, int h, int n, float scale_log2)
{
    constexpr int ROWS = 16 * AF_TILES;
    const int b = pair / h, head = pair - b * h;
    const int64_t row0 = offsets[b];
    const int Lb = (int)(offsets[b + 1] - row0);
    if (chunk * ROWS >= Lb) return true;
    const int tiles = min(AF_TILES, (Lb - chunk * ROWS + 15) / 16);
    if (tiles <= AF_TILES / 2) return false;                  // two waves a tile do better there

    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l = lane & 15, g = lane >> 4;
    const bool live = wid < tiles;

    // This thread's part of a stage: 8 values of a row of K and of V
    const int srow = tid >> 3, schunk = tid & 7;
    const float *kp = k + (int64_t)b * kv_bs + (int64_t)head * kv_hs + 8 * schunk;
    const float *vp = v + (int64_t)b * kv_bs + (int64_t)head * kv_hs + 8 * schunk;
    float rk[8], rv[8];
    bool large = false;                                      // a value of this wave's that is
    auto load_stage = [&](int st) {                          // rows past the last key repeat it
        const int64_t off = (int64_t)min(st * AS_KEYS + srow, n - 1) * kv_ts;
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const f32x4 a = *reinterpret_cast<const f32x4 *>(kp + off + 4 * i), c = *reinterpret_cast<const f32x4 *>(vp + off + 4 * i);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                rk[4 * i + e] = a[e];
                rv[4 * i + e] = c[e];
            }
        }
    };
    const int kdst = srow * 128 + ((schunk ^ ((srow >> 1) & 7)) * 16);
    const int vdst = 3 * AS_PLANE + srow * 128 + ((schunk ^ (2 * ((srow >> 1) & 3))) * 16);
    auto store_stage = [&](int st) {
        if (st * AS_KEYS + AS_KEYS > n) {                    // nothing of a repeated row, not even 0 * infinity
            const bool past = st * AS_KEYS + srow >= n;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                rk[e] = past ? 0.f : rk[e];
                rv[e] = past ? 0.f : rv[e];
            }
        }
        u32x4 p[3];
        split8(rk, p);
#pragma unroll
        for (int i = 0; i < 3; i++) *reinterpret_cast<u32x4 *>(smem + kdst + i * AS_PLANE) = p[i];
        float most = 0.f;
#pragma unroll
        for (int e = 0; e < 8; e++) most = __builtin_amdgcn_fmed3f(fabsf(rv[e]), most, INFINITY);            // the maximum
        large = large || __builtin_amdgcn_ballot_w64(!(most < AS_LARGE)) != 0;
        split8(rv, p);
#pragma unroll
        for (int i = 0; i < 3; i++) *reinterpret_cast<u32x4 *>(smem + vdst + i * AS_PLANE) = p[i];
    };

    load_stage(0);
    // queries times scale * log2(e), split: step t of the contraction takes d = 32 t + 8 g + (0 .. 7)
    const int qrow = chunk * ROWS + wid * 16 + l;
    const bool row_live = qrow < Lb;
    u32x4 qf[2][3];
    bool odd = false;                                        // something the split is not exact for
    {
        const float *qp = q + (row0 + qrow) * q_rs + (int64_t)head * q_hs + 8 * g;
#pragma unroll
        for (int t = 0; t < 2; t++) {
            float x[8];
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const f32x4 a = row_live ? *reinterpret_cast<const f32x4 *>(qp + 32 * t + 4 * j) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    x[4 * j + e] = a[e] * scale_log2;
                    const float m = fabsf(x[4 * j + e]);
                    odd = odd || !(m <= AS_FAR) || (m < 1.f / AS_FAR && a[e] != 0.f && scale_log2 != 0.f);
                }
            }
            split8(x, qf[t]);
        }
        odd = fresh(odd) != 0;                               // here: the compiler would keep the queries for a test at the end
    }
    f32x4 o[4];
#pragma unroll
    for (int db = 0; db < 4; db++) o[db] = f32x4{0.f, 0.f, 0.f, 0.f};
    float neg_m = 0.f, l_run = 0.f;                          // the reference and the row sum, as in attention_f32_rows
    bool first = true;
    int koff[2], voff[4];
#pragma unroll
    for (int t = 0; t < 2; t++) koff[t] = l * 128 + (((4 * t + g) ^ ((l >> 1) & 7)) * 16);      // K row l, chunk 4 t + g
    {
        // the transposing reads of V: source lane 4 e + r of a block of 16 names key 4 g + e (+ 16), channels 4 r ..
        const int key = 4 * g + (l >> 2), r = l & 3;
#pragma unroll
        for (int db = 0; db < 4; db++)
            voff[db] = 3 * AS_PLANE + key * 128 + (((2 * db + (r >> 1)) ^ (2 * ((key >> 1) & 3))) * 16) + 8 * (r & 1);
    }
    constexpr int PA[6] = {2, 0, 1, 1, 0, 0}, PB[6] = {0, 2, 1, 0, 1, 0};     // partial products, the small ones first

    // the 32 keys of a stage; those >= n are masked (their K and V are zero)
    auto compute = [&](int st) {
        f32x4 s[2];
#pragma unroll
        for (int kb = 0; kb < 2; kb++) {
            s[kb] = f32x4{neg_m, neg_m, neg_m, neg_m};
#pragma unroll
            for (int t = 0; t < 2; t++) {
                u32x4 kf[3];
#pragma unroll
                for (int p = 0; p < 3; p++) kf[p] = *reinterpret_cast<const u32x4 *>(smem + koff[t] + kb * 16 * 128 + p * AS_PLANE);
#pragma unroll
                for (int x = 0; x < 6; x++) s[kb] = mma_bf16_16(kf[PA[x]], qf[t][PB[x]], s[kb]);
            }
        }
        if (st * AS_KEYS + AS_KEYS > n) {
            const int left = n - st * AS_KEYS - 4 * g;       // keys from this lane's first one on
#pragma unroll
            for (int e = 0; e < 8; e++)
                if (16 * (e / 4) + e % 4 >= left) s[e / 4][e % 4] = -INFINITY;
        }
        // whether a score is that far above the reference: the largest bit pattern orders positive floats as floats do
        int bits = __float_as_int(s[0][0]);
#pragma unroll
        for (int e = 1; e < 8; e++) bits = max(bits, __float_as_int(s[e / 4][e % 4]));
        if (__any(first || __int_as_float(bits) > AF_RAISE)) {
            float mx = -INFINITY;
#pragma unroll
            for (int e = 0; e < 8; e++) mx = fmaxf(mx, s[e / 4][e % 4]);
            mx = fmaxf(mx, __shfl_xor(mx, 16, WAVE));
            mx = fmaxf(mx, __shfl_xor(mx, 32, WAVE));
            const float d = !first ? fmaxf(mx, 0.f) : mx == -INFINITY ? 0.f : mx;
            const float alpha = first ? 1.f : __builtin_amdgcn_exp2f(-d);
            first = first && mx == -INFINITY;
            neg_m -= d;
            s[0] -= d;
            s[1] -= d;
            l_run *= alpha;
#pragma unroll
            for (int db = 0; db < 4; db++) o[db] *= alpha;
        }
        u32x4 pf[3];
        float p[8];
#pragma unroll
        for (int e = 0; e < 8; e++) {
            p[e] = __builtin_amdgcn_exp2f(s[e / 4][e % 4]);
            l_run += p[e];
        }
        split8(p, pf);
#pragma unroll
        for (int db = 0; db < 4; db++) {
            u32x4 vf[3];
#pragma unroll
            for (int i = 0; i < 3; i++) {
                const unsigned char *vs = smem + voff[db] + i * AS_PLANE;
                const u32x2 lo = lds_read_tr16(vs), hi = lds_read_tr16(vs + 16 * 128);
                vf[i] = u32x4{lo.x, lo.y, hi.x, hi.y};
            }
#pragma unroll
            for (int x = 0; x < 6; x++) o[db] = mma_bf16_16(vf[PA[x]], pf[PB[x]], o[db]);
        }
    };

    const int stages = (n + AS_KEYS - 1) / AS_KEYS;
    for (int st = 0; st < stages; st++) {
        if (st > 0) lds_barrier();                           // the stage before has been read
        store_stage(st);
        if (st + 1 < stages) load_stage(st + 1);
        lds_barrier();                                       // stage st is whole
        if (live) compute(st);
    }
    l_run += __shfl_xor(l_run, 16, WAVE);
    l_run += __shfl_xor(l_run, 32, WAVE);
    odd = odd || large;
    if (row_live) {
        odd = odd || !(l_run < INFINITY);
#pragma unroll
        for (int e = 0; e < 16; e++) {
            const float m = fabsf(o[e / 4][e % 4]);
            odd = odd || !(m <= AS_FAR) || (m < AS_TINY && m != 0.f);
        }
    }
    if (__syncthreads_or(odd ? 1 : 0)) return false;
    if (!row_live) return true;
    const float inv = 1.0f / l_run;
    float *op = out + (row0 + qrow) * o_rs + (int64_t)head * o_hs + 4 * g;
#pragma unroll
    for (int db = 0; db < 4; db++)
        *reinterpret_cast<f32x4 *>(op + 16 * db) = f32x4{o[db][0] * inv, o[db][1] * inv, o[db][2] * inv, o[db][3] * inv};
    return true;
}

template <bool WIDE>
__global__ __launch_bounds__(64 * AF_TILES, 4) void attention_f32_split_kernel(
    const float *__restrict__ q, int64_t q_rs, int64_t q_hs, const float *__restrict__ k, const float *__restrict__ v,
    int64_t kv_bs, int64_t kv_ts, int64_t kv_hs, const int64_t *__restrict__ offsets, float *__restrict__ out,
    int64_t o_rs, int64_t o_hs, int pairs, int h, int n, float scale_log2)
{
    extern __shared__ __attribute__((aligned(128))) unsigned char smem[];
    const int rest = blockIdx.x >> 3, pairs_x = (pairs + 7) / 8;
    const int pair = (rest % pairs_x) * 8 + (blockIdx.x & 7), chunk = rest / pairs_x;
    if (pair >= pairs) return;
    if (!attention_f32_split_rows(smem, q, q_rs, q_hs, k, v, kv_bs, kv_ts, kv_hs, offsets, out, o_rs, o_hs, pair, chunk, h, n,
                                  scale_log2))
        attention_f32_rows<64, WIDE>(smem, q, q_rs, q_hs, k, v, kv_bs, kv_ts, kv_hs, offsets, out, o_rs, o_hs, pair, chunk, h, n,
                                     scale_log2);
}

template <int D, bool WIDE, bool SPLIT>
static int go_attention_f32(const void *q, int64_t q_rs, int64_t q_hs, const void *k, const void *v, int64_t kv_bs,
                            int64_t kv_ts, int64_t kv_hs, const int64_t *offsets, void *out, int64_t o_rs, int64_t o_hs,
                            int B, int h, int n, int max_rows, float scale, hipStream_t st)
{
    constexpr size_t lds = 2 * AttnF32<D>::BUF;
    static_assert(!SPLIT || lds >= AS_BUF, "a stage of split keys and values");
    const int64_t pairs = (int64_t)B * h, chunks = ceil_div(max_rows, 16 * AF_TILES);
    const int64_t grid = ceil_div(pairs, 8) * 8 * chunks;
    VT_REQUIRE(grid < (1ll << 31), VTDGE_ERR_UNSUPPORTED, "sparse_attention: %lld workgroups exceed one launch",
               (long long)grid);
    constexpr auto kern = [] {
        if constexpr (SPLIT) return attention_f32_split_kernel<WIDE>;
        else return attention_f32_kernel<D, WIDE>;
    }();
    VT_RESERVE_LDS(kern, lds, "sparse_attention");
    note_kernel(reinterpret_cast<const void *>(kern));
    kern<<<dim3((unsigned)grid), dim3(64 * AF_TILES), lds, st>>>(
        (const float *)q, q_rs, q_hs, (const float *)k, (const float *)v, kv_bs, kv_ts, kv_hs, offsets, (float *)out,
        o_rs, o_hs, (int)pairs, h, n, scale * 1.44269504088896340736f);
    return check_launch("sparse_attention");
}
template <int D>
int launch_attention_f32(const void *q, int64_t q_rs, int64_t q_hs, const void *k, const void *v, int64_t kv_bs,
                         int64_t kv_ts, int64_t kv_hs, const int64_t *offsets, void *out, int64_t o_rs, int64_t o_hs,
                         int B, int h, int n, int max_rows, float scale, hipStream_t st)
{
    const bool wide = !(kv_ts >= 0 && kv_ts < (1 << 23));
    auto go = wide ? go_attention_f32<D, true, false> : go_attention_f32<D, false, false>;
    // The bf16 instructions from about as many workgroups on as put one on every compute unit and some beside it, and for long
    // chains of keys.  Us, fp32 / bf16 instructions (samples, heads, keys, live rows): 128, 3, 257, 14146: 44.1 / 34.5;
    // 64, 6, 257, 6596: 44.2 / 33.7; 64, 6, 145, 4834: 25.8 / 20.3; 64, 6, 64, 16384: 25.3 / 21.6; 16, 6, 257, 2021: 23.6 /
    // 19.9; 6, 1, 144, 24192: 16.8 / 15.2; 32, 6, 1025, 15106: 302 / 191; 8, 6, 1025, 3169: 77.0 / 60.0.  Below the line:
    // 8, 6, 257, 862: 15.3 / 15.8; 6, 5, 144, 1512: 10.1 / 10.9; 64, 3, 65, 2033: 8.4 / 9.2.
    const int64_t wgs = (int64_t)B * h * ceil_div(max_rows, 16 * AF_TILES);
    if constexpr (D == 64)
        if (n > 512 || (wgs >= 320 && wgs * n >= 48000))
            go = wide ? go_attention_f32<D, true, true> : go_attention_f32<D, false, true>;
    return go(q, q_rs, q_hs, k, v, kv_bs, kv_ts, kv_hs, offsets, out, o_rs, o_hs, B, h, n, max_rows, scale, st);
}
template int launch_attention_f32<64>(const void *, int64_t, int64_t, const void *, const void *, int64_t, int64_t,
                                      int64_t, const int64_t *, void *, int64_t, int64_t, int, int, int, int, float,
                                      hipStream_t);
template int launch_attention_f32<32>(const void *, int64_t, int64_t, const void *, const void *, int64_t, int64_t,
                                      int64_t, const int64_t *, void *, int64_t, int64_t, int, int, int, int, float,
                                      hipStream_t);

}  // namespace vtdge
