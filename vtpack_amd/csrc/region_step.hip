// From the packed queries of one block to those of the next in one launch, a workgroup per 4 x 4 region (gfx950): scatter
// back, the next block's router, its index -> patch and compress, and whatever its first LayerNorm wants of tokens and rows.
//
// With few regions the launches this replaces - decompress_route_kernel, compress_regions or patch_write + compress,
// layernorm - are chains of round trips to memory by four waves on four regions each: 300 instructions a token one after the other
// in a wave that has its SIMD for itself; with many, up to 50 a compute unit, they are the passes over the tokens that this one
// does not repeat (vtdge_region_step_fits has the line).  Here a wave has one row of four tokens; the sixteen meet
// in LDS, where wave 0 adds them up for the router in the one order all kernels use while the other waves write what
// LayerNorm wants of theirs.  What the router needs is requested first of all, and its decision is published before
// anything that can wait.  Every value has the arithmetic, the order and the rounding of the kernels named above: the
// results are theirs bit for bit.
//
// The first packed row of a region is the number of queries of all regions before it: handed along in launch order through
// status words (handover.h), a workgroup waits for workgroups with smaller numbers only.
#include "region_pack.h"

namespace vtdge {

namespace {

template <typename T> struct RegionStep {
    const T *in, *sub, *ref;               // packed queries after and before the block, tokens before it
    const int64_t *cur_indices, *splits, *offsets;
    const int32_t *region_rows;            // with cur_counts (nullable): this block's first packed rows
    const uint8_t *cur_counts;
    T *out;
    const T *weight, *bias;                // the next router
    T *gate;                               // nullable
    int64_t *indices;
    const int64_t *next_splits;
    uint8_t *next_counts;
    u32x4 *records;                        // nullable: statistics records of the tokens
    T *out_ln;                             // nullable: their LayerNorm
    const T *ln_w, *ln_b;
    float eps;
    T *comp;
    u32x4 *comp_records;                   // nullable, with records
    T *comp_ln;                            // nullable, with out_ln
    int64_t *patches;
    int64_t capacity;
    int64_t *next_offsets;
    int32_t *next_region_rows;
    unsigned long long *status;
    int B, H, W, C, extra, S, S2;
};

// The sums of NN rows, every lane a piece of each, in all lanes.  NARROW, rows of at most 32 vectors: in the order of the kernels
// that give such a row to a group of 8, 16 or 32 lanes, the lane half a group away first (more than half a group away there is
// nothing but zeros), so that both ways give the same bits.
template <bool NARROW, int NN> __device__ __forceinline__ void row_sums(float (&v)[NN])
{
    if constexpr (!NARROW) {
        wave_sum_n<NN>(v);
        return;
    }
#pragma unroll
    for (int i = 0; i < NN; i++) {
        const auto r16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[i]), __float_as_uint(v[i]), false, false);
        v[i] = __uint_as_float(r16[0]) + __uint_as_float(r16[1]);
    }
#pragma unroll
    for (int i = 0; i < NN; i++) v[i] += dpp_move<0x128>(v[i]);                    // lane ^ 8
#pragma unroll
    for (int i = 0; i < NN; i++) v[i] += dpp_move<0x141>(dpp_move<0x1B>(v[i]));    // lane ^ 4
#pragma unroll
    for (int i = 0; i < NN; i++) v[i] += dpp_move<0x4E>(v[i]);                     // lane ^ 2
#pragma unroll
    for (int i = 0; i < NN; i++) v[i] += dpp_move<0xB1>(v[i]);                     // lane ^ 1
#pragma unroll
    for (int i = 0; i < NN; i++)
        v[i] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v[i]), 0));
}
template <bool NARROW> __device__ __forceinline__ float row_sum(float v)
{
    if constexpr (!NARROW) return wave_sum(v);
    float one[1] = {v};
    row_sums<NARROW, 1>(one);
    return one[0];
}

// layernorm_kernel's arithmetic for one row held by a wave, a vector or several a lane
template <typename T, int NV, bool NARROW>
__device__ __forceinline__ void norm_row(const u32x4 (&row)[NV], const bool (&act)[NV], const u32x4 (&w)[NV],
                                         const u32x4 (&bb)[NV], float eps, int C, T *dst)
{
    constexpr int VEC = Elem<T>::VEC;
    float vals[NV][VEC];
    float s = 0.f, q = 0.f;
#pragma unroll
    for (int it = 0; it < NV; it++)
        if (act[it]) {
            Elem<T>::unpack(row[it], vals[it]);
#pragma unroll
            for (int c = 0; c < VEC; c++) s += vals[it][c];
        }
    const float mean = row_sum<NARROW>(s) / (float)C;
#pragma unroll
    for (int it = 0; it < NV; it++)
        if (act[it]) {
#pragma unroll
            for (int c = 0; c < VEC; c++) {
                const float dlt = vals[it][c] - mean;
                q += dlt * dlt;
            }
        }
    const float rstd = 1.0f / sqrtf(row_sum<NARROW>(q) / (float)C + eps);
#pragma unroll
    for (int it = 0; it < NV; it++)
        if (act[it]) {
            float y[VEC], wf[VEC], bf[VEC];
            Elem<T>::unpack(w[it], wf);
            Elem<T>::unpack(bb[it], bf);
#pragma unroll
            for (int c = 0; c < VEC; c++) y[c] = (vals[it][c] - mean) * rstd * wf[c] + bf[c];
            *reinterpret_cast<u32x4 *>(dst + it * WAVE * VEC) = Elem<T>::pack(y);
        }
}

// The same for the four rows of a wave, one step of all of them after the other: their sums are four independent chains, and
// their quotients and roots are taken once, in four lanes side by side (the same operations on the same values).  With that,
// the LayerNorm of a region that stays 16 queries taken over from its tokens, and registers for four waves a SIMD, a launch at
// 2048 regions of 192 fp32 channels went from 39.9 to 36.3 us (119 MB), at 80 regions of 768 bf16 channels from 15.5 to 13.9.
template <typename T, int NV, bool NARROW>
__device__ __forceinline__ void norm_rows4(const u32x4 (&row)[4][NV], const bool (&act)[NV], const u32x4 (&w)[NV],
                                           const u32x4 (&bb)[NV], float eps, int C, T *dst, u32x4 (&y4)[4][NV])
{
    constexpr int VEC = Elem<T>::VEC;
    const int lane = threadIdx.x & 63;
    // (the values come by value: behind a reference the selection turns into a load through a computed address)
    auto per_row = [&](float v0, float v1, float v2, float v3, auto f, float (&out)[4]) {
        const float r = f(lane & 2 ? (lane & 1 ? v3 : v2) : (lane & 1 ? v1 : v0));
#pragma unroll
        for (int t = 0; t < 4; t++)
            out[t] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, r), t));
    };
    float vals[4][NV][VEC], s[4], q[4], mean[4], rstd[4];
#pragma unroll
    for (int t = 0; t < 4; t++) {
        s[t] = 0.f;
#pragma unroll
        for (int it = 0; it < NV; it++)
            if (act[it]) {
                Elem<T>::unpack(row[t][it], vals[t][it]);
#pragma unroll
                for (int c = 0; c < VEC; c++) s[t] += vals[t][it][c];
            }
    }
    row_sums<NARROW, 4>(s);
    per_row(s[0], s[1], s[2], s[3], [&](float v) { return v / (float)C; }, mean);
#pragma unroll
    for (int t = 0; t < 4; t++) {
        q[t] = 0.f;
#pragma unroll
        for (int it = 0; it < NV; it++)
            if (act[it]) {
#pragma unroll
                for (int c = 0; c < VEC; c++) {
                    const float dlt = vals[t][it][c] - mean[t];
                    q[t] += dlt * dlt;
                }
            }
    }
    row_sums<NARROW, 4>(q);
    per_row(q[0], q[1], q[2], q[3], [&](float v) { return 1.0f / sqrtf(v / (float)C + eps); }, rstd);
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
        for (int it = 0; it < NV; it++)
            if (act[it]) {
                float y[VEC], wf[VEC], bf[VEC];
                Elem<T>::unpack(w[it], wf);
                Elem<T>::unpack(bb[it], bf);
#pragma unroll
                for (int c = 0; c < VEC; c++) y[c] = (vals[t][it][c] - mean[t]) * rstd[t] * wf[c] + bf[c];
                y4[t][it] = Elem<T>::pack(y);
                *reinterpret_cast<u32x4 *>(dst + (int64_t)t * C + it * WAVE * VEC) = y4[t][it];
            }
}

// the record of one row, from wave-wide sums
template <typename T>
__device__ __forceinline__ void record_row(const u32x4 &row, bool act, float eps, int C, u32x4 *rec)
{
    const int lane = threadIdx.x & 63;
    float pivot, st[2];
    lane_sums<T>(row, act, pivot, st[0], st[1]);
    wave_sum_n<2>(st);
    u32x4 lo, hi;
    row_record(pivot, st[0], st[1], C, eps, lo, hi);
    if (lane < 2) rec[lane] = lane ? hi : lo;
}

}  // namespace

template <typename T, int NV, bool REC, bool NARROW>
__global__ __launch_bounds__(256, NV == 1 ? (REC ? 6 : 5) : NV == 2 ? 3 : 2) void region_step_kernel(const RegionStep<T> a)
{
    static_assert(!REC || (NV == 1 && sizeof(T) == 2 && !NARROW), "records: bf16 rows of one vector a lane");
    constexpr int VEC = Elem<T>::VEC;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    u32x4 *const held = reinterpret_cast<u32x4 *>(smem);          // [16 tokens][vectors]
    __shared__ int s_split;
    __shared__ long long s_before;

    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int Hr = a.H / 4, Wr = a.W / 4, nreg = Hr * Wr, region = blockIdx.x;
    const int b = region / nreg, rr = region % nreg, ry = rr / Wr, rx = rr % Wr;
    const int C = a.C, nvec = C / VEC, extra = a.extra, N = extra + a.H * a.W;
    bool act[NV];
#pragma unroll
    for (int it = 0; it < NV; it++) act[it] = it * WAVE + lane < nvec;
    const u32x4 z = {0u, 0u, 0u, 0u};

    // ---- what depends on nothing before: the router (wave 0) and the LayerNorm's parameters.  The weights of more than four
    // splits are read where they are used, and the LayerNorm's of rows of three vectors a lane behind the scatter: the registers,
    // 96, 167 and 225 where all eight splits took 123, 201 and 290; rows with records read two ahead and the third behind the scatter
    // (80 registers, six workgroups: 120 pictures of 384 channels 1787 -> 1764 us, 176: 2323 -> 2280).  A forward with four and five workgroups a compute unit for rows
    // of one vector, two and three for two, us (pictures): DeiT-S bf16 80: 1302 / 1260, 130: 1853 / 1840; DeiT-Ti bf16 200: 1492 /
    // 1458, 400: 2581 / 2523; fp32 300: 5446 / 5412; DeiT-B bf16 99: 3965 / 3889, 5: 978 / 975; DeiT-S fp32 33: 2386 / 2351.  With
    // scratch memory instead (three workgroups, all eight early) 99 pictures took 4266 where 4116 were taken.
    constexpr int EARLY = REC ? 3 : 4, FIRST = REC ? 2 : EARLY;
    u32x4 rw[EARLY][NV];
    float rbias = 0.f;
    int rsplit = 1;
    if (wv == 0) {
#pragma unroll
        for (int s = 0; s < FIRST; s++)
            if (s < a.S2) {
#pragma unroll
                for (int it = 0; it < NV; it++) {
                    rw[s][it] = z;
                    if (act[it])
                        rw[s][it] = *reinterpret_cast<const u32x4 *>(a.weight + (int64_t)s * C + (it * WAVE + lane) * VEC);
                }
            }
        if (lane < a.S2) {
            rbias = Elem<T>::load(a.bias + lane);
            rsplit = (int)a.next_splits[lane];
        }
    }
    u32x4 lw[NV], lb[NV];
    const bool normed = !REC && a.out_ln != nullptr;
    auto norm_parameters = [&]() {
#pragma unroll
        for (int it = 0; it < NV; it++)
            if (act[it]) {
                lw[it] = *reinterpret_cast<const u32x4 *>(a.ln_w + (it * WAVE + lane) * VEC);
                lb[it] = *reinterpret_cast<const u32x4 *>(a.ln_b + (it * WAVE + lane) * VEC);
            }
    };
    if (NV <= 2 && normed) norm_parameters();

    // ---- this block's place of the region
    int64_t r0, row_b;
    int ps;
    if (a.region_rows != nullptr) {
        r0 = a.region_rows[region];
        row_b = r0 - extra;                     // used for a sample's first region only
        const int cnt = a.cur_counts[region];
        ps = cnt == 16 ? 4 : cnt == 4 ? 2 : 1;
    } else {
        auto split_of = [&](int reg) {
            int64_t g = a.cur_indices[(int64_t)b * nreg + reg];
            g = g < 0 ? 0 : (g >= a.S ? a.S - 1 : g);
            return (int)a.splits[g];
        };
        float before = 0.f;
        for (int r2 = lane; r2 < rr; r2 += WAVE) {
            const int ps2 = split_of(r2);
            before += (float)(ps2 * ps2);
        }
        row_b = a.offsets[b];
        r0 = row_b + extra + (int64_t)wave_sum(before);
        ps = split_of(rr);
    }
    ps = __builtin_amdgcn_readfirstlane(ps);

    // ---- this wave's row of four tokens: out = (in - sub) + ref, each step rounded to the storage type (nothing reads in,
    // sub and ref again: nontemporal loads)
    u32x4 tok[4][NV];
    const int64_t tok0 = ((int64_t)b * N + extra + (int64_t)(ry * 4 + wv) * a.W + rx * 4) * C + lane * VEC;
    auto scatter = [&](auto ps_c) {
        constexpr int PS = decltype(ps_c)::value, STEP = 4 / PS;
        const int64_t q0 = (r0 + (wv / STEP) * PS) * C + lane * VEC;
        u32x4 ir[PS][NV], sr[PS][NV];
        auto read = [&](const T *p) { return __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(p)); };
#pragma unroll
        for (int it = 0; it < NV; it++) {
            const int at = it * WAVE * VEC;
#pragma unroll
            for (int j = 0; j < PS; j++) {
                ir[j][it] = sr[j][it] = z;
                if (act[it]) {
                    ir[j][it] = read(a.in + q0 + (int64_t)j * C + at);
                    sr[j][it] = read(a.sub + q0 + (int64_t)j * C + at);
                }
            }
#pragma unroll
            for (int t = 0; t < 4; t++) {
                tok[t][it] = z;
                if (act[it]) tok[t][it] = read(a.ref + tok0 + (int64_t)t * C + at);
            }
        }
#pragma unroll
        for (int it = 0; it < NV; it++) {
            float d[PS][VEC];
#pragma unroll
            for (int j = 0; j < PS; j++) {
                float sv[VEC];
                Elem<T>::unpack(ir[j][it], d[j]);
                Elem<T>::unpack(sr[j][it], sv);
#pragma unroll
                for (int c = 0; c < VEC; c++) d[j][c] -= sv[c];
                Elem<T>::unpack(Elem<T>::pack(d[j]), d[j]);
            }
#pragma unroll
            for (int t = 0; t < 4; t++) {
                float r[VEC];
                Elem<T>::unpack(tok[t][it], r);
#pragma unroll
                for (int c = 0; c < VEC; c++) r[c] += d[t / STEP][c];
                tok[t][it] = Elem<T>::pack(r);
                if (act[it]) {
                    held[(4 * wv + t) * nvec + it * WAVE + lane] = tok[t][it];
                    *reinterpret_cast<u32x4 *>(a.out + tok0 + (int64_t)t * C + it * WAVE * VEC) = tok[t][it];
                }
            }
        }
    };
    if (ps == 4) scatter(std::integral_constant<int, 4>{});
    else if (ps == 2) scatter(std::integral_constant<int, 2>{});
    else scatter(std::integral_constant<int, 1>{});
    if (NV > 2 && normed) norm_parameters();
    if constexpr (FIRST < EARLY)
        if (wv == 0) {
#pragma unroll
            for (int s = FIRST; s < EARLY; s++)
                if (s < a.S2) {
                    rw[s][0] = z;
                    if (act[0]) rw[s][0] = *reinterpret_cast<const u32x4 *>(a.weight + (int64_t)s * C + lane * VEC);
                }
        }
    lds_barrier();

    // ---- the next router on the tokens as stored (wave 0), published at once
    u32x4 pooled[NV];
    int nq = 0;
    if (wv == 0) {
        float part[VTDGE_MAX_SPLITS];
#pragma unroll
        for (int s = 0; s < VTDGE_MAX_SPLITS; s++) part[s] = 0.f;
#pragma unroll
        for (int it = 0; it < NV; it++) {
            float acc[VEC];
#pragma unroll
            for (int c = 0; c < VEC; c++) acc[c] = 0.f;
            pooled[it] = z;
            if (act[it]) {
#pragma unroll
                for (int h = 0; h < 16; h += 8) {
                    u32x4 t8[8];
#pragma unroll
                    for (int t = 0; t < 8; t++) t8[t] = held[(h + t) * nvec + it * WAVE + lane];
#pragma unroll
                    for (int t = 0; t < 8; t++) add_vector<T>(acc, t8[t]);
                }
#pragma unroll
                for (int c = 0; c < VEC; c++) acc[c] = Elem<T>::round(acc[c] / 16.f);
                pooled[it] = Elem<T>::pack(acc);
#pragma unroll
                for (int s = 0; s < VTDGE_MAX_SPLITS; s++)
                    if (s < a.S2) {
                        float w[VEC];
                        if (s < EARLY) Elem<T>::unpack(rw[s < EARLY ? s : 0][it], w);
                        else Elem<T>::unpack(*reinterpret_cast<const u32x4 *>(a.weight + (int64_t)s * C + (it * WAVE + lane) * VEC), w);
#pragma unroll
                        for (int c = 0; c < VEC; c++) part[s] += acc[c] * w[c];
                    }
            }
        }
        float best = 0.f;
        int best_s = 0;
#pragma unroll
        for (int s = 0; s < VTDGE_MAX_SPLITS; s++)
            if (s < a.S2) {
                float logit =
                    row_sum<NARROW>(part[s]) + __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(rbias), s));
                logit = Elem<T>::round(logit);
                if (a.gate != nullptr && lane == 0) Elem<T>::store(a.gate + (int64_t)region * a.S2 + s, logit);
                if (s == 0 || logit > best) {      // strict >: lowest index wins a tie
                    best = logit;
                    best_s = s;
                }
            }
        best_s = __builtin_amdgcn_readfirstlane(best_s);
        const int ps_n = __builtin_amdgcn_readlane(rsplit, best_s);
        nq = ps_n == 4 ? 16 : ps_n == 2 ? 4 : 1;
        chain_publish(a.status + 1, region, nq);
        if (lane == 0) {
            a.indices[region] = best_s;
            if (a.next_counts != nullptr) a.next_counts[region] = (uint8_t)(ps_n * ps_n);
            s_split = ps_n;
        }
    }

    // ---- the sample's extra tokens, by the waves in turn (the last first: wave 0 has the router, and every workgroup behind this
    // one waits for the count it publishes: not before that; a forward of 1 picture, 384 channels, 478 -> 472 us, of 99, 768
    // channels, 4221 -> 4160)
    if (rr == 0)
        for (int e = 3 - wv; e < extra; e += 4) {
            u32x4 row[NV];
#pragma unroll
            for (int it = 0; it < NV; it++) {
                row[it] = z;
                if (act[it]) {
                    const int64_t at = (row_b + e) * (int64_t)C + (it * WAVE + lane) * VEC;
                    const int64_t oe = ((int64_t)b * N + e) * C + (it * WAVE + lane) * VEC;
                    float d[VEC], sv[VEC], r[VEC];
                    Elem<T>::unpack(*reinterpret_cast<const u32x4 *>(a.in + at), d);
                    Elem<T>::unpack(*reinterpret_cast<const u32x4 *>(a.sub + at), sv);
#pragma unroll
                    for (int c = 0; c < VEC; c++) d[c] -= sv[c];
                    Elem<T>::unpack(Elem<T>::pack(d), d);
                    Elem<T>::unpack(*reinterpret_cast<const u32x4 *>(a.ref + oe), r);
#pragma unroll
                    for (int c = 0; c < VEC; c++) r[c] += d[c];
                    row[it] = Elem<T>::pack(r);
                    *reinterpret_cast<u32x4 *>(a.out + oe) = row[it];
                }
            }
            const int64_t at = (int64_t)b * N + e;
            if constexpr (REC) record_row<T>(row[0], act[0], a.eps, C, a.records + at * 2);
            else if (normed) norm_row<T, NV, NARROW>(row, act, lw, lb, a.eps, C, a.out_ln + at * C + lane * VEC);
        }

    // ---- what LayerNorm wants of this wave's tokens
    u32x4 y4[4][NV];                                               // their LayerNorm, which rows of one token take over
    const int64_t row0 = (int64_t)b * N + extra + (int64_t)(ry * 4 + wv) * a.W + rx * 4;
    if constexpr (REC) {
        float pivot[4], st[8];
#pragma unroll
        for (int t = 0; t < 4; t++) lane_sums<T>(tok[t][0], act[0], pivot[t], st[2 * t], st[2 * t + 1]);
        write_records4(st, pivot[0], pivot[1], pivot[2], pivot[3], C, a.eps, a.records + row0 * 2);
    } else if (normed) {
        norm_rows4<T, NV, NARROW>(tok, act, lw, lb, a.eps, C, a.out_ln + row0 * C + lane * VEC, y4);
    }

    // ---- the region's place among the next block's queries
    if (wv == 0) {
        const long long before = chain_rows_before(a.status, region, nq, a.capacity, a.next_offsets + a.B);
        if (lane == 0) s_before = before;
    }
    lds_barrier();
    const int ps_n = __builtin_amdgcn_readfirstlane(s_split);
    nq = ps_n == 4 ? 16 : ps_n == 2 ? 4 : 1;
    const int64_t n0 = s_before + (int64_t)extra * (b + 1);        // first packed row of the region
    if (wv == 3) {                                                 // descriptors, offsets
        if (a.next_region_rows != nullptr && lane == 0) a.next_region_rows[region] = (int32_t)n0;
        if (lane < nq && n0 + lane < a.capacity) {
            const int step = 4 / ps_n, dy = lane / ps_n, dx = lane - dy * ps_n;
            int64_t *p = a.patches + 4 * (n0 + lane);
            p[0] = b; p[1] = ry * 4 + dy * step; p[2] = rx * 4 + dx * step; p[3] = step;
        }
        if (rr == 0) {
            if (lane == 0) a.next_offsets[b] = n0 - extra;
            if (lane < extra && n0 - extra + lane < a.capacity) {
                int64_t *p = a.patches + 4 * (n0 - extra + lane);
                p[0] = b; p[1] = -(int64_t)lane - 1; p[2] = 0; p[3] = 1;
            }
        }
        if (region == a.B * nreg - 1 && lane == 0) chain_total(a.status, a.next_offsets + a.B, n0 + nq, a.capacity);
    }
    if (n0 + nq > a.capacity) return;                              // never outside the buffers

    // ---- the queries themselves: 16, four a wave; 4, one a wave; or the mean that the router has taken
    auto store = [&](T *to, const u32x4 (&row)[NV], int64_t r) {
#pragma unroll
        for (int it = 0; it < NV; it++)
            if (act[it]) *reinterpret_cast<u32x4 *>(to + r * C + (it * WAVE + lane) * VEC) = row[it];
    };
    auto put = [&](const u32x4 (&row)[NV], int64_t r) {
        store(a.comp, row, r);
        if (normed) norm_row<T, NV, NARROW>(row, act, lw, lb, a.eps, C, a.comp_ln + r * C + lane * VEC);
    };
    if (ps_n == 4) {
        float pivot[4], st[8];
#pragma unroll
        for (int t = 0; t < 4; t++) {
#pragma unroll
            for (int it = 0; it < NV; it++) {
                float acc[VEC];
#pragma unroll
                for (int c = 0; c < VEC; c++) acc[c] = 0.f;
                add_vector<T>(acc, tok[t][it]);                    // 0 + x: the mean of a window of one
                tok[t][it] = Elem<T>::pack(acc);
            }
            store(a.comp, tok[t], n0 + 4 * wv + t);
            if (normed) store(a.comp_ln, y4[t], n0 + 4 * wv + t);
            if constexpr (REC) lane_sums<T>(tok[t][0], act[0], pivot[t], st[2 * t], st[2 * t + 1]);
        }
        if constexpr (REC)
            write_records4(st, pivot[0], pivot[1], pivot[2], pivot[3], C, a.eps, a.comp_records + (n0 + 4 * wv) * 2);
    } else if (ps_n == 2) {
        const int t0 = (wv / 2) * 8 + (wv % 2) * 2;
        u32x4 row[NV];
#pragma unroll
        for (int it = 0; it < NV; it++) {
            float acc[VEC];
#pragma unroll
            for (int c = 0; c < VEC; c++) acc[c] = 0.f;
            row[it] = z;
            if (act[it]) {
                const int v = it * WAVE + lane;
                add_vector<T>(acc, held[t0 * nvec + v]);
                add_vector<T>(acc, held[(t0 + 1) * nvec + v]);
                add_vector<T>(acc, held[(t0 + 4) * nvec + v]);
                add_vector<T>(acc, held[(t0 + 5) * nvec + v]);
#pragma unroll
                for (int c = 0; c < VEC; c++) acc[c] *= 0.25f;
                row[it] = Elem<T>::pack(acc);
            }
        }
        put(row, n0 + wv);
        if constexpr (REC) {
            float pivot, st[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            lane_sums<T>(row[0], act[0], pivot, st[0], st[1]);
            write_records4(st, pivot, 0.f, 0.f, 0.f, C, a.eps, a.comp_records + (n0 + wv) * 2, 1);
        }
    } else if (wv == 0) {
        put(pooled, n0);
        if constexpr (REC) record_row<T>(pooled[0], act[0], a.eps, C, a.comp_records + n0 * 2);
    }
    if (rr == 0)               // the extra tokens again, by the lanes that stored them
        for (int e = 3 - wv; e < extra; e += 4) {
            u32x4 row[NV];
#pragma unroll
            for (int it = 0; it < NV; it++) {
                row[it] = z;
                if (act[it]) row[it] = *reinterpret_cast<const u32x4 *>(a.out + ((int64_t)b * N + e) * C + (it * WAVE + lane) * VEC);
            }
            put(row, n0 - extra + e);
            if constexpr (REC) record_row<T>(row[0], act[0], a.eps, C, a.comp_records + (n0 - extra + e) * 2);
        }
}

}  // namespace vtdge

using namespace vtdge;

extern "C" int vtdge_region_step_fits(int B, int H, int W, int C, int extra, int dtype)
{
    if (B <= 0 || H <= 0 || W <= 0 || C <= 0 || extra < 0 || extra > WAVE || H % 4 || W % 4) return 0;
    if (dtype != VTDGE_F32 && dtype != VTDGE_BF16) return 0;
    const int vec = dtype == VTDGE_BF16 ? 8 : 4, nvec = C / vec;
    const int64_t regions = (int64_t)B * (H / 4) * (W / 4);
    if (C % vec != 0 || nvec > 192) return 0;
    // Up to where a wave for every four tokens is faster than one for sixteen that repeats nothing (the router's sums are
    // made from LDS again).  A forward, us, without it / with it (channels, regions): bf16 384: 256: 816 / 728, 512: 944 / 882,
    // 1024: 1348 / 1304, 2048: 1872 / 1853, 2560: 2126 / 2073, 3200: 2486 / 2436, 3904: 2871 / 2853 (of 512 px 3254 / 3263), 4096:
    // 2972 / 2968 (3394 / 3395), 4224: 3206 / 3090, 5120: 3738 / 3638, 6144: 4393 / 4327, 8192: 5739 / 5708, 10240: 7188 / 7059; 768: 512: 2204 / 2090, 1408: 3965 / 3847, 3072: 7152 / 7113, 5120: 10542 / 10259; 192: 16: 541 / 437, 512: 997 / 847, 1536: 1311 / 1202,
    // 4096: 1778 / 1758, 8192: 3177 / 3135, 11200: 4287 / 4176, 14400: 5535 / 5626; fp32 192: 512: 1302 / 1196, 2080: 3200 / 3034,
    // 6400: 7892 / 7338, 12800: 15009 / 14762; 384: 528: 2418 / 2395, 1280: 4901 / 4749, 2240: 7373 / 7166, 3200: 10060 / 9847, 4096:
    // 12813 / 12864; 768: 384: 5296 / 5280, 768: 8269 / 8182, 1280: 12039 / 11820; pyramids with 320 channels in their third stage,
    // bf16 1600: 2507 / 2471, 2240: 3029 / 2996, 4096: 4597 / 4549, 9600: 9847 / 9805; fp32 864: 4626 / 4547, 1440: 6677 / 6562.  Rows of up to 16 vectors, whose other
    // kernels give several regions to a wave, lose sooner: pyramids of 64 to 512 channels by pictures of 256 px, bf16 2: 582 / 549,
    // 14: 1419 / 1425, 20: 1479 / 1503; fp32 with 2304 regions of 64 and 576 of 128 channels 1049 / 1043, 3072 and 768: 1125 / 1126.
    const int most = dtype == VTDGE_BF16 ? (nvec <= 16 ? 3072 : nvec <= 32 ? 11200 : nvec <= WAVE ? 10240 : 5120)
                                         : (nvec <= 32 ? 2048 : nvec <= WAVE ? 12800 : nvec <= 128 ? 3200 : 1280);
    return regions <= most ? 1 : 0;
}

extern "C" int64_t vtdge_region_step_workspace(int B, int H, int W)
{
    return B > 0 && H > 0 && W > 0 ? 8 * (1 + (int64_t)B * (H / 4) * (W / 4)) : 0;
}

extern "C" int vtdge_region_step(const void *in, const void *sub, const int64_t *cur_indices, const int64_t *splits,
                                 const int64_t *offsets, const int32_t *region_rows, const uint8_t *cur_counts, const void *ref,
                                 void *out, const void *next_weight, const void *next_bias, void *next_gate,
                                 int64_t *next_indices, const int64_t *next_splits, uint8_t *next_counts, void *out_records,
                                 void *out_ln, const void *ln_weight, const void *ln_bias, float eps, void *next_comp,
                                 void *next_comp_records, void *next_comp_ln, int64_t *next_patches, int64_t capacity_rows,
                                 int64_t *next_offsets, int32_t *next_region_rows, void *workspace, int64_t workspace_bytes,
                                 int B, int H, int W, int C, int extra, int S, int S2, int dtype, void *stream)
{
    VT_REQUIRE(in && sub && cur_indices && splits && offsets && ref && out && next_weight && next_bias && next_indices &&
                   next_splits && next_comp && next_patches && next_offsets && workspace,
               VTDGE_ERR_ARG, "region_step: NULL operand");
    VT_REQUIRE((region_rows == nullptr) == (cur_counts == nullptr), VTDGE_ERR_ARG,
               "region_step: the regions' first rows and their query counts come together");
    VT_REQUIRE((out_records == nullptr) == (next_comp_records == nullptr) && (out_ln == nullptr) == (next_comp_ln == nullptr) &&
                   (out_ln == nullptr || (ln_weight && ln_bias && out_records == nullptr)),
               VTDGE_ERR_ARG, "region_step: records or LayerNorms, of tokens and rows together");
    VT_REQUIRE(vtdge_region_step_fits(B, H, W, C, extra, dtype) && S >= 1 && S <= VTDGE_MAX_SPLITS && S2 >= 1 &&
                   S2 <= VTDGE_MAX_SPLITS,
               VTDGE_ERR_UNSUPPORTED, "region_step: no kernel for %d samples of a %dx%d grid of %d channels (dtype %d)", B, H, W, C,
               dtype);
    VT_REQUIRE(out_records == nullptr || (dtype == VTDGE_BF16 && C > 256 && C <= 512), VTDGE_ERR_UNSUPPORTED,
               "region_step: statistics records are written for bf16 rows of 264 to 512 channels (C=%d)", C);
    VT_REQUIRE(capacity_rows >= (int64_t)B * (extra + (int64_t)H * W) && workspace_bytes >= vtdge_region_step_workspace(B, H, W),
               VTDGE_ERR_ARG, "region_step: buffers too small");
    VT_REQUIRE((((uintptr_t)in | (uintptr_t)sub | (uintptr_t)ref | (uintptr_t)out | (uintptr_t)next_weight | (uintptr_t)out_records |
                 (uintptr_t)out_ln | (uintptr_t)ln_weight | (uintptr_t)ln_bias | (uintptr_t)next_comp |
                 (uintptr_t)next_comp_records | (uintptr_t)next_comp_ln) & 15) == 0,
               VTDGE_ERR_ARG, "region_step: operands must be 16-byte aligned");
    const unsigned grid = (unsigned)(B * (H / 4) * (W / 4));
    const int vec = dtype == VTDGE_BF16 ? 8 : 4, nv = (C / vec + WAVE - 1) / WAVE;
    const bool narrow = C / vec <= 32;
    const size_t lds = (size_t)16 * (C / vec) * 16;
#define VT_GO(T, NV, REC, NARROW)                                                                                              \
    do {                                                                                                                    \
        const RegionStep<T> a{(const T *)in, (const T *)sub, (const T *)ref, cur_indices, splits, offsets, region_rows,     \
                              cur_counts, (T *)out, (const T *)next_weight, (const T *)next_bias, (T *)next_gate,           \
                              next_indices, next_splits, next_counts, (u32x4 *)out_records, (T *)out_ln,                    \
                              (const T *)ln_weight, (const T *)ln_bias, eps, (T *)next_comp, (u32x4 *)next_comp_records,    \
                              (T *)next_comp_ln, next_patches, capacity_rows, next_offsets, next_region_rows,               \
                              (unsigned long long *)workspace, B, H, W, C, extra, S, S2};                                   \
        note_kernel(reinterpret_cast<const void *>(region_step_kernel<T, NV, REC, NARROW>));                                        \
        region_step_kernel<T, NV, REC, NARROW><<<grid, 256, lds, (hipStream_t)stream>>>(a);                                         \
        return check_launch("region_step");                                                                                 \
    } while (0)
    if (dtype == VTDGE_F32) {
        if (narrow) VT_GO(float, 1, false, true);
        if (nv == 1) VT_GO(float, 1, false, false);
        if (nv == 2) VT_GO(float, 2, false, false);
        VT_GO(float, 3, false, false);
    }
    if (out_records != nullptr) VT_GO(bf16_t, 1, true, false);
    if (narrow) VT_GO(bf16_t, 1, false, true);
    if (nv == 1) VT_GO(bf16_t, 1, false, false);
    if (nv == 2) VT_GO(bf16_t, 2, false, false);
    VT_GO(bf16_t, 3, false, false);
#undef VT_GO
}
