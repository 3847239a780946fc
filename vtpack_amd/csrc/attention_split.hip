// Sparse attention, bf16 / head_dim 64, of few (sample, head) pairs (gfx950).
//
// What bounds it is latency: a workgroup per pair (attention_dma.hip) leaves most of the chip idle and walks its keys in one
// chain.  Here the waves of a workgroup split the keys: each brings blocks of 32 keys (K and V) into an LDS region of its own
// by direct loads, turns the scores of a 32-query tile into probabilities against its own maximum and multiplies them with V,
// without meeting the others; maxima, sums and outputs meet in LDS once a tile and are added up in the order of the waves.
//   * Up to 288 keys there is a wave for every block (257 keys: nine), which keeps its fragments of K and V in registers while
//     the workgroup takes a tile after another; a pair has as many workgroups as give every compute unit one.  A tile costs
//     1.1 us (2.2 with the parts read in a loop over a number of waves that the compiler does not know).
//   * Beyond, eight waves go through the blocks of one tile in turn, with a second region to load into.
// Consecutive workgroups share a pair and run on different XCDs: its keys and values are fetched up to eight times, but a
// number of pairs that is no multiple of eight fills the chip (1 sample, 6 heads, 1025 keys and queries: 8.6 against 14 us
// with the workgroups of a pair on one XCD).
#include "attention_tile.h"

namespace vtdge {

constexpr int SP_BLOCK = 2 * 32 * 128;      // bytes of a block: 32 rows of K, then 32 of V
constexpr int SP_RESIDENT = 9;              // blocks, and waves, of a sequence without a second region
constexpr int SP_WAVES = 8;                 // waves of a longer one

// NW = waves; LONG: more blocks than waves
template <int NW, bool LONG>
__global__ __launch_bounds__(NW * 64) void sparse_attention_bf16_d64_split_kernel(
    const bf16_t *__restrict__ q, int64_t q_rs, int64_t q_hs, const bf16_t *__restrict__ k, const bf16_t *__restrict__ v,
    int64_t kv_bs, int64_t kv_ts, int64_t kv_hs, const int64_t *__restrict__ offsets, bf16_t *__restrict__ out, int64_t o_rs,
    int64_t o_hs, int n, int groups, float scale, int items, int h)
{
    extern __shared__ __attribute__((aligned(128))) unsigned char smem[];
    const int item = blockIdx.x / groups;
    int qt = blockIdx.x - item * groups;                          // tiles qt, qt + groups, ... of the pair
    const int b = item / h, head = item - b * h;
    const int64_t row0 = offsets[b];
    const int Lb = (int)(offsets[b + 1] - row0);
    if (qt * 32 >= Lb) return;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int blocks = (n + 31) / 32;                             // NW of them at least: every wave has one
    const int lr = lane & 31, lg = lane >> 5;
    unsigned char *mine = smem + wid * 2 * SP_BLOCK;              // two regions a wave
    const uint32_t lds = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uintptr_t)mine);

    // block kb into region `reg`: load j covers rows 8 j .. 8 j + 7 of K (j < 4) or of V; rows past the last key repeat it.
    // 16-byte chunks are XOR-ed by the row as attention_tile.h reads them.
    const void *kbase = uniform_ptr(k + (int64_t)b * kv_bs + (int64_t)head * kv_hs);
    const void *vbase = uniform_ptr(v + (int64_t)b * kv_bs + (int64_t)head * kv_hs);
    const uint32_t row_bytes = (uint32_t)(kv_ts * 2);
    auto issue = [&](int kb, int reg) {
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int r = (j & 3) * 8 + (lane >> 3);
            const int chunk = (lane & 7) ^ (j < 4 ? (r >> 1) & 7 : 2 * (r & 3));
            const uint32_t off = (uint32_t)min(kb * 32 + r, n - 1) * row_bytes + chunk * 16;
            dma16(j < 4 ? kbase : vbase, off, lds + reg * SP_BLOCK + j * 1024);
        }
    };
    u32x4 qf[4];
    auto load_q = [&](int t) {
        const int qrow = t * 32 + lr;
        const unsigned char *qp =
            reinterpret_cast<const unsigned char *>(q + (row0 + qrow) * q_rs + (int64_t)head * q_hs) + lg * 16;
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const u32x4 z = {0u, 0u, 0u, 0u};
            qf[s] = qrow < Lb ? *reinterpret_cast<const u32x4 *>(qp + s * 32) : z;
        }
    };
    auto scale_q = [&]() {                     // scores come out of the matrix pipe in log2 units
#pragma unroll
        for (int s = 0; s < 4; s++) qf[s] = att_scale_frag(qf[s], scale * 1.44269504088896340736f);
    };
    const int sw = (lr >> 1) & 7;
    int cs[4];
#pragma unroll
    for (int s = 0; s < 4; s++) cs[s] = ((2 * s + lg) ^ sw) * 16;

    const f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    f32x16 o[2];
    float l, m;                                 // this lane's part of the row sum; the query's maximum so far
    u32x4 kf[4], vf[4];
    auto fetch = [&](int reg) {
        unsigned char *buf = mine + reg * SP_BLOCK;
        const AttnTile t = {buf + lr * 128, att_v_lane(buf + 32 * 128, lane), nullptr, n, lg};
#pragma unroll
        for (int sl = 0; sl < 4; sl++) kf[sl] = att_read_k(t, cs, 0, sl);
        att_read_v<false>(t, 0, vf);
    };
    auto block = [&](int kb, bool first) {      // block kb, whose fragments are in kf and vf
        f32x16 s = zero;
#pragma unroll
        for (int sl = 0; sl < 4; sl++) s = att_mfma(kf[sl], qf[sl], s);
        if (kb * 32 + 32 > n) {
            const int lim = n - kb * 32 - 4 * lg;
#pragma unroll
            for (int e = 0; e < 16; e++)
                if (8 * (e >> 2) + (e & 3) >= lim) s[e] = -INFINITY;
        }
        float mx = att_max16(s);
        mx = fmaxf(m, fmaxf(mx, __shfl_xor(mx, 32, WAVE)));
        // scores of -infinity only: their probabilities are zero against any reference
        const float ref = mx == -INFINITY ? 0.f : mx;
        if (!first) {
            const float alpha = __builtin_amdgcn_exp2f(m - ref);
            l *= alpha;
#pragma unroll
            for (int e = 0; e < 16; e++) {
                o[0][e] *= alpha;
                o[1][e] *= alpha;
            }
        }
        m = mx;
        u32x4 pf[2];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            uint32_t w[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                w[e] = pack_bf16x2(__builtin_amdgcn_exp2f(s[8 * i + 2 * e] - ref), __builtin_amdgcn_exp2f(s[8 * i + 2 * e + 1] - ref));
                l = bf16_pair_sum(w[e], l);     // the values the second product multiplies with
            }
            pf[i] = u32x4{w[0], w[1], w[2], w[3]};
        }
#pragma unroll
        for (int i = 0; i < 2; i++) {
            o[0] = att_mfma(vf[2 * i], pf[i], o[0]);
            o[1] = att_mfma(vf[2 * i + 1], pf[i], o[1]);
        }
    };
    // The parts of tile t meet: outputs as fp32 [query][channel] in the waves' regions `reg` (16-byte chunks XOR-ed by the
    // query), maxima and sums in a table behind the regions, one for each `reg`.
    auto meet = [&](int t, int reg) {
        float *mt = reinterpret_cast<float *>(smem + NW * 2 * SP_BLOCK) + reg * NW * 64, *lt = mt + NW * 32;
        l += __shfl_xor(l, 32, WAVE);
        if (lg == 0) {
            mt[wid * 32 + lr] = m;
            lt[wid * 32 + lr] = l;
        }
#pragma unroll
        for (int db = 0; db < 2; db++)
#pragma unroll
            for (int g4 = 0; g4 < 4; g4++) {
                const int chunk = db * 8 + 2 * g4 + lg;
                *reinterpret_cast<f32x4 *>(mine + reg * SP_BLOCK + lr * 256 + ((chunk ^ (lr & 15)) * 16)) =
                    f32x4{o[db][4 * g4], o[db][4 * g4 + 1], o[db][4 * g4 + 2], o[db][4 * g4 + 3]};
            }
        lds_barrier();
        for (int i = tid; i < 512; i += NW * 64) {            // four channels of a query
            const int row = i >> 4, chunk = i & 15;
            if (t * 32 + row >= Lb) break;                       // rows only grow with i
            float f[NW], top = -INFINITY, sum = 0.f;
            f32x4 part[NW], acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w = 0; w < NW; w++) {
                f[w] = mt[w * 32 + row];
                part[w] = *reinterpret_cast<const f32x4 *>(smem + (w * 2 + reg) * SP_BLOCK + row * 256 + ((chunk ^ (row & 15)) * 16));
            }
#pragma unroll
            for (int w = 0; w < NW; w++) top = fmaxf(top, f[w]);
#pragma unroll
            for (int w = 0; w < NW; w++) {
                f[w] = __builtin_amdgcn_exp2f(f[w] - top);
                sum += f[w] * lt[w * 32 + row];
                acc += f[w] * part[w];
            }
            const float inv = 1.0f / sum;
            u32x2 r;
            r.x = pack_bf16x2(acc[0] * inv, acc[1] * inv);
            r.y = pack_bf16x2(acc[2] * inv, acc[3] * inv);
            *reinterpret_cast<u32x2 *>(out + (row0 + t * 32 + row) * o_rs + (int64_t)head * o_hs + 4 * chunk) = r;
        }
    };

    issue(wid, 0);
    load_q(qt);
    if constexpr (LONG) {
        scale_q();
        o[0] = o[1] = zero;
        l = 0.f;
        m = -INFINITY;
        for (int kb = wid, reg = 0; kb < blocks; kb += NW, reg ^= 1) {
            if (kb + NW < blocks) {
                issue(kb + NW, reg ^ 1);
                wait_vmcnt<8>();                // the loads before these eight have landed
            } else {
                wait_vmcnt<0>();
            }
            asm volatile("" ::: "memory");
            fetch(reg);
            block(kb, kb == wid);
        }
        asm volatile("" ::: "memory");
        meet(qt, 0);
    } else {
        wait_vmcnt<0>();
        asm volatile("" ::: "memory");
        fetch(0);
        for (int reg = 1; qt * 32 < Lb; qt += groups, reg ^= 1) {
            scale_q();
            o[0] = o[1] = zero;
            l = 0.f;
            m = -INFINITY;
            block(wid, true);
            if ((qt + groups) * 32 < Lb) load_q(qt + groups);
            meet(qt, reg);
        }
    }
}

// Which calls the kernel is taken for: those whose workgroups are on the chip all at once, which makes it no slower than the
// kernels of attention_dma.hip with every query live (as a router that keeps the finest split leaves them).  Measured, us,
// those / this one (samples, heads, keys, live queries of a sample):
//   1, 6, 257, 128: 7.1 / 5.1           5, 12, 257, 90: 7.2 / 5.6      13, 6, 257, 118: 9.2 / 8.8    1, 2, 144, 2304: 33.8 / 11.0
//   14, 6, 257, 257: 11.5 / 9.9         85, 1, 145, 145: 6.8 / 6.5     85, 1, 65, 65: 4.7 / 4.1      1, 1, 256, 4096: 70.7 / 16.0
//   beyond the line: 21, 6, 257, 257: 11.9 / 13.6 (two tiles and more for each of 9 waves), 80, 1, 144, 576: 12.4 / 14.0
//   longer: 1, 6, 1025, 1025: 14.8 / 8.6      1, 12, 577, 577: 10.7 / 6.6      3, 3, 785, 785: 12.5 / 7.5
//   beyond the line: 1, 12, 1025, 1025: 15.3 / 15.5     4, 3, 785, 785: 12.7 / 12.6
bool attention_split_wanted(int64_t items, int n, int max_rows)
{
    const int64_t cus = compute_units(), qtiles = ceil_div(max_rows, 32);
    if (n > 32 * SP_RESIDENT) return items * qtiles <= cus;
    return 3 * items <= cus && qtiles <= 3 * (cus / items);
}

template <int NW, bool LONG>
static int go_attention_split(const void *q, int64_t q_rs, int64_t q_hs, const void *k, const void *v, int64_t kv_bs,
                              int64_t kv_ts, int64_t kv_hs, const int64_t *offsets, void *out, int64_t o_rs, int64_t o_hs,
                              int items, int h, int n, int groups, float scale, hipStream_t st)
{
    constexpr size_t lds = (size_t)NW * 2 * (SP_BLOCK + 256);
    auto kern = sparse_attention_bf16_d64_split_kernel<NW, LONG>;
    VT_RESERVE_LDS(kern, lds, "sparse_attention");
    note_kernel(reinterpret_cast<const void *>(kern));
    kern<<<dim3((unsigned)(items * groups)), dim3(NW * 64), lds, st>>>(
        (const bf16_t *)q, q_rs, q_hs, (const bf16_t *)k, (const bf16_t *)v, kv_bs, kv_ts, kv_hs, offsets, (bf16_t *)out,
        o_rs, o_hs, n, groups, scale, items, h);
    return check_launch("sparse_attention");
}

int launch_attention_split(const void *q, int64_t q_rs, int64_t q_hs, const void *k, const void *v, int64_t kv_bs,
                           int64_t kv_ts, int64_t kv_hs, const int64_t *offsets, void *out, int64_t o_rs, int64_t o_hs, int B,
                           int h, int n, int max_rows, float scale, hipStream_t st)
{
    const int qtiles = (int)ceil_div(max_rows, 32), items = B * h;
#define VT_SPLIT_GO(NW, LONG, groups)                                                                               \
    return go_attention_split<NW, LONG>(q, q_rs, q_hs, k, v, kv_bs, kv_ts, kv_hs, offsets, out, o_rs, o_hs, items, h, n,    \
                                        groups, scale, st)
    if (n > 32 * SP_RESIDENT) VT_SPLIT_GO(SP_WAVES, true, qtiles);
    // as many workgroups a pair as give every compute unit one
    int groups = compute_units() / items;
    groups = groups < qtiles ? groups : qtiles;
    switch ((int)ceil_div(n, 32)) {
    case 1: VT_SPLIT_GO(1, false, groups);
    case 2: VT_SPLIT_GO(2, false, groups);
    case 3: VT_SPLIT_GO(3, false, groups);
    case 4: VT_SPLIT_GO(4, false, groups);
    case 5: VT_SPLIT_GO(5, false, groups);
    case 6: VT_SPLIT_GO(6, false, groups);
    case 7: VT_SPLIT_GO(7, false, groups);
    case 8: VT_SPLIT_GO(8, false, groups);
    default: VT_SPLIT_GO(SP_RESIDENT, false, groups);
    }
#undef VT_SPLIT_GO
}

}  // namespace vtdge
