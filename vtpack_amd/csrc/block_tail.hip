// What a block does with its packed queries behind attention, as one kernel (bf16, gfx950):
//   q1 = o Wp^T + bp + comp,   out = q1 + gelu(LayerNorm(q1) W1^T + b1) W2^T + b2.
//
// For narrow models the four launches this stands in for (projection, LayerNorm, fc1, fc2) are bound by HBM: the hidden rows,
// 4 to 8 times as wide as the tokens, are written and read back, 470 MB each way at 459 000 rows of 64 channels.  Here a
// wave takes 32 rows through all of it in registers, and only o and comp come in and out leaves.
//
// Every product is formed transposed, D = W_block * rows^T with v_mfma_f32_32x32x16_bf16: a lane holds one row (column of
// D), 16 of the block's 32 output channels.  The rows of the weights are dealt to the MFMA's rows with their middle groups
// of four swapped (within 16: 0-3, 8-11, 4-7, 12-15), so that those 16 are two runs of 8 consecutive channels - which is
// the operand layout of the next product, whose contraction runs over these channels.  So nothing moves between lanes from
// the projection to the result but two sums of the LayerNorm; residuals and biases are what the accumulators start from.
//
// The weights go through LDS in stages that all waves share, two buffers, by direct loads: first Wp, then per 64 hidden
// channels the 64 rows of W1 and the 64 columns of W2.  128-byte row pieces, their 16-byte chunks XOR-ed by the row against
// bank conflicts.
//
// What bounds it: the GELU (11 vector instructions a hidden value: 69 us of the 103 below, 35 of 87, 10 of 35), the LDS reads
// of the weights' fragments (one a matrix instruction, which is all LDS delivers) and a tile's first loads, in turns.  Three
// waves a SIMD at 64 channels and two at 128 overlap them in part; at 192 a workgroup takes 101 KB of LDS and more, so there is
// one wave a SIMD.  Measured against the launches it stands in for (rows, C, hidden):
//   459000,  64,  512: 103 against 393 us     7000: 13.5 against 27     1800: 13.5 against 16     200: 13.5 against 12
//   115000, 128, 1024:  87 against 190        7000: 29.5 against 40     1800: 29.5 against 23
//    29000, 192,  768:  35 against  69       14000: 33 against 45       3600: 32 against 34        800: 32 against 17
// Tried: 64 rows a wave (half the LDS reads): 116, 144 (spills); four waves a SIMD at 64 channels: 123; eight waves on one
// buffer pair: 87 at 128 channels, 45 at 192; the parameters by a load each instead of the table: 118, 92, 47.
#include "common.h"

namespace vtdge {

struct TailArgs {
    const bf16_t *o, *comp, *wp, *bp, *lnw, *lnb, *w1, *b1, *w2, *b2;
    bf16_t *out;
    const int64_t *rows_dev;
    int64_t rows;
    float eps;
    int hidden;
};

// the weight row that goes to MFMA row r (an involution)
__device__ __forceinline__ int dealt_row(int r) { return (r & ~12) | ((r & 4) << 1) | ((r & 8) >> 1); }

template <int C> struct Tail {
    static constexpr int T = C / 16;                       // K steps over the channels = 8-channel runs of a lane
    static constexpr int SLABS = C / 64;                   // 128-byte pieces of a row
    static constexpr int STAGE = 2 * C * 128;              // bytes: 64 rows x SLABS of W1 and C rows x 1 of W2
    static constexpr int UNITS = STAGE / 1024;             // direct loads a stage
    static constexpr int PROJ = (SLABS + 1) / 2;           // stages of Wp, two slabs of C rows each
};

template <int C, int NW, int WPE> __global__ __launch_bounds__(NW * 64, WPE) void block_tail_kernel(TailArgs a)
{
    using G = Tail<C>;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int64_t M = live_rows(a.rows_dev, a.rows);
    const int64_t first = (int64_t)blockIdx.x * (NW * 32);
    if (first >= M) return;
    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 31, lg = lane >> 5;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int stages = G::PROJ + a.hidden / 64;
    float *const table = reinterpret_cast<float *>(smem + 2 * G::STAGE);      // bp, lnw, lnb, b2, b1 as floats
    const uint32_t lds0 = (uint32_t)(uintptr_t)smem;

    // direct loads of a stage: unit u is 8 rows of 128 bytes, of Wp or of W1 and W2
    auto unit = [&](const bf16_t *base, int r, int pitch, int st, int u) {
        dma16(uniform_ptr(base), (uint32_t)dealt_row(r) * (uint32_t)pitch + (uint32_t)(((lane & 7) ^ (r >> 1)) & 7) * 16u,
              lds0 + (uint32_t)((st & 1) * G::STAGE + u * 1024));
    };
    auto load_proj = [&](int st) {
#pragma unroll
        for (int i = 0; i < G::UNITS / NW; i++) {
            const int u = i * NW + wid, slab = st * 2 + u / (C / 8);
            if (slab < G::SLABS) unit(a.wp + slab * 64, (u % (C / 8)) * 8 + (lane >> 3), C * 2, st, u);
        }
    };
    auto load_hidden = [&](int st) {
        const int h = st - G::PROJ;
#pragma unroll
        for (int i = 0; i < G::UNITS / NW; i++) {
            const int u = i * NW + wid;
            if (i * NW < 8 * G::SLABS) unit(a.w1 + (int64_t)h * 64 * C + (u / 8) * 64, (u % 8) * 8 + (lane >> 3), C * 2, st, u);
            else unit(a.w2 + h * 64, (u - 8 * G::SLABS) * 8 + (lane >> 3), a.hidden * 2, st, u);
        }
    };
    static_assert(G::UNITS % NW == 0 && (8 * G::SLABS) % NW == 0, "units are dealt out evenly");
    load_proj(0);

    const bool wave_live = first + wid * 32 < M;
    const int64_t row = first + wid * 32 + lr, at = (row < M ? row : M - 1) * C + 8 * lg;
    u32x4 x[G::T];                                         // o, then LayerNorm(q1), as the products take them
    f32x16 acc[C / 32];
#pragma unroll
    for (int t = 0; t < G::T; t++) x[t] = *reinterpret_cast<const u32x4 *>(a.o + at + 16 * t);
    // all parameters that are vectors go to LDS in one round trip
    for (int i = tid; i < (4 * C + a.hidden) / 8; i += NW * 64) {
        const int which = i / (C / 8), at8 = which < 4 ? i % (C / 8) : i - C / 2;
        const bf16_t *p = which == 0 ? a.bp : which == 1 ? a.lnw : which == 2 ? a.lnb : which == 3 ? a.b2 : a.b1;
        float f[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (p != nullptr) Elem<bf16_t>::unpack(*reinterpret_cast<const u32x4 *>(p + 8 * at8), f);
        *reinterpret_cast<f32x4 *>(table + 8 * i) = f32x4{f[0], f[1], f[2], f[3]};
        *reinterpret_cast<f32x4 *>(table + 8 * i + 4) = f32x4{f[4], f[5], f[6], f[7]};
    }
    const float *const lane_table = table + 8 * lg;
    // value e of vector `which` at this lane's channels 16 t + 8 lg ..
    auto param = [&](int which, int t, int e) { return lane_table[which * C + 16 * t + e]; };
    const int sw = (lr >> 1) & 7;
    int cs[4];
#pragma unroll
    for (int s = 0; s < 4; s++) cs[s] = lr * 128 + ((2 * s + lg) ^ sw) * 16;

#pragma unroll
    for (int t = 0; t < G::T; t++) {
        float r[8];
        Elem<bf16_t>::unpack(*reinterpret_cast<const u32x4 *>(a.comp + at + 16 * t), r);
#pragma unroll
        for (int e = 0; e < 8; e++) acc[t / 2][8 * (t & 1) + e] = r[e];
    }
    // ---- projection
#pragma unroll
    for (int st = 0; st < G::PROJ; st++) {
        wait_vmcnt<0>();
        lds_barrier();                                     // (the first one also publishes the table)
        if (st + 1 < G::PROJ) load_proj(st + 1);
        else load_hidden(st + 1);
        if (!wave_live) continue;
        const unsigned char *S = smem + (st & 1) * G::STAGE;
#pragma unroll
        for (int sl = 0; sl < 2; sl++) {
            if (2 * st + sl >= G::SLABS) break;
#pragma unroll
            for (int s = 0; s < 4; s++)
#pragma unroll
                for (int cb = 0; cb < C / 32; cb++)
                    Slab<bf16_t>::mma(*reinterpret_cast<const u32x4 *>(S + (sl * C + cb * 32) * 128 + cs[s]),
                                      x[(2 * st + sl) * 4 + s], acc[cb]);
        }
    }
    // ---- q1 as stored, its LayerNorm, and what fc2's accumulators start from
    {
        float sum = 0.f;
#pragma unroll
        for (int t = 0; t < G::T; t++) {
            float f[8];
#pragma unroll
            for (int e = 0; e < 8; e++) f[e] = acc[t / 2][8 * (t & 1) + e] + param(0, t, e);
            Elem<bf16_t>::unpack(Elem<bf16_t>::pack(f), f);
#pragma unroll
            for (int e = 0; e < 8; e++) {
                acc[t / 2][8 * (t & 1) + e] = f[e];
                sum += f[e];
            }
        }
        const float mean = (sum + __shfl_xor(sum, 32, WAVE)) / (float)C;
        float sq = 0.f;
#pragma unroll
        for (int cb = 0; cb < C / 32; cb++)
#pragma unroll
            for (int e = 0; e < 16; e++) {
                const float d = acc[cb][e] - mean;
                sq += d * d;
            }
        const float rstd = 1.0f / sqrtf((sq + __shfl_xor(sq, 32, WAVE)) / (float)C + a.eps);
#pragma unroll
        for (int t = 0; t < G::T; t++) {
            float f[8];
#pragma unroll
            for (int e = 0; e < 8; e++)
                f[e] = (acc[t / 2][8 * (t & 1) + e] - mean) * rstd * param(1, t, e) + param(2, t, e);
            x[t] = Elem<bf16_t>::pack(f);
#pragma unroll
            for (int e = 0; e < 8; e++) acc[t / 2][8 * (t & 1) + e] += param(3, t, e);
        }
    }
    // ---- 64 hidden channels a stage
    for (int st = G::PROJ; st < stages; st++) {
        wait_vmcnt<0>();
        block_barrier();                                   // stage st is whole; the buffer of st - 1 is free
        if (st + 1 < stages) load_hidden(st + 1);
        if (!wave_live) continue;
        const unsigned char *S1 = smem + (st & 1) * G::STAGE, *S2 = S1 + G::SLABS * 64 * 128;
        const float *b1 = lane_table + 4 * C + (st - G::PROJ) * 64;
        // two blocks of 32 hidden channels: the GELU of the first under the first product of the second, that of the second
        // under the second product of the first
        f32x16 d[2];
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const f32x4 z = *reinterpret_cast<const f32x4 *>(b1 + 32 * j + 16 * (v >> 1) + 4 * (v & 1));
#pragma unroll
                for (int e = 0; e < 4; e++) d[j][4 * v + e] = z[e];
            }
        // 4 T matrix instructions, each with its share of the vector work and the LDS read of the one two steps on
        uint32_t hb[2][8];
        auto fragment = [&](int k) {                       // what step k multiplies by
            const int j = (k / G::T) & 1, t = k % G::T;
            return *reinterpret_cast<const u32x4 *>(k < 2 * G::T ? S1 + ((t >> 2) * 64 + j * 32) * 128 + cs[t & 3]
                                                                 : S2 + (t / 2) * 32 * 128 + cs[2 * j + (t & 1)]);
        };
        u32x4 w[3];
        w[0] = fragment(0);
        w[1] = fragment(1);
        static_for<4 * G::T>([&](auto kc) {
            constexpr int k = decltype(kc)::value, j = (k / G::T) & 1, t = k % G::T;
            if constexpr (k + 2 < 4 * G::T) w[(k + 2) % 3] = fragment(k + 2);
            if constexpr (k < 2 * G::T) Slab<bf16_t>::mma(w[k % 3], x[t], d[j]);
            else {
                constexpr int e = 4 * (t & 1);
                Slab<bf16_t>::mma(w[k % 3], u32x4{hb[j][e], hb[j][e + 1], hb[j][e + 2], hb[j][e + 3]}, acc[t / 2]);
            }
            if constexpr (k >= G::T && k < 3 * G::T) {
                constexpr int u = k / G::T - 1;            // the block whose GELU goes here
#pragma unroll
                for (int e = t * 8 / G::T; e < (t + 1) * 8 / G::T; e++)
                    hb[u][e] = pack_bf16x2(gelu_fn<bf16_t>(d[u][2 * e]), gelu_fn<bf16_t>(d[u][2 * e + 1]));
            }
            __builtin_amdgcn_sched_barrier(0);
        });
    }
    if (row >= M) return;
#pragma unroll
    for (int t = 0; t < G::T; t++) {
        float f[8];
#pragma unroll
        for (int e = 0; e < 8; e++) f[e] = acc[t / 2][8 * (t & 1) + e];
        *reinterpret_cast<u32x4 *>(a.out + at + 16 * t) = Elem<bf16_t>::pack(f);
    }
}

template <int C, int NW, int WPE> static int go(const TailArgs &a, hipStream_t st)
{
    const size_t lds = 2 * Tail<C>::STAGE + (size_t)(4 * C + a.hidden) * 4;
    auto kern = block_tail_kernel<C, NW, WPE>;
    VT_RESERVE_LDS(kern, 160 * 1024, "block_tail");
    const int64_t grid = ceil_div(a.rows, NW * 32);
    VT_REQUIRE(grid < (1ll << 31), VTDGE_ERR_UNSUPPORTED, "block_tail: %lld rows exceed one launch", (long long)a.rows);
    note_kernel(reinterpret_cast<const void *>(kern));
    kern<<<dim3((unsigned)grid), dim3(NW * 64), lds, st>>>(a);
    return check_launch("block_tail");
}

}  // namespace vtdge

using namespace vtdge;

extern "C" int vtdge_block_tail_fits(int64_t rows, int C, int hidden, int dtype)
{
    return dtype == VTDGE_BF16 && (C == 64 || C == 128 || C == 192) && hidden > 0 && hidden % 64 == 0 && hidden <= 4096 &&
           rows >= 0 && ceil_div(rows, 128) < (1ll << 31);
}

// Few rows are left to the kernels that deal a product to more compute units: the live rows are about 0.44 of `rows`, and
// at those the two are even near 500 (64 channels) and 3500 (128, 192; figures above).
extern "C" int vtdge_block_tail_wanted(int64_t rows, int C, int hidden, int dtype)
{
    return vtdge_block_tail_fits(rows, C, hidden, dtype) && rows >= (C == 64 ? 1024 : 8192);
}

extern "C" int vtdge_block_tail(const void *o, const void *comp, const void *proj_weight, const void *proj_bias,
                                const void *ln_weight, const void *ln_bias, float ln_eps, const void *fc1_weight,
                                const void *fc1_bias, const void *fc2_weight, const void *fc2_bias, void *out,
                                const int64_t *rows_dev, int64_t rows, int C, int hidden, int dtype, void *stream)
{
    VT_REQUIRE(o && comp && proj_weight && ln_weight && ln_bias && fc1_weight && fc2_weight && out, VTDGE_ERR_ARG,
               "block_tail: NULL operand");
    VT_REQUIRE(vtdge_block_tail_fits(rows, C, hidden, dtype), VTDGE_ERR_UNSUPPORTED,
               "block_tail: built for bf16, 64, 128 or 192 channels and a multiple of 64 hidden ones, at most 4096 (rows=%lld "
               "C=%d hidden=%d dtype=%d)", (long long)rows, C, hidden, dtype);
    VT_REQUIRE((((uintptr_t)o | (uintptr_t)comp | (uintptr_t)proj_weight | (uintptr_t)proj_bias | (uintptr_t)ln_weight |
                 (uintptr_t)ln_bias | (uintptr_t)fc1_weight | (uintptr_t)fc1_bias | (uintptr_t)fc2_weight | (uintptr_t)fc2_bias |
                 (uintptr_t)out) &
                15) == 0,
               VTDGE_ERR_ARG, "block_tail: operands must be 16-byte aligned");
    if (rows == 0) return VTDGE_OK;
    const TailArgs a{(const bf16_t *)o, (const bf16_t *)comp, (const bf16_t *)proj_weight, (const bf16_t *)proj_bias,
                     (const bf16_t *)ln_weight, (const bf16_t *)ln_bias, (const bf16_t *)fc1_weight, (const bf16_t *)fc1_bias,
                     (const bf16_t *)fc2_weight, (const bf16_t *)fc2_bias, (bf16_t *)out, rows_dev, rows, ln_eps, hidden};
    hipStream_t st = (hipStream_t)stream;
    // waves a SIMD the registers are held to: what LDS lets in at 64 and 128 channels; at 192, where that is one, two only
    // keeps the kernel within 256 registers
    if (C == 64) return go<64, 4, 3>(a, st);
    if (C == 128) return go<128, 4, 2>(a, st);
    return go<192, 4, 2>(a, st);
}
