// LayerNorm inside the Linear over blocks of tokens (gfx950): norm1 in front of the spatial reduction of the key/value
// projection, out[(b, gy, gx), :] = sum over (dy, dx) of LayerNorm(token (gy P + dy, gx P + dx)) W[:, dy, dx, :]^T + bias.
// Separately the LayerNorm reads and writes every token and the product reads them again; here each token passes once,
// from memory through registers, where it is normalised and rounded as the LayerNorm kernel does it, into LDS.
//
// A workgroup of four waves makes 32 rows of the product, all C columns, two workgroups a compute unit whose phases fill each
// other (one of eight waves and 64 rows: 44.7 us where this took 41.4).  A step is TS tokens of each of its 32 blocks,
// K = 256: the tokens of the next step are normalised into the other of two LDS tiles while the matrix instructions read
// this one, those of the two steps after that are on their way to registers, and so are the next step's weights, fragments
// straight from L2, which the workgroups of an XCD share.  The weights of a step are asked for before the tokens of a
// later one: loads come back in order, and a fragment asked for behind a token would wait for memory.
// Bound by memory with whole chips of work, the tokens at 3.6 TB/s (a forward's other stream reads them at the same time),
// below by a step's chain of waits, 1.4 us.  Us, LayerNorm and Linear / this (rows, channels, P): 16384, 64, 8: 78.7 / 39.3;
// 16384, 128, 4: 44.4 / 27.6; 8192: 41.3 / 25.2 and 27.7 / 19.0; 6144: 35.4 / 24.1 and 25.8 / 18.2; 4096: 24.6 / 23.7 and 27.1 / 17.5;
// 2048: 25.4 / 23.3 and 16.3 / 17.4; 50176, 64, 4: 56.1 / 36.3; 25088, 128, 2: 24.5 / 18.6; 4096, 128, 8: 52.6 / 60.0.  PVT-Small at 256
// pictures, a pass: 4786 -> 4517 us.
#include "common.h"

namespace vtdge {

constexpr int LNP_ROWS = 32, LNP_K = 256, LNP_PITCH = LNP_K * 2 + 16;      // LDS row: the pad turns the banks a row further
constexpr int LNP_THREADS = 256;

// Weights [C, P P C] as the product reads them: fragment (step of 32 along K, 16 columns) after fragment, 64 vectors each, a
// weight a grid row.  In rows of a power of two of bytes a step's pieces all lie in the same two channels of an L2: 47 us
// whatever the batch, from 64 channels and P = 8 on.
constexpr int LNP_WEIGHTS = 16;
struct PatchWeights { const u32x4 *w[LNP_WEIGHTS]; };
__global__ __launch_bounds__(256) void patch_weight_pack_kernel(const PatchWeights weights, u32x4 *__restrict__ packed, int C, int K)
{
    const int i = blockIdx.x * 256 + threadIdx.x, lane = i & 63, tile = i / WAVE % (C / 16), k = i / WAVE / (C / 16);
    if (k < K / 32)
        packed[(int64_t)blockIdx.y * (C / 8) * K + i] = weights.w[blockIdx.y][(tile * 16 + (lane & 15)) * (K / 8) + k * 4 + (lane >> 4)];
}

template <int C>
__global__ __launch_bounds__(LNP_THREADS, 2) void layernorm_patch_linear_kernel(
    const bf16_t *__restrict__ x, const bf16_t *__restrict__ ln_w, const bf16_t *__restrict__ ln_b, float eps,
    const u32x4 *__restrict__ packed, const bf16_t *__restrict__ bias, const bf16_t *__restrict__ out_w,
    const bf16_t *__restrict__ out_b, float out_eps, bf16_t *__restrict__ out, int rows, int H, int W, int P)
{
    constexpr int TS = LNP_K / C;                                          // tokens of a block a step
    constexpr int GS = C / 8;                                              // lanes a token: a 16-byte vector each
    constexpr int RPW = WAVE / GS;                                         // tokens a wave reads with one load
    constexpr int LOADS = LNP_ROWS * TS / (4 * RPW);                       // of which it makes so many a step
    constexpr int NT = C / 64;                                             // tiles of 16 columns a wave
    constexpr int KS = LNP_K / 32;                                         // matrix instructions along K a step
    __shared__ __attribute__((aligned(16))) unsigned char tile[2][LNP_ROWS * LNP_PITCH];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row0 = blockIdx.x * LNP_ROWS;
    const int steps = P * P / TS;

    // where this lane's tokens lie: token `t` of a step in block `blk` of the workgroup (past the last row: the last)
    const int vec = lane % GS;
    const bf16_t *src[LOADS];
    int at[LOADS];
    const int gw = W / P, g2 = (H / P) * gw;
#pragma unroll
    for (int i = 0; i < LOADS; i++) {
        const int token = (i * 4 + wave) * RPW + lane / GS, blk = token / TS, t = token % TS;
        const int row = row0 + blk < rows ? row0 + blk : rows - 1;
        const int b = row / g2, r = row - b * g2, gy = r / gw, gx = r - gy * gw;
        src[i] = x + (((int64_t)b * H + gy * P) * W + gx * P + t) * C + vec * 8;
        at[i] = blk * LNP_PITCH + t * C * 2 + vec * 16;
    }
    // the first token of a step: P is a multiple of TS, a step stays in one row of its block
    auto load_tokens = [&](int step, u32x4 (&raw)[LOADS]) {
        const int first = step * TS, dy = first / P;
        const int64_t off = (int64_t)(dy * W + first - dy * P) * C;
#pragma unroll
        for (int i = 0; i < LOADS; i++) raw[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(src[i] + off));
    };
    // a wave's columns: 16 NT from 16 NT `wave` on
    const int fr = lane & 15, fk = lane >> 4;
    const u32x4 *wsrc = packed + wave * NT * WAVE + lane;
    auto load_weights = [&](int step, u32x4 (&wf)[KS][NT]) {
#pragma unroll
        for (int k = 0; k < KS; k++)
#pragma unroll
            for (int j = 0; j < NT; j++)
                wf[k][j] = wsrc[((step * KS + k) * (C / 16) + j) * WAVE];
    };
    float ww[8], bb[8];
    Elem<bf16_t>::unpack(*reinterpret_cast<const u32x4 *>(ln_w + vec * 8), ww);
    Elem<bf16_t>::unpack(*reinterpret_cast<const u32x4 *>(ln_b + vec * 8), bb);
    // A token's quotient and root are taken once a quad of lanes, each lane's of the load of its number: the same bits in a
    // fourth of the instructions.
    static_assert(LOADS == 4, "load i in lane i of a quad");
    auto each_load = [&](float (&v)[LOADS], auto &&f) {
        const float lo = lane & 1 ? v[1] : v[0], hi = lane & 1 ? v[3] : v[2];
        const float r = f(lane & 2 ? hi : lo);
        v[0] = dpp_move<0x00>(r);
        v[1] = dpp_move<0x55>(r);
        v[2] = dpp_move<0xAA>(r);
        v[3] = dpp_move<0xFF>(r);
    };
    auto normalise = [&](const u32x4 (&raw)[LOADS], unsigned char *to) {
        float f[LOADS][8], mean[LOADS], rstd[LOADS];
#pragma unroll
        for (int i = 0; i < LOADS; i++) {
            Elem<bf16_t>::unpack(raw[i], f[i]);
            mean[i] = 0.f;
#pragma unroll
            for (int c = 0; c < 8; c++) mean[i] += f[i][c];
        }
        group_sum_n<GS, LOADS>(mean);
        each_load(mean, [&](float s) { return s / (float)C; });
#pragma unroll
        for (int i = 0; i < LOADS; i++) {
            rstd[i] = 0.f;
#pragma unroll
            for (int c = 0; c < 8; c++) {
                f[i][c] -= mean[i];
                rstd[i] += f[i][c] * f[i][c];
            }
        }
        group_sum_n<GS, LOADS>(rstd);
        each_load(rstd, [&](float q) { return 1.0f / sqrtf(q / (float)C + eps); });
#pragma unroll
        for (int i = 0; i < LOADS; i++) {
#pragma unroll
            for (int c = 0; c < 8; c++) f[i][c] = f[i][c] * rstd[i] * ww[c] + bb[c];
            *reinterpret_cast<u32x4 *>(to + at[i]) = Elem<bf16_t>::pack(f[i]);
        }
    };
    f32x4 acc[2][NT];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < NT; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int frag = fr * LNP_PITCH + fk * 16;
    auto multiply = [&](const unsigned char *from, const u32x4 (&wf)[KS][NT]) {
#pragma unroll
        for (int k = 0; k < KS; k++)
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const bf16x8 a = __builtin_bit_cast(
                    bf16x8, *reinterpret_cast<const u32x4 *>(from + frag + i * 16 * LNP_PITCH + k * 64));
#pragma unroll
                for (int j = 0; j < NT; j++)        // the weights as first operand: a lane holds four columns of one row
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wf[k][j]), a, acc[i][j], 0, 0, 0);
            }
    };

    u32x4 raw_a[LOADS], raw_b[LOADS], wf_a[KS][NT], wf_b[KS][NT];
    load_tokens(0, raw_a);
    load_weights(0, wf_a);
    load_tokens(1, raw_b);
    normalise(raw_a, tile[0]);
    load_tokens(2 < steps ? 2 : 1, raw_a);
    lds_barrier();
    // `steps` is even.  Past the end nothing new is asked for: the last step's tokens and weights again.
    for (int s = 0; s < steps; s += 2) {
        load_weights(s + 1, wf_b);
        __builtin_amdgcn_sched_barrier(0);
        multiply(tile[0], wf_a);
        normalise(raw_b, tile[1]);
        load_tokens(s + 3 < steps ? s + 3 : steps - 1, raw_b);
        lds_barrier();
        load_weights(s + 2 < steps ? s + 2 : steps - 1, wf_a);
        __builtin_amdgcn_sched_barrier(0);
        multiply(tile[1], wf_b);
        if (s + 2 < steps) {
            normalise(raw_a, tile[0]);
            load_tokens(s + 4 < steps ? s + 4 : steps - 1, raw_a);
        }
        lds_barrier();
    }
    // the product's rows, rounded, through LDS: stored whole, or their LayerNorm instead
#pragma unroll
    for (int j = 0; j < NT; j++) {
        const int n = (wave * NT + j) * 16 + fk * 4;
        const u32x2 braw = *reinterpret_cast<const u32x2 *>(bias + n);
        const float b4[4] = {bf16lo(braw.x), bf16hi(braw.x), bf16lo(braw.y), bf16hi(braw.y)};
#pragma unroll
        for (int i = 0; i < 2; i++) {
            u32x2 r;
            r.x = pack_bf16x2(acc[i][j][0] + b4[0], acc[i][j][1] + b4[1]);
            r.y = pack_bf16x2(acc[i][j][2] + b4[2], acc[i][j][3] + b4[3]);
            *reinterpret_cast<u32x2 *>(tile[0] + (i * 16 + fr) * LNP_PITCH + n * 2) = r;
        }
    }
    lds_barrier();
#pragma unroll
    for (int i = 0; i < LNP_ROWS / (4 * RPW); i++) {
        const int blk = (i * 4 + wave) * RPW + lane / GS, row = row0 + blk;
        u32x4 r = *reinterpret_cast<const u32x4 *>(tile[0] + blk * LNP_PITCH + vec * 16);
        if (out_w != nullptr) {
            float f[8], w2[8], b2[8], s = 0.f, q = 0.f;
            Elem<bf16_t>::unpack(r, f);
            Elem<bf16_t>::unpack(*reinterpret_cast<const u32x4 *>(out_w + vec * 8), w2);
            Elem<bf16_t>::unpack(*reinterpret_cast<const u32x4 *>(out_b + vec * 8), b2);
#pragma unroll
            for (int c = 0; c < 8; c++) s += f[c];
            const float mean = group_sum<GS>(s) / (float)C;
#pragma unroll
            for (int c = 0; c < 8; c++) {
                f[c] -= mean;
                q += f[c] * f[c];
            }
            const float rstd = 1.0f / sqrtf(group_sum<GS>(q) / (float)C + out_eps);
#pragma unroll
            for (int c = 0; c < 8; c++) f[c] = f[c] * rstd * w2[c] + b2[c];
            r = Elem<bf16_t>::pack(f);
        }
        if (row < rows) *reinterpret_cast<u32x4 *>(out + (int64_t)row * C + vec * 8) = r;
    }
}

}  // namespace vtdge

using namespace vtdge;

extern "C" int vtdge_layernorm_patch_linear_fits(int B, int H, int W, int C, int P, int dtype)
{
    if (B <= 0 || H <= 0 || W <= 0 || P <= 0 || P > 32 || dtype != VTDGE_BF16 || (C != 64 && C != 128)) return 0;
    if (H % P != 0 || W % P != 0 || (int64_t)B * H * W >= (1ll << 31)) return 0;
    const int per_step = LNP_K / C;
    return P % per_step == 0 && (P * P / per_step) % 2 == 0 ? 1 : 0;
}

extern "C" int vtdge_layernorm_patch_linear_wanted(int B, int H, int W, int C, int P, int dtype)
{
    // from three eighths of a chip of workgroups on, with long sums from three fourths: the times above, and a forward of PVT-Small,
    // two kernels / this (pictures, 64 rows each): 32: 1642 / 1643, 40: 1779 / 1772, 48: 1866 / 1853, 56: 1966 / 1913, 64: 2076 / 2011,
    // 92: 2477 / 2349; 24: 1556 / 1570
    return vtdge_layernorm_patch_linear_fits(B, H, W, C, P, dtype) &&
                   (int64_t)B * (H / P) * (W / P) >= (P * P * C <= 4096 ? 96 : 192) * LNP_ROWS ? 1 : 0;
}

extern "C" int vtdge_layernorm_patch_pack(const void *const *weights_host, int count, void *packed, int C, int P, void *stream)
{
    VT_REQUIRE(weights_host && packed && count > 0, VTDGE_ERR_ARG, "layernorm_patch_pack: NULL operand");
    VT_REQUIRE((C == 64 || C == 128) && P > 0 && P <= 32, VTDGE_ERR_UNSUPPORTED, "layernorm_patch_pack: %d channels, P = %d", C, P);
    VT_REQUIRE(((uintptr_t)packed & 15) == 0, VTDGE_ERR_ARG, "layernorm_patch_pack: operands must be 16-byte aligned");
    const int K = P * P * C;
    for (int at = 0; at < count; at += LNP_WEIGHTS) {
        const int n = count - at < LNP_WEIGHTS ? count - at : LNP_WEIGHTS;
        PatchWeights pw = {};
        for (int i = 0; i < n; i++) {
            VT_REQUIRE(weights_host[at + i] && ((uintptr_t)weights_host[at + i] & 15) == 0, VTDGE_ERR_ARG,
                       "layernorm_patch_pack: operands must be 16-byte aligned");
            pw.w[i] = (const u32x4 *)weights_host[at + i];
        }
        note_kernel(reinterpret_cast<const void *>(patch_weight_pack_kernel));
        patch_weight_pack_kernel<<<dim3((unsigned)ceil_div(K / 8 * C, 256), (unsigned)n), 256, 0, (hipStream_t)stream>>>(
            pw, (u32x4 *)packed + (int64_t)at * (C / 8) * K, C, K);
        if (int rc = check_launch("layernorm_patch_pack")) return rc;
    }
    return VTDGE_OK;
}

extern "C" int vtdge_layernorm_patch_linear(const void *tokens, const void *ln_weight, const void *ln_bias, float eps,
                                            const void *packed, const void *bias, const void *out_ln_weight,
                                            const void *out_ln_bias, float out_eps, void *out, int B, int H, int W, int C, int P,
                                            int dtype, void *stream)
{
    VT_REQUIRE(tokens && ln_weight && ln_bias && packed && bias && out && (out_ln_weight == nullptr) == (out_ln_bias == nullptr),
               VTDGE_ERR_ARG, "layernorm_patch_linear: NULL operand");
    VT_REQUIRE(vtdge_layernorm_patch_linear_fits(B, H, W, C, P, dtype), VTDGE_ERR_UNSUPPORTED,
               "layernorm_patch_linear: no kernel for %d x %d blocks of a %d x %d grid of %d channels", P, P, H, W, C);
    VT_REQUIRE((((uintptr_t)tokens | (uintptr_t)ln_weight | (uintptr_t)ln_bias | (uintptr_t)packed | (uintptr_t)bias |
                 (uintptr_t)out_ln_weight | (uintptr_t)out_ln_bias | (uintptr_t)out) & 15) == 0, VTDGE_ERR_ARG,
               "layernorm_patch_linear: operands must be 16-byte aligned");
    const int rows = B * (H / P) * (W / P);
    const unsigned grid = (unsigned)ceil_div(rows, LNP_ROWS);
    hipStream_t st = (hipStream_t)stream;
#define VT_LAUNCH(CC)                                                                                               \
    note_kernel(reinterpret_cast<const void *>(layernorm_patch_linear_kernel<CC>)),                                 \
    layernorm_patch_linear_kernel<CC><<<grid, LNP_THREADS, 0, st>>>(                                                \
        (const bf16_t *)tokens, (const bf16_t *)ln_weight, (const bf16_t *)ln_bias, eps, (const u32x4 *)packed,     \
        (const bf16_t *)bias, (const bf16_t *)out_ln_weight, (const bf16_t *)out_ln_bias, out_eps, (bf16_t *)out, rows, H, W, P)
    if (C == 64) VT_LAUNCH(64); else VT_LAUNCH(128);
#undef VT_LAUNCH
    return check_launch("layernorm_patch_linear");
}
