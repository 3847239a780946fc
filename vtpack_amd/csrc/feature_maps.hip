// Token rows of a stage to feature maps: out[b, c, t] = x[b, t, c] (gfx950).
//
// Bound by memory once both sides are coalesced: tiles of 64 tokens by 64 channels go through LDS, read in 16-byte pieces along
// the channels and written in 16-byte pieces along the tokens, 256 bytes of a row or a map side by side in fp32.  The LDS rows
// are one word longer than a tile, so that neither side meets a bank twice.  Us, a general strided copy, which reads 4
// bytes at a time across the rows / so (samples, tokens, channels): fp32 24, 16384, 64: 92.9 / 32.2 (201 MB); 6, 9216, 64: 19.1 /
// 6.6; 256, 3136, 64: 258 / 60.7; bf16 24, 16384, 64: 97.0 / 18.4; 256, 49, 512: 17.1 / 11.7.
#include "common.h"

namespace vtdge {

constexpr int FM_TILE = 64;

// VIN, VOUT: rows of x, maps of out lie on 16-byte boundaries
template <typename U, bool VIN, bool VOUT>
__global__ __launch_bounds__(256) void rows_to_maps_kernel(const U *__restrict__ x, int64_t batch_stride, U *__restrict__ out,
                                                           int tokens, int C, int token_tiles, int channel_tiles)
{
    constexpr int VEC = 16 / sizeof(U), LPR = FM_TILE / VEC, ROWS = 256 / LPR, STRIDE = FM_TILE + 4 / (int)sizeof(U);
    struct Vec {
        U v[VEC];
    };
    __shared__ U tile[FM_TILE * STRIDE];
    const int of_sample = token_tiles * channel_tiles;
    const int b = blockIdx.x / of_sample, rest = blockIdx.x - b * of_sample;
    const int t0 = (rest / channel_tiles) * FM_TILE, c0 = (rest % channel_tiles) * FM_TILE;
    const int piece = (threadIdx.x % LPR) * VEC, row = threadIdx.x / LPR;
    const U *const from = x + b * batch_stride;
    U *const to = out + (int64_t)b * C * tokens;

    Vec got[FM_TILE / ROWS] = {};
#pragma unroll
    for (int i = 0; i < FM_TILE / ROWS; i++) {
        const int t = t0 + row + i * ROWS, c = c0 + piece;
        const U *const p = from + (int64_t)t * C + c;
        if (t >= tokens) continue;
        if constexpr (VIN) {
            if (c < C) got[i] = __builtin_bit_cast(Vec, __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(p)));
        } else {
#pragma unroll
            for (int e = 0; e < VEC; e++)
                if (c + e < C) got[i].v[e] = p[e];
        }
    }
#pragma unroll
    for (int i = 0; i < FM_TILE / ROWS; i++)
#pragma unroll
        for (int e = 0; e < VEC; e++) tile[(row + i * ROWS) * STRIDE + piece + e] = got[i].v[e];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < FM_TILE / ROWS; i++) {
        const int c = c0 + row + i * ROWS, t = t0 + piece;
        if (c >= C) continue;
        Vec put;
#pragma unroll
        for (int e = 0; e < VEC; e++) put.v[e] = tile[(piece + e) * STRIDE + row + i * ROWS];
        U *const p = to + (int64_t)c * tokens + t;
        if constexpr (VOUT) {
            if (t < tokens) *reinterpret_cast<u32x4 *>(p) = __builtin_bit_cast(u32x4, put);
        } else {
#pragma unroll
            for (int e = 0; e < VEC; e++)
                if (t + e < tokens) p[e] = put.v[e];
        }
    }
}

template <typename U>
static int go_rows_to_maps(const void *x, int64_t batch_stride, void *out, int B, int tokens, int C, hipStream_t st)
{
    constexpr int VEC = 16 / sizeof(U);
    const int64_t tt = ceil_div(tokens, FM_TILE), ct = ceil_div(C, FM_TILE), blocks = tt * ct * B;
    VT_REQUIRE(blocks < (int64_t)1 << 31, VTDGE_ERR_UNSUPPORTED, "rows_to_maps: %lld tiles", (long long)blocks);
    const bool vin = C % VEC == 0 && batch_stride % VEC == 0 && ((uintptr_t)x & 15) == 0;
    const bool vout = tokens % VEC == 0 && ((uintptr_t)out & 15) == 0;
    auto kern = vin ? (vout ? rows_to_maps_kernel<U, true, true> : rows_to_maps_kernel<U, true, false>)
                    : (vout ? rows_to_maps_kernel<U, false, true> : rows_to_maps_kernel<U, false, false>);
    note_kernel(reinterpret_cast<const void *>(kern));
    kern<<<dim3((unsigned)blocks), dim3(256), 0, st>>>((const U *)x, batch_stride, (U *)out, tokens, C, (int)tt, (int)ct);
    return check_launch("rows_to_maps");
}

}  // namespace vtdge

using namespace vtdge;

extern "C" int vtdge_rows_to_maps(const void *x, int64_t batch_stride, void *out, int B, int tokens, int C, int dtype, void *stream)
{
    VT_REQUIRE(x && out, VTDGE_ERR_ARG, "rows_to_maps: NULL operand");
    VT_REQUIRE(B > 0 && tokens > 0 && C > 0 && batch_stride >= (int64_t)tokens * C, VTDGE_ERR_ARG, "rows_to_maps: bad sizes");
    VT_REQUIRE(dtype == VTDGE_F32 || dtype == VTDGE_BF16, VTDGE_ERR_UNSUPPORTED, "rows_to_maps: dtype %d", dtype);
    if (dtype == VTDGE_F32) return go_rows_to_maps<uint32_t>(x, batch_stride, out, B, tokens, C, (hipStream_t)stream);
    return go_rows_to_maps<uint16_t>(x, batch_stride, out, B, tokens, C, (hipStream_t)stream);
}
