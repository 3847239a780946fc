// Where the rows of a Linear over patches come from, shared by the kernels that read them in place (gfx950).
//
// The Linear is a patch embedding (a convolution whose stride is its kernel size, as a Linear over the
// patches).  A is the image batch [B, Cin, S, S] itself: row (b, gy, gx) of the product is patch (gy, gx) of image b
// and its K index runs over (channel, row of the patch, pixel), so a 128-byte K slab of a row is a few consecutive
// pixel rows of one channel of the patch and the loader waves fetch them straight from the image - nothing but
// their per-lane source addresses differs from the plain kernel, no unfolded copy of the images exists.  The output
// row goes to token `extra + gy G + gx` of sample b in [B, extra + G G, N], and the residual is row
// `extra + gy G + gx` of one [extra + G G, N] table for every sample (the position embedding).
//
// The same mode reads patches of a channels-last token grid (cl_C > 0): A is [B, cl_H cl_W, cl_C] tokens, row
// (b, gy, gx) of the product is the P x P block of tokens at (gy P, gx P) and its K index runs over (token row of
// the block, token of that row, channel), i.e. a 128-byte K slab is a piece of one token's channels (cl_C values
// must fill whole slabs).  This is a stride-P P x P convolution over the grid with its weight in [O, kh, kw, C]
// order; rows of the product are stored densely (extra = 0) and there is no residual.
#pragma once
#include "common.h"

namespace vtdge {

struct PatchGeom {
    int P, S, G, Cin, extra;     // patch edge, image edge, patches per edge, input channels, tokens in front
    int cl_C, cl_H, cl_W;        // channels-last source: channels and token grid (cl_C = 0: an image batch)
};

constexpr int SLAB_BYTES = 128;   // of a row of A per stage of the kernels' K loops

// byte offset in A of 16-byte chunk `chunk` of slab 0 of row `row`
template <typename T> __device__ __forceinline__ int64_t patch_row_offset(const PatchGeom &pg, int row, int chunk)
{
    constexpr int ESZ = sizeof(T);
    if (pg.cl_C > 0) {
        // block (b, gy, gx) of the token grid: its first token; the slab's piece is added per stage
        const int gw = pg.cl_W / pg.P, g2 = (pg.cl_H / pg.P) * gw;
        const int b = row / g2, t = row - b * g2, gy = t / gw, gx = t - gy * gw;
        return (((int64_t)b * pg.cl_H + gy * pg.P) * pg.cl_W + gx * pg.P) * pg.cl_C * ESZ + chunk * 16;
    }
    // patch (b, gy, gx); the chunk is pixels `cc` of patch row `cr` of the slab's first rows
    const int g2 = pg.G * pg.G, cpr = pg.P * ESZ / 16;      // chunks per patch row
    const int b = row / g2, t = row - b * g2, gy = t / pg.G, gx = t - gy * pg.G;
    const int cr = chunk / cpr, cc = chunk % cpr;
    return (((int64_t)b * pg.Cin * pg.S + gy * pg.P + cr) * pg.S + gx * pg.P) * ESZ + cc * 16;
}
// what slab `kt` adds to that offset
template <typename T> __device__ __forceinline__ int64_t patch_slab_offset(const PatchGeom &pg, int kt)
{
    constexpr int ESZ = sizeof(T);
    if (pg.cl_C > 0) {
        // slab kt of a block of tokens: which token of the block and where in its channels
        const int spt = pg.cl_C * ESZ / SLAB_BYTES;                       // slabs per token
        const int tk = kt / spt, dy = tk / pg.P, dx = tk - dy * pg.P;
        return ((int64_t)(dy * pg.cl_W + dx) * pg.cl_C) * ESZ + (int64_t)(kt - tk * spt) * SLAB_BYTES;
    }
    // slab kt of a patch: its channel and its first row in the patch
    const int rps = SLAB_BYTES / (pg.P * ESZ), spc = pg.P / rps;          // rows per slab, slabs per channel
    return ((int64_t)(kt / spc) * pg.S + (kt % spc) * rps) * pg.S * ESZ;
}
// where row `row` of the product is stored and which row of the residual table it takes
// (32-bit arithmetic: the patch count of a batch fits, and a 64-bit division costs a hundred instructions)
__device__ __forceinline__ int64_t patch_out_row(const PatchGeom &pg, int row)
{
    return row + (int64_t)(row / (pg.G * pg.G) + 1) * pg.extra;
}
__device__ __forceinline__ int64_t patch_res_row(const PatchGeom &pg, int row) { return row % (pg.G * pg.G) + pg.extra; }

}  // namespace vtdge
