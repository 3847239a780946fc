// What the bf16 / head_dim 64 attention kernels share (attention_dma.hip, attention_split.hip): how a lane reads its
// fragments of K and V from LDS, and small pieces of the softmax.
#pragma once
#include "common.h"

namespace vtdge {

struct AttnTile {
    const unsigned char *krow;      // K row `lr` of block 0 in LDS
    const unsigned char *vlane;     // this lane's source address for the transposing reads of V, block 0, d < 32
    const unsigned char *vlane_hi;  // HI: the same for d >= 32, vlane ^ 64 (key offsets are multiples of 128 bytes,
                                    // so the XOR can be taken once and every read is a base plus a constant)
    int n, lg;
};

__device__ __forceinline__ u32x4 att_read_k(const AttnTile &t, const int (&cs)[4], int kb, int sl)
{
    return *reinterpret_cast<const u32x4 *>(t.krow + kb * 32 * 128 + cs[sl]);
}
// V stays row-major in LDS ([key][d], 128-byte rows like K) and is transposed on the way to the registers:
// ds_read_b64_tr_b16 works on blocks of 16 lanes; source lane 4e + r of a block names four consecutive 16-bit
// elements, and lane i of the block receives, as its element e, column (i & 3) of source lane 4e + (i >> 2).  With
// source lane 4e + r pointing at key k0 + e, channels d0 + 4r .. d0 + 4r + 3, lane i receives keys k0 .. k0 + 3 of
// channel d0 + i: four K-elements of a row of V^T.  The first operand of O^T += V^T P^T wants, in lane (lr, lg),
// channel 32 db + lr and the eight keys the lane's own P fragment holds (16 h + 4 lg + j and 16 h + 8 + 4 lg + j,
// j < 4): two such reads, with k0 = 16 h + 4 lg (+ 8) and d0 = 32 db + 16 (block & 1).  Rows are stored with their
// 16-byte chunks XOR-ed by 2 (key & 3), so the sixteen 8-byte pieces of a block come from sixteen different bank
// groups; the XOR constant of a lane does not depend on kb, h or the +8, and db = 1 is the address XOR 64.
__device__ __forceinline__ const unsigned char *att_v_lane(const unsigned char *vbase, int lane)
{
    const int blk = lane >> 4, i = lane & 15;
    const int e = i >> 2, r = i & 3;                   // role of this lane as a source
    const int key = 4 * (blk >> 1) + e;                 // + 32 kb + 16 h (+ 8)
    const int chunk = (2 * (blk & 1) + (r >> 1)) ^ (2 * (key & 3));
    return vbase + key * 128 + chunk * 16 + 8 * (r & 1);
}
// HI: the tile carries the address for d >= 32 (two instructions a block less; in the resident kernel the extra
// register costs more than they do: 45 against 38 us)
template <bool HI>
__device__ __forceinline__ void att_read_v(const AttnTile &t, int kb, u32x4 (&vf)[4])
{
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int db = 0; db < 2; db++) {
            const unsigned char *p =
                HI ? (db ? t.vlane_hi : t.vlane) + (kb * 32 + 16 * h) * 128
                   : reinterpret_cast<const unsigned char *>((uintptr_t)(t.vlane + (kb * 32 + 16 * h) * 128) ^ (64u * db));
            const u32x2 lo = lds_read_tr16(p), hi = lds_read_tr16(p + 8 * 128);
            vf[2 * h + db].x = lo.x;
            vf[2 * h + db].y = lo.y;
            vf[2 * h + db].z = hi.x;
            vf[2 * h + db].w = hi.y;
        }
}
__device__ __forceinline__ f32x16 att_mfma(const u32x4 &a, const u32x4 &b, const f32x16 &acc)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), acc, 0,
                                                   0, 0);
}
// q * f for the packed bf16 pairs of a fragment (round to nearest even)
__device__ __forceinline__ u32x4 att_scale_frag(const u32x4 &q, float f)
{
    u32x4 r;
    r.x = pack_bf16x2(bf16lo(q.x) * f, bf16hi(q.x) * f);
    r.y = pack_bf16x2(bf16lo(q.y) * f, bf16hi(q.y) * f);
    r.z = pack_bf16x2(bf16lo(q.z) * f, bf16hi(q.z) * f);
    r.w = pack_bf16x2(bf16lo(q.w) * f, bf16hi(q.w) * f);
    return r;
}
__device__ __forceinline__ float att_max16(const f32x16 &s)
{
    const float a = fmaxf(fmaxf(fmaxf(s[0], s[1]), s[2]), fmaxf(fmaxf(s[3], s[4]), s[5]));
    const float b = fmaxf(fmaxf(fmaxf(s[6], s[7]), s[8]), fmaxf(fmaxf(s[9], s[10]), s[11]));
    return fmaxf(fmaxf(a, b), fmaxf(fmaxf(fmaxf(s[12], s[13]), s[14]), s[15]));
}
// The largest of a lane's 16 scores IF one of them is positive (else some negative value): the maximum of their bit
// patterns as signed integers, which orders positive floats as floats and puts every negative one below them.  That
// is all the test against the (positive) rescaling threshold needs, and it takes eight v_max3_i32, where fmaxf() on
// values whose origin the compiler cannot see (the output of an MFMA) brings one more instruction per operand to
// quiet signalling NaNs: 14 instructions for the same decision, a quarter of the softmax's full-rate vector work.
__device__ __forceinline__ float att_max16_if_positive(const f32x16 &s)
{
    const auto bits = [&](int e) { return __float_as_int(s[e]); };
    const auto max3 = [](int a, int b, int c) { return max(max(a, b), c); };
    int a = max3(bits(0), bits(1), bits(2)), b = max3(bits(8), bits(9), bits(10));
    a = max3(a, bits(3), bits(4));
    b = max3(b, bits(11), bits(12));
    a = max3(a, bits(5), bits(6));
    b = max3(b, bits(13), bits(14));
    a = max3(a, bits(7), bits(15));
    return __int_as_float(max(a, b));
}

}  // namespace vtdge
