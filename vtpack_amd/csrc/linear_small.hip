// Linear over few rows (gfx950), with the LayerNorm in front of it where there is one.
//
// What bounds it is latency: below some thousand rows a Linear of these models has a few dozen tiles, each of them a
// chain of dependent round trips (row count -> operands -> multiply, stage after stage -> store), and the 128-row tiles
// of the streaming kernel give it few workgroups with long chains.  So here
//   * tiles are 32 rows x 32 columns, for as many workgroups as the product has;
//   * the waves of a workgroup split K: wave w multiplies the 128-byte K slabs w, w + NW, ... of the whole tile, from a
//     ring of its own in LDS that it fills by direct loads - as many slabs in flight as fit, no barrier in the K loop -
//     and the partial tiles meet in LDS at the end.  Slab s always belongs to partial sum s mod 8 (four waves keep two
//     each) and the eight are added in order: the same bytes on every call and for either number of waves;
//   * with LN the rows of A (all of K) go to LDS first, are normalised there in place by the LayerNorm kernel's own
//     arithmetic and rounding (the same bits), and multiplied: a LayerNorm costs no launch and no copy of the rows;
//   * two independent problems over the same K (keys/values on the tokens, queries on the packed rows) can share a
//     launch.
// Consecutive tile numbers walk down the rows of one column strip and are dealt to an XCD in one run, so an XCD reads
// an eighth of the weights.  Where the rows are bf16 blocks of tokens and more than the weights they go along the columns of
// one row strip instead, an XCD reading an eighth of the rows (4096 blocks of 4096 values, 64 outputs: 11.6 against 14.3 us;
// 4096 of 2048, 128: 12.2 against 14.7).  Dense rows and fp32 lose by that (DeiT-Base, five pictures: 1473 against 1303 us;
// PVT-Tiny fp32, six of 384 px: 1628 against 1568).
#include "patch_source.h"

namespace vtdge {

constexpr int SM_BM = 32, SM_BN = 32;   // rows and columns of a tile
constexpr int SM_PITCH = 68;         // floats between the accumulator registers of a partial tile in LDS (64 lanes + 4)

struct SmallProblem {
    const void *A, *W, *bias, *res;
    void *out;
    const int64_t *rows_dev;
    int64_t lda, ldr, ldo;
    int rows, N, tiles_m, tiles_n;
};

// sums over groups of GS lanes, returned in each lane: for GS = 64 and below as group_sum_n of the LayerNorm kernels adds
// them (lane ^ 16, 8, 4, 2, 1 in that order), without their trips through LDS
template <int GS, int NV> __device__ __forceinline__ void small_group_sum(float (&v)[NV])
{
    if constexpr (GS == 64) {
        wave_sum_n<NV>(v);
        return;
    }
#pragma unroll
    for (int i = 0; i < NV; i++) {
        if constexpr (GS >= 32) {
            const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[i]), __float_as_uint(v[i]), false, false);
            v[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
        }
        if constexpr (GS >= 16) v[i] += dpp_move<0x128>(v[i]);      // the row rotated by eight
        v[i] += dpp_move<0x141>(dpp_move<0x1B>(v[i]));               // lane ^ 4: the quad reversed, the half row mirrored
        v[i] += dpp_move<0x4E>(v[i]);                                // lane ^ 2
        v[i] += dpp_move<0xB1>(v[i]);                                // lane ^ 1
    }
}

// LN: 0, or how a row lies while it is normalised: the lanes that share it (up to 64), times the 16-byte vectors of each
template <typename T, int NW, int ACT, int LN, bool PATCH>
__global__ __launch_bounds__(NW * 64) void linear_small_kernel(SmallProblem p0, SmallProblem p1, int K,
                                                               const T *__restrict__ ln_w, const T *__restrict__ ln_b,
                                                               float eps, PatchGeom pg, int ring)
{
    constexpr int ESZ = sizeof(T), VEC = Elem<T>::VEC;
    constexpr int WROWS = LN ? SM_BN : SM_BM + SM_BN;              // rows of a ring slot
    constexpr int NLW = WROWS / 8;                           // direct loads that fill it
    constexpr int GS = LN == 0 || LN > 64 ? 64 : LN, NV = LN > 64 ? LN / 64 : 1;
    constexpr int PARTS = 8, PW = PARTS / NW;                // partial sums of a tile, and a wave's share of them
    constexpr int NQ = (8 * SM_BN + NW * 64 - 1) / (NW * 64);   // four-column pieces of the output per thread
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

    const int total0 = p0.tiles_m * p0.tiles_n, total = total0 + p1.tiles_m * p1.tiles_n;
    const int per_xcd = (total + 7) / 8;
    int v = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (v >= total || (int)(blockIdx.x >> 3) >= per_xcd) return;
    const bool second = v >= total0;
    if (second) v -= total0;
    const SmallProblem &p = second ? p1 : p0;
    const int tiles_m = p.tiles_m, N = p.N;
    const bool down = !PATCH || ESZ == 4 || pg.cl_C == 0 || p.rows <= N;
    const int m0 = (down ? v % tiles_m : v / p.tiles_n) * SM_BM, n0 = (down ? v / tiles_m : v % p.tiles_n) * SM_BN;
    const int M = (int)live_rows(p.rows_dev, p.rows);
    if (m0 >= M) return;

    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int slabs = K * ESZ / SLAB_BYTES;
    const int nj = slabs > w ? (slabs - w + NW - 1) / NW : 0;      // slabs of this wave: w, w + NW, ...
    const uint32_t lds0 = (uint32_t)(uintptr_t)smem;
    const uint32_t ring0 = (LN ? slabs * SM_BM * SLAB_BYTES : 0) + w * ring * WROWS * SLAB_BYTES;

    // per-lane source offsets: a direct load brings 8 rows of a slab, LDS slot c of row r holding chunk c ^ ((r >> 1) & 7)
    uint32_t va[SM_BM / 8], vw[SM_BN / 8];
#pragma unroll
    for (int i = 0; i < SM_BM / 8; i++) {
        const int r = i * 8 + (lane >> 3), chunk = (lane & 7) ^ ((r >> 1) & 7), row = min(m0 + r, M - 1);
        if constexpr (PATCH) va[i] = (uint32_t)patch_row_offset<T>(pg, row, chunk);
        else va[i] = (uint32_t)row * (uint32_t)(p.lda * ESZ) + chunk * 16;
    }
#pragma unroll
    for (int i = 0; i < SM_BN / 8; i++) {
        const int r = i * 8 + (lane >> 3), chunk = (lane & 7) ^ ((r >> 1) & 7);
        vw[i] = (uint32_t)min(n0 + r, N - 1) * (uint32_t)(K * ESZ) + chunk * 16;
    }
    auto load_a = [&](int slab, uint32_t dst) {
        int64_t off = (int64_t)slab * SLAB_BYTES;
        if constexpr (PATCH) off = patch_slab_offset<T>(pg, slab);
        const void *base = uniform_ptr((const unsigned char *)p.A + off);
#pragma unroll
        for (int i = 0; i < SM_BM / 8; i++) dma16(base, va[i], dst + i * 1024);
    };
    auto issue = [&](int j) {
        const int slab = w + NW * j;
        uint32_t dst = lds0 + ring0 + (uint32_t)(j % ring) * WROWS * SLAB_BYTES;
        if constexpr (!LN) {
            load_a(slab, dst);
            dst += SM_BM * SLAB_BYTES;
        }
        const void *base = uniform_ptr((const unsigned char *)p.W + (int64_t)slab * SLAB_BYTES);
#pragma unroll
        for (int i = 0; i < SM_BN / 8; i++) dma16(base, vw[i], dst + i * 1024);
    };
    if constexpr (LN)
        for (int j = 0; j < nj; j++) load_a(w + NW * j, lds0 + (uint32_t)(w + NW * j) * SM_BM * SLAB_BYTES);
    for (int j = 0; j < ring && j < nj; j++) issue(j);

    if constexpr (LN) {
        // ---- LayerNorm of the tile's rows in LDS: a wave takes 32 / NW of them, 64 / GS groups of lanes side by side
        constexpr int RW = SM_BM / NW, GR = 64 / GS < RW ? 64 / GS : RW, RG = RW / GR;      // rows: wave, groups, group
        static_assert(RG <= 4, "rows side by side in a group");
        const int chunks = K / VEC, gl = lane & (GS - 1), grp = lane / GS;
        const bool mine = grp < GR;
        float gw[NV][VEC], gb[NV][VEC];
#pragma unroll
        for (int i = 0; i < NV; i++) {
            if (i * 64 + gl < chunks) {
                Elem<T>::unpack(*reinterpret_cast<const u32x4 *>(ln_w + (i * 64 + gl) * VEC), gw[i]);
                Elem<T>::unpack(*reinterpret_cast<const u32x4 *>(ln_b + (i * 64 + gl) * VEC), gb[i]);
            }
        }
        wait_vmcnt<0>();
        block_barrier();
        const int r0 = w * RW + (mine ? grp : 0) * RG;
        // of four rows a division or square root is taken once, in four lanes side by side (the rows' values by value: behind a
        // reference the selection turns into a load through a computed address, and the array into scratch memory, which every
        // launch pays for: DeiT-Small, one picture, a pass: 483 us; 476 without)
        auto in_one = [&](float v0, float v1, float v2, float v3, auto f) {
            return f(lane & 2 ? (lane & 1 ? v3 : v2) : (lane & 1 ? v1 : v0));
        };
        auto per_row = [&](const float (&v)[RG], auto f, float (&out)[RG]) {
            if constexpr (RG == 4) {
                const float r = in_one(v[0], v[1], v[2], v[3], f);
#pragma unroll
                for (int t = 0; t < RG; t++)
                    out[t] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, r), t));
            } else {
#pragma unroll
                for (int t = 0; t < RG; t++) out[t] = f(v[t]);
            }
        };
        float x[RG][NV][VEC], s[RG], mean[RG], q[RG], rstd[RG];
        unsigned char *at[RG][NV];
#pragma unroll
        for (int t = 0; t < RG; t++) {
            s[t] = 0.f;
#pragma unroll
            for (int i = 0; i < NV; i++) {
                const int c = i * 64 + gl, r = r0 + t;
                at[t][i] = smem + (c >> 3) * (SM_BM * SLAB_BYTES) + r * SLAB_BYTES + (((c & 7) ^ ((r >> 1) & 7)) * 16);
                if (c < chunks) {
                    Elem<T>::unpack(*reinterpret_cast<const u32x4 *>(at[t][i]), x[t][i]);
#pragma unroll
                    for (int e = 0; e < VEC; e++) s[t] += x[t][i][e];
                }
            }
        }
        small_group_sum<GS, RG>(s);
        per_row(s, [&](float v) { return v / (float)K; }, mean);
#pragma unroll
        for (int t = 0; t < RG; t++) {
            q[t] = 0.f;
#pragma unroll
            for (int i = 0; i < NV; i++)
                if (i * 64 + gl < chunks)
#pragma unroll
                    for (int e = 0; e < VEC; e++) {
                        const float d = x[t][i][e] - mean[t];
                        q[t] += d * d;
                    }
        }
        small_group_sum<GS, RG>(q);
        per_row(q, [&](float v) { return 1.0f / sqrtf(v / (float)K + eps); }, rstd);
#pragma unroll
        for (int t = 0; t < RG; t++)
#pragma unroll
            for (int i = 0; i < NV; i++)
                if (mine && i * 64 + gl < chunks) {
                    float y[VEC];
#pragma unroll
                    for (int e = 0; e < VEC; e++) y[e] = (x[t][i][e] - mean[t]) * rstd[t] * gw[i][e] + gb[i][e];
                    *reinterpret_cast<u32x4 *>(at[t][i]) = Elem<T>::pack(y);
                }
        lds_barrier();
    }

    // ---- this wave's share of K.  acc[v] = C[row lr][column 8 (v / 4) + 4 lg + v % 4]
    const int lr = lane & 31, lg = lane >> 5, sw = (lr >> 1) & 7;
    int cs[4];
#pragma unroll
    for (int s = 0; s < 4; s++) cs[s] = lr * SLAB_BYTES + ((2 * s + lg) ^ sw) * 16;
    f32x16 acc[PW];
#pragma unroll
    for (int h = 0; h < PW; h++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[h][e] = 0.f;
    auto multiply = [&](int j, f32x16 &ac) {
        // the slab has landed once only the loads of the younger ones are outstanding
        const int younger = min(nj, j + ring) - 1 - j;
        if (younger >= 3) wait_vmcnt<3 * NLW>();
        else if (younger == 2) wait_vmcnt<2 * NLW>();
        else if (younger == 1) wait_vmcnt<NLW>();
        else wait_vmcnt<0>();
        asm volatile("" ::: "memory");
        const unsigned char *slot = smem + ring0 + (j % ring) * WROWS * SLAB_BYTES;
        const unsigned char *As = LN ? smem + (w + NW * j) * SM_BM * SLAB_BYTES : slot;
        const unsigned char *Ws = LN ? slot : slot + SM_BM * SLAB_BYTES;
        if constexpr (ESZ == 2) {
            // all fragments are asked for before the first product: left to itself the compiler waits for two at a time (DeiT-Base,
            // 5 pictures, a pass: 999 us; 989 this way).  Not in fp32, whose products are long (PVT-Tiny, 6 of 384 px: 1272; 1283)
            u32x4 fa[4], fw[4];
#pragma unroll
            for (int s = 0; s < 4; s++) {
                fa[s] = *reinterpret_cast<const u32x4 *>(As + cs[s]);
                fw[s] = *reinterpret_cast<const u32x4 *>(Ws + cs[s]);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s = 0; s < 4; s++) Slab<T>::mma(fw[s], fa[s], ac);
        } else {
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const u32x4 fa = *reinterpret_cast<const u32x4 *>(As + cs[s]);
                Slab<T>::mma(*reinterpret_cast<const u32x4 *>(Ws + cs[s]), fa, ac);
            }
        }
        if (j + ring < nj) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");       // the slot has been read
            issue(j + ring);
        }
    };
    for (int j = 0; j < nj; j += PW) {
        multiply(j, acc[0]);
        if constexpr (PW == 2)
            if (j + 1 < nj) multiply(j + 1, acc[1]);
    }

    // ---- the partial tiles meet in LDS; a thread finishes four consecutive columns of a row
    float *sh = reinterpret_cast<float *>(smem);
    lds_barrier();
#pragma unroll
    for (int h = 0; h < PW; h++)
        for (int e = 0; e < 16; e++) sh[((h * NW + w) * 16 + e) * SM_PITCH + lane] = acc[h][e];
    lds_barrier();
#pragma unroll
    for (int i = 0; i < NQ; i++) {
        const int qd = tid + i * NW * 64;
        if (8 * SM_BN % (NW * 64) != 0 && qd >= 8 * SM_BN) return;
        const int r = qd / (SM_BN / 4), c4 = qd % (SM_BN / 4), src = (c4 & 1) * 32 + r, e0 = 4 * (c4 >> 1);
        const int row = m0 + r, col = n0 + 4 * c4;
        if (row >= M || col >= N) continue;
        float f[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ww = 0; ww < PARTS; ww++)
#pragma unroll
            for (int e = 0; e < 4; e++) f[e] += sh[(ww * 16 + e0 + e) * SM_PITCH + src];
        const int64_t orow = PATCH ? patch_out_row(pg, row) : row;
        if (p.bias != nullptr) {
#pragma unroll
            for (int e = 0; e < 4; e++) f[e] += Elem<T>::load((const T *)p.bias + col + e);
        }
        if constexpr (ACT == VTDGE_ACT_GELU) {
#pragma unroll
            for (int e = 0; e < 4; e++) f[e] = gelu_fn<T>(f[e]);
        }
        if (p.res != nullptr) {
            const T *rp = (const T *)p.res + (PATCH ? patch_res_row(pg, row) : (int64_t)row) * p.ldr + col;
#pragma unroll
            for (int e = 0; e < 4; e++) f[e] += Elem<T>::load(rp + e);
        }
        T *op = (T *)p.out + orow * p.ldo + col;
        if constexpr (ESZ == 2) {
            u32x2 o2;
            o2.x = pack_bf16x2(f[0], f[1]);
            o2.y = pack_bf16x2(f[2], f[3]);
            *reinterpret_cast<u32x2 *>(op) = o2;
        } else {
            *reinterpret_cast<f32x4 *>(op) = f32x4{f[0], f[1], f[2], f[3]};
        }
    }
}

// ----------------------------------------------------------------------------- host
template <typename T, int NW, int ACT, int LN, bool PATCH>
static int go_small(const SmallProblem &p0, const SmallProblem &p1, int K, const void *ln_w, const void *ln_b, float eps,
                    const PatchGeom &pg, hipStream_t st)
{
    constexpr int WROWS = LN ? SM_BN : SM_BM + SM_BN;
    const int slabs = K * (int)sizeof(T) / SLAB_BYTES;
    const size_t a_bytes = LN ? (size_t)slabs * SM_BM * SLAB_BYTES : 0, slot = (size_t)NW * WROWS * SLAB_BYTES;
    // as many slots per wave as it has slabs, up to four, within half a compute unit's LDS (two workgroups share it)
    // where that leaves at least two, else within all of it
    int ring = (slabs + NW - 1) / NW;
    ring = ring < 4 ? ring : 4;
    while (ring > (LN ? 1 : 2) && a_bytes + ring * slot > 80 * 1024) ring--;
    while (ring > 1 && a_bytes + ring * slot > 160 * 1024) ring--;
    const size_t reduce = (size_t)8 * 16 * SM_PITCH * 4;
    const size_t lds = a_bytes + ring * slot > reduce ? a_bytes + ring * slot : reduce;
    VT_REQUIRE(lds <= 160 * 1024, VTDGE_ERR_UNSUPPORTED, "linear: %d values of K do not fit the LDS", K);
    auto kern = linear_small_kernel<T, NW, ACT, LN, PATCH>;
    VT_RESERVE_LDS(kern, 160 * 1024, "linear");
    const int64_t total = (int64_t)p0.tiles_m * p0.tiles_n + (int64_t)p1.tiles_m * p1.tiles_n;
    note_kernel(reinterpret_cast<const void *>(kern));
    kern<<<dim3((unsigned)(ceil_div(total, 8) * 8)), dim3(NW * 64), lds, st>>>(p0, p1, K, (const T *)ln_w, (const T *)ln_b,
                                                                               eps, pg, ring);
    return check_launch("linear");
}

static SmallProblem small_problem(const void *A, int64_t lda, const void *W, const void *bias, const void *res, int64_t ldr,
                                  void *out, int64_t ldo, const int64_t *rows_dev, int64_t rows, int N)
{
    return SmallProblem{A, W, bias, res, out, rows_dev, lda, ldr, ldo, (int)rows, N, (int)ceil_div(rows, SM_BM),
                        (int)ceil_div(N, SM_BN)};
}

// What the kernel needs of one problem: whole 128-byte slabs of K, four-column pieces of the output, 32-bit offsets.
bool linear_small_fits(int64_t lda, int64_t ldr, int64_t ldo, int64_t rows, int N, int K, int esz, const void *bias,
                       const void *res, const void *out)
{
    const int64_t piece = 4 * esz - 1;
    return ((int64_t)K * esz) % SLAB_BYTES == 0 && N % 4 == 0 && ldo % 4 == 0 && rows * lda * esz < (1ll << 31) &&
           (int64_t)N * K * esz < (1ll << 31) && ((uintptr_t)out & piece) == 0;
}

// Which products the kernel is taken for, by their 32x32 tiles at full row capacity: where it is no slower than the streaming
// kernel with every row live, as a router that keeps the finest split (an untrained one) leaves them.  Of packed rows about
// 0.44 are live for a trained mix; that only adds to its lead.  Measured, us, this kernel / streaming, all rows live and 0.44
// of them, by tiles (rows, N, K):
//   bf16  768 (4091, 192, 192) 5.7 / 6.1, 4.8 / 6.0     768 (507, 1536, 384) 7.3 / 8.1, 5.4 / 7.9
//         760 (2427, 320, 1280) 13.7 / 14.0, 7.6 / 13.5 768 (1531, 512, 2048) 17.7 / 20.1, 9.2 / 19.2
//        1008 (2011, 512, 2048) 24.0 / 19.9, 10.7 / 19.1   2016 (1339, 1536, 384) 15.1 / 8.8, 8.9 / 8.0
//        1500 (4795, 320, 320) 12.7 / 7.3, 8.5 / 7.0    768 (4091, 192, 768) 11.7 / 10.3, 6.5 / 10.0 (narrow: half a tile
//        of the streaming kernel's is empty, but it has many)
//   long rows of 768 values and more, with as many outputs, leave the streaming kernel few tiles and long chains:
//        1008 (1339, 768, 768) 10.4 / 10.0, 6.4 / 9.7   1008 (1339, 768, 3072) 30.9 / 27.7, 13.5 / 27.2 (30.2 on the tiles
//        before the present ones)  960 (315, 3072, 768) 10.4 / 12.5, 8.3 / 12.1
//        1488 (1979, 768, 768) 15.2 / 10.0, 8.4 / 9.6   1488 (1979, 768, 3072) 46.2 / 27.9, 20.2 / 27.2
//   fp32 1024 (2043, 512, 2048) 54.6 / 45.7, 25.8 / 42.1   1020 (2715, 384, 1536) 42.5 / 58.0, 33.8 / 32.3
//        1008 (1339, 768, 768) 23.7 / 31.4, 12.1 / 18.6    1020 (5435, 192, 768) 26.1 / 31.6, 19.3 / 18.1
//        1398 (7451, 192, 192) 18.0 / 11.6, 10.9 / 7.5     2040 (5435, 384, 1536) 81.7 / 85.1, 52.0 / 33.1
//        2700 (7195, 384, 384) 38.7 / 26.3, 25.4 / 17.9    4080 (13051, 320, 1280) 128.9 / 113.5, 70.4 / 48.3
static int64_t small_tiles(int64_t rows, int N) { return ceil_div(rows, SM_BM) * ceil_div(N, SM_BN); }
bool linear_small_wanted(int64_t rows, int N, int K, int esz)
{
    const int64_t most = esz == 4 || (N >= 768 && K >= 768) ? 1024 : N >= 256 ? 768 : 640;
    return small_tiles(rows, N) <= most;
}

template <typename T>
int launch_linear_small(const void *A, int64_t lda, const void *W, const void *bias, const void *res, int64_t ldr,
                        void *out, int64_t ldo, const int64_t *rows_dev, int64_t rows, int N, int K, int act,
                        hipStream_t st)
{
    const PatchGeom none{0, 0, 0, 0, 0, 0, 0, 0};
    const SmallProblem p = small_problem(A, lda, W, bias, res, ldr, out, ldo, rows_dev, rows, N);
    // eight waves where a tile has two slabs of K for each of them and there are too few tiles to fill the chip
    const bool deep = K * (int)sizeof(T) / SLAB_BYTES >= 16 && small_tiles(rows, N) <= 256;
#define VT_SMALL(NW, ACT) return go_small<T, NW, ACT, 0, false>(p, SmallProblem{}, K, nullptr, nullptr, 0.f, none, st)
    if (act == VTDGE_ACT_GELU) {
        if (deep) VT_SMALL(8, VTDGE_ACT_GELU);
        VT_SMALL(4, VTDGE_ACT_GELU);
    }
    if (deep) VT_SMALL(8, VTDGE_ACT_NONE);
    VT_SMALL(4, VTDGE_ACT_NONE);
#undef VT_SMALL
}
template int launch_linear_small<float>(const void *, int64_t, const void *, const void *, const void *, int64_t, void *,
                                        int64_t, const int64_t *, int64_t, int, int, int, hipStream_t);
template int launch_linear_small<bf16_t>(const void *, int64_t, const void *, const void *, const void *, int64_t, void *,
                                         int64_t, const int64_t *, int64_t, int, int, int, hipStream_t);

// The patch embedding and the strided convolution over tokens (patch_source.h) for few rows, by the same tiles (all rows
// live).  Measured, us, this kernel / streaming (rows, N, K): images, bf16 480 (1280, 384, 768) 8.3 / 11.7, 576 12.0 / 11.8,
// 960 14.5 / 11.9; fp32 480 15.0 / 21.1, 768 (1024, 768, 768) 21.6 / 21.8, 1920 52.0 / 37.0.  Blocks of tokens, bf16 512
// (1024, 512, 1280) 10.3 / 10.8, (4096, 128, 256) 6.7 / 5.9; fp32 700 (2240, 320, 1280) 31.0 / 33.4, (11200, 64, 4096)
// 79 / 93, 1000 (1984, 512, 1280) 40 / 35, 2000 74 / 54.
bool patch_small_wanted(int64_t rows, int N, int K, int esz, int64_t source_bytes)
{
    return small_tiles(rows, N) <= (esz == 2 ? 512 : 768) && (int64_t)K * esz % SLAB_BYTES == 0 && N % 4 == 0 &&
           source_bytes < (1ll << 31) && (int64_t)N * K * esz < (1ll << 31);
}
template <typename T>
int launch_patch_small(const void *source, const void *W, const void *bias, const void *res, void *out, int64_t rows, int N,
                       int K, const PatchGeom &pg, hipStream_t st)
{
    const SmallProblem p = small_problem(source, 0, W, bias, res, N, out, N, nullptr, rows, N);
    if (K * (int)sizeof(T) / SLAB_BYTES >= 16 && small_tiles(rows, N) <= 256)
        return go_small<T, 8, VTDGE_ACT_NONE, 0, true>(p, SmallProblem{}, K, nullptr, nullptr, 0.f, pg, st);
    return go_small<T, 4, VTDGE_ACT_NONE, 0, true>(p, SmallProblem{}, K, nullptr, nullptr, 0.f, pg, st);
}
template int launch_patch_small<float>(const void *, const void *, const void *, const void *, void *, int64_t, int, int,
                                       const PatchGeom &, hipStream_t);
template int launch_patch_small<bf16_t>(const void *, const void *, const void *, const void *, void *, int64_t, int, int,
                                        const PatchGeom &, hipStream_t);

// act(LayerNorm(A) W^T + bias): one problem, or two over the same K with the same LayerNorm (rows1 = 0: none).
bool layernorm_linear_fits(int64_t rows0, int N0, int64_t rows1, int N1, int K, int esz)
{
    const int64_t row = (int64_t)K * esz, tiles = small_tiles(rows0, N0) + small_tiles(rows1, N1);
    return row % SLAB_BYTES == 0 && row <= 2048 && N0 % 4 == 0 && N1 % 4 == 0 &&
           tiles <= (row > 1536 ? 512 : rows1 > 0 ? 2048 : 1024);
}
// Which of them the kernel is taken for: every column tile normalises its rows again, so what the LayerNorm kernels' launches
// cost is given back from some number of tiles on, the sooner the longer the rows.  The line lies where the separate kernels
// (streaming Linears) are even with all packed rows live, as an untrained router leaves them.  Measured, us, this kernel /
// separate kernels (rows, K; tiles), all rows live: keys/values and queries, bf16 257, 384: 8.4 / 20.4; 1285, 384 (1476):
// 19.8 / 21.1; 1028, 512 (1584): 23.4 / 22.8; 1285, 512 (1968): 26.4 / 23.4; 514, 768 (1224): 24.2 / 29.1; 771, 768 (1800):
// 33.5 / 30.0; fp32 257, 384: 11.7 / 28.6; 1285, 384 (1476): 31.5 / 36.7; 3000, 192 (1692): 27.5 / 26.4; 2056, 320
// (1950): 39.7 / 34.1.  fc1, bf16 1285, 192 (984): 9.6 / 11.4; 514, 320 (680): 11.1 / 11.2; 771, 320 (1000): 13.6 / 11.3; 514, 384
// (816): 14.5 / 11.9; 257, 512 (576): 12.9 / 12.8; 64, 768 (192): 8.5 / 16.3; 257, 768 (864): 19.6 / 17.1; fp32 514, 192
// (408): 10.2 / 12.0; 771, 192 (600): 15.0 / 12.4; 514, 320 (680): 18.3 / 20.0; 514, 384 (816): 22.2 / 22.3.
static bool layernorm_linear_wanted(int64_t rows0, int N0, int64_t rows1, int N1, int K, int esz)
{
    const int64_t row = (int64_t)K * esz, tiles = small_tiles(rows0, N0) + small_tiles(rows1, N1);
    if (!layernorm_linear_fits(rows0, N0, rows1, N1, K, esz)) return false;
    if (esz == 4) return tiles <= (rows1 > 0 ? 1536 : row > 1024 ? 768 : 512);
    if (rows1 > 0) return tiles <= (row > 1024 ? 1280 : row == 1024 ? 1600 : 2048);
    return tiles <= (row <= 384 ? 1024 : row <= 1024 ? 640 : 512);
}
template <typename T>
static int launch_layernorm_linear(const void *A0, int64_t lda0, const void *W0, const void *bias0, void *out0,
                                   const int64_t *rows_dev0, int64_t rows0, int N0, const void *A1, int64_t lda1,
                                   const void *W1, const void *bias1, void *out1, const int64_t *rows_dev1, int64_t rows1,
                                   int N1, const void *ln_w, const void *ln_b, float eps, int K, int act, hipStream_t st)
{
    const PatchGeom none{0, 0, 0, 0, 0, 0, 0, 0};
    const SmallProblem p0 = small_problem(A0, lda0, W0, bias0, nullptr, 0, out0, N0, rows_dev0, rows0, N0);
    const SmallProblem p1 = rows1 > 0 ? small_problem(A1, lda1, W1, bias1, nullptr, 0, out1, N1, rows_dev1, rows1, N1)
                                      : SmallProblem{};
    const int vecs = K * (int)sizeof(T) / 16;
#define VT_SMALL(LN)                                                                                                    \
    do {                                                                                                                \
        if (act == VTDGE_ACT_GELU)                                                                                      \
            return go_small<T, 8, VTDGE_ACT_GELU, LN, false>(p0, p1, K, ln_w, ln_b, eps, none, st);                 \
        return go_small<T, 8, VTDGE_ACT_NONE, LN, false>(p0, p1, K, ln_w, ln_b, eps, none, st);                     \
    } while (0)
    if (vecs <= 8) VT_SMALL(8);
    if (vecs <= 16) VT_SMALL(16);
    if (vecs <= 32) VT_SMALL(32);
    if (vecs <= 64) VT_SMALL(64);
    VT_SMALL(128);
#undef VT_SMALL
}

// A0 W0^T + bias0 and A1 W1^T + bias1 over the same K in one launch
template <typename T>
static int launch_pair(const SmallProblem &p0, const SmallProblem &p1, int K, hipStream_t st)
{
    const PatchGeom none{0, 0, 0, 0, 0, 0, 0, 0};
    return go_small<T, 4, VTDGE_ACT_NONE, 0, false>(p0, p1, K, nullptr, nullptr, 0.f, none, st);
}

}  // namespace vtdge

using namespace vtdge;

extern "C" int vtdge_layernorm_linear_fits(int64_t rows0, int N0, int64_t rows1, int N1, int K, int dtype)
{
    if (rows0 < 0 || rows1 < 0 || N0 <= 0 || N1 < 0 || K <= 0 || (dtype != VTDGE_F32 && dtype != VTDGE_BF16)) return 0;
    return layernorm_linear_fits(rows0, N0, rows1, N1, K, dtype == VTDGE_BF16 ? 2 : 4) ? 1 : 0;
}

extern "C" int vtdge_layernorm_linear_wanted(int64_t rows0, int N0, int64_t rows1, int N1, int K, int dtype)
{
    if (rows0 < 0 || rows1 < 0 || N0 <= 0 || N1 < 0 || K <= 0 || (dtype != VTDGE_F32 && dtype != VTDGE_BF16)) return 0;
    return layernorm_linear_wanted(rows0, N0, rows1, N1, K, dtype == VTDGE_BF16 ? 2 : 4) ? 1 : 0;
}

extern "C" int vtdge_layernorm_linear(const void *A0, int64_t lda0, const void *W0, const void *bias0, void *out0,
                                      const int64_t *rows_dev0, int64_t rows0, int N0, const void *A1, int64_t lda1,
                                      const void *W1, const void *bias1, void *out1, const int64_t *rows_dev1,
                                      int64_t rows1, int N1, const void *ln_weight, const void *ln_bias, float ln_eps, int K,
                                      int act, int dtype, void *stream)
{
    VT_REQUIRE(A0 && W0 && out0 && ln_weight && ln_bias, VTDGE_ERR_ARG, "layernorm_linear: NULL operand");
    VT_REQUIRE(rows1 == 0 || (A1 && W1 && out1), VTDGE_ERR_ARG, "layernorm_linear: NULL operand of the second product");
    VT_REQUIRE(dtype == VTDGE_F32 || dtype == VTDGE_BF16, VTDGE_ERR_ARG, "layernorm_linear: unknown dtype %d", dtype);
    VT_REQUIRE(act == VTDGE_ACT_NONE || act == VTDGE_ACT_GELU, VTDGE_ERR_ARG, "layernorm_linear: unknown activation %d",
               act);
    const int esz = dtype == VTDGE_BF16 ? 2 : 4;
    VT_REQUIRE(rows0 >= 0 && rows1 >= 0 && N0 > 0 && N1 >= 0 && K > 0 && lda0 >= K && (rows1 == 0 || lda1 >= K),
               VTDGE_ERR_ARG, "layernorm_linear: bad sizes");
    VT_REQUIRE(layernorm_linear_fits(rows0, N0, rows1, N1, K, esz) && rows0 * lda0 * esz < (1ll << 31) &&
                   rows1 * lda1 * esz < (1ll << 31) && (lda0 * esz) % 16 == 0 && (rows1 == 0 || (lda1 * esz) % 16 == 0),
               VTDGE_ERR_UNSUPPORTED, "layernorm_linear: %lld x %d and %lld x %d outputs over %d values (see "
               "vtdge_layernorm_linear_fits)", (long long)rows0, N0, (long long)rows1, N1, K);
    VT_REQUIRE((((uintptr_t)A0 | (uintptr_t)W0 | (uintptr_t)out0 | (uintptr_t)A1 | (uintptr_t)W1 | (uintptr_t)out1 |
                 (uintptr_t)ln_weight | (uintptr_t)ln_bias) & 15) == 0,
               VTDGE_ERR_ARG, "layernorm_linear: operands must be 16-byte aligned");
    if (rows0 == 0 && rows1 == 0) return VTDGE_OK;
    hipStream_t st = (hipStream_t)stream;
    if (dtype == VTDGE_F32)
        return launch_layernorm_linear<float>(A0, lda0, W0, bias0, out0, rows_dev0, rows0, N0, A1, lda1, W1, bias1, out1,
                                              rows_dev1, rows1, N1, ln_weight, ln_bias, ln_eps, K, act, st);
    return launch_layernorm_linear<bf16_t>(A0, lda0, W0, bias0, out0, rows_dev0, rows0, N0, A1, lda1, W1, bias1, out1,
                                           rows_dev1, rows1, N1, ln_weight, ln_bias, ln_eps, K, act, st);
}

extern "C" int vtdge_linear_pair(const void *A0, int64_t lda0, const void *W0, const void *bias0, void *out0,
                                 const int64_t *rows_dev0, int64_t rows0, int N0, const void *A1, int64_t lda1, const void *W1,
                                 const void *bias1, void *out1, const int64_t *rows_dev1, int64_t rows1, int N1, int K, int dtype,
                                 void *stream)
{
    VT_REQUIRE(A0 && W0 && out0 && A1 && W1 && out1, VTDGE_ERR_ARG, "linear_pair: NULL operand");
    VT_REQUIRE(dtype == VTDGE_F32 || dtype == VTDGE_BF16, VTDGE_ERR_ARG, "linear_pair: unknown dtype %d", dtype);
    const int esz = dtype == VTDGE_BF16 ? 2 : 4;
    VT_REQUIRE(rows0 > 0 && rows1 > 0 && N0 > 0 && N1 > 0 && K > 0 && lda0 >= K && lda1 >= K, VTDGE_ERR_ARG,
               "linear_pair: bad sizes");
    VT_REQUIRE(layernorm_linear_fits(rows0, N0, rows1, N1, K, esz) && rows0 * lda0 * esz < (1ll << 31) &&
                   rows1 * lda1 * esz < (1ll << 31) && (lda0 * esz) % 16 == 0 && (lda1 * esz) % 16 == 0,
               VTDGE_ERR_UNSUPPORTED, "linear_pair: %lld x %d and %lld x %d outputs over %d values (see "
               "vtdge_layernorm_linear_fits)", (long long)rows0, N0, (long long)rows1, N1, K);
    VT_REQUIRE((((uintptr_t)A0 | (uintptr_t)W0 | (uintptr_t)out0 | (uintptr_t)A1 | (uintptr_t)W1 | (uintptr_t)out1) & 15) == 0,
               VTDGE_ERR_ARG, "linear_pair: operands must be 16-byte aligned");
    hipStream_t st = (hipStream_t)stream;
    const SmallProblem p0 = small_problem(A0, lda0, W0, bias0, nullptr, 0, out0, N0, rows_dev0, rows0, N0);
    const SmallProblem p1 = small_problem(A1, lda1, W1, bias1, nullptr, 0, out1, N1, rows_dev1, rows1, N1);
    return dtype == VTDGE_F32 ? launch_pair<float>(p0, p1, K, st) : launch_pair<bf16_t>(p0, p1, K, st);
}
