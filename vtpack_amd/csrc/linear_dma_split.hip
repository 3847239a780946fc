// fp32 Linear on the bf16 matrix instructions, as exact as on the fp32 ones (gfx950).
//
// The fp32 matrix instructions multiply at 1/16 of the rate of v_mfma_f32_32x32x16_bf16.  An fp32 value is the sum of three bf16
// values, exactly (8 + 8 + 8 significant bits, each part rounded to nearest, so the remainders are signed): x = x1 + x2 + x3 with
// |x2| <= 2^-8 |x| and |x3| <= 2^-17 |x|.  Of the nine partial products of two such sums the six of weight 2^-17 and above are
// multiplied, each exactly, and added in fp32; what is left out is up to 2^-24 of the product where both operands are as far from a
// bf16 value as they can be and all terms have one sign (one rounding of fp32), 2^-26 or less in 97 of 100 pairs of mantissas.
// Against float64 the sums are closer than those of the fp32 instructions: over unit normals 0.82 to 0.86 of the error (2-norm, K =
// 192 to 1536), over values of one sign 0.65 to 0.82.  That is 16/6 of the fp32 instructions' rate if the splitting (11 vector
// instructions for two values) hides behind the products: a wave splits the operands of one step of 16 columns of K while it
// multiplies those of the step before and the ones of the step after are on their way out of LDS, one matrix instruction (32
// clocks) and then the vector instructions that fit its shadow. Split first and multiplied then, the two add up.
//
// Operands go to LDS as in linear_dma.hip: loader waves stream 128-byte slabs of both by direct loads into a ring, one
// barrier a stage, the ring running on across the tiles of a persistent workgroup.
//
// Not covered by the split: an infinity or NaN (the remainders become NaN), a value that rounds to infinity in bf16, and sums
// that live below the precision of small bf16 values.  All of them show in the result: a block with a sum that is not
// finite, or not zero and below 2^-80, is worked out again with the fp32 instructions from the operands in memory.  A sum of
// 2^-80 and above hides what small bf16 values lose (2^-134 of an operand) only where the other operand is not huge: weights
// from 2^20 on, whose activations may be that small, and those below 2^-100, are put down as NaN and so join the others.
// Such a block walks all of K from memory behind its products, unpipelined.  Us, no such weight / one in one of the blocks of 32
// columns / one in all of them / the fp32 instructions' kernel (rows, N, K; the split of the weight among them, 3.3 to 5.7):
// 32896, 384, 192: 47 / 60 / 119 / 60; 16448, 1536, 384: 134 / 194 / 474 / 186; 4112, 3072, 768: 162 / 244 / 525 / 200.
#include "common.h"

namespace vtdge {

namespace {

constexpr int DKB = 128;                   // bytes of a row of A per stage

}  // namespace

// Byte offset of plane `p` of row `n`, columns 32 kt .. 32 kt + 31 of K, in the packed copy of a weight: 1 KB blocks of 16
// rows, three planes after one another, K next, rows last.  A block is what one direct load brings into LDS: 64 bytes a
// row, whose 16-byte pieces q = 2 t + g hold what lane half g multiplies in step t (columns 16 t + 4 g + 0..3 and 16 t + 8
// + 4 g + 0..3, as it finds them in two pieces of a row of A), piece q of row n in place q ^ (n / 4 % 4): 16 rows at one q,
// a phase of a fragment read, lie in 16 different bank groups.
__device__ __forceinline__ int64_t packed_block(int n16, int kt, int nk, int p) { return (((int64_t)n16 * nk + kt) * 3 + p) * 1024; }

// Weights of one launch, and the workgroups up to and including each one's (vtdge_linear_split_set)
constexpr int SPLIT_SET = 80;
struct SplitSet {
    struct {
        const float *W;
        unsigned char *packed;
        int N, K;
    } of[SPLIT_SET];
    int end[SPLIT_SET], count;
};

__global__ __launch_bounds__(256) void split_weights_kernel(const SplitSet set)
{
    int j = 0;
    for (int step = 64; step > 0; step >>= 1)               // the first weight that ends behind this workgroup
        if (j + step <= set.count - 1 && (int)blockIdx.x >= set.end[j + step - 1]) j += step;
    const float *W = set.of[j].W;
    unsigned char *packed = set.of[j].packed;
    const int K = set.of[j].K;
    const int i = ((int)blockIdx.x - (j > 0 ? set.end[j - 1] : 0)) * 256 + threadIdx.x;      // piece q of (row, slab)
    const int nk = K / 32, q = i & 3, n = i / 4 / nk, kt = i / 4 - n * nk;
    if (n >= set.of[j].N) return;
    const float *src = W + (int64_t)n * K + kt * 32 + 16 * (q >> 1) + 4 * (q & 1);
    const u32x4 lo = *reinterpret_cast<const u32x4 *>(src), hi = *reinterpret_cast<const u32x4 *>(src + 8);
    u32x4 part[3];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        float x = __uint_as_float(e < 2 ? lo[2 * e] : hi[2 * e - 4]), y = __uint_as_float(e < 2 ? lo[2 * e + 1] : hi[2 * e - 3]);
        x = x == 0.f || (fabsf(x) >= 0x1p-100f && fabsf(x) < 0x1p20f) ? x : __builtin_nanf("");
        y = y == 0.f || (fabsf(y) >= 0x1p-100f && fabsf(y) < 0x1p20f) ? y : __builtin_nanf("");
#pragma unroll
        for (int p = 0; p < 3; p++) {
            part[p][e] = pack_bf16x2(x, y);
            x -= bf16lo(part[p][e]);
            y -= bf16hi(part[p][e]);
        }
    }
#pragma unroll
    for (int p = 0; p < 3; p++)
        *reinterpret_cast<u32x4 *>(packed + packed_block(n / 16, kt, nk, p) + (n & 15) * 64 + ((q ^ (n >> 2 & 3)) << 4)) = part[p];
}

// The walk over the tiles is that of linear_dma_kernel: m-tile t on XCD t % 8, n-fastest inside an XCD.
template <int BM, int BN, int WGM, int WGN, int NWP, int NSTAGE, int ACT, bool HAS_BIAS, bool HAS_RES>
__global__ __launch_bounds__((WGM * WGN + NWP) * 64) void linear_dma_split_kernel(
    const float *__restrict__ A, int64_t lda, const float *__restrict__ Wt, const unsigned char *__restrict__ packed,
    const float *__restrict__ bias, const float *__restrict__ res, int64_t ldr, float *__restrict__ out, int64_t ldo,
    const int64_t *__restrict__ rows_dev, int64_t rows, int N, int K)
{
    constexpr int NWC = WGM * WGN;                   // MFMA waves
    constexpr int TM = BM / WGM, TN = BN / WGN;      // wave tile
    constexpr int IM = TM / 32, JN = TN / 32;        // 32x32 blocks per wave
    constexpr int STAGE_A = BM * DKB, PLANE = BN * 64, STAGE = STAGE_A + 3 * PLANE;
    constexpr int NLA = BM / 8 / NWP, NLB = 3 * BN / 16 / NWP, NLW = NLA + NLB;      // direct loads per loader wave and stage
    static_assert(BM % (8 * NWP) == 0 && (3 * BN / 16) % NWP == 0 && TM % 32 == 0 && TN % 32 == 0, "tile shape");
    static_assert((NSTAGE - 2) * NLW < 64, "6-bit vmcnt");

    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

    const int64_t M = live_rows(rows_dev, rows);
    const int tiles_n = N / BN;
    const int tiles_m = (int)((M + BM - 1) / BM);
    const int xcd = blockIdx.x & 7, wg = blockIdx.x >> 3, nwg = gridDim.x >> 3;
    const int mt_x = tiles_m > xcd ? (tiles_m - xcd + 7) / 8 : 0;
    const int U = mt_x * tiles_n;
    const int nt = U > wg ? (U - wg + nwg - 1) / nwg : 0;
    if (nt == 0) return;
    const int nk = K / 32;
    const int G = nt * nk;                           // stages this workgroup consumes

    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;

    if (wid >= NWC) {
        // ------------------------------------------------------------------ loader waves
        const int lw = wid - NWC;
        const unsigned char *src[NLA], *wsrc[NLB];
        auto set_tile = [&](int k) {
            const int u = wg + k * nwg;
            const int64_t m0 = (int64_t)((u / tiles_n) * 8 + xcd) * BM;
            const int n0 = (u % tiles_n) * BN;
#pragma unroll
            for (int i = 0; i < NLA; i++) {
                const int r = (lw * NLA + i) * 8 + (lane >> 3);
                const int chunk = (lane & 7) ^ ((r >> 1) & 7);
                int64_t gm = m0 + r;
                gm = gm < M ? gm : M - 1;
                src[i] = reinterpret_cast<const unsigned char *>(A + gm * lda) + chunk * 16;
            }
#pragma unroll
            for (int i = 0; i < NLB; i++) {
                const int b = lw * NLB + i, p = b / (BN / 16);       // plane and block of 16 rows
                wsrc[i] = packed + packed_block(n0 / 16 + b % (BN / 16), 0, nk, p) + lane * 16;
            }
        };
        int it_tile = 0, it_kt = 0, issued = 0;
        set_tile(0);
        auto issue_next = [&]() {
            unsigned char *dst = smem + (issued % NSTAGE) * STAGE;
#pragma unroll
            for (int i = 0; i < NLA; i++) VT_GLOBAL_TO_LDS(src[i] + (int64_t)it_kt * DKB, dst + (lw * NLA + i) * 1024);
#pragma unroll
            for (int i = 0; i < NLB; i++)
                VT_GLOBAL_TO_LDS(wsrc[i] + (int64_t)it_kt * 3072, dst + STAGE_A + (lw * NLB + i) * 1024);
            issued++;
            if (++it_kt == nk) {
                it_kt = 0;
                if (++it_tile < nt) set_tile(it_tile);
            }
        };
#pragma unroll
        for (int i = 0; i < NSTAGE - 1; i++)
            if (issued < G) issue_next();
        for (int g = 0; g < G; g++) {
            // stage g has landed once at most the loads of the younger stages in flight are outstanding
            if (G - 1 - g >= NSTAGE - 2) wait_vmcnt<(NSTAGE - 2) * NLW>();
            else wait_vmcnt<0>();
            block_barrier();                         // stage g visible to the MFMA waves; slot of g-1 is free
            if (issued < G) issue_next();            // stage g + NSTAGE - 1
        }
        block_barrier();                             // the MFMA waves look one stage past the end (and use nothing of it)
        return;
    }

    // ---------------------------------------------------------------------- MFMA waves
    const int wm = wid / WGN, wn = wid % WGN;
    const int lr = lane & 31, lg = lane >> 5;
    int cs[4];
#pragma unroll
    for (int s = 0; s < 4; s++) cs[s] = (wm * TM + lr) * DKB + ((2 * s + lg) ^ ((lr >> 1) & 7)) * 16;
    int ws[2];
#pragma unroll
    for (int t = 0; t < 2; t++) ws[t] = STAGE_A + (wn * TN + lr) * 64 + ((2 * t + lg) ^ ((lr >> 2) & 3)) * 16;

    f32x16 acc[IM][JN];
#pragma unroll
    for (int i = 0; i < IM; i++)
#pragma unroll
        for (int j = 0; j < JN; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[i][j][v] = 0.f;

    float raw[IM][8];                   // A of the next step as read, then what is left of it to split
    u32x4 pa[2][IM][3], pw[2][JN][3];   // the split operands of this step and of the next
    auto read_step = [&](const unsigned char *st, int t) {
#pragma unroll
        for (int i = 0; i < IM; i++)
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const u32x4 r = *reinterpret_cast<const u32x4 *>(st + cs[2 * t + h] + i * 32 * DKB);
#pragma unroll
                for (int e = 0; e < 4; e++) raw[i][4 * h + e] = __uint_as_float(r[e]);
            }
#pragma unroll
        for (int p = 0; p < 3; p++)
#pragma unroll
            for (int j = 0; j < JN; j++) pw[t][j][p] = *reinterpret_cast<const u32x4 *>(st + ws[t] + p * PLANE + j * 32 * 64);
    };
    // One of the 28 small steps in which a fragment's four pairs of values are split, the four pairs in turn so that what
    // depends on each other lies apart: convert, widen the halves, subtract, twice over, and convert what is left.
    uint32_t wide[IM][4][2];
    auto split_part = [&](int t, int m) {
        const int i = m / 28, what = m % 28 / 4, e = m % 4;
        float &x = raw[i][2 * e], &y = raw[i][2 * e + 1];
        if (what % 3 == 0) {
            pa[t][i][what / 3][e] = pack_bf16x2(x, y);
        } else if (what % 3 == 1) {
            wide[i][e][0] = pa[t][i][what / 3][e] << 16;
            wide[i][e][1] = pa[t][i][what / 3][e] & 0xffff0000u;
        } else {
            x -= __uint_as_float(wide[i][e][0]);
            y -= __uint_as_float(wide[i][e][1]);
        }
    };
    constexpr int PARTS = 28 * IM, NM = 6 * IM * JN, FIRST = NM / 4;
    // The products of step t, the small ones first and the blocks in turn; between them, from the FIRST on (the values are on
    // their way out of LDS before), the split of the other step.  Held in this order: left to itself the compiler puts the
    // vector instructions behind the matrix instructions, and the two times add up.
    auto multiply_and_split = [&](auto t_c) {
        constexpr int t = decltype(t_c)::value;
        constexpr int PA[6] = {2, 0, 1, 1, 0, 0}, PW[6] = {0, 2, 1, 0, 1, 0};
        static_for<NM>([&](auto x_c) {
            constexpr int x = decltype(x_c)::value, pr = x / (IM * JN), i = x / JN % IM, j = x % JN;
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, pw[t][j][PW[pr]]),
                                                                __builtin_bit_cast(bf16x8, pa[t][i][PA[pr]]), acc[i][j], 0, 0, 0);
            if constexpr (x >= FIRST) {
                constexpr int from = PARTS * (x - FIRST) / (NM - FIRST), to = PARTS * (x + 1 - FIRST) / (NM - FIRST);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int m = from; m < to; m++) split_part(t ^ 1, m);
                __builtin_amdgcn_sched_barrier(0);
            }
        });
    };

    auto epilogue = [&](int tk) {
        const int u = wg + tk * nwg;
        const int64_t m0 = (int64_t)((u / tiles_n) * 8 + xcd) * BM;
        const int n0 = (u % tiles_n) * BN;
        const int er = fresh(lr), eg = fresh(lg);    // lane constants of the epilogue: not kept in registers in between
#pragma unroll
        for (int i = 0; i < IM; i++) {
            const int64_t row = m0 + wm * TM + i * 32 + er;
#pragma unroll
            for (int j = 0; j < JN; j++) {
                __builtin_amdgcn_sched_barrier(0);
                // acc[i][j][v] = C[row i*32 + lr][col j*32 + 8*(v/4) + 4*lg + v%4]
                u32x4 bv[4], rv[4];
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int col = n0 + wn * TN + j * 32 + 4 * eg + 8 * q;
                    bv[q] = rv[q] = u32x4{0u, 0u, 0u, 0u};
                    if constexpr (HAS_BIAS) bv[q] = *reinterpret_cast<const u32x4 *>(bias + col);
                    if constexpr (HAS_RES)
                        if (row < M) rv[q] = *reinterpret_cast<const u32x4 *>(res + row * ldr + col);
                }
                // a sum that is not finite makes `odd` NaN; a small one that is not zero has the smallest bits, zero the largest
                float odd = 0.f;
                uint32_t small = ~0u;
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    odd = __builtin_fmaf(acc[i][j][v], 0.f, odd);
                    const uint32_t m = 2 * __float_as_uint(acc[i][j][v]) - 1;
                    small = m < small ? m : small;
                }
                if (__any(odd != 0.f || small < (47u << 24) - 1)) {
#pragma unroll
                    for (int v = 0; v < 16; v++) acc[i][j][v] = 0.f;
                    const int64_t ar = row < M ? row : M - 1;
                    const int wr = n0 + wn * TN + j * 32 + er;
                    for (int c = 0; c < nk * 4; c++) {
                        const int chunk = 2 * c + eg;
                        Slab<float>::mma(*reinterpret_cast<const u32x4 *>(Wt + (int64_t)wr * K + 4 * chunk),
                                         *reinterpret_cast<const u32x4 *>(A + ar * lda + 4 * chunk), acc[i][j]);
                    }
                }
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int col = n0 + wn * TN + j * 32 + 4 * eg + 8 * q;
                    float f[4];
#pragma unroll
                    for (int e = 0; e < 4; e++) f[e] = acc[i][j][4 * q + e];
                    if constexpr (HAS_BIAS)
#pragma unroll
                        for (int e = 0; e < 4; e++) f[e] += __uint_as_float(bv[q][e]);
                    if constexpr (ACT == VTDGE_ACT_GELU)
#pragma unroll
                        for (int e = 0; e < 4; e++) f[e] = gelu_fn<float>(f[e]);
                    if constexpr (HAS_RES)
#pragma unroll
                        for (int e = 0; e < 4; e++) f[e] += __uint_as_float(rv[q][e]);
                    if (row < M) *reinterpret_cast<u32x4 *>(out + row * ldo + col) = Elem<float>::pack(f);
                }
#pragma unroll
                for (int v = 0; v < 16; v++) acc[i][j][v] = 0.f;
            }
        }
    };

    // Every step's operands are read and split while the step before is multiplied; the barrier that lets the first step of a
    // stage be read also tells the loaders that all of the stage before has been.
    using std::integral_constant;
    block_barrier();
    const unsigned char *st = smem;
    read_step(st, 0);
#pragma unroll
    for (int m = 0; m < PARTS; m++) split_part(0, m);
    int slot = 0;
    for (int tk = 0; tk < nt; tk++) {
        for (int kt = 0; kt < nk; kt++) {
            read_step(st, 1);
            __builtin_amdgcn_sched_barrier(0);
            multiply_and_split(integral_constant<int, 0>{});
            lds_barrier();
            slot = slot + 1 == NSTAGE ? 0 : slot + 1;
            st = smem + slot * STAGE;
            read_step(st, 0);
            __builtin_amdgcn_sched_barrier(0);
            multiply_and_split(integral_constant<int, 1>{});
        }
        epilogue(tk);
    }
}

// ----------------------------------------------------------------------------- host
template <int BM, int BN, int WGM, int WGN, int NWP, int NSTAGE, int ACT, bool HB, bool HR>
static int go(const float *A, int64_t lda, const float *W, const void *packed, const float *bias, const float *res, int64_t ldr,
              float *out, int64_t ldo, const int64_t *rows_dev, int64_t rows, int N, int K, hipStream_t st)
{
    constexpr size_t lds = (size_t)NSTAGE * (BM * DKB + BN * 192);
    static_assert(lds <= 160 * 1024, "LDS budget");
    constexpr int WGS_PER_CU = lds <= 40 * 1024 ? 4 : lds <= 53 * 1024 ? 3 : lds <= 80 * 1024 ? 2 : 1;
    auto kern = linear_dma_split_kernel<BM, BN, WGM, WGN, NWP, NSTAGE, ACT, HB, HR>;
    VT_RESERVE_LDS(kern, lds, "linear");
    const int64_t tiles_per_xcd = ceil_div(ceil_div(rows, BM), 8) * ceil_div(N, BN);
    int64_t wgs_per_xcd = 32 * WGS_PER_CU;
    if (wgs_per_xcd > tiles_per_xcd) wgs_per_xcd = tiles_per_xcd;
    note_kernel(reinterpret_cast<const void *>(kern));
    kern<<<dim3((unsigned)(wgs_per_xcd * 8)), dim3((WGM * WGN + NWP) * 64), lds, st>>>(
        A, lda, W, (const unsigned char *)packed, bias, res, ldr, out, ldo, rows_dev, rows, N, K);
    return check_launch("linear");
}

int64_t linear_split_size(int N, int K)
{
    return N % 64 == 0 && K % 32 == 0 && (int64_t)N * K < (1ll << 33) ? (int64_t)N * K * 6 : 0;      // pieces in 31 bits
}

int split_linear_weights(const void *const *W, const int32_t *N, const int32_t *K, const int64_t *at, int count, void *split,
                         hipStream_t st)
{
    for (int first = 0; first < count; first += SPLIT_SET) {
        SplitSet set;
        int64_t end = 0;
        set.count = count - first < SPLIT_SET ? count - first : SPLIT_SET;
        for (int j = 0; j < set.count; j++) {
            const int x = first + j;
            set.of[j] = {(const float *)W[x], (unsigned char *)split + at[x], N[x], K[x]};
            end += ceil_div((int64_t)N[x] * K[x] / 8, 256);
            VT_REQUIRE(end < (1ll << 31), VTDGE_ERR_UNSUPPORTED, "linear_split: too many workgroups for one launch");
            set.end[j] = (int)end;
        }
        note_kernel(reinterpret_cast<const void *>(split_weights_kernel));
        split_weights_kernel<<<(unsigned)end, 256, 0, st>>>(set);
        const int rc = check_launch("linear_split");
        if (rc != VTDGE_OK) return rc;
    }
    return VTDGE_OK;
}

int launch_linear_dma_split(const void *A, int64_t lda, const void *W, const void *split, const void *bias, const void *res, int64_t ldr,
                      void *out, int64_t ldo, const int64_t *rows_dev, int64_t rows, int N, int K, int act, hipStream_t st)
{
#define VT_GO(ACT, HB, HR, ...)                                                                                             \
    go<__VA_ARGS__, ACT, HB, HR>((const float *)A, lda, (const float *)W, split, (const float *)bias, (const float *)res,   \
                                 ldr, (float *)out, ldo, rows_dev, rows, N, K, st)
#define VT_PICK(HR, ...)                                                                                                    \
    do {                                                                                                                    \
        if (act == VTDGE_ACT_GELU)                                                                                          \
            return bias ? VT_GO(VTDGE_ACT_GELU, true, HR, __VA_ARGS__) : VT_GO(VTDGE_ACT_GELU, false, HR, __VA_ARGS__);     \
        return bias ? VT_GO(VTDGE_ACT_NONE, true, HR, __VA_ARGS__) : VT_GO(VTDGE_ACT_NONE, false, HR, __VA_ARGS__);         \
    } while (0)
    // 64x64 tiles, two workgroups a compute unit; from some number of tiles on larger ones, whose operands are split for
    // more columns, and with a long K 128x128.  Measured, us (rows live of rows, N, K; the fp32 instructions' 64x64 tiles of
    // linear_dma.hip, 256x128 for the last / 64x64 / 128x64 / 128x128): 32896, 384, 192: 59 / 45 / 40 / 46; 14300 of 32896,
    // 192, 192: 16.5 / 12.2 / 14.2 / 14.6; 768, 192 + GELU: 56 / 45 / 44 / 46; 192, 768: 48 / 33 / 44 / 38; 24000 of 55296,
    // 512, 64 + GELU: 31 / 27.6 / 25.8 / 30; 64, 512: 22.7 / 18.4 / 19.4 / 25; 6000 of 13824, 1024, 128 + GELU: 24.5 / 20.6 /
    // 18.8 / 25; 128, 1024: 23 / 17.7 / 28 / 38; 1500 of 3456, 1280, 320 + GELU: 18 / 13.7 / 20.7 / 20.5; 320, 1280: 27 /
    // 20.3 / 34 / 46; 16448, 768, 384: 100 / 70 / 67 / 70; 7200 of 16448, 1536, 384 + GELU: 96 / 72 / 70 / 65; 384, 1536: 89 /
    // 60 / 80 / 60; 4112, 1536, 768: 95 / 72 / 74 / 64; 1800 of 4112, 3072, 768 + GELU: 88 / 76 / 64 / 69; 768, 3072: 111 /
    // 73 / 76 / 100; 65536, 1536, 384: 637 / 572 / 525 / 477.
    if (res != nullptr) VT_PICK(true, 64, 64, 2, 2, 4, 3);
    if (N % 128 == 0 && K >= 384 && ceil_div(rows, 128) * (N / 128) >= 1024) VT_PICK(false, 128, 128, 2, 2, 4, 3);
    if (ceil_div(rows, 128) * (N / 64) >= 1536) {
        // a short K: waves of 32x64, which split half as many operands a product (14300 of 32896, 768, 192 + GELU: 41.2 on waves
        // of 64x32, 38.0 on these; 24000 of 55296, 512, 64 + GELU: 23.5 / 21.8; 6000 of 13824, 1024, 128 + GELU: 17.2 / 16.7;
        // from K = 384 on the others are even or faster: 7200 of 16448, 1536, 384 + GELU: 59.3 / 62.9)
        if (K <= 256) VT_PICK(false, 128, 64, 4, 1, 4, 2);
        VT_PICK(false, 128, 64, 2, 2, 4, 2);
    }
    VT_PICK(false, 64, 64, 2, 2, 4, 3);
#undef VT_PICK
#undef VT_GO
}

}  // namespace vtdge
