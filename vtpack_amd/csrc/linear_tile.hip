// Packed-M Linear over long rows (bf16, K and N from 768 on: the Linears of the 768-channel models), gfx950.
//
// What bounds it is what a compute unit issues and moves per product.  Four waves, one a SIMD, so that each may hold 128 x 128
// fp32 sums in the 256 accumulation registers: of a 256 x 256 tile a K slab of 64 costs 64 KB of direct loads and 128 KB of LDS
// reads for 2048 clocks of products, where the 128 x 256 tiles of linear_dma.hip take 48 + 128 KB for 1024.  A wave that has its
// SIMD for itself issues a ds_read_b128 or a direct load in about 14 clocks during which no matrix instruction starts unless
// one is running: eight reads in a row cost 108 clocks on top of 512 of products (measured, registers and LDS only), single
// ones between the products nothing.  So fragments of the next step and direct loads go out one at a time between the products,
// across the stages' barriers too (11200 rows, 768, 3072: 72 us with reads and loads in a row, 63 like this).  A normal-valued
// product loop alone, out of registers, runs at 1.65 PFLOP/s here (the clock falls to 1.65 GHz); this kernel reaches 0.93 to
// 1.0 at K = 3072 with 25443 live rows, 0.87 with 11195, and 0.5 to 0.8 at K = 768.
//   * A runs through a ring of three 64-value slabs, W of two (160 KB for 256 x 256), direct loads swizzled as in
//     linear_dma.hip; one barrier a slab, before it a counted wait for this wave's loads of the next one.
//   * An XCD takes an eighth of the rows, in units of 64, and walks the column tiles of a block of rows first.  As many whole
//     rounds of 256 x 256 as its workgroups have go first, the rest in the tile shape that ends first: the live row count is
//     known to the kernel only.
//   * The sums start from the bias; the results leave in 16-byte pieces after half-wave swaps, residuals come a block of rows
//     ahead.
// Launches one behind the other against the tiles of linear_dma.hip (live rows, N, K, us there / here): 25443, 1536, 768: 69.8 /
// 67.8; 25443, 768, 3072 + residual: 158 / 129, 11195: 78.6 / 61.0; 32896, 4096, 1024 + GELU: 346 / 294; 25443, 1024, 4096 + residual:
// 277 / 204.  Which calls take it: linear_tile_wanted below.
#include "common.h"

namespace vtdge {

constexpr int TILE_SLAB = 128;                  // bytes of K a stage
constexpr int TILE_LDS = 160 * 1024;

struct TileArgs {
    const bf16_t *A; int64_t lda; const bf16_t *W; const bf16_t *bias; const bf16_t *res; int64_t ldr;
    bf16_t *out; int64_t ldo; const int64_t *rows_dev; int64_t rows; int N; int K;
};

__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ float acc_read(float a)
{
    float v;
    asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(v) : "a"(a));
    return v;
}

// a direct load of 1 KB to LDS byte `lds` + AT, from a wave-uniform pointer and an offset per lane
template <int AT> __device__ __forceinline__ void dma16_at(const void *base, uint32_t off, uint32_t lds)
{
    asm volatile("s_add_u32 m0, %0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(uniform(lds)), "v"(off),
                 "s"(uniform_ptr(base)), "n"(AT)
                 : "memory", "m0", "scc");
}

// Tiles of 64 IM rows and 64 JN columns: tile t of the list covers rows from row0 + (t / tn) * 64 IM, columns from (t % tn) * 64 JN.
// This workgroup takes tiles first, first + step, ... below `tiles`.
template <int ACT, bool HAS_RES, int IM, int JN, int NA, int NW>
__device__ __forceinline__ void tile_phase(const TileArgs &p, unsigned char *smem, int row0, int rows_end, int tn, int first,
                                           int step, int tiles)
{
    static_assert((NA * 64 * IM + NW * 64 * JN) * TILE_SLAB <= TILE_LDS && (NA == NW || NA == NW + 1), "operand rings");
    if (first >= tiles) return;
    constexpr int A_PART = 64 * IM * TILE_SLAB, W_PART = 64 * JN * TILE_SLAB, W_RING = NA * A_PART;
    constexpr int LA = 2 * IM, LW = 2 * JN;          // direct loads of a wave per stage
    const int nk = p.K / 64;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = uniform(tid >> 6);
    const int wm = wid >> 1, wn = wid & 1;
    const uint32_t lds0 = (uint32_t)(uintptr_t)smem;
    const uint32_t a_lds = lds0 + wid * 8 * TILE_SLAB;
    const int count = uniform((tiles - first + step - 1) / step);

    // ---- direct loads: 8 rows of 128 bytes each; wave w takes rows 8 w .. 8 w + 7 of every 32
    const int lrow = wid * 8 + (lane >> 3);
    const int lchunk = ((lane & 7) ^ ((lrow >> 1) & 7)) * 16;
    const int a_pitch = (int)p.lda * 2, w_pitch = p.K * 2;
    const unsigned char *a_ptr, *w_ptr;
    uint32_t a_off[LA], w_off[LW];              // of a tile's rows, clamped to those there are
    int a_t = first, a_kt = 0, a_slot = 0, w_t = first, w_kt = 0, w_slot = 0;
    auto set_a = [&]() {
        const int r = row0 + uniform(a_t / tn) * (64 * IM);
        a_ptr = reinterpret_cast<const unsigned char *>(p.A + (int64_t)r * p.lda);
#pragma unroll
        for (int d = 0; d < LA; d++) a_off[d] = __umul24(min(d * 32 + lrow, rows_end - 1 - r), a_pitch) + lchunk;
    };
    auto set_w = [&]() {
        const int n0 = (w_t - uniform(w_t / tn) * tn) * (64 * JN);
        w_ptr = reinterpret_cast<const unsigned char *>(p.W + (int64_t)n0 * p.K);
#pragma unroll
        for (int d = 0; d < LW; d++) w_off[d] = __umul24(min(d * 32 + lrow, p.N - 1 - n0), w_pitch) + lchunk;
    };
    auto load_a = [&](auto D) {
        constexpr int d = decltype(D)::value;
        dma16_at<d * 32 * TILE_SLAB>(a_ptr, a_off[d], a_lds + a_slot * A_PART);
    };
    auto load_w = [&](auto D) {
        constexpr int d = decltype(D)::value;
        dma16_at<W_RING + d * 32 * TILE_SLAB>(w_ptr, w_off[d], a_lds + w_slot * W_PART);
    };
    auto next_a = [&]() {
        a_slot = a_slot == NA - 1 ? 0 : a_slot + 1;
        a_ptr += TILE_SLAB;
        if (++a_kt == nk) {
            a_kt = 0;
            a_t += step;
            if (a_t < tiles) set_a();
        }
    };
    auto next_w = [&]() {
        w_slot = w_slot == NW - 1 ? 0 : w_slot + 1;
        w_ptr += TILE_SLAB;
        if (++w_kt == nk) {
            w_kt = 0;
            w_t += step;
            if (w_t < tiles) set_w();
        }
    };
    auto all_a = [&]() {
        if (a_t >= tiles) return;
        static_for<LA>([&](auto D) { load_a(D); });
        next_a();
    };
    auto all_w = [&]() {
        if (w_t >= tiles) return;
        static_for<LW>([&](auto D) { load_w(D); });
        next_w();
    };
    // this wave's loads of a stage have landed when at most those of the `r` stages behind it that exist are outstanding
    auto wait_stage = [&](int r) {
        static_for<NA - 1>([&](auto X) {
            constexpr int x = decltype(X)::value;
            constexpr int n = (x < NW - 2 ? x : NW - 2) * LW + (x < NA - 2 ? x : NA - 2) * LA;
            if (x == NA - 2 ? r >= x : r == x) wait_vmcnt<n>();
        });
    };
    int left = count * nk;                       // stages not yet multiplied
    bool more_w = false, more_a = false;         // whether there is a stage of each to load
    set_a();
    set_w();
    if (NA > NW) all_a();
#pragma unroll
    for (int s = 0; s < NW; s++) {
        all_w();
        all_a();
    }
    // stage 0: one stage more than in the loop is in flight
    if (NW >= 2 && left >= 2) wait_vmcnt<LW + LA>();
    else wait_vmcnt<0>();
    block_barrier();

    const int lr = lane & 31, lg = lane >> 5;
    const int sw = (lr >> 1) & 7;
    int cs[4];
#pragma unroll
    for (int s = 0; s < 4; s++) cs[s] = ((2 * s + lg) ^ sw) * 16;
    int ra = 0, rw = 0;                          // slots read from
    const int a_row = (wm * 32 * IM + lr) * TILE_SLAB, w_row = W_RING + (wn * 32 * JN + lr) * TILE_SLAB;

    for (int t = first; t < tiles; t += step) {
        const int tm = uniform(t / tn);
        const int n0 = (t - tm * tn) * (64 * JN), m0 = row0 + tm * (64 * IM);
        f32x16 acc[IM][JN];
        u32x4 fa[2][IM], fw[2][JN];
        // fragment f of step s: those of W, then those of A
        auto fetch1 = [&](int set, int s, int f) {
            if (f < JN)
                fw[set][f] = *reinterpret_cast<const u32x4 *>(smem + rw * W_PART + w_row + cs[s] + f * 32 * TILE_SLAB);
            else
                fa[set][f - JN] = *reinterpret_cast<const u32x4 *>(smem + ra * A_PART + a_row + cs[s] + (f - JN) * 32 * TILE_SLAB);
        };
        // the products of a step; between them the fragments of the next one and a quarter of a stage's direct loads, one at a
        // time: a wave that has its SIMD for itself issues them while the matrix unit works
        auto multiply = [&](int set, int next, bool more, auto Q) {
            constexpr int q = decltype(Q)::value, LOADS = LW + LA;
            constexpr int d0 = q * LOADS / 4, n = (q + 1) * LOADS / 4 - d0, P = JN * IM, R = JN + IM;
            static_for<P>([&](auto X) {
                constexpr int x = decltype(X)::value;
                Slab<bf16_t>::mma(fw[set][x % JN], fa[set][x / JN], acc[x / JN][x % JN]);
                __builtin_amdgcn_sched_barrier(0);
                static_for<(x + 1) * R / P - x * R / P>([&](auto Y) {
                    if (more) fetch1(set ^ 1, next, x * R / P + decltype(Y)::value);
                });
                __builtin_amdgcn_sched_barrier(0);
                static_for<(x + 1) * n / P - x * n / P>([&](auto Y) {
                    constexpr int d = d0 + x * n / P + decltype(Y)::value;
                    if constexpr (d < LW) {
                        if (more_w) load_w(std::integral_constant<int, d>{});
                    } else {
                        if (more_a) load_a(std::integral_constant<int, d - LW>{});
                    }
                });
                __builtin_amdgcn_sched_barrier(0);
            });
        };
        // the accumulators start from the bias: acc[i][j][v] = C[row i*32 + lr][col j*32 + 8*(v/4) + 4*lg + v%4]
        const int cw = n0 + wn * 32 * JN;
#pragma unroll
        for (int j = 0; j < JN; j++) {
            f32x16 b;
#pragma unroll
            for (int v4 = 0; v4 < 4; v4++) {
                const int col = cw + j * 32 + 8 * v4 + 4 * lg;
                u32x2 w = {0u, 0u};
                if (p.bias != nullptr && col < p.N) w = *reinterpret_cast<const u32x2 *>(p.bias + col);
                b[4 * v4] = bf16lo(w.x);
                b[4 * v4 + 1] = bf16hi(w.x);
                b[4 * v4 + 2] = bf16lo(w.y);
                b[4 * v4 + 3] = bf16hi(w.y);
            }
#pragma unroll
            for (int i = 0; i < IM; i++) acc[i][j] = b;
        }
#pragma unroll
        for (int f = 0; f < JN + IM; f++) fetch1(0, 0, f);
        for (int kt = 0; kt < nk; kt++) {
            static_for<3>([&](auto S) {
                constexpr int st = decltype(S)::value;
                multiply(st & 1, st + 1, true, std::integral_constant<int, st + 1>{});
            });
            if (more_w) next_w();
            if (more_a) next_a();
            // the last fragments are in registers: this stage's slots are free behind the barrier, the next stage is there
            wait_stage(left - 2);
            lds_barrier();
            left--;
            ra = ra == NA - 1 ? 0 : ra + 1;
            rw = rw == NW - 1 ? 0 : rw + 1;
            more_w = w_t < tiles;
            more_a = a_t < tiles;
            multiply(1, 0, kt + 1 < nk, std::integral_constant<int, 0>{});
        }
        // ---- epilogue: half-wave swaps leave a lane 8 consecutive columns
        // (the wait states between a matrix instruction and the reads of its result)
        asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        const int c0 = cw + 8 * lg;
        u32x4 rraw[2][JN][2];                    // the residual of a block of rows, requested a block ahead
        auto read_res = [&](int i) {
            const int row = m0 + wm * 32 * IM + i * 32 + lr;
#pragma unroll
            for (int j = 0; j < JN; j++)
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    const int col = c0 + j * 32 + 16 * q;
                    const u32x4 z = {0u, 0u, 0u, 0u};
                    rraw[i & 1][j][q] = z;
                    if (row < rows_end && col < p.N)
                        rraw[i & 1][j][q] = *reinterpret_cast<const u32x4 *>(p.res + (int64_t)row * p.ldr + col);
                }
        };
        if constexpr (HAS_RES) read_res(0);
#pragma unroll
        for (int i = 0; i < IM; i++) {
            const int row = m0 + wm * 32 * IM + i * 32 + lr;
            const bool in = row < rows_end;
            bf16_t *orow = p.out + (int64_t)row * p.ldo + c0;
            if constexpr (HAS_RES)
                if (i + 1 < IM) read_res(i + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < JN; j++)
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    float f[8];
#pragma unroll
                    for (int e = 0; e < 8; e++) f[e] = acc_read(acc[i][j][8 * q + e]);
                    if constexpr (ACT == VTDGE_ACT_GELU) {
#pragma unroll
                        for (int e = 0; e < 8; e++) f[e] = gelu_fn<bf16_t>(f[e]);
                    }
                    if constexpr (HAS_RES) {
                        // the residual's vector back to the accumulators' columns
                        const auto r0 = __builtin_amdgcn_permlane32_swap(rraw[i & 1][j][q].x, rraw[i & 1][j][q].z, false, false);
                        const auto r1 = __builtin_amdgcn_permlane32_swap(rraw[i & 1][j][q].y, rraw[i & 1][j][q].w, false, false);
                        f[0] += bf16lo(r0[0]);
                        f[1] += bf16hi(r0[0]);
                        f[2] += bf16lo(r1[0]);
                        f[3] += bf16hi(r1[0]);
                        f[4] += bf16lo(r0[1]);
                        f[5] += bf16hi(r0[1]);
                        f[6] += bf16lo(r1[1]);
                        f[7] += bf16hi(r1[1]);
                    }
                    const auto s0 = __builtin_amdgcn_permlane32_swap(pack_bf16x2(f[0], f[1]), pack_bf16x2(f[4], f[5]),
                                                                     false, false);
                    const auto s1 = __builtin_amdgcn_permlane32_swap(pack_bf16x2(f[2], f[3]), pack_bf16x2(f[6], f[7]),
                                                                     false, false);
                    const u32x4 o = {s0[0], s1[0], s0[1], s1[1]};
                    if (in && c0 + j * 32 + 16 * q < p.N) *reinterpret_cast<u32x4 *>(orow + j * 32 + 16 * q) = o;
                    __builtin_amdgcn_sched_barrier(0);
                }
        }
    }
}

template <int ACT, bool HAS_RES>
__global__ __launch_bounds__(256, 1) void linear_tile_kernel(TileArgs p)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int64_t live = live_rows(p.rows_dev, p.rows);
    const int M = uniform(live > 0 ? (int)live : 0);
    const int units = (M + 63) >> 6;
    const int xcd = blockIdx.x & 7, wg = blockIdx.x >> 3, nwg = gridDim.x >> 3;
    const int tn = (p.N + 255) / 256;
    const int u0 = (int)((int64_t)units * xcd >> 3), u1 = (int)((int64_t)units * (xcd + 1) >> 3);
    const int rows_end = u1 * 64 < M ? u1 * 64 : M;
    const int u = u1 - u0;
    const int full = uniform(u * tn / (nwg * 4));
    const int nb = uniform(full * nwg / tn);
    const int left = u - 4 * nb, spare = full * nwg - nb * tn;
    // the rest in the tiles that end first: 4, 3, 2 or 1 units of rows by 256 columns, 2 or 1 by 128.  What a round of each
    // takes per slab of K, in hundredths of a microsecond, was measured at K = 3072.
    int best = 0x7fffffff, tail = 0, shape = 0;
    for (int h = 0; h < 6; h++) {
        const int im = h < 4 ? 4 - h : h == 4 ? 2 : 1, cols = h < 4 ? tn : (p.N + 127) / 128;
        const int tiles = uniform((left + im - 1) / im) * cols;
        const int more = tiles > spare ? uniform((tiles - spare + nwg - 1) / nwg) : 0;
        const int cost = more * (h == 0 ? 151 : h == 1 ? 119 : h == 2 ? 89 : h == 3 ? 64 : h == 4 ? 55 : 42);
        if (cost < best) best = cost, shape = h, tail = tiles;
    }
    // the rest starts with the workgroups that the last round of large tiles has left out
    int tail_first = wg - (nb * tn - uniform(nb * tn / nwg) * nwg);
    if (tail_first < 0) tail_first += nwg;
    const int tail_row = (u0 + 4 * nb) * 64, cols = shape < 4 ? tn : (p.N + 127) / 128;
    tile_phase<ACT, HAS_RES, 4, 4, 3, 2>(p, smem, u0 * 64, rows_end, tn, wg, nwg, nb * tn);
    block_barrier();
#define VT_REST(...) tile_phase<ACT, HAS_RES, __VA_ARGS__>(p, smem, tail_row, rows_end, cols, tail_first, nwg, tail)
    if (shape == 0) VT_REST(4, 4, 3, 2);
    else if (shape == 1) VT_REST(3, 4, 3, 2);
    else if (shape == 2) VT_REST(2, 4, 3, 3);
    else if (shape == 3) VT_REST(1, 4, 4, 4);
    else if (shape == 4) VT_REST(2, 2, 4, 4);
    else VT_REST(1, 2, 4, 4);
#undef VT_REST
}

template <int ACT, bool HAS_RES> static int go_tile(const TileArgs &a, hipStream_t st)
{
    auto kern = linear_tile_kernel<ACT, HAS_RES>;
    VT_RESERVE_LDS(kern, TILE_LDS, "linear");
    note_kernel(reinterpret_cast<const void *>(kern));
    kern<<<256, 256, TILE_LDS, st>>>(a);
    return check_launch("linear");
}

// Which products the kernel is taken for (beyond what linear_dma_applicable asks and linear_small_wanted leaves).  Shorter rows
// and narrower outputs leave its tiles few slabs and many epilogues: 28000, 1280, 320 + GELU: 48.0 / 49.4 us (linear_dma.hip /
// here) with all rows live, 23.6 / 30.5 with 0.44 of them; 16640, 2048, 512 + GELU: 57.4 / 52.3 and 25.8 / 25.8; 16640, 512,
// 2048: 58.1 / 47.0 and 22.5 / 24.6; 32896, 768, 192 + GELU: 23.7 / 30.5.
// From 768 on, us of a launch inside a pass of the 768-channel model (256 px pictures of 257 rows, the mean of its blocks, whose
// live rows are about 7 in 16), linear_dma.hip / here, at 8, 20, 44, 64, 99 and 128 pictures:
//   keys and values (1536, 768, all rows live): 16.9 / 14.3, 25.1 / 22.7, 43.9 / 37.7, 55.2 / 49.0, 75.7 / 71.0, 98.4 / 89.8; 16: 18.7 / 19.3
//   queries (768, 768):             10.0 / 9.7, 10.6 / 10.4, 16.8 / 13.8, 18.3 / 16.6, 24.7 / 21.4, 28.1 / 25.0; 40: 13.3 / 13.4
//   proj (768, 768 + residual):     10.6 / 10.9, 11.2 / 11.8, 15.2 / 16.6, 17.4 / 19.8, 25.2 / 27.3, 30.2 / 32.2
//   fc1 (3072, 768 + GELU):         13.6 / 15.1, 23.4 / 22.7, 36.4 / 36.6, 44.6 / 46.2, 64.4 / 68.0, 79.6 / 84.0
//   fc2 (768, 3072 + residual):     26.3 / 25.1, 28.8 / 26.8, 39.9 / 37.4, 46.0 / 44.3, 67.5 / 59.3, 80.6 / 71.0; 32: 31.3 / 31.6
// These are of a card that rests between a few passes; one that runs without a rest lowers its clock, by less for the fewer
// instructions and loads of this kernel, and fc1 is ahead here too then.  A pass without a rest, us: without this kernel / with it wherever K and N
// allow / without proj and fc1 / without proj, which is the rule: 10 pictures: 1396 / 1386 / 1379 / 1395; 28: 2018 / 1965 / 1975 /
// 1953; 48: 2758 / 2670 / 2702 / 2664; 64: 3257 / 3138 / 3172 / 3133; 80: 3819 / 3743 / 3779 / 3725; 99: 4560 / 4418 / 4429 / 4403; 128: 5630 /
// 5402 / 5360 / 5373.
// What the rule costs: with 2000 to 4700 rows of 768 and about 7 in 16 live, proj here as well takes 0.5 to 1 percent off a pass (one
// model, builds in turn; 12 pictures 1497 / 1487, three of 512 px 1607 / 1595), and from 5100 rows on it adds as much (28 pictures
// 1892 / 1900).  But where a router keeps every row it adds 1 to 2 percent from 2570 rows on (12 pictures 1808 / 1844), and queries
// here as well 1 more (1857); the host does not know how many rows live, so that the rule takes the smaller loss.
// Against a pass without this kernel, at 6168 to 12336 rows and 7 in 16, all or only the coarse ones live (48 passes): level or up to 11
// percent faster, but for one in the band below (16 pictures of 384 px, 2297 / 2265 without), where fc2 elsewhere adds 2 percent if
// every row lives.
// Where the 128x128 tiles of linear_dma.hip fill the chip once at most and 64x128 here do not, long K lose a fifth (4000 live rows of
// 768, 3072: 27.1 / 32.7).  With all rows live outputs of 2 to 4 M values lie in that band altogether and are left out.  Packed rows
// are taken: blocks of routed samples only touch it (12 to 20 pictures, a pass: 1539 / 1499 to 1723 / 1695), a router that
// keeps every row - an untrained one - loses about 3 percent of a pass there.  Left out are also keys and values of 5 to
// 7.5 M, where 128x128 tiles there are one and a half rounds.  Wider K, launches one behind the other: 4096, 1024 + GELU: 0.91 of
// linear_dma.hip on average over 28 sizes with a quarter to all rows live, 2048, 1024 and 3072, 1536 0.91 and 0.88.
bool linear_tile_wanted(int64_t lda, bool packed, int64_t rows, int N, int K, int act, const void *res)
{
    if (rows < 2048 || N < 768 || K < 768 || K % 64 != 0 || (act != VTDGE_ACT_NONE && res != nullptr) || rows >= (1ll << 30) ||
        lda >= (1 << 23) || K >= (1 << 23) || compute_units() != 256)      // its rounds are counted for a workgroup on each of 256
        return false;
    if (res != nullptr && K < 1536) return false;
    const int64_t out = rows * N, M = 1 << 20;
    if (N < 1536 || K >= 2048 || res != nullptr)                           // 128x128 tiles there
        return K >= 1536 ? packed || out <= 2 * M || out > 4 * M : out >= 8 * M;
    return act != VTDGE_ACT_NONE || K >= 1024 || out <= 5 * M || out > 7 * M + M / 2;
}

int launch_linear_tile(const void *A, int64_t lda, const void *W, const void *bias, const void *res, int64_t ldr, void *out,
                       int64_t ldo, const int64_t *rows_dev, int64_t rows, int N, int K, int act, hipStream_t st)
{
    const TileArgs a{(const bf16_t *)A, lda, (const bf16_t *)W, (const bf16_t *)bias, (const bf16_t *)res, ldr, (bf16_t *)out,
                     ldo, rows_dev, rows, N, K};
    if (act == VTDGE_ACT_GELU) return go_tile<VTDGE_ACT_GELU, false>(a, st);
    if (res != nullptr) return go_tile<VTDGE_ACT_NONE, true>(a, st);
    return go_tile<VTDGE_ACT_NONE, false>(a, st);
}

}  // namespace vtdge
