// Single fp32 products in bf16 terms (bf16x3.h) whose operands are cut once: a first launch writes both operands as planes of terms in the
// order in which the matrix core reads them, a second one multiplies planes and nothing else.
//
// The staged tiles (gemm_staged.hip) cut a value again in every tile that reads it: 2000 x 4096 x 1024 takes 133 M cuts for 6.2 M values, beside which the
// matrix core is busy 49 % of the cycles.  Here a value is cut once (2000 x 4096 x 1024: 11 us, 25 MB read and 37 written, the rate of a copy), and what is
// left is what the int8 kernels do: loads straight to LDS, reads of whole fragments without a bank conflict, products; no vector instruction in the loop.
// v_mfma_f32_16x16x32_bf16, not 32x32x16: its accumulators are read and written half as often, and at full load the matrix core runs into the
// power cap (2000 x 4096 x 1024 the product alone 80 -> 72 us, 1.4 PFLOP/s of bf16 products; with 64 of 256 CUs at work it is at 87 % of the peak).
// us, staged tiles -> this, both launches, back to back, on one card: 2000 x 4096 x 1024 105 -> 85, 2000 x 3072 x 1024 98 -> 79, 2048 x 4096 x 4096 366 -> 311, A B^T
// 2112 x 2432 x 2403 192 -> 157, A^T B 1288 x 3985 x 767 85 -> 65.
// Bound: 256x128 tiles, power with every CU at work (zeros for operands 65 and 224 us in place of 82 and 288 at 2000 x 4096 x 1024 and 2048 x 4096 x 4096; the matrix core is busy 63 and 81 % of
// the cycles); 128x64 ones, what L2 hands to the CUs (36 KiB per tile and 32 k: 2000 x 3072 x 1024 906 MB in 59 us, 15.4 TB/s, 936 MB by its counter, the matrix core busy 51 %;
// the same rate where A's fragments go to registers without LDS, where sets of waves share K, and with a ring of four stages), and power too (zeros 62 in place of 75).
// Measured and dropped: four waves of 128x64 on a 256x128 tile (one wave a SIMD leaves its waits bare: 72 -> 92), 128x128 on four waves (86), and for one
// 128x64 tile a CU two sets of waves over K, or fragments of A straight to registers (2000 x 1024 x 4096 98 and 117 where the staged tiles take 104).
#include "gemm_planes.h"

#include "bf16x3.h"

namespace {
using namespace axhip;

// ---- planes ----------------------------------------------------------------------------------------------------------
// An operand of `rows` rows (of A, columns of B) and K: blocks of 16 rows x 32 k, the blocks of 16 rows one after another along k, each as
// its three terms, a term as the 64 x 16 bytes of a matrix instruction's operand: lane l holds row l & 15, k = 8 (l >> 4) + 0..7.
// Rows and k past the end are zero.
constexpr int BLOCK = 3 * 1024;

struct CutSide {
    const float *x;
    unsigned char *out;
    int64_t rows, ld;
    int across;          // stored across k: element (row, k) at k * ld + row
    int blocks;          // of 16 rows
};

// A wave cuts four blocks: of an operand stored along k, four along k; of one stored across it, two by two, so that its loads are 128 bytes long.
__device__ __forceinline__ void cut_along(const CutSide &s, int64_t K, int kblocks, int rb, int kb0, int lane) {
    const int64_t row = (int64_t)rb * 16 + (lane & 15), at = row < s.rows ? row : s.rows - 1;
    float x[4][8];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int64_t k = (int64_t)(kb0 + q) * 32 + 8 * (lane >> 4);
        if (k + 8 <= K) __builtin_memcpy(x[q], s.x + at * s.ld + k, 32);
        else {
#pragma unroll
            for (int e = 0; e < 8; e++) x[q][e] = k + e < K ? s.x[at * s.ld + k + e] : 0.0f;
        }
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
        if (kb0 + q >= kblocks) break;
        if (row >= s.rows) {
#pragma unroll
            for (int e = 0; e < 8; e++) x[q][e] = 0.0f;
        }
        v4i t[3];
        cut(x[q], TERMS_UP, t);
        unsigned char *d = s.out + ((int64_t)rb * kblocks + kb0 + q) * BLOCK + lane * 16;
#pragma unroll
        for (int p = 0; p < 3; p++) *reinterpret_cast<v4i *>(d + p * 1024) = t[p];
    }
}
__device__ __forceinline__ void cut_across(const CutSide &s, int64_t K, int kblocks, int rb, int kb0, int lane) {
    const int c = lane & 31, kh = lane >> 5, mine = rb + (c >> 4);      // this lane's block of rows; its half of 32 k
    const int64_t row = (int64_t)rb * 16 + c, at = row < s.rows ? row : s.rows - 1;
    float x[2][2][8];
#pragma unroll
    for (int q = 0; q < 2; q++)
#pragma unroll
        for (int e = 0; e < 16; e++) {
            const int64_t k = (int64_t)(kb0 + q) * 32 + 16 * kh + e;
            x[q][e >> 3][e & 7] = s.x[(k < K ? k : K - 1) * s.ld + at];
            if (k >= K || row >= s.rows) x[q][e >> 3][e & 7] = 0.0f;
        }
#pragma unroll
    for (int q = 0; q < 2; q++)
#pragma unroll
        for (int half = 0; half < 2; half++) {
            if (kb0 + q >= kblocks || mine >= s.blocks) continue;
            v4i t[3];
            cut(x[q][half], TERMS_UP, t);
            unsigned char *d = s.out + ((int64_t)mine * kblocks + kb0 + q) * BLOCK + ((c & 15) + 16 * (2 * kh + half)) * 16;
#pragma unroll
            for (int p = 0; p < 3; p++) *reinterpret_cast<v4i *>(d + p * 1024) = t[p];
        }
}
// workgroups of an operand: 16 rows and 16 blocks of k, or 32 rows and 8
__host__ __device__ constexpr int cut_groups(int across, int blocks, int kblocks) {
    return across ? (blocks + 1) / 2 * ((kblocks + 7) / 8) : blocks * ((kblocks + 15) / 16);
}
__global__ void __launch_bounds__(256) k_cut_planes(CutSide a, CutSide b, int64_t K, int kblocks) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int first = cut_groups(a.across, a.blocks, kblocks);
    const bool second = (int)blockIdx.x >= first;
    const int id = second ? blockIdx.x - first : blockIdx.x;
    const CutSide &s = second ? b : a;
    if (s.across) {                                  // neighbours along the rows share lines
        const int pairs = (s.blocks + 1) / 2, run = id / pairs, kb0 = run * 8 + wave * 2;
        if (kb0 < kblocks) cut_across(s, K, kblocks, (id - run * pairs) * 2, kb0, lane);
    } else {
        const int runs = (kblocks + 15) / 16, rb = id / runs, kb0 = (id - rb * runs) * 16 + wave * 4;
        if (kb0 < kblocks) cut_along(s, K, kblocks, rb, kb0, lane);
    }
}

// ---- the product -----------------------------------------------------------------------------------------------------
struct PlanesArgs {
    StagedArgs g;
    const unsigned char *a, *b;
    int a_blocks, b_blocks, kblocks;
};

__device__ __forceinline__ void load_lds(unsigned lds_at, unsigned offset, const unsigned char *base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_at), "v"(offset), "s"(base) : "memory");
}

__device__ __forceinline__ v4f mfma16(const v4i &a, const v4i &b, const v4f &c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
}

// WM x WN waves of TI x TJ blocks of 16 x 16 each; two stages of 32 k.
template <int WM, int WN, int TI, int TJ>
struct Tile {
    static constexpr int WAVES = WM * WN, BM = 16 * TI * WM, BN = 16 * TJ * WN, RA = BM / 16, RB = BN / 16;
    static constexpr int A_BYTES = RA * BLOCK, STAGE = (RA + RB) * BLOCK;
    static constexpr int PIECES = STAGE / 1024, MINE = PIECES / WAVES;    // loads of a stage, of a wave
    static_assert(PIECES % WAVES == 0 && WAVES % 4 == 0, "loads of a stage");
    static_assert(TI % 2 == 0 && TJ % 2 == 0, "written back in blocks of 32 x 32");
    static constexpr int WORDS = 2 * STAGE, SMEM = WORDS + 4 * WAVES;
    static_assert(WAVES * 4096 <= WORDS && SMEM <= 160 * 1024, "LDS budget");
};

// TURNS: the large products of neighbouring stages go into two sums.
template <int WM, int WN, int TI, int TJ, bool TURNS, bool A_KC, bool B_KC>
__global__ void __launch_bounds__(64 * WM * WN, 2) k_gemm_planes(PlanesArgs p) {
    using T = Tile<WM, WN, TI, TJ>;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const StagedArgs &g = p.g;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN;
    int tm, tn;
    tile_of_block(blockIdx.x, (int)((g.M + T::BM - 1) / T::BM), (int)((g.N + T::BN - 1) / T::BN), tm, tn);
    const int64_t m0 = (int64_t)tm * T::BM + wm * 16 * TI, n0 = (int64_t)tn * T::BN + wn * 16 * TJ;      // of the wave
    const int steps = p.kblocks;

    // ---- planes -> LDS: piece q of a stage is 1 KiB of one block of rows; a block of rows that does not exist reads the last one ----
    const unsigned lds0 = (unsigned)(uintptr_t)lds;
    const unsigned char *from[T::MINE];
#pragma unroll
    for (int j = 0; j < T::MINE; j++) {
        const int q = j * T::WAVES + wave, rb = q / 3, rem = q % 3;
        const bool is_a = rb < T::RA;
        const int64_t block = is_a ? (int64_t)tm * T::RA + rb : (int64_t)tn * T::RB + rb - T::RA;
        const int64_t last = (is_a ? p.a_blocks : p.b_blocks) - 1;
        from[j] = (is_a ? p.a : p.b) + (block < last ? block : last) * p.kblocks * BLOCK + rem * 1024;
    }
    const unsigned lane16 = lane * 16;
    auto stage_at = [&](int s) { return (int64_t)(s < steps ? s : steps - 1) * BLOCK; };
    auto issue_one = [&](int j, int64_t at, unsigned to) { load_lds(to + (j * T::WAVES + wave) * 1024, lane16, from[j] + at); };

    // ---- LDS -> fragments -> products ----
    const unsigned char *fa = lds + wm * TI * BLOCK + lane16, *fb = lds + T::A_BYTES + wn * TJ * BLOCK + lane16;
    struct FragsA {
        v4i x[TI];
    };
    struct FragsB {
        v4i x[TJ];
    };
    auto read_one = [&](auto &f, const unsigned char *from, unsigned at, int t, int i) {
        f.x[i] = *reinterpret_cast<const v4i *>(from + at + i * BLOCK + t * 1024);
    };
    v4f acc[TI][TJ], low[TI][TJ], other[TURNS ? TI : 1][TURNS ? TJ : 1];
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
        for (int j = 0; j < TJ; j++) {
            acc[i][j] = low[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
            if constexpr (TURNS) other[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
        }
    // the products of the wave's blocks of A and of B (in a serpentine: neighbours share an operand), with `between(n)` after each
    constexpr int NP = TI * TJ;
    auto products = [&](const FragsA &a, const FragsB &b, v4f (&to)[TI][TJ], auto between) {
#pragma unroll
        for (int n = 0; n < NP; n++) {
            const int i = n / TJ, j = (i & 1) ? TJ - 1 - n % TJ : n % TJ;
            to[i][j] = mfma16(b.x[j], a.x[i], to[i][j]);
            __builtin_amdgcn_sched_barrier(0);
            between(n);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // One stage.  a2 and b0 are in registers; the fragments of the next products are read during those before them.
    auto step = [&](int s, unsigned at, const FragsA &a2, const FragsB &b0, FragsA &a2_next, FragsB &b0_next, v4f (&large)[TI][TJ]) {
        const unsigned after = T::STAGE - at;
        const int64_t mem = stage_at(s + 2);
        FragsA a1, a0;
        FragsB b1, b2;
        auto every_other = [&](int n, int count) { return !(n & 1) && n < 2 * count; };
        products(a2, b0, low, [&](int n) { if (every_other(n, TI)) read_one(a1, fa, at, 1, n >> 1); });
        products(a1, b0, low, [&](int n) { if (every_other(n, TJ)) read_one(b1, fb, at, 1, n >> 1); });
        products(a1, b1, low, [&](int n) { if (every_other(n, TI)) read_one(a0, fa, at, 0, n >> 1); });
        products(a0, b1, low, [&](int n) { if (every_other(n, TJ)) read_one(b2, fb, at, 2, n >> 1); });
        // the next stage has arrived for every wave, and every wave has read this one
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        constexpr int HALF = (T::MINE + 1) / 2;
        products(a0, b2, low, [&](int n) {
            if (every_other(n, TI)) read_one(a2_next, fa, after, 2, n >> 1);
            if (NP - 1 - n < HALF) issue_one(n - (NP - HALF), mem, lds0 + at);
        });
        products(a0, b0, large, [&](int n) {
            if (every_other(n, TJ)) read_one(b0_next, fb, after, 0, n >> 1);
            if (n >= NP - (T::MINE - HALF)) issue_one(HALF + n - (NP - (T::MINE - HALF)), mem, lds0 + at);
        });
    };
    static_assert((T::MINE + 1) / 2 <= NP, "a load after a product");
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
        for (int j = 0; j < T::MINE; j++) issue_one(j, stage_at(s), lds0 + s * T::STAGE);
    asm volatile("s_waitcnt vmcnt(%0)" ::"i"(T::MINE) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    FragsA a2, a2_other;
    FragsB b0, b0_other;
#pragma unroll
    for (int i = 0; i < TI; i++) read_one(a2, fa, 0, 2, i);
#pragma unroll
    for (int i = 0; i < TJ; i++) read_one(b0, fb, 0, 0, i);
    int s = 0;
    auto &second = [&]() -> v4f (&)[TI][TJ] {
        if constexpr (TURNS) return other;
        else return acc;
    }();
    for (; s + 2 <= steps; s += 2) {
        step(s, 0, a2, b0, a2_other, b0_other, acc);
        step(s + 1, T::STAGE, a2_other, b0_other, a2, b0, second);
    }
    if (s < steps) step(s, 0, a2, b0, a2_other, b0_other, acc);
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");       // loads past the last stage still write the buffers

    // ---- finite?  else again with fp32 instructions, straight from memory ----
    float seen = 0.0f;
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
        for (int j = 0; j < TJ; j++) {
            if constexpr (TURNS) acc[i][j] += other[i][j];
            acc[i][j] += low[i][j];
#pragma unroll
            for (int v = 0; v < 4; v++) seen = __builtin_fmaf(acc[i][j][v], 0.0f, seen);
        }
    const int r16 = lane & 15, h = lane >> 4;
    if (any_wave<T::WAVES>(!(seen == 0.0f), lds + T::WORDS, wave)) {
        const float *a[TI], *b[TJ];
#pragma unroll
        for (int i = 0; i < TI; i++) {
            const int64_t row = m0 + i * 16 + r16, at = row < g.M ? row : g.M - 1;
            a[i] = static_cast<const float *>(g.A) + (A_KC ? at * g.lda : at);
        }
#pragma unroll
        for (int j = 0; j < TJ; j++) {
            const int64_t col = n0 + j * 16 + r16, at = col < g.N ? col : g.N - 1;
            b[j] = static_cast<const float *>(g.B) + (B_KC ? at * g.ldb : at);
        }
#pragma unroll
        for (int i = 0; i < TI; i++)
#pragma unroll
            for (int j = 0; j < TJ; j++) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
        // 16 k at a time, those of lane group h: 4 h + e.  (Not the next ones meanwhile: two sets of operands beside the sums would not fit the registers, and what is
        // kept in memory for this rare pass is stored and read again on every call: A B^T 18560 x 14592 x 480 1263 -> 1588 us, 7477 x 9353 x 1028 686 -> 781.)
        struct Raw {
            float a[TI][4], b[TJ][4];
        };
        auto four = [&](auto kc, const float *x, int64_t ld, int64_t k0, float (&to)[4]) {
            const int64_t k = k0 + 4 * h;
            if (decltype(kc)::value && k + 4 <= g.K) __builtin_memcpy(to, x + k, 16);
            else {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float y = x[(k + e < g.K ? k + e : g.K - 1) * (decltype(kc)::value ? 1 : ld)];
                    to[e] = k + e < g.K ? y : 0.0f;
                }
            }
        };
        auto load = [&](Raw &r, int64_t k0) {
#pragma unroll
            for (int i = 0; i < TI; i++) four(std::integral_constant<bool, A_KC>(), a[i], g.lda, k0, r.a[i]);
#pragma unroll
            for (int j = 0; j < TJ; j++) four(std::integral_constant<bool, B_KC>(), b[j], g.ldb, k0, r.b[j]);
        };
        auto multiply = [&](const Raw &r) {
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int i = 0; i < TI; i++)
#pragma unroll
                    for (int j = 0; j < TJ; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(r.b[j][e], r.a[i][e], acc[i][j], 0, 0, 0);
        };
        for (int64_t k0 = 0; k0 < g.K; k0 += 16) {                    // uniform
            Raw r;
            load(r, k0);
            multiply(r);
        }
    } else {
#pragma unroll
        for (int i = 0; i < TI; i++)
#pragma unroll
            for (int j = 0; j < TJ; j++) acc[i][j] *= TERMS_DOWN;
    }

    // ---- blocks of 32 x 32 in whole rows of 128 bytes, turned through 4 KiB of the wave's own (as turn_tile_and_store, for any alignment of C).
    // Register v of lane l: row l & 15, column 4 (l >> 4) + v of a 16 x 16 block ----
    unsigned char *turn = lds + wave * 4096;
#pragma unroll
    for (int ci = 0; ci < TI / 2; ci++)
#pragma unroll
        for (int cj = 0; cj < TJ / 2; cj++) {
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int row = 16 * (q >> 1) + r16, chunk = 4 * (q & 1) + h;
                *reinterpret_cast<v4f *>(turn + row * 128 + ((chunk ^ ((row >> 1) & 7)) << 4)) = acc[2 * ci + (q >> 1)][2 * cj + (q & 1)];
            }
            order_in_wave();
            const int64_t col = n0 + cj * 32 + (lane & 7) * 4;
            const int have = g.N - col >= 4 ? 4 : (int)(g.N - col);
            v4f bias = {0.f, 0.f, 0.f, 0.f};
            if (g.bias) {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (e < have) bias[e] = g.bias[col + e];
            }
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int row = r * 8 + (lane >> 3);
                const int64_t m = m0 + ci * 32 + row;
                v4f o = *reinterpret_cast<const v4f *>(turn + row * 128 + (((lane & 7) ^ ((row >> 1) & 7)) << 4));
                if (m >= g.M || have <= 0) continue;
                float *cp = g.C + m * g.ldc + col;
                if (g.alpha != 1.0f) o *= g.alpha;
                if (g.beta != 0.0f) {
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        if (e < have) o[e] += g.beta * cp[e];
                }
                if (g.bias) o += bias;
#pragma unroll
                for (int e = 0; e < 4; e++) o[e] = apply_act(o[e], g.act);
                if (have == 4) __builtin_memcpy(cp, &o, 16);
                else {
#pragma unroll
                    for (int e = 0; e < 3; e++)
                        if (e < have) cp[e] = o[e];
                }
            }
            order_in_wave();
        }
}

template <int WM, int WN, int TI, int TJ, bool TURNS, bool A_KC, bool B_KC>
int launch_planes(const char *name, const PlanesArgs &p) {
    using T = Tile<WM, WN, TI, TJ>;
    auto kern = k_gemm_planes<WM, WN, TI, TJ, TURNS, A_KC, B_KC>;
    static bool attr_set = false;
    if (!attr_set) {
        AXHIP_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, T::SMEM), "hipFuncSetAttribute");
        attr_set = true;
    }
    const int64_t tiles = ((p.g.M + T::BM - 1) / T::BM) * ((p.g.N + T::BN - 1) / T::BN);
    note_kernel(name);
    hipLaunchKernelGGL(kern, dim3((unsigned)tiles), dim3(64 * T::WAVES), T::SMEM, kStream, p);
    return check_launch(name);
}
}  // namespace

namespace axhip {
// Tiles of 256x128 (a workgroup a CU) and 128x64 (two a CU), each priced by a line fitted to 420 products of 1.2e9 to 4e10 multiply-adds in every storage order, and
// taken where that is a twentieth below the price of the staged tiles (plan_staged).  The prices are for this comparison; as times both are too low where the chip runs into its
// power cap (2048 x 4096 x 4096 241 for 311 us, staged 320 for 366; over 79 products of up to 2e11 multiply-adds 0.70 to 0.98, staged 0.77 to 1.05).  On these
// 79 planes are 1.24 times as fast (0.99 to 1.43), on 145 more near the line, of K up to 7300, 1.15 (0.999 and more).  Near the line with a K above 4096 planes of 128x64 are
// behind but for A^T B (A B^T 1498 x 2020 x 7312 270 -> 292, 2208 x 1248 x 6112 218 -> 238, A B 2368 x 1248 x 6304 245 -> 256; A^T B 1495 x 1819 x 5230 226 -> 215, A B
// 1706 x 3467 x 5049, priced at 0.90, 456 -> 388): a twelfth there.  K below 480, left out: 2122 x 3008 x 320 35.4 -> 38.0.  Elsewhere
// cutting costs what it saves: up to a tile or two a CU (1024^3 21 -> 34, 2000 x 1024 x 1024 31 -> 37), and a long K with few columns (2000 x 1024 x 4096
// 104 -> 113; its planes take 20).
// The error against 64 bits is no larger than before on any of them: 128x64 has as many sums as the staged 128x64 and 64x64 tiles (1.19e-7 at K = 1024,
// 2.5e-7 at 4096), 256x128 fewer (1.70 and 3.75e-7), and stands only for 128x128 ones (3.4 and 7.0e-7); ranges of K on smaller tiles, which have more, stay.
int planes_f32(const StagedArgs &g, int transa, int transb) {
    if ((transa && transb) || g.K < 480 || g.K > (1 << 20) || g.M > (1 << 20) || g.N > (1 << 20)) return -1;
    const StagedChoice staged = split_choice(g);
    if (staged.ranges > 1 && !staged.is_128x128) return -1;
    auto up = [](int64_t n, int64_t by) { return (n + by - 1) / by; };
    const int64_t cus = cu_count();
    const float cut_mb = (float)(g.M + g.N) * (float)g.K * 10.0e-6f, slabs = (float)up(g.K, 32);
    const float large = (float)up(up(g.M, 256) * up(g.N, 128), cus), small = (float)up(up(g.M, 128) * up(g.N, 64), cus);
    const float pairs = (float)((int)small / 2), single = small - 2.0f * pairs;
    const float us[2] = {4.6f + 0.357f * cut_mb + large * (1.042f * slabs + 13.7f),
                         8.7f + 0.207f * cut_mb + pairs * (0.851f * slabs + 5.6f) + single * (0.567f * slabs + 3.3f)};
    const int tile = staged.is_128x128 && us[0] < us[1] ? 0 : 1, kblocks = (int)up(g.K, 32);
    if (us[tile] > (tile == 1 && !transa && g.K > 4096 ? 0.92f : 0.95f) * staged.us) return -1;
    PlanesArgs p{g, nullptr, nullptr, (int)up(g.M, 16), (int)up(g.N, 16), kblocks};
    const size_t a_bytes = (size_t)p.a_blocks * kblocks * BLOCK, b_bytes = (size_t)p.b_blocks * kblocks * BLOCK;
    if (a_bytes + b_bytes > kWorkspaceStart || a_bytes + b_bytes > workspace_bytes()) return -1;     // never grown for planes
    unsigned char *ws = static_cast<unsigned char *>(workspace(a_bytes + b_bytes));
    if (!ws) return AXHIP_ERR_ALLOC;
    p.a = ws;
    p.b = ws + a_bytes;
    const CutSide a{static_cast<const float *>(g.A), ws, g.M, g.lda, transa, p.a_blocks}, b{static_cast<const float *>(g.B), ws + a_bytes, g.N, g.ldb, !transb, p.b_blocks};
    const int groups = cut_groups(a.across, a.blocks, kblocks) + cut_groups(b.across, b.blocks, kblocks);
    hipLaunchKernelGGL(k_cut_planes, dim3((unsigned)groups), dim3(256), 0, kStream, a, b, g.K, kblocks);
    if (int rc = check_launch("sgemm planes")) return rc;
    auto launch = [&](auto a_kc, auto b_kc, const char *const names[2]) {
        constexpr bool A_KC = decltype(a_kc)::value, B_KC = decltype(b_kc)::value;
        return tile == 0 ? launch_planes<4, 2, 4, 4, false, A_KC, B_KC>(names[0], p) : launch_planes<2, 2, 4, 2, true, A_KC, B_KC>(names[1], p);
    };
    static const char *const nn[2] = {"sgemm_nn_planes256x128x3", "sgemm_nn_planes128x64x3"};
    static const char *const nt[2] = {"sgemm_nt_planes256x128x3", "sgemm_nt_planes128x64x3"};
    static const char *const tn[2] = {"sgemm_tn_planes256x128x3", "sgemm_tn_planes128x64x3"};
    const std::true_type yes;
    const std::false_type no;
    if (!transa && !transb) return launch(yes, no, nn);
    if (!transa) return launch(yes, yes, nt);
    return launch(no, no, tn);
}
}  // namespace axhip
