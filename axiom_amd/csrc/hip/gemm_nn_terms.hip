// Batches of A * B with N up to 32 or from 65 to 128 columns (P V of attention heads) on the bf16 matrix core: both operands in
// three bf16 terms, six products of terms for one of values (bf16x3.h).
//
// What bounds it: reading A (every float once, for 2 N operations), beside the matrix core for the wider N.  A wave takes 32 rows and
// every column, so that a value of A is cut once; A comes in 128-byte pieces of rows (the 16 bytes a lane needs would be 64 rows of
// 16: under half the rate), turned through 4 KiB of LDS of the wave's own.  B is cut once per workgroup, a unit of 32 k ahead in the
// other half of its LDS, and both operands are two units ahead in registers.  Four waves leave room for a second workgroup on the CU,
// which fills the other's barriers; eight cut B half as often.
// us, before (64x64 tiles; N = 128: 128x64 streams) -> this, and the error against 64 bits relative to C: 512 heads of 512 x 512,
// N = 32 157 -> 116 (2.9e-7 -> 1.2e-7), N = 80 293 -> 199 (2.9e-7 -> 1.6e-7), N = 128 284 -> 248 (4.1e-7 -> 1.6e-7); 128 of 500 x 500,
// N = 17 46 -> 27, N = 80 79 -> 48; 512 of 100 x 100, N = 32 13.4 -> 10.0.  N = 33..64 stays with the tiles and
// streams (N = 64 157 -> 154 here, 96 of 640 x 640 slower).
// A workgroup with a sum that is not finite does its rows again with fp32 instructions.
#include "gemm_staged.h"

#include "bf16x3.h"

namespace {
using namespace axhip;

// A workgroup of WAVES waves owns 32 * WAVES rows and all NB blocks of 32 columns of one member of the batch; K goes in units of 32.
template <int NB, int WAVES>
struct NnGeom {
    static constexpr int T = 64 * WAVES, COLS = 32 * NB;
    static constexpr int PLANE = COLS * 64, STAGE = 3 * PLANE;          // B of a unit: a column's 32 k of one term, 64 bytes
    static constexpr int TURN_AT = 2 * STAGE, FLAGS_AT = TURN_AT + WAVES * 4096, SMEM = FLAGS_AT + 4 * WAVES;
    static constexpr int E = COLS * 32 % (8 * T) == 0 ? 8 : COLS * 32 % (4 * T) == 0 ? 4 : 2, PIECES = COLS * 32 / (E * T);       // a thread's pieces of B: E k of a column
    static_assert(E >= 2 && PIECES * E * T == COLS * 32, "a unit of B divides over the threads");
    // where the 16-byte chunk c (8 k) of column r lies
    __device__ static unsigned at(int r, int c) { return (unsigned)(r * 64 + ((c ^ ((r >> 2) & 3)) << 4)); }
};

template <int NB, int WAVES>
__global__ void __launch_bounds__(64 * WAVES, NB == 1 ? 3 : 2) k_nn_terms(StagedArgs g) {
    using G = NnGeom<NB, WAVES>;
    constexpr int E = G::E, PIECES = G::PIECES;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r32 = lane & 31, h = lane >> 5;
    int tm, tn;
    int64_t batch;
    tile_of_batched_block((int)((g.M + 32 * WAVES - 1) / (32 * WAVES)), 1, tm, tn, batch);
    const int64_t row0 = (int64_t)tm * 32 * WAVES + wave * 32, lda4 = g.lda * 4, ldb4 = g.ldb * 4;
    const bool idle = row0 >= g.M;                     // such a wave brings its share of B all the same
    const int rows = idle ? 0 : (int)(g.M - row0 < 32 ? g.M - row0 : 32);
    const char *A = reinterpret_cast<const char *>(static_cast<const float *>(g.A) + batch * g.stride_a + (idle ? 0 : row0) * g.lda);
    const char *B = reinterpret_cast<const char *>(static_cast<const float *>(g.B) + batch * g.stride_b);
    // What is fetched past the last unit is not multiplied: it is the unit before it, since the last one may end inside and is slow then (us, last -> before:
    // 512 of 136 x 32 x 136 20.9 -> 19.7, 300 of 200 x 96 x 200 42.9 -> 41.7, 40 of 777 x 32 x 777 37.3 -> 36.5; level where K is a multiple of 32).
    const int units = (int)((g.K + 31) / 32), last = units - 1, before = last > 0 ? last - 1 : 0;

    // ---- A: 128-byte pieces of rows, eight rows a load, turned through 4 KiB of this wave's own ----
    unsigned char *turn = lds + G::TURN_AT + wave * 4096;
    unsigned oa[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int r = 8 * q + (lane >> 3);
        oa[q] = (unsigned)(r < rows ? r : rows > 0 ? rows - 1 : 0) * (unsigned)lda4 + (lane & 7) * 16;
    }
    auto load_a = [&](float (&x)[16], int u) {
        const int64_t k = (int64_t)(u <= last ? u : before) * 32;
        const char *p = A + k * 4;
        const int end = (int)(g.K - 1 - k) - (lane & 7) * 4;                   // the last k there is, from this lane's first
        if (k + 32 <= g.K) {
#pragma unroll
            for (int q = 0; q < 4; q++) __builtin_memcpy(&x[4 * q], p + oa[q], 16);
        } else {                                       // past the end of K: zero
#pragma unroll
            for (int q = 0; q < 4; q++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float y = *reinterpret_cast<const float *>(p + oa[q] + (e <= end ? e : end) * 4);
                    x[4 * q + e] = e <= end ? y : 0.0f;
                }
        }
    };
    // ---- B: a thread takes E k of a column ----
    unsigned ob[PIECES];
    int kb[PIECES];
    unsigned wb[PIECES];
#pragma unroll
    for (int i = 0; i < PIECES; i++) {
        const int q = tid + i * G::T, col = q % G::COLS, c = q / G::COLS;
        ob[i] = (unsigned)(col < g.N ? col : g.N - 1) * 4;
        kb[i] = c * E;
        wb[i] = G::at(col, c * E / 8) + c * E % 8 * 2;
    }
    auto load_b = [&](float (&x)[PIECES][E], int u) {
        const int64_t k = (int64_t)(u <= last ? u : before) * 32;
        const int end = (int)(g.K - 1 - k);
        const char *p = B + k * ldb4;
#pragma unroll
        for (int i = 0; i < PIECES; i++)
#pragma unroll
            for (int e = 0; e < E; e++) x[i][e] = *reinterpret_cast<const float *>(p + (unsigned)(kb[i] + e < end ? kb[i] + e : end) * (uint64_t)ldb4 + ob[i]);
    };
    auto stage_b = [&](const float (&x)[PIECES][E], unsigned at) {
#pragma unroll
        for (int i = 0; i < PIECES; i++) {
            if constexpr (E >= 4) {
                Term<E> t[3];
                cut(x[i], TERMS_UP, t);
#pragma unroll
                for (int p = 0; p < 3; p++) *reinterpret_cast<Term<E> *>(lds + at + wb[i] + p * G::PLANE) = t[p];
            } else {
                int t[3];
                bf16x3_nearest(x[i][0] * TERMS_UP, x[i][1] * TERMS_UP, t[0], t[1], t[2]);
#pragma unroll
                for (int p = 0; p < 3; p++) *reinterpret_cast<int *>(lds + at + wb[i] + p * G::PLANE) = t[p];
            }
        }
    };

    // The five smaller products in a sum of their own: one for all of K where there are registers for it, else one for each step, which
    // the sum takes in with one addition (512 x 512, N = 128: error 3.4e-7 with all six in one sum, 1.6e-7 so).
    constexpr bool APART = NB == 1;
    v16f acc[NB], sums[APART ? NB : 1], zero;
#pragma unroll
    for (int j = 0; j < NB; j++)
#pragma unroll
        for (int v = 0; v < 16; v++) {
            acc[j][v] = 0.0f;
            if constexpr (APART) sums[j][v] = 0.0f;
            zero[v] = 0.0f;
        }
    auto multiply = [&](const float (&x)[16], unsigned cur) {
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int row = 8 * q + (lane >> 3);
            *reinterpret_cast<v4f *>(turn + row * 128 + (((lane & 7) ^ ((row >> 1) & 7)) << 4)) = v4f{x[4 * q], x[4 * q + 1], x[4 * q + 2], x[4 * q + 3]};
        }
        order_in_wave();                               // (the next writes come after a barrier of the workgroup)
#pragma unroll
        for (int s = 0; s < 2; s++) {                  // k 16 s + 8 h + e
            const unsigned at = r32 * 128 + (((4 * s + 2 * h) ^ ((r32 >> 1) & 7)) << 4);
            const v4f y = *reinterpret_cast<const v4f *>(turn + at), z = *reinterpret_cast<const v4f *>(turn + (at ^ 16));
            const float v[8] = {y[0], y[1], y[2], y[3], z[0], z[1], z[2], z[3]};
            v4i fa[3];
            cut(v, TERMS_UP, fa);
#pragma unroll
            for (int j = 0; j < NB; j++) {
                v4i fb[3];
                v16f of_step;
#pragma unroll
                for (int p = 2; p >= 0; p--) fb[p] = *reinterpret_cast<const v4i *>(lds + cur + G::at(r32, 2 * s + h) + j * 2048 + p * G::PLANE);
                v16f &low = APART ? sums[APART ? j : 0] : of_step;
                if constexpr (!APART) low = zero;
#pragma unroll
                for (int sum = 2; sum > 0; sum--)      // the small products first
#pragma unroll
                    for (int p = sum; p >= 0; p--) low = mfma_terms(fa[p], fb[sum - p], low);
                acc[j] = mfma_terms(fa[0], fb[0], acc[j]);
                if constexpr (!APART) acc[j] += low;
            }
        }
    };

    // ---- units: B of the next one is cut beside the products of this one, both operands are two ahead in registers ----
    float a0[16], a1[16], b[PIECES][E];
    load_b(b, 0);
    load_a(a0, 0);
    load_a(a1, 1);
    stage_b(b, 0);
    load_b(b, 1);
    __syncthreads();
    unsigned cur = 0;
    auto step = [&](int u, float (&a)[16]) {
        if (!idle) multiply(a, cur);
        stage_b(b, cur ^ G::STAGE);
        load_a(a, u + 2);
        load_b(b, u + 2);
        __syncthreads();
        cur ^= G::STAGE;
    };
    int u = 0;
    for (; u + 2 <= last; u += 2) {
        step(u, a0);
        step(u + 1, a1);
    }
    if (u < last) {
        step(u, a0);
        if (!idle) multiply(a1, cur);
    } else if (!idle) multiply(a0, cur);

    float seen = 0.0f;
#pragma unroll
    for (int j = 0; j < NB; j++) {
        if constexpr (APART) acc[j] += sums[j];
        look_at(acc[j], seen);
    }
    float scale = TERMS_DOWN;
    if (any_wave<WAVES>(!(seen == 0.0f), lds + G::FLAGS_AT, wave)) {
        if (idle) return;
        // what the terms cannot hold, with fp32 instructions
        scale = 1.0f;
#pragma unroll
        for (int j = 0; j < NB; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[j][v] = 0.0f;
        const char *arow = A + (int64_t)(r32 < rows ? r32 : rows - 1) * lda4;
        for (int64_t k0 = 0; k0 < g.K; k0 += 2) {
            const int64_t k = k0 + h, ke = k < g.K ? k : g.K - 1;
            const float x = *reinterpret_cast<const float *>(arow + ke * 4), fa = k < g.K ? x : 0.0f;
#pragma unroll
            for (int j = 0; j < NB; j++) {
                const int col = 32 * j + r32;
                const float y = *reinterpret_cast<const float *>(B + ke * ldb4 + (col < g.N ? col : g.N - 1) * 4);
                acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa, k < g.K ? y : 0.0f, acc[j], 0, 0, 0);
            }
        }
    }
    if (idle) return;
    // register v of lane l: row 8 (v >> 2) + 4 (l >> 5) + (v & 3), column l & 31: a store instruction writes two whole 128-byte pieces of rows
    float *C = g.C + batch * g.stride_c + row0 * g.ldc;
#pragma unroll
    for (int j = 0; j < NB; j++) {
        const int col = 32 * j + r32;
        if (col >= g.N) continue;
#pragma unroll
        for (int v = 0; v < 16; v++) {
            const int row = 8 * (v >> 2) + 4 * h + (v & 3);
            if (row < rows) C[(int64_t)row * g.ldc + col] = g.alpha * (acc[j][v] * scale);
        }
    }
}

template <int NB, int WAVES>
int launch(const StagedArgs &g, int64_t batch) {
    using G = NnGeom<NB, WAVES>;
    static bool attr_set = false;
    if (!attr_set) {
        AXHIP_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(k_nn_terms<NB, WAVES>), hipFuncAttributeMaxDynamicSharedMemorySize, G::SMEM),
                      "hipFuncSetAttribute");
        attr_set = true;
    }
    constexpr const char *name = WAVES == 8 ? "sgemm_nn_rows256x3" : "sgemm_nn_rows128x3";
    note_kernel(name);
    hipLaunchKernelGGL((k_nn_terms<NB, WAVES>), dim3((unsigned)((g.M + 32 * WAVES - 1) / (32 * WAVES)), (unsigned)batch), dim3(64 * WAVES), G::SMEM, kStream, g);
    return check_launch(name);
}
}  // namespace

namespace axhip {
int nn_terms(const StagedArgs &g, int64_t batch) {
    if (g.K < 64 || g.M < 96 || g.N < 1 || g.N > 128 || g.beta != 0.0f || g.bias || g.col_scale || g.act != AXHIP_ACT_NONE || g.lda >= (1 << 22) ||
        g.ldb >= (1 << 22) || batch > 65535)
        return -1;
    // Under 96 rows idle waves cost more than the tiles (N = 32, 256 of 64 x 500 13.8 -> 16.1, 16 x 1024 22.5 -> 24.7).
    const int64_t cus = cu_count(), tiles4 = (g.M + 127) / 128 * batch, tiles8 = (g.M + 255) / 256 * batch;
    // whether the kernels before load straight to LDS, and are on fp32 instructions
    const bool on_grid = (g.K | g.N | g.lda | g.ldb | g.ldc | g.stride_a | g.stride_b | g.stride_c) % 4 == 0 &&
                         ((uintptr_t)g.A | (uintptr_t)g.B | (uintptr_t)g.C) % 16 == 0;
    if (g.N <= 32) {
        // From three quarters of the CUs on (1000 x 1000, 32 of them 39 -> 32; 64 of 256 x 256, 128 workgroups, level); from one and a half
        // where three of eight waves would have no rows and the kernels before have 32-row tiles (132 x 936, N = 4, 99 of them 22.0 -> 28.8, 144 x 144,
        // N = 4, 146 of them 8.7 -> 11.3).  Cached operands gain more than such from HBM (497 random batches, any N: 1.34 and 1.23).
        const bool short_rows = on_grid && g.M > 128 && g.M <= 160;
        return tiles4 * 4 >= cus * (short_rows ? 6 : 3) ? launch<1, 4>(g, batch) : -1;
    }
    // N = 33..64 as above.  Wider ones need 0.7 of two workgroups a CU (N = 80, 64 of 512 x 512, half of them, 0.97; 96 of 384 x 384,
    // 0.56, 1.16; off the grid, where the kernels before are faster, 0.75), N > 96 K >= 256 (256 of 1024 x 128 82.5 -> 84.1, 200 x 200
    // 109 -> 111).
    if (g.N <= 64 || tiles4 * 20 <= 2 * cus * (on_grid ? 14 : 15) || (g.N > 96 && g.K < 256)) return -1;
    // Off the grid they stand before tiles in terms, whose error is the larger one on 128x128 tiles only: elsewhere those have the five smaller
    // products in a sum of their own over all of K (129 of 959 x 181, N = 69 9.6e-8 here and 5.9e-8 there, 284 of 176 x 990, N = 73 2.2e-7 and
    // 1.15e-7; on 128x128 tiles 1.4 to 1.5 times the error here).
    if (!on_grid && !split_is_128x128(g, batch)) return -1;
    // Four waves or eight: rounds of workgroups over the chip, of which one with a workgroup on each CU at most is 0.72 (N = 80: 96 of
    // 640 x 640 82 with eight and 59 with four, 64 of 1000 x 1000 86 and 100).
    const int64_t left = tiles4 % (2 * cus), cost4 = tiles4 / (2 * cus) * 107 + (left == 0 ? 0 : left <= cus ? 72 : 105);
    const bool eight = (tiles8 + cus - 1) / cus * 100 <= cost4;
    if (g.N <= 96) return eight ? launch<3, 8>(g, batch) : launch<3, 4>(g, batch);
    return eight ? launch<4, 8>(g, batch) : launch<4, 4>(g, batch);
}
}  // namespace axhip
