// Products whose operands pass through registers on their way to LDS: fp32 matrices at any alignment and any K, as they are or
// cut into three bf16 terms each on the way, and W8A32 (fp32 activations against int8 weights), where the activations are.
//
// fp32 products in bf16 terms (SPLIT): six bf16 products per fp32 one (bf16x3_nearest) still take 6/16 of the matrix-core time of
// the fp32 instructions, and as an instruction adds 16 products before it rounds, the sums are nearer to 64 bits than those of
// the fp32 tiles on every shape measured (relative error 1024^3 4.1e-7 -> 1.2e-7 on 64x64 tiles, 2048 x 4096 x 4096 1.15e-6 ->
// 7.0e-7 on 128x128).  us, fp32 tiles -> split: 2000 x 4096 x 1024 142 -> 98, 2000 x 1024 x 4096 134 -> 98, 4096^3 931 -> 686
// (200 TFLOP/s), 8192^3 7370 -> 5440, 8 x 1024^3 155 -> 98, a feed-forward block 2048 x 1024 x 4096 250 -> 200.  Bound on 128x128: of
// the cycles of that block's products the matrix core is busy 49 %, the vector pipe some 40 %, the LDS pipe 32 % (a fifth of that bank
// conflicts); 64x64: the reads of fragments from LDS.  The conversions
// (some 8 instructions a value) are put between the products of the same wave (interleave), worth 4 to 10 %.
// A tile whose sums are not all finite is computed again with fp32 instructions by the same workgroup: infinities, NaNs and values
// near the largest float come out as fp32 products give them.
//
// Why not direct to LDS: those loads move whole 16-byte pieces to their final place, so rows that start off the 16-byte grid,
// a K that ends inside a slab and a conversion all need the register.  A slab is fetched two slabs ahead into registers,
// converted and written to the other LDS buffer while the current one is multiplied.  Eight waves: two sets of four that share
// the tile and take its 16-wide k-steps in turn; on every SIMD one wave of each set, which do the slab's two halves of work
// (convert and write; read and multiply) in opposite order, so that vector and matrix instructions come from different waves.
// Operands lie in LDS as rows of one slab each (an operand stored the other way is transposed by the register: a thread takes
// consecutive k of one column), fragments are 16-byte reads; rows are spread over the banks (Geom::at).
// Bound: fp32 instructions (forced tiles, K below 64 off the 16-byte grid, narrow batches), the matrix core: 2001 x 2003 x 2005 runs at
// 119 TFLOP/s (76 % of the datasheet rate; guarded 64x64 tiles without
// prefetch 75), 1024^3 at 24 us against 19.6 of the direct-to-LDS kernel, which keeps every shape it can take.  Small products
// are latency: one 64x64 tile with K = 92 takes 7 us, of which 2.3 are the launch.  W8A32, 250 x 4096 x 4096 in 35.6 us (235
// TFLOP/s of products, three bf16 terms each): matrix core busy 28 % of the cycles, LDS and vector pipe 24 % each, at idle clocks; without
// the conversions 27 us, without products 24, without global loads 27, products alone 20 - three pipes that overlap in part.
// Activations are cut as in SPLIT, so that small ones keep their bits (they ran on fp32 instructions before these tiles); the second
// pass over tiles with sums that are not finite reads its operands straight from memory (no room for fp32 slabs in the same LDS).
// Measured and dropped: reading the fragments of both k-steps ahead of the products (35.7 us, 29 spills), 64-wide fp32 slabs
// (2001 x 2003 x 2005 144 us against 135 with 32-wide ones).
#include "gemm_staged.h"

#include "bf16x3.h"

namespace {
using namespace axhip;


// How a product is formed: fp32 on the fp32 matrix core; fp32 activations in three bf16 terms against int8 weights in one;
// both operands in three bf16 terms.
enum Op { F32, I8W, SPLIT };

// One BM x BN tile of C per workgroup of eight waves: WM x WN waves over the tile, and two sets of them (wk) that take
// the 16-wide k-steps of a slab in turn and are added through LDS at the end.
template <int BM, int BN, int WM, int WN, int BK, Op OP>
struct Geom {
    static_assert(WM * WN == 4, "two sets of four waves");
    static constexpr int TM = BM / WM / 32, TN = BN / WN / 32;      // 32x32 blocks per wave
    static constexpr int ROW = BK * (OP == F32 ? 4 : 2);            // bytes of a row of a slab in LDS: fp32, or bf16 terms
    static constexpr int A_PLANE = BM * ROW, A_BYTES = (OP == F32 ? 1 : 3) * A_PLANE;
    static constexpr int B_PLANE = BN * ROW, B_BYTES = (OP == SPLIT ? 3 : 1) * B_PLANE;
    static constexpr int STAGE = A_BYTES + B_BYTES;
    static constexpr int CPITCH = BN + 4;                           // floats per row of the tile in LDS
    static constexpr int BUFFERS = 2 * STAGE > BM * CPITCH * 4 ? 2 * STAGE : BM * CPITCH * 4;
    // In bf16 terms a word per wave besides: are its sums finite.  Where 32 bytes more would keep a second workgroup off the CU (I8W,
    // 64x128) the words lie in the buffers, past the tile, and are written when all waves have read the last slab.
    static constexpr bool WORDS_INSIDE = 160 * 1024 / (BUFFERS + 32) < 160 * 1024 / BUFFERS;
    static constexpr int SMEM = BUFFERS + (OP == F32 || WORDS_INSIDE ? 0 : 32), WORDS_AT = WORDS_INSIDE ? BUFFERS - 32 : BUFFERS;
    static_assert(OP == F32 || BM * CPITCH * 4 <= WORDS_AT, "the words outlive the start of the write-back");
    static_assert(SMEM <= 160 * 1024, "LDS budget");
    // Where the 16-byte chunk c of row r lies in its row: rows are spread so that the 16 lanes that a 16-byte access
    // serves together (16 rows of one chunk, or the chunks of neighbouring rows) fall on distinct banks.
    __host__ __device__ static constexpr int at(int row, int chunk) {
        return row * ROW + ((chunk ^ ((row / (256 / ROW)) & (ROW / 16 - 1))) << 4);
    }
};

// The sum over this workgroup's range of K, into acc: per wave TM x TN blocks of 32x32, register v of lane l: row (l & 31),
// column 8 * (v >> 2) + 4 * (l >> 5) + (v & 3).  Returns whether any wave found its part of a product
// in bf16 terms unfit.
template <int BM, int BN, int WM, int WN, int BK, Op OP, bool A_KC, bool B_KC>
__device__ __forceinline__ bool
sum_range(const StagedArgs &g, unsigned char *lds, int wave, int64_t m0, int64_t n0, int64_t batch,
          v16f (&acc)[BM / WM / 32][BN / WN / 32]) {
    using G = Geom<BM, BN, WM, WN, BK, OP>;
    constexpr bool I8 = OP == I8W, TERMS = OP != F32;   // int8 B; bf16 terms in LDS
    constexpr int TM = G::TM, TN = G::TN, T = 512;
    // a thread stages NTA pieces of EA k values of a row of A per slab, NTB of EB of B
    constexpr int EA = BM * BK >= 8 * T ? 8 : 4, NTA = BM * BK / T / EA;
    constexpr int EB = I8 ? (BN * BK >= 16 * T ? 16 : 8) : (BN * BK >= 8 * T ? 8 : 4), NTB = BN * BK / T / EB;
    static_assert(NTA * EA * T == BM * BK && NTB * EB * T == BN * BK, "a slab divides over the threads");

    const int tid = threadIdx.x, lane = tid & 63;
    const int wk = wave >> 2, wm = (wave & 3) / WN, wn = (wave & 3) % WN;
    const int64_t kbeg = (int64_t)blockIdx.z * g.k_range, kend = kbeg + g.k_range < g.K ? kbeg + g.k_range : g.K;
    const int slabs = (int)((kend - kbeg + BK - 1) / BK), last = slabs - 1;

    // ---- where each piece is read and written: 32-bit byte offsets from a base that is the same for the whole workgroup ----
    const char *abase = reinterpret_cast<const char *>(static_cast<const float *>(g.A) + batch * g.stride_a +
                                                       (A_KC ? m0 * g.lda + kbeg : m0 + kbeg * g.lda));
    const char *bbase = static_cast<const char *>(g.B) + (int64_t)(I8 ? 1 : 4) * (batch * g.stride_b + (B_KC ? n0 * g.ldb + kbeg : n0 + kbeg * g.ldb));
    const int64_t astep = A_KC ? BK * 4 : BK * 4 * g.lda, bstep = I8 ? BK : B_KC ? BK * 4 : BK * 4 * g.ldb;   // bytes per slab
    // A last slab that would run past the range is fetched from so much further to the left that it ends with the range,
    // and the `skip` values that the slab before it already held are zeroed in LDS before it is multiplied: every load is
    // a whole vector load, whatever K is (K >= BK).
    const int skip = slabs * BK - (int)(kend - kbeg);
    const int64_t aback = astep / BK * skip, bback = bstep / BK * skip;
    const unsigned lda4 = (unsigned)g.lda * 4, ldb4 = (unsigned)g.ldb * 4;
    unsigned oa[NTA], wa[NTA], ob[NTB], wb[NTB];     // byte offsets in memory, in LDS
    const int mlast = (int)(g.M - 1 - m0), nlast = (int)(g.N - 1 - n0);
#pragma unroll
    for (int i = 0; i < NTA; i++) {
        constexpr int PER = BK / EA;                 // pieces per row
        const int q = tid + i * T, row = A_KC ? q / PER : q % BM, c = A_KC ? q % PER : q / BM;
        const unsigned r = row < mlast ? row : mlast;
        oa[i] = A_KC ? r * lda4 + c * EA * 4 : r * 4 + c * EA * lda4;
        wa[i] = TERMS ? G::at(row, c * EA / 8) + (c * EA % 8) * 2 : G::at(row, c * EA / 4);
    }
#pragma unroll
    for (int i = 0; i < NTB; i++) {
        constexpr int PER = BK / EB;
        const int q = tid + i * T, row = B_KC ? q / PER : q % BN, c = B_KC ? q % PER : q / BN;
        const unsigned r = row < nlast ? row : nlast;
        if constexpr (I8) ob[i] = r * (unsigned)g.ldb + c * EB;
        else ob[i] = B_KC ? r * ldb4 + c * EB * 4 : r * 4 + c * EB * ldb4;
        wb[i] = TERMS ? G::at(row, c * EB / 8) + (c * EB % 8) * 2 : G::at(row, c * EB / 4);
    }

    struct Regs {
        float a[NTA][EA];
        float b[NTB][I8 ? 1 : EB];
        int q[NTB][I8 ? EB / 4 : 1];
    };
    Regs set0, set1;
    auto load = [&](Regs &r, int s) {                // slab s (the last one for any s past it) from memory
        const int t = s < last ? s : last;
        const char *ab = abase + t * astep - (s < last ? 0 : aback), *bb = bbase + t * bstep - (s < last ? 0 : bback);
#pragma unroll
        for (int i = 0; i < NTA; i++) {
            if constexpr (A_KC) __builtin_memcpy(r.a[i], ab + oa[i], EA * 4);
            else {
#pragma unroll
                for (int e = 0; e < EA; e++) r.a[i][e] = *reinterpret_cast<const float *>(ab + (uint64_t)e * lda4 + oa[i]);
            }
        }
#pragma unroll
        for (int i = 0; i < NTB; i++) {
            if constexpr (I8) __builtin_memcpy(r.q[i], bb + ob[i], EB);
            else if constexpr (B_KC) __builtin_memcpy(r.b[i], bb + ob[i], EB * 4);
            else {
#pragma unroll
                for (int e = 0; e < EB; e++) r.b[i][e] = *reinterpret_cast<const float *>(bb + (uint64_t)e * ldb4 + ob[i]);
            }
        }
    };
    auto put_terms = [&](unsigned char *d, int plane, const auto &x) {
        constexpr int E = sizeof(x) / sizeof(float);
        Term<E> t[3];
        cut(x, TERMS_UP, t);
#pragma unroll
        for (int p = 0; p < 3; p++) *reinterpret_cast<Term<E> *>(d + p * plane) = t[p];
    };
    auto stage = [&](const Regs &r, unsigned at) {   // ... into LDS buffer `at`
#pragma unroll
        for (int i = 0; i < NTA; i++) {
            const float *x = r.a[i];
            if constexpr (TERMS) {
                put_terms(lds + at + wa[i], G::A_PLANE, r.a[i]);
            } else {
#pragma unroll
                for (int h = 0; h < EA / 4; h++)
                    *reinterpret_cast<v4f *>(lds + at + (wa[i] ^ (h * 16))) = v4f{x[4 * h], x[4 * h + 1], x[4 * h + 2], x[4 * h + 3]};
            }
        }
#pragma unroll
        for (int i = 0; i < NTB; i++) {
            if constexpr (I8) {
#pragma unroll
                for (int h = 0; h < EB / 8; h++)
                    *reinterpret_cast<v4i *>(lds + at + G::A_BYTES + (wb[i] ^ (h * 16))) = bf16_of_i8(r.q[i][2 * h], r.q[i][2 * h + 1]);
            } else if constexpr (OP == SPLIT) {
                put_terms(lds + at + G::A_BYTES + wb[i], G::B_PLANE, r.b[i]);
            } else {
                const float *x = r.b[i];
#pragma unroll
                for (int h = 0; h < EB / 4; h++)
                    *reinterpret_cast<v4f *>(lds + at + G::A_BYTES + (wb[i] ^ (h * 16))) = v4f{x[4 * h], x[4 * h + 1], x[4 * h + 2], x[4 * h + 3]};
            }
        }
    };

    // ---- LDS -> fragments -> products ----
    const int frow = lane & 31, fhalf = lane >> 5;
    // SPLIT, up to 128x64: the five smaller products in a sum of their own, so that the large one is rounded once per 16 k and not
    // six times (relative error of 139 x 192 x 320, 288 x 3561 x 703: one sum 1.9e-7, 2.8e-7); 128x128 has no registers left for it
    constexpr bool APART = OP == SPLIT && TM * TN < 4;
    v16f low[APART ? TM : 1][APART ? TN : 1];
    if constexpr (APART) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int v = 0; v < 16; v++) low[i][j][v] = 0.0f;
    }
    const int arow = wm * TM * 32 + frow, brow = wn * TN * 32 + frow;     // + 32 t: the swizzle is that of the first
    // byte addresses of this lane's chunks in its wave's k-steps (wk, and wk + 2 of a 64-wide slab; fp32: the first of two)
    constexpr int STEPS = BK / 32;
    unsigned ra[STEPS], rb[STEPS];
#pragma unroll
    for (int it = 0; it < STEPS; it++) {
        const int ks = 2 * it + wk, c = TERMS ? 2 * ks + fhalf : 4 * ks + 2 * fhalf;
        ra[it] = G::at(arow, c);
        rb[it] = G::A_BYTES + G::at(brow, c);
    }
    auto multiply = [&](unsigned at) {
#pragma unroll
        for (int it = 0; it < STEPS; it++) {
            if constexpr (I8) {
                v4i fa[TM][3], fb[TN];
#pragma unroll
                for (int j = 0; j < TN; j++) fb[j] = *reinterpret_cast<const v4i *>(lds + at + rb[it] + j * 32 * G::ROW);
#pragma unroll
                for (int p = 2; p >= 0; p--)
#pragma unroll
                    for (int i = 0; i < TM; i++) fa[i][p] = *reinterpret_cast<const v4i *>(lds + at + ra[it] + p * G::A_PLANE + i * 32 * G::ROW);
#pragma unroll
                for (int p = 2; p >= 0; p--)                              // the small terms first
#pragma unroll
                    for (int i = 0; i < TM; i++)
#pragma unroll
                        for (int j = 0; j < TN; j++)
                            acc[i][j] = mfma_terms(fb[j], fa[i][p], acc[i][j]);
            } else if constexpr (OP == SPLIT) {
                v4i fa[TM][3], fb[TN][3];
#pragma unroll
                for (int p = 2; p >= 0; p--) {                            // in the order of use
#pragma unroll
                    for (int j = 0; j < TN; j++) fb[j][2 - p] = *reinterpret_cast<const v4i *>(lds + at + rb[it] + (2 - p) * G::B_PLANE + j * 32 * G::ROW);
#pragma unroll
                    for (int i = 0; i < TM; i++) fa[i][p] = *reinterpret_cast<const v4i *>(lds + at + ra[it] + p * G::A_PLANE + i * 32 * G::ROW);
                }
#pragma unroll
                for (int sum = 2; sum >= 0; sum--)                        // the small products first
#pragma unroll
                    for (int p = sum; p >= 0; p--)
#pragma unroll
                        for (int i = 0; i < TM; i++)
#pragma unroll
                            for (int j = 0; j < TN; j++) {
                                v16f &to = APART && sum > 0 ? low[APART ? i : 0][APART ? j : 0] : acc[i][j];
                                to = mfma_terms(fb[j][sum - p], fa[i][p], to);
                            }
            } else {
                v4f fa[TM][2], fb[TN][2];
#pragma unroll
                for (int h = 0; h < 2; h++) {
#pragma unroll
                    for (int i = 0; i < TM; i++) fa[i][h] = *reinterpret_cast<const v4f *>(lds + at + (ra[it] ^ (h * 16)) + i * 32 * G::ROW);
#pragma unroll
                    for (int j = 0; j < TN; j++) fb[j][h] = *reinterpret_cast<const v4f *>(lds + at + (rb[it] ^ (h * 16)) + j * 32 * G::ROW);
                }
#pragma unroll
                for (int e = 0; e < 8; e++)
#pragma unroll
                    for (int i = 0; i < TM; i++)
#pragma unroll
                        for (int j = 0; j < TN; j++)
                            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fb[j][e >> 2][e & 3], fa[i][e >> 2][e & 3], acc[i][j], 0, 0, 0);
            }
        }
    };

    // SPLIT: the conversions go between the products of the same wave: a product keeps the matrix core for eight times as long
    // as it takes to issue
    auto interleave = [&]() {
        constexpr int PRODUCTS = 6 * TM * TN, CUTS = (NTA * EA + NTB * EB) * 8 / STEPS, PER = CUTS / PRODUCTS;
#pragma unroll
        for (int it = 0; it < STEPS; it++) {
            __builtin_amdgcn_sched_group_barrier(0x100, 3 * (TM + TN), 0);
#pragma unroll
            for (int q = 0; q < PRODUCTS; q++) {
                __builtin_amdgcn_sched_group_barrier(0x002, PER, 0);
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            }
        }
    };

    // One slab: multiply the one in LDS, put the next one (already in registers) beside it, request the one three ahead.
    // The two wave sets of a SIMD do the first two in opposite order, so that one converts and writes while the other
    // multiplies.  No branch inside: past the last slab the last one is requested again, unused.
    auto walk = [&](auto set_number) {
        constexpr bool stage_first = decltype(set_number)::value;
        auto step = [&](int s, Regs &next, unsigned cur, unsigned nxt) {
            if constexpr (OP == SPLIT) {
                multiply(cur);
                stage(next, nxt);
                load(next, s + 3);
                interleave();
            } else if constexpr (stage_first) {
                stage(next, nxt);
                load(next, s + 3);
                multiply(cur);
            } else {
                multiply(cur);
                stage(next, nxt);
                load(next, s + 3);
            }
            __syncthreads();
        };
        int s = 0;
        for (; s + 2 <= last; s += 2) {
            step(s, set1, 0, G::STAGE);
            step(s + 1, set0, G::STAGE, 0);
        }
        if (s < last) step(s, set1, 0, G::STAGE);
    };
    load(set0, 0);
    load(set1, 1);
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[i][j][v] = 0.0f;
    stage(set0, 0);
    load(set0, 2);
    __syncthreads();
    if (wk == 0) walk(std::integral_constant<bool, false>());
    else walk(std::integral_constant<bool, true>());
    const unsigned end = (last & 1) ? G::STAGE : 0;
    if (skip) {                                       // uniform; a row's first values by four threads
        constexpr int ROWS = I8 ? BM : BM + BN;       // (an int8 B times zeros is zero)
        for (int q = tid; q < ROWS * 4; q += T) {
            const int row = q % ROWS, r = row < BM ? row : row - BM;
            for (int k = q / ROWS; k < skip; k += 4) {
                if constexpr (TERMS) {
                    const unsigned base = end + (row < BM ? 0 : G::A_BYTES), plane = row < BM ? G::A_PLANE : G::B_PLANE;
#pragma unroll
                    for (int p = 0; p < 3; p++) *reinterpret_cast<unsigned short *>(lds + base + p * plane + G::at(r, k >> 3) + (k & 7) * 2) = 0;
                } else {
                    *reinterpret_cast<float *>(lds + end + (row < BM ? 0 : G::A_BYTES) + G::at(r, k >> 2) + (k & 3) * 4) = 0.0f;
                }
            }
        }
        __syncthreads();
    }
    multiply(end);
    if constexpr (OP == F32 || G::WORDS_INSIDE) __syncthreads();
    if constexpr (OP == F32) return false;
    if constexpr (APART) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) acc[i][j] += low[i][j];
    }
    float seen = 0.0f;
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) look_at(acc[i][j], seen);
    if (any_wave<8>(!(seen == 0.0f), lds + G::WORDS_AT, wave)) return true;
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] *= I8 ? 1.0f / TERMS_UP : TERMS_DOWN;      // (an int8 value is taken as it is)
    return false;
}

// The same sum for fp32 against int8 with fp32 instructions, operands straight from memory: the rare second pass.  The wave sets
// take pairs of k in turn.
template <int TM, int TN, int WN>
__device__ __forceinline__ void sum_range_i8_f32(const StagedArgs &g, int wave, int lane, int64_t m0, int64_t n0, v16f (&acc)[TM][TN]) {
    const int wk = wave >> 2, wm = (wave & 3) / WN, wn = (wave & 3) % WN, frow = lane & 31, fhalf = lane >> 5;
    const int64_t kbeg = (int64_t)blockIdx.z * g.k_range, kend = kbeg + g.k_range < g.K ? kbeg + g.k_range : g.K;
    const float *a[TM];
    const int8_t *b[TN];
#pragma unroll
    for (int i = 0; i < TM; i++) {
        const int64_t row = m0 + (wm * TM + i) * 32 + frow;
        a[i] = static_cast<const float *>(g.A) + (row < g.M ? row : g.M - 1) * g.lda;
    }
#pragma unroll
    for (int j = 0; j < TN; j++) {
        const int64_t col = n0 + (wn * TN + j) * 32 + frow;
        b[j] = static_cast<const int8_t *>(g.B) + (col < g.N ? col : g.N - 1) * g.ldb;
    }
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[i][j][v] = 0.0f;
    for (int64_t k0 = kbeg + 2 * wk; k0 < kend; k0 += 4) {           // uniform
        const int64_t k = k0 + fhalf;
        float fa[TM], fb[TN];
#pragma unroll
        for (int i = 0; i < TM; i++) fa[i] = k < kend ? a[i][k] : 0.0f;
#pragma unroll
        for (int j = 0; j < TN; j++) fb[j] = k < kend ? (float)b[j][k] : 0.0f;
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fb[j], fa[i], acc[i][j], 0, 0, 0);
    }
}

template <int BM, int BN, int WM, int WN, int BK, Op OP, bool A_KC, bool B_KC, int WAVES>
__global__ void __launch_bounds__(512, WAVES) k_gemm_staged(StagedArgs g) {
    using G = Geom<BM, BN, WM, WN, BK, OP>;
    constexpr int TM = G::TM, TN = G::TN, T = 512;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wk = wave >> 2, wm = (wave & 3) / WN, wn = (wave & 3) % WN;
    const int tiles_m = (int)((g.M + BM - 1) / BM), tiles_n = (int)((g.N + BN - 1) / BN);
    int tm, tn;
    int64_t batch = 0;
    if (gridDim.y == 1) tile_of_block(blockIdx.x, tiles_m, tiles_n, tm, tn);
    else tile_of_batched_block(tiles_m, tiles_n, tm, tn, batch);
    const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
    float *C = g.C + batch * g.stride_c + blockIdx.z * g.stride_z;
    v16f acc[TM][TN];
    const bool unfit = sum_range<BM, BN, WM, WN, BK, OP, A_KC, B_KC>(g, lds, wave, m0, n0, batch, acc);
    if constexpr (OP == SPLIT) {
        static_assert(2 * Geom<BM, BN, WM, WN, BK, F32>::STAGE <= G::BUFFERS, "the fp32 pass runs in the same LDS");
        if (unfit) sum_range<BM, BN, WM, WN, BK, F32, A_KC, B_KC>(g, lds, wave, m0, n0, batch, acc);
    }
    if constexpr (OP == I8W) {
        if (unfit) sum_range_i8_f32<TM, TN, WN>(g, wave, lane, m0, n0, acc);
    }

    // ---- the two sets added in LDS, then whole rows written back ----
    const int frow = lane & 31, fhalf = lane >> 5, arow = wm * TM * 32 + frow;
    float *tile = reinterpret_cast<float *>(lds);
    if (wk == 1) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int q = 0; q < 4; q++)
                    *reinterpret_cast<v4f *>(tile + (arow + 32 * i) * G::CPITCH + wn * TN * 32 + 32 * j + 8 * q + 4 * fhalf) =
                        v4f{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
    }
    __syncthreads();
    if (wk == 0) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    v4f *d = reinterpret_cast<v4f *>(tile + (arow + 32 * i) * G::CPITCH + wn * TN * 32 + 32 * j + 8 * q + 4 * fhalf);
                    *d = *d + v4f{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
                }
    }
    __syncthreads();
    constexpr int GROUPS = BN / 4, RSTEP = T / GROUPS;
    const int64_t col = n0 + (tid % GROUPS) * 4;
    const int have = g.N - col >= 4 ? 4 : (int)(g.N - col);               // columns of this thread's group that exist
    if (have <= 0) return;
    v4f cs = {1.f, 1.f, 1.f, 1.f}, bv = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 4; e++) {
        if (g.col_scale && e < have) cs[e] = g.col_scale[col + e];
        if (g.bias && e < have) bv[e] = g.bias[col + e];
    }
#pragma unroll
    for (int r = 0; r < BM / RSTEP; r++) {
        const int row = tid / GROUPS + r * RSTEP;
        if (m0 + row >= g.M) break;
        v4f o = *reinterpret_cast<const v4f *>(tile + row * G::CPITCH + (tid % GROUPS) * 4);
        float *cp = C + (m0 + row) * g.ldc + col;
        if (g.alpha != 1.0f) o *= g.alpha;
        if (g.col_scale) o *= cs;
        if (g.beta != 0.0f) {
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (e < have) o[e] += g.beta * cp[e];
        }
        if (g.bias) o += bv;
#pragma unroll
        for (int e = 0; e < 4; e++) o[e] = apply_act(o[e], g.act);
        if (have == 4) __builtin_memcpy(cp, &o, 16);
        else {
#pragma unroll
            for (int e = 0; e < 3; e++)
                if (e < have) cp[e] = o[e];
        }
    }
}

template <int BM, int BN, int WM, int WN, int BK, Op OP, bool A_KC, bool B_KC, int WAVES>
int launch_staged(const char *name, const StagedArgs &g, int64_t batch, int64_t splits) {
    using G = Geom<BM, BN, WM, WN, BK, OP>;
    auto kern = k_gemm_staged<BM, BN, WM, WN, BK, OP, A_KC, B_KC, WAVES>;
    // what the kernel relies on: a last slab is fetched from further left, never from before the row; 32-bit offsets
    if (g.K < BK || g.k_range < 1 || (g.k_range % BK != 0 && g.k_range < g.K) || (splits - 1) * g.k_range >= g.K || splits * g.k_range < g.K ||
        g.lda >= (1 << 22) || g.ldb >= (1 << 22))
        return fail(AXHIP_ERR_SHAPE, "%s: shape outside the staged tiles", name);
    static bool attr_set = false;
    if (!attr_set) {
        AXHIP_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, G::SMEM),
                      "hipFuncSetAttribute");
        attr_set = true;
    }
    const int64_t tiles = ((g.M + BM - 1) / BM) * ((g.N + BN - 1) / BN);
    note_kernel(name);
    hipLaunchKernelGGL(kern, dim3((unsigned)tiles, (unsigned)batch, (unsigned)splits), dim3(512), G::SMEM, kStream, g);
    return check_launch(name);
}

// ---- which tile, and into how many ranges of K -----------------------------------------------------------------------
// A tile and a number of ranges are chosen by the time they should take: what a launch costs once, and the rounds of workgroups
// over the CUs, times the slabs of a range at what a slab of that tile costs plus what a round costs besides (first loads,
// write-back); and for more than one range the finishing launch and its traffic.  The figures (us) of the fp32 and SPLIT tiles are
// fitted to some 1900 products and batches, every tile timed on each, K from 32 to 3000: predictions are within 6 % (64x64) to 10 %
// (128x128) on average, and the tile that is chosen within 1 % of the best one.  A round of the large tiles costs five times one of
// 64x64, two of which share a CU: with a K of one to eight slabs that decides (us, 128x128 -> 64x64: 338 x 294 x 294, K = 64 97 ->
// 80, 176 x 132 x 132, K = 34 32 -> 18, 383 x 279 x 279, K = 80 140 -> 112).
struct Plan {
    int tile;
    int64_t splits;
    float us;
};
struct TileCost {
    int bm, bn, bk;
    float slab_us, round_us, once_us;
};
Plan plan_staged(const StagedArgs &g, int64_t batch, const TileCost *tiles, int n, bool may_split) {
    const int64_t cus = cu_count(), forced = tuning().f32_splitk;     // 0: no AX_HIP_F32_SPLITK
    Plan best{-1, 1, 0.0f};
    for (int t = 0; t < n; t++) {
        const TileCost &c = tiles[t];
        if (g.K < c.bk) continue;
        const int64_t count = ((g.M + c.bm - 1) / c.bm) * ((g.N + c.bn - 1) / c.bn) * batch, slabs = (g.K + c.bk - 1) / c.bk;
        if (count > 0x7fffff) continue;                          // 512 threads each, and a grid holds fewer than 2^32: the guarded tiles have 256
        int64_t last = 0;
        for (int64_t per_cu = 0; per_cu <= 2; per_cu++) {        // no split, or as many ranges as give every CU one or two workgroups
            int64_t z = forced ? (count * 2 > cus ? 1 : forced) : per_cu == 0 ? 1 : per_cu * cus / count;
            if (z > g.K / 128) z = g.K / 128;
            if (z > 16) z = 16;
            if (z < 1 || (z > 1 && !may_split)) z = 1;
            if (z == last) continue;
            last = z;
            const int64_t per = (slabs + z - 1) / z;
            z = (slabs + per - 1) / per;                          // no empty range
            float us = c.once_us + (float)((count * z + cus - 1) / cus) * ((float)per * c.slab_us + c.round_us);
            if (z > 1) us += 3.0f + (float)(g.M * g.N) * (float)(z + 1) * (4.0f / 3.0e6f);
            if (best.tile < 0 || us < best.us) best = {t, z, us};
        }
    }
    return best;
}

template <typename F>
int run_plan(const StagedArgs &g, const Plan &p, int bk, const char *split_name, F &&launch) {
    if (p.splits == 1) return launch(g);
    float *part = static_cast<float *>(workspace((size_t)p.splits * g.M * g.N * sizeof(float)));
    if (!part) return AXHIP_ERR_ALLOC;
    StagedArgs a = g;
    const int64_t slabs = (g.K + bk - 1) / bk;
    a.k_range = (slabs + p.splits - 1) / p.splits * bk;
    a.C = part;
    a.ldc = g.N;
    a.stride_z = g.M * g.N;
    a.alpha = 1.0f;
    a.beta = 0.0f;
    a.bias = nullptr;
    a.act = AXHIP_ACT_NONE;
    if (int rc = launch(a)) return rc;
    const int rc = splitk_finish(part, p.splits, g.M, g.N, g.alpha, g.beta, g.bias, g.act, g.C, g.ldc);
    note_kernel(split_name);
    return rc;
}

const TileCost kF32Tiles[] = {{64, 64, 32, 0.56f, 1.1f, 3.3f}, {128, 128, 32, 1.92f, 6.5f, 0.8f}};
const TileCost kSplitTiles[] = {{128, 128, 32, 1.20f, 6.5f, 0.3f}, {128, 64, 32, 0.74f, 5.0f, 0.4f}, {64, 128, 32, 0.77f, 4.8f, 0.9f}, {64, 64, 32, 0.45f, 1.4f, 3.0f}};
const TileCost kI8Tiles[] = {{32, 128, 64, 0.57f, 2.5f, 1.0f}, {64, 128, 64, 0.90f, 2.5f, 1.0f}, {64, 256, 64, 1.52f, 2.5f, 1.0f}};

template <bool A_KC, bool B_KC>
int run_f32(const StagedArgs &g, int64_t batch, bool may_split, const char *const names[2], const char *split_name) {
    const Plan p = plan_staged(g, batch, kF32Tiles, 2, may_split && batch == 1);
    if (p.tile < 0) return -1;
    return run_plan(g, p, kF32Tiles[p.tile].bk, split_name, [&](const StagedArgs &a) {
        return p.tile == 0 ? launch_staged<64, 64, 2, 2, 32, F32, A_KC, B_KC, 4>(names[0], a, batch, p.splits)
                           : launch_staged<128, 128, 2, 2, 32, F32, A_KC, B_KC, 2>(names[1], a, batch, p.splits);
    });
}
template <bool A_KC, bool B_KC>
int run_split(const StagedArgs &g, int64_t batch, bool may_split, const char *const names[4], const char *split_name) {
    const Plan p = plan_staged(g, batch, kSplitTiles, 4, may_split && batch == 1);
    if (p.tile < 0) return -1;
    return run_plan(g, p, kSplitTiles[p.tile].bk, split_name, [&](const StagedArgs &a) {
        switch (p.tile) {
            case 0: return launch_staged<128, 128, 2, 2, 32, SPLIT, A_KC, B_KC, 2>(names[0], a, batch, p.splits);
            case 1: return launch_staged<128, 64, 2, 2, 32, SPLIT, A_KC, B_KC, 2>(names[1], a, batch, p.splits);
            case 2: return launch_staged<64, 128, 2, 2, 32, SPLIT, A_KC, B_KC, 2>(names[2], a, batch, p.splits);
            default: return launch_staged<64, 64, 2, 2, 32, SPLIT, A_KC, B_KC, 4>(names[3], a, batch, p.splits);
        }
    });
}
}  // namespace

namespace axhip {
int split_f32(const StagedArgs &g, int transa, int transb, int64_t batch, bool may_split) {
    static const char *const nn[4] = {"sgemm_nn_128x128x3_staged", "sgemm_nn_128x64x3_staged", "sgemm_nn_64x128x3_staged", "sgemm_nn_64x64x3_staged"};
    static const char *const nt[4] = {"sgemm_nt_128x128x3_staged", "sgemm_nt_128x64x3_staged", "sgemm_nt_64x128x3_staged", "sgemm_nt_64x64x3_staged"};
    static const char *const tn[4] = {"sgemm_tn_128x128x3_staged", "sgemm_tn_128x64x3_staged", "sgemm_tn_64x128x3_staged", "sgemm_tn_64x64x3_staged"};
    if ((transa && transb) || g.K < 32 || g.lda >= (1 << 22) || g.ldb >= (1 << 22) || batch > 65535) return -1;
    if (!transa && !transb) return run_split<true, false>(g, batch, may_split, nn, kSplitTermsName);
    if (!transa) return run_split<true, true>(g, batch, may_split, nt, kSplitTermsName);
    return run_split<false, false>(g, batch, may_split, tn, kSplitTermsName);
}

StagedChoice split_choice(const StagedArgs &g) {
    const Plan p = plan_staged(g, 1, kSplitTiles, 4, true);
    return {p.tile == 0, p.splits, p.us};
}
bool split_is_128x128(const StagedArgs &g, int64_t batch) { return g.K >= 64 && plan_staged(g, batch, kSplitTiles, 4, false).tile == 0; }

int staged_f32(const StagedArgs &g, int transa, int transb, int64_t batch, bool may_split) {
    static const char *const nn[2] = {"sgemm_nn_64x64k2_staged", "sgemm_nn_128x128k2_staged"};
    static const char *const nt[2] = {"sgemm_nt_64x64k2_staged", "sgemm_nt_128x128k2_staged"};
    static const char *const tn[2] = {"sgemm_tn_64x64k2_staged", "sgemm_tn_128x128k2_staged"};
    if ((transa && transb) || g.K < 32 || g.lda >= (1 << 22) || g.ldb >= (1 << 22) || batch > 65535) return -1;
    if (!transa && !transb) return run_f32<true, false>(g, batch, may_split, nn, "sgemm_splitk");
    if (!transa) return run_f32<true, true>(g, batch, may_split, nt, "sgemm_splitk");
    return run_f32<false, false>(g, batch, may_split, tn, "sgemm_splitk");
}

int staged_i8w(const StagedArgs &g) {
    if (g.K < 64 || g.lda >= (1 << 22) || g.ldb >= (1 << 22)) return -1;
    const Plan p = plan_staged(g, 1, kI8Tiles, 3, true);
    if (p.tile < 0) return -1;
    return run_plan(g, p, 64, "qgemm_w8a32_mfma_splitk", [&](const StagedArgs &a) {
        switch (p.tile) {
            case 0: return launch_staged<32, 128, 1, 4, 64, I8W, true, true, 4>("qgemm_w8a32_mfma_32x128k2_staged", a, 1, p.splits);
            case 1: return launch_staged<64, 128, 2, 2, 64, I8W, true, true, 4>("qgemm_w8a32_mfma_64x128k2_staged", a, 1, p.splits);
            default: return launch_staged<64, 256, 1, 4, 64, I8W, true, true, 2>("qgemm_w8a32_mfma_64x256k2_staged", a, 1, p.splits);
        }
    });
}
}  // namespace axhip
