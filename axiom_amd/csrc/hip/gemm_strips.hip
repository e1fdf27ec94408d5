// Single fp32 products with few tiles, in one launch: a workgroup of four to sixteen waves owns one 32x32 tile of C, or one range of K of it, and
// every wave forms the whole tile over its own strip of K, straight from memory, in three bf16 terms per operand (bf16x3.h); the strips meet
// in LDS, in a fixed order, and the ranges in memory, where the last workgroup of a tile to arrive adds them, in a fixed order too.
//
// What bounds such products is not the matrix core but latency: the launch, the first trip to memory, the loop's barriers where waves
// share slabs through LDS, and a second launch where K is cut into ranges to fill the chip.  Here the chip is filled by small tiles, no wave
// waits for another before the end, and a value is cut once per tile.  Two steps of 16 k are under way per wave.
// us, before -> here (on what), cached operands: 128 x 1024 x 784 11.6 -> 7.9, 300 x 333 x 777 11.1 -> 8.6, 1024 x 256 x 1024 12.3 -> 8.6 (two launches: ranges of K), 40 x
// 500 x 300 9.5 -> 5.9 (64x64 tiles in bf16 terms), 1024 x 256 x 256 5.9 -> 5.1 (32x64 tiles on fp32 instructions), 128 x 1024 x 10 6.6 -> 3.9 (guarded
// tiles), 1024 x 256 x 256 A^T B 9.5 -> 5.0; geometric mean over 2612 random products that the rule below takes 1.33, operands from HBM 1.31 (in terms 1.41
// and 1.38).  Past it the vector pipe (6.5 instructions a value and 64 values a column of k) and the loads (64 rows a tile) take over: 1024^3 20 ->
// 25, 100 x 10 x 4096 11 -> 22.
// The five smaller products of terms have a sum of their own, the others one, or two in turn where a wave has the registers (eight waves with one
// tile a CU), and the strips are added in pairs: relative error against 64 bits 7.1e-8 at K = 1024 on eight or sixteen waves (ranges of K in terms
// 7.6e-8, 64x64 tiles in terms 1.2e-7, fp32 instructions 4.1e-7), on four 8.1e-8 at K = 784 (ranges 8.1e-8).  A sum with a single product that is
// not zero is off by up to 1.7 units of 2^-24, where fp32 instructions round it (1.0).
//
// Loads.  An operand stored along K against one stored across it: a lane reads its 32 bytes of its row in place.  Both along K
// (A B^T): twice as many scattered lines would bound the kernel (1024 x 256 x 1024 21 us), so 64-byte pieces are loaded 16 rows at a time and
// turned through 2 KiB of LDS of the wave's own (9.3).  Stored across K: one k of 32 rows a load.  Rows and columns past the end are
// read as the last one, k past the end as the last one with A zero, and B too on fp32 instructions: zero times an infinity there would be
// a NaN, which in terms shows in the sum and sends the tile through the second pass.  Every alignment and every K is taken.
#include "gemm_strips.h"

#include "bf16x3.h"

namespace {
using namespace axhip;

constexpr int TILE = 32, CPITCH = TILE + 4, PART = TILE * CPITCH;        // floats of a wave's part of the tile

struct Meeting {                 // of ranges of K: a part of each tile for each, a counter for each tile
    float *parts;
    int *arrivals;
};

// RANGES: the workgroup has the range blockIdx.y of K (an argument of the kernel without it costs one with K = 256 0.3 us).
template <int WAVES, bool TERMS, bool A_KC, bool B_KC, int PER_SIMD, bool RANGES>
__global__ void __launch_bounds__(64 * WAVES, PER_SIMD) k_gemm_strips(StagedArgs g, std::conditional_t<RANGES, Meeting, int> meeting) {
    constexpr bool TURN = A_KC && B_KC;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r32 = lane & 31, h = lane >> 5;
    int tm, tn;
    tile_of_block(blockIdx.x, (int)((g.M + TILE - 1) / TILE), (int)((g.N + TILE - 1) / TILE), tm, tn);
    const int64_t m0 = (int64_t)tm * TILE, n0 = (int64_t)tn * TILE, lda4 = g.lda * 4, ldb4 = g.ldb * 4;
    const char *abase = reinterpret_cast<const char *>(static_cast<const float *>(g.A) + (A_KC ? m0 * g.lda : m0));
    const char *bbase = reinterpret_cast<const char *>(static_cast<const float *>(g.B) + (B_KC ? n0 * g.ldb : n0));
    const int mlast = (int)(g.M - 1 - m0 < TILE - 1 ? g.M - 1 - m0 : TILE - 1), nlast = (int)(g.N - 1 - n0 < TILE - 1 ? g.N - 1 - n0 : TILE - 1);
    // steps of 16 k; this workgroup's are `steps` from `first` on, this wave's strip of them is [s0, s1)
    int first = 0, steps = (int)((g.K + 15) / 16);
    if constexpr (RANGES) {
        const int64_t all = steps;
        first = (int)(all * blockIdx.y / gridDim.y);
        steps = (int)(all * (blockIdx.y + 1) / gridDim.y) - first;
    }
    const int s0 = first + (int)((int64_t)steps * wave / WAVES), s1 = first + (int)((int64_t)steps * (wave + 1) / WAVES);

    // ---- loads: in place, a lane's 8 k (8 h + e) of row r32; turned, four k of rows 16 q + lane / 4 ----
    std::integral_constant<bool, A_KC> akc;
    std::integral_constant<bool, B_KC> bkc;
    auto chunk = [&](int q) { return TURN ? lane & 3 : 2 * h + q; };
    auto offset = [&](auto kc, int64_t ld4, int last, int q) {
        constexpr bool KC = decltype(kc)::value;
        const int r = TURN ? 16 * q + (lane >> 2) : r32, row = r < last ? r : last;
        return (unsigned)row * (unsigned)(KC ? ld4 : 4) + (KC ? chunk(q) * 16 : (unsigned)(8 * h) * (unsigned)ld4);
    };
    const unsigned oa[2] = {offset(akc, lda4, mlast, 0), offset(akc, lda4, mlast, 1)}, ob[2] = {offset(bkc, ldb4, nlast, 0), offset(bkc, ldb4, nlast, 1)};
    auto load_rows = [&](auto kc, const char *base, int64_t ld4, const unsigned (&o)[2], int s, bool zero_past, float (&x)[8]) {
        const int64_t k = (int64_t)s * 16;
        const int end = (int)(g.K - 1 - k);            // the last k there is, from this step's first
        if constexpr (decltype(kc)::value) {
            const char *p = base + k * 4;
            if (end >= 15) {
#pragma unroll
                for (int q = 0; q < 2; q++) __builtin_memcpy(&x[4 * q], p + o[q], 16);
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const int past = end - (4 * chunk(e >> 2) + (e & 3));          // below zero: past the end
                    const float y = *reinterpret_cast<const float *>(p + o[e >> 2] + ((e & 3) + (past < 0 ? past : 0)) * 4);
                    x[e] = zero_past && past < 0 ? 0.0f : y;
                }
            }
        } else {
            const char *p = base + k * ld4;
            if (end >= 15) {
#pragma unroll
                for (int e = 0; e < 8; e++) x[e] = *reinterpret_cast<const float *>(p + e * ld4 + o[0]);
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const int past = end - (8 * h + e);
                    const float y = *reinterpret_cast<const float *>(p + (int64_t)(e + (past < 0 ? past : 0)) * ld4 + o[0]);
                    x[e] = zero_past && past < 0 ? 0.0f : y;
                }
            }
        }
    };
    struct Raw {
        float a[8], b[8];
    };
    auto load = [&](Raw &r, int s) {
        load_rows(akc, abase, lda4, oa, s, true, r.a);
        load_rows(bkc, bbase, ldb4, ob, s, !TERMS, r.b);
    };
    // chunks lie in rows of 64 bytes, exchanged by the row so that the 16 lanes that an access serves together fall on distinct banks
    auto turn = [&](unsigned char *d, float (&a)[8], float (&b)[8]) {
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const int row = 16 * q + (lane >> 2);
            const unsigned at = row * 64 + (((lane & 3) ^ ((row >> 2) & 3)) << 4);
            *reinterpret_cast<v4f *>(d + at) = v4f{a[4 * q], a[4 * q + 1], a[4 * q + 2], a[4 * q + 3]};
            *reinterpret_cast<v4f *>(d + 2048 + at) = v4f{b[4 * q], b[4 * q + 1], b[4 * q + 2], b[4 * q + 3]};
        }
        order_in_wave();
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const unsigned at = r32 * 64 + (((2 * h + q) ^ ((r32 >> 2) & 3)) << 4);
            const v4f y = *reinterpret_cast<const v4f *>(d + at), z = *reinterpret_cast<const v4f *>(d + 2048 + at);
#pragma unroll
            for (int e = 0; e < 4; e++) a[4 * q + e] = y[e], b[4 * q + e] = z[e];
        }
        order_in_wave();
    };

    // steps in turn into two sums, where there are registers for them
    constexpr bool TURNS = TERMS && PER_SIMD <= 2;
    v16f acc, other, low;
#pragma unroll
    for (int v = 0; v < 16; v++) acc[v] = other[v] = low[v] = 0.0f;
    auto multiply = [&](Raw &r, v16f &acc) {
        if constexpr (TURN) turn(lds + wave * 4096, r.a, r.b);
        if constexpr (!TERMS) {
#pragma unroll
            for (int e = 0; e < 8; e++) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(r.b[e], r.a[e], acc, 0, 0, 0);
            return;
        }
        v4i fa[3], fb[3];
        cut(r.a, TERMS_UP, fa);
        cut(r.b, TERMS_UP, fb);
#pragma unroll
        for (int sum = 2; sum > 0; sum--)              // the small products first
#pragma unroll
            for (int p = sum; p >= 0; p--) low = mfma_terms(fb[sum - p], fa[p], low);
        acc = mfma_terms(fb[0], fa[0], acc);
    };
    if (s0 < s1) {
        Raw r0, r1;
        load(r0, s0);
        load(r1, s0 + 1 < s1 ? s0 + 1 : s0);
        int s = s0;
        for (; s + 2 < s1; s += 2) {
            multiply(r0, acc);
            load(r0, s + 2);
            multiply(r1, TURNS ? other : acc);
            load(r1, s + 3 < s1 ? s + 3 : s);          // (not the last step twice, which is slow where K ends inside it: 500 x 300 x 300 5.9 -> 5.7)
        }
        multiply(r0, acc);
        if (s + 1 < s1) multiply(r1, TURNS ? other : acc);
    }
    if constexpr (TURN) __syncthreads();               // the parts lie where values were turned

    // ---- the strips together: register v of lane l holds row l & 31, column 8 (v >> 2) + 4 (l >> 5) + (v & 3) ----
    float seen = 0.0f;
    if constexpr (TERMS) {
        if constexpr (TURNS) acc += other;
        acc += low;
        look_at(acc, seen);
    }
    float *part = reinterpret_cast<float *>(lds);
    auto put = [&](float by) {
#pragma unroll
        for (int q = 0; q < 4; q++)
            *reinterpret_cast<v4f *>(part + wave * PART + r32 * CPITCH + 8 * q + 4 * h) =
                v4f{acc[4 * q] * by, acc[4 * q + 1] * by, acc[4 * q + 2] * by, acc[4 * q + 3] * by};
    };
    // Strips that are finite in themselves may exceed the largest float together while they hold the factor of the terms: each gives up a
    // WAVES-th of it first (exactly: nothing that reaches C is that small), the rest goes once they are added.
    put(TERMS ? 1.0f / WAVES : 1.0f);
    float down = TERMS ? TERMS_DOWN * WAVES : 1.0f;
    if constexpr (!TERMS) __syncthreads();
    else if (any_wave<WAVES>(!(seen == 0.0f), lds + WAVES * PART * 4, wave)) {
        // what the terms cannot hold, with fp32 instructions: the waves take pairs of k in turn
        down = 1.0f;
#pragma unroll
        for (int v = 0; v < 16; v++) acc[v] = 0.0f;
        const int row = r32 < mlast ? r32 : mlast, col = r32 < nlast ? r32 : nlast;
        const int64_t kend = RANGES && (int64_t)(first + steps) * 16 < g.K ? (int64_t)(first + steps) * 16 : g.K;
        for (int64_t k0 = (int64_t)first * 16 + 2 * wave; k0 < kend; k0 += 2 * WAVES) {
            const int64_t k = k0 + h, ke = k < kend ? k : kend - 1;
            const float a = *reinterpret_cast<const float *>(abase + (A_KC ? row * lda4 + ke * 4 : ke * lda4 + row * 4));
            const float b = *reinterpret_cast<const float *>(bbase + (B_KC ? col * ldb4 + ke * 4 : ke * ldb4 + col * 4));
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(k < kend ? b : 0.0f, k < kend ? a : 0.0f, acc, 0, 0, 0);
        }
        put(1.0f);
        __syncthreads();
    }
    const int row = tid / 8, cg = (tid & 7) * 4;       // four columns of a row each, from the first 256 threads
    const int64_t m = m0 + row, col = n0 + cg;
    if (tid >= TILE * TILE / 4) return;                // (whole waves: they no longer count at barriers)
    v4f p[WAVES];                                      // added in pairs (sixteen in a row: error 8.9e-8 at K = 1024)
#pragma unroll
    for (int w = 0; w < WAVES; w++) p[w] = *reinterpret_cast<const v4f *>(part + w * PART + row * CPITCH + cg);
#pragma unroll
    for (int by = 1; by < WAVES; by *= 2)
#pragma unroll
        for (int w = 0; w < WAVES; w += 2 * by) p[w] += p[w + by];
    v4f o = p[0];
    o *= down;
    if constexpr (RANGES) {
        // The ranges meet in memory: every workgroup leaves its part, and the last one to arrive on the tile's counter adds them in order.  Parts, counter
        // and the reads below are device-scope accesses (the workgroups run on XCDs with an L2 each); the wait makes a thread's stores complete before the
        // barrier, the barrier orders them before thread 0's increment.
        typedef float v2f __attribute__((ext_vector_type(2)));
        const int ranges = gridDim.y;
        int64_t *slots = reinterpret_cast<int64_t *>(meeting.parts + (int64_t)blockIdx.x * ranges * (TILE * TILE)) + 2 * tid;
        constexpr int STRIDE = TILE * TILE / 2;
        __hip_atomic_store(slots + blockIdx.y * STRIDE, __builtin_bit_cast(int64_t, v2f{o[0], o[1]}), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(slots + blockIdx.y * STRIDE + 1, __builtin_bit_cast(int64_t, v2f{o[2], o[3]}), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        int *last = reinterpret_cast<int *>(lds + WAVES * PART * 4);
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        if (tid == 0) *last = __hip_atomic_fetch_add(meeting.arrivals + blockIdx.x, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == ranges - 1;
        __syncthreads();
        if (!*last) return;
        o = v4f{0.f, 0.f, 0.f, 0.f};
        for (int r0 = 0; r0 < ranges; r0 += 8) {
            v2f x[8][2];
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const int r = r0 + u < ranges ? r0 + u : ranges - 1;
#pragma unroll
                for (int e = 0; e < 2; e++) x[u][e] = __builtin_bit_cast(v2f, __hip_atomic_load(slots + r * STRIDE + e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
                if (r0 + u >= ranges) x[u][0] = x[u][1] = v2f{0.f, 0.f};
            }
#pragma unroll
            for (int by = 1; by < 8; by *= 2)
#pragma unroll
                for (int u = 0; u < 8; u += 2 * by) {
                    x[u][0] += x[u + by][0];
                    x[u][1] += x[u + by][1];
                }
            o += v4f{x[0][0][0], x[0][0][1], x[0][1][0], x[0][1][1]};
        }
        if (tid == 0) __hip_atomic_store(meeting.arrivals + blockIdx.x, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);      // ready for the next launch
    }
    if (m >= g.M || col >= g.N) return;
    const int have = g.N - col >= 4 ? 4 : (int)(g.N - col);
    float *cp = g.C + m * g.ldc + col;
    if (g.alpha != 1.0f) o *= g.alpha;
#pragma unroll
    for (int e = 0; e < 4; e++)
        if (e < have) {
            if (g.beta != 0.0f) o[e] += g.beta * cp[e];
            if (g.bias) o[e] += g.bias[col + e];
            o[e] = apply_act(o[e], g.act);
        }
    if (have == 4) __builtin_memcpy(cp, &o, 16);
    else {
#pragma unroll
        for (int e = 0; e < 3; e++)
            if (e < have) cp[e] = o[e];
    }
}

template <int WAVES, bool TERMS, bool A_KC, bool B_KC, int PER_SIMD, bool RANGES = false>
int launch(const char *name, const StagedArgs &g, int64_t ranges = 1) {
    constexpr int SMEM = WAVES * PART * 4 + 4 * WAVES;
    static_assert(!(A_KC && B_KC) || WAVES * 4096 <= SMEM, "values are turned where the parts come to lie");
    auto kern = k_gemm_strips<WAVES, TERMS, A_KC, B_KC, PER_SIMD, RANGES>;
    static bool attr_set = false;
    if (!attr_set) {
        AXHIP_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, SMEM), "hipFuncSetAttribute");
        attr_set = true;
    }
    const int64_t tiles = ((g.M + TILE - 1) / TILE) * ((g.N + TILE - 1) / TILE);
    std::conditional_t<RANGES, Meeting, int> meeting{};
    if constexpr (RANGES) {
        meeting.parts = static_cast<float *>(workspace((size_t)(tiles * ranges * TILE * TILE) * sizeof(float)));
        meeting.arrivals = strip_counters((size_t)tiles);
        if (!meeting.parts || !meeting.arrivals) return AXHIP_ERR_ALLOC;
    }
    note_kernel(name);
    hipLaunchKernelGGL(kern, dim3((unsigned)tiles, (unsigned)ranges), dim3(64 * WAVES), SMEM, kStream, g, meeting);
    return check_launch(name);
}
}  // namespace

namespace axhip {
// In terms from K = 113 on.  The limits to K lie where the geometric mean of the gains with operands cached and operands from HBM falls to one: two
// steps under way wait longer for memory than the kernels behind, which gain as much there as they lose cached, and have a second launch to be issued
// (a training step of a 384-896-216 classifier, batch 160, 70.6 us with 160 x 216 x 896 here and 74.3 on ranges of K).  us, before -> here, cached / from
// HBM: 1024 x 256 x 1024 12.3 / 12.7 -> 8.5 / 10.1, 384 x 128 x 700 10.5 / 11.0 -> 7.3 / 9.0, 128 x 10 x 1024 9.4 / 9.6 -> 7.8 / 8.4, A B^T 256 x 768 x 896 11.5 / 12.5
// -> 8.3 / 9.6, 500 x 300 x 640 11.0 / 11.9 -> 7.1 / 8.4, A^T B 1024 x 256 x 1280 13.1 / 13.5 -> 10.4 / 11.7, 97 x 31 x 1000 9.9 / 10.1 -> 8.3 / 8.9; near the limits 1588 x
// 22 x 973 9.8 / 10.5 -> 8.6 / 12.0, 1446 x 65 x 1208 11.8 / 12.8 -> 10.2 / 14.0, past them A B^T 57 x 1598 x 893 9.9 / 11.3 -> 8.9 / 12.7, 96 x 64 x 896 7.3 / 7.4 -> 7.8 / 8.2, 72 x 1354 x 1317 12.3 / 13.6 -> 13.4 / 14.7;
// 1024 x 1024 x 256 cached 8.2 -> 9.5, and A B^T on 336 tiles with K = 476, with its extra turn, 8.9 -> 9.7.
// Two workgroups share a CU from 257 tiles on: four waves each (86 x 3584 x 300: eight 6.4, four 5.6); but
// eight on up to a third of the CUs with K above 400, where ranges of K on 64x64 tiles would have the smaller error than four long strips (geometric
// mean over 51 products 1.03 of theirs with four, at most 1.09; 0.94 with eight, times 1.05 in A B and 0.96 in A^T B of four's), and none there above
// K = 640 (127 x 2125 x 705 13.7 -> 15.3, 2186 x 104 x 699 from HBM 13.0 -> 14.9).  Off the 16-byte grid four too up to K = 176,
// where eight strips of a step or two leave a larger error than the staged tiles in terms that they stand before (geometric means over some
// hundred products: eight 1.05 of theirs at K = 129..144, 1.02 at 145..160, 1.01 at 161..168, 0.99 from 177 on, four 0.99, 0.98, 0.96 and, of
// uniform values, 1.00 at 121..128), and none up to K = 120 (four 1.07 at 64..80, 1.01 at 113..120).  On the grid the kernels before were on fp32 instructions, with three times the error.
// Sixteen pay where A is stored across K, whose loads are the slowest, above K = 256 (256 x 1000 x 500 6.6 -> 6.1; 250 x 500 x 256 4.5 -> 5.2).
// A K past that, or past 760 with up to 64 tiles, in ranges, which meet in the same launch: for a narrow result two launches had cost their floor twice, and a few
// workgroups of eight waves each wait for memory through their strip.  us, before -> here: 100 x 10 x 4096 10.8 -> 7.9, 128 x 10 x 1024 8.6 -> 5.7, 64 x
// 256 x 2048 A^T B 8.7 -> 7.7, 100 x 100 x 4096 9.2 -> 8.9 (on the 16-byte grid with whole K from fp32 instructions: fewer bits in a sum of one product, 1.7 in place of 1 unit of 2^-24).  Geometric means over 800 random products, before over here, and the error over that of before: up to 32 tiles
// K = 761..960 1.18 to 1.28 (four ranges of four waves, 1.00 of the strips' and 0.7 of the others' error), ..1300 1.36 to 1.45 (eight), ..4608 1.14 to 1.43
// (eight of eight waves, 0.6 to 0.8); 33 to 64 tiles ..1024 1.07 to 1.36, ..2600 1.03 to 1.31; 65 to 100 tiles, cached and
// from HBM, A B 961..1600 1.12 and 1.07, A^T B ..1950 1.13 and 1.10 (on the grid ..2600 1.10 and 1.08), A B^T ..1280 1.05 and 1.06; past these A B 0.94 to 1.1 and 0.87 to 1.06, A^T B off the grid 0.86 to 1.1, A B^T 0.78 to 1.0
// and 0.70 to 0.88 (86 tiles, K = 2322 10.7 -> 13.9, from HBM 12.5 -> 17.5: three workgroups a CU, each with a turn through LDS).  Below K = 760 the parts are
// so short that adding them costs accuracy (1.01 to 1.05 for 1.0 to 1.2 of the speed), past 100 tiles the chip is full (0.7 to 1.0); sixteen ranges 0.8 to 1.0 of eight.  A longer K on
// 33 to 100 tiles is behind (2610 to 3320 0.92 to 1.09, 4700 to 8000 0.72 to 0.93); up to 32 tiles it is ahead still (49 of 50 up to 15900 1.06 to 1.45), but its error is not compared there.
// On fp32 instructions up to K = 63 off the grid and 112 on it, where the kernels before are on them too: there is little to multiply and nothing to
// cut.  Four waves, up to two tiles a CU (geometric means over some hundred products a range, cached / from HBM, and the error over that of the
// kernels before: K below 32 1.3 / 1.3, 0.99; 32..63 off the grid 1.31 / 1.29, 0.86, on it 1.22 / 1.21, 0.74; 64..112 on the grid 1.32 / 1.31, 0.64; strips in
// terms 1.17 / 1.18 there.  us: 128 x 1024 x 10 6.6 -> 3.9, A B^T 6.3 -> 3.5, 784 x 40 x 20 A^T B 4.5 -> 4.1).
int strips_f32(const StagedArgs &g, int transa, int transb, bool on_grid) {
    if ((transa && transb) || g.K < 1 || g.lda >= (1 << 22) || g.ldb >= (1 << 22)) return -1;
    const int64_t tiles = ((g.M + TILE - 1) / TILE) * ((g.N + TILE - 1) / TILE), cus = cu_count();
    const bool one = tiles <= cus, two = tiles <= 2 * cus;
    if (two && g.K < (on_grid ? 113 : 64)) {
        if (!transa && !transb) return launch<4, false, true, false, 4>("sgemm_nn_strips32", g);
        if (!transa) return launch<4, false, true, true, 4>("sgemm_nt_strips32", g);
        return launch<4, false, false, false, 4>("sgemm_tn_strips32", g);
    }
    const bool many = tiles >= 128;
    const bool ranges_in_terms = !on_grid || g.K % 32 != 0;      // what stands behind a longer K: ranges on the staged tiles in terms, or on fp32 ones
    const int64_t most = many              ? (transb ? 1088 : g.M < 96 ? 1024 : 1536)
                         : ranges_in_terms ? (transb ? 864 : 1024)
                                           : (transb ? 832 : 896);
    const bool third = tiles * 3 <= cus * 4;                   // two workgroups on a third of the CUs at most
    const bool strips = (one && g.K <= most) || (two && !transb && g.K <= (third ? 640 : 800));
    // Few tiles and a long K: ranges of it, four to eight workgroups a tile.
    const int64_t waves = tiles <= 32 ? (g.K > 1300 ? 8 : 4) : tiles <= 64 && g.K > 1024 ? 8 : 4;
    const int64_t farthest = transb ? 1280 : !transa ? 1600 : on_grid ? 2600 : 1950;
    const int64_t ranges = g.K <= 760                ? 1
                           : tiles <= 32             ? (g.K <= 960 ? 4 : g.K <= 4608 ? 8 : 1)
                           : tiles <= 64             ? (g.K <= 2600 ? 4 : 1)
                           : tiles <= 100            ? (g.K > 960 && g.K <= farthest ? 8 : 1)
                                                     : 1;
    if (ranges > 1) {
        const char *name = transa ? "sgemm_tn_ranges32x3" : transb ? "sgemm_nt_ranges32x3" : "sgemm_nn_ranges32x3";
        if (!transa && !transb) return waves == 8 ? launch<8, true, true, false, 2, true>(name, g, ranges) : launch<4, true, true, false, 4, true>(name, g, ranges);
        if (!transa) return waves == 8 ? launch<8, true, true, true, 2, true>(name, g, ranges) : launch<4, true, true, true, 4, true>(name, g, ranges);
        return waves == 8 ? launch<8, true, false, false, 2, true>(name, g, ranges) : launch<4, true, false, false, 4, true>(name, g, ranges);
    }
    if (g.K <= (on_grid ? 112 : 120) || !strips) return -1;
    if (!one && third && g.K > 400)
        return transa ? launch<8, true, false, false, 4>("sgemm_tn_strips32x3", g) : launch<8, true, true, false, 4>("sgemm_nn_strips32x3", g);
    const bool four = !one || (!on_grid && g.K <= 176);
    if (!transa && !transb)
        return four ? launch<4, true, true, false, 4>("sgemm_nn_strips32x3", g) : launch<8, true, true, false, 2>("sgemm_nn_strips32x3", g);
    if (!transa) return four ? launch<4, true, true, true, 4>("sgemm_nt_strips32x3", g) : launch<8, true, true, true, 2>("sgemm_nt_strips32x3", g);
    if (four) return launch<4, true, false, false, 4>("sgemm_tn_strips32x3", g);
    return g.K <= 256 ? launch<8, true, false, false, 2>("sgemm_tn_strips32x3", g) : launch<16, true, false, false, 4>("sgemm_tn_strips32x3", g);
}
}  // namespace axhip
