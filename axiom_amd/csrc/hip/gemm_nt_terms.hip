// C = alpha * A * B^T for batches of products with a short K (Q K^T of attention heads: K = the head size) on the bf16 matrix
// core: both operands in three bf16 terms, six products of terms for one of values (bf16x3.h).
//
// What bounds it: writing C (one float for every K products), beside the matrix core.  A workgroup of eight waves owns 256 columns
// of one entry and walks its rows: a wave keeps the terms of its 32 columns of B in registers for the whole walk, blocks of 64
// rows of A are cut once per workgroup on their way from registers to LDS (two blocks there, the next one in registers), and a
// lane owns one column of the 32x32 tiles, so that a store instruction writes two whole 128-byte rows.
// us, fp32 instructions -> this: 512 heads of 512 x 512, K = 64 167 -> 131 (4.6 TB/s; with plain stores 153), K = 128 with 256 of
// them 147 -> 115, 128 of 1024 x 1024, K = 64 163 -> 124, K = 128 276 -> 213; off the 256 grid 256 of 333 x 333, K = 64 69 -> 43, 64 of
// 1000 x 1000 116 -> 84, 512 of 200 x 200 55 -> 29.  Non-temporal stores where rows are no whole lines: 84 -> 111 (1000 x 1000).
// A walk with a sum that is not finite is done again with fp32 instructions.
#include "gemm_staged.h"

#include "bf16x3.h"

namespace {
using namespace axhip;

template <int K>
struct NtGeom {
    static constexpr int BM = 64, ROW = K * 2, PLANE = BM * ROW, STAGE = 3 * PLANE;      // rows of a block; bytes
    static constexpr int FLAGS_AT = 2 * STAGE, SMEM = FLAGS_AT + 32;
    static constexpr int E = K % 64 ? 4 : 8, PIECES = BM * K / 512 / E;                 // what a thread stages of a block
    // where the 16-byte chunk c of row r lies: the 16 lanes that an access serves fall on distinct banks
    __device__ static unsigned at(int row, int chunk) {
        const int key = ROW == 256 ? row & 15 : ROW == 128 ? (row >> 1) & 7 : (row >> 2) & 3;
        return (unsigned)(row * ROW + ((chunk ^ key) << 4));
    }
};

template <int E>
__device__ __forceinline__ void load_row(float (&x)[E], const float *p) {
#pragma unroll
    for (int h = 0; h < E / 4; h++) {
        const v4f a = *reinterpret_cast<const v4f *>(p + 4 * h);
#pragma unroll
        for (int e = 0; e < 4; e++) x[4 * h + e] = a[e];
    }
}

// LINES: the rows of C lie on 128-byte lines.  Whole lines go out past the caches, which keep A and B; pieces of lines must not.
template <int K, bool LINES>
__global__ void __launch_bounds__(512, (K > 64 ? 2 : 4)) k_nt_terms(StagedArgs g) {
    using G = NtGeom<K>;
    constexpr int KS = K / 16;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int frow = lane & 31, fhalf = lane >> 5;
    const float *A = static_cast<const float *>(g.A) + blockIdx.y * g.stride_a, *B = static_cast<const float *>(g.B) + blockIdx.y * g.stride_b;
    float *C = g.C + blockIdx.y * g.stride_c;
    const int64_t n0 = (int64_t)blockIdx.x * 256 + wave * 32, col = n0 + frow;
    const float *brow = B + (col < g.N ? col : g.N - 1) * g.ldb;         // columns past the end repeat the last one and are not stored
    const bool idle = n0 >= g.N;
    const int64_t nblocks = (g.M + G::BM - 1) / G::BM;

    int prow[G::PIECES], pcol[G::PIECES];
    unsigned put[G::PIECES];
#pragma unroll
    for (int i = 0; i < G::PIECES; i++) {
        const int q = tid + i * 512, c = q % (K / G::E);
        prow[i] = q / (K / G::E);
        pcol[i] = c * G::E;
        put[i] = G::at(prow[i], c * G::E / 8) + c * G::E % 8 * 2;
    }
    float ar[G::PIECES][G::E];
    auto load = [&](int64_t blk) {
        const char *a = reinterpret_cast<const char *>(A + blk * G::BM * g.lda);
        const int64_t left = g.M - blk * G::BM;
        const int end = left < G::BM ? (int)left - 1 : G::BM - 1;
#pragma unroll
        for (int i = 0; i < G::PIECES; i++) load_row(ar[i], reinterpret_cast<const float *>(a + ((unsigned)(prow[i] < end ? prow[i] : end) * (unsigned)g.lda + pcol[i]) * 4));
    };
    auto stage = [&](unsigned at) {
#pragma unroll
        for (int i = 0; i < G::PIECES; i++) {
            Term<G::E> t[3];
            cut(ar[i], TERMS_UP, t);
#pragma unroll
            for (int p = 0; p < 3; p++) *reinterpret_cast<Term<G::E> *>(lds + at + put[i] + p * G::PLANE) = t[p];
        }
    };
    // register v of lane l: row 8*(v>>2) + 4*(l>>5) + (v&3), column l & 31
    const unsigned coff = (unsigned)(4 * fhalf * g.ldc + col) * 4;      // bytes from a row that is the same for the whole wave
    auto store = [&](const v16f &acc, int64_t row0) {
        if (col >= g.N) return;
        auto at = [&](int v) { return reinterpret_cast<float *>(reinterpret_cast<char *>(C + (row0 + 8 * (v >> 2) + (v & 3)) * g.ldc) + coff); };
        if (row0 + 32 <= g.M) {
#pragma unroll
            for (int v = 0; v < 16; v++) {
                if constexpr (LINES) __builtin_nontemporal_store(g.alpha * acc[v], at(v));
                else *at(v) = g.alpha * acc[v];
            }
        } else {
#pragma unroll
            for (int v = 0; v < 16; v++)
                if (row0 + 4 * fhalf + 8 * (v >> 2) + (v & 3) < g.M) *at(v) = g.alpha * acc[v];
        }
    };

    load(0);
    v4i bf[KS][3];
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
        float x[8];
        load_row(x, brow + 16 * ks + 8 * fhalf);
        cut(x, TERMS_UP, bf[ks]);
    }
    stage(0);
    if (nblocks > 1) load(1);
    __syncthreads();
    float seen = 0.0f;
    unsigned cur = 0;
    for (int64_t blk = 0; blk < nblocks; blk++, cur ^= G::STAGE) {
        if (blk + 1 < nblocks) {
            stage(cur ^ G::STAGE);
            if (blk + 2 < nblocks) load(blk + 2);
        }
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const int64_t row0 = blk * G::BM + 32 * t;
            if (idle || row0 >= g.M) break;
            v16f acc, low;                            // the five smaller products of terms in a sum of their own
#pragma unroll
            for (int v = 0; v < 16; v++) acc[v] = low[v] = 0.0f;
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {
                v4i af[3];
#pragma unroll
                for (int p = 0; p < 3; p++) af[p] = *reinterpret_cast<const v4i *>(lds + cur + G::at(frow, 2 * ks + fhalf) + t * 32 * G::ROW + p * G::PLANE);
#pragma unroll
                for (int sum = 2; sum > 0; sum--)
#pragma unroll
                    for (int p = sum; p >= 0; p--) low = mfma_terms(af[p], bf[ks][sum - p], low);
                acc = mfma_terms(af[0], bf[ks][0], acc);
            }
            acc += low;
            look_at(acc, seen);
            store(acc * TERMS_DOWN, row0);
        }
        __syncthreads();
    }

    if (!any_wave<8>(!(seen == 0.0f), lds + G::FLAGS_AT, wave) || idle) return;
    for (int64_t row0 = 0; row0 < g.M; row0 += 32) {
        const float *arow = A + (row0 + frow < g.M ? row0 + frow : g.M - 1) * g.lda;
        v16f acc;
#pragma unroll
        for (int v = 0; v < 16; v++) acc[v] = 0.0f;
        for (int k = 4 * fhalf; k < K; k += 8) {
            const v4f a = *reinterpret_cast<const v4f *>(arow + k), b = *reinterpret_cast<const v4f *>(brow + k);
#pragma unroll
            for (int e = 0; e < 4; e++) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], b[e], acc, 0, 0, 0);
        }
        store(acc, row0);
    }
}

template <int K, bool LINES>
int launch(const StagedArgs &g, int64_t batch) {
    using G = NtGeom<K>;
    static bool attr_set = false;
    if (!attr_set) {
        AXHIP_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(k_nt_terms<K, LINES>), hipFuncAttributeMaxDynamicSharedMemorySize, G::SMEM),
                      "hipFuncSetAttribute");
        attr_set = true;
    }
    note_kernel("sgemm_nt_cols256x3");
    hipLaunchKernelGGL((k_nt_terms<K, LINES>), dim3((unsigned)((g.N + 255) / 256), (unsigned)batch), dim3(512), G::SMEM, kStream, g);
    return check_launch("sgemm_nt_cols256x3");
}
template <int K>
int launch(const StagedArgs &g, int64_t batch) {
    const bool lines = ((uintptr_t)g.C & 127) == 0 && g.ldc % 32 == 0 && g.stride_c % 32 == 0;
    return lines ? launch<K, true>(g, batch) : launch<K, false>(g, batch);
}
}  // namespace

namespace axhip {
int nt_terms(const StagedArgs &g, int64_t batch) {
    if (g.K % 32 != 0 || g.K < 32 || g.K > 128 || g.M < 1 || g.N < 1 || g.beta != 0.0f || g.bias || g.col_scale || g.act != AXHIP_ACT_NONE) return -1;
    if ((((uintptr_t)g.A | (uintptr_t)g.B) & 15) != 0 || g.lda % 4 != 0 || g.ldb % 4 != 0 || g.stride_a % 4 != 0 || g.stride_b % 4 != 0 ||
        g.lda >= (1 << 22) || g.ldc >= (1 << 24) || g.N >= (1 << 24) || batch > 65535 || (g.N + 255) / 256 > 0x7fffffff)
        return -1;
    switch (g.K / 32) {
        case 1: return launch<32>(g, batch);
        case 2: return launch<64>(g, batch);
        case 3: return launch<96>(g, batch);
        default: return launch<128>(g, batch);
    }
}
}  // namespace axhip
