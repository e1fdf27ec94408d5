// Scaled dot-product attention forward: O = softmax(scale * Q K^T [+ causal mask]) V per head,
// Q, K, V, O [BH, S, dk] row-major fp32, L [BH, S] = log-sum-exp of each score row (or NULL).
//
// Fused kernel (dk a multiple of 4 up to 128, on the geometry of the next size among 32, 64, 96 and
// 128; any S): the score matrix never leaves the chip.  A workgroup of four or eight waves owns 128 or 256
// query rows of one head, a wave 32 of them; keys and values stream through LDS in blocks of 64 (32 for dk 128).
// Both products run on the bf16 matrix core with every fp32 operand cut into three bf16 terms (six
// products of terms for one of values, bf16x3.h): 6/16 of the matrix-core time of the fp32 instructions,
// which also share their lanes with the softmax's vector instructions.  K and V are cut once per
// workgroup on their way from registers to LDS, Q once per tile, a probability when it is used.  The
// query index is on the MFMA's column side, so lane l of a wave owns query (l & 31) in the score tile
// *and* in the output accumulator:
//   S^T tile:  A = K rows (32 keys), B = the wave's Q rows (terms held in registers for the whole tile);
//              register v of lane l = score(query l&31, key 8*(v>>2) + 4*(l>>5) + (v&3)).
//   softmax:   running maximum m and sum per query, the online form: the accumulator is
//              rescaled by 2^(m_old - m_new) when the maximum moves.  Row reductions are within
//              a lane plus one exchange with lane l^32.  Scores are kept in base-2 units
//              (scale * log2(e) folded in) so the exponential is the hardware's 2^x.
//   O^T tile:  A = V^T, B = the probabilities exactly where the score MFMA left them: registers 8s .. 8s+7
//              are the eight k of a 16-key step, V^T lies in LDS in that order of keys, and a sum over
//              keys does not care about their order.
// V is transposed by the registers (a thread loads eight keys of one column).  Rows of both operands
// are XOR-swizzled in 16-byte chunks, so the 16 lanes that a 16-byte access serves fall on distinct banks.
// A tile with a sum that is not finite is computed again with fp32 instructions by the same workgroup:
// infinities, NaNs and values near the largest float come out as fp32 products give them.
// us, fp32 instructions -> terms: 512 heads of [512, 64] 269 -> 194 (causal 178 -> 126), 64 of [1024, 128] 273 -> 174, 96 causal
// ones of [1000, 80] 324 -> 113 (a quarter of that from the 96-wide geometry; the matrix core is busy 43 % of the cycles, vector instructions some 34, and on zeros it takes 97), 512 of [256, 32] 41 -> 33; with few query tiles for the
// CUs k_sdpa_few cuts a head along its keys too (32 heads of [128, 64] 11.4 -> 6.6).  O is nearer to 64 bits on every shape measured (relative error 4.9e-7 -> 3.7e-7 at [512, 64]).  Bound: the matrix core is
// busy 49 % of the cycles, vector instructions (cutting, softmax) take some 44 ([512, 64]).  Measured and dropped: two key tiles at a time,
// the scores of one interleaved with the exponentials of the other by instruction groups ([512, 64] 194, [1024, 96] 126 -> 128).
//
// Every other head size: scores through a workspace, one batched NT GEMM, a row softmax kernel and
// one batched NN GEMM over as many heads at a time as fit 256 MiB (the structure of
// ax_cuda_sdpa_fwd, cuda/ops_attention.cu:299-392).
#include "bf16x3.h"
#include "sdpa_order.h"

namespace {
using namespace axhip;

template <int DK, int WAVES>
struct SdGeom {
    static_assert(DK == 32 || DK == 64 || DK == 96 || DK == 128, "head dimension");
    static constexpr int BQ = 32 * WAVES;               // queries per workgroup
    static constexpr int BKV = DK == 128 ? 32 : 64;             // keys per block
    static constexpr int KROW = DK * 2, VROW = BKV * 2; // bytes of a row of one term: a key's, a column's
    static constexpr int KPLANE = BKV * KROW, VPLANE = DK * VROW;
    static constexpr int V_AT = 3 * KPLANE, STAGE = V_AT + 3 * VPLANE;
    static constexpr bool DOUBLE = WAVES == 8;          // two blocks in LDS, or two workgroups per CU
    static constexpr int PER_SIMD = DK == 128 && WAVES == 4 ? 1 : 2;     // waves: with two, 64 registers would spill
    static constexpr int FLAGS_AT = (DOUBLE ? 2 : 1) * STAGE;
    static constexpr int SMEM = FLAGS_AT + 4 * WAVES;   // a word per wave: are its sums finite
    static constexpr int E = BKV * DK % (512 * WAVES) == 0 ? 8 : 4;      // values of a piece that a thread stages
    static constexpr int PIECES = BKV * DK / E / (64 * WAVES);          // pieces of K, and of V
    static_assert(PIECES * E * 64 * WAVES == BKV * DK, "a block divides over the threads");
    static_assert(SMEM * (DOUBLE ? 1 : 2) <= 160 * 1024, "eight waves per CU");
    // where the 16-byte chunk c of row r lies
    template <int ROW>
    __device__ static unsigned at(int row, int chunk) {
        const int key = ROW == 256 ? row & 15 : ROW == 128 ? (row >> 1) & 7 : (row >> 2) & 3;
        return (unsigned)(row * ROW + ((chunk ^ key) << 4));
    }
    __device__ static unsigned k_at(int row, int chunk) { return at<KROW>(row, chunk); }
    __device__ static unsigned v_at(int col, int chunk) { return V_AT + at<VROW>(col, chunk); }
};

// The online softmax of a 32-key tile of scores (log2 units once taken times `down`, masked ones -infinity): scores become
// probabilities times `up`.  The reference point m_run of the exponentials only moves when some query's
// maximum exceeds it by more than 2^8: until then p = 2^(s - m_run) <= 256 is safe in fp32 and exact in
// the quotient O = sum(p v) / sum(p), and the accumulator needs no rescaling pass (which costs as many
// vector instructions as the exponentials themselves).  It starts at SD_LOWEST, the lowest finite value and not
// -infinity: scores of -infinity then weigh nothing also where a row has met no other yet.
constexpr float SD_LOWEST = -3.402823466e+38f;
template <int DT>
__device__ __forceinline__ void softmax_step(v16f &s, v16f (&acc_o)[DT], float &m_run, float &l_run, float up, float down) {
    float m_blk = -INFINITY;
#pragma unroll
    for (int v = 0; v < 16; v++) m_blk = fmaxf(m_blk, s[v]);
    m_blk = fmaxf(m_blk, __shfl_xor(m_blk, 32, 64)) * down;
    if (__builtin_amdgcn_ballot_w64(m_blk > m_run + 8.0f)) {      // wave-uniform; always taken for the first finite scores
        const float m_new = fmaxf(m_run, m_blk);
        const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
        l_run *= alpha;
        m_run = m_new;
#pragma unroll
        for (int d = 0; d < DT; d++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc_o[d][v] *= alpha;
    }
    float l_blk = 0.0f;
#pragma unroll
    for (int v = 0; v < 16; v++) {
        const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[v], down, -m_run)) * up;
        s[v] = p;
        l_blk += p;
    }
    l_run += l_blk;
}

// A wave's 32 queries with fp32 instructions, operands straight from memory: the rare second pass.  Rows
// past the end of the head are read as its last row, columns past dkr as zero (K, Q) or as the last one
// (V: they feed output columns that are not stored).
template <int DK, bool CAUSAL>
__device__ __forceinline__ void attend_f32(const float *Qh, const float *Kh, const float *Vh, int64_t ld, int64_t S, int dkr, float scale_log2e,
                                           int64_t wq_lo, int lane, v16f (&acc_o)[DK / 32], float &m_run, float &l_run) {
    constexpr int DT = DK / 32;
    const int frow = lane & 31, fhalf = lane >> 5;
    const int64_t qg = wq_lo + frow;
    const float *q = Qh + (qg < S ? qg : S - 1) * ld;
    m_run = SD_LOWEST;
    l_run = 0.0f;
#pragma unroll
    for (int d = 0; d < DT; d++)
#pragma unroll
        for (int v = 0; v < 16; v++) acc_o[d][v] = 0.0f;
    const int64_t end = CAUSAL && wq_lo + 32 < S ? wq_lo + 32 : S;
    for (int64_t k0 = 0; k0 < end; k0 += 32) {
        const float *k = Kh + (k0 + frow < S ? k0 + frow : S - 1) * ld;
        v16f s;
#pragma unroll
        for (int v = 0; v < 16; v++) s[v] = 0.0f;
        for (int c = 4 * fhalf; c < DK; c += 8) {
            v4f kf = {0.f, 0.f, 0.f, 0.f}, qf = kf;
            if (c < dkr) {
                kf = *reinterpret_cast<const v4f *>(k + c);
                qf = *reinterpret_cast<const v4f *>(q + c) * scale_log2e;
            }
#pragma unroll
            for (int e = 0; e < 4; e++) s = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[e], qf[e], s, 0, 0, 0);
        }
        const int64_t seen = (CAUSAL && qg < S ? qg : S - 1) - k0;
#pragma unroll
        for (int v = 0; v < 16; v++)
            if (8 * (v >> 2) + 4 * fhalf + (v & 3) > seen) s[v] = -INFINITY;
        softmax_step<DT>(s, acc_o, m_run, l_run, 1.0f, 1.0f);
#pragma unroll
        for (int v = 0; v < 16; v++) {
            const int64_t key = k0 + 8 * (v >> 2) + 4 * fhalf + (v & 3);
            const float *row = Vh + (key < S ? key : S - 1) * ld;
#pragma unroll
            for (int d = 0; d < DT; d++) {
                const int col = d * 32 + frow;
                acc_o[d] = __builtin_amdgcn_mfma_f32_32x32x2f32(row[col < dkr ? col : dkr - 1], s[v], acc_o[d], 0, 0, 0);
            }
        }
    }
}

constexpr int64_t FAR = 7168;                            // queries: K and V of such a head are more than an XCD's L2 holds
constexpr int ORDER_GROUPS = -1, ORDER_PAIRS = -2;       // of query tiles, where they go out in groups of eight heads

// Rows past the end of a head are never read (such a row is redirected to the head's last row, which keeps
// V finite), keys past the end are masked like causal ones, and queries past the end are computed but not stored.
// PAD: the head size dkr is below DK (a multiple of 4): chunks of Q and K past column dkr are zero, columns
// of V past it repeat the last one and feed output columns that are not stored.
template <int DK, int WAVES, bool CAUSAL, bool PAD>
__global__ void __launch_bounds__(64 * WAVES, (SdGeom<DK, WAVES>::PER_SIMD))
k_sdpa(const float *__restrict__ Q, const float *__restrict__ K, const float *__restrict__ V,
       float *__restrict__ O, float *__restrict__ L, int64_t BH, int64_t S, float scale_log2e,
       int64_t H, int64_t ld, int64_t ldo, int dkr, int order) {
    using G = SdGeom<DK, WAVES>;
    constexpr int BQ = G::BQ, BKV = G::BKV, E = G::E;
    constexpr int KS = DK / 16;                  // 16-wide steps of the score product
    constexpr int DT = DK / 32;                  // 32-wide column tiles of the output
    // the five smaller products of a score's terms in a sum of their own, where there are registers for it
    constexpr bool APART = DK <= 64;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int64_t nq = (S + BQ - 1) / BQ;
    // Workgroups go to the 8 XCDs round-robin by linear index.  Eight heads form a group: workgroup r of a group works on head r % 8 (every query tile of a
    // head then runs on the same XCD and shares its L2 copy of K and V) and on unit r / 8: a query tile, or a pair of causal tiles p and nq - 1 - p, which together
    // visit the same number of keys whatever p is (the middle tile of an odd nq stands alone).  `order` >= 0: single causal tiles in the order of sdpa_order.h.
    const bool paired = CAUSAL && order == ORDER_PAIRS;
    int64_t head, unit;
    if (CAUSAL && order >= 0) {
        const CausalTile o = causal_tile(blockIdx.x, (unsigned)BH, (unsigned)nq, (unsigned)order);
        head = o.head;
        unit = o.tile;
    } else {
        const int64_t units = paired ? (nq + 1) / 2 : nq;
        const int64_t lin = blockIdx.x, group = lin / (8 * units), left = BH - group * 8;
        const int64_t r = lin - group * 8 * units, hpg = left < 8 ? left : 8;
        head = group * 8 + r % hpg;
        unit = r / hpg;
    }
    const int passes = (paired && unit != nq - 1 - unit) ? 2 : 1;
    // head b * H + h starts at row b * S, column h * DK of matrices with row pitch ld (Q, K, V)
    // and ldo (O): H = 1, ld = DK is one matrix per head; H heads side by side in rows of
    // ld >= H * DK floats is the layout a fused projection writes and the output projection reads
    const int64_t hb = head / H, hh = head - hb * H;
    const int width = PAD ? dkr : DK;
    const int64_t in0 = hb * S * ld + hh * width;
    const float *Qh = Q + in0, *Kh = K + in0, *Vh = V + in0;
    const unsigned rowb = (unsigned)ld * 4;      // bytes between rows in global memory

    for (int pass = 0; pass < passes; pass++) {
        int t = threadIdx.x;                         // opaque: addresses are formed for each tile, not held from one to the next
        asm volatile("" : "+v"(t));
        const int lane = t & 63, frow = lane & 31, fhalf = lane >> 5;
        // the pieces this thread stages of each block: E columns of a key's row of K, E keys of a column of V
        // (a chunk holds those of registers 8s .. 8s+7 of a lane half: 16s + 4 * half + 0..3 and 8 further on)
        int krow[G::PIECES], kcol[G::PIECES], vcol[G::PIECES], vkey[G::PIECES];
        unsigned kput[G::PIECES], vput[G::PIECES];
#pragma unroll
        for (int i = 0; i < G::PIECES; i++) {
            const int q = t + i * 64 * WAVES, kc = q % (DK / E), vd = q % DK, vc = q / DK;
            krow[i] = q / (DK / E);
            kcol[i] = kc * E;
            kput[i] = G::k_at(krow[i], kc * E / 8) + kc * E % 8 * 2;
            vcol[i] = PAD && vd >= dkr ? dkr - 1 : vd;
            vkey[i] = E == 8 ? 16 * (vc >> 1) + 4 * (vc & 1) : 16 * (vc >> 2) + 4 * (vc >> 1 & 1) + 8 * (vc & 1);
            vput[i] = G::v_at(vd, vc * E / 8) + vc * E % 8 * 2;
        }
        float kr[G::PIECES][E], vr[G::PIECES][E];
        auto load_row = [&](auto &x, const char *base, unsigned off, int col) {      // columns from `col` on
            constexpr int N = sizeof(x) / 16;
#pragma unroll
            for (int h = 0; h < N; h++) {
                v4f a = {0.f, 0.f, 0.f, 0.f};
                if (!PAD || col + 4 * h < dkr) a = *reinterpret_cast<const v4f *>(base + off + 16 * h);
#pragma unroll
                for (int e = 0; e < 4; e++) x[4 * h + e] = a[e];
            }
        };
        auto load = [&](int64_t blk) {
            const char *kg = reinterpret_cast<const char *>(Kh + blk * BKV * ld), *vg = reinterpret_cast<const char *>(Vh + blk * BKV * ld);
            const int64_t valid = S - blk * BKV;
            if (valid >= BKV) {
#pragma unroll
                for (int i = 0; i < G::PIECES; i++) load_row(kr[i], kg, krow[i] * rowb + kcol[i] * 4, kcol[i]);
#pragma unroll
                for (int i = 0; i < G::PIECES; i++) {
                    const unsigned off = vkey[i] * rowb + vcol[i] * 4;
#pragma unroll
                    for (int e = 0; e < E; e++) vr[i][e] = *reinterpret_cast<const float *>(vg + (uint64_t)(e + (e & 4)) * rowb + off);
                }
            } else {
                const int end = (int)valid - 1;
#pragma unroll
                for (int i = 0; i < G::PIECES; i++) load_row(kr[i], kg, (krow[i] < end ? krow[i] : end) * rowb + kcol[i] * 4, kcol[i]);
#pragma unroll
                for (int i = 0; i < G::PIECES; i++) {
#pragma unroll
                    for (int e = 0; e < E; e++) {
                        const int key = vkey[i] + e + (e & 4);
                        vr[i][e] = *reinterpret_cast<const float *>(vg + (key < end ? key : end) * rowb + vcol[i] * 4);
                    }
                }
            }
        };
        auto put = [&](const float (&x)[E], unsigned at, unsigned plane) {
            Term<E> terms[3];
            cut(x, TERMS_UP, terms);
#pragma unroll
            for (int p = 0; p < 3; p++) *reinterpret_cast<Term<E> *>(lds + at + p * plane) = terms[p];
        };
        auto stage = [&](unsigned at) {              // the block in registers, to LDS
#pragma unroll
            for (int i = 0; i < G::PIECES; i++) put(kr[i], at + kput[i], G::KPLANE);
#pragma unroll
            for (int i = 0; i < G::PIECES; i++) put(vr[i], at + vput[i], G::VPLANE);
        };
        const int64_t q0 = (paired && pass == 0 ? nq - 1 - unit : unit) * BQ;
        const int64_t all_blocks = (S + BKV - 1) / BKV;
        const int64_t nblocks = CAUSAL && (q0 + BQ) / BKV < all_blocks ? (q0 + BQ) / BKV : all_blocks;
        const int64_t wq_lo = q0 + wave * 32, qg = wq_lo + frow;      // this wave's first query, this lane's query
        load(0);
        v4i qf[KS][3];                               // step ks: dk 16*ks + 8*fhalf .. +7 of this lane's query
        {
            const char *q = reinterpret_cast<const char *>(Qh + (qg < S ? qg : S - 1) * ld);
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {        // scale * log2(e) goes into Q once: scores come out in log2 units
                float x[8];
                load_row(x, q, (16 * ks + 8 * fhalf) * 4, 16 * ks + 8 * fhalf);
#pragma unroll
                for (int e = 0; e < 8; e++) x[e] *= scale_log2e;
                cut(x, TERMS_UP, qf[ks]);
            }
        }
        stage(0);
        if (G::DOUBLE && nblocks > 1) load(1);
        __syncthreads();

        v16f acc_o[DT];
#pragma unroll
        for (int d = 0; d < DT; d++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc_o[d][v] = 0.0f;
        float m_run = SD_LOWEST, l_run = 0.0f;       // l_run: this lane half's share of the row sum

        auto attend = [&](int64_t blk, unsigned at) {
            const int64_t kb0 = blk * BKV;
#pragma unroll 1
            for (int kt = 0; kt < BKV / 32; kt++) {
                // a wave past the end of the head has nothing to do; causal: a 32-key tile entirely above this wave's 32 queries is
                // skipped, and only tiles that straddle the diagonal pay for the mask (all wave-uniform decisions)
                const int64_t kt0 = kb0 + 32 * kt;
                if ((CAUSAL && kt0 > wq_lo + 31) || kt0 >= S || wq_lo >= S) break;
                const bool need_mask = CAUSAL ? kt0 + 31 > wq_lo : kt0 + 32 > S;

                // ---- scores ----
                v16f s, low;
#pragma unroll
                for (int v = 0; v < 16; v++) s[v] = low[v] = 0.0f;
                __builtin_amdgcn_s_setprio(1);  // matrix phases go ahead of the co-resident wave's vector work
#pragma unroll
                for (int ks = 0; ks < KS; ks++) {
                    v4i kf[3];
#pragma unroll
                    for (int p = 0; p < 3; p++)
                        kf[p] = *reinterpret_cast<const v4i *>(lds + at + G::k_at(frow, 2 * ks + fhalf) + kt * 32 * G::KROW + p * G::KPLANE);
#pragma unroll
                    for (int sum = 2; sum > 0; sum--)
#pragma unroll
                        for (int p = sum; p >= 0; p--) (APART ? low : s) = mfma_terms(kf[sum - p], qf[ks][p], APART ? low : s);
                    s = mfma_terms(kf[0], qf[ks][0], s);
                }
                __builtin_amdgcn_s_setprio(0);
                if (APART) s += low;
                if (need_mask) {
                    // keys of this tile with index > qrel are masked: those after the query (causal; such a query
                    // lies inside the head, so they cover the keys past its end too) or past the end
                    const int qrel = (int)((CAUSAL ? qg : S - 1) - kt0);
#pragma unroll
                    for (int v = 0; v < 16; v++)
                        if (8 * (v >> 2) + 4 * fhalf + (v & 3) > qrel) s[v] = -INFINITY;
                }
                softmax_step<DT>(s, acc_o, m_run, l_run, TERMS_UP, TERMS_DOWN);

                // ---- O^T += V^T P^T ----
#pragma unroll
                for (int st = 0; st < 2; st++) {
                    float x[8];
#pragma unroll
                    for (int e = 0; e < 8; e++) x[e] = s[8 * st + e];
                    v4i pf[3];
                    cut(x, 1.0f, pf);                     // (a probability is zero or from 2^-126 up, and was taken times 2^24)
#pragma unroll
                    for (int d = 0; d < DT; d++) {
                        v4i vf[3];
#pragma unroll
                        for (int p = 2; p >= 0; p--)
                            vf[p] = *reinterpret_cast<const v4i *>(lds + at + G::v_at(d * 32 + frow, 4 * kt + 2 * st + fhalf) + p * G::VPLANE);
#pragma unroll
                        for (int sum = 2; sum >= 0; sum--)                // the small products first
#pragma unroll
                            for (int p = sum; p >= 0; p--) acc_o[d] = mfma_terms(vf[p], pf[sum - p], acc_o[d]);
                    }
                }
            }
        };
        if constexpr (G::DOUBLE) {
            // Two blocks in LDS and the next one in registers.  The two waves of a SIMD (w, w + 4) put it beside the current
            // block before and after that is multiplied, so that one cuts while the other's products run.
            unsigned cur = 0;
            for (int64_t blk = 0; blk < nblocks; blk++, cur ^= G::STAGE) {
                const bool more = blk + 1 < nblocks;
                auto next = [&]() {
                    stage(cur ^ G::STAGE);
                    if (blk + 2 < nblocks) load(blk + 2);
                };
                if (more && wave >= 4) next();
                attend(blk, cur);
                if (more && wave < 4) next();
                __syncthreads();
            }
        } else {
            for (int64_t blk = 0; blk < nblocks; blk++) {
                const bool more = blk + 1 < nblocks;
                if (more) load(blk + 1);
                attend(blk, 0);
                __syncthreads();                      // the block has been read
                if (more) {
                    stage(0);
                    __syncthreads();
                }
            }
        }

        // ---- did every sum come out finite?  Scores past 2^80 below zero are infinite too: they weigh nothing, as they should,
        // unless a row has no others ----
        float seen = l_run * 0.0f, up = TERMS_UP, down = 1.0f / TERMS_UP;
#pragma unroll
        for (int d = 0; d < DT; d++) look_at(acc_o[d], seen);
        float l_tot = l_run + __shfl_xor(l_run, 32, 64);
        if (any_wave<WAVES>(!(seen == 0.0f) || (l_tot == 0.0f && wq_lo < S), lds + G::FLAGS_AT, wave)) {
            int again = lane;                        // opaque, so that no address of this pass is held through the loop above
            asm volatile("" : "+v"(again));
            attend_f32<DK, CAUSAL>(Qh, Kh, Vh, ld, S, width, scale_log2e, wq_lo, again, acc_o, m_run, l_run);
            l_tot = l_run + __shfl_xor(l_run, 32, 64);
            up = down = 1.0f;
        }

        // ---- normalise and write: lane owns query qg, dk columns 32*d + 8*g + 4*fhalf .. +3 ----
        const float inv = 1.0f / l_tot * down;       // the sums hold the factors of V and of the probabilities, l_tot the latter's
        float *orow = O + (hb * S + qg) * ldo + hh * width;
        if (qg < S) {
#pragma unroll
            for (int d = 0; d < DT; d++)
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    v4f o;
#pragma unroll
                    for (int e = 0; e < 4; e++) o[e] = acc_o[d][4 * g + e] * inv;
                    if (!PAD || d * 32 + 8 * g + 4 * fhalf < dkr) *reinterpret_cast<v4f *>(orow + d * 32 + 8 * g + 4 * fhalf) = o;
                }
            // (a row that saw nothing but -infinity: 0 / 0 above, and NaN here)
            if (L && fhalf == 0) L[head * S + qg] = l_tot == 0.0f ? NAN : (m_run + __builtin_amdgcn_logf(l_tot / up)) * 0.6931471805599453f;
        }
    }
}

// A kernel's name: geometry, mask, waves (four unless it says eight), and whether tiles go out in pairs; or the form for few tiles.
enum Form { FOUR, EIGHT, FOUR_PAIRS, EIGHT_PAIRS, FEW };
const char *sdpa_name(int dk, int causal, Form form) {
#define AX_NAMES(DK)                                                                                                                          \
    {{"sdpa_fused_dk" DK, "sdpa_fused_dk" DK "_w8", "", "", "sdpa_fused_few_dk" DK},                                                             \
     {"sdpa_fused_dk" DK "_causal", "sdpa_fused_dk" DK "_causal_w8", "sdpa_fused_dk" DK "_causal_pairs", "sdpa_fused_dk" DK "_causal_w8_pairs",   \
      "sdpa_fused_few_dk" DK "_causal"}}
    static const char *const names[4][2][5] = {AX_NAMES("32"), AX_NAMES("64"), AX_NAMES("96"), AX_NAMES("128")};
#undef AX_NAMES
    return names[dk / 32 - 1][causal != 0][form];
}

// Few tiles: four waves share 32 queries of one head and take its 32-key tiles in turn, each with an online softmax of its own; the
// sets of maxima, sums and outputs meet in LDS.  Each wave reads its keys and values straight into fragment registers and cuts them itself,
// so a key is cut once per 32 queries and not once per 128 or 256: more vector work in all, on four (or eight) times the workgroups and with
// a quarter of the serial key tiles.
template <int DK, bool CAUSAL, bool PAD>
__global__ void __launch_bounds__(256, DK <= 64 ? 2 : 1)
k_sdpa_few(const float *__restrict__ Q, const float *__restrict__ K, const float *__restrict__ V, float *__restrict__ O, float *__restrict__ L,
           int64_t BH, int64_t S, float scale_log2e, int64_t H, int64_t ld, int64_t ldo, int dkr) {
    constexpr int KS = DK / 16, DT = DK / 32, PIECES = 4 * DT, WAVES = 4;
    constexpr bool APART = DK <= 64;             // as in k_sdpa
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    auto part = reinterpret_cast<v4f (*)[PIECES][64]>(lds);              // [WAVES]: sums; then maxima and row sums; then a word per wave
    auto ml = reinterpret_cast<float (*)[2][32]>(lds + WAVES * PIECES * 1024);
    unsigned char *flags = lds + WAVES * (PIECES * 1024 + 256);
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63, frow = lane & 31, fhalf = lane >> 5;
    const int64_t nq = (S + 31) / 32;            // workgroups as in k_sdpa: the tiles of a head on one XCD
    const int64_t lin = blockIdx.x, group = lin / (8 * nq), left = BH - group * 8;
    const int64_t r = lin - group * 8 * nq, hpg = left < 8 ? left : 8;
    const int64_t head = group * 8 + r % hpg, q0 = (CAUSAL ? nq - 1 - r / hpg : r / hpg) * 32;       // causal: the longest first
    const int64_t hb = head / H, hh = head - hb * H;
    const int width = PAD ? dkr : DK;
    const int64_t in0 = hb * S * ld + hh * width;
    const float *Qh = Q + in0, *Kh = K + in0, *Vh = V + in0;
    const unsigned rowb = (unsigned)ld * 4;
    const int64_t qg = q0 + frow;
    const int tiles = (int)(CAUSAL ? q0 / 32 + 1 : nq);

    auto load_row = [&](float (&x)[8], const char *row, int col) {       // columns col .. col + 7, zero from width on
#pragma unroll
        for (int h = 0; h < 2; h++) {
            v4f a = {0.f, 0.f, 0.f, 0.f};
            if (!PAD || col + 4 * h < dkr) a = *reinterpret_cast<const v4f *>(row + (col + 4 * h) * 4);
#pragma unroll
            for (int e = 0; e < 4; e++) x[4 * h + e] = a[e];
        }
    };
    float kr[KS][8], vr[2][DT][8];
    // a key past the end is read as the last one (its score is masked)
    auto load_k = [&](int t) {
        const int64_t key = (int64_t)t * 32 + frow;
        const char *row = reinterpret_cast<const char *>(Kh + (key < S ? key : S - 1) * ld);
#pragma unroll
        for (int ks = 0; ks < KS; ks++) load_row(kr[ks], row, 16 * ks + 8 * fhalf);
    };
    auto load_v = [&](int t) {
        const char *base = reinterpret_cast<const char *>(Vh + (int64_t)t * 32 * ld);
        const int end = (int)(S - 1 - (int64_t)t * 32 < 31 ? S - 1 - (int64_t)t * 32 : 31);
#pragma unroll
        for (int st = 0; st < 2; st++)
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const int key = 16 * st + 4 * fhalf + e + (e & 4);
                const char *row = base + (unsigned)(key < end ? key : end) * rowb;
#pragma unroll
                for (int d = 0; d < DT; d++) {
                    const int col = d * 32 + frow;
                    vr[st][d][e] = *reinterpret_cast<const float *>(row + (PAD && col >= dkr ? dkr - 1 : col) * 4);
                }
            }
    };
    v4i qf[KS][3];
    v16f acc_o[DT];
#pragma unroll
    for (int d = 0; d < DT; d++)
#pragma unroll
        for (int v = 0; v < 16; v++) acc_o[d][v] = 0.0f;
    float m_run = SD_LOWEST, l_run = 0.0f;
    if (wave < tiles) {
        load_k(wave);
        const char *q = reinterpret_cast<const char *>(Qh + (qg < S ? qg : S - 1) * ld);
        float x[KS][8];
#pragma unroll
        for (int ks = 0; ks < KS; ks++) load_row(x[ks], q, 16 * ks + 8 * fhalf);
        load_v(wave);
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
#pragma unroll
            for (int e = 0; e < 8; e++) x[ks][e] *= scale_log2e;
            cut(x[ks], TERMS_UP, qf[ks]);
        }
    }
    auto attend = [&](int t, auto more, int next) {  // more: tile `next` is fetched meanwhile
        v16f s, low;
#pragma unroll
        for (int v = 0; v < 16; v++) s[v] = low[v] = 0.0f;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            v4i kf[3];
            cut(kr[ks], TERMS_UP, kf);
#pragma unroll
            for (int sum = 2; sum > 0; sum--)
#pragma unroll
                for (int p = sum; p >= 0; p--) (APART ? low : s) = mfma_terms(kf[sum - p], qf[ks][p], APART ? low : s);
            s = mfma_terms(kf[0], qf[ks][0], s);
        }
        if constexpr (decltype(more)::value) load_k(next);
        if (APART) s += low;
        if (CAUSAL ? t == tiles - 1 : (int64_t)t * 32 + 32 > S) {
            const int qrel = (int)((CAUSAL ? qg : S - 1) - (int64_t)t * 32);
#pragma unroll
            for (int v = 0; v < 16; v++)
                if (8 * (v >> 2) + 4 * fhalf + (v & 3) > qrel) s[v] = -INFINITY;
        }
        softmax_step<DT>(s, acc_o, m_run, l_run, TERMS_UP, TERMS_DOWN);
#pragma unroll
        for (int st = 0; st < 2; st++) {
            float x[8];
#pragma unroll
            for (int e = 0; e < 8; e++) x[e] = s[8 * st + e];
            v4i pf[3];
            cut(x, 1.0f, pf);
#pragma unroll
            for (int d = 0; d < DT; d++) {
                v4i vf[3];
                cut(vr[st][d], TERMS_UP, vf);
#pragma unroll
                for (int sum = 2; sum >= 0; sum--)
#pragma unroll
                    for (int p = sum; p >= 0; p--) acc_o[d] = mfma_terms(vf[p], pf[sum - p], acc_o[d]);
            }
        }
        if constexpr (decltype(more)::value) load_v(next);
    };
    // The last tile stands apart and fetches nothing: with one tile a wave, fetching it again was half of all loads, and a branch about the fetch cuts
    // the loop in two for the scheduler.  us, fetched again -> branch -> apart: 32 heads of [128, 64] 6.85 -> 6.60 -> 6.55, 16 of [128, 128] 11.8 -> 10.9 -> 10.1, 32
    // of [500, 128] 49.6 -> 47.9 -> 45.6, 8 of [288, 32] 7.05 -> 7.18 -> 6.95, 4 of [2048, 64] 40.0 -> 40.9 -> 39.0.
    // Only geometry 96 at its full width under the mask is slower apart: more registers than a wave addresses directly (9 of [2312, 96] 119 -> 125, 5 of [2206, 96] 53 -> 56).
    int t = wave;
    if constexpr (DK == 96 && CAUSAL && !PAD) {
        for (; t < tiles; t += WAVES) attend(t, std::true_type(), t + WAVES < tiles ? t + WAVES : t);
    } else {
        for (; t + WAVES < tiles; t += WAVES) attend(t, std::true_type(), t + WAVES);
        if (t < tiles) attend(t, std::false_type(), t);
    }

    // ---- the waves' parts together, each at an eighth (exactly): outputs that are finite in themselves may exceed the largest float when
    // four are added with the factors of the terms still in them ----
    constexpr float PART_DOWN = 0.125f;
    float seen = l_run * 0.0f;
#pragma unroll
    for (int d = 0; d < DT; d++) look_at(acc_o[d], seen);
    const float l_wave = l_run + __shfl_xor(l_run, 32, 64);
#pragma unroll
    for (int d = 0; d < DT; d++)
#pragma unroll
        for (int g = 0; g < 4; g++) part[wave][d * 4 + g][lane] = v4f{acc_o[d][4 * g], acc_o[d][4 * g + 1], acc_o[d][4 * g + 2], acc_o[d][4 * g + 3]} * PART_DOWN;
    if (fhalf == 0) {
        ml[wave][0][frow] = m_run;
        ml[wave][1][frow] = l_wave;
    }
    bool unfit = any_wave<WAVES>(!(seen == 0.0f), flags, wave);
    float m_all = ml[0][0][frow], weight[WAVES], l_all = 0.0f;
#pragma unroll
    for (int w = 1; w < WAVES; w++) m_all = fmaxf(m_all, ml[w][0][frow]);
#pragma unroll
    for (int w = 0; w < WAVES; w++) {
        weight[w] = __builtin_amdgcn_exp2f(ml[w][0][frow] - m_all);
        l_all += ml[w][1][frow] * weight[w];
    }
    unfit |= __builtin_amdgcn_ballot_w64(l_all == 0.0f && qg < S) != 0;  // the same in every wave
    float *orow = O + (hb * S + qg) * ldo + hh * width;
    if (unfit) {
        if (wave != 0) return;
        attend_f32<DK, CAUSAL>(Qh, Kh, Vh, ld, S, width, scale_log2e, q0, lane, acc_o, m_run, l_run);
        const float l_tot = l_run + __shfl_xor(l_run, 32, 64), inv = 1.0f / l_tot;
        if (qg >= S) return;
#pragma unroll
        for (int d = 0; d < DT; d++)
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const int col = d * 32 + 8 * g + 4 * fhalf;
                if (!PAD || col < dkr)
                    *reinterpret_cast<v4f *>(orow + col) = v4f{acc_o[d][4 * g] * inv, acc_o[d][4 * g + 1] * inv, acc_o[d][4 * g + 2] * inv, acc_o[d][4 * g + 3] * inv};
            }
        if (L && fhalf == 0) L[head * S + qg] = l_tot == 0.0f ? NAN : (m_run + __builtin_amdgcn_logf(l_tot)) * 0.6931471805599453f;
        return;
    }
    if (qg >= S) return;
    const float inv = 1.0f / l_all * (1.0f / (TERMS_UP * PART_DOWN));
    for (int piece = wave; piece < PIECES; piece += WAVES) {
        v4f o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < WAVES; w++) o += part[w][piece][lane] * weight[w];
        const int col = (piece >> 2) * 32 + 8 * (piece & 3) + 4 * fhalf;
        if (!PAD || col < dkr) *reinterpret_cast<v4f *>(orow + col) = o * inv;
    }
    if (L && wave == 0 && fhalf == 0) L[head * S + qg] = (m_all + __builtin_amdgcn_logf(l_all / TERMS_UP)) * 0.6931471805599453f;
}

// Where the few-tiles form pays, by the key tiles that a wave walks one after the other: the longest walk is a quarter of a head's 32-key
// tiles, and all walks together are shared by the CUs.  `limit` is four times the longest walks a CU up to which it is ahead of k_sdpa, whose
// four waves each walk all of a head's tiles: two rounds of workgroups and a little where two share a CU (geometries 32 and 64), two where one has
// it, one where a walk is two tiles and mostly start and end; causal walks differ in length, and the shorter they all are the sooner the
// longer geometries fall behind (us, k_sdpa -> this as it was before its last tile stood apart: 32 heads of [128, 64] 11.4 -> 6.9, 4 of [2048, 64] 111 -> 36, 32 of [512, 64] 33.3 -> 22.0, 8 causal ones of
// [2048, 128] 204 -> 74, 32 causal of [1024, 80] 81.6 -> 74.4; past it 64 of [512, 64] 35.7 -> 38.6, 64 causal of [512, 80] 44.6 -> 55.6, 81 of [216, 128]
// 30.4 -> 43.2, 100 of [160, 128] 23.6 -> 28.7, 53 of [294, 96] 29.8 -> 37.7, causal 113 of [208, 80] 23.8 -> 34.1, 57 of [507, 128] 60.6 -> 70.8; over 2804 random
// ones within it 0.91 to 2.8 times as fast).  A single key tile per wave (S up to 128): one workgroup a CU, or two of the smaller geometries from three
// tiles on (128 of [128, 64] 12.1 -> 11.5, but 128 of [128, 128] 21.3 -> 23.2, 256 of [64, 64] 8.1 -> 8.9).  A head of one tile gains nothing (4.6 us
// either way).
// With the last tile apart from the loop the line moved out: random ones of the two smaller geometries with walks of ten tiles and more, up to 1.3 times the limit, 0.99 to 1.65
// times as fast (17 of [1256, 32] 47.7 -> 36.8, 14 of [1571, 32] 58.6 -> 48.3, causal 28 of [1386, 32] 53.1 -> 47.6, 39 of [1166, 32] 46.3 -> 46.8); walks of nine 0.95 to 1.2, the larger geometries
// 0.93 to 1.3 (causal 18 of [1908, 112] 192 -> 206), at 1.4 times and beyond 0.7 to 1.3: these stay.  One tile a wave of the geometry 96 with four tiles: 24 random
// ones 0.98 to 1.16 (78 of [99, 96] causal 16.1 -> 14.0, 127 of [100, 80] causal 14.9 -> 15.2); the geometry 128 keeps one (four tiles would gain 2 to 13 %, three lose 5: 150 of
// [96, 128] 17.0 -> 17.9).
// Eight waves on 32 queries: level or behind (32 of [512, 64] 22.0 -> 27.2, 1 of [2048, 64] 32.7 -> 31.1): the vector pipe is the bound.
template <int DK>
bool few_tiles(int64_t BH, int64_t S, int causal) {
    const int64_t tiles = (S + 31) / 32, walk = (tiles + 3) / 4, cus = cu_count();
    if (tiles < 2 || BH > 4 * cus || tiles > 0xffff) return false;
    if (walk == 1) return tiles * BH <= (tiles == 4 ? (DK < 128 ? 2 : 1) : tiles == 3 && DK <= 64 ? 2 : 1) * cus;
    const int64_t q = tiles / 4, all = causal ? 2 * q * (q + 1) + tiles % 4 * (q + 1) : tiles * walk;
    int64_t limit = 9;
    if (causal && DK > 64) limit = walk + (DK == 96 ? 2 : 1) < 7 ? walk + (DK == 96 ? 2 : 1) : 7;
    else if (causal && DK == 64 && walk == 2) limit = 5;
    else if (!causal && DK > 64) limit = walk == 2 ? 4 : 8;
    else if (!causal && DK == 64 && walk <= 3) limit = 8;
    const bool further = walk > 9 && DK <= 64;
    return all * BH * 40 <= limit * (further ? 13 : 10) * walk * cus;
}

template <int DK>
int launch_sdpa_few(const float *Q, const float *K, const float *V, float *O, float *L, int64_t BH, int64_t S,
                    float scale, int causal, int64_t H, int64_t ld, int64_t ldo, int dkr) {
    constexpr int SMEM = 4 * (DK / 8 * 1024 + 256 + 4);
    static bool attr_set = false;
    if (!attr_set) {
        for (const void *k : {reinterpret_cast<const void *>(k_sdpa_few<DK, false, false>), reinterpret_cast<const void *>(k_sdpa_few<DK, true, false>),
                              reinterpret_cast<const void *>(k_sdpa_few<DK, false, true>), reinterpret_cast<const void *>(k_sdpa_few<DK, true, true>)})
            AXHIP_HIP_TRY(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, SMEM), "hipFuncSetAttribute");
        attr_set = true;
    }
    const float sl2 = scale * 1.4426950408889634f;
    const dim3 grid((unsigned)((S + 31) / 32 * BH)), block(256);
    note_kernel(sdpa_name(DK, causal, FEW));
#define AX_FEW(C, P) hipLaunchKernelGGL((k_sdpa_few<DK, C, P>), grid, block, SMEM, kStream, Q, K, V, O, L, BH, S, sl2, H, ld, ldo, dkr)
    if (causal && dkr == DK) AX_FEW(true, false);
    else if (causal) AX_FEW(true, true);
    else if (dkr == DK) AX_FEW(false, false);
    else AX_FEW(false, true);
#undef AX_FEW
    return check_launch("sdpa_fwd");
}

template <int DK, int WAVES, bool PAD>
int launch_sdpa_p(const float *Q, const float *K, const float *V, float *O, float *L, int64_t BH, int64_t S,
                  float scale, int causal, int64_t H, int64_t ld, int64_t ldo, int dkr) {
    using G = SdGeom<DK, WAVES>;
    static bool attr_set = false;
    if (!attr_set) {
        for (const void *k : {reinterpret_cast<const void *>(k_sdpa<DK, WAVES, false, PAD>), reinterpret_cast<const void *>(k_sdpa<DK, WAVES, true, PAD>)})
            AXHIP_HIP_TRY(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, G::SMEM), "hipFuncSetAttribute");
        attr_set = true;
    }
    const float sl2 = scale * 1.4426950408889634f;
    const int64_t nq = (S + G::BQ - 1) / G::BQ;
    // Causal tiles p and nq - 1 - p in one workgroup where there are more tiles than CUs and the pairs, up to two a CU, give every CU the same number of keys or
    // nearly ([8192, 64] x 8 single 486 us, paired 462, [16384, 64] x 8 1520 and 1416, [1024, 128] x 64 136.5 and 134.2; but [8192, 32] x 16 433 and 457); and up to one a CU
    // where K and V of a head are more than an XCD's L2 holds ([7662, 80] x 12 734 and 696, [8192, 96] x 12 802 and 776, [7000, 80] x 12 648 and 652, but [6000, 80] x 12 524
    // and 548).  With a CU for every tile there is nothing to even out.
    const int64_t cus = cu_count(), pairs = (nq + 1) / 2 * BH, rounds = (pairs + cus - 1) / cus;
    const bool even = WAVES == 4 && (DK == 64 || DK == 128) && rounds <= 2 && rounds * cus * 30 <= nq * BH * 16, far = DK >= 96 && rounds == 1 && S > FAR;
    const bool pair = causal && nq * BH > cus && (even || far);
    const dim3 block(64 * WAVES);
    // A grid holds fewer than 2^32 threads: more heads go in pieces, of whole batches where those fit (head h of a launch lies in batch h / H of its pointers).
    const int64_t a_head = pair ? (nq + 1) / 2 : nq;
    int64_t most = 0xffffffffll / (64 * WAVES) / a_head;
    if (most < 1) return fail(AXHIP_ERR_SHAPE, "sdpa_fwd: too many tiles");
    note_kernel(sdpa_name(DK, causal, pair ? (WAVES == 8 ? EIGHT_PAIRS : FOUR_PAIRS) : WAVES == 8 ? EIGHT : FOUR));
    if (most > H) most -= most % H;
    for (int64_t h0 = 0, n; h0 < BH; h0 += n) {
        n = BH - h0 < most ? BH - h0 : most;
        if (most < H && n > H - h0 % H) n = H - h0 % H;
        const int64_t in = h0 / H * S * ld + h0 % H * dkr, out = h0 / H * S * ldo + h0 % H * dkr;
        const dim3 grid((unsigned)(a_head * n));
        const int order = pair ? ORDER_PAIRS : nq * n > cus ? (int)causal_last(n, nq, cus * (WAVES == 8 || DK == 128 ? 1 : 2)) : ORDER_GROUPS;
        float *lse = L ? L + h0 * S : nullptr;
        if (causal) hipLaunchKernelGGL((k_sdpa<DK, WAVES, true, PAD>), grid, block, G::SMEM, kStream, Q + in, K + in, V + in, O + out, lse, n, S, sl2, H, ld, ldo, dkr, order);
        else hipLaunchKernelGGL((k_sdpa<DK, WAVES, false, PAD>), grid, block, G::SMEM, kStream, Q + in, K + in, V + in, O + out, lse, n, S, sl2, H, ld, ldo, dkr, order);
        if (int rc = check_launch("sdpa_fwd")) return rc;
    }
    return AXHIP_OK;
}

template <int DK>
int launch_sdpa(const float *Q, const float *K, const float *V, float *O, float *L, int64_t BH, int64_t S,
                float scale, int causal, int64_t H, int64_t ld, int64_t ldo, int dkr) {
    // Eight waves on 256 queries cut half as much of K and V for each of them, four on 128 waste less of a short head and
    // of the diagonal.  us, four waves -> eight: 64 heads of [1024, 128] 191 -> 174, 64 of [1024, 96]
    // 141 -> 126, 85 causal ones of [1099, 80] 154 -> 149, 512 of [512, 64] 201 -> 194; but causal 128 -> 142, 512 of [256, 32]
    // 33 -> 37, 256 causal ones of [333, 48] 40 -> 44.  Geometry
    // 128 has the registers of one wave per SIMD with four waves, so it takes eight as soon as there is more than one tile a CU.
    if constexpr (DK > 32) {
        const int64_t half_tiles = (S + 127) / 128, tiles = (S + 255) / 256, cus = cu_count();
        const bool fits = tiles * 8 <= half_tiles * 5;
        bool eight;
        if (!causal) eight = DK == 128 ? half_tiles * BH > cus : DK >= 64 && tiles * BH >= cus && fits;
        else {
            // single causal tiles: three of 128 queries or two of 256, where the latter have a CU each (us, four -> eight: 99 heads of [381, 96] 40 -> 31, 95 of
            // [322, 64] 27 -> 23, 120 of [314, 128] 57 -> 49 but 50 of [316, 128], whose three have one too, 43 -> 48; 129 of [280, 80] 35 -> 48); geometry 128
            // a little under two rounds of them, too (219 of [384, 128] 103 -> 97, 186 of [448, 128] 119 -> 113), and from nine blocks of 128 x 128 a CU on (238 of [512, 128] 163 -> 134, 60 of [832, 128] 109 -> 113)
            // geometry 128 two or one by their rounds (178 of [192, 128] 46 -> 37, 430 of [208, 128] 98 -> 87, but 124 of [190, 128] 28 -> 37)
            eight = half_tiles == 3 && 2 * BH <= cus && (DK != 128 || 3 * BH > cus);
            if (DK == 128 && half_tiles == 2) eight = (BH + cus - 1) / cus * 5 < (2 * BH + cus - 1) / cus * 3;
            else if (DK == 128) eight = eight || (half_tiles == 3 && BH <= cus && 6 * BH > 5 * cus) || (half_tiles == 4 && 10 * BH >= 7 * cus) || (half_tiles + 1) * half_tiles * BH > 18 * cus;
            // geometry 96 from half a tile of 256 a CU on, with more than three tiles a head from three quarters on, and where heads are so long that tiles of 128 go out in pairs (launch_sdpa_p)
            // from one (four -> eight: 90 of [400, 96] 47 -> 44, 90 of [595, 96] 71 -> 64, 34 of [1786, 96] 177 -> 173, but 32 of [1024, 96] 85 -> 95, 14 of [3002, 80] 245 -> 260, 24 of [2000, 96] 178 -> 185,
            // 8 of [7662, 80] 590 -> 650)
            if (DK == 96) eight = eight || ((tiles == 1 ? BH > cus : tiles <= 3 ? tiles * BH * 2 >= cus : S > FAR ? tiles * BH >= cus : tiles * BH * 4 > cus * 3) && fits);
        }
        if (eight)
            return dkr == DK ? launch_sdpa_p<DK, 8, false>(Q, K, V, O, L, BH, S, scale, causal, H, ld, ldo, dkr)
                             : launch_sdpa_p<DK, 8, true>(Q, K, V, O, L, BH, S, scale, causal, H, ld, ldo, dkr);
    }
    return dkr == DK ? launch_sdpa_p<DK, 4, false>(Q, K, V, O, L, BH, S, scale, causal, H, ld, ldo, dkr)
                     : launch_sdpa_p<DK, 4, true>(Q, K, V, O, L, BH, S, scale, causal, H, ld, ldo, dkr);
}

// One workgroup per score row: mask, maximum, exponentials, sum, normalise in place; L = max + log(sum).
__global__ void __launch_bounds__(256)
k_softmax_lse_rows(float *__restrict__ score, float *__restrict__ L, int64_t S, int causal) {
    __shared__ float red[256];
    const int64_t row = blockIdx.x;               // head * S + query
    const int64_t qi = row % S;
    float *p = score + row * S;
    const int64_t n = causal ? qi + 1 : S;        // keys this query sees
    float mx = -INFINITY;
    for (int64_t j = threadIdx.x; j < n; j += 256) mx = fmaxf(mx, p[j]);
    red[threadIdx.x] = mx;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) red[threadIdx.x] = fmaxf(red[threadIdx.x], red[threadIdx.x + s]);
        __syncthreads();
    }
    mx = red[0];
    __syncthreads();
    float sum = 0.0f;
    for (int64_t j = threadIdx.x; j < S; j += 256) {
        const float e = j < n ? expf(p[j] - mx) : 0.0f;
        p[j] = e;
        sum += e;
    }
    red[threadIdx.x] = sum;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    sum = red[0];
    const float inv = 1.0f / sum;
    for (int64_t j = threadIdx.x; j < n; j += 256) p[j] *= inv;
    if (L && threadIdx.x == 0) L[row] = mx + logf(sum);
}

int sdpa_unfused(const float *Q, const float *K, const float *V, float *O, float *L, int64_t BH,
                 int64_t S, int64_t dk, float scale, int causal) {
    const size_t per_head = (size_t)S * (size_t)S * sizeof(float);
    int64_t chunk = (int64_t)((size_t(256) << 20) / per_head);
    if (chunk < 1) chunk = 1;
    if (chunk > BH) chunk = BH;
    if (chunk > 65535) chunk = 65535;
    float *score = static_cast<float *>(workspace((size_t)chunk * per_head));
    if (!score) return AXHIP_ERR_ALLOC;
    for (int64_t h0 = 0; h0 < BH; h0 += chunk) {
        const int64_t nb = BH - h0 < chunk ? BH - h0 : chunk;
        const float *q = Q + h0 * S * dk, *k = K + h0 * S * dk, *v = V + h0 * S * dk;
        int rc = sgemm_batched(0, 1, S, S, dk, scale, q, dk, S * dk, k, dk, S * dk, 0.0f, score, S, S * S, nb, false);
        if (rc) return rc;
        if (nb * S > 0x7fffffff) return fail(AXHIP_ERR_SHAPE, "sdpa: too many score rows per chunk");
        hipLaunchKernelGGL(k_softmax_lse_rows, dim3((unsigned)(nb * S)), dim3(256), 0, kStream, score,
                           L ? L + h0 * S : nullptr, S, causal);
        if ((rc = check_launch("sdpa softmax"))) return rc;
        rc = sgemm_batched(0, 0, S, dk, S, 1.0f, score, S, S * S, v, dk, S * dk, 0.0f, O + h0 * S * dk, dk, S * dk, nb, false);
        if (rc) return rc;
    }
    note_kernel("sdpa_unfused");
    return AXHIP_OK;
}

}  // namespace

// shared by both entry points: H heads side by side in rows of ld (Q, K, V) / ldo (O) floats.  A head
// size that is a multiple of 4 up to 128 runs on the kernel of the next size among 32, 64, 96, 128.
static bool sdpa_fusable(int64_t dk) { return dk >= 4 && dk <= 128 && dk % 4 == 0; }

static int sdpa_fused(const float *Q, const float *K, const float *V, float *O, float *L, int64_t BH, int64_t S,
                      int64_t dk, float scale, int causal, int64_t H, int64_t ld, int64_t ldo) {
    auto run = [&](auto geometry) {
        constexpr int DK = decltype(geometry)::value;
        return few_tiles<DK>(BH, S, causal) ? launch_sdpa_few<DK>(Q, K, V, O, L, BH, S, scale, causal, H, ld, ldo, (int)dk)
                                            : launch_sdpa<DK>(Q, K, V, O, L, BH, S, scale, causal, H, ld, ldo, (int)dk);
    };
    if (dk <= 32) return run(std::integral_constant<int, 32>());
    if (dk <= 64) return run(std::integral_constant<int, 64>());
    if (dk <= 96) return run(std::integral_constant<int, 96>());
    return run(std::integral_constant<int, 128>());
}

extern "C" int axhip_sdpa_fwd(const float *Q, const float *K, const float *V, float *O, float *L, int64_t BH,
                              int64_t S, int64_t dk, float scale, int causal) {
    if (int rc = axhip::ensure_ready()) return rc;
    if (!Q || !K || !V || !O) return fail(AXHIP_ERR_NULL_ARG, "sdpa_fwd: NULL tensor");
    if (BH < 0 || S < 0 || dk <= 0) return fail(AXHIP_ERR_SHAPE, "sdpa_fwd: bad extent");
    if (BH == 0 || S == 0) return AXHIP_OK;
    const bool aligned = ((((uintptr_t)Q | (uintptr_t)K | (uintptr_t)V | (uintptr_t)O) & 15) == 0);
    if (sdpa_fusable(dk) && aligned && (S + 127) / 128 * BH <= 0x7fffffff)
        return sdpa_fused(Q, K, V, O, L, BH, S, dk, scale, causal, 1, dk, dk);
    return sdpa_unfused(Q, K, V, O, L, BH, S, dk, scale, causal);
}

extern "C" int axhip_sdpa_fwd_rows(const float *Q, const float *K, const float *V, int64_t ld, float *O, int64_t ldo,
                                   float *L, int64_t B, int64_t H, int64_t S, int64_t dk, float scale, int causal) {
    if (int rc = axhip::ensure_ready()) return rc;
    if (!Q || !K || !V || !O) return fail(AXHIP_ERR_NULL_ARG, "sdpa_fwd_rows: NULL tensor");
    if (B < 0 || H <= 0 || S < 0) return fail(AXHIP_ERR_SHAPE, "sdpa_fwd_rows: bad extent");
    if (!sdpa_fusable(dk))
        return fail(AXHIP_ERR_NOT_IMPLEMENTED, "sdpa_fwd_rows: head size %lld (multiples of 4 up to 128 only)", (long long)dk);
    if (ld < H * dk || ldo < H * dk || ld % 4 != 0 || ldo % 4 != 0 || ld > (1 << 22))
        return fail(AXHIP_ERR_SHAPE, "sdpa_fwd_rows: row pitch must hold H * dk floats and be a multiple of 4");
    if ((((uintptr_t)Q | (uintptr_t)K | (uintptr_t)V | (uintptr_t)O) & 15) != 0)
        return fail(AXHIP_ERR_SHAPE, "sdpa_fwd_rows: tensors must be 16-byte aligned");
    if (B == 0 || S == 0) return AXHIP_OK;
    if (B > 0x7fffffff / H || (S + 127) / 128 * (B * H) > 0x7fffffff)
        return fail(AXHIP_ERR_SHAPE, "sdpa_fwd_rows: too many tiles");
    return sdpa_fused(Q, K, V, O, L, B * H, S, dk, scale, causal, H, ld, ldo);
}
