// float32 fused self-attention for head dim 64 on the bf16 matrix pipe (gfx950):
//   ctx = softmax(Q K^T * scale + maskadd) V        per (batch, head)
// with Q, K, V float32 as three bf16 planes (common.h: split_bf16x3), six plane products per float32 product, and the
// probabilities split the same way in registers.
//
// Block arithmetic as in attention.hip: one wave owns 32 queries and walks the keys in blocks of 32, scores transposed
// (keys x queries) so that a lane owns one query, online softmax in the exp2 domain with a lazily moved reference
// exponent, key blocks without a visible key skipped.  A block costs 48 MFMAs against some 800 clocks of vector work, so
// the matrix pipe is what the kernel runs on; K and V of a key block are 12 KiB each and are brought into the LDS once for
// the workgroup's four waves, one block ahead (two stages), which leaves room for three workgroups per CU.
//
// Operand layout, written by the QKV GEMM's epilogue (gemm_split.hip) and chosen so that it is the register layout of the
// MFMA operand: per (batch, head) and block of 32 positions twelve 1 KiB units, unit (kk, plane) = features 16 kk .. + 15;
// the 16 bytes of position r, features 16 kk + 8 g .. + 7 at 512 g + 16 (r % 32).  V needs its second MFMA operand
// transposed: ds_read_b64_tr_b16 takes, per group of 16 lanes, four features' pieces of 8 bytes of four positions, and
// with position r of V at slot r ^ (4 g + 8 (kk & 1)) (attn_v_slot) the pieces of two groups lie in distinct banks.
//
// 128 sequences of up to 200 positions, 16 heads, a quarter of it padding: 137 us; 16 x 512, 12 heads: 73 us.  (Float32 MFMA,
// K and V read from memory by every wave, attention.hip: 310 and 157 us.)
#include <algorithm>

#include "kernels.h"
#include "l2_touch.h"

namespace cubert {
namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(16))) float f32x16_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4_t;
typedef __attribute__((ext_vector_type(4))) short s16x4_t;
typedef __attribute__((ext_vector_type(8))) short s16x8_t;
typedef __attribute__((address_space(3))) void* lds_ptr_t;

constexpr int kUnit = 1024, kBlockBytes = 12 * kUnit;      // one key block of one operand
constexpr int kStage = 2 * kBlockBytes + 256;

__device__ __forceinline__ bf16x8_t tr_read(const unsigned char* stage, int piece) {
    const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        reinterpret_cast<__attribute__((address_space(3))) s16x4_t*>((__attribute__((address_space(3))) unsigned char*)(stage + piece)));
    // the same features of the positions 8 further: bit 3 of the slot
    const s16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        reinterpret_cast<__attribute__((address_space(3))) s16x4_t*>((__attribute__((address_space(3))) unsigned char*)(stage + (piece ^ 128))));
    return __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

// My piece of a transposing read in a block of V (f = 0): position 4 g + (i >> 2), features 4 (i & 3) .. + 3 of unit row kk = 2 db + (l32 >> 4).
__device__ __forceinline__ void v_pieces(int l32, int g, int (&vpiece)[2]) {
#pragma unroll
    for (int db = 0; db < 2; ++db) {
        const int i16 = l32 & 15, kk = 2 * db + (l32 >> 4), half = (i16 & 3) >> 1;
        vpiece[db] = kk * 3 * kUnit + half * 512 + attn_v_slot(4 * g + (i16 >> 2), half, kk) * 16 + (i16 & 1) * 8;
    }
}

// One block of 32 keys for the wave's 32 queries: kfrag(kk, p) is the fragment of K (features 16 kk .., plane p), vblk the block
// of V and mask its mask terms, both in the LDS.  plain: all 32 keys are visible, with a zero mask term.
template <class KFrag>
__device__ __forceinline__ void key_block(const KFrag& kfrag, const u32x4_t (&qf)[4][3], const unsigned char* vblk, const int (&vpiece)[2],
                                      const unsigned char* mask, bool plain, int g, float scale_log2e, f32x16_t (&o)[2],
                                      float& run_max, float& run_sum) {
    f32x16_t sc;
#pragma unroll
    for (int e = 0; e < 16; ++e) sc[e] = 0.0f;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
        u32x4_t kf[3];
#pragma unroll
        for (int p = 0; p < 3; ++p) kf[p] = kfrag(kk, p);
#define CUBERT_QK(a, c) sc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, kf[a]), __builtin_bit_cast(bf16x8_t, qf[kk][c]), sc, 0, 0, 0)
        CUBERT_QK(0, 0); CUBERT_QK(0, 1); CUBERT_QK(1, 0); CUBERT_QK(1, 1); CUBERT_QK(0, 2); CUBERT_QK(2, 0);
#undef CUBERT_QK
    }
    float blk_max = -INFINITY;
    if (plain) {
#pragma unroll
        for (int e = 0; e < 16; ++e) blk_max = fmaxf(blk_max, sc[e]);
        blk_max *= scale_log2e;                          // scale_log2e > 0
    } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const f32x4_t m4 = *reinterpret_cast<const f32x4_t*>(mask + (8 * j + 4 * g) * 4);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float t = fmaf(sc[4 * j + e], scale_log2e, m4[e] * 1.4426950408889634f);
                sc[4 * j + e] = t;
                blk_max = fmaxf(blk_max, t);
            }
        }
    }
    blk_max = half_swap_max(blk_max);
    if (__ballot(blk_max > run_max + 20.0f) != 0ull) {
        const float new_max = fmaxf(run_max, blk_max);
        const float alpha = __builtin_amdgcn_exp2f(run_max - new_max);     // 1 for the lanes that stay
        run_sum *= alpha;
        run_max = new_max;
#pragma unroll
        for (int db = 0; db < 2; ++db)
#pragma unroll
            for (int e = 0; e < 16; ++e) o[db][e] *= alpha;
    }
    const float neg_ref = -run_max, mul = plain ? scale_log2e : 1.0f;
    float blk_sum = 0.0f;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        const float pv = __builtin_amdgcn_exp2f(fmaf(sc[e], mul, neg_ref));
        sc[e] = pv;
        blk_sum += pv;
    }
    run_sum += half_swap_sum(blk_sum);
    // ctx^T += V^T (rows = head features) x P^T (column = my query): positions 16 f + {4g..4g+3, 8+4g..8+4g+3}
#pragma unroll
    for (int f = 0; f < 2; ++f) {
        bf16x8_t pf[3];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            __bf16 s0, s1, s2;
            split_bf16x3(sc[8 * f + e], s0, s1, s2);
            pf[0][e] = s0; pf[1][e] = s1; pf[2][e] = s2;
        }
#pragma unroll
        for (int db = 0; db < 2; ++db) {
            bf16x8_t vf[3];
#pragma unroll
            for (int p = 0; p < 3; ++p) vf[p] = tr_read(vblk, (vpiece[db] + p * kUnit) ^ (f * 256));      // 16 positions further: bit 4 of the slot
#define CUBERT_PV(a, c) o[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[a], pf[c], o[db], 0, 0, 0)
            CUBERT_PV(0, 0); CUBERT_PV(0, 1); CUBERT_PV(1, 0); CUBERT_PV(1, 1); CUBERT_PV(0, 2); CUBERT_PV(2, 0);
#undef CUBERT_PV
        }
    }
}

__global__ __launch_bounds__(256, 2) void attention_f32_kernel(
    const unsigned char* __restrict__ q, const unsigned char* __restrict__ k, const unsigned char* __restrict__ v,
    const float* __restrict__ maskadd, unsigned char* __restrict__ ctx, int heads, int S, int Sp, float scale_log2e,
    const int* __restrict__ cu, int first_only) {
    __shared__ __attribute__((aligned(1024))) unsigned char stage0[kStage];      // K block, V block, mask terms
    __shared__ __attribute__((aligned(1024))) unsigned char stage1[kStage];

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l32 = lane & 31, g = lane >> 5;
    const int h = blockIdx.y, b = blockIdx.z;
    const int q0 = (blockIdx.x * 4 + wave) * 32;
    const int qlen = cu ? cu[b + 1] - cu[b] : S;
    if ((int)blockIdx.x * 128 >= qlen) return;                        // the whole workgroup: no barrier has been met
    const bool active = q0 < qlen && !(first_only && q0 != 0);        // idle waves still fetch their share of K and V
    const int nblk = Sp >> 5;
    const size_t bh = ((size_t)b * heads + h) * nblk * kBlockBytes;
    const float* mrow = maskadd + (size_t)b * Sp;

    // a wave fetches three units of K and three of V of every block
    const __amdgpu_buffer_rsrc_t kres = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char*>(k + bh), 0, nblk * kBlockBytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t vres = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char*>(v + bh), 0, nblk * kBlockBytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t mres = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(mrow), 0, Sp * 4, 0x00020000);
    auto issue = [&](unsigned char* stage, int blk) {
        // (lanes 32 and up fetch what nobody reads)
        if (wave == 0) __builtin_amdgcn_raw_ptr_buffer_load_lds(mres, (lds_ptr_t)(stage + 2 * kBlockBytes), 4, (blk * 32 + lane) * 4, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const int unit = wave * 3 + i;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(kres, (lds_ptr_t)(stage + unit * kUnit), 16, blk * kBlockBytes + unit * kUnit + lane * 16, 0, 0, 0);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(vres, (lds_ptr_t)(stage + kBlockBytes + unit * kUnit), 16, blk * kBlockBytes + unit * kUnit + lane * 16, 0, 0, 0);
        }
    };
    issue(stage0, 0);

    u32x4_t qf[4][3];
    {
        const unsigned char* qb = q + bh + (size_t)(q0 < Sp ? q0 >> 5 : 0) * kBlockBytes + lane * 16;
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
#pragma unroll
            for (int p = 0; p < 3; ++p) qf[kk][p] = *reinterpret_cast<const u32x4_t*>(qb + (kk * 3 + p) * kUnit);
    }

    // live: a key of the block is visible; plain: all 32 are, with a zero mask term
    unsigned long long live = 0ull, plain = 0ull;
#pragma unroll 4
    for (int i = 0; i < nblk && i < 64; i += 2) {
        const int col = i * 32 + lane;
        const float m = col < Sp ? mrow[col] : -INFINITY;
        const unsigned long long vis = __ballot(m > -5000.0f), zero = __ballot(m == 0.0f);
        if ((unsigned)vis) live |= 1ull << i;
        if (vis >> 32) live |= 2ull << i;
        if ((unsigned)zero == 0xffffffffu) plain |= 1ull << i;
        if ((zero >> 32) == 0xffffffffull) plain |= 2ull << i;
    }
    if (live == 0ull || nblk > 64) { live = ~0ull; plain = nblk > 64 ? 0ull : plain; }
    auto next_block = [&](int from) {
        if (nblk > 64) return from;
        const unsigned long long rest = from < 64 ? live & (~0ull << from) : 0ull;
        return rest ? __builtin_ctzll(rest) : nblk;
    };

    f32x16_t o[2];
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[db][e] = 0.0f;
    float run_max = -INFINITY, run_sum = 0.0f;
    int vpiece[2];
    v_pieces(l32, g, vpiece);

    auto compute = [&](const unsigned char* stage, int blk) {
        key_block([&](int kk, int p) { return *reinterpret_cast<const u32x4_t*>(stage + (kk * 3 + p) * kUnit + lane * 16); }, qf, stage + kBlockBytes, vpiece,
                  stage + 2 * kBlockBytes, nblk <= 64 && ((plain >> blk) & 1ull), g, scale_log2e, o, run_max, run_sum);
    };
    // everything I asked for has landed, and so has everybody else's after the barrier (the transposing reads are not
    // ordered behind the memory-to-LDS loads by the compiler)
    auto landed = [&]() {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    };

    landed();
    // (the compiler, which does not know that, would wait for the queries inside the loop and with them for the loads in flight there)
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
#pragma unroll
        for (int p = 0; p < 3; ++p) asm volatile("" : "+v"(qf[kk][p]));
    for (int blk = 0;;) {
        int next = next_block(blk + 1);
        if (next < nblk) issue(stage1, next);
        if (active) compute(stage0, blk);
        if (next >= nblk) break;
        landed();
        blk = next;
        next = next_block(blk + 1);
        if (next < nblk) issue(stage0, next);
        if (active) compute(stage1, blk);
        if (next >= nblk) break;
        landed();
        blk = next;
    }

    // ---- normalise and store, split: after exchanging halves a lane holds eight features of its query ----
    const int qi = q0 + l32;
    if (!active) return;                                     // wave-uniform
    const float inv = 1.0f / run_sum;
    const bool store = qi < qlen && !(first_only && qi != 0);
    const size_t row = first_only ? (size_t)b : (cu ? (size_t)cu[b] : (size_t)b * S) + qi;
    const int hidden = heads * 64;
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            float x[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = o[db][8 * u + e] * inv;
            u32x4_t pl[3];
            split_unit_rows(x, pl);
            unsigned char* dst = ctx + split_offset((int)row, h * 64 + 32 * db + 16 * u + 8 * g, hidden);
            if (store) {
#pragma unroll
                for (int p = 0; p < 3; ++p) *reinterpret_cast<u32x4_t*>(dst + p * kUnit) = pl[p];
            }
        }
}

// Short batches: one workgroup of the kernel above owns 128 queries, so a line or a few occupy a fraction of the CUs and every
// wave walks all key blocks in turn, a round trip and a barrier for each.  Here a workgroup owns 32 queries of a (batch, head)
// and its NW waves share the KEYS: wave w takes the blocks w, w + NW, ...  A wave requests its queries, its fragments of K
// (the layout in memory is the operand's), its block of V and the mask terms (both straight into wave-private LDS) in one round
// trip and meets the others once, at the end, where the partials (reference exponent, row sum, context) are merged:
// ctx = sum_w 2^(ref_w - top) o_w / sum_w 2^(ref_w - top) sum_w, top the largest reference.  No key block is skipped: a masked
// key's probability underflows to exactly zero and a wave all of whose keys are masked gets weight zero.
template <int NW>
__global__ __launch_bounds__(NW * 64, NW == 4 ? 2 : 1) void attention_f32_split_kernel(
    const unsigned char* __restrict__ q, const unsigned char* __restrict__ k, const unsigned char* __restrict__ v,
    const float* __restrict__ maskadd, const int* __restrict__ cu, int heads, int S, int Sp, int query_blocks,
    unsigned char* __restrict__ ctx, float scale_log2e, int first_only, const WeightsAhead ahead) {
    constexpr int OSTRIDE = 68;                          // floats per query row of a partial context
    constexpr int WBYTES = kBlockBytes + 256;            // a block of V, later the partial context (8.5 KiB), and 64 mask terms
    static_assert(32 * OSTRIDE * 4 <= kBlockBytes, "the partial context takes the place of V");
    __shared__ __attribute__((aligned(1024))) unsigned char sW[NW * WBYTES];
    __shared__ float sRef[NW][32], sSum[NW][32];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, g = lane >> 5;
    const int h = blockIdx.x, b = blockIdx.y, q0 = blockIdx.z * 32;
    if ((int)blockIdx.z >= query_blocks) {               // the workgroups after the queries: weights for the next launch
        l2_touch<true>(ahead, l2_share_after_planes(h, b, blockIdx.z, gridDim.x, gridDim.y, gridDim.z, query_blocks, NW, wave), lane);
        return;
    }
    const int qlen = cu ? cu[b + 1] - cu[b] : S;
    if (q0 >= qlen) return;                              // the whole workgroup: no barrier has been met
    const int nblk = Sp >> 5;
    const size_t bh = ((size_t)b * heads + h) * nblk * kBlockBytes;
    unsigned char* myV = sW + wave * WBYTES;
    unsigned char* myM = myV + kBlockBytes;
    const __amdgpu_buffer_rsrc_t vres = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char*>(v + bh), 0, nblk * kBlockBytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t mres = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(maskadd + (size_t)b * Sp), 0, Sp * 4, 0x00020000);

    u32x4_t qf[4][3], kf[4][3];
    const unsigned char* qb = q + bh + (size_t)blockIdx.z * kBlockBytes + lane * 16;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
#pragma unroll
        for (int p = 0; p < 3; ++p) qf[kk][p] = *reinterpret_cast<const u32x4_t*>(qb + (kk * 3 + p) * kUnit);

    f32x16_t o[2];
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[db][e] = 0.0f;
    float run_max = -INFINITY, run_sum = 0.0f;
    int vpiece[2];
    v_pieces(l32, g, vpiece);

    for (int blk = wave; blk < nblk; blk += NW) {
        const unsigned char* kb = k + bh + (size_t)blk * kBlockBytes + lane * 16;
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
#pragma unroll
            for (int p = 0; p < 3; ++p) kf[kk][p] = *reinterpret_cast<const u32x4_t*>(kb + (kk * 3 + p) * kUnit);
#pragma unroll
        for (int i = 0; i < 12; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(vres, (lds_ptr_t)(myV + i * kUnit), 16, blk * kBlockBytes + i * kUnit + lane * 16, 0, 0, 0);
        // (lanes 32 and up fetch what nobody reads)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(mres, (lds_ptr_t)myM, 4, (blk * 32 + lane) * 4, 0, 0, 0);
        // nothing below may read this wave's LDS before all of it has landed (the transposing reads are not ordered behind the
        // memory-to-LDS loads by the compiler)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        const bool plain = __ballot(reinterpret_cast<const float*>(myM)[l32] == 0.0f) == ~0ull;
        key_block([&](int kk, int p) { return kf[kk][p]; }, qf, myV, vpiece, myM, plain, g, scale_log2e, o, run_max, run_sum);
        // the next round's memory-to-LDS loads stay behind this round's LDS reads, and those are done
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }

    // ---- the partials meet: wave w's context as [query][feature] over its V space ----
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    float* myO = reinterpret_cast<float*>(myV);
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
        for (int j = 0; j < 4; ++j)
            *reinterpret_cast<f32x4_t*>(myO + l32 * OSTRIDE + 32 * db + 8 * j + 4 * g) =
                f32x4_t{o[db][4 * j], o[db][4 * j + 1], o[db][4 * j + 2], o[db][4 * j + 3]};
    if (g == 0) { sRef[wave][l32] = run_max; sSum[wave][l32] = run_sum; }
    __syncthreads();
    constexpr int FPT = 32 / NW, TQ = 64 / FPT;          // features per thread, threads per query
    const int qi = tid / TQ, f0 = tid % TQ * FPT, qrow = q0 + qi;
    if (qrow >= qlen || (first_only && qrow != 0)) return;
    const int nw = nblk < NW ? nblk : NW;                // waves that held a key block
    float top = -INFINITY;
    for (int w = 0; w < nw; ++w) top = fmaxf(top, sRef[w][qi]);
    float den = 0.0f, acc[FPT];
#pragma unroll
    for (int e = 0; e < FPT; ++e) acc[e] = 0.0f;
    for (int w = 0; w < nw; ++w) {
        const float wgt = __builtin_amdgcn_exp2f(sRef[w][qi] - top);
        den = fmaf(wgt, sSum[w][qi], den);
        const float* src = reinterpret_cast<const float*>(sW + w * WBYTES) + qi * OSTRIDE + f0;
#pragma unroll
        for (int e = 0; e < FPT; e += 4) {
            const f32x4_t x4 = *reinterpret_cast<const f32x4_t*>(src + e);
#pragma unroll
            for (int c = 0; c < 4; ++c) acc[e + c] = fmaf(wgt, x4[c], acc[e + c]);
        }
    }
    const float inv = 1.0f / den;
    typedef __attribute__((ext_vector_type(FPT))) __bf16 bf16_t_v;
    bf16_t_v pl[3];
#pragma unroll
    for (int e = 0; e < FPT; ++e) {
        __bf16 s0, s1, s2;
        split_bf16x3(acc[e] * inv, s0, s1, s2);
        pl[0][e] = s0; pl[1][e] = s1; pl[2][e] = s2;
    }
    const size_t row = first_only ? (size_t)b : (cu ? (size_t)cu[b] : (size_t)b * S) + qrow;
    unsigned char* dst = ctx + split_offset((int)row, h * 64 + f0, heads * 64);
#pragma unroll
    for (int p = 0; p < 3; ++p) *reinterpret_cast<bf16_t_v*>(dst + p * kUnit) = pl[p];
}

}  // namespace

// The key-split kernel wins up to 768 blocks of 32 queries (B * heads * ceil(S / 32)), the eight-wave form of it while every
// workgroup has a CU to itself and there are more than four key blocks.  Microseconds, queries in fours / split by 4 / by 8:
// B=1 S=128 16 heads 8.7 / 5.0 / -, B=1 S=200 13.7 / 8.1 / 6.9, B=1 S=512 26.1 / 13.9 / 10.8 (256 blocks), B=4 S=200 14.9 / 10.4 / 12.8
// (448), B=8 S=200 12 heads 16.1 / 13.4 / 18.9 (672), B=16 S=128 12 heads 11.7 / 11.4 / - (768), 16 heads 13.8 / 17.9 / - (1024).
int attn_f32_variant(int B, int heads, int S, int max_blocks) {
    const int nblk = (S + 31) / 32;
    const long blocks = (long)B * heads * nblk;
    if (blocks > max_blocks || nblk > 65535) return kAttnPerHead;
    return nblk > 4 && blocks <= 256 ? kAttnSplitKeys8 : kAttnSplitKeys;
}

bool launch_attention_f32(const void* q, const void* k, const void* v, const float* maskadd, void* ctx, int B, int heads,
                          int S, int Sp, float scale, hipStream_t stream, const int* cu, bool first_only, int variant, const WeightsAhead& ahead) {
    if (B <= 0 || heads <= 0 || S <= 0) { set_error("attention: empty problem"); return false; }
    if (!(scale > 0.0f)) { set_error("attention: scale must be positive"); return false; }
    if (Sp % 32 != 0 || Sp < S || Sp - S >= 32 || (long)Sp * 384 >= (1L << 31)) {
        set_error("attention: Sp must be S rounded up to a multiple of 32");
        return false;
    }
    if (B > 65535 || heads > 65535) { set_error("attention: grid too large"); return false; }
    if (!q || !k || !v || !maskadd || !ctx ||
        ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(v) |
          reinterpret_cast<uintptr_t>(maskadd) | reinterpret_cast<uintptr_t>(ctx)) & 15)) {
        set_error("attention: null or misaligned operand");
        return false;
    }
    if (variant < kAttnAuto || variant > kAttnSplitKeys8) { set_error("attention: unknown variant"); return false; }
    if (variant == kAttnAuto) variant = attn_f32_variant(B, heads, S, kAttnSplitMaxWorkgroups);
    if (variant != kAttnPerHead) {
        if ((S + 31) / 32 > 65535) { set_error("attention: grid too large"); return false; }
        const bool eight = variant == kAttnSplitKeys8;
        const int blocks = first_only ? 1 : (S + 31) / 32;
        const dim3 sgrid(heads, B, std::min(65535, blocks + (l2_touch_workgroups<true>(ahead) / (eight ? 2 : 1) + heads * B - 1) / (heads * B)));
        auto kernel = eight ? attention_f32_split_kernel<8> : attention_f32_split_kernel<4>;
        hipLaunchKernelGGL(kernel, sgrid, dim3(eight ? 512 : 256), 0, stream, static_cast<const unsigned char*>(q), static_cast<const unsigned char*>(k),
                           static_cast<const unsigned char*>(v), maskadd, cu, heads, S, Sp, blocks, static_cast<unsigned char*>(ctx),
                           scale * 1.4426950408889634f, first_only ? 1 : 0, ahead);
        CUBERT_HIP_OK(hipGetLastError());
        return true;
    }
    const dim3 grid(first_only ? 1 : (S + 127) / 128, heads, B);
    hipLaunchKernelGGL(attention_f32_kernel, grid, dim3(256), 0, stream, static_cast<const unsigned char*>(q),
                       static_cast<const unsigned char*>(k), static_cast<const unsigned char*>(v), maskadd,
                       static_cast<unsigned char*>(ctx), heads, S, Sp, scale * 1.4426950408889634f, cu, first_only ? 1 : 0);
    CUBERT_HIP_OK(hipGetLastError());
    return true;
}

}  // namespace cubert
