// Shared host/device definitions for the gfx950 BERT encoder engine.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>

namespace cubert {

enum Precision : int { kF32 = 0, kBF16 = 1, kF32Split = 2 };   // kF32Split: GEMM operands only, float32 in the split layout below

struct Dims {
    int hidden = 768;
    int layers = 12;
    int heads = 12;
    int inter = 3072;
    int vocab = 30522;
    int max_pos = 512;
    int type_vocab = 2;
};

// bf16 storage type used on the host side of the launch interface.
typedef uint16_t bf16_t;

// Round-to-nearest-even float -> bf16 (host).
inline bf16_t f32_to_bf16_host(float f) {
    uint32_t u;
    __builtin_memcpy(&u, &f, 4);
    if ((u & 0x7fffffffu) > 0x7f800000u) return bf16_t((u >> 16) | 0x40);   // quiet NaN
    u += 0x7fffu + ((u >> 16) & 1u);
    return bf16_t(u >> 16);
}

inline int round_up(int x, int m) { return (x + m - 1) / m * m; }

// ---- packed operand layout ----------------------------------------------
// A matrix [rows, row_bytes] that feeds a GEMM as a K-contiguous operand can be
// kept "packed": 16 KiB blocks of 256 rows x 64 bytes, block (rt, kb) at
// (rt * KB + kb) * 16384 with KB = row_bytes / 64, and inside a block the
// 16-byte chunk c of row r at r * 64 + ((c ^ swz(r)) * 16),
// swz(r) = (r >> 2) & 3.  A block is exactly the LDS image the GEMM kernels
// compute from, so a tile load is a contiguous copy made of full cache lines.
// Rows are padded to a multiple of 256.  With this swizzle the kernels'
// ds_read_b128 fragment reads (lane = row, 64-byte row pitch) run at the full
// 256 bytes per clock of the LDS; measured alternatives: none 85, xor of
// (r>>1)^(r>>3) 158 bytes per clock.
//
// The "units" layout (bf16) has the same 16 KiB blocks of 256 rows x 32 k, but inside a block 1 KiB units of 32 rows x 16 k in
// the register layout of the 32x32x16 MFMA operand (lane 32 (k / 8 % 2) + row % 32 owns 16 bytes): unit (r / 32 % 8, k / 16
// % 2).  A GEMM epilogue writes it straight from the accumulators, a kernel without an LDS-staged loop loads its operands from
// it as they are, and LDS fragment reads are linear in the lane; writers that hold whole rows (LayerNorm) prefer the
// packed layout, whose pieces of a row are 64 bytes instead of 16.
// Attention kernels (launch_attention's `variant`).
constexpr int kAttnAuto = 0, kAttnPerHead = 1, kAttnSplitKeys = 2, kAttnSplitKeys8 = 3;      // 8: float32 only, eight waves instead of four
constexpr int kAttnSplitMaxWorkgroups = 768; // B * heads * ceil(S / 32) up to which kAttnAuto takes the key-split kernel

__host__ __device__ inline int packed_swizzle(int r) { return (r >> 2) & 3; }
__host__ __device__ inline size_t packed_bytes(size_t rows, size_t row_bytes) {
    return (rows + 255) / 256 * (row_bytes / 64) * 16384;
}
// Byte offset of the byte `kbyte` (within its row) of row r; KB = row_bytes / 64.
__host__ __device__ inline size_t packed_offset(int r, int kbyte, int KB) {
    const int rp = r & 255;
    const int sw = packed_swizzle(rp);
    return ((size_t)(r >> 8) * KB + (kbyte >> 6)) * 16384 + rp * 64 + ((((kbyte >> 4) & 3) ^ sw) << 4) +
           (kbyte & 15);
}

__host__ __device__ inline size_t units_offset(int r, int kbyte, int KB) {
    return ((size_t)(r >> 8) * KB + (kbyte >> 6)) * 16384 + ((r >> 5) & 7) * 2048 + ((kbyte >> 4) & 3) * 512 + (r & 31) * 16 + (kbyte & 15);
}

// ---- split operand layout --------------------------------------------------
// float32 operands of a GEMM, every element as the exact sum of three bfloat16 numbers (split_bf16x3): plane 0 is the
// element rounded to bf16, plane 1 what is left rounded to bf16, plane 2 the rest (at most 7 bits, so exact).  Six of the
// nine products of two such elements give their float32 product: the dropped ones (planes 1 and 2, 2 and 2) are below
// 2^-24 of it at the worst and 2^-28 typically, less than one rounding of a float32 multiply-add chain.  gfx950 multiplies
// bf16 sixteen times as fast as float32 on the matrix pipe, so six products take 0.375 of the time of one.
// Layout: 1 KiB units of 32 rows x 16 k x one plane, in the register layout of the 32x32x16 MFMA operand (lane
// 32 (k / 8 % 2) + row % 32 owns 16 bytes), unit (row / 32, k / 16, plane) at ((row / 32 * (K / 16) + k / 16) * 3 + plane).
// Rows are padded to a multiple of 32.
enum OperandLayout : int { kRowMajor = 0, kPacked = 1, kSplit = 2, kUnits = 3 };
__host__ __device__ inline size_t split_bytes(size_t rows, size_t K) { return (rows + 31) / 32 * (K / 16) * 3072; }
// Byte offset of plane 0 of element (r, k); planes 1 and 2 follow 1024 and 2048 bytes further.
__host__ __device__ inline size_t split_offset(int r, int k, int K) {
    return ((size_t)(r >> 5) * (K >> 4) + (k >> 4)) * 3072 + ((k >> 3) & 1) * 512 + (r & 31) * 16 + (k & 7) * 2;
}
// float32 Q, K, V of the attention (attention_f32.hip): per (batch, head) and block of 32 positions twelve units (four
// groups of 16 features x three planes).  V's positions are permuted inside a half unit (half: features 8 half .. + 7 of the
// 16) so that its transposing LDS reads spread over the banks.
__host__ __device__ inline int attn_v_slot(int pos, int half, int kk) { return pos ^ (4 * half + 8 * (kk & 1)); }
#if defined(__HIPCC__)
// (Within 0.4 % of the largest float the first plane rounds to infinity; infinities and NaNs end as NaN.)
__device__ __forceinline__ void split_bf16x3(float x, __bf16& p0, __bf16& p1, __bf16& p2) {
#pragma clang fp contract(off)
    p0 = (__bf16)x;
    const float r1 = x - (float)p0;
    p1 = (__bf16)r1;
    p2 = (__bf16)(r1 - (float)p1);
}
#endif

// ---- LayerNorm statistics -------------------------------------------------
// Every LayerNorm of the engine (the row kernels and the GEMM epilogue that normalises) forms its
// row statistics the same way, so that a row gets the same bits whichever kernel handles it.
// The row is cut into slots of 128 features; in a slot 32 lanes hold four consecutive features each.
// Per slot (ln_slot_stats): the sum, (a + b) + (c + d) per lane combined by ln_half_wave_sum, and M2, the
// sum of squared distances from the slot's own mean, taken the same way.  ln_row_mean adds the slot sums
// in slot order starting from zero; ln_merge_slot adds, again in slot order, M2_s + n_s (mean_s - mean)^2
// (the pairwise update of Chan et al. for a known total mean); ln_finalize turns the total into
// 1 / sigma (biased variance, eps 1e-12 inside the square root: modeling.py:168-172).  No difference of
// large squares is formed anywhere, so a row whose mean is many sigma away from zero keeps its
// precision, as with the running (Welford) statistics of cuda_bert/ops/layernorm.cu:27-67, 100-135.
// The helpers spell out their fused multiply-adds so that every caller compiles to the same arithmetic.
#if defined(__HIPCC__)
template <int CTRL>
__device__ __forceinline__ float ln_dpp_lanes(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
// v combined with the value of the lane 32 further (or back): gfx950's v_permlane32_swap exchanges the upper half of
// one register with the lower half of another, so of two copies of v one ends up holding v of the lower lane of each
// pair in both halves and the other v of the upper lane; sum and maximum commute, so the result has the bits of
// v + shfl_xor(v, 32) / max(v, shfl_xor(v, 32)) without the trip through the LDS crossbar.  (Inline asm, with the wait
// states the instruction needs after a vector write of its operands and before a vector read of its results: the
// compiler's builtin returns the first register twice.)
__device__ __forceinline__ void half_swap(float& a, float& b) {
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
}
// The same for lanes 16 apart (rows of 16 lanes: the odd rows of one register with the even rows of the other).
__device__ __forceinline__ float row_swap_sum(float v) {
    float a = v, b = v;
    asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
    return a + b;
}
// Accumulator layout -> split layout.  x: four consecutive values (features or k) of group 2 u and four of group 2 u + 1 of
// my row, the halves lane / 32 of the two groups of eight; after exchanging with lane ^ 32 a lane holds all eight of group
// 2 u + lane / 32, i.e. the 16 bytes per plane of a unit that are its own.  Every lane of the wave takes part.
typedef __attribute__((ext_vector_type(4))) unsigned int split_u32x4_t;
__device__ __forceinline__ void split_unit_rows(const float (&x)[8], split_u32x4_t (&planes)[3]) {
    typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;
    float w[3][4];                       // [plane][pairs 0 1, 2 3 of group 2 u; of group 2 u + 1], as bits
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        __bf16 a0, a1, a2, b0, b1, b2;
        split_bf16x3(x[2 * i], a0, a1, a2);
        split_bf16x3(x[2 * i + 1], b0, b1, b2);
        w[0][i] = __builtin_bit_cast(float, bf16x2_t{a0, b0});
        w[1][i] = __builtin_bit_cast(float, bf16x2_t{a1, b1});
        w[2][i] = __builtin_bit_cast(float, bf16x2_t{a2, b2});
    }
#pragma unroll
    for (int p = 0; p < 3; ++p) {
        half_swap(w[p][0], w[p][2]);
        half_swap(w[p][1], w[p][3]);
        planes[p] = split_u32x4_t{__builtin_bit_cast(unsigned, w[p][0]), __builtin_bit_cast(unsigned, w[p][1]),
                                  __builtin_bit_cast(unsigned, w[p][2]), __builtin_bit_cast(unsigned, w[p][3])};
    }
}
__device__ __forceinline__ float half_swap_sum(float v) {
    float a = v, b = v;
    half_swap(a, b);
    return a + b;
}
__device__ __forceinline__ float half_swap_max(float v) {
    float a = v, b = v;
    half_swap(a, b);
    return fmaxf(a, b);
}
// Sum over the 32 lanes that share lane / 32; every lane gets the same bits (the additions are
// pairwise and commutative).  The pairs: lanes 8, 4, 2, 16 and last 1 apart.  The GEMM epilogue that normalises
// holds a row in the MFMA accumulator layout, where quad 8 i + 2 qd + g of a slot is block i, group qd of lane half g: with the
// neighbours last it adds a lane's sixteen quads in registers and crosses lanes once (ln_tree16, then half_swap_sum).
__device__ __forceinline__ float ln_half_wave_sum(float v) {
    v += ln_dpp_lanes<0x128>(v);      // row_ror 8: lane ^ 8
    v += ln_dpp_lanes<0x124>(v);      // row_ror 4: lane ^ 4, now that lanes 8 apart agree
    v += ln_dpp_lanes<0x122>(v);      // row_ror 2: lane ^ 2
    v = row_swap_sum(v);              // lane ^ 16
    v += ln_dpp_lanes<0xB1>(v);       // quad_perm [1,0,3,2]: lane ^ 1
    return v;
}
// The same sum, but for the last step, of values one lane holds: v[4 i + qd] is what lane 8 i + 2 qd would hold above.
__device__ __forceinline__ float ln_tree16(const float (&v)[16]) {
    const float a = ((v[0] + v[4]) + (v[2] + v[6])) + ((v[1] + v[5]) + (v[3] + v[7]));
    const float b = ((v[8] + v[12]) + (v[10] + v[14])) + ((v[9] + v[13]) + (v[11] + v[15]));
    return a + b;
}
__device__ __forceinline__ float ln_sum4(float a, float b, float c, float d) { return (a + b) + (c + d); }
__device__ __forceinline__ float ln_sumsq4(float a, float b, float c, float d) {
#pragma clang fp contract(off)
    return __builtin_fmaf(a, a, b * b) + __builtin_fmaf(c, c, d * d);
}
// Statistics of one slot.  (a, b, c, d): this lane's four features, zeros if the lane lies past the end of
// the row (`in` false); inv_count = 1 / (features of the row inside this slot), 1 / 128 for a full slot.
__device__ __forceinline__ void ln_slot_stats(float a, float b, float c, float d, bool in, float inv_count, float* sum,
                                              float* m2) {
#pragma clang fp contract(off)
    const float s = ln_half_wave_sum(ln_sum4(a, b, c, d));
    const float mu = s * inv_count;
    const float da = in ? a - mu : 0.0f, db = in ? b - mu : 0.0f, dc = in ? c - mu : 0.0f, dd = in ? d - mu : 0.0f;
    *sum = s;
    *m2 = ln_half_wave_sum(ln_sumsq4(da, db, dc, dd));
}
__device__ __forceinline__ float ln_row_mean(float sum_of_slot_sums, float inv_n) {
#pragma clang fp contract(off)
    return sum_of_slot_sums * inv_n;
}
// m2 + (M2 of a slot about the row mean); count = features in the slot (0: the slot lies past the row).
__device__ __forceinline__ float ln_merge_slot(float m2, float slot_sum, float slot_m2, float count, float inv_count, float mean) {
#pragma clang fp contract(off)
    const float dm = slot_sum * inv_count - mean;
    return m2 + __builtin_fmaf(count * dm, dm, slot_m2);
}
__device__ __forceinline__ float ln_finalize(float m2, float inv_n) {
#pragma clang fp contract(off)
    return 1.0f / sqrtf(m2 * inv_n + 1e-12f);
}
__device__ __forceinline__ float ln_scale(float x, float mean, float rstd) {
#pragma clang fp contract(off)
    return (x - mean) * rstd;
}
__device__ __forceinline__ float ln_affine(float z, float gamma, float beta) { return __builtin_fmaf(gamma, z, beta); }
__device__ __forceinline__ float ln_apply(float x, float mean, float rstd, float gamma, float beta) {
    return ln_affine(ln_scale(x, mean, rstd), gamma, beta);
}
#endif

// Thread-local last error text (returned by cubert_last_error()).
void set_error(const std::string& msg);
const char* get_error();

#define CUBERT_HIP_OK(expr)                                                              \
    do {                                                                                 \
        hipError_t _e = (expr);                                                          \
        if (_e != hipSuccess) {                                                          \
            ::cubert::set_error(std::string(#expr) + " failed: " + hipGetErrorString(_e)); \
            return false;                                                                \
        }                                                                                \
    } while (0)

}  // namespace cubert
